"""The work that users of this framework have it do, as cases that can be timed and checked.

Six kinds, each through the package's public entry points:

  prefill   a prompt of S positions through the Talker (hip.Talker.prefill): the time before
            the first frame.  Output: the last position's residual, and where "then" is 1 also
            the hidden state of the decode step that follows on the cache rows just written.
  step      one decode step at a given cache length with host vectors in and out
            (hip.Talker.step), as the C engine's frame loop calls it.
  batch     one step of B streams at ragged positions over one copy of the weights
            (hip.TalkerBatch.step), the serving case.
  frames    whole frames on the device (hip.generate): codec head, sampling at the engine's
            defaults, the Code Predictor's 15 codes, the next input, the Talker step.
  decode    codes to 24 kHz audio in one call (hip.SpeechDecoder.decode).
  stream    the same, a few frames at a time (hip.SpeechDecoderStream), from a new utterance.

Models are the two of qwen3_tts_amd.synth (0.6B and 1.7B, 28 layers) and the speech decoder of
synth_sd, with random weights; weight types are the engine's three (bf16, int8 per row, q4_0).
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """qwen3-tts_amd has a hyphen in its folder's name: loaded by path as qwen3_tts_amd."""
    if "qwen3_tts_amd" not in sys.modules:
        d = os.path.join(ROOT, "qwen3-tts_amd")
        spec = importlib.util.spec_from_file_location("qwen3_tts_amd", os.path.join(d, "__init__.py"),
                                                      submodule_search_locations=[d])
        m = importlib.util.module_from_spec(spec)
        sys.modules["qwen3_tts_amd"] = m
        spec.loader.exec_module(m)
    from qwen3_tts_amd import hip, synth, synth_sd
    return hip, synth, synth_sd


hip, synth, synth_sd = _package()
DEV = "cuda"


def listed():
    return [
        # the smallest call: one decode step of the small model, short cache
        {"name": "step-0.6B-bf16-L256", "kind": "step", "model": "0.6B", "prec": "bf16", "L": 256},
        # the benchmark's headline setting, through the step entry that a C engine calls
        {"name": "step-1.7B-int8-L2048", "kind": "step", "model": "1.7B", "prec": "int8", "L": 2048},
        # a few frames of speech at the engine's sampling defaults
        {"name": "frames-0.6B-bf16-L256", "kind": "frames", "model": "0.6B", "prec": "bf16", "L": 256, "n": 4},
        # a busy server: 32 utterances in flight, from just begun to very long
        {"name": "batch-1.7B-int8-B32", "kind": "batch", "model": "1.7B", "prec": "int8", "B": 32, "lo": 128, "hi": 4000},
        # a small server in four-bit weights
        {"name": "batch-1.7B-q4-B12", "kind": "batch", "model": "1.7B", "prec": "q4", "B": 12, "lo": 200, "hi": 900},
        # a handful of streams of the small model in its checkpoint's own type
        {"name": "batch-0.6B-bf16-B6", "kind": "batch", "model": "0.6B", "prec": "bf16", "B": 6, "lo": 60, "hi": 500},
        # a short sentence, an odd length, up to the first step on its cache
        {"name": "prefill-0.6B-S45", "kind": "prefill", "model": "0.6B", "S": 45, "then": 1},
        # a sentence or two with a speaker prompt
        {"name": "prefill-1.7B-S128", "kind": "prefill", "model": "1.7B", "S": 128, "then": 0},
        # a paragraph with a reference recording (voice cloning)
        {"name": "prefill-1.7B-S512", "kind": "prefill", "model": "1.7B", "S": 512, "then": 0},
        # ten seconds of speech in one call
        {"name": "decode-125", "kind": "decode", "n": 125},
        # a long paragraph, 32 seconds: the largest call
        {"name": "decode-400", "kind": "decode", "n": 400},
        # live playback: the first 2.4 seconds in pieces of 0.8
        {"name": "stream-3x10", "kind": "stream", "chunk": 10, "chunks": 3},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("prefill", "prefill", "step", "batch", "frames", "decode", "decode", "stream"))
    model = rng.choice(("0.6B", "1.7B"))
    prec = rng.choice(("bf16", "int8", "q4"))
    if kind == "prefill":
        return {"kind": kind, "model": model, "S": _log(rng, 12, 1100), "then": rng.randint(0, 1)}
    if kind == "step":
        return {"kind": kind, "model": model, "prec": prec, "L": _log(rng, 1, 6000)}
    if kind == "batch":
        lo = _log(rng, 16, 400)
        return {"kind": kind, "model": model, "prec": prec, "B": _log(rng, 2, 48), "lo": lo, "hi": lo + _log(rng, 16, 2500)}
    if kind == "frames":
        return {"kind": kind, "model": model, "prec": rng.choice(("bf16", "int8")), "L": _log(rng, 16, 3000), "n": rng.randint(1, 4)}
    if kind == "decode":
        return {"kind": kind, "n": _log(rng, 4, 390)}
    return {"kind": kind, "chunk": _log(rng, 1, 48), "chunks": rng.randint(1, 4)}


# ---- the Talker's weights and inputs, from a seed --------------------------------------------


def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + stream) & 0x7FFFFFFFFFFF)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _quantize(w, prec):
    """w f32 [rows][cols] in the reference's encoding: bf16 bits; int8 rows and their scales;
    or q4_0 blocks of 32 (f16 scale, then byte i = element 2i low, 2i + 1 high, each + 8)."""
    if prec == "bf16":
        return w.bfloat16(), None
    if prec == "int8":
        s = w.abs().amax(1) / 127.0
        return (w / s[:, None]).round().clamp(-127, 127).to(torch.int8), s
    b = w.view(w.shape[0], -1, 32)
    s = (b.abs().amax(2) / 7.5).half()
    q = ((b / s.float()[..., None]).round().clamp(-8, 7) + 8).to(torch.uint8)
    qs = q[..., 0::2] | (q[..., 1::2] << 4)
    return torch.cat((s.view(torch.uint8).view(*s.shape, 2), qs), 2).contiguous(), None


def _dequantize(m, prec):
    """float64 [rows][cols] of what _quantize made."""
    w, s = m
    if prec == "bf16":
        return w.double()
    if prec == "int8":
        return w.double() * s.double()[:, None]
    sc = w[..., :2].contiguous().view(torch.float16)[..., 0].double()
    q = torch.stack((w[..., 2:] & 15, w[..., 2:] >> 4), 3).flatten(2).double() - 8.0
    return (q * sc[..., None]).flatten(1)


def _dims(model, cp=False):
    s = synth.SHAPES[model]
    if cp:
        return s.cp_hidden, s.cp_inter, s.cp_heads, s.cp_kv_heads, s.cp_layers
    return s.hidden, s.inter, s.heads, s.kv_heads, s.layers


def _layers(model, prec, seed):
    """The Talker's layers on the GPU: matrices ~ N(0, 0.02), gains 1 + N(0, 0.1)."""
    H, F, nh, nkv, nl = _dims(model)
    g = _gen(seed, 1)
    out = []
    for _ in range(nl):
        d = {}
        for nm, r, c in (("q", nh * 128, H), ("k", nkv * 128, H), ("v", nkv * 128, H), ("o", H, nh * 128),
                         ("gate_up", 2 * F, H), ("down", H, F)):
            d[nm] = _quantize(0.02 * _randn(g, r, c), prec)
        for nm, n in (("input_norm", H), ("post_attn_norm", H), ("q_norm", 128), ("k_norm", 128)):
            d[nm] = 1.0 + 0.1 * _randn(g, n)
        out.append(d)
    return out, 1.0 + 0.1 * _randn(g, H)


class _Mem:
    """Device memory in the place of a host array: hip.Talker takes its address."""

    def __init__(self, t):
        self.t = t
        self.ctypes = self

    @property
    def data(self):
        return self.t.data_ptr()


ROPE_LEN = 8192
_ROPE = synth.rope_tables(128, 1e6, ROPE_LEN)


def _kv_cap(n):
    """The cache's capacity for n positions: doubled from 512 as the engine's cache grows."""
    c = 512
    while c < n:
        c *= 2
    return min(c, ROPE_LEN)


def _talker(model, prec, seed, kv_max):
    layers, fn = _layers(model, prec, seed)
    put = []
    for d in layers:
        e = {nm: d[nm].cpu().numpy() for nm in ("input_norm", "post_attn_norm", "q_norm", "k_norm")}
        for nm in ("q", "k", "v", "o", "gate_up", "down"):
            w, s = d[nm]
            e[nm] = (_Mem(w), None if s is None else _Mem(s))
        put.append(e)
    torch.cuda.synchronize()
    return hip.Talker(synth.SHAPES[model], put, fn.cpu().numpy(), *_ROPE, hip.PREC["q4_0" if prec == "q4" else prec], kv_max)


def _cache(model, seed, n):
    """K and V rows of n positions, bf16 [layers][n][kv_dim]: keys are normed per head
    (about N(0, 1)), values are a projection's (about N(0, 0.7))."""
    _, _, _, nkv, nl = _dims(model)
    g = _gen(seed, 2)
    k = torch.randn(nl, n, nkv * 128, generator=g, device=DEV, dtype=torch.bfloat16)
    v = 0.7 * torch.randn(nl, n, nkv * 128, generator=g, device=DEV, dtype=torch.bfloat16)
    return k, v


def _bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def _embeds(model, seed, n):
    """Inputs: sums of 16 embedding rows ~ N(0, 0.02)."""
    return 0.08 * _randn(_gen(seed, 3), n, _dims(model)[0])


def _lens(c):
    """The streams' lengths, evenly from lo to hi, in an order with no trend."""
    B = c["B"]
    v = [c["lo"] + (c["hi"] - c["lo"]) * i // max(1, B - 1) for i in range(B)]
    step = next(s for s in (7, 5, 3, 11, 13, 1) if math.gcd(s, B) == 1)
    return [v[i * step % B] for i in range(B)]


def _starts(c, lens):
    """Where each stream's rows begin in the one pool of cache rows that is drawn."""
    return [37 * b % 256 for b in range(len(lens))], max(lens) + 256


CP_KEYS = ("talker.code_predictor.", "talker.model.codec_embedding.", "talker.codec_head.")


def _cp_tensors(model, seed):
    """The Code Predictor's tensors and the codec embeddings and head, bf16 bits on the host."""
    g = _gen(seed, 4)
    out = {}
    for name, shape, kind in synth.tensor_specs(synth.SHAPES[model]):
        if name.startswith(CP_KEYS):
            t = _randn(g, *shape)
            out[name] = _bits((1.0 + 0.1 * t if kind == "n" else 0.02 * t).bfloat16())
    return out


FRAME0 = 50                       # the frame index that a "frames" case starts at
SAMPLING = dict(temp=0.9, top_k=50, top_p=1.0, rep=1.05)


def _frame_inputs(c, seed):
    H = _dims(c["model"])[0]
    g = _gen(seed, 5)
    prev = torch.randint(0, 2048, (FRAME0,), generator=g, device=DEV).cpu().numpy().astype(np.int32)
    return (0.02 * _randn(g, H)).cpu().numpy(), _randn(g, H).cpu().numpy(), prev, int(seed) & 0x7FFFFFFF


# ---- the speech decoder's weights and codes ----------------------------------------------------


def _sd_tensors(seed):
    """synth_sd's tensors and distributions, drawn on the GPU."""
    g = _gen(seed, 6)
    out = {}
    for name, shape, kind, sc in synth_sd.sd_specs():
        t = _randn(g, *shape)
        out[name] = (sc * (1.0 + 0.1 * t) if kind == "c" else 1.0 + sc * t if kind == "g" else
                     4.0 * torch.exp(sc * t) if kind == "u" else sc * t)
    for name in out:
        if name.endswith("embedding_sum"):
            out[name] = out[name] * out[name.replace("embedding_sum", "cluster_usage")][:, None]
    return out


def _sd_frames(c):
    return c["n"] if c["kind"] == "decode" else c["chunk"] * c["chunks"]


def _sd_codes(c, seed):
    return torch.randint(0, 2048, (_sd_frames(c), 16), generator=_gen(seed, 7), device=DEV, dtype=torch.int32).cpu().numpy()


# ---- prepare and run -----------------------------------------------------------------------------


def prepare(case, seed):
    c = case
    k = c["kind"]
    if k in ("decode", "stream"):
        dec = hip.SpeechDecoder.from_tensors({n: t.cpu().numpy() for n, t in _sd_tensors(seed).items()})
        return _Owner(kind=k, case=c, codes=_sd_codes(c, seed), dec=dec,
                      stream=hip.SpeechDecoderStream(dec) if k == "stream" else None)
    if k == "prefill":
        x = _embeds(c["model"], seed, c["S"] + 1).cpu().numpy()
        return _Owner(kind=k, t=_talker(c["model"], "bf16", seed, _kv_cap(c["S"] + 512)), x=x[:-1],
                      after=x[-1] if c["then"] else None)
    if k == "batch":
        lens = _lens(c)
        t = _talker(c["model"], c["prec"], seed, _kv_cap(max(lens) + 1))
        b = hip.TalkerBatch(t, c["B"])
        at, pool = _starts(c, lens)
        kk, vv = (_bits(x) for x in _cache(c["model"], seed, pool))
        row, slot = kk.shape[2] * 2, kk.nbytes
        for i, n in enumerate(lens):   # slot i's rows are the pool's rows from at[i]: the entry adds i slots to the address
            p, q = (ctypes.c_void_p(a.ctypes.data + at[i] * row - i * slot) for a in (kk, vv))
            hip.check(hip.lib().qwen_hip_talker_batch_upload_slot(b.h, i, p, q, pool, n), "upload_slot")
        return _Owner(kind=k, t=t, b=b, pos=np.array(lens, np.int32), x=_embeds(c["model"], seed, c["B"]).cpu().numpy())
    t = _talker(c["model"], c["prec"], seed, _kv_cap(c["L"] + c.get("n", 1)))
    kk, vv = (_bits(x) for x in _cache(c["model"], seed, c["L"]))
    t.upload_kv(kk, vv, c["L"])
    if k == "step":
        return _Owner(kind=k, t=t, pos=c["L"], x=_embeds(c["model"], seed, 1)[0].cpu().numpy())
    tens = _cp_tensors(c["model"], seed)
    return _Owner(kind=k, t=t, cp=hip.cp_from_tensors(tens, synth.SHAPES[c["model"]]), n=c["n"], pos=c["L"],
                  head=tens["talker.codec_head.weight"], emb=tens["talker.model.codec_embedding.weight"],
                  inputs=_frame_inputs(c, seed))


class _Owner(dict):
    """A case's state; what it holds on the device goes with it."""

    def __del__(self):
        for k in ("stream", "b", "cp", "dec", "t"):
            if self.get(k) is not None:
                self[k].free()


def run(state):
    s = state
    k = s["kind"]
    if k == "prefill":
        last = s["t"].prefill(s["x"])
        return {"last": last} if s["after"] is None else {"last": last, "hidden": s["t"].step(s["after"], len(s["x"]))}
    if k == "step":
        return s["t"].step(s["x"], s["pos"])
    if k == "batch":
        return s["b"].step(s["x"], s["pos"])
    if k == "frames":
        pad, hidden, prev, lcg = s["inputs"]
        codes, _, hid, after = hip.generate(s["t"], s["cp"], s["head"], s["emb"], pad, hidden, s["pos"], FRAME0, s["n"],
                                            prev=prev, seed=lcg, **SAMPLING)
        return {"codes": codes, "hidden": hid, "lcg": after}
    if k == "decode":
        return s["dec"].decode(s["codes"])
    s["stream"].reset()
    n = s["case"]["chunk"]
    return [s["stream"].decode(s["codes"][i * n:(i + 1) * n]) for i in range(s["case"]["chunks"])]


# ---- the work of one pass --------------------------------------------------------------------------

WEIGHT_BYTES = {"bf16": 2.0, "int8": 1.0, "q4": 18.0 / 32.0}


def _params(model, cp=False):
    H, F, nh, nkv, nl = _dims(model, cp)
    return nl * (H * (nh + 2 * nkv) * 128 + H * nh * 128 + 3 * H * F)


def work(case):
    c = case
    k = c["kind"]
    if k in ("decode", "stream"):
        macs = weights = 0
        rows = 1                       # output rows per frame
        for name, shape, kind, _ in synth_sd.sd_specs():
            if kind != "w":
                continue
            n = math.prod(shape)
            weights += n
            if name.startswith("decoder.upsample."):
                rows = 2 ** (int(name.split(".")[2]) + 1)
            elif name.startswith("decoder.decoder."):
                rows = 4 * math.prod(synth_sd.UP_RATES[:min(4, int(name.split(".")[2]))])
            # a transposed conv's kernel column meets each input row once
            up = name.endswith(".1.conv.weight") or name.endswith(".0.conv.weight") and "upsample" in name
            macs += n * (rows // (2 if "upsample" in name else synth_sd.UP_RATES[int(name.split(".")[2]) - 1]) if up else rows)
        f = _sd_frames(c)
        return {"bytes": 4.0 * weights + f * (16 * 1025 + 1920 * 4), "flops": 2.0 * macs * f}
    H, _, nh, nkv, nl = _dims(c["model"])
    P = _params(c["model"])
    if k == "prefill":
        S = c["S"]
        if c["then"]:
            nxt = work({"kind": "step", "model": c["model"], "prec": "bf16", "L": S})
            one = work({**c, "then": 0})
            return {m: one[m] + nxt[m] for m in one}
        return {"bytes": 2.0 * P + 4.0 * S * H + 2.0 * 2 * nl * S * nkv * 128,
                "flops": 2.0 * P * S + nl * 4.0 * nh * 128 * S * (S + 1) / 2}
    kv = lambda L: 2.0 * 2 * nl * L * nkv * 128        # noqa: E731
    at = lambda L: nl * 4.0 * nh * 128 * (L + 1)       # noqa: E731
    w = P * WEIGHT_BYTES[c["prec"]]
    if k == "step":
        return {"bytes": w + kv(c["L"] + 1) + 8.0 * H, "flops": 2.0 * P + at(c["L"])}
    if k == "batch":
        ls = _lens(c)
        return {"bytes": w + sum(kv(n + 1) for n in ls) + 8.0 * H * c["B"], "flops": 2.0 * P * c["B"] + sum(at(n) for n in ls)}
    s = synth.SHAPES[c["model"]]
    heads = 2.0 * (s.codec_vocab * H + 15 * s.codebook * s.cp_hidden)
    pc = _params(c["model"], cp=True)
    return {"bytes": c["n"] * (w + 2.0 * pc + heads + kv(c["L"] + 1)),
            "flops": c["n"] * (2.0 * P + at(c["L"]) + 16 * 2.0 * pc + heads)}


def tolerance(case):
    """About four times what the path is off the 64-bit result: 5e-6 for a prefill, whose sums
    are f32 throughout, and 9e-6 for the audio.  A decode step's new cache rows are cut to bf16
    on the way, so that now and then an f32 rounding moves an element by a whole bf16 unit:
    3e-4 seen where a cache is long enough to average it, 1e-3 where it holds a few rows."""
    k = case["kind"]
    if k == "prefill" and not case["then"]:
        return {"rel": 2e-5, "max": 4e-4}
    if k in ("decode", "stream"):
        return {"rel": 4e-5, "max": 1e-3}
    shortest = case["S"] if k == "prefill" else case["lo"] if k == "batch" else case["L"]
    return {"rel": 4e-3 if shortest < 64 else 1.2e-3, "max": 4e-2, "differ": 0.0}


# ---- the same in 64 bits -----------------------------------------------------------------------------


def _rms(x, g, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * g.double()


def _rope64(x, pos):
    """x [n][heads][128] rotated at its rows' positions (split halves)."""
    c, s = (torch.from_numpy(t).to(DEV).double()[pos][:, None, :] for t in _ROPE)
    a, b = x[..., :64], x[..., 64:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _cut(x):
    """The cache's bf16: a float's upper half."""
    return (x.float().view(torch.int32) & -65536).view(torch.float32).double()


def _layer64(d, prec, x, pos, dims, attend):
    """One layer over the rows x [n][H]; attend(q, k, v) -> [n][nh * 128] from the normed and
    rotated q and k and the projected v."""
    H, F, nh, nkv, _ = dims
    n = x.shape[0]
    xn = _rms(x, d["input_norm"])
    q, k, v = (xn @ _dequantize(d[m], prec).T for m in ("q", "k", "v"))
    q = _rope64(_rms(q.view(n, nh, 128), d["q_norm"]), pos)
    k = _rope64(_rms(k.view(n, nkv, 128), d["k_norm"]), pos)
    x = x + attend(q, k, v.view(n, nkv, 128)).reshape(n, nh * 128) @ _dequantize(d["o"], prec).T
    gu = _rms(x, d["post_attn_norm"]) @ _dequantize(d["gate_up"], prec).T
    g, u = gu[:, 0::2], gu[:, 1::2]
    return x + (g / (1 + torch.exp(-g)) * u) @ _dequantize(d["down"], prec).T


def _over_cache(cache, nh):
    """One row's attention over cache = [K, V], [L][nkv][128] each, to which its own rows are added."""
    def attend(q, k, v):
        cache[0], cache[1] = torch.cat((cache[0], _cut(k))), torch.cat((cache[1], _cut(v)))
        kk, vv = (t.repeat_interleave(nh // t.shape[1], 1).transpose(0, 1).contiguous() for t in cache)
        p = torch.softmax(torch.matmul(kk, q[0][:, :, None])[..., 0] / math.sqrt(128), 1)
        return torch.matmul(p[:, None], vv)[None, :, 0]
    return attend


def _talker_step64(layers, fn, prec, dims, caches, x, pos):
    """x [H] at position pos over the layers' caches [K, V]; returns the normed hidden."""
    x = x[None]
    p = torch.tensor([pos], device=DEV)
    for d, cache in zip(layers, caches):
        x = _layer64(d, prec, x, p, dims, _over_cache(cache, dims[2]))
    return _rms(x, fn)[0]


def _rows(kv, l, a, n):
    """Layer l's cache rows [a, a + n) as [K, V]."""
    return [t[l, a:a + n].double().view(n, -1, 128) for t in kv]


def _prefill64(case, seed):
    c = case
    layers, fn = _layers(c["model"], "bf16", seed)
    dims = _dims(c["model"])
    e = _embeds(c["model"], seed, c["S"] + 1).double()
    x, caches = e[:-1], []
    pos = torch.arange(c["S"], device=DEV)
    mask = torch.full((c["S"], c["S"]), -math.inf, device=DEV, dtype=torch.float64).triu(1)

    def attend(q, k, v):
        caches.append([_cut(k), _cut(v)])
        r = q.shape[1] // k.shape[1]
        k, v = (t.transpose(0, 1).repeat_interleave(r, 0).contiguous() for t in (k, v))
        s = torch.matmul(q.transpose(0, 1).contiguous(), k.transpose(1, 2).contiguous()) / math.sqrt(128) + mask
        return torch.matmul(torch.softmax(s, 2), v).transpose(0, 1)
    for d in layers:
        x = _layer64(d, "bf16", x, pos, dims, attend)
    last = {"last": x[-1].cpu().numpy()}
    if not c["then"]:
        return last
    return {**last, "hidden": _talker_step64(layers, fn, "bf16", dims, caches, e[-1], c["S"]).cpu().numpy()}


def _sample64(logits, frame, prev, lcg):
    """The codec-head rule and the engine's sampler (repetition penalty, temperature, top-k, LCG draw)."""
    lg = logits.clamp(-100, 100)
    lg[2048:2150] = -1e30
    lg[2151:] = -1e30
    if frame < 2:
        lg[2150] = -1e30
    for t in prev:
        lg[t] = lg[t] / SAMPLING["rep"] if lg[t] > 0 else lg[t] * SAMPLING["rep"]
    p = torch.softmax(lg / SAMPLING["temp"], 0)
    p = torch.where(p < p.topk(SAMPLING["top_k"]).values[-1], torch.zeros_like(p), p)
    lcg = (lcg * 1103515245 + 12345) & 0xFFFFFFFF
    r = ((lcg >> 16) & 0x7FFF) / 32768.0
    hit = torch.nonzero(torch.cumsum(p / p.sum(), 0) > r)
    return (int(hit[0]) if len(hit) else lg.numel() - 1), lcg


def _frames64(case, seed):
    c = case
    m = c["model"]
    dims, cdims = _dims(m), _dims(m, cp=True)
    layers, fn = _layers(m, c["prec"], seed)
    kv = _cache(m, seed, c["L"])
    caches = [_rows(kv, l, 0, c["L"]) for l in range(dims[4])]
    bf = lambda a: torch.from_numpy(a.view(np.int16).copy()).to(DEV).view(torch.bfloat16)   # noqa: E731
    t = {n: bf(a) for n, a in _cp_tensors(m, seed).items()}
    P = "talker.code_predictor."
    cls = []
    for l in range(cdims[4]):
        q = f"{P}model.layers.{l}."
        gu = torch.stack((t[q + "mlp.gate_proj.weight"], t[q + "mlp.up_proj.weight"]), 1).flatten(0, 1)
        cls.append({"q": (t[q + "self_attn.q_proj.weight"], None), "k": (t[q + "self_attn.k_proj.weight"], None),
                    "v": (t[q + "self_attn.v_proj.weight"], None), "o": (t[q + "self_attn.o_proj.weight"], None),
                    "gate_up": (gu, None), "down": (t[q + "mlp.down_proj.weight"], None),
                    "input_norm": t[q + "input_layernorm.weight"], "post_attn_norm": t[q + "post_attention_layernorm.weight"],
                    "q_norm": t[q + "self_attn.q_norm.weight"], "k_norm": t[q + "self_attn.k_norm.weight"]})
    emb, head = t["talker.model.codec_embedding.weight"].double(), t["talker.codec_head.weight"].double()
    cemb = [t[f"{P}model.codec_embedding.{g}.weight"].double() for g in range(15)]
    lm = [t[f"{P}lm_head.{g}.weight"].double() for g in range(15)]
    mtp = t.get(P + "small_to_mtp_projection.weight")
    into = (lambda x: x) if mtp is None else (lambda x: mtp.double() @ x + t[P + "small_to_mtp_projection.bias"].double())
    pad, hidden, prev, lcg = _frame_inputs(c, seed)
    pad, h = torch.from_numpy(pad).to(DEV).double(), torch.from_numpy(hidden).to(DEV).double()
    prev, codes = list(prev), []
    for f in range(c["n"]):
        c0, lcg = _sample64(head @ h, FRAME0 + f, prev, lcg)
        if c0 == 2150:
            break
        prev.append(c0)
        row = [c0]
        cc = [[torch.zeros(0, cdims[3], 128, device=DEV, dtype=torch.float64)] * 2 for _ in cls]
        x = into(h)
        for p in range(16):
            if p == 1:
                x = into(emb[c0])
            y = _talker_step64(cls, t[P + "model.norm.weight"], "bf16", cdims, cc, x, p)
            if p:
                row.append(int(torch.argmax(lm[p - 1] @ y)))
                x = into(cemb[p - 1][row[-1]])
        codes.append(row)
        e = emb[c0] + sum(cemb[g][row[g + 1]] for g in range(15)) + pad
        h = _talker_step64(layers, fn, c["prec"], dims, caches, e, c["L"] + f)
    return {"codes": np.array(codes, np.int32).reshape(-1, 16), "hidden": h.cpu().numpy(), "lcg": lcg}


def _sd64(codes, t):
    """The speech decoder, time-major [T][C]."""
    w = lambda n: t[n].double()                        # noqa: E731
    D = "decoder."
    codes = torch.from_numpy(codes).to(DEV).long()

    def conv(x, p, dil=1):
        W = w(p + ".weight")
        k = W.shape[2]
        xp = torch.cat((torch.zeros((k - 1) * dil, x.shape[1], device=DEV, dtype=torch.float64), x))
        return sum(xp[j * dil:j * dil + x.shape[0]] @ W[:, :, j].T for j in range(k)) + w(p + ".bias")

    def conv_up(x, p, r):
        W = w(p + ".weight")
        y = torch.zeros(x.shape[0] + 1, r, W.shape[1], device=DEV, dtype=torch.float64)
        for j in range(W.shape[2]):
            y[j // r:j // r + x.shape[0], j % r] += x @ W[:, :, j]
        return y[:-1].reshape(-1, W.shape[1]) + w(p + ".bias")

    def snake(x, p):
        return x + torch.exp(-w(p + "beta")) * torch.sin(torch.exp(w(p + "alpha")) * x) ** 2
    q = D + "quantizer.rvq_"
    book = lambda p: w(p + ".embedding_sum") / w(p + ".cluster_usage").clamp(min=1e-5)[:, None]      # noqa: E731
    a = book(q + "first.vq.layers.0._codebook")[codes[:, 0]] @ w(q + "first.output_proj.weight").view(512, 256).T
    b = sum(book(f"{q}rest.vq.layers.{i}._codebook")[codes[:, i + 1]] for i in range(15))
    h = conv(a + b @ w(q + "rest.output_proj.weight").view(512, 256).T, D + "pre_conv.conv")
    P = D + "pre_transformer"
    h = h @ w(P + ".input_proj.weight").T + w(P + ".input_proj.bias")
    n = h.shape[0]
    ang = torch.arange(n, device=DEV, dtype=torch.float64)[:, None] / 10000.0 ** (torch.arange(32, device=DEV, dtype=torch.float64) / 32)
    cs, sn = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    rot = lambda x: torch.cat((x[..., :32] * cs - x[..., 32:] * sn, x[..., 32:] * cs + x[..., :32] * sn), -1)   # noqa: E731
    i = torch.arange(n, device=DEV)
    off = (i[None] > i[:, None]) | (i[None] <= i[:, None] - 72)
    for l in range(8):
        p = f"{P}.layers.{l}."
        xn = _rms(h, t[p + "input_layernorm.weight"], 1e-5)
        Q, K, V = ((xn @ w(p + f"self_attn.{m}_proj.weight").T).view(n, 16, 64) for m in "qkv")
        s = torch.matmul(rot(Q).transpose(0, 1).contiguous(), rot(K).permute(1, 2, 0).contiguous()) / 8.0
        s = torch.softmax(s.masked_fill(off, -math.inf), 2)
        o = torch.matmul(s, V.transpose(0, 1).contiguous()).transpose(0, 1).reshape(n, 1024)
        h = h + o @ w(p + "self_attn.o_proj.weight").T * w(p + "self_attn_layer_scale.scale")
        xn = _rms(h, t[p + "post_attention_layernorm.weight"], 1e-5)
        g, u = (xn @ w(p + f"mlp.{m}_proj.weight").T for m in ("gate", "up"))
        h = h + (g / (1 + torch.exp(-g)) * u) @ w(p + "mlp.down_proj.weight").T * w(p + "mlp_layer_scale.scale")
    x = _rms(h, t[P + ".norm.weight"], 1e-5) @ w(P + ".output_proj.weight").T + w(P + ".output_proj.bias")
    for b in range(2):
        p = f"{D}upsample.{b}."
        x = conv_up(x, p + "0.conv", 2)
        W = w(p + "1.dwconv.conv.weight")[:, 0]
        xp = torch.cat((torch.zeros(6, 1024, device=DEV, dtype=torch.float64), x))
        d = sum(xp[j:j + x.shape[0]] * W[:, j] for j in range(7)) + w(p + "1.dwconv.conv.bias")
        d = torch.nn.functional.layer_norm(d, (1024,), w(p + "1.norm.weight"), w(p + "1.norm.bias"), 1e-5)
        d = torch.nn.functional.gelu(d @ w(p + "1.pwconv1.weight").T + w(p + "1.pwconv1.bias"))
        x = x + (d @ w(p + "1.pwconv2.weight").T + w(p + "1.pwconv2.bias")) * w(p + "1.gamma")
    x = conv(x, D + "decoder.0.conv")
    for b in range(4):
        p = f"{D}decoder.{b + 1}.block."
        x = conv_up(snake(x, p + "0."), p + "1.conv", synth_sd.UP_RATES[b])
        for r in range(3):
            y = conv(snake(x, f"{p}{r + 2}.act1."), f"{p}{r + 2}.conv1.conv", synth_sd.DILATIONS[r])
            x = x + conv(snake(y, f"{p}{r + 2}.act2."), f"{p}{r + 2}.conv2.conv")
    return conv(snake(x, D + "decoder.5."), D + "decoder.6.conv")[:, 0].clamp(-1, 1).cpu().numpy()


def exact(case, seed):
    c = case
    k = c["kind"]
    if k == "prefill":
        return _prefill64(c, seed)
    if k in ("decode", "stream"):
        y = _sd64(_sd_codes(c, seed), _sd_tensors(seed))
        return y if k == "decode" else np.split(y, c["chunks"])
    if k == "frames":
        return _frames64(c, seed)
    layers, fn = _layers(c["model"], c["prec"], seed)
    dims = _dims(c["model"])
    if k == "step":
        kv = _cache(c["model"], seed, c["L"])
        caches = [_rows(kv, l, 0, c["L"]) for l in range(dims[4])]
        x = _embeds(c["model"], seed, 1)[0].double()
        return _talker_step64(layers, fn, c["prec"], dims, caches, x, c["L"]).cpu().numpy()
    lens = _lens(c)
    at, pool = _starts(c, lens)
    kv = _cache(c["model"], seed, pool)
    x = _embeds(c["model"], seed, c["B"]).double()
    pos = torch.tensor(lens, device=DEV)
    for l, d in enumerate(layers):
        def attend(q, k, v, l=l):
            return torch.cat([_over_cache(_rows(kv, l, at[i], lens[i]), dims[2])(q[i:i + 1], k[i:i + 1], v[i:i + 1])
                              for i in range(len(lens))])
        x = _layer64(d, c["prec"], x, pos, dims, attend)
    return _rms(x, fn).cpu().numpy()
