"""GPU parity of the batched (B-stream, ragged) step and its MFMA projection.

Oracle: the C restatement (oracle/), one independent decode per stream on that
stream's own KV cache, over the reference-loaded weights (oracle_talker).  The
reference's batched step computes exactly these per-stream single steps
(qwen_tts_talker.c:1192-1270: per-sequence norm/RoPE/KV/attention, weights shared), so
each stream is held to the north-star tolerance (max-abs 2e-2, rel-L2 1e-3 of the
hidden state) and its KV rows to the single-step KV checks.
"""
import ctypes as C

import numpy as np
import pytest

from conftest import model_dir, need_ref, rel_l2

pytestmark = pytest.mark.gpu

from qwen3_tts_amd import hip, synth  # noqa: E402


def _matmat(q, s, X):
    rows, cols = q.shape
    B = X.shape[1]
    Y = np.empty((rows, B), np.float32)
    Xc = np.ascontiguousarray(X, np.float32)
    hip.check(hip.lib().qwen_hip_op_matmat_int8(Y.ctypes.data, q.ctypes.data, s.ctypes.data, Xc.ctypes.data,
                                               rows, cols, B), "matmat_int8")
    return Y


@pytest.mark.parametrize("rows,cols,B", [(16, 64, 1), (64, 2048, 32), (4096, 1024, 16), (2048, 6144, 32),
                                         (257, 320, 5), (100, 2048, 33), (48, 8192, 64), (12288, 2048, 8)])
def test_op_matmat_int8(oracle, rows, cols, B):
    """Y = (W*scale) @ X against the f64 product of the dequantised weights: the exact
    int8-piece contraction leaves only the activation split (|e| <= max|x| 2^-20) and
    the final roundings."""
    print(f"[case] matmat int8 {rows}x{cols} B={B}", flush=True)
    rng = np.random.default_rng(rows + cols + B)
    w = synth.f32_to_bf16_rne((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    q, s = oracle.quantize_int8(w)
    X = rng.standard_normal((cols, B)).astype(np.float32)
    X[:, 0] *= 1e-3                                     # streams of very different magnitude
    if B > 2:
        X[:, 2] = 0.0                                   # an all-zero stream
    Y = _matmat(q, s, X)
    Wf = q.astype(np.float64) * s.astype(np.float64)[:, None]
    Y64 = Wf @ X.astype(np.float64)
    for j in range(B):
        den = np.abs(Y64[:, j]).max()
        if den == 0:
            assert np.all(Y[:, j] == 0)
            continue
        err = np.abs(Y[:, j] - Y64[:, j]).max() / den
        assert err < 1e-5, (j, err)


def test_op_matmat_int8_exact_inputs(oracle):
    """Activations that the three int8 planes hold exactly (multiples of 2^-14 of a
    power-of-two scale): the product is the exact dot product rounded once, so it
    equals the f64 result rounded to f32 (times the row scale)."""
    rows, cols, B = 64, 2048, 16
    rng = np.random.default_rng(4)
    q = rng.integers(-127, 128, (rows, cols)).astype(np.int8)
    s = np.ones(rows, np.float32)
    X = (rng.integers(-(1 << 20), 1 << 20, (cols, B)) * 2.0 ** -14).astype(np.float32)   # |x| < 64
    Y = _matmat(q, s, X)
    exact = q.astype(np.float64) @ X.astype(np.float64)
    assert np.array_equal(Y, exact.astype(np.float32))


def test_op_matmat_int8_tiny_negative_activations(oracle):
    """Activations just below zero next to O(1) ones (SwiGLU outputs of very negative
    gates): y = x/s in (-2^-25, 0) makes y - floor(y) round up to 1.0 in f32, which once
    turned piece plane 2 into 128 (an int8 -128, an error of 2s on that element).  Every
    stream, and each of the four tall-tile / split-K plans (K = 1024, 2048, 3072, 6144),
    against the f64 product."""
    rng = np.random.default_rng(0x71C)
    for rows, cols, B in [(64, 1024, 32), (256, 2048, 32), (128, 3072, 16), (2048, 6144, 32)]:
        print(f"[case] matmat int8 tiny negatives {rows}x{cols} B={B}", flush=True)
        w = synth.f32_to_bf16_rne((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
        q, s = oracle.quantize_int8(w)
        X = rng.standard_normal((cols, B)).astype(np.float32)
        tiny = rng.random((cols, B)) < 0.25
        X[tiny] = -(rng.random(int(tiny.sum())) * 1e-9 + 1e-12).astype(np.float32)
        Y = _matmat(q, s, X)
        Y64 = (q.astype(np.float64) * s.astype(np.float64)[:, None]) @ X.astype(np.float64)
        for j in range(B):
            err = np.abs(Y[:, j] - Y64[:, j]).max() / np.abs(Y64[:, j]).max()
            assert err < 1e-5, (rows, cols, j, err)


def test_op_matmat_matches_matvec_per_column(oracle):
    """Each column of the batched product is the single-stream matvec of that column
    (qwen_tts_kernels.h:117-122: 'with B==1 it equals matvec'), to the f32 rounding of
    the matvec's own 3072-term accumulation."""
    rows, cols, B = 1024, 3072, 6
    rng = np.random.default_rng(9)
    w = synth.f32_to_bf16_rne((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    q, s = oracle.quantize_int8(w)
    X = rng.standard_normal((cols, B)).astype(np.float32)
    Y = _matmat(q, s, X)
    for j in range(B):
        y = np.empty(rows, np.float32)
        xj = np.ascontiguousarray(X[:, j])
        hip.check(hip.lib().qwen_hip_op_matvec_int8(y.ctypes.data, q.ctypes.data, s.ctypes.data,
                                                   xj.ctypes.data, rows, cols), "mv")
        assert rel_l2(Y[:, j], y) < 5e-6


def _matmat_q4(blocks, rows, cols, X):
    B = X.shape[1]
    Y = np.empty((rows, B), np.float32)
    Xc = np.ascontiguousarray(X, np.float32)
    hip.check(hip.lib().qwen_hip_op_matmat_q4_0(Y.ctypes.data, blocks.ctypes.data, Xc.ctypes.data, rows, cols, B),
              "matmat_q4_0")
    return Y


@pytest.mark.parametrize("rows,cols,B", [(16, 64, 1), (64, 2048, 32), (4096, 1024, 16), (2048, 6144, 32),
                                         (257, 320, 5), (100, 2048, 33), (48, 8192, 64), (12288, 2048, 8)])
def test_op_matmat_q4_0(oracle, rows, cols, B):
    """Y = dequant(W_q4) @ X (weights read once for all B columns) against the f64 product
    of the dequantised weights (oracle dequant_q4_0, k.c:2810-2819): each block's dot
    product is an exact integer sum rounded once, so only f32 roundings remain."""
    print(f"[case] matmat q4_0 {rows}x{cols} B={B}", flush=True)
    rng = np.random.default_rng(rows * 7 + cols + B)
    w = synth.f32_to_bf16_rne((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    blocks = oracle.quantize_q4_0(w)
    X = rng.standard_normal((cols, B)).astype(np.float32)
    X[:, 0] *= 1e-3
    if B > 2:
        X[:, 2] = 0.0
    Y = _matmat_q4(blocks, rows, cols, X)
    Wf = oracle.dequant_q4_0(blocks, rows, cols).astype(np.float64)
    Y64 = Wf @ X.astype(np.float64)
    for j in range(B):
        den = np.abs(Y64[:, j]).max()
        if den == 0:
            assert np.all(Y[:, j] == 0)
            continue
        err = np.abs(Y[:, j] - Y64[:, j]).max() / den
        assert err < 1e-5, (j, err)


def test_op_matmat_q4_0_exact_inputs(oracle):
    """Power-of-two block scales (the second block of each row scaled by zero) and
    activations that the int8 planes hold exactly: every block's integer dot product, its
    conversion and its scaling are exact, so Y equals the f64 product."""
    rows, cols, B = 32, 64, 16
    rng = np.random.default_rng(5)
    nib = rng.integers(0, 16, (rows, cols))
    blocks = np.zeros((rows, cols // 32, 18), np.uint8)
    for r in range(rows):
        for j in range(cols // 32):
            e = int(rng.integers(-6, 3))
            h = np.float16(2.0 ** e) if j == 0 else np.float16(0.0)
            blocks[r, j, :2] = np.frombuffer(h.tobytes(), np.uint8)
            q = nib[r, 32 * j:32 * j + 32]
            blocks[r, j, 2:] = (q[0::2] | (q[1::2] << 4)).astype(np.uint8)
    X = (rng.integers(-(1 << 14), 1 << 14, (cols, B)) * 2.0 ** -10).astype(np.float32)
    Y = _matmat_q4(blocks, rows, cols, X)
    Wf = oracle.dequant_q4_0(blocks.reshape(-1), rows, cols).astype(np.float64)
    assert np.array_equal(Y, (Wf @ X.astype(np.float64)).astype(np.float32))


# ------------------------------------------------------------------ batched Talker step

def _ref(name, prec):
    from oracle.oracle import RefModel
    d, shape, _ = model_dir(name)
    return RefModel(d, shape, prec=prec, threads=8), shape


def _streams(ref, prec_code, B, kv_max):
    from oracle.oracle import oracle_talker
    return [oracle_talker(ref, prec_code, kv_max) for _ in range(B)]


@need_ref
@pytest.mark.parametrize("prec,B", [("int8", 5), ("int8", 32), ("bf16", 3), ("bf16", 32), ("int4", 2), ("int4", 17), ("int4", 32)])
def test_batch_step_ragged_vs_oracle(oracle, prec, B):
    """B streams prefilled to different lengths (upload_slot), then stepped together,
    each at its own position; every stream against its own oracle decode."""
    print(f"[case] batch step {prec} B={B}", flush=True)
    ref, shape = _ref("mini", prec)
    pc = hip.PREC[prec]
    kv_max = 96
    layers = hip.layers_from_ref(ref, pc)
    cos, sin = ref.rope()
    g = hip.Talker(shape, layers, ref.final_norm(), cos, sin, pc, kv_max)
    bt = hip.TalkerBatch(g, B)
    streams = _streams(ref, pc, B, kv_max)
    emb = ref.codec_emb()
    rng = np.random.default_rng(100 + B)
    pre = [int(rng.integers(0, 40)) for _ in range(B)]
    pre[0] = 0
    H, L, kvd = shape.hidden, shape.layers, shape.kv_dim
    kvk = np.zeros((B, L, kv_max, kvd), np.uint16)
    kvv = np.zeros_like(kvk)
    for b in range(B):
        t, keep = streams[b]
        for p in range(pre[b]):
            oracle.talker_step(t, synth.bf16_to_f32(emb[int(rng.integers(0, 2048))]), p)
        kvk[b], kvv[b] = keep["kv_k"], keep["kv_v"]
    for b in range(B):
        bt.upload_slot(b, kvk, kvv, pre[b])
        if pre[b]:
            k2, v2 = bt.download_slot(b, pre[b])
            assert np.array_equal(k2[:, :pre[b]], kvk[b][:, :pre[b]]) and np.array_equal(v2[:, :pre[b]], kvv[b][:, :pre[b]])
    pos = np.array(pre, np.int32)
    worst = 0.0
    for it in range(6):
        E = np.stack([synth.bf16_to_f32(emb[int(rng.integers(0, 2048))]) for _ in range(B)])
        got = bt.step(E, pos)
        for b in range(B):
            want, _ = oracle.talker_step(streams[b][0], E[b], int(pos[b]))
            assert np.abs(got[b] - want).max() <= 2e-2, (it, b)
            err = rel_l2(got[b], want)
            assert err <= 1e-3, (it, b, err)
            worst = max(worst, err)
        pos += 1
    # KV rows written by the batched step: truncated bf16 of the stream's own k/v
    for b in range(B):
        n = int(pos[b])
        kg, vg = bt.download_slot(b, n)
        kr, vr = streams[b][1]["kv_k"], streams[b][1]["kv_v"]
        for a_, b_ in [(kg, kr), (vg, vr)]:
            fa, fb = synth.bf16_to_f32(a_[:, :n]), synth.bf16_to_f32(b_[:, :n])
            num = np.linalg.norm((fa - fb).astype(np.float64), axis=-1)
            den = np.linalg.norm(fb.astype(np.float64), axis=-1)
            assert (num <= 1e-2 * den + 1e-6).all(), float((num / np.maximum(den, 1e-30)).max())
    print(f"[result] batch {prec} B={B}: worst hidden rel-L2 {worst:.2e}")
    bt.free()
    g.free()


@pytest.mark.parametrize("prec", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("name,B", [("tiny", 1), ("tiny", 31), ("mini", 5), ("mini", 16), ("mini", 49), ("mini17", 17),
                                    ("mini17", 64)])
def test_batch_row_tiles_vs_oracle(oracle, name, B, prec):
    """Projections of B rows: whole and partial tiles of 16, K from a slice per wave up to 24,
    every weight tile width.  Each stream is at one of three positions with that position's cache;
    the bars are the ragged test's."""
    from oracle.oracle import talker_from_tensors
    print(f"[case] batch {prec} {name} B={B}", flush=True)
    _, shape, t = model_dir(name)
    cos, sin = synth.rope_tables(shape.head_dim, shape.rope_theta, 64)
    g = hip.Talker(shape, hip.layers_from_tensors(t, shape), synth.bf16_to_f32(t["talker.model.norm.weight"]), cos, sin,
                   hip.BF16, 64, quantize_to=-1 if prec == "bf16" else hip.PREC[prec])
    ot, keep = talker_from_tensors(oracle, t, shape, prec, 64, cos, sin)
    rng = np.random.default_rng(B)
    at = [0, 3, 21]
    for p in range(at[-1]):
        oracle.talker_step(ot, rng.normal(0, 0.5, shape.hidden).astype(np.float32), p)
    kvk, kvv = keep["kv_k"].copy(), keep["kv_v"].copy()
    bt = hip.TalkerBatch(g, B)
    pos = np.array([at[b % 3] for b in range(B)], np.int32)
    ks, vs = np.stack([kvk] * B), np.stack([kvv] * B)
    for b in range(B):
        bt.upload_slot(b, ks, vs, int(pos[b]))
    E = rng.normal(0, 0.5, (B, shape.hidden)).astype(np.float32)
    got = bt.step(E, pos)
    for b in range(B):
        keep["kv_k"][:], keep["kv_v"][:] = kvk, kvv
        want, _ = oracle.talker_step(ot, E[b], int(pos[b]))
        assert rel_l2(got[b], want) <= 1e-3 and np.abs(got[b] - want).max() <= 2e-2, (b, rel_l2(got[b], want))
    bt.free()
    g.free()


@pytest.mark.parametrize("prec,pieces", [("bf16", False), ("int8", False), ("int8", True), ("int4", False)])
@pytest.mark.parametrize("name,at", [("mini", (383, 767, 1000)),
                                     ("tiny", (382, 383, 384, 385, 0, 766, 767, 768, 769, 31, 1000, 1150, 1151, 1152, 400, 800, 1))])
def test_batch_long_caches_vs_oracle(oracle, name, at, prec, pieces):
    """Caches around the edges of the 384-key chunks that at most 128 (stream, kv head) pairs are split
    into, so that the last chunk's workgroup merges up to four of them, into planes (three, or
    seventeen rows: two row tiles) or, on the int8 pieces, into f32 rows; two steps, so that the second one's
    chunks hold the first one's keys and the arrival counters are used again."""
    print(f"[case] batch long caches {prec} {name} pieces={pieces}", flush=True)
    from oracle.oracle import talker_from_tensors
    _, shape, t = model_dir(name)
    B, kv_max = len(at), 1200
    cos, sin = synth.rope_tables(shape.head_dim, shape.rope_theta, kv_max)
    g = hip.Talker(shape, hip.layers_from_tensors(t, shape), synth.bf16_to_f32(t["talker.model.norm.weight"]), cos, sin,
                   hip.BF16, kv_max, quantize_to=-1 if prec == "bf16" else hip.PREC[prec])
    ot, keep = talker_from_tensors(oracle, t, shape, prec, kv_max, cos, sin)
    rng = np.random.default_rng(B)
    kv = [synth.f32_to_bf16_rne(rng.standard_normal((B,) + keep["kv_k"].shape, dtype=np.float32)) for _ in range(2)]
    bt = hip.TalkerBatch(g, B)
    if pieces:
        bt.fold_pieces(True)
    for b in range(B):
        bt.upload_slot(b, kv[0], kv[1], at[b])
    pos = np.array(at, np.int32)
    E = rng.normal(0, 0.5, (2, B, shape.hidden)).astype(np.float32)
    got = [bt.step(E[i], pos + i) for i in range(2)]
    for b in range(B):
        keep["kv_k"][:], keep["kv_v"][:] = kv[0][b], kv[1][b]
        for i in range(2):
            want, _ = oracle.talker_step(ot, E[i, b], at[b] + i)
            assert rel_l2(got[i][b], want) <= 1e-3 and np.abs(got[i][b] - want).max() <= 2e-2, (i, b, rel_l2(got[i][b], want))
    bt.free()
    g.free()


@pytest.mark.parametrize("prec", ["bf16", "int8", "int4"])
def test_batch_non_finite_stream_alone(prec):
    """An input with an infinity, a NaN or squares that overflow ends in its own stream's row."""
    print(f"[case] batch non-finite stream {prec}", flush=True)
    _, shape, t = model_dir("tiny")
    cos, sin = synth.rope_tables(shape.head_dim, shape.rope_theta, 64)
    g = hip.Talker(shape, hip.layers_from_tensors(t, shape), synth.bf16_to_f32(t["talker.model.norm.weight"]), cos, sin,
                   hip.BF16, 64, quantize_to=-1 if prec == "bf16" else hip.PREC[prec])
    B, pos = 19, np.zeros(19, np.int32)
    bt = hip.TalkerBatch(g, B)
    E = np.random.default_rng(1).normal(0, 0.5, (B, shape.hidden)).astype(np.float32)
    clean = bt.step(E, pos)
    E[3, 7], E[17, 0] = np.inf, np.nan
    E[11] *= 1e25
    E[12] = np.sign(E[12]) * np.finfo(np.float32).max
    got = bt.step(E, pos)
    rest = np.delete(np.arange(B), [3, 11, 12, 17])
    assert np.array_equal(got[rest], clean[rest]) and np.isnan(got[[3, 17]]).all() and not got[[11, 12]].any()
    bt.free()
    g.free()


@need_ref
def test_batch_of_identical_streams_matches_single_step():
    """B copies of one stream (the reference's batch self-test, cu:657-730 /
    t.c:1301-1402): every row equals the single-state step to the tolerance."""
    ref, shape = _ref("mini", "int8")
    layers = hip.layers_from_ref(ref, hip.INT8)
    cos, sin = ref.rope()
    g = hip.Talker(shape, layers, ref.final_norm(), cos, sin, hip.INT8, 64)
    B = 4
    bt = hip.TalkerBatch(g, B)
    emb = ref.codec_emb()
    for pos in range(8):
        e = synth.bf16_to_f32(emb[pos * 41 + 3])
        single = g.step(e, pos)
        got = bt.step(np.tile(e, (B, 1)), np.full(B, pos, np.int32))
        # rows of the batch are bit-identical to each other; against the single step
        # (VALU f32 sums) they differ by f32 rounding, which can flip a truncated bf16
        # K/V bit (2^-8 relative) and so reach ~1e-4 after 2 layers
        for b in range(B):
            assert np.array_equal(got[b], got[0])
            assert rel_l2(got[b], single) <= 1e-3, (pos, rel_l2(got[b], single))
    bt.free()
    g.free()


@need_ref
@pytest.mark.parametrize("B", [5, 20, 32])
def test_batch_fold_pieces_matches_separate_launch(B):
    """int8: the activation pieces made inside each projection launch (the default) and
    in a launch of their own are the same bytes, so the outputs are the same bit for bit:
    every layer's residual (ungraphed step) and the graphed step's hidden state.  B = 5 and
    20 have padding streams (16 and 32 columns)."""
    print(f"[case] fold pieces B={B}", flush=True)
    ref, shape = _ref("mini", "int8")
    layers = hip.layers_from_ref(ref, hip.INT8)
    cos, sin = ref.rope()
    g = hip.Talker(shape, layers, ref.final_norm(), cos, sin, hip.INT8, 64)
    bt = hip.TalkerBatch(g, B)
    assert bt.fold_pieces(True)
    emb = ref.codec_emb()
    rng = np.random.default_rng(7 + B)
    pos = rng.integers(0, 40, B).astype(np.int32)
    for it in range(3):
        E = np.stack([synth.bf16_to_f32(emb[int(rng.integers(0, 2048))]) for _ in range(B)])
        assert bt.fold_pieces(True)
        r1, h1 = bt.step_layers(E, pos)
        g1 = bt.step(E, pos)
        assert not bt.fold_pieces(False)
        r2, h2 = bt.step_layers(E, pos)     # same position: rewrites the same KV rows
        g2 = bt.step(E, pos)
        assert np.array_equal(r1, r2) and np.array_equal(h1, h2), it
        assert np.array_equal(g1, g2) and np.array_equal(g1, h1), it
        pos += 1
    bt.free()
    g.free()


@pytest.mark.parametrize("B,created", [(5, 2), (48, 2), (49, 1)])
def test_batch_fold_pieces_and_back(B, created):
    """int8: the pieces give the same bytes inside the launches and apart, and a batch comes back to the
    route that it was created with, bit for bit (the bf16 planes up to 48 streams of the 0.6B shape)."""
    print(f"[case] fold pieces and back B={B}", flush=True)
    _, shape, t = model_dir("mini")
    cos, sin = synth.rope_tables(shape.head_dim, shape.rope_theta, 64)
    g = hip.Talker(shape, hip.layers_from_tensors(t, shape), synth.bf16_to_f32(t["talker.model.norm.weight"]), cos, sin,
                   hip.BF16, 64, quantize_to=hip.INT8)
    bt = hip.TalkerBatch(g, B)
    rng = np.random.default_rng(B)
    pos = np.zeros(B, np.int32)
    E = rng.normal(0, 0.5, (B, shape.hidden)).astype(np.float32)
    first = bt.step(E, pos)
    assert bt.fold_pieces(True)
    inside = bt.step(E, pos)
    assert not bt.fold_pieces(False)
    apart = bt.step(E, pos)
    assert bt.fold_pieces(None) == created
    again, (_, layers) = bt.step(E, pos), bt.step_layers(E, pos)
    assert np.array_equal(inside, apart) and np.array_equal(again, first) and np.array_equal(layers, first)
    assert np.array_equal(inside, first) == (created == 1)
    assert max(rel_l2(inside[b], first[b]) for b in range(B)) <= 1e-3
    bt.free()
    g.free()


def test_batch_rejects_bad_arguments():
    shape = synth.SHAPES["tiny"]
    t = synth.generate(shape, 0x5EED0009, 0.0, threads=4, only=lambda n: n.startswith("talker.model."))
    layers = hip.layers_from_tensors(t, shape)
    cos, sin = synth.rope_tables(shape.head_dim, shape.rope_theta, 32)
    g = hip.Talker(shape, layers, synth.bf16_to_f32(t["talker.model.norm.weight"]), cos, sin, hip.BF16, 32,
                   quantize_to=hip.INT8)
    L = hip.lib()
    assert not L.qwen_hip_talker_batch_init(g.h, 0)
    assert not L.qwen_hip_talker_batch_init(g.h, 65)
    assert not L.qwen_hip_talker_batch_init(None, 4)
    bt = hip.TalkerBatch(g, 2)
    E = np.zeros((2, shape.hidden), np.float32)
    with pytest.raises(RuntimeError):
        bt.step(E, np.array([0, 32], np.int32))        # position past kv_max
    bt.free()
    g.free()


@need_ref
@pytest.mark.parametrize("prec", ["bf16", "int8"])
def test_cp_batch_step_vs_oracle(oracle, prec):
    """CP batch twin: B residual streams, one 2-layer pass each at its own position,
    against the oracle's CP pass per stream."""
    from test_gpu_parity import _gpu_cp
    from oracle.oracle import oracle_talker
    ref, shape = _ref("mini", prec)
    pc = hip.PREC[prec]
    cp = _gpu_cp(ref, shape, pc)
    B = 6
    streams = [oracle_talker(ref, pc, 64, cp=True) for _ in range(B)]
    rng = np.random.default_rng(3)
    for p in range(5):
        x = rng.standard_normal((B, shape.cp_hidden)).astype(np.float32)
        got = cp.batch_step(x, np.full(B, p, np.int32))
        for b in range(B):
            want = np.array(x[b], copy=True)
            assert oracle.lib.qo_cp_pass(C.byref(streams[b][0]), want.ctypes.data, p) == 0
            assert rel_l2(got[b], want) <= 1e-3, (p, b, rel_l2(got[b], want))
    cp.free()


@pytest.mark.parametrize("prec", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("name,B", [("tiny", 33), ("mini", 6), ("mini", 17), ("mini", 50)])
def test_cp_batch_tiles_vs_oracle(oracle, name, B, prec):
    """The batched Code Predictor pass over whole and partial row tiles, at ragged positions, up to and
    past the stream counts of the few-rows projections (int8: 48): every stream's residual after each of
    three passes, and at 0, against the oracle's pass on that stream's own cache."""
    from oracle.oracle import talker_from_tensors
    print(f"[case] CP batch {prec} {name} B={B}", flush=True)
    _, shape, t = model_dir(name)
    cp = hip.cp_from_tensors(t, shape, hip.PREC[prec])
    cos, sin = synth.rope_tables(shape.cp_head_dim, shape.rope_theta, 64)
    ot, keep = talker_from_tensors(oracle, t, shape, prec, 64, cos, sin, cp=True)
    cache = [np.zeros((B,) + keep["kv_k"].shape, np.uint16) for _ in range(2)]
    rng = np.random.default_rng(B)
    pos = np.zeros(B, np.int32)
    for it in range(3):
        x = rng.standard_normal((B, shape.cp_hidden)).astype(np.float32)
        got = cp.batch_step(x, pos)
        for b in range(B):
            keep["kv_k"][:], keep["kv_v"][:] = cache[0][b], cache[1][b]
            want = np.array(x[b], copy=True)
            assert oracle.lib.qo_cp_pass(C.byref(ot), want.ctypes.data, int(pos[b])) == 0
            cache[0][b], cache[1][b] = keep["kv_k"], keep["kv_v"]
            assert rel_l2(got[b], want) <= 1e-3, (it, b, rel_l2(got[b], want))
        pos += np.arange(B, dtype=np.int32) % 2         # half of the streams take position 0 again
    cp.free()


@need_ref
def test_cp_prefill2_vs_oracle_and_reference(oracle):
    """Two-position prefill (cp_prefill2, qwen_tts_code_predictor.c:816-902): the
    two-column pass against two sequential oracle passes at positions 0 and 1 (the
    reference's own definition: 'the same math', its matmat only reorders rounding),
    then whole frames with the prefill on against the compiled reference's
    qwen_cp_predict with QWEN_CP_PREFILL2=1 (its mode is probed once per thread, so the
    reference runs in a fresh thread)."""
    import os
    import threading
    from test_gpu_parity import _gpu_cp
    from oracle.oracle import oracle_talker
    print("[case] cp prefill2 int8", flush=True)
    ref, shape = _ref("mini", "int8")
    cp = _gpu_cp(ref, shape, hip.INT8)
    with pytest.raises(RuntimeError):
        cp.prefill2(np.zeros(shape.cp_hidden, np.float32), np.zeros(shape.cp_hidden, np.float32))   # not enabled
    cp.set_prefill2(1)
    rng = np.random.default_rng(21)
    for trial in range(3):
        x0 = rng.standard_normal(shape.cp_hidden).astype(np.float32)
        x1 = rng.standard_normal(shape.cp_hidden).astype(np.float32)
        g0, g1 = cp.prefill2(x0, x1)
        t, _ = oracle_talker(ref, hip.INT8, 64, cp=True)
        w0, w1 = np.array(x0, copy=True), np.array(x1, copy=True)
        assert oracle.lib.qo_cp_pass(C.byref(t), w0.ctypes.data, 0) == 0
        assert oracle.lib.qo_cp_pass(C.byref(t), w1.ctypes.data, 1) == 0
        for g, w in [(g0, w0), (g1, w1)]:
            assert np.abs(g - w).max() <= 2e-2 and rel_l2(g, w) <= 1e-3, (trial, rel_l2(g, w))
    frames = []
    for f in range(4):
        th = rng.standard_normal(shape.hidden).astype(np.float32)
        th /= np.sqrt((th ** 2).mean())
        frames.append((th, int(rng.integers(0, 2048))))
    got = [list(cp.frame(th, c0)) for th, c0 in frames]
    want = []
    old = os.environ.get("QWEN_CP_PREFILL2")
    os.environ["QWEN_CP_PREFILL2"] = "1"
    try:
        th_ = threading.Thread(target=lambda: want.extend(list(ref.cp_predict(th, c0)) for th, c0 in frames))
        th_.start()
        th_.join()
    finally:
        if old is None:
            del os.environ["QWEN_CP_PREFILL2"]
        else:
            os.environ["QWEN_CP_PREFILL2"] = old
    assert len(want) == len(frames)
    assert got == want, (got, want)
    cp.set_prefill2(0)                                  # back to sequential passes
    assert [list(cp.frame(th, c0)) for th, c0 in frames] == [list(ref.cp_predict(th, c0)) for th, c0 in frames]
    cp.free()


@need_ref
def test_cp_prefill2_needs_int8():
    from test_gpu_parity import _gpu_cp
    ref, shape = _ref("mini", "bf16")
    cp = _gpu_cp(ref, shape, hip.BF16)
    with pytest.raises(RuntimeError):
        cp.set_prefill2(1)
    cp.free()
