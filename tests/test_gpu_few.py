"""One projection of a few rows (qt_few.hip: the batched steps of few streams, short prompts)
against float64, with the planes and the sums of squares that it hands on."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

from qwen3_tts_amd import hip, synth  # noqa: E402

EPS = 1e-6
STORE, RESID, SWIGLU = 0, 1, 2


def _weights(oracle, prec, w):
    """(device form, its scales, float64 values) of the bf16 matrix w."""
    if prec == "bf16":
        return w, None, synth.bf16_to_f32(w).astype(np.float64)
    if prec == "int8":
        q, s = oracle.quantize_int8(w)
        return q, s, q.astype(np.float64) * s.astype(np.float64)[:, None]
    b = oracle.quantize_q4_0(w)
    return b, None, oracle.dequant_q4_0(b, *w.shape).reshape(w.shape).astype(np.float64)


def _few(prec, epi, W, scale, X, N, gain, Y=None, next_gain=None):
    S, K = X.shape
    C = N // 2 if epi == SWIGLU else N
    Y = np.zeros((S, N), np.float32) if Y is None else np.array(Y, np.float32, copy=True)
    planes, sums = np.empty((3, S, C), np.float32), np.empty((S, N // 16), np.float32)
    p = lambda a: None if a is None else a.ctypes.data  # noqa: E731
    X, W = np.ascontiguousarray(X, np.float32), np.ascontiguousarray(W)
    hip.check(hip.lib().qwen_hip_op_few_gemm(hip.PREC[prec], epi, p(Y), p(W), p(scale), p(X), S, N, K, p(gain), EPS, p(next_gain),
                                             p(planes), p(sums)), "op_few_gemm")
    return Y, planes, sums


def _two_planes(x):
    """x without what its third plane holds."""
    u = x.view(np.uint32) & np.uint32(0xFFFF0000)
    r = x - u.view(np.float32)
    return u.view(np.float32) + (r.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)


@pytest.mark.parametrize("prec", ["bf16", "int8", "q4_0"])
@pytest.mark.parametrize("S,N,K", [(1, 64, 64), (15, 192, 192), (16, 128, 3072), (17, 2048, 2048), (33, 64, 6144),
                                   (64, 256, 1024), (64, 2048, 6144), (17, 12288, 2048), (1, 4096, 320)])
def test_op_few_gemm_vs_f64(oracle, S, N, K, prec):
    """Whole and partial row tiles, K from less than a slice per wave up to 24, every weight tile
    width.  Bound: a wave adds 3 K / 256 matrix instructions (K / 256 more for a q4_0 block's scale), the
    workgroup eight waves, x gain and 1/rms round once: that many roundings of 2^-24, of either sign,
    times 4.  Operands without their third plane would be past it."""
    print(f"[case] few {prec} S={S} N={N} K={K}", flush=True)
    rng = np.random.default_rng(S * 131 + N + K)
    W, scale, W64 = _weights(oracle, prec, synth.f32_to_bf16_rne((rng.standard_normal((N, K)) * 0.05).astype(np.float32)))
    X = (rng.standard_normal((S, K)) * np.exp(rng.uniform(-3, 3, (S, 1)))).astype(np.float32)
    gain = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32)
    ng = (1 + 0.1 * rng.standard_normal(N)).astype(np.float32)
    bound = 4 * 2.0 ** -24 * np.sqrt(4 * K / 256 + 8 + 3)
    xg = X.astype(np.float64) * gain
    rms = 1.0 / np.sqrt((X.astype(np.float64) ** 2).mean(1, keepdims=True) + EPS)
    want = xg @ W64.T
    lost = rel_l2(_two_planes(X * gain).astype(np.float64) @ W64.T, want)
    assert lost > bound, (lost, bound)

    Y, _, _ = _few(prec, STORE, W, scale, X, N, gain)
    assert rel_l2(Y, want * rms) <= bound, (rel_l2(Y, want * rms), bound)

    if N <= 4096:                                    # the widest residual row
        Y0 = (rng.standard_normal((S, N)) * np.abs(want).mean()).astype(np.float32)
        Y, planes, sums = _few(prec, RESID, W, scale, X, N, gain, Y0, ng)
        assert np.linalg.norm(Y - (Y0 + want)) <= bound * (np.linalg.norm(want) + np.linalg.norm(Y0))
        assert np.array_equal(planes.astype(np.float64).sum(0), (Y * ng).astype(np.float64))      # exact planes
        sq = (Y.astype(np.float64) ** 2).reshape(S, N // 16, 16).sum(2)
        assert np.abs(sums - sq).max() <= 16 * 2.0 ** -24 * sq.max()

    _, planes, _ = _few(prec, SWIGLU, W, scale, X, N, gain)
    h = planes.astype(np.float64).sum(0)
    g, u = (want * rms)[:, 0::2], (want * rms)[:, 1::2]
    e = np.exp(-g)
    # the gate's error passes through the sigmoid's slope, expf and the division add a few roundings
    scale_g = np.linalg.norm(want * rms) / np.sqrt(g.size * 2)
    slope = np.abs((1 + e * (1 + g)) / (1 + e) ** 2 * u) + np.abs(g / (1 + e))
    assert np.linalg.norm(h - g / (1 + e) * u) <= 2 * bound * scale_g * np.linalg.norm(slope) + 8 * 2.0 ** -24 * np.linalg.norm(h)
    assert np.array_equal(h.astype(np.float32).astype(np.float64), h)


@pytest.mark.parametrize("prec", ["bf16", "int8", "q4_0"])
def test_op_few_gemm_planes_are_exact(prec):
    """A weight of 1 at column k picks x[k] out bit for bit: the planes hold all of it, over forty
    binary orders of magnitude."""
    K, N, S = 320, 64, 21
    at = (7 * np.arange(N)) % K
    scale = None
    if prec == "bf16":
        W = np.zeros((N, K), np.uint16)
        W[np.arange(N), at] = 0x3F80
    elif prec == "int8":
        W, scale = np.zeros((N, K), np.int8), np.ones(N, np.float32)
        W[np.arange(N), at] = 1
    else:
        n = np.full((N, K), 8)
        n[np.arange(N), at] = 9
        n = n.reshape(N, K // 32, 32)
        W = np.zeros((N, K // 32, 18), np.uint8)
        W[..., :2] = np.frombuffer(np.float16(1).tobytes(), np.uint8)
        W[..., 2:] = n[..., 0::2] | (n[..., 1::2] << 4)
    rng = np.random.default_rng(9)
    X = (rng.standard_normal((S, K)) * np.exp(rng.uniform(-14, 14, (S, K)))).astype(np.float32)
    one = np.ones(K, np.float32)
    Y, planes, _ = _few(prec, RESID, W, scale, X, N, one, None, np.ones(N, np.float32))
    assert np.array_equal(Y, X[:, at])
    assert np.array_equal(planes.astype(np.float64).sum(0), X[:, at].astype(np.float64))


@pytest.mark.parametrize("prec", ["bf16", "int8", "q4_0"])
def test_op_few_gemm_non_finite_rows(oracle, prec):
    """An infinity or a NaN makes its row NaN (the norm's 0 times infinity), a row whose squares overflow
    becomes 0 as x * (1 / rms) does, up to the largest float, and no other row changes by a bit."""
    S, N, K = 37, 128, 512
    rng = np.random.default_rng(3)
    W, scale, _ = _weights(oracle, prec, synth.f32_to_bf16_rne((rng.standard_normal((N, K)) * 0.05).astype(np.float32)))
    X = rng.standard_normal((S, K)).astype(np.float32)
    gain, ng = (1 + 0.1 * rng.standard_normal(K)).astype(np.float32), (1 + 0.1 * rng.standard_normal(N)).astype(np.float32)
    Y0 = rng.standard_normal((S, N)).astype(np.float32)
    clean = [_few(prec, e, W, scale, X, N, gain, Y0, ng) for e in (STORE, RESID, SWIGLU)]
    X[2, 5], X[17, 511], X[36, 0] = np.inf, np.nan, -np.inf
    X[20] *= 1e25
    X[21] = np.sign(X[21]) * np.finfo(np.float32).max
    Y0[20], Y0[21] = 1e25, np.finfo(np.float32).max
    nan, big, rest = [2, 17, 36], [20, 21], np.delete(np.arange(S), [2, 17, 20, 21, 36])
    y, _, _ = _few(prec, STORE, W, scale, X, N, gain)
    assert np.isnan(y[nan]).all() and not y[big].any() and np.array_equal(y[rest], clean[0][0][rest])
    _, h, _ = _few(prec, SWIGLU, W, scale, X, N, gain)
    assert np.isnan(h.sum(0)[nan]).all() and not h[:, big].any() and np.array_equal(h[:, rest], clean[2][1][:, rest])
    X[big] = 0.0
    y, p, ss = _few(prec, RESID, W, scale, X, N, gain, Y0, ng)
    assert not np.isfinite(y[nan]).any() and not np.isfinite(ss[nan]).any()
    assert np.array_equal(y[big], Y0[big]) and np.isinf(ss[big]).all() and np.isfinite(p[:, big]).all()
    for got, want in zip((y, p.swapaxes(0, 1), ss), (clean[1][0], clean[1][1].swapaxes(0, 1), clean[1][2])):
        assert np.array_equal(got[rest], want[rest])
