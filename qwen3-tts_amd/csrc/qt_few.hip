// qt_few.hip — projections of a few rows (the batched step's streams, a short
// prompt's positions: at most 64) on gfx950.
//
// Y = X . W^T with W bf16 [N][K] as stored and X f32, as the exact products of qt_prefill.hip:
// each activation is the sum of three bf16 planes, a plane times a weight is exact in f32, and
// the matrix cores sum in f32.  Such a product is a stream of the weights, and what it costs
// beyond that is latency: a launch is done in one pass, with nothing summed by another one.
//
// bf16, 0.6B, 28 layers: six streams 1.79 -> 1.08 ms a step; 45 positions 1.83 -> 1.47 ms.
// q4_0 (before: int8 pieces of the activations on the integer matrix cores): 1.7B, 2 streams 2.09 ->
// 1.53, 12 2.23 -> 1.70, 32 2.63 -> 2.1 ms; 0.6B, 4 1.65 -> 1.1, 48 2.46 -> 1.7; error against 64 bits
// of 12 streams 3.2e-5 -> 1.1e-5.
// int8 (before: the same pieces, made inside each projection's launch): 0.6B, 2 streams 1.18 -> 0.99, 16
// 1.34 -> 1.15, 32 1.64 -> 1.39, 48 1.94 -> 1.75; 1.7B, 2 1.40 -> 1.35, 8 1.51 -> 1.44; error against 64
// bits 3.2e-5 -> 3e-6.
//
//   * a workgroup owns 16 NT weight rows for all of K; its eight waves take an eighth of K each
//     and their sums meet in LDS;
//   * the activations come as planes in operand order (qt_frag_at), written so by whoever
//     made them;
//   * int8 weights are exact in bf16 as well, their row scale multiplies the sums;
//   * a q4_0 block is 32 k, one matrix instruction deep: its weights n - 8 are exact in bf16, its
//     sums start from zero, and its f16 scale multiplies them in f32;
//   * RMSNorm is applied around the product: the planes are those of x * gain, each maker of
//     16 columns of x leaves the sum of their squares (one float a row), and the consumer
//     scales its sums by 1/rms: the row's statistic needs no launch of its own.  (An x whose
//     square overflows is cut, qf_cut.)
#include "qt_planes.h"

#define QF_W 8                   // waves of a workgroup, and parts of K
#define QF_T (64 * QF_W)
#define QF_ROWS 64               // rows at most
#define QF_QPER 32               // q4_0: K slices of a wave at most (K <= 8192)
#define QF_PART 256              // partial sums of squares at most (hidden <= 4096)

// (the values of qt_launch.h, which the .hip sources do not include)
enum { QF_STORE = 0, QF_RESID = 1, QF_SWIGLU = 2 };
enum { QF_BF16 = 0, QF_INT8 = 1, QF_Q4 = 2 };

struct QtFewArgs {
    const void *W;               // bf16 [N][K]; int8 [N][K]; or q4_0 nibbles [N][K / 2] ...
    const uint16_t *s16;         // ... and f16 block scales [N][K / 32]
    const float *scale;          // int8: row scales [N]
    const uint16_t *P;           // the input's planes
    int N, K, S, RT;             // RT: row tiles of the planes
    const float *ssp; int np;    // STORE, SWIGLU: the rows' partial sums of squares [row][np] (the input is normed)
    float eps;
    float *Y; int ldy;           // STORE: Y = v; RESID: Y += v
    const float *gain;           // RESID with Pout: the next norm's gain
    uint16_t *Pout; float *sspo; // RESID (may be NULL): planes of Y * gain and its partial sums; SWIGLU: planes of h
};

// planes of four neighbouring values (columns k..k+3 of a row, k a multiple of 4)
__device__ __forceinline__ void qf_put4(uint16_t *P, int RT, int row, int k, qt_f32x4 v) {
    uint16_t pc[3][4];
#pragma unroll
    for (int e = 0; e < 4; e++) qt_put_pieces(&pc[0][e], 4, v[e]);
    uint16_t *d = P + qt_frag_at(RT, row, k);
#pragma unroll
    for (int p = 0; p < 3; p++)
        *reinterpret_cast<uint2 *>(d + 512 * p) =
            make_uint2((uint32_t)pc[p][0] | ((uint32_t)pc[p][1] << 16), (uint32_t)pc[p][2] | ((uint32_t)pc[p][3] << 16));
}

// x as the planes of x * gain take it: past 2^64 its square alone is past f32's range, the row's 1/rms
// is 0 and its result 0 (as x (1/rms) is), whatever finite value x has; cut there, the sums that the 0
// multiplies stay finite.  An infinity or a NaN stays one.
__device__ __forceinline__ float qf_cut(float x) { return fabsf(x) > 0x1p64f && fabsf(x) < INFINITY ? copysignf(0x1p64f, x) : x; }
__device__ __forceinline__ qt_f32x4 qf_cut4(qt_f32x4 v) { return qt_f32x4{qf_cut(v[0]), qf_cut(v[1]), qf_cut(v[2]), qf_cut(v[3])}; }

// 8 weights as a lane's operand: bf16 as they are, int8 converted (exact), q4_0 nibbles (element e in bits 4 e, + 8) unpacked
template <int PREC> struct QfWord { using t = qt_u32x4; };
template <> struct QfWord<QF_INT8> { using t = uint2; };
template <> struct QfWord<QF_Q4> { using t = uint32_t; };
__device__ __forceinline__ qt_u32x4 qf_i8(uint2 w) {
    qt_u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int v = (int)(i < 2 ? w.x : w.y) << (16 * (1 - (i & 1)));   // the pair in the upper half
        r[i] = qt_bf16x2((float)(v << 8 >> 24), (float)(v >> 24));
    }
    return r;
}
__device__ __forceinline__ qt_u32x4 qf_q4(uint32_t n) {
    const int v = (int)(n ^ 0x88888888u);           // two's complement nibbles of n - 8
    qt_u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = qt_bf16x2((float)(v << (28 - 8 * i) >> 28), (float)(v << (24 - 8 * i) >> 28));
    return r;
}

// A workgroup computes 16 NT weight rows for 16 activation rows; each wave has D slices of 32 k of
// both in flight (all of its eighth of K where the registers hold it: one memory latency).
template <int NT, int D, int EPI, int PREC>
__global__ __launch_bounds__(QF_T) void k_few(QtFewArgs a) {
    constexpr bool Q4 = PREC == QF_Q4;
    __shared__ __align__(16) qt_f32x4 part[QF_W][NT][64];
    __shared__ float s_inv[16];
    // q4_0: the block scales of each wave's slices, [slice][weight row], filled and read by that wave
    __shared__ __align__(16) float s_sc[Q4 ? QF_W : 1][Q4 ? QF_QPER : 1][16 * NT];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, kg = lane >> 4;
    const int n0 = blockIdx.x * 16 * NT, rt = blockIdx.y, ns = a.K / 32;
    const int s0 = ns * wave / QF_W, s1 = ns * (wave + 1) / QF_W;
    // what the epilogue needs is asked for first: the rows' partial sums of squares (16 threads a
    // row), and, in the waves that finish a tile, the residual and the next gain
    constexpr bool NORM = EPI != QF_RESID;
    qt_f32x4 sv[QF_PART / 64];
    if (NORM) {
        const float *ss = a.ssp + (size_t)min(16 * rt + ((tid >> 4) & 15), a.S - 1) * a.np;
#pragma unroll
        for (int i = 0; i < QF_PART / 64; i++) sv[i] = *reinterpret_cast<const qt_f32x4 *>(ss + min(64 * i + 4 * (tid & 15), a.np - 4));
    }
    const int row = 16 * rt + li, n = n0 + 16 * wave + 4 * kg;       // the output of a finishing wave
    const bool mine = wave < NT && row < a.S;
    qt_f32x4 old = {0.f, 0.f, 0.f, 0.f}, gn = old, rs = old;
    if (PREC == QF_INT8 && mine) rs = *reinterpret_cast<const qt_f32x4 *>(a.scale + n);
    if (EPI == QF_RESID && mine) {
        old = *reinterpret_cast<const qt_f32x4 *>(a.Y + (size_t)row * a.ldy + n);
        if (a.Pout) gn = *reinterpret_cast<const qt_f32x4 *>(a.gain + n);
    }
    // rows past S repeat the last one: nothing more is read for them
    using wt = typename QfWord<PREC>::t;            // 8 weights of a lane
    const uint8_t *wp[NT];
    const uint16_t *xp = a.P + (size_t)rt * 1536 + 8 * (min(li, a.S - 1 - 16 * rt) + 16 * kg);
#pragma unroll
    for (int j = 0; j < NT; j++)
        wp[j] = (const uint8_t *)a.W + (size_t)(n0 + 16 * j + li) * (a.K / 32) * (4 * sizeof(wt)) + kg * sizeof(wt);
    wt w[D][NT];
    qt_u32x4 x[D][3];
    const size_t xs = (size_t)a.RT * 1536;
    auto fetch = [&](int s, int d) {
#pragma unroll
        for (int j = 0; j < NT; j++) w[d][j] = *reinterpret_cast<const wt *>(wp[j] + s * (int)(4 * sizeof(wt)));
#pragma unroll
        for (int p = 0; p < 3; p++) x[d][p] = *reinterpret_cast<const qt_u32x4 *>(xp + s * xs + 512 * p);
    };
    qt_f32x4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[j] = qt_f32x4{0.f, 0.f, 0.f, 0.f};
    auto mul = [&](int s, int d) {
        if constexpr (Q4) {
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const qt_u32x4 q = qf_q4(w[d][j]);
                qt_f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int p = 0; p < 3; p++) c = qt_mfma_bf16(q, x[d][2 - p], c);
                const qt_f32x4 sc = *reinterpret_cast<const qt_f32x4 *>(&s_sc[wave][s - s0][16 * j + 4 * kg]);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[j][r] = fmaf(c[r], sc[r], acc[j][r]);
            }
        } else {
            qt_u32x4 q[NT];
#pragma unroll
            for (int j = 0; j < NT; j++) {
                if constexpr (PREC == QF_INT8) q[j] = qf_i8(w[d][j]);
                else q[j] = w[d][j];
            }
#pragma unroll
            for (int p = 0; p < 3; p++)
#pragma unroll
                for (int j = 0; j < NT; j++) acc[j] = qt_mfma_bf16(q[j], x[d][2 - p], acc[j]);
        }
    };
    // q4_0: four blocks' scales of a weight row a load, asked for ahead of the weights (K a multiple of
    // 1024: a wave's slices are whole fours)
    const bool fours = Q4 && a.K % 1024 == 0;
    uint2 sr[QF_QPER / 16][NT];
    if (fours) {
#pragma unroll
        for (int i = 0; i < QF_QPER / 16; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
                sr[i][j] = *reinterpret_cast<const uint2 *>(a.s16 + (size_t)(n0 + 16 * j + li) * ns + s0 + min(4 * kg + 16 * i, s1 - s0 - 4));
    }
    // loads past the wave's last slice repeat it: no load is behind a branch, so that the waits count them
    const int last = max(s1 - 1, 0);
#pragma unroll
    for (int d = 0; d < D; d++) fetch(min(s0 + d, last), d);
    if constexpr (Q4) {
        if (fours) {
#pragma unroll
            for (int i = 0; i < QF_QPER / 16; i++)
                if (4 * kg + 16 * i < s1 - s0)
#pragma unroll
                    for (int j = 0; j < NT; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            s_sc[wave][4 * kg + 16 * i + e][16 * j + li] =
                                ref_f16_to_f32(((e < 2 ? sr[i][j].x : sr[i][j].y) >> (16 * (e & 1))) & 0xFFFFu);
        } else {
            for (int i = kg; i < s1 - s0; i += 4)
#pragma unroll
                for (int j = 0; j < NT; j++)
                    s_sc[wave][i][16 * j + li] = ref_f16_to_f32(a.s16[(size_t)(n0 + 16 * j + li) * ns + s0 + i]);
        }
        __builtin_amdgcn_wave_barrier();
    }
    int s = s0;
    for (; s + D < s1; s += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            mul(s + d, d);
            fetch(min(s + d + D, last), d);
        }
    }
#pragma unroll
    for (int d = 0; d < D; d++)
        if (s + d < s1) mul(s + d, d);
#pragma unroll
    for (int j = 0; j < NT; j++) part[wave][j][lane] = acc[j];
    if (NORM) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < QF_PART / 64; i++) ss += 64 * i + 4 * (tid & 15) < a.np ? (sv[i][0] + sv[i][1]) + (sv[i][2] + sv[i][3]) : 0.f;
        ss = group_sum<16>(ss);
        if (tid < 256 && (tid & 15) == 0) s_inv[tid >> 4] = 1.0f / sqrtf(ss / (float)a.K + a.eps);
    }
    __syncthreads();
    if (!mine) return;
    qt_f32x4 v = part[0][wave][lane];
#pragma unroll
    for (int g = 1; g < QF_W; g++) v += part[g][wave][lane];
    if (PREC == QF_INT8) v *= rs;
    if (NORM) v *= s_inv[li];
    if (EPI == QF_SWIGLU) {                        // rows 2i, 2i + 1 of W are gate_i, up_i
        // rounded products, split as they are
        const float h0 = __fmul_rn(v[0] / (1.0f + expf(-v[0])), v[1]), h1 = __fmul_rn(v[2] / (1.0f + expf(-v[2])), v[3]);
        uint16_t pc[3][2];
        qt_put_pieces(&pc[0][0], 2, h0);
        qt_put_pieces(&pc[0][1], 2, h1);
        uint16_t *d = a.Pout + qt_frag_at(a.RT, row, n >> 1);
#pragma unroll
        for (int p = 0; p < 3; p++) *reinterpret_cast<uint32_t *>(d + 512 * p) = (uint32_t)pc[p][0] | ((uint32_t)pc[p][1] << 16);
    } else if (EPI == QF_RESID) {
        v = old + v;
        *reinterpret_cast<qt_f32x4 *>(a.Y + (size_t)row * a.ldy + n) = v;
        if (a.Pout) {
            float sq = fmaf(v[3], v[3], fmaf(v[2], v[2], fmaf(v[1], v[1], v[0] * v[0])));
            qt_f32x4 c = v;
            if (__any(!(sq < INFINITY))) c = qf_cut4(v);
            qf_put4(a.Pout, a.RT, row, n, c * gn);
            sq += __shfl_xor(sq, 16);              // a row's four lanes are all in the tile or all past S
            sq += __shfl_xor(sq, 32);
            if (kg == 0) a.sspo[(size_t)row * (a.N / 16) + blockIdx.x * NT + wave] = sq;
        }
    } else {
        *reinterpret_cast<qt_f32x4 *>(a.Y + (size_t)row * a.ldy + n) = v;
    }
}

// planes of x * gain and each row's sum of squares (as QF_FIRST partial sums, all but one zero)
#define QF_FIRST 4
__global__ __launch_bounds__(256) void k_few_planes(const float *X, int ldx, int K, int RT, const float *gain, uint16_t *P,
                                                    float *ssp) {
    __shared__ float red[QT_WAVES];
    const int row = blockIdx.x;
    const float *x = X + (size_t)row * ldx;
    float ss = 0.f;
    for (int k = 4 * threadIdx.x; k < K; k += 1024) {
        qt_f32x4 v = *reinterpret_cast<const qt_f32x4 *>(x + k);
        ss = fmaf(v[3], v[3], fmaf(v[2], v[2], fmaf(v[1], v[1], fmaf(v[0], v[0], ss))));
        qf_put4(P, RT, row, k, qf_cut4(v) * *reinterpret_cast<const qt_f32x4 *>(gain + k));
    }
    ss = block_sum(ss, red);
    if (threadIdx.x < QF_FIRST) ssp[row * QF_FIRST + threadIdx.x] = threadIdx.x ? 0.f : ss;
}

// ---- launchers ----------------------------------------------------------------------------
// The rows fit while the widest projection has few enough tiles that its workgroups (of up to four)
// run in about one round; with more rounds of one latency each the prefill's tiles are the faster ones.
// 28 layers, 0.6B / 1.7B: 16 rows 1.23 against 1.75 / 1.80 against 2.21 ms, 32 rows - / 2.09 against
// 2.32, 64 rows 1.48 against 1.93 / 2.80 against 2.55 (1.7B: 32 rows are the most).  int8 has the integer
// matrix cores on the other side and goes up to three quarters of that: a step of 16 streams 1.15 against
// 1.34 / 1.57 against 1.58 ms, 17 - / 1.92 against 1.91, 32 1.39 against 1.64 / 3.10 against 2.99, 48 1.75
// against 1.94 / -.
extern "C" int qt_few_ok(int prec, int S, int H, int F, int qd, int qkvr) {
    return S >= 1 && S <= QF_ROWS && H % 64 == 0 && F % 64 == 0 && qd % 64 == 0 && qkvr % 64 == 0 && H / 16 <= QF_PART &&
           (long long)(F / 8 > qkvr / 16 ? F / 8 : qkvr / 16) * ((S + 15) / 16) <= (prec == QF_INT8 ? 1152 : 1536) &&
           (prec != QF_Q4 || (H <= 256 * QF_QPER && F <= 256 * QF_QPER && qd <= 256 * QF_QPER));
}
extern "C" int qt_few_first(void) { return QF_FIRST; }
extern "C" size_t qt_few_planes_elems(int S, int K) { return (size_t)((S + 15) / 16) * 16 * K * 3; }

extern "C" hipError_t qt_launch_few_planes(const float *X, int ldx, int S, int K, const float *gain, uint16_t *P, float *ssp,
                                           hipStream_t st) {
    if (!X || !P || !gain || !ssp || S < 1 || S > QF_ROWS || K < 64 || K % 64 || ldx < K || ldx % 4) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_few_planes, dim3(S), dim3(256), 0, st, X, ldx, K, (S + 15) / 16, gain, P, ssp);
    return hipGetLastError();
}

template <int NT, int D, int PREC>
static hipError_t few_launch(int epi, const QtFewArgs &a, hipStream_t st) {
    const dim3 grid(a.N / (16 * NT), a.RT);
    if (epi == QF_STORE) hipLaunchKernelGGL((k_few<NT, D, QF_STORE, PREC>), grid, dim3(QF_T), 0, st, a);
    else if (epi == QF_RESID) hipLaunchKernelGGL((k_few<NT, D, QF_RESID, PREC>), grid, dim3(QF_T), 0, st, a);
    else hipLaunchKernelGGL((k_few<NT, D, QF_SWIGLU, PREC>), grid, dim3(QF_T), 0, st, a);
    return hipGetLastError();
}

// nt weight tiles a workgroup, `per` K slices a wave: the fewest slices in flight that hold them all,
// as far as the registers go
template <int PREC>
static hipError_t few_pick(int epi, int nt, int per, const QtFewArgs &a, hipStream_t st) {
    if (nt == 1)
        return per <= 4 ? few_launch<1, 4, PREC>(epi, a, st) : per <= 8 ? few_launch<1, 8, PREC>(epi, a, st)
                                                                        : few_launch<1, 12, PREC>(epi, a, st);
    if (nt == 2) return per <= 4 ? few_launch<2, 4, PREC>(epi, a, st) : few_launch<2, 8, PREC>(epi, a, st);
    if (nt == 3) return per <= 4 ? few_launch<3, 4, PREC>(epi, a, st) : few_launch<3, 8, PREC>(epi, a, st);
    if constexpr (PREC != QF_BF16)
        if (per > 4) return few_launch<4, 8, PREC>(epi, a, st);
    return few_launch<4, 4, PREC>(epi, a, st);
}

// prec: QT_BF16, QT_INT8 (scale: row scales) or QT_Q4 (s16: block scales)
extern "C" hipError_t qt_launch_few_gemm(int prec, int epi, const void *W, const float *scale, const uint16_t *s16, int N, int K,
                                         const uint16_t *P, int S, const float *ssp, int np, float eps, float *Y, int ldy,
                                         const float *gain, uint16_t *Pout, float *sspo, hipStream_t st) {
    if (!W || !P || S < 1 || S > QF_ROWS || N < 64 || N % 64 || K < 64 || K % 64 || epi < 0 || epi > 2 || prec < QF_BF16 || prec > QF_Q4 ||
        (prec == QF_INT8 && !scale) || (prec == QF_Q4 && (!s16 || K > 256 * QF_QPER)) ||
        (epi != QF_RESID && (!ssp || np < 4 || np % 4 || np > QF_PART)) ||
        (epi != QF_SWIGLU && (!Y || ldy < N || ldy % 4)) ||
        (epi == QF_SWIGLU && !Pout) || (epi == QF_RESID && Pout && (!gain || !sspo || N / 16 > QF_PART)))
        return hipErrorInvalidValue;
    const QtFewArgs a = {W, s16, scale, P, N, K, S, (S + 15) / 16, ssp, np, eps, Y, ldy, gain, Pout, sspo};
    // the tile whose busiest CU reads the fewest bytes (16 K (2 NT + 6) a workgroup; int8 NT + 6, q4_0
    // NT / 2 + 6), one workgroup a CU
    int nt = 1;
    long long best = -1;
    for (int t = 1; t <= 4; t++) {
        if (N % (16 * t)) continue;
        const long long c = ((long long)(N / (16 * t)) * a.RT + 255) / 256 * ((prec == QF_BF16 ? 4 * t : prec == QF_INT8 ? 2 * t : t) + 12);
        if (best < 0 || c < best) { best = c; nt = t; }
    }
    const int per = (K / 32 + QF_W - 1) / QF_W;    // slices of a wave
    return prec == QF_Q4 ? few_pick<QF_Q4>(epi, nt, per, a, st) : prec == QF_INT8 ? few_pick<QF_INT8>(epi, nt, per, a, st)
                                                                                  : few_pick<QF_BF16>(epi, nt, per, a, st);
}
