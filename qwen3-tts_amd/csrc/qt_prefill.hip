// qt_prefill.hip — Talker prefill (qwen_talker_prefill, qwen_tts_talker.c:730-1038) on gfx950.
//
// The reference runs the prompt's positions as dense projections Y[seq][out] =
// Xn[seq][in] . W^T over the bf16 layer weights with f32 sums (sgemm or
// qwen_matmat_bf16, t.c:845-847, 913, 964, 990), per-head q/k RMSNorm, NeoX RoPE at each
// position, the bf16-truncated K/V store (t.c:897-899), causal attention over the f32
// q/k/v (t.c:901-907), O + residual, RMSNorm + gate|up + SwiGLU, down + residual.
//
// Projections here run on the bf16 matrix cores.  The f32 activations are split
// into three bf16 planes whose sum is each value exactly (x truncated to bf16, the
// truncated rest, the remaining <= 8 significant bits; qt_attn_mf.h); W . x = sum over
// the planes of W . x_p, and each bf16 x bf16 product is exact in f32, so the three
// MFMAs per k-step accumulate, in f32, the exact products of the f32 activations with
// the bf16 weights.  Both operands are read row-major exactly as stored: the MFMA A
// operand is 16 weight rows x 8 consecutive k, the B operand 16 positions x 8
// consecutive k of one plane, so neither needs a transpose.
#include "qt_planes.h"

#define QT_PF_WG 256

// ---- activation planes ---------------------------------------------------------------
// Row s < S of X (ldx floats apart), optionally RMS-normalised with gain (the reference's
// qwen_rms_norm: out = (x * inv) * w, inv = 1/sqrt(mean(x^2) + eps), k.c:292-382), as
// three bf16 planes P[p][s][K] (plane stride Sp*K); rows S <= s < Sp are zero.
__global__ __launch_bounds__(QT_PF_WG) void k_pf_pieces(const float *X, int ldx, int S, int Sp, int K,
                                                         const float *gain, float eps, uint16_t *P) {
    __shared__ float red[QT_WAVES];
    const int s = blockIdx.x, tid = threadIdx.x;
    const size_t plane = (size_t)Sp * K;
    uint16_t *p0 = P + (size_t)s * K;
    if (s >= S) {
        for (int k = tid * 8; k < K; k += QT_PF_WG * 8)
#pragma unroll
            for (int p = 0; p < 3; p++) *reinterpret_cast<uint4 *>(p0 + p * plane + k) = make_uint4(0u, 0u, 0u, 0u);
        return;
    }
    const float *x = X + (size_t)s * ldx;
    float inv = 1.0f;
    if (gain) {
        float ss = 0.f;
        for (int k = tid; k < K; k += QT_PF_WG) ss = fmaf(x[k], x[k], ss);
        ss = block_sum(ss, red);
        inv = 1.0f / sqrtf(ss / (float)K + eps);
    }
    for (int k = tid * 4; k < K; k += QT_PF_WG * 4) {
        float4 v = *reinterpret_cast<const float4 *>(x + k);
        if (gain) {
            const float4 g = *reinterpret_cast<const float4 *>(gain + k);
            v.x = (v.x * inv) * g.x; v.y = (v.y * inv) * g.y; v.z = (v.z * inv) * g.z; v.w = (v.w * inv) * g.w;
        }
        uint16_t pc[3][4];
        const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) qt_put_pieces(&pc[0][i], 4, e[i]);
#pragma unroll
        for (int p = 0; p < 3; p++)
            *reinterpret_cast<uint2 *>(p0 + p * plane + k) =
                make_uint2((uint32_t)pc[p][0] | ((uint32_t)pc[p][1] << 16), (uint32_t)pc[p][2] | ((uint32_t)pc[p][3] << 16));
    }
}

// ---- projection GEMM ------------------------------------------------------------------
// Y = X . W^T: W bf16 [N][K] row-major, X as the planes P[3][Sp][K].  Workgroup tile:
// 64*NR weight rows x 64 positions; wave w takes rows [16*NR*w, 16*NR*(w+1)) of it and
// every position; the weight fragments go straight from HBM to registers (each wave reads
// its own rows once), the planes' tile is shared through LDS.
//   PF_STORE   Y[s][n] = acc
//   PF_RESID   Y[s][n] += acc                     (O, down: the residual stream)
//   PF_SWIGLU  rows 2i, 2i+1 are gate_i, up_i (the reference's interleaved gate|up,
//              t.c:378-388): Y[s][i] = g / (1 + e^-g) * u  (qwen_swiglu_inplace, k.c:3857)
// (the same values as in qt_launch.h, which the .hip sources do not include)
enum { QT_PF_STORE = 0, QT_PF_RESID = 1, QT_PF_SWIGLU = 2 };

// NST chunks of 64 k are in flight: each chunk's planes (3 x 64
// positions x 128 B) go straight from HBM into LDS stage c % NST by global_load_lds (no
// registers; lane L of a 1-KiB copy fills slot L%8 of row 8b + L/8 and fetches the chunk
// that belongs there: chunk c of row r sits at slot c ^ ((r >> 1) & 7), so the 16 lanes of
// a B-operand read (rows j, one chunk) hit 16 different bank groups), and its weight
// fragments into registers, NST - 1 chunks ahead.  One barrier per chunk: after the wait
// for chunk c, every wave is also done with chunk c - 1, whose stage takes chunk
// c + NST - 1.  blockIdx.z selects one of gridDim.z equal K ranges (split K): with
// PF_PART the workgroup stores its partial tile at Y + z * S * ldy (k_pf_reduce adds the
// ranges in order).
enum { QT_PF_PART = 3 };
template <int N>
__device__ __forceinline__ void qt_vmcnt() {   // wait until at most N vector-memory ops are outstanding
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Two waves per SIMD for the two-stage tile (amdgpu_waves_per_eu(2)): the 256-row tile
// with two stages fits in 202 registers per lane, so two workgroups share a CU and hide
// each other's chunk waits (the three-stage 256-row tile held 304 registers, one wave per
// SIMD); the four-stage tiles' 96 KB of LDS allow one workgroup per CU anyway.
template <int EPI, int NR, int NST>
__global__ __launch_bounds__(QT_PF_WG) __attribute__((amdgpu_waves_per_eu(NST == 2 ? 2 : 1))) void k_pf_gemm2(const uint16_t *__restrict__ W, const uint16_t *__restrict__ P,
                                                        int S, int Sp, int K, float *Y, int ldy) {
    constexpr int KC = 64, ST = 64, STB = 3 * ST * KC * 2;      // one stage: 24 KiB
    constexpr int NB = STB / 1024 / QT_WAVES;                   // 1-KiB copies per wave per chunk (6)
    constexpr int OPS = NB + 2 * NR;                            // vector-memory ops per wave per chunk
    static_assert(NB * 1024 * QT_WAVES == STB, "copy split");
    __shared__ __align__(16) uint8_t sp[NST * STB];             // NST stages
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 15, kg = lane >> 4;
    const int n0 = blockIdx.x * (64 * NR) + wave * 16 * NR;
    const int s0 = blockIdx.y * ST;
    const int kr = K / gridDim.z, k0 = blockIdx.z * kr, nch = kr / KC;
    const size_t plane = (size_t)Sp * K;
    if (EPI == QT_PF_PART) Y += (size_t)blockIdx.z * S * ldy;

    // this lane's source of each 1-KiB copy (chunk offset added per chunk)
    const uint16_t *src[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int row = 8 * (wave * NB + b) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        src[b] = P + (row / ST) * plane + (size_t)(s0 + row % ST) * K + k0 + 8 * c;
    }
    const uint16_t *wrow[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) wrow[r] = W + (size_t)(n0 + 16 * r + j) * K + k0 + 8 * kg;
    qt_u32x4 a[NST][2][NR];
    auto issue = [&](int c, int st) {   // chunk c into stage st (compile-time st)
        uint8_t *dst = sp + st * STB + (wave * NB) * 1024;
#pragma unroll
        for (int b = 0; b < NB; b++)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src[b] + c * KC),
                                             (__attribute__((address_space(3))) void *)(dst + b * 1024), 16, 0, 0);
    };
    qt_f32x4 acc[NR][4];
#pragma unroll
    for (int r = 0; r < NR; r++)
#pragma unroll
        for (int t = 0; t < 4; t++) acc[r][t] = qt_f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int c = 0; c < NST - 1; c++)
        if (c < nch) {
            issue(c, c);
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int r = 0; r < NR; r++) a[c][ks][r] = *reinterpret_cast<const qt_u32x4 *>(wrow[r] + c * KC + 32 * ks);
        }
    const int f = j >> 1;                               // row swizzle of this lane's B rows
    for (int cb = 0; cb < nch; cb += NST) {
#pragma unroll
        for (int u = 0; u < NST; u++) {
            const int c = cb + u;
            if (c >= nch) break;
            if (c + NST - 2 < nch) qt_vmcnt<(NST - 2) * OPS>();
            else qt_vmcnt<0>();
            __syncthreads();
            const int cn = c + NST - 1;                  // stage (u + NST - 1) % NST held chunk c - 1
            if (cn < nch) {
                issue(cn, (u + NST - 1) % NST);
#pragma unroll
                for (int ks = 0; ks < 2; ks++)
#pragma unroll
                    for (int r = 0; r < NR; r++)
                        a[(u + NST - 1) % NST][ks][r] = *reinterpret_cast<const qt_u32x4 *>(wrow[r] + cn * KC + 32 * ks);
            }
            const uint8_t *stg = sp + u * STB;
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                qt_u32x4 b[4][3];
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int p = 0; p < 3; p++)
                        b[t][p] = qt_lds16(stg + (p * ST + 16 * t + j) * (KC * 2) + 16 * ((4 * ks + kg) ^ f));
#pragma unroll
                for (int r = 0; r < NR; r++)
#pragma unroll
                    for (int t = 0; t < 4; t++)
#pragma unroll
                        for (int p = 0; p < 3; p++) acc[r][t] = qt_mfma_bf16(a[u][ks][r], b[t][p], acc[r][t]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < NR; r++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int s = s0 + 16 * t + j, n = n0 + 16 * r + 4 * kg;
            if (s >= S) continue;
            const qt_f32x4 v = acc[r][t];
            if constexpr (EPI == QT_PF_SWIGLU) {
                const float g0 = v[0], u0 = v[1], g1 = v[2], u1 = v[3];
                *reinterpret_cast<float2 *>(Y + (size_t)s * ldy + (n >> 1)) =
                    make_float2(g0 / (1.0f + expf(-g0)) * u0, g1 / (1.0f + expf(-g1)) * u1);
            } else {
                float4 *y = reinterpret_cast<float4 *>(Y + (size_t)s * ldy + n);
                if constexpr (EPI == QT_PF_RESID) {
                    const float4 o = *y;
                    *y = make_float4(o.x + v[0], o.y + v[1], o.z + v[2], o.w + v[3]);
                } else {
                    *y = make_float4(v[0], v[1], v[2], v[3]);
                }
            }
        }
}

// acc = sum over the nz K ranges of part[z][s][n..n+3], ranges in order (each range's
// loads issued before the adds), then the projection's epilogue: Y = acc (STORE),
// Y += acc (RESID), or the SwiGLU of the interleaved gate|up pairs into Y[s][n/2..n/2+1].
__device__ __forceinline__ float4 pf_sum_ranges(const float *part, int nz, int S, int N, int s, int n) {
    float4 acc = *reinterpret_cast<const float4 *>(part + (size_t)s * N + n);
    constexpr int ZB = 8;
    for (int z0 = 1; z0 < nz; z0 += ZB) {
        float4 v[ZB];
#pragma unroll
        for (int k = 0; k < ZB; k++)
            if (z0 + k < nz) v[k] = *reinterpret_cast<const float4 *>(part + ((size_t)(z0 + k) * S + s) * N + n);
#pragma unroll
        for (int k = 0; k < ZB; k++)
            if (z0 + k < nz) { acc.x += v[k].x; acc.y += v[k].y; acc.z += v[k].z; acc.w += v[k].w; }
    }
    return acc;
}

template <int EPI>
__global__ __launch_bounds__(QT_PF_WG) void k_pf_reduce(const float *part, int nz, int S, int N, float *Y, int ldy) {
    const int i = blockIdx.x * QT_PF_WG + threadIdx.x;
    if (i >= S * N / 4) return;
    const int s = i / (N / 4), n = 4 * (i % (N / 4));
    const float4 acc = pf_sum_ranges(part, nz, S, N, s, n);
    if constexpr (EPI == QT_PF_SWIGLU) {
        *reinterpret_cast<float2 *>(Y + (size_t)s * ldy + (n >> 1)) =
            make_float2(acc.x / (1.0f + expf(-acc.x)) * acc.y, acc.z / (1.0f + expf(-acc.z)) * acc.w);
    } else {
        float4 *y = reinterpret_cast<float4 *>(Y + (size_t)s * ldy + n);
        if constexpr (EPI == QT_PF_RESID) {
            const float4 o = *y;
            *y = make_float4(o.x + acc.x, o.y + acc.y, o.z + acc.z, o.w + acc.w);
        } else {
            *y = acc;
        }
    }
}

// The SwiGLU epilogue of the summed K ranges written straight as the three planes of h,
// the down projection's input (F = N/2 columns, P[p][s][F], plane stride Sp*F; rows
// S <= s < Sp zero): the same h values and the same pieces as k_pf_reduce<SWIGLU> followed
// by k_pf_pieces, one launch fewer.
__global__ __launch_bounds__(QT_PF_WG) void k_pf_reduce_swiglu_planes(const float *part, int nz, int S, int Sp, int N,
                                                                      uint16_t *P) {
    const int i = blockIdx.x * QT_PF_WG + threadIdx.x;
    if (i >= Sp * N / 4) return;
    const int s = i / (N / 4), n = 4 * (i % (N / 4));
    const int F = N / 2;
    const size_t plane = (size_t)Sp * F;
    uint16_t *dst = P + (size_t)s * F + (n >> 1);
    if (s >= S) {
#pragma unroll
        for (int p = 0; p < 3; p++) *reinterpret_cast<uint32_t *>(dst + p * plane) = 0u;
        return;
    }
    const float4 acc = pf_sum_ranges(part, nz, S, N, s, n);
    // rounded products (__fmul_rn: no contraction into the piece split), as stored by k_pf_reduce
    const float h0 = __fmul_rn(acc.x / (1.0f + expf(-acc.x)), acc.y), h1 = __fmul_rn(acc.z / (1.0f + expf(-acc.z)), acc.w);
    uint16_t pc[3][2];
    qt_put_pieces(&pc[0][0], 2, h0);
    qt_put_pieces(&pc[0][1], 2, h1);
#pragma unroll
    for (int p = 0; p < 3; p++)
        *reinterpret_cast<uint32_t *>(dst + p * plane) = (uint32_t)pc[p][0] | ((uint32_t)pc[p][1] << 16);
}

// The residual epilogue of the summed K ranges for one position row per workgroup (Y[s] +=
// acc, as k_pf_reduce<RESID>), then that row RMS-normalised with `gain` and written as the
// next projection's three input planes (P[p][s][N], plane stride Sp*N; rows S <= s < Sp
// zero): one launch fewer than with k_pf_pieces.  A hundred rows leave most of the chip idle and
// the time is the row's chain of latencies, so a row has eight waves (hidden 2048: one round of
// loads, all of them issued before the sums) and a thread norms the elements that it summed: no
// barrier but the statistic's.  1.7B: 128
// positions 7.2 -> 5.8 us with eight waves for four, 512 8.1 -> 7.3.
#define PF_ROW_T 512
__global__ __launch_bounds__(PF_ROW_T) void k_pf_reduce_resid_planes(const float *part, int nz, int S, int Sp, int N,
                                                                     float *Y, int ldy, const float *gain, float eps,
                                                                     uint16_t *P) {
    extern __shared__ __align__(16) float xr[];                // a thread's own elements, past its first four
    __shared__ float red[PF_ROW_T / 64];
    const int s = blockIdx.x, tid = threadIdx.x, n0 = 4 * tid;
    const size_t plane = (size_t)Sp * N;
    uint16_t *p0 = P + (size_t)s * N;
    if (s >= S) {
        for (int k = tid * 8; k < N; k += PF_ROW_T * 8)
#pragma unroll
            for (int p = 0; p < 3; p++) *reinterpret_cast<uint4 *>(p0 + p * plane + k) = make_uint4(0u, 0u, 0u, 0u);
        return;
    }
    float4 first = make_float4(0.f, 0.f, 0.f, 0.f), g0 = first;
    if (n0 < N) g0 = *reinterpret_cast<const float4 *>(gain + n0);
    float ss = 0.f;
    for (int n = n0; n < N; n += 4 * PF_ROW_T) {
        float4 *y = reinterpret_cast<float4 *>(Y + (size_t)s * ldy + n);
        const float4 o = *y;
        const float4 acc = pf_sum_ranges(part, nz, S, N, s, n);
        const float4 r = make_float4(o.x + acc.x, o.y + acc.y, o.z + acc.z, o.w + acc.w);
        *y = r;
        if (n == n0) first = r;
        else *reinterpret_cast<float4 *>(xr + n) = r;
        ss = fmaf(r.w, r.w, fmaf(r.z, r.z, fmaf(r.y, r.y, fmaf(r.x, r.x, ss))));
    }
    ss = group_sum<64>(ss);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < PF_ROW_T / 64; i++) ss += red[i];
    const float inv = 1.0f / sqrtf(ss / (float)N + eps);
    for (int k = n0; k < N; k += 4 * PF_ROW_T) {
        float4 v = k == n0 ? first : *reinterpret_cast<const float4 *>(xr + k);
        const float4 g = k == n0 ? g0 : *reinterpret_cast<const float4 *>(gain + k);
        v.x = (v.x * inv) * g.x; v.y = (v.y * inv) * g.y; v.z = (v.z * inv) * g.z; v.w = (v.w * inv) * g.w;
        uint16_t pc[3][4];
        const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) qt_put_pieces(&pc[0][i], 4, e[i]);
#pragma unroll
        for (int p = 0; p < 3; p++)
            *reinterpret_cast<uint2 *>(p0 + p * plane + k) =
                make_uint2((uint32_t)pc[p][0] | ((uint32_t)pc[p][1] << 16), (uint32_t)pc[p][2] | ((uint32_t)pc[p][3] << 16));
    }
}

// ---- per-head q/k norm, RoPE, KV store ---------------------------------------------
// Position s = blockIdx.x of QKV [S][ld] (q | k | v rows as the projection wrote them):
// q and k heads RMS-normalised with their [128] gains (qwen_rms_norm_per_head,
// k.c:486-577) and rotated at position s (apply_rope_neox_inplace, t.c:203-251:
// x1' = x1 c - x2 s, x2' = x2 c + x1 s), in place; the cache rows s of kv head g get the
// bf16 truncation of k and v (t.c:897-899).  One wave per head row, lane d holding
// elements d and d + 64 (the RoPE pair).
__global__ __launch_bounds__(QT_PF_WG) void k_pf_qkv_post(float *QKV, int ld, int nh, int nkv, const float *qn,
                                                           const float *kn, const float *rc, const float *rs, float eps,
                                                           uint16_t *kc, uint16_t *vc, long long kv_max) {
    const int s = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float *row = QKV + (size_t)s * ld;
    const float c = rc[(size_t)s * 64 + lane], sn = rs[(size_t)s * 64 + lane];
    for (int hr = wave; hr < nh + 2 * nkv; hr += QT_WAVES) {
        float *x = row + hr * 128;
        const float x0 = x[lane], x1 = x[lane + 64];
        if (hr < nh + nkv) {
            const bool isk = hr >= nh;
            const float *w = isk ? kn : qn;
            const float ss = group_sum<64>(x0 * x0 + x1 * x1);
            const float inv = 1.0f / sqrtf(ss / 128.0f + eps);
            const float n0 = (x0 * inv) * w[lane], n1 = (x1 * inv) * w[lane + 64];
            const float r0 = fmaf(n0, c, -(n1 * sn)), r1 = fmaf(n1, c, n0 * sn);
            x[lane] = r0;
            x[lane + 64] = r1;
            if (isk) {
                uint16_t *kd = kc + ((size_t)(hr - nh) * kv_max + s) * 128;
                kd[lane] = f2bf_trunc(r0);
                kd[lane + 64] = f2bf_trunc(r1);
            }
        } else {
            uint16_t *vd = vc + ((size_t)(hr - nh - nkv) * kv_max + s) * 128;
            vd[lane] = f2bf_trunc(x0);
            vd[lane + 64] = f2bf_trunc(x1);
        }
    }
}

// The q|k|v projection's summed K ranges for one position row per workgroup, kept in LDS,
// then k_pf_qkv_post's work on that row (per-head q/k norm, RoPE, KV store) with the same
// arithmetic; the row (q, k rotated, v as summed) is written once.  One launch fewer.  Sixteen
// waves a row, for the same reason: one round of loads, two heads a wave.  1.7B: 128 positions 7.7 ->
// 5.5 us with sixteen for four, 512 7.9 -> 6.9.
struct PfQkvPost {
    int nh, nkv;
    const float *qn, *kn, *rc, *rs;
    float eps;
    uint16_t *kc, *vc;
    long long kv_max;
};
#define PF_QKV_T 1024
__global__ __launch_bounds__(PF_QKV_T) void k_pf_reduce_qkv_post(const float *part, int nz, int S, int N, float *QKV,
                                                                 int ld, PfQkvPost a) {
    extern __shared__ __align__(16) float xr[];
    const int s = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float c = a.rc[(size_t)s * 64 + lane], sn = a.rs[(size_t)s * 64 + lane];
    const float qn0 = a.qn[lane], qn1 = a.qn[lane + 64], kn0 = a.kn[lane], kn1 = a.kn[lane + 64];
    for (int n = 4 * tid; n < N; n += 4 * PF_QKV_T)
        *reinterpret_cast<float4 *>(xr + n) = pf_sum_ranges(part, nz, S, N, s, n);
    __syncthreads();
    float *row = QKV + (size_t)s * ld;
    for (int hr = wave; hr < a.nh + 2 * a.nkv; hr += PF_QKV_T / 64) {
        float *x = row + hr * 128;
        const float x0 = xr[hr * 128 + lane], x1 = xr[hr * 128 + lane + 64];
        if (hr < a.nh + a.nkv) {
            const bool isk = hr >= a.nh;
            const float ss = group_sum<64>(x0 * x0 + x1 * x1);
            const float inv = 1.0f / sqrtf(ss / 128.0f + a.eps);
            const float n0 = (x0 * inv) * (isk ? kn0 : qn0), n1 = (x1 * inv) * (isk ? kn1 : qn1);
            const float r0 = fmaf(n0, c, -(n1 * sn)), r1 = fmaf(n1, c, n0 * sn);
            x[lane] = r0;
            x[lane + 64] = r1;
            if (isk) {
                uint16_t *kd = a.kc + ((size_t)(hr - a.nh) * a.kv_max + s) * 128;
                kd[lane] = f2bf_trunc(r0);
                kd[lane + 64] = f2bf_trunc(r1);
            }
        } else {
            x[lane] = x0;
            x[lane + 64] = x1;
            uint16_t *vd = a.vc + ((size_t)(hr - a.nh - a.nkv) * a.kv_max + s) * 128;
            vd[lane] = f2bf_trunc(x0);
            vd[lane + 64] = f2bf_trunc(x1);
        }
    }
}

// ---- causal attention ------------------------------------------------------------------------
// A workgroup of eight waves takes 16 queries of the HPK heads of one kv head; wave w takes the
// 32-key blocks w, w + 8, ..., each with its own running softmax, and the waves' sums are merged
// through LDS at the end: no barrier in the key loop, and a prompt of a few hundred positions
// gives every CU a workgroup (16 queries of 512 positions: 256 workgroups, the longest of two
// blocks a wave).  Both products are f32 products on the bf16 matrix cores (qt_planes.h); K and V
// are read from the f32 rows and split in registers, once for the HPK heads.
//   scores: A = 16 keys, B = 16 queries: lane l ends with query l % 16 and keys 4 (l / 16) + r of
//           each of the block's two 16-key tiles: the eight k of its group in the A operand of
//           P.V, when k-index 8 g + e stands for key 16 (e / 4) + 4 g + e % 4.
//   P.V:    column n of dim tile d is dim 8 n + d, so that a lane reads 8 neighbouring dims of
//           its 8 keys (two 16-byte loads a key) and holds one column of all eight dim tiles;
//           it ends with queries 4 (l / 16) + r and those 8 dims.
// Bound by the latency of a wave's few blocks up to some 500 positions, then by the splitting of K
// and V (VALU) next to the products.  16 heads, against 64 queries a workgroup over 64-key blocks in LDS on
// the f32 matrix cores (16 to 64 queries on the VALU below 256 positions): 45 positions 8.6 -> 7.4 us,
// 128 15.8 -> 8.8, 512 63 -> 26.7, 1024 122 -> 81, 4096 1622 -> 637; error against 64 bits at 1000 positions
// 8.6e-7 -> 2.5e-7.
#define QT_PF_AW 8
#define QT_PF_AT (64 * QT_PF_AW)

// One query of one head, one key after the other in f32: where an operand has no planes
// (infinite or NaN).  One wave; sp: 64 floats of its own.
__device__ __forceinline__ void pf_att_serial(const float *q, const float *K, const float *V, int ld, int n, float scale,
                                              float *out, float *sp, int lane) {
    float m = -INFINITY, l = 0.f, o0 = 0.f, o1 = 0.f;
    for (int j0 = 0; j0 < n; j0 += 64) {
        float s = -INFINITY;
        if (j0 + lane < n) {
            s = 0.f;
            for (int d = 0; d < 128; d++) s = fmaf(q[d], K[(size_t)(j0 + lane) * ld + d], s);
            s *= scale;
        }
        const float mn = fmaxf(m, group_max<64>(s)), mr = mn == -INFINITY ? 0.f : mn, c = expf(m - mr);
        const float p = j0 + lane < n ? expf(s - mr) : 0.f;
        __builtin_amdgcn_wave_barrier();
        sp[lane] = p;
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_wave_barrier();
        l = l * c + group_sum<64>(p);
        o0 *= c; o1 *= c;
        for (int j = 0; j < min(64, n - j0); j++) {
            o0 = fmaf(sp[j], V[(size_t)(j0 + j) * ld + lane], o0);
            o1 = fmaf(sp[j], V[(size_t)(j0 + j) * ld + 64 + lane], o1);
        }
        m = mn;
    }
    out[lane] = o0 / l;
    out[64 + lane] = o1 / l;
}

// P != NULL: the output goes out as the three planes of the O projection's input: RT == 0:
// P[p][s][nh*128], plane stride Sp*nh*128 (the same pieces k_pf_pieces makes of the f32 output), and
// the workgroup of the last query tile zeroes rows S <= s < Sp of its heads; RT > 0: in operand
// order over RT row tiles (qt_frag_at).
template <int HPK>
__global__ __launch_bounds__(QT_PF_AT) __attribute__((amdgpu_waves_per_eu(2))) void k_pf_att(
    const float *QKV, int ld, int S, int nh, int nkv, float scale, float *A, int lda, uint16_t *P, int Sp, int RT) {
    constexpr int QB = HPK * 3 * 16 * 256;             // the queries' planes: [head][plane][16][128] bf16
    constexpr int OB = HPK * 16 * 128 * 4;             // one wave's sums
    static_assert(QB <= OB * QT_PF_AW, "the queries' planes and the sums share the LDS");
    __shared__ __align__(16) uint8_t sm[OB * QT_PF_AW];
    __shared__ float sst[2][QT_PF_AW][HPK][16];        // the waves' running maximum and sum
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, g = lane >> 4;
    const int h0 = blockIdx.y * HPK, kvh = h0 / (nh / nkv);
    const int qt = gridDim.x - 1 - blockIdx.x, q0 = 16 * qt;         // the longest first
    const int qd = nh * 128, kvd = nkv * 128;
    const float *Kb = QKV + qd + kvh * 128, *Vb = Kb + kvd;
    // each 32-k product is summed by itself: one rounding at the running sum's size, not six
    const qt_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    float chk = 0.f;
    for (int u = tid; u < HPK * 16 * 16; u += QT_PF_AT) {
        const int h = u >> 8, row = (u >> 4) & 15, c = u & 15, q = q0 + row;
        float v[8];
        const float *src = QKV + (size_t)min(q, S - 1) * ld + (h0 + h) * 128 + 8 * c;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const float4 f = *reinterpret_cast<const float4 *>(src + 4 * e);
            v[4 * e] = f.x; v[4 * e + 1] = f.y; v[4 * e + 2] = f.z; v[4 * e + 3] = f.w;
        }
        qt_u32x4 pl[3];
        qt_planes8(v, pl, chk);
#pragma unroll
        for (int p = 0; p < 3; p++)
            *reinterpret_cast<qt_u32x4 *>(sm + (h * 3 + p) * 4096 + row * 256 + 16 * (c ^ row)) = pl[p];
    }
    __syncthreads();
    float m[HPK], l[HPK];
    qt_f32x4 o[HPK][8];
#pragma unroll
    for (int h = 0; h < HPK; h++) {
        m[h] = -INFINITY; l[h] = 0.f;
#pragma unroll
        for (int d = 0; d < 8; d++) o[h][d] = zero;
    }
    float4 vr[8][2];
    auto values = [&](int j0) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float *src = Vb + (size_t)min(j0 + 16 * (e >> 2) + 4 * g + (e & 3), S - 1) * ld + 8 * li;
            vr[e][0] = *reinterpret_cast<const float4 *>(src);
            vr[e][1] = *reinterpret_cast<const float4 *>(src + 4);
        }
    };
    const int q = q0 + li, nkb = min(q0 + 15, S - 1) / 32 + 1;
    for (int kb = wave; kb < nkb; kb += QT_PF_AW) {
        const int j0 = 32 * kb;
        if (HPK == 1) values(j0);
        qt_f32x4 sc[HPK][2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const float *src = Kb + (size_t)min(j0 + 16 * t + li, S - 1) * ld + 8 * g;
            float4 kr[4][2];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                kr[s][0] = *reinterpret_cast<const float4 *>(src + 32 * s);
                kr[s][1] = *reinterpret_cast<const float4 *>(src + 32 * s + 4);
            }
#pragma unroll
            for (int h = 0; h < HPK; h++) sc[h][t] = zero;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const float v[8] = {kr[s][0].x, kr[s][0].y, kr[s][0].z, kr[s][0].w, kr[s][1].x, kr[s][1].y, kr[s][1].z, kr[s][1].w};
                qt_u32x4 kp[3], qp[3];
                qt_planes8(v, kp, chk);
#pragma unroll
                for (int h = 0; h < HPK; h++) {
#pragma unroll
                    for (int p = 0; p < 3; p++)
                        qp[p] = qt_lds16(sm + (h * 3 + p) * 4096 + li * 256 + 16 * ((4 * s + g) ^ li));
                    sc[h][t] += qt_mma6(kp, qp, zero);
                }
            }
        }
        if (HPK == 2) {                                 // two heads' sums leave no room for them earlier
            __builtin_amdgcn_sched_barrier(0);
            values(j0);
            __builtin_amdgcn_sched_barrier(0);
        }
        qt_u32x4 pp[HPK][3];
#pragma unroll
        for (int h = 0; h < HPK; h++) {
            float bm = -INFINITY;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float sv = j0 + 16 * t + 4 * g + r <= q ? sc[h][t][r] * scale : -INFINITY;
                    sc[h][t][r] = sv;
                    bm = fmaxf(bm, sv);
                }
            bm = fmaxf(bm, __shfl_xor(bm, 16));
            bm = fmaxf(bm, __shfl_xor(bm, 32));
            const float mn = fmaxf(m[h], bm), mr = mn == -INFINITY ? 0.f : mn, alpha = expf(m[h] - mr);
            float p8[8], rs = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                p8[e] = expf(sc[h][e >> 2][e & 3] - mr);
                rs += p8[e];
            }
            rs += __shfl_xor(rs, 16);
            rs += __shfl_xor(rs, 32);
            l[h] = l[h] * alpha + rs;
            m[h] = mn;
            qt_planes8(p8, pp[h], chk);
            float ar[4];
#pragma unroll
            for (int r = 0; r < 4; r++) ar[r] = __shfl(alpha, 4 * g + r);
#pragma unroll
            for (int d = 0; d < 8; d++)
#pragma unroll
                for (int r = 0; r < 4; r++) o[h][d][r] *= ar[r];
        }
#pragma unroll
        for (int d = 0; d < 8; d++) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float4 f = vr[e][d >> 2];
                v[e] = (d & 3) == 0 ? f.x : (d & 3) == 1 ? f.y : (d & 3) == 2 ? f.z : f.w;
            }
            qt_u32x4 vp[3];
            qt_planes8(v, vp, chk);
#pragma unroll
            for (int h = 0; h < HPK; h++) o[h][d] += qt_mma6(pp[h], vp, zero);
        }
    }
    // merge: the waves' maxima and sums, each wave's output scaled to the common maximum
#pragma unroll
    for (int h = 0; h < HPK; h++)
        if (g == 0) { sst[0][wave][h][li] = m[h]; sst[1][wave][h][li] = l[h]; }
    const bool serial = __syncthreads_or(chk != chk);
    const int nw = min(nkb, QT_PF_AW);
    if (!serial) {
        float *os = reinterpret_cast<float *>(sm + wave * OB);
#pragma unroll
        for (int h = 0; h < HPK; h++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 4 * g + r;
                float M = -INFINITY;
                for (int w = 0; w < nw; w++) M = fmaxf(M, sst[0][w][h][row]);
                const float f = expf(sst[0][wave][h][row] - M);
                if (wave < nw) {
                    float *d = os + (h * 16 + row) * 128 + 8 * li;
                    *reinterpret_cast<float4 *>(d) = make_float4(o[h][0][r] * f, o[h][1][r] * f, o[h][2][r] * f, o[h][3][r] * f);
                    *reinterpret_cast<float4 *>(d + 4) = make_float4(o[h][4][r] * f, o[h][5][r] * f, o[h][6][r] * f, o[h][7][r] * f);
                }
            }
        __syncthreads();
    }
    const size_t plane = RT ? 512 : (size_t)Sp * qd;
    const auto at = [&](int row, int col) { return RT ? qt_frag_at(RT, row, col) : (size_t)row * qd + col; };
    for (int u = tid; u < HPK * 16 * 32; u += QT_PF_AT) {
        const int h = u >> 9, row = (u >> 5) & 15, c = 4 * (u & 31);
        if (serial || q0 + row >= S) continue;
        float M = -INFINITY, L = 0.f;
        for (int w = 0; w < nw; w++) M = fmaxf(M, sst[0][w][h][row]);
        qt_f32x4 v = {0.f, 0.f, 0.f, 0.f};
        for (int w = 0; w < nw; w++) {
            L += sst[1][w][h][row] * expf(sst[0][w][h][row] - M);
            v += *reinterpret_cast<const qt_f32x4 *>(sm + w * OB + ((h * 16 + row) * 128 + c) * 4);
        }
        const float inv = 1.0f / L;
        const int col = (h0 + h) * 128 + c;
        if (P) {
            uint16_t pc[3][4];
#pragma unroll
            for (int e = 0; e < 4; e++) qt_put_pieces(&pc[0][e], 4, __fmul_rn(v[e], inv));
#pragma unroll
            for (int p = 0; p < 3; p++)
                *reinterpret_cast<uint2 *>(P + p * plane + at(q0 + row, col)) =
                    make_uint2((uint32_t)pc[p][0] | ((uint32_t)pc[p][1] << 16), (uint32_t)pc[p][2] | ((uint32_t)pc[p][3] << 16));
        } else {
            *reinterpret_cast<qt_f32x4 *>(A + (size_t)(q0 + row) * lda + col) = v * inv;
        }
    }
    if (serial) {
        float *out = reinterpret_cast<float *>(sm) + wave * 256;
        for (int u = wave; u < HPK * 16; u += QT_PF_AW) {
            const int h = u >> 4, qq = q0 + (u & 15);
            if (qq >= S) continue;
            pf_att_serial(QKV + (size_t)qq * ld + (h0 + h) * 128, Kb, Vb, ld, qq + 1, scale, out, out + 128, lane);
            __builtin_amdgcn_s_waitcnt(0);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int col = (h0 + h) * 128 + 64 * e + lane;
                if (P) qt_put_pieces(P + at(qq, col), (int)plane, out[64 * e + lane]);
                else A[(size_t)qq * lda + col] = out[64 * e + lane];
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (P && !RT && qt == (int)gridDim.x - 1)
        for (int i = tid; i < (Sp - S) * 32 * HPK; i += QT_PF_AT) {
            uint16_t *dst = P + (size_t)(S + i / (32 * HPK)) * qd + h0 * 128 + 4 * (i % (32 * HPK));
#pragma unroll
            for (int p = 0; p < 3; p++) *reinterpret_cast<uint2 *>(dst + p * plane) = make_uint2(0u, 0u);
        }
}

// ---- launchers -------------------------------------------------------------------------
// Positions are padded to a multiple of QT_PF_SPAD for the planes (the GEMM's position
// tile); weight rows must be a multiple of 64 and K a multiple of 64.
#define QT_PF_SPAD 64

extern "C" int qt_pf_spad(int S) { return (S + QT_PF_SPAD - 1) / QT_PF_SPAD * QT_PF_SPAD; }

extern "C" hipError_t qt_launch_pf_pieces(const float *X, int ldx, int S, int K, const float *gain, float eps,
                                          uint16_t *P, hipStream_t st) {
    if (S <= 0 || K <= 0 || K % 8 || ldx % 4) return hipErrorInvalidValue;
    const int Sp = qt_pf_spad(S);
    hipLaunchKernelGGL(k_pf_pieces, dim3(Sp), dim3(QT_PF_WG), 0, st, X, ldx, S, Sp, K, gain, eps, P);
    return hipGetLastError();
}

// part: workspace of 4 * S * N floats for split K (nullable: no split).  The residual
// projections (few weight rows) split K so the grid fills the CUs; the partial ranges
// are added in order (deterministic).
// Tile and K split of a projection: a weight tile of 256, 192, 128 or 64 rows (a taller
// tile reuses each LDS read of the planes over more rows and runs more MFMAs per barrier)
// with its K split where needed into 2^k equal ranges of at least four 64-k chunks whose
// partials fit in part_cap floats (added in order by k_pf_reduce), so that the grid
// reaches 256 workgroups; among such plans the one with the least work on the busiest CU,
// else the largest grid.  Measured on the 1.7B prefill (128 / 512 positions): with the
// three-stage 256-row tile 4.16 / 9.46 ms against 4.53 / 10.72 preferring an unsplit
// shorter tile, 4.50 / 10.22 splitting to 512 workgroups, 4.27 / 9.46 with two-chunk
// ranges; with the two-stage tiles at two waves per SIMD 3.94 / 8.73 (splitting to 512
// workgroups 4.50 / 9.56); choosing by the busiest CU's work (192-row tiles for gate|up:
// 512 workgroups, two on every CU, where 256-row tiles gave 384) 3.64 / 7.79.
static void qt_pf_plan(int S, int Sp, int N, int K, long long part_cap, int &nr, int &sk) {
    // per-CU load of a plan: workgroups per CU (ceil over 256) x rows per workgroup / K ranges;
    // among the plans that reach 256 workgroups the lightest, the taller tile on a tie
    const long long sy = Sp / 64;
    long long best = -1;
    double bcost = 1e30;
    bool reach = false;
    nr = 1; sk = 1;
    const int rs[4] = {4, 3, 2, 1};
    for (int ri = 0; ri < 4; ri++) {
        const int r = rs[ri];
        if (N % (64 * r)) continue;
        const long long g = (long long)(N / (64 * r)) * sy;
        int k = 1;
        while (g * k < 256 && (K / 64) % (2 * k) == 0 && K / 64 / (2 * k) >= 4 && 2LL * k * S * N <= part_cap) k *= 2;
        if (g * k >= 256) {
            const double cost = (double)((g * k + 255) / 256) * r / k;
            if (!reach || cost < bcost) { nr = r; sk = k; bcost = cost; }
            reach = true;
        } else if (!reach && g * k > best) {
            best = g * k; nr = r; sk = k;
        }
    }
}

// Pout != NULL (SwiGLU only): h goes out as the three planes of the next projection's
// input (k_pf_reduce_swiglu_planes) instead of f32 rows; needs part with S*N <= part_cap.
// Pout with RESID: Y += the product as usual, then RMSNorm(Y row) * gain goes out as the
// next projection's input planes (k_pf_reduce_resid_planes); needs part, S*N <= part_cap.
// qp != NULL (STORE into the q|k|v rows Y): k_pf_reduce_qkv_post finishes the rows.
static hipError_t pf_gemm(int epi, const uint16_t *W, const uint16_t *P, int S, int N, int K, float *Y, int ldy,
                          float *part, long long part_cap, uint16_t *Pout, const float *gain, float eps,
                          hipStream_t st, const PfQkvPost *qp = nullptr) {
    constexpr int NST = 4;
    if (qp && (epi != QT_PF_STORE || Pout || !part || (long long)S * N > part_cap || N != (qp->nh + 2 * qp->nkv) * 128 ||
               (size_t)N * 4 > 64 * 1024 || S > qp->kv_max))
        return hipErrorInvalidValue;
    if (S <= 0 || N <= 0 || K <= 0 || N % 64 || K % 64 || epi < 0 || epi > 2) return hipErrorInvalidValue;
    if (Pout ? ((epi != QT_PF_SWIGLU && !(epi == QT_PF_RESID && gain && Y && ldy >= N && ldy % 4 == 0 &&
                                          (size_t)N * 4 <= 64 * 1024)) ||
                !part || (long long)S * N > part_cap)
             : (epi != QT_PF_SWIGLU ? (ldy < N || ldy % 4) : (ldy < N / 2 || ldy % 2)))
        return hipErrorInvalidValue;
    const int Sp = qt_pf_spad(S);
    int nr, sk;
    qt_pf_plan(S, Sp, N, K, part ? part_cap : 0, nr, sk);
    const int gx = N / (64 * nr);
    const dim3 grid(gx, Sp / 64, sk);
#define QT_PF_GEMM(E, OUT, LD)                                                                                         \
    if (nr == 4) hipLaunchKernelGGL((k_pf_gemm2<E, 4, 2>), grid, dim3(QT_PF_WG), 0, st, W, P, S, Sp, K, OUT, LD);    \
    else if (nr == 3) hipLaunchKernelGGL((k_pf_gemm2<E, 3, 2>), grid, dim3(QT_PF_WG), 0, st, W, P, S, Sp, K, OUT, LD); \
    else if (nr == 2) hipLaunchKernelGGL((k_pf_gemm2<E, 2, NST>), grid, dim3(QT_PF_WG), 0, st, W, P, S, Sp, K, OUT, LD); \
    else hipLaunchKernelGGL((k_pf_gemm2<E, 1, NST>), grid, dim3(QT_PF_WG), 0, st, W, P, S, Sp, K, OUT, LD);
    if (qp) {
        QT_PF_GEMM(QT_PF_PART, part, N)
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_pf_reduce_qkv_post, dim3(S), dim3(PF_QKV_T), (size_t)N * sizeof(float), st, part, sk, S, N, Y,
                           ldy, *qp);
    } else if (Pout) {
        QT_PF_GEMM(QT_PF_PART, part, N)
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        if (epi == QT_PF_SWIGLU)
            hipLaunchKernelGGL(k_pf_reduce_swiglu_planes, dim3((Sp * N / 4 + QT_PF_WG - 1) / QT_PF_WG), dim3(QT_PF_WG), 0,
                               st, part, sk, S, Sp, N, Pout);
        else
            hipLaunchKernelGGL(k_pf_reduce_resid_planes, dim3(Sp), dim3(PF_ROW_T), (size_t)N * sizeof(float), st, part, sk,
                               S, Sp, N, Y, ldy, gain, eps, Pout);
    } else if (sk > 1) {
        QT_PF_GEMM(QT_PF_PART, part, N)
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const dim3 rg((S * N / 4 + QT_PF_WG - 1) / QT_PF_WG);
        if (epi == QT_PF_STORE) hipLaunchKernelGGL(k_pf_reduce<QT_PF_STORE>, rg, dim3(QT_PF_WG), 0, st, part, sk, S, N, Y, ldy);
        else if (epi == QT_PF_RESID) hipLaunchKernelGGL(k_pf_reduce<QT_PF_RESID>, rg, dim3(QT_PF_WG), 0, st, part, sk, S, N, Y, ldy);
        else hipLaunchKernelGGL(k_pf_reduce<QT_PF_SWIGLU>, rg, dim3(QT_PF_WG), 0, st, part, sk, S, N, Y, ldy);
    } else if (epi == QT_PF_STORE) {
        QT_PF_GEMM(QT_PF_STORE, Y, ldy)
    } else if (epi == QT_PF_RESID) {
        QT_PF_GEMM(QT_PF_RESID, Y, ldy)
    } else {
        QT_PF_GEMM(QT_PF_SWIGLU, Y, ldy)
    }
#undef QT_PF_GEMM
    return hipGetLastError();
}

extern "C" hipError_t qt_launch_pf_gemm(int epi, const uint16_t *W, const uint16_t *P, int S, int N, int K, float *Y,
                                        int ldy, float *part, long long part_cap, hipStream_t st) {
    return pf_gemm(epi, W, P, S, N, K, Y, ldy, part, part_cap, NULL, NULL, 0.f, st);
}
extern "C" hipError_t qt_launch_pf_gemm_swiglu_planes(const uint16_t *W, const uint16_t *P, int S, int N, int K,
                                                      uint16_t *Pout, float *part, long long part_cap, hipStream_t st) {
    return pf_gemm(QT_PF_SWIGLU, W, P, S, N, K, NULL, 0, part, part_cap, Pout, NULL, 0.f, st);
}
extern "C" hipError_t qt_launch_pf_gemm_qkv_post(const uint16_t *W, const uint16_t *P, int S, int N, int K, float *QKV,
                                                  int ld, int nh, int nkv, const float *qn, const float *kn,
                                                  const float *rc, const float *rs, float eps, uint16_t *kc, uint16_t *vc,
                                                  long long kv_max, float *part, long long part_cap, hipStream_t st) {
    if (nh <= 0 || nkv <= 0 || nh % nkv) return hipErrorInvalidValue;
    const PfQkvPost qp = {nh, nkv, qn, kn, rc, rs, eps, kc, vc, kv_max};
    return pf_gemm(QT_PF_STORE, W, P, S, N, K, QKV, ld, part, part_cap, NULL, NULL, 0.f, st, &qp);
}
extern "C" hipError_t qt_launch_pf_gemm_resid_planes(const uint16_t *W, const uint16_t *P, int S, int N, int K, float *Y,
                                                     int ldy, const float *gain, float eps, uint16_t *Pout, float *part,
                                                     long long part_cap, hipStream_t st) {
    return pf_gemm(QT_PF_RESID, W, P, S, N, K, Y, ldy, part, part_cap, Pout, gain, eps, st);
}

extern "C" hipError_t qt_launch_pf_qkv_post(float *QKV, int ld, int S, int nh, int nkv, const float *qn,
                                            const float *kn, const float *rc, const float *rs, float eps, uint16_t *kc,
                                            uint16_t *vc, long long kv_max, hipStream_t st) {
    if (S <= 0 || nh <= 0 || nkv <= 0 || nh % nkv || S > kv_max) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_pf_qkv_post, dim3(S), dim3(QT_PF_WG), 0, st, QKV, ld, nh, nkv, qn, kn, rc, rs, eps, kc, vc,
                       kv_max);
    return hipGetLastError();
}

static hipError_t pf_attn(const float *QKV, int ld, int S, int nh, int nkv, float scale, float *A, int lda,
                          uint16_t *P, int frag, hipStream_t st) {
    if (S <= 0 || nh <= 0 || nkv <= 0 || nh % nkv) return hipErrorInvalidValue;
    const int Sp = qt_pf_spad(S), rt = frag ? (S + 15) / 16 : 0;
    // One head a workgroup while every such workgroup has a CU of its own, then two heads of a kv
    // head, which split its keys and values once (16 heads: 8.8 us against 11.9 at 128 positions, 13.4
    // against 17.3 at 256, then 28.2 against 21.1 at 384 and 40.1 against 26.7 at 512)
    if ((nh / nkv) % 2 == 0 && (long long)((S + 15) / 16) * nh > 256)
        hipLaunchKernelGGL(k_pf_att<2>, dim3((S + 15) / 16, nh / 2), dim3(QT_PF_AT), 0, st, QKV, ld, S, nh, nkv, scale, A, lda, P, Sp, rt);
    else
        hipLaunchKernelGGL(k_pf_att<1>, dim3((S + 15) / 16, nh), dim3(QT_PF_AT), 0, st, QKV, ld, S, nh, nkv, scale, A, lda, P, Sp, rt);
    return hipGetLastError();
}

extern "C" hipError_t qt_launch_pf_attn(const float *QKV, int ld, int S, int nh, int nkv, float scale, float *A,
                                        int lda, hipStream_t st) {
    return pf_attn(QKV, ld, S, nh, nkv, scale, A, lda, NULL, 0, st);
}
// the output as the O projection's input planes: P[p][s][nh*128] (rows padded to qt_pf_spad(S)), or,
// with frag, in operand order (qt_frag_at)
extern "C" hipError_t qt_launch_pf_attn_planes(const float *QKV, int ld, int S, int nh, int nkv, float scale, uint16_t *P,
                                               int frag, hipStream_t st) {
    return pf_attn(QKV, ld, S, nh, nkv, scale, NULL, 0, P, frag, st);
}
