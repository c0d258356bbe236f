// qt_sd.hip — the speech decoder (codes -> 24 kHz audio) on gfx950.
//
// The reference's one-shot decode (qwen_speech_decoder_decode, qwen_tts_speech_decoder.c:
// 579-1290) is a VQ lookup, an 8-layer windowed-attention transformer over the frames and
// a convolutional upsampler (ConvNeXt x2, then four blocks of transposed conv + dilated
// residual units) to 1920 samples per frame.  All of it is f32.  Here every activation is
// kept time-major ([T][C], channels contiguous), and every projection, convolution and
// transposed convolution is one implicit GEMM:
//
//   Y[t*os + z][n] = epi( sum over channels k, taps p of X[t + off_p][k] * W[z][p][k][n] )
//
// (rows of X outside [xlo, Tx) read as zero: the causal left padding; the streaming decode
// keeps the previous chunk's last rows at negative indices, xlo < 0).  A causal conv of
// kernel K and dilation d has taps off_p = (p - K + 1) d; a transposed conv of stride s
// and kernel 2s is s phases z (output rows t*s + z), each with taps at offsets 0 and -1
// (kernel columns z and z + s); a linear layer is one tap.  The epilogue adds a bias,
// applies GELU, scales per column (layer scale, ConvNeXt gamma), adds a residual and
// applies the snake activation that the next layer needs on its input (so no separate
// pass over the activation: the upsampler's snakes all live in the producing GEMM).
//
// The products run on the bf16 matrix cores, sixteen times as fast as the f32 ones: each f32
// operand is the exact sum of three bf16 planes, a product of two planes is exact in f32,
// and the six largest of the nine plane products of an f32 product are accumulated in f32
// (the rest are under 2^-25 of it, below its own rounding).  The weights' planes are made
// once, when the decoder is loaded; an input's on its way into LDS.
#include "qt_planes.h"

#define SD_WG 256
#define SD_MAXTAP 8
#define SD_HALO 54               // staged rows before a tile's own: a 7-tap conv of dilation 9

enum { SD_EPI_BIAS = 1, SD_EPI_GELU = 2, SD_EPI_CSCALE = 4, SD_EPI_RESID = 8, SD_EPI_SNAKE = 16, SD_EPI_SNAKE2 = 32 };

// ---- the GEMM's weights: three bf16 planes in the matrix core's order ----------------------
// v_mfma_f32_16x16x32_bf16 takes A = 16 output channels x 32 k and B = 32 k x 16 output rows;
// lane l supplies 8 consecutive k (group l / 16) of channel (row) l % 16 and receives
// D[channel 4 (l / 16) + r][row l % 16], r < 4.  A weight tile of 16 channels x 32 k is
// stored as its three planes, 64 lanes x 16 bytes each (3 KiB), in the order that a
// workgroup walks: [K slice][tap][phase][channel tile].  K and the channels of a phase are
// padded with zeros to 32 and 16.
// One tensor of the reference's layout (element [n][k][column] at n * sn + k * sk + column * sc)
// into channels [n0, n0 + nn) and k [k0, k0 + kk) of the packed weights (n0, k0: whole tiles).
// Tap p of phase z is column p (stride 0: a conv or linear layer) or z + p * stride (zero past the
// kernel's columns).  The planes of an infinite or NaN value give NaN sums (sd_redo).
struct SdPackArgs {
    const float *src;
    long long sn, sk, sc;
    int cols, stride, ntap, phases, tiles;         // tiles: channel tiles of a phase
    int n0, nn, k0, kk;
    uint16_t *dst;
};
__global__ __launch_bounds__(SD_WG) void k_sd_pack(SdPackArgs a) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nt = (a.nn + 15) / 16;
    const int t = blockIdx.x * QT_WAVES + wave, z = blockIdx.z;
    const int kc = t / (a.ntap * nt), r = t - kc * a.ntap * nt, p = r / nt, j = r - p * nt;
    if (kc >= (a.kk + 31) / 32) return;
    const int n = 16 * j + (lane & 15), k = 32 * kc + 8 * (lane >> 4), col = a.stride ? z + p * a.stride : p;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++)
        v[i] = (n < a.nn && k + i < a.kk && col < a.cols) ? a.src[n * a.sn + (k + i) * a.sk + col * a.sc] : 0.f;
    // a finite value that rounds past bf16's range: its planes are cut instead of rounded (qt_put_pieces)
    float big[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        big[i] = fabsf(v[i]) > 0x1.fep127f && fabsf(v[i]) < INFINITY ? v[i] : 0.f;
        if (big[i] != 0.f) v[i] = 0.f;
    }
    qt_u32x4 pl[3];
    qt_planes8(v, pl);
#pragma unroll
    for (int i = 0; i < 8; i++)
        if (big[i] != 0.f) {
            uint16_t pc[3];
            qt_put_pieces(pc, 1, big[i]);
#pragma unroll
            for (int q = 0; q < 3; q++) pl[q][i / 2] |= (uint32_t)pc[q] << (16 * (i & 1));
        }
    uint16_t *d = a.dst + ((((size_t)(a.k0 / 32 + kc) * a.ntap + p) * a.phases + z) * a.tiles + a.n0 / 16 + j) * 1536 + 8 * lane;
#pragma unroll
    for (int q = 0; q < 3; q++) *reinterpret_cast<qt_u32x4 *>(d + 512 * q) = pl[q];
}

struct SdGemmArgs {
    const float *X; int ldx, Tx, xlo;     // input rows [xlo, Tx) of a [.][ldx] buffer (xlo <= 0: history rows)
    const uint16_t *W;                    // packed planes
    int K, N, ntap;
    int slices, tiles, phases;            // K slices of 32; channel tiles of a phase
    int off[SD_MAXTAP];
    int omin, span;                       // smallest offset; largest minus smallest
    int tps;                              // taps that share a staged slice (ntap, or 1 where span is too long)
    int T;                                // output rows per phase (t < T)
    float *Y; int ldy, os;                // output row t*os + phase
    const float *bias, *cscale;
    const float *R;                       // residual, same indexing as Y (may alias Y)
    const float *sa, *sib;                // SNAKE: Y = snake(v) with per-column a, 1/b
    float *Y2;                            // SNAKE2: Y = v and Y2 = snake(v) (same indexing)
    int epi;
};

__device__ __forceinline__ float sd_gelu(float x) {
    return 0.5f * x * (1.0f + erff(x * 0.7071067811865476f));
}

// snake (k.c:4472-4600): x + (1/b) sin(a x)^2 with a = e^alpha, 1/b = e^-beta per channel
__device__ __forceinline__ float sd_snake(float x, float a, float ib) {
    const float s = sinf(a * x);
    return fmaf(ib, s * s, x);
}

// Channels n..n+3 of output row t from the f32 operands, by a whole wave: each lane takes units of
// 8 k, in an order of their own that depends on nothing but the layer.  A channel's NaN is final:
// the sum ends once every channel in `want` (bits) has one.
__device__ __forceinline__ qt_f32x4 sd_redo(const SdGemmArgs &a, int t, int tile, int n, unsigned want, int lane) {
    qt_f32x4 s = {0.f, 0.f, 0.f, 0.f};
    const int units = 4 * a.slices * a.ntap;
    for (int u0 = 0; u0 < units; u0 += 64) {
        const int u = u0 + lane, kg = u & 3, kc = (u >> 2) / a.ntap, p = (u >> 2) - kc * a.ntap, k = 32 * kc + 8 * kg;
        if (u < units && k < a.K) {
            const int xr = t + a.off[p];
            float4 x[2] = {make_float4(0.f, 0.f, 0.f, 0.f), make_float4(0.f, 0.f, 0.f, 0.f)};
            if (xr >= a.xlo && xr < a.Tx) {
                const float4 *src = reinterpret_cast<const float4 *>(a.X + (ptrdiff_t)xr * a.ldx + k);
                x[0] = src[0]; x[1] = src[1];
            }
            const float xv[8] = {x[0].x, x[0].y, x[0].z, x[0].w, x[1].x, x[1].y, x[1].z, x[1].w};
            const uint16_t *w = a.W + (((size_t)kc * a.ntap + p) * a.phases * a.tiles + tile) * 1536 + 8 * ((n & 15) + 16 * kg);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                qt_u32x4 wq[3];
#pragma unroll
                for (int q = 0; q < 3; q++) wq[q] = *reinterpret_cast<const qt_u32x4 *>(w + 8 * r + 512 * q);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    float wf[3];
#pragma unroll
                    for (int q = 0; q < 3; q++) wf[q] = e & 1 ? qt_bf_hi(wq[q][e / 2]) : qt_bf_lo(wq[q][e / 2]);
                    // an infinite or NaN weight is its first plane
                    s[r] = fmaf(xv[e], fabsf(wf[0]) < INFINITY ? wf[0] + (wf[1] + wf[2]) : wf[0], s[r]);
                }
            }
        }
        bool open = false;
#pragma unroll
        for (int r = 0; r < 4; r++) open = open || ((want >> r & 1) && !__any(s[r] != s[r]));
        if (!open) break;
    }
#pragma unroll
    for (int r = 0; r < 4; r++) s[r] = group_sum<64>(s[r]);
    return s;
}

// A sum of plane products is finite unless an operand is infinite, NaN or past bf16's range, or the
// sum itself is out of range: then the planes cannot say whether the result is an infinity, a NaN or
// a finite value, and that output is taken again from the f32 operands.  An output is redone for its
// own operands only, so every other one keeps the bits that it has in any call and any tile; and what
// it costs is a matter of the outputs concerned (a wave's latency each, the first product where the row is
// NaN throughout).  Every lane of the wave calls this (v, t, tile, n: its own; live: its output exists).
__device__ __forceinline__ qt_f32x4 sd_finite(const SdGemmArgs &a, qt_f32x4 v, int t, int tile, int n, bool live, int lane) {
    unsigned bad = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) bad |= fabsf(v[r]) < INFINITY ? 0u : 1u << r;
    for (unsigned long long m = __ballot(live && bad); m; m &= m - 1) {
        const int l = __builtin_ctzll(m);
        const unsigned want = __builtin_amdgcn_readlane(bad, l);
        const qt_f32x4 s = sd_redo(a, __builtin_amdgcn_readlane(t, l), __builtin_amdgcn_readlane(tile, l),
                                   __builtin_amdgcn_readlane(n, l), want, lane);
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (lane == l && (want >> r & 1)) v[r] = s[r];
    }
    return v;
}

// The four channels n..n+3 (n: channel of the phase) of output row t: bias, GELU, column
// scale, residual, snake.
__device__ __forceinline__ void sd_epilogue(const SdGemmArgs &a, int t, int z, int n, qt_f32x4 v) {
    if (t >= a.T || n >= a.N) return;
    const size_t o = (size_t)(t * a.os + z) * a.ldy + n;
    const auto ld = [](const float *p) { return *reinterpret_cast<const qt_f32x4 *>(p); };
    if (a.epi & SD_EPI_BIAS) v += ld(a.bias + n);
    if (a.epi & SD_EPI_GELU)
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = sd_gelu(v[r]);
    if (a.epi & SD_EPI_CSCALE) v *= ld(a.cscale + n);
    if (a.epi & SD_EPI_RESID) v = ld(a.R + o) + v;
    if (a.epi & (SD_EPI_SNAKE | SD_EPI_SNAKE2)) {
        const qt_f32x4 pa = ld(a.sa + n), pb = ld(a.sib + n);
        qt_f32x4 s;
#pragma unroll
        for (int r = 0; r < 4; r++) s[r] = sd_snake(v[r], pa[r], pb[r]);
        if (a.epi & SD_EPI_SNAKE2) *reinterpret_cast<qt_f32x4 *>(a.Y2 + o) = s;
        else v = s;
    }
    *reinterpret_cast<qt_f32x4 *>(a.Y + o) = v;
}

// Where a layer has at least SD_GROUP_SLICES slices of 32 k (512), its slices are SD_GROUPS
// equal runs whose sums are added in order.  That is a property of the layer alone, so a
// small call can give the runs to different waves and still return the bits of a large one.
#define SD_GROUPS 8
#define SD_GROUP_SLICES 16

// swizzle of the 16-byte unit kg of an LDS row of 32 k: 8 (and 16) consecutive rows read one
// unit each from different banks
__device__ __forceinline__ int sd_unit(int row, int kg) { return 16 * (kg ^ (((row >> 2) & 3) ^ (row & 2))); }

// ---- tiles for many rows ---------------------------------------------------------------------
// A workgroup of WN x WT waves computes 16 NT WN channels x 16 MT WT rows.  A slice of 32 k of
// the rows that all its taps read (the tile's rows and the taps' span before them) is
// loaded once, split into planes on the way into LDS, and every tap runs from there, so a
// 7-tap conv stages each input once; the weights' planes come straight from L2 in operand
// order, one (slice, tap) ahead.  Two LDS buffers, one barrier per slice.
// Bound by the matrix cores where there are rows enough: 7 taps of 384 -> 384 channels over 20 000
// rows take 175 us = 236 TFLOP/s of f32 products, 1.42 PFLOP/s of plane products (the f32 matrix
// cores: 450 us, 92 TFLOP/s; a 4096 x 4096 library product in bf16 reaches 1.13 PFLOP/s here); the
// 96-channel convs are held by their f32 traffic as well (240 000 rows: 167 us, 185 TFLOP/s).
// Weight planes two or three items ahead, in a loop unrolled over a ring: no faster.
template <int WN, int NT, int WT, int MT, bool GRP>
__global__ __launch_bounds__(SD_WG) __attribute__((amdgpu_waves_per_eu(2))) void k_sd_tile(SdGemmArgs a) {
    static_assert(WN * WT == QT_WAVES, "four waves");
    constexpr int TT = 16 * MT * WT, RM = TT + SD_HALO, PS = RM * 64, BUF = 3 * PS, NU = (RM * 4 + SD_WG - 1) / SD_WG;
    __shared__ __align__(16) uint8_t xs[2 * BUF];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, kg = lane >> 4;
    const int t0 = blockIdx.x * TT, all = a.phases * a.tiles;
    const int j0 = (blockIdx.y * WN + wave % WN) * NT, tw = 16 * MT * (wave / WN);
    const int rows = TT + (a.tps > 1 ? a.span : 0), ns = a.slices * (a.ntap / a.tps);
    float st[NU][8];
    unsigned ok = 0;
    auto fetch = [&](int s) {
        const int per = a.ntap / a.tps, kc = s / per, o = a.tps > 1 ? a.omin : a.off[s - kc * per];
#pragma unroll
        for (int i = 0; i < NU; i++) {
            const int u = tid + i * SD_WG, row = u >> 2, k = 32 * kc + 8 * (u & 3), xr = t0 + row + o;
            const bool in = row < rows && xr >= a.xlo && xr < a.Tx && k < a.K;
            ok = in ? ok | (1u << i) : ok & ~(1u << i);
            // in bounds either way; the value is dropped when !in
            const float *src = a.X + (ptrdiff_t)min(max(xr, a.xlo), a.Tx - 1) * a.ldx + min(k, a.K - 8);
            const float4 p = *reinterpret_cast<const float4 *>(src), q = *reinterpret_cast<const float4 *>(src + 4);
            st[i][0] = p.x; st[i][1] = p.y; st[i][2] = p.z; st[i][3] = p.w;
            st[i][4] = q.x; st[i][5] = q.y; st[i][6] = q.z; st[i][7] = q.w;
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NU; i++) {
            const int u = tid + i * SD_WG, row = u >> 2;
            if ((i + 1) * SD_WG > RM * 4 && row >= RM) continue;
            const unsigned m = 0u - ((ok >> i) & 1u);
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = __uint_as_float(__float_as_uint(st[i][e]) & m);
            qt_u32x4 pl[3];
            qt_planes8(v, pl);
            uint8_t *d = xs + buf * BUF + row * 64 + sd_unit(row, u & 3);
#pragma unroll
            for (int p = 0; p < 3; p++) *reinterpret_cast<qt_u32x4 *>(d + p * PS) = pl[p];
        }
    };
    const uint16_t *wp[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) wp[j] = a.W + (size_t)min(j0 + j, all - 1) * 1536 + 8 * lane;
    const size_t step = (size_t)all * 1536;
    const int items = a.slices * a.ntap;
    qt_u32x4 w[NT][3], wn[NT][3];
    auto weights = [&](int it, qt_u32x4 (&d)[NT][3]) {
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int p = 0; p < 3; p++) d[j][p] = *reinterpret_cast<const qt_u32x4 *>(wp[j] + it * step + 512 * p);
    };
    qt_f32x4 acc[NT][MT], tot[GRP ? NT : 1][GRP ? MT : 1];
    const qt_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = zero;
    fetch(0);
    weights(0, w);
    put(0);
    __syncthreads();
    int g = 0;
    for (int s = 0, it = 0; s < ns; s++) {
        if (s + 1 < ns) fetch(s + 1);
        const uint8_t *b = xs + (s & 1) * BUF;
        for (int p = 0; p < a.tps; p++, it++) {
            weights(min(it + 1, items - 1), wn);
            const int row = tw + li + (a.tps > 1 ? a.off[p] - a.omin : 0);
            const uint8_t *x0 = b + row * 64 + sd_unit(row, kg);
#pragma unroll
            for (int i = 0; i < MT; i++) {
                qt_u32x4 x[3];
#pragma unroll
                for (int q = 0; q < 3; q++) x[q] = qt_lds16(x0 + i * 1024 + q * PS);
#pragma unroll
                for (int j = 0; j < NT; j++) acc[j][i] = qt_mma6(w[j], x, acc[j][i]);
            }
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int q = 0; q < 3; q++) w[j][q] = wn[j][q];
        }
        if constexpr (GRP) {
            if (it == (a.slices * (g + 1) / SD_GROUPS) * a.ntap) {   // a run ends here
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        tot[j][i] = g ? tot[j][i] + acc[j][i] : acc[j][i];
                        acc[j][i] = zero;
                    }
                g++;
            }
        }
        if (s + 1 < ns) put((s + 1) & 1);
        __syncthreads();
    }
    // the sums through LDS (free: the last slice's barrier is behind), so that a row's channels go out (and its residual comes in) together
    constexpr int TN = 16 * WN * NT, LD = TN + 4;
    static_assert(TT * LD * 4 <= 2 * BUF, "the tile's sums fit in the staging buffers");
    static_assert(TT * TN / 4 % SD_WG == 0, "no thread leaves the last loop early");
    float *ys = reinterpret_cast<float *>(xs);
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++)
            *reinterpret_cast<qt_f32x4 *>(ys + (tw + 16 * i + li) * LD + 16 * (wave % WN * NT + j) + 4 * kg) =
                GRP ? tot[GRP ? j : 0][GRP ? i : 0] : acc[j][i];
    __syncthreads();
    for (int e = tid; e < TT * TN / 4; e += SD_WG) {
        const int row = e / (TN / 4), c = 4 * (e % (TN / 4)), t = t0 + row, tile = blockIdx.y * (WN * NT) + c / 16;
        const int z = tile / a.tiles, n = 16 * (tile - z * a.tiles) + c % 16;
        const bool live = tile < all && t < a.T && n < a.N;
        const qt_f32x4 v = sd_finite(a, *reinterpret_cast<qt_f32x4 *>(ys + row * LD + c), t, tile, n, live, lane);
        if (live) sd_epilogue(a, t, z, n, v);
    }
}

// ---- few rows ---------------------------------------------------------------------------------
// A workgroup of eight waves computes 16 NT channels x 16 MT rows; wave g takes the layer's g-th
// run of slices, with its operands straight from memory (no staging, no barrier until the
// runs' sums meet in LDS), D (slice, tap) pairs in flight.  A call of a few frames leaves the
// long-K layers with a few dozen such tiles: the time is the latency of one run (10 rows: 512 -> 3072
// 6.0 us, 1024 -> 512 5.8 us, where one wave per tile walked all of K in f32 in 16 to 21 us).  With more
// rows it is held by L2: every tile reads its own operands, 550 TFLOP/s of plane products.
template <int NT, int MT, int D>
__global__ __launch_bounds__(64 * SD_GROUPS) void k_sd_split(SdGemmArgs a) {
    __shared__ __align__(16) qt_f32x4 part[SD_GROUPS][NT * MT][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, kg = lane >> 4;
    const int t0 = blockIdx.x * 16 * MT, all = a.phases * a.tiles, j0 = blockIdx.y * NT;
    const int i0 = (a.slices * wave / SD_GROUPS) * a.ntap, i1 = (a.slices * (wave + 1) / SD_GROUPS) * a.ntap;
    const size_t step = (size_t)all * 1536;
    const uint16_t *wp[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) wp[j] = a.W + (size_t)min(j0 + j, all - 1) * 1536 + 8 * lane;
    qt_u32x4 w[D][NT][3];
    float4 xa[D][MT], xb[D][MT];
    unsigned ok[D];
    auto fetch = [&](int it, int d) {
        const int kc = it / a.ntap, p = it - kc * a.ntap, k = 32 * kc + 8 * kg, o = a.off[p];
        unsigned m = 0;
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const int xr = t0 + 16 * i + li + o;
            if (xr >= a.xlo && xr < a.Tx && k < a.K) m |= 1u << i;
            const float *src = a.X + (ptrdiff_t)min(max(xr, a.xlo), a.Tx - 1) * a.ldx + min(k, a.K - 8);
            xa[d][i] = *reinterpret_cast<const float4 *>(src);
            xb[d][i] = *reinterpret_cast<const float4 *>(src + 4);
        }
        ok[d] = m;
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int q = 0; q < 3; q++) w[d][j][q] = *reinterpret_cast<const qt_u32x4 *>(wp[j] + it * step + 512 * q);
    };
    qt_f32x4 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = qt_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < D; d++) fetch(min(i0 + d, i1 - 1), d);
    for (int it = i0; it < i1; it += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (it + d < i1) {
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const unsigned m = 0u - ((ok[d] >> i) & 1u);
                    const float4 p = xa[d][i], q = xb[d][i];
                    float v[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] = __uint_as_float(__float_as_uint(v[e]) & m);
                    qt_u32x4 pl[3];
                    qt_planes8(v, pl);
#pragma unroll
                    for (int j = 0; j < NT; j++) acc[j][i] = qt_mma6(w[d][j], pl, acc[j][i]);
                }
            }
            fetch(min(it + d + D, i1 - 1), d);
        }
    }
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) part[wave][j * MT + i][lane] = acc[j][i];
    __syncthreads();
    for (int c = wave; c < NT * MT; c += SD_GROUPS) {
        const int j = c / MT, i = c - j * MT;
        if (j0 + j >= all) continue;
        const int z = (j0 + j) / a.tiles, n = 16 * (j0 + j - z * a.tiles) + 4 * kg, t = t0 + 16 * i + li;
        qt_f32x4 v = part[0][c][lane];
#pragma unroll
        for (int g = 1; g < SD_GROUPS; g++) v += part[g][c][lane];
        v = sd_finite(a, v, t, j0 + j, n, t < a.T && n < a.N, lane);
        sd_epilogue(a, t, z, n, v);
    }
}

// ---- elementwise / small kernels ---------------------------------------------------------

// codebook = embedding_sum / max(cluster_usage, 1e-5) (sd.c:383-405), [rows][dim]
__global__ void k_sd_cb_dequant(const float *es, const float *cu, float *cb, int rows, int dim) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (size_t)rows * dim) cb[i] = es[i] / fmaxf(cu[i / dim], 1e-5f);
}

// exp of the snake log-parameters: a = e^alpha, ib = e^-beta (k.c:4475-4476)
__global__ void k_sd_snake_params(const float *la, const float *lb, float *a, float *ib, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { a[i] = expf(la[i]); ib[i] = expf(-lb[i]); }
}

// per frame: E[f][0:256] = codebook 0 row, E[f][256:512] = sum of codebooks 1..15 rows in
// order (sd.c:604-625); codes outside [0, 2048) add nothing
__global__ void k_sd_vq(const int *codes, const float *cb, float *E, int cbsize) {
    const int f = blockIdx.x, d = threadIdx.x;        // 256 threads = codebook dim
    const int *c = codes + f * 16;
    const int c0 = c[0];
    E[(size_t)f * 512 + d] = (c0 >= 0 && c0 < cbsize) ? cb[(size_t)c0 * 256 + d] : 0.f;
    float s = 0.f;
    for (int k = 1; k < 16; k++) {
        const int ck = c[k];
        if (ck >= 0 && ck < cbsize) s += cb[((size_t)k * cbsize + ck) * 256 + d];
    }
    E[(size_t)f * 512 + 256 + d] = s;
}

// RMSNorm of rows (qwen_rms_norm, k.c:292-382): out = x * (1/sqrt(mean(x^2) + eps)) * w
__global__ __launch_bounds__(SD_WG) void k_sd_rmsnorm(const float *x, const float *w, float *out, int C, float eps) {
    __shared__ float red[QT_WAVES];
    const float *xr = x + (size_t)blockIdx.x * C;
    float ss = 0.f;
    for (int i = threadIdx.x; i < C; i += SD_WG) ss = fmaf(xr[i], xr[i], ss);
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)C + eps);
    for (int i = threadIdx.x; i < C; i += SD_WG) out[(size_t)blockIdx.x * C + i] = (xr[i] * inv) * w[i];
}

// NeoX split-half RoPE of q and k (columns [0, 1024) and [1024, 2048) of a [.][3072] row),
// 16 heads of 64, tables [pos][32] (sd.c:790-860): rows row0 .. row0 + T - 1 at positions
// pos0 .. pos0 + T - 1
__global__ void k_sd_rope(float *qkv, const float *cs, const float *sn, int T, int row0, int pos0) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;      // (t, which, head, pair)
    if (i >= T * 2 * 16 * 32) return;
    const int pr = i & 31, h = (i >> 5) & 15, which = (i >> 9) & 1, t = i >> 10;
    float *v = qkv + (size_t)(row0 + t) * 3072 + which * 1024 + h * 64;
    const int p = pos0 + t;
    const float c = cs[p * 32 + pr], s = sn[p * 32 + pr];
    const float x1 = v[pr], x2 = v[pr + 32];
    v[pr] = x1 * c - x2 * s;
    v[pr + 32] = x2 * c + x1 * s;
}

// windowed causal attention (qwen_causal_attention_windowed, k.c:3579-3700; seq_q == seq_k,
// q_offset 0): the query at buffer row q0 + t of head h over keys [max(kmin, q0 + t + 1 -
// window), q0 + t] (kmin: the first row holding a key; the streaming decode keeps the
// previous chunks' last window - 1 keys in rows [kmin, q0)).  One wave per (t, h): lanes take
// keys for the scores (dot over 64 dims), then lanes take dims for the weighted sum of values.
__global__ __launch_bounds__(SD_WG) void k_sd_attn(const float *qkv, float *out, int T, int q0, int kmin, int window,
                                                   float scale) {
    __shared__ float sq[QT_WAVES][64];
    __shared__ float sp[QT_WAVES][128];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int item = blockIdx.x * QT_WAVES + wave;
    if (item >= T * 16) return;
    const int t = item >> 4, h = item & 15, qr = q0 + t;
    const int j0 = max(kmin, qr + 1 - window), nk = qr + 1 - j0;   // nk <= window <= 128
    sq[wave][lane] = qkv[(size_t)qr * 3072 + h * 64 + lane];
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    float sc[2];
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int j = r * 64 + lane;
        float s = -INFINITY;
        if (j < nk) {
            const float *kr = qkv + (size_t)(j0 + j) * 3072 + 1024 + h * 64;
            float d = 0.f;
            for (int e = 0; e < 64; e += 4) {
                const float4 kv = *reinterpret_cast<const float4 *>(kr + e);
                d = fmaf(sq[wave][e], kv.x, d); d = fmaf(sq[wave][e + 1], kv.y, d);
                d = fmaf(sq[wave][e + 2], kv.z, d); d = fmaf(sq[wave][e + 3], kv.w, d);
            }
            s = d * scale;
        }
        sc[r] = s;
        mx = fmaxf(mx, s);
    }
    mx = group_max<64>(mx);
    float l = 0.f;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int j = r * 64 + lane;
        const float p = j < nk ? expf(sc[r] - mx) : 0.f;
        sp[wave][j] = p;
        l += p;
    }
    l = group_sum<64>(l);
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    float o = 0.f;
    for (int j = 0; j < nk; j++) o = fmaf(sp[wave][j], qkv[(size_t)(j0 + j) * 3072 + 2048 + h * 64 + lane], o);
    out[(size_t)t * 1024 + h * 64 + lane] = o * (1.0f / l);
}

// m[t][i] = g / (1 + e^-g) * u for the [T][2C] gate|up rows (sd.c:946-950)
__global__ void k_sd_swiglu(const float *gu, float *m, int T, int C) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)T * C) return;
    const size_t t = i / C, c = i % C;
    const float g = gu[t * 2 * C + c], u = gu[t * 2 * C + C + c];
    m[i] = g / (1.0f + expf(-g)) * u;
}

// ConvNeXt: depthwise causal conv (k = 7, pad 6) + LayerNorm over the channels of each
// time step (mean and E[x^2] - mean^2, eps 1e-5), sd.c:1086-1116.  One workgroup per t;
// input rows before xlo (<= 0) read as zero.
__global__ __launch_bounds__(SD_WG) void k_sd_dwln(const float *x, const float *dw, const float *db, const float *lw,
                                                   const float *lb, float *out, int T, int C, int xlo) {
    __shared__ float red[QT_WAVES];
    const int t = blockIdx.x;
    float v[4];
    float s = 0.f, s2 = 0.f;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int c = threadIdx.x + q * SD_WG;
        float d = 0.f;
        if (c < C) {
            d = db[c];
            for (int j = 0; j < 7; j++) {
                const int ti = t - 6 + j;
                if (ti >= xlo) d = fmaf(dw[c * 7 + j], x[(size_t)ti * C + c], d);
            }
        }
        v[q] = d;
        s += d;
        s2 = fmaf(d, d, s2);
    }
    s = block_sum(s, red);
    __syncthreads();
    s2 = block_sum(s2, red);
    const float mean = s / (float)C;
    const float var = s2 / (float)C - mean * mean;
    const float inv = 1.0f / sqrtf(var + 1e-5f);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int c = threadIdx.x + q * SD_WG;
        if (c < C) out[(size_t)t * C + c] = (v[q] - mean) * inv * lw[c] + lb[c];
    }
}

// final conv to one channel (k = 7, pad 6) + clamp to [-1, 1] (sd.c:1259-1279); x [T][C]
// already through the final snake (rows before xlo <= 0 read as zero).  A workgroup takes
// 64 samples: the 70 input rows they
// need go to LDS (row stride C + 1, so the 64 lanes of a read, one row each, hit distinct
// banks); wave w sums channels [w C/4, (w+1) C/4) for its lane's sample, and the four
// partial sums are added in wave order.
#define SD_FIN_T 64
__global__ __launch_bounds__(SD_WG) void k_sd_final(const float *x, const float *w, const float *b, float *audio, int T,
                                                    int C, int xlo) {
    extern __shared__ float xs[];                        // [70][C + 1]
    __shared__ float part[QT_WAVES][SD_FIN_T];
    const int t0 = blockIdx.x * SD_FIN_T, ld = C + 1;
    for (int i = threadIdx.x; i < (SD_FIN_T + 6) * C; i += SD_WG) {
        const int r = i / C, c = i % C, ti = t0 - 6 + r;
        xs[r * ld + c] = (ti >= xlo && ti < T) ? x[(size_t)ti * C + c] : 0.f;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cw = C / QT_WAVES, c0 = wave * cw;
    float s = 0.f;
    for (int c = c0; c < c0 + cw; c++)
#pragma unroll
        for (int j = 0; j < 7; j++) s = fmaf(w[c * 7 + j], xs[(lane + j) * ld + c], s);
    part[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && t0 + lane < T) {
        const float v = b[0] + part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
        audio[t0 + lane] = fminf(fmaxf(v, -1.0f), 1.0f);
    }
}

// streaming history: the last H rows of a buffer's [H + T] rows become its first H rows.
// Source and destination overlap when T < H (a chunk of fewer new rows than the history),
// so a workgroup owns 64 columns whole: its four waves read all H rows of them into
// registers (loads of every row in flight at once), wait for the data, meet at one
// barrier, and only then store.  No other workgroup touches those columns.  All of a
// chunk's buffers (29) go in one launch: each alone is a latency of 3.7 us, with a launch's
// boundary before it (30 frames streamed by 10: 4.53 -> 4.31 ms).
#define SD_SHIFT_MAXH 96
#define SD_SHIFT_N 32
struct SdShiftArgs {
    int n;
    struct { float *buf; int H, T, C, end; } b[SD_SHIFT_N];    // end: workgroups up to this buffer's last
};
__global__ __launch_bounds__(SD_WG) void k_sd_shift(SdShiftArgs a) {
    constexpr int NR = SD_SHIFT_MAXH / 4;
    int j = 0;
    while (j + 1 < a.n && (int)blockIdx.x >= a.b[j].end) j++;
    float *const buf = a.b[j].buf;
    const int H = a.b[j].H, T = a.b[j].T, C = a.b[j].C;
    const int c = ((int)blockIdx.x - (j ? a.b[j - 1].end : 0)) * 64 + (threadIdx.x & 63), r0 = threadIdx.x >> 6;
    float v[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const int r = r0 + 4 * i;
        v[i] = (c < C && r < H) ? buf[(size_t)(T + r) * C + c] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < NR; i++) asm volatile("" : "+v"(v[i]));   // every load has returned
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const int r = r0 + 4 * i;
        if (c < C && r < H) buf[(size_t)r * C + c] = v[i];
    }
}

// ---- launchers ----------------------------------------------------------------------------

// bf16 values of a layer's packed weights
extern "C" size_t qt_sd_pack_elems(int K, int N, int ntap, int phases) {
    return (size_t)((K + 31) / 32) * ntap * phases * ((N + 15) / 16) * 1536;
}
extern "C" hipError_t qt_launch_sd_pack(const float *src, long long sn, long long sk, long long sc, int cols, int stride,
                                        int ntap, int phases, int N, int n0, int nn, int k0, int kk, uint16_t *dst,
                                        hipStream_t st) {
    if (!src || !dst || n0 % 16 || k0 % 32 || nn <= 0 || kk <= 0 || n0 + nn > N) return hipErrorInvalidValue;
    const SdPackArgs a = {src, sn, sk, sc, cols, stride, ntap, phases, (N + 15) / 16, n0, nn, k0, kk, dst};
    const int t = (kk + 31) / 32 * ntap * ((nn + 15) / 16);
    hipLaunchKernelGGL(k_sd_pack, dim3((t + QT_WAVES - 1) / QT_WAVES, 1, phases), dim3(SD_WG), 0, st, a);
    return hipGetLastError();
}

// tile: 0 = by size, 16, 32, 64 or 128 = rows per workgroup.  Every tile sums each output's
// products in the same order, and takes an output again (sd_finite) for that output's own operands
// alone, so the choice never changes a result bit.
extern "C" hipError_t qt_launch_sd_gemm(const float *X, int ldx, int Tx, int xlo, const uint16_t *W, int K, int N,
                                        int ntap, const int *off, int phases, int T, float *Y, int ldy, const float *bias,
                                        const float *cscale, const float *R, const float *sa, const float *sib,
                                        float *Y2, int epi, int tile, hipStream_t st) {
    if (!X || !W || !Y || K <= 0 || K % 16 || N <= 0 || N % 4 || ntap < 1 || ntap > SD_MAXTAP || phases < 1 ||
        T <= 0 || Tx <= 0 || xlo > 0 || ldx % 4 || ldx < K || ldy < N || ldy % 4)
        return hipErrorInvalidValue;
    if (((epi & 1) && !bias) || ((epi & 4) && !cscale) || ((epi & 8) && !R)) return hipErrorInvalidValue;
    if ((epi & (SD_EPI_SNAKE | SD_EPI_SNAKE2)) && (!sa || !sib)) return hipErrorInvalidValue;
    if ((epi & SD_EPI_SNAKE2) && (!Y2 || (epi & SD_EPI_SNAKE))) return hipErrorInvalidValue;
    SdGemmArgs a;
    a.X = X; a.ldx = ldx; a.Tx = Tx; a.xlo = xlo; a.W = W; a.K = K; a.N = N; a.ntap = ntap;
    a.slices = (K + 31) / 32; a.tiles = (N + 15) / 16; a.phases = phases;
    int omax = off[0];
    a.omin = off[0];
    for (int i = 0; i < SD_MAXTAP; i++) {
        a.off[i] = i < ntap ? off[i] : 0;
        if (i < ntap && off[i] < a.omin) a.omin = off[i];
        if (i < ntap && off[i] > omax) omax = off[i];
    }
    a.span = omax - a.omin;
    a.tps = a.span <= SD_HALO ? ntap : 1;
    a.T = T; a.Y = Y; a.ldy = ldy; a.os = phases; a.bias = bias; a.cscale = cscale; a.R = R; a.epi = epi;
    a.sa = sa; a.sib = sib; a.Y2 = Y2;
    const bool grp = a.slices >= SD_GROUP_SLICES;
    const int all = phases * a.tiles;
    const auto wgs = [&](int tt, int nt) { return (long long)((T + tt - 1) / tt) * ((all + nt - 1) / nt); };
    if (tile == 0) {
        // 64-row tiles from about one a CU on; below that the layers with runs take k_sd_split
        // (32 rows reach 550 TFLOP/s of plane products from L2; 16 rows while every tile has a CU of its
        // own: 768 -> 768 channels, 7 taps, 320 rows: 74 us with 16, 37 with 32, 121 with 64, and at 32 rows
        // 20 / 32 / 118) and the others the narrow tiles (384 channels, 1600 rows: 42 us against 59).
        // 64 or 128 rows: by the rounds that the resident workgroups need, three of 64 rows a
        // CU or two of 128 (768 -> 5 x 384 channels: 4000 rows 129 us with 128, 146 with 64; 768 -> 768,
        // 12800 rows: 488 and 462)
        const long long w64 = wgs(64, 8), w128 = wgs(128, 8);
        if (grp && w64 < 224) tile = wgs(16, 1) <= 256 ? 16 : 32;
        else if (!grp && w64 < 256) tile = wgs(32, 4) >= 256 ? 32 : 16;
        else tile = 4 * ((w128 + 511) / 512) <= 3 * ((w64 + 767) / 768) ? 128 : 64;
    }
#define SD_TILE(WN, NT, WT, MT, G)                                                                                          \
    hipLaunchKernelGGL((k_sd_tile<WN, NT, WT, MT, G>),                                                                      \
                       dim3((T + 16 * MT * WT - 1) / (16 * MT * WT), (all + WN * NT - 1) / (WN * NT)), dim3(SD_WG), 0, st, a)
#define SD_SPLIT(NT, MT, D)                                                                                                 \
    hipLaunchKernelGGL((k_sd_split<NT, MT, D>), dim3((T + 16 * MT - 1) / (16 * MT), (all + NT - 1) / NT),                   \
                       dim3(64 * SD_GROUPS), 0, st, a)
    // 96 channels a tile where 128 would be half empty (the decoder's last two blocks: 192 and 96)
    const bool n96 = !grp && all % 8 && all % 6 == 0;
    if (tile == 128) {
        if (grp) SD_TILE(4, 2, 1, 8, true);
        else if (n96) SD_TILE(2, 3, 2, 4, false);
        else SD_TILE(4, 2, 1, 8, false);
    } else if (tile == 64) {
        if (grp) SD_TILE(4, 2, 1, 4, true);
        else if (n96) SD_TILE(2, 3, 2, 2, false);
        else SD_TILE(4, 2, 1, 4, false);
    } else if (tile == 32) {
        if (grp) SD_SPLIT(2, 2, 2);
        else SD_TILE(4, 1, 1, 2, false);
    } else if (tile == 16) {
        if (grp) SD_SPLIT(1, 1, 4);
        else SD_TILE(4, 1, 1, 1, false);
    } else {
        return hipErrorInvalidValue;
    }
#undef SD_TILE
#undef SD_SPLIT
    return hipGetLastError();
}

extern "C" hipError_t qt_launch_sd_cb_dequant(const float *es, const float *cu, float *cb, int rows, int dim,
                                              hipStream_t st) {
    const size_t n = (size_t)rows * dim;
    hipLaunchKernelGGL(k_sd_cb_dequant, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, es, cu, cb, rows, dim);
    return hipGetLastError();
}
extern "C" hipError_t qt_launch_sd_snake_params(const float *la, const float *lb, float *a, float *ib, int n,
                                                hipStream_t st) {
    hipLaunchKernelGGL(k_sd_snake_params, dim3((n + 255) / 256), dim3(256), 0, st, la, lb, a, ib, n);
    return hipGetLastError();
}
extern "C" hipError_t qt_launch_sd_vq(const int *codes, const float *cb, float *E, int n, int cbsize, hipStream_t st) {
    hipLaunchKernelGGL(k_sd_vq, dim3(n), dim3(256), 0, st, codes, cb, E, cbsize);
    return hipGetLastError();
}
extern "C" hipError_t qt_launch_sd_rmsnorm(const float *x, const float *w, float *out, int T, int C, float eps,
                                           hipStream_t st) {
    hipLaunchKernelGGL(k_sd_rmsnorm, dim3(T), dim3(SD_WG), 0, st, x, w, out, C, eps);
    return hipGetLastError();
}
extern "C" hipError_t qt_launch_sd_rope(float *qkv, const float *cs, const float *sn, int T, int row0, int pos0,
                                        hipStream_t st) {
    const int n = T * 1024;
    hipLaunchKernelGGL(k_sd_rope, dim3((n + 255) / 256), dim3(256), 0, st, qkv, cs, sn, T, row0, pos0);
    return hipGetLastError();
}
extern "C" hipError_t qt_launch_sd_attn(const float *qkv, float *out, int T, int q0, int kmin, int window, float scale,
                                        hipStream_t st) {
    if (window <= 0 || window > 128 || kmin < 0 || kmin > q0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_sd_attn, dim3((T * 16 + QT_WAVES - 1) / QT_WAVES), dim3(SD_WG), 0, st, qkv, out, T, q0, kmin,
                       window, scale);
    return hipGetLastError();
}
extern "C" hipError_t qt_launch_sd_swiglu(const float *gu, float *m, int T, int C, hipStream_t st) {
    const size_t n = (size_t)T * C;
    hipLaunchKernelGGL(k_sd_swiglu, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, gu, m, T, C);
    return hipGetLastError();
}
extern "C" hipError_t qt_launch_sd_dwln(const float *x, const float *dw, const float *db, const float *lw, const float *lb,
                                        float *out, int T, int C, int xlo, hipStream_t st) {
    if (C > 4 * SD_WG || xlo > 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_sd_dwln, dim3(T), dim3(SD_WG), 0, st, x, dw, db, lw, lb, out, T, C, xlo);
    return hipGetLastError();
}
extern "C" hipError_t qt_launch_sd_final(const float *x, const float *w, const float *b, float *audio, int T, int C,
                                         int xlo, hipStream_t st) {
    if (C % QT_WAVES || C > 256 || xlo > 0) return hipErrorInvalidValue;
    const size_t lds = (size_t)(SD_FIN_T + 6) * (C + 1) * sizeof(float);
    hipLaunchKernelGGL(k_sd_final, dim3((T + SD_FIN_T - 1) / SD_FIN_T), dim3(SD_WG), lds, st, x, w, b, audio, T, C, xlo);
    return hipGetLastError();
}

// n distinct buffers [H[i] + T[i]][C[i]]
extern "C" hipError_t qt_launch_sd_shift(int n, float *const *buf, const int *H, const int *T, const int *C, hipStream_t st) {
    if (n < 0 || n > SD_SHIFT_N) return hipErrorInvalidValue;
    SdShiftArgs a = {};
    int end = 0;
    for (int i = 0; i < n; i++) {
        if (H[i] <= 0) continue;
        if (!buf[i] || H[i] > SD_SHIFT_MAXH || T[i] <= 0 || C[i] <= 0) return hipErrorInvalidValue;
        end += (C[i] + 63) / 64;
        a.b[a.n++] = {buf[i], H[i], T[i], C[i], end};
    }
    if (!a.n) return hipSuccess;
    hipLaunchKernelGGL(k_sd_shift, dim3(end), dim3(SD_WG), 0, st, a);
    return hipGetLastError();
}
