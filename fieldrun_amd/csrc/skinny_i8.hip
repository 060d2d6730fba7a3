// skinny_i8.hip — int8 W8A8 linear for decode batches (2 <= M <= 16), gfx950.
//
// Restates the M > 1 arm of Bundle::mm's I8 path on pre-quantised rows
// (/root/reference/src/bundle.rs:709-715): acc = i8dot(a8[i], wt[j]) in i32,
// corr = sum over row i's outliers of av * (wt[j, ch] as f32) in ascending
// channel order from -0.0, out = scale[j] * (sa[i] * acc + corr) (separate
// mul / add).  Every output is bit-exact to that order.
//
// HBM-bound: the weights stream once.  A workgroup owns CB blocks of 16
// output rows (16 CB weight rows) over all of K; its KS waves split the
// k-blocks.  Per k-block a wave issues one A operand (the M <= 16 token rows
// of a8, 64 bytes each, L2-resident and shared by every workgroup) and CB B
// operands from the blocked weight copy wblk (each a contiguous 1 KB wave
// load), and CB v_mfma_i32_16x16x64_i8: C[token][weight row].  The waves'
// int32 partials are added through LDS (exact in any order).  The outlier
// correction runs on VALU in the reference's order: the 16-byte runs
// W[j0 .. j0 + 16 CB), ch] of the (K, Np) copy for the rows' 32 outlier
// channels are loaded at the start (they do not depend on the dot) and wait
// in registers until the epilogue.
#include "frq_internal.h"

namespace frq {

namespace {

template <int CB, int KS>
__global__ __launch_bounds__(64 * KS) void skinny_i8_kernel(
    const int8_t* __restrict__ Wb, const int8_t* __restrict__ Wkn, const float* __restrict__ scale,
    int N, int Np, int Kp, const int8_t* __restrict__ a8, int M, const float* __restrict__ sa,
    const uint32_t* __restrict__ oidx, const float* __restrict__ oval, int t,
    float* __restrict__ out, int32_t* __restrict__ acc_dbg) {
    constexpr int NT = 64 * KS, TC = 16 * CB;  // threads, tile columns (weight rows)
    __shared__ v4i red[KS - 1][CB][64];
    __shared__ int tot[16][TC + 1];
    __shared__ __attribute__((aligned(16))) int8_t gat[16 * FRQ_T][TC];  // W[j0 + c, ch(i, q)]
    __shared__ float ovs[16][FRQ_T];

    const int tid = threadIdx.x, lane = tid & 63;
    const int ks = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int jb0 = blockIdx.x * CB, j0 = jb0 * 16;
    // outlier gathers first: pair p = (row i, outlier q), TC bytes each
    constexpr int PPT = (16 * FRQ_T + NT - 1) / NT;  // pairs per thread
    v4i gv[PPT][CB];
    float ovv[PPT];
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
        const int pr = tid + NT * u, i = pr / FRQ_T, q = pr % FRQ_T;
        const bool ok = pr < 16 * FRQ_T && i < M && q < t;
        const uint32_t ch = ok ? min(oidx[(size_t)i * FRQ_T + q], (uint32_t)(Kp - 1)) : 0u;
        ovv[u] = ok ? oval[(size_t)i * FRQ_T + q] : 0.0f;
#pragma unroll
        for (int c = 0; c < CB; ++c)
            gv[u][c] = ok ? *reinterpret_cast<const v4i*>(Wkn + (size_t)ch * Np + j0 + 16 * c)
                          : v4i{0, 0, 0, 0};
    }
    // main loop: lane 16g + r reads token row r (zero past M), k-bytes 16g..
    const int nkb = Kp / 64;
    const int kb0 = nkb * ks / KS, kb1 = nkb * (ks + 1) / KS;
    const int r = lane & 15, g = lane >> 4;
    const bool arow = r < M;
    const int8_t* ap = a8 + (size_t)(arow ? r : 0) * Kp + 16 * g;
    const int8_t* wp = Wb + (size_t)jb0 * 1024 + lane * 16;
    const size_t kstride = (size_t)(Np / 16) * 1024;
    v4i acc[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[c] = v4i{0, 0, 0, 0};
    constexpr int U = 4;
    for (int kb = kb0; kb < kb1; kb += U) {
        v4i av[U], bv[U][CB];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = kb + u < kb1;
            av[u] = (in && arow) ? *reinterpret_cast<const v4i*>(ap + (size_t)(kb + u) * 64) : v4i{0, 0, 0, 0};
#pragma unroll
            for (int c = 0; c < CB; ++c)
                bv[u][c] = in ? ntload_v4i(wp + (size_t)(kb + u) * kstride + (size_t)c * 1024) : v4i{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < CB; ++c)
                acc[c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[u], bv[u][c], acc[c], 0, 0, 0);
    }
    if (ks > 0) {
#pragma unroll
        for (int c = 0; c < CB; ++c) red[ks - 1][c][lane] = acc[c];
    }
    // the gathered bytes and outlier values to LDS
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
        const int pr = tid + NT * u;
        if (pr < 16 * FRQ_T) {
#pragma unroll
            for (int c = 0; c < CB; ++c) *reinterpret_cast<v4i*>(&gat[pr][16 * c]) = gv[u][c];
            ovs[pr / FRQ_T][pr % FRQ_T] = ovv[u];
        }
    }
    __syncthreads();
    if (ks == 0) {
#pragma unroll
        for (int w = 0; w < KS - 1; ++w)
#pragma unroll
            for (int c = 0; c < CB; ++c) acc[c] += red[w][c][lane];
        // C lane l: tokens 4 (l / 16) + e, weight row l % 16
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) tot[4 * (lane >> 4) + e][16 * c + (lane & 15)] = acc[c][e];
    }
    __syncthreads();
    // epilogue: one thread per (token, column), the reference's order
    for (int o = tid; o < M * TC; o += NT) {
        const int i = o / TC, cl = o % TC, j = j0 + cl;
        if (j >= N) continue;
        const int total = tot[i][cl];
        float corr = -0.0f;
        for (int q = 0; q < t; ++q) corr = corr + ovs[i][q] * (float)gat[i * FRQ_T + q][cl];
        out[(size_t)i * N + j] = scale[j] * (sa[i] * (float)total + corr);
        if (acc_dbg) acc_dbg[(size_t)i * N + j] = total;
    }
}

// 17 .. a few hundred rows, in the same order: a wave owns 16 token rows x CB
// column blocks over all of K (A and B operands straight from a8 and wblk, U
// k-blocks in flight; the four waves of a workgroup share the columns, so the
// weights come to them from L1) and forms its outputs itself: the outliers'
// weight bytes (16 rows x 32 channels x 16 CB columns from wkn, requested
// before the k loop) wait in the wave's LDS and each lane adds the 32 terms
// of its outputs in order.  No second pass over the sums, no barrier.  Bound
// by the correction's three VALU instructions a term and, at long K, by L1
// (1 KB + CB KB an MFMA pair).
template <int CB>
__global__ __launch_bounds__(256) void mid_i8_kernel(
    const int8_t* __restrict__ Wb, const int8_t* __restrict__ Wkn, const float* __restrict__ scale, int N, int Np,
    int Kp, const int8_t* __restrict__ a8, int M, const float* __restrict__ sa, const uint32_t* __restrict__ oidx,
    const float* __restrict__ oval, int t, float* __restrict__ out, int32_t* __restrict__ acc_dbg) {
    constexpr int TC = 16 * CB, RS = FRQ_T * TC + 16;  // RS: bytes a token's gathered rows (+16: other banks)
    __shared__ __attribute__((aligned(16))) int8_t gat_[4][16 * RS];
    __shared__ __attribute__((aligned(16))) float ovs_[4][16 * FRQ_T];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = ((int)blockIdx.y * 4 + wave) * 16, jb0 = blockIdx.x * CB, j0 = jb0 * 16;
    if (m0 >= M) return;  // whole waves, no barrier below
    int8_t* gat = gat_[wave];
    float* ovs = ovs_[wave];
    // the outlier gathers: pair p = (token p / 32, outlier p % 32)
    v4i gv[8][CB];
    float ovv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int p = lane + 64 * u, i = m0 + p / FRQ_T;
        const bool ok = i < M && p % FRQ_T < t;
        const size_t at = (size_t)(ok ? i : 0) * FRQ_T + p % FRQ_T;
        const uint32_t ch = ok ? min(oidx[at], (uint32_t)(Kp - 1)) : 0u;
        ovv[u] = ok ? oval[at] : 0.0f;
#pragma unroll
        for (int c = 0; c < CB; ++c) gv[u][c] = *reinterpret_cast<const v4i*>(Wkn + (size_t)ch * Np + j0 + 16 * c);
    }
    // lane 16 g + r: token row r (the last row past M), k-bytes 16 g ..
    const int nkb = Kp / 64;
    const int8_t* ap = a8 + (size_t)min(m0 + (lane & 15), M - 1) * Kp + 16 * (lane >> 4);
    const int8_t* wp = Wb + (size_t)jb0 * 1024 + lane * 16;
    const size_t kstride = (size_t)(Np / 16) * 1024;
    v4i acc[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[c] = v4i{0, 0, 0, 0};
    constexpr int U = 4;
    v4i an[U], bn[U][CB];
    auto load = [&](int u, int kb) {  // unconditional: past the end the last block again
        const int k = min(kb, nkb - 1);
        an[u] = *reinterpret_cast<const v4i*>(ap + (size_t)k * 64);
#pragma unroll
        for (int c = 0; c < CB; ++c) bn[u][c] = *reinterpret_cast<const v4i*>(wp + (size_t)k * kstride + (size_t)c * 1024);
    };
#pragma unroll
    for (int u = 0; u < U; ++u) load(u, u);
    for (int kb = 0; kb < nkb; kb += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (kb + u < nkb) {
#pragma unroll
                for (int c = 0; c < CB; ++c)
                    acc[c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(an[u], bn[u][c], acc[c], 0, 0, 0);
            }
            load(u, kb + u + U);
        }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int p = lane + 64 * u;
#pragma unroll
        for (int c = 0; c < CB; ++c)
            *reinterpret_cast<v4i*>(gat + (p / FRQ_T) * RS + (p % FRQ_T) * TC + 16 * c) = gv[u][c];
        ovs[p] = ovv[u];
    }
    wave_sync();
    // lane l: tokens 4 (l / 16) + e, column l % 16 of each block
    const int i0 = 4 * (lane >> 4);
    float corr[4][CB];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < CB; ++c) corr[e][c] = -0.0f;
    for (int q = 0; q < t; ++q) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float ov = ovs[(i0 + e) * FRQ_T + q];
#pragma unroll
            for (int c = 0; c < CB; ++c)
                corr[e][c] = corr[e][c] + ov * (float)gat[(i0 + e) * RS + q * TC + 16 * c + (lane & 15)];
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = m0 + i0 + e;
        if (i >= M) continue;
        const float s = sa[i];
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const int j = j0 + 16 * c + (lane & 15);
            if (j >= N) continue;
            out[(size_t)i * N + j] = scale[j] * (s * (float)acc[c][e] + corr[e][c]);
            if (acc_dbg) acc_dbg[(size_t)i * N + j] = acc[c][e];
        }
    }
}

template <int CB, int KS>
hipError_t launch_s(const Weight& w, size_t m, const int8_t* a8, const float* sa,
                    const uint32_t* oidx, const float* oval, float* out, int32_t* acc, hipStream_t s) {
    const unsigned grid = (unsigned)(w.np / (16 * CB));
    const int t = (int)(w.k < FRQ_T ? w.k : FRQ_T);
    skinny_i8_kernel<CB, KS><<<dim3(grid), dim3(64 * KS), 0, s>>>(
        w.wblk, w.wkn, w.scale, (int)w.n, (int)w.np, (int)w.kp, a8, (int)m, sa, oidx, oval, t, out, acc);
    return hipGetLastError();
}

template <int CB>
hipError_t launch_m(const Weight& w, size_t m, const int8_t* a8, const float* sa, const uint32_t* oidx,
                    const float* oval, float* out, int32_t* acc, hipStream_t s) {
    const int t = (int)(w.k < FRQ_T ? w.k : FRQ_T);
    const dim3 grid((unsigned)((w.n + 16 * CB - 1) / (16 * CB)), (unsigned)((m + 63) / 64));
    mid_i8_kernel<CB><<<grid, dim3(256), 0, s>>>(w.wblk, w.wkn, w.scale, (int)w.n, (int)w.np, (int)w.kp, a8, (int)m,
                                                 sa, oidx, oval, t, out, acc);
    return hipGetLastError();
}

}  // namespace

// The middling batches that this kernel takes from the GEMM (with the union
// correction for frq_mm_dev, with the exact epilogue for frq_mm_exact_dev):
// by an estimate of its tiles, 3.2 ns + 1.9 ps a k each over the whole card,
// up to 30 us.  Its time is that and 6 .. 12 us (the quant and the launches;
// at long K the walk of one wave, which the estimate leaves out: 64 us at 32 x
// 18944 x 3584, estimated at 18), the GEMM's at least 34 us from K = 512 on and
// more with K (56 at 9216, 75 at 18944; 77 at that product), so the tiles are
// the faster there; a higher cut would still gain (512 x 896 x 4864: 48
// against 68).  Shorter K is cheap for the GEMM (K = 128:
// 24 us however many rows, 256: 28), and outputs wider than 32768 run half-empty
// workgroups in a third round (32 x 512 x 40000: 43 against 34 exact).  Timed on
// both routes at 1800 products of K 32 .. 20480, N 64 .. 65000, M 17 .. 4096:
// none that this rule picks is slower by more than 7% (K = 384; 3% from 512).
// K beyond 20480, which the GEMM does not hold, is served here alone.
bool mid_i8_ok(const Weight& w, size_t m) {
    if (m <= 16 || m > 65535 || !w.wblk || !w.wkn || w.kp == 0 || w.kp % 64 || w.n > 32768) return false;
    const double tiles = (double)((w.n + 15) / 16) * (double)((m + 15) / 16);
    const double cut = w.kp < 256 ? 13000.0 : w.kp < 512 ? 17000.0 : 30000.0;
    return tiles * (3.2 + 0.0019 * (double)w.kp) <= cut;
}

hipError_t launch_mid_i8(const Weight& w, size_t m, const int8_t* a8, const float* sa, const uint32_t* oidx,
                         const float* oval, float* out, int32_t* acc, hipStream_t s) {
    // a8: m rows of pitch Kp; wblk / wkn padded to Np (a multiple of 256)
    if (m < 1 || m > 65535 || !w.wblk || !w.wkn || w.kp % 64 || w.kp == 0) return hipErrorInvalidValue;
    // two column blocks a wave from 1500 tiles on (us of the kernel, one / two: K=896 N=4864
    // M=48 11.8 / 11.4, M=129 19.9 / 17.9, M=512 55 / 41; K=4096 N=14336 M=20
    // 31.7 / 21.1; K=2048 N=2048 M=129 12.3 / 15.5, M=256 20.0 / 15.9)
    if ((w.n + 15) / 16 * ((m + 15) / 16) > 1500) return launch_m<2>(w, m, a8, sa, oidx, oval, out, acc, s);
    return launch_m<1>(w, m, a8, sa, oidx, oval, out, acc, s);
}

hipError_t launch_skinny_i8(const Weight& w, size_t m, const int8_t* a8, const float* sa,
                            const uint32_t* oidx, const float* oval, float* out, int32_t* acc,
                            hipStream_t s) {
    // a8: m rows of pitch Kp; wblk / wkn padded to Np (a multiple of 256)
    if (m < 1 || m > 16 || !w.wblk || w.kp % 64) return hipErrorInvalidValue;
    // enough workgroups to fill the chip: two column blocks per workgroup
    // when N is large, and the k-blocks split over more waves when K is long
    const size_t blocks = w.np / 16;
    if (w.kp > 8192) return launch_s<1, 8>(w, m, a8, sa, oidx, oval, out, acc, s);
    if (blocks >= 2048) return launch_s<2, 4>(w, m, a8, sa, oidx, oval, out, acc, s);
    return launch_s<1, 4>(w, m, a8, sa, oidx, oval, out, acc, s);
}

}  // namespace frq
