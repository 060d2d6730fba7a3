// mm_f32.hip — the M > 1 products of dequantised weights in a.dot's own f32
// order, on the f32 matrix cores (gfx950).
//
// out[m, n] = sum over k of a[m, k] * W[n, k] as matrixmultiply's sgemm sums
// it: MM_KC-long k blocks, each an FMA chain from +0 with k ascending, the
// block values added in order.  W is formed in registers from its stored
// bytes: int4 s4 * scale (/root/reference/src/bundle.rs:777-798), q4a
// scale * u4 + min (802-845), and the expert banks' f16 / f32 (404-454).
//
// v_mfma_f32_16x16x4_f32 advances each output by fma(a_k, w_k, c) with k
// ascending and one rounding a step (checked bit for bit against fmaf chains
// over normal, subnormal, zero and non-finite values), so a block's chain is
// a run of MFMAs on an accumulator that starts at +0.  It runs at 69 T FMA/s
// on the card against 50 for v_fma_f32 and 25 for its DPP-broadcast form,
// and one operand register serves 16 rows.
//
// A wave owns MT row tiles x NT column tiles of 16 x 16 outputs and takes k
// in chunks of 32, whose operands pass through its own LDS buffer (no barrier
// in the k loop): activations and packed weights are loaded in whole cache
// lines under the MFMAs of the chunk before.  What bounds it: the f32 MFMAs
// share the SIMD's pipe with the VALU, which forms the weights (two
// to three instructions a value): 1500 clocks a chunk of 1024 MFMA clocks at MT = 1.
// Measured against the kernels it replaced (a lane a row of the output's
// columns; DPP-broadcast weights), us: int4 300 x 2304 x 9216 3250 (frq_mm)
// / 240 -> 153 (42 T FMA/s), 1024 x 2304 x 9216 -> 438 (50), q4a 64 x 9216 x
// 2304 400 -> 83.
//
// P == 1: four independent waves a workgroup, each keeping the running block
// sums of its tile in registers.  P > 1: the P waves of a workgroup share
// one tile and take blocks p, p + P, ...; after each P blocks their values
// meet in LDS and are added in block order (the chains of different blocks
// are independent, so this split is exact).  mm_plan picks the form.
#include <cmath>
#include <type_traits>

#include "frq_internal.h"

namespace frq {

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // rows of any K: 4-byte aligned
typedef unsigned u4u __attribute__((ext_vector_type(4), aligned(1)));  // packed rows: any alignment
typedef unsigned u2u __attribute__((ext_vector_type(2), aligned(1)));
typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));

// A 16 x 16 output tile's MFMAs over a 32-long chunk of k: MFMA s takes k =
// 4 s + h of lane group h = lane / 16, and accumulator element v of a lane is
// row 4 (lane / 16) + v, column lane % 16.
constexpr int TT = 16, G = 4, VX = 8, SEG = 128;
__device__ __forceinline__ f4v mma(float a, float b, f4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// ---- a wave's weights -------------------------------------------------------
// Packed rows (int4, q4a) with groups of a multiple of 32: a segment of 128 k
// of the wave's R = NT TT rows is loaded at once, whole 64-byte pieces of a
// row by four lanes, a row's four scales by one lane, and waits in the wave's
// LDS buffer for its four chunks (a lane per row and chunk instead made every
// load touch 32 or 64 cache lines: 339 -> 657 us of a 1024 x 2304 x 9216
// product).  Column tile c's lane i has row n0 + TT c + i.  RAG: K ends
// inside a chunk.
template <int DT, int NT, bool RAG_>
struct Packed {
    static constexpr bool RAG = RAG_, Q = DT == FRQ_DT_Q4A;
    static constexpr int R = NT * TT, RL = R / 16;
    static constexpr int LDS = R * 16 + (Q ? 8 : 4) * R;  // words: nibbles, scales (and mins)
    const uint8_t* p[RL];
    const uint16_t *s, *m;
    int lane, K, g, ss, ng;
    v4u wn[RL];
    u2v sn, mn;  // the four chunks' f16 scales and mins
    __device__ __forceinline__ Packed(const MmWeight& v, size_t e, int n0, int lane_) : lane(lane_) {
        K = v.k; g = v.g; ss = v.ss; ng = v.ng;
#pragma unroll
        for (int i = 0; i < RL; ++i) {
            const size_t row = (size_t)min(n0 + 16 * i + (lane >> 2), v.n - 1);
            p[i] = reinterpret_cast<const uint8_t*>(v.w) + e * v.per + row * v.pitch + 16 * (lane & 3);
        }
        const size_t row = e * v.sper + (size_t)min(n0 + lane % R, v.n - 1) * v.ng;
        s = v.sc + row * v.ss;
        m = Q ? v.mn + row * v.ss : nullptr;
    }
    __device__ __forceinline__ void load_seg(int k0) {
#pragma unroll
        for (int i = 0; i < RL; ++i) wn[i] = *reinterpret_cast<const u4u*>(p[i] + k0 / 2);
        u2v sv, mv = {0, 0};
        if (g == 32 && (!Q || ss == 1)) {  // uniform: the four in one load (past the row's last: not used)
            sv = *reinterpret_cast<const u2u*>(s + k0 / 32);
            if constexpr (Q) mv = *reinterpret_cast<const u2u*>(m + k0 / 32);
        } else if (Q && g == 32) {  // scale | min words
            const v4u w = *reinterpret_cast<const u4u*>(s + k0 / 32 * 2);
            sv = u2v{(w.x & 0xffffu) | (w.y << 16), (w.z & 0xffffu) | (w.w << 16)};
            mv = u2v{(w.x >> 16) | (w.y & 0xffff0000u), (w.z >> 16) | (w.w & 0xffff0000u)};
        } else {
            auto at = [&](int c) { return min((k0 + 32 * c) / g, ng - 1) * ss; };
            auto four = [&](const uint16_t* q) {
                return u2v{(uint32_t)q[at(0)] | ((uint32_t)q[at(1)] << 16),
                           (uint32_t)q[at(2)] | ((uint32_t)q[at(3)] << 16)};
            };
            sv = four(s);
            if constexpr (Q) mv = four(m);
        }
        sn = sv;
        mn = mv;
    }
    __device__ __forceinline__ void put_seg(float* buf) const {
        v4u* w = reinterpret_cast<v4u*>(buf);
#pragma unroll
        for (int i = 0; i < RL; ++i) {
            const int r = 16 * i + (lane >> 2);
            w[r * 4 + ((lane & 3) ^ ((r >> 2) & 3))] = wn[i];
        }
        float* sl = buf + R * 16;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            sl[c * R + lane % R] = h2f((uint16_t)((c < 2 ? sn.x : sn.y) >> (16 * (c % 2))));
            if constexpr (Q) sl[(4 + c) * R + lane % R] = h2f((uint16_t)((c < 2 ? mn.x : mn.y) >> (16 * (c % 2))));
        }
    }
    __device__ __forceinline__ void load(int) {}
    // chunk c of the segment, k0 its first k
    __device__ __forceinline__ void form(const float* buf, int c, float (&x)[NT][VX]) const {
        const v4u* w4 = reinterpret_cast<const v4u*>(buf);
        const float* sl = buf + R * 16;
        const int h = lane / TT;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int r = TT * t + lane % TT;
            const v4u q = w4[r * 4 + (c ^ ((r >> 2) & 3))];
            const uint32_t w[4] = {q.x >> (4 * h), q.y >> (4 * h), q.z >> (4 * h), q.w >> (4 * h)};
            const float sc = sl[c * R + r], mi = Q ? sl[(4 + c) * R + r] : 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {  // word i: k = 8 i + h and 8 i + 4 + h, nibble h of each half
                if constexpr (Q) {  // u as f16 pairs, then scale * u (exact) + min in one rounding
                    const h2v u = __builtin_bit_cast(h2v, (w[i] & 0x000F000Fu) | 0x64006400u) - h2v{1024, 1024};
                    x[t][2 * i] = __builtin_fmaf((float)u.x, sc, mi);
                    x[t][2 * i + 1] = __builtin_fmaf((float)u.y, sc, mi);
                } else {  // s4 from the f16 1032 + s4, then one product: exact, and s4 * scale for any scale
                    const h2v u = __builtin_bit_cast(h2v, (w[i] & 0x000F000Fu) ^ 0x64086408u) - h2v{1032, 1032};
                    x[t][2 * i] = __builtin_fmaf((float)u.x, sc, mi);
                    x[t][2 * i + 1] = __builtin_fmaf((float)u.y, sc, mi);
                }
            }
        }
    }
    __device__ __forceinline__ void form_end(float* buf, int k0, float (&x)[NT][VX]) {
        load_seg(k0);
        wave_sync();
        put_seg(buf);
        wave_sync();
        form(buf, 0, x);
    }
    static __device__ __forceinline__ int col(int n0, int c, int lane, int) { return n0 + TT * c + lane % TT; }
};

// Packed rows with any other group: a lane per row and chunk, a scale (and
// min) a value.
template <int DT, int NT>
struct PackedAny {
    static constexpr bool RAG = true, Q = DT == FRQ_DT_Q4A;
    static constexpr int LDS = 0;
    const uint8_t* p[NT];
    const uint16_t *s[NT], *m[NT];
    int h, g, ss, ng;
    v4u wn[NT];
    uint16_t sn[NT][VX], mn[NT][Q ? VX : 1];
    __device__ __forceinline__ PackedAny(const MmWeight& v, size_t e, int n0, int lane) {
        h = lane / TT;
        g = v.g; ss = v.ss; ng = v.ng;
#pragma unroll
        for (int c = 0; c < NT; ++c) {
            const size_t row = (size_t)min(n0 + TT * c + lane % TT, v.n - 1);
            p[c] = reinterpret_cast<const uint8_t*>(v.w) + e * v.per + row * v.pitch;
            s[c] = v.sc + (e * v.sper + row * (size_t)v.ng) * v.ss;
            m[c] = Q ? v.mn + (e * v.sper + row * (size_t)v.ng) * v.ss : nullptr;
        }
    }
    __device__ __forceinline__ void load_seg(int) {}
    __device__ __forceinline__ void put_seg(float*) const {}
    __device__ __forceinline__ void load(int k0) {
#pragma unroll
        for (int c = 0; c < NT; ++c) wn[c] = *reinterpret_cast<const u4u*>(p[c] + k0 / 2);
        int gi = (k0 + h) / g, in = k0 + h - gi * g;
#pragma unroll
        for (int i = 0; i < VX; ++i) {
            const int at = min(gi, ng - 1) * ss;  // past K: the last group's
#pragma unroll
            for (int c = 0; c < NT; ++c) {
                sn[c][i] = s[c][at];
                if constexpr (Q) mn[c][i] = m[c][at];
            }
            for (in += G; in >= g; in -= g) ++gi;
        }
    }
    __device__ __forceinline__ void form(const float*, int, float (&x)[NT][VX]) const {
#pragma unroll
        for (int c = 0; c < NT; ++c)
#pragma unroll
            for (int i = 0; i < VX; ++i) {
                const uint32_t v = wn[c][i / 2] >> (4 * h);
                const int b = 16 * (i % 2);
                if constexpr (Q) x[c][i] = h2f(sn[c][i]) * (float)((v >> b) & 15u) + h2f(mn[c][i]);
                else x[c][i] = (float)(int)__builtin_amdgcn_sbfe((int)v, b, 4) * h2f(sn[c][i]);
            }
    }
    __device__ __forceinline__ void form_end(float*, int k0, float (&x)[NT][VX]) {
        load(k0);
        form(nullptr, 0, x);
    }
    static __device__ __forceinline__ int col(int n0, int c, int lane, int) { return n0 + TT * c + lane % TT; }
};

// (in, out) rows (f16, f32): a lane's NT columns are adjacent, n0 + NT i ..;
// past the matrix they are its last NT (stored twice, the same values).
template <int DT, int NT>
struct Columns {
    static constexpr bool RAG = true;
    static constexpr int LDS = 0;
    using E = std::conditional_t<DT == FRQ_DT_F16, uint16_t, float>;
    typedef E V __attribute__((ext_vector_type(NT)));
    typedef E VU __attribute__((ext_vector_type(NT), aligned(sizeof(E))));  // rows of any width
    const E* p;
    int h, K;
    size_t n;
    V wn[VX];
    __device__ __forceinline__ Columns(const MmWeight& v, size_t e, int n0, int lane) {
        h = lane / TT;
        K = v.k;
        n = (size_t)v.n;
        p = reinterpret_cast<const E*>(v.w) + e * v.per + col(n0, 0, lane, v.n);
    }
    __device__ __forceinline__ void load_seg(int) {}
    __device__ __forceinline__ void put_seg(float*) const {}
    __device__ __forceinline__ void load(int k0) {
        const E* q = p + (size_t)(k0 + h) * n;
#pragma unroll
        for (int i = 0; i < VX; ++i) wn[i] = *reinterpret_cast<const VU*>(q + (size_t)(G * i) * n);
    }
    __device__ __forceinline__ void form(const float*, int, float (&x)[NT][VX]) const {
#pragma unroll
        for (int c = 0; c < NT; ++c)
#pragma unroll
            for (int i = 0; i < VX; ++i) {
                if constexpr (DT == FRQ_DT_F16) x[c][i] = h2f(wn[i][c]);
                else x[c][i] = wn[i][c];
            }
    }
    __device__ __forceinline__ void form_end(float*, int k0, float (&x)[NT][VX]) {
#pragma unroll
        for (int i = 0; i < VX; ++i)
            wn[i] = *reinterpret_cast<const VU*>(p + (size_t)min(k0 + G * i + h, K - 1) * n);
        form(nullptr, 0, x);
    }
    static __device__ __forceinline__ int col(int n0, int c, int lane, int n) {
        return max(0, min(n0 + NT * (lane % TT), n - NT)) + c;
    }
};

// GM 0: Packed, K a multiple of 32; 1: Packed, any K; 2: PackedAny.
template <int DT, int NT, int GM>
using Weights = std::conditional_t<
    DT == FRQ_DT_F16 || DT == FRQ_DT_F32, Columns<DT == FRQ_DT_F16 ? FRQ_DT_F16 : FRQ_DT_F32, NT>,
    std::conditional_t<GM == 2, PackedAny<DT, NT>, Packed<DT, NT, GM == 1>>>;

// GR: the rows of one expert's tile (MmGroup), else rows 0 .. M - 1.  Two forms
// spill a register or two (q4a 1 x 4 over 16 waves, f16 2 x 4 grouped).
template <int DT, int MT, int NT, int P, int GM, bool GR>
__global__ __launch_bounds__(64 * (P == 1 ? 4 : P), P == 16 ? 4 : MT * NT >= 8 || GM || P == 8 ? 2 : 3) void mm_f32_kernel(
    MmWeight w, MmGroup grp, const float* __restrict__ a, int M, int tm, int tn, float* __restrict__ out) {
    using L = Weights<DT, NT, GM>;
    constexpr int AV = 4, E = MT * NT * TT * TT;
    constexpr int PPT = P == 1 ? 1 : (E + 64 * P - 1) / (64 * P);  // output elements a thread sums
    constexpr int NW = P == 1 ? 4 : P, ABUF = MT * TT * 32, BUF = ABUF + L::LDS;
    constexpr int WB = P > 1 && E > BUF ? E : BUF;  // a wave's buffer; a slice's end: its block values
    __shared__ __align__(16) float wl[NW * WB];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int K = w.k, nb = (K + MM_KC - 1) / MM_KC;
    int it, ct, rows, pbase = 0;
    size_t e = 0;
    if constexpr (GR) {
        it = 0;
        ct = P == 1 ? (int)blockIdx.y * 4 + wave : (int)blockIdx.y;
        if ((int)blockIdx.x >= grp.ntile[0]) return;  // uniform
        e = (size_t)grp.tile_e[blockIdx.x];
        const int r0 = grp.tile_r[blockIdx.x];
        rows = min(grp.rows, grp.cnt[e] - r0);
        pbase = grp.off[e] + r0;
    } else {
        // contiguous tile ranges an XCD (workgroups go round the 8 XCDs), rows
        // fastest: an XCD's L2 holds its share of the columns' weights while
        // the rows pass; the waves of a workgroup share activation rows
        const int nwg = gridDim.x, x = blockIdx.x & 7, q = nwg >> 3, rem = nwg & 7;
        const int wg = x * q + min(x, rem) + (blockIdx.x >> 3);
        ct = wg / tm;
        it = wg - ct * tm;
        if (P == 1) ct = ct * 4 + wave;
        rows = min(MT * TT, M - it * MT * TT);
    }
    if (P == 1 && ct >= tn) return;  // whole waves, and no barrier below
    const int n0 = ct * NT * TT;
    L ld(w, e, n0, lane);
    // The tile's activations of a chunk: lane 8 r + q loads 16 bytes (k0 +
    // 4 q ..) of rows r, r + 8, ..., so a load covers whole 128-byte lines,
    // and the wave's own LDS buffer hands them to the MFMA lanes: row r is
    // 128 bytes in lane-group order (k = h, G + h, 2 G + h, ... of group h
    // together), its 16-byte slots exchanged by the row so that 16 lanes
    // reading one slot number of 16 rows meet all banks.
    constexpr int RL = MT * TT / 8;
    float* const abuf = wl + wave * WB;
    float* const wbuf = abuf + ABUF;
    const int lq = lane & 7;
    const float* ar[RL];
#pragma unroll
    for (int i = 0; i < RL; ++i) {
        int r = min(8 * i + (lane >> 3), rows - 1);
        if constexpr (GR) r = grp.gather ? grp.ptok[pbase + r] : pbase + r;
        else r += it * MT * TT;
        ar[i] = a + (size_t)r * K + 4 * lq;
    }
    auto load_a = [&](int k0, f4v (&x)[RL]) {
#pragma unroll
        for (int i = 0; i < RL; ++i) x[i] = *reinterpret_cast<const f4u*>(ar[i] + k0);
    };
    auto put_a = [&](const f4v (&x)[RL]) {
#pragma unroll
        for (int i = 0; i < RL; ++i) {
            const int r = 8 * i + (lane >> 3), sw = (r >> 1) & 7;
            float* row = abuf + r * 32;
#pragma unroll
            for (int g = 0; g < 4; ++g) row[(((2 * g + (lq >> 2)) ^ sw) * 4) + (lq & 3)] = x[i][g];
        }
    };
    f4v acc[MT][NT];
    auto multiply = [&](float (&y)[NT][VX]) {
        auto tiles = [&](auto n) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                f4v x[MT];
#pragma unroll
                for (int t = 0; t < decltype(n)::value; ++t) {
                    const int r = t * TT + lane % TT, slot = 2 * (lane / TT) + u;
                    x[t] = *reinterpret_cast<const f4v*>(abuf + r * 32 + (slot ^ ((r >> 1) & 7)) * 4);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int t = 0; t < decltype(n)::value; ++t)
#pragma unroll
                        for (int c = 0; c < NT; ++c) acc[t][c] = mma(x[t][i], y[c][4 * u + i], acc[t][c]);
            }
        };
        if (GR && MT > 1 && rows <= TT) tiles(std::integral_constant<int, 1>{});  // a short tile (uniform)
        else tiles(std::integral_constant<int, MT>{});
    };
    // this wave's whole chunks: those of blocks p, p + P, ... in order, each
    // (a segment's weights) loaded under the MFMAs before; past the last one
    // that one again, not used
    const int p = P == 1 ? 0 : wave;
    const int kw = K / 32 * 32, last = kw - 32;
    auto after = [&](int k1, int k0) {  // k1 > k0: on in k0's block, or the wave's next block
        return min((k1 % MM_KC) && k1 < kw ? k1 : (k0 / MM_KC + P) * MM_KC, last);
    };
    f4v an[RL];
    int k0 = min(p * MM_KC, last);
    if (kw) {
        load_a(k0, an);
        ld.load(k0);
        ld.load_seg(k0 / SEG * SEG);
    }
    auto block = [&](int b) {  // the chain of block b into acc
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int v = 0; v < AV; ++v) acc[t][c][v] = 0.0f;
        const int end = min(kw, (b + 1) * MM_KC);
        for (int ks = b * MM_KC; ks < end; ks += SEG) {
            wave_sync();  // the wave's LDS accesses run in order
            ld.put_seg(wbuf);
            ld.load_seg(after(ks + SEG, ks) / SEG * SEG);
            const int nc = min(SEG, end - ks) / 32;
            for (int c = 0; c < nc; ++c) {
                float y[NT][VX];
                wave_sync();
                put_a(an);
                wave_sync();
                ld.form(wbuf, c, y);
                k0 = after(k0 + 32, k0);
                load_a(k0, an);
                ld.load(k0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(y);
            }
        }
        if (L::RAG && b == nb - 1 && kw < K) {  // the row's ragged end, zeros past it: fma(0, 0, c) = c
            float y[NT][VX];
            f4v z[RL];
#pragma unroll
            for (int i = 0; i < RL; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) z[i][j] = kw + 4 * lq + j < K ? ar[i][kw + j] : 0.0f;
            wave_sync();
            put_a(z);
            ld.form_end(wbuf, kw, y);
            wave_sync();
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int i = 0; i < VX; ++i) y[c][i] = kw + G * i + lane / TT < K ? y[c][i] : 0.0f;
            multiply(y);
        }
    };
    auto store = [&](int t, int c, int v, int ln, float val) {
        const int r = t * TT + 4 * (ln >> 4) + v;
        const int n = L::col(n0, c, ln, w.n);
        const size_t orow = GR ? (size_t)(pbase + r) : (size_t)(it * MT * TT + r);
        if (r < rows && n < w.n) out[orow * w.n + n] = val;
    };
    if constexpr (P == 1) {
        f4v tot[MT][NT];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int v = 0; v < AV; ++v) tot[t][c][v] = 0.0f;
        for (int b = 0; b < nb; ++b) {
            block(b);
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int c = 0; c < NT; ++c)
#pragma unroll
                    for (int v = 0; v < AV; ++v) tot[t][c][v] = tot[t][c][v] + acc[t][c][v];
        }
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int v = 0; v < AV; ++v) store(t, c, v, lane, tot[t][c][v]);
    } else {
        float sum[PPT];
#pragma unroll
        for (int i = 0; i < PPT; ++i) sum[i] = 0.0f;
        for (int b0 = 0; b0 < nb; b0 += P) {
            if (b0 + p < nb) {
                block(b0 + p);
                wave_sync();
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int c = 0; c < NT; ++c)
#pragma unroll
                        for (int v = 0; v < AV; ++v)
                            abuf[((t * NT + c) * AV + v) * 64 + lane] = acc[t][c][v];
            }
            __syncthreads();
            const int np = min(P, nb - b0);
#pragma unroll
            for (int i = 0; i < PPT; ++i)
                for (int j = 0; j < np; ++j)
                    sum[i] = sum[i] + wl[j * WB + min((int)threadIdx.x + 64 * P * i, E - 1)];
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < PPT; ++i) {
            const int el = threadIdx.x + 64 * P * i, tcv = el >> 6;
            if (el < E) store(tcv / AV / NT, tcv / AV % NT, tcv % AV, el & 63, sum[i]);
        }
    }
}

// The forms: MT x NT tiles a wave, P waves over the blocks of k.
struct Plan {
    int mt, nt, p;
};

// The form that takes the fewest clocks: every CU's SIMDs run
// ceil(workgroups / CUs) x ceil(P / 4) waves, each ceil(nb / P) blocks of 8
// chunks.  A chunk's clocks a wave are measured (the f32 MFMAs and VALU
// instructions of all waves of a SIMD share its pipe, so they add up): 1500
// at MT = 1 and 2800 at MT = 2 (1024 and 2048 of them in the MFMAs), 400
// more where a wave is alone on its SIMD and waits for its own loads.
Plan mm_plan(const Plan* forms, int nf, size_t m, size_t n, size_t k, size_t groups, int cus) {
    const size_t nb = (k + MM_KC - 1) / MM_KC;
    Plan best = forms[0];
    double bt = 0;
    for (int f = 0; f < nf; ++f) {
        const Plan& q = forms[f];
        const size_t rt = (size_t)TT * q.mt, ct = (size_t)TT * q.nt * (q.p == 1 ? 4 : 1);
        const double wgs = (double)((m + rt - 1) / rt) * (double)((n + ct - 1) / ct) * (double)groups;
        const double wps = std::ceil(wgs * (q.p == 1 ? 4 : q.p) / 4.0 / cus) * (q.p > 4 && wgs < cus ? q.p / 4 : 1);
        const double chunk = (q.mt == 1 ? 1500 : 2800) * q.nt / 4.0 * wps + (wps <= 1 ? 400 : 0);
        const double t = (double)((nb + q.p - 1) / q.p) * (8 * chunk + 800);
        if (f == 0 || t < bt) {
            bt = t;
            best = q;
        }
    }
    return best;
}

template <int DT, int MT, int NT, int P, int GM, bool GR>
hipError_t go(const MmWeight& w, const MmGroup& grp, unsigned ntile, const float* a, size_t m, float* out,
              hipStream_t s) {
    const int tm = (int)((m + TT * MT - 1) / (TT * MT)), tn = (w.n + TT * NT - 1) / (TT * NT);
    constexpr int TPW = P == 1 ? 4 : 1;  // tiles a workgroup
    const dim3 grid = GR ? dim3(ntile, (unsigned)((tn + TPW - 1) / TPW))
                         : dim3((unsigned)((size_t)tm * ((tn + TPW - 1) / TPW)));
    mm_f32_kernel<DT, MT, NT, P, GM, GR><<<grid, dim3(64 * (P == 1 ? 4 : P)), 0, s>>>(w, grp, a, (int)m, tm, tn, out);
    return hipGetLastError();
}

#define FRQ_MM(mt_, nt_, p_) \
    if (q.mt == mt_ && q.nt == nt_ && q.p == p_) return go<DT, mt_, nt_, p_, GM, GR>(w, grp, ntile, a, m, out, s);

// int4 / q4a: the whole set for K in whole chunks, fewer forms elsewhere
template <int DT, int GM, bool GR>
hipError_t packed(const MmWeight& w, const MmGroup& grp, unsigned ntile, const float* a, size_t m, float* out,
                  int cus, hipStream_t s) {
    if constexpr (GR || GM == 2) {
        static const Plan few[] = {{1, 2, 1}, {1, 2, 8}, {1, 1, 8}}, many[] = {{2, 2, 1}, {2, 2, 8}};
        const Plan q = mm_plan(m > TT ? many : few, m > TT ? 2 : 3, m, (size_t)w.n, (size_t)w.k, ntile, cus);
        FRQ_MM(1, 2, 1) FRQ_MM(1, 2, 8) FRQ_MM(1, 1, 8) FRQ_MM(2, 2, 1) FRQ_MM(2, 2, 8)
    } else if constexpr (GM == 1) {
        static const Plan all[] = {{1, 4, 1}, {1, 4, 4}, {1, 4, 8}, {1, 2, 8}, {1, 1, 4}, {1, 1, 8}};
        const Plan q = mm_plan(all, 6, m, (size_t)w.n, (size_t)w.k, 1, cus);
        FRQ_MM(1, 4, 1) FRQ_MM(1, 4, 4) FRQ_MM(1, 4, 8) FRQ_MM(1, 2, 8) FRQ_MM(1, 1, 4) FRQ_MM(1, 1, 8)
    } else {
        static const Plan all[] = {{1, 4, 1}, {1, 4, 4}, {1, 4, 8}, {1, 4, 16}, {2, 4, 1}, {2, 4, 2},
                                   {1, 2, 4}, {1, 2, 8}, {1, 1, 4}, {1, 1, 8}};
        const Plan q = mm_plan(all, 10, m, (size_t)w.n, (size_t)w.k, 1, cus);
        FRQ_MM(1, 4, 1) FRQ_MM(1, 4, 4) FRQ_MM(1, 4, 8) FRQ_MM(1, 4, 16) FRQ_MM(2, 4, 1) FRQ_MM(2, 4, 2)
        FRQ_MM(1, 2, 4) FRQ_MM(1, 2, 8) FRQ_MM(1, 1, 4) FRQ_MM(1, 1, 8)
    }
    return hipErrorInvalidValue;
}

// f16 / f32 banks: four adjacent columns a lane (one where there are fewer)
template <int DT, bool GR>
hipError_t columns(const MmWeight& w, const MmGroup& grp, unsigned ntile, const float* a, size_t m, float* out,
                   int cus, hipStream_t s) {
    constexpr int GM = 1;
    static const Plan one[] = {{2, 1, 1}, {2, 1, 8}}, few[] = {{1, 4, 1}, {1, 4, 8}}, many[] = {{2, 4, 1}, {2, 4, 8}};
    const Plan q = mm_plan(w.n < 4 ? one : m > TT ? many : few, 2, m, (size_t)w.n, (size_t)w.k, ntile, cus);
    FRQ_MM(2, 1, 1) FRQ_MM(2, 1, 8) FRQ_MM(1, 4, 1) FRQ_MM(1, 4, 8) FRQ_MM(2, 4, 1) FRQ_MM(2, 4, 8)
    return hipErrorInvalidValue;
}
#undef FRQ_MM

__global__ void zero_kernel(float* out, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = 0.0f;
}

template <bool GR>
hipError_t launch(int dt, const MmWeight& w, const MmGroup& grp, unsigned ntile, const float* a, size_t m,
                  float* out, int cus, hipStream_t s) {
    if (dt == FRQ_DT_F16) return columns<FRQ_DT_F16, GR>(w, grp, ntile, a, m, out, cus, s);
    if (dt == FRQ_DT_F32) return columns<FRQ_DT_F32, GR>(w, grp, ntile, a, m, out, cus, s);
    auto run = [&](auto d) {
        constexpr int DT = decltype(d)::value;
        return w.g % 32 ? packed<DT, 2, GR>(w, grp, ntile, a, m, out, cus, s)
               : w.k % 32 ? packed<DT, 1, GR>(w, grp, ntile, a, m, out, cus, s)
                          : packed<DT, 0, GR>(w, grp, ntile, a, m, out, cus, s);
    };
    if (dt == FRQ_DT_I4) return run(std::integral_constant<int, FRQ_DT_I4>{});
    if (dt == FRQ_DT_Q4A) return run(std::integral_constant<int, FRQ_DT_Q4A>{});
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_mm_f32(int dt, const MmWeight& w, const float* a, size_t m, float* out, int cus, hipStream_t s) {
    if (m == 0 || w.n == 0) return hipSuccess;
    if (w.k == 0) {
        zero_kernel<<<dim3(256), dim3(256), 0, s>>>(out, m * (size_t)w.n);
        return hipGetLastError();
    }
    if (m > (size_t)INT32_MAX - 64) return hipErrorInvalidValue;
    return launch<false>(dt, w, MmGroup{}, 1, a, m, out, cus, s);
}

hipError_t launch_mm_f32_group(int dt, const MmWeight& w, const MmGroup& grp, unsigned ntile, const float* a,
                               float* out, int cus, hipStream_t s) {
    if (ntile == 0 || w.n == 0 || w.k == 0) return hipSuccess;
    if (grp.rows < 1 || grp.rows > MM_GROUP_ROWS) return hipErrorInvalidValue;
    return launch<true>(dt, w, grp, ntile, a, (size_t)grp.rows, out, cus, s);
}

}  // namespace frq
