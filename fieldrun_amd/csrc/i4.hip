// i4.hip — group-wise int4 W4A32 linear (gfx950).
//
// Restates the I4 arm of Bundle::mm (/root/reference/src/bundle.rs:760-799):
//  M == 1 (767-776): out[j] = i4_dot(row j), which on x86 is i4_dot_avx2
//    (199-225): per group, 8 lane accumulators each an FMA chain over the
//    group's 8-nibble chunks, then hsum256 ((l0+l4)+(l2+l6))+((l1+l5)+(l3+l7))
//    (146-153), a scalar mul+add tail, then sum += scale[g] * gsum.
//  M > 1 (777-798): w[kk,j] = s4 * scale[j, kk/g] (f32) then a.dot(w),
//    matrixmultiply's sgemm: per output, k in blocks of MM_KC, each an FMA
//    chain from +0, the blocks added in order; the exact M > 1 kernels below
//    reproduce that order.
//
// Blocked shapes (g == 32, K % 32 == 0, 1 <= M <= 16) run on the int8
// MFMA.  At upload the nibbles are re-laid out so that the B operand of
// v_mfma_i32_16x16x32_i8 (16 weight rows x 32 k = one group) for four
// consecutive groups is one 16-byte load per lane and a wave load is 1 KB of
// contiguous memory; in registers each packed dword (8 nibbles) becomes two
// dwords of sign-extended int8 with 8 VALU operations.  The f32 activations
// of each (token, group) are written as X = round(a / s), s = max|a| /
// (127 * 2^16), |X| <= 127 * 2^16, split into three int8 digits
// X = d2*2^16 + d1*2^8 + d0; token m's digits are A rows 4m, 4m+1, 4m+2, so
// one MFMA gives the exact integer group dots of 4 tokens, and
//   gsum = s * (C2 * 2^16 + C1 * 2^8 + C0),   out += scale[j,g] * gsum.
// The 24-bit fixed point per group keeps the result within ~1e-7 of
// max|a| * sum|w| of the group (the reference's own sums differ between its
// M == 1 and M > 1 arms by more); a (token, group) with a non-finite or
// extreme activation takes the group sum in the reference arm's own order
// instead (i4_dot_avx2 for M == 1, the dequantised a * (s4 * scale) chain
// for M > 1).  The digits are written once per call by a small kernel
// (L2-resident, read by every row block); K is split across the waves of
// one workgroup and the parts are added in order through LDS: a split across
// workgroups would need device-scope fences, which on this part write back
// and invalidate the whole L2.
// Other shapes run i4_gemv_generic (M == 1, bit-identical to i4_dot_avx2)
// or, M > 1 in the exact order, the f32 matrix cores (mm_f32.hip).  Up to 16
// independent M == 1 rows (a batched decode) run i4_rows_mfma, of narrow
// outputs i4_rows_dpp.
#include "frq_internal.h"

namespace frq {

namespace {

__device__ __forceinline__ float s4f(uint32_t word, int nib) {
    return (float)((int)(word << (28 - 4 * nib)) >> 28);
}

// One group of 32 nibbles (4 words) against 32 activations, AVX2 order.
__device__ __forceinline__ float group_avx2(const uint4 w, const float* __restrict__ a) {
    float l[8];
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int q = 0; q < 8; ++q) l[q] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int q = 0; q < 8; ++q)
            l[q] = __builtin_fmaf(s4f(ws[c], q), a[8 * c + q], l[q]);
    const float q0 = l[0] + l[4], q1 = l[1] + l[5], q2 = l[2] + l[6], q3 = l[3] + l[7];
    return (q0 + q2) + (q1 + q3);
}

// Generic M == 1 (any K, g): one thread per output row, i4_dot_avx2 order.
__global__ void i4_gemv_generic(const uint8_t* __restrict__ packed,
                                const uint16_t* __restrict__ scale, int N,
                                int K, int g, const float* __restrict__ a,
                                float* __restrict__ out) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= N) return;
    const int rb = (K + 1) / 2, ng = (K + g - 1) / g;
    const uint8_t* prow = packed + (size_t)j * rb;
    auto nib = [&](int i) -> float {
        const uint8_t byte = prow[i >> 1];
        const int v = (i & 1) ? (byte >> 4) : (byte & 0x0F);
        return (float)((int)((uint32_t)v << 28) >> 28);
    };
    float sum = 0.0f;
    int kk = 0, gi = 0;
    while (kk < K) {
        const int hi = min(kk + g, K);
        float l[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        while (kk + 8 <= hi) {
            const int base = (kk / 2) * 2;
            for (int q = 0; q < 8; ++q) l[q] = __builtin_fmaf(nib(base + q), a[kk + q], l[q]);
            kk += 8;
        }
        const float q0 = l[0] + l[4], q1 = l[1] + l[5], q2 = l[2] + l[6], q3 = l[3] + l[7];
        float gs = (q0 + q2) + (q1 + q3);
        for (; kk < hi; ++kk) gs = gs + a[kk] * nib(kk);
        sum = sum + h2f(scale[(size_t)j * ng + gi]) * gs;
        ++gi;
    }
    out[j] = sum;
}

// M == 1 for any K and g (int4 in i4_dot_avx2's order, Q: q4a in
// q4a_dot_avx2's): a thread a (row, group), adjacent threads adjacent groups,
// the packed words read eight nibbles at a time at whatever byte they start,
// the activation row in LDS (36 floats a 32, so lanes a group apart meet
// other banks), and a lane a row adding its group terms in order.  Bound by
// the VALU at wide outputs and by the latency of a group's chain at narrow
// ones; a thread a row instead (i4_gemv_generic, kept up to K = 64 and where
// LDS does not hold the row and its terms) walks all of K alone: 184 x 6346
// 334 -> 8 us.  q4a keeps its own form at most sizes (launch_q4a).
__device__ __forceinline__ int any_pad(int k) { return k + (k >> 5) * 4; }

template <bool Q>
__global__ __launch_bounds__(256) void pack_gemv_any(const uint8_t* __restrict__ packed, size_t pitch,
                                                     const uint16_t* __restrict__ sc, const uint16_t* __restrict__ mn,
                                                     int ss, int N, int K, int g, int rb,
                                                     const float* __restrict__ a, float* __restrict__ out) {
    typedef uint32_t word_u __attribute__((aligned(1)));
    extern __shared__ float4 any_lds[];
    float* as = reinterpret_cast<float*>(any_lds);
    const int ng = (K + g - 1) / g, ngp = (ng + 3) & ~3;
    float* cg = as + (any_pad(K) + 7) / 4 * 4;
    const int r0 = blockIdx.x * rb, nr = min(rb, N - r0), items = nr * ng;
    for (int i = threadIdx.x; i < K; i += 256) as[any_pad(i)] = a[i];
    __syncthreads();
    for (int p = threadIdx.x; p < items; p += 256) {
        const int r = p / ng, gi = p - r * ng;
        const uint8_t* prow = packed + (size_t)(r0 + r) * pitch;
        int kk = gi * g;
        const int hi = min(kk + g, K);
        float l[8] = {0, 0, 0, 0, 0, 0, 0, 0}, m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (; kk + 8 <= hi; kk += 8) {
            const uint32_t w = *reinterpret_cast<const word_u*>(prow + (kk >> 1));  // from an even index on
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const float av = as[any_pad(kk + q)];
                const float wv = Q ? (float)((w >> (4 * q)) & 15u) : s4f(w, q);
                l[q] = __builtin_fmaf(wv, av, l[q]);
                if (Q) m[q] = m[q] + av;
            }
        }
        float qs = ((l[0] + l[4]) + (l[2] + l[6])) + ((l[1] + l[5]) + (l[3] + l[7]));
        float ms = ((m[0] + m[4]) + (m[2] + m[6])) + ((m[1] + m[5]) + (m[3] + m[7]));
        for (; kk < hi; ++kk) {
            const int v = (kk & 1) ? prow[kk >> 1] >> 4 : prow[kk >> 1] & 15;
            const float av = as[any_pad(kk)];
            qs = qs + av * (float)(Q ? v : (v ^ 8) - 8);
            if (Q) ms = ms + av;
        }
        const size_t at = ((size_t)(r0 + r) * ng + gi) * ss;
        cg[r * ngp + gi] = Q ? h2f(sc[at]) * qs + h2f(mn[at]) * ms : h2f(sc[at]) * qs;
    }
    __syncthreads();
    for (int r = threadIdx.x; r < nr; r += 256) out[r0 + r] = lds_seq_sum(cg + r * ngp, ng, 0.0f);
}

// M == 1 in i4_dot_avx2's order, fast: a group's term scale * gsum is
// independent of the others until the in-order sum, so a thread takes one
// (row, group) at a time (adjacent threads adjacent groups: the G4 16-byte
// nibble loads and the f16 scales arrive coalesced), the activations come
// from the workgroup's LDS copy (padded 4 floats per 32 against bank
// conflicts), and one lane per row adds its row's terms in order.  Needs
// K % 32 == 0 (16-byte aligned rows) and g == 32 G4.
template <int G4>
__global__ __launch_bounds__(256) void i4_gemv_terms(const uint8_t* __restrict__ packed,
                                                     const uint16_t* __restrict__ scale, int N, int K, int rb,
                                                     const float* __restrict__ a, float* __restrict__ out) {
    extern __shared__ float4 lds4[];
    float* cg = reinterpret_cast<float*>(lds4);
    constexpr int g = 32 * G4;
    const int ng = K / g, pitch = K / 2;
    const int r0 = blockIdx.x * rb;
    const int nr = min(rb, N - r0);
    const int items = nr * ng;
    const int ngp = (ng + 3) & ~3;  // row stride of the terms: 16-byte aligned rows
    float* as = cg + rb * ngp;
    for (int i = threadIdx.x; i < K / 4; i += 256)
        *reinterpret_cast<float4*>(as + (4 * i) / 32 * 36 + (4 * i) % 32) = reinterpret_cast<const float4*>(a)[i];
    __syncthreads();
    // the next item's nibbles and scale load while this one computes (the
    // index clamped to the last item, so every load is unconditional)
    auto fetch = [&](int p, uint4 (&w)[G4], float& sc) {
        const int r = p / ng, gi = p - r * ng;
        const uint8_t* pg = packed + (size_t)(r0 + r) * pitch + (size_t)gi * 16 * G4;
#pragma unroll
        for (int h = 0; h < G4; ++h) w[h] = *reinterpret_cast<const uint4*>(pg + 16 * h);
        sc = h2f(scale[(size_t)(r0 + r) * ng + gi]);
    };
    if (threadIdx.x < items) {
        uint4 wn[G4];
        float sn;
        fetch(threadIdx.x, wn, sn);
        for (int p = threadIdx.x; p < items; p += 256) {
            uint4 wc[G4];
#pragma unroll
            for (int h = 0; h < G4; ++h) wc[h] = wn[h];
            const float sc = sn;
            fetch(min(p + 256, items - 1), wn, sn);
            const int rr = p / ng, gi = p - rr * ng;
            float l[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int h = 0; h < G4; ++h) {
                const uint32_t ws[4] = {wc[h].x, wc[h].y, wc[h].z, wc[h].w};
                const float* ab = as + (gi * g + 32 * h) / 32 * 36;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float4 a0 = *reinterpret_cast<const float4*>(ab + 8 * c);
                    const float4 a1 = *reinterpret_cast<const float4*>(ab + 8 * c + 4);
                    const float av[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
                    for (int q = 0; q < 8; ++q) l[q] = __builtin_fmaf(s4f(ws[c], q), av[q], l[q]);
                }
            }
            const float q0 = l[0] + l[4], q1 = l[1] + l[5], q2 = l[2] + l[6], q3 = l[3] + l[7];
            cg[rr * ngp + gi] = sc * ((q0 + q2) + (q1 + q3));
        }
    }
    __syncthreads();
    for (int r = threadIdx.x; r < nr; r += 256) out[r0 + r] = lds_seq_sum(cg + r * ngp, ng, 0.0f);
}

// M == 1 in i4_dot_avx2's order, streamed: a persistent grid of about one
// workgroup per CU, each owning a contiguous range of R rows, so its
// R * ng items (row, group) are one contiguous run of the packed weights
// and of the scales.  A thread takes items tid + NT i; every one of its
// nibble and scale loads is issued up front, right after the direct-to-LDS
// loads of the activation row (32-float units padded to 36 against bank
// conflicts), and items are consumed in issue order as the loads land.  A
// group's term scale * gsum goes to LDS; after one barrier a lane per row
// adds its row's terms in order.
//   Nibbles to f32: (x & 0x000F000F) ^ 0x64086408 puts (q ^ 8) of nibbles
// 0 and 4 of a word under the f16 exponent of 1024 (one bit operation),
// a packed f16 add of -1032 leaves the exact signed values q - 16 [q >= 8]
// in both halves, and v_fma_mix_f32 takes either half as an exactly
// widened f32 operand of the FMA: the products and their rounding are
// those of fma(float(s4), a, acc).
__device__ __forceinline__ void nib_f16x2(uint32_t x, uint32_t (&d)[4]) {
    d[0] = (x & 0x000F000Fu) ^ 0x64086408u;
    d[1] = ((x >> 4) & 0x000F000Fu) ^ 0x64086408u;
    d[2] = ((x >> 8) & 0x000F000Fu) ^ 0x64086408u;
    d[3] = ((x >> 12) & 0x000F000Fu) ^ 0x64086408u;
}

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// One 32-nibble unit (4 words) against 32 activations into the eight AVX2
// lane chains l[q] (element 8c + q is nibble q of word c).
__device__ __forceinline__ void unit_fma(const uint4 w, const float* __restrict__ ab, float (&l)[8]) {
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
    const f16x2 off = {(_Float16)-1032.0f, (_Float16)-1032.0f};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        uint32_t d[4];
        nib_f16x2(ws[c], d);
        f16x2 h[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) h[j] = __builtin_bit_cast(f16x2, d[j]) + off;
        const float4 a0 = *reinterpret_cast<const float4*>(ab + 8 * c);
        const float4 a1 = *reinterpret_cast<const float4*>(ab + 8 * c + 4);
        const float av[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
        for (int q = 0; q < 8; ++q) l[q] = __builtin_fmaf((float)(q < 4 ? h[q].x : h[q - 4].y), av[q], l[q]);
    }
}

// LDS bytes of the staged activation row: 16-byte slots of 9 a unit (8 of
// data, 1 of padding), whole 1 KB loads of 64 slots.
__host__ __device__ inline size_t i4_stream_as_bytes(int K) { return (size_t)(K / 32 * 9 + 63) / 64 * 1024; }

template <int G4, int IPT, int NT>
__global__ __launch_bounds__(NT) void i4_m1_stream(const uint8_t* __restrict__ packed,
                                                    const uint16_t* __restrict__ scale, int N, int K, int R,
                                                    const float* __restrict__ a, float* __restrict__ out) {
    extern __shared__ float4 lds4[];
    constexpr int g = 32 * G4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ng = K / g, nu = K / 32;
    constexpr int NW = NT / 64;
    const int r0 = blockIdx.x * R;
    if (r0 >= N) return;  // workgroup-uniform, before any barrier
    const int nr = min(R, N - r0), items = nr * ng;
    const int ngp = (ng + 3) & ~3;  // terms row stride: 16-byte aligned rows
    char* lds = reinterpret_cast<char*>(lds4);
    const float* as = reinterpret_cast<const float*>(lds);                // unit u at 36 u floats
    float* terms = reinterpret_cast<float*>(lds + i4_stream_as_bytes(K));  // nr rows of ngp floats, 1 dummy
    const float4* a4 = reinterpret_cast<const float4*>(a);
    // 1. the activation row straight into LDS (L2-resident, shared by every
    //    workgroup): load q of the workgroup fills slots 64 q .. 64 q + 63,
    //    slot k = 9 u + j holding float4 8 u + j (j == 8: padding, a dummy)
    const int nslot = nu * 9, nld = (nslot + 63) / 64;
    for (int q = wave; q < nld; q += NW) {
        const int k = q * 64 + lane, u = k / 9, j = k - 9 * u;
        dma16_lds(u < nu && j < 8 ? a4 + 8 * u + j : a4, lds + (size_t)q * 1024);
    }
    __builtin_amdgcn_sched_barrier(0);
    // 2. every item's nibbles and scale (indices clamped: unconditional)
    const uint4* wp = reinterpret_cast<const uint4*>(packed + (size_t)r0 * ng * 16 * G4);
    const uint16_t* sp = scale + (size_t)r0 * ng;
    uint4 w[IPT][G4];
    uint16_t sc[IPT];
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
        const int p = min(tid + NT * i, items - 1);
#pragma unroll
        for (int h = 0; h < G4; ++h) w[i][h] = wp[(size_t)p * G4 + h];
        sc[i] = sp[p];
    }
    asm volatile("" ::: "memory");  // no load sinks below this point
    __builtin_amdgcn_sched_barrier(0);
    // 3. the row's loads were issued before these IPT (G4 + 1): once at most
    //    that many are outstanding, this wave's share of the row is in LDS,
    //    and after the barrier every wave's is
    wait_vmcnt<IPT * (G4 + 1)>();
    __builtin_amdgcn_s_barrier();
    // item p = tid + NT i: row r = p / ng and group gi = p % ng, kept
    // incrementally; every item is computed (past the end: a copy of the
    // last, stored to a dummy slot)
    const int q256 = NT / ng, m256 = NT % ng;
    int r = tid / ng, gi = tid % ng;
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
        const int p = tid + NT * i;
        const int gc = p < items ? gi : ng - 1;
        float l[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int h = 0; h < G4; ++h) unit_fma(w[i][h], as + (gc * G4 + h) * 36, l);
        const float q0 = l[0] + l[4], q1 = l[1] + l[5], q2 = l[2] + l[6], q3 = l[3] + l[7];
        const float t = h2f(sc[i]) * ((q0 + q2) + (q1 + q3));
        terms[p < items ? r * ngp + gi : nr * ngp] = t;  // past the end: a dummy slot (the compute
                                                         // stays live, so its loads stay hoisted)
        r += q256;
        gi += m256;
        if (gi >= ng) {
            gi -= ng;
            ++r;
        }
    }
    __syncthreads();
    for (int rr = tid; rr < nr; rr += NT) out[r0 + rr] = lds_seq_sum(terms + rr * ngp, ng, 0.0f);
}

constexpr int ROWS_GW = 4;  // groups a wave of i4_rows_mfma takes a round, at most

// The activation layout of i4_rows_mfma and i4_rows_dpp: the 16 token rows interleaved by
// k-quads, a4[64 (k / 4) + 4 t + k % 4] = a[t][k] (rows t >= M zero), so
// that 16 token lanes read 256 contiguous bytes a load.
__global__ void rows_to_a4_kernel(const float* __restrict__ a, int M, int K, float* __restrict__ a4) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;  // float4 i of a4: k-quad i / 16, token i % 16
    const int kq = i >> 4, t = i & 15;
    if (kq >= K / 4) return;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (t < M) v = *reinterpret_cast<const float4*>(a + (size_t)t * K + 4 * kq);
    reinterpret_cast<float4*>(a4)[i] = v;
}

// 16 FMAs of one weight register v of a 32-unit into lane chains
// l[4 v .. 4 v + 3]: v_fmac_f32_dpp with row_newbcast:n gives each token
// lane of a 16-lane DPP row the weight held by lane n of that row.  Lane n
// holds element e = 8 (n & 3) + (n >> 2) + 4 v, which is nibble
// (n >> 2) + 4 v of word n & 3 (chain q = e & 7, chunk c = e >> 3), and its
// product takes av[e]; the FMAs go c-major so each chain advances in chunk
// order.  START begins the chains: chunk 0 is a v_mul_f32_dpp, which
// differs from fma(w, a, +0) only in giving -0 for a -0 product; a chain
// is exact otherwise, the lane sums of i4_dot_avx2 then differ at most in
// the sign of a zero, and so does a group term, which the running sum from
// +0 absorbs (+0 + -0 == +0): the row sums are bit-identical.  The s_nop
// gives the two wait states a DPP read needs after the VALU write of w,
// which the compiler does not see inside the asm.
#define FRQ_DPPF(op, acc, n, src) #op "_f32_dpp %" #acc ", %4, %" #src " row_newbcast:" #n " row_mask:0xf bank_mask:0xf\n\t"
#define FRQ_DPP_C0(op) FRQ_DPPF(op, 0, 0, 5) FRQ_DPPF(op, 1, 4, 9) FRQ_DPPF(op, 2, 8, 13) FRQ_DPPF(op, 3, 12, 17)
#define FRQ_DPP_C123                                                                                          \
    FRQ_DPPF(v_fmac, 0, 1, 6) FRQ_DPPF(v_fmac, 1, 5, 10) FRQ_DPPF(v_fmac, 2, 9, 14) FRQ_DPPF(v_fmac, 3, 13, 18) \
    FRQ_DPPF(v_fmac, 0, 2, 7) FRQ_DPPF(v_fmac, 1, 6, 11) FRQ_DPPF(v_fmac, 2, 10, 15)                            \
    FRQ_DPPF(v_fmac, 3, 14, 19) FRQ_DPPF(v_fmac, 0, 3, 8) FRQ_DPPF(v_fmac, 1, 7, 12)                            \
    FRQ_DPPF(v_fmac, 2, 11, 16) FRQ_DPPF(v_fmac, 3, 15, 20)
#define FRQ_DPP_OPS(V)                                                                              \
    : "+v"(l[4 * V]), "+v"(l[4 * V + 1]), "+v"(l[4 * V + 2]), "+v"(l[4 * V + 3])                    \
    : "v"(w), "v"(av[4 * V]), "v"(av[8 + 4 * V]), "v"(av[16 + 4 * V]), "v"(av[24 + 4 * V]),         \
      "v"(av[1 + 4 * V]), "v"(av[9 + 4 * V]), "v"(av[17 + 4 * V]), "v"(av[25 + 4 * V]),             \
      "v"(av[2 + 4 * V]), "v"(av[10 + 4 * V]), "v"(av[18 + 4 * V]), "v"(av[26 + 4 * V]),            \
      "v"(av[3 + 4 * V]), "v"(av[11 + 4 * V]), "v"(av[19 + 4 * V]), "v"(av[27 + 4 * V])
template <int V, bool START>
__device__ __forceinline__ void dpp_fma16(float (&l)[8], float w, const float (&av)[32]) {
    if constexpr (START)
        asm("s_nop 1\n\t" FRQ_DPP_C0(v_mul) FRQ_DPP_C123 FRQ_DPP_OPS(V));
    else
        asm("s_nop 1\n\t" FRQ_DPP_C0(v_fmac) FRQ_DPP_C123 FRQ_DPP_OPS(V));
}
#undef FRQ_DPP_OPS
#undef FRQ_DPP_C123
#undef FRQ_DPP_C0
#undef FRQ_DPPF

// M independent rows (M <= 16), each in the M == 1 order (i4_dot_avx2),
// with the weights broadcast across tokens: lane 16 d + t of a wave is token
// t in DPP row d, and the workgroup's ND = 4 NW DPP rows D = 4 wave + d take
// a slice of 2 ND groups in two rounds (groups 2 ND s + ND i + D, i = 0, 1).
// A lane holds its token's 32 activations of the current 32-unit (read from
// the a4 layout) and, for each of the workgroup's R weight rows, the packed
// word t & 3 of the unit, whose nibbles t >> 2 and 4 + (t >> 2) become its
// two f32 weight registers (dpp_fma16): each activation register serves R
// rows and each weight register 16 tokens.  A group's term scale * gsum goes
// to LDS (+0 for the groups past the end, which the running sum absorbs
// exactly: it is never -0); after the slice's one barrier the lane of (row,
// token) adds the slice's 2 ND terms to its running sum in group order (two
// term buffers, so the next slice's writes never meet this slice's reads).
// Activations and scales are loaded one step ahead, weights two.  Needs
// K % (32 G4) == 0.  Bound by the DPP FMAs' issue.  It takes the narrow
// outputs, where the 16-row tiles of i4_rows_mfma leave most CUs idle and
// these 4-row ones do not; 16 rows, us here / there: 896 x 4864 12.3 / 14.8,
// 512 x 9216 (groups of 64) 15.6 / 22.6, 512 x 2304 8.5 / 9.9; from a second
// workgroup a CU on it loses (1536 x 2304 10.6 / 10.0, 2304 x 4864 20.3 /
// 14.8).
template <int G4, int NW>
__global__ __launch_bounds__(64 * NW) void i4_rows_dpp(const uint8_t* __restrict__ packed,
                                                       const uint16_t* __restrict__ scale, int N, int K,
                                                       const float* __restrict__ a4, int M, float* __restrict__ out) {
    static_assert(G4 == 1 || G4 == 2, "a group is one or two 32-units");
    constexpr int R = 4;                       // weight rows a workgroup
    constexpr int ND = 4 * NW;                 // DPP rows
    constexpr int GPS = 3 - G4;                // groups a DPP row takes a slice (two steps a slice)
    constexpr int SG = ND * GPS;               // groups a slice
    constexpr int TS = SG + 1;                 // term row stride (floats), odd: conflict-free reads
    constexpr int L = (16 * R + NW - 1) / NW;  // serial lanes a wave
    static_assert(L <= 64, "one (row, token) pair a lane");
    __shared__ float tb[2][16 * R][TS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t = lane & 15, D = 4 * wave + (lane >> 4);
    const int ng = K / (32 * G4), r0 = blockIdx.x * R;
    const int nst = (ng + SG - 1) / SG * 2;  // unit steps: two a slice
    const int sh = 4 * (t >> 2);
    const size_t pitch = (size_t)K / 2;
    const uint8_t* wrow[R];
    const uint16_t* srow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t row = (size_t)min(r0 + r, N - 1);  // clamped: loads stay unconditional
        wrow[r] = packed + row * pitch;
        srow[r] = scale + row * ng;
    }
    const float* at = a4 + 4 * t;
    // serial lane: pair p = wave L + lane -> (row p >> 4, token p & 15)
    const int p = wave * L + lane;
    const bool ser = lane < L && p < 16 * R;
    float sum = 0.0f;
    struct WB {
        uint32_t w[R];
    };
    struct AB {
        float4 a[8];
        uint32_t sc[R];
    };
    // step j: slice j / 2; with G4 == 1 round j % 2 of the slice, with G4 == 2
    // unit j % 2 of the DPP row's one group
    auto group_of = [&](int j) { return (j >> 1) * SG + (G4 == 1 ? (j & 1) * ND : 0) + D; };
    auto unit_of = [&](int j, int gi) { return min(gi, ng - 1) * G4 + (G4 == 2 ? (j & 1) : 0); };
    auto load_w = [&](int j, WB& b) {
        const uint32_t wo = (uint32_t)unit_of(j, group_of(j)) * 16 + 4 * (t & 3);
#pragma unroll
        for (int r = 0; r < R; ++r) b.w[r] = *reinterpret_cast<const uint32_t*>(wrow[r] + wo);
    };
    auto load_a = [&](int j, AB& b) {
        const int gi = group_of(j);
        const float* ap = at + (size_t)unit_of(j, gi) * 512;
#pragma unroll
        for (int i = 0; i < 8; ++i) b.a[i] = *reinterpret_cast<const float4*>(ap + 64 * i);
        const uint32_t so = 2 * (uint32_t)min(gi, ng - 1);
#pragma unroll
        for (int r = 0; r < R; ++r)
            b.sc[r] = *reinterpret_cast<const uint16_t*>(reinterpret_cast<const uint8_t*>(srow[r]) + so);
    };
    float l[R][8];  // each group's chains start with a product (dpp_fma16<., true>)
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int q = 0; q < 8; ++q) l[r][q] = 0.0f;  // defined inputs for the first asm
    // ODD: the slice's second step, which ends every chain and the slice
    auto step = [&](auto odd, int j, const WB& wb, const AB& ab) {
        constexpr bool O = decltype(odd)::value;
        constexpr bool START = G4 == 1 || !O;
        float av[32];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            av[4 * i] = ab.a[i].x;
            av[4 * i + 1] = ab.a[i].y;
            av[4 * i + 2] = ab.a[i].z;
            av[4 * i + 3] = ab.a[i].w;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float w0 = (float)(int)__builtin_amdgcn_sbfe((int)wb.w[r], sh, 4);
            const float w1 = (float)(int)__builtin_amdgcn_sbfe((int)wb.w[r], sh + 16, 4);
            dpp_fma16<0, START>(l[r], w0, av);
            dpp_fma16<1, START>(l[r], w1, av);
        }
        if constexpr (G4 == 2 && !O) return;  // the group goes on in the odd step
        float(&tbs)[16 * R][TS] = tb[(j >> 1) & 1];
        const int gi = group_of(j);
        const int col = gi - (j >> 1) * SG;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float q0 = l[r][0] + l[r][4], q1 = l[r][1] + l[r][5], q2 = l[r][2] + l[r][6],
                        q3 = l[r][3] + l[r][7];
            const float term = h2f((uint16_t)ab.sc[r]) * ((q0 + q2) + (q1 + q3));
            tbs[r * 16 + t][col] = gi < ng ? term : 0.0f;
        }
        if constexpr (!O) return;
        __syncthreads();
        if (ser) {
            float v[SG];
#pragma unroll
            for (int i = 0; i < SG; ++i) v[i] = tbs[p][i];
#pragma unroll
            for (int i = 0; i < SG; ++i) sum = sum + v[i];
        }
    };
    using T = std::true_type;
    using F = std::false_type;
    // The loads are unconditional (past the end: the last step again), so
    // the wait for a step's data never covers a later one's, and fenced so
    // that they issue before the step they run ahead of.
    auto issued = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    WB wc, wn, w2;
    AB a0, a1;
    load_w(0, wc);
    load_a(0, a0);
    load_w(1, wn);
    for (int j = 0; j < nst; j += 2) {
        load_w(min(j + 2, nst - 1), w2);
        load_a(j + 1, a1);
        issued();
        step(F{}, j, wc, a0);
        load_w(min(j + 3, nst - 1), wc);
        load_a(min(j + 2, nst - 1), a0);
        issued();
        step(T{}, j + 1, wn, a1);
        wn = wc;
        wc = w2;
    }
    if (ser) {
        const int pr = p >> 4, pt = p & 15;
        if (pt < M && r0 + pr < N) out[(size_t)pt * N + r0 + pr] = sum;
    }
}

// M independent rows (M <= 16), each in the M == 1 order (i4_dot_avx2), on
// the f32 matrix cores: v_mfma_f32_16x16x4_f32 advances an output by four
// FMAs in ascending lane group, so with lane group h feeding k = 8 h + q of a
// 32-unit, MFMA q is the lane chain l[q] of 16 tokens x 16 weight rows (from
// +0; a 64-long group goes on in the same accumulators).  A lane's weights of
// a unit are one packed word, its activations two float4 of the a4 layout.
// The lane sums and scale give a group's term, which goes to LDS; after the
// barrier that ends a round of 8 gw groups (gw <= 4 a wave) a thread a (row,
// token) adds the round's terms in group order, two term buffers, so the next
// round's writes never meet these reads.  Loads run
// two units ahead.  Bound by the f32 MFMAs (256 of about 460 clocks a unit)
// and the VALU that forms the weights and the terms, on the same pipe; the
// DPP-broadcast FMAs this replaced issue at half the plain rate.  16 rows with
// the a4 copy, us before / now: 18432 x 2304 39.9 / 31.7, 2304 x 9216 31.7 /
// 24.9, 4096 x 2304 14.5 / 10.0, 2304 x 2048 11.2 / 9.2, 512 x 512 6.1 / 6.1;
// 3 rows cost the same.
template <int G4>
__global__ __launch_bounds__(512, 4) void i4_rows_mfma(const uint8_t* __restrict__ packed,
                                                       const uint16_t* __restrict__ scale, int N, int K, int gw,
                                                       const float* __restrict__ a4, int M, float* __restrict__ out) {
    static_assert(G4 == 1 || G4 == 2, "a group is one or two 32-units");
    typedef float f4v __attribute__((ext_vector_type(4)));
    constexpr int P = 8;
    __shared__ float tb[2][P * ROWS_GW][256];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lh = lane >> 4;
    const int ng = K / (32 * G4), R = P * gw, n0 = blockIdx.x * 16;
    const size_t row = (size_t)min(n0 + li, N - 1);  // clamped: loads stay unconditional
    const uint8_t* wp = packed + row * ((size_t)K / 2) + 4 * lh;
    const uint16_t* sp = scale + row * ng;
    const float* ap = a4 + 4 * li + 128 * lh;
    // unit j of the wave: units j % G4 of its groups, gw adjacent ones a round
    // (past the end the last group again)
    const int rounds = (ng + R - 1) / R, nj = rounds * gw * G4;
    int lg = wave * gw, lp = 0;  // the group to load next, its place in the round
    auto unit = [&](int s) { return (size_t)(min(lg, ng - 1) * G4 + s); };
    uint32_t w[2];
    uint16_t sc[2];
    f4v a[2][2];
    auto load_w = [&](int u) {
        w[u] = *reinterpret_cast<const uint32_t*>(wp + unit(G4 == 2 ? u : 0) * 16);
        sc[u] = sp[min(lg, ng - 1)];
    };
    auto load_a = [&](int u) {  // and on
        const float* q = ap + unit(G4 == 2 ? u : 0) * 512;
        a[u][0] = *reinterpret_cast<const f4v*>(q);
        a[u][1] = *reinterpret_cast<const f4v*>(q + 64);
        if (G4 == 2 && u == 0) return;
        const bool on = lp + 1 < gw;
        lg += on ? 1 : 1 + R - gw;
        lp = on ? lp + 1 : 0;
    };
#pragma unroll
    for (int u = 0; u < 2; ++u) {  // in the loop's order, so its waits count the same loads
        load_w(u);
        __builtin_amdgcn_sched_barrier(0);
        load_a(u);
        __builtin_amdgcn_sched_barrier(0);
    }
    float sum = 0.0f;  // tid < 256: token 4 (lane / 16) + tid / 64, row lane % 16
    int r = 0, i = 0;
    f4v l[8];
    auto step = [&](auto uc) {
        constexpr int u = decltype(uc)::value, s = G4 == 2 ? u : 0;
        const int g = r * R + wave * gw + i;
        float wv[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) wv[q] = (float)(int)__builtin_amdgcn_sbfe((int)w[u], 4 * q, 4);
        const float sv = h2f(sc[u]);
        load_w(u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const f4v c = s == 0 ? f4v{0.0f, 0.0f, 0.0f, 0.0f} : l[q];
            l[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][q / 4][q % 4], wv[q], c, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_a(u);
        if (s < G4 - 1) return;
        float(&t)[P * ROWS_GW][256] = tb[r & 1];
        if (g < ng) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float q0 = l[0][v] + l[4][v], q1 = l[1][v] + l[5][v], q2 = l[2][v] + l[6][v],
                            q3 = l[3][v] + l[7][v];
                t[wave * gw + i][64 * v + lane] = sv * ((q0 + q2) + (q1 + q3));
            }
        }
        if (++i < gw) return;
        __syncthreads();  // every wave ends the round here
        if (wave < 4) {
            const int n = min(R, ng - r * R);
            int j = 0;
            for (; j + 8 <= n; j += 8) {
                float x[8];
#pragma unroll
                for (int v = 0; v < 8; ++v) x[v] = t[j + v][tid];
#pragma unroll
                for (int v = 0; v < 8; ++v) sum = sum + x[v];
            }
            for (; j < n; ++j) sum = sum + t[j][tid];
        }
        i = 0;
        ++r;
    };
    for (int j = 0; j < nj; j += 2) {
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});  // past the last unit: no term (g >= ng), in every wave
    }
    if (wave < 4) {
        const int tok = 4 * lh + wave, n = n0 + li;
        if (tok < M && n < N) out[(size_t)tok * N + n] = sum;
    }
}

constexpr float XMAX4 = 8323072.0f;  // 127 * 2^16

// Sign-extend the 8 nibbles of w (k = 0..7, low nibble first) into int8:
// lo = bytes for k = 0,2,4,6, hi = k = 1,3,5,7.  Per byte, with y = x ^ 8:
// ((y + 0x78) ^ 0x80) == x as a signed nibble, and y + 0x78 <= 0x87 never
// carries into the next byte.
__device__ __forceinline__ void nib_unpack(uint32_t w, uint32_t& lo, uint32_t& hi) {
    const uint32_t y = w ^ 0x88888888u;
    lo = ((y & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
    hi = (((y >> 4) & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
}

// Activation digits, four threads (chunks q = 0..3 of 8 k) per (token m <
// 4*MT4, group g < 4*ng4).  The A operand of token group tg = m/4 and group
// g = 4*g4 + gi is, for lane l, the 8 bytes at ((tg*ng4 + g4)*64 + l)*32 +
// 8*gi (a lane's 4 groups of a quad are one 32-byte run); lane
// 16q + 4(m%4) + d holds digit d of token m at k = 8q + {0,2,4,6,1,3,5,7}
// (the nibble order of the unpacked weights), lane 16q + 4(m%4) + 3 is zero.
// so[(m*ng4 + g4)*4 + gi] = s, -1 for a group that takes the exact path, 0
// for padding tokens and groups.
__global__ void i4_digits_kernel(const float* __restrict__ a, int M, int Mp, int K, int ng4,
                                 uint8_t* __restrict__ adig, float* __restrict__ so_out) {
    const int ng = K / 32, ngp = 4 * ng4;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    const int mg = idx >> 2, q = idx & 3;  // the 4 threads of (m, g) are adjacent lanes
    const bool act = mg < Mp * ngp;
    const int m = act ? mg / ngp : 0, g = act ? mg % ngp : 0;
    const bool real = act && m < M && g < ng;
    float v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (real) {
        const float4* ap = reinterpret_cast<const float4*>(a + (size_t)m * K + (size_t)g * 32 + 8 * q);
        const float4 x0 = ap[0], x1 = ap[1];
        v[0] = x0.x; v[1] = x0.y; v[2] = x0.z; v[3] = x0.w;
        v[4] = x1.x; v[5] = x1.y; v[6] = x1.z; v[7] = x1.w;
    }
    float mx = 0.0f;
    int nf = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        nf |= !(fabsf(v[k]) <= 3.0e38f);
        mx = fmaxf(mx, fabsf(v[k]));
    }
    mx = fmaxf(mx, __shfl_xor(mx, 1, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 2, 64));
    nf |= __shfl_xor(nf, 1, 64);
    nf |= __shfl_xor(nf, 2, 64);
    if (!act) return;
    // |group sum| <= 32 * 8 * mx stays finite for s <= 1e28
    const float s = mx > 0.0f ? mx / XMAX4 : 1.0f;
    const bool ok = real && !nf && s >= 1.0e-30f && s <= 1.0e28f;
    uint32_t dw[3][2] = {{0, 0}, {0, 0}, {0, 0}};
    if (ok) {
        const float r = 1.0f / s;  // any rounding of a / s keeps |a - s X| <= ~s/2
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float xf = rintf(v[j] * r);
            xf = fminf(fmaxf(xf, -XMAX4), XMAX4);
            const int X = (int)xf;
            const int d0 = (int)(int8_t)(X & 0xFF);
            const int X1 = (X - d0) >> 8;
            const int d1 = (int)(int8_t)(X1 & 0xFF);
            const int d2 = (X1 - d1) >> 8;
            const int p = (j & 1) ? 4 + (j >> 1) : (j >> 1);  // byte within the lane's 8
            const int wsel = p >> 2, sh = 8 * (p & 3);
            dw[0][wsel] |= (uint32_t)(d2 & 0xFF) << sh;
            dw[1][wsel] |= (uint32_t)(d1 & 0xFF) << sh;
            dw[2][wsel] |= (uint32_t)(d0 & 0xFF) << sh;
        }
    }
    const int g4 = g >> 2, gi = g & 3;
    uint8_t* blk = adig + ((size_t)(m >> 2) * ng4 + g4) * 64 * 32 + 8 * gi;
    const int l0 = 16 * q + 4 * (m & 3);
#pragma unroll
    for (int d = 0; d < 3; ++d)
        *reinterpret_cast<uint2*>(blk + (l0 + d) * 32) = make_uint2(dw[d][0], dw[d][1]);
    *reinterpret_cast<uint2*>(blk + (l0 + 3) * 32) = make_uint2(0u, 0u);
    if (q == 0) so_out[((size_t)m * ng4 + g4) * 4 + gi] = real ? (ok ? s : -1.0f) : 0.0f;
}

// acc plus one group of a (token, weight row) in the reference arm's own
// order, for activations the digits cannot carry (non-finite or extreme):
// M == 1: scale * i4_dot_avx2 group sum; M > 1: a * (s4 * scale), k ascending.
template <bool INL = false>
__device__ __attribute__((noinline)) float exact_group(float acc, const uint8_t* wrow, const float* ag,
                                                       float sc, bool m1);
template <>
__device__ __attribute__((noinline)) float exact_group<false>(float acc, const uint8_t* wrow, const float* ag,
                                                              float sc, bool m1);
__device__ __forceinline__ float exact_group_body(float acc, const uint8_t* wrow, const float* ag,
                                                  float sc, bool m1) {
    const uint4 wr = *reinterpret_cast<const uint4*>(wrow);
    if (m1) return acc + sc * group_avx2(wr, ag);
    const uint32_t ws[4] = {wr.x, wr.y, wr.z, wr.w};
    float e = 0.0f;
    for (int k = 0; k < 32; ++k) e = __builtin_fmaf(ag[k], s4f(ws[k >> 3], k & 7) * sc, e);
    return acc + e;
}
template <>
__device__ __attribute__((noinline)) float exact_group<false>(float acc, const uint8_t* wrow, const float* ag,
                                                              float sc, bool m1) {
    return exact_group_body(acc, wrow, ag, sc, m1);
}

// Dot of one group for the MT4 token groups of a wave, acc += scale * gsum.
template <int MT4, bool INL = false>
__device__ __forceinline__ void group_mfma(float (&acc)[MT4], uint32_t wd, float sc, const long* aop,
                                           const float* so, int g, int row, int N, int K, int M,
                                           const uint8_t* __restrict__ raw, const float* __restrict__ a,
                                           int ml) {
    uint32_t lo, hi;
    nib_unpack(wd, lo, hi);
    const long bop = (long)(((unsigned long long)hi << 32) | lo);
#pragma unroll
    for (int t = 0; t < MT4; ++t) {
        const v4i cr = __builtin_amdgcn_mfma_i32_16x16x32_i8(aop[t], bop, v4i{0, 0, 0, 0}, 0, 0, 0);
        if (__builtin_amdgcn_ballot_w64(so[t] < 0.0f)) {  // wave-uniform, rare
            if (so[t] < 0.0f && row < N) {
                const uint8_t* wr = raw + (size_t)row * (K / 2) + (size_t)g * 16;
                const float* ag = a + (size_t)(4 * t + ml) * K + (size_t)g * 32;
                if constexpr (INL) acc[t] = exact_group_body(acc[t], wr, ag, sc, M == 1);
                else acc[t] = exact_group<false>(acc[t], wr, ag, sc, M == 1);
                continue;
            }
        }
        const float gs = so[t] * ((float)cr[0] * 65536.0f + ((float)cr[1] * 256.0f + (float)cr[2]));
        acc[t] = acc[t] + sc * gs;
    }
}

// int4 x f32 on the int8 MFMA.  A workgroup of KS waves covers 16-row
// blocks rb = blockIdx.x, + gridDim.x, ...; wave ks owns the ks-th part (at
// most GQ group quads) of K.  It loads that part's activation operands once
// (only the lanes whose A rows carry a token's digit; with M == 1 the digit
// scales are wave-uniform) and keeps them in registers; per block it issues
// all of the part's weight loads at once.  The KS partial sums of a block are
// added in part order through LDS.  MT4 = token groups of 4 (M <= 4 * MT4).
template <int MT4, int KS, int GQ, bool M1>
__global__ __launch_bounds__(64 * KS) void i4_mfma_kernel(
    const uint8_t* __restrict__ q4m, const uint16_t* __restrict__ s4m,
    const uint8_t* __restrict__ raw, const float* __restrict__ a,
    const uint8_t* __restrict__ adig, const float* __restrict__ sog, int M, int K,
    int N, int ng4, float* __restrict__ out) {
    __shared__ float red[2][KS][MT4][64];
    const int lane = threadIdx.x & 63;
    const int ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nrb = (N + 15) / 16, ng = K / 32;
    const int q0 = (int)((long)ng4 * ks / KS), q1 = (int)((long)ng4 * (ks + 1) / KS);
    const int col = lane & 15, ml = M1 ? 0 : lane >> 4;
    // resident activation operands and digit scales of this part
    long ao[GQ][4][MT4];
    float sv[GQ][4][MT4];
#pragma unroll
    for (int i = 0; i < GQ; ++i)
#pragma unroll
        for (int t = 0; t < MT4; ++t) {
            const int mt = M1 ? 1 : min(M - 4 * t, 4);  // tokens in this token group
            const bool need = ((col >> 2) < mt) && ((col & 3) < 3) && q0 + i < q1;
            uint4 h0 = make_uint4(0, 0, 0, 0), h1 = make_uint4(0, 0, 0, 0);
            if (need) {
                const uint4* ap = reinterpret_cast<const uint4*>(adig + (((size_t)t * ng4 + q0 + i) * 64 + lane) * 32);
                h0 = ap[0];
                h1 = ap[1];
            }
            ao[i][0][t] = (long)(((unsigned long long)h0.y << 32) | h0.x);
            ao[i][1][t] = (long)(((unsigned long long)h0.w << 32) | h0.z);
            ao[i][2][t] = (long)(((unsigned long long)h1.y << 32) | h1.x);
            ao[i][3][t] = (long)(((unsigned long long)h1.w << 32) | h1.z);
            float4 s4v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (q0 + i < q1 && (M1 || 4 * t + ml < M))
                s4v = *reinterpret_cast<const float4*>(sog + ((size_t)(4 * t + ml) * ng4 + q0 + i) * 4);
            sv[i][0][t] = s4v.x; sv[i][1][t] = s4v.y; sv[i][2][t] = s4v.z; sv[i][3][t] = s4v.w;
        }

    int buf = 0;
    for (int rb = blockIdx.x; rb < nrb; rb += gridDim.x) {  // workgroup-uniform
        const int row = 16 * rb + col;
        uint4 wq[GQ];
        uint2 wsc[GQ];
#pragma unroll
        for (int i = 0; i < GQ; ++i)
            if (q0 + i < q1) {
                const size_t blk = (size_t)rb * ng4 + q0 + i;
                wq[i] = *reinterpret_cast<const uint4*>(q4m + (blk * 64 + lane) * 16);
                wsc[i] = *reinterpret_cast<const uint2*>(s4m + (blk * 16 + col) * 4);
            }
        float acc[MT4];
#pragma unroll
        for (int t = 0; t < MT4; ++t) acc[t] = 0.0f;
#pragma unroll
        for (int i = 0; i < GQ; ++i) {
            if (q0 + i >= q1) continue;  // no break, so the loop unrolls
            const uint32_t wd[4] = {wq[i].x, wq[i].y, wq[i].z, wq[i].w};
            const uint32_t sd[2] = {wsc[i].x, wsc[i].y};
#pragma unroll
            for (int gi = 0; gi < 4; ++gi) {
                const int g = 4 * (q0 + i) + gi;
                if (g >= ng) continue;  // zero padding groups of the last quad
                const float sc = h2f((uint16_t)(sd[gi >> 1] >> (16 * (gi & 1))));
                group_mfma<MT4>(acc, wd[gi], sc, ao[i][gi], sv[i][gi], g, row, N, K, M, raw, a, ml);
            }
        }
        if (KS == 1) {
#pragma unroll
            for (int t = 0; t < MT4; ++t) {
                const int m = 4 * t + (lane >> 4);
                if (m < M && row < N) out[(size_t)m * N + row] = acc[t];
            }
            continue;
        }
        // parts of this block through LDS; the two buffers alternate between
        // consecutive blocks, so one barrier per block suffices
#pragma unroll
        for (int t = 0; t < MT4; ++t) red[buf][ks][t][lane] = acc[t];
        __syncthreads();
        if (ks == 0) {
#pragma unroll
            for (int t = 0; t < MT4; ++t) {
                float v = red[buf][0][t][lane];
#pragma unroll
                for (int q = 1; q < KS; ++q) v = v + red[buf][q][t][lane];
                const int m = 4 * t + (lane >> 4);
                if (m < M && row < N) out[(size_t)m * N + row] = v;
            }
        }
        buf ^= 1;
    }
}

// Fused M <= 4 path (one launch, one 16-row block per workgroup).  The
// workgroup first writes the activation digits of all K into LDS in compact
// form: for group g < 4*ng4 (groups past K are zero), chunk q (k = 8q..8q+7),
// token m and digit d, the 8 bytes at (((g*4 + q)*M + m)*3 + d)*8, plus
// so[g*M + m] (-1: a group the digits cannot carry), and one zero slot.
// Then its KS waves, wave ks owning the ks-th part (at most GQ quads) of K,
// issue all of their part's weight loads at once (before the digit pass, so
// the latencies overlap); the A operand of a group is an 8-byte LDS read (the
// zero slot for lanes whose A row 4m + d has m >= M or d == 3).  The KS
// partial sums are added in part order through LDS.
template <int M, int KS, int GQ>
__global__ __launch_bounds__(64 * KS) void i4_fused_kernel(
    const uint8_t* __restrict__ q4m, const uint16_t* __restrict__ s4m,
    const uint8_t* __restrict__ raw, const float* __restrict__ a, int K, int N,
    int ng4, float* __restrict__ out) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int ng = K / 32, ngp = 4 * ng4;
    uint2* adl = reinterpret_cast<uint2*>(smem);  // [ngp*4*M*3 + 1 zero slot]
    const int zslot = ngp * 4 * M * 3;
    float* sol = reinterpret_cast<float*>(smem + (size_t)(zslot + 2) * 8);  // [ngp*M]
    float* red = sol + ((ngp * M + 3) & ~3);                                // [KS][64]
    const int tid = threadIdx.x, lane = tid & 63;
    const int ks = __builtin_amdgcn_readfirstlane(tid >> 6);

    // the weight loads of this wave's part do not depend on the digits: issue
    // them first, so their latency overlaps the digit pass
    const int rb = blockIdx.x;
    const int q0 = (int)((long)ng4 * ks / KS), q1 = (int)((long)ng4 * (ks + 1) / KS);
    const int nq = q1 - q0;  // <= GQ
    const int col = lane & 15, ml = lane >> 4;
    uint4 wq[GQ];
    uint2 wsc[GQ];
#pragma unroll
    for (int i = 0; i < GQ; ++i)
        if (i < nq) {
            const size_t blk = (size_t)rb * ng4 + q0 + i;
            wq[i] = *reinterpret_cast<const uint4*>(q4m + (blk * 64 + lane) * 16);
            wsc[i] = *reinterpret_cast<const uint2*>(s4m + (blk * 16 + col) * 4);
        }

    // 1. digits: four adjacent threads per (m, g), one chunk q each; a
    //    thread's items of a pass are loaded together, then digitised
    constexpr int IPT = 2;
    const int nitems = 4 * M * ngp;
    if (tid == 0) adl[zslot] = make_uint2(0u, 0u);
    for (int base = 0; base < nitems; base += 64 * KS * IPT) {  // uniform trip count
        float v[IPT][8];
#pragma unroll
        for (int it = 0; it < IPT; ++it) {
            const int idx = base + it * 64 * KS + tid;
            const int mg = idx >> 2, q = idx & 3;
            const int m = mg / ngp, g = mg % ngp;
#pragma unroll
            for (int k = 0; k < 8; ++k) v[it][k] = 0.0f;
            if (mg < M * ngp && g < ng) {
                const float4* ap = reinterpret_cast<const float4*>(a + (size_t)m * K + (size_t)g * 32 + 8 * q);
                const float4 x0 = ap[0], x1 = ap[1];
                v[it][0] = x0.x; v[it][1] = x0.y; v[it][2] = x0.z; v[it][3] = x0.w;
                v[it][4] = x1.x; v[it][5] = x1.y; v[it][6] = x1.z; v[it][7] = x1.w;
            }
        }
#pragma unroll
        for (int it = 0; it < IPT; ++it) {
            const int idx = base + it * 64 * KS + tid;
            const int mg = idx >> 2, q = idx & 3;
            const bool act = mg < M * ngp;
            const int m = act ? mg / ngp : 0, g = act ? mg % ngp : 0;
            float mx = 0.0f;
            int nf = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                nf |= !(fabsf(v[it][k]) <= 3.0e38f);
                mx = fmaxf(mx, fabsf(v[it][k]));
            }
            mx = fmaxf(mx, __shfl_xor(mx, 1, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 2, 64));
            nf |= __shfl_xor(nf, 1, 64);
            nf |= __shfl_xor(nf, 2, 64);
            if (!act) continue;
            // |group sum| <= 32 * 8 * mx stays finite for s <= 1e28
            const float sg = mx > 0.0f ? mx / XMAX4 : 1.0f;
            const bool ok = !nf && sg >= 1.0e-30f && sg <= 1.0e28f;
            uint32_t dw[3][2] = {{0, 0}, {0, 0}, {0, 0}};
            if (ok) {
                const float r = 1.0f / sg;  // any rounding of a / s keeps |a - s X| <= ~s/2
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float xf = rintf(v[it][j] * r);
                    xf = fminf(fmaxf(xf, -XMAX4), XMAX4);
                    const int X = (int)xf;
                    const int d0 = (int)(int8_t)(X & 0xFF);
                    const int X1 = (X - d0) >> 8;
                    const int d1 = (int)(int8_t)(X1 & 0xFF);
                    const int d2 = (X1 - d1) >> 8;
                    const int p = (j & 1) ? 4 + (j >> 1) : (j >> 1);
                    const int wsel = p >> 2, sh = 8 * (p & 3);
                    dw[0][wsel] |= (uint32_t)(d2 & 0xFF) << sh;
                    dw[1][wsel] |= (uint32_t)(d1 & 0xFF) << sh;
                    dw[2][wsel] |= (uint32_t)(d0 & 0xFF) << sh;
                }
            }
#pragma unroll
            for (int d = 0; d < 3; ++d) adl[((g * 4 + q) * M + m) * 3 + d] = make_uint2(dw[d][0], dw[d][1]);
            if (q == 0) sol[g * M + m] = g < ng ? (ok ? sg : -1.0f) : 0.0f;
        }
    }
    __syncthreads();

    // 2. this workgroup's 16-row block, the groups of the wave's part in order
    const int am = col >> 2, ad = col & 3;  // A row of this lane: token am, digit ad
    const int row = 16 * rb + col;
    const int mtok = ml < M ? ml : 0;       // token of this lane's result (lanes >= M: junk)
    // LDS slot of the lane's A operand for group g: abase + g * 12M (the zero
    // slot, stride 0, for lanes without a digit row)
    const bool arow = am < M && ad < 3;
    const int abase = arow ? (ml * M + am) * 3 + ad : zslot;
    const int astep = arow ? 12 * M : 0;
    const int g0 = 4 * q0;
    // any group of the part that the digits cannot carry?  (wave-uniform)
    int xg = 0;
    for (int i = lane; i < 4 * nq * M; i += 64) xg |= sol[g0 * M + i] < 0.0f;
    float acc = 0.0f;
    if (__builtin_amdgcn_ballot_w64(xg) == 0) {
        // fast path: straight-line digit MFMAs, four groups per weight quad
#pragma unroll
        for (int i = 0; i < GQ; ++i) {
            if (i >= nq) continue;  // wave-uniform; no break, so the loop unrolls
            const int gq = 4 * (q0 + i);
            const uint32_t wd[4] = {wq[i].x, wq[i].y, wq[i].z, wq[i].w};
            v4i cr[4];
#pragma unroll
            for (int gi = 0; gi < 4; ++gi) {
                uint32_t lo, hi;
                nib_unpack(wd[gi], lo, hi);
                const long bop = (long)(((unsigned long long)hi << 32) | lo);
                const uint2 av = adl[abase + (gq + gi) * astep];
                const long aop = (long)(((unsigned long long)av.y << 32) | av.x);
                cr[gi] = __builtin_amdgcn_mfma_i32_16x16x32_i8(aop, bop, v4i{0, 0, 0, 0}, 0, 0, 0);
            }
            const uint32_t sd[2] = {wsc[i].x, wsc[i].y};
#pragma unroll
            for (int gi = 0; gi < 4; ++gi) {
                const float sgi = sol[(gq + gi) * M + mtok];
                const float sc = h2f((uint16_t)(sd[gi >> 1] >> (16 * (gi & 1))));
                const float gs = sgi * ((float)cr[gi][0] * 65536.0f + ((float)cr[gi][1] * 256.0f + (float)cr[gi][2]));
                acc = acc + sc * gs;
            }
        }
    } else {
        // some group needs the exact path: a compact loop over the part, the
        // weights read again from global memory
        for (int g = g0; g < min(4 * q1, ng); ++g) {
            const size_t blk = (size_t)rb * ng4 + (g >> 2);
            const uint32_t wd = *reinterpret_cast<const uint32_t*>(q4m + (blk * 64 + lane) * 16 + 4 * (g & 3));
            const uint16_t sh = s4m[(blk * 16 + col) * 4 + (g & 3)];
            const uint2 av = adl[abase + g * astep];
            const long aop[1] = {(long)(((unsigned long long)av.y << 32) | av.x)};
            const float so[1] = {sol[g * M + mtok]};
            float a1[1] = {acc};
            group_mfma<1, true>(a1, wd, h2f(sh), aop, so, g, row, N, K, M, raw, a, ml);
            acc = a1[0];
        }
    }
    if (KS == 1) {
        if (ml < M && row < N) out[(size_t)ml * N + row] = acc;
        return;
    }
    red[ks * 64 + lane] = acc;
    __syncthreads();
    if (ks == 0) {
        float v = red[lane];
#pragma unroll
        for (int q = 1; q < KS; ++q) v = v + red[q * 64 + lane];
        if (ml < M && row < N) out[(size_t)ml * N + row] = v;
    }
}

// LDS bytes of the fused path (compact digits + zero slot + scales + reduction).
size_t fused_lds(size_t m, size_t k, int ks) {
    const size_t ngp = 4 * ((k / 32 + 3) / 4);
    return (ngp * 4 * m * 3 + 2) * 8 + ((ngp * m + 3) & ~(size_t)3) * 4 + (size_t)ks * 64 * 4;
}

// (N, K/2) packed nibbles + (N, ng) f16 scales -> the MFMA layout: for row
// block rb and group quad g4, lane l = 16q + r holds, for groups 4g4..4g4+3,
// the 4 bytes of row 16rb + r at k = 8q..8q+7 of each group (16 bytes at
// ((rb*ng4 + g4)*64 + l)*16), and the scales (rb, g4, r) as 4 halves.
// Rows >= N and groups >= ng are zero.
__global__ void i4_block_kernel(const uint8_t* __restrict__ raw, const uint16_t* __restrict__ sraw,
                                int N, int K, int ng4, uint8_t* __restrict__ q4m,
                                uint16_t* __restrict__ s4m) {
    const int ng = K / 32, nrb = (N + 15) / 16;
    const size_t total = (size_t)nrb * ng4 * 64;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total;
         i += (size_t)gridDim.x * blockDim.x) {
        const int l = (int)(i % 64);
        const size_t bg = i / 64;
        const int g4 = (int)(bg % ng4), rb = (int)(bg / ng4);
        const int r = l & 15, q = l >> 4, row = 16 * rb + r;
        uint32_t v[4] = {0, 0, 0, 0};
        for (int gi = 0; gi < 4; ++gi) {
            const int g = 4 * g4 + gi;
            if (row < N && g < ng)
                v[gi] = *reinterpret_cast<const uint32_t*>(raw + (size_t)row * (K / 2) + (size_t)g * 16 + 4 * q);
        }
        reinterpret_cast<uint4*>(q4m)[i] = make_uint4(v[0], v[1], v[2], v[3]);
        if (q == 0) {
            for (int gi = 0; gi < 4; ++gi) {
                const int g = 4 * g4 + gi;
                s4m[(bg * 16 + r) * 4 + gi] = (row < N && g < ng) ? sraw[(size_t)row * ng + g] : (uint16_t)0;
            }
        }
    }
}

}  // namespace

static bool mfma_fits(size_t k, size_t m);

static bool fused_fits(size_t k, size_t m);

size_t i4_ws_floats(const Weight& w, size_t m) {
    if (!w.i4_blocked || fused_fits(w.k, m) || !mfma_fits(w.k, m)) return 0;
    const size_t mp = round_up(m, 4), ng4 = (w.k / 32 + 3) / 4;
    return (mp / 4) * ng4 * 64 * 32 / sizeof(float) + mp * ng4 * 4 + 64;  // digits + scales
}

size_t i4_blocked_bytes(size_t n, size_t k) {
    return (n + 15) / 16 * ((k / 32 + 3) / 4) * 1024;
}

hipError_t launch_i4_block(const uint8_t* raw, const uint16_t* sraw, size_t n,
                           size_t k, uint8_t* blk, uint16_t* sblk,
                           hipStream_t s) {
    const int ng4 = (int)((k / 32 + 3) / 4);
    i4_block_kernel<<<dim3(1024), dim3(256), 0, s>>>(raw, sraw, (int)n, (int)k, ng4, blk, sblk);
    return hipGetLastError();
}

template <int MT4, int KS, int GQ>
static hipError_t launch_mfma_t(const Weight& w, size_t m, const float* a, const uint8_t* adig,
                                const float* sog, float* out, hipStream_t s) {
    const size_t ng4 = (w.k / 32 + 3) / 4, nrb = (w.n + 15) / 16;
    // about 8 waves per CU on 256 CUs, the blocks spread evenly
    const size_t want = 2048 / KS;
    const size_t per = (nrb + want - 1) / want;
    const size_t grid = (nrb + per - 1) / per;
    if constexpr (MT4 == 1)
        if (m == 1) {
            i4_mfma_kernel<1, KS, GQ, true><<<dim3((unsigned)grid), dim3(64 * KS), 0, s>>>(
                w.q4, w.s4, w.q4raw, a, adig, sog, (int)m, (int)w.k, (int)w.n, (int)ng4, out);
            return hipGetLastError();
        }
    i4_mfma_kernel<MT4, KS, GQ, false><<<dim3((unsigned)grid), dim3(64 * KS), 0, s>>>(
        w.q4, w.s4, w.q4raw, a, adig, sog, (int)m, (int)w.k, (int)w.n, (int)ng4, out);
    return hipGetLastError();
}

// Group quads per K part (register budget: GQ * 4 * MT4 resident operands).
constexpr int gq_of(int mt4) { return mt4 == 1 ? 9 : (mt4 == 2 ? 5 : 3); }

// KS waves per workgroup, the fewest whose parts hold at most GQ quads.
template <int MT4>
static hipError_t launch_mfma(const Weight& w, size_t m, const float* a, const uint8_t* adig,
                              const float* sog, float* out, hipStream_t s) {
    constexpr int GQ = gq_of(MT4);
    const size_t ng4 = (w.k / 32 + 3) / 4;
    if (ng4 <= GQ) return launch_mfma_t<MT4, 1, GQ>(w, m, a, adig, sog, out, s);
    if (ng4 <= 2 * GQ) return launch_mfma_t<MT4, 2, GQ>(w, m, a, adig, sog, out, s);
    if (ng4 <= 4 * GQ) return launch_mfma_t<MT4, 4, GQ>(w, m, a, adig, sog, out, s);
    if (ng4 <= 8 * GQ) return launch_mfma_t<MT4, 8, GQ>(w, m, a, adig, sog, out, s);
    return hipErrorInvalidValue;  // mfma_fits() sends longer K to the generic path
}

// Shapes the MFMA path takes at m tokens: m <= 16 and K in at most 8 parts.
static bool mfma_fits(size_t k, size_t m) {
    if (m < 1 || m > 16) return false;
    const size_t ng4 = (k / 32 + 3) / 4, mt4 = (m + 3) / 4;
    return ng4 <= 8 * (size_t)gq_of((int)mt4);
}

template <int M, int KS>
static hipError_t launch_fused_t(const Weight& w, const float* a, float* out, hipStream_t s) {
    constexpr int GQ = 9;
    const size_t ng4 = (w.k / 32 + 3) / 4, nrb = (w.n + 15) / 16;
    const size_t lds = fused_lds(M, w.k, KS);
    i4_fused_kernel<M, KS, GQ><<<dim3((unsigned)nrb), dim3(64 * KS), lds, s>>>(
        w.q4, w.s4, w.q4raw, a, (int)w.k, (int)w.n, (int)ng4, out);
    return hipGetLastError();
}

// KS waves per workgroup: parts of at most 5 group quads (more waves per CU
// to overlap the MFMA -> VALU chains), at most 9 when K needs 16 parts.
template <int M>
static hipError_t launch_fused_m(const Weight& w, const float* a, float* out, hipStream_t s) {
    const size_t ng4 = (w.k / 32 + 3) / 4;
    if (ng4 <= 5) return launch_fused_t<M, 1>(w, a, out, s);
    if (ng4 <= 10) return launch_fused_t<M, 2>(w, a, out, s);
    if (ng4 <= 20) return launch_fused_t<M, 4>(w, a, out, s);
    if (ng4 <= 40) return launch_fused_t<M, 8>(w, a, out, s);
    return launch_fused_t<M, 16>(w, a, out, s);
}

// The fused path: M <= 4, K in at most 16 parts of 9 quads, digits within 64 KB of LDS.
static bool fused_fits(size_t k, size_t m) {
    const size_t ng4 = (k / 32 + 3) / 4;
    return m >= 1 && m <= 4 && ng4 <= 144 && fused_lds(m, k, 16) <= 64 * 1024;
}

static hipError_t launch_fused(const Weight& w, size_t m, const float* a, float* out, hipStream_t s) {
    switch (m) {
        case 1: return launch_fused_m<1>(w, a, out, s);
        case 2: return launch_fused_m<2>(w, a, out, s);
        case 3: return launch_fused_m<3>(w, a, out, s);
        default: return launch_fused_m<4>(w, a, out, s);
    }
}

template <int G4, int IPT, int NT>
hipError_t launch_stream_t(const Weight& w, int R, unsigned grid, size_t lds, const float* a, float* out,
                           hipStream_t s) {
    // the attribute once per instantiation, at the full 160 KB (later calls
    // issue the launch only)
    static bool attr = false;
    if (lds > 64 * 1024 && !attr) {
        const hipError_t e = hipFuncSetAttribute((const void*)i4_m1_stream<G4, IPT, NT>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        attr = true;
    }
    i4_m1_stream<G4, IPT, NT><<<dim3(grid), dim3(NT), lds, s>>>(w.q4raw, w.s4raw, (int)w.n, (int)w.k, R, a, out);
    return hipGetLastError();
}

template <int G4, int NT>
hipError_t launch_stream_g(const Weight& w, int ipt, int R, unsigned grid, size_t lds, const float* a, float* out,
                           hipStream_t s) {
    switch (ipt) {
        case 2: return launch_stream_t<G4, 2, NT>(w, R, grid, lds, a, out, s);
        case 4: return launch_stream_t<G4, 4, NT>(w, R, grid, lds, a, out, s);
        case 6: return launch_stream_t<G4, 6, NT>(w, R, grid, lds, a, out, s);
        case 8: return launch_stream_t<G4, 8, NT>(w, R, grid, lds, a, out, s);
        case 12: return launch_stream_t<G4, 12, NT>(w, R, grid, lds, a, out, s);
        default: return launch_stream_t<G4, 16, NT>(w, R, grid, lds, a, out, s);
    }
}

// The streamed M == 1 kernel: rows split evenly over the workgroups (one a
// CU, of 512 threads; more where a thread would hold over 16 items),
// the activation row and the terms within 160 KB of LDS (else
// hipErrorNotSupported).
hipError_t launch_i4_stream(const Weight& w, const float* a, float* out, hipStream_t s) {
    if (w.k % 32 || (w.g != 32 && w.g != 64) || w.k % w.g || w.k > (1u << 24) || w.n > (size_t)INT32_MAX ||
        ((uintptr_t)a & 15))
        return hipErrorNotSupported;
    const size_t ng = w.k / w.g, n = w.n;
    constexpr int nt = 512;  // 8 waves: two a SIMD, one activation row staged a CU
    const size_t nwg = (size_t)device_cus(w.device);
    size_t R = (n + nwg - 1) / nwg;
    if (R * ng > (size_t)nt * 16) R = std::max<size_t>(1, (size_t)nt * 16 / ng);
    const size_t items = R * ng, ipt0 = (items + nt - 1) / nt;
    const int ipt = ipt0 <= 2 ? 2 : ipt0 <= 4 ? 4 : ipt0 <= 6 ? 6 : ipt0 <= 8 ? 8 : ipt0 <= 12 ? 12 : 16;
    if (ipt0 > 16) return hipErrorNotSupported;
    const size_t lds = i4_stream_as_bytes((int)w.k) + (R * ((ng + 3) & ~(size_t)3) + 4) * sizeof(float);
    if (lds > 160 * 1024) return hipErrorNotSupported;
    const unsigned grid = (unsigned)((n + R - 1) / R);
    return w.g == 32 ? launch_stream_g<1, nt>(w, ipt, (int)R, grid, lds, a, out, s)
                     : launch_stream_g<2, nt>(w, ipt, (int)R, grid, lds, a, out, s);
}

// The exact M == 1 kernel when the shape allows it (else hipErrorNotSupported).
hipError_t launch_i4_terms(const Weight& w, const float* a, float* out, hipStream_t s) {
    {
        const hipError_t e = launch_i4_stream(w, a, out, s);
        if (e != hipErrorNotSupported) return e;
    }
    if (w.k % 32 || (w.g != 32 && w.g != 64) || w.k > (size_t)INT32_MAX || w.n > (size_t)INT32_MAX)
        return hipErrorNotSupported;
    const int ng = (int)(w.k / w.g);
    int rb = std::min(64, std::max(1, 8192 / std::max(ng, 1)));
    while (rb > 8 && (w.n + rb - 1) / rb < 512) rb /= 2;
    const size_t cgb = (size_t)rb * ((ng + 3) & ~3) * sizeof(float);
    const size_t asb = (w.k / 32) * 36 * sizeof(float);
    if (cgb + asb > 64 * 1024) return hipErrorNotSupported;
    const unsigned grid = (unsigned)((w.n + rb - 1) / rb);
    if (w.g == 32)
        i4_gemv_terms<1><<<dim3(grid), dim3(256), cgb + asb, s>>>(w.q4raw, w.s4raw, (int)w.n, (int)w.k, rb, a, out);
    else
        i4_gemv_terms<2><<<dim3(grid), dim3(256), cgb + asb, s>>>(w.q4raw, w.s4raw, (int)w.n, (int)w.k, rb, a, out);
    return hipGetLastError();
}

// Whether launch_i4_rows_a4 takes this weight (else launch_i4_m1_rows runs
// the rows one M == 1 launch at a time: other shapes, and matrices of 4 GB and
// more, at which the batched kernels have not been run).
bool i4_rows_a4_ok(const Weight& w) {
    return (w.g == 32 || w.g == 64) && w.k > 0 && w.k % w.g == 0 && w.k <= (size_t)INT32_MAX &&
           w.n <= (size_t)INT32_MAX && w.n * w.k / 2 < ((size_t)1 << 32);
}

size_t i4_a4_floats(size_t k) { return 16 * k; }

hipError_t launch_rows_to_a4(const float* a, size_t m, size_t k, float* a4, hipStream_t s) {
    const size_t n4 = 4 * k;  // float4 of a4
    rows_to_a4_kernel<<<dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s>>>(a, (int)m, (int)k, a4);
    return hipGetLastError();
}

namespace {
// Workgroups of 3 or 4 waves (12 or 16 DPP rows), whichever leaves the fewer
// idle groups in the last slice; 4 on a tie.
template <int G4>
hipError_t rows_dpp(const Weight& w, size_t m, const float* a4, float* out, hipStream_t s) {
    const size_t ng = w.k / w.g, gps = 3 - G4;  // groups a DPP row takes a slice
    const unsigned grid = (unsigned)((w.n + 3) / 4);
    if ((ng + 12 * gps - 1) / (12 * gps) * 12 < (ng + 16 * gps - 1) / (16 * gps) * 16)
        i4_rows_dpp<G4, 3><<<dim3(grid), dim3(192), 0, s>>>(w.q4raw, w.s4raw, (int)w.n, (int)w.k, a4, (int)m, out);
    else
        i4_rows_dpp<G4, 4><<<dim3(grid), dim3(256), 0, s>>>(w.q4raw, w.s4raw, (int)w.n, (int)w.k, a4, (int)m, out);
    return hipGetLastError();
}
}  // namespace

// m <= 16 rows in the a4 layout (launch_rows_to_a4), each in the M == 1
// order.  Narrow outputs take i4_rows_dpp; i4_rows_mfma the fewest rounds of 8 waves x ROWS_GW groups
// (64 KB of terms, two workgroups a CU), the groups spread evenly over them
// (72: 3 rounds of 24).
hipError_t launch_i4_rows_a4(const Weight& w, size_t m, const float* a4, float* out, hipStream_t s) {
    if (m == 0 || w.n == 0) return hipSuccess;
    if (m > 16 || !i4_rows_a4_ok(w)) return hipErrorNotSupported;
    if (w.n <= 4 * (size_t)device_cus(w.device))  // i4_rows_dpp's workgroups in one round
        return w.g == 32 ? rows_dpp<1>(w, m, a4, out, s) : rows_dpp<2>(w, m, a4, out, s);
    const size_t ng = w.k / w.g, rounds = (ng + 8 * ROWS_GW - 1) / (8 * ROWS_GW);
    const int gw = rounds ? (int)((ng + 8 * rounds - 1) / (8 * rounds)) : 1;
    const unsigned grid = (unsigned)((w.n + 15) / 16);
    if (w.g == 32)
        i4_rows_mfma<1><<<dim3(grid), dim3(512), 0, s>>>(w.q4raw, w.s4raw, (int)w.n, (int)w.k, gw, a4, (int)m, out);
    else
        i4_rows_mfma<2><<<dim3(grid), dim3(512), 0, s>>>(w.q4raw, w.s4raw, (int)w.n, (int)w.k, gw, a4, (int)m, out);
    return hipGetLastError();
}

// m rows, each in the M == 1 order (bit-identical to m launches at M == 1);
// a4 is scratch of i4_a4_floats(K) floats (16-byte aligned).
hipError_t launch_i4_m1_rows(const Weight& w, size_t m, const float* a, float* out, float* a4, hipStream_t s) {
    if (m == 0 || w.n == 0) return hipSuccess;
    for (size_t r0 = 0; r0 < m; r0 += 16) {
        const size_t mm = std::min<size_t>(16, m - r0);
        if (a4 && i4_rows_a4_ok(w)) {
            if (hipError_t e = launch_rows_to_a4(a + r0 * w.k, mm, w.k, a4, s)) return e;
            if (hipError_t e = launch_i4_rows_a4(w, mm, a4, out + r0 * w.n, s)) return e;
            continue;
        }
        for (size_t i = r0; i < r0 + mm; ++i)
            if (hipError_t e = launch_i4_exact(w, 1, a + i * w.k, out + i * w.n, s)) return e;
    }
    return hipSuccess;
}

// Any K and g at M == 1; hipErrorNotSupported where a row's activations and
// terms exceed 64 KB of LDS (K past about 14000).  Rows a workgroup: as many as fit beside the
// activations, fewer while the grid is short and a row still fills half the
// threads.
hipError_t launch_pack_m1_any(bool q4a, const uint8_t* packed, size_t pitch, const uint16_t* sc, const uint16_t* mn,
                              int ss, size_t n, size_t k, size_t g, const float* a, float* out, hipStream_t s) {
    if (k == 0 || g == 0 || n > (size_t)INT32_MAX || k > 64 * 1024 / 4) return hipErrorNotSupported;
    const size_t gg = std::min(g, k), ng = (k + gg - 1) / gg, row = ((ng + 3) & ~(size_t)3) * 4;
    const size_t act = ((k + k / 32 * 4) / 4 + 4) * 16;
    if (act + row > 64 * 1024) return hipErrorNotSupported;
    size_t rb = std::min<size_t>(64, (64 * 1024 - act) / row);
    while (rb > 1 && (n + rb - 1) / rb < 512 && rb * ng > 256) rb = (rb + 1) / 2;
    const unsigned grid = (unsigned)((n + rb - 1) / rb);
    const size_t lds = act + rb * row;
    if (q4a)
        pack_gemv_any<true><<<dim3(grid), dim3(256), lds, s>>>(packed, pitch, sc, mn, ss, (int)n, (int)k, (int)gg,
                                                               (int)rb, a, out);
    else
        pack_gemv_any<false><<<dim3(grid), dim3(256), lds, s>>>(packed, pitch, sc, mn, ss, (int)n, (int)k, (int)gg,
                                                                (int)rb, a, out);
    return hipGetLastError();
}

namespace {
hipError_t i4_m1_any(const Weight& w, const float* a, float* out, hipStream_t s) {
    if (w.k > 64) {  // a thread a row is the faster below: 37 x 2000 3.5 against 3.9 us, 65 x 2000 5.3 against 4.3
        const hipError_t e = launch_pack_m1_any(false, w.q4raw, (w.k + 1) / 2, w.s4raw, nullptr, 1, w.n, w.k, w.g, a,
                                                out, s);
        if (e != hipErrorNotSupported) return e;
    }
    i4_gemv_generic<<<dim3((unsigned)((w.n + 255) / 256)), dim3(256), 0, s>>>(w.q4raw, w.s4raw, (int)w.n, (int)w.k,
                                                                             (int)w.g, a, out);
    return hipGetLastError();
}

// M > 1: the dequantised weights on the f32 matrix cores, in a.dot's order.
hipError_t mm_dequant(const Weight& w, size_t m, const float* a, float* out, hipStream_t s) {
    if (w.n > (size_t)INT32_MAX || w.k > (size_t)INT32_MAX) return hipErrorInvalidValue;
    MmWeight v{};
    v.w = w.q4raw;
    v.sc = w.s4raw;
    v.ss = 1;
    v.n = (int)w.n;
    v.k = (int)w.k;
    v.g = (int)std::min(w.g, std::max<size_t>(w.k, 1));  // a longer group is one group
    v.ng = (int)((w.k + w.g - 1) / w.g);
    v.pitch = (w.k + 1) / 2;
    return launch_mm_f32(FRQ_DT_I4, v, a, m, out, device_cus(w.device), s);
}
}  // namespace

hipError_t launch_i4_exact(const Weight& w, size_t m, const float* a, float* out, hipStream_t s) {
    if (m == 0 || w.n == 0) return hipSuccess;
    if (m == 1) {
        const hipError_t e = launch_i4_terms(w, a, out, s);
        if (e != hipErrorNotSupported) return e;
        return i4_m1_any(w, a, out, s);
    }
    return mm_dequant(w, m, a, out, s);
}

hipError_t launch_i4(const Weight& w, size_t m, const float* a, float* out,
                     float* wsf, hipStream_t s) {
    if (m == 0) return hipSuccess;
    if (m == 1) {  // the reference's decode order, bit for bit, where the shape allows
        const hipError_t e = launch_i4_terms(w, a, out, s);
        if (e != hipErrorNotSupported) return e;
    }
    if (w.i4_blocked && fused_fits(w.k, m)) return launch_fused(w, m, a, out, s);
    if (w.i4_blocked && mfma_fits(w.k, m)) {
        const size_t mp = round_up(m, 4), ng4 = (w.k / 32 + 3) / 4;
        uint8_t* adig = reinterpret_cast<uint8_t*>(wsf);
        float* sog = reinterpret_cast<float*>(adig + (mp / 4) * ng4 * 64 * 32);
        const size_t nth = 4 * mp * 4 * ng4;
        i4_digits_kernel<<<dim3((unsigned)((nth + 255) / 256)), dim3(256), 0, s>>>(
            a, (int)m, (int)mp, (int)w.k, (int)ng4, adig, sog);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        switch (mp / 4) {
            case 1: return launch_mfma<1>(w, m, a, adig, sog, out, s);
            case 2: return launch_mfma<2>(w, m, a, adig, sog, out, s);
            case 3: return launch_mfma<3>(w, m, a, adig, sog, out, s);
            default: return launch_mfma<4>(w, m, a, adig, sog, out, s);
        }
    }
    if (m == 1) return i4_m1_any(w, a, out, s);
    return mm_dequant(w, m, a, out, s);
}

}  // namespace frq
