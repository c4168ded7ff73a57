// VALU GEMVs for the weight formats without a fused matrix-core kernel:
// F32, F16, Q2_K and Q3_K.
//
//  * GGUF order (AETH_ORDER_GGUF): load_quant keeps these formats as the file
//    holds them, [k][n] (model_loader.rs:344-350), and quantized_matmul_impl
//    multiplies them by dequantize(b, [k, n]) + matmul_f32_gguf
//    (dispatch.rs:126-133, 541-574): c[j] = fma(a_i, b[i·n + j], c[j]) over i,
//    rows with a_i == 0 skipped. Here workgroup (unit u, split s, row group)
//    owns outputs j ∈ [256u, 256u + 256) and inputs i ∈ split s; its four waves
//    take every fourth i, each lane four outputs, one FMA per (row, output) per
//    i with the same zero skip (n % 4 == 0; K-quant blocks may straddle rows). Q2_K / Q3_K of whole blocks per input
//    run k_colk instead. Partials [s][row][j] are then summed by k_col_reduce in a
//    fixed order, which also applies accumulate and the argmax key.
//  * Rows (AETH_ORDER_ROWS): matmul_f16 / matmul_q2_k / matmul_q3_k on [n][k]
//    row blocks (f16.rs, q2_k.rs, q3_k.rs; x86: avx2.rs:210-389). A wave per
//    output row, lanes four elements of each 256-element unit, a wave sum at
//    the end.
//
// Weights are formed exactly as dequant.rs rounds them (contraction off):
// Q2_K d·(sc & 15)·q − dmin·(sc >> 4), Q3_K (d·sc)·q, F16 exact; only the
// summation order differs from the reference.
//
// Lanes own four consecutive elements of the weight's flat element run
// (f, f+1, f+2, f+3 with f % 4 == 0, so they share one K-quant block and
// sub-block): lane l of a 256-wide unit takes its elements 4l .. 4l+3.
#include <algorithm>

#include "aeth_common.hpp"
#include "aeth_internal.hpp"
#include "aeth_ops_internal.hpp"

#pragma clang fp contract(off)

namespace {

template <int F> struct XU;

// Each format splits into load (the raw words a lane needs, issued for a whole
// batch of inputs before any is used) and expand (the four f32 weights).

// dequant_q2_k (dequant.rs:350-398): 84-byte block [d][dmin][scales 16][qs 64];
// element e = 128h + 32t + 16v + i is bits 2t of qs[32h + 16v + i], sub-block
// 8h + 2t + v. Blocks are 4-byte aligned (84 = 4·21) and so are the lane's 4 qs bytes.
template <> struct XU<AETH_DTYPE_Q2_K> {
    struct Raw { uint32_t dd, sc, q; int t; };
    __device__ static Raw load(const uint8_t* W, int64_t f) {
        const uint8_t* b = W + (f >> 8) * Q2K_BLOCK_BYTES;
        const int e = (int)(f & 255), h = e >> 7, t = (e >> 5) & 3, v = (e >> 4) & 1;
        Raw r;
        r.dd = *(const uint32_t*)b;
        r.sc = b[4 + 8 * h + 2 * t + v];
        r.q = *(const uint32_t*)(b + 20 + 32 * h + 16 * v + (e & 15));
        r.t = t;
        return r;
    }
    __device__ static void expand(const Raw& r, float (&w)[4]) {
        const float d = aeth_decode_d(r.dd & 0xFFFFu), dmin = aeth_decode_d(r.dd >> 16);
        const float dl = d * (float)(r.sc & 0xF), ml = dmin * (float)(r.sc >> 4);
#pragma unroll
        for (int c = 0; c < 4; c++) w[c] = dl * (float)((r.q >> (8 * c + 2 * r.t)) & 3) - ml;
    }
};

// dequant_q3_k (dequant.rs:400-451): 110-byte block [hmask 32][qs 64][scales 12][d]
// (2-byte aligned); element e = 128h + 32t + 16v + i: bits 2t of
// qs[32h + 16v + i], bit 4h + t of hmask[16v + i], 6-bit scale of sub-block
// s = 8h + 2t + v (low nibble of scales[s % 8], high pair from scales[8 + s % 4]),
// q = ql − 4·(1 − hbit), w = (d·(scale − 32))·q.
template <> struct XU<AETH_DTYPE_Q3_K> {
    struct Raw { uint32_t q, hm, lob, hib, d; int e; };
    __device__ static Raw load(const uint8_t* W, int64_t f) {
        const uint8_t* b = W + (f >> 8) * Q3K_BLOCK_BYTES;
        const int e = (int)(f & 255), h = e >> 7, t = (e >> 5) & 3, v = (e >> 4) & 1, i = e & 15;
        const uint16_t* qp = (const uint16_t*)(b + 32 + 32 * h + 16 * v + i);
        const uint16_t* hp = (const uint16_t*)(b + 16 * v + i);
        const int s = 8 * h + 2 * t + v;
        Raw r;
        r.q = (uint32_t)qp[0] | ((uint32_t)qp[1] << 16);
        r.hm = (uint32_t)hp[0] | ((uint32_t)hp[1] << 16);
        r.lob = b[96 + (s & 7)];
        r.hib = b[104 + (s & 3)];
        r.d = *(const uint16_t*)(b + 108);
        r.e = e;
        return r;
    }
    __device__ static void expand(const Raw& r, float (&w)[4]) {
        const int h = r.e >> 7, t = (r.e >> 5) & 3, v = (r.e >> 4) & 1, s = 8 * h + 2 * t + v;
        const int sc = (int)((s < 8 ? (r.lob & 0xF) : (r.lob >> 4)) | (((r.hib >> (2 * (s >> 2))) & 3) << 4)) - 32;
        const float dl = aeth_decode_d(r.d) * (float)sc;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const int ql = (int)((r.q >> (8 * c + 2 * t)) & 3), hb = (int)((r.hm >> (8 * c + 4 * h + t)) & 1);
            w[c] = dl * (float)(ql - ((hb ^ 1) << 2));
        }
    }
};

template <> struct XU<AETH_DTYPE_F16> {
    typedef uint2 Raw;
    __device__ static Raw load(const uint8_t* W, int64_t f) { return *(const uint2*)(W + 2 * f); }
    __device__ static void expand(const Raw& v, float (&w)[4]) {
        w[0] = aeth_f16_to_f32(v.x & 0xFFFFu);
        w[1] = aeth_f16_to_f32(v.x >> 16);
        w[2] = aeth_f16_to_f32(v.y & 0xFFFFu);
        w[3] = aeth_f16_to_f32(v.y >> 16);
    }
};

template <> struct XU<AETH_DTYPE_F32> {
    typedef float4 Raw;
    __device__ static Raw load(const uint8_t* W, int64_t f) { return *(const float4*)(W + 4 * f); }
    __device__ static void expand(const Raw& v, float (&w)[4]) {
        w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
    }
};

// GGUF order: partials part[s][row][j] of Σ_{i ∈ split s} x[row][i]·W[i][j]
// (element (i, j) is flat element i·n + j; n % 4 == 0). NW waves take every
// NW-th input of the split, NB inputs per batch with all loads issued first.
template <int F, int R, int NW>
__global__ void __launch_bounds__(64 * NW) k_col(const uint8_t* __restrict__ W, int64_t n, int64_t k,
                                                 const float* __restrict__ x, int64_t ldx, int m, int S,
                                                 float* __restrict__ part) {
    constexpr int NB = 8;
    typedef typename XU<F>::Raw Raw;
    __shared__ float4 red[NW][R][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t j0 = (int64_t)blockIdx.x * 256 + 4 * lane;  // this lane's first output
    const int s = blockIdx.y, r0 = blockIdx.z * R;
    const int64_t i0 = k * s / S, i1 = k * (s + 1) / S;
    float acc[R][4];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int t = 0; t < 4; t++) acc[r][t] = 0.0f;
    const float* xr[R];
#pragma unroll
    for (int r = 0; r < R; r++) xr[r] = x + (int64_t)min(r0 + r, m - 1) * ldx;
    const int64_t jl = j0 < n ? j0 : n - 4;  // lanes past n read the last valid group, discarded
    for (int64_t ib = i0 + wave; ib < i1; ib += NW * NB) {
        Raw raw[NB];
        float xv[NB][R];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int64_t i = ib + (int64_t)b * NW, ic = i < i1 ? i : i1 - 1;
            raw[b] = XU<F>::load(W, ic * n + jl);
#pragma unroll
            for (int r = 0; r < R; r++) xv[b][r] = i < i1 ? xr[r][ic] : 0.0f;  // past the split: skipped as 0
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
            float w[4];
            XU<F>::expand(raw[b], w);
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float a = xv[b][r];
                if (a != 0.0f) {  // matmul_f32_gguf skips zero activations (dispatch.rs:548)
#pragma unroll
                    for (int t = 0; t < 4; t++) acc[r][t] = fmaf(a, w[t], acc[r][t]);
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) red[wave][r][lane] = make_float4(acc[r][0], acc[r][1], acc[r][2], acc[r][3]);
    __syncthreads();
    const float* rf = (const float*)red;
    for (int idx = threadIdx.x; idx < R * 256; idx += 64 * NW) {
        const int r = idx >> 8, e = idx & 255;
        const int64_t j = (int64_t)blockIdx.x * 256 + e;
        if (j >= n || r0 + r >= m) continue;
        float v = rf[r * 256 + e];
#pragma unroll
        for (int wv = 1; wv < NW; wv++) v += rf[(wv * R + r) * 256 + e];
        part[((int64_t)s * m + r0 + r) * n + j] = v;
    }
}

// GGUF order, Q2_K / Q3_K with whole blocks per input (n % 256 == 0): the form
// of k_col for packed quants. A wave takes four neighbouring blocks (1024
// outputs) of one input, 16 lanes a block: lane u holds qs dword u, i.e. the
// 4 × 4 elements (t, c) at outputs 128h + 32t + 4(u % 8) + c, h = u / 8, whose
// four scales (sub-blocks 8h + 2t + v, v = (u % 8) / 4) come out of two or
// three dwords with one v_perm each. sc·q is an exact fp16 integer (Q2_K at
// most 45, Q3_K −124 .. 128), formed two at a time; the f32 weight then takes
// one v_fma_mix and is the one dequant.rs rounds (dl·q is exact in f32), and the
// product one more. What bounds it is the VALU, ≈ 5 instructions per weight (≈ 8 µs
// of issue for 14336 × 4096, whose bytes take 5) against ≈ 12 and five narrow
// loads in k_col. Q3_K, one row: 14336 × 4096 53.5 → 17.7 µs, 4096 × 4096 17.9 →
// 8.9, 1024 × 4096 7.9 → 6.4; eight rows of 4096 × 4096 41.5 → 20.9.
typedef _Float16 xh2 __attribute__((ext_vector_type(2)));
// Bytes (0, 1) or (2, 3) of w as the half pair b·2^-24 (the half with bits b: a subnormal, exact, and so are
// its products with integers up to 2^10 in all), and as 1024 + b.
template <int HI> __device__ __forceinline__ xh2 xk_tiny(uint32_t w) {
    return __builtin_bit_cast(xh2, __builtin_amdgcn_perm(0u, w, HI ? 0x0C030C02u : 0x0C010C00u));
}
template <int HI> __device__ __forceinline__ xh2 xk_1024(uint32_t w) {
    return __builtin_bit_cast(xh2, __builtin_amdgcn_perm(0x64646464u, w, HI ? 0x07030702u : 0x07010700u));
}
__device__ __forceinline__ xh2 xk_both(_Float16 v) { return (xh2){v, v}; }

template <int F> struct XK;
template <> struct XK<AETH_DTYPE_Q2_K> {
    static constexpr int BB = Q2K_BLOCK_BYTES;
    struct Raw { uint32_t dd, q; uint2 sc; };
    __device__ static Raw load(const uint8_t* b, int u) {
        Raw r;
        r.dd = *(const uint32_t*)b;  // blocks are 4-byte aligned
        const uint32_t* sp = (const uint32_t*)(b + 4 + (u & 8));
        r.sc = make_uint2(sp[0], sp[1]);
        r.q = *(const uint32_t*)(b + 20 + 4 * u);
        return r;
    }
    uint32_t q, sc4;
    xh2 s01, s23;  // the sub-blocks' scales
    float d, dmin;
    __device__ XK(const Raw& r, int u) {
        // bytes v, 2 + v, 4 + v, 6 + v: sub-blocks t = 0..3
        sc4 = __builtin_amdgcn_perm(r.sc.y, r.sc.x, (u & 4) ? 0x07050301u : 0x06040200u);
        s01 = xk_1024<0>(sc4 & 0x0F0F0F0Fu) - xk_both((_Float16)1024.0f);
        s23 = xk_1024<1>(sc4 & 0x0F0F0F0Fu) - xk_both((_Float16)1024.0f);
        q = r.q;
        d = aeth_decode_d(r.dd & 0xFFFFu) * 0x1p24f;  // over the quants' 2^-24
        dmin = aeth_decode_d(r.dd >> 16);
    }
    __device__ __forceinline__ void weights(int t, float (&w)[4]) const {  // d·(sc·q) − dmin·m, one rounding
        const uint32_t b = (q >> (2 * t)) & 0x03030303u;
        const xh2 s = xk_both(t < 2 ? s01[t & 1] : s23[t & 1]);
        const xh2 a = xk_tiny<0>(b) * s, c = xk_tiny<1>(b) * s;
        const float ml = -(dmin * (float)((sc4 >> (8 * t + 4)) & 15));
        w[0] = fmaf((float)a[0], d, ml);
        w[1] = fmaf((float)a[1], d, ml);
        w[2] = fmaf((float)c[0], d, ml);
        w[3] = fmaf((float)c[1], d, ml);
    }
};
template <> struct XK<AETH_DTYPE_Q3_K> {
    static constexpr int BB = Q3K_BLOCK_BYTES;
    struct Raw { uint32_t q, hm, s0, s1, s2, d; };
    __device__ static uint32_t ld32(const uint8_t* p) {  // blocks are 2-byte aligned
        uint32_t v;
        __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 4);
        return v;
    }
    __device__ static Raw load(const uint8_t* b, int u) {
        Raw r;
        r.q = ld32(b + 32 + 4 * u);
        r.hm = ld32(b + 4 * (u & 7));
        r.s0 = ld32(b + 96);
        r.s1 = ld32(b + 100);
        r.s2 = ld32(b + 104);
        r.d = *(const uint16_t*)(b + 108);
        return r;
    }
    uint32_t q, hm;
    xh2 s01, s23;
    float d;
    __device__ XK(const Raw& r, int u) {
        // sub-block s = 8h + 2t + v: low nibble h of byte 2t + v, high pair h·2 + t/2 of byte 8 + 2(t % 2) + v
        const int h = u >> 3;
        const uint32_t lo = __builtin_amdgcn_perm(r.s1, r.s0, (u & 4) ? 0x07050301u : 0x06040200u) >> (4 * h);
        const uint32_t hi = __builtin_amdgcn_perm(0u, r.s2, (u & 4) ? 0x03010301u : 0x02000200u) >> (4 * h);
        const uint32_t sc4 = (lo & 0x0F0F0F0Fu) | (((hi & 0x0303u) | ((hi >> 2) & 0x03030000u)) << 4);
        s01 = xk_1024<0>(sc4) - xk_both((_Float16)1056.0f);  // sc − 32
        s23 = xk_1024<1>(sc4) - xk_both((_Float16)1056.0f);
        q = r.q;
        hm = h ? r.hm >> 2 : r.hm << 2;  // bit 4h + t of a byte at 2 + t
        d = aeth_decode_d(r.d);
    }
    __device__ __forceinline__ void weights(int t, float (&w)[4]) const {  // d·((sc − 32)·(q − 4))
        // q = low pair | high bit · 4 selects the high byte of the half q − 4 (its low byte is 0)
        const uint32_t b = ((q >> (2 * t)) & 0x03030303u) | ((hm >> t) & 0x04040404u);
        const uint32_t v = __builtin_amdgcn_perm(0x42403C00u, 0xBCC0C2C4u, b);
        const xh2 s = xk_both(t < 2 ? s01[t & 1] : s23[t & 1]);
        const xh2 a = __builtin_bit_cast(xh2, __builtin_amdgcn_perm(0u, v, 0x010C000Cu)) * s;
        const xh2 c = __builtin_bit_cast(xh2, __builtin_amdgcn_perm(0u, v, 0x030C020Cu)) * s;
        w[0] = fmaf((float)a[0], d, 0.0f);
        w[1] = fmaf((float)a[1], d, 0.0f);
        w[2] = fmaf((float)c[0], d, 0.0f);
        w[3] = fmaf((float)c[1], d, 0.0f);
    }
};

#define COLK_WAVES 8
constexpr int colk_nb(int R) { return R > 4 ? 2 : 4; }  // inputs of a wave in flight

// Split s of k: inputs [chunk·s, chunk·(s + 1)).
template <int F, int R>
__global__ void __launch_bounds__(64 * COLK_WAVES) k_colk(const uint8_t* __restrict__ W, int64_t n, int k, int chunk,
                                                          const float* __restrict__ x, int64_t ldx, int m,
                                                          float* __restrict__ part) {
    constexpr int NB = colk_nb(R);
    __shared__ __attribute__((aligned(16))) float red[COLK_WAVES][1024];
    const int lane = threadIdx.x & 63, u = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nbk = (int)(n >> 8), blk = min((int)blockIdx.x * 4 + (lane >> 4), nbk - 1);  // past n: discarded
    const int s = blockIdx.y, r0 = blockIdx.z * R;
    const int i0 = chunk * s, i1 = min(k, i0 + chunk);
    const uint8_t* Wb = W + (int64_t)blk * XK<F>::BB;
    const int64_t row = (int64_t)nbk * XK<F>::BB;
    float acc[R][16];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[r][e] = 0.0f;
    for (int ib = i0 + wave; ib < i1; ib += COLK_WAVES * NB) {
        typename XK<F>::Raw raw[NB];
        float xv[NB][R];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int i = ib + b * COLK_WAVES, ic = min(i, i1 - 1);
            raw[b] = XK<F>::load(Wb + ic * row, u);
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float v = x[(int64_t)min(r0 + r, m - 1) * ldx + ic];
                xv[b][r] = i < i1 ? v : 0.0f;  // past the split: counts nothing (the weights are finite)
            }
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const XK<F> wk(raw[b], u);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                float w[4];
                wk.weights(t, w);
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[r][4 * t + e] = fmaf(xv[b][r], w[e], acc[r][4 * t + e]);
            }
        }
    }
    // the waves' sums meet in LDS, a row at a time
    float* mine = red[wave] + 256 * (lane >> 4) + 128 * (u >> 3) + 4 * (u & 7);
    const int64_t j0 = (int64_t)blockIdx.x * 1024;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (r) __syncthreads();
#pragma unroll
        for (int t = 0; t < 4; t++)
            *(float4*)(mine + 32 * t) = make_float4(acc[r][4 * t], acc[r][4 * t + 1], acc[r][4 * t + 2], acc[r][4 * t + 3]);
        __syncthreads();
        if (r0 + r < m)
            for (int e = threadIdx.x; e < 1024 && j0 + e < n; e += 64 * COLK_WAVES) {
                static_assert(COLK_WAVES == 8, "summed as a tree");
                part[((int64_t)s * m + r0 + r) * n + j0 + e] =
                    ((red[0][e] + red[1][e]) + (red[2][e] + red[3][e])) + ((red[4][e] + red[5][e]) + (red[6][e] + red[7][e]));
            }
    }
}

// Σ over the S splits, then y = (accumulate ? y : 0) + Σ, and the argmax key.
// A workgroup takes 4·LN consecutive outputs of the [m][n] result (n % 4 == 0:
// a float4 never crosses a row), G groups of LN threads every G-th split each,
// 8 loads in flight a thread, met through LDS in group order: fixed order,
// contiguous reads (LN = 16 with 16 groups: 1024 outputs of 128 splits spread
// over 16 workgroups; 256-output workgroups of 1024 threads took 0.6 µs more). The sums run in f64, free beside the loads: with up to
// 128 partials they were most of a product's rounding error.
template <int G, int LN>
__global__ void __launch_bounds__(LN * G) k_col_reduce(const float* __restrict__ part, int S, int64_t m, int64_t n,
                                                       float* __restrict__ y, int64_t ldy, int accumulate,
                                                       unsigned long long* __restrict__ amax) {
    static_assert(4 * LN % 64 == 0 && LN * G % 64 == 0, "whole waves");
    __shared__ __attribute__((aligned(16))) double red[G][4 * LN];
    const int l = threadIdx.x % LN, g = threadIdx.x / LN;
    const int64_t total = m * n, base = (int64_t)blockIdx.x * (4 * LN);
    {
        const float* src = part + min(base + 4 * l, total - 4);  // past the end: discarded below
        double a[4] = {0.0, 0.0, 0.0, 0.0};
        for (int s = g; s < S; s += 8 * G) {
            float4 p[8];
#pragma unroll
            for (int u = 0; u < 8; u++) p[u] = *(const float4*)(src + min(s + u * G, S - 1) * total);
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const bool in = s + u * G < S;
                a[0] += in ? p[u].x : 0.0f; a[1] += in ? p[u].y : 0.0f;
                a[2] += in ? p[u].z : 0.0f; a[3] += in ? p[u].w : 0.0f;
            }
        }
        *(double2*)&red[g][4 * l] = make_double2(a[0], a[1]);
        *(double2*)&red[g][4 * l + 2] = make_double2(a[2], a[3]);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 4 * LN; e += LN * G) {  // whole waves
        const int64_t idx = base + e;
        double a = red[0][e];
#pragma unroll
        for (int q = 1; q < G; q++) a += red[q][e];
        unsigned long long best = 0;
        if (idx < total) {
            const int64_t row = idx / n, j = idx - row * n;
            float* dst = y + row * ldy + j;
            float v = (float)a;
            if (accumulate) v = *dst + v;
            *dst = v;
            if (amax) best = aeth_amax_key(v, j);
        }
        if (amax) {
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) {
                const unsigned long long o = __shfl_xor(best, off, 64);
                best = o > best ? o : best;
            }
            if ((threadIdx.x & 63) == 0 && best) atomicMax(amax, best);
        }
    }
}

// Rows: y[row][j] = Σ_e x[row][e]·W[j][e], a wave per output j, R rows.
// Row j's elements start at flat element j·row_elems (K-quants: k/256 whole
// blocks per row; F16: k values, k % 4 == 0); NB units per batch, loads first.
template <int F, int R>
__global__ void __launch_bounds__(256) k_row(const uint8_t* __restrict__ W, int64_t n, int64_t kr, int64_t row_elems,
                                             const float* __restrict__ x, int64_t ldx, int m, float* __restrict__ y,
                                             int64_t ldy, int accumulate) {
    constexpr int NB = 4;
    typedef typename XU<F>::Raw Raw;
    const int lane = threadIdx.x & 63;
    const int64_t j = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = blockIdx.y * R;
    if (j >= n) return;
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
    const float* xr[R];
#pragma unroll
    for (int r = 0; r < R; r++) xr[r] = x + (int64_t)min(r0 + r, m - 1) * ldx;
    for (int64_t eb = 4 * lane; eb < kr + 4 * lane; eb += 256 * NB) {  // kr: elements per row (a multiple of 4)
        Raw raw[NB];
        float4 xv[NB][R];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int64_t e = eb + 256 * b, ec = e < kr ? e : kr - 4;
            raw[b] = XU<F>::load(W, j * row_elems + ec);
#pragma unroll
            for (int r = 0; r < R; r++) {
                xv[b][r] = *(const float4*)(xr[r] + ec);
                if (e >= kr) xv[b][r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
            float w[4];
            XU<F>::expand(raw[b], w);
#pragma unroll
            for (int r = 0; r < R; r++) {
                acc[r] = fmaf(xv[b][r].x, w[0], acc[r]);
                acc[r] = fmaf(xv[b][r].y, w[1], acc[r]);
                acc[r] = fmaf(xv[b][r].z, w[2], acc[r]);
                acc[r] = fmaf(xv[b][r].w, w[3], acc[r]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const float v = aeth_wave_sum(acc[r]);
        if (lane == 0 && r0 + r < m) {
            float* dst = y + (int64_t)(r0 + r) * ldy + j;
            *dst = accumulate ? *dst + v : v;
        }
    }
}

// Q2_K / Q3_K whose inputs are whole blocks run k_colk (every GGUF tensor with n % 256 == 0)
bool col_packed(const aeth_weight* w) {
    return (w->dtype == AETH_DTYPE_Q2_K || w->dtype == AETH_DTYPE_Q3_K) && w->n % 256 == 0 && w->k <= INT32_MAX / 2 &&
           w->n <= INT32_MAX;
}
int colk_rows(int64_t m) { return m == 1 ? 1 : m <= 4 ? 4 : 8; }  // rows a workgroup forms from one read of the weight

// Inputs per split of a k_colk launch: whole batches of every wave (no wave's last batch is part
// empty), as few as leave 2 workgroups per CU for one row, 1 for more (a partial row of results per split
// costs the reduction more than it gives there), at most 128 splits. 14336 × 4096 / 4096 × 4096 Q3_K, one
// row: 1 per CU 19.8 / 10.0 µs, 2 18.7 / 9.8, 3 19.4 / 9.8; four rows of 4096 × 4096: 14.9, 16.7, 16.7.
int colk_chunk(const aeth_weight* w, int64_t m) {
    const int R = colk_rows(m), batch = COLK_WAVES * colk_nb(R);
    const int64_t per_cu = R == 1 ? 2 : 1;
    const int64_t wgs = aeth_cdiv(w->n, 1024) * aeth_cdiv(m, R), fit = std::max<int64_t>(1, per_cu * aeth_num_cus() / wgs);
    const int64_t S = std::min<int64_t>(fit, 128);
    return (int)(aeth_cdiv(aeth_cdiv(w->k, S), batch) * batch);
}

template <int F, int R>
void launch_colk(const aeth_weight* w, const float* x, int64_t m, float* part, int S, hipStream_t s) {
    const dim3 grid((unsigned)aeth_cdiv(w->n, 1024), (unsigned)S, (unsigned)aeth_cdiv(m, R));
    hipLaunchKernelGGL((k_colk<F, R>), grid, dim3(64 * COLK_WAVES), 0, s, w->p0, w->n, (int)w->k,
                       colk_chunk(w, m), x, w->k, (int)m, part);
}

template <int F>
int launch_col(const aeth_weight* w, const float* x, int64_t m, float* y, int64_t ldy, const GemvEpi& e,
               float* part, int S, hipStream_t s) {
    const int64_t units = aeth_cdiv(w->n, 256);
    bool done = false;
    if constexpr (F == AETH_DTYPE_Q2_K || F == AETH_DTYPE_Q3_K) {
        if ((done = col_packed(w))) {
            const int R = colk_rows(m);
            if (R == 1) launch_colk<F, 1>(w, x, m, part, S, s);
            else if (R == 4) launch_colk<F, 4>(w, x, m, part, S, s);
            else launch_colk<F, 8>(w, x, m, part, S, s);
        }
    }
    if (!done && m == 1) {
        const dim3 grid((unsigned)units, (unsigned)S, 1);
        hipLaunchKernelGGL((k_col<F, 1, 8>), grid, dim3(512), 0, s, w->p0, w->n, w->k, x, w->k, 1, S, part);
    } else if (!done) {
        const dim3 grid((unsigned)units, (unsigned)S, (unsigned)aeth_cdiv(m, 8));
        hipLaunchKernelGGL((k_col<F, 8, 4>), grid, dim3(256), 0, s, w->p0, w->n, w->k, x, w->k, (int)m, S, part);
    }
    AETH_LAUNCH_CHECK();
    const int64_t tot = m * w->n;
    const int acc = (e.flags & AETH_MM_ACCUMULATE) ? 1 : 0;
    // 16 groups where there are splits for them to share
    if (S > 8) hipLaunchKernelGGL((k_col_reduce<16, 16>), dim3((unsigned)aeth_cdiv(tot, 64)), dim3(256), 0, s, part, S, m, w->n, y, ldy, acc, e.amax);
    else hipLaunchKernelGGL((k_col_reduce<1, 64>), dim3((unsigned)aeth_cdiv(tot, 256)), dim3(64), 0, s, part, S, m, w->n, y, ldy, acc, e.amax);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}

template <int F>
int launch_row(const aeth_weight* w, const float* x, int64_t m, float* y, int64_t ldy, unsigned flags, hipStream_t s) {
    const bool f16 = F == AETH_DTYPE_F16;
    const int64_t kr = f16 ? w->k : w->k / 256 * 256, row_elems = kr;
    const int R = m == 1 ? 1 : 8;
    const dim3 grid((unsigned)aeth_cdiv(w->n, 4), (unsigned)aeth_cdiv(m, R));
    const int acc = (flags & AETH_MM_ACCUMULATE) ? 1 : 0;
    if (R == 1)
        hipLaunchKernelGGL((k_row<F, 1>), grid, dim3(256), 0, s, w->p0, w->n, kr, row_elems, x, w->k, (int)m, y, ldy,
                           acc);
    else
        hipLaunchKernelGGL((k_row<F, 8>), grid, dim3(256), 0, s, w->p0, w->n, kr, row_elems, x, w->k, (int)m, y, ldy,
                           acc);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}

// Splits of k for a GGUF-order launch: enough workgroups to cover the chip
// (≈ 4 per CU), at least one batch of inputs (8 per wave) per wave.
int col_splits(const aeth_weight* w, int64_t m) {
    const int64_t units = aeth_cdiv(w->n, 256), groups = m == 1 ? 1 : aeth_cdiv(m, 8);
    const int64_t per_wave_batch = m == 1 ? 64 : 32;  // NW·NB inputs
    if (col_packed(w)) return (int)aeth_cdiv(w->k, colk_chunk(w, m));
    int64_t S = aeth_cdiv(4LL * aeth_num_cus(), units * groups);
    const int64_t smax = w->k / per_wave_batch > 1 ? w->k / per_wave_batch : 1;
    S = S < 1 ? 1 : S > 128 ? 128 : S;
    return (int)(S < smax ? S : smax);
}

}  // namespace

int64_t aeth_xgemv_ws_floats(const aeth_weight* w, int64_t m) {
    if (!w || w->order != AETH_ORDER_GGUF || m <= 0) return 0;
    return (int64_t)col_splits(w, m) * m * w->n + m * w->k;  // partials + a normed copy of x
}

int aeth_xgemv_launch(const aeth_weight* w, const float* d_x, int64_t m, float* d_y, const GemvEpi& e,
                      hipStream_t s) {
    if (m <= 0 || m > 65535) return aeth_set_error(AETH_EINVAL, "gemv: m=%lld out of range", (long long)m);
    if (e.swiglu) return aeth_set_error(AETH_EUNSUPPORTED, "gemv: fused SwiGLU needs a planar weight");
    const int64_t ldy = e.ldc ? e.ldc : w->n;
    if (w->order == AETH_ORDER_ROWS) {
        if (((uintptr_t)d_x & 15) || (m > 1 && (w->k & 3)))  // float4 activation loads
            return aeth_set_error(AETH_EINVAL, "gemv: x rows must be 16-byte aligned");
        if (e.norm_w || e.amax)
            return aeth_set_error(AETH_EUNSUPPORTED, "gemv: row-order weights take no fused norm or argmax");
        switch (w->dtype) {
            case AETH_DTYPE_F16: return launch_row<AETH_DTYPE_F16>(w, d_x, m, d_y, ldy, e.flags, s);
            case AETH_DTYPE_Q2_K: return launch_row<AETH_DTYPE_Q2_K>(w, d_x, m, d_y, ldy, e.flags, s);
            case AETH_DTYPE_Q3_K: return launch_row<AETH_DTYPE_Q3_K>(w, d_x, m, d_y, ldy, e.flags, s);
            default: return aeth_set_error(AETH_EUNSUPPORTED, "gemv: no row kernel for dtype %d", w->dtype);
        }
    }
    if (w->order != AETH_ORDER_GGUF) return aeth_set_error(AETH_EINVAL, "gemv: weight order %d", w->order);
    const int S = col_splits(w, m);
    const int64_t need = aeth_xgemv_ws_floats(w, m);
    float* ws = e.ws;
    if (ws && e.ws_floats < need)
        return aeth_set_error(AETH_EINVAL, "gemv: scratch of %lld floats < %lld needed", (long long)e.ws_floats,
                              (long long)need);
    if (!ws) {  // the library's scratch of this stream
        void* p = nullptr;
        int rc = aeth_stream_scratch(s, AETH_SCRATCH_XGEMV, (size_t)need * sizeof(float), &p);
        if (rc) return rc;
        ws = (float*)p;
    }
    float* part = ws;
    const float* x = d_x;
    if (e.norm_w) {  // rmsnorm_inplace (runner.rs:1739-1746) into the scratch, then the product
        float* xn = ws + (int64_t)S * m * w->n;
        int rc = aeth_rmsnorm_launch(d_x, e.norm_w, m, w->k, e.eps, xn, s);
        if (rc) return rc;
        x = xn;
    }
    switch (w->dtype) {
        case AETH_DTYPE_F32: return launch_col<AETH_DTYPE_F32>(w, x, m, d_y, ldy, e, part, S, s);
        case AETH_DTYPE_F16: return launch_col<AETH_DTYPE_F16>(w, x, m, d_y, ldy, e, part, S, s);
        case AETH_DTYPE_Q2_K: return launch_col<AETH_DTYPE_Q2_K>(w, x, m, d_y, ldy, e, part, S, s);
        case AETH_DTYPE_Q3_K: return launch_col<AETH_DTYPE_Q3_K>(w, x, m, d_y, ldy, e, part, S, s);
        default: return aeth_set_error(AETH_EUNSUPPORTED, "gemv: no GGUF-order kernel for dtype %d", w->dtype);
    }
}
