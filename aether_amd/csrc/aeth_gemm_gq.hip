// Prefill product of GGUF-order Q2_K / Q3_K weights (m rows from aeth_gq_gemm_rows on):
//   C[r][j] = Σ_i A[r][i]·W[i][j],  W = dequantize(b, [k, n]) (quantized_matmul_impl's fallback,
//   src/quant/matmul/dispatch.rs:126-133, 541-574),
// on the int8 matrix cores, exact up to the rounding of A·d to 31 bits. Blocks run along n, so input i has one
// d (and dmin) per 256 outputs and W[i][j] = d_i·v_ij (Q3_K, v = (sc − 32)·(q − 4)) or d_i·v_ij − dmin_i·m_ij
// (Q2_K, v = sc·q, m the 4-bit min of j's 16 outputs), where v and m are small integers:
//   C[r][j] = Σ_i (A[r][i]·d_i)·v_ij − Σ_i (A[r][i]·dmin_i)·m_ij.
// Per (row, 256 outputs, K part) x_i = A[r][i]·d_i becomes an integer of 31 bits against the largest |x_i| of
// those inputs — formed from the product and its rounding error, so the conversion truncates once, below 2^-29 of
// that maximum — and four balanced signed byte digits of it are four A operands of v_mfma_i32_32x32x32_i8. The i32
// sums are exact (2^14·k), the digits meet in f64 and one rounding to f32 is left: 2.5e-8 of a result, what the
// f64 product (a dequantized weight and rocBLAS DGEMM) gave before. 31 bits do as long as the maximum is not far above
// the rest, an activation or a block scale out of proportion, whose integer weight may well be 0 in an output: a unit
// is to stay below 2^-24 of the geometric mean of the sums of four |x_i|, that is, the maximum below 2^5 of it (normal
// activations under half-normal scales reach 2^2.5, behind a SiLU gate 2^4). Where some row of a workgroup has more, it
// takes a second product, of the next 30 bits (one run, Q3_K 203 × 4096 × 4096: 49.5 µs without, 75 .. 82 with).
//
//  1. k_gq_prep: the blocks unpacked to v (int8) in MFMA operand order, and d as f32.
//  2. k_gq_gemm: workgroup = 64 rows × 256 outputs. A first pass over its A finds each row's largest |A·d|; then
//     its 8 waves convert 64 × 64 of A to digits in LDS (each thread 8 elements) and multiply them, each wave 32
//     rows by 64 outputs, 16 MFMAs between two barriers; of the two waves of a SIMD one converts the next
//     64 inputs while the other multiplies. When the tiles are few, K is split over workgroups and the f64
//     partial results (scaled by their own exponents) are added in order (k_narrow).
// A row of whose products one is not finite (an infinite or NaN activation, or an overflow), or of which 61 bits would
// not do, is summed in f64 element by element instead, as the f64 product did.
//
// What bounds it: bytes into the CUs (per 64 inputs 16 KiB of A and twice 16 KiB of v for 1024 clocks of MFMA;
// without the products the kernel still takes three quarters of its time), then the first pass over A. Q3_K, m =
// 203, 4096 × 4096: 189 → 45 µs (unpack 9.3, product 33, sum 6.3), m = 512, 14336 × 4096: 1197 → 196 µs.
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "aeth_common.hpp"
#include "aeth_gemm_common.hpp"
#include "aeth_internal.hpp"

#pragma clang fp contract(off)

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

#define GQ_KS 64        // inputs per step
#define GQ_BAD 0x7FFF   // exponent of a row that is summed element by element
#define GQ_NAN 0x7FFE   // exponent of a row with a NaN activation: its outputs are NaN
#define GQ_LOW 30       // bits of the second product

struct GqArgs {
    const uint8_t* raw;   // [k][n/256] blocks
    const float* A;       // [m][k]
    int m, n, k, kp, nB;  // kp: k rounded up to GQ_KS
    int8_t* v;            // [nB][kp/32][8 column tiles][64 lanes][16]
    float* d;             // [nB][kp]
    int8_t* mins;         // Q2_K: [nB][kp/32][64 lanes][16], 16 columns of 32 used
    float* dmin;
    int gm, ksplit;
    double* part;         // [ksplit][m][n]: the parts' results, or those of a first product
    float* C;
    int64_t ldc;
    int accumulate;
};

template <int F> struct Gq;
template <> struct Gq<AETH_DTYPE_Q2_K> {
    static constexpr int BB = Q2K_BLOCK_BYTES, D = 0;
    static constexpr bool MIN = true;
};
template <> struct Gq<AETH_DTYPE_Q3_K> {
    static constexpr int BB = Q3K_BLOCK_BYTES, D = 108;
    static constexpr bool MIN = false;
};

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
// (b0·s, b1·s, b2·s, b3·s) mod 256 of a dword's bytes less `off`
__device__ __forceinline__ uint32_t gq_mul4(uint32_t b, uint16_t off, uint16_t s) {
    const u16x2 o = {off, off}, sv = {s, s};
    const u16x2 lo = (__builtin_bit_cast(u16x2, __builtin_amdgcn_perm(0u, b, 0x0C010C00u)) - o) * sv;
    const u16x2 hi = (__builtin_bit_cast(u16x2, __builtin_amdgcn_perm(0u, b, 0x0C030C02u)) - o) * sv;
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x06040200u);
}
// four dwords of four bytes → their transpose
__device__ __forceinline__ void gq_transpose(const uint32_t (&r)[4], uint32_t (&c)[4]) {
    const uint32_t a = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u), b = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);
    const uint32_t e = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u), f = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
    c[0] = __builtin_amdgcn_perm(e, a, 0x05040100u);
    c[1] = __builtin_amdgcn_perm(e, a, 0x07060302u);
    c[2] = __builtin_amdgcn_perm(f, b, 0x05040100u);
    c[3] = __builtin_amdgcn_perm(f, b, 0x07060302u);
}
__device__ __forceinline__ uint32_t gq_ld32(const uint8_t* p) {  // Q3_K blocks are 2-byte aligned
    uint32_t v;
    __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 4);
    return v;
}

// One block's qs dword u: for t = 0..3 the products of its four elements at outputs 128h + 32t + 4(u % 8) + c,
// and the mins of sub-blocks 8h + 2t + v in the bytes of mn (Q2_K).
template <int F>
__device__ __forceinline__ void gq_block(const uint8_t* b, int u, uint32_t (&p)[4], uint32_t& mn) {
    const uint32_t sel = (u & 4) ? 0x07050301u : 0x06040200u;  // bytes v, 2 + v, 4 + v, 6 + v
    if constexpr (F == AETH_DTYPE_Q2_K) {
        const uint32_t* sp = (const uint32_t*)(b + 4 + (u & 8));
        const uint32_t sc = __builtin_amdgcn_perm(sp[1], sp[0], sel), q = *(const uint32_t*)(b + 20 + 4 * u);
        mn = (sc >> 4) & 0x0F0F0F0Fu;
#pragma unroll
        for (int t = 0; t < 4; t++) p[t] = gq_mul4((q >> (2 * t)) & 0x03030303u, 0, (sc >> (8 * t)) & 15);
    } else {
        const int h = u >> 3;
        const uint32_t q = gq_ld32(b + 32 + 4 * u), hm = gq_ld32(b + 4 * (u & 7));
        const uint32_t s0 = gq_ld32(b + 96), s1 = gq_ld32(b + 100), s2 = gq_ld32(b + 104);
        const uint32_t lo = __builtin_amdgcn_perm(s1, s0, sel) >> (4 * h);
        const uint32_t hi = __builtin_amdgcn_perm(0u, s2, (u & 4) ? 0x03010301u : 0x02000200u) >> (4 * h);
        const uint32_t sc = (lo & 0x0F0F0F0Fu) | (((hi & 0x0303u) | ((hi >> 2) & 0x03030000u)) << 4);
        const uint32_t h2 = h ? hm >> 2 : hm << 2;  // bit 4h + t of a byte at 2 + t
        mn = 0;
        // (32 − sc)·(q − 4): the negative of v, whose range −124 .. 128 is one past a signed byte's
#pragma unroll
        for (int t = 0; t < 4; t++)
            p[t] = gq_mul4(((q >> (2 * t)) & 0x03030303u) | ((h2 >> t) & 0x04040404u), 4,
                           (uint16_t)(32 - (int)((sc >> (8 * t)) & 63)));
    }
}

template <int F>
__device__ __forceinline__ float gq_scale(const uint8_t* b, int which) {
    return aeth_decode_d(*(const uint16_t*)(b + Gq<F>::D + 2 * which));
}

template <int F>
__global__ void __launch_bounds__(256) k_gq_prep(GqArgs G) {
    constexpr int BB = Gq<F>::BB, NT = Gq<F>::MIN ? 2 : 1;
    __shared__ __attribute__((aligned(16))) uint32_t sh[4096 * NT];
    const int tid = threadIdx.x;
    const int64_t row = (int64_t)G.nB * BB;
    // block column B, inputs [64·ks, +64): thread = 4 inputs × qs dword u
    const int kst = G.kp / GQ_KS, B = blockIdx.x / kst, ks = blockIdx.x - B * kst;
    const int u = tid & 15, g = tid >> 4, i0 = GQ_KS * ks + 4 * g;
    const uint8_t* src = G.raw + (int64_t)B * BB;
    uint32_t p[4][4], mn[4];  // [input][t]
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const bool in = i0 + r < G.k;
        const uint8_t* b = src + min(i0 + r, G.k - 1) * row;
        gq_block<F>(b, u, p[r], mn[r]);
#pragma unroll
        for (int t = 0; t < 4; t++) p[r][t] = in ? p[r][t] : 0u;
        mn[r] = in ? mn[r] : 0u;
        if (u == 0) {
            G.d[(int64_t)B * G.kp + i0 + r] = in ? gq_scale<F>(b, 0) : 0.0f;
            if (Gq<F>::MIN) G.dmin[(int64_t)B * G.kp + i0 + r] = in ? gq_scale<F>(b, 1) : 0.0f;
        }
    }
    // operand bytes: (32-input step, column tile, lane = column + 32·(input half), input % 16)
    const int kk = 4 * g, at = ((kk >> 5) * 8 * 64 + 32 * ((kk >> 4) & 1)) * 4 + ((kk & 15) >> 2);
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const uint32_t r[4] = {p[0][t], p[1][t], p[2][t], p[3][t]};
        uint32_t c[4];
        gq_transpose(r, c);
#pragma unroll
        for (int e = 0; e < 4; e++) sh[at + ((4 * (u >> 3) + t) * 64 + 4 * (u & 7) + e) * 4] = c[e];
    }
    if (Gq<F>::MIN) {
        uint32_t* shm = sh + 4096;  // [step 2][64 lanes][16 B]
        for (int i = tid; i < 512; i += 256) shm[i] = 0u;
        __syncthreads();
        if ((u & 3) == 0) {
            uint32_t c[4];  // column t: the four inputs' mins of sub-block 8h + 2t + v
            gq_transpose(mn, c);
#pragma unroll
            for (int t = 0; t < 4; t++)
                shm[((kk >> 5) * 64 + 32 * ((kk >> 4) & 1) + 8 * (u >> 3) + 2 * t + ((u >> 2) & 1)) * 4 + ((kk & 15) >> 2)] = c[t];
        }
    }
    __syncthreads();
    uint4* dst = (uint4*)(G.v + ((int64_t)B * G.kp + GQ_KS * ks) * 256);
#pragma unroll
    for (int i = 0; i < 4; i++) dst[tid + 256 * i] = ((const uint4*)sh)[tid + 256 * i];
    if (Gq<F>::MIN && tid < 128)
        ((uint4*)(G.mins + ((int64_t)B * G.kp + GQ_KS * ks) * 32))[tid] = ((const uint4*)(sh + 4096))[tid];
}

__device__ __forceinline__ int gq_trunc(float f) {  // the instruction's own rule for what does not fit (NaN: 0)
    int i;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(f));
    return i;
}

// a·d's integer part as bytes of four digits, 0 .. 2 biased by 128; LOW: the GQ_LOW bits behind it
template <bool LOW> __device__ __forceinline__ uint32_t gq_digits(float a, float d) {
    const float p = a * d, er = fmaf(a, d, -p);
    if (!LOW) return (uint32_t)(gq_trunc(p) + gq_trunc(rintf(er))) + 0x808080u;
    constexpr float up = (float)(1 << GQ_LOW);  // both fractions are exact, their sum is below 1.5
    return (uint32_t)(gq_trunc((p - truncf(p)) * up) + gq_trunc((er - rintf(er)) * up)) + 0x808080u;
}

struct GqShared {
    // digit operands [buffer 2][32-input step 2][m-tile 2][digit 4][64 lanes][16 B]: 32 KiB
    uint8_t dig[2][16384];
    int Sx[2][64];  // the rows' exponents over this workgroup's inputs: of A·d, of A·dmin
};

// Four floats of A and the scales of a step's inputs, by thread (row tid/8, inputs 4·(tid%8) and 32 on)
struct GqRaw { float4 a[2], d[2]; };
template <bool AL16>
__device__ __forceinline__ void gq_load(const GqArgs& G, const float* a_src, const float* sc, int s, int kq, GqRaw& R) {
#pragma unroll
    for (int j = 0; j < 2; j++) {  // inputs past k read any value: their d is 0
        const int i = GQ_KS * s + 32 * j + kq;
        R.d[j] = *(const float4*)(sc + i);
        if (AL16) R.a[j] = *(const float4*)(a_src + min(i, G.k - 4));
        else R.a[j] = make_float4(a_src[min(i, G.k - 1)], a_src[min(i + 1, G.k - 1)], a_src[min(i + 2, G.k - 1)],
                                  a_src[min(i + 3, G.k - 1)]);
    }
}

// The product of one digit set over the steps [s0, s1) of a workgroup. LOW: the second one, added to what the first left
// in `part`; `more`: a second one follows.
template <int F, bool AL16, bool LOW>
__device__ __forceinline__ void gq_product(const GqArgs& G, int tid, int m0, int B, int ks, int s0, int s1, int Srow,
                                           int Srowm, bool more, GqShared& sh, int* msum) {
    constexpr bool MIN = Gq<F>::MIN;
    auto& dig = sh.dig;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rr = tid >> 3, row = min(m0 + rr, G.m - 1), kq = 4 * (tid & 7);  // this thread's row and inputs of A
    const float* a_src = G.A + (int64_t)row * G.k;
    const float* ds = G.d + (int64_t)B * G.kp;
    const float* dm = G.dmin + (int64_t)B * G.kp;  // MIN only
    auto loadA = [&](int s, const float* sc, GqRaw& R) { gq_load<AL16>(G, a_src, sc, s, kq, R); };
    auto convert = [&](const GqRaw& R, int S, uint8_t* buf) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float a[4] = {R.a[j].x, R.a[j].y, R.a[j].z, R.a[j].w}, d[4] = {R.d[j].x, R.d[j].y, R.d[j].z, R.d[j].w};
            uint32_t y[4], c[4];
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = gq_digits<LOW>(__builtin_amdgcn_ldexpf(a[e], S), d[e]);
            gq_transpose(y, c);
            uint32_t* o = (uint32_t*)(buf + j * 8192 + (rr >> 5) * 4096) + ((rr & 31) + 32 * (kq >> 4)) * 4 + ((kq & 15) >> 2);
            o[0] = c[0] ^ 0x80808080u;
            o[256] = c[1] ^ 0x80808080u;
            o[512] = c[2] ^ 0x80808080u;
            o[768] = c[3];
        }
    };

    const int mt = wave & 1, cp = wave >> 1;  // this wave's 32 rows, and column tiles 2cp, 2cp + 1
    i32x16 acc[2][4];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int q = 0; q < 4; q++) acc[c][q] = (i32x16){};
    {
        const i32x4* vb = (const i32x4*)(G.v + (int64_t)B * G.kp * 256) + 2 * cp * 64 + lane;  // + (2s + j)·512 + 64·c
        GqRaw P, Q;
        i32x4 b0[2][2], b1[2][2];
        const int last = s1 - 1;
        auto loadB = [&](int s, i32x4 (&o)[2][2]) {
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int c = 0; c < 2; c++) o[j][c] = vb[(2 * s + j) * 512 + 64 * c];
        };
        auto product = [&](const uint8_t* buf, const i32x4 (&b)[2][2]) {
            i32x4 a[2][4];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) a[j][q] = *(const i32x4*)(buf + ((j * 2 + mt) * 4 + q) * 1024 + lane * 16);
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
#pragma unroll
                    for (int c = 0; c < 2; c++) acc[c][q] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[j][q], b[j][c], acc[c][q], 0, 0, 0);
        };
        // step s: its digits are in `cur`; of a SIMD's waves w and w + 4 one multiplies while the other converts step
        // s + 1 (past the last one into a buffer nobody reads). The loads run two steps ahead.
        auto step = [&](int s, const uint8_t* cur, uint8_t* nxt, i32x4 (&b)[2][2], GqRaw& R) {
            __syncthreads();  // cur is written, and nxt read by every wave
            if (wave < 4) product(cur, b);
            __builtin_amdgcn_sched_barrier(0);
            convert(R, Srow, nxt);
            __builtin_amdgcn_sched_barrier(0);
            if (wave >= 4) product(cur, b);
            loadB(min(s + 2, last), b);
            loadA(min(s + 3, last), ds, R);
            __builtin_amdgcn_sched_barrier(0);
        };
        loadA(s0, ds, P);
        loadB(s0, b0);
        loadB(min(s0 + 1, last), b1);
        convert(P, Srow, dig[0]);
        loadA(min(s0 + 1, last), ds, P);
        loadA(min(s0 + 2, last), ds, Q);
        int s = s0;
        for (; s + 1 < s1; s += 2) {
            step(s, dig[0], dig[1], b0, P);
            step(s + 1, dig[1], dig[0], b1, Q);
        }
        if (s < s1) step(s, dig[0], dig[1], b0, P);
    }
    if constexpr (MIN) {  // the mins' product, 16 columns: wave = (m-tile, digit)
        const i32x4* vb = (const i32x4*)(G.mins + (int64_t)B * G.kp * 32) + lane;
        const int q = wave >> 1;
        i32x16 am = (i32x16){};
        GqRaw R;
        loadA(s0, dm, R);
        __syncthreads();  // the main loop's operands are read
        convert(R, Srowm, dig[0]);
        loadA(min(s0 + 1, s1 - 1), dm, R);
        for (int s = s0; s < s1; s++) {
            const int cur = (s - s0) & 1;
            const i32x4 b0 = vb[(int64_t)(2 * s) * 64], b1 = vb[(int64_t)(2 * s + 1) * 64];
            __syncthreads();
            am = __builtin_amdgcn_mfma_i32_32x32x32_i8(*(const i32x4*)(dig[cur] + (mt * 4 + q) * 1024 + lane * 16), b0, am, 0, 0, 0);
            am = __builtin_amdgcn_mfma_i32_32x32x32_i8(*(const i32x4*)(dig[cur] + ((2 + mt) * 4 + q) * 1024 + lane * 16), b1, am, 0, 0, 0);
            convert(R, Srowm, dig[cur ^ 1]);
            loadA(min(s + 2, s1 - 1), dm, R);
        }
        if ((lane & 31) < 16)
#pragma unroll
            for (int r = 0; r < 16; r++)
                msum[(q * 64 + 32 * mt + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * 16 + (lane & 31)] = am[r];
        __syncthreads();
    }
    const int64_t mn = (int64_t)G.m * G.n;
    constexpr int LB = LOW ? GQ_LOW : 0;
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int lr = 32 * mt + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), cr = m0 + lr;
            const int ce = 32 * (2 * cp + c) + (lane & 31);  // output within the block
            if (cr >= G.m) continue;
            const int S = sh.Sx[0][lr];
            double v = fma((double)acc[c][3][r], 16777216.0,
                           fma((double)acc[c][2][r], 65536.0, fma((double)acc[c][1][r], 256.0, (double)acc[c][0][r])));
            v = ldexp(F == AETH_DTYPE_Q3_K ? 0.0 - v : v, -S - LB);
            if constexpr (MIN) {
                const int* p = msum + lr * 16 + (ce >> 4);
                v -= ldexp(fma((double)p[3072], 16777216.0, fma((double)p[2048], 65536.0, fma((double)p[1024], 256.0, (double)p[0]))),
                           -sh.Sx[1][lr] - LB);
            }
            const int64_t col = 256LL * B + ce;
            double* part = G.part + ks * mn + (int64_t)cr * G.n + col;
            if (LOW) v += *part;
            if (S >= GQ_NAN && !more) {  // rare: element by element in f64
                v = S == GQ_NAN ? __builtin_nan("") : 0.0;
                const int i1 = S == GQ_NAN ? 0 : min(GQ_KS * s1, G.k);
                for (int i = GQ_KS * s0; i < i1 && v == v; i++) {
                    const int8_t q = G.v[((int64_t)B * G.kp + (i & ~31)) * 256 + ((ce >> 5) * 64 + (ce & 31) + 32 * ((i >> 4) & 1)) * 16 + (i & 15)];
                    double w = (double)ds[i] * (double)(F == AETH_DTYPE_Q3_K ? -(int)q : (int)q);
                    if constexpr (MIN)
                        w -= (double)dm[i] *
                             (double)G.mins[((int64_t)B * G.kp + (i & ~31)) * 32 + ((ce >> 4) + 32 * ((i >> 4) & 1)) * 16 + (i & 15)];
                    v += (double)G.A[(int64_t)cr * G.k + i] * w;
                }
            }
            if (G.ksplit > 1 || more) {
                *part = v;
            } else {
                float* dst = G.C + (int64_t)cr * G.ldc + col;
                *dst = G.accumulate ? *dst + (float)v : (float)v;
            }
        }
}

template <int F, bool AL16>
__global__ void __launch_bounds__(512) k_gq_gemm(GqArgs G) {
    constexpr bool MIN = Gq<F>::MIN;
    __shared__ __attribute__((aligned(16))) GqShared sh;
    __shared__ int msum[MIN ? 4 * 64 * 16 : 1];
    const int tid = threadIdx.x;
    // the XCDs take workgroup ids round robin: each gets a contiguous run of tiles, the row tiles of a block column
    // next to each other, so that an XCD reads its part of v once
    const int T = G.gm * G.nB, ks = blockIdx.x / T, id = blockIdx.x - ks * T;
    const int tile = (T & 7) == 0 ? (id & 7) * (T >> 3) + (id >> 3) : id;
    const int tm = tile % G.gm, B = tile / G.gm, m0 = 64 * tm;
    const int nst = G.kp / GQ_KS, s0 = nst * ks / G.ksplit, s1 = nst * (ks + 1) / G.ksplit;

    int Srow, Srowm = 0;
    bool wide = false;
    {  // max |A·d| of the row over this workgroup's inputs: the row's eight threads are neighbouring lanes
        const int rr = tid >> 3, row = min(m0 + rr, G.m - 1), kq = 4 * (tid & 7);
        const float* a_src = G.A + (int64_t)row * G.k;
        const float* ds = G.d + (int64_t)B * G.kp;
        const float* dm = G.dmin + (int64_t)B * G.kp;
        float mx = 0.0f, mxm = 0.0f;
        // sums of four: the upper halves of their bits (2^7·(log2 + 127), about) summed, and how many are not zero
        uint32_t lg = 0, lgm = 0;
        int nz = 0, nzm = 0;
        bool bad = false;
        auto most = [&](const float4& a, const float4& d, float& m, uint32_t& lg, int& nz) {
            const float x = fmaxf(fmaxf(fabsf(a.x * d.x), fabsf(a.y * d.y)), fmaxf(fabsf(a.z * d.z), fabsf(a.w * d.w)));
            const float t = fabsf(a.x * d.x) + fabsf(a.y * d.y) + fabsf(a.z * d.z) + fabsf(a.w * d.w);
            bad |= !(t < INFINITY);  // a NaN or an infinity among them (or four products near overflow)
            lg = __builtin_amdgcn_udot2(__builtin_bit_cast(u16x2, t), (u16x2){0, 1}, lg, false);
            nz += t > 0.0f ? 1 : 0;
            m = fmaxf(m, x);
        };
#pragma unroll 4
        for (int s = s0; s < s1; s++) {
            GqRaw R;
            gq_load<AL16>(G, a_src, ds, s, kq, R);
            most(R.a[0], R.d[0], mx, lg, nz);
            most(R.a[1], R.d[1], mx, lg, nz);
            if constexpr (MIN) {
                most(R.a[0], *(const float4*)(dm + GQ_KS * s + kq), mxm, lgm, nzm);
                most(R.a[1], *(const float4*)(dm + GQ_KS * s + 32 + kq), mxm, lgm, nzm);
            }
        }
        auto sum8 = [](int v) {
            v += aeth_dpp_xor1(v);
            v += aeth_dpp_xor2(v);
            return v + __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, false);
        };
        bool far = false;  // past what the second product holds too
        auto exponent = [&](float v, uint32_t lg, int nz) {  // S with |x|·2^S < 2^30
            v = fmaxf(v, aeth_dpp_xor1f(v));
            v = fmaxf(v, aeth_dpp_xor2f(v));
            v = fmaxf(v, aeth_dpp_mirror8f(v));
            const int over = (int)(__float_as_uint(v) >> 16), sum = sum8((int)lg), n = sum8(nz);
            wide |= (over - 5 * 128) * n > sum;
            far |= (over - (5 + GQ_LOW) * 128) * n > sum;
            int E = 0;
            if (v > 0.0f) (void)frexpf(v, &E);
            return 30 - E;
        };
        Srow = exponent(mx, lg, nz);
        if (MIN) Srowm = exponent(mxm, lgm, nzm);
        bad = sum8(bad ? 1 : 0) != 0;
        bool nan = false;
        if (bad) {
            wide = false;
            for (int s = s0; s < s1; s++) {
                GqRaw R;
                gq_load<AL16>(G, a_src, ds, s, kq, R);
#pragma unroll
                for (int j = 0; j < 2; j++) nan |= R.a[j].x != R.a[j].x || R.a[j].y != R.a[j].y || R.a[j].z != R.a[j].z || R.a[j].w != R.a[j].w;
            }
            nan = sum8(nan ? 1 : 0) != 0;
        }
        if ((tid & 7) == 0) {
            sh.Sx[0][rr] = nan ? GQ_NAN : bad || far ? GQ_BAD : Srow;
            if (MIN) sh.Sx[1][rr] = Srowm;
        }
    }
    wide = __builtin_amdgcn_readfirstlane(__syncthreads_or(wide));
    gq_product<F, AL16, false>(G, tid, m0, B, ks, s0, s1, Srow, Srowm, wide, sh, msum);
    if (wide) {
        int t = tid;  // the second product's addresses are formed anew: nothing of it stays in registers through the first
        asm volatile("" : "+v"(t));
        __syncthreads();
        gq_product<F, AL16, true>(G, t, m0, B, ks, s0, s1, Srow, Srowm, false, sh, msum);
    }
}

bool aeth_gq_gemm_rows(const aeth_weight* w, int64_t m) {
    if (!w || (w->dtype != AETH_DTYPE_Q2_K && w->dtype != AETH_DTYPE_Q3_K) || w->order != AETH_ORDER_GGUF) return false;
    // whole blocks per input; i32 sums of 2^14 a product; one row's offsets in an int
    if (w->n % 256 != 0 || w->k < 4 || w->k > 65536 || w->n > (1LL << 28) || m > (1LL << 20)) return false;
    // grids below 2^32 threads (a larger product goes on as blocks that straddle inputs do)
    if (aeth_cdiv(m, 64) * (w->n / 256) > (1LL << 22) || w->n / 256 * aeth_cdiv(w->k, GQ_KS) > (1LL << 23)) return false;
    // From the rows that had the f64 product, always (its precision). Below: k_colk goes through the weight once per 8
    // rows, g times, here it is unpacked and read whole, plus a fixed ≈ 20 µs of launches; both times grow with the weight,
    // in M = 10^6 weights ≈ 0.45·g·M + 8 there and 0.62·M + 20 here (Q2_K: 1.0·M + 24, the mins' product too). So from
    // (g − 1.3)·M = 23 on (Q2_K: (g − 1.95)·M = 26). µs here / there, last row count there and first here:
    // Q3_K 4096 × 2048 (8.4) 24 rows 28.8 / 25.6, 32 29.4 / 27.9; 4096 × 4096 (16.8) 16 36.3 / 26.7, 24 34.6 / 35.2; 6144 ×
    // 4096 (25) 16 36.3 / 36.4, 24 36.0 / 45.6; 2048 × 14336 (29) 16 42.5 / 36.9, 24 41.8 / 47.2; 8192 × 4096 (34) 8 38.7 /
    // 27.7, 16 37.4 / 42.3; 4096 × 14336 (59) 8 54.6 / 35.5, 16 56.0 / 59.1; 28672 × 4096 (117) 8 93 / 65, 16 95 / 122.
    // Q2_K 4096 × 4096 24 39.6 / 36.8, 32 37.7 / 42.8; 6144 × 4096 16 45.9 / 37.0, 24 45.7 / 48.2; 14336 × 2048 16 49.8 / 42.5,
    // 24 50.5 / 52.2; 14336 × 4096 16 75.9 / 67.4, 24 78.2 / 88.7; 28672 × 4096 16 134 / 128, 24 137 / 164.
    const bool q2 = w->dtype == AETH_DTYPE_Q2_K;
    const int64_t g = aeth_cdiv(m, 8), weights = w->n * w->k;
    if (m >= (q2 ? 40 : 32)) return true;
    return q2 ? (20 * g - 39) * weights >= 520000000 : (10 * g - 13) * weights >= 230000000;
}

// bytes of the four unpacked arrays, rounded to 256
static int64_t gq_up(int64_t b) { return aeth_cdiv(b, 256) * 256; }

int aeth_gemm_gq_launch(const aeth_weight* w, const float* d_a, int64_t m, float* d_c, unsigned flags, hipStream_t s,
                        int64_t ldc) {
    if (!aeth_gq_gemm_rows(w, m))
        return aeth_set_error(AETH_EINVAL, "gemm q2_k/q3_k: shape not taken (m=%lld)", (long long)m);
    const bool q2 = w->dtype == AETH_DTYPE_Q2_K;
    const int64_t kp = aeth_cdiv(w->k, GQ_KS) * GQ_KS, nB = w->n / 256, gm = aeth_cdiv(m, 64), T = gm * nB;
    // K split over workgroups while they all fit the chip at once, at least 4 steps each
    const int64_t ksplit = std::max<int64_t>(1, std::min<int64_t>(aeth_num_cus() / T, kp / (4 * GQ_KS)));
    const int64_t uw = nB * (kp / GQ_KS);
    const int64_t vb = gq_up(nB * kp * 256), db = gq_up(nB * kp * 4), mb = gq_up(nB * kp * 32);
    const int64_t pb = ksplit * m * w->n * 8;  // (with K whole, for a first of two products)
    void* ws = nullptr;
    if (!aeth_stream_scratch_try(s, AETH_SCRATCH_DEQ, (size_t)(vb + db + (q2 ? mb + db : 0) + pb), &ws)) return AETH_NO_SCRATCH;
    uint8_t* p = (uint8_t*)ws;
    GqArgs G{};
    G.raw = w->p0; G.A = d_a; G.m = (int)m; G.n = (int)w->n; G.k = (int)w->k; G.kp = (int)kp; G.nB = (int)nB;
    G.v = (int8_t*)p; p += vb;
    G.d = (float*)p; p += db;
    if (q2) {
        G.mins = (int8_t*)p; p += mb;
        G.dmin = (float*)p; p += db;
    }
    G.gm = (int)gm; G.ksplit = (int)ksplit; G.part = (double*)p;
    G.C = d_c; G.ldc = ldc > 0 ? ldc : w->n; G.accumulate = (flags & AETH_MM_ACCUMULATE) ? 1 : 0;
    const dim3 pg((unsigned)uw), gg((unsigned)(T * ksplit));
    const bool al = ((uintptr_t)d_a & 15) == 0 && (w->k & 3) == 0;
    if (q2) hipLaunchKernelGGL(k_gq_prep<AETH_DTYPE_Q2_K>, pg, dim3(256), 0, s, G);
    else hipLaunchKernelGGL(k_gq_prep<AETH_DTYPE_Q3_K>, pg, dim3(256), 0, s, G);
    AETH_LAUNCH_CHECK();
    if (q2 && al) hipLaunchKernelGGL((k_gq_gemm<AETH_DTYPE_Q2_K, true>), gg, dim3(512), 0, s, G);
    else if (q2) hipLaunchKernelGGL((k_gq_gemm<AETH_DTYPE_Q2_K, false>), gg, dim3(512), 0, s, G);
    else if (al) hipLaunchKernelGGL((k_gq_gemm<AETH_DTYPE_Q3_K, true>), gg, dim3(512), 0, s, G);
    else hipLaunchKernelGGL((k_gq_gemm<AETH_DTYPE_Q3_K, false>), gg, dim3(512), 0, s, G);
    AETH_LAUNCH_CHECK();
    if (ksplit > 1) return aeth_narrow_launch(G.part, m, w->n, (int)ksplit, d_c, G.ldc, G.accumulate, s);
    return AETH_OK;
}
