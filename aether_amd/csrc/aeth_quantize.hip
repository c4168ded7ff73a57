// f32 → GGUF blocks on the device: the load-time re-quantizers and the Q8_0
// activation quantizer, byte-exact with the reference.
//
//  * requantize_{q8_0,q4_k,q5_k,q6_k} (src/quant/matmul/dispatch.rs:149-184,
//    186-300, 302-429, 431-537): f32 rows → blocks, used by load_quant to transpose
//    quantized weights (model_loader.rs:330-386).
//  * quantize_q8_0_block / quantize_activations_q8_0[_batched]
//    (src/quant/matmul/neon.rs:45-155): the Q8_0 activation scheme.
//  * load_quant's transpose (model_loader.rs:372-385): dequantize the GGUF
//    [k][n] tensor, transpose to [n][k], re-quantize row by row.
//
// Every step is a single f32 operation with IEEE rounding (contraction off,
// correctly rounded division; minima and maxima do not depend on order), Rust's
// f32::round is C roundf (half away from zero), f32::max / f32::min ignore a NaN
// operand like fmaxf / fminf, and `as u8 / as i8` after the clamps is exact. The f16
// scale bytes follow half::f16::from_f32: round-to-nearest-even, NaN keeps its sign and top payload bits with the
// quiet bit set.
#include <algorithm>
#include <type_traits>

#include "aeth_common.hpp"
#include "aeth_internal.hpp"

#pragma clang fp contract(off)

__device__ __forceinline__ uint32_t f16_bits(float f) { return aeth_f32_to_f16_bits(f); }

// ── re-quantizers ─────────────────────────────────────────────────────────
// Four threads share a super-block of 256 elements (a Q8_0 one: eight blocks of
// 32): `part` p holds 64 of them in registers, whole sub-blocks each, so the
// minima, maxima and quants of a sub-block never leave a thread and only the
// super-block's two maxima and its packed scales go through LDS. A thread per
// 256-block, as these kernels once were, kept 1 of 16 lanes' cache line and read
// every float twice from memory: a 14336 × 4096 Q4_K load took 1954 µs there.
//
// What bounds it now is the VALU: ≈ 20 instructions per element, five of them
// the division. RN(a/d) comes from r = RN(1/d), q0 = a·r and two residual steps
// (the first leaves q within an ulp of a/d; from there one more step with a
// correctly rounded reciprocal gives the correctly rounded quotient, Markstein
// 1990), taken where no step can overflow or lose bits to underflow:
// 2^-60 <= d <= 2^60 and |a| <= 2^60. Elsewhere, and for infinities, the IEEE
// division itself. A NaN goes through either form and ends as the least quant.
template <int F> __device__ __forceinline__ constexpr int rq_index(int p, int c) {
    // Q6_K: 16 elements of each of the four sub-blocks whose bits share ql / qh bytes
    return F == AETH_DTYPE_Q6_K ? 128 * (p >> 1) + 32 * (c >> 4) + 16 * (p & 1) + (c & 15) : 64 * p + c;
}
template <int F> struct Rq;  // BB bytes a super-block, OSD its LDS stride in dwords (odd: no bank conflicts)
template <> struct Rq<AETH_DTYPE_Q8_0> { static constexpr int BB = 8 * Q8_BLOCK_BYTES, OSD = 69; };
template <> struct Rq<AETH_DTYPE_Q4_K> { static constexpr int BB = Q4K_BLOCK_BYTES, OSD = 37; };
template <> struct Rq<AETH_DTYPE_Q5_K> { static constexpr int BB = Q5K_BLOCK_BYTES, OSD = 45; };
template <> struct Rq<AETH_DTYPE_Q6_K> { static constexpr int BB = Q6K_BLOCK_BYTES, OSD = 53; };

template <int SLOTS> struct RqShared {
    float2 mx[4][SLOTS];    // per part: max d_s, max m_s of its sub-blocks
    uint32_t sm[4][SLOTS];  // per part: sc, sc, m, m of its two sub-blocks (Q4_K / Q5_K)
};

struct RqDiv {
    float d, r;
    bool fast;
    // amax: at least the largest |a| divided by d; dead: the caller discards every quotient
    __device__ __forceinline__ RqDiv(float d_, float amax, bool dead = false) : d(d_), r(1.0f / d_) {
        const float ad = fabsf(d_);
        fast = dead || (ad >= 0x1p-60f && ad <= 0x1p60f && amax <= 0x1p60f);
    }
    template <bool FAST> __device__ __forceinline__ float div(float a) const {
        if (!FAST) return a / d;
        float q = a * r;
        q = fmaf(fmaf(-q, d, a), r, q);
        return fmaf(fmaf(-q, d, a), r, q);
    }
};
// f(true_type) where every lane of the wave may take the quick form, else f(false_type): one
// uniform branch per sub-block instead of both quotients per element
template <class Fn> __device__ __forceinline__ void rq_either(const RqDiv& dv, Fn&& f) {
    if (__all(dv.fast)) f(std::true_type{});
    else f(std::false_type{});
}
// clamp(round(v), LO, HI), round half away from zero: 0.5 − 2^-25 is the largest float that
// carries exactly the values from n + 0.5 on to n + 1 (0.49999997 + 0.49999997 < 1, and the
// sum of a tie n + 0.5 rounds up); a NaN ends as max(LO, ·)
template <int LO, int HI> __device__ __forceinline__ int rq_round(float v) {
    const float t = LO < 0 ? v + copysignf(0x1.fffffep-2f, v) : v + 0x1.fffffep-2f;
    return (int)fminf(fmaxf(t, (float)LO), (float)HI);
}

// One part's 64 elements → its bytes of the super-block in `ob` (LDS). `actual` elements of
// the super-block exist (RAGGED; else all 256). Every thread of the workgroup calls it
// (barriers inside); the caller's next barrier publishes ob.
//  Q8_0 (dispatch.rs:149-184): d = max|x|/127 (1 if the block is 0), q = clamp(round(x/d), −128, 127).
//  Q4_K / Q5_K (:186-300, :302-429): per 32-element sub-block m_s = |min(min, 0)|, d_s = (max +
//   m_s)/15 (31); d = max d_s / 63, dmin = max m_s / 63 (1 when 0); sc, m = clamp(round(d_s/d)),
//   clamp(round(m_s/dmin)) in [0, 63], packed as get_scale_min_k4 reads them; q =
//   clamp(round((x + dmin·m)/(d·sc)), 0, 15 (31)). Q5_K: the low nibbles fill qs (byte 48 on), the
//   fifth bit of element e bit e % 8 of qh[e / 8] (bytes 16..47).
//  Q6_K (:431-537): per 16-element sub-block s_max = max|x|; d = max s_max / (32·127) (1 when 0);
//   sc = clamp(round(s_max/(32·d)), 0, 127); q = clamp(round(x/(d·sc)), −32, 31) + 32 (0 + 32 where
//   sc = 0), split into ql nibbles and qh 2-bit fields as dequant_q6_k reads them.
template <int F, bool RAGGED, int SLOTS>
__device__ __forceinline__ void rq_part(const float (&v)[64], int p, int slot, int actual, RqShared<SLOTS>& sh,
                                        uint32_t* ob) {
    if constexpr (F == AETH_DTYPE_Q8_0) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int s0 = 64 * p + 32 * u;
            if (RAGGED && s0 >= actual) continue;
            float mx = 0.0f;
#pragma unroll
            for (int i = 0; i < 32; i++)
                if (!RAGGED || s0 + i < actual) mx = fmaxf(mx, fabsf(v[32 * u + i]));
            const RqDiv dv(mx == 0.0f ? 1.0f : mx / 127.0f, mx);
            uint16_t* o = (uint16_t*)ob + 17 * (2 * p + u);
            o[0] = (uint16_t)f16_bits(dv.d);
            rq_either(dv, [&](auto fast) {
#pragma unroll
                for (int i = 0; i < 32; i += 2) {
                    uint32_t w = 0;
#pragma unroll
                    for (int b = 0; b < 2; b++) {
                        const int q = rq_round<-128, 127>(dv.div<decltype(fast)::value>(v[32 * u + i + b]));
                        if (!RAGGED || s0 + i + b < actual) w |= (uint32_t)(q & 0xFF) << (8 * b);
                    }
                    o[1 + i / 2] = (uint16_t)w;
                }
            });
        }
    } else if constexpr (F == AETH_DTYPE_Q6_K) {
        const int h = p >> 1, is = p & 1;
        float sub[4], mp = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int s0 = rq_index<F>(p, 16 * t);
            float mx = 0.0f;
            if (!RAGGED || s0 < actual) {
                mx = fabsf(v[16 * t]);
#pragma unroll
                for (int i = 1; i < 16; i++)
                    if (!RAGGED || s0 + i < actual) mx = fmaxf(mx, fabsf(v[16 * t + i]));
            }
            sub[t] = mx;
            mp = fmaxf(mp, mx);
        }
        sh.mx[p][slot].x = mp;
        __syncthreads();
        float mv = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) mv = fmaxf(mv, sh.mx[q][slot].x);
        const float d = mv == 0.0f ? 1.0f : mv / (32.0f * 127.0f);
        uint8_t* o8 = (uint8_t*)ob;
        if (p == 0) ((uint16_t*)ob)[104] = (uint16_t)f16_bits(d);
        uint32_t lo0[4] = {}, lo1[4] = {}, hi[4] = {};  // ql[l], ql[l + 32], qh[l] of l = 16·is + (0..15)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint32_t sc = (uint32_t)rq_round<0, 127>(sub[t] / (32.0f * d));
            o8[192 + 8 * h + is + 2 * t] = (uint8_t)sc;
            const float s = (float)sc;
            const RqDiv dv(d * s, mv, !(s > 0.0f));
            rq_either(dv, [&](auto fast) {
#pragma unroll
                for (int l = 0; l < 16; l++) {
                    int q = rq_round<-32, 31>(dv.div<decltype(fast)::value>(v[16 * t + l]));
                    if (!(s > 0.0f) || (RAGGED && rq_index<F>(p, 16 * t + l) >= actual)) q = 0;
                    const uint32_t u = (uint32_t)(q + 32), at = 8 * (l & 3);
                    (t & 1 ? lo1 : lo0)[l >> 2] |= (u & 15) << (at + 4 * (t >> 1));
                    hi[l >> 2] |= (u >> 4) << (at + 2 * t);
                }
            });
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            ob[16 * h + 4 * is + i] = lo0[i];
            ob[16 * h + 8 + 4 * is + i] = lo1[i];
            ob[32 + 8 * h + 4 * is + i] = hi[i];
        }
    } else {
        constexpr bool Q5 = F == AETH_DTYPE_Q5_K;
        constexpr int LVI = Q5 ? 31 : 15;
        float msub[2], dsub[2], big[2];
        float2 mp = make_float2(0.0f, 0.0f);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int s0 = 64 * p + 32 * u;
            float mn = 0.0f, mx = 0.0f;
            if (!RAGGED || s0 < actual) {
                mn = mx = v[32 * u];
#pragma unroll
                for (int i = 1; i < 32; i++)
                    if (!RAGGED || s0 + i < actual) {
                        mn = fminf(mn, v[32 * u + i]);
                        mx = fmaxf(mx, v[32 * u + i]);
                    }
            }
            msub[u] = fabsf(fminf(mn, 0.0f));
            dsub[u] = (mx + msub[u]) / (float)LVI;
            big[u] = fmaxf(fabsf(mn), fabsf(mx));
            mp.x = fmaxf(mp.x, dsub[u]);
            mp.y = fmaxf(mp.y, msub[u]);
        }
        sh.mx[p][slot] = mp;
        __syncthreads();
        float maxd = 0.0f, maxm = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            maxd = fmaxf(maxd, sh.mx[q][slot].x);
            maxm = fmaxf(maxm, sh.mx[q][slot].y);
        }
        const float d = maxd == 0.0f ? 1.0f : maxd / 63.0f;
        const float dmin = maxm == 0.0f ? 1.0f : maxm / 63.0f;
        uint32_t sc[2], mm[2], qs[8] = {};
#pragma unroll
        for (int u = 0; u < 2; u++) {
            sc[u] = (uint32_t)rq_round<0, 63>(dsub[u] / d);
            mm[u] = (uint32_t)rq_round<0, 63>(msub[u] / dmin);
        }
        sh.sm[p][slot] = sc[0] | (sc[1] << 8) | (mm[0] << 16) | (mm[1] << 24);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const float d1 = d * (float)sc[u], m1 = dmin * (float)mm[u];
            const RqDiv dv(d1, fmaxf(big[u], m1) * 2.0f, !(d1 != 0.0f));
            uint32_t fifth = 0;
            rq_either(dv, [&](auto fast) {
#pragma unroll
                for (int l = 0; l < 32; l++) {
                    uint32_t q = (uint32_t)rq_round<0, LVI>(dv.div<decltype(fast)::value>(v[32 * u + l] + m1));
                    if (!(d1 != 0.0f) || (RAGGED && 64 * p + 32 * u + l >= actual)) q = 0;
                    qs[l >> 2] |= (q & 15) << (8 * (l & 3) + 4 * u);
                    if (Q5) fifth |= (q >> 4) << l;
                }
            });
            if (Q5) ob[4 + 2 * p + u] = fifth;
        }
#pragma unroll
        for (int i = 0; i < 8; i++) ob[(Q5 ? 12 : 4) + 8 * p + i] = qs[i];
        __syncthreads();
        if (p == 0) {  // the 16-byte header
            uint32_t s[8], m[8], hd[3] = {};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t w = sh.sm[q][slot];
                s[2 * q] = w & 0xFF; s[2 * q + 1] = (w >> 8) & 0xFF;
                m[2 * q] = (w >> 16) & 0xFF; m[2 * q + 1] = w >> 24;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                hd[0] |= (s[q] | ((s[q + 4] >> 4) << 6)) << (8 * q);
                hd[1] |= (m[q] | ((m[q + 4] >> 4) << 6)) << (8 * q);
                hd[2] |= ((s[q + 4] & 15) | ((m[q + 4] & 15) << 4)) << (8 * q);
            }
            ob[0] = f16_bits(d) | (f16_bits(dmin) << 16);
            ob[1] = hd[0]; ob[2] = hd[1]; ob[3] = hd[2];
        }
    }
}

// f32 rows → blocks: a workgroup takes SLOTS consecutive super-blocks, staged through LDS so that
// a wave's loads are contiguous and part p of 64 super-blocks is one conflict-free column read.
// A row's last super-block may be partial (RAGGED): its missing elements read as 0. With 16 slots
// the threads past 4 · 16 form the same parts again (the same values to the same places).
template <int F, bool RAGGED, int SLOTS>
__global__ void __launch_bounds__(256) k_requant(const float* __restrict__ src, int64_t rows, int64_t cols, int64_t sbr,
                                                 int64_t row_bytes, uint8_t* __restrict__ out) {
    constexpr int XS = 257, OSD = Rq<F>::OSD;
    __shared__ __attribute__((aligned(16))) uint32_t buf[SLOTS * XS];
    __shared__ RqShared<SLOTS> sh;
    const int tid = threadIdx.x, slot = tid % SLOTS, p = tid / SLOTS & 3;
    const int64_t b0 = (int64_t)blockIdx.x * SLOTS, total = rows * sbr;
    float* x = (float*)buf;
#pragma unroll 8
    for (int s = 0; s < SLOTS; s++) {
        const int64_t b = min(b0 + s, total - 1), r = b / sbr, c = (b - r * sbr) * 256 + tid;
        x[s * XS + tid] = !RAGGED || c < cols ? src[r * cols + c] : 0.0f;
    }
    __syncthreads();
    float v[64];
#pragma unroll
    for (int c = 0; c < 64; c++) v[c] = x[slot * XS + rq_index<F>(p, c)];
    __syncthreads();  // the tile is in registers: its LDS takes the blocks
    const int64_t b = min(b0 + slot, total - 1);
    const int actual = RAGGED ? (int)min((int64_t)256, cols - (b % sbr) * 256) : 256;
    rq_part<F, RAGGED, SLOTS>(v, p, slot, actual, sh, buf + slot * OSD);
    __syncthreads();
    constexpr int HW = Rq<F>::BB / 2;  // blocks hold whole halfwords
    const bool odd = (uintptr_t)out & 1;
    for (int i = tid; i < SLOTS * HW; i += 256) {
        const int s = i / HW, w = i - s * HW;
        const int64_t bb = b0 + s;
        if (bb >= total) break;
        const int64_t r = bb / sbr, at = (bb - r * sbr) * Rq<F>::BB + 2 * w;
        if (F == AETH_DTYPE_Q8_0 && RAGGED && at >= row_bytes) continue;
        const uint16_t hw = ((const uint16_t*)(buf + s * OSD))[w];
        uint8_t* o = out + r * row_bytes + at;
        if (!odd) *(uint16_t*)o = hw;
        else o[0] = (uint8_t)hw, o[1] = (uint8_t)(hw >> 8);
    }
}

// ── load_quant in one pass ────────────────────────────────────────────────
// GGUF blocks of a [k][n] tensor → blocks of its [n][k] transpose, for whole super-blocks both
// ways (n % 256 == 0, k % 256 == 0). A workgroup takes 256 inputs × 256 outputs: the 256 source
// blocks stay packed in LDS (36 .. 70 KiB), each thread dequantizes its 64 elements of one output
// straight from there into registers, exactly as aeth_dequant.hip rounds them (the products
// d·sc and dmin·m once per sub-block, in a table), and the re-quantizer above takes them. The f32
// tensor and its transpose (8 bytes an element written and read back twice) never exist. 14336 × 4096:
// Q4_K 2136 → 58 µs, Q5_K 75, Q6_K 88, Q8_0 57 (a copy of the 66 MB of Q4_K bytes: 13 µs; the rest
// is the VALU above). 16 waves a workgroup, one workgroup a CU: 64 values a thread want 128 VGPRs.
// Lanes are neighbouring outputs, so a row's bytes and its scale are one broadcast-friendly LDS
// read each. Other shapes run dequantize, transpose, re-quantize.
template <int F> struct Ld;  // SEG source bytes of a row's 256 outputs, RS their LDS stride, SUB sub-blocks
template <> struct Ld<AETH_DTYPE_Q8_0> { static constexpr int SEG = 272, RS = 272, SUB = 8; };
template <> struct Ld<AETH_DTYPE_Q4_K> { static constexpr int SEG = 144, RS = 144, SUB = 8; };
template <> struct Ld<AETH_DTYPE_Q5_K> { static constexpr int SEG = 176, RS = 176, SUB = 8; };
template <> struct Ld<AETH_DTYPE_Q6_K> { static constexpr int SEG = 210, RS = 212, SUB = 16; };

__device__ __forceinline__ void ld_scale_min(int j, const uint8_t* s, float& sc, float& m) {  // get_scale_min_k4
    const uint32_t a = s[j & 3], b = s[4 + (j & 3)], c = s[8 + (j & 3)];
    sc = (float)(j < 4 ? (a & 63) : ((c & 15) | ((a >> 6) << 4)));
    m = (float)(j < 4 ? (b & 63) : ((c >> 4) | ((b >> 6) << 4)));
}

template <int F>
__global__ void __launch_bounds__(1024, 4) k_load_tile(const uint8_t* __restrict__ src, int64_t k, int64_t n,
                                                   uint8_t* __restrict__ dst) {
    constexpr int SLOTS = 256, OSD = Rq<F>::OSD, BB = Rq<F>::BB, SEG = Ld<F>::SEG, RS = Ld<F>::RS, SUB = Ld<F>::SUB;
    constexpr bool MIN = F == AETH_DTYPE_Q4_K || F == AETH_DTYPE_Q5_K;
    constexpr int OUT = SLOTS * OSD * 4;
    __shared__ __attribute__((aligned(16))) uint8_t raw[256 * RS < OUT ? OUT : 256 * RS];  // then the new blocks
    __shared__ float tab[256 * SUB * (MIN ? 2 : 1)];
    uint32_t* obuf = (uint32_t*)raw;
    __shared__ RqShared<SLOTS> sh;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int64_t kt = k / 256, b = blockIdx.x % kt, jt = blockIdx.x / kt, rowb = n / 256 * SEG;
    const uint8_t* base = src + 256 * b * rowb + jt * SEG;
    if constexpr (F == AETH_DTYPE_Q6_K) {  // blocks are 2-byte aligned only
#pragma unroll 8
        for (int i = tid; i < 256 * (SEG / 2); i += 1024) {
            const int r = i / (SEG / 2), c = i - r * (SEG / 2);
            *(uint16_t*)(raw + r * RS + 2 * c) = *(const uint16_t*)(base + r * rowb + 2 * c);
        }
    } else {
#pragma unroll
        for (int it = 0; it < (256 * (SEG / 16) + 1024 - 1) / 1024; it++) {
            const int i = min(tid + 1024 * it, 256 * (SEG / 16) - 1);  // surplus lanes repeat the last piece
            const int r = i / (SEG / 16), c = i - r * (SEG / 16);
            *(uint4*)(raw + r * RS + 16 * c) = *(const uint4*)(base + r * rowb + 16 * c);
        }
    }
    __syncthreads();
#pragma unroll 4
    for (int i = tid; i < 256 * SUB; i += 1024) {
        const int r = i / SUB, s = i % SUB;
        const uint8_t* q = raw + r * RS;
        if constexpr (MIN) {
            float sc, m;
            ld_scale_min(s, q + 4, sc, m);
            const uint32_t dd = *(const uint32_t*)q;
            tab[2 * i] = aeth_decode_d(dd & 0xFFFFu) * sc;
            tab[2 * i + 1] = aeth_decode_d(dd >> 16) * m;
        } else if constexpr (F == AETH_DTYPE_Q6_K) {
            tab[i] = aeth_decode_d(*(const uint16_t*)(q + 208)) * (float)(int8_t)q[192 + s];
        } else {
            tab[i] = aeth_f16_to_f32(*(const uint16_t*)(q + 34 * s));
        }
    }
    __syncthreads();
    const int p = w & 3, slot = 64 * (w >> 2) + lane;
    const int e = slot;  // this thread's output within the source blocks
    float v[64];
#pragma unroll
    for (int c = 0; c < 64; c++) {
        const int r = rq_index<F>(p, c);
        const uint8_t* q = raw + r * RS;
        if constexpr (F == AETH_DTYPE_Q8_0) {
            v[c] = (float)(int8_t)q[2 * (e >> 5) + 2 + e] * tab[r * SUB + (e >> 5)];
        } else if constexpr (F == AETH_DTYPE_Q6_K) {
            const int t = (e >> 5) & 3;
            const uint32_t lo = q[64 * (e >> 7) + (e & 31) + 32 * (t & 1)], hi = q[128 + 32 * (e >> 7) + (e & 31)];
            const int qi = (int)(((lo >> (4 * (t >> 1))) & 15) | (((hi >> (2 * t)) & 3) << 4)) - 32;
            v[c] = tab[r * SUB + (e >> 4)] * (float)qi;
        } else {
            constexpr int QS = F == AETH_DTYPE_Q5_K ? 48 : 16;
            uint32_t qi = (q[QS + 32 * (e >> 6) + (e & 31)] >> ((e >> 3) & 4)) & 15;
            if (F == AETH_DTYPE_Q5_K) qi |= ((q[16 + (e >> 3)] >> (e & 7)) & 1u) << 4;
            const float2 dm = *(const float2*)(tab + 2 * (r * SUB + (e >> 5)));
            v[c] = dm.x * (float)qi - dm.y;
        }
        if ((c & 7) == 7) __builtin_amdgcn_sched_barrier(0);  // bounds the reads in flight: 128 VGPRs
    }
    __syncthreads();  // raw is read
    rq_part<F, false, SLOTS>(v, p, slot, 256, sh, obuf + slot * OSD);
    __syncthreads();
    const int64_t j0 = 256 * jt;
    if constexpr (F == AETH_DTYPE_Q6_K) {
#pragma unroll 4
        for (int i = tid; i < SLOTS * (BB / 2); i += 1024) {
            const int s = i / (BB / 2), c = i - s * (BB / 2);
            *(uint16_t*)(dst + ((j0 + s) * kt + b) * BB + 2 * c) = ((const uint16_t*)(obuf + s * OSD))[c];
        }
    } else {
#pragma unroll 4
        for (int i = tid; i < SLOTS * (BB / 4); i += 1024) {
            const int s = i / (BB / 4), c = i - s * (BB / 4);
            *(uint32_t*)(dst + ((j0 + s) * kt + b) * BB + 4 * c) = obuf[s * OSD + c];
        }
    }
}

__global__ void k_zero_f32(float* __restrict__ p, int n) {
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0.0f;
}

// quantize_q8_0_block, neon.rs:45-104, over rows of k (quantize_activations_q8_0
// [_batched], neon.rs:106-155: a partial last block is zero-padded).
// d = max|x|/127 with a NaN-propagating max (vmaxq_f32); stored as f16, while
// the quants use the f32 d: q = sat_i8(RNE(x·(1/d))) (vcvtnq_s32_f32 then two
// saturating narrows); d = 0 or NaN → zero quants. A block holding a NaN
// stores the quiet NaN 0x7E00 as its scale (the sign and payload that
// vmaxq_f32 would carry over from the input NaN are not reproduced).
__global__ void __launch_bounds__(256) k_quant_act_q8_0(const float* __restrict__ a, int64_t m, int64_t k,
                                                        int64_t bpr, uint8_t* __restrict__ out) {
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= m * bpr) return;
    const int64_t r = b / bpr, blk = b - r * bpr;
    const float* x = a + r * k + blk * 32;
    const int actual = (int)min((int64_t)32, k - blk * 32);
    float v[32];
    for (int i = 0; i < 32; i++) v[i] = i < actual ? x[i] : 0.0f;
    bool nan = false;
    float mx = 0.0f;
    for (int i = 0; i < 32; i++) {
        nan |= v[i] != v[i];
        mx = fmaxf(mx, fabsf(v[i]));
    }
    const float d = nan ? __uint_as_float(0x7FC00000u) : mx / 127.0f;
    uint8_t* o = out + b * 34;
    const uint32_t db = f16_bits(d);
    o[0] = (uint8_t)db;
    o[1] = (uint8_t)(db >> 8);
    if (d > 0.0f) {
        const float inv = 1.0f / d;
        for (int i = 0; i < 32; i++) {
            const float p = v[i] * inv;
            // RNE to integer with i32 saturation, NaN → 0 (vcvtnq_s32_f32), then clamp to i8
            int32_t q = p != p ? 0 : p >= 2147483648.0f ? INT32_MAX : p < -2147483648.0f ? INT32_MIN : (int32_t)rintf(p);
            q = max(-128, min(127, q));
            o[2 + i] = (uint8_t)(int8_t)q;
        }
    } else {
        for (int i = 0; i < 32; i++) o[2 + i] = 0;
    }
}

// [rows][cols] → [cols][rows] through 32 × 33 LDS tiles.
__global__ void __launch_bounds__(256) k_transpose_f32(const float* __restrict__ src, int64_t rows, int64_t cols,
                                                       float* __restrict__ dst) {
    __shared__ float t[32][33];
    const int64_t c0 = (int64_t)blockIdx.x * 32, r0 = (int64_t)blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 × 8
    for (int j = ty; j < 32; j += 8) {
        const int64_t r = r0 + j, c = c0 + tx;
        if (r < rows && c < cols) t[j][tx] = src[r * cols + c];
    }
    __syncthreads();
    for (int j = ty; j < 32; j += 8) {
        const int64_t c = c0 + j, r = r0 + tx;
        if (r < rows && c < cols) dst[c * rows + r] = t[tx][j];
    }
}

template <int F>
static void requant_go(const float* src, int64_t rows, int64_t cols, uint8_t* dst, hipStream_t s) {
    const int64_t sbr = aeth_cdiv(cols, 256), n = rows * sbr;
    const int64_t row_bytes = F == AETH_DTYPE_Q8_0 ? aeth_cdiv(cols, 32) * Q8_BLOCK_BYTES : sbr * Rq<F>::BB;
    // 16 super-blocks a workgroup (64 left most CUs idle up to 16384 of them, and put two a CU by their LDS after that): Q8_0
    // 16 × 4096 21.6 → 8.1 µs, 1024 × 4096 24.7 → 16.2, 14336 × 4096 291 → 170; Q4_K 19 → 7.9, 21.4 → 16.0, 209 → 156, between
    // (2048 rows) 25.9 → 28.0. The 64 stay for many ragged rows of Q4_K / Q5_K, where each super-block is mostly VALU
    // work for absent elements: Q4_K 4096 × 300 24.9 → 15.0, but 32768 × 50 27.9 → 41.3, 65536 × 300 143 → 170.
    constexpr bool wide = F == AETH_DTYPE_Q4_K || F == AETH_DTYPE_Q5_K;
    const int64_t step = std::max<int64_t>(1, (1LL << 27) / sbr);  // rows a launch: below 2^32 threads
    for (int64_t r = 0; r < rows; r += step) {
        const float* x = src + r * cols;
        uint8_t* o = dst + r * row_bytes;
        const int64_t m = std::min(step, rows - r);
        const dim3 grid((unsigned)aeth_cdiv(m * sbr, 16)), grid64((unsigned)aeth_cdiv(m * sbr, 64));
        if (cols % 256 == 0)
            hipLaunchKernelGGL((k_requant<F, false, 16>), grid, dim3(256), 0, s, x, m, cols, sbr, row_bytes, o);
        else if (!wide || n < 64LL * aeth_num_cus())
            hipLaunchKernelGGL((k_requant<F, true, 16>), grid, dim3(256), 0, s, x, m, cols, sbr, row_bytes, o);
        else if constexpr (wide)
            hipLaunchKernelGGL((k_requant<F, true, 64>), grid64, dim3(256), 0, s, x, m, cols, sbr, row_bytes, o);
    }
}

static int requant_launch(int dtype, const float* src, int64_t rows, int64_t cols, uint8_t* dst, hipStream_t s) {
    if (dtype == AETH_DTYPE_Q8_0 && cols % 32 == 0) {  // whole blocks a row: one run of blocks, no row's end to pad
        cols *= rows;
        rows = 1;
    }
    if (rows == 0 || cols == 0) return AETH_OK;
    if (dtype == AETH_DTYPE_Q8_0) requant_go<AETH_DTYPE_Q8_0>(src, rows, cols, dst, s);
    else if (dtype == AETH_DTYPE_Q4_K) requant_go<AETH_DTYPE_Q4_K>(src, rows, cols, dst, s);
    else if (dtype == AETH_DTYPE_Q5_K) requant_go<AETH_DTYPE_Q5_K>(src, rows, cols, dst, s);
    else requant_go<AETH_DTYPE_Q6_K>(src, rows, cols, dst, s);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}

static bool requant_dtype(int dtype) {
    return dtype == AETH_DTYPE_Q8_0 || dtype == AETH_DTYPE_Q4_K || dtype == AETH_DTYPE_Q5_K || dtype == AETH_DTYPE_Q6_K;
}

extern "C" AETH_API int aeth_requantize(int dtype, const float* d_src, int64_t rows, int64_t cols, void* d_dst,
                                        void* stream) {
    if (!requant_dtype(dtype)) return aeth_set_error(AETH_EUNSUPPORTED, "aeth_requantize: unsupported dtype %d", dtype);
    if (rows < 0 || cols <= 0 || (rows > 0 && (!d_src || !d_dst)))
        return aeth_set_error(AETH_EINVAL, "aeth_requantize: bad argument");
    return requant_launch(dtype, d_src, rows, cols, (uint8_t*)d_dst, (hipStream_t)stream);
}

extern "C" AETH_API int aeth_quantize_activations_q8_0(const float* d_a, int64_t m, int64_t k, void* d_dst,
                                                       void* stream) {
    if (m < 0 || k <= 0 || (m > 0 && (!d_a || !d_dst)))
        return aeth_set_error(AETH_EINVAL, "aeth_quantize_activations_q8_0: bad argument");
    const int64_t bpr = aeth_cdiv(k, 32), nblk = m * bpr;
    if (nblk == 0) return AETH_OK;
    hipLaunchKernelGGL(k_quant_act_q8_0, dim3((unsigned)aeth_cdiv(nblk, 256)), dim3(256), 0, (hipStream_t)stream, d_a,
                       m, k, bpr, (uint8_t*)d_dst);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}

extern "C" AETH_API int aeth_transpose_f32(const float* d_src, int64_t rows, int64_t cols, float* d_dst,
                                           void* stream) {
    if (rows < 0 || cols < 0 || (rows * cols > 0 && (!d_src || !d_dst)) || d_src == d_dst)
        return aeth_set_error(AETH_EINVAL, "aeth_transpose_f32: bad argument");
    if (rows == 0 || cols == 0) return AETH_OK;
    if (aeth_cdiv(rows, 32) > 65535) return aeth_set_error(AETH_EINVAL, "aeth_transpose_f32: rows=%lld too large", (long long)rows);
    hipLaunchKernelGGL(k_transpose_f32, dim3((unsigned)aeth_cdiv(cols, 32), (unsigned)aeth_cdiv(rows, 32)), dim3(256),
                       0, (hipStream_t)stream, d_src, rows, cols, d_dst);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}

extern "C" AETH_API int64_t aeth_load_quant_ws_bytes(int64_t k, int64_t n) {
    if (k <= 0 || n <= 0) return 0;
    int64_t kn = 0;
    if (!aeth_mul_ok(k, n, &kn) || kn > INT64_MAX / 8) return -1;  // too large for any device
    return 2 * kn * (int64_t)sizeof(float);
}

// load_quant for a 2-D quantized tensor, model_loader.rs:330-386: GGUF shape
// [k, n] (k·n elements, dequantized as one flat run of blocks and read as a
// row-major [k][n] matrix) → [n][k] f32 → requantized rows of k.
extern "C" AETH_API int aeth_load_quant(int dtype, const void* d_src, int64_t k, int64_t n, void* d_dst,
                                        void* d_ws, void* stream) {
    if (!requant_dtype(dtype)) return aeth_set_error(AETH_EUNSUPPORTED, "aeth_load_quant: unsupported dtype %d", dtype);
    if (k <= 0 || n <= 0 || !d_src || !d_dst || !d_ws) return aeth_set_error(AETH_EINVAL, "aeth_load_quant: bad argument");
    hipStream_t s = (hipStream_t)stream;
    // One pass where both ways are whole super-blocks and its accesses are aligned (a file's tensors
    // are; only Q6_K's 210-byte blocks do with 2 bytes): 14336 × 4096 Q4_K 56 µs, 14336 × 4100 425 in the
    // three passes below. A destination that overlaps the source (bytes loaded in place) needs the
    // copies those make: here a workgroup would overwrite blocks that another has yet to read. k past
    // 65535 · 32 stays with the transpose, which refuses it; the grid holds under 2^32 threads.
    const int64_t bytes = n * (k / (dtype == AETH_DTYPE_Q8_0 ? 32 : 256)) *
                          (dtype == AETH_DTYPE_Q8_0 ? Q8_BLOCK_BYTES : dtype == AETH_DTYPE_Q4_K ? Q4K_BLOCK_BYTES :
                           dtype == AETH_DTYPE_Q5_K ? Q5K_BLOCK_BYTES : Q6K_BLOCK_BYTES);
    const uintptr_t sa = (uintptr_t)d_src, da = (uintptr_t)d_dst;
    const bool apart = sa + (uintptr_t)bytes <= da || da + (uintptr_t)bytes <= sa;
    if (n % 256 == 0 && k % 256 == 0 && k <= 65535 * 32 && (n / 256) * (k / 256) <= 0x3FFFFF && apart &&
        ((sa | da) & (dtype == AETH_DTYPE_Q6_K ? 1 : 15)) == 0) {
        const dim3 grid((unsigned)((n / 256) * (k / 256)));
        const uint8_t* src = (const uint8_t*)d_src;
        uint8_t* dst = (uint8_t*)d_dst;
        if (dtype == AETH_DTYPE_Q8_0) hipLaunchKernelGGL(k_load_tile<AETH_DTYPE_Q8_0>, grid, dim3(1024), 0, s, src, k, n, dst);
        else if (dtype == AETH_DTYPE_Q4_K) hipLaunchKernelGGL(k_load_tile<AETH_DTYPE_Q4_K>, grid, dim3(1024), 0, s, src, k, n, dst);
        else if (dtype == AETH_DTYPE_Q5_K) hipLaunchKernelGGL(k_load_tile<AETH_DTYPE_Q5_K>, grid, dim3(1024), 0, s, src, k, n, dst);
        else hipLaunchKernelGGL(k_load_tile<AETH_DTYPE_Q6_K>, grid, dim3(1024), 0, s, src, k, n, dst);
        AETH_LAUNCH_CHECK();
        return AETH_OK;
    }
    float* flat = (float*)d_ws;
    float* tr = flat + k * n;
    // the K-quants dequantize whole blocks only; the reference's output starts zeroed
    const int tail = dtype == AETH_DTYPE_Q8_0 ? 0 : (int)(k * n % 256);
    if (tail) {
        hipLaunchKernelGGL(k_zero_f32, dim3(1), dim3(256), 0, s, flat + (k * n - tail), tail);
        AETH_LAUNCH_CHECK();
    }
    int rc = aeth_dequant(dtype, d_src, k * n, flat, stream);
    if (rc != AETH_OK) return rc;
    rc = aeth_transpose_f32(flat, k, n, tr, stream);
    if (rc != AETH_OK) return rc;
    return requant_launch(dtype, tr, n, k, (uint8_t*)d_dst, s);
}
