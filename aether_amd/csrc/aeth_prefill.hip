// Batched prefill kernels (LlamaRunner::forward_batch, src/inference/runner.rs:833-993):
// the n prompt tokens go through each layer together, token i at position i,
// its K/V written to cache slot i. The projections run on the quantized GEMM
// (aeth_gemm.hip, Q4_K) or the row-batched GEMV (other formats); these kernels
// are the glue around them:
//  * k_embed_rows: token embeddings → rows of x;
//  * k_prefill_rope_kv: RoPE of q and k at each token's position
//    (apply_rope_inplace, runner.rs:1886-1909) and the cache writes (:890-906);
//  * k_attn_prefill_mf: causal attention (attention_batch, runner.rs:1809-1883)
//    on the f32 matrix cores, flash-style (online softmax over 16-key blocks);
//    k_attn_prefill, the f32 VALU form (64-query blocks, 4×4 score and 4×8
//    output register tiles per thread), serves group sizes the MFMA form does
//    not take;
//  * k_silu_pairs: h = g·σ(g)·u on the interleaved gate/up GEMM output
//    (runner.rs:1617-1625 form).
#include <limits.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>

#include "aeth_common.hpp"
#include "aeth_gemm_common.hpp"
#include "aeth_internal.hpp"
#include "aeth_ops_internal.hpp"

typedef float f32x4 __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(256) k_embed_rows(const float* __restrict__ table, const int* __restrict__ tokens,
                                                    int64_t d, float* __restrict__ x) {
    const int64_t i = blockIdx.x;
    const float* src = table + (int64_t)tokens[i] * d;
    float* dst = x + i * d;
    for (int64_t e = threadIdx.x; e < d; e += 256) dst[e] = src[e];
}

int aeth_embed_rows_launch(const float* table, const int* d_tokens, int64_t n, int64_t d, float* x, hipStream_t s) {
    if (n <= 0) return AETH_OK;
    hipLaunchKernelGGL(k_embed_rows, dim3((unsigned)n), dim3(256), 0, s, table, d_tokens, d, x);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}

// qkv: [n][nh·hd | nkv·hd | nkv·hd]; q and k rotated in place, k and v copied to
// the layer's cache [2][nkv][max_seq][hd] at slot i.
__global__ void __launch_bounds__(256) k_prefill_rope_kv(float* __restrict__ qkv, int64_t stride, int nh, int nkv,
                                                         int hd, const float* __restrict__ sin_t,
                                                         const float* __restrict__ cos_t, int64_t max_seq,
                                                         float* __restrict__ layer_kv) {
    const int64_t i = blockIdx.x;
    const int half = hd / 2;
    const int64_t p = i < max_seq ? i : max_seq - 1;
    float* row = qkv + i * stride;
    const float* sn = sin_t + p * half;
    const float* cs = cos_t + p * half;
    const int64_t hs = max_seq * hd;
    for (int idx = threadIdx.x; idx < (nh + nkv) * half; idx += 256) {
        const int h = idx / half, e = idx - h * half;
        float* v = row + (int64_t)h * hd;  // heads nh.. are the k heads (they follow q in the row)
        const float x0 = v[e], x1 = v[e + half];
        const float r0 = x0 * cs[e] - x1 * sn[e], r1 = x0 * sn[e] + x1 * cs[e];
        v[e] = r0;
        v[e + half] = r1;
        if (h >= nh) {
            float* kd = layer_kv + (int64_t)(h - nh) * hs + i * hd;
            kd[e] = r0;
            kd[e + half] = r1;
        }
    }
    const float* vsrc = row + (int64_t)(nh + nkv) * hd;
    for (int idx = threadIdx.x; idx < nkv * hd; idx += 256) {
        const int h = idx / hd, e = idx - h * hd;
        layer_kv[(int64_t)(nkv + h) * hs + i * hd + e] = vsrc[idx];
    }
}

// The same for hd % 8 == 0 on 16-byte aligned rows: float4 pieces (four rotation
// pairs, or four v elements), 4 per thread per batch with every load issued
// before the first store.
__global__ void __launch_bounds__(256) k_prefill_rope_kv4(float* __restrict__ qkv, int64_t stride, int nh, int nkv,
                                                          int hd, const float* __restrict__ sin_t,
                                                          const float* __restrict__ cos_t, int64_t max_seq,
                                                          float* __restrict__ layer_kv) {
    const int64_t i = blockIdx.x;
    const int half = hd / 2, q4 = half / 4;
    const int64_t p = i < max_seq ? i : max_seq - 1;
    float* row = qkv + i * stride;
    const float* sn = sin_t + p * half;
    const float* cs = cos_t + p * half;
    const int64_t hs = max_seq * hd;
    const int units = (nh + nkv) * q4, vunits = nkv * hd / 4;
    for (int u0 = 0; u0 < units; u0 += 1024) {
        float4 a[4], b[4], c[4], t[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int u = min(u0 + (int)threadIdx.x + 256 * k, units - 1), h = u / q4, e = 4 * (u - h * q4);
            a[k] = *(const float4*)(row + (int64_t)h * hd + e);
            b[k] = *(const float4*)(row + (int64_t)h * hd + e + half);
            c[k] = *(const float4*)(cs + e);
            t[k] = *(const float4*)(sn + e);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int u = u0 + (int)threadIdx.x + 256 * k;
            if (u < units) {
                const int h = u / q4, e = 4 * (u - h * q4);
                const float4 r0 = make_float4(a[k].x * c[k].x - b[k].x * t[k].x, a[k].y * c[k].y - b[k].y * t[k].y,
                                              a[k].z * c[k].z - b[k].z * t[k].z, a[k].w * c[k].w - b[k].w * t[k].w);
                const float4 r1 = make_float4(a[k].x * t[k].x + b[k].x * c[k].x, a[k].y * t[k].y + b[k].y * c[k].y,
                                              a[k].z * t[k].z + b[k].z * c[k].z, a[k].w * t[k].w + b[k].w * c[k].w);
                *(float4*)(row + (int64_t)h * hd + e) = r0;
                *(float4*)(row + (int64_t)h * hd + e + half) = r1;
                if (h >= nh) {
                    float* kd = layer_kv + (int64_t)(h - nh) * hs + i * hd;
                    *(float4*)(kd + e) = r0;
                    *(float4*)(kd + e + half) = r1;
                }
            }
        }
    }
    const float* vsrc = row + (int64_t)(nh + nkv) * hd;
    for (int u = threadIdx.x; u < vunits; u += 256) {
        const int h = (4 * u) / hd, e = 4 * u - h * hd;
        *(float4*)(layer_kv + (int64_t)(nkv + h) * hs + i * hd + e) = *(const float4*)(vsrc + 4 * u);
    }
}

int aeth_prefill_rope_kv_launch(float* qkv, int64_t n, int64_t nh, int64_t nkv, int64_t hd, const float* sin_t,
                                const float* cos_t, int64_t max_seq, float* layer_kv, hipStream_t s) {
    if (n <= 0) return AETH_OK;
    if (n > max_seq) return aeth_set_error(AETH_EINVAL, "prefill: %lld tokens exceed the cache", (long long)n);
    const bool al16 = (((uintptr_t)qkv | (uintptr_t)sin_t | (uintptr_t)cos_t | (uintptr_t)layer_kv) & 15) == 0;
    if (al16 && hd % 8 == 0)
        hipLaunchKernelGGL(k_prefill_rope_kv4, dim3((unsigned)n), dim3(256), 0, s, qkv, (nh + 2 * nkv) * hd, (int)nh,
                           (int)nkv, (int)hd, sin_t, cos_t, max_seq, layer_kv);
    else
        hipLaunchKernelGGL(k_prefill_rope_kv, dim3((unsigned)n), dim3(256), 0, s, qkv, (nh + 2 * nkv) * hd, (int)nh,
                           (int)nkv, (int)hd, sin_t, cos_t, max_seq, layer_kv);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}

#define PA_BQ 64
#define PA_BK 64

// Causal attention of queries [64·blockIdx.x, +64) of head blockIdx.y over keys
// 0..i of the layer cache (slots written by k_prefill_rope_kv); with a sliding
// window w > 0, keys i - w + 1 ..= i (attention_batch, runner.rs:1825-1845).
template <int HD>
__global__ void __launch_bounds__(256) k_attn_prefill(const float* __restrict__ qkv, int64_t qkv_stride,
                                                      const float* __restrict__ layer_kv, int n, int nh, int nkv,
                                                      int64_t max_seq, int window, float* __restrict__ out) {
    constexpr int LD = HD + 4;  // row stride (floats): 16-byte aligned rows
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float* Qs = sm;
    float* Ks = Qs + PA_BQ * LD;
    float* Vs = Ks + PA_BK * LD;
    float* Ps = Vs + PA_BK * LD;  // [BQ][BK + 1]
    float* mrow = Ps + PA_BQ * (PA_BK + 1);
    float* lrow = mrow + PA_BQ;
    float* arow = lrow + PA_BQ;
    const int tid = threadIdx.x;
    const int h = blockIdx.y, kvh = h / (nh / nkv);
    const int q0 = blockIdx.x * PA_BQ;
    const float* K = layer_kv + (int64_t)kvh * max_seq * HD;
    const float* V = layer_kv + (int64_t)(nkv + kvh) * max_seq * HD;
    const float scale = 1.0f / sqrtf((float)HD);

    for (int idx = tid; idx < PA_BQ * HD / 4; idx += 256) {
        const int r = idx / (HD / 4), c = idx - r * (HD / 4);
        const int qi = min(q0 + r, n - 1);
        *(float4*)(Qs + r * LD + 4 * c) = *(const float4*)(qkv + (int64_t)qi * qkv_stride + (int64_t)h * HD + 4 * c);
    }
    if (tid < PA_BQ) {
        mrow[tid] = -INFINITY;
        lrow[tid] = 0.0f;
    }
    const int qq = tid >> 4, kq = tid & 15;  // score tile: queries 4qq.., keys 4kq..
    const int dq = tid & 15;                 // output tile: queries 4qq.., dims 8dq..
    float o[4][8];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int e = 0; e < 8; e++) o[a][e] = 0.0f;
    const int nkb = (min(q0 + PA_BQ, n) - 1) / PA_BK + 1;
    const int kb0 = window > 0 ? max(0, q0 - window + 1) / PA_BK : 0;  // blocks before every query's window: none
    for (int kb = kb0; kb < nkb; kb++) {
        const int k0 = kb * PA_BK;
        __syncthreads();  // the previous block's K/V/P are no longer read
        for (int idx = tid; idx < PA_BK * HD / 4; idx += 256) {
            const int r = idx / (HD / 4), c = idx - r * (HD / 4);
            const int kj = min(k0 + r, n - 1);
            *(float4*)(Ks + r * LD + 4 * c) = *(const float4*)(K + (int64_t)kj * HD + 4 * c);
            *(float4*)(Vs + r * LD + 4 * c) = *(const float4*)(V + (int64_t)kj * HD + 4 * c);
        }
        __syncthreads();
        float sacc[4][4];
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int b = 0; b < 4; b++) sacc[a][b] = 0.0f;
        for (int dd = 0; dd < HD; dd += 4) {
            float4 qv[4], kv[4];
#pragma unroll
            for (int a = 0; a < 4; a++) qv[a] = *(const float4*)(Qs + (4 * qq + a) * LD + dd);
#pragma unroll
            for (int b = 0; b < 4; b++) kv[b] = *(const float4*)(Ks + (4 * kq + b) * LD + dd);
#pragma unroll
            for (int a = 0; a < 4; a++)
#pragma unroll
                for (int b = 0; b < 4; b++)
                    sacc[a][b] += qv[a].x * kv[b].x + qv[a].y * kv[b].y + qv[a].z * kv[b].z + qv[a].w * kv[b].w;
        }
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int qi = q0 + 4 * qq + a, kj = k0 + 4 * kq + b;
                Ps[(4 * qq + a) * (PA_BK + 1) + 4 * kq + b] =
                    (kj <= qi && kj < n && (window <= 0 || kj > qi - window)) ? sacc[a][b] * scale : -INFINITY;
            }
        __syncthreads();
        {  // online softmax: 4 threads per query row, 16 keys each
            const int r = tid >> 2, pp = tid & 3;
            float* pr = Ps + r * (PA_BK + 1) + 16 * pp;
            float mx = -INFINITY;
#pragma unroll
            for (int j = 0; j < 16; j++) mx = fmaxf(mx, pr[j]);
            mx = fmaxf(mx, __shfl_xor(mx, 1, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 2, 64));
            const float m_old = mrow[r];
            const float m_new = fmaxf(m_old, mx);
            float ps = 0.0f;
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const float e = m_new == -INFINITY ? 0.0f : expf(pr[j] - m_new);
                pr[j] = e;
                ps += e;
            }
            ps += __shfl_xor(ps, 1, 64);
            ps += __shfl_xor(ps, 2, 64);
            if (pp == 0) {
                const float alpha = m_new == -INFINITY ? 1.0f : expf(m_old - m_new);
                lrow[r] = lrow[r] * alpha + ps;
                mrow[r] = m_new;
                arow[r] = alpha;
            }
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const float al = arow[4 * qq + a];
#pragma unroll
            for (int e = 0; e < 8; e++) o[a][e] *= al;
        }
        for (int j = 0; j < PA_BK; j++) {
            const float4 v0 = *(const float4*)(Vs + j * LD + 8 * dq);
            const float4 v1 = *(const float4*)(Vs + j * LD + 8 * dq + 4);
#pragma unroll
            for (int a = 0; a < 4; a++) {
                const float p = Ps[(4 * qq + a) * (PA_BK + 1) + j];
                o[a][0] += p * v0.x; o[a][1] += p * v0.y; o[a][2] += p * v0.z; o[a][3] += p * v0.w;
                o[a][4] += p * v1.x; o[a][5] += p * v1.y; o[a][6] += p * v1.z; o[a][7] += p * v1.w;
            }
        }
    }
#pragma unroll
    for (int a = 0; a < 4; a++) {
        const int qi = q0 + 4 * qq + a;
        if (qi < n) {
            const float inv = 1.0f / lrow[4 * qq + a];
            float* dst = out + (int64_t)qi * nh * HD + (int64_t)h * HD + 8 * dq;
            *(float4*)dst = make_float4(o[a][0] * inv, o[a][1] * inv, o[a][2] * inv, o[a][3] * inv);
            *(float4*)(dst + 4) = make_float4(o[a][4] * inv, o[a][5] * inv, o[a][6] * inv, o[a][7] * inv);
        }
    }
}

// Causal attention on the f32 matrix cores, v_mfma_f32_16x16x4_f32 (lane l
// holds A[l%16][l/16] and B[l/16][l%16]; result register r of lane l is
// D[4(l/16) + r][l%16]). Scores are computed transposed, Sᵀ = K·Qᵀ, so that a
// lane's accumulator holds 4 keys of one score column; those registers are
// then directly the B operand of Oᵀ = Vᵀ·Pᵀ (no transposes). The 16 columns
// are QB = 16/G queries × the G query heads of one KV head (column c: query
// c/G, head c%G), so every K/V element loaded serves all G heads.
// K-index maps: in Sᵀ step i, lane group g (= l/16) contracts d = 32g + i;
// in Oᵀ step j it contracts key t0 + 4g + j (its own score register j), and
// Oᵀ row m of d-tile dt is d = 8m + dt, so a lane (c, g) ends with d = 32g +
// 8r + dt of column c.
// Work: workgroup (KV head, query-block pair {p, nqb−1−p}), which balances the
// causal triangle; its 4 waves take the 16-key blocks of a query block round
// robin, each keeping an online softmax, and merge the partials through LDS.
// Per key block the softmax runs in log2 units (v_exp_f32) and rescales the
// partials only when some column's running max grows by more than 2^8: below
// that the probabilities are taken against the stale max (at most 2^8 each;
// the result o / l does not depend on which max is used). K and V are read as
// buffers of the n filled rows, so the loads of rows ≥ n (the last block's
// tail) return zeros; those keys are masked. Two register sets alternate, the
// next block's loads in flight during the current block. With a sliding window
// w > 0 (attention_batch, runner.rs:1825-1845) query i sees keys i - w + 1 ..= i:
// the waves start at the first key block some query of the block sees, and the
// keys before a query's window are masked like those past it.
// Max / sum of a value over the lane pairs (l, l ^ 16) and (l, l ^ 32): v_permlane16_swap and
// v_permlane32_swap with the same register as both operands leave each lane of a pair the
// lower lane's value in the first result and the upper lane's in the second (register moves,
// no LDS round trip); both lanes then compute lower ∘ upper, the same bits.
__device__ __forceinline__ float pa_max16(float a) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(a), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pa_max32(float a) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(a), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pa_sum16(float a) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(a), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float pa_sum32(float a) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(a), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ float4 pa_ld4(__amdgpu_buffer_rsrc_t r, int off) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}

template <int G>
__global__ void __launch_bounds__(256, 2) k_attn_prefill_mf(const float* __restrict__ qkv, int64_t qkv_stride,
                                                         const float* __restrict__ layer_kv, int n, int nh, int nkv,
                                                         int64_t max_seq, int window, float* __restrict__ out) {
    constexpr int QB = 16 / G, HD = 128, PLD = HD + 4;
    constexpr float TH = 8.0f;  // log2 units a running max may grow before the partials are rescaled
    __shared__ __attribute__((aligned(16))) float po[4][16][PLD];  // per wave: column c, d
    __shared__ float pm[4][16], pl[4][16];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int c = lane & 15, grp = lane >> 4;
    const int g = blockIdx.x % nkv, p = blockIdx.x / nkv;
    const int nqb = (n + QB - 1) / QB;
    const int head = g * G + c % G;
    const float* K = layer_kv + (int64_t)g * max_seq * HD;
    const float* V = layer_kv + (int64_t)(nkv + g) * max_seq * HD;
    const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc((void*)K, (short)0, n * HD * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rV = __builtin_amdgcn_make_buffer_rsrc((void*)V, (short)0, n * HD * 4, 0x00020000);
    const float sl2 = 1.4426950408889634f / sqrtf((float)HD);  // scale · log2(e)
    for (int pass = 0; pass < 2; pass++) {
        const int qb = pass == 0 ? p : nqb - 1 - p;
        if (pass == 1 && qb == p) break;  // the middle block of an odd count (uniform)
        const int q0 = qb * QB, query = q0 + c / G;
        float qv[32];
        {
            const float* src = qkv + (int64_t)min(query, n - 1) * qkv_stride + (int64_t)head * HD + 32 * grp;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float4 t = *(const float4*)(src + 4 * i);
                qv[4 * i] = t.x; qv[4 * i + 1] = t.y; qv[4 * i + 2] = t.z; qv[4 * i + 3] = t.w;
            }
        }
        const int kb_end = (min(q0 + QB, n) - 1) / 16;  // last key block, inclusive
        const int kb_beg = window > 0 ? max(0, q0 - window + 1) / 16 : 0;  // first key block any query sees
        // keys t with t > query - window are visible: t ≥ lo_all for every query of the block
        const int lo_all = window > 0 ? q0 + QB - window : INT_MIN;
        // loads of one key block: K rows t0 + c (A of Sᵀ), V rows t0 + 4·grp + j,
        // floats [8c, 8c + 8) (A of Oᵀ)
        auto load = [&](int kb, float4* kk, float4 (*vv)[2]) {
            const int ko = ((16 * kb + c) * HD + 32 * grp) * 4, vo = ((16 * kb + 4 * grp) * HD + 8 * c) * 4;
#pragma unroll
            for (int i = 0; i < 8; i++) kk[i] = pa_ld4(rK, ko + 16 * i);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                vv[j][0] = pa_ld4(rV, vo + j * HD * 4);
                vv[j][1] = pa_ld4(rV, vo + j * HD * 4 + 16);
            }
        };
        float m = -INFINITY, l = 0.0f;
        f32x4 o[8];
#pragma unroll
        for (int dt = 0; dt < 8; dt++) o[dt] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        auto step = [&](int kb, const float4* kr, const float4 (*vr)[2]) {
            const int t0 = 16 * kb;
            // four independent chains of 8 MFMAs (d ≡ i mod 4 of each lane group's 32), summed
            f32x4 s4[4];
#pragma unroll
            for (int u = 0; u < 4; u++) s4[u] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                s4[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[i].x, qv[4 * i], s4[0], 0, 0, 0);
                s4[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[i].y, qv[4 * i + 1], s4[1], 0, 0, 0);
                s4[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[i].z, qv[4 * i + 2], s4[2], 0, 0, 0);
                s4[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[i].w, qv[4 * i + 3], s4[3], 0, 0, 0);
            }
            f32x4 s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
            if (t0 + 15 <= q0 && t0 + 15 < n && t0 >= lo_all) {  // no key of the block is masked (uniform)
#pragma unroll
                for (int r = 0; r < 4; r++) s[r] *= sl2;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int t = t0 + 4 * grp + r;
                    s[r] = (t <= query && t < n && (window <= 0 || t > query - window)) ? s[r] * sl2 : -INFINITY;
                }
            }
            float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
            mx = pa_max32(pa_max16(mx));
            if (__any(mx > m + TH)) {  // uniform
                const float m_new = fmaxf(m, mx);
                const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
                l *= alpha;
#pragma unroll
                for (int dt = 0; dt < 8; dt++) o[dt] *= alpha;
                m = m_new;
            }
            float ps = 0.0f;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                s[r] = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(s[r] - m);
                ps += s[r];
            }
            l += pa_sum32(pa_sum16(ps));
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float vj[8] = {vr[j][0].x, vr[j][0].y, vr[j][0].z, vr[j][0].w,
                                     vr[j][1].x, vr[j][1].y, vr[j][1].z, vr[j][1].w};
#pragma unroll
                for (int dt = 0; dt < 8; dt++) o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vj[dt], s[j], o[dt], 0, 0, 0);
            }
        };
        float4 ka[8], va[4][2], kn[8], vn[4][2];
        if (kb_beg + w <= kb_end) load(kb_beg + w, ka, va);
        for (int kb = kb_beg + w; kb <= kb_end; kb += 8) {  // two blocks per trip, the register sets alternating
            load(min(kb + 4, kb_end), kn, vn);
            step(kb, ka, va);
            if (kb + 4 > kb_end) break;
            load(min(kb + 8, kb_end), ka, va);
            step(kb + 4, kn, vn);
        }
        // this wave's partial: column c, d = 32·grp + 8r + dt
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int dt = 0; dt < 8; dt += 4)
                *(float4*)&po[w][c][32 * grp + 8 * r + dt] = make_float4(o[dt][r], o[dt + 1][r], o[dt + 2][r], o[dt + 3][r]);
        if (grp == 0) {
            pm[w][c] = m;
            pl[w][c] = l;
        }
        __syncthreads();
        {  // merge the 4 waves: thread → column tid/16, d [8·(tid%16), +8)
            const int cc = tid >> 4, d0 = 8 * (tid & 15);
            float M = -INFINITY;
#pragma unroll
            for (int v = 0; v < 4; v++) M = fmaxf(M, pm[v][cc]);
            float wgt[4], L = 0.0f;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                wgt[v] = pm[v][cc] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(pm[v][cc] - M);
                L += wgt[v] * pl[v][cc];
            }
            float acc[8] = {};
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float4 a = *(const float4*)&po[v][cc][d0];
                const float4 b = *(const float4*)&po[v][cc][d0 + 4];
                acc[0] += wgt[v] * a.x; acc[1] += wgt[v] * a.y; acc[2] += wgt[v] * a.z; acc[3] += wgt[v] * a.w;
                acc[4] += wgt[v] * b.x; acc[5] += wgt[v] * b.y; acc[6] += wgt[v] * b.z; acc[7] += wgt[v] * b.w;
            }
            const int qq = q0 + cc / G, hh = g * G + cc % G;
            if (qq < n) {
                const float inv = 1.0f / L;
                float* dst = out + (int64_t)qq * nh * HD + (int64_t)hh * HD + d0;
                *(float4*)dst = make_float4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
                *(float4*)(dst + 4) = make_float4(acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv);
            }
        }
        __syncthreads();  // LDS is reused by the second query block
    }
}

// ── Long prompts: the same attention on the fp16 matrix cores ─────────────
// The f32 matrix cores run at a sixteenth of the fp16 rate. Here q, k, v and the
// probabilities are each split into two fp16 parts, x·2^-e = hi + lo (22
// significant bits), and a product takes three passes, lo·hi, hi·lo and hi·hi
// (the dropped lo·lo is 2^-24 of it), on v_mfma_f32_32x32x16_f16: the error
// against f64 is below the f32 kernel's (n = 1000 / 2000 / 4000: 1.7 / 1.8 / 1.9e-7
// of a result against 1.9 / 2.3 / 2.7e-7).
//  * k_attn_split lays K and V out once per call, per KV head and tile of 32
//    keys, as MFMA fragments with one power of two each for the tile's K and V
//    (32 KiB a tile; its exponents beside). Keys past the last are zero.
//  * k_attn_prefill_sp: workgroup = 128 columns (128/G queries × G heads of a KV
//    head, the query-block pair {p, last − p}); wave = 32 columns × every other
//    key tile. A stage of two tiles (64 KiB) is loaded to LDS while the stage
//    before it is used. Sᵀ = K·Qᵀ leaves a lane 16 keys of one column; V's
//    fragments take their keys in that order, so the probabilities are the B
//    operand of Oᵀ = Vᵀ·Pᵀ as they stand. Probabilities are taken against a
//    maximum that may be 2^8 stale, and a tile's enter its product times a power
//    of two of their column's largest, so that neither a flat row nor a tile far
//    below the maximum has them in fp16's subnormals.
// What bounds it: at n = 2000 (32 / 8 heads: 325 → 117 µs, 7 of it k_attn_split) the matrix cores are busy a third
// of the time, 30 % of the waves' time goes to waits for LDS and the stage barrier, 37 % to dependencies. Not the
// phases of a SIMD's two waves: an odd wave that multiplies its values a stage late took 138 µs, four
// independent chains in place of two 153; without the stage loads it would take 115.
// The parts are 22 bits of a value while it is no smaller than 2^-16 of the largest that shares its power of two (below
// that a fixed 2^-39 of the largest). Where that would show, f32 sums on the VALU run instead (sp_plain, 880 .. 980 µs for
// that prompt): for a KV head of which some tile has SP_FEW groups of eight (eight dimensions of a key; a dimension of eight
// values' rows) below 2^-16 of its largest and not all zero, so that a key or a dimension is out of proportion (a key has 16
// such groups, a dimension of the values 4; of normal numbers a group with one key left in the last tile is one in 10^4
// times), or an infinity or NaN (the split has none, and a masked key's must not reach the queries before it); and for
// 128 columns with a query of which, of a lane's eight groups of eight dimensions, five stay below 2^-13 of its largest.
#define SP_TILE 32768  // bytes of a key tile's fragments: K [8 k-steps][hi, lo][1 KiB], V [4 d-tiles][2 halves][hi, lo][1 KiB]
#define SP_BAD 0x7FFF  // exponent of a tile for sp_plain: an infinity or NaN, too wide a range, or numbers past 2^64
#define SP_MAXE 50     // largest exponent of a score's factors: no product of their scales overflows
#define SP_FEW 4       // groups of eight numbers below 2^-16 of the largest that make a tile's range too wide

typedef _Float16 sp_h8 __attribute__((ext_vector_type(8)));
typedef float sp_f16 __attribute__((ext_vector_type(16)));

// 8 floats·2^-e → hi and lo
__device__ __forceinline__ void sp_split(const float (&x)[8], float inv, sp_h8& hi, sp_h8& lo) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float v = x[i] * inv;
        hi[i] = (_Float16)v;
        lo[i] = (_Float16)(v - (float)hi[i]);
    }
}
// e with |x|·2^-e < 2^14 for |x| <= mx (2^14 at most 2^100 away: the factors below stay normal)
__device__ __forceinline__ int sp_exponent(float mx) {
    int E = 14;
    if (mx > 0.0f) (void)frexpf(mx, &E);
    return max(E - 14, -100);
}

// a group's largest number g below 2^-bits of the largest mx, and not zero
__device__ __forceinline__ bool sp_small(float g, float mx, int bits) { return g > 0.0f && g < ldexpf(mx, -bits); }

__global__ void __launch_bounds__(256) k_attn_split(const float* __restrict__ layer_kv, int n, int nkv, int64_t max_seq,
                                                    int ntiles, uint8_t* __restrict__ frag, int2* __restrict__ exps) {
    __shared__ float red[2][4];
    __shared__ int bad, few;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int g = blockIdx.x % nkv, t = blockIdx.x / nkv, k0 = 32 * t;
    const float* K = layer_kv + (int64_t)g * max_seq * 128;
    const float* V = layer_kv + (int64_t)(nkv + g) * max_seq * 128;
    if (tid == 0) bad = few = 0;
    // K: k-steps w and w + 4, lane = key lane%32, d 16·ks + 8·(lane/32) + i. V: (d-tile, half) pairs w and w + 4,
    // lane = d 32·dt + lane%32, element i = key 16·half + 8·(i/4) + 4·(lane/32) + i%4 (Sᵀ's result order)
    float kx[2][8], vx[2][8], km = 0.0f, vm = 0.0f, kg[2] = {}, vg[2] = {};
    bool nf = false;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int ks = w + 4 * u, key = k0 + (lane & 31);
        const float* src = K + (int64_t)min(key, n - 1) * 128 + 16 * ks + 8 * (lane >> 5);
        const float4 a = *(const float4*)src, b = *(const float4*)(src + 4);
        const float r[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        const int dt = ks >> 1, hf = ks & 1;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            kx[u][i] = key < n ? r[i] : 0.0f;
            const int vk = k0 + 16 * hf + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
            const float x = V[(int64_t)min(vk, n - 1) * 128 + 32 * dt + (lane & 31)];
            vx[u][i] = vk < n ? x : 0.0f;
            nf |= !(fabsf(kx[u][i]) < INFINITY) || !(fabsf(vx[u][i]) < INFINITY);
            kg[u] = fmaxf(kg[u], fabsf(kx[u][i]));
            vg[u] = fmaxf(vg[u], fabsf(vx[u][i]));
        }
    }
    km = fmaxf(kg[0], kg[1]);
    vm = fmaxf(vg[0], vg[1]);
    km = aeth_wave_max(km);
    vm = aeth_wave_max(vm);
    __syncthreads();
    if (nf) bad = 1;
    if (lane == 0) {
        red[0][w] = km;
        red[1][w] = vm;
    }
    __syncthreads();
    km = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    vm = fmaxf(fmaxf(red[1][0], red[1][1]), fmaxf(red[1][2], red[1][3]));
    const int ek = sp_exponent(km), ev = sp_exponent(vm);
    const int c = sp_small(kg[0], km, 16) + sp_small(kg[1], km, 16) + sp_small(vg[0], vm, 16) + sp_small(vg[1], vm, 16);
    if (c) atomicAdd(&few, c);
    const float ki = ldexpf(1.0f, -ek), vi = ldexpf(1.0f, -ev);
    uint8_t* dst = frag + ((int64_t)g * ntiles + t) * SP_TILE + lane * 16;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        sp_h8 hi, lo;
        sp_split(kx[u], ki, hi, lo);
        *(sp_h8*)(dst + (w + 4 * u) * 2048) = hi;
        *(sp_h8*)(dst + (w + 4 * u) * 2048 + 1024) = lo;
        sp_split(vx[u], vi, hi, lo);
        *(sp_h8*)(dst + 16384 + (w + 4 * u) * 2048) = hi;
        *(sp_h8*)(dst + 16384 + (w + 4 * u) * 2048 + 1024) = lo;
    }
    __syncthreads();
    if (tid == 0) {
        const bool wide = few >= SP_FEW || ek > SP_MAXE || ev > SP_MAXE;
        exps[g * ntiles + t] = bad || wide ? make_int2(SP_BAD, SP_BAD) : make_int2(ek, ev);
    }
}

// 128 columns in f32 on the VALU (rare), the queries from q0 on: tiles of 32 keys through LDS, thread = (two columns
// 2·(tid/8), dimensions [16·(tid%8), +16)), a score summed over eight lanes. A masked key's value enters nothing.
struct SpPlain {
    float k[32][132], v[32][132], p[128][33];
};
template <int G>
__device__ __forceinline__ void sp_plain(const float* qkv, int64_t qkv_stride, const float* K, const float* V, int n, int nh,
                                      int g, int q0, int window, float* out, SpPlain* sh) {
    const int tid = threadIdx.x, c0 = 2 * (tid >> 3), part = tid & 7, d0 = 16 * part;
    const float scale = 1.0f / sqrtf(128.0f);
    int query[2], lo[2];  // keys [lo, query] are visible
    float q[2][16], o[2][16] = {}, m[2] = {-INFINITY, -INFINITY}, l[2] = {};
#pragma unroll
    for (int c = 0; c < 2; c++) {
        query[c] = q0 + (c0 + c) / G;
        lo[c] = window > 0 ? query[c] - window + 1 : 0;
        const float* src = qkv + (int64_t)min(query[c], n - 1) * qkv_stride + (int64_t)(g * G + (c0 + c) % G) * 128 + d0;
#pragma unroll
        for (int d = 0; d < 16; d += 4) {
            const float4 x = *(const float4*)(src + d);
            q[c][d] = x.x; q[c][d + 1] = x.y; q[c][d + 2] = x.z; q[c][d + 3] = x.w;
        }
    }
    const int kb_end = (min(q0 + 128 / G, n) - 1) / 32, kb_beg = window > 0 ? max(0, q0 - window + 1) / 32 : 0;
    for (int kb = kb_beg; kb <= kb_end; kb++) {
        __syncthreads();
        for (int i = tid; i < 32 * 32; i += 512) {
            const int t = i >> 5, d = 4 * (i & 31);
            *(float4*)&sh->k[t][d] = *(const float4*)(K + (int64_t)min(32 * kb + t, n - 1) * 128 + d);
            *(float4*)&sh->v[t][d] = *(const float4*)(V + (int64_t)min(32 * kb + t, n - 1) * 128 + d);
        }
        __syncthreads();
        float s[2][4], mx[2] = {-INFINITY, -INFINITY};  // of this lane's keys part + 8u
#pragma unroll
        for (int t = 0; t < 32; t++) {
            float a[2] = {0.0f, 0.0f};
#pragma unroll
            for (int d = 0; d < 16; d += 4) {
                const float4 y = *(const float4*)&sh->k[t][d0 + d];
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    a[c] = fmaf(q[c][d], y.x, a[c]);
                    a[c] = fmaf(q[c][d + 1], y.y, a[c]);
                    a[c] = fmaf(q[c][d + 2], y.z, a[c]);
                    a[c] = fmaf(q[c][d + 3], y.w, a[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < 2; c++) {
                a[c] += aeth_dpp_xor1f(a[c]);
                a[c] += aeth_dpp_xor2f(a[c]);
                a[c] += aeth_dpp_mirror8f(a[c]);
                s[c][t >> 3] = (t & 7) == part ? a[c] * scale : s[c][t >> 3];
            }
            if ((t & 3) == 3) __builtin_amdgcn_sched_barrier(0);  // four keys' reads in flight
        }
        float al[2];
#pragma unroll
        for (int c = 0; c < 2; c++) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int t = 32 * kb + part + 8 * u;
                if (t < lo[c] || t > query[c]) s[c][u] = -INFINITY;
                mx[c] = fmaxf(mx[c], s[c][u]);
            }
            mx[c] = fmaxf(mx[c], aeth_dpp_xor1f(mx[c]));
            mx[c] = fmaxf(mx[c], aeth_dpp_xor2f(mx[c]));
            mx[c] = fmaxf(mx[c], aeth_dpp_mirror8f(mx[c]));
            const float mn = fmaxf(m[c], mx[c]);
            al[c] = mn == -INFINITY ? 1.0f : expf(m[c] - mn);
            m[c] = mn;
            l[c] *= al[c];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int t = 32 * kb + part + 8 * u;
                const float p = t >= lo[c] && t <= query[c] && mn != -INFINITY ? expf(s[c][u] - mn) : 0.0f;
                sh->p[c0 + c][part + 8 * u] = p;
                l[c] += p;
            }
#pragma unroll
            for (int d = 0; d < 16; d++) o[c][d] *= al[c];
        }
        __syncthreads();
        const int t0 = max(min(lo[0], lo[1]) - 32 * kb, 0), t1 = min(max(query[0], query[1]) - 32 * kb, 31);
#pragma unroll 4
        for (int t = t0; t <= t1; t++) {
            float4 y[4];
#pragma unroll
            for (int d = 0; d < 4; d++) y[d] = *(const float4*)&sh->v[t][d0 + 4 * d];
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int key = 32 * kb + t;
                const float p = sh->p[c0 + c][t];
                if (key < lo[c] || key > query[c]) continue;
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    o[c][4 * d] = fmaf(p, y[d].x, o[c][4 * d]);
                    o[c][4 * d + 1] = fmaf(p, y[d].y, o[c][4 * d + 1]);
                    o[c][4 * d + 2] = fmaf(p, y[d].z, o[c][4 * d + 2]);
                    o[c][4 * d + 3] = fmaf(p, y[d].w, o[c][4 * d + 3]);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 2; c++) {
        l[c] += aeth_dpp_xor1f(l[c]);
        l[c] += aeth_dpp_xor2f(l[c]);
        l[c] += aeth_dpp_mirror8f(l[c]);
        const float inv = 1.0f / l[c];
        if (query[c] < n) {
            float* dst = out + (int64_t)query[c] * nh * 128 + (int64_t)(g * G + (c0 + c) % G) * 128 + d0;
#pragma unroll
            for (int d = 0; d < 16; d += 4)
                *(float4*)(dst + d) = make_float4(o[c][d] * inv, o[c][d + 1] * inv, o[c][d + 2] * inv, o[c][d + 3] * inv);
        }
    }
    __syncthreads();  // LDS is used again
}

template <int G>
__global__ void __launch_bounds__(512, 2) k_attn_prefill_sp(const float* __restrict__ qkv, int64_t qkv_stride,
                                                            const float* __restrict__ layer_kv,
                                                            const uint8_t* __restrict__ frag,
                                                            const int2* __restrict__ exps, int n, int nh, int nkv,
                                                            int64_t max_seq, int ntiles, int window,
                                                            float* __restrict__ out) {
    constexpr int QB = 128 / G, PLD = 132;
    constexpr float TH = 8.0f;  // log2: how stale a maximum may be
    // two stages of two tiles (128 KiB), then the partial results [key parity][column][PLD] and their statistics
    __shared__ __attribute__((aligned(1024))) char smem[2 * 128 * PLD * 4];
    static_assert(sizeof(SpPlain) <= sizeof(smem), "the f32 form's LDS");
    __shared__ float pm[2][128], pl[2][128];
    __shared__ int pe[2][4];
    __shared__ __attribute__((aligned(16))) int far[2][8];  // [pass][wave]: a query of the wave's is for sp_plain
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), cg = w & 3, par = w >> 2;
    const int c = 32 * cg + (lane & 31), hf = lane >> 5;
    const int g = blockIdx.x % nkv, p = blockIdx.x / nkv;
    const int nqb = (n + QB - 1) / QB;
    const int head = g * G + c % G;
    const uint8_t* fr = frag + (int64_t)g * ntiles * SP_TILE;
    const int2* ex = exps + g * ntiles;
    bool bad = false;
    for (int t = lane; t < ntiles; t += 64) bad |= ex[t].x == SP_BAD;
    bad = __any(bad);
    if (lane < 2) far[lane][w] = 0;  // (a wave's own: no barrier; a store to LDS under the stage's loads would wait for them)
    const uint32_t sm0 = lds_addr(smem);
    const float sl2 = 1.4426950408889634f / sqrtf(128.0f);  // scale · log2(e)
    for (int pass = 0; pass < 2; pass++) {
        const int qb = pass == 0 ? p : nqb - 1 - p;
        if (pass == 1 && qb == p) break;  // the middle block of an odd count (uniform)
        const int q0 = qb * QB, query = q0 + c / G;
        bool again = bad;
        if (!bad) {
        const int kb_end = (min(q0 + QB, n) - 1) / 32;                           // last key tile, inclusive
        const int kb_beg = window > 0 ? max(0, q0 - window + 1) / 32 : 0;        // first one any query sees
        const int w_lo = q0 + 32 * cg / G, w_hi = q0 + (32 * cg + 31) / G;       // this wave's queries
        // tiles kb_beg + 2·st + {0, 1} (past the last: the last again) → buffer st%2, 8 of the 64 KiB a wave
        auto issue = [&](int st) {
            const uint8_t* src = fr + (int64_t)min(kb_beg + 2 * st + (w >> 2), kb_end) * SP_TILE + (w & 3) * 8192 + lane * 16;
            char* dst = smem + (st & 1) * 65536 + w * 8192;
#pragma unroll
            for (int i = 0; i < 8; i++) __builtin_amdgcn_global_load_lds(src + i * 1024, (lds_void*)(dst + i * 1024), 16, 0, 0);
        };
        issue(0);
        sp_h8 qh[8], ql[8];
        float fq;
        {
            const float* src = qkv + (int64_t)min(query, n - 1) * qkv_stride + (int64_t)head * 128 + 8 * hf;
            float x[8][8], xg[8], mx = 0.0f;
#pragma unroll
            for (int ks = 0; ks < 8; ks++) {
                const float4 a = *(const float4*)(src + 16 * ks), b = *(const float4*)(src + 16 * ks + 4);
                x[ks][0] = a.x; x[ks][1] = a.y; x[ks][2] = a.z; x[ks][3] = a.w;
                x[ks][4] = b.x; x[ks][5] = b.y; x[ks][6] = b.z; x[ks][7] = b.w;
#pragma unroll
                for (int i = 0; i < 8; i++) xg[ks] = i ? fmaxf(xg[ks], fabsf(x[ks][i])) : fabsf(x[ks][0]);
                mx = fmaxf(mx, xg[ks]);
            }
            mx = pa_max32(mx);
            const int eq = sp_exponent(mx < INFINITY ? mx : 0.0f);  // an infinity makes the column NaN
            int few = eq > SP_MAXE ? 8 : 0;
#pragma unroll
            for (int ks = 0; ks < 8; ks++) few += sp_small(xg[ks], mx, 13) ? 1 : 0;
            if (__any(few > 4)) far[pass][w] = 1;  // (a branch: the store waits for the loads in flight) read after the pass
            __builtin_amdgcn_sched_barrier(0);
            const float inv = ldexpf(1.0f, -eq);
#pragma unroll
            for (int ks = 0; ks < 8; ks++) sp_split(x[ks], inv, qh[ks], ql[ks]);
            fq = ldexpf(sl2, eq);
        }
        float m = -INFINITY, l = 0.0f;
        int eo = -1000;  // the output's exponent: V tiles with a larger one raise it
        sp_f16 o[4];
#pragma unroll
        for (int dt = 0; dt < 4; dt++) o[dt] = (sp_f16){};
        const int nst = (kb_end - kb_beg) / 2 + 1;
        sp_h8 ph[2], plo[2];  // the probabilities of a tile, hi and lo
        float ve = 0.0f;      // and the scale of their product with its values against the output's
        // o += Vᵀ·Pᵀ of the tile whose V is at vb. A tile's product forms apart, takes the tile's exponent and is added
        // once: six roundings of a small sum and one of o, not six of o
        auto values = [&](uint32_t vb) {
            constexpr int LA = 2;  // fragments read ahead
            sp_h8 f[LA + 1][2];
            sp_f16 t4[2];
#pragma unroll
            for (int u = 0; u < LA; u++) {
                f[u][0] = lds_b128h<0>(vb + u * 2048);
                f[u][1] = lds_b128h<1024>(vb + u * 2048);
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {  // (d-tile u/2, key half u%2)
                const int dt = u >> 1, c = u % (LA + 1);
                if (u < 8 - LA) {
                    f[(u + LA) % (LA + 1)][0] = lds_b128h<0>(vb + (u + LA) * 2048);
                    f[(u + LA) % (LA + 1)][1] = lds_b128h<1024>(vb + (u + LA) * 2048);
                    lgkm_wait<2 * LA>();
                } else if (u == 6) {
                    lgkm_wait<2>();
                } else {
                    lgkm_wait<0>();
                }
                pin(f[c][0]);
                pin(f[c][1]);
                sp_f16 x = (u & 1) ? t4[dt & 1] : (sp_f16){};
                x = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[c][1], ph[u & 1], x, 0, 0, 0);
                x = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[c][0], plo[u & 1], x, 0, 0, 0);
                t4[dt & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[c][0], ph[u & 1], x, 0, 0, 0);
                if ((u & 1) == 0 && dt > 0) o[dt - 1] += t4[(dt - 1) & 1] * ve;  // under this d-tile's products
            }
            o[3] += t4[1] * ve;
        };
        // Sᵀ of the tile whose K is at kb, and its probabilities
        auto scores = [&](uint32_t kb, int t0, int2 e) {
            sp_f16 s0[2] = {(sp_f16){}, (sp_f16){}}, s1 = (sp_f16){};  // hi·hi in two chains, the lo passes
            constexpr int LA = 2;
            sp_h8 f[LA + 1][2];
#pragma unroll
            for (int u = 0; u < LA; u++) {
                f[u][0] = lds_b128h<0>(kb + u * 2048);
                f[u][1] = lds_b128h<1024>(kb + u * 2048);
            }
#pragma unroll
            for (int ks = 0; ks < 8; ks++) {
                const int c = ks % (LA + 1);
                if (ks < 8 - LA) {
                    f[(ks + LA) % (LA + 1)][0] = lds_b128h<0>(kb + (ks + LA) * 2048);
                    f[(ks + LA) % (LA + 1)][1] = lds_b128h<1024>(kb + (ks + LA) * 2048);
                    lgkm_wait<2 * LA>();
                } else if (ks == 6) {
                    lgkm_wait<2>();
                } else {
                    lgkm_wait<0>();
                }
                pin(f[c][0]);
                pin(f[c][1]);
                s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[c][1], qh[ks], s1, 0, 0, 0);
                s0[ks & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[c][0], qh[ks], s0[ks & 1], 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[c][0], ql[ks], s1, 0, 0, 0);
            }
            const float fs = ldexpf(fq, e.x);
            float s[16], mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = ((s0[0][r] + s0[1][r]) + s1[r]) * fs;
            if (!(t0 + 31 <= w_lo && t0 + 31 < n && (window <= 0 || t0 > w_hi - window))) {  // some key is masked (uniform)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int key = t0 + 8 * (r >> 2) + 4 * hf + (r & 3);
                    if (!(key <= query && key < n && (window <= 0 || key > query - window))) s[r] = -INFINITY;
                }
            }
#pragma unroll
            for (int r = 0; r < 16; r++) mx = fmaxf(mx, s[r]);
            mx = pa_max32(mx);
            if (__any(mx > m + TH)) {  // uniform
                const float mn = fmaxf(m, mx), al = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
                l *= al;
#pragma unroll
                for (int dt = 0; dt < 4; dt++) o[dt] *= al;
                m = mn;
            }
            if (e.y > eo) {  // uniform
                const float al = ldexpf(1.0f, max(eo - e.y, -250));
#pragma unroll
                for (int dt = 0; dt < 4; dt++) o[dt] *= al;
                eo = e.y;
            }
            const float mo = m == -INFINITY ? 0.0f : m;  // every key masked so far: s − mo is −Inf
            // the tile's largest probability of this column times 2^j lies in (2^12, 2^13]
            const int j = mx == -INFINITY ? 0 : 13 - max((int)ceilf(mx - mo), -100);
            const float fj = ldexpf(1.0f, j);
            ve = ldexpf(1.0f, max(e.y - eo, -120) - j);
#pragma unroll
            for (int r = 0; r < 16; r++) {
                s[r] = __builtin_amdgcn_exp2f(s[r] - mo);
                const float pv = s[r] * fj;
                ph[r >> 3][r & 7] = (_Float16)pv;
                plo[r >> 3][r & 7] = (_Float16)(pv - (float)ph[r >> 3][r & 7]);
            }
#pragma unroll
            for (int h = 8; h >= 1; h /= 2)  // the tile's sum as a tree: one rounding of l a tile
#pragma unroll
                for (int r = 0; r < h; r++) s[r] += s[r + h];
            l += s[0];
        };
        for (int st = 0; st < nst; st++) {
            const int t = kb_beg + 2 * st + par, t0 = 32 * t;
            vm_wait<0>();                 // this wave's part of stage st has landed
            __builtin_amdgcn_s_barrier();  // and every wave's; the other stage's buffers are read
            if (st + 1 < nst) issue(st + 1);
            if (t > kb_end || t0 > w_hi || (window > 0 && t0 + 31 <= w_lo - window)) continue;  // nothing visible (uniform)
            const uint32_t at = sm0 + (st & 1) * 65536 + par * 32768 + lane * 16;
            scores(at, t0, ex[t]);
            values(at + 16384);
        }
        __syncthreads();  // the stages are read: their LDS takes the partial results
        float* po = (float*)smem + (par * 128 + c) * PLD;
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int r = 0; r < 16; r += 4)  // d = 32·dt + 2·r + 4·hf
                *(float4*)(po + 32 * dt + 2 * r + 4 * hf) = make_float4(o[dt][r], o[dt][r + 1], o[dt][r + 2], o[dt][r + 3]);
        l = pa_sum32(l);
        if (hf == 0) {
            pm[par][c] = m;
            pl[par][c] = l;
        }
        if (lane == 0) pe[par][cg] = eo;
        __syncthreads();
        {  // merge the two key parities: thread → column tid/4, d 4·(tid%4) + 16·i
            const int cc = tid >> 2, qq = q0 + cc / G, hh = g * G + cc % G;
            const float m0 = pm[0][cc], m1 = pm[1][cc], M = fmaxf(m0, m1);
            const float w0 = m0 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m0 - M);
            const float w1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - M);
            const float inv = 1.0f / (w0 * pl[0][cc] + w1 * pl[1][cc]);
            const float a0 = ldexpf(w0 * inv, pe[0][cc >> 5]), a1 = ldexpf(w1 * inv, pe[1][cc >> 5]);
            const float* x0 = (const float*)smem + cc * PLD;
            const float* x1 = x0 + 128 * PLD;
            if (qq < n) {
                float* dst = out + (int64_t)qq * nh * 128 + (int64_t)hh * 128;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int d = 4 * (tid & 3) + 16 * i;
                    const float4 u = *(const float4*)(x0 + d), v = *(const float4*)(x1 + d);
                    *(float4*)(dst + d) = make_float4(a0 * u.x + a1 * v.x, a0 * u.y + a1 * v.y, a0 * u.z + a1 * v.z,
                                                      a0 * u.w + a1 * v.w);
                }
            }
        }
        __syncthreads();  // LDS is reused by the second query block
        const int4 f0 = *(const int4*)&far[pass][0], f1 = *(const int4*)&far[pass][4];
        if (__builtin_amdgcn_readfirstlane(f0.x | f0.y | f0.z | f0.w | f1.x | f1.y | f1.z | f1.w)) again = true;
        }
        if (again)  // the pass's rows in f32
            sp_plain<G>(qkv, qkv_stride, layer_kv + (int64_t)g * max_seq * 128, layer_kv + (int64_t)(nkv + g) * max_seq * 128, n,
                        nh, g, q0, window, out, (SpPlain*)smem);
    }
}

// The split form where it is the faster one: once the f32 kernel's workgroups (eight for one of these) no longer fit the
// chip at once, two a CU. µs here and on the f32 kernel by its workgroups on 256 CUs: 512 (32 / 8 heads, n = 512) 43.7 / 35.4,
// (16 / 8, 1024) 63.3 / 51.4, (16 / 2, 1024) 62.6 / 51.9, (64 / 8, 256) 34.0 / 24.5; 544 (32 / 8, 544) 45.5 / 50.7, 576 46.7 / 51.2,
// 552 (16 / 8, 1100) 68 / 79, 600 (32 / 4, 600) 48.8 / 52.7, 640 (64 / 8, 320) 37.0 / 37.4, (32 / 8, 640) 49 / 54; 1200 (32 / 4,
// 1200) 74 / 136, n = 2000 at 32 / 8 heads 117 / 330, 4000 414 / 1318.
// It needs a scratch of 32 KiB per KV head and 32 keys, the stream's own; under graph capture, where that could not grow
// and a recorded address would not outlive a later growth, and where there is no memory for it, the f32 kernel runs.
// Two host threads may call on one stream: from the fetch of the scratch to the launch that reads it a call holds a
// lock, or another's fragments (or a growth that frees the buffer) could come between its two kernels.
static std::mutex g_split_mu;
template <int G>
static bool attn_split_launch(const float* qkv, int64_t stride, const float* layer_kv, int64_t n, int64_t nh, int64_t nkv,
                              int64_t max_seq, int win, float* out, hipStream_t s, int* rc) {
    *rc = AETH_OK;
    const int64_t nqb = aeth_cdiv(n, 128 / G), wgs = nkv * aeth_cdiv(nqb, 2), nt = aeth_cdiv(n, 32);
    if (nkv * aeth_cdiv(aeth_cdiv(n, 16 / G), 2) <= 2 * aeth_num_cus()) return false;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cs) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (cs != hipStreamCaptureStatusNone) return false;
    const int64_t fb = nkv * nt * SP_TILE;
    void* ws = nullptr;
    std::lock_guard<std::mutex> lk(g_split_mu);
    if (!aeth_stream_scratch_try(s, AETH_SCRATCH_PATTN, (size_t)(fb + nkv * nt * sizeof(int2)), &ws)) return false;
    int2* ex = (int2*)((uint8_t*)ws + fb);
    hipLaunchKernelGGL(k_attn_split, dim3((unsigned)(nkv * nt)), dim3(256), 0, s, layer_kv, (int)n, (int)nkv, max_seq, (int)nt,
                       (uint8_t*)ws, ex);
    hipLaunchKernelGGL(k_attn_prefill_sp<G>, dim3((unsigned)wgs), dim3(512), 0, s, qkv, stride, layer_kv, (const uint8_t*)ws, ex,
                       (int)n, (int)nh, (int)nkv, max_seq, (int)nt, win, out);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) *rc = aeth_set_error(AETH_EHIP, "prefill attention: launch failed: %s", hipGetErrorString(e));
    return true;
}

int aeth_attn_prefill_launch(const float* qkv, int64_t stride, const float* layer_kv, int64_t n, int64_t nh,
                             int64_t nkv, int64_t hd, int64_t max_seq, int64_t window, float* out, hipStream_t s) {
    if (n <= 0) return AETH_OK;
    const int win = window > 0 && window < n ? (int)window : 0;  // a window reaching back past key 0 masks nothing
    if (hd != 128 || nh % nkv != 0)
        return aeth_set_error(AETH_EUNSUPPORTED, "prefill attention: head_dim %lld (needs 128)", (long long)hd);
    // AETH_PREFILL_ATTN=valu selects the f32 VALU kernel (comparison, tests)
    static const bool force_valu = getenv("AETH_PREFILL_ATTN") && !strcmp(getenv("AETH_PREFILL_ATTN"), "valu");
    const int64_t G = nh / nkv;
    if (!force_valu && (G == 1 || G == 2 || G == 4 || G == 8)) {
        int rc;
        if (G == 1 ? attn_split_launch<1>(qkv, stride, layer_kv, n, nh, nkv, max_seq, win, out, s, &rc)
            : G == 2 ? attn_split_launch<2>(qkv, stride, layer_kv, n, nh, nkv, max_seq, win, out, s, &rc)
            : G == 4 ? attn_split_launch<4>(qkv, stride, layer_kv, n, nh, nkv, max_seq, win, out, s, &rc)
                     : attn_split_launch<8>(qkv, stride, layer_kv, n, nh, nkv, max_seq, win, out, s, &rc))
            return rc;
        const int64_t nqb = aeth_cdiv(n, 16 / G);
        const dim3 grid((unsigned)(nkv * aeth_cdiv(nqb, 2)));
        if (G == 1) hipLaunchKernelGGL(k_attn_prefill_mf<1>, grid, dim3(256), 0, s, qkv, stride, layer_kv, (int)n, (int)nh, (int)nkv, max_seq, win, out);
        else if (G == 2) hipLaunchKernelGGL(k_attn_prefill_mf<2>, grid, dim3(256), 0, s, qkv, stride, layer_kv, (int)n, (int)nh, (int)nkv, max_seq, win, out);
        else if (G == 4) hipLaunchKernelGGL(k_attn_prefill_mf<4>, grid, dim3(256), 0, s, qkv, stride, layer_kv, (int)n, (int)nh, (int)nkv, max_seq, win, out);
        else hipLaunchKernelGGL(k_attn_prefill_mf<8>, grid, dim3(256), 0, s, qkv, stride, layer_kv, (int)n, (int)nh, (int)nkv, max_seq, win, out);
        AETH_LAUNCH_CHECK();
        return AETH_OK;
    }
    const size_t lds = sizeof(float) * ((size_t)(PA_BQ + 2 * PA_BK) * (128 + 4) + PA_BQ * (PA_BK + 1) + 3 * PA_BQ);
    static bool opted = false;
    if (!opted) {
        AETH_HIP_CHECK(hipFuncSetAttribute((const void*)k_attn_prefill<128>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)lds));
        opted = true;
    }
    hipLaunchKernelGGL(k_attn_prefill<128>, dim3((unsigned)aeth_cdiv(n, PA_BQ), (unsigned)nh), dim3(256), lds, s, qkv,
                       stride, layer_kv, (int)n, (int)nh, (int)nkv, max_seq, win, out);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}

// h[i][j] = g·σ(g)·u with (g, u) = gu[i][2j], gu[i][2j+1] (gate/up rows interleaved).
__global__ void k_silu_pairs(const float* __restrict__ gu, int64_t total, float* __restrict__ h) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const float2 p = *(const float2*)(gu + 2 * idx);
    h[idx] = p.x * (1.0f / (1.0f + expf(-p.x))) * p.y;
}

int aeth_silu_pairs_launch(const float* gu, int64_t total, float* h, hipStream_t s) {
    if (total <= 0) return AETH_OK;
    hipLaunchKernelGGL(k_silu_pairs, dim3((unsigned)aeth_cdiv(total, 256)), dim3(256), 0, s, gu, total, h);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}
