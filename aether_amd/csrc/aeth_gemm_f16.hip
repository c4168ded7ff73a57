// F16 prefill GEMM (m rows from aeth_f16_gemm_rows on):  C[m][n] = Σ_k A[m][k]·W[k][n], W the GGUF-order
// [k][n] halves load_quant keeps (quantized_matmul_impl's dequantize + matmul_f32_gguf route,
// src/quant/matmul/dispatch.rs:126-133, 541-574).
//
// The exact mode of the Q4_K GEMM: A·2^-e split into fp16 hi/lo MFMA fragments (k_gemm_prep in
// aeth_gemm.hip), f32 accumulation on v_mfma_f32_32x32x16_f16, two passes per product; the weights are
// their own exact operands. The reference skips a zero activation, which matters to weights that are
// infinite or NaN: weights holding one keep k_col (aeth_f16_gemm_rows). Rows that the two parts do not hold (an
// infinity; a largest value far above the others) come with zero fragments and the scale −1: the epilogue puts the
// negative of their f64 sum in place of the tile's, element by element over this workgroup's part of K.
//
// Work split as aeth_gemm_q80.hip: 64 × 128 workgroup tiles, 8 waves over eighths of the 16-position
// slices (and K over several workgroups when the tiles are few). Nothing is shared between waves and
// nothing is unpacked, so operands go straight into registers, the next slice's loads in flight under this
// slice's 16 MFMAs: an A fragment is 1 KiB in operand order, and lane (n, kg) reads columns 4n .. 4n + 3 of
// the eight k rows of its half (rows of 256 contiguous bytes). Operand column n of tile c is output column
// 4n + c, so the transpose is 16 v_perm a slice and a lane ends with four neighbouring outputs.
// What bounds it: operand bytes, 8 KiB per wave and slice (64 B per CU and clock at the full MFMA rate; the
// L2s deliver about a third of that). m = 333, 4096 × 4096: 456 → 40.5 µs with the prep;
// m = 512, 14336 × 4096: 1834 → 162 µs.
#include <math.h>
#include <stdint.h>

#include "aeth_common.hpp"
#include "aeth_gemm_common.hpp"
#include "aeth_internal.hpp"

#define F16_W 8

__global__ void __launch_bounds__(64 * F16_W) k_gemm_f16(F16Args G) {
    __shared__ __attribute__((aligned(16))) float red[4 * 2 * 4 * 16 * 64];  // 128 KiB
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tile, ks, nsplit, tm, tn;
    g2_work((int)blockIdx.x, G.gm, G.gn, G.ksplit, G.t_full, G.tsplit, tile, ks, nsplit);
    g2_tile(tile, G.gm, G.gn, tm, tn);
    const int n0 = tn * 128, m0 = tm * 64, nks = G.k >> 4;
    const int lo = nks * ks / nsplit, len = nks * (ks + 1) / nsplit - lo;  // this split's slices
    const int s0 = lo + len * wave / F16_W, s1 = lo + len * (wave + 1) / F16_W;

    const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc((void*)G.frag, (short)0, G.a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc((void*)G.w, (short)0, G.w_bytes, 0x00020000);
    const int a_v = lane * 16, aB[2] = {2 * tm * nks * 2048, (2 * tm + 1) * nks * 2048};
    // columns past n read the last four (never stored)
    const int ldw = G.n * 2, w_v = 8 * (lane >> 5) * ldw + min(n0 + 4 * (lane & 31), G.n - 4) * 2;

    f32x16 U[2][4];
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int c = 0; c < 4; c++) U[mt][c] = (f32x16){};
    struct Slice {
        u32x4 a[2][2];  // [m-tile][hi/lo]
        u32x2 w[8];     // k row i of this lane's half, columns 4n .. 4n + 3
    };
    auto load = [&](int s, Slice& S) {
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int p = 0; p < 2; p++)
                S.a[mt][p] = __builtin_amdgcn_raw_buffer_load_b128(rA, a_v, aB[mt] + s * 2048 + p * 1024, 0);
#pragma unroll
        for (int i = 0; i < 8; i++) S.w[i] = __builtin_amdgcn_raw_buffer_load_b64(rW, w_v, (16 * s + i) * ldw, 0);
    };
    auto step = [&](const Slice& S) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            // halves in k order [0, 2, 1, 3] per 4, as the prep orders A
            const uint32_t sel = (c & 1) ? 0x07060302u : 0x05040100u;
            u32x4 b;
            b[0] = __builtin_amdgcn_perm(S.w[2][c >> 1], S.w[0][c >> 1], sel);
            b[1] = __builtin_amdgcn_perm(S.w[3][c >> 1], S.w[1][c >> 1], sel);
            b[2] = __builtin_amdgcn_perm(S.w[6][c >> 1], S.w[4][c >> 1], sel);
            b[3] = __builtin_amdgcn_perm(S.w[7][c >> 1], S.w[5][c >> 1], sel);
            const half8_t bh = __builtin_bit_cast(half8_t, b);
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
                    U[mt][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, S.a[mt][p]), bh,
                                                                      U[mt][c], 0, 0, 0);
        }
    };
    Slice P, Q;
    if (s0 < s1) load(s0, P);
    int s = s0;
    for (; s + 1 < s1; s += 2) {  // two slices a trip, the register sets alternating
        load(s + 1, Q);
        __builtin_amdgcn_sched_barrier(0);
        step(P);
        __builtin_amdgcn_sched_barrier(0);
        load(min(s + 2, s1 - 1), P);
        __builtin_amdgcn_sched_barrier(0);
        step(Q);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (s < s1) step(P);

    // the eight K-eighth tiles meet in LDS: wave → m-tile wave/4, result registers [4·(wave%4), +4)
    const int mt = wave >> 2, r0 = 4 * (wave & 3), lr = lane & 31, col = n0 + 4 * lr;
    const int row0 = m0 + 32 * mt + 2 * r0 + 4 * (lane >> 5);  // row of register r0 + r: row0 + r
    float es[4];  // in flight during the reduction
#pragma unroll
    for (int r = 0; r < 4; r++) es[r] = G.escale[row0 + r];
    if (wave >= 4) {
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int r = 0; r < 16; r++) red[((((wave - 4) * 2 + q) * 4 + c) * 16 + r) * 64 + lane] = U[q][c][r];
    }
    __syncthreads();
    if (wave < 4) {
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int i = (((wave * 2 + q) * 4 + c) * 16 + r) * 64 + lane;
                    red[i] = U[q][c][r] + red[i];
                }
    }
    __syncthreads();
    float4 sum[4];
    float4 pv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float* p = red + ((mt * 4 + c) * 16 + r0 + r) * 64 + lane;
            v[c] = (p[0] + p[2 * 4 * 16 * 64]) + (p[2 * 2 * 4 * 16 * 64] + p[3 * 2 * 4 * 16 * 64]);
        }
        sum[r] = make_float4(v[0], v[1], v[2], v[3]);
    }
#pragma unroll
    for (int r = 0; r < 4; r++)
        if (es[r] < 0.0f) {  // rare (and then row0 + r < m)
            const float* a = G.A + (int64_t)(row0 + r) * G.k;
            const uint8_t* wc = G.w + 2 * (int64_t)min(col, G.n - 4);
            double d[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
            for (int i = 16 * lo; i < 16 * (lo + len); i++) {
                const uint2 h = *(const uint2*)(wc + (int64_t)i * ldw);
                const double x = (double)a[i];
                d[0] += x * (double)aeth_f16_to_f32(h.x & 0xFFFFu);
                d[1] += x * (double)aeth_f16_to_f32(h.x >> 16);
                d[2] += x * (double)aeth_f16_to_f32(h.y & 0xFFFFu);
                d[3] += x * (double)aeth_f16_to_f32(h.y >> 16);
            }
            sum[r] = make_float4((float)-d[0], (float)-d[1], (float)-d[2], (float)-d[3]);
        }
    if (nsplit > 1) {  // the split's partial tile (rows < mp, columns < pld: no bounds to check)
        int ld;
        float* P = g2_part(G.part, ks, tile, G.t_full, G.tsplit, G.gm * G.gn, G.mp, G.pld, m0, n0, ld) + 4 * lr;
#pragma unroll
        for (int r = 0; r < 4; r++) *(float4*)(P + (int64_t)(row0 + r - m0) * ld) = sum[r];
        return;
    }
    // n % 4 == 0: a lane's four columns are all below n or none. The loads precede the first store (it may alias).
    if (col >= G.n) return;
    if (G.accumulate) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float* p = G.C + (int64_t)min(row0 + r, G.m - 1) * G.ldc + col;
            pv[r] = G.c16 ? *(const float4*)p : make_float4(p[0], p[1], p[2], p[3]);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (row0 + r >= G.m) break;
        float4 v = make_float4(sum[r].x * es[r], sum[r].y * es[r], sum[r].z * es[r], sum[r].w * es[r]);
        if (G.accumulate) v = make_float4(pv[r].x + v.x, pv[r].y + v.y, pv[r].z + v.z, pv[r].w + v.w);
        float* p = G.C + (int64_t)(row0 + r) * G.ldc + col;
        if (G.c16) {
            *(float4*)p = v;
        } else {
            p[0] = v.x; p[1] = v.y; p[2] = v.z; p[3] = v.w;
        }
    }
}

int aeth_gemm_f16_kernel_launch(const F16Args& G, hipStream_t s) {
    hipLaunchKernelGGL(k_gemm_f16, dim3(g2_grid(G)), dim3(64 * F16_W), 0, s, G);
    AETH_LAUNCH_CHECK();
    return g2_split_sum(G, s);
}
