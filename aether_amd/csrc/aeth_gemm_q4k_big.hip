// Q4_K prefill GEMM for large products (aeth_q4k_big_ok):  C[m][n] = Σ_k A[m][k]·W[n][k]
// (avx2::matmul_q4_k with m rows, src/quant/avx2.rs:23-57; quantized_matmul_impl).
//
// The exact mode of aeth_gemm.hip on the same operands as aeth_gemm_kq.hip, tiled for operand bytes. There
// every wave streams its own operands for a 64 × 128 tile, 5.1 KiB a slice of 16 K positions for 16 MFMAs, and
// the chip's L2s deliver about 13 TB/s of that: 40 B per CU and clock wanted at the full matrix rate, 22 had.
// Here a workgroup owns 128 × 256 of C and shares its operands through LDS, 10.3 KiB a slice for 64 MFMAs
// (20 B per clock): wave (wm, wn) of 2 × 4 computes rows 64·wm, columns 64·wn, and each A fragment is read by four
// waves, each quant by two.
//
// A stage is 32 K positions, the two slices (low and high nibbles) of one 16-byte quant piece: 16 KiB of A
// fragments, 4 KiB of quants; a super-block's first stage also brings its headers and the rows' sub-block sums
// (8 KiB). Four stages are in the ring (six or seven measured the same); one barrier a stage, in its middle: then every
// wave has the next slice's operands to read while it multiplies, dequantising between the MFMAs (reading and
// dequantising before the MFMAs instead: 137 µs at 512 × 14336 × 4096, now 126).
// P holds the products of one super-block, U the result: leaving a super-block, U += d·P − 32·dmin·Q
// (Q = Σ_s m_s·S_s, one more MFMA), so a sum runs through 32 MFMAs and one add per super-block; against 64 bits
// the relative error is 1.9e-7 (the 64 × 128 kernel 2.2e-7).
// What bounds it: 512 × 14336 × 4096 takes 121 µs after the prep, 0.99 PFLOP/s of fp16 MFMAs with 224 of 256 CUs
// at work (a library bf16 product reaches 1.21 on the whole card); the 64 × 128 kernel takes 152.
#include <math.h>
#include <stdint.h>

#include "aeth_common.hpp"
#include "aeth_gemm_common.hpp"
#include "aeth_internal.hpp"

#define QB_A 16384               // a stage's A fragments: [m-tile 4][slice 2][hi, lo][1 KiB]
#define QB_STAGE (QB_A + 4096)   // + quants [tile 16][row 16][16 B]
#define QB_NST 4
#define QB_HDR (QB_NST * QB_STAGE)   // headers [tile 16][row 16][16 B], then sums [m-tile 4][hi, lo][row 32][16 B]
#define QB_LDS (QB_HDR + 2 * 8192)  // two super-blocks'

// loads a wave issues for stage position j of a super-block, and for the QB_NST − 2 stages after position j + 1
__host__ __device__ constexpr int qb_loads(int j) { return 4 + ((j & 7) == 0 ? 4 : 0); }
__host__ __device__ constexpr int qb_after(int j) {
    int v = 0;
    for (int i = 2; i < QB_NST; i++) v += qb_loads(j + i);
    return v;
}

__global__ void __launch_bounds__(512) k_gemm_q4k_big(KqArgs G) {
    __shared__ __attribute__((aligned(1024))) char smem[QB_LDS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
    int tm, tn;
    g2_tile((int)blockIdx.x, G.gm, G.gn, tm, tn);
    const int n0 = tn * 256, m0 = tm * 128, t0 = n0 >> 4;
    const int nb = G.nb, nks = G.k >> 4, ksb = G.k >> 5, mtiles = G.mp >> 5;
    const uint32_t lds = lds_addr(smem);

    const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc((void*)G.frag, (short)0, G.a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rS = __builtin_amdgcn_make_buffer_rsrc((void*)G.sums, (short)0, G.s_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rQ = __builtin_amdgcn_make_buffer_rsrc((void*)G.qs, (short)0, G.q_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rH = __builtin_amdgcn_make_buffer_rsrc((void*)G.hdr, (short)0, G.h_bytes, 0x00020000);
    // this wave's share of a stage: the hi and lo fragment of (m-tile wave/2, slice wave%2), the 256 B of quants and
    // headers of row tiles 2·wave, +1 (past the last: the last, never stored), the sums of m-tile wave/2, half
    // wave%2 of its rows, hi and lo. M-tiles past mp: the last, never stored.
    const int amt = min(4 * tm + (wave >> 1), mtiles - 1), aB = amt * nks * 2048;
    const int q0 = min(t0 + 2 * wave, G.ntiles - 1), q1 = min(t0 + 2 * wave + 1, G.ntiles - 1);
    const uint32_t a_v = lane * 16, q_v = lane * 4;
    // sums: lane → row 16·(wave%2) + lane/4 of the m-tile, dword lane%4 of its 16 bytes
    const uint32_t s_v = (uint32_t)((32 * amt + 16 * (wave & 1) + (lane >> 2)) * ksb * 2 + (lane & 3) * 4);
    // stage position j = 2·J + kg of super-block sb (past the last one: that again, unused)
    auto issue = [&](int sb, int j, int slot) {
        const int b = min(sb, nb - 1);
        char* st = smem + slot * QB_STAGE;
        const int J = j >> 1, kg = j & 1, kso = b * 32768 + (4 * J + 2 * (wave & 1) + kg) * 2048;
#pragma unroll
        for (int p = 0; p < 2; p++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, (lds_void*)(st + wave * 2048 + p * 1024), 16, a_v,
                                                     aB + kso + p * 1024, 0, 0);
        const int qo = b * 2048 + (J >> 1) * 1024 + (2 * (J & 1) + kg) * 256;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rQ, (lds_void*)(st + QB_A + 2 * wave * 256), 4, q_v, q0 * nb * 2048 + qo, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rQ, (lds_void*)(st + QB_A + (2 * wave + 1) * 256), 4, q_v, q1 * nb * 2048 + qo, 0, 0);
        if (j == 0) {
            char* h = smem + QB_HDR + (sb & 1) * 8192;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rH, (lds_void*)(h + 2 * wave * 256), 4, q_v, (q0 * nb + b) * 256, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rH, (lds_void*)(h + (2 * wave + 1) * 256), 4, q_v, (q1 * nb + b) * 256, 0, 0);
#pragma unroll
            for (int p = 0; p < 2; p++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rS, (lds_void*)(h + 4096 + (wave >> 1) * 1024 + p * 512 + (wave & 1) * 256), 4, s_v,
                    p * G.mp * ksb * 2 + b * 16, 0, 0);
        }
    };

    // LDS offsets: quants / header of this lane's column 64·wn + 32·c + lane%32 (tile 4·wn + 2·c + (lane%32)/16), k half
    // lane/32; A fragments and sums (lane/32: hi or lo) of m-tile 2·wm + mt
    const uint32_t h_off = (4 * wn + ((lane & 31) >> 4)) * 256 + (lane & 15) * 16, b_off = QB_A + h_off + 8 * (lane >> 5);
    const uint32_t a_off = 2 * wm * 4096 + a_v;
    const uint32_t s_off = 4096 + 2 * wm * 1024 + (lane >> 5) * 512 + (lane & 31) * 16;

    f32x16 U[2][2], P[2][2];
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int c = 0; c < 2; c++) U[mt][c] = (f32x16){};
    u32x4 hd[2], hn[2];  // headers of this super-block; of the next one
    half2_t sp[2], zp[2];
    uint32_t c64;  // 0x64006400 in a VGPR (see dq8s)
    asm("v_mov_b32 %0, 0x64006400" : "=v"(c64));
    half8_t a[2][2][2];  // [slice][m-tile][part]
    u32x2 raw[2];
    half8_t bv[2][2];  // [slice][column tile]
    auto read_a = [&](uint32_t st, int s) {
        a[s][0][0] = lds_b128h<0>(st + a_off + s * 2048);
        a[s][0][1] = lds_b128h<1024>(st + a_off + s * 2048);
        a[s][1][0] = lds_b128h<4096>(st + a_off + s * 2048);
        a[s][1][1] = lds_b128h<5120>(st + a_off + s * 2048);
    };
    auto read_raw = [&](uint32_t st) {
        raw[0] = lds_b64<0>(st + b_off);
        raw[1] = lds_b64<512>(st + b_off);
    };
    auto read_hd = [&](int b) {
        const uint32_t hs = lds + QB_HDR + (b & 1) * 8192 + h_off;
        hn[0] = lds_b128<0>(hs);
        hn[1] = lds_b128<512>(hs);
    };
    auto scales = [&](const u32x4* h, int J) {  // of sub-blocks 2J and 2J + 1 (as aeth_gemm_kq.hip)
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const uint32_t y = h[c][1], w = h[c][3];
            const uint32_t sc4 = J < 2 ? (y & 0x3F3F3F3Fu) : ((w & 0x0F0F0F0Fu) | ((y >> 2) & 0x30303030u));
            half2_t p01, p23;
            bytes_to_h2(sc4, p01, p23);
            const half2_t pr = (J & 1) ? p23 : p01;
            const half2_t k_s = {(_Float16)1.0f, (_Float16)0.0625f}, k_z = {(_Float16)-1024.0f, (_Float16)-64.0f};
            sp[c] = pr * k_s;
            zp[c] = pr * k_z;
        }
    };
    auto deq = [&](int s) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const uint32_t x8 = raw[c][0] >> 8, y8 = raw[c][1] >> 8;
            if (s == 0)
                bv[0][c] = dq8s<0x000F000Fu>(raw[c][0], raw[c][1], x8, y8, c64, __builtin_shufflevector(sp[c], sp[c], 0, 0),
                                             __builtin_shufflevector(zp[c], zp[c], 0, 0));
            else
                bv[1][c] = dq8s<0x00F000F0u>(raw[c][0], raw[c][1], x8, y8, c64, __builtin_shufflevector(sp[c], sp[c], 1, 1),
                                             __builtin_shufflevector(zp[c], zp[c], 1, 1));
        }
    };
#pragma unroll
    for (int i = 0; i < QB_NST; i++) issue(0, i, i);
    vm_wait<4 * (QB_NST - 1)>();  // the first stage, its headers and sums are here
    __builtin_amdgcn_s_barrier();
    read_raw(lds);
    read_hd(0);
    read_a(lds, 0);
    lgkm_wait<4>();
#pragma unroll
    for (int c = 0; c < 2; c++) {
        pin(raw[c]);
        pin(hn[c]);
    }
    scales(hn, 0);
    deq(0);
    int slot = 0;  // of the stage being computed
    for (int b = 0; b < nb; b++) {
#pragma unroll
        for (int c = 0; c < 2; c++) hd[c] = hn[c];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            // slice 0, dequantised before; meanwhile slice 1's fragments are read and its quants dequantised
            read_a(lds + slot * QB_STAGE, 1);
            lgkm_wait<4>();
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                pin(a[0][mt][0]);
                pin(a[0][mt][1]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
#pragma unroll
                    for (int c = 0; c < 2; c++)
                        P[mt][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][mt][p], bv[0][c],
                                                                          j == 0 && p == 0 ? (f32x16){} : P[mt][c], 0, 0, 0);
            deq(1);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            // slice 1's fragments are here: this wave is done with the slot. The next stage's loads have landed (those
            // of the QB_NST − 2 after it may be in flight); after the barrier every wave's have, and every wave is
            // done with the slot, which takes stage j + QB_NST.
            lgkm_wait<0>();
            if (qb_after(j) == 4 * QB_NST - 4) vm_wait<4 * QB_NST - 4>();
            else vm_wait<4 * QB_NST - 8>();
            __builtin_amdgcn_s_barrier();
            issue(b + (j + QB_NST) / 8, (j + QB_NST) & 7, slot);
            slot = slot + 1 == QB_NST ? 0 : slot + 1;
            read_raw(lds + slot * QB_STAGE);
            if (j == 7) read_hd(b + 1);
            read_a(lds + slot * QB_STAGE, 0);
#pragma unroll
            for (int mt = 0; mt < 2; mt++) {
                pin(a[1][mt][0]);
                pin(a[1][mt][1]);
            }
            __builtin_amdgcn_sched_barrier(0);
            auto slice1 = [&](int p) {
#pragma unroll
                for (int mt = 0; mt < 2; mt++)
#pragma unroll
                    for (int c = 0; c < 2; c++)
                        P[mt][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1][mt][p], bv[1][c], P[mt][c], 0, 0, 0);
            };
            slice1(0);
            __builtin_amdgcn_sched_barrier(0);
            lgkm_wait<4>();  // the next stage's quants: its slice 0 is dequantised under the rest
#pragma unroll
            for (int c = 0; c < 2; c++) {
                pin(raw[c]);
                if (j == 7) pin(hn[c]);
            }
            __builtin_amdgcn_sched_barrier(0);
            slice1(1);
            if (j & 1) scales(j == 7 ? hn : hd, ((j + 1) & 7) >> 1);
            deq(0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (j == 7) {  // U += d·P − 32·dmin·Σ_s m_s·S_s (S carries 2^-(e+5))
                half8_t sv[2];
                const uint32_t ss = lds + QB_HDR + (b & 1) * 8192 + s_off;
                sv[0] = lds_b128h<0>(ss);
                sv[1] = lds_b128h<1024>(ss);
                lgkm_wait<0>();
                pin(sv[0]);
                pin(sv[1]);
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const float d = aeth_decode_d(hd[c][0]), ndm = -32.0f * aeth_decode_d(hd[c][0] >> 16);
                    const uint32_t z = hd[c][2], w = hd[c][3];
                    half2_t m01, m23, m45, m67;
                    bytes_to_h2(z & 0x3F3F3F3Fu, m01, m23);
                    bytes_to_h2(((w >> 4) & 0x0F0F0F0Fu) | ((z >> 2) & 0x30303030u), m45, m67);
                    const half8_t mv = {m01[0], m01[1], m23[0], m23[1], m45[0], m45[1], m67[0], m67[1]};
#pragma unroll
                    for (int mt = 0; mt < 2; mt++) {
                        const f32x16 q = __builtin_amdgcn_mfma_f32_32x32x16_f16(sv[mt], mv, (f32x16){}, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 16; r++) U[mt][c][r] = fmaf(d, P[mt][c][r], fmaf(ndm, q[r], U[mt][c][r]));
                    }
                }
            }
        }
    }
    vm_wait<0>();  // the tail's loads have landed: the LDS outlives them
    lgkm_wait<0>();  // and its reads: their registers are free

#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int col = n0 + 64 * wn + 32 * c + (lane & 31);
            int rows[16];
#pragma unroll
            for (int r = 0; r < 16; r++)
                rows[r] = min(m0 + 64 * wm + 32 * mt + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), G.mp - 1);
            G2Epi E;
            g2_epi_load(E, G.escale, G.C, G.ldc, G.m, G.n, rows, col, G.accumulate);
            // rows past mp share the last one's scale and are past m: not stored
            if (m0 + 64 * wm + 32 * mt >= G.mp) continue;
            if (G.swiglu) {
#pragma unroll
                for (int r = 0; r < 16; r += 2)
                    g2_store_swiglu(E, r, G.C, G.ldc, G.m, G.n, rows[r], col, U[mt][c][r], U[mt][c][r + 1]);
            } else {
#pragma unroll
                for (int r = 0; r < 16; r++) g2_store(E, r, G.C, G.ldc, G.m, G.n, rows[r], col, U[mt][c][r], G.accumulate);
            }
        }
}

// A round of these workgroups (one a CU) takes 2.9 .. 3.1 times as long as a round of aeth_gemm_kq.hip's, which
// holds a quarter of the outputs; a last round costs as much as a full one. So from three rounds there for each one here:
// measured there / here, k = 4096, with prep: 512 × 12288 126.6 / 121.9 µs, × 14336 157.9 / 126.4, × 28672 283 /
// 235, 256 × 28672 157 / 126, 100 × 49152 127 / 123; on the other side 512 × 8192 89 / 108, × 20480 200 / 224, 100 ×
// 32000 86 / 104, 1024 × 10240 201 / 223 (512 × 10240, 2.5 rounds: 116 / 114).
bool aeth_q4k_big_ok(int64_t m, int64_t n) {
    const int64_t cus = aeth_num_cus(), T = aeth_cdiv(m, 128) * aeth_cdiv(n, 256);
    return aeth_cdiv(m, 64) * aeth_cdiv(n, 128) >= 3 * cus * aeth_cdiv(T, cus);
}

int aeth_gemm_q4k_big_launch(KqArgs G, hipStream_t s) {
    G.gm = (int)aeth_cdiv(G.m, 128);
    G.gn = (int)aeth_cdiv(G.n, 256);
    hipLaunchKernelGGL(k_gemm_q4k_big, dim3((unsigned)(G.gm * G.gn)), dim3(512), 0, s, G);
    AETH_LAUNCH_CHECK();
    return AETH_OK;
}
