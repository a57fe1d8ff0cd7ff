// Device side of the small-tile GEMMs that more than one translation unit runs (gemm_tile.hip, recurrent.hip).
#pragma once
#include "gemm.h"

namespace flstm_hip {
namespace {

constexpr int BK = 64;
constexpr int kTileThreads = 256;

typedef __attribute__((address_space(3))) char lds_char;

// 1 KiB from (base + lane_off) into LDS at lds_block, lane l to byte 16 * l.  Issued by hand, so that the compiler does
// not wait for it in front of LDS reads of other buffers; the kernels' own waits and barriers order copies and reads.
__device__ __forceinline__ void copy_1k(const char* base, unsigned lane_off, char* lds_block) {
    const unsigned m = unsigned(reinterpret_cast<unsigned long>((lds_char*)(lds_block)));
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :: "v"(lane_off), "s"(base), "s"(m) : "m0", "memory");
}
template <int N>
__device__ __forceinline__ void wait_copies() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void barrier_here() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// fma in fp32, then one rounding to fp16 (as in gemm.hip: the same bits whichever kernel forms an element)
__device__ __forceinline__ half_t round16(float alpha, float acc, float bias) {
    float v = __builtin_fmaf(alpha, acc, bias);
    asm volatile("" : "+v"(v));
    return (half_t)v;
}

// Accumulators of a wave -> the staged tile.  Register r of MFMA tile (i, j) holds row i*32 + lane%32, column
// j*32 + 8*(r/4) + 4*(lane/32) + r%4 of the wave's part (operands swapped, D = B * A^T).
template <int MI, int PITCH>
__device__ __forceinline__ void stage16(half_t* stage, const floatx16 (&acc)[MI][MI], float alpha, const float* bias, int n0,
                                        int N, int row, int col, int lane) {
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = col + j * 32 + 8 * q + 4 * (lane / 32);
            float b[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) b[e] = (bias && n0 + c + e < N) ? bias[n0 + c + e] : 0.f;
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                half4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = round16(alpha, acc[i][j][4 * q + e], b[e]);
                *reinterpret_cast<half4*>(stage + (row + i * 32 + lane % 32) * PITCH + c) = v;
            }
        }
}
// acc = `rows` (at most TM) rows of A times as many of B, both from their first row and K-contiguous, over nk slabs of 64: the
// product of a tile, by four waves.  Slabs sit in LDS (ST of them, tile_lds_bytes), rows of 128 bytes, 16-byte chunk c of row r at
// c ^ (r/2) % 8 (as in gemm_nt_stream).  Rows past the operand's are fetched from its last one.
// ALONE: the workgroup has its CU to itself, so nothing else covers the way of its fragments from LDS; all of a slab's are read
// ahead of its MFMAs (registers allow it).
template <int TM, int ST, bool ALONE = false>
__device__ __forceinline__ void nt_tile_product(floatx16 (&acc)[TM / 64][TM / 64], char* lds, const half_t* A, size_t lda, int rows,
                                                const half_t* B, size_t ldb, int cols, int nk, int wave, int lane) {
    constexpr int MI = TM / 64;                    // 32 x 32 MFMA tiles per wave and direction
    constexpr int OPERAND = TM * BK * 2, SLAB = 2 * OPERAND;
    constexpr int CP = TM / 32;                    // copies per wave, operand and slab
    // copy i of this wave fills rows 8 * (wave * CP + i) .. +7: lane l lands at row l / 8, chunk position l % 8
    unsigned off_a[CP], off_b[CP];
#pragma unroll
    for (int i = 0; i < CP; ++i) {
        const int r = 8 * (wave * CP + i) + lane / 8;
        const unsigned chunk = unsigned((lane % 8) ^ ((r >> 1) & 7)) * 16u;
        off_a[i] = unsigned(min(r, rows - 1)) * unsigned(lda * 2) + chunk;
        off_b[i] = unsigned(min(r, cols - 1)) * unsigned(ldb * 2) + chunk;
    }
    const char* src_a = reinterpret_cast<const char*>(A);
    const char* src_b = reinterpret_cast<const char*>(B);
    auto request = [&](int k) {
        char* dst = lds + (k % ST) * SLAB + wave * CP * 1024;
#pragma unroll
        for (int i = 0; i < CP; ++i) {
            copy_1k(src_a + size_t(k) * (BK * 2), off_a[i], dst + i * 1024);
            copy_1k(src_b + size_t(k) * (BK * 2), off_b[i], dst + OPERAND + i * 1024);
        }
    };

    const int wm = wave / 2, wn = wave % 2;
    const int a_frag = (wm * 32 * MI + lane % 32) * (BK * 2), b_frag = OPERAND + (wn * 32 * MI + lane % 32) * (BK * 2);
    int pos[BK / 16];
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) pos[kk] = ((2 * kk + lane / 32) ^ ((lane % 32) >> 1 & 7)) * 16;

#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

#pragma unroll
    for (int k = 0; k < ST - 1; ++k)
        if (k < nk) request(k);
    for (int k = 0; k < nk; ++k) {
        // (near the end fewer slabs are in flight than the count allows for: everything is awaited)
        if (k + ST - 2 < nk) wait_copies<(ST - 2) * 2 * CP>();
        else wait_copies<0>();
        barrier_here();
        if (k + ST - 1 < nk) request(k + ST - 1);
        const char* st = lds + (k % ST) * SLAB;
        constexpr int AHEAD = ALONE ? BK / 16 : 1;   // k-steps whose fragments are read before the first is multiplied
#pragma unroll
        for (int k0 = 0; k0 < BK / 16; k0 += AHEAD) {
            half8 af[AHEAD][MI], bf[AHEAD][MI];
#pragma unroll
            for (int a = 0; a < AHEAD; ++a)
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    af[a][i] = *reinterpret_cast<const half8*>(st + a_frag + i * 32 * BK * 2 + pos[k0 + a]);
                    bf[a][i] = *reinterpret_cast<const half8*>(st + b_frag + i * 32 * BK * 2 + pos[k0 + a]);
                }
            if constexpr (ALONE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int a = 0; a < AHEAD; ++a)
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < MI; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[a][j], af[a][i], acc[i][j], 0, 0, 0);
        }
    }
}

}  // namespace
}  // namespace flstm_hip
