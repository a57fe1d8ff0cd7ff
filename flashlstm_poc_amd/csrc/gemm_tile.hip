// The fp16 MFMA GEMMs of gemm.hip for problems that do not fill the chip with 256 x 256 tiles: one workgroup of four
// waves per tile of 64 x 64 or 128 x 128, several workgroups per CU.
//
// A 256 x 256 tile of gemm.hip takes its CU 2 us per 64-wide slab of K whether or not the other CUs have work, so a
// product of few tiles runs on few CUs for a long time: 2048 x 1024 outputs over K = 4096 are 32 tiles, 64 slabs,
// 140 us at an eighth of the chip.  Here the same product is 512 tiles of 64 x 64 (or 128 of 128 x 128).  What bounds
// these kernels is the latency of a slab (about a microsecond from memory), covered by ST slabs in LDS -- ST - 1
// requested ahead -- and by the other workgroups of the CU; the MFMA rate of a CU is reached by the 128 x 128 tile
// only.  launch_gemm_nt / launch_gemm_tn take whichever size a cost model prefers (gemm_tile_choice).
//
// Both kernels: slabs of 64 k go from global memory straight into LDS (1 KiB per copy instruction), one barrier per
// slab: wait for this wave's copies of slab k, barrier (everybody's copies have landed and everybody is done with slab
// k - 1), request slab k + ST - 1 into the buffer of slab k - 1, multiply slab k.  The finished tile is turned through
// LDS so that rows leave in whole lines whatever their pitch.
#include "gemm_tile_device.h"

namespace flstm_hip {
namespace {

// Workgroup -> tile.  Workgroups are dealt round-robin to the 8 XCDs; each XCD gets a contiguous run of tiles, walked
// in bands of four tile rows, so that the workgroups that share an L2 share operand panels.
__device__ __forceinline__ void tile_of(int lin, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int total = tiles_m * tiles_n;
    // (XCD x has the workgroups x, x + 8, ...: the first total % 8 of them one more than the others)
    const int xcd = lin % 8, rem = total % 8;
    const int t = xcd * (total / 8) + (xcd < rem ? xcd : rem) + lin / 8;
    const int band = t / (4 * tiles_n), r = t % (4 * tiles_n);
    const int rows = tiles_m - band * 4 < 4 ? tiles_m - band * 4 : 4;
    tm = band * 4 + r % rows;
    tn = r / rows;
}

// The tile, row by row, from LDS (`stage`: [TM][TN] of T with rows of TN + pad elements) to global memory: `cols` valid
// columns of `rows` valid rows, 16 bytes per lane where the rows allow it.
template <int TM, int TN, int PITCH, typename T>
__device__ __forceinline__ void store_rows(const T* stage, T* dst, size_t ldc, int rows, int cols, int tid) {
    constexpr int V = 16 / sizeof(T);
    const bool vec = (ldc % V == 0) && (reinterpret_cast<uintptr_t>(dst) % 16 == 0) && cols % V == 0;
    if (vec) {
        constexpr int PER_ROW = TN / V;
#pragma unroll 4
        for (int i = tid; i < TM * PER_ROW; i += kTileThreads) {
            const int r = i / PER_ROW, c = (i % PER_ROW) * V;
            if (r < rows && c < cols)
                *reinterpret_cast<uint4*>(dst + size_t(r) * ldc + c) = *reinterpret_cast<const uint4*>(stage + r * PITCH + c);
        }
    } else {
        for (int i = tid; i < TM * TN; i += kTileThreads) {
            const int r = i / TN, c = i % TN;
            if (r < rows && c < cols) dst[size_t(r) * ldc + c] = stage[r * PITCH + c];
        }
    }
}

// (stage16's counterpart for fp32 outputs)
template <int MI, int PITCH>
__device__ __forceinline__ void stage32(float* stage, const floatx16 (&acc)[MI][MI], float alpha, const float* bias, int n0,
                                        int N, int row, int col, int lane) {
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = col + j * 32 + 8 * q + 4 * (lane / 32);
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                floatx4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = __builtin_fmaf(alpha, acc[i][j][4 * q + e], (bias && n0 + c + e < N) ? bias[n0 + c + e] : 0.f);
                *reinterpret_cast<floatx4*>(stage + (row + i * 32 + lane % 32) * PITCH + c) = v;
            }
        }
}

// Rows of the staged tile are TN + 4 (fp32) / TN + 8 (fp16) elements: the 32 rows a store instruction touches then start
// 4 banks apart.
template <int TM, int ST>
constexpr size_t tile_lds_bytes() {
    constexpr size_t slabs = size_t(ST) * 2 * TM * BK * 2, stage = size_t(TM) * (TM + 4) * 4;
    return slabs > stage ? slabs : stage;
}

// Tile `lin` of C[M][N] = alpha * A[M][K] * B[N][K]^T (+ bias), see nt_tile_product.
template <int TM, int ST>
__device__ __forceinline__ void nt_tile(const GemmNT& g, char* lds, int lin, int tiles_m, int tiles_n) {
    constexpr int MI = TM / 64;                    // 32 x 32 MFMA tiles per wave and direction
    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    if (g.stamp && lin == 0 && tid == 0) *g.stamp = wall_clock64();
    int tm, tn;
    tile_of(lin, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * TM, n0 = tn * TM, nk = g.K / BK;

    const int wm = wave / 2, wn = wave % 2;
    floatx16 acc[MI][MI];
    nt_tile_product<TM, ST>(acc, lds, g.A + size_t(m0) * g.lda, g.lda, g.M - m0, g.B + size_t(n0) * g.ldb, g.ldb, g.N - n0, nk, wave, lane);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier_here();   // the slabs are done with: their LDS takes the tile
    const int rows = min(TM, g.M - m0), cols = min(TM, g.N - n0);
    if (g.C16) {
        constexpr int PITCH = TM + 8;
        half_t* stage = reinterpret_cast<half_t*>(lds);
        stage16<MI, PITCH>(stage, acc, g.alpha, g.bias, n0, g.N, wm * 32 * MI, wn * 32 * MI, lane);
        __syncthreads();
        store_rows<TM, TM, PITCH>(stage, g.C16 + size_t(m0) * g.ldc + n0, g.ldc, rows, cols, tid);
    } else {
        constexpr int PITCH = TM + 4;
        float* stage = reinterpret_cast<float*>(lds);
        stage32<MI, PITCH>(stage, acc, g.alpha, g.bias, n0, g.N, wm * 32 * MI, wn * 32 * MI, lane);
        __syncthreads();
        store_rows<TM, TM, PITCH>(stage, g.C32 + size_t(m0) * g.ldc + n0, g.ldc, rows, cols, tid);
    }
}

typedef short short4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v lds_short4;

// Tile `lin` of C[M][N] = alpha * sum_k A[k][m] * B[k][n] over K split `split`.  Slabs sit in LDS as they sit in memory, 64 k-rows of TM
// columns per operand; fragments are read with the transposing LDS load (see gemm_tn_stream).  The four k-rows that 32
// lanes read together are kept in different quarters of a 256-byte bank row: the 64-byte chunk c of k-row r sits at
// c ^ (r % 4) where a row is 256 bytes, at c ^ (r / 2 % 2) where it is 128 (two rows share a bank row).
template <int TM, int ST>
__device__ __forceinline__ void tn_tile(const GemmNT& g, char* lds, int lin, int split, int tiles_m, int tiles_n, int slabs_per_split) {
    constexpr int MI = TM / 64;
    constexpr int ROWB = TM * 2;                   // bytes of an LDS row
    constexpr int OPERAND = BK * ROWB, SLAB = 2 * OPERAND;
    constexpr int CP = TM / 32;                    // copies per wave, operand and slab
    constexpr int RPC = 1024 / ROWB;               // k-rows per copy
    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    if (g.stamp && lin == 0 && tid == 0) *g.stamp = wall_clock64();
    int tm, tn;
    tile_of(lin, tiles_m, tiles_n, tm, tn);
    const int tiles_n1 = g.B2 ? (g.N1 + TM - 1) / TM : (1 << 30);
    const bool side = tn >= tiles_n1;              // columns [N1, N) of C: the second B operand
    const int m0 = tm * TM, n0 = (tn - (side ? tiles_n1 : 0)) * TM;
    const half_t* B = side ? g.B2 : g.B;
    const size_t ldb = side ? g.ldb2 : g.ldb;
    const int nside = g.B2 ? (side ? g.N - g.N1 : g.N1) : g.N;
    const int slab0 = split * slabs_per_split;
    const int nk = min((g.K + BK - 1) / BK - slab0, slabs_per_split);
    if (nk <= 0) return;

    // swizzle of k-row r (the same for r and r + RPC: both are multiples of 4 apart)
    auto sw = [](int r) { return TM == 128 ? r % 4 : (r / 2) % 2; };
    const int lr = lane / (64 / RPC), lp = lane % (64 / RPC);           // k-row inside a copy, 16-byte position
    const int lc = (((lp / 4) ^ sw(lr)) * 4 + lp % 4) * 8;               // column (halfs) fetched by this lane
    const unsigned col_a = unsigned(min(m0 + lc, g.M - 8)) * 2u, col_b = unsigned(min(n0 + lc, nside - 8)) * 2u;
    const unsigned pa = unsigned(g.lda * 2), pb = unsigned(ldb * 2);
    const char* src_a = reinterpret_cast<const char*>(g.A) + size_t(slab0) * BK * pa;
    const char* src_b = reinterpret_cast<const char*>(B) + size_t(slab0) * BK * pb;
    auto rows_of = [&](int k) { return min(BK, g.K - (slab0 + k) * BK); };   // valid k-rows of a slab
    auto request = [&](int k) {
        char* dst = lds + (k % ST) * SLAB + wave * CP * 1024;
        const char* a = src_a + size_t(k) * BK * pa;
        const char* b = src_b + size_t(k) * BK * pb;
        const int last = rows_of(k) - 1;
#pragma unroll
        for (int i = 0; i < CP; ++i) {
            const unsigned r = unsigned(min((wave * CP + i) * RPC + lr, last));
            copy_1k(a, r * pa + col_a, dst + i * 1024);
            copy_1k(b, r * pb + col_b, dst + OPERAND + i * 1024);
        }
    };
    // k-rows past K of the slab, as far as this wave copied them, are cleared (its copies have landed)
    auto clear_tail = [&](int k) {
        const int rows = rows_of(k);
        if (rows >= BK) return;
        char* st = lds + (k % ST) * SLAB + wave * CP * 1024;
#pragma unroll
        for (int i = 0; i < CP; ++i)
            if ((wave * CP + i) * RPC + lr >= rows) {
                *reinterpret_cast<uint4*>(st + i * 1024 + lane * 16) = uint4{0u, 0u, 0u, 0u};
                *reinterpret_cast<uint4*>(st + OPERAND + i * 1024 + lane * 16) = uint4{0u, 0u, 0u, 0u};
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };

    const int wm = wave / 2, wn = wave % 2;
    const int gq = lane / 16, jq = lane % 16;
    const int frag_lane = (8 * (gq / 2) + jq / 4) * ROWB + 32 * (gq % 2) + 8 * (jq % 4);
    int a_frag[MI], b_frag[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        a_frag[i] = frag_lane + ((wm * MI + i) ^ sw(jq / 4)) * 64;
        b_frag[i] = OPERAND + frag_lane + ((wn * MI + i) ^ sw(jq / 4)) * 64;
    }
    auto read_frag = [&](const char* at) {
        union { short4v s[2]; half8 h; } u;
        u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at));
        u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(at + 4 * ROWB));
        return u.h;
    };

    floatx16 acc[MI][MI];
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
        if (k + ST - 2 < nk) wait_copies<(ST - 2) * 2 * CP>();
        else wait_copies<0>();
        clear_tail(k);
        barrier_here();
        if (k + ST - 1 < nk) request(k + ST - 1);
        const char* st = lds + (k % ST) * SLAB;
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk) {
            half8 af[MI], bf[MI];
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                af[i] = read_frag(st + a_frag[i] + kk * 16 * ROWB);
                bf[i] = read_frag(st + b_frag[i] + kk * 16 * ROWB);
            }
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < MI; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[j], af[i], acc[i][j], 0, 0, 0);
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier_here();
    constexpr int PITCH = TM + 4;
    float* stage = reinterpret_cast<float*>(lds);
    stage32<MI, PITCH>(stage, acc, g.alpha, nullptr, 0, 0, wm * 32 * MI, wn * 32 * MI, lane);
    __syncthreads();
    float* dst = g.C32 + size_t(split) * g.split_stride + size_t(m0) * g.ldc + n0 + (side ? g.N1 : 0);
    store_rows<TM, TM, PITCH>(stage, dst, g.ldc, min(TM, g.M - m0), min(TM, nside - n0), tid);
}

template <int TM, int ST>
__global__ __launch_bounds__(kTileThreads) void gemm_nt_tile(GemmNT g, int tiles_m, int tiles_n) {
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    nt_tile<TM, ST>(g, lds, blockIdx.x, tiles_m, tiles_n);
}

template <int TM, int ST>
__global__ __launch_bounds__(kTileThreads) void gemm_tn_tile(GemmNT g, int tiles_m, int tiles_n, int slabs_per_split) {
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    tn_tile<TM, ST>(g, lds, blockIdx.x, blockIdx.y, tiles_m, tiles_n, slabs_per_split);
}

// A TN and an NT product of the same pass in one launch (launch_gemm_tn_and_nt): workgroups [0, tn_first) and those from
// tn_first + tn_m * tn_n * splits on have the NT product's tiles, those between the TN product's.  tn_first is 0 or all of the NT
// product's: the product whose tiles take longer comes first, so that the other's fill up its end (297 rows x 1920 units: 120 slabs
// an NT tile, 5 a TN one).
struct PairTiles {
    int tn_m, tn_n, splits, slabs_per_split, nt_m, nt_n, tn_first;
};
template <int TN, int SN, int TT, int SS>
__global__ __launch_bounds__(kTileThreads) void gemm_pair_tile(GemmNT tn, GemmNT nt, PairTiles t) {
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int lin = int(blockIdx.x) - t.tn_first, per_split = t.tn_m * t.tn_n, all = per_split * t.splits;
    if (lin >= 0 && lin < all) tn_tile<TN, SN>(tn, lds, lin % per_split, lin / per_split, t.tn_m, t.tn_n, t.slabs_per_split);
    else nt_tile<TT, SS>(nt, lds, t.tn_first ? int(blockIdx.x) : lin - all, t.nt_m, t.nt_n);
}

template <typename K>
hipError_t with_lds(K kernel, size_t bytes) {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes));
}

template <int TM, int ST>
hipError_t run_nt(const GemmNT& g, hipStream_t s) {
    const int tm = (g.M + TM - 1) / TM, tn = (g.N + TM - 1) / TM;
    hipError_t e = with_lds(gemm_nt_tile<TM, ST>, tile_lds_bytes<TM, ST>());
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((gemm_nt_tile<TM, ST>), dim3(unsigned(tm) * unsigned(tn)), dim3(kTileThreads), (tile_lds_bytes<TM, ST>()), s,
                       g, tm, tn);
    return hipGetLastError();
}

template <int TM, int ST>
hipError_t run_tn(const GemmNT& g, int splits, int slabs_per_split, hipStream_t s) {
    const int tm = (g.M + TM - 1) / TM;
    const int tn = g.B2 ? (g.N1 + TM - 1) / TM + (g.N - g.N1 + TM - 1) / TM : (g.N + TM - 1) / TM;
    hipError_t e = with_lds(gemm_tn_tile<TM, ST>, tile_lds_bytes<TM, ST>());
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((gemm_tn_tile<TM, ST>), dim3(unsigned(tm) * unsigned(tn), unsigned(splits)), dim3(kTileThreads),
                       (tile_lds_bytes<TM, ST>()), s, g, tm, tn, slabs_per_split);
    return hipGetLastError();
}

template <int TN, int SN, int TT, int SS>
hipError_t run_pair(const GemmNT& tn, const GemmNT& nt, int splits, int slabs_per_split, hipStream_t s) {
    PairTiles t;
    t.tn_m = (tn.M + TN - 1) / TN;
    t.tn_n = tn.B2 ? (tn.N1 + TN - 1) / TN + (tn.N - tn.N1 + TN - 1) / TN : (tn.N + TN - 1) / TN;
    t.splits = splits;
    t.slabs_per_split = slabs_per_split;
    t.nt_m = (nt.M + TT - 1) / TT;
    t.nt_n = (nt.N + TT - 1) / TT;
    t.tn_first = (nt.K / BK) * TT > slabs_per_split * TN ? t.nt_m * t.nt_n : 0;   // (a slab of a 128 x 128 tile takes twice as long)
    constexpr size_t lds = tile_lds_bytes<TN, SN>() > tile_lds_bytes<TT, SS>() ? tile_lds_bytes<TN, SN>() : tile_lds_bytes<TT, SS>();
    hipError_t e = with_lds(gemm_pair_tile<TN, SN, TT, SS>, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((gemm_pair_tile<TN, SN, TT, SS>), dim3(unsigned(t.tn_m) * unsigned(t.tn_n) * unsigned(splits) + unsigned(t.nt_m) * unsigned(t.nt_n)),
                       dim3(kTileThreads), lds, s, tn, nt, t);
    return hipGetLastError();
}

}  // namespace

// Estimated microseconds of a product on 256 CUs.  A tile of T x T takes a CU `slab` us per 64-wide slab when the CU is
// shared by as many workgroups as fit and `alone` us when it has one, plus `tail` us for its output; tiles are dealt
// evenly.  The constants are fits to timings of 40 shapes (products of 0.03 to 1100 GFLOP) on random operands; what
// matters of them is where the lines cross: 128 x 128 from about 256 tiles of that size on, 256 x 256 once those fill
// the chip for a round.  Measured on both sides, us, 64 / 128 / 256: NT 2048 x 4096 over 1024: 32 / 29 / 38; 2048 x
// 16384 over 1024: 124 / 91 / 71; 2048 x 1024 over 4096: 31 / 50 / 94; 14000 x 1152 over 128: 19 / 17 / 83; 12288 x
// 512 over 6144: 126 / 98 / 181.  TN 1024 x 384 over 512: 4.2 / 5.6 / 29; 4096 x 2048 over 2000: 60 / 42 / 44; 6144 x
// 2048 over 12288: 530 / 324 / 308.
static double tiles_cost(double tiles, double slabs, double fixed, double alone, double slab, double tail) {
    const double load = tiles / 256.0, one = slabs * alone + tail, many = load * (slabs * slab + tail);
    return fixed + (one > many ? one : many);
}
static double big_cost(long blocks_of_32, double slabs, bool ragged) {
    const double rounds = double((blocks_of_32 + 7) / 8);
    return 8.0 + rounds * (slabs * 2.0 + (ragged ? 15.0 : 2.0));   // (ragged tiles leave element by element there)
}
static double tiles_of(int M, int N, int T) { return double((M + T - 1) / T) * double((N + T - 1) / T); }

static double nt_cost(int M, int N, int K, int tile) {
    const double nk = double(K) / BK;
    if (tile == 64) return tiles_cost(tiles_of(M, N, 64), nk, 2.5, 0.27, 0.22, 0.5);
    if (tile == 128) return tiles_cost(tiles_of(M, N, 128), nk, 3.0, 0.78, 0.62, 1.6);
    return big_cost(gemm_blocks_of_32(M, N, 0), nk, M % 256 != 0 || N % 256 != 0);
}
int gemm_nt_tile_size(int M, int N, int K) {
    const double c64 = nt_cost(M, N, K, 64), c128 = nt_cost(M, N, K, 128), c256 = nt_cost(M, N, K, 256);
    return c64 <= c128 && c64 <= c256 ? 64 : (c128 <= c256 ? 128 : 256);
}
double gemm_nt_cost(int M, int N, int K) { return nt_cost(M, N, K, gemm_nt_tile_size(M, N, K)); }

static double tn_cost(int M, int N1, int N2, int K, int splits, int tile) {
    const double nk = double(((K + BK - 1) / BK + splits - 1) / splits);
    // partial tiles are written and read back once at about 3 TB/s
    const double reduce = 2.5 + 8.0 * splits * double(M) * double(N1 + N2) / 3e6;
    const double tiles = (tiles_of(M, N1, tile) + tiles_of(M, N2, tile)) * splits;
    if (tile == 64) return reduce + tiles_cost(tiles, nk, 2.5, 0.27, 0.25, 0.5);
    if (tile == 128) return reduce + tiles_cost(tiles, nk, 3.0, 0.56, 0.56, 1.6);
    return reduce + big_cost(gemm_blocks_of_32(M, N1, N2) * splits, nk, M % 256 != 0 || N1 % 256 != 0 || N2 % 256 != 0);
}
int gemm_tn_tile_size(int M, int N1, int N2, int K, int splits) {
    int best = 256;
    for (int tile : {128, 64})
        if (tn_cost(M, N1, N2, K, splits, tile) < tn_cost(M, N1, N2, K, splits, best)) best = tile;
    return best;
}
int gemm_tn_plan_splits(int M, int N1, int N2, int K, int max_splits) {
    // the large tiles with the split count their own schedule prefers, against the small ones at every count
    int best = gemm_tn_auto_splits(M, N1, N2, K, max_splits);
    double best_cost = tn_cost(M, N1, N2, K, best, 256);
    const int nslab = (K + BK - 1) / BK;
    for (int sp = 1; sp <= max_splits && sp <= nslab; ++sp) {
        if (gemm_effective_splits(K, sp) != sp) continue;
        for (int tile : {128, 64}) {
            const double c = tn_cost(M, N1, N2, K, sp, tile);
            if (c < best_cost) { best_cost = c; best = sp; }
        }
    }
    return best;
}

hipError_t launch_gemm_nt_tile(const GemmNT& g, int tile, hipStream_t s) {
    // four slabs in LDS where few workgroups share a CU, two -- twice the workgroups -- where many could
    if (tile == 64) return tiles_of(g.M, g.N, 64) <= 512 ? run_nt<64, 4>(g, s) : run_nt<64, 2>(g, s);
    return run_nt<128, 2>(g, s);
}
hipError_t launch_gemm_tn_tile(const GemmNT& g, int tile, int splits, int slabs_per_split, hipStream_t s) {
    const double tiles = (tiles_of(g.M, g.B2 ? g.N1 : g.N, 64) + (g.B2 ? tiles_of(g.M, g.N - g.N1, 64) : 0.0)) * splits;
    if (tile == 64) return tiles <= 512 ? run_tn<64, 4>(g, splits, slabs_per_split, s) : run_tn<64, 2>(g, splits, slabs_per_split, s);
    return run_tn<128, 2>(g, splits, slabs_per_split, s);
}

bool gemm_pair_possible(const GemmNT& tn, int tn_tile, int splits, const GemmNT& nt, int nt_tile) {
    const double tn_tiles = (tiles_of(tn.M, tn.B2 ? tn.N1 : tn.N, 64) + (tn.B2 ? tiles_of(tn.M, tn.N - tn.N1, 64) : 0.0)) * splits;
    return (tn_tile == 128 || (tn_tile == 64 && tn_tiles <= 512)) && (nt_tile == 128 || (nt_tile == 64 && tiles_of(nt.M, nt.N, 64) <= 512));
}
hipError_t launch_gemm_pair_tile(const GemmNT& tn, int tn_tile, int splits, int slabs_per_split, const GemmNT& nt, int nt_tile,
                                 hipStream_t s) {
    if (tn_tile == 64)
        return nt_tile == 64 ? run_pair<64, 4, 64, 4>(tn, nt, splits, slabs_per_split, s) : run_pair<64, 4, 128, 2>(tn, nt, splits, slabs_per_split, s);
    return nt_tile == 64 ? run_pair<128, 2, 64, 4>(tn, nt, splits, slabs_per_split, s) : run_pair<128, 2, 128, 2>(tn, nt, splits, slabs_per_split, s);
}

}  // namespace flstm_hip
