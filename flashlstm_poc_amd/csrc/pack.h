// Layout kernels around the GEMMs and the recurrence: weight packing, dtype conversion with
// padding, transposes, and the reductions that turn scaled/padded internals into caller tensors.
#pragma once
#include "common.h"

namespace flstm_hip {

// Packed gate order of the gate arrays (x-projection / gate cache, dG) and of everything indexed like them (rows
// of the packed W_ih, bias, contraction index of the backward products): the four gates of a hidden unit are
// neighbours, q = 4 * j + gate.   PyTorch row of (gate, j) is gate*H + j.
struct Dims {
    int B, I, H;     // caller sizes
    int Ip, Hp;      // I rounded up to 64, H to 32 (above 2048: to 64)
};

// Replaces src/kernels.cu:57-84 (pack_weights_kernel) and :45-55 (combine_bias_kernel): fp32
// PyTorch-layout weights -> the fp16 operand layouts of the kernels in this library.
struct FragLayout {   // where a recurrence kernel expects its weight fragments: RecLayout's description of them
    half8* out = nullptr;   // (null: not wanted)
    int ks = 0, nt = 0, rot_div = 0, nw = 0, unit_major = 0, wide = 0, kq = 0, split = 0;
    size_t fragments = 0;   // of 64 lanes
};
// Forward: the one-way kernels' and those of the kernel for short contractions, for few rows, or with slices of 32 units
// (RecLayout::split, few, broad); backward the one-way kernels' (which those for few rows use as well), with slices of 32 units, and those of
// the recurrence that splits its product two ways.
enum Frag : int { kFragFwd, kFragFwdSplit, kFragBwd, kFragBwdBroad, kFragBwdTwoD, kFragKinds };
// W_ih twice (as it is for the projection, transposed for dX) and W_hh as every kind of fragments asked for; one launch.
hipError_t pack_weights(const Dims& d, const float* w_ih, const float* w_hh, half_t* wih_p /*[4Hp][Ip]*/,
                        half_t* wih_t /*[Ip][4Hp]*/, const FragLayout (&frag)[kFragKinds], hipStream_t s);
// Forward fragments of slices of 32 units, up to 1024 units: those of columns 32 * gate + unit (gate_major, the one-way kernel's) from those of
// columns 4 * unit + gate, or the other way round.
hipError_t reorder_fragments(const half8* in, half8* out, size_t fragments, bool gate_major, hipStream_t s);
hipError_t pack_bias(const Dims& d, const float* b_ih, const float* b_hh, float* bias_p, hipStream_t s);

// dst[r][c] (pitch ldc) = sum over z < splits of partial[z * per + r * cols + c]: split-K partials of a plain GEMM.
hipError_t reduce_partials(const float* partial, int splits, size_t per, int rows, int cols, size_t ldc, float* dst,
                           hipStream_t s);

// *out += a position-weighted 64-bit sum over the 16-bit units of a device buffer (`salt` tells buffers apart when
// several are folded into one sum); null or empty buffers add nothing.  Evidence that device tensors still hold what
// an earlier call saw.
hipError_t checksum_add(const void* p, size_t bytes, u64 salt, u64* out, hipStream_t s);

hipError_t fill_zero(void* p, size_t bytes, hipStream_t s);

// The largest |value| of n elements (NaN if there is one), left in pinned host memory; `partial`: kAbsmaxBlocks words of
// device memory.
constexpr int kAbsmaxBlocks = 256;
hipError_t absmax(const void* t, int f32, size_t n, unsigned* partial, float* host_out, hipStream_t s);

// The layout operations around the GEMMs and the recurrence, up to kMaxOps of them in ONE launch.  A pass starts with
// half a dozen of them (state rows, rings, counters, operand conversion) and ends with as many (outputs, final states,
// gradient reductions); each is a few microseconds of kernel plus a launch of its own when issued one by one.
constexpr int kMaxOps = 12;
struct LayoutOp {
    enum Kind : int { kFill = 1, kToHalf, kToFloat, kUnpad, kToExchange, kReduceDw, kReduceDb };
    int kind = 0;
    int in_f32 = 0, out_f32 = 0, vec = 1;   // vec: elements per work item (8 or 4 where alignment allows, else 1; kUnpad: 16 bytes of output then)
    void* dst = nullptr;
    void* dst2 = nullptr;
    const void* src = nullptr;              // null reads as zeros (kToHalf, kToFloat, kToExchange)
    size_t n = 0;                           // work items
    size_t rows = 0, ld_in = 0, ld_out = 1; // elements
    size_t rows_per_block = 0, block_stride = 0;
    int cols = 0;
    unsigned word = 0;                      // kFill
    float scale = 1.f;
    int splits = 0, H = 0, accumulate = 0;  // kReduceDw, kReduceDb (kToExchange: splits = rows a block, RecLayout::few)
    size_t per = 0;
    unsigned first_block = 0, blocks = 0;   // set by run_ops
};
// Time stamps and status of a pass.  Device side: word 0 of `status` is the recurrence's status, `stamps` hold ticks of
// the constant-rate clock.  A list with `publish` set copies both to pinned host memory, so that the wait that ends the
// pass is also the one that makes them readable: no copy command and no second round trip.  Only the pass's own stamps are copied,
// and a forward pass's share a line of 64 bytes with the status: each further line of host memory written at its end costs 1 us
// (one step of 24 rows of 2144 units: three lines 51.0 us, two 50.0, one 48.7).
enum Stamp : int { kStampFwdBegin, kStampFwdStart, kStampFwdRec, kStampFwdRecEnd, kStampFwdEnd,
                   kStampBwdBegin, kStampBwdStart, kStampBwdRecEnd, kStampBwdDw, kStampBwdEnd, kStampCount };
struct HostStatus {
    int status;
    float absmax;   // (absmax())
    long long stamps[kStampCount];
};
struct OpList {
    int count = 0;
    int stamp = -1;                   // which stamp block 0 writes when it is done (-1: none)
    int begin = -1;                   // ... and which when it starts
    const int* status = nullptr;      // device status word (with `publish`)
    long long* stamps = nullptr;
    HostStatus* publish = nullptr;    // (the stamps of the direction whose last one `stamp` is)
    bool only_if_ok = false;          // (with `status`) the operations are left out if that word is not 0
    LayoutOp op[kMaxOps];

    void fill(void* p, size_t bytes, unsigned word);   // bytes: a multiple of 4
    // rows x cols (pitch ld_in, fp32 when in_f32 else fp16; null reads as zeros), times `scale`, -> fp16 [rows_out][ld_out], zero padded
    void to_half(const void* in, int in_f32, size_t rows, int cols, size_t ld_in, float scale, half_t* out, size_t rows_out, size_t ld_out);
    // ... -> fp32 [rows][ld_out], zero padded (the input's pitch is cols)
    void to_float(const void* in, int in_f32, size_t rows, int cols, float scale, float* out, size_t ld_out);
    // padded internals -> caller tensors: out[r][c] = scale * in[row(r)][c], c < cols, with
    // row(r) = (r / rows_per_block) * block_stride + r % rows_per_block (rows_per_block = 0: row(r) = r): a gather of row
    // blocks pulls the states at every R-th step out of the state arrays.  A null `out` adds nothing.
    void unpad(const void* in, int in_f32, size_t ld_in, size_t rows, int cols, float scale, void* out, int out_f32,
               size_t rows_per_block = 0, size_t block_stride = 0);
    // rows x cols (pitch cols; null reads as zeros) -> a whole slot of an exchange ring (fragment-major, rows padded to 32, kcols
    // columns), zero elsewhere.  few: the ring of rec_fwd_few_kernel, blocks of that many rows (RecLayout::few)
    void to_exchange(const void* in, int in_f32, size_t rows, int cols, int kcols, half_t* slot, int few = 0);
    // Sums columns [col0, col0 + out_cols) of the split-K partials [splits][4Hp][ld] (packed gate rows) into dst
    // [4H][out_cols] (PyTorch row order), times `scale`; `accumulate` adds to dst instead of overwriting it (the beta=1
    // accumulation over chunks of flashlstm_v2/src/lstm_backward.cu:1112-1142).  A null dst adds nothing.
    void reduce_dw(const Dims& d, const float* partial, int splits, size_t ld, int col0, int out_cols, float scale, bool accumulate, float* dst);
    // db_part [ng][4Hp] packed -> db_ih == db_hh (4H), times scale (flashlstm_v2/src/lstm_backward.cu:1218-1231)
    void reduce_db(const Dims& d, const float* db_part, int ng, float scale, bool accumulate, float* db_ih, float* db_hh);
};
hipError_t run_ops(OpList& list, hipStream_t s);
// one operation as a launch of its own
hipError_t gather_from_half(const half_t* in, size_t ld_in, size_t rows, int cols, void* out, int out_f32,
                            size_t rows_per_block, size_t block_stride, hipStream_t s);
hipError_t gather_from_float(const float* in, size_t ld_in, size_t rows, int cols, float scale, void* out, int out_f32,
                             size_t rows_per_block, size_t block_stride, hipStream_t s);
// fp16 values spread over (-amp, amp) from a hash of the index (operands for timing runs)
hipError_t fill_noise(half_t* p, size_t n, unsigned seed, float amp, hipStream_t s);
// Fills a buffer (multiple of 4 bytes) with one 32-bit pattern; a kernel, so it may be captured in a graph.
hipError_t fill_words(void* p, size_t bytes, unsigned value, hipStream_t s);

}  // namespace flstm_hip
