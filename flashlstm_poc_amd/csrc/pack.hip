// Layout kernels: weight packing, padded dtype conversion, transposes and output reductions.
// All are pure HBM-bandwidth work; each thread moves a few elements with coalesced accesses.
#include "layout_device.h"
#include "pack.h"
#include "recurrent.h"

namespace flstm_hip {
namespace {

constexpr int kT = 256;

__host__ __device__ inline int grid_for(size_t n) { return int((n + kT - 1) / kT); }

// Column q of the gate arrays (x-projection / gate cache, dG, and with them the rows of the packed W_ih, the bias
// and the contraction index of the backward products) -> PyTorch weight row, or -1 for a padding unit.  The four
// gates of a hidden unit are neighbours, q = 4 * unit + gate, so a thread that owns a few consecutive units moves
// all of their gate values with one 16-byte access.
__device__ __forceinline__ int torch_row(int q, int H) {
    const int j = q / 4, gate = q % 4;
    return j < H ? gate * H + j : -1;
}

// Everything that becomes of the weights, one launch; blocks [first[i], first[i + 1]) of the grid make operand i.  A thread
// makes eight consecutive halfs (one 16-byte store).  One element per thread and one launch per operand took 28 us of
// kernels and the gaps between them at 650 units, every pass of a training loop.
struct PackJob {
    Dims d;
    const float *w_ih, *w_hh;
    half_t *wih_p, *wih_t;
    FragLayout frag[kFragKinds];
    unsigned first[kFragKinds + 3];
};

__device__ __forceinline__ half8 frag_values_fwd(const Dims& d, const float* __restrict__ w_hh, const FragLayout& f, size_t item) {
    // B operand of  gates[b][c] += h[b][k] * W_hh[row(c)][k].  The product's columns are local to a workgroup (they only
    // meet the pointwise stage through LDS) and stay gate-major within the slice of JB = 4*NT units: column
    // c = gate * JB + unit.  In the kernels with one cell per thread (rec_fwd_il_kernel, rec_fwd_wide_kernel) they are
    // unit-major, column c = 4 * unit + gate: the four accumulation registers of a lane are then the four gates of one
    // unit.  Fragment (hs, wave, ks, n): lane l holds column c = n*16 + l%16 of slice hs, k = (ks*nw + wave)*32 + 8*(l/16)
    // + e, e = 0..7 (nw = wavefronts per workgroup, 4 or 8).
    // split (rec_fwd_split_kernel): a wave has two tiles over the whole contraction, column c of tile n is gate c % 4 of
    // its unit 2 (c / 4) + n.
    const int tiles = f.split ? 2 : f.nt;
    unsigned r = unsigned(item);
    const int lane = int(r % kWave); r /= kWave;
    const int n = int(r % tiles); r /= tiles;
    const int ks = int(r % f.ks); r /= f.ks;
    const int nw = f.split ? f.split : f.nw;
    const int wave = int(r % nw);
    const int hs = int(r / nw);
    const int jb = f.split ? 8 * f.split : 4 * f.nt, c = n * 16 + lane % 16, nh = d.Hp / jb;
    const int gate = f.unit_major || f.split ? c % 4 : c / jb;
    const int unit = hs * jb + (f.split ? wave * 8 + 2 * ((c % 16) / 4) + n : f.unit_major ? c / 4 : c % jb);
    // (slot ks of slice hs holds a rotated k-step: recurrent.h, rec_kstep_rotation, rec_wide_rotation)
    const int kstep = f.wide ? (ks ^ rec_wide_rotation(ks, hs / 8, f.ks)) : rec_kstep_of_slot(ks, rec_kstep_rotation(hs, nh, f.ks, f.rot_div), f.ks);
    const int k = (f.split ? ks : kstep * f.nw + wave) * 32 + 8 * (lane / 16);
    half8 v{};
    if (unit < d.H) {
        const float* row = w_hh + size_t(gate * d.H + unit) * d.H;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (k + e < d.H) v[e] = (half_t)row[k + e];
    }
    return v;
}

// eight consecutive packed gate rows q .. q+7 (two units) of column k of W_hh
__device__ __forceinline__ half8 gate_rows(const Dims& d, const float* __restrict__ w_hh, int q, int k) {
    half8 v{};
    if (k < d.H) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int row = torch_row(q + e, d.H);
            if (row >= 0) v[e] = (half_t)w_hh[size_t(row) * d.H + k];
        }
    }
    return v;
}

__device__ __forceinline__ half8 frag_values_bwd(const Dims& d, const float* __restrict__ w_hh, const FragLayout& f, size_t item) {
    // B operand of  dh[b][k] += dG[b][q] * W_hh[row(q)][k].  Fragment (hs, wave, ks, n): lane l holds output column
    // k = hs*16*NT + n*16 + l%16, contraction index q = (ks*nw + wave)*32 + 8*(l/16) + e.
    unsigned r = unsigned(item);
    const int lane = int(r % kWave); r /= kWave;
    const int n = int(r % f.nt); r /= f.nt;
    const int ks = int(r % f.ks); r /= f.ks;
    const int wave = int(r % f.nw);
    const int hs = int(r / f.nw), nh = d.Hp / (16 * f.nt);
    const int k = hs * 16 * f.nt + n * 16 + lane % 16;
    const int kstep = rec_kstep_of_slot(ks, rec_kstep_rotation(hs, nh, f.ks, f.rot_div), f.ks);
    const int q = (kstep * f.nw + wave) * 32 + 8 * (lane / 16);
    return q < 4 * d.Hp ? gate_rows(d, w_hh, q, k) : half8{};
}

__device__ __forceinline__ half8 frag_values_two_d(const Dims& d, const float* __restrict__ w_hh, const FragLayout& f, size_t item) {
    // [Hp / 64 column slices s][kq contraction slices q][4 waves][ks k-steps][4 tiles][64 lanes][8]: lane l of tile n holds
    // column 64 s + 16 n + l % 16 of W_hh (hidden unit k of dh = dG * W_hh^T-packed) and the eight packed gate rows
    // (4 Hp / kq) q + 32 (4 ks + wave) + 8 (l / 16) .. +7.
    unsigned r = unsigned(item);
    const int lane = int(r % kWave); r /= kWave;
    const int n = int(r % 4); r /= 4;
    const int ks = int(r % f.ks); r /= f.ks;
    const int wave = int(r % 4); r /= 4;
    const int qs = int(r % f.kq);
    const int sl = int(r / f.kq);
    const int k = sl * 64 + n * 16 + lane % 16;
    // (slot ks of a wave holds the k-step the kernel fetches there: rotated per column slice)
    const int kstep = f.wide ? (ks ^ rec_wide_rotation(ks, sl / 8, f.ks)) : rec_kstep_of_slot(ks, rec_bwd2d_rotation(sl, f.ks, f.kq), f.ks);
    const int in_slice = (kstep * 4 + wave) * 32 + 8 * (lane / 16), q = qs * (4 * d.Hp / f.kq) + in_slice;
    return in_slice < 4 * d.Hp / f.kq ? gate_rows(d, w_hh, q, k) : half8{};
}

__global__ __launch_bounds__(kT) void pack_kernel(PackJob job) {
    const Dims& d = job.d;
    int which = 0;
    while (blockIdx.x >= job.first[which + 1]) ++which;
    const size_t item = size_t(blockIdx.x - job.first[which]) * kT + threadIdx.x;
    if (which == 0) {          // wih_p: eight columns of a packed row
        const unsigned per_row = unsigned(d.Ip) / 8;
        if (item >= size_t(4) * d.Hp * per_row) return;
        const int q = int(unsigned(item) / per_row), i = int(unsigned(item) % per_row) * 8, row = torch_row(q, d.H);
        half8 v{};
        if (row >= 0) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (i + e < d.I) v[e] = (half_t)job.w_ih[size_t(row) * d.I + i + e];
        }
        st_half8(job.wih_p + size_t(q) * d.Ip + i, v);
    } else if (which == 1) {   // wih_t: eight packed gate columns of a row; 16 rows by 4 chunks per wave, so that reads and writes come in 64-byte pieces
        const unsigned chunks = unsigned(4 * d.Hp) / 8, lane = unsigned(item) % 64, tile = unsigned(item) / 64, across = chunks / 4;
        const int i = int(tile / across * 16 + lane % 16), q = int((tile % across) * 4 + lane / 16) * 8;
        if (i >= d.Ip) return;
        half8 v{};
        if (i < d.I) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int row = torch_row(q + e, d.H);
                if (row >= 0) v[e] = (half_t)job.w_ih[size_t(row) * d.I + i];
            }
        }
        st_half8(job.wih_t + size_t(i) * 4 * d.Hp + q, v);
    } else {
        const FragLayout& f = job.frag[which - 2];
        if (item >= f.fragments * kWave) return;
        const int kind = which - 2;
        f.out[item] = kind <= kFragFwdSplit ? frag_values_fwd(d, job.w_hh, f, item) : kind <= kFragBwdBroad ? frag_values_bwd(d, job.w_hh, f, item) : frag_values_two_d(d, job.w_hh, f, item);
    }
}

// Fragment `tile` of a slice's 128 columns in one order, 32 * gate + unit or 4 * unit + gate, from those in the other: lane l of it, column
// 16 tile + l % 16, is a lane of the other order's tile that holds the same column and the same eight k.
__global__ __launch_bounds__(kT) void reorder_kernel(const half8* __restrict__ in, half8* __restrict__ out, unsigned items, int gate_major) {
    const unsigned i = blockIdx.x * kT + threadIdx.x;
    if (i >= items) return;
    const unsigned lane = i % kWave, tile = i / kWave % 8, column = 16 * tile + lane % 16;
    const unsigned other = gate_major ? column % 32 * 4 + column / 32 : column % 4 * 32 + column / 4;
    out[i] = in[(i / (8 * kWave) * 8 + other / 16) * kWave + lane / 16 * 16 + other % 16];
}

__global__ void pack_bias_kernel(Dims d, const float* __restrict__ b_ih, const float* __restrict__ b_hh,
                                 float* __restrict__ out) {
    const int q = blockIdx.x * kT + threadIdx.x;
    if (q >= 4 * d.Hp) return;
    const int row = torch_row(q, d.H);
    out[q] = row >= 0 ? b_ih[row] + b_hh[row] : 0.f;
}

__global__ void fill_words_kernel(unsigned* p, size_t words, unsigned value) {
    const size_t stride = size_t(gridDim.x) * kT;
    for (size_t i = size_t(blockIdx.x) * kT + threadIdx.x; i < words; i += stride) p[i] = value;
}

// kToHalf / kToFloat: V consecutive elements of an output row (V = 8: ld_out is a multiple of 8)
template <int V>
__device__ __forceinline__ void op_convert(const LayoutOp& o, size_t first, size_t stride) {
    const int out_f32 = o.kind == LayoutOp::kToFloat;
    const bool aligned = (o.ld_in % V == 0) && (reinterpret_cast<uintptr_t>(o.src) % 16 == 0);   // whole 16-byte loads
    for (size_t i = first; i < o.n; i += stride) {
        size_t r, c;
        split_index(i, o.ld_out / V, r, c);
        c *= V;
        float v[V];
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = 0.f;
        if (o.src != nullptr && r < o.rows) {
            const size_t at = r * o.ld_in + c;
            if (aligned && c + V <= size_t(o.cols)) {
                load_floats<V>(o.src, at, o.in_f32, v);
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (c + e < size_t(o.cols)) { float one[1]; load_floats<1>(o.src, at + e, o.in_f32, one); v[e] = one[0]; }
            }
#pragma unroll
            for (int e = 0; e < V; ++e) v[e] *= o.scale;
        }
        store_values<V>(o.dst, r * o.ld_out + c, out_f32, v);
    }
}

// kReduceDw: V consecutive columns of a gradient row (V = 4: pitches and first column multiples of 4).  The partials of an element are
// added in the order of the splits.
template <int V>
__device__ __forceinline__ void op_reduce_dw(const LayoutOp& o, size_t first, size_t stride) {
    const float* partial = static_cast<const float*>(o.src);
    float* dst = static_cast<float*>(o.dst);
    for (size_t i = first; i < o.n; i += stride) {
        size_t row, c;
        split_index(i, size_t(o.cols) / V, row, c);
        c *= V;
        const unsigned gate = unsigned(row) / unsigned(o.H), j = unsigned(row) % unsigned(o.H);
        const size_t at = (size_t(4) * j + gate) * o.ld_in + c;
        float s[V];
#pragma unroll
        for (int e = 0; e < V; ++e) s[e] = 0.f;
        for (int z = 0; z < o.splits; ++z) {
            const float* p = partial + size_t(z) * o.per + at;
            if constexpr (V == 4) {
                const floatx4 q = *reinterpret_cast<const floatx4*>(p);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] += q[e];
            } else {
                s[0] += p[0];
            }
        }
        float* out = dst + row * size_t(o.cols) + c;
#pragma unroll
        for (int e = 0; e < V; ++e) out[e] = o.accumulate ? out[e] + o.scale * s[e] : o.scale * s[e];
    }
}

// Blocks [first_block, first_block + blocks) of the grid walk an operation with a grid stride.  All of it is memory
// traffic or launch latency: eight elements per thread in 16-byte accesses where the pitches allow (fp32 sequence of
// 65536 x 1024 from fp16 rows: 2.1 TB/s with one element per thread and 64-bit index arithmetic).
__global__ __launch_bounds__(kT) void layout_ops_kernel(OpList list) {
    // (stored at the end: a store in front of the operations' loads keeps block 0 waiting for its way to memory, 1 us a pass)
    const long long begun = blockIdx.x == 0 && list.begin >= 0 ? wall_clock64() : 0;
    int which = 0;
    while (which + 1 < list.count && blockIdx.x >= list.op[which + 1].first_block) ++which;
    if (list.count > 0 && !(list.only_if_ok && *list.status != 0)) {
        const LayoutOp& o = list.op[which];
        const size_t stride = size_t(o.blocks) * kT;
        const size_t first = size_t(blockIdx.x - o.first_block) * kT + threadIdx.x;
        if (o.kind == LayoutOp::kFill) {
            if (o.vec == 4) {
                uint4* p = static_cast<uint4*>(o.dst);
                for (size_t i = first; i < o.n; i += stride) p[i] = uint4{o.word, o.word, o.word, o.word};
            } else {
                unsigned* p = static_cast<unsigned*>(o.dst);
                for (size_t i = first; i < o.n; i += stride) p[i] = o.word;
            }
        } else if (o.kind == LayoutOp::kToHalf || o.kind == LayoutOp::kToFloat) {
            if (o.vec == 8) op_convert<8>(o, first, stride);
            else op_convert<1>(o, first, stride);
        } else if (o.kind == LayoutOp::kUnpad) {
            op_unpad(o, first, stride);
        } else if (o.kind == LayoutOp::kToExchange) {
            // item i = eight halfs of one lane: [16-row tile][32-wide k-step][lane] (recurrent.hip, xch_offset); with `splits` rows a block
            // and pack = 16 / rows: [block][pack of k-steps 4 (pack P + s) + w at 4 P + w][lane], rows * s .. k-step s (rec_fwd_few_kernel)
            const unsigned rb = o.splits ? unsigned(o.splits) : 16u, pack = 16u / rb, nks = unsigned(o.ld_out) / 32;
            const unsigned per_tile = o.splits ? (nks + 4 * pack - 1) / (4 * pack) * 4 : nks;
            for (size_t i = first; i < o.n; i += stride) {
                const unsigned lane = unsigned(i) % 64, at = (unsigned(i) / 64) % per_tile, tile = unsigned(i) / 64 / per_tile;
                const size_t r = size_t(tile) * rb + lane % rb;
                const unsigned k = (4 * (at / 4 * pack + lane % 16 / rb) + at % 4) * 32 + (lane / 16) * 8;
                half8 h{};
                if (o.src != nullptr && r < o.rows) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (k + e < unsigned(o.cols)) { float one[1]; load_floats<1>(o.src, r * o.cols + k + e, o.in_f32, one); h[e] = (half_t)one[0]; }
                }
                st_half8(static_cast<half_t*>(o.dst) + i * 8, h);
            }
        } else if (o.kind == LayoutOp::kReduceDw) {
            if (o.vec == 4) op_reduce_dw<4>(o, first, stride);
            else op_reduce_dw<1>(o, first, stride);
        } else if (o.kind == LayoutOp::kReduceDb) {
            const float* part = static_cast<const float*>(o.src);
            float *db_ih = static_cast<float*>(o.dst), *db_hh = static_cast<float*>(o.dst2);
            for (size_t q = first; q < o.n; q += stride) {
                const int row = torch_row(int(q), o.H);
                if (row < 0) continue;
                float s = 0.f;
                int g = 0;
                for (; g + 8 <= o.splits; g += 8) {   // (eight on their way at a time: small layers have up to 256 groups)
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = part[size_t(g + e) * o.n + q];
#pragma unroll
                    for (int e = 0; e < 8; ++e) s += v[e];
                }
                for (; g < o.splits; ++g) s += part[size_t(g) * o.n + q];
                s *= o.scale;
                if (db_ih) db_ih[row] = o.accumulate ? db_ih[row] + s : s;
                if (db_hh && db_hh != db_ih) db_hh[row] = o.accumulate ? db_hh[row] + s : s;
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && list.stamps) {
        const long long now = wall_clock64();
        if (list.begin >= 0) list.stamps[list.begin] = begun;
        if (list.stamp >= 0) list.stamps[list.stamp] = now;
        if (list.publish) {   // (what earlier launches left: this launch writes neither the status nor the other stamps)
            __hip_atomic_store(&list.publish->status, *list.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            for (int i = list.stamp == kStampFwdEnd ? kStampFwdBegin : kStampBwdBegin; i <= list.stamp; ++i)
                __hip_atomic_store(&list.publish->stamps[i], i == list.stamp ? now : list.stamps[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

}  // namespace

hipError_t pack_weights(const Dims& d, const float* w_ih, const float* w_hh, half_t* wih_p, half_t* wih_t,
                        const FragLayout (&frag)[kFragKinds], hipStream_t s) {
    PackJob job{};
    job.d = d;
    job.w_ih = w_ih; job.w_hh = w_hh; job.wih_p = wih_p; job.wih_t = wih_t;
    // (Hp is a multiple of 32 and Ip of 64: whole chunks of eight, and of four chunks, everywhere)
    for (int i = 0; i < kFragKinds + 2; ++i) {
        size_t items = size_t(4) * d.Hp * d.Ip / 8;
        if (i >= 2) {
            job.frag[i - 2] = frag[i - 2];
            items = frag[i - 2].out ? frag[i - 2].fragments * kWave : 0;
        }
        if (items >> 32) return hipErrorInvalidValue;
        job.first[i + 1] = job.first[i] + unsigned(ceil_div(items, kT));
    }
    hipLaunchKernelGGL(pack_kernel, dim3(job.first[kFragKinds + 2]), dim3(kT), 0, s, job);
    return hipGetLastError();
}

hipError_t reorder_fragments(const half8* in, half8* out, size_t fragments, bool gate_major, hipStream_t s) {
    const size_t items = fragments * kWave;
    if (items == 0 || fragments % 8 != 0 || items >> 32) return hipErrorInvalidValue;
    hipLaunchKernelGGL(reorder_kernel, dim3(unsigned(ceil_div(items, kT))), dim3(kT), 0, s, in, out, unsigned(items), int(gate_major));
    return hipGetLastError();
}

hipError_t pack_bias(const Dims& d, const float* b_ih, const float* b_hh, float* bias_p, hipStream_t s) {
    hipLaunchKernelGGL(pack_bias_kernel, dim3(grid_for(size_t(4) * d.Hp)), dim3(kT), 0, s, d, b_ih, b_hh, bias_p);
    return hipGetLastError();
}

namespace {

// a work item's elements: 8 where rows and bases allow 16-byte accesses
bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

void OpList::fill(void* p, size_t bytes, unsigned w) {
    if (bytes == 0) return;
    LayoutOp& o = op[count++];
    o.kind = LayoutOp::kFill; o.dst = p; o.word = w;
    o.vec = (aligned16(p) && bytes % 16 == 0) ? 4 : 1;
    o.n = bytes / 4 / o.vec;
}

void OpList::to_half(const void* in, int in_f32, size_t rows, int cols, size_t ld_in, float scale, half_t* out, size_t rows_out, size_t ld_out) {
    if (rows_out * ld_out == 0) return;
    LayoutOp& o = op[count++];
    o.kind = LayoutOp::kToHalf; o.in_f32 = in_f32; o.dst = out; o.src = in;
    o.vec = (ld_out % 8 == 0 && aligned16(out)) ? 8 : 1;
    o.n = rows_out * ld_out / o.vec;
    o.rows = rows; o.cols = cols; o.ld_in = ld_in; o.ld_out = ld_out; o.scale = scale;
}

void OpList::to_float(const void* in, int in_f32, size_t rows, int cols, float scale, float* out, size_t ld_out) {
    if (rows * ld_out == 0) return;
    LayoutOp& o = op[count++];
    o.kind = LayoutOp::kToFloat; o.in_f32 = in_f32; o.dst = out; o.src = in;
    o.vec = (ld_out % 8 == 0 && aligned16(out)) ? 8 : 1;
    o.n = rows * ld_out / o.vec;
    o.rows = rows; o.cols = cols; o.ld_in = size_t(cols); o.ld_out = ld_out; o.scale = scale;
}

void OpList::unpad(const void* in, int in_f32, size_t ld_in, size_t rows, int cols, float scale, void* out, int out_f32,
                   size_t rows_per_block, size_t block_stride) {
    if (out == nullptr || rows * size_t(cols) == 0) return;
    if (rows_per_block >= rows) rows_per_block = 0;
    if (ld_in == size_t(cols) && rows_per_block == 0 && rows * size_t(cols) <= size_t(1) << 30) {   // contiguous: one row
        cols = int(rows * size_t(cols));
        ld_in = round_up(size_t(cols), 8);
        rows = 1;
    }
    LayoutOp& o = op[count++];
    o.kind = LayoutOp::kUnpad; o.in_f32 = in_f32; o.out_f32 = out_f32; o.dst = out; o.src = in;
    o.vec = (cols % 8 == 0 && ld_in % 8 == 0 && aligned16(in) && aligned16(out)) ? 8 : 1;
    if (o.vec == 8) {
        o.n = rows * size_t(cols) / 8;
    } else {   // 16 aligned bytes of the output per item (op_unpad_flat)
        const size_t esz = out_f32 ? 4 : 2;
        o.n = ceil_div(reinterpret_cast<uintptr_t>(out) % 16 + rows * size_t(cols) * esz, 16);
    }
    o.rows = rows; o.cols = cols; o.ld_in = ld_in; o.scale = scale;
    o.rows_per_block = rows_per_block; o.block_stride = block_stride;
}

void OpList::to_exchange(const void* in, int in_f32, size_t rows, int cols, int kcols, half_t* slot, int few) {
    LayoutOp& o = op[count++];
    o.kind = LayoutOp::kToExchange; o.in_f32 = in_f32; o.dst = slot; o.src = in;
    o.splits = few;
    o.n = few ? ceil_div(rows, size_t(few)) * ceil_div(size_t(kcols) / 32, size_t(4 * 16 / few)) * 4 * kWave : exchange_slot_halfs(int(rows), kcols) / 8;
    o.rows = rows; o.cols = cols; o.ld_out = size_t(kcols);
}

void OpList::reduce_dw(const Dims& d, const float* partial, int splits, size_t ld, int col0, int out_cols, float scale,
                       bool accumulate, float* dst) {
    if (dst == nullptr || out_cols <= 0) return;
    LayoutOp& o = op[count++];
    o.kind = LayoutOp::kReduceDw; o.src = partial + col0; o.dst = dst;
    o.vec = (out_cols % 4 == 0 && ld % 4 == 0 && col0 % 4 == 0 && aligned16(dst)) ? 4 : 1;
    o.n = size_t(4) * d.H * out_cols / o.vec;
    o.cols = out_cols; o.ld_in = ld; o.splits = splits; o.per = size_t(4) * d.Hp * ld; o.H = d.H; o.scale = scale;
    o.accumulate = accumulate ? 1 : 0;
}

void OpList::reduce_db(const Dims& d, const float* db_part, int ng, float scale, bool accumulate, float* db_ih, float* db_hh) {
    if (!db_ih && !db_hh) return;
    LayoutOp& o = op[count++];
    o.kind = LayoutOp::kReduceDb; o.src = db_part; o.dst = db_ih; o.dst2 = db_hh;
    o.n = size_t(4) * d.Hp; o.splits = ng; o.H = d.H; o.scale = scale; o.accumulate = accumulate ? 1 : 0;
}

hipError_t run_ops(OpList& list, hipStream_t s) {
    if (list.count > kMaxOps) return hipErrorInvalidValue;
    if (list.count <= 0 && !list.publish) return hipSuccess;
    unsigned total = 0;
    for (int i = 0; i < list.count; ++i) {
        LayoutOp& o = list.op[i];
        size_t blocks = (o.n + kT - 1) / kT;
        if (blocks > 4096) blocks = 4096;   // (more work than that is walked with the grid stride)
        if (blocks < 1) blocks = 1;
        o.first_block = total;
        o.blocks = unsigned(blocks);
        total += o.blocks;
    }
    hipLaunchKernelGGL(layout_ops_kernel, dim3(total ? total : 1), dim3(kT), 0, s, list);
    return hipGetLastError();
}

hipError_t gather_from_half(const half_t* in, size_t ld_in, size_t rows, int cols, void* out, int out_f32,
                            size_t rows_per_block, size_t block_stride, hipStream_t s) {
    OpList list;
    list.unpad(in, 0, ld_in, rows, cols, 1.f, out, out_f32, rows_per_block, block_stride);
    return run_ops(list, s);
}

hipError_t gather_from_float(const float* in, size_t ld_in, size_t rows, int cols, float scale, void* out, int out_f32,
                             size_t rows_per_block, size_t block_stride, hipStream_t s) {
    OpList list;
    list.unpad(in, 1, ld_in, rows, cols, scale, out, out_f32, rows_per_block, block_stride);
    return run_ops(list, s);
}

__global__ void reduce_partials_kernel(const float* __restrict__ partial, int splits, size_t per, int rows, int cols,
                                       size_t ldc, float* __restrict__ dst) {
    const size_t idx = size_t(blockIdx.x) * kT + threadIdx.x;
    if (idx >= size_t(rows) * cols) return;
    float s = 0.f;
    for (int z = 0; z < splits; ++z) s += partial[size_t(z) * per + idx];
    dst[(idx / cols) * ldc + idx % cols] = s;
}

hipError_t reduce_partials(const float* partial, int splits, size_t per, int rows, int cols, size_t ldc, float* dst,
                           hipStream_t s) {
    if (rows <= 0 || cols <= 0) return hipSuccess;
    hipLaunchKernelGGL(reduce_partials_kernel, dim3(grid_for(size_t(rows) * cols)), dim3(kT), 0, s, partial, splits, per,
                       rows, cols, ldc, dst);
    return hipGetLastError();
}

// Position-weighted sum of the 16-bit units of a buffer, added to *out: any changed, moved or swapped element
// changes the sum (up to a 2^-64 accident); the order of the additions does not matter, so atomics may be used.
// Eight units per thread and 16-byte load (one 2-byte load per thread and iteration read 16 MiB at 160 GB/s, 104 us).
__device__ __forceinline__ u64 checksum_unit(unsigned v16, size_t i, u64 salt) {
    u64 v = (u64(v16) + 1u) * (2 * (i + salt) + 1) * 0x9E3779B97F4A7C15ull;
    v ^= v >> 29;
    return v * 0xBF58476D1CE4E5B9ull;
}
__global__ __launch_bounds__(kT) void checksum_kernel(const unsigned short* __restrict__ p, size_t n, u64 salt, u64* out) {
    __shared__ u64 wave_sum[kT / 64];
    u64 acc = 0;
    const size_t stride = size_t(gridDim.x) * blockDim.x, first = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t n8 = (reinterpret_cast<uintptr_t>(p) % 16 == 0) ? n / 8 : 0;
    for (size_t i = first; i < n8; i += stride) {
        const uint4 q = reinterpret_cast<const uint4*>(p)[i];
        const unsigned w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) acc += checksum_unit((w[e / 2] >> (16 * (e % 2))) & 0xffffu, i * 8 + e, salt);
    }
    for (size_t i = n8 * 8 + first; i < n; i += stride) acc += checksum_unit(p[i], i, salt);
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
    if (threadIdx.x % 64 == 0) wave_sum[threadIdx.x / 64] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kT / 64; ++w) acc += wave_sum[w];
        atomicAdd(reinterpret_cast<unsigned long long*>(out), acc);
    }
}

hipError_t checksum_add(const void* p, size_t bytes, u64 salt, u64* out, hipStream_t s) {
    if (p == nullptr || bytes < 2) return hipSuccess;
    const size_t n = bytes / 2;   // every tensor of this library is made of 2- or 4-byte elements
    int blocks = grid_for(ceil_div(n, 8));
    if (blocks > 512) blocks = 512;
    hipLaunchKernelGGL(checksum_kernel, dim3(blocks), dim3(kT), 0, s, static_cast<const unsigned short*>(p), n, salt, out);
    return hipGetLastError();
}

// |value| as an unsigned word orders like the value, NaN above infinity.
__global__ __launch_bounds__(kT) void absmax_kernel(const void* t, int f32, size_t n, unsigned* partial) {
    __shared__ unsigned wave_max[kT / 64];
    unsigned m = 0;
    const size_t stride = size_t(gridDim.x) * kT, first = size_t(blockIdx.x) * kT + threadIdx.x;
    const int V = f32 ? 4 : 8;
    const size_t nv = reinterpret_cast<uintptr_t>(t) % 16 == 0 ? n / V : 0;
    for (size_t i = first; i < nv; i += stride) {
        const uint4 q = static_cast<const uint4*>(t)[i];
        const unsigned w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (f32) m = max(m, w[e] & 0x7fffffffu);
            else m = max(m, max(w[e] & 0x7fffu, (w[e] >> 16) & 0x7fffu));
        }
    }
    for (size_t i = nv * V + first; i < n; i += stride)
        m = max(m, f32 ? static_cast<const unsigned*>(t)[i] & 0x7fffffffu : unsigned(static_cast<const unsigned short*>(t)[i]) & 0x7fffu);
    for (int off = 32; off > 0; off >>= 1) m = max(m, unsigned(__shfl_down(int(m), off, 64)));
    if (threadIdx.x % 64 == 0) wave_max[threadIdx.x / 64] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kT / 64; ++w) m = max(m, wave_max[w]);
        partial[blockIdx.x] = m;
    }
}
__global__ __launch_bounds__(64) void absmax_finish_kernel(const unsigned* partial, int blocks, int f32, float* host_out) {
    unsigned m = 0;
    for (int i = threadIdx.x; i < blocks; i += 64) m = max(m, partial[i]);
    for (int off = 32; off > 0; off >>= 1) m = max(m, unsigned(__shfl_down(int(m), off, 64)));
    if (threadIdx.x == 0) {
        const float v = f32 ? __builtin_bit_cast(float, m) : (float)__builtin_bit_cast(half_t, (unsigned short)m);
        __hip_atomic_store(host_out, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
hipError_t absmax(const void* t, int f32, size_t n, unsigned* partial, float* host_out, hipStream_t s) {
    int blocks = grid_for(ceil_div(n, 8));
    if (blocks > kAbsmaxBlocks) blocks = kAbsmaxBlocks;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(absmax_kernel, dim3(blocks), dim3(kT), 0, s, t, f32, n, partial);
    hipLaunchKernelGGL(absmax_finish_kernel, dim3(1), dim3(64), 0, s, partial, blocks, f32, host_out);
    return hipGetLastError();
}

hipError_t fill_words(void* p, size_t bytes, unsigned value, hipStream_t s) {
    if (bytes == 0) return hipSuccess;
    const size_t words = bytes / 4;  // all buffers of this library are multiples of 4 bytes
    int blocks = grid_for(words);
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(fill_words_kernel, dim3(blocks), dim3(kT), 0, s, static_cast<unsigned*>(p), words, value);
    return hipGetLastError();
}

hipError_t fill_zero(void* p, size_t bytes, hipStream_t s) { return fill_words(p, bytes, 0u, s); }

// n fp16 values spread over (-amp, amp) from a hash of the index: operands for timing runs (the matrix cores draw
// more power, and run slower, on varied operands than on constant ones)
__global__ void fill_noise_kernel(half_t* p, size_t n, unsigned seed, float amp) {
    const size_t stride = size_t(gridDim.x) * kT;
    for (size_t i = size_t(blockIdx.x) * kT + threadIdx.x; i < n; i += stride) {
        unsigned h = unsigned(i) * 0x9E3779B1u + unsigned(i >> 32) * 0x85EBCA77u + seed;
        h ^= h >> 15; h *= 0x2C1B3C6Du; h ^= h >> 12; h *= 0x297A2D39u; h ^= h >> 15;
        p[i] = (half_t)(amp * (float(h >> 8) * (2.f / 16777216.f) - 1.f));
    }
}

hipError_t fill_noise(half_t* p, size_t n, unsigned seed, float amp, hipStream_t s) {
    if (n == 0) return hipSuccess;
    int blocks = grid_for(n);
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(fill_noise_kernel, dim3(blocks), dim3(kT), 0, s, p, n, seed, amp);
    return hipGetLastError();
}

}  // namespace flstm_hip
