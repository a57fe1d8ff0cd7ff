// Device side of the layout operations that more than one translation unit runs (pack.hip, recurrent.hip).
#pragma once
#include "pack.h"

namespace flstm_hip {

// Index arithmetic of the operations in 32 bits where the counts allow: a 64-bit division is a hundred instructions,
// more than the memory traffic of the 16 bytes it addresses.
__device__ __forceinline__ void split_index(size_t i, size_t width, size_t& r, size_t& c) {
    if ((i | width) >> 32) { r = i / width; c = i % width; }
    else { const unsigned q = unsigned(i) / unsigned(width); r = q; c = unsigned(i) - q * unsigned(width); }
}

template <int V>
__device__ __forceinline__ void load_floats(const void* src, size_t at, int in_f32, float (&v)[V]) {
    if constexpr (V == 8) {
        if (in_f32) {
            const floatx4* p = reinterpret_cast<const floatx4*>(static_cast<const float*>(src) + at);
            const floatx4 a = p[0], b = p[1];
#pragma unroll
            for (int e = 0; e < 4; ++e) { v[e] = a[e]; v[4 + e] = b[e]; }
        } else {
            const half8 h = ld_half8(static_cast<const half_t*>(src) + at);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (float)h[e];
        }
    } else {
        v[0] = in_f32 ? static_cast<const float*>(src)[at] : (float)static_cast<const half_t*>(src)[at];
    }
}
template <int V>
__device__ __forceinline__ void store_values(void* dst, size_t at, int out_f32, const float (&v)[V]) {
    if constexpr (V == 8) {
        if (out_f32) {
            floatx4* p = reinterpret_cast<floatx4*>(static_cast<float*>(dst) + at);
            p[0] = floatx4{v[0], v[1], v[2], v[3]};
            p[1] = floatx4{v[4], v[5], v[6], v[7]};
        } else {
            half8 h;
#pragma unroll
            for (int e = 0; e < 8; ++e) h[e] = (half_t)v[e];
            st_half8(static_cast<half_t*>(dst) + at, h);
        }
    } else {
        if (out_f32) static_cast<float*>(dst)[at] = v[0];
        else static_cast<half_t*>(dst)[at] = (half_t)v[0];
    }
}

// kUnpad: input row of output row r
__device__ __forceinline__ size_t unpad_row(const LayoutOp& o, size_t r) {
    if (!o.rows_per_block) return r;
    size_t blk, rest;
    split_index(r, o.rows_per_block, blk, rest);
    return blk * o.block_stride + rest;
}

// Eight consecutive elements of an output row per work item: both pitches multiples of 8, both bases 16-byte aligned.
__device__ __forceinline__ void op_unpad_rows(const LayoutOp& o, size_t first, size_t stride) {
    for (size_t i = first; i < o.n; i += stride) {
        size_t r, c;
        split_index(i, size_t(o.cols) / 8, r, c);
        float v[8];
        load_floats<8>(o.src, unpad_row(o, r) * o.ld_in + c * 8, o.in_f32, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= o.scale;
        store_values<8>(o.dst, i * 8, o.out_f32, v);
    }
}

// Any width, pitch and alignment: the output is one contiguous array, and a work item is E elements, 16 aligned bytes of it
// (fewer at its ends), which may lie across rows of the input.  Stores of an element per thread kept a link to host memory
// an eighth as busy: 1024 steps of 32 rows of 257 units streamed from and to the host, forward and backward, 57 -> 4.6 ms a pass; 512 steps of
// 128 rows, 1023 features and 256 units 9.0 -> 7.0, with 1024 features (whole 16-byte accesses throughout) 6.9.
template <int E>
__device__ __forceinline__ void op_unpad_flat(const LayoutOp& o, size_t first, size_t stride) {
    const size_t total = o.rows * size_t(o.cols), cols = size_t(o.cols);
    const size_t shift = reinterpret_cast<uintptr_t>(o.dst) % 16 / (16 / E);   // elements of the first item that are not there
    for (size_t i = first; i < o.n; i += stride) {
        const size_t lo = i == 0 ? 0 : i * E - shift, hi = min((i + 1) * E - shift, total);
        size_t r, c;
        split_index(lo, cols, r, c);
        float v[E];
        if (hi - lo == E && c + E <= cols) {   // within a row, at any alignment of the input
            const size_t at = unpad_row(o, r) * o.ld_in + c;
            if (o.in_f32) {
                float raw[E];
                __builtin_memcpy(raw, static_cast<const float*>(o.src) + at, sizeof(raw));
#pragma unroll
                for (int e = 0; e < E; ++e) v[e] = raw[e];
            } else {
                half_t raw[E];
                __builtin_memcpy(raw, static_cast<const half_t*>(o.src) + at, sizeof(raw));
#pragma unroll
                for (int e = 0; e < E; ++e) v[e] = (float)raw[e];
            }
        } else {
            size_t row = unpad_row(o, r) * o.ld_in;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                v[e] = 0.f;
                if (lo + e < hi) {
                    float one[1];
                    load_floats<1>(o.src, row + c, o.in_f32, one);
                    v[e] = one[0];
                    if (++c == cols) { c = 0; row = unpad_row(o, ++r) * o.ld_in; }
                }
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] *= o.scale;
        if (hi - lo == E) {
            if constexpr (E == 4) {
                *reinterpret_cast<floatx4*>(static_cast<float*>(o.dst) + lo) = floatx4{v[0], v[1], v[2], v[3]};
            } else {
                half8 h;
#pragma unroll
                for (int e = 0; e < 8; ++e) h[e] = (half_t)v[e];
                st_half8(static_cast<half_t*>(o.dst) + lo, h);
            }
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (lo + e < hi) { const float one[1] = {v[e]}; store_values<1>(o.dst, lo + e, o.out_f32, one); }
        }
    }
}

__device__ __forceinline__ void op_unpad(const LayoutOp& o, size_t first, size_t stride) {
    if (o.vec == 8) op_unpad_rows(o, first, stride);
    else if (o.out_f32) op_unpad_flat<4>(o, first, stride);
    else op_unpad_flat<8>(o, first, stride);
}

}  // namespace flstm_hip
