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

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
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
    } else if constexpr (V == 2) {
        if (in_f32) {
            const float2 q = *reinterpret_cast<const float2*>(static_cast<const float*>(src) + at);
            v[0] = q.x; v[1] = q.y;
        } else {
            const half2v q = *reinterpret_cast<const half2v*>(static_cast<const half_t*>(src) + at);
            v[0] = (float)q[0]; v[1] = (float)q[1];
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
    } else if constexpr (V == 2) {
        if (out_f32) *reinterpret_cast<float2*>(static_cast<float*>(dst) + at) = float2{v[0], v[1]};
        else *reinterpret_cast<half2v*>(static_cast<half_t*>(dst) + at) = half2v{(half_t)v[0], (half_t)v[1]};
    } else {
        if (out_f32) static_cast<float*>(dst)[at] = v[0];
        else static_cast<half_t*>(dst)[at] = (half_t)v[0];
    }
}

// kUnpad: V consecutive elements of an output row (V = 8: both pitches multiples of 8, both bases 16-byte aligned;
// V = 2: even pitches, bases 8-byte aligned)
template <int V>
__device__ __forceinline__ void op_unpad(const LayoutOp& o, size_t first, size_t stride) {
    for (size_t i = first; i < o.n; i += stride) {
        size_t r, c;
        split_index(i, size_t(o.cols) / V, r, c);
        size_t rin = r;
        if (o.rows_per_block) {
            size_t blk, rest;
            split_index(r, o.rows_per_block, blk, rest);
            rin = blk * o.block_stride + rest;
        }
        float v[V];
        load_floats<V>(o.src, rin * o.ld_in + c * V, o.in_f32, v);
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] *= o.scale;
        store_values<V>(o.dst, i * V, o.out_f32, v);
    }
}

__device__ __forceinline__ void op_unpad_any(const LayoutOp& o, size_t first, size_t stride) {
    if (o.vec == 8) op_unpad<8>(o, first, stride);
    else if (o.vec == 2) op_unpad<2>(o, first, stride);
    else op_unpad<1>(o, first, stride);
}

}  // namespace flstm_hip
