// What the contraction kernels share of their epilogue: the stored output
// element and the bias element, in each storage type.
#pragma once

#include <type_traits>

#include "devfmt.hpp"
#include "gemm.hpp"

namespace presk {

// The storage-type store of an output element with the epilogue: f32 storage
// adds the bias to the sum; narrow storage stores the sum rounded, reads it
// back and adds (lower.rs:1053-1060), each store under the overflow guard.
template <int ST>
__device__ __forceinline__ void store_out(void* C, long long off, float sum, bool has_bias, float bias, bool& ovf) {
    if (ST == kF32) {
        ((float*)C)[off] = has_bias ? sum + bias : sum;
    } else if (ST == kBF16) {
        unsigned short h = pk_f32_to_bf16(sum);
        if (has_bias) h = pk_f32_to_bf16(pk_bf16_to_f32(h) + bias);
        ((unsigned short*)C)[off] = h;
    } else {
        ovf |= pk_overflows_f16(sum);
        unsigned short h = pk_f32_to_f16(sum);
        if (has_bias) {
            const float v = pk_f16_to_f32(h) + bias;
            ovf |= pk_overflows_f16(v);
            h = pk_f32_to_f16(v);
        }
        ((unsigned short*)C)[off] = h;
    }
}

// The stored value of an output element (as store_out computes it).
template <int ST>
__device__ __forceinline__ typename std::conditional<ST == kF32, float, unsigned short>::type round_out(float sum, bool has_bias, float bias, bool& ovf) {
    if constexpr (ST == kF32) {
        return has_bias ? sum + bias : sum;
    } else if constexpr (ST == kBF16) {
        unsigned short h = pk_f32_to_bf16(sum);
        if (has_bias) h = pk_f32_to_bf16(pk_bf16_to_f32(h) + bias);
        return h;
    } else {
        ovf |= pk_overflows_f16(sum);
        unsigned short h = pk_f32_to_f16(sum);
        if (has_bias) {
            const float v = pk_f16_to_f32(h) + bias;
            ovf |= pk_overflows_f16(v);
            h = pk_f32_to_f16(v);
        }
        return h;
    }
}

template <int ST>
__device__ __forceinline__ float load_bias(const void* p, long long off) {
    if (ST == kF32) return ((const float*)p)[off];
    if (ST == kBF16) return pk_bf16_to_f32(((const unsigned short*)p)[off]);
    return pk_f16_to_f32(((const unsigned short*)p)[off]);
}

}  // namespace presk
