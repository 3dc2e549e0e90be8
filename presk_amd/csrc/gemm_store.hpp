// What the contraction kernels share of their epilogue: the stored output
// element and the bias element, in each storage type.
#pragma once

#include <hip/hip_runtime.h>

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

namespace {

// The split partial sums added in increasing split order, then the epilogue.
// Each source has its own: a source's code is loaded whole the first time one
// of its kernels is, and gemm.hip's is 3 MB (the first recording of a dense
// layer's reverse mode, whose products gemm_split.hip holds, took 11.2 ms with the
// partials summed there and takes 5.5).
template <int ST>
__global__ void __launch_bounds__(256) split_reduce_kernel(GemmArgs g) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= g.M * g.N) return;
    // M * N < 2^31 (the plan's bound): 32-bit division
    const unsigned nn = (unsigned)g.N, mq = (unsigned)idx / nn;
    const long long m = mq, n = (unsigned)idx - mq * nn;
    // the partials in increasing split order, eight loads in flight
    const long long mn = g.M * g.N;
    float s = g.work[idx];
    int p = 1;
    for (; p + 8 <= g.splits; p += 8) {
        float w[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) w[q] = g.work[(long long)(p + q) * mn + idx];
#pragma unroll
        for (int q = 0; q < 8; ++q) s = s + w[q];
    }
    for (; p < g.splits; ++p) s = s + g.work[(long long)p * mn + idx];
    bool ovf = false;
    float b = 0.f;
    // an e8m15 plan keeps bias_kind but passes no bias here: its own last
    // kernel adds the bias after narrowing the sum
    if (g.bias) {
        if (g.bias_kind == 1) b = load_bias<ST>(g.bias, n);
        else if (g.bias_kind == 2) b = load_bias<ST>(g.bias, idx);
        else if (g.bias_kind == 3) b = load_bias<ST>(g.bias, 0);
    }
    store_out<ST>(g.C, m * g.sc_m + n, s, g.bias != nullptr, b, ovf);
    if (ovf && g.flag) atomicOr(g.flag, 1u);
}

// (nothing to do where K is not split)
template <int ST>
hipError_t split_reduce(const GemmArgs& g, hipStream_t stream) {
    if (g.splits <= 1) return hipSuccess;
    split_reduce_kernel<ST><<<(unsigned)((g.M * g.N + 255) / 256), 256, 0, stream>>>(g);
    return hipGetLastError();
}

}  // namespace

}  // namespace presk
