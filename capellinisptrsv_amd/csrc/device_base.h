// Types and small device functions shared by the kernels' headers and sources.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cap {

constexpr int kWave = 64;
constexpr int kBlock = 256;       // 4 wavefronts per workgroup

template <typename T>
struct VBits;
template <>
struct VBits<double> {
    typedef unsigned long long U;
    static constexpr U kSentinel = 0xFFF0000000000001ULL;  // negative signalling NaN
    static constexpr U kQNaN = 0x7FF8000000000000ULL;
};
template <>
struct VBits<float> {
    typedef unsigned int U;
    static constexpr U kSentinel = 0xFF800001u;
    static constexpr U kQNaN = 0x7FC00000u;
};

__device__ __forceinline__ double as_val(unsigned long long u) { return __longlong_as_double((long long)u); }
__device__ __forceinline__ float as_val(unsigned int u) { return __uint_as_float(u); }
__device__ __forceinline__ unsigned long long as_bits(double v) { return (unsigned long long)__double_as_longlong(v); }
__device__ __forceinline__ unsigned int as_bits(float v) { return __float_as_uint(v); }
__device__ __forceinline__ double fmac(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmac(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// Workgroup barrier that orders LDS only: the plain __syncthreads would also
// wait for the acknowledgement of the published values.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace cap
