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

// v, the same in every lane, in scalar registers: a product of 64 bits is
// formed in vector ones, and a buffer descriptor made from it would be read
// back lane by lane at every use.
__device__ __forceinline__ long long uniform(long long v)
{
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)v);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32));
    return (long long)((unsigned long long)hi << 32 | lo);
}

// Loads and stores through buffer descriptors: a uniform byte offset in a
// scalar register plus the thread's own 32-bit offset, so walking a table
// costs no vector instruction.  Reads past the descriptor's bytes give 0 and
// writes there are dropped.
typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef unsigned Words4 __attribute__((ext_vector_type(4)));
typedef unsigned Words2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ Rsrc make_rsrc(const void *p, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void load_value(Rsrc r, unsigned own, unsigned off, double *v)
{
    const Words2 w = __builtin_amdgcn_raw_buffer_load_b64(r, (int)own, (int)off, 0);
    __builtin_memcpy(v, &w, 8);
}
__device__ __forceinline__ void load_value(Rsrc r, unsigned own, unsigned off, float *v)
{
    const unsigned w = __builtin_amdgcn_raw_buffer_load_b32(r, (int)own, (int)off, 0);
    __builtin_memcpy(v, &w, 4);
}
__device__ __forceinline__ void store_value(Rsrc r, unsigned own, unsigned off, double v)
{
    Words2 w;
    __builtin_memcpy(&w, &v, 8);
    __builtin_amdgcn_raw_buffer_store_b64(w, r, (int)own, (int)off, 0);
}
__device__ __forceinline__ void store_value(Rsrc r, unsigned own, unsigned off, float v)
{
    unsigned w;
    __builtin_memcpy(&w, &v, 4);
    __builtin_amdgcn_raw_buffer_store_b32(w, r, (int)own, (int)off, 0);
}

}  // namespace cap
