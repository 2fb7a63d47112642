// 16 x 16 matrix-core tiles (gfx950) and device-memory views shared by the sigma kernels.
#pragma once
#include <hip/hip_runtime.h>

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// device-memory (global address space) views of pointers read from descriptors, so their
// loads are global loads (vector-memory counter only) rather than flat ones, which a later
// LDS wait would also have to drain
template <typename T> __device__ __forceinline__ const __attribute__((address_space(1))) T *
gptr(const T *p)
{
    return (const __attribute__((address_space(1))) T *)p;
}
template <typename T> __device__ __forceinline__ __attribute__((address_space(1))) T *gptr_w(T *p)
{
    return (__attribute__((address_space(1))) T *)p;
}

// 16x16 output tile, 4-deep reduction per instruction.  Operand lanes: A[l % 16][l / 16],
// B[l / 16][l % 16]; accumulator element v of lane l sits in column l % 16 and row row(l, v).
template <typename T> struct Mf;
template <> struct Mf<double> {
    typedef v4d acc;
    static __device__ __forceinline__ acc zero() { return (v4d){0.0, 0.0, 0.0, 0.0}; }
    static __device__ __forceinline__ acc mma(double a, double b, acc c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int v) { return l / 16 + 4 * v; }
    static constexpr int LROW = 1, VROW = 4;   // row(l, v) = LROW (l / 16) + VROW v
};
template <> struct Mf<float> {
    typedef v4f acc;
    static __device__ __forceinline__ acc zero() { return (v4f){0.0f, 0.0f, 0.0f, 0.0f}; }
    static __device__ __forceinline__ acc mma(float a, float b, acc c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int v) { return 4 * (l / 16) + v; }
    static constexpr int LROW = 4, VROW = 1;
};

__device__ __forceinline__ void wave_sync()
{
    // LDS accesses of one wave execute in order; this keeps the compiler from moving them
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// a value that all lanes share, in scalar registers (divisions leave theirs in vector registers)
__device__ __forceinline__ int wave_uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ long long wave_uni(long long v)
{
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)v);
    return (long long)(int)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 | lo;
}
