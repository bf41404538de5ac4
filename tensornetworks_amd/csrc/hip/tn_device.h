// tn_device.h -- device helpers shared by the kernel files: scalar conversions,
// bfloat16 splitting and the matrix-instruction traits.
#pragma once
#include <type_traits>

#include "tn_kernels.h"

namespace tn {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// scalar conversions
__device__ __forceinline__ bf16 f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (bf16)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
    return (bf16)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16 h) { return __uint_as_float(((uint32_t)h) << 16); }

template <typename T> __device__ __forceinline__ T cvt_from_d(double v);
template <> __device__ __forceinline__ double cvt_from_d<double>(double v) { return v; }
template <> __device__ __forceinline__ float cvt_from_d<float>(double v) { return (float)v; }
template <> __device__ __forceinline__ bf16 cvt_from_d<bf16>(double v) { return f2bf((float)v); }
template <typename T> __device__ __forceinline__ T cvt_from_f(float v);
template <> __device__ __forceinline__ double cvt_from_f<double>(float v) { return (double)v; }
template <> __device__ __forceinline__ float cvt_from_f<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 cvt_from_f<bf16>(float v) { return f2bf(v); }
__device__ __forceinline__ double to_d(double v) { return v; }
__device__ __forceinline__ double to_d(float v) { return (double)v; }
__device__ __forceinline__ double to_d(bf16 v) { return (double)bf2f(v); }
__device__ __forceinline__ float to_f(double v) { return (float)v; }
__device__ __forceinline__ float to_f(float v) { return v; }
__device__ __forceinline__ float to_f(bf16 v) { return bf2f(v); }
template <typename A, typename T> __device__ __forceinline__ A to_acc(T v)
{
    if constexpr (std::is_same<A, double>::value) return to_d(v);
    else return to_f(v);
}

// v = h0 + h1 + h2 + O(2^-24 |v|): each bfloat16 piece is the rounding of what
// the previous ones leave (the differences are exact in the wider type)
__device__ __forceinline__ void split3_val(double v, bf16& h0, bf16& h1, bf16& h2)
{
    h0 = f2bf((float)v);
    double r = v - (double)bf2f(h0);
    h1 = f2bf((float)r);
    r -= (double)bf2f(h1);
    h2 = f2bf((float)r);
}
__device__ __forceinline__ void split3_val(float v, bf16& h0, bf16& h1, bf16& h2)
{
    h0 = f2bf(v);
    float r = v - bf2f(h0);
    h1 = f2bf(r);
    r -= bf2f(h1);
    h2 = f2bf(r);
}

// ---------------------------------------------------------------------------
// MFMA traits: 16x16 output block per wave instruction
//   A frag: lane l holds A[l%16][kbase + (l/16)*KPL + 0..KPL-1]
//   B frag: lane l holds B[kbase + (l/16)*KPL + ..][l%16]
//          (KPL = 1 for f64 and f32)
//   C    : lane l holds C[row(l, r)][l%16], r = 0..3, with
//          row = (l/16)*4 + r for the f32/bf16 instructions and
//          row = (l/16) + 4*r for f64 (measured on gfx950 with a one-wave probe)
template <typename TI> struct MT;
template <> struct MT<double> {
    static __device__ __forceinline__ int crow(int lane, int r) { return (lane >> 4) + 4 * r; }
    typedef v4d acc_t;
};
template <> struct MT<float> {
    static __device__ __forceinline__ int crow(int lane, int r) { return (lane >> 4) * 4 + r; }
    typedef v4f acc_t;
};
template <> struct MT<bf16> {
    static constexpr int KPL = 8, MK = 32, VEC = 8, PAD = 8;
    static __device__ __forceinline__ int crow(int lane, int r) { return (lane >> 4) * 4 + r; }
    typedef v8bf frag_t;
    typedef v4f acc_t;
};

__device__ __forceinline__ v4d mma(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4f mma(float a, float b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4f mma(v8bf a, v8bf b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

}  // namespace tn
