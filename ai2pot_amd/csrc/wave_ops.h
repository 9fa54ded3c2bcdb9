// Pieces of the kernels that give an atom a wavefront: 16-byte LDS accesses, 16 x 16 x 4 matrix instructions of either
// precision.
#pragma once
#include "a2p_common.h"

namespace a2p {
namespace wave {

// ---- LDS -----------------------------------------------------------------------------------------
__device__ __forceinline__ void lds_load4(const float* p, float (&o)[4])
{
    const float4 v = *reinterpret_cast<const float4*>(p);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
}
__device__ __forceinline__ void lds_load4(const double* p, double (&o)[4])
{
    const double2 v0 = *reinterpret_cast<const double2*>(p);
    const double2 v1 = *reinterpret_cast<const double2*>(p + 2);
    o[0] = v0.x; o[1] = v0.y; o[2] = v1.x; o[3] = v1.y;
}
__device__ __forceinline__ void lds_store4(float* p, float a, float b, float c, float d)
{
    *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
}
__device__ __forceinline__ void lds_store4(double* p, double a, double b, double c, double d)
{
    *reinterpret_cast<double2*>(p) = make_double2(a, b);
    *reinterpret_cast<double2*>(p + 2) = make_double2(c, d);
}
// tile entries: [x y z species]
__device__ __forceinline__ void ent_store(float* p, float x, float y, float z, int w)
{
    *reinterpret_cast<float4*>(p) = make_float4(x, y, z, __int_as_float(w));
}
__device__ __forceinline__ void ent_load(const float* p, float& x, float& y, float& z, int& w)
{
    const float4 v = *reinterpret_cast<const float4*>(p);
    x = v.x; y = v.y; z = v.z; w = __float_as_int(v.w);
}
__device__ __forceinline__ void ent_store(double* p, double x, double y, double z, int w)
{
    *reinterpret_cast<double2*>(p) = make_double2(x, y);
    *reinterpret_cast<double2*>(p + 2) = make_double2(z, __longlong_as_double((long long)w));
}
__device__ __forceinline__ void ent_load(const double* p, double& x, double& y, double& z, int& w)
{
    const double2 v0 = *reinterpret_cast<const double2*>(p);
    const double2 v1 = *reinterpret_cast<const double2*>(p + 2);
    x = v0.x; y = v0.y; z = v1.x; w = (int)__double_as_longlong(v1.y);
}

// ---- D[16][16] += A[16][4] B[4][16] --------------------------------------------------------------------
// Lane l holds A[l % 16][l / 16] and B[l / 16][l % 16]; register v of the result is D[mma_row(v, l)][l % 16].
template <typename T> struct Acc;
template <> struct Acc<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct Acc<double> { typedef double type __attribute__((ext_vector_type(4))); };
__device__ __forceinline__ Acc<float>::type mma(float a, float b, Acc<float>::type c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ Acc<double>::type mma(double a, double b, Acc<double>::type c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
template <typename T>
__device__ __forceinline__ int mma_row(int v, int lane)
{
    return sizeof(T) == 4 ? 4 * (lane >> 4) + v : 4 * v + (lane >> 4);
}

}  // namespace wave
}  // namespace a2p
