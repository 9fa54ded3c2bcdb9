// Pieces of the kernels that give an atom a wavefront: sums across lanes, 16-byte LDS accesses, 16 x 16 x 4 matrix
// instructions of either precision.
#pragma once
#include "a2p_common.h"

namespace a2p {
namespace wave {

// ---- cross-lane sums -----------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ int dpp_move(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) { return __int_as_float(dpp_move<CTRL>(__float_as_int(v))); }
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = dpp_move<CTRL>((int)(b & 0xffffffffll));
    const int hi = dpp_move<CTRL>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// v[lane] + v[lane ^ 16] and v[lane] + v[lane ^ 32]: the swap of a value with its copy leaves one half's rows in the
// first and the other half's in the second
template <int ROWS>
__device__ __forceinline__ void swap_rows(unsigned v, unsigned& a, unsigned& b)
{
    const auto r = ROWS == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false)
                              : __builtin_amdgcn_permlane32_swap(v, v, false, false);
    a = r[0]; b = r[1];
}
template <int ROWS>
__device__ __forceinline__ float add_rows(float v)
{
    unsigned a, b;
    swap_rows<ROWS>(__float_as_uint(v), a, b);
    return __uint_as_float(a) + __uint_as_float(b);
}
template <int ROWS>
__device__ __forceinline__ double add_rows(double v)
{
    const unsigned long long w = (unsigned long long)__double_as_longlong(v);
    unsigned al, bl, ah, bh;
    swap_rows<ROWS>((unsigned)w, al, bl);
    swap_rows<ROWS>((unsigned)(w >> 32), ah, bh);
    return __longlong_as_double((long long)((unsigned long long)ah << 32 | al)) +
           __longlong_as_double((long long)((unsigned long long)bh << 32 | bl));
}
template <typename T>
__device__ __forceinline__ T quad_sum(T v)          // the four lanes of a quad
{
    v += dpp_move<0xB1>(v);    // quad_perm [1,0,3,2]
    v += dpp_move<0x4E>(v);    // quad_perm [2,3,0,1]
    return v;
}
template <typename T>
__device__ __forceinline__ T sum_over_quads(T v)    // the sixteen lanes with the same place in their quad
{
    v += dpp_move<0x124>(v);   // row_ror:4
    v += dpp_move<0x128>(v);   // row_ror:8
    v = add_rows<16>(v);
    return add_rows<32>(v);
}
template <typename T>
__device__ __forceinline__ T all_sum(T v) { return sum_over_quads(quad_sum(v)); }

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
