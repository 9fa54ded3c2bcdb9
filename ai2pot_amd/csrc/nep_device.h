// Device-side pieces shared by the NEP kernels: argument block, three-body weights, Chebyshev
// radial functions with cosine cutoff, and the 24 real solid harmonics b_lm with their gradients.
// Formulas follow the reference's source/descriptor/nep/include/{basis.h:137-158,300-332,
// 519-530; nep_utilities.h:25-31,100-379}.
#pragma once
#include "a2p_common.h"

namespace a2p {
namespace nepdev {

// three-body weights, nep_utilities.h:25-31 (a double table whose odd entries carry an `f`
// suffix in the reference; kept so that fp64 results agree to the last digits)
__device__ constexpr double kC3B[24] = {
    0.238732414637843, 0.119366207318922f, 0.119366207318922f, 0.099471839432435f,
    0.596831036594608, 0.596831036594608f, 0.149207759148652f, 0.149207759148652f,
    0.139260575205408, 0.104445431404056f, 0.104445431404056f, 1.044454314040563f,
    1.044454314040563, 0.174075719006761f, 0.174075719006761f, 0.011190581936149f,
    0.223811638722978, 0.223811638722978f, 0.111905819361489f, 0.111905819361489f,
    1.566681471060845, 1.566681471060845f, 0.195835183882606f, 0.195835183882606f};

// weights of the four- and five-body invariants of the extension (source/descriptor/ace/include/nep_descriptor.h:43-54;
// the reference never evaluates them)
__device__ constexpr double kC4B[5] = {-0.007499480826664, -0.134990654879954, 0.067495327439977, 0.404971964639861,
                                       -0.809943929279723};
__device__ constexpr double kC5B[3] = {0.026596810706114, 0.053193621412227, 0.026596810706114};

template <typename T>
struct NepArgs {
    int K, n_r, n_a, l_max, H, ntypes, D;
    const T *coeffs, *w0, *b0, *w1, *bias, *q_scaler;
    T rr, ra;
    int B, P, U, nghost, nblocks;
    const int *binum, *bilist, *bnumneigh, *bfirstneigh;
    const T* brcs;
    const int* btypes;
    T* force;        // [B, P+nghost, 3] or null
    T* pair_g;       // [B*P, U, 3] or null (needed when force != null)
    T* desc;         // [B, P, D] or null
    double* partial; // energy and virial per workgroup (ev_partial)
    int* status;
    int want_virial;
    int w_in_lds;    // network weights staged in LDS (else read from global memory)
    // optional: places of the pairs in their targets' reduction segments, kept by the caller from
    // call to call while the list stays the same: brank[B, P, U], and bincoming[B, P+nghost] pairs
    // naming each atom.  ranks_valid = 0: this call claims the places and records them there;
    // 1: it uses what an earlier call recorded.
    int* brank;
    int* bincoming;
    int ranks_valid;
    int mb4 = 0, mb5 = 0;   // extension (generic kernel only): four- / five-body invariant per angular channel
};

// What the kernels that store a pair derivative straight into its target's segment know of the segments (PairCsr).
struct SegArgs {
    int* cursor;   // [B * NF] entries claimed so far in each target's reduction segment, or null (no forces)
    int cap;       // capacity of a segment
    int spare;     // entry that takes what overflows a segment
    int mark;      // own sums are marked in the cursors (PairCsr)
};

// The model's tables in LDS, staged by the workgroup: w0 in rows of WROW values, the coefficients of a species pair in rows of
// NB * KC + CPAD.  The first W0 and four values of every thread, four to a load, are all on their way before one is stored, behind
// them whatever `early` asks for.  No load stands behind a branch: a thread beyond the end takes the last four again.
template <int KC, int NB, int D, int WROW, int CPAD, int W0, typename T, typename Args, typename Lds, typename Early>
__device__ __forceinline__ void stage_tables(Args& a, const Lds& L, int tid, int nthreads, Early early)
{
    constexpr int W4 = W0 / 4, NC = NB * KC;
    static_assert(W0 % 4 == 0 && D >= 4 && NC >= 4, "four values cross one end of a row at most");
    struct alignas(sizeof(T)) Four { T v[4]; };
    const int nt = a.ntypes, H = a.H, nw0 = nt * H * D, nc = nt * nt * NC, nh = nt * H;
    auto take = [&](const T* p, int n, int u) __attribute__((always_inline)) {
        return *reinterpret_cast<const Four*>(p + min((tid + u * nthreads) * 4, n - 4));
    };
    auto put = [&](T* dst, auto row, auto pad, int n, int u, const Four& o) __attribute__((always_inline)) {
        constexpr int ROW = decltype(row)::value, PAD = decltype(pad)::value;
        const int i = min((tid + u * nthreads) * 4, n - 4), r = i / ROW, c = i - r * ROW;
#pragma unroll
        for (int k = 0; k < 4; k++) dst[i + k + (r + (c + k >= ROW ? 1 : 0)) * PAD] = o.v[k];
    };
    auto put_w0 = [&](int u, const Four& o) __attribute__((always_inline)) {
        put(L.w0, std::integral_constant<int, D>{}, std::integral_constant<int, WROW - D>{}, nw0, u, o);
    };
    auto put_coef = [&](int u, const Four& o) __attribute__((always_inline)) {
        put(L.coef, std::integral_constant<int, NC>{}, std::integral_constant<int, CPAD>{}, nc, u, o);
    };
    const Four c0 = take(a.coeffs, nc, 0);
    Four w0[W4];
#pragma unroll
    for (int u = 0; u < W4; u++) w0[u] = take(a.w0, nw0, u);
    const T b0 = a.b0[min(tid, nh - 1)], w1 = a.w1[min(tid, nh - 1)], qs = a.q_scaler[min(tid, D - 1)];
    early();
    put_coef(0, c0);
#pragma unroll
    for (int u = 0; u < W4; u++)
        if (u * nthreads * 4 < nw0) put_w0(u, w0[u]);
    if (tid < nh) { L.b0[tid] = b0; L.w1[tid] = w1; }
    if (tid < WROW) L.qs[tid] = tid < D ? (T)1 / qs : (T)0;
    for (int u = 1; (tid + u * nthreads) * 4 < nc; u++) put_coef(u, take(a.coeffs, nc, u));
    for (int u = W4; (tid + u * nthreads) * 4 < nw0; u++) put_w0(u, take(a.w0, nw0, u));
    for (int i = tid + nthreads; i < nh; i += nthreads) { L.b0[i] = a.b0[i]; L.w1[i] = a.w1[i]; }
}

// r and 1 / r from r^2: the estimate of 1 / r and a Newton step for each, a third of the operations of square root and
// division, and no further from fp64 (forces 4.65e-7 with either).  Adjoint kernel of 1,048,576 atoms 631 -> 620 us, gather
// kernel, which waits for memory, 334 -> 331.  r^2 = 0 gives NaN, as 0 / 0 does; MIN keeps it from that.
template <bool MIN>
__device__ __forceinline__ float length(float d2, float& rinv)
{
    if (MIN) d2 = d2 < 1e-30f ? 1e-30f : d2;                    // (NaN stays)
    const float y = __builtin_amdgcn_rsqf(d2), r0 = d2 * y;
    const float r = r0 + (d2 - r0 * r0) * (0.5f * y);
    rinv = y + y * (1.0f - r * y);
    return r;
}
template <bool MIN>
__device__ __forceinline__ double length(double d2, double& rinv)
{
    const double r = sqrt(d2);
    rinv = 1.0 / r;
    return r;
}

// sin(pi u / 2) on [-1, 1]: u + u p(u^2), p + 1 the polynomial of least relative error (5e-9; 2.6e-19) for sin(pi sqrt(y) / 2) / sqrt(y)
__device__ __forceinline__ float quarter_sine(float u)
{
    const float y = u * u;
    float p = 0.000151485130733f;
    p = p * y - 0.0046737666124f;
    p = p * y + 0.0796896789478f;
    p = p * y - 0.6459637106f;
    p = p * y + 0.57079631845f;
    return u * p + u;
}
__device__ __forceinline__ double quarter_sine(double u)
{
    const double y = u * u;
    double p = 5.8706109783952470938e-12;
    p = p * y - 6.684321720453320249e-10;
    p = p * y + 5.6921348727149338656e-8;
    p = p * y - 3.5988430072086468421e-6;
    p = p * y + 0.00016044118470682204322;
    p = p * y - 0.0046817541353026425916;
    p = p * y + 0.079692626246165435628;
    p = p * y - 0.64596409750624619109;
    p = p * y + 0.5707963267948966188;
    return u * p + u;
}
// cos(pi t) and sin(pi t) for t in [0, 1] (a dummy neighbour's larger t is taken for 1).  The library's pair reduces any
// argument first: 660 instead of 631 us for the adjoint kernel of 1,048,576 atoms, 96 instead of 90 for a wavefront per atom at
// 20,011; forces against fp64 differ by 4.7e-7 with either.
template <typename T>
__device__ __forceinline__ void cos_sin_pi(T t, T& c, T& s)
{
    t = min(t, (T)1);
    const T m = min(t, (T)1 - t);
    c = quarter_sine((T)1 - (t + t));
    s = quarter_sine(m + m);
}
// tanh: below 0.7 x + x^3 p(x^2), p of least relative error (1.6e-8), else 1 - 2 / (exp(2 |x|) + 1) by the chip's exp2 and
// reciprocal; both and a choice, 20 operations.  The library's takes a branch for either side and an argument of exp in two parts,
// 35 operations of which a wavefront with both kinds of argument issues all.  Error over every float, in units of the last place, largest
// and mean, against the library's: below 0.35 0.74 and 0.58, to 0.7 0.91 and 1.41 (mean 0.269 and 0.273), to 1 1.61 and 1.18 (0.373 and 0.329), to
// 2 1.35 and 1.00, beyond alike; that of forces against fp64 8.83e-7 with it, 8.86e-7 before (120,000 atoms, with the other changes of that step),
// energies and virials alike.
__device__ __forceinline__ float tanh_t(float x)
{
    const float a = fabsf(x), y = a * a;
    float p = -0.00513857882f;
    p = p * y + 0.0200918801f;
    p = p * y - 0.0535588302f;
    p = p * y + 0.133291095f;
    p = p * y - 0.333331913f;
    const float small = a * y * p + a;
    const float large = 1.0f - 2.0f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(a * 2.88539008f) + 1.0f);
    return copysignf(a < 0.7f ? small : large, x);
}
__device__ __forceinline__ double tanh_t(double x) { return tanh(x); }
__device__ __forceinline__ float sqrt_t(float x) { return sqrtf(x); }
__device__ __forceinline__ double sqrt_t(double x) { return sqrt(x); }

// f_k(r) = 1/2 (T_k(x)+1) fc(r), x = 2 (r/rc - 1)^2 - 1, fc = 1/2 (1 + cos(pi r/rc));
// basis.h:137-158, 300-332, 519-530.  Caller guarantees r <= rc.
template <typename T, int KC, bool DER>
__device__ __forceinline__ void radial_basis(T r, T rc_inv, int K, T (&f)[KC], T (&df)[KC])
{
    const T t = r * rc_inv;
    const T xr = t - (T)1;
    const T x = (T)2 * xr * xr - (T)1, x2 = x + x;
    T cs, sn;
    cos_sin_pi(t, cs, sn);
    const T h = (T)0.25 * cs + (T)0.25;                                           // 1/2 fc
    const T dh = (T)(-0.25 * 3.14159265358979323846) * rc_inv * sn;               // 1/2 fc'
    const T w = h * ((T)4 * rc_inv * xr);                                         // 1/2 fc dx/dr
    T t0 = (T)1, t1 = x, d0 = (T)0, d1 = (T)1;
#pragma unroll
    for (int k = 0; k < KC; k++) {
        T tv = k == 0 ? t0 : t1, dv = k == 0 ? d0 : d1;
        if (k >= 2) {
            tv = x2 * t1 - t0;
            dv = (T)2 * t1 + (x2 * d1 - d0);
            t0 = t1; t1 = tv; d0 = d1; d1 = dv;
        }
        f[k] = (k < K) ? (k == 0 ? h + h : h * tv + h) : (T)0;
        if (DER) df[k] = (k < K) ? (k == 0 ? dh + dh : (dh * tv + dh) + w * dv) : (T)0;
    }
}

// h = fc / 2 and T_k, so that f_k = h (T_k + 1): for sums of the functions themselves, sum h T_k + sum h.
template <typename T, int KC>
__device__ __forceinline__ T radial_terms(T r, T rc_inv, T (&t)[KC])
{
    const T u = r * rc_inv;
    const T xr = u - (T)1;
    const T x = (T)2 * xr * xr - (T)1, x2 = x + x;
    T cs, sn;
    cos_sin_pi(u, cs, sn);
    t[0] = (T)1; t[1] = x;
#pragma unroll
    for (int k = 2; k < KC; k++) t[k] = x2 * t[k - 1] - t[k - 2];
    return (T)0.25 * cs + (T)0.25;
}

// b_lm(u) for unit vector u, flat index l*l-1+mp (nep_utilities.h:110-203 with r = 1).  With C_m + i S_m = (x + i y)^m the pair
// of mp = 2 m - 1, 2 m is C_m and S_m times a polynomial in z of degree l - m: 37 operations for the 24 of l <= 4.
template <typename T, int LC>
__device__ __forceinline__ void blm_values(T x, T y, T z, T (&b)[LC * LC + 2 * LC])
{
    const T z2 = z * z, c2 = x * x - y * y, s2 = (x + x) * y;
    if (LC >= 1) { b[0] = z; b[1] = x; b[2] = y; }
    if (LC >= 2) {
        b[3] = (T)3 * z2 - (T)1; b[4] = x * z; b[5] = y * z; b[6] = c2; b[7] = s2;
    }
    const T c3 = x * c2 - y * s2, s3 = x * s2 + y * c2;
    if (LC >= 3) {
        const T p1 = (T)5 * z2 - (T)1;
        b[8] = (p1 - (T)2) * z; b[9] = p1 * x; b[10] = p1 * y; b[11] = c2 * z; b[12] = s2 * z; b[13] = c3; b[14] = s3;
    }
    if (LC >= 4) {
        const T p1 = ((T)7 * z2 - (T)3) * z, p2 = (T)7 * z2 - (T)1;
        b[15] = ((T)35 * z2 - (T)30) * z2 + (T)3;
        b[16] = p1 * x; b[17] = p1 * y; b[18] = p2 * c2; b[19] = p2 * s2; b[20] = c3 * z; b[21] = s3 * z;
        b[22] = c2 * c2 - s2 * s2; b[23] = (c2 + c2) * s2;
    }
}

// Gradient of sum_lm a[lm] b_lm, the b_lm as blm_values forms them.  They are the solid harmonics on the unit sphere only, so
// what counts is the part across u (across()).  With P_m(z), Q_m(z) the sums of the a[lm] that go with C_m and S_m it is
//   x: sum m (C_{m-1} P_m + S_{m-1} Q_m),  y: sum m (C_{m-1} Q_m - S_{m-1} P_m),  z: sum C_m P_m' + S_m Q_m'
// Some 60 operations; the gradients of the homogeneous polynomials (nep_utilities.h:206-379) taken one by one are 150.
template <typename T, int LC>
__device__ __forceinline__ void blm_gradient(T x, T y, T z, const T (&a)[LC * LC + 2 * LC], T& wx, T& wy, T& wz)
{
    const T z2 = z * z, c2 = x * x - y * y, s2 = (x + x) * y;
    const T c3 = x * c2 - y * s2, s3 = x * s2 + y * c2;
    T P1 = a[1], Q1 = a[2];                                   // m = 1
    wz = a[0];
    T dP1 = (T)0, dQ1 = (T)0;
    if (LC >= 2) {
        P1 += a[4] * z; Q1 += a[5] * z;
        wz += a[3] * ((T)6 * z);
        dP1 = a[4]; dQ1 = a[5];
    }
    if (LC >= 3) {
        const T p1 = (T)5 * z2 - (T)1, d1 = (T)10 * z;
        P1 += a[9] * p1; Q1 += a[10] * p1;
        wz += a[8] * ((T)15 * z2 - (T)3);
        dP1 += a[9] * d1; dQ1 += a[10] * d1;
    }
    if (LC >= 4) {
        const T p1 = ((T)7 * z2 - (T)3) * z, d1 = (T)21 * z2 - (T)3;
        P1 += a[16] * p1; Q1 += a[17] * p1;
        wz += a[15] * (((T)140 * z2 - (T)60) * z);
        dP1 += a[16] * d1; dQ1 += a[17] * d1;
    }
    wx = P1; wy = Q1;
    if (LC >= 2) wz += x * dP1 + y * dQ1;
    if (LC >= 2) {
        T P2 = a[6], Q2 = a[7];
        if (LC >= 3) { P2 += a[11] * z; Q2 += a[12] * z; }
        if (LC >= 4) { const T p2 = (T)7 * z2 - (T)1; P2 += a[18] * p2; Q2 += a[19] * p2; }
        const T x2 = x + x, y2 = y + y;
        wx += x2 * P2 + y2 * Q2;
        wy += x2 * Q2 - y2 * P2;
    }
    if (LC >= 3) {
        T P3 = a[13], Q3 = a[14], dP2 = a[11], dQ2 = a[12];
        if (LC >= 4) {
            const T d2 = (T)14 * z;
            P3 += a[20] * z; Q3 += a[21] * z;
            dP2 += a[18] * d2; dQ2 += a[19] * d2;
        }
        wz += c2 * dP2 + s2 * dQ2;
        const T c23 = (T)3 * c2, s23 = (T)3 * s2;
        wx += c23 * P3 + s23 * Q3;
        wy += c23 * Q3 - s23 * P3;
    }
    if (LC >= 4) {
        wz += c3 * a[20] + s3 * a[21];
        const T c34 = (T)4 * c3, s34 = (T)4 * s3;
        wx += c34 * a[22] + s34 * a[23];
        wy += c34 * a[23] - s34 * a[22];
    }
}

// The compiler forms what depends on x from here on anew, instead of holding what blm_values has formed of it already (the
// kernels whose registers are full).
template <typename T>
__device__ __forceinline__ void forget(T& x, T& y, T& z) { asm volatile("" : "+v"(x), "+v"(y), "+v"(z)); }

// Derivative along the pair vector of a function g(r) b(u): `along` = g' b for its length, w = g grad b for its direction, of
// which the part across u counts: along u + (w - (w . u) u) / r.
template <typename T>
__device__ __forceinline__ void pair_gradient(T along, T wx, T wy, T wz, T ux, T uy, T uz, T rinv, T& gx, T& gy, T& gz)
{
    const T s = along - (wx * ux + wy * uy + wz * uz) * rinv;
    gx = s * ux + wx * rinv;
    gy = s * uy + wy * rinv;
    gz = s * uz + wz * rinv;
}

// d[lm] = w . grad b_lm(u): the directional derivative of every homogeneous polynomial b_lm along
// w, evaluated on the unit sphere (the gradients of nep_utilities.h:206-379 with r = 1)
template <typename T, int LC>
__device__ __forceinline__ void blm_dir_derivs(T x, T y, T z, T wx, T wy, T wz, T (&d)[LC * LC + 2 * LC])
{
    const T x2 = x * x, y2 = y * y, z2 = z * z;
    const T xy = x * y, xz = x * z, yz = y * z;
    if (LC >= 1) { d[0] = wz; d[1] = wx; d[2] = wy; }
    if (LC >= 2) {
        d[3] = (T)-2 * x * wx + (T)-2 * y * wy + (T)4 * z * wz;
        d[4] = z * wx + x * wz;
        d[5] = z * wy + y * wz;
        d[6] = (T)2 * x * wx - (T)2 * y * wy;
        d[7] = (T)2 * y * wx + (T)2 * x * wy;
    }
    if (LC >= 3) {
        const T c = (T)5 * z2 - (T)1;
        d[8] = (T)-6 * xz * wx + (T)-6 * yz * wy + ((T)9 * z2 - (T)3) * wz;
        d[9] = (c - (T)2 * x2) * wx + (T)-2 * xy * wy + (T)8 * xz * wz;
        d[10] = (T)-2 * xy * wx + (c - (T)2 * y2) * wy + (T)8 * yz * wz;
        d[11] = (T)2 * xz * wx + (T)-2 * yz * wy + (x2 - y2) * wz;
        d[12] = (T)2 * yz * wx + (T)2 * xz * wy + (T)2 * xy * wz;
        d[13] = (T)3 * (x2 - y2) * wx + (T)-6 * xy * wy;
        d[14] = (T)6 * xy * wx + (T)3 * (x2 - y2) * wy;
    }
    if (LC >= 4) {
        const T z3 = z2 * z, x3 = x2 * x, y3 = y2 * y;
        const T c73 = (T)7 * z3 - (T)3 * z;
        d[15] = ((T)-60 * x * z2 + (T)12 * x) * wx + ((T)-60 * y * z2 + (T)12 * y) * wy +
                ((T)80 * z3 - (T)48 * z) * wz;
        d[16] = ((T)-6 * x2 * z + c73) * wx + ((T)-6 * xy * z) * wy + ((T)15 * x * z2 - (T)3 * x) * wz;
        d[17] = ((T)-6 * xy * z) * wx + ((T)-6 * y2 * z + c73) * wy + ((T)15 * y * z2 - (T)3 * y) * wz;
        d[18] = ((T)-2 * x3 + (T)2 * x * y2 + (T)14 * x * z2 - (T)2 * x) * wx +
                ((T)-2 * x2 * y + (T)2 * y3 - (T)14 * y * z2 + (T)2 * y) * wy + ((T)12 * z * (x2 - y2)) * wz;
        d[19] = ((T)-4 * x2 * y + (T)14 * y * z2 - (T)2 * y) * wx +
                ((T)-4 * x * y2 + (T)14 * x * z2 - (T)2 * x) * wy + ((T)24 * xy * z) * wz;
        d[20] = ((T)3 * (x2 - y2) * z) * wx + ((T)-6 * xy * z) * wy + ((x2 - (T)3 * y2) * x) * wz;
        d[21] = ((T)6 * xy * z) * wx + ((T)3 * (x2 - y2) * z) * wy + (((T)3 * x2 - y2) * y) * wz;
        d[22] = ((T)4 * x3 - (T)12 * x * y2) * wx + ((T)4 * y3 - (T)12 * x2 * y) * wy;
        d[23] = ((T)12 * x2 * y - (T)4 * y3) * wx + ((T)4 * x3 - (T)12 * x * y2) * wy;
    }
}

}  // namespace nepdev

// The staged kernel for the common model shape (nep_staged.hip).  staged_supported() tells
// whether it applies; nep_staged_run() performs forces' zero-fill, pair counting, the kernel and
// the pair reduction, whose launch also sums the workgroup partial sums of a.partial (a.nblocks
// is set by staged_nblocks()) into etot and virial.
// Four atoms per wavefront (nep_quad.hip); also l_max 3, and any number of species whose tables fit the LDS.
template <typename T>
bool nep_quad_supported(const nepdev::NepArgs<T>& a);
template <typename T>
int nep_quad_nblocks(const nepdev::NepArgs<T>& a);
template <typename T>
int nep_quad_run(const nepdev::NepArgs<T>& a, T* etot, T* virial, hipStream_t stream);
// A wavefront per atom (nep_wave.hip), the same shapes, for batches too small to give every SIMD a few wavefronts.
template <typename T>
bool nep_wave_supported(const nepdev::NepArgs<T>& a, size_t* lds_bytes);
int nep_wave_nblocks(int P, int B);
template <typename T>
int nep_wave_run(const nepdev::NepArgs<T>& a, size_t lds_bytes, T* etot, T* virial, hipStream_t stream);

template <typename T>
bool nep_staged_supported(const nepdev::NepArgs<T>& a, size_t* lds_bytes);
int nep_staged_nblocks(int P);
template <typename T>
int nep_staged_run(const nepdev::NepArgs<T>& a, size_t lds_bytes, T* etot, T* virial, hipStream_t stream);

}  // namespace a2p
