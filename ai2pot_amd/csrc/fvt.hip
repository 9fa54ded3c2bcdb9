// Short-range force and virial from per-pair derivatives dE_i/dr_ij, and their
// vector-Jacobian products, for gfx950.
//
//   force : F[c] = sum_s g[ii,s] - sum over pairs whose neighbour is c of g   (c = ilist[ii])
//           reference: source/fvt/include/force_sr.h:50-84.  a2p::pair_reduce: the own-row sum is formed by the
//           wavefront that deals out the row's places (no floating-point atomics).
//   virial: V[a,b] = - sum_{ii,s} g[ii,s,a] r[ii,s,b]          source/fvt/include/virial_sr.h:24-51
// The reference materialises dense Jacobians [(nlocal+nghost)*3, nlocal*umax] and
// [9, nlocal*umax] (src/force_sr_op.cc:44, src/virial_sr_op.cc:31-32) and multiplies by them
// in backward; the Jacobian entries are +-1, -r and -g, so the products are written directly:
//   dL/dg[ii,s,k]  = gF[c,k] - gF[j,k]                         (force_sr.h:99-124)
//   dL/dg[ii,s,a]  = - sum_b gV[a,b] r[ii,s,b],   dL/dr[ii,s,b] = - sum_a gV[a,b] g[ii,s,a]
#include "a2p_common.h"

#include <mutex>
#include <vector>

namespace a2p {
namespace {

// Rows of three values to a slot, a lane to a slot.  Many rows in fp64 are bound by what they write: 64 slots' values pass through the
// wavefront's LDS (WHOLE), so that each store writes whole lines, where three stores would write every third value each.  Few are
// bound by the wavefront's chain, which that makes longer, and so are rows in fp32, whose lines the L2 puts together as they come.
// Kernels without and with it, us, force and virial: fp64, 200 slots, 600 rows 3.40 and 3.52, 4.04 and 3.80; 900 3.68 and 3.60, 4.64 and 4.08;
// 2,000 5.3 and 4.8, 7.4 and 5.7; 4,000 7.6 and 6.4, 10.6 and 8.6; 32,000 43.7 and 39.4, 92.6 and 60.2; 64 slots, 1,400 rows 3.28 and 3.40, 3.76 and
// 3.60; 2,400 3.80 and 3.76, 4.64 and 4.40; 32,000 15.3 and 15.2, 23.6 and 23.9.  fp32, 200 slots, 2,000 rows 3.56 and 3.72, 4.28 and 4.68;
// 4,000 5.0 and 4.8, 6.0 and 6.1; 32,000 18.6 and 19.0, 30.8 and 35.3; 64 slots, 4,000 rows 3.3 and 3.6, 3.7 and 4.1.
constexpr long long FVT_WHOLE = 1 << 17;                 // slots, fp64
template <typename T>
constexpr bool whole_lines() { return sizeof(T) == 8; }
template <typename T, bool WHOLE>
__device__ __forceinline__ void store_slots(T* __restrict__ out, T* sh, int lane, int n, T v0, T v1, T v2)
{
    if (!WHOLE) {
        if (lane < n) { out[lane * 3] = v0; out[lane * 3 + 1] = v1; out[lane * 3 + 2] = v2; }
        return;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    sh[lane * 3] = v0; sh[lane * 3 + 1] = v1; sh[lane * 3 + 2] = v2;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int i = 0; i < 3; i++)
        if (lane + i * 64 < n * 3) out[lane + i * 64] = sh[lane + i * 64];
}

// zeros behind a row's last neighbour: slots from .. U
template <typename T>
__device__ __forceinline__ void pad_slots(T* __restrict__ out, int lane, int from, int U)
{
    for (int e = from * 3 + lane; e < U * 3; e += 64) out[e] = (T)0;
}

template <typename T, bool WHOLE>
__global__ void __launch_bounds__(256)
force_bwd_kernel(T* __restrict__ gout, const T* __restrict__ gF, int B, int P, int U, int NF,
                 const int* __restrict__ binum, const int* __restrict__ bilist,
                 const int* __restrict__ bnumneigh, const int* __restrict__ bfirstneigh)
{
    __shared__ T sh[4][WHOLE ? 64 * 3 : 1];
    const int row = (blockIdx.x * 256 + threadIdx.x) >> 6, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (row >= B * P) return;
    const int b = row / P, ii = row - b * P;
    int nn = 0, c = 0;
    if (ii < binum[b]) {
        nn = min(bnumneigh[row], U);
        c = bilist[row];
        if ((unsigned)c >= (unsigned)NF) nn = 0;
    }
    T* out = gout + (size_t)row * U * 3;
    const T* fc = gF + ((size_t)b * NF + c) * 3;
    const int* first = bfirstneigh + (size_t)row * U;
    const int own = WHOLE ? max(min((nn + 63) / 64 * 64, U), 0) : U;
    pad_slots(out, lane, own, U);
    for (int s0 = 0; s0 < own; s0 += 64) {
        const int s = s0 + lane;
        T v0 = 0, v1 = 0, v2 = 0;
        if (s < nn) {
            const int j = first[s];
            if ((unsigned)j < (unsigned)NF) {
                const T* fj = gF + ((size_t)b * NF + j) * 3;
                v0 = fc[0] - fj[0]; v1 = fc[1] - fj[1]; v2 = fc[2] - fj[2];
            }
        }
        store_slots<T, WHOLE>(out + s0 * 3, sh[wave], lane, min(U - s0, 64), v0, v1, v2);
    }
}

// one wavefront per row -> 9 partial sums per row (fp64), reduced by finish_partials; too_long (a word of host memory)
// is set when a row claims more than U neighbours
template <typename T>
__global__ void __launch_bounds__(256)
virial_rows_kernel(double* __restrict__ partial, const T* __restrict__ g, const T* __restrict__ r, int B,
                   int P, int U, const int* __restrict__ bnumneigh, int* too_long)
{
    const int row = (blockIdx.x * 256 + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (row >= B * P) return;
    const int nn = min(bnumneigh[row], U);
    if (too_long && lane == 0 && bnumneigh[row] > U) __hip_atomic_store(too_long, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    const T* gr = g + (size_t)row * U * 3;
    const T* rr = r + (size_t)row * U * 3;
    double v[9];
#pragma unroll
    for (int q = 0; q < 9; q++) v[q] = 0.0;
    for (int s = lane; s < nn; s += 64) {
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int c = 0; c < 3; c++) v[a * 3 + c] -= (double)gr[s * 3 + a] * (double)rr[s * 3 + c];
    }
#pragma unroll
    for (int q = 0; q < 9; q++) {
        const double t = wave_sum(v[q]);
        if (lane == 0) partial[(size_t)row * 9 + q] = t;
    }
}

template <typename T, bool WHOLE>
__global__ void __launch_bounds__(256)
virial_bwd_kernel(T* __restrict__ gg, T* __restrict__ gr, const T* __restrict__ gV, const T* __restrict__ g,
                  const T* __restrict__ r, int B, int P, int U, const int* __restrict__ bnumneigh)
{
    __shared__ T sh[4][2][WHOLE ? 64 * 3 : 1];
    const int row = (blockIdx.x * 256 + threadIdx.x) >> 6, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (row >= B * P) return;
    const int b = row / P;
    const int nn = min(bnumneigh[row], U);
    T m[9];
#pragma unroll
    for (int q = 0; q < 9; q++) m[q] = gV[b * 9 + q];
    const size_t base = (size_t)row * U * 3;
    const int own = WHOLE ? max(min((nn + 63) / 64 * 64, U), 0) : U;
    if (gg) pad_slots(gg + base, lane, own, U);
    if (gr) pad_slots(gr + base, lane, own, U);
    for (int s0 = 0; s0 < own; s0 += 64) {
        const int s = s0 + lane, n = min(U - s0, 64);
        T og[3] = {0, 0, 0}, orr[3] = {0, 0, 0};
        if (s < nn) {
            const T g0 = g[base + s * 3], g1 = g[base + s * 3 + 1], g2 = g[base + s * 3 + 2];
            const T r0 = r[base + s * 3], r1 = r[base + s * 3 + 1], r2 = r[base + s * 3 + 2];
#pragma unroll
            for (int a = 0; a < 3; a++) og[a] = -(m[a * 3] * r0 + m[a * 3 + 1] * r1 + m[a * 3 + 2] * r2);
#pragma unroll
            for (int c = 0; c < 3; c++) orr[c] = -(m[c] * g0 + m[3 + c] * g1 + m[6 + c] * g2);
        }
        if (gg) store_slots<T, WHOLE>(gg + base + s0 * 3, sh[wave][0], lane, n, og[0], og[1], og[2]);
        if (gr) store_slots<T, WHOLE>(gr + base + s0 * 3, sh[wave][1], lane, n, orr[0], orr[1], orr[2]);
    }
}

int check_shape(int B, int P, int U, int nghost)
{
    A2P_REQUIRE(B >= 0 && P >= 0 && U >= 1 && nghost >= 0, A2P_ERR_INVALID, "fvt: bad shape");
    A2P_REQUIRE((long long)B * P * U < (1ll << 31), A2P_ERR_INVALID, "fvt: batch too large");
    return A2P_OK;
}

template <typename T>
int force_fwd(int B, int P, int U, int nghost, const int* binum, const int* bilist, const int* bnumneigh,
              const int* bfirstneigh, const T* dei, T* force, hipStream_t stream)
{
    int rc = check_shape(B, P, U, nghost);
    if (rc) return rc;
    A2P_REQUIRE(binum && bilist && bnumneigh && bfirstneigh && dei && force, A2P_ERR_INVALID,
                "fvt force: null pointer");
    if (B == 0 || P == 0) return A2P_OK;
    return pair_reduce<T>(force, dei, B, P, U, nghost, binum, bilist, bnumneigh, bfirstneigh, true, stream);
}

template <typename T>
int force_bwd(int B, int P, int U, int nghost, const int* binum, const int* bilist, const int* bnumneigh,
              const int* bfirstneigh, const T* grad_force, T* grad_dei, hipStream_t stream)
{
    int rc = check_shape(B, P, U, nghost);
    if (rc) return rc;
    A2P_REQUIRE(binum && bilist && bnumneigh && bfirstneigh && grad_force && grad_dei, A2P_ERR_INVALID,
                "fvt force backward: null pointer");
    if (B == 0 || P == 0) return A2P_OK;
    prof_begin("fvt_force_bwd", stream);
    auto kern = (long long)B * P * U >= FVT_WHOLE ? force_bwd_kernel<T, whole_lines<T>()> : force_bwd_kernel<T, false>;
    hipLaunchKernelGGL(kern, dim3(ceil_div((long long)B * P * 64, 256)), dim3(256), 0, stream,
                       grad_dei, grad_force, B, P, U, P + nghost, binum, bilist, bnumneigh, bfirstneigh);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

template <typename T>
int virial_fwd(int B, int P, int U, const int* bnumneigh, const T* rcs, const T* dei, T* virial,
               hipStream_t stream)
{
    int rc = check_shape(B, P, U, 0);
    if (rc) return rc;
    A2P_REQUIRE(bnumneigh && rcs && dei && virial, A2P_ERR_INVALID, "fvt virial: null pointer");
    if (B == 0) return A2P_OK;
    if (P == 0) return fill_zero(virial, (size_t)B * 9 * sizeof(T), stream);
    void* ws = nullptr;
    rc = ws_get(WS_PARTIAL, (size_t)B * P * 9 * sizeof(double), &ws);
    if (rc) return rc;
    bool no_slot = false;
    int* const too_long = early_word(stream, &no_slot);
    prof_begin("fvt_virial_rows", stream);
    hipLaunchKernelGGL(virial_rows_kernel<T>, dim3(ceil_div((long long)B * P * 64, 256)), dim3(256), 0, stream,
                       (double*)ws, dei, rcs, B, P, U, bnumneigh, too_long);
    prof_end(stream);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess && too_long) early_word_drop();
    A2P_HIP_CHECK(err);
    if (too_long) {
        rc = early_word_post(stream);
        if (rc) return rc;
    } else if (no_slot) {                    // more calls waiting than there are slots
        std::vector<int> nn((size_t)B * P);
        A2P_HIP_CHECK(hipMemcpyAsync(nn.data(), bnumneigh, nn.size() * sizeof(int), hipMemcpyDeviceToHost, stream));
        A2P_HIP_CHECK(hipStreamSynchronize(stream));
        early_word_known(*std::max_element(nn.begin(), nn.end()) > U ? 1 : 0);
    }
    return finish_partials<T>(virial, (const double*)ws, B, P, 9, 9, 9, stream);
}

template <typename T>
int virial_bwd(int B, int P, int U, const int* bnumneigh, const T* rcs, const T* dei, const T* grad_virial,
               T* grad_dei, T* grad_rcs, hipStream_t stream)
{
    int rc = check_shape(B, P, U, 0);
    if (rc) return rc;
    A2P_REQUIRE(bnumneigh && rcs && dei && grad_virial && (grad_dei || grad_rcs), A2P_ERR_INVALID,
                "fvt virial backward: null pointer");
    if (B == 0 || P == 0) return A2P_OK;
    prof_begin("fvt_virial_bwd", stream);
    auto kern = (long long)B * P * U >= FVT_WHOLE ? virial_bwd_kernel<T, whole_lines<T>()> : virial_bwd_kernel<T, false>;
    hipLaunchKernelGGL(kern, dim3(ceil_div((long long)B * P * 64, 256)), dim3(256), 0, stream,
                       grad_dei, grad_rcs, grad_virial, dei, rcs, B, P, U, bnumneigh);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

// ---- virial without any allocation ------------------------------------------------------------
// The row partial sums of virial_fwd live in a per-device workspace that is allocated on demand.
// Callers that must not allocate (HIP graph capture, serving loops, harnesses that forbid it) get
// the same two kernels on a buffer that is part of the library's image: each GPU the library runs
// on holds its own copy of `scratch` from the first use until the process ends.
constexpr int kNoAllocMaxRows = 65536;                           // batch * nlocal, 4.5 MiB of partial sums
static __device__ __align__(256) double scratch[(size_t)kNoAllocMaxRows * 9];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
double* g_scratch_ptr[kMaxDevices];                              // device address of `scratch`, per device

// Device address of `scratch` on the current device (its name is only a host-side stand-in).
int scratch_address(double** out)
{
    int dev = -1;
    A2P_HIP_CHECK(hipGetDevice(&dev));
    A2P_REQUIRE(dev >= 0 && dev < kMaxDevices, A2P_ERR_INVALID, "fvt virial (no allocation): device %d not supported", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        A2P_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        A2P_REQUIRE(p != nullptr, A2P_ERR_HIP, "fvt virial (no allocation): scratch has no device address");
        g_scratch_ptr[dev] = (double*)p;
    }
    *out = g_scratch_ptr[dev];
    return A2P_OK;
}

int virial_fwd_noalloc(int B, int P, int U, const int* bnumneigh, const float* rcs, const float* dei, float* virial,
                       hipStream_t stream)
{
    int rc = check_shape(B, P, U, 0);
    if (rc) return rc;
    A2P_REQUIRE(bnumneigh && rcs && dei && virial, A2P_ERR_INVALID, "fvt virial: null pointer");
    A2P_REQUIRE((long long)B * P <= kNoAllocMaxRows, A2P_ERR_INVALID,
                "fvt virial (no allocation): batch * nlocal = %lld exceeds the %d rows of the built-in scratch; "
                "use a2p_fvt_virial_fwd_f32", (long long)B * P, kNoAllocMaxRows);
    if (B == 0) return A2P_OK;
    double* partial = nullptr;
    rc = scratch_address(&partial);
    if (rc) return rc;
    rc = enter_stream(stream);          // the scratch is shared by every stream of the device
    if (rc) return rc;
    // every row below batch * nlocal is written by the first kernel before the second reads it, so
    // what an earlier call left in the buffer never shows; nlocal == 0 leaves nothing to sum (zeros)
    if (P > 0) {
        hipLaunchKernelGGL(virial_rows_kernel<float>, dim3(ceil_div((long long)B * P * 64, 256)), dim3(256), 0, stream,
                           partial, dei, rcs, B, P, U, bnumneigh, (int*)nullptr);
        A2P_HIP_CHECK(hipGetLastError());
    }
    return finish_partials<float>(virial, (const double*)partial, B, P, 9, 9, 9, stream, false);
}

}  // namespace
}  // namespace a2p

#define FVT_LIST const int* binum, const int* bilist, const int* bnumneigh, const int* bfirstneigh

extern "C" {
int a2p_fvt_force_fwd_f32(int B, int P, int U, int nghost, FVT_LIST, const float* dei, float* force, void* s)
{ return a2p::force_fwd<float>(B, P, U, nghost, binum, bilist, bnumneigh, bfirstneigh, dei, force, (hipStream_t)s); }
int a2p_fvt_force_fwd_f64(int B, int P, int U, int nghost, FVT_LIST, const double* dei, double* force, void* s)
{ return a2p::force_fwd<double>(B, P, U, nghost, binum, bilist, bnumneigh, bfirstneigh, dei, force, (hipStream_t)s); }
int a2p_fvt_force_bwd_f32(int B, int P, int U, int nghost, FVT_LIST, const float* gF, float* gdei, void* s)
{ return a2p::force_bwd<float>(B, P, U, nghost, binum, bilist, bnumneigh, bfirstneigh, gF, gdei, (hipStream_t)s); }
int a2p_fvt_force_bwd_f64(int B, int P, int U, int nghost, FVT_LIST, const double* gF, double* gdei, void* s)
{ return a2p::force_bwd<double>(B, P, U, nghost, binum, bilist, bnumneigh, bfirstneigh, gF, gdei, (hipStream_t)s); }
int a2p_fvt_virial_fwd_f32(int B, int P, int U, const int* bnumneigh, const float* rcs, const float* dei,
                           float* virial, void* s)
{ return a2p::virial_fwd<float>(B, P, U, bnumneigh, rcs, dei, virial, (hipStream_t)s); }
int a2p_fvt_virial_fwd_f64(int B, int P, int U, const int* bnumneigh, const double* rcs, const double* dei,
                           double* virial, void* s)
{ return a2p::virial_fwd<double>(B, P, U, bnumneigh, rcs, dei, virial, (hipStream_t)s); }
int a2p_fvt_virial_fwd_noalloc_f32(int B, int P, int U, const int* bnumneigh, const float* rcs, const float* dei,
                                   float* virial, void* s)
{ return a2p::virial_fwd_noalloc(B, P, U, bnumneigh, rcs, dei, virial, (hipStream_t)s); }
int a2p_fvt_virial_bwd_f32(int B, int P, int U, const int* bnumneigh, const float* rcs, const float* dei,
                           const float* gV, float* gdei, float* grcs, void* s)
{ return a2p::virial_bwd<float>(B, P, U, bnumneigh, rcs, dei, gV, gdei, grcs, (hipStream_t)s); }
int a2p_fvt_virial_bwd_f64(int B, int P, int U, const int* bnumneigh, const double* rcs, const double* dei,
                           const double* gV, double* gdei, double* grcs, void* s)
{ return a2p::virial_bwd<double>(B, P, U, bnumneigh, rcs, dei, gV, gdei, grcs, (hipStream_t)s); }
}
