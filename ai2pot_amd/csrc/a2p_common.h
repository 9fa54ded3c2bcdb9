// Internal helpers shared by the HIP translation units of libai2pot_hip.so:
// error reporting, a per-device growable workspace, launch checks and wave-level
// primitives for 64-wide wavefronts (gfx950).
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdarg>
#include <cstring>
#include <string>

#include "../../include/ai2pot_hip.h"

namespace a2p {

// ---- error state (thread local, read back through a2p_last_error) ---------------------
void set_error(const char* fmt, ...);
const char* last_error();

#define A2P_HIP_CHECK(expr)                                                              \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess) {                                                          \
            a2p::set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_),        \
                           __FILE__, __LINE__);                                          \
            return A2P_ERR_HIP;                                                          \
        }                                                                                \
    } while (0)

#define A2P_REQUIRE(cond, code, ...)                                                     \
    do {                                                                                 \
        if (!(cond)) {                                                                   \
            a2p::set_error(__VA_ARGS__);                                                 \
            return code;                                                                 \
        }                                                                                \
    } while (0)

// ---- workspace: a few named device buffers per device, grown on demand -----------------
enum WsSlot {
    WS_PAIR_G = 0,     // per-pair derivative buffer [rows, U, 3]
    WS_CSR,            // counts / offsets / cursors / incoming pair ids
    WS_PARTIAL,        // per-block partial sums (energy, virial, loss terms)
    WS_NBL_A,          // neighbor-list: images, bins
    WS_NBL_B,
    WS_MTP,            // MTP per-atom scratch
    WS_FLAGS,          // device-side status words
    WS_MISC,
    WS_GRID,           // neighbor-list: the bin grid derived on the device (builds without read-back)
    WS_NEP_CLAIMS,     // NEP on compact lists: counters of claimed places and spare rows; zero between calls
    WS_HOST_LISTS,     // neighbour lists on their way to host arrays
    WS_CURSORS,        // pair reduction: cursors and chain heads of the targets; zero between calls
    WS_NSLOTS
};
// Returns a device pointer valid until the next ws_get on the same slot with a larger size.
// Growth synchronises the device (hipFree); steady-state calls do not allocate.
// WS_FLAGS, WS_NEP_CLAIMS and WS_CURSORS are zero-filled when they are allocated; their users leave them zero.
int ws_get(int slot, size_t bytes, void** out);
int ws_drop(int slot); // synchronises the device and frees one buffer of the current device (its contents are suspect)
size_t ws_bytes();     // held on the current device
int ws_release();      // synchronises the device, frees the current device's buffers

// Pinned host memory for one call's copies from or to the device, or null beyond the library's share of it; given back,
// from any thread, when nothing queued reads or writes it any more.
constexpr size_t PINNED_BLOCK = (size_t)64 << 20;      // the largest
void* pinned_take(size_t bytes);
void pinned_give(void* p);

// Device status word bits written by kernels when inputs violate the contract.
enum StatusBits {
    ST_BAD_NEIGHBOR = 1,   // neighbour index outside [0, natoms_pad + nghost)
    ST_BAD_TYPE = 2,       // type index outside [0, ntypes)
    ST_NEIGH_OVERFLOW = 4, // numneigh larger than the row capacity
    ST_SEG_OVERFLOW = 8,   // more pairs name one atom than its reduction segment holds (a list that is not symmetric)
    ST_GRID_BOUND = 16,    // neighbour list built without reading the extents back: the bin box outgrew its bound
};

// Copies nwords (< 32) 4-byte words from device memory to the host behind the work queued on `stream` and waits for
// them; not for streams under capture.
int read_back(const void* device_src, int nwords, void* host_dst, hipStream_t stream);
// The same in two steps, so that the host can queue more work in between.  Every post is waited for, once.
struct ReadBack {
    const void* src;
    int nwords, slot, seq;
    hipStream_t stream;
};
int read_back_post(const void* device_src, int nwords, hipStream_t stream, ReadBack* rb);
int read_back_wait(const ReadBack& rb, void* host_dst);
// For a kernel that posts by itself: the slot's words (1.. are the data, word 0 the number rb->seq, written last and
// with system scope: read_back_store), or null when no slot is free; the caller launches and then waits as above.
int* read_back_take(int nwords, hipStream_t stream, ReadBack* rb);
void read_back_drop(const ReadBack& rb);       // a taken slot whose kernel was not launched
// By one lane.
__device__ __forceinline__ void read_back_store(int* slot, int seq, const int* words, int n)
{
    for (int i = 0; i < n; i++) __hip_atomic_store(slot + 1 + i, words[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(slot, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
// Called where every check of the call's inputs has been queued: posts the status word if the calling thread asked
// for it (a2p_status_early).
int status_post_early(hipStream_t stream);
// The same for a kernel that is launched at that point anyway and posts the word itself (read_back_store of *flags, by one
// lane): slot is null when nothing was asked for or no slot is free.  early_posted tells whether the kernel was launched.
struct EarlyPost {
    int* slot;
    int seq;
    const int* flags;
};
int early_take(hipStream_t stream, EarlyPost* post);
void early_posted(const EarlyPost& post, bool launched);
// The same for a call whose own check is all that is asked for: its kernel stores a non-zero value to the word of pinned
// memory that early_word gives (null: nothing was asked for, or no slot is free; the latter is *no_slot), and
// early_word_post, behind that kernel, ends the report.  The shared status word is left alone.  early_word_known reports
// what the host found by itself, early_word_drop gives the word back when the kernel was not launched.
int* early_word(hipStream_t stream, bool* no_slot);
int early_word_post(hipStream_t stream);
void early_word_known(int word);
void early_word_drop();

inline int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

// ---- optional per-kernel timing with HIP events on the launching stream --------------------
// While profiling is enabled (a2p_profile_enable), a ProfScope around a launch records an
// event before and after it on `stream`; a2p_profile_report resolves them into per-label
// totals.  Disabled (the default) it costs one branch.
void prof_begin(const char* label, hipStream_t stream);
void prof_end(hipStream_t stream);
// Orders this library's work across streams of a device (device synchronisation when the stream changes; a stream
// under capture is left alone).  prof_begin calls it; entry points that launch without prof_begin call it first.
int enter_stream(hipStream_t stream);
struct ProfScope {
    hipStream_t s;
    ProfScope(const char* label, hipStream_t stream) : s(stream) { prof_begin(label, stream); }
    ~ProfScope() { prof_end(s); }
};

// ---- wave64 primitives -------------------------------------------------------------------
__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63); }

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
template <int CTRL>
__device__ __forceinline__ long long dpp_move(long long v)
{
    return (long long)((unsigned long long)(unsigned)dpp_move<CTRL>((int)(v >> 32)) << 32 | (unsigned)dpp_move<CTRL>((int)v));
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
__device__ __forceinline__ int add_rows(int v)
{
    unsigned a, b;
    swap_rows<ROWS>((unsigned)v, a, b);
    return (int)(a + b);
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
    // the longer way round first: lanes eight apart then hold the same bits, and so do, behind the shorter one, lanes four apart
    // (the other way about, neighbouring quads add the same four values in two orders, and end a rounding apart)
    v += dpp_move<0x128>(v);   // row_ror:8
    v += dpp_move<0x124>(v);   // row_ror:4
    v = add_rows<16>(v);
    return add_rows<32>(v);
}
template <typename T>
__device__ __forceinline__ T all_sum(T v) { return sum_over_quads(quad_sum(v)); }
// `take(o)` with the value of the lane 8, 4, 2 and 1 behind in the row of sixteen, which folds it into v: in the end v is folded over
// the row, in each of its lanes, with the same bits (each way round is half of the one before, as in sum_over_quads)
template <typename T, typename Take>
__device__ __forceinline__ void over_row(T& v, Take&& take)
{
    take(dpp_move<0x128>(v));      // row_ror
    take(dpp_move<0x124>(v));
    take(dpp_move<0x122>(v));
    take(dpp_move<0x121>(v));
}
}  // namespace wave

// By data-parallel moves: through the LDS, six round trips and two moves a double each, a wavefront's nine virial sums took most of
// their kernel (virial_rows_kernel, 4,000 rows, 8.2 -> 4.7 us; reduce_kernel at 20,011 atoms, over rows of sixteen, 6.7 -> 6.1).
// Every lane holds the sum, with the same bits.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) { return wave::all_sum(v); }

template <typename T>
__device__ __forceinline__ T wave_max(T v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        T o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    return v;
}


// inclusive prefix sum across the 64 lanes of a wave: shifts by 1, 2, 4, 8 inside each row of
// 16 lanes, then the last lane of row 0 / 2 is added to row 1 / 3 and lane 31 to rows 2 and 3
__device__ __forceinline__ int wave_inclusive_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);    // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);    // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);    // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);    // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 -> rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 -> rows 2, 3
    return v;
}

// ---- shared device routines (pair_reduce.hip) --------------------------------------------
// Deterministic reduction of per-pair derivatives g[row, slot, 3] onto atoms:
//   force[b, j] = own[b, j] - sum over pairs (row, slot) of structure b whose neighbour is j.
// With `own` the sum over the row of centre j is formed here; otherwise `force` must already hold it (zero for atoms
// without a row) and bilist is not read.  Integer atomics deal out the places of the pairs in their targets'
// segments; the floating-point sums are order-independent (terms rounded to a common quantum chosen from the
// per-target maximum, then added exactly), so results are reproducible run to run.  Any list is summed in full.
template <typename T>
int pair_reduce(T* force, const T* pair_g, int B, int P, int U, int nghost, const int* binum, const int* bilist,
                const int* bnumneigh, const int* bfirstneigh, bool own, hipStream_t stream);

// A kernel's argument block, taken anew from the segment it was passed in: a kernel of many phases holds each value in a
// register from its first to its last use otherwise, and what does not fit moves between lanes of vector registers.  S is the
// kernel's first parameter; the empty statement keeps the compiler from carrying an earlier phase's values over.
#define A2P_CONSTANT __attribute__((address_space(4)))
template <typename S>
__device__ __forceinline__ const A2P_CONSTANT S& again(const A2P_CONSTANT S* args)
{
    asm volatile("" : "+s"(args));
    return *args;
}
template <typename S>
__device__ __forceinline__ const A2P_CONSTANT S* kernel_args() { return (const A2P_CONSTANT S*)__builtin_amdgcn_kernarg_segment_ptr(); }
// An array that a wavefront reads uniformly: by scalar loads.
template <typename S>
__device__ __forceinline__ const A2P_CONSTANT S* uniform_array(const S* p) { return (const A2P_CONSTANT S*)(uintptr_t)p; }

// Workgroups are handed to the 8 XCDs round robin; giving XCD k the k-th contiguous run of blocks
// keeps neighbours in space on one L2.
__device__ __forceinline__ int xcd_block(int w, int nb)
{
    const int per = nb >> 3, rem = nb & 7, k = w & 7;
    return k * per + min(k, rem) + (w >> 3);
}

// The same reduction for a producer that stores each pair derivative straight into its target's segment, without the
// intermediate [row, slot, 3] array (pair_fixed_begin, the producer, pair_csr_finish).
// Capacity of the fixed reduction segments: umax unless the calling thread asked for more with
// a2p_pair_segment_capacity (lists in which an atom is named by more pairs than a row holds).
int pair_segment_capacity(int U);
// pair_fixed_begin: every target owns a segment of fixed capacity seg_cap (umax by default)
// (a cutoff-built list sends an atom no more pairs than its own row could hold); the producer
// claims  rank = pair_claim(&cursor[t]),  stores at  pos = t*seg_cap + rank  when rank < seg_cap
// and otherwise raises ST_SEG_OVERFLOW and stores at the spare entry n*seg_cap.  Where it stores an atom's own sum to
// `force` it calls pair_mark_own on the atom's cursor when `mark` is set: the reduction then takes every other atom's own
// sum for zero, so that `force` needs no clearing, and leaves the cursors zero for the next call.
constexpr int PAIR_OWN = (int)0x80000000;          // counts stay below 2^31
__device__ __forceinline__ int pair_claim_raw(int* cursor) { return atomicAdd(cursor, 1); }
__device__ __forceinline__ int pair_rank(int raw) { return raw & ~PAIR_OWN; }       // (where the rank is used: it waits for the claim)
__device__ __forceinline__ int pair_claim(int* cursor) { return pair_rank(pair_claim_raw(cursor)); }
__device__ __forceinline__ void pair_mark_own(int* cursor) { atomicOr(cursor, PAIR_OWN); }
struct PairCsr {
    int* cursor = nullptr;
    void* seg_g = nullptr;
    int n = 0;          // B * (P + nghost) targets
    int seg_cap = 0;
    int runs = 0;       // no ghosts among the targets
    int mark = 0;
    PairCsr() = default;
    PairCsr(const PairCsr&) = delete;
    PairCsr& operator=(const PairCsr&) = delete;
    ~PairCsr() { if (mark) (void)ws_drop(WS_CURSORS); }     // begun and not finished (a launch failed): not known to be zero
};
template <typename T>
int pair_fixed_begin(PairCsr* csr, int B, int P, int U, int nghost, hipStream_t stream, T* force, int* cursor_ext = nullptr,
                     bool cursor_final = false);
// cursor_ext (optional): the caller's array takes the place of the cursors, so that the counts
// survive the call; cursor_final: it already holds the final counts (every pair's place is known
// from an earlier call), so it is neither zeroed nor written.  Nothing is marked then: `force` is cleared by a launch.

// rank[B, P, U] = index of pair (row, slot) among the pairs naming the same neighbour (-1 for an
// index out of range), incoming[B, P+nghost] = number of pairs naming each atom.
int pair_ranks(int B, int P, int U, int nghost, const int* binum, const int* bnumneigh, const int* bfirstneigh,
               int* rank, int* incoming, hipStream_t stream);
// Posts the status word if the calling thread asked for it (status_post_early).
// With etot or virial given, the same launch also sums the energy / virial partials
// (finish_energy_virial's work, in workgroups of its own behind those of the segments).
template <typename T>
int pair_csr_finish(T* force, PairCsr& csr, hipStream_t stream, T* etot = nullptr, T* virial = nullptr,
                    const double* partial = nullptr, int B = 0, int nblocks = 0);

// out[b*out_stride + c] = sum over blocks of partial[(b*nblocks + block)*src_stride + c], c < ncomp,
// with a fixed summation tree (fp64).  timed = false: the launch is never bracketed by timing events
// (which are created on first use), for the callers that must not allocate.
template <typename T>
int finish_partials(T* out, const double* partial, int B, int nblocks, int ncomp, int src_stride,
                    int out_stride, hipStream_t stream, bool timed = true);

// One workgroup of 256 threads, `sh` for its four wavefronts: component c (0 energy, 1..9 virial) of structure b from
// partial[ev_partial(..)], summed over the blocks by a fixed tree (fp64).  A component's shares lie together: with the ten
// of a block together, a workgroup fetched ten times the lines it used (8192 blocks of an MTP call: 9.4 -> 5.3 us for the
// reduction they share a launch with, 12.7 before the sixteen loads in flight).
__host__ __device__ __forceinline__ size_t ev_partial(int nblocks, int b, int block, int c)
{
    return ((size_t)b * 10 + c) * nblocks + block;
}
template <typename T>
__device__ __forceinline__ void finish_ev_body(T* etot, T* virial, const double* partial, int nblocks, int b, int c,
                                               double* sh)
{
    if (c == 0 ? etot == nullptr : virial == nullptr) return;      // uniform over the workgroup
    const double* src = partial + ev_partial(nblocks, b, 0, c);
    double acc = 0.0;
    for (int k0 = threadIdx.x; k0 < nblocks; k0 += 256 * 16) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = k0 + 256 * u < nblocks ? src[k0 + 256 * u] : 0.0;
#pragma unroll
        for (int u = 0; u < 16; u++) acc += v[u];
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        acc = (sh[0] + sh[1]) + (sh[2] + sh[3]);
        if (c == 0) etot[b] = (T)acc;
        else virial[(size_t)b * 9 + c - 1] = (T)acc;
    }
}

// etot[b] and virial[b*9 + c] from partial[ev_partial(nblocks, b, block, 0 | 1 + c)], one launch; either
// output may be null.
template <typename T>
int finish_energy_virial(T* etot, T* virial, const double* partial, int B, int nblocks, hipStream_t stream);

int fill_zero(void* ptr, size_t bytes, hipStream_t stream);
int fill_zero2(void* ptr, size_t bytes, void* ptr2, size_t bytes2, hipStream_t stream);   // two ranges, one launch

// out[i] = in[0] + ... + in[i-1] for i < n (out must not alias in); tmp holds scan_tmp_ints(n) ints.
int scan_tmp_ints(int n);
int exclusive_scan_i32(const int* in, int* out, int n, int* tmp, hipStream_t stream);

}  // namespace a2p
