// Deterministic neighbour-pair reduction: every pair (row, slot) of a structure holds a
// derivative g = dE_row/dr_(row,slot); atom j receives  -sum of g over the pairs whose
// neighbour is j  on top of the sum over its own row that the producing kernel stored.
//
// Steps (all on `stream`):
//   1. claim  : every pair takes an entry of its target's segment (a returning integer atomic; the order inside a
//               segment is therefore arbitrary) and leaves its number there.  Segments hold as many pairs as a row: a
//               list built with one cutoff never needs more.  What does not fit (half lists, ghosts that collect the pairs
//               of several rows) is chained behind the target, its pairs dealt to the sixteen chains in turn
//   2. reduce : per target, order-independent sum over the pairs named: every term is converted to 64-bit fixed
//               point against the segment's largest magnitude, integers are added (exact,
//               associative), the total is converted back.  The result is identical for
//               any arrival order, so the output is bit-reproducible run to run; the
//               conversion error per term is below 2^-37 (fp32 inputs) / 2^-52 (fp64 inputs)
//               of the largest term, i.e. below the rounding error of a floating sum.
// The cursors and chain heads are zero between calls: step 2 clears what step 1 wrote.  Step 1 also marks in its cursor
// an atom whose own sum it stored, so the output needs no clearing either.  With the status word leaving by step 2 as well
// (instead of a kernel behind it), an energy / force call of 216 atoms takes 32.2 instead of 37.8 us (level-10 MTP), of
// 20,011 atoms and their ghosts 102.8 instead of 113 (NEP).
// Two short launches, bound by their latency for systems of a few thousand atoms.  Force and virial of 4 x 1000 atoms with
// their gradients, fp64: 59 us of kernels, of which claim 10.8 and reduce 5.5 (65 with a launch that cleared and one that
// sent the status).
// No floating-point atomics are used.
#include "a2p_common.h"

namespace a2p {

namespace {

constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 8;   // items per thread
constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;
constexpr int SCAN_ONE_BLOCK = 512, SCAN_ONE_TILES = 16, SCAN_OWN_TILES = 2048;

__global__ void count_kernel(int* __restrict__ counts, int* __restrict__ rank, int B, int P, int U, int NF,
                             const int* __restrict__ binum, const int* __restrict__ bnumneigh,
                             const int* __restrict__ bfirstneigh, int* __restrict__ status)
{
    // one wave per row; lanes stride the valid slots (coalesced over the row).  With `rank` the
    // pair also learns its place inside its target's segment.
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (wave >= B * P) return;
    const int b = wave / P, ii = wave - b * P;
    if (ii >= binum[b]) return;
    int nn = bnumneigh[wave];
    if (nn > U) {
        if (lane == 0) atomicOr(status, ST_NEIGH_OVERFLOW);
        nn = U;
    }
    const int* row = bfirstneigh + (size_t)wave * U;
    for (int s = lane; s < nn; s += 64) {
        int j = row[s];
        if ((unsigned)j >= (unsigned)NF) {
            atomicOr(status, ST_BAD_NEIGHBOR);
            if (rank) rank[(size_t)wave * U + s] = -1;
            continue;
        }
        if (rank) rank[(size_t)wave * U + s] = atomicAdd(&counts[(size_t)b * NF + j], 1);
        else atomicAdd(&counts[(size_t)b * NF + j], 1);
    }
}

// ---- exclusive scan over int32 ----------------------------------------------------------------
// Bound by its launches (each waits for the one before) until the array is large.  Up to SCAN_ONE_TILES tiles every workgroup
// adds up all that stands before its tile, in one launch; up to SCAN_OWN_TILES what stands before it of the tiles' sums, which
// a first launch forms; beyond, one workgroup scans those sums in between.  22,000 values: 9.2 us in three launches, 5.0 in one;
// 150,000: 10.2 in three, 5.8 in two (in one a workgroup would read up to 600 KB).
struct Four { int v[4]; };                       // (one load, however the array is aligned)

// sum over a workgroup of BLOCK threads, in all of them; `sh` is free again behind the next barrier
template <int BLOCK>
__device__ __forceinline__ int block_sum(int v, int* sh)
{
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; w++) t += sh[w];
    return t;
}

// the thread's SCAN_ITEMS values of the tile (zero beyond the end)
__device__ __forceinline__ void scan_load(const int* __restrict__ in, size_t base, int n, int (&v)[SCAN_ITEMS])
{
    if (base + SCAN_ITEMS <= (size_t)n) {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; k += 4) {
            const Four f = *reinterpret_cast<const Four*>(in + base + k);
#pragma unroll
            for (int i = 0; i < 4; i++) v[k + i] = f.v[i];
        }
    } else {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; k++) v[k] = base + k < (size_t)n ? in[base + k] : 0;
    }
}

// out of the thread's values: what stands before the tile, and before the thread in it
template <int BLOCK>
__device__ __forceinline__ void scan_store(int* __restrict__ out, size_t base, int n, const int (&v)[SCAN_ITEMS], int before, int* sh)
{
    int acc = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) acc += v[k];
    const int incl = wave_inclusive_scan(acc);
    if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = incl;
    __syncthreads();
    int off = before + incl - acc;
    for (int w = 0; w < (int)(threadIdx.x >> 6); w++) off += sh[w];
    if (base + SCAN_ITEMS <= (size_t)n) {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; k += 4) {
            Four f;
#pragma unroll
            for (int i = 0; i < 4; i++) { f.v[i] = off; off += v[k + i]; }
            *reinterpret_cast<Four*>(out + base + k) = f;
        }
    } else {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; k++) {
            if (base + k < (size_t)n) out[base + k] = off;
            off += v[k];
        }
    }
}

__global__ void __launch_bounds__(SCAN_ONE_BLOCK)
scan_one(const int* __restrict__ in, int* __restrict__ out, int n)
{
    __shared__ int sh[2][SCAN_ONE_BLOCK / 64];
    const size_t base = (size_t)blockIdx.x * (SCAN_ONE_BLOCK * SCAN_ITEMS) + (size_t)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    scan_load(in, base, n, v);
    int before = 0;
    static_assert(SCAN_ITEMS == 8, "two loads of four to a thread and tile");
#pragma unroll 4
    for (int t = 0; t < 2 * (int)blockIdx.x; t++) {
        const Four f = *reinterpret_cast<const Four*>(in + ((size_t)t * SCAN_ONE_BLOCK + threadIdx.x) * 4);
        before += (f.v[0] + f.v[1]) + (f.v[2] + f.v[3]);
    }
    before = block_sum<SCAN_ONE_BLOCK>(before, sh[0]);
    scan_store<SCAN_ONE_BLOCK>(out, base, n, v, before, sh[1]);
}

__global__ void __launch_bounds__(SCAN_BLOCK)
scan_tile_sums(const int* __restrict__ in, int* __restrict__ tile_sums, int n)
{
    __shared__ int sh[SCAN_BLOCK / 64];
    int v[SCAN_ITEMS], acc = 0;
    scan_load(in, (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS, n, v);
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; k++) acc += v[k];
    acc = block_sum<SCAN_BLOCK>(acc, sh);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = acc;
}

// single block: exclusive scan of the tile sums
__global__ void scan_tile_offsets(int* __restrict__ tile_sums, int ntiles)
{
    __shared__ int sh[1024 / 64];
    __shared__ int carry_sh;
    if (threadIdx.x == 0) carry_sh = 0;
    __syncthreads();
    for (int base = 0; base < ntiles; base += 1024) {
        int i = base + threadIdx.x;
        int v = i < ntiles ? tile_sums[i] : 0;
        int incl = wave_inclusive_scan(v);
        if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = incl;
        __syncthreads();
        int wave_off = 0;
        for (int w = 0; w < (int)(threadIdx.x >> 6); w++) wave_off += sh[w];
        int carry = carry_sh;
        if (i < ntiles) tile_sums[i] = carry + wave_off + incl - v;
        __syncthreads();
        if (threadIdx.x == 1023) carry_sh = carry + wave_off + incl;
        __syncthreads();
    }
}

// OWN: `tiles` holds the tiles' sums, of which the workgroup adds up its own predecessors'; otherwise their offsets
template <bool OWN>
__global__ void __launch_bounds__(SCAN_BLOCK)
scan_apply(const int* __restrict__ in, int* __restrict__ out, const int* __restrict__ tiles, int n)
{
    __shared__ int sh[2][SCAN_BLOCK / 64];
    const size_t base = (size_t)blockIdx.x * SCAN_TILE + (size_t)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    scan_load(in, base, n, v);
    int before = 0;
    if (OWN) {
#pragma unroll 4
        for (int t = threadIdx.x; t < (int)blockIdx.x; t += SCAN_BLOCK) before += tiles[t];
        before = block_sum<SCAN_BLOCK>(before, sh[0]);
    } else {
        before = tiles[blockIdx.x];
    }
    scan_store<SCAN_BLOCK>(out, base, n, v, before, sh[1]);
}

// Chains of a target that is named by more pairs than a row holds: one for each lane that sums it, so that a chain's
// dependent loads are a sixteenth of what ran over.  Force of 50,000 rows of 32 neighbours, fp64, whole operator: 231 us
// where every segment fits, 328 where an eighth of the atoms collects all pairs (7/8 of them chained), 10 ms where one atom
// collects the pairs of 6,250 rows.
constexpr int SPILL_CHAINS = 16;

// Claims of step 1, one wavefront per row.  With OWN the wavefront also sums the row itself and stores it as the force
// on the row's centre (a centre has one row).
template <typename T, bool OWN>
__global__ void __launch_bounds__(256)
claim_kernel(int B, int P, int U, int NF, int cap, const int* __restrict__ binum, const int* __restrict__ bilist,
             const int* __restrict__ bnumneigh, const int* __restrict__ bfirstneigh, const T* __restrict__ pair_g,
             int* __restrict__ cursor, int* __restrict__ seg, int* __restrict__ heads, int* __restrict__ next,
             T* __restrict__ force, int* __restrict__ status)
{
    const int row = (blockIdx.x * 256 + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (row >= B * P) return;
    const int b = row / P, ii = row - b * P;
    if (ii >= binum[b]) return;
    int nn = bnumneigh[row];
    if (nn > U) {
        if (lane == 0) atomicOr(status, ST_NEIGH_OVERFLOW);
        nn = U;
    }
    const int* first = bfirstneigh + (size_t)row * U;
    const T* g = pair_g + (size_t)row * U * 3;
    T sx = (T)0, sy = (T)0, sz = (T)0;
    for (int s = lane; s < nn; s += 64) {
        const int j = first[s];
        if (OWN) { sx += g[s * 3]; sy += g[s * 3 + 1]; sz += g[s * 3 + 2]; }
        if ((unsigned)j >= (unsigned)NF) {
            atomicOr(status, ST_BAD_NEIGHBOR);
            continue;
        }
        const int t = b * NF + j;
        const int k = pair_claim(&cursor[t]);
        const int pair = row * U + s;
        if (k < cap) seg[(size_t)t * cap + k] = pair;
        else next[pair] = atomicExch(&heads[(size_t)t * SPILL_CHAINS + (k - cap) % SPILL_CHAINS], pair + 1);   // 0 ends a chain
    }
    if (OWN) {
        sx = wave_sum(sx); sy = wave_sum(sy); sz = wave_sum(sz);
        const int c = bilist[row];
        if ((unsigned)c >= (unsigned)NF) {
            if (lane == 0) atomicOr(status, ST_BAD_NEIGHBOR);
        } else if (lane == 0) {
            T* f = force + ((size_t)b * NF + c) * 3;
            f[0] = sx; f[1] = sy; f[2] = sz;
            pair_mark_own(&cursor[b * NF + c]);
        }
    }
}

// 16 lanes per target atom.  Workgroups from `reduce_blocks` on sum the energy / virial partials
// instead (one component of one structure each), which saves small systems a launch.
// With `clear` the cursors (and the heads of the chains in use) are left zero; with `marked` an atom without its producer's
// mark has no own sum in `force` yet.  The status word leaves with the first workgroup when it was asked for: every check of the
// producers is behind this launch, so a caller that waits for it waits for no launch of its own, nor for the sums.
// NAMED: the segments hold the numbers of the pairs (claim_kernel), otherwise the derivatives themselves.
// The first four entries of every lane stay in registers between the two passes (largest magnitude, then the sum).
// With `runs` the workgroups go to the XCDs in runs, so that neighbouring targets' segments come through one L2: 8 structures of 2,500
// atoms 5.0 -> 4.3 us, 4,096 atoms 4.07 -> 3.94.  Not with ghosts, which stand last, have few entries and would leave some XCDs idle
// (20,011 atoms and their ghosts 6.1 -> 6.9).
template <typename T, bool NAMED>
__global__ void __launch_bounds__(256)
reduce_kernel(T* __restrict__ force, const T* __restrict__ seg_g, int* __restrict__ counts, int clear, int marked, int NT, int runs, int seg_cap,
              const int* __restrict__ seg_pair, int* __restrict__ heads, const int* __restrict__ next,
              const EarlyPost post, int reduce_blocks, T* __restrict__ etot, T* __restrict__ virial, const double* __restrict__ partial,
              int nblocks)
{
    if (post.slot && blockIdx.x == 0 && threadIdx.x == 0) {
        const int word = *post.flags;
        read_back_store(post.slot, post.seq, &word, 1);
    }
    if ((int)blockIdx.x >= reduce_blocks) {
        __shared__ double sh[4];
        const int id = (int)blockIdx.x - reduce_blocks;
        finish_ev_body<T>(etot, virial, partial, nblocks, id / 10, id % 10, sh);
        return;
    }
    const int t = (runs ? xcd_block(blockIdx.x, reduce_blocks) : (int)blockIdx.x) * 16 + (int)(threadIdx.x >> 4);       // 256 threads
    const int sub = threadIdx.x & 15;
    // target t owns entries [t*seg_cap, (t+1)*seg_cap); uniform over the 16 lanes of a target
    int all = t < NT ? counts[t] : 0;
    T* const fo = force + (size_t)t * 3;
    bool own = true;
    if (clear) {
        own = !marked || all < 0;
        if (all != 0 && sub == 0) counts[t] = 0;         // the lanes of a target read it in one instruction
        all &= ~PAIR_OWN;
        if (!own && all == 0 && t < NT && sub == 0) fo[0] = fo[1] = fo[2] = (T)0;
    }
    const int cnt = min(all, seg_cap);
    if (all == 0) return;
    const size_t beg = (size_t)t * seg_cap;
    auto entry = [&](int e) __attribute__((always_inline)) -> const T* {
        return seg_g + (NAMED ? (size_t)seg_pair[beg + e] : beg + e) * 3;
    };
    // calls f on every entry beyond the four in registers: the rest of the segment, then this lane's chain of those that
    // did not fit
    auto others = [&](auto&& f) __attribute__((always_inline)) {
        for (int e = sub + 64; e < cnt; e += 16) f(entry(e));
        if (NAMED && all > seg_cap)
            for (int e = heads[(size_t)t * SPILL_CHAINS + sub]; e > 0; e = next[e - 1]) f(seg_g + (size_t)(e - 1) * 3);
    };
    T gx[4], gy[4], gz[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int e = sub + 16 * k;
        gx[k] = (T)0; gy[k] = (T)0; gz[k] = (T)0;
        if (e < cnt) {
            const T* g = entry(e);
            gx[k] = g[0]; gy[k] = g[1]; gz[k] = g[2];
        }
    }
    if constexpr (sizeof(T) == 4) {
        // fp32 segments: every value is rounded to a multiple of 2^q, q chosen from the segment's
        // largest magnitude and its length so that any partial sum of the rounded values fits the
        // 53 bits of a double: the additions are then exact in whatever order they happen.
        float mf = 0.0f;
        auto larger = [&](float a0, float a1, float a2) __attribute__((always_inline)) {
            // fmaxf drops a NaN operand: keep it
            if (!(mf != mf)) mf = fmaxf(mf, fmaxf(fabsf(a0), fmaxf(fabsf(a1), fabsf(a2))));
            if (a0 != a0 || a1 != a1 || a2 != a2) mf = NAN;
        };
#pragma unroll
        for (int k = 0; k < 4; k++) larger(gx[k], gy[k], gz[k]);
        others([&](const T* g) __attribute__((always_inline)) { larger(g[0], g[1], g[2]); });
        wave::over_row(mf, [&](float o) __attribute__((always_inline)) { mf = (mf != mf || o != o) ? NAN : fmaxf(mf, o); });
        const bool finite = mf < 3.0e38f && mf == mf;
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        const bool any = finite && mf > 0.0f;
        if (any) {
            // |v| < 2^(ex+1), fewer than 2^hb of them: sums stay below 2^(ex+1+hb), so q = ex + hb - 52;
            // (v + C) - C with C = 1.5 * 2^(52+q) rounds v to a multiple of 2^q (needs hb >= 2)
            const int hb = max(32 - __clz(all), 2);
            const double C = ldexp(1.5, ilogbf(mf) + hb);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                s0 += ((double)gx[k] + C) - C;
                s1 += ((double)gy[k] + C) - C;
                s2 += ((double)gz[k] + C) - C;
            }
            others([&](const T* g) __attribute__((always_inline)) {
                s0 += ((double)g[0] + C) - C;
                s1 += ((double)g[1] + C) - C;
                s2 += ((double)g[2] + C) - C;
            });
        }
        wave::over_row(s0, [&](double o) __attribute__((always_inline)) { s0 += o; });
        wave::over_row(s1, [&](double o) __attribute__((always_inline)) { s1 += o; });
        wave::over_row(s2, [&](double o) __attribute__((always_inline)) { s2 += o; });
        if (sub == 0) {
            if (!finite) {
                fo[0] = fo[1] = fo[2] = (T)NAN;
            } else if (any || !own) {
                fo[0] = (T)((own ? (double)fo[0] : 0.0) - s0);
                fo[1] = (T)((own ? (double)fo[1] : 0.0) - s1);
                fo[2] = (T)((own ? (double)fo[2] : 0.0) - s2);
            }
        }
    } else {
        double m = 0.0;
        auto larger = [&](double a0, double a1, double a2) __attribute__((always_inline)) {
            m = fmax(m, fmax(fabs(a0), fmax(fabs(a1), fabs(a2))));
        };
#pragma unroll
        for (int k = 0; k < 4; k++) larger(gx[k], gy[k], gz[k]);
        others([&](const T* g) __attribute__((always_inline)) { larger(g[0], g[1], g[2]); });
        wave::over_row(m, [&](double o) __attribute__((always_inline)) { m = fmax(m, o); });
        long long s0 = 0, s1 = 0, s2 = 0;
        double scale = 0.0;
        const bool finite = m < 1.0e300 && m == m;
        if (m < 1.0e-280) m = 0.0;          // nothing but (sub)normal dust: contributes zero
        if (m > 0.0 && finite) {
            const int bits = 61 - (32 - __clz(all));    // head-room for that many additions
            scale = ldexp(1.0, bits - 1 - ilogb(m));
#pragma unroll
            for (int k = 0; k < 4; k++) {
                s0 += __double2ll_rn(gx[k] * scale);
                s1 += __double2ll_rn(gy[k] * scale);
                s2 += __double2ll_rn(gz[k] * scale);
            }
            others([&](const T* g) __attribute__((always_inline)) {
                s0 += __double2ll_rn(g[0] * scale);
                s1 += __double2ll_rn(g[1] * scale);
                s2 += __double2ll_rn(g[2] * scale);
            });
        }
        wave::over_row(s0, [&](long long o) __attribute__((always_inline)) { s0 += o; });
        wave::over_row(s1, [&](long long o) __attribute__((always_inline)) { s1 += o; });
        wave::over_row(s2, [&](long long o) __attribute__((always_inline)) { s2 += o; });
        if (sub == 0) {
            if (!finite) {
                fo[0] = fo[1] = fo[2] = (T)NAN;
            } else if (m > 0.0) {
                fo[0] = (T)((own ? (double)fo[0] : 0.0) - (double)s0 / scale);
                fo[1] = (T)((own ? (double)fo[1] : 0.0) - (double)s1 / scale);
                fo[2] = (T)((own ? (double)fo[2] : 0.0) - (double)s2 / scale);
            } else if (!own) {
                fo[0] = fo[1] = fo[2] = (T)0;
            }
        }
    }
    if (NAMED && clear && all > seg_cap) heads[(size_t)t * SPILL_CHAINS + sub] = 0;     // each lane its own chain's
}

}  // namespace

int scan_tmp_ints(int n) { return ceil_div(n, SCAN_TILE) + 8; }

int exclusive_scan_i32(const int* in, int* out, int n, int* tmp, hipStream_t stream)
{
    if (n <= 0) return A2P_OK;
    const int one = ceil_div(n, SCAN_ONE_BLOCK * SCAN_ITEMS), ntiles = ceil_div(n, SCAN_TILE);
    prof_begin("scan", stream);
    if (one <= SCAN_ONE_TILES) {
        hipLaunchKernelGGL(scan_one, dim3(one), dim3(SCAN_ONE_BLOCK), 0, stream, in, out, n);
    } else {
        hipLaunchKernelGGL(scan_tile_sums, dim3(ntiles), dim3(SCAN_BLOCK), 0, stream, in, tmp, n);
        if (ntiles <= SCAN_OWN_TILES) {
            hipLaunchKernelGGL(scan_apply<true>, dim3(ntiles), dim3(SCAN_BLOCK), 0, stream, in, out, (const int*)tmp, n);
        } else {
            hipLaunchKernelGGL(scan_tile_offsets, dim3(1), dim3(1024), 0, stream, tmp, ntiles);
            hipLaunchKernelGGL(scan_apply<false>, dim3(ntiles), dim3(SCAN_BLOCK), 0, stream, in, out, (const int*)tmp, n);
        }
    }
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

static thread_local int g_seg_capacity = 0;

int pair_segment_capacity(int U) { return g_seg_capacity > U ? g_seg_capacity : U; }

template <typename T>
int pair_fixed_begin(PairCsr* csr, int B, int P, int U_rows, int nghost, hipStream_t stream, T* force, int* cursor_ext,
                     bool cursor_final)
{
    const int U = pair_segment_capacity(U_rows);
    const long long NT = (long long)B * (P + nghost);
    A2P_REQUIRE(NT * U + 1 < (1ll << 31), A2P_ERR_INVALID,
                "pair_reduce: (natoms_pad + nghost) * segment capacity exceeds 32-bit pair indexing");
    const int n = (int)NT;
    // seg_g[(n*U + 1) * 3]: the last entry takes what overflows
    void* ws = nullptr;
    int rc = ws_get(WS_CSR, ((size_t)n * U + 1) * 3 * sizeof(T), &ws);
    if (rc) return rc;
    csr->n = n;
    csr->seg_cap = U;
    csr->runs = nghost == 0 ? 1 : 0;
    csr->seg_g = ws;
    if (cursor_ext) {                                    // the caller keeps the counts
        csr->cursor = cursor_ext;
        const size_t force_bytes = (size_t)n * 3 * sizeof(T);
        if (cursor_final) return fill_zero(force, force_bytes, stream);      // ... and every pair's place is known
        return fill_zero2(cursor_ext, (size_t)n * sizeof(int), force, force_bytes, stream);
    }
    rc = ws_get(WS_CURSORS, (size_t)n * sizeof(int), &ws);
    if (rc) return rc;
    csr->cursor = (int*)ws;
    csr->mark = 1;
    return A2P_OK;
}

int pair_ranks(int B, int P, int U, int nghost, const int* binum, const int* bnumneigh, const int* bfirstneigh,
               int* rank, int* incoming, hipStream_t stream)
{
    A2P_REQUIRE(B >= 0 && P >= 0 && U >= 1 && nghost >= 0, A2P_ERR_INVALID, "pair_ranks: bad shape");
    A2P_REQUIRE(binum && bnumneigh && bfirstneigh && rank && incoming, A2P_ERR_INVALID, "pair_ranks: null pointer");
    if (B == 0 || P == 0) return A2P_OK;
    const int NF = P + nghost;
    void* flags = nullptr;
    int rc = ws_get(WS_FLAGS, 64, &flags);
    if (rc) return rc;
    rc = fill_zero(incoming, (size_t)B * NF * sizeof(int), stream);
    if (rc) return rc;
    prof_begin("pair_ranks", stream);
    hipLaunchKernelGGL(count_kernel, dim3(ceil_div((long long)B * P * 64, 256)), dim3(256), 0, stream, incoming, rank,
                       B, P, U, NF, binum, bnumneigh, bfirstneigh, (int*)flags);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

template <typename T>
int pair_csr_finish(T* force, PairCsr& csr, hipStream_t stream, T* etot, T* virial, const double* partial,
                    int B, int nblocks)
{
    EarlyPost post;
    const int rc = early_take(stream, &post);
    if (rc) return rc;
    const int reduce_blocks = ceil_div((long long)csr.n * 16, 256);
    const int ev_blocks = (etot || virial) ? 10 * B : 0;
    prof_begin("reduce_sum", stream);
    hipLaunchKernelGGL((reduce_kernel<T, false>), dim3(reduce_blocks + ev_blocks), dim3(256), 0, stream,
                       force, (const T*)csr.seg_g, csr.cursor, csr.mark, csr.mark, csr.n, csr.runs, csr.seg_cap, (const int*)nullptr,
                       (int*)nullptr, (const int*)nullptr, post, reduce_blocks, etot, virial, partial, nblocks);
    prof_end(stream);
    const hipError_t err = hipGetLastError();
    early_posted(post, err == hipSuccess);
    A2P_HIP_CHECK(err);
    csr.mark = 0;                                        // the cursors are zero again behind this launch
    return A2P_OK;
}

template <typename T>
int pair_reduce(T* force, const T* pair_g, int B, int P, int U, int nghost, const int* binum, const int* bilist,
                const int* bnumneigh, const int* bfirstneigh, bool own, hipStream_t stream)
{
    const int NF = P + nghost;
    const long long NT = (long long)B * NF, rows = (long long)B * P;
    A2P_REQUIRE(NT < (1ll << 31) - 1 && rows * U < (1ll << 31), A2P_ERR_INVALID,
                "pair_reduce: batch too large for 32-bit pair indexing");
    const int n = (int)NT;
    // workspace: seg[n*U] | next[rows*U] (by pair), and cursor[n] | heads[n*16]
    const size_t seg_bytes = ((size_t)n * U * sizeof(int) + 255) / 256 * 256;
    void *ws = nullptr, *cursors = nullptr;
    int rc = ws_get(WS_CSR, seg_bytes + (size_t)rows * U * sizeof(int), &ws);
    if (rc) return rc;
    int* seg = (int*)ws;
    int* next = (int*)((char*)ws + seg_bytes);
    rc = ws_get(WS_FLAGS, 64, &ws);
    if (rc) return rc;
    rc = ws_get(WS_CURSORS, (size_t)n * (1 + SPILL_CHAINS) * sizeof(int), &cursors);
    if (rc) return rc;
    PairCsr csr;                                         // (gives the cursors up when a launch fails)
    csr.cursor = (int*)cursors;
    csr.mark = 1;
    int* const cursor = csr.cursor;
    int* const heads = cursor + n;
    prof_begin("reduce_claim", stream);
    hipLaunchKernelGGL((own ? claim_kernel<T, true> : claim_kernel<T, false>), dim3(ceil_div(rows * 64, 256)), dim3(256), 0,
                       stream, B, P, U, NF, U, binum, bilist, bnumneigh, bfirstneigh, pair_g, cursor, seg, heads, next,
                       force, (int*)ws);
    prof_end(stream);
    EarlyPost post;
    rc = early_take(stream, &post);
    if (rc) return rc;
    const int reduce_blocks = ceil_div((long long)n * 16, 256);
    prof_begin("reduce_sum", stream);
    hipLaunchKernelGGL((reduce_kernel<T, true>), dim3(reduce_blocks), dim3(256), 0, stream, force, pair_g,
                       cursor, 1, own ? 1 : 0, n, nghost == 0 ? 1 : 0, U, (const int*)seg, heads, (const int*)next, post, reduce_blocks,
                       (T*)nullptr, (T*)nullptr, (const double*)nullptr, 0);
    prof_end(stream);
    const hipError_t err = hipGetLastError();
    early_posted(post, err == hipSuccess);
    A2P_HIP_CHECK(err);
    csr.mark = 0;
    return A2P_OK;
}

template int pair_fixed_begin<float>(PairCsr*, int, int, int, int, hipStream_t, float*, int*, bool);
template int pair_fixed_begin<double>(PairCsr*, int, int, int, int, hipStream_t, double*, int*, bool);
template int pair_csr_finish<float>(float*, PairCsr&, hipStream_t, float*, float*, const double*, int, int);
template int pair_csr_finish<double>(double*, PairCsr&, hipStream_t, double*, double*, const double*, int, int);
template int pair_reduce<float>(float*, const float*, int, int, int, int, const int*, const int*, const int*, const int*,
                                bool, hipStream_t);
template int pair_reduce<double>(double*, const double*, int, int, int, int, const int*, const int*, const int*,
                                 const int*, bool, hipStream_t);

}  // namespace a2p

// largest number of pairs naming one atom: counts (the histogram of a2p_pair_ranks without the ranks), then the maximum
__global__ void incoming_max_kernel(const int* __restrict__ v, int n, int* __restrict__ out)
{
    __shared__ int sh[4];
    int m = 0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) m = max(m, v[i]);
    m = a2p::wave_max(m);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) atomicMax(out, max(max(sh[0], sh[1]), max(sh[2], sh[3])));
}

extern "C" int a2p_pair_segment_capacity(int capacity)
{
    const int old = a2p::g_seg_capacity;
    a2p::g_seg_capacity = capacity > 0 ? capacity : 0;
    return old;
}

extern "C" int a2p_pair_incoming_max(int batch, int natoms_pad, int umax, int nghost, const int* binum,
                                     const int* bnumneigh, const int* bfirstneigh, int* max_incoming, void* stream_)
{
    using namespace a2p;
    hipStream_t stream = (hipStream_t)stream_;
    A2P_REQUIRE(batch >= 0 && natoms_pad >= 0 && umax >= 1 && nghost >= 0, A2P_ERR_INVALID, "pair_incoming_max: bad shape");
    A2P_REQUIRE(binum && bnumneigh && bfirstneigh && max_incoming, A2P_ERR_INVALID, "pair_incoming_max: null pointer");
    *max_incoming = 0;
    if (batch == 0 || natoms_pad == 0) return A2P_OK;
    int rc = enter_stream(stream);
    if (rc) return rc;
    const int NF = natoms_pad + nghost;
    const size_t n = (size_t)batch * NF;
    void* ws = nullptr;
    rc = ws_get(WS_CSR, (n + 64) * sizeof(int), &ws);
    if (rc) return rc;
    void* flags = nullptr;
    rc = ws_get(WS_FLAGS, 64, &flags);
    if (rc) return rc;
    int* counts = (int*)ws;
    rc = fill_zero(counts, (n + 64) * sizeof(int), stream);
    if (rc) return rc;
    hipLaunchKernelGGL(count_kernel, dim3(ceil_div((long long)batch * natoms_pad * 64, 256)), dim3(256), 0, stream, counts,
                       (int*)nullptr, batch, natoms_pad, umax, NF, binum, bnumneigh, bfirstneigh, (int*)flags);
    hipLaunchKernelGGL(incoming_max_kernel, dim3(std::min(ceil_div((long long)n, 256), 1024)), dim3(256), 0, stream,
                       (const int*)counts, (int)n, counts + n);
    A2P_HIP_CHECK(hipGetLastError());
    return read_back(counts + n, 1, max_incoming, stream);
}

extern "C" int a2p_pair_ranks(int batch, int natoms_pad, int umax, int nghost, const int* binum, const int* bnumneigh,
                              const int* bfirstneigh, int* rank, int* incoming, void* stream)
{
    return a2p::pair_ranks(batch, natoms_pad, umax, nghost, binum, bnumneigh, bfirstneigh, rank, incoming,
                           (hipStream_t)stream);
}
