// NEP energy / force / virial, four atoms per wavefront, for the common model shapes (chebyshev_size 8, n_radial 4 or 6,
// n_angular 4, l_max 3 or 4) on lists in the padded layout.
//
// What bounds it is the issue of vector instructions once a SIMD holds three wavefronts, and an atom's chain of dependent steps
// before that.  A wavefront per atom (1900 instructions an atom) repeated radial functions and b_lm in every channel's lanes,
// summed 24 moments over the wavefront, and left lanes idle wherever an atom has fewer than 64 of something.  Here sixteen
// lanes are an atom's, four atoms share an instruction (3600 for the four), and every step has its own division:
//   * slots of the row: lane = slot, two in flight per lane; radial sums on the way; pairs inside the angular cutoff are
//     compacted to the front of the atom's entries in LDS, pairs between the cutoffs to their back;
//   * angular pairs of all four atoms, 64 at a time: lane = pair, so that each radial function and b_lm is evaluated once; rows
//     [g | b_lm] in LDS turn them over to
//   * moments: lane = (atom, channel, quarter of the moments), which runs through the atom's pairs: no sums across lanes;
//   * hidden layer: lane = neuron, then lane = descriptor for dE/dq;
//   * angular forces: lane = pair again, from the moments' adjoints contracted over the channels; radial forces: lane = entry.
// A pair claims its place in its target's reduction segment with one integer atomic (a2p::PairCsr), issued as soon as the
// pairs are known and waited for behind the read-out (the atomics of all rows take some 5 us at 4096 atoms).  The model's
// tables lie in LDS once per workgroup.  Systems of up to some thousand atoms are faster with a wavefront per atom (nep_wave.hip).
// Registers decide how many wavefronts a SIMD holds: each phase takes arguments, LDS addresses and the lane's place anew.  With
// 60 values spilled for three wavefronts the kernel took 89 us at 20,011 atoms, with two 72, so 58.
//
// Measured (fp32, 6 radial functions, l_max 4, 47 neighbours) against a wavefront per atom: 4096 atoms in lattice order 34 -> 20.7 us
// (28 for the same atoms in no spatial order, when those took 22), 20,011 with skin lists 94 -> 52, 64 structures of 128 atoms 43 -> 24.
// Of the 42 thousand cycles of a wavefront at 4096 atoms the tables took 5.2 (8.2 with a load to a value and the number of rows
// waited for before the first), its rows' heads 1, slots 7.3, angular pairs and moments 6, read-out 9, angular forces 2, radial forces 6,
// and the claims with their answers 3, a row behind the last 1.3, before their entries were read four at a time and it was not begun:
// 21.4 -> 20.7 us, 53.2 -> 51.9 at 20,011.
// Taken back: two neurons a lane at a time (8 values spilled: 61 us), the neurons of dE/dq by fours (57 -> 58), the first entries
// of the radial forces ahead of the angular ones (20 bytes spilled), descriptors scaled by the lane that sums them (no change).
//
// Formulas: source/descriptor/nep/include/{nepBasis.h:57-196; nep.h:320-529}.
#include "a2p_common.h"
#include "nep_device.h"
#include "wave_ops.h"

#include <type_traits>

namespace a2p {
using namespace nepdev;
using namespace wave;
namespace {

template <typename T>
constexpr int wave_cap() { return sizeof(T) == 4 ? 12 : 4; }     // wavefronts of a compute unit: three (fp64: one) per SIMD by registers
constexpr int NW_ATOMS = 4, NW_LANES = 64 / NW_ATOMS;      // atoms of a wavefront, lanes of an atom
constexpr int NW_CAP = 128;                  // slots of a row per tile
constexpr int NW_TRIPS = NW_CAP / NW_LANES;
constexpr int KC = 8, NAC = 4;
constexpr int WROW = 24;                     // row of w0 in LDS: 16-byte reads by 8 lanes with consecutive rows touch
                                             // each bank once
constexpr int CPAD = 4;                      // values behind the coefficients of a species pair (bank spread)

// Shape of the angular part: a lane holds MG moments of a channel, four lanes a channel's (l_max 4: 24, l_max 3: 15 + 1).
template <int LC>
struct Angular {
    static constexpr int NLM = LC * LC + 2 * LC, MG = (NLM + 3) / 4;
    static constexpr int ROW = NAC + 4 * MG;               // of a pair: g of the channels, b_lm
    static constexpr int XYZ = 64 * ROW / (3 * NW_ATOMS);  // angular pairs of an atom whose vectors wait there for their turn
    static constexpr int SCH = 4 * MG, SAT = NAC * SCH + 4;        // moments of a channel, of an atom (banks of the four atoms apart)
};

// Where things lie in LDS, in bytes: the model's tables of the workgroup (w0 first), behind them `own` bytes for each wavefront.
struct WaveAt {
    int coef, b0, w1, qs, cw, bias, shared;        // (cw: w_m C_lm of the 24 moments)
    int own, rows, ang, mom, cc, q, dq, sde;       // of a wavefront, whose entries come first; mom .. sde in the place of rows
};
template <typename T, int LC>
WaveAt wave_at(int nt, int H, int nb)
{
    typedef Angular<LC> A;
    static_assert(64 * A::ROW * sizeof(T) >= 64 * 10 * sizeof(double), "room for the sums at the end");
    WaveAt at;
    size_t off = 0;
    auto take = [&](size_t n, size_t size) { const int at = (int)off; off += (n * size + 15) / 16 * 16; return at; };
    take((size_t)nt * H * WROW, sizeof(T));
    at.coef = take((size_t)nt * nt * (nb * KC + CPAD), sizeof(T));
    at.b0 = take((size_t)nt * H, sizeof(T));
    at.w1 = take((size_t)nt * H, sizeof(T));
    at.qs = take(WROW, sizeof(T));
    at.cw = take(4 * A::MG, sizeof(T));
    at.bias = take((size_t)nt, sizeof(T));
    at.shared = (int)std::min(off, (size_t)1 << 20);      // (beyond the LDS in any case)
    off = 0;
    take(NW_ATOMS * NW_CAP, sizeof(int2));
    at.rows = at.mom = take(NW_ATOMS * A::SAT, sizeof(T));
    at.cc = take((size_t)NW_ATOMS * nt * KC, sizeof(T));
    at.q = take(NW_ATOMS * WROW, sizeof(T));
    at.dq = take(NW_ATOMS * WROW, sizeof(T));
    at.sde = take((size_t)NW_ATOMS * ((H + 3) / 4 * 4), sizeof(T));
    off = std::max(off, at.rows + 64 * A::ROW * sizeof(T));
    at.ang = take(64 * 3, sizeof(T));
    at.own = (int)std::min(off, (size_t)1 << 20);
    return at;
}
template <typename T>
struct WaveLds {
    T *w0, *coef, *b0, *w1, *qs, *cw, *bias;
    int2* ent;                       // pairs of the four atoms' tiles (neighbour, later its place; slot | species << 16)
    T *rows, *ang;                   // angular pairs for the moments; their forces
    T *mom, *cc;                     // moments' adjoints; radial coefficients contracted with dE/dq
    T *q, *dq, *sde;                 // of the read-out
    template <typename At>
    __device__ __forceinline__ WaveLds(const At& at, unsigned char* base, int wave)
    {
        w0 = (T*)base; coef = (T*)(base + at.coef); b0 = (T*)(base + at.b0); w1 = (T*)(base + at.w1); qs = (T*)(base + at.qs);
        cw = (T*)(base + at.cw); bias = (T*)(base + at.bias);
        unsigned char* const mine = base + at.shared + at.own * wave;
        ent = (int2*)mine; rows = (T*)(mine + at.rows); ang = (T*)(mine + at.ang); mom = (T*)(mine + at.mom); cc = (T*)(mine + at.cc);
        q = (T*)(mine + at.q); dq = (T*)(mine + at.dq); sde = (T*)(mine + at.sde);
    }
};

// N values (N even) behind an address aligned to two of them
template <typename T, int N>
__device__ __forceinline__ void lds_load_even(const T* p, T (&o)[N])
{
    typedef T Two __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < N; i += 2) {
        const Two v = *reinterpret_cast<const Two*>(p + i);
        o[i] = v.x; o[i + 1] = v.y;
    }
}

// What a lane of the wavefront wrote to LDS is read by the others behind this.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ int of_atom(int v, int g) { return __builtin_amdgcn_readlane(v, g * NW_LANES); }
__device__ __forceinline__ int most_of_atoms(int v) { return max(max(of_atom(v, 0), of_atom(v, 1)), max(of_atom(v, 2), of_atom(v, 3))); }
__device__ __forceinline__ int pick(int g, int v0, int v1, int v2, int v3) { return g < 2 ? (g == 0 ? v0 : v1) : (g == 2 ? v2 : v3); }

template <typename T>
__device__ __forceinline__ T row_sum(T v)          // the sixteen lanes of a row
{
    v += dpp_move<0x128>(v);                       // row_ror: 8, 4, 2, 1
    v += dpp_move<0x124>(v);
    v += dpp_move<0x122>(v);
    return v + dpp_move<0x121>(v);
}

template <typename T>
struct WaveArgs {
    NepArgs<T> nep;
    SegArgs seg;
    T* seg_g;
    WaveAt at;
    int runs;                        // rows dealt to the workgroups in runs (wave_shape)
};
// The lane's place, found anew by each phase as well (again() of a2p_common.h): what the phases derive from it does not fit the registers
// of three wavefronts per SIMD either.
__device__ __forceinline__ int lane_again()
{
    int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane));
    return lane;
}
#define NW_PHASE                                                                                                            \
    [[maybe_unused]] auto& K_ = again(kernel_args<WaveArgs<T>>());                                                          \
    [[maybe_unused]] auto& a = K_.nep;                                                                                      \
    [[maybe_unused]] auto& seg = K_.seg;                                                                                    \
    [[maybe_unused]] const WaveLds<T> L(K_.at, smem_raw, wave);                                                         \
    [[maybe_unused]] const int H = a.H, nt = a.ntypes, U = a.U, NF = a.P + a.nghost;                                    \
    [[maybe_unused]] const int lane = lane_again();                                                                     \
    [[maybe_unused]] const int g = lane / NW_LANES, s = lane % NW_LANES;       /* atom of the wavefront, lane of the atom */\
    [[maybe_unused]] const int chan = s & 3, mg = s >> 2;                      /* angular channel, MG of its moments */ \
    [[maybe_unused]] int2* const ent = L.ent + g * NW_CAP

// RUNS: rows dealt to the workgroups in runs (wave_shape).  An instance of its own: the loads that only it makes on the way to the first
// rows cost the others a wait (fp64, 4,019 atoms 21.6 -> 22.4 us).  The others ask for `runs` all the same, which is never set there: without
// that branch the compiler lays their first loads out otherwise, at 21.8.
template <typename T, int NR, int LC, bool RUNS>
__global__ void __launch_bounds__(64 * wave_cap<T>(), sizeof(T) == 4 ? 3 : 1)
nep_quad_kernel(const WaveArgs<T>)
{
    typedef Angular<LC> A;
    constexpr int NLM = A::NLM, MG = A::MG, XYZ = A::XYZ, NB = NR + NAC, D = NR + NAC * LC, CROW = NB * KC + CPAD;
    static_assert(D <= WROW && D <= 16 + 8, "descriptor count exceeds the padded row or the lanes of dE/dq");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    int b, blk, inum, last, first, stride;         // structure, workgroup of it; rows, and of the wavefront: end, first, distance
    bool derivs, claims;
    auto run_of = [&](int rows, int nblocks) __attribute__((always_inline)) {              // the workgroup's share of so many
        const int sets = (rows + NW_ATOMS - 1) / NW_ATOMS, per = sets / nblocks, more = sets - per * nblocks, set0 = blk * per + min(blk, more);
        first = NW_ATOMS * (set0 + wave);
        last = NW_ATOMS * (set0 + per + (blk < more ? 1 : 0));
    };
    {
        NW_PHASE;
        const int nblocks = a.nblocks;
        b = blockIdx.y; blk = blockIdx.x; last = a.P;
        first = NW_ATOMS * (wave * nblocks + blk); stride = NW_ATOMS * nwaves * nblocks;
        if (RUNS || K_.runs) {
            const int at = xcd_block(b * nblocks + blk, nblocks * gridDim.y);
            b = at / nblocks; blk = at - b * nblocks;
            run_of(last, nblocks);
            stride = NW_ATOMS * nwaves;
        }
    }
    double e_sum = 0.0, v_sum[9];
#pragma unroll
    for (int i = 0; i < 9; i++) v_sum[i] = 0.0;

    // What the next four rows begin with, on its way while the rows before are worked on: the atom, its number of neighbours,
    // the first 2 * STEP slots (whether they hold a neighbour or not).
    constexpr int V = 2, STEP = V * NW_LANES;              // slots of a lane in flight, of an atom per trip
    int center1, nn1, ti1, nj[V], nj1[V], tj[V];
    T x[V], y[V], z[V], x1[V], y1[V], z1[V];
    auto load = [&](auto& a, int s, int base, int room, int slot0, int (&n)[V], T (&px)[V], T (&py)[V], T (&pz)[V]) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < V; v++) {
            const int slot = slot0 + v * NW_LANES + s;
            n[v] = -1; px[v] = py[v] = pz[v] = (T)0;
            if (slot < room) {
                n[v] = a.bfirstneigh[base + slot];
                const T* p = a.brcs + (size_t)(base + slot) * 3;
                px[v] = p[0]; py[v] = p[1]; pz[v] = p[2];
            }
        }
    };
    auto begin = [&](int i0) __attribute__((always_inline)) {
        NW_PHASE;
        const int row = b * a.P + min(i0 + g, a.P - 1);
        center1 = a.bilist[row];
        nn1 = a.bnumneigh[row];
        load(a, s, row * U, U, 0, nj, x, y, z);
        load(a, s, row * U, U, STEP, nj1, x1, y1, z1);
    };
    auto species = [&](const int (&n)[V], int (&t)[V]) __attribute__((always_inline)) {
        NW_PHASE;
        const int* const types = a.btypes + (size_t)b * NF;
#pragma unroll
        for (int v = 0; v < V; v++) t[v] = (unsigned)n[v] < (unsigned)NF ? types[n[v]] : 0;
    };
    // Their species too, asked for when the tables have been stored: what comes before them in the wavefront's loads is there by then.
    auto begin_species = [&]() __attribute__((always_inline)) {
        NW_PHASE;
        ti1 = a.btypes[(size_t)b * NF + ((unsigned)center1 < (unsigned)NF ? center1 : 0)];
        species(nj, tj);
    };
    begin(first);
    {
        NW_PHASE;
        const int tid = threadIdx.x, nthreads = blockDim.x;
        T bias;
        double c3b;
        [[maybe_unused]] int sample = 0;
        stage_tables<KC, NB, D, WROW, CPAD, 16, T>(a, L, tid, nthreads, [&]() __attribute__((always_inline)) {
            bias = a.bias[min(tid, nt - 1)];
            c3b = kC3B[min(tid, NLM - 1)];
            derivs = a.force != nullptr || a.want_virial;
            claims = derivs && seg.cursor;
            inum = min(uniform_array(a.binum)[b], a.P);       // (the loop below strides over the rows: none beyond the last)
            if (RUNS) sample = a.binum[(unsigned)lane * gridDim.y / 64];
        });
        if (tid < 4 * MG) L.cw[tid] = tid < NLM ? ((tid == 0 || tid == 3 || tid == 8 || tid == 15) ? (T)1 : (T)2) * (T)c3b : (T)0;
        if (tid < nt) L.bias[tid] = bias;
        for (int i = tid + nthreads; i < nt; i += nthreads) L.bias[i] = a.bias[i];
        // Where all structures (of up to 64 looked at) leave a quarter of their places empty, they are divided by their own numbers of rows,
        // now that these are there (wave_shape).
        if (RUNS && !__any(sample > a.P - a.P / 4)) {
            run_of(max(inum, 0), a.nblocks);
            begin(first);
            begin_species();
        } else {
            begin_species();
        }
    }
    __syncthreads();

    last = min(inum, last);
    for (int i0 = first; i0 < last;) {
        int center = center1, nn = nn1, ti, base0;
        {
            NW_PHASE;
            const bool act = i0 + g < inum;
            base0 = (b * a.P + min(i0 + g, a.P - 1)) * U;                    // first pair of the row (pairs: below 2^31)
            if (!act) { center = 0; nn = 0; }
            if (nn > U) { if (s == 0) atomicOr(a.status, ST_NEIGH_OVERFLOW); nn = U; }
            if ((unsigned)center >= (unsigned)NF) { if (s == 0) atomicOr(a.status, ST_BAD_NEIGHBOR); center = 0; nn = 0; }
            ti = center == center1 ? ti1 : a.btypes[(size_t)b * NF + center];
            if ((unsigned)ti >= (unsigned)nt) { if (s == 0 && act) atomicOr(a.status, ST_BAD_TYPE); ti = 0; nn = 0; }
        }
        const int ntiles = max(1, (most_of_atoms(nn) + NW_CAP - 1) / NW_CAP);
        const int ti0 = of_atom(ti, 0), ti1 = of_atom(ti, 1), ti2 = of_atom(ti, 2), ti3 = of_atom(ti, 3);

        T S[MG], q[NR];
#pragma unroll
        for (int m = 0; m < MG; m++) S[m] = (T)0;
#pragma unroll
        for (int n = 0; n < NR; n++) q[n] = (T)0;
        T fx = (T)0, fy = (T)0, fz = (T)0;

        // Tile by tile for the sums (mom), behind the last one the read-out, from the last one on tile by tile for the
        // forces (frc).  Rows of one tile, nearly all, are passed once.
        for (int jt = 0; jt < (derivs ? 2 * ntiles - 1 : ntiles); jt++) {
            const int t = jt < ntiles ? jt : jt - ntiles;
            const bool mom = jt < ntiles, frc = derivs && jt >= ntiles - 1;
            const bool claim = frc && claims;
            const int base = base0 + t * NW_CAP;
            const int tn = min(max(nn - t * NW_CAP, 0), NW_CAP);

            // ---- slots of the tile: radial sums; pairs inside the angular cutoff to the front of the atom's entries, pairs
            // between the cutoffs to their back
            int nA = 0, nR = 0;
            {
                NW_PHASE;
                T* const seg_g = K_.seg_g;
                const T* const cti = L.coef + ti * nt * CROW;
                const T rr = a.rr, ra = a.ra, rr_inv = (T)1 / rr;
                const unsigned below = (1u << s) - 1u;
                const int room = min(U - t * NW_CAP, NW_CAP);
                if (jt > 0) {
                    load(a, s, base, room, 0, nj, x, y, z);
                    load(a, s, base, room, STEP, nj1, x1, y1, z1);
                    species(nj, tj);
                }
                const int trips = (most_of_atoms(tn) + STEP - 1) / STEP;
#pragma unroll 1
                for (int k = 0; k < trips; k++) {
                    const int slot0 = k * STEP + s;
                    int nj2[V];
                    T x2[V], y2[V], z2[V];
                    load(a, s, base, tn, (k + 2) * STEP, nj2, x2, y2, z2);
                    int tj1[V];
                    species(nj1, tj1);
                    bool valid[V], inA[V], inR[V];
                    T r[V];
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        valid[v] = slot0 + v * NW_LANES < tn;
                        if (valid[v] && (unsigned)nj[v] >= (unsigned)NF) { atomicOr(a.status, ST_BAD_NEIGHBOR); valid[v] = false; }
                        if (valid[v] && (unsigned)tj[v] >= (unsigned)nt) { atomicOr(a.status, ST_BAD_TYPE); tj[v] = 0; }
                        T unused;
                        r[v] = length<true>(x[v] * x[v] + y[v] * y[v] + z[v] * z[v], unused);
                        inA[v] = valid[v] && r[v] <= ra && r[v] <= rr;   // nepBasis.h:106, 135: beyond the radial cutoff a neighbour is skipped
                        inR[v] = valid[v] && !inA[v] && r[v] <= rr;
                    }
                    if (mom) {
                        T f[V][KC], df[KC];
#pragma unroll
                        for (int v = 0; v < V; v++) {
                            radial_basis<T, KC, false>(r[v], rr_inv, KC, f[v], df);
#pragma unroll
                            for (int i = 0; i < KC; i++) f[v][i] = inA[v] || inR[v] ? f[v][i] : (T)0;
                        }
#pragma unroll
                        for (int n = 0; n < NR; n++) {
#pragma unroll
                            for (int v = 0; v < V; v++) {
                                T c0[4], c1[4];
                                lds_load4(cti + tj[v] * CROW + n * KC, c0);
                                lds_load4(cti + tj[v] * CROW + n * KC + 4, c1);
                                T u = (T)0;
#pragma unroll
                                for (int i = 0; i < 4; i++) u += c0[i] * f[v][i];
#pragma unroll
                                for (int i = 0; i < 4; i++) u += c1[i] * f[v][4 + i];
                                q[n] += u;
                            }
                        }
                    }
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        const int slot = slot0 + v * NW_LANES;
                        // A pair beyond the cutoffs (a list with a skin) needs no place in this call; when the places are
                        // kept with the list it has one all the same and stores a zero.
                        if (claim && a.brank && valid[v] && !inA[v] && !inR[v]) {
                            const int tg = b * NF + nj[v];
                            int rk;
                            if (a.ranks_valid) rk = a.brank[base + slot];
                            else a.brank[base + slot] = rk = pair_claim(&seg.cursor[tg]);
                            if ((unsigned)rk >= (unsigned)seg.cap) atomicOr(a.status, ST_SEG_OVERFLOW);
                            T* dst = seg_g + (size_t)((unsigned)rk < (unsigned)seg.cap ? tg * seg.cap + rk : seg.spare) * 3;
                            dst[0] = (T)0; dst[1] = (T)0; dst[2] = (T)0;
                        }
                        const unsigned long long bA = __ballot(inA[v]), bR = __ballot(inR[v]);
                        const unsigned mA = (unsigned)(bA >> (g * NW_LANES)) & 0xffffu, mR = (unsigned)(bR >> (g * NW_LANES)) & 0xffffu;
                        if (mom && inA[v]) {                       // (behind the read-out its results lie there)
                            const int k = nA + __popc(mA & below);
                            if (k < XYZ) {
                                T* const p = L.rows + (g * XYZ + k) * 3;
                                p[0] = x[v]; p[1] = y[v]; p[2] = z[v];
                            }
                        }
                        if (inA[v] || inR[v])
                            ent[inA[v] ? nA + __popc(mA & below) : NW_CAP - 1 - (nR + __popc(mR & below))] = make_int2(nj[v], slot | tj[v] << 16);
                        nA += __popc(mA);
                        nR += __popc(mR);
                    }
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        nj[v] = nj1[v]; x[v] = x1[v]; y[v] = y1[v]; z[v] = z1[v]; tj[v] = tj1[v];
                        nj1[v] = nj2[v]; x1[v] = x2[v]; y1[v] = y2[v]; z1[v] = z2[v];
                    }
                }
            }
            wave_sync();
            const int n_own = nA + nR, n_most = most_of_atoms(n_own);
            auto entry = [&](int e) __attribute__((always_inline)) { return e < nA ? e : NW_CAP - 1 - (e - nA); };

            // ---- angular pairs, 64 at a time over the four atoms
            const int n0 = of_atom(nA, 0), n1 = of_atom(nA, 1), n2 = of_atom(nA, 2), n3 = of_atom(nA, 3);
            const int o1 = n0, o2 = n0 + n1, o3 = o2 + n2, total = o3 + n3;
            const int nch = max(1, (total + 63) / 64);
            const bool xyz_held = mom && max(max(n0, n1), max(n2, n3)) <= XYZ;
            int rk[NW_TRIPS];
            for (int it = 0; it < nch + (mom && frc ? nch - 1 : 0); it++) {
                const int c0 = (it < nch ? it : it - nch) * 64;
                const int p = c0 + lane_again();
                // -- lane = pair: direction, radial functions, b_lm
                const int pg = (p >= o1) + (p >= o2) + (p >= o3);
                const bool on = p < total;
                T ux = (T)0, uy = (T)0, uz = (T)0, rinv = (T)0, ga[NAC], dg[NAC];
#pragma unroll
                for (int c = 0; c < NAC; c++) ga[c] = dg[c] = (T)0;
                if (on) {
                    NW_PHASE;
                    const int row0 = b * a.P + i0;
                    const T ra_inv = (T)1 / a.ra;
                    const int w = L.ent[pg * NW_CAP + (p - pick(pg, 0, o1, o2, o3))].y;
                    T x, y, z;
                    if (it == 0 && xyz_held) {
                        const T* const xp = L.rows + (pg * XYZ + (p - pick(pg, 0, o1, o2, o3))) * 3;
                        x = xp[0]; y = xp[1]; z = xp[2];
                    } else {
                        const T* const xp = a.brcs + (size_t)((row0 + pg) * U + t * NW_CAP + (w & 0xffff)) * 3;
                        x = xp[0]; y = xp[1]; z = xp[2];
                    }
                    const T r = length<false>(x * x + y * y + z * z, rinv);
                    ux = x * rinv; uy = y * rinv; uz = z * rinv;
                    T f[KC], df[KC];
                    radial_basis<T, KC, true>(r, ra_inv, KC, f, df);
                    const T* c = L.coef + (size_t)(pick(pg, ti0, ti1, ti2, ti3) * nt + (w >> 16)) * CROW + NR * KC;
#pragma unroll
                    for (int n = 0; n < NAC; n++) {
                        T v0[4], v1[4];
                        lds_load4(c + n * KC, v0);
                        lds_load4(c + n * KC + 4, v1);
#pragma unroll
                        for (int i = 0; i < 4; i++) { ga[n] += v0[i] * f[i]; dg[n] += v0[i] * df[i]; }
#pragma unroll
                        for (int i = 0; i < 4; i++) { ga[n] += v1[i] * f[4 + i]; dg[n] += v1[i] * df[4 + i]; }
                    }
                }
                if (claim && it == (mom ? nch - 1 : 0)) {
                    // -- the pairs claim their places; the answers are stored when the forces' turn comes (the loads above
                    // would wait for them)
                    NW_PHASE;
                    // (half of the entries read at a time, and then their claims)
#pragma unroll
                    for (int k0 = 0; k0 < NW_TRIPS; k0 += NW_TRIPS / 2) {
                        if (k0 * NW_LANES >= n_most && k0 > 0) {
#pragma unroll
                            for (int k = k0; k < k0 + NW_TRIPS / 2; k++) rk[k] = 0;
                            break;
                        }
                        int2 w[NW_TRIPS / 2];
#pragma unroll
                        for (int k = 0; k < NW_TRIPS / 2; k++) w[k] = ent[entry(min((k0 + k) * NW_LANES + s, max(n_own - 1, 0)))];
#pragma unroll
                        for (int k = k0; k < k0 + NW_TRIPS / 2; k++) {
                            rk[k] = 0;
                            if (k * NW_LANES + s < n_own) {
                                if (a.brank && a.ranks_valid) rk[k] = a.brank[base + (w[k - k0].y & 0xffff)];
                                else rk[k] = pair_claim_raw(&seg.cursor[b * NF + w[k - k0].x]);
                            }
                        }
                    }
                }
                if (mom && it < nch) {
                    NW_PHASE;
                    // -- moments: lane = (atom, channel, MG of the moments), the atom's pairs one after the other
                    wave_sync();
                    if (on) {
                        T bl[NLM];
                        blm_values<T, LC>(ux, uy, uz, bl);
                        T* const rw = L.rows + lane * A::ROW;
                        lds_store4(rw, ga[0], ga[1], ga[2], ga[3]);
#pragma unroll
                        for (int m = 0; m < 4 * MG; m += 4)
                            lds_store4(rw + NAC + m, bl[m], bl[m + 1], bl[m + 2], m + 3 < NLM ? bl[m + 3 < NLM ? m + 3 : 0] : (T)0);
                    }
                    wave_sync();
                    const int o_own = pick(g, 0, o1, o2, o3), lo = max(o_own, c0) - c0, n = max(min(o_own + nA, c0 + 64) - c0 - lo, 0), trips = most_of_atoms(n);
                    if (n > 0) {
                        const T* const rw = L.rows + lo * A::ROW;
                        for (int k0 = 0; k0 < trips; k0 += 4) {
                            T gc[4], bm[4][MG];
#pragma unroll
                            for (int u = 0; u < 4; u++) {
                                const T* const r = rw + min(k0 + u, n - 1) * A::ROW;
                                gc[u] = r[chan];
                                lds_load_even(r + NAC + mg * MG, bm[u]);
                            }
#pragma unroll
                            for (int u = 0; u < 4; u++) gc[u] = k0 + u < n ? gc[u] : (T)0;
#pragma unroll
                            for (int m = 0; m < MG; m++)
                                S[m] += (gc[0] * bm[0][m] + gc[1] * bm[1][m]) + (gc[2] * bm[2][m] + gc[3] * bm[3][m]);
                        }
                    }
                    wave_sync();
                }
                if (mom && jt == ntiles - 1 && it == nch - 1) {
                    NW_PHASE;
                    // ---- descriptors.  q_{n,l} = sum_m w_m C_lm S^2  (nepBasis.h:174-190)
                    T cw[MG];
                    lds_load_even(L.cw + mg * MG, cw);
                    const bool act = i0 + g < inum;
                    const T* const cti = L.coef + ti * nt * CROW;
                    T* const mo = L.mom + g * A::SAT + chan * A::SCH;
#pragma unroll
                    for (int m = 0; m < MG; m++) mo[mg * MG + m] = cw[m] * S[m] * S[m];
#pragma unroll
                    for (int n = 0; n < NR; n++) q[n] = row_sum(q[n]);
                    wave_sync();
                    T* const Q = L.q + g * WROW;
                    T qr = (T)0;
#pragma unroll
                    for (int n = 0; n < NR; n++) qr = s == n ? q[n] : qr;
                    if (s < NR) Q[s] = qr;
                    if (mg < LC) {
                        const int l = mg + 1;
                        T acc = (T)0;
#pragma unroll
                        for (int i = 0; i < 2 * LC + 1; i++)
                            if (i < 2 * l + 1) acc += mo[l * l - 1 + i];
                        Q[NR + chan * LC + mg] = acc;
                    }
                    wave_sync();
#pragma unroll
                    for (int d0 = 0; d0 < WROW; d0 += NW_LANES) {
                        const int d = d0 + s;
                        if (d < D) {
                            const T v = Q[d];
                            if (a.desc && act) a.desc[((size_t)b * a.P + i0 + g) * D + d] = v;
                            Q[d] = v * L.qs[d];
                        } else if (d < WROW) {
                            Q[d] = (T)0;
                        }
                    }
                    wave_sync();

                    // ---- hidden layer (nep.h:415-447): lane = neuron -------------------------------------------------
                    T qv[(D + 3) / 4 * 4], e_site = (T)0;
#pragma unroll
                    for (int j = 0; j < D; j += 4) {
                        T v[4];
                        lds_load4(Q + j, v);
#pragma unroll
                        for (int i = 0; i < 4; i++) qv[j + i] = v[i];
                    }
                    T* const sde = L.sde + g * ((H + 3) / 4 * 4);
#pragma unroll 1
                    for (int n = s; n < H; n += NW_LANES) {
                        const T* wrow = L.w0 + (size_t)(ti * H + n) * WROW;
                        T h = L.b0[ti * H + n];
#pragma unroll
                        for (int j = 0; j < D; j += 4) {
                            T w[4];
                            lds_load4(wrow + j, w);
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                if (j + i < D) h += w[i] * qv[j + i];
                        }
                        const T th = tanh_t(h), w1p = L.w1[ti * H + n];
                        e_site += w1p * th;
                        sde[n] = w1p * ((T)1 - th * th);
                    }
                    e_site = row_sum(e_site);
                    if (act && s == 0) e_sum += (double)e_site + (double)L.bias[ti];         // (rounded to fp32 the bias shifts every atom alike)
                    if (derivs) {
                        wave_sync();
                        // dE/dq: lane = descriptor; of those from the sixteenth on a lane takes half of the neurons
                        T* const DQ = L.dq + g * WROW;
                        const T* col = L.w0 + (size_t)ti * H * WROW;
                        T acc = (T)0, acc1 = (T)0, acc2 = (T)0;
                        const int half = H >> 1, d2 = NW_LANES + (s & 7), h2 = s < 8 ? 0 : half;
#pragma unroll 5
                        for (int n = 0; n < half; n++) {
                            acc += sde[n] * col[n * WROW + s];
                            acc1 += sde[half + n] * col[(half + n) * WROW + s];
                            if (D > NW_LANES) acc2 += sde[h2 + n] * col[(h2 + n) * WROW + d2];
                        }
                        if (H & 1) {
                            acc += sde[H - 1] * col[(H - 1) * WROW + s];
                            if (D > NW_LANES && s < 8) acc2 += sde[H - 1] * col[(H - 1) * WROW + d2];
                        }
                        if (D > NW_LANES) {
                            acc2 += dpp_move<0x128>(acc2);
                            if (s < 8) DQ[d2] = acc2 * L.qs[d2];
                        }
                        DQ[s] = (acc + acc1) * L.qs[s];
                        wave_sync();
                        // ---- dE/dS (nep.h:450-466); radial coefficients contracted with dE/dq
#pragma unroll
                        for (int m = 0; m < MG; m++) {
                            const int lm = mg * MG + m;
                            const int l1 = lm < 3 ? 0 : lm < 8 ? 1 : lm < 15 ? 2 : 3;
                            mo[lm] = S[m] * DQ[NR + chan * LC + min(l1, LC - 1)] * ((T)2 * cw[m]);
                        }
                        for (int i = s; i < nt * KC; i += NW_LANES) {
                            const T* c = cti + (i >> 3) * CROW + (i & 7);
                            T v = (T)0;
#pragma unroll
                            for (int n = 0; n < NR; n++) v += DQ[n] * c[n * KC];
                            L.cc[g * nt * KC + i] = v;
                        }
                    }
                    wave_sync();
                }
                if (!frc || (mom && it < nch - 1)) continue;

                // ---- pair derivatives ------------------------------------------------------------------------------
                if (claim && it == (mom ? nch - 1 : 0)) {
                    NW_PHASE;
#pragma unroll
                    for (int k0 = 0; k0 < NW_TRIPS; k0 += NW_TRIPS / 2) {
                        if (k0 * NW_LANES >= n_most) break;
                        int2 w[NW_TRIPS / 2];
#pragma unroll
                        for (int k = 0; k < NW_TRIPS / 2; k++) w[k] = ent[entry(min((k0 + k) * NW_LANES + s, max(n_own - 1, 0)))];
#pragma unroll
                        for (int k = k0; k < k0 + NW_TRIPS / 2; k++) {
                            const int e = k * NW_LANES + s;
                            if (e >= n_own) continue;
                            const int tg = b * NF + w[k - k0].x, r = pair_rank(rk[k]);
                            if (a.brank && !a.ranks_valid) a.brank[base + (w[k - k0].y & 0xffff)] = r;
                            const bool fits = (unsigned)r < (unsigned)seg.cap;
                            if (!fits) atomicOr(a.status, ST_SEG_OVERFLOW);
                            ent[entry(e)].x = fits ? tg * seg.cap + r : seg.spare;
                        }
                    }
                }
                // -- lane = pair: F = g' T u + (w - (w . u) u) / r with the moments' adjoints s, T = s . b and w = s . grad b
                if (on) {
                    NW_PHASE;
                    const T* mo = L.mom + pg * A::SAT;
                    T bl[NLM];                                    // (again: held over the read-out they would cost a wavefront per SIMD)
                    asm volatile("" : "+v"(ux), "+v"(uy), "+v"(uz));
                    blm_values<T, LC>(ux, uy, uz, bl);
                    T P[NLM], srad = (T)0;
#pragma unroll
                    for (int m = 0; m < NLM; m++) P[m] = (T)0;
#pragma unroll
                    for (int c = 0; c < NAC; c++) {
                        T tc = (T)0;
#pragma unroll
                        for (int m = 0; m < 4 * MG; m += 4) {
                            T v[4];
                            lds_load4(mo + c * A::SCH + m, v);
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                if (m + i < NLM) { P[m + i] += ga[c] * v[i]; tc += v[i] * bl[m + i]; }
                        }
                        srad += dg[c] * tc;
                    }
                    T wx, wy, wz;
                    forget(ux, uy, uz);
                    blm_gradient<T, LC>(ux, uy, uz, P, wx, wy, wz);
                    T* const rw = L.ang + lane * 3;
                    pair_gradient(srad, wx, wy, wz, ux, uy, uz, rinv, rw[0], rw[1], rw[2]);
                }
                wave_sync();
                // -- lane = neighbour of the atom: the radial part, the pair's force; behind the last angular pairs also the
                // pairs between the cutoffs
                const bool tail = it == nch - 1;
                NW_PHASE;
                const int o_own = pick(g, 0, o1, o2, o3);
                const T rr_inv = (T)1 / a.rr;
                const int f0 = min(max(c0 - o_own, 0), nA), f1 = min(max(c0 + 64 - o_own, 0), nA);
                const int nf = f1 - f0, nr = tail ? nR : 0, trips = (most_of_atoms(nf + nr) + 2 * NW_LANES - 1) / (2 * NW_LANES);
                T* const seg_g = K_.seg_g;
                auto fetch = [&](int k, int2& w, T& x, T& y, T& z) __attribute__((always_inline)) {
                    w = make_int2(0, 0); x = (T)1; y = z = (T)0;
                    if (k < nf + nr) {
                        w = ent[k < nf ? f0 + k : NW_CAP - 1 - (k - nf)];
                        const T* xp = a.brcs + (size_t)(base + (w.y & 0xffff)) * 3;
                        x = xp[0]; y = xp[1]; z = xp[2];
                    }
                };
                T vir[9];
#pragma unroll
                for (int i = 0; i < 9; i++) vir[i] = (T)0;
                int2 w1[V];
                T xn[V], yn[V], zn[V];
#pragma unroll
                for (int v = 0; v < V; v++) fetch(v * NW_LANES + s, w1[v], xn[v], yn[v], zn[v]);
#pragma unroll 1
                for (int k0 = 0; k0 < trips; k0++) {
                    const int k = k0 * STEP + s;
                    int2 w[V];
                    T px[V], py[V], pz[V], gx[V], gy[V], gz[V];
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        w[v] = w1[v]; px[v] = xn[v]; py[v] = yn[v]; pz[v] = zn[v];
                        fetch(k + STEP + v * NW_LANES, w1[v], xn[v], yn[v], zn[v]);
                    }
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        T ri;
                        const T r = length<false>(px[v] * px[v] + py[v] * py[v] + pz[v] * pz[v], ri);
                        T f[KC], df[KC];
                        radial_basis<T, KC, true>(r, rr_inv, KC, f, df);
                        T v0[4], v1[4], sr = (T)0;
                        const T* cc = L.cc + (g * nt + (w[v].y >> 16)) * KC;
                        lds_load4(cc, v0);
                        lds_load4(cc + 4, v1);
#pragma unroll
                        for (int i = 0; i < 4; i++) sr += v0[i] * df[i];
#pragma unroll
                        for (int i = 0; i < 4; i++) sr += v1[i] * df[4 + i];
                        sr *= ri;
                        gx[v] = sr * px[v]; gy[v] = sr * py[v]; gz[v] = sr * pz[v];
                    }
#pragma unroll
                    for (int v = 0; v < V; v++) {
                        const int kv = k + v * NW_LANES;
                        if (kv < nf + nr) {
                            if (kv < nf) {
                                const T* rw = L.ang + (o_own + f0 + kv - c0) * 3;
                                gx[v] += rw[0]; gy[v] += rw[1]; gz[v] += rw[2];
                            }
                            if (seg_g) {
                                T* dst = seg_g + (size_t)w[v].x * 3;
                                dst[0] = gx[v]; dst[1] = gy[v]; dst[2] = gz[v];
                            }
                        } else {
                            gx[v] = gy[v] = gz[v] = (T)0;
                        }
                    }
                    static_assert(V == 2, "sums two by two: as many roundings as over 64 lanes");
                    fx += gx[0] + gx[1]; fy += gy[0] + gy[1]; fz += gz[0] + gz[1];
                    vir[0] -= gx[0] * px[0] + gx[1] * px[1]; vir[1] -= gx[0] * py[0] + gx[1] * py[1]; vir[2] -= gx[0] * pz[0] + gx[1] * pz[1];
                    vir[3] -= gy[0] * px[0] + gy[1] * px[1]; vir[4] -= gy[0] * py[0] + gy[1] * py[1]; vir[5] -= gy[0] * pz[0] + gy[1] * pz[1];
                    vir[6] -= gz[0] * px[0] + gz[1] * px[1]; vir[7] -= gz[0] * py[0] + gz[1] * py[1]; vir[8] -= gz[0] * pz[0] + gz[1] * pz[1];
                }
#pragma unroll
                for (int i = 0; i < 9; i++) v_sum[i] += (double)vir[i];
                wave_sync();
            }
        }
        NW_PHASE;
        if (a.force) {
            fx = row_sum(fx); fy = row_sum(fy); fz = row_sum(fz);
            const bool act = i0 + g < inum;
            if (act && s < 3) a.force[((size_t)b * NF + center) * 3 + s] = s == 0 ? fx : s == 1 ? fy : fz;
            if (act && seg.mark && s == 3) pair_mark_own(&seg.cursor[b * NF + center]);
        }
        i0 += stride;
        if (i0 >= last) break;                           // (no row behind the last one is waited for)
        begin(i0);
        begin_species();
    }

    // ---- workgroup partial sums of energy and virial (fp64): 16 threads to a sum, lanes 4 k .. 4 k + 3 of every wavefront
    // to the k-th
    {
        NW_PHASE;
        double* const mine = (double*)L.rows;              // (of the wavefront; the read-out's scratch is no longer in use)
        mine[lane] = e_sum;
#pragma unroll
        for (int i = 0; i < 9; i++) mine[(1 + i) * 64 + lane] = v_sum[i];
    }
    __syncthreads();
    NW_PHASE;
    for (int c = threadIdx.x >> 4; c < 10; c += nwaves * 4) {
        double v = 0.0;
        for (int w = 0; w < nwaves; w++) {
            const double* theirs = (const double*)((const unsigned char*)L.rows + (w - wave) * K_.at.own) + c * 64 + s * 4;
#pragma unroll
            for (int i = 0; i < 4; i++) v += theirs[i];
        }
        v = row_sum(v);
        if (s == 0) a.partial[ev_partial(a.nblocks, b, blk, c)] = v;
    }
}
#undef NW_PHASE

// Wavefronts of a workgroup, workgroups of a structure.  A workgroup to a compute unit, which shares the model's tables, or two
// where they have room; as many rows for each wavefront as it takes with the most wavefronts a compute unit holds, and then no
// more wavefronts than that takes (four stage the tables faster than one).
// Up to eight sets to a compute unit the rows are dealt out one set to a workgroup in turn; beyond, every workgroup takes a run of
// consecutive rows and every XCD a run of workgroups, so that neighbours in the list's order share their species, cursors and
// segments' lines in one cache.  In turn and in runs, us: one structure of 9,000 atoms 34.9 and 32.1, 20,011 with ghosts 57.0
// and 52.9, 32,768 68.1 and 66.0; 8 of 2,500 61.4 and 47.6, 32 of 640 60.1 and 47.7, 64 of 400 66.2 and 59.7, 128 of 128 44.4
// and 41.1; fp64 20,011 100 and 98.  With fewer sets all rows of a neighbourhood claim their places at once, from one XCD: 4,096
// atoms 21.9 and 23.1, 6,000 25.0 and 26.0, 8,192 26.6 and 26.7, 64 structures of 128 24.8 and 29.4.  (XCDs in runs and workgroups in
// turn: 20,011 atoms 51.4, 32,768 82.9.)  Runs go by the lists' places, for the numbers of rows in use
// come with the tables; where these show that all structures leave a quarter of their places empty, by those numbers, which takes the first rows'
// loads once more.  In turn, by places alone and so, us: 8 structures of 2,500 places with 1,870 in use 43.8, 38.9 and 41.4, with 1,500 36.2,
// 38.0 and 35.3, with 800 28.4, 36.3 and 28.1; 64 of 400 with 300 43.2, 48.7 and 41.2, with 150 27.5, 46.1 and 27.6; one of 20,000 with 5,000 23.3, 37.4
// and 24.0; fp64 8 of 2,500 with 800 42.3, 91.0 and 42.1.  A structure with all of its places in use takes as long whatever the others do: sizes
// from a third of the places up, 32 of 640 45.8 in turn, 39.6 by places, 42.0 with the smaller ones by their rows, 128 of 128 34.7, 34.1 and 34.8.
struct WaveShape { int waves, nblocks, runs; size_t lds; WaveAt at; };
template <typename T>
WaveShape wave_shape(const NepArgs<T>& a)
{
    const WaveAt at = a.l_max == 3 ? wave_at<T, 3>(a.ntypes, a.H, a.n_r + NAC) : wave_at<T, 4>(a.ntypes, a.H, a.n_r + NAC);
    const int most = std::min(wave_cap<T>(), (160 * 1024 - std::min(at.shared, 160 * 1024)) / at.own);
    if (most < 1) return {0, 0, 0, 0, at};
    const int per = std::max(1, ceil_div(a.P, NW_ATOMS));                    // sets of four rows of a structure
    const long long sets = (long long)a.B * per;
    int waves = std::min(most, (int)std::min<long long>((sets + 256 * 4 - 1) / (256 * 4) * 4, wave_cap<T>())), held = 1;
    if (waves == 8 && 2 * (at.shared + 4 * at.own) <= 160 * 1024) { waves = 4; held = 2; }
    const int nblocks = std::min(ceil_div(per, waves), std::max(1, held * 256 / std::max(a.B, 1)));
    return {waves, nblocks, sets > 8 * 256, (size_t)at.shared + (size_t)waves * at.own, at};
}

template <typename T, int NR, int LC>
int launch_wave(const NepArgs<T>& a, const PairCsr& csr, hipStream_t stream)
{
    SegArgs seg{csr.cursor, csr.seg_cap, csr.n * csr.seg_cap, csr.mark};
    const WaveShape w = wave_shape<T>(a);
    auto kern = w.runs ? nep_quad_kernel<T, NR, LC, true> : nep_quad_kernel<T, NR, LC, false>;
    if (w.lds > 48 * 1024)
        A2P_HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)w.lds));
    prof_begin("nep_quad_kernel", stream);
    hipLaunchKernelGGL(kern, dim3(a.nblocks, a.B), dim3(64 * w.waves), w.lds, stream, WaveArgs<T>{a, seg, (T*)csr.seg_g, w.at, w.runs});
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

}  // namespace

template <typename T>
int nep_quad_nblocks(const NepArgs<T>& a)
{
    return wave_shape<T>(a).nblocks;
}

template <typename T>
bool nep_quad_supported(const NepArgs<T>& a)
{
    return a.K == KC && (a.n_r == 4 || a.n_r == 6) && a.n_a == NAC && (a.l_max == 3 || a.l_max == 4) && wave_shape<T>(a).waves > 0;
}

template <typename T>
int nep_quad_run(const NepArgs<T>& a, T* etot, T* virial, hipStream_t stream)
{
    PairCsr csr;
    int rc;
    if (a.force) {
        rc = pair_fixed_begin<T>(&csr, a.B, a.P, a.U, a.nghost, stream, a.force, a.bincoming,
                                 a.bincoming != nullptr && a.ranks_valid != 0);
        if (rc) return rc;
    }
    if (a.n_r == 4) rc = a.l_max == 3 ? launch_wave<T, 4, 3>(a, csr, stream) : launch_wave<T, 4, 4>(a, csr, stream);
    else rc = a.l_max == 3 ? launch_wave<T, 6, 3>(a, csr, stream) : launch_wave<T, 6, 4>(a, csr, stream);
    if (rc) return rc;
    if (a.force) return pair_csr_finish<T>(a.force, csr, stream, etot, virial, a.partial, a.B, a.nblocks);
    return finish_energy_virial<T>(etot, virial, a.partial, a.B, a.nblocks, stream);
}

template bool nep_quad_supported<float>(const NepArgs<float>&);
template bool nep_quad_supported<double>(const NepArgs<double>&);
template int nep_quad_nblocks<float>(const NepArgs<float>&);
template int nep_quad_nblocks<double>(const NepArgs<double>&);
template int nep_quad_run<float>(const NepArgs<float>&, float*, float*, hipStream_t);
template int nep_quad_run<double>(const NepArgs<double>&, double*, double*, hipStream_t);

}  // namespace a2p
