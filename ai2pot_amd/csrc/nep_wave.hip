// NEP energy / force / virial, one wavefront per atom, for the common model shapes (chebyshev_size 8, n_radial 4 or 6,
// n_angular 4, l_max 3 or 4) on lists in the padded layout, for systems of up to some thousand atoms.
//
// What bounds such systems is the serial chain of an atom and the first fetch of the code: every SIMD holds three wavefronts at
// most.  Here every step has its own division over the 64 lanes:
//   * a row is read once, lane = slot, 128 slots at a time; pairs inside the angular cutoff are compacted to the front of
//     the wavefront's tile in LDS, pairs between the cutoffs to its back (ballots); a pair claims its place in its
//     target's reduction segment with one integer atomic (a2p::PairCsr);
//   * radial functions and radial forces: lane = neighbour (47 of 64 lanes at the benchmark's density);
//   * angular moments and forces: lane = (neighbour, angular channel), 16 neighbours at a time; a lane holds the 24
//     moments of its channel, summed over the neighbours with four cross-lane additions;
//   * hidden layer: lane = neuron, then lane = (descriptor, half of the neurons) for dE/dq.
// About 1900 vector instructions per atom (6 radial, l_max 4, 48 + 12 neighbours); nep_quad.hip shares most of them between four
// atoms and takes over where their issue counts.  The model's tables lie in LDS once per workgroup of four wavefronts.
//
// Measured, fp32, 6 radial functions, l_max 4, 40 neurons, one species: 108 atoms with 72 neighbours 19.6 -> 16.0 us, 1000 22.3 ->
// 18.3 (fp64 22.7 -> 19.9, 26.4 -> 22.9), by first slots and tables all on their way at the start (0.8 us) and by as many
// registers as it asks for (with the 128 of four wavefronts per SIMD 42 values are spilled).
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

constexpr int NW_THREADS = 256, NW_WAVES = NW_THREADS / 64;
constexpr int NW_CAP = 128;                  // slots of a row per tile
constexpr int KC = 8, NAC = 4;
constexpr int WROW = 28;                     // row of w0 in LDS: 16-byte reads by 8 lanes with consecutive rows touch
                                             // each bank once
constexpr int CPAD = 4;                      // values behind the coefficients of a species pair (bank spread)

template <typename T>
struct WaveLds {
    T *w0, *coef, *b0, *w1, *qs;     // model tables, shared by the workgroup
    double* red;
    T *ent, *ang, *q, *dq, *sde, *cc;       // of the wavefront: tile, angular forces of its front, read-out scratch
    int* pos;
};

template <typename T>
__host__ __device__ __forceinline__ size_t wave_lds_layout(int nt, int H, int nb, int wave, unsigned char* base,
                                                           WaveLds<T>& L)
{
    size_t off = 0;
    auto take = [&](size_t n, size_t size) {
        unsigned char* p = base + off;
        off += (n * size + 15) / 16 * 16;
        return p;
    };
    L.w0 = (T*)take((size_t)nt * H * WROW, sizeof(T));
    L.coef = (T*)take((size_t)nt * nt * (nb * KC + CPAD), sizeof(T));
    L.b0 = (T*)take((size_t)nt * H, sizeof(T));
    L.w1 = (T*)take((size_t)nt * H, sizeof(T));
    L.qs = (T*)take(WROW, sizeof(T));
    L.red = (double*)take(NW_WAVES * 10, sizeof(double));
    const size_t shared = off;
    L.ent = (T*)take(NW_CAP * 4, sizeof(T));
    L.ang = (T*)take(NW_CAP * 3, sizeof(T));
    L.pos = (int*)take(NW_CAP, sizeof(int));
    L.q = (T*)take(WROW, sizeof(T));
    L.dq = (T*)take(WROW, sizeof(T));
    L.sde = (T*)take(H, sizeof(T));
    L.cc = (T*)take(nt * KC, sizeof(T));
    const size_t own = off - shared;
    const size_t shift = own * wave;
    L.ent = (T*)((unsigned char*)L.ent + shift); L.ang = (T*)((unsigned char*)L.ang + shift);
    L.pos = (int*)((unsigned char*)L.pos + shift); L.q = (T*)((unsigned char*)L.q + shift);
    L.dq = (T*)((unsigned char*)L.dq + shift); L.sde = (T*)((unsigned char*)L.sde + shift);
    L.cc = (T*)((unsigned char*)L.cc + shift);
    return shared + own * NW_WAVES;
}

// Slots [128 t, 128 t + 128) of a row, of which `room` are read: lane = slot, both halves in flight.
template <typename T>
struct Slots {
    int nj[2], tj[2];
    T x[2], y[2], z[2];
};
template <typename T>
__device__ __forceinline__ void load_slots(const NepArgs<T>& a, int t, int lane, size_t row, int room, Slots<T>& o)
{
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int slot = t * NW_CAP + h * 64 + lane;
        o.nj[h] = -1;
        o.x[h] = o.y[h] = o.z[h] = (T)0;
        if (slot < room) {
            const size_t pr = row * a.U + slot;
            o.nj[h] = a.bfirstneigh[pr];
            const T* p = a.brcs + pr * 3;
            o.x[h] = p[0]; o.y[h] = p[1]; o.z[h] = p[2];
        }
    }
}
// ... and the species of the neighbours
template <typename T>
__device__ __forceinline__ void load_species(const int* types, int NF, Slots<T>& o)
{
#pragma unroll
    for (int h = 0; h < 2; h++) o.tj[h] = (unsigned)o.nj[h] < (unsigned)NF ? types[o.nj[h]] : -1;
}
// They into the wavefront's tile; nA / nR: entries at its front / back.
template <typename T>
__device__ __forceinline__ void load_tile(const NepArgs<T>& a, const SegArgs& seg, T* __restrict__ seg_g,
                                          const WaveLds<T>& L, int t, int lane, size_t row, int b, int NF, int nn, T rr,
                                          T ra, bool claim, const Slots<T>& in, int& nA, int& nR)
{
    const unsigned long long lt = (1ull << lane) - 1ull;
    nA = 0; nR = 0;
    const int (&nj)[2] = in.nj;
    const T (&x)[2] = in.x, (&y)[2] = in.y, (&z)[2] = in.z;
    int tj[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int slot = t * NW_CAP + h * 64 + lane;
        const bool bad = slot < nn && (unsigned)nj[h] >= (unsigned)NF;
        if (bad) atomicOr(a.status, ST_BAD_NEIGHBOR);
        tj[h] = slot < nn && !bad ? in.tj[h] : -1;
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        if (t * NW_CAP + h * 64 >= nn) break;          // uniform
        const int slot = t * NW_CAP + h * 64 + lane;
        const bool valid = slot < nn && (unsigned)nj[h] < (unsigned)NF;
        if (valid && (unsigned)tj[h] >= (unsigned)a.ntypes) { atomicOr(a.status, ST_BAD_TYPE); tj[h] = 0; }
        T unused;
        const T r = length<true>(x[h] * x[h] + y[h] * y[h] + z[h] * z[h], unused);
        const bool inA = valid && r <= ra && r <= rr;   // nepBasis.h:106, 135: beyond the radial cutoff a neighbour is skipped
        const bool inR = valid && !inA && r <= rr;
        int pos = 0;
        // A pair beyond the cutoffs (a list with a skin) needs no place in this call; when the places are kept with
        // the list it has one all the same and stores a zero.
        if (valid && claim && seg.cursor && (inA || inR || a.brank)) {
            const size_t pr = row * a.U + slot;
            const int tg = b * NF + nj[h];
            int rk;
            if (a.brank && a.ranks_valid) {
                rk = a.brank[pr];
            } else {
                rk = pair_claim(&seg.cursor[tg]);
                if (a.brank) a.brank[pr] = rk;
            }
            pos = (unsigned)rk < (unsigned)seg.cap ? tg * seg.cap + rk : seg.spare;
            if ((unsigned)rk >= (unsigned)seg.cap) atomicOr(a.status, ST_SEG_OVERFLOW);
            if (!(inA || inR)) {
                T* dst = seg_g + (size_t)pos * 3;
                dst[0] = (T)0; dst[1] = (T)0; dst[2] = (T)0;
            }
        }
        const unsigned long long mA = __ballot(inA), mR = __ballot(inR);
        if (inA || inR) {
            const int k = inA ? nA + __popcll(mA & lt) : NW_CAP - 1 - (nR + __popcll(mR & lt));
            ent_store(L.ent + k * 4, x[h], y[h], z[h], tj[h]);
            L.pos[k] = pos;
        }
        nA += __popcll(mA);
        nR += __popcll(mR);
    }
    __builtin_amdgcn_wave_barrier();
}

template <typename T, int NR, int LC>
__global__ void __launch_bounds__(NW_THREADS, 1)
nep_wave_kernel(const NepArgs<T> a, const SegArgs seg, T* __restrict__ seg_g)
{
    constexpr int NLM = LC * LC + 2 * LC, NB = NR + NAC, D = NR + NAC * LC, CROW = NB * KC + CPAD;
    static_assert(D <= WROW, "descriptor count exceeds the padded row");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.y, H = a.H, nt = a.ntypes, NF = a.P + a.nghost;
    WaveLds<T> L;
    wave_lds_layout<T>(nt, H, NB, wave, smem_raw, L);

    // What the wavefront's first atom begins with, on its way while the tables are: the atom, its number of neighbours, its
    // first 128 slots (whether they hold a neighbour or not).
    const int first = blockIdx.x * NW_WAVES + wave;
    const size_t row1 = (size_t)b * a.P + min(first, a.P - 1);
    const int center1 = a.bilist[row1], nn1 = a.bnumneigh[row1];
    Slots<T> slots;
    load_slots<T>(a, 0, lane, row1, a.U, slots);
    const int* const types = a.btypes + (size_t)b * NF;
    int ti1, inum;
    stage_tables<KC, NB, D, WROW, CPAD, sizeof(T) == 4 ? 16 : 8, T>(a, L, tid, NW_THREADS, [&]() __attribute__((always_inline)) {
        ti1 = types[(unsigned)center1 < (unsigned)NF ? center1 : 0];
        load_species<T>(types, NF, slots);
        inum = min(uniform_array(a.binum)[b], a.P);   // (the loop below strides over the rows: none beyond the last)
    });
    __syncthreads();

    const T rr = a.rr, ra = a.ra, rr_inv = (T)1 / rr, ra_inv = (T)1 / ra;
    const bool derivs = a.force != nullptr || a.want_virial;
    const int quad = lane >> 2, chan = lane & 3;       // neighbour within a round of 16, angular channel
    double e_sum = 0.0, v_sum[9];
#pragma unroll
    for (int i = 0; i < 9; i++) v_sum[i] = 0.0;

    for (int ii = first; ii < inum; ii += gridDim.x * NW_WAVES) {
        const size_t row = (size_t)b * a.P + ii;
        int center = ii == first ? center1 : a.bilist[row], nn = ii == first ? nn1 : a.bnumneigh[row];
        if (nn > a.U) { if (lane == 0) atomicOr(a.status, ST_NEIGH_OVERFLOW); nn = a.U; }
        if ((unsigned)center >= (unsigned)NF) { if (lane == 0) atomicOr(a.status, ST_BAD_NEIGHBOR); center = 0; nn = 0; }
        int ti = ii == first && center == center1 ? ti1 : types[center];
        if ((unsigned)ti >= (unsigned)nt) { if (lane == 0) atomicOr(a.status, ST_BAD_TYPE); ti = 0; nn = 0; }
        const int ntiles = (nn + NW_CAP - 1) / NW_CAP;
        const T* const cti = L.coef + (size_t)ti * nt * CROW;

        // ---- radial sums, angular moments ------------------------------------------------------------
        T S[NLM], q[NR];
#pragma unroll
        for (int m = 0; m < NLM; m++) S[m] = (T)0;
#pragma unroll
        for (int n = 0; n < NR; n++) q[n] = (T)0;
        int nA = 0, nR = 0;
        for (int t = 0; t < ntiles; t++) {
            // (a row of several tiles is read again for the forces, and its pairs claim their places then)
            if (t > 0 || ii != first) {
                load_slots<T>(a, t, lane, row, nn, slots);
                load_species<T>(types, NF, slots);
            }
            load_tile<T>(a, seg, seg_g, L, t, lane, row, b, NF, nn, rr, ra, ntiles == 1, slots, nA, nR);
            for (int e = lane; e < nA + nR; e += 64) {
                T x, y, z;
                int tj;
                ent_load(L.ent + (e < nA ? e : NW_CAP - 1 - (e - nA)) * 4, x, y, z, tj);
                T f[KC], df[KC];
                T unused;
                radial_basis<T, KC, false>(length<true>(x * x + y * y + z * z, unused), rr_inv, KC, f, df);
                const T* c = cti + tj * CROW;
#pragma unroll
                for (int n = 0; n < NR; n++) {
                    T c0[4], c1[4];
                    lds_load4(c + n * KC, c0);
                    lds_load4(c + n * KC + 4, c1);
#pragma unroll
                    for (int k = 0; k < 4; k++) q[n] += c0[k] * f[k];
#pragma unroll
                    for (int k = 0; k < 4; k++) q[n] += c1[k] * f[4 + k];
                }
            }
            for (int e0 = 0; e0 < nA; e0 += 16) {
                const int e = e0 + quad;
                T x, y, z;
                int tj;
                ent_load(L.ent + min(e, nA - 1) * 4, x, y, z, tj);
                T rinv;
                const T r = length<false>(x * x + y * y + z * z, rinv);
                T f[KC], df[KC];
                radial_basis<T, KC, false>(r, ra_inv, KC, f, df);
                T c0[4], c1[4], g = (T)0;
                lds_load4(cti + tj * CROW + (NR + chan) * KC, c0);
                lds_load4(cti + tj * CROW + (NR + chan) * KC + 4, c1);
#pragma unroll
                for (int k = 0; k < 4; k++) g += c0[k] * f[k];
#pragma unroll
                for (int k = 0; k < 4; k++) g += c1[k] * f[4 + k];
                if (e >= nA) g = (T)0;
                T bl[NLM];
                blm_values<T, LC>(x * rinv, y * rinv, z * rinv, bl);
#pragma unroll
                for (int m = 0; m < NLM; m++) S[m] += g * bl[m];
            }
            __builtin_amdgcn_wave_barrier();          // the tile is overwritten by the next one
        }
#pragma unroll
        for (int n = 0; n < NR; n++) q[n] = all_sum(q[n]);
#pragma unroll
        for (int m = 0; m < NLM; m++) S[m] = sum_over_quads(S[m]);

        // ---- descriptors: the radial ones in every lane, the angular ones of a channel in its lanes -----------
#pragma unroll
        for (int n = 0; n < NR; n++)
            if (lane == n) L.q[n] = q[n];
        // q_{n,l} = sum_m w_m C_lm S^2  (nepBasis.h:174-190)
#pragma unroll
        for (int l = 1; l <= LC; l++) {
            T acc = (T)0;
#pragma unroll
            for (int mp = 0; mp < 2 * l + 1; mp++) {
                const int m = l * l - 1 + mp;
                acc += (T)(mp == 0 ? 1.0 : 2.0) * (T)kC3B[m] * S[m] * S[m];
            }
            if (lane < NAC) L.q[NR + chan * LC + (l - 1)] = acc;
        }
        __builtin_amdgcn_wave_barrier();
        if (lane < D) {
            const T v = L.q[lane];
            if (a.desc) a.desc[row * D + lane] = v;
            L.q[lane] = v * L.qs[lane];
        } else if (lane < WROW) {
            L.q[lane] = (T)0;
        }
        __builtin_amdgcn_wave_barrier();

        // ---- hidden layer (nep.h:415-447): lane = neuron -------------------------------------------------
        T e_site = (T)0;
        for (int p = lane; p < H; p += 64) {
            const T* wrow = L.w0 + (size_t)(ti * H + p) * WROW;
            T h = L.b0[ti * H + p];
#pragma unroll
            for (int j = 0; j < D; j += 4) {
                T w[4], v[4];
                lds_load4(wrow + j, w);
                lds_load4(L.q + j, v);
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (j + i < D) h += w[i] * v[i];
            }
            const T th = tanh_t(h), w1p = L.w1[ti * H + p];
            e_site += w1p * th;
            L.sde[p] = w1p * ((T)1 - th * th);
        }
        e_site = all_sum(e_site) + a.bias[ti];
        e_sum += (double)e_site;
        if (!derivs) { __builtin_amdgcn_wave_barrier(); continue; }
        __builtin_amdgcn_wave_barrier();
        {
            // dE/dq: lane = (descriptor, half of the neurons); the halves meet in lanes 0 .. D-1
            const int half = lane >> 5, d = lane & 31;
            T acc = (T)0;
            if (d < D) {
                const T* col = L.w0 + (size_t)ti * H * WROW + d;
                const int mid = (H + 1) / 2, p1 = half ? H : mid;
#pragma unroll 5
                for (int p = half ? mid : 0; p < p1; p++) acc += L.sde[p] * col[(size_t)p * WROW];
            }
            acc = add_rows<32>(acc);
            if (lane < D) L.dq[lane] = acc * L.qs[lane];
        }
        __builtin_amdgcn_wave_barrier();

        // ---- dE/dS (nep.h:450-466), overwriting S; radial coefficients contracted with dE/dq ---------------
#pragma unroll
        for (int l = 1; l <= LC; l++) {
            const T dl = L.dq[NR + chan * LC + (l - 1)];
#pragma unroll
            for (int mp = 0; mp < 2 * l + 1; mp++) {
                const int m = l * l - 1 + mp;
                S[m] *= dl * (T)(mp == 0 ? 2.0 : 4.0) * (T)kC3B[m];
            }
        }
        for (int i = lane; i < nt * KC; i += 64) {
            const T* c = cti + (i >> 3) * CROW + (i & 7);
            T v = (T)0;
#pragma unroll
            for (int n = 0; n < NR; n++) v += L.dq[n] * c[n * KC];
            L.cc[i] = v;
        }
        __builtin_amdgcn_wave_barrier();

        // ---- pair derivatives ------------------------------------------------------------------------------
        T fx = (T)0, fy = (T)0, fz = (T)0, vir[9];
#pragma unroll
        for (int i = 0; i < 9; i++) vir[i] = (T)0;
        for (int t = 0; t < ntiles; t++) {
            if (ntiles > 1) {
                load_slots<T>(a, t, lane, row, nn, slots);
                load_species<T>(types, NF, slots);
                load_tile<T>(a, seg, seg_g, L, t, lane, row, b, NF, nn, rr, ra, true, slots, nA, nR);
            }
            for (int e0 = 0; e0 < nA; e0 += 16) {
                const int e = e0 + quad;
                T x, y, z;
                int tj;
                ent_load(L.ent + min(e, nA - 1) * 4, x, y, z, tj);
                T rinv;
                const T r = length<false>(x * x + y * y + z * z, rinv);
                const T ux = x * rinv, uy = y * rinv, uz = z * rinv;
                T f[KC], df[KC];
                radial_basis<T, KC, true>(r, ra_inv, KC, f, df);
                T c0[4], c1[4], g = (T)0, dg = (T)0;
                lds_load4(cti + tj * CROW + (NR + chan) * KC, c0);
                lds_load4(cti + tj * CROW + (NR + chan) * KC + 4, c1);
#pragma unroll
                for (int k = 0; k < 4; k++) { g += c0[k] * f[k]; dg += c0[k] * df[k]; }
#pragma unroll
                for (int k = 0; k < 4; k++) { g += c1[k] * f[4 + k]; dg += c1[k] * df[4 + k]; }
                T bl[NLM];
                blm_values<T, LC>(ux, uy, uz, bl);
                T sb = (T)0, wx, wy, wz, gx, gy, gz;
#pragma unroll
                for (int m = 0; m < NLM; m++) sb += S[m] * bl[m];
                blm_gradient<T, LC>(ux, uy, uz, S, wx, wy, wz);
                pair_gradient(dg * sb, wx, wy, wz, ux, uy, uz, g * rinv, gx, gy, gz);
                gx = quad_sum(gx); gy = quad_sum(gy); gz = quad_sum(gz);
                if (e < nA && chan == 0) { L.ang[e * 3] = gx; L.ang[e * 3 + 1] = gy; L.ang[e * 3 + 2] = gz; }
            }
            __builtin_amdgcn_wave_barrier();
            for (int e = lane; e < nA + nR; e += 64) {
                const int k = e < nA ? e : NW_CAP - 1 - (e - nA);
                T x, y, z;
                int tj;
                ent_load(L.ent + k * 4, x, y, z, tj);
                T rinv;
                const T r = length<false>(x * x + y * y + z * z, rinv);
                T f[KC], df[KC];
                radial_basis<T, KC, true>(r, rr_inv, KC, f, df);
                T c0[4], c1[4], sr = (T)0;
                lds_load4(L.cc + tj * KC, c0);
                lds_load4(L.cc + tj * KC + 4, c1);
#pragma unroll
                for (int i = 0; i < 4; i++) sr += c0[i] * df[i];
#pragma unroll
                for (int i = 0; i < 4; i++) sr += c1[i] * df[4 + i];
                sr *= rinv;
                T gx = sr * x, gy = sr * y, gz = sr * z;
                if (e < nA) { gx += L.ang[e * 3]; gy += L.ang[e * 3 + 1]; gz += L.ang[e * 3 + 2]; }
                if (seg_g) {
                    T* dst = seg_g + (size_t)L.pos[k] * 3;
                    dst[0] = gx; dst[1] = gy; dst[2] = gz;
                }
                fx += gx; fy += gy; fz += gz;
                vir[0] -= gx * x; vir[1] -= gx * y; vir[2] -= gx * z;
                vir[3] -= gy * x; vir[4] -= gy * y; vir[5] -= gy * z;
                vir[6] -= gz * x; vir[7] -= gz * y; vir[8] -= gz * z;
            }
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int i = 0; i < 9; i++) v_sum[i] += (double)vir[i];
        if (a.force) {
            fx = all_sum(fx); fy = all_sum(fy); fz = all_sum(fz);
            if (lane < 3) a.force[((size_t)b * NF + center) * 3 + lane] = lane == 0 ? fx : lane == 1 ? fy : fz;
            if (seg.mark && lane == 3) pair_mark_own(&seg.cursor[b * NF + center]);
        }
    }

    // ---- workgroup partial sums of energy and virial (fp64) ---------------------------------
    if (lane == 0) L.red[wave * 10] = e_sum;
#pragma unroll
    for (int i = 0; i < 9; i++) {
        const double v = all_sum(v_sum[i]);
        if (lane == 0) L.red[wave * 10 + 1 + i] = v;
    }
    __syncthreads();
    if (tid < 10) {
        double v = 0.0;
        for (int w = 0; w < NW_WAVES; w++) v += L.red[w * 10 + tid];
        a.partial[ev_partial(a.nblocks, b, blockIdx.x, tid)] = v;
    }
}

template <typename T, int NR, int LC>
int launch_wave(const NepArgs<T>& a, size_t lds, const PairCsr& csr, hipStream_t stream)
{
    SegArgs seg{csr.cursor, csr.seg_cap, csr.n * csr.seg_cap, csr.mark};
    auto kern = nep_wave_kernel<T, NR, LC>;
    if (lds > 48 * 1024)
        A2P_HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    prof_begin("nep_wave_kernel", stream);
    hipLaunchKernelGGL(kern, dim3(a.nblocks, a.B), dim3(NW_THREADS), lds, stream, a, seg, (T*)csr.seg_g);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

}  // namespace

// Workgroups per structure: an atom per wavefront until the batch has some 1024 workgroups (four per compute unit), from
// there on several, so that the tables are staged once for all of them.
int nep_wave_nblocks(int P, int B)
{
    return std::max(1, std::min(ceil_div(P, NW_WAVES), 1024 / std::max(B, 1)));
}

template <typename T>
bool nep_wave_supported(const NepArgs<T>& a, size_t* lds_bytes)
{
    if (!(a.K == KC && (a.n_r == 4 || a.n_r == 6) && a.n_a == NAC && (a.l_max == 3 || a.l_max == 4))) return false;
    WaveLds<T> unused;
    *lds_bytes = wave_lds_layout<T>(a.ntypes, a.H, a.n_r + NAC, 0, nullptr, unused);
    return *lds_bytes <= 150 * 1024;
}

template <typename T>
int nep_wave_run(const NepArgs<T>& a, size_t lds_bytes, T* etot, T* virial, hipStream_t stream)
{
    PairCsr csr;
    int rc;
    if (a.force) {
        rc = pair_fixed_begin<T>(&csr, a.B, a.P, a.U, a.nghost, stream, a.force, a.bincoming,
                                 a.bincoming != nullptr && a.ranks_valid != 0);
        if (rc) return rc;
    }
    if (a.n_r == 4) rc = a.l_max == 3 ? launch_wave<T, 4, 3>(a, lds_bytes, csr, stream) : launch_wave<T, 4, 4>(a, lds_bytes, csr, stream);
    else rc = a.l_max == 3 ? launch_wave<T, 6, 3>(a, lds_bytes, csr, stream) : launch_wave<T, 6, 4>(a, lds_bytes, csr, stream);
    if (rc) return rc;
    if (a.force) return pair_csr_finish<T>(a.force, csr, stream, etot, virial, a.partial, a.B, a.nblocks);
    return finish_energy_virial<T>(etot, virial, a.partial, a.B, a.nblocks, stream);
}

template bool nep_wave_supported<float>(const NepArgs<float>&, size_t*);
template bool nep_wave_supported<double>(const NepArgs<double>&, size_t*);
template int nep_wave_run<float>(const NepArgs<float>&, size_t, float*, float*, hipStream_t);
template int nep_wave_run<double>(const NepArgs<double>&, size_t, double*, double*, hipStream_t);

}  // namespace a2p
