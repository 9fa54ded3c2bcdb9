// Gradient of the NEP training loss, one wavefront per atom, for the common model shapes (chebyshev_size 8, n_radial 4 or
// 6, n_angular 4, l_max 3 or 4).  The formulas and their names (alpha, beta, a, b, sigma, tau, P, Q) stand in nep_loss.hip.
//
// Every sum over an atom's neighbours is a small matrix product and runs on the matrix cores (16 x 16 x 4, the precision
// of the call; A is [row][pair], or [row][component] with the pairs as columns):
//   F, Fdot    [species][pair] one-hot  x  [pair][f_k | f'_k (u.w)]
//   S, Sdot    [g_n | g'_n (u.w)][pair]  x  [pair][Y_lm | Ydot_lm]
//   P, Q       [sigma tau ; tau 0][lm]  x  [lm][pair]
//   dc         [(species, n)][pair] of P and Q  x  [pair][fa_k], [fa'_k]
// The vector ALUs compute the table of an angular pair (Y, Ydot, basis functions) with lane = pair, 32 pairs at a time,
// and the hidden layer with lane = neuron, then lane = (descriptor, half of the neurons).  While a row has at most 64 pairs
// of which at most 32 are inside the angular cutoff, the table of the first pass still stands in the second.
// dPhi/dW0 = sum over the atoms of a species of alpha q^T + beta qdot^T is left to the second kernel, as a matrix product
// over the atoms: an atom's row carries the four vectors (144 values at 50 neurons) instead of the product (1100).
//
// Bound: issue of the vector instructions and the chain of an atom, with two workgroups (fp64: one) of four wavefronts per
// compute unit (LDS).  64 structures of 128 atoms, fp32, 3 species, 50 neurons: 179 -> 59 us against 128 threads per atom, and
// 25 -> 9.8 us for the sums over the atoms.  59 -> 52 by the next atom's first slots and the tables on their way early (tables
// 8.9 -> 5.1 thousand cycles) and by a descriptor's moments read together (4.5 -> 2.3 of 25.6 thousand cycles an atom).
#include "a2p_common.h"
#include "nep_device.h"
#include "nep_loss.h"
#include "wave_ops.h"
#include <climits>

namespace a2p {
using namespace nepdev;
using namespace wave;
namespace {

constexpr int LW_THREADS = 256, LW_WAVES = LW_THREADS / 64;
// Workgroups per compute unit, what the LDS leaves: 53 KB of an fp32 workgroup's wavefronts and the tables, twice that in fp64.
// A bound of two in fp64 buys no second workgroup and costs the loop over the atoms up to 63 spilled registers; and a grid for
// two of them loads the tables a second time, with half of the atoms.  64 structures of 128 atoms, fp64, 3 species: 135 -> 117
// us by the registers, -> 113 by the grid; 5 of 500: 71 -> 61 -> 48; 8 of 60 (one atom per wavefront): 21 -> 18.
template <typename T>
constexpr int LW_GROUPS = sizeof(T) == 4 ? 2 : 1;
constexpr int KC = 8, NAC = 4;
constexpr int WROW = 28;                     // row of w0 in LDS: see nep_wave.hip
constexpr int CPAD = 4;
constexpr int CH = 32;                       // angular pairs per table
constexpr int TS = 52;                       // row of the table, [Y 24 | Ydot 24]: 16 rows by 4 columns, and 4 rows four apart
                                             // by 16 columns, touch each bank once
constexpr int RS = 2 * KC;                   // row of the radial table: consecutive rows fill the banks in turn
constexpr int LM = 24;

template <typename T>
struct LossWaveLds {
    T *w0, *coef, *b0, *w1, *qs, *wc;        // model tables, shared by the workgroup
    T *tab, *G, *SS, *F, *gca, *ent, *W, *q, *ab, *alpha, *beta;
    int *tj, *tja;                           // species of the slots and of the angular pairs
};

template <typename T>
__host__ __device__ __forceinline__ size_t loss_wave_layout(int nt, int H, int nb, int wave, unsigned char* base,
                                                            LossWaveLds<T>& L)
{
    T* p = (T*)base;
    auto take = [&](size_t n) { T* r = p; p += (n + 3) / 4 * 4; return r; };
    L.w0 = take((size_t)nt * H * WROW);
    L.coef = take((size_t)nt * nt * (nb * KC + CPAD));
    L.b0 = take((size_t)nt * H);
    L.w1 = take((size_t)nt * H);
    L.qs = take(WROW);
    L.wc = take(LM);
    T* const own = p;
    L.tab = take(CH * TS);                   // (holds the radial table of 64 slots before the angular one)
    L.G = take(CH * 8);
    L.SS = take(8 * TS);
    L.F = take(nt * RS);
    L.gca = take(nt * NAC * KC);
    L.ent = take(64 * 4);
    L.W = take(64 * 4);
    L.q = take(2 * WROW);
    L.ab = take(2 * WROW);
    L.alpha = take(H);
    L.beta = take(H);
    L.tj = (int*)p;
    L.tja = L.tj + 64;
    const size_t n = (size_t)(p - own) + 128 * sizeof(int) / sizeof(T), shift = n * wave;
    L.tab += shift; L.G += shift; L.SS += shift; L.F += shift; L.gca += shift; L.ent += shift; L.W += shift;
    L.q += shift; L.ab += shift; L.alpha += shift; L.beta += shift;
    L.tj = (int*)((T*)L.tj + shift); L.tja = (int*)((T*)L.tja + shift);
    return ((size_t)(own - (T*)base) + n * LW_WAVES) * sizeof(T);
}
static_assert(CH * TS >= 64 * RS, "the radial table uses the angular one's place");

template <typename T, int NR, int LC>
__global__ void __launch_bounds__(LW_THREADS, LW_GROUPS<T>) nep_loss_wave_kernel(const NepLossArgs<T> a)
{
    constexpr int NLM = LC * LC + 2 * LC, NB = NR + NAC, D = NR + NAC * LC, CROW = NB * KC + CPAD;
    static_assert(D <= WROW && D <= 32, "descriptor count exceeds the padded row");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, k4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.y, H = a.H, nt = a.ntypes;
    LossWaveLds<T> L;
    loss_wave_layout<T>(nt, H, NB, wave, smem_raw, L);
    // What the next atom begins with, on its way while the one before is worked on: the atom, its number of neighbours, its
    // first 64 slots (whether they hold a neighbour or not).
    int center1, nn1, nj1;
    T x1, y1, z1;
    auto begin = [&](int ii) __attribute__((always_inline)) {
        const size_t row = (size_t)b * a.P + min(ii, a.P - 1), pr = row * a.U + min(lane, a.U - 1);
        center1 = a.bilist[row];
        nn1 = a.bnumneigh[row];
        nj1 = a.bfirstneigh[pr];
        x1 = a.brcs[pr * 3]; y1 = a.brcs[pr * 3 + 1]; z1 = a.brcs[pr * 3 + 2];
    };
    begin(blockIdx.x * LW_WAVES + wave);
    int inum;
    T cE;
    stage_tables<KC, NB, D, WROW, CPAD, sizeof(T) == 4 ? 16 : 8, T>(a, L, tid, LW_THREADS, [&]() __attribute__((always_inline)) {
        inum = min(uniform_array(a.binum)[b], a.P);
        cE = uniform_array(a.cE)[b];
    });
    if (tid < LM) {
        const int l = l_of_lm(tid);
        L.wc[tid] = tid < NLM ? (T)(tid == l * l - 1 ? 1.0 : 2.0) * (T)kC3B[tid] : (T)0;
    }
    const int* types = a.btypes + (size_t)b * a.P;
    // The species of the next atom is asked for ahead of its turn too.
    auto species = [&]() __attribute__((always_inline)) { return types[(unsigned)center1 < (unsigned)a.P ? center1 : 0]; };
    int ti1 = species();
    __syncthreads();

    const T rr = a.rr, ra = a.ra, rr_inv = (T)1 / rr, ra_inv = (T)1 / ra;
    const T* dv = a.dVs + (size_t)b * 9;
    const unsigned long long lt = (1ull << lane) - 1ull;

    for (int ii = blockIdx.x * LW_WAVES + wave; ii < inum; ii += gridDim.x * LW_WAVES) {
        const size_t row = (size_t)b * a.P + ii;
        int center = center1, nn = nn1;
        if (nn > a.U) { if (lane == 0) atomicOr(a.status, ST_NEIGH_OVERFLOW); nn = a.U; }
        if ((unsigned)center >= (unsigned)a.P) { if (lane == 0) atomicOr(a.status, ST_BAD_NEIGHBOR); center = 0; nn = 0; }
        int ti = center == center1 ? ti1 : types[center];
        if ((unsigned)ti >= (unsigned)nt) { if (lane == 0) atomicOr(a.status, ST_BAD_TYPE); ti = 0; nn = 0; }
        if (nn == 0) begin(ii + gridDim.x * LW_WAVES);        // (no first slots below, behind which the next row is fetched)
        const T* const cti = L.coef + (size_t)ti * nt * CROW;
        T* const grow = a.gpart + row * a.nrow;
        T* const g_alpha = grow + nt * NB * KC;

        for (int o = lane; o < nt * RS; o += 64) L.F[o] = (T)0;
        for (int o = lane; o < nt * NAC * KC; o += 64) L.gca[o] = (T)0;
        typename Acc<T>::type s[3];
#pragma unroll
        for (int t = 0; t < 3; t++) s[t] = {0, 0, 0, 0};
        T fa[KC], fad[KC];                             // of the lane's angular pair
        int nA = 0;

#pragma unroll 1
        for (int pass = 0; pass < 2; pass++) {
#pragma unroll 1
            for (int slot0 = 0; slot0 < nn; slot0 += 64) {
                if (pass == 0 || nn > 64) {
                    // ---- 64 slots: displacement, residual field w, angular pairs compacted; the radial sums
                    const int slot = slot0 + lane;
                    T x = (T)1, y = (T)0, z = (T)0, w[3] = {(T)0, (T)0, (T)0};
                    int tj = -1;
                    int nj = nj1;
                    if (slot < nn) { x = x1; y = y1; z = z1; }
                    if ((pass > 0 || slot0 > 0) && slot < nn) {
                        const size_t pr = row * a.U + slot;
                        nj = a.bfirstneigh[pr];
                        x = a.brcs[pr * 3]; y = a.brcs[pr * 3 + 1]; z = a.brcs[pr * 3 + 2];
                    }
                    if (pass == 0 && slot0 == 0) begin(ii + gridDim.x * LW_WAVES);
                    if (slot < nn) {
                        if ((unsigned)nj >= (unsigned)a.P) { atomicOr(a.status, ST_BAD_NEIGHBOR); nj = center; }
                        tj = types[nj];
                        const T* fc = a.dFs + ((size_t)b * a.P + center) * 3;
                        const T* fn = a.dFs + ((size_t)b * a.P + nj) * 3;
#pragma unroll
                        for (int q = 0; q < 3; q++)
                            w[q] = fc[q] - fn[q] - (dv[q * 3] * x + dv[q * 3 + 1] * y + dv[q * 3 + 2] * z);
                        if ((unsigned)tj >= (unsigned)nt) { atomicOr(a.status, ST_BAD_TYPE); tj = 0; }
                    }
                    T rinv;
                    const T r = length<false>(x * x + y * y + z * z, rinv);
                    const T uw = (w[0] * x + w[1] * y + w[2] * z) * rinv;
                    const bool in = slot < nn && r <= rr, inA = in && r <= ra;   // nepBasis.h:106, 135
                    const unsigned long long mA = __ballot(inA);
                    nA = __popcll(mA);
                    if (inA) {
                        const int k = __popcll(mA & lt);
                        ent_store(L.ent + k * 4, x, y, z, tj);
                        lds_store4(L.W + k * 4, w[0], w[1], w[2], uw);
                        L.tja[k] = tj;
                    }
                    if (pass == 0) {
                        T f[KC], df[KC];
                        radial_basis<T, KC, true>(in ? r : rr, rr_inv, KC, f, df);
#pragma unroll
                        for (int k = 0; k < KC; k++) { f[k] = in ? f[k] : (T)0; df[k] = in ? df[k] * uw : (T)0; }
                        T* t = L.tab + lane * RS;
                        lds_store4(t, f[0], f[1], f[2], f[3]);
                        lds_store4(t + 4, f[4], f[5], f[6], f[7]);
                        lds_store4(t + 8, df[0], df[1], df[2], df[3]);
                        lds_store4(t + 12, df[4], df[5], df[6], df[7]);
                        L.tj[lane] = tj;
                        __builtin_amdgcn_wave_barrier();
                        const int steps = (min(nn - slot0, 64) + 3) >> 2;
                        for (int t0 = 0; t0 < nt; t0 += 16) {
                            typename Acc<T>::type o = {0, 0, 0, 0};
                            for (int st = 0; st < steps; st++) {
                                const int k = 4 * st + k4;
                                o = mma(L.tj[k] == t0 + c16 ? (T)1 : (T)0, L.tab[k * RS + c16], o);
                            }
#pragma unroll
                            for (int v = 0; v < 4; v++) {
                                const int t_ = t0 + mma_row<T>(v, lane);
                                if (t_ < nt) L.F[t_ * RS + c16] += o[v];
                            }
                        }
                    }
                    __builtin_amdgcn_wave_barrier();
                }
#pragma unroll 1
                for (int c0 = 0; c0 < nA; c0 += CH) {
                    const int n = min(CH, nA - c0), groups = (n + 15) >> 4;
                    if ((pass == 0 || nn > 64 || nA > CH) && lane < CH) {
                        // ---- table of the angular pairs (a lane beyond the last repeats it, with zero functions)
                        T x, y, z, w[4];
                        int tj;
                        const int e = c0 + min(lane, n - 1);
                        ent_load(L.ent + e * 4, x, y, z, tj);
                        lds_load4(L.W + e * 4, w);
                        T rinv;
                        const T r = length<false>(x * x + y * y + z * z, rinv);
                        x *= rinv; y *= rinv; z *= rinv;
                        radial_basis<T, KC, true>(r, ra_inv, KC, fa, fad);
#pragma unroll
                        for (int k = 0; k < KC; k++) { fa[k] = lane < n ? fa[k] : (T)0; fad[k] = lane < n ? fad[k] : (T)0; }
                        if (pass == 0) {
                            T g[NAC], dg[NAC];
#pragma unroll
                            for (int q = 0; q < NAC; q++) {
                                T c[KC];
                                const T* src = cti + tj * CROW + (NR + q) * KC;
                                g[q] = (T)0; dg[q] = (T)0;
#pragma unroll
                                for (int k = 0; k < KC; k += 4) {
                                    T cc[4];
                                    lds_load4(src + k, cc);
#pragma unroll
                                    for (int i = 0; i < 4; i++) c[k + i] = cc[i];
                                }
#pragma unroll
                                for (int k = 0; k < KC; k++) { g[q] += c[k] * fa[k]; dg[q] += c[k] * fad[k]; }
                            }
                            lds_store4(L.G + lane * 8, g[0], g[1], g[2], g[3]);
                            lds_store4(L.G + lane * 8 + 4, dg[0] * w[3], dg[1] * w[3], dg[2] * w[3], dg[3] * w[3]);
                        }
                        T Y[LM], Yd[LM], Yv[NLM], Gd[NLM];
                        blm_values<T, LC>(x, y, z, Yv);
                        blm_dir_derivs<T, LC>(x, y, z, w[0], w[1], w[2], Gd);
#pragma unroll
                        for (int m = 0; m < LM; m++) {
                            Y[m] = m < NLM ? Yv[m < NLM ? m : 0] : (T)0;
                            Yd[m] = m < NLM ? rinv * (Gd[m < NLM ? m : 0] - (T)l_of_lm(m) * Y[m] * w[3]) : (T)0;
                        }
                        T* t = L.tab + lane * TS;
#pragma unroll
                        for (int m = 0; m < LM; m += 4) {
                            lds_store4(t + m, Y[m], Y[m + 1], Y[m + 2], Y[m + 3]);
                            lds_store4(t + LM + m, Yd[m], Yd[m + 1], Yd[m + 2], Yd[m + 3]);
                        }
                    }
                    __builtin_amdgcn_wave_barrier();
                    if (pass == 0) {
                        for (int st = 0; st < 4 * groups; st++) {
                            const int k = 16 * (st >> 2) + 4 * k4 + (st & 3);
                            const T g = c16 < 8 ? L.G[k * 8 + (c16 & 7)] : (T)0;
                            const T* t = L.tab + k * TS + c16;
#pragma unroll
                            for (int q = 0; q < 3; q++) s[q] = mma(g, t[16 * q], s[q]);
                        }
                        __builtin_amdgcn_wave_barrier();
                        continue;
                    }
                    // ---- P and Q of the pairs
                    typename Acc<T>::type o[2];
                    o[0] = {0, 0, 0, 0}; o[1] = {0, 0, 0, 0};
                    const T* t0 = L.tab + c16 * TS + k4;
#pragma unroll 4
                    for (int st = 0; st < 2 * LM / 4; st++) {
                        const T sg = c16 < 8 ? L.SS[(c16 & 7) * TS + 4 * st + k4] : (T)0;
                        o[0] = mma(sg, t0[4 * st], o[0]);
                        if (groups > 1) o[1] = mma(sg, t0[16 * TS + 4 * st], o[1]);
                    }
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int et = 0; et < 2; et++) {
                        const int e = et * 16 + c16;
                        const T uw = L.W[min(c0 + e, nA - 1) * 4 + 3];
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            const int q = mma_row<T>(v, lane);
                            if (q < 8 && et < groups) L.G[e * 8 + q] = q < 4 ? o[et][v] : o[et][v] * uw;
                        }
                    }
                    if (lane < CH) {
                        T* t = L.tab + lane * TS;
                        lds_store4(t, fa[0], fa[1], fa[2], fa[3]);
                        lds_store4(t + 4, fa[4], fa[5], fa[6], fa[7]);
                        lds_store4(t + 8, fad[0], fad[1], fad[2], fad[3]);
                        lds_store4(t + 12, fad[4], fad[5], fad[6], fad[7]);
                    }
                    __builtin_amdgcn_wave_barrier();
                    // ---- their share of the angular coefficients' gradient: rows (species, n), four species at a time
                    for (int s0 = 0; s0 < nt; s0 += 4) {
                        typename Acc<T>::type d = {0, 0, 0, 0};
                        for (int st = 0; st < 4 * groups; st++) {
                            const int k = 16 * (st >> 2) + 4 * k4 + (st & 3);
                            const bool mine = L.tja[min(c0 + k, 63)] == s0 + (c16 >> 2);
                            const T pv = L.G[k * 8 + (c16 & 3)], qv = L.G[k * 8 + 4 + (c16 & 3)];
                            d = mma(mine ? pv : (T)0, L.tab[k * TS + (c16 & 7)], d);
                            d = mma(mine ? qv : (T)0, L.tab[k * TS + KC + (c16 & 7)], d);
                        }
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            const int q = s0 * NAC + mma_row<T>(v, lane);
                            if (q < nt * NAC && c16 < KC) L.gca[q * KC + c16] += d[v];
                        }
                    }
                    __builtin_amdgcn_wave_barrier();
                }
            }
            if (pass == 1) break;

            // ---- descriptors and their tangents (nepBasis.h:153-190): lane = (descriptor, value or tangent)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int q = mma_row<T>(v, lane);
                if (q < 8)
#pragma unroll
                    for (int t = 0; t < 3; t++) L.SS[q * TS + t * 16 + c16] = s[t][v];
            }
            __builtin_amdgcn_wave_barrier();
            const int half = lane >> 5, d = lane & 31;
            if (d < D) {
                T acc = (T)0;
                if (d < NR) {
#pragma unroll 2
                    for (int t = 0; t < nt; t++) {
                        const T *c = cti + t * CROW + d * KC, *f = L.F + t * RS + half * KC;
#pragma unroll
                        for (int k = 0; k < KC; k += 4) {
                            T cv[4], fv[4];
                            lds_load4(c + k, cv);
                            lds_load4(f + k, fv);
#pragma unroll
                            for (int i = 0; i < 4; i++) acc += cv[i] * fv[i];
                        }
                    }
                } else {
                    const int n = (d - NR) / LC, l = (d - NR) % LC + 1;
                    // (a degree's moments all read before they are summed; beyond its last the weight is left out)
                    const T* const sv = L.SS + n * TS + l * l - 1;
                    const T* const wc = L.wc + l * l - 1;
                    T v[2 * LC + 1], u[2 * LC + 1], w[2 * LC + 1];
#pragma unroll
                    for (int i = 0; i < 2 * LC + 1; i++) {
                        const int m = min(i, 2 * l);
                        v[i] = sv[m];
                        u[i] = sv[NAC * TS + m] + sv[LM + m];
                        w[i] = wc[m];
                    }
#pragma unroll
                    for (int i = 0; i < 2 * LC + 1; i++)
                        if (i <= 2 * l) acc += w[i] * v[i] * (half ? (T)2 * u[i] : v[i]);
                }
                acc *= L.qs[d];                        // scaled descriptor and tangent
                L.q[half * WROW + d] = acc;
                g_alpha[3 * H + half * D + d] = acc;
            } else if (d < WROW) {
                L.q[half * WROW + d] = (T)0;
            }
            __builtin_amdgcn_wave_barrier();

            // ---- hidden layer, alpha / beta, gradients of b0 (alpha itself) and w1
            for (int p = lane; p < H; p += 64) {
                const T* wrow = L.w0 + (size_t)(ti * H + p) * WROW;
                T h = L.b0[ti * H + p], hd = (T)0;
#pragma unroll
                for (int j = 0; j < D; j += 4) {
                    T wv[4], qv[4], qd[4];
                    lds_load4(wrow + j, wv);
                    lds_load4(L.q + j, qv);
                    lds_load4(L.q + WROW + j, qd);
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (j + i < D) { h += wv[i] * qv[i]; hd += wv[i] * qd[i]; }
                }
                const T t = tanh_t(h), sd = (T)1 - t * t, be = L.w1[ti * H + p] * sd;
                const T al = be * (cE - (T)2 * t * hd);
                L.alpha[p] = al; L.beta[p] = be;
                g_alpha[p] = al;
                g_alpha[H + p] = cE * t + sd * hd;
                g_alpha[2 * H + p] = be;
            }
            __builtin_amdgcn_wave_barrier();
            {
                T av = (T)0, bv = (T)0;
                if (d < D) {
                    const T* col = L.w0 + (size_t)ti * H * WROW + d;
                    const int mid = (H + 1) / 2, p1 = half ? H : mid;
#pragma unroll 5
                    for (int p = half ? mid : 0; p < p1; p++) {
                        const T wv = col[(size_t)p * WROW];
                        av += L.alpha[p] * wv; bv += L.beta[p] * wv;
                    }
                }
                av = add_rows<32>(av);
                bv = add_rows<32>(bv);
                if (lane < D) { L.ab[lane] = av * L.qs[lane]; L.ab[WROW + lane] = bv * L.qs[lane]; }
            }
            __builtin_amdgcn_wave_barrier();

            ti1 = species();                           // (of the next row, which was fetched behind the first slots of this)

            // ---- radial coefficients' gradient; [sigma tau ; tau 0] over the moments
            for (int o = lane; o < nt * NR * KC; o += 64) {
                const int t = o / (NR * KC), n = (o - t * NR * KC) / KC, k = o % KC;
                grow[(t * NB + n) * KC + k] = L.ab[n] * L.F[t * RS + k] + L.ab[WROW + n] * L.F[t * RS + KC + k];
            }
            for (int o = lane; o < NAC * LM; o += 64) {
                const int n = o / LM, m = o - n * LM;
                T sg = (T)0, ta = (T)0;
                if (m < NLM) {
                    const int dd = NR + n * LC + l_of_lm(m) - 1;
                    const T sv = L.SS[n * TS + m], sdv = L.SS[(NAC + n) * TS + m] + L.SS[n * TS + LM + m];
                    const T w2 = (T)2 * L.wc[m];
                    sg = w2 * (L.ab[dd] * sv + L.ab[WROW + dd] * sdv);
                    ta = w2 * L.ab[WROW + dd] * sv;
                }
                L.SS[n * TS + m] = sg;
                L.SS[n * TS + LM + m] = ta;
                L.SS[(NAC + n) * TS + m] = ta;
                L.SS[(NAC + n) * TS + LM + m] = (T)0;
            }
            __builtin_amdgcn_wave_barrier();
        }
        for (int o = lane; o < nt * NAC * KC; o += 64) {
            const int t = o / (NAC * KC);
            grow[(t * NB + NR) * KC + (o - t * NAC * KC)] = L.gca[o];
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Sums of the rows over the atoms of one species (blockIdx.y) of one structure (blockIdx.z).  The first workgroups take 64
// elements each of the entries that are summed as they are, a quarter of the atoms per wavefront; the others 64 rows of
// dPhi/dW0 each, a wavefront sixteen, as a matrix product over the atoms.  The atoms are gathered 256 at a time in atom
// order, so every sum has a fixed order.
template <typename T>
__global__ void __launch_bounds__(256)
nep_loss_wave_reduce_kernel(const NepLossArgs<T> a, int sum_blocks, T* __restrict__ dcoeffs, T* __restrict__ dw0,
                            T* __restrict__ db0, T* __restrict__ dw1, T* __restrict__ dbias)
{
    __shared__ int list[256], count[4];
    __shared__ T red[4][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c16 = lane & 15, k4 = lane >> 4;
    const int t = blockIdx.y, b = blockIdx.z, nt = a.ntypes, H = a.H, D = a.D;
    const int ncl = nt * (a.n_r + a.n_a) * a.K, job = blockIdx.x;
    if (job >= sum_blocks + (H + 63) / 64) {                   // (one more for the batch's errors)
        if (t == 0 && b == 0 && wave == 0) losskern::loss_rmse(a.errors, lane);
        return;
    }
    const bool sums = job < sum_blocks;
    const int e = min(job * 64 + lane, ncl + 2 * H - 1);         // element of a row
    const int p0 = (job - sum_blocks) * 64 + wave * 16, p = min(p0 + c16, H - 1);
    const int d1 = min(16 + c16, D - 1);
    const int inum = min(a.binum[b], a.P);
    const T* const rows = a.gpart + (size_t)b * a.P * a.nrow;
    T acc = (T)0;
    typename Acc<T>::type o[2];
    o[0] = {0, 0, 0, 0}; o[1] = {0, 0, 0, 0};
    int all = 0;
    for (int i0 = 0; i0 < inum; i0 += 256) {
        const int i = i0 + tid;
        bool mine = false;
        if (i < inum) {
            const int c = a.bilist[(size_t)b * a.P + i];
            mine = (unsigned)c < (unsigned)a.P && a.btypes[(size_t)b * a.P + c] == t;
        }
        const unsigned long long m = __ballot(mine);
        if (lane == 0) count[wave] = __popcll(m);
        __syncthreads();
        int before = 0, n = 0;
        for (int w = 0; w < 4; w++) { if (w < wave) before += count[w]; n += count[w]; }
        if (mine) list[before + __popcll(m & ((1ull << lane) - 1ull))] = i;
        __syncthreads();
        all += n;
        if (sums) {
            for (int k0 = wave; k0 < n; k0 += 32) {
                T v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = rows[(size_t)list[min(k0 + 4 * u, n - 1)] * a.nrow + e];
#pragma unroll
                for (int u = 0; u < 8; u++) acc += k0 + 4 * u < n ? v[u] : (T)0;
            }
        } else if (p0 < H) {
            for (int k0 = 0; k0 < n; k0 += 16) {
                T al[4], be[4], q[4][2], qd[4][2];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const T* r = rows + (size_t)list[min(k0 + 4 * u + k4, n - 1)] * a.nrow + ncl;
                    al[u] = r[p]; be[u] = r[2 * H + p];
                    q[u][0] = r[3 * H + c16]; q[u][1] = r[3 * H + d1];
                    qd[u][0] = r[3 * H + D + c16]; qd[u][1] = r[3 * H + D + d1];
                }
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const bool ok = k0 + 4 * u + k4 < n;
                    const T av = ok ? al[u] : (T)0, bv = ok ? be[u] : (T)0;
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        o[h] = mma(av, q[u][h], o[h]);
                        o[h] = mma(bv, qd[u][h], o[h]);
                    }
                }
            }
        }
        __syncthreads();
    }
    if (sums) {
        red[wave][lane] = acc;
        __syncthreads();
        if (wave == 0 && job * 64 + lane < ncl + 2 * H) {
            const T v = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
            if (e < ncl) { if (dcoeffs) dcoeffs[((size_t)b * nt + t) * ncl + e] = v; }
            else if (e < ncl + H) { if (db0) db0[((size_t)b * nt + t) * H + e - ncl] = v; }
            else { if (dw1) dw1[((size_t)b * nt + t) * H + e - ncl - H] = v; }
        }
        if (job == 0 && tid == 0 && dbias) dbias[(size_t)b * nt + t] = (T)all * a.cE[b];
    } else if (dw0) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int pr = p0 + mma_row<T>(v, lane), d = 16 * h + c16;
                if (pr < H && d < D) dw0[(((size_t)b * nt + t) * H + pr) * D + d] = o[h][v];
            }
    }
}

// Workgroups per structure: the number with the shortest way through the device, in rounds of `room` workgroups, each the
// atoms of a wavefront and the tables (a quarter of an atom: 4 of 14 us in fp64, 5 of 26 thousand cycles in fp32).  One round
// unless the batch does not divide the room well: room / B workgroups each left 129 structures of 64 atoms on half of the device
// (fp64: 208 us, now 151), 200 of 40 on 400 of the 512 places (fp32: 60 us, now 53), 300 of 30 in two rounds of which the second
// was nearly empty (fp64 244 -> 152, fp32 89 -> 70).
int loss_wave_blocks(int P, int B, int room)
{
    const int most = ceil_div(P, LW_WAVES);
    int best = 1;
    long long least = LLONG_MAX;
    for (int round = 1; round <= ceil_div(B, room) + 3; round++) {
        const int n = std::max(1, std::min<int>(most, (long long)round * room / B));
        const long long way = (long long)ceil_div((long long)n * B, (long long)room) * (4ll * ceil_div(P, n * LW_WAVES) + 1);
        if (way < least) { least = way; best = n; }
    }
    return best;
}

template <typename T, int NR, int LC>
int launch_loss_wave(const NepLossArgs<T>& a, size_t lds, hipStream_t stream)
{
    auto kern = nep_loss_wave_kernel<T, NR, LC>;
    if (lds > 48 * 1024)
        A2P_HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int nblk = loss_wave_blocks(a.P, a.B, LW_GROUPS<T> * 256);
    prof_begin("nep_loss_bwd_kernel", stream);
    hipLaunchKernelGGL(kern, dim3(nblk, a.B), dim3(LW_THREADS), lds, stream, a);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

}  // namespace

template <typename T>
bool nep_loss_wave_supported(const NepLossArgs<T>& a, size_t* lds_bytes)
{
    if (!(a.K == KC && (a.n_r == 4 || a.n_r == 6) && a.n_a == NAC && (a.l_max == 3 || a.l_max == 4))) return false;
    if (a.ntypes > 65535 || a.B > 65535) return false;
    LossWaveLds<T> unused;
    *lds_bytes = loss_wave_layout<T>(a.ntypes, a.H, a.n_r + NAC, 0, nullptr, unused);
    return *lds_bytes <= 150 * 1024;
}

template <typename T>
int nep_loss_wave_row(const NepLossArgs<T>& a)
{
    return a.ntypes * (a.n_r + a.n_a) * a.K + 3 * a.H + 2 * a.D;
}

template <typename T>
int nep_loss_wave_run(const NepLossArgs<T>& a, size_t lds_bytes, T* dcoeffs, T* dw0, T* db0, T* dw1, T* dbias,
                      hipStream_t stream)
{
    int rc;
    if (a.n_r == 4) rc = a.l_max == 3 ? launch_loss_wave<T, 4, 3>(a, lds_bytes, stream) : launch_loss_wave<T, 4, 4>(a, lds_bytes, stream);
    else rc = a.l_max == 3 ? launch_loss_wave<T, 6, 3>(a, lds_bytes, stream) : launch_loss_wave<T, 6, 4>(a, lds_bytes, stream);
    if (rc) return rc;
    const int sum_blocks = ceil_div(a.ntypes * (a.n_r + a.n_a) * a.K + 2 * a.H, 64);
    prof_begin("nep_grad_reduce", stream);
    hipLaunchKernelGGL(nep_loss_wave_reduce_kernel<T>, dim3(sum_blocks + ceil_div(a.H, 64) + (a.errors.rmse ? 1 : 0), a.ntypes, a.B), dim3(256), 0,
                       stream, a, sum_blocks, dcoeffs, dw0, db0, dw1, dbias);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

template bool nep_loss_wave_supported<float>(const NepLossArgs<float>&, size_t*);
template bool nep_loss_wave_supported<double>(const NepLossArgs<double>&, size_t*);
template int nep_loss_wave_row<float>(const NepLossArgs<float>&);
template int nep_loss_wave_row<double>(const NepLossArgs<double>&);
template int nep_loss_wave_run<float>(const NepLossArgs<float>&, size_t, float*, float*, float*, float*, float*, hipStream_t);
template int nep_loss_wave_run<double>(const NepLossArgs<double>&, size_t, double*, double*, double*, double*, double*,
                                       hipStream_t);

}  // namespace a2p
