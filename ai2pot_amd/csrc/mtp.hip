// Linear Moment Tensor Potential for gfx950: energy / force / virial, and the analytic
// gradient of the training loss w.r.t. coeffs, linear_coeffs and type_bias.
//
// One workgroup (64 threads, or 256 for the larger levels) per centre atom; the moment vector M,
// its adjoint and (for the loss gradient) the tangent and mixed vectors live in LDS.  Neighbours
// are processed in equal chunks of at most 16 to 48: a per-neighbour table (powers of the unit vector, contracted
// radial functions g_mu(r) = sum_k c[ti,tj,mu,k] f_k(r) and their r-derivatives) is staged
// in LDS, then
//   basic moments : M_(mu,a,b,c) = sum_j g_mu(r_j) ux^a uy^b uz^c as products of matrices over the neighbours, rows (a, b)
//                   and columns (mu, c)     (x^a y^b z^c / r^(a+b+c) of the reference, include/mtpBasis.h:472-519,
//                    written with the unit vector u = r_ij / r)
//   products      : level-ordered gather over the host-built plan (mtp_plan.h)
//   energy        : E_i = bias[t] + sum_s lin[s] M[map[s]] / q_scaler[s]  (linearMtp.h:281-285)
//   adjoint       : seed + reverse gather                                  (linearMtp.h:292-306)
//   pair forces   : lane <- neighbour (or half of one), wavefronts share the (mu, c):
//                   dE_i/dr_ij = u sum_i adj_i m_i (g' - k g / r) + (1/r) sum_i adj_i g grad_u m_i
//                   by polynomials nested in (x, y, z) whose coefficients are the adjoints
//                   -> reduction segments of the neighbours (a2p::PairCsr), summed without float atomics
// Tables that the products and the nested polynomials do not fit (mtp_plan.h: ntiles) go by basic moments and by polynomials in z.
// The loss gradient adds the tangent sweep (include/linearMtpLoss.h:371-398), the mixed
// adjoint (:417-434) and the coefficient-gradient pass (:438-536) in the same structure;
// per-structure gradients are accumulated per workgroup and summed by a second kernel.
#include "a2p_common.h"
#include "mtp_plan.h"
#include "loss_kernels.h"
#include "wave_ops.h"

#include <algorithm>
#include <array>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <type_traits>

namespace a2p {
namespace {

constexpr int MTP_NC = 32;        // neighbours per chunk (rows of the LDS table); the energy / force / virial
constexpr int MTP_NC_MAX = 48;    // the launch picks between MTP_NC_MIN and MTP_NC_MAX rows (launch_atoms)
constexpr int MTP_NC_MIN = 16;
constexpr int MTP_SCRATCH = 16;

// The group sums of the last pass over the neighbours (four per thread for the pair derivatives, two
// for the loss gradient) live in the moment vector (loss mode: moments and tangents) when it is long
// enough, else behind the neighbour table.
__host__ __device__ inline bool mtp_gred_in_moments(bool loss, int n_moms)
{
    return loss ? 2 * n_moms >= 512 : n_moms >= 1024;
}
// General tables (a kernel that is not TILED): entries of the region that holds the neighbour table (+ group sums).
// In the energy / force / virial kernel the group sums (4 per thread) are written over the table once every
// thread has finished reading it.
// The adjoints live in this region too: they are needed from the end of
// the forward sweep to the last pass over the neighbours, which is when the neighbour table is not.  That pass needs
// the adjoints of the basic moments only: the energy / force / virial kernel moves them to its polynomials, the
// loss kernel moves them behind the region first.
__host__ __device__ inline int mtp_table_region(int nc, int E, bool loss, int n_moms, int nt)
{
    int a = loss ? nc * E + (mtp_gred_in_moments(loss, n_moms) ? 0 : (256 / 32) * 32 * 4) : nc * E;
    if (!loss && a < nt * 4) a = nt * 4;          // four group sums per thread
    a = (a + 1) & ~1;
    const int b = (loss ? 2 : 1) * n_moms;         // loss mode: the adjoints and the mixed adjoints
    return a > b ? a : b;
}
// the coefficients of the pair-derivative pass's polynomials take the place of the moments when they fit
__host__ __device__ inline bool mtp_polys_in_moments(int ncoef, int n_moms) { return ncoef <= n_moms; }
// the tangents of a network's inputs wait in the place of P and Q (loss gradient) when they fit
__host__ __device__ inline bool mtp_tangents_at_pq(int n_scalar, int nc, int nmus) { return n_scalar <= 2 * nc * nmus + nc; }
constexpr int MTP_NGMAX = 16;     // most thread groups that share the basic moments of a chunk
constexpr int MTP_KMAX = 16;      // radial basis size limit
constexpr int MTP_NMUS_MAX = 8;   // radial function count limit
constexpr int MTP_NODE_CAP = 4094; // most (scalar moment, ancestor) nodes of one launch of the components kernel

template <typename T>
struct MtpArgs {
    MtpPlanDevice p;
    int K, ntypes;
    T scaling, rmax, rmin, inv_span;     // inv_span = 1 / (rmax - rmin)
    const T *coeffs, *lin, *bias, *q_scaler;
    int B, P, U, nghost;
    const int *binum, *bilist, *bnumneigh, *bfirstneigh;
    const T* brcs;
    const int* btypes;
    T* force;          // [B, P+nghost, 3]
    int* seg_cursor;   // reduction segments of fixed capacity U (a2p::PairCsr): entries claimed per target,
    T* seg_g;          // the entries, and the entry that takes what overflows a segment;
    int seg_spare;     // seg_cursor is null when no forces are wanted
    int seg_cap;       // capacity of a segment
    int seg_mark;      // own sums are marked in the cursors
    double* partial;   // energy and virial per atom (ev_partial, a block per row)
    int* status;
    int E;             // table entries per neighbour
    // loss gradient mode
    const T* cE;       // [B]        2 e_w / N (E - E_dft)
    const T* dFs;      // [B, P, 3]  2 f_w / (3N) (F - F_dft)
    const T* dVs;      // [B, 9]     2 v_w / (9N) (V - V_dft)
    T* gpart;          // [B, P, ngrad] per-atom gradient rows: coefficient block of the centre's species | bias | linear coefficients
    int ngrad;
    // Places in LDS, in entries (AtomLds), and in a row of the neighbour table: worked out once for the launch.
    int at_Tg, at_cf, at_tab, at_A, at_Bm, at_gred, at_Ab, at_Bb, at_pq, at_polys, at_net, at_part, at_scratch;
    int OY, OZ, OG, ODG, OU, OW, OF, ODF;
    int PE;             // entries of a neighbour's powers: a table of their own at the beginning of the LDS, or E
    int lds_basic_off;  // byte offset of the packed basic-moment table in LDS (general tables)
    int grad_parts;     // loss gradient: parts of a chunk's neighbours that are summed at the same time
    int nc_cap;         // rows of the LDS neighbour table: a row is processed in chunks of at most nc_cap
    int leaves_late;    // the streams are fwd_core and rev_leaf: moments that only the read-out reads are formed in the reverse sweep
    // site-energy / descriptor mode (linearMtp.h:514-611, 821-890)
    T* e_sites;        // [B, P] per-row energies, or null
    T* desc;           // [B, P, n_scalar] scalar moments, or null
    int energy_only;   // stop after the energy: no adjoint, no pair derivatives
    int cE_per_atom;   // loss-gradient mode: cE is indexed per row (weights of the site energies)
    int no_tangent;    // loss-gradient mode: the force and virial residuals are zero (site-energy and basis backward),
                       // so the tangents and mixed adjoints vanish: their sweeps and terms are left out
    // neural-network read-out (source/descriptor/nnmtp/include/nnMtp.h:470-507) when H > 0:
    // e_i = bias + sum_p w1[t,p] tanh(sum_k w0[t,p,k] (M_k - q_shift[k]) / q_scaler[k]); `lin` is unused
    int H;
    const T *w0, *w1, *q_shift;
    int nn_exact;      // loss mode: 1 = complete derivative, 0 = the reference's formulas (see nnmtp_loss)
    // backward of the legacy basis operator (mtpBasis.h:359-394): the adjoint sweep starts from the caller's
    // weights of each row's scalar moments instead of a read-out (`lin`, `bias`, `q_scaler` are unused)
    const T* row_seed; // [B, P, n_scalar], or null
    T* pair_out;       // [B, P, U, 3] derivative of the row's weighted moments along each pair vector, or null
};

// a / b for small integers, 0 <= a < 2^20, b > 0 (the exact quotient is at least 0.5 / b away from the next integer, the
// rounding here below 2^-22 of it)
__device__ __forceinline__ int small_div(int a, int b) { return (int)(((float)a + 0.5f) * __builtin_amdgcn_rcpf((float)b)); }

__device__ __forceinline__ float tanh_t(float x) { return tanhf(x); }
__device__ __forceinline__ double tanh_t(double x) { return tanh(x); }

__device__ __forceinline__ float sqrt_t(float x) { return sqrtf(x); }
__device__ __forceinline__ double sqrt_t(double x) { return sqrt(x); }

// Per-neighbour table for neighbours [c0, c0+nc) of the row.
// Layout per neighbour: in `pw` (stride a.PE) ux^0..kmax | uy^.. | uz^..; in `tab` (E entries of T, the places in MtpArgs) ux uy uz 1/r |
// g[nmus] | dg[nmus] | (loss mode) vx vy vz w.u | f[K] | df[K].  The two are one table where a.PE is E.
// PASS says what the passes that follow read: TAB_MOMENTS powers, g, dg; TAB_TANGENTS also w; TAB_ALL also f, df; TAB_GRADIENT powers, w,
// f, df.  Without `powers` the powers are left out.
// The threads form groups of nc, a neighbour to a thread.  Groups share the radial functions, two to a Chebyshev
// recurrence (coefficients from the LDS copy `cf` of the centre species' block); more than two where the workgroup has no
// room for their groups beside those of the powers, of w and of f.  What bounds it is the issue of fp64 instructions, so a
// group for every function, which would be no faster, is no gain.
// (One task per radial function and per axis, with every value in every pass, took 333 instead of 324 us for the whole
// kernel at level 20, 8192 atoms, 118 instead of 111 at level 16, 64 structures of 128 atoms, and 252 instead of 244 for
// the loss gradient there; early claims and row-swap sums at the end included.)
// Lanes j < nc also return the neighbour's index, validity and displacement.
enum TablePass { TAB_MOMENTS, TAB_TANGENTS, TAB_ALL, TAB_GRADIENT };

// An array on its way to LDS: the first U entries of every thread are asked for together, and stored when the caller says.
template <typename V, int NT, int U>
struct Staged {
    V v[U];
    __device__ __forceinline__ void load(const V* src, int n, int lane)
    {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (lane + u * NT < n) v[u] = src[lane + u * NT];
    }
    __device__ __forceinline__ void store(V* dst, const V* src, int n, int lane)
    {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (lane + u * NT < n) dst[lane + u * NT] = v[u];
        for (int i = lane + U * NT; i < n; i += NT) dst[i] = src[i];
    }
};

// `ahead`: what a thread's first task begins with, read while the workgroup set itself up (is_ahead).
template <typename T>
struct TableAhead {
    T x, y, z;
    int nj, tj;          // the neighbour as it is listed, and the species of it (of the centre, where it is none)
    __device__ __forceinline__ void entries(const T* rcs, const int* first, int lane, int c0, int nc)
    {
        const int jj = c0 + lane - small_div(lane, nc) * nc;
        x = rcs[jj * 3 + 0]; y = rcs[jj * 3 + 1]; z = rcs[jj * 3 + 2];
        nj = first[jj];
    }
    __device__ __forceinline__ void species(const int* types, int NF, int center)
    {
        tj = types[(unsigned)nj < (unsigned)NF ? nj : center];
    }
};
template <typename T, TablePass PASS, int NT, typename Args>
__device__ __forceinline__ void build_table(Args& a, T* tab, T* pw, const T* cf, int lane, int nc, int c0,
                                            const T* rcs, const int* first, const int* types, int center,
                                            int b, int NF, int* nj_out, bool* valid_out, T* d_out, bool fill = true, bool powers = true,
                                            const TableAhead<T>& ahead = TableAhead<T>(), bool is_ahead = false)
{
    const int kmax = a.p.kmax, nmus = a.p.nmus, K = a.K;
    const int OG = a.OG, ODG = a.ODG, OU = a.OU, OW = a.OW, OF = a.OF, ODF = a.ODF;
    *valid_out = false;
    *nj_out = center;
    if (lane < nc) {
        const int jj = c0 + lane;
        T x, y, z;
        int nj;
        if (is_ahead) { x = ahead.x; y = ahead.y; z = ahead.z; nj = ahead.nj; }
        else { x = rcs[jj * 3 + 0]; y = rcs[jj * 3 + 1]; z = rcs[jj * 3 + 2]; nj = first[jj]; }
        d_out[0] = x; d_out[1] = y; d_out[2] = z;
        if ((unsigned)nj >= (unsigned)NF) { atomicOr(a.status, ST_BAD_NEIGHBOR); nj = center; }
        if ((unsigned)(is_ahead ? ahead.tj : types[nj]) >= (unsigned)a.ntypes) atomicOr(a.status, ST_BAD_TYPE);
        *nj_out = nj;
        *valid_out = !(sqrt_t(x * x + y * y + z * z) > a.rmax);      // mtpBasis.h:457, linearMtp.h:316
    }
    if (!fill) return;                      // the table is in place, only the lanes' own neighbours are returned
    // groups [0, nrad) radial functions, then powers, then w, then f
    constexpr bool WITH_W = PASS != TAB_MOMENTS, WITH_F = PASS == TAB_ALL || PASS == TAB_GRADIENT;
    constexpr int OTHERS = 1 + (WITH_W ? 1 : 0) + (WITH_F ? 1 : 0);
    int share = 0, nrad = 0;
    if (PASS != TAB_GRADIENT) {
        nrad = max(1, min((nmus + 1) / 2, __builtin_amdgcn_readfirstlane(small_div(NT, nc)) - OTHERS));
        share = (__builtin_amdgcn_readfirstlane(small_div(nmus + nrad - 1, nrad)) + 1) & ~1;
        nrad = __builtin_amdgcn_readfirstlane(small_div(nmus + share - 1, share));
    }
    const int ntask = nc * (nrad + OTHERS);
    for (int task = lane; task < ntask; task += NT) {
        const int role = small_div(task, nc), j = task - role * nc;
        const int jj = c0 + j;
        const bool known = is_ahead && task < NT;                         // (uniform: the first round)
        T x, y, z;
        if (known) { x = ahead.x; y = ahead.y; z = ahead.z; }
        else { x = rcs[jj * 3 + 0]; y = rcs[jj * 3 + 1]; z = rcs[jj * 3 + 2]; }
        const T r = sqrt_t(x * x + y * y + z * z);
        T* t = tab + j * a.E;
        if (role == nrad) {                                            // powers of the unit vector
            const T rinv = (T)1 / r;
            const T ux = x * rinv, uy = y * rinv, uz = z * rinv;
            T px = (T)1, py = (T)1, pz = (T)1;
            if (powers) {
                T* const q = pw + j * a.PE;
                for (int k = 0; k <= kmax; k++) {
                    q[k] = px; q[kmax + 1 + k] = py; q[2 * (kmax + 1) + k] = pz;
                    px *= ux; py *= uy; pz *= uz;
                }
            }
            t[OU + 0] = ux; t[OU + 1] = uy; t[OU + 2] = uz; t[OU + 3] = rinv;
            continue;
        }
        int nj = known ? ahead.nj : first[jj];
        if ((unsigned)nj >= (unsigned)NF) nj = center;
        if (WITH_W && role == nrad + 1) {
            // w_a = dFs[centre]_a - dFs[neighbour]_a - sum_b dVs[a,b] r_b   (linearMtpLoss.h:371-386), kept as w . u and
            // v = (w - (w . u) u) / r: the monomials are homogeneous, k m = u . grad m, so D_w m = (w . u) m' + v . grad m
            const T* fc = a.dFs + ((size_t)b * a.P + center) * 3;
            const T* fn = a.dFs + ((size_t)b * a.P + nj) * 3;
            const T* dv = a.dVs + (size_t)b * 9;
            T w[3];
#pragma unroll
            for (int q = 0; q < 3; q++)
                w[q] = fc[q] - fn[q] - (dv[q * 3 + 0] * x + dv[q * 3 + 1] * y + dv[q * 3 + 2] * z);
            const T rinv = (T)1 / r, wu = (w[0] * x + w[1] * y + w[2] * z) * rinv;
            t[OW + 0] = (w[0] - wu * (x * rinv)) * rinv;
            t[OW + 1] = (w[1] - wu * (y * rinv)) * rinv;
            t[OW + 2] = (w[2] - wu * (z * rinv)) * rinv;
            t[OW + 3] = wu;
            continue;
        }
        // radial functions, basis.h:154-196, 351-381, 620-637
        // quotients by the span: a product and one correction step, which restores the last bit
        const T span = a.rmax - a.rmin;
        auto over_span = [&](T v) { const T q = v * a.inv_span; return fma(fma(-q, span, v), a.inv_span, q); };
        const T xx = over_span((T)2 * r - (a.rmax + a.rmin)), x2 = (T)2 * xx;
        const T u = over_span(r - a.rmin);
        T s = (T)0, ds = (T)0;
        if (!(r > a.rmax) && r >= a.rmin && r < a.rmax) {
            s = a.scaling * (u * u * u * ((T)-6 * u * u + (T)15 * u - (T)10) + (T)1);
            ds = a.scaling * a.inv_span * ((T)-30 * u * u * u * u + (T)60 * u * u * u - (T)30 * u * u);
        }
        const T sx = s * (T)2 * a.inv_span;
        if (WITH_F && role == nrad + 2) {
            T t0 = (T)1, t1 = xx, d0 = (T)0, d1 = (T)1;
            for (int k = 0; k < K; k++) {
                t[OF + k] = s * t0;
                t[ODF + k] = ds * t0 + sx * d0;
                const T tv = x2 * t1 - t0, dv = (T)2 * t1 + x2 * d1 - d0;
                t0 = t1; t1 = tv; d0 = d1; d1 = dv;
            }
            continue;
        }
        if (PASS == TAB_GRADIENT) continue;
        int tj = known ? ahead.tj : types[nj];
        if ((unsigned)tj >= (unsigned)a.ntypes) tj = 0;
        const int m1 = min(nmus, (role + 1) * share);
        for (int mu = role * share; mu < m1; mu += 2) {
            const int two = mu + 1 < m1;
            const T* ca = cf + (tj * nmus + mu) * K;
            const T* cb = ca + two * K;
            T t0 = (T)1, t1 = xx, d0 = (T)0, d1 = (T)1;
            T ga = (T)0, gb = (T)0, ha = (T)0, hb = (T)0;
#pragma unroll 4
            for (int k = 0; k < K; k++) {
                const T c0k = ca[k], c1k = cb[k];
                ga += c0k * t0; ha += c0k * d0;
                gb += c1k * t0; hb += c1k * d0;
                const T tv = x2 * t1 - t0, dv = (T)2 * t1 + x2 * d1 - d0;
                t0 = t1; t1 = tv; d0 = d1; d1 = dv;
            }
            t[OG + mu] = s * ga; t[ODG + mu] = ds * ga + sx * ha;
            if (two) { t[OG + mu + 1] = s * gb; t[ODG + mu + 1] = ds * gb + sx * hb; }
        }
    }
}

// Basic moments M_(mu,a,b,c) = sum_j (x^a y^b)_j (g_mu z^c)_j of a chunk's neighbours as products of matrices, tile by tile of rows (a, b)
// and columns (mu, c) (mtp_plan.h), and, with tangents, D_w M = sum_j (x^a y^b) ((w . u) g' z^c + g v_z c z^(c-1)) + (v_x a x^(a-1) y^b +
// v_y b x^a y^(b-1)) (g z^c).  Four neighbours to an instruction; the sums stay in its accumulators over all chunks of the row.  A
// wavefront takes up to tiles_of tiles; with fewer tiles than wavefronts these share the neighbours.
// What bounds it: the matrix instructions, 64 cycles each in fp64 during which the SIMD issues nothing else (as many FMAs as the vector
// instructions make in that time), with a third of the places of the tiles in use; but the operands of a tile cost 6 LDS reads and some 14
// vector instructions per four neighbours, where a thread per polynomial in z read four values per neighbour and moment row.
constexpr int tiles_of(bool loss, int nt) { return loss && nt == 64 ? 1 : 2; }
struct TileShare {
    int first, split, nsplit;            // the wavefront's first tile; its share of the neighbours and how many there are
    template <int NT>
    static __device__ __forceinline__ TileShare of(int ntiles, int wave)
    {
        constexpr int W = NT / 64;
        if (ntiles >= W) return {wave, 0, 1};
        const int s = wave >= 2 * ntiles ? (wave >= 3 * ntiles ? 3 : 2) : (wave >= ntiles ? 1 : 0);       // (at most three tiles)
        return {wave - s * ntiles, s, ntiles == 1 ? W : W / 2 >= ntiles ? 2 : 1};
    }
};
// The exponents of the lane's row and column of a tile.
template <typename T>
__device__ __forceinline__ unsigned tile_word(const unsigned* ops, int tile, int lane)
{
    // (in single precision the lane's places are rows 4 (l / 16) + v of the product: its rows in the order that makes them those of the plan)
    const unsigned own = ops[tile * 64 + lane];
    if (sizeof(T) == 8) return own;
    return (ops[tile * 64 + (lane & 3) * 4 + (lane >> 2 & 3)] & 0x3ffu) | (own & ~0x3ffu);
}
template <typename T, bool TANGENT, int NT, int TILES, typename Args>
__device__ __forceinline__ void tile_products(Args& a, const T* tab, const T* pw, int tid, int nc, const TileShare& ts, const unsigned (&word)[TILES],
                                              typename wave::Acc<T>::type (&m)[TILES], typename wave::Acc<T>::type (&d)[TILES])
{
    const int kq = (tid & 63) >> 4, E = a.E, PE = a.PE, n1 = a.p.kmax + 1, ntiles = a.p.ntiles;
    if (ts.split >= ts.nsplit) return;
    const int steps = (nc + 3) >> 2;
    const int k0 = ts.nsplit == 1 ? 0 : ts.split * steps / ts.nsplit, k1 = ts.nsplit == 1 ? steps : (ts.split + 1) * steps / ts.nsplit;
#pragma unroll
    for (int u = 0; u < TILES; u++) {
        if (ts.first + u * (NT / 64) >= ntiles || (u > 0 && ts.nsplit > 1)) break;
        const int ea = word[u] & 31, eb = word[u] >> 5 & 31, mu = word[u] >> 10 & 7, ec = word[u] >> 13;
        const T *const px = pw + ea, *const py = pw + n1 + eb, *const pz = pw + 2 * n1 + ec, *const pg = tab + a.OG + mu;
        for (int k = k0; k < k1; k++) {
            const int j = k * 4 + kq;
            const bool on = j < nc;
            const unsigned jj = on ? j : nc - 1, ap = __umul24(jj, PE), at = __umul24(jj, E);
            const T xa = px[ap], yb = py[ap], zc = pz[ap], g = pg[at];
            const T row = xa * yb, col = on ? g * zc : (T)0;
            m[u] = wave::mma(row, col, m[u]);
            if (TANGENT) {
                const T xm = px[(int)ap - (ea > 0)], ym = py[(int)ap - (eb > 0)], zm = pz[(int)ap - (ec > 0)], dg = pg[at + a.ODG - a.OG];
                const T *const w = tab + at + a.OW;
                const T rowd = ((T)ea * w[0]) * (xm * yb) + ((T)eb * w[1]) * (xa * ym);
                const T cold = on ? (w[3] * dg) * zc + ((T)ec * w[2]) * (g * zm) : (T)0;
                d[u] = wave::mma(row, cold, d[u]);
                d[u] = wave::mma(rowd, col, d[u]);
            }
        }
    }
}
// A wavefront's sums to their moments.
template <typename T, int NT, int TILES, typename Plan>
__device__ __forceinline__ void tile_store(Plan& p, T* dst, const TileShare& ts, const uint2 (&place)[TILES], const typename wave::Acc<T>::type (&m)[TILES])
{
    if (ts.split >= ts.nsplit) return;
#pragma unroll
    for (int u = 0; u < TILES; u++) {
        const int tile = ts.first + u * (NT / 64);
        if (tile >= p.ntiles || (u > 0 && ts.nsplit > 1)) break;
        const uint2 at = place[u];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const unsigned i = (v < 2 ? at.x : at.y) >> (v & 1 ? 16 : 0) & 0xffffu;
            if (i != MTP_NO_MOMENT) dst[i] = m[u][v];
        }
    }
}

// A unit (mtp_plan.h): the polynomial of degree M in x and t whose coefficients stand at `c`, with its derivatives, and, with BOTH, the
// value of the one at `cb`.  G lanes to a neighbour: with one, t = y; with two, t = xy and the powers of t take two degrees each.
// Nested Horner's rule without a branch: two FMAs per coefficient (three), three per power of t (four).
template <typename T>
struct UnitSums { T v, x, t, b; };
template <int G>
constexpr int unit_size(int M)
{
    int n = 0;
    for (int b = 0; b <= (G == 2 ? M / 2 : M); b++) n += M - G * b + 1;
    return n;
}
// The coefficients come by lots, one ahead of the one in use (all at once they take a hundred registers).
template <typename T, int G, int M, bool BOTH>
__device__ __forceinline__ UnitSums<T> unit_poly(const T* c, const T* cb, T x, T t)
{
    constexpr int TOP = G == 2 ? M / 2 : M, N = unit_size<G>(M), AHEAD = BOTH ? 2 : 4;
    UnitSums<T> s = {(T)0, (T)0, (T)0, (T)0};
    T lot[2][AHEAD], lotb[2][BOTH ? AHEAD : 1];
    auto fetch = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            if (i0 + u >= N) continue;
            lot[i0 / AHEAD & 1][u] = c[i0 + u];
            if (BOTH) lotb[i0 / AHEAD & 1][u] = cb[i0 + u];
        }
    };
    fetch(0);
    T v = (T)0, d = (T)0, vb = (T)0;
    int b = TOP, k = 0;                                 // row, place in it
#pragma unroll
    for (int i = 0; i < N; i++) {
        if (i % AHEAD == 0) {
            // (nothing of the lots before is left for later, and no later lot is asked for yet)
            if (i > 0) asm volatile("" : "+v"(v), "+v"(d), "+v"(s.v), "+v"(s.x), "+v"(s.t) : : "memory");
            if (BOTH && i > 0) asm volatile("" : "+v"(vb), "+v"(s.b) : : "memory");
            fetch(i + AHEAD);
        }
        const T ci = lot[i / AHEAD & 1][i % AHEAD];
        const T cbi = BOTH ? lotb[i / AHEAD & 1][BOTH ? i % AHEAD : 0] : (T)0;
        if (k == 0) {
            v = ci; d = (T)0; vb = cbi;
        } else {
            d = k == 1 ? v : d * x + v;
            v = v * x + ci;
            if (BOTH) vb = vb * x + cbi;
        }
        if (++k == M - G * b + 1) {
            if (b == TOP) {
                s.v = v; s.x = d; s.b = vb;
            } else {
                s.t = b == TOP - 1 ? s.v : s.t * t + s.v;
                s.v = s.v * t + v;
                s.x = s.x * t + d;
                if (BOTH) s.b = s.b * t + vb;
            }
            b--;
            k = 0;
        }
    }
    return s;
}
template <typename T, int G, bool BOTH>
__device__ __forceinline__ UnitSums<T> unit_sums(int M, const T*& c, const T*& cb, T x, T t)
{
    UnitSums<T> s;
#define MTP_UNIT(N) case N: s = unit_poly<T, G, N, BOTH>(c, cb, x, t); c += unit_size<G>(N); if (BOTH) cb += unit_size<G>(N); break;
    switch (M) {
        MTP_UNIT(1) MTP_UNIT(2) MTP_UNIT(3) MTP_UNIT(4) MTP_UNIT(5) MTP_UNIT(6) MTP_UNIT(7) MTP_UNIT(8) MTP_UNIT(9)
        default: s = unit_poly<T, G, 0, BOTH>(c, cb, x, t); c++; if (BOTH) cb++;
    }
#undef MTP_UNIT
    static_assert(MTP_NEST_MAX == 9, "a case for every degree");
    return s;
}

// The wavefront's units at the lane's neighbour, whose table row is t: with A = sum adj m over the basic moments m of a mu, taken as a
// polynomial in (x, y, z), `done` receives mu, the share's number, A, its gradient, and, with BOTH, the value B of the second coefficients.
// With two lanes to a neighbour (G), the upper 32 lanes of the wavefront have x and y exchanged, and each lane the sums of its half.
// All lanes of a wavefront take the same way, so that what describes a unit costs scalar instructions only, and read the same one or two
// coefficients.  What bounds it is the issue of the FMAs: a lane per (neighbour, share of the polynomials in z of all rows (a, b)) before
// took six LDS reads and some thirty instructions per polynomial beside its FMAs, of which polynomials of different lengths left some idle.
template <typename T, int G, bool BOTH, typename Done>
__device__ __forceinline__ void nested(const T* coef, const T* coefb, int prog, int n, T x, T y, T z, Done&& done)
{
    const T t = G == 2 ? x * y : y;
    T r = (T)0, rx = (T)0, rt = (T)0, rz = (T)0, rb = (T)0;
#pragma unroll 1
    for (int i = 0; i < n; i++) {
        const int w = __builtin_amdgcn_readlane(prog, i);
        const UnitSums<T> s = unit_sums<T, G, BOTH>(w & 15, coef, coefb, x, t);
        rz = rz * z + r;
        r = r * z + s.v;
        rx = rx * z + s.x;
        rt = rt * z + s.t;
        if (BOTH) rb = rb * z + s.b;
        if (w & 128) {
            for (int k = w >> 8 & 31; k > 0; k--) {            // (the next powers of z are another wavefront's)
                rz = rz * z + r;
                r *= z; rx *= z; rt *= z;
                if (BOTH) rb *= z;
            }
            done(w >> 4 & 7, w >> 13, r, rx, rt, rz, rb);
            r = rx = rt = rz = rb = (T)0;
        }
    }
}
// The moments behind a thread's first coefficients of the units, on their way during the reverse sweep (with the places of the tiles'
// sums during these: level 20, 8192 atoms 176 -> 174 us, level 12, 64 x 128 atoms 43.2 -> 40.9), and the coefficients out of the
// adjoints of the basic moments: set(place, moment) for each.
template <int NT>
struct UnitSources {
    static constexpr int U = NT == 64 ? 4 : 2;
    int m[U];
    template <typename Plan>
    __device__ __forceinline__ void load(Plan& p, int G, int tid)
    {
        const int n = p.nstream[G - 1];
#pragma unroll
        for (int u = 0; u < U; u++) m[u] = p.stream_src[G - 1][min(tid + u * NT, n - 1)];
    }
    template <typename Plan, typename Set>
    __device__ __forceinline__ void each(Plan& p, int G, int tid, Set&& set) const
    {
        const int n = p.nstream[G - 1];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (tid + u * NT < n) set(tid + u * NT, m[u]);
        for (int i = tid + U * NT; i < n; i += NT) set(i, (int)p.stream_src[G - 1][i]);
    }
};

template <typename T>
__device__ __forceinline__ T group_sum(const T* src, int ng, int ncoef)
{
    T v = src[0];
    for (int k = 1; k < ng; k++) v += src[k * ncoef];
    return v;
}

// Sum over the pieces of a list (mtp_plan.h: MtpStream): `rem` is the number of pieces behind the lane's own in its list;
// after `steps` doubling steps the lane of a list's first piece holds the list's sum (pieces in a fixed tree order).  Within
// a row of sixteen lanes by data-parallel moves, which bring a zero from beyond the row.  All 64 lanes take part.
template <typename T>
__device__ __forceinline__ T piece_sum(T v, int rem, int steps)
{
    T o = wave::dpp_move<0x101>(v);                   // row_shl:1
    v += rem >= 1 ? o : (T)0;
    if (steps > 1) { o = wave::dpp_move<0x102>(v); v += rem >= 2 ? o : (T)0; }
    if (steps > 2) { o = wave::dpp_move<0x104>(v); v += rem >= 4 ? o : (T)0; }
    if (steps > 3) { o = wave::dpp_move<0x108>(v); v += rem >= 8 ? o : (T)0; }
    for (int d = 16; d < 1 << steps; d <<= 1) {
        o = __shfl_down(v, d, 64);
        v += rem >= d ? o : (T)0;
    }
    return v;
}

// The same for several values, a step for all of them at a time, so that their moves overlap.
template <typename T, int N>
__device__ __forceinline__ void piece_sums(T (&v)[N], int rem, int steps)
{
    T o[N];
    auto add = [&](bool on) __attribute__((always_inline)) {        // (selected values: twelve instructions more for six)
        if (on) {
#pragma unroll
            for (int q = 0; q < N; q++) v[q] += o[q];
        }
    };
#pragma unroll
    for (int q = 0; q < N; q++) o[q] = wave::dpp_move<0x101>(v[q]);
    add(rem >= 1);
    if (steps <= 1) return;
#pragma unroll
    for (int q = 0; q < N; q++) o[q] = wave::dpp_move<0x102>(v[q]);
    add(rem >= 2);
    if (steps <= 2) return;
#pragma unroll
    for (int q = 0; q < N; q++) o[q] = wave::dpp_move<0x104>(v[q]);
    add(rem >= 4);
    if (steps <= 3) return;
#pragma unroll
    for (int q = 0; q < N; q++) o[q] = wave::dpp_move<0x108>(v[q]);
    add(rem >= 8);
    for (int d = 16; d < 1 << steps; d <<= 1) {
#pragma unroll
        for (int q = 0; q < N; q++) o[q] = __shfl_down(v[q], d, 64);
        add(rem >= d);
    }
}

// Sums of items by neighbouring lanes: log2 of how many lanes an item gets of `nt` threads (at most sixteen), and the sum over
// an item's lanes, in all of them.
__device__ __forceinline__ int parts_log2(int nt, int items)
{
    int l = 0;
    while (l < 4 && (items << (l + 1)) <= nt) l++;
    return l;
}
template <typename T>
__device__ __forceinline__ T parts_sum(T v, int log2_parts)
{
    if (log2_parts > 0) v += wave::dpp_move<0xB1>(v);      // quad_perm [1,0,3,2]
    if (log2_parts > 1) v += wave::dpp_move<0x4E>(v);      // quad_perm [2,3,0,1]
    if (log2_parts > 2) v += wave::dpp_move<0x141>(v);     // row_half_mirror
    if (log2_parts > 3) v += wave::dpp_move<0x140>(v);     // row_mirror
    return v;
}

// A plan term names its two moments by byte offsets into an array of doubles (index * 8): no shift between the
// word and the LDS address in fp64.
template <typename T>
__device__ __forceinline__ T plan_entry(const T* base, unsigned off)
{
    return *(const T*)((const char*)base + (sizeof(T) == 8 ? off : off >> 1));
}

// A gather (mtp_plan.h: MtpStream): terms(words, leaf, next) for a step, with next() where it has read its words, and done(moment,
// rem, steps, leaf) behind the last of a group; a barrier behind every level.  What bounds it is the instructions a wavefront issues
// one after the other and, with few wavefronts, the way of a step through one, so the plan holds everything in the order of use, and
// the words of the next two steps are on their way, also across a barrier (the plan does not depend on the moments).
// That takes some care, or the compiler waits for what it has only just asked for: every load of the loop is made in every step
// (with one that only some make, the next group's moments or control words, it does not know how many lie behind the words it waits
// for), the loop has one way out, what is loaded into is free by then (or it goes elsewhere, and copies wait for it), and none of a
// load's registers is lent to something else meanwhile.  So a step brings its moments along in the multiplicities, the
// control words of 64 steps lie in a vector register, and an odd step is walked ahead of the loop.
// Kernel of energies and forces, level 20, 8192 atoms, 236 -> 222 us (216 atoms: 28.3 -> 26.9), of level 16, 64 structures of 128 atoms,
// 90.3 -> 87.7, the loss gradient there 161 -> 159.5; with two products to a multiplicity (step_terms), 14 instead of 24 vector
// instructions for the four of a step; with the words' address formed without vector instructions and the second multiplicity as it was
// loaded, level 20, 8192 atoms 174 -> 169.5, the components of level 16 134 -> 131.  (The words of a step in an order that keeps the LDS free of bank conflicts, 1.2 lanes to a
// bank instead of 2.1: no change.)
template <typename Stream, typename Terms, typename Done>
__device__ __forceinline__ void walk(Stream& g, int tid, Terms&& terms, Done&& done)
{
    typedef int int4_t __attribute__((ext_vector_type(4)));
    struct Step { int4_t w[2]; };
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const A2P_CONSTANT int* const head = uniform_array((const int*)g.head) + wave * 4;
    const int first = head[0], n = head[1];
    const A2P_CONSTANT char* at = (const A2P_CONSTANT char*)(const A2P_CONSTANT int4*)uniform_array(g.words + (size_t)first * MTP_STEP_WORDS);
    unsigned at_lane = (unsigned)lane * 16u;
    auto load = [&](Step& s, int k) __attribute__((always_inline)) {       // (two steps behind the last)
        s.w[0] = *(const A2P_CONSTANT int4_t*)(at + k * MTP_STEP_WORDS * 16 + at_lane);
        s.w[1] = *(const A2P_CONSTANT int4_t*)(at + k * MTP_STEP_WORDS * 16 + 64 * 16 + at_lane);
    };
    // An odd step is walked ahead of the loop, which takes two at a time and has one way out (on another one the compiler sees
    // the loads of one step alone behind the words it waits for).
    const int odd = n & 1;
    Step a, b, single;
    int ctrl = 0;
    if (n > 0) {                                       // in the order in which they are waited for
        ctrl = g.ctrl[first + lane];                   // (64 words behind the last)
        __builtin_amdgcn_sched_barrier(0);
        if (odd) {
            load(single, 0);
            at += MTP_STEP_WORDS * 16;
        }
        __builtin_amdgcn_sched_barrier(0);
        load(a, 0);
        __builtin_amdgcn_sched_barrier(0);
        load(b, 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (int k = head[3]; k > 0; k--) __syncthreads();
    auto step = [&](Step& s, int i, bool ahead) __attribute__((always_inline)) {
        const int c = __builtin_amdgcn_readlane(ctrl, i);
        int slot;
        const bool leaf = (c & MTP_CTRL_LEAF) != 0;
        terms(s.w, leaf, [&]() __attribute__((always_inline)) {
            slot = s.w[0].z - 1;
            // (w[1].z, of no use, keeps its register: given to another value, this one would wait for the load)
            asm volatile("" : "+v"(slot) : "v"(s.w[1].z) : "memory");
            if (!ahead) return;
            // (a lane's address takes no vector instruction where it is formed anew each step, of the wavefront's and 32 bits of
            // the lane's, with an offset of less than 4096 bytes)
            at += MTP_STEP_WORDS * 16;
            asm volatile("" : "+s"(at), "+v"(at_lane));
            load(s, 1);
        });
        if (__builtin_expect(c & 1, 0)) {
            done((int)(short)slot, slot >> 16, (c >> 1) & 7, leaf);
            for (int k = c >> 4 & 0xffff; k > 0; k--) __syncthreads();
        }
    };
    if (n == 0) return;
    if (odd) step(single, 0, false);
    for (int i = odd, base = 0; i < n; base = i) {
        if (base > 0) ctrl = g.ctrl[first + base + lane];
        asm volatile("" : "+v"(ctrl));                 // (waited for here, not in the loop)
        const int end = min(n, base + 64 - (i - base));
#pragma unroll 1
        for (; i < end; i += 2) {
            step(a, i - base, true);
            step(b, i - base + 1, true);
        }
    }
}

// The terms of a step, two pairs of products (mtp_plan.h): acc += mult (a[x0] b[y0] + a[x1] b[y1]), and, with BOTH,
// tac += mult (ta[x0] b[y0] + a[x0] tb[y0] + ta[x1] b[y1] + a[x1] tb[y1]).  next() stands where the words have been read: the
// multiplicities are taken out of them before, for words that are held beyond the load of the next ones send these to other
// registers, and the copies at the end of a step wait for them.
template <typename T, bool BOTH, typename Words, typename Next>
__device__ __forceinline__ void step_terms(const Words (&w)[2], const T* a, const T* b, const T* ta, const T* tb, T& acc, T& tac, Next&& next)
{
    constexpr int C = MTP_DEPTH_STEP;
    T v0[C], v1[C], t0[C], t1[C], mult[C / 2];
#pragma unroll
    for (int u = 0; u < C; u++) {
        const unsigned x = u & 1 ? w[u / 2].y : w[u / 2].x, i0 = x & 0xffffu, i1 = x >> 16;
        v0[u] = plan_entry(a, i0); v1[u] = plan_entry(b, i1);
        if (BOTH) { t0[u] = plan_entry(ta, i0); t1[u] = plan_entry(tb, i1); }
    }
#pragma unroll
    for (int u = 0; u < C / 2; u++) {
        mult[u] = (T)__hiloint2double(w[u].w, u == 0 ? 0 : w[u].z);
        asm volatile("" : "+v"(mult[u]));
    }
    next();
#pragma unroll
    for (int u = 0; u < C; u += 2) {
        acc += mult[u / 2] * (v0[u] * v1[u] + v0[u + 1] * v1[u + 1]);
        if (BOTH) tac += mult[u / 2] * ((t0[u] * v1[u] + v0[u] * t1[u]) + (t0[u + 1] * v1[u + 1] + v0[u + 1] * t1[u + 1]));
    }
}

// forward products: M[dst] = sum mult M[m0] M[m1]; with TANGENT also the product rule on Tg.
template <typename T, bool TANGENT, typename Stream>
__device__ __forceinline__ void sweep_forward(Stream& g, T* M, T* Tg, int tid)
{
    T acc = (T)0, tacc = (T)0;
    walk(g, tid,
        [&](const auto& w, bool, auto next) __attribute__((always_inline)) {
            step_terms<T, TANGENT>(w, M, M, Tg, Tg, acc, tacc, next);
        },
        [&](int dst, int rem, int steps, bool) __attribute__((always_inline)) {
            if (steps) {
                acc = piece_sum(acc, rem, steps);
                if (TANGENT) tacc = piece_sum(tacc, rem, steps);
            }
            if (dst >= 0) {                                  // the first piece of a list
                M[dst] = acc;
                if (TANGENT) Tg[dst] = tacc;
            }
            acc = tacc = (T)0;
        });
}

// reverse gather: A[m] += sum mult A[dst] M[other], and, when MIXED, X[m] += sum mult (X[dst] M[other] + A[dst] Tg[other]) in
// the same walk: its words and the reads of M and A serve both (a walk for each: 285 instead of 273 us for the training step of
// level 16, 64 structures of 128 atoms).
// LEAF: the stream also holds the products that nothing but the read-out reads (mtp_plan.h: rev_leaf): sums mult M[m0] M[m1],
// and, when MIXED, their tangents sum mult (Tg[m0] M[m1] + M[m0] Tg[m1]); a leaf's sums go to leaf().
template <typename T, bool MIXED, bool LEAF, typename Stream, typename Leaf>
__device__ __forceinline__ void sweep_reverse(Stream& g, const T* M, T* A, T* X, const T* Tg, int tid, Leaf&& at_leaf)
{
    T acc = (T)0, xacc = (T)0;
    walk(g, tid,
        [&](const auto& w, bool leaf, auto next) __attribute__((always_inline)) {
            step_terms<T, MIXED>(w, LEAF && leaf ? M : A, M, LEAF && leaf ? Tg : X, Tg, acc, xacc, next);
        },
        [&](int src, int rem, int steps, bool leaf) __attribute__((always_inline)) {
            if (steps) {
                acc = piece_sum(acc, rem, steps);
                if (MIXED) xacc = piece_sum(xacc, rem, steps);
            }
            if (src >= 0) {
                if (LEAF && leaf) at_leaf(src, acc, xacc);
                else {
                    A[src] += acc;
                    if (MIXED) X[src] += xacc;
                }
            }
            acc = xacc = (T)0;
        });
}
template <typename T, typename Stream>
__device__ __forceinline__ void sweep_reverse(Stream& g, const T* M, T* X, int tid)
{
    sweep_reverse<T, false, false>(g, M, X, (T*)nullptr, (const T*)nullptr, tid, [](int, T, T) {});
}

// sum over the NT threads of a workgroup in a fixed order (wave sums, then wave 0 .. last)
template <typename T, int NT>
__device__ __forceinline__ T block_sum(T v, T* scratch, int tid)
{
    v = wave::all_sum(v);
    if (NT == 64) return v;
    __syncthreads();
    if ((tid & 63) == 0) scratch[tid >> 6] = v;
    __syncthreads();
    T t = (T)0;
#pragma unroll
    for (int w = 0; w < NT / 64; w++) t += scratch[w];
    return t;
}

// The adjoints of the basic moments as coefficients of the row polynomials (mtp_plan.h).  Ends without a barrier.
template <typename T, int NT, typename Plan>
__device__ __forceinline__ void scatter_polys(Plan& p, T* __restrict__ dst, const T* __restrict__ src, int tid)
{
    if (p.poly_unique && p.ncoef_poly == p.n_basic) {        // the usual case: a permutation
        for (int i = tid; i < p.n_basic; i += NT) dst[p.poly_pos[i]] = src[i];
        return;
    }
    for (int e = tid; e < p.ncoef_poly; e += NT) {
        const int one = p.poly_src[e];
        T v = (T)0;
        if (one >= 0) v = src[one];
        else if (one == -2)
            for (int q = p.poly_off[e]; q < p.poly_off[e + 1]; q++) v += src[p.poly_items[q]];
        dst[e] = v;
    }
}

// Pair derivatives of one neighbour by a walk over the monomial rows (mtp_plan.h): the lane owns the
// neighbour whose table row is `t`, takes every ng-th row and returns its share of
//   gs = sum_i adj_i m_i (g' - k g / r),   w = sum_i adj_i g grad_u m_i.
// A row (a, b) and a radial function mu make a polynomial in z, P(z) = sum_c adj z^c over the basic moments
// (mu, a, b, c), whose value and derivative come from one Horner walk: two FMAs per basic moment and neighbour.  With
// s1 = sum_mu g P, s2 = sum_mu g P', sd = sum_mu g' P (and z P' = sum_c c adj z^c) the row adds
//   gs += x^a y^b (sd - ((a + b) s1 + z s2) / r),  w_x += a x^(a-1) y^b s1,  w_y += b x^a y^(b-1) s1,  w_z += x^a y^b s2.
// What bounds it: the vector ALUs' issue and the LDS reads of the coefficients (uniform over a group's lanes).  A walk
// over all monomials with every mu (a dense array of adjoints, 2 nmus + 12 operations per monomial) took
// 356 instead of 334 us for the whole kernel at level 20, 8192 atoms, and 125 instead of 118 us at level 16.
template <typename T>
__device__ __forceinline__ void pair_walk(const T* __restrict__ t, const T* __restrict__ coef, const int* __restrict__ rows,
                                          const int* __restrict__ polys, int nrows, int h, int ng, int OX, int OY, int OZ,
                                          int OG, int ODG, T rinv, T& gs, T& wx, T& wy, T& wz)
{
    const T z = t[OZ + 1];
    // the rows are sorted by length: groups take them in alternating direction, which evens out their shares
    for (int pass = 0, r = h; r < nrows; pass++, r = pass * ng + (pass & 1 ? ng - 1 - h : h)) {
        const int rw = rows[r];
        const int ea = rw & 255, eb = (rw >> 8) & 255;
        const int s_end = rows[r + 1] >> 16;
        T s1 = (T)0, s2 = (T)0, sd = (T)0;
        for (int s = rw >> 16; s < s_end; s++) {
            const int pw = polys[s];
            const T g = t[OG + (pw & 15)], dg = t[ODG + (pw & 15)];
            const T* c = coef + (pw >> 12);                  // highest power first
            int len = (pw >> 4) & 255;
            T v = (T)0, d = (T)0;
            if (len & 1) v = *c++;
            for (len >>= 1; len > 0; len--, c += 2) {
                const T c0 = c[0], c1 = c[1];
                d = d * z + v;
                v = v * z + c0;
                d = d * z + v;
                v = v * z + c1;
            }
            s1 += g * v;
            s2 += g * d;
            sd += dg * v;
        }
        const T xa = t[OX + ea], yb = t[OY + eb];
        const T xy = xa * yb;
        gs += xy * (sd - ((T)(ea + eb) * s1 + z * s2) * rinv);
        wx += (T)ea * t[OX + max(ea - 1, 0)] * yb * s1;
        wy += (T)eb * xa * t[OY + max(eb - 1, 0)] * s1;
        wz += xy * s2;
    }
}

// The polynomials of a neighbour for the loss gradient: every ng-th one of a radial function's from the s-th on.  With
// A = sum adj m, B = sum (cE adj + mixed) m over the basic moments of mu and k m = u . grad m (m is homogeneous),
//   P_mu = B + (w - (w . u) u) . grad A / r,   Q_mu = (w . u) A.
// Three FMAs per basic moment and neighbour; forming each monomial with its gradient from the table of powers instead
// took about thirty operations and nine LDS reads (263 -> 252 us for the kernel, level 16, 64 structures of 128 atoms).
template <typename T>
__device__ __forceinline__ void loss_walk(const T* __restrict__ t, const T* __restrict__ Ac, const T* __restrict__ Bc,
                                          const int* __restrict__ polys, int& s, int end, int ng, int OX, int OY, int OZ,
                                          int OW, T cE, bool no_tan, T& P, T& Q)
{
    P = Q = (T)0;
    if (s >= end) return;
    const T z = t[OZ + 1];
    const T wu = no_tan ? (T)0 : t[OW + 3];
    const T vx = no_tan ? (T)0 : t[OW + 0], vy = no_tan ? (T)0 : t[OW + 1], vz = no_tan ? (T)0 : t[OW + 2];
    for (; s < end; s += ng) {
        const int pw = polys[s];
        const int ea = pw & 31, eb = (pw >> 5) & 31;
        int len = (pw >> 10) & 31;
        const T* ca = Ac + (pw >> 15);
        const T* cb = Bc + (pw >> 15);
        const T xa = t[OX + ea], yb = t[OY + eb], xm = t[OX + max(ea - 1, 0)], ym = t[OY + max(eb - 1, 0)];
        T va = (T)0, da = (T)0, vb = (T)0;
        if (len & 1) { va = *ca++; vb = *cb++; }
        for (len >>= 1; len > 0; len--, ca += 2, cb += 2) {
            const T a0 = ca[0], a1 = ca[1], b0 = cb[0], b1 = cb[1];
            da = da * z + va;
            va = va * z + a0;
            vb = vb * z + b0;
            da = da * z + va;
            va = va * z + a1;
            vb = vb * z + b1;
        }
        const T xy = xa * yb;
        P += xy * (cE * va + vb) + va * (vx * ((T)ea * xm * yb) + vy * ((T)eb * xa * ym)) + da * (vz * xy);
        Q += xy * va;
    }
    Q *= wu;
}

// Wavefronts per SIMD that the registers are kept to.  Energies and forces with 256 threads: five (four: level 20, 8192 atoms 174 -> 195
// us; six spill: 266), with 64: four (five: level 16, 64 structures of 128 atoms 67 -> 90).  Loss gradient in fp64: five, which takes 95
// registers without a spill (six, as long as its sums went by polynomials in z: 136 registers spilled, level 16 165 -> 133; four: 149), in
// fp32 six (without a limit some went to the accumulation registers and back: level 20, 32 x 128 atoms 123 -> 115).
constexpr int waves_of(bool fp64, bool loss, int nt) { return loss ? (fp64 ? 5 : 6) : nt == 256 ? 5 : 4; }

// The workgroup's LDS (launch_atoms): moments | (loss mode: their tangents) | adjoints | (mixed adjoints), in whose place the powers of the
// neighbours' unit vectors stand before | coefficients of the centre species | neighbour table | ...
// General tables: moments | tangents | coefficients | neighbour table, in whose place the adjoints come after it | ...
template <typename T, bool LOSS>
struct AtomLds {
    T *M, *Tg, *cf, *tab, *A, *Bm, *gred, *Ab, *Bb, *pq, *polys, *net, *part, *scratch;
    unsigned* bas;
    int* rws;
    template <typename Args>
    __device__ __forceinline__ AtomLds(Args& a, unsigned char* smem)
    {
        M = (T*)smem;
        Tg = M + a.at_Tg;
        cf = M + a.at_cf;                       // [ntypes][nmus][K]
        tab = M + a.at_tab;
        A = M + a.at_A;
        Bm = M + a.at_Bm;
        gred = M + a.at_gred;                   // partial sums of the thread groups
        // loss mode: adjoints and mixed adjoints of the basic moments (as coefficients of the polynomials) | P[nc][nmus] |
        // Q[nc][nmus] | ...
        Ab = M + a.at_Ab;
        Bb = M + a.at_Bb;
        pq = M + a.at_pq;
        polys = M + a.at_polys;                 // energy / force / virial: coefficients of the polynomials
        net = M + a.at_net;                     // network inputs and per-neuron values
        part = M + a.at_part;                   // sums of the basic moments by wavefronts that share a tile
        scratch = M + a.at_scratch;             // a value per wavefront; sums over the pairs of a row's chunks so far
        // general tables, behind everything else: (mu, a, b, c) of every basic moment, one byte each; monomial rows and polynomials of
        // the pair-derivative walk
        bas = (unsigned*)(smem + a.lds_basic_off);
        rws = (int*)(bas + a.p.n_basic);
    }
};

// What a phase of the atom kernel works with, under the names of the formulas.
// The kernels' arguments are some eighty scalars, and the plan names two dozen arrays: held in registers from the first
// use to the last they do not fit, and what did not (some 150 values) moved between lanes of vector registers all the time:
// 300 instead of 281 us for the energies and forces of level 20, 8192 atoms, 238 instead of 222 for the loss gradient of
// level 16, 64 structures of 128 atoms.  Each phase takes the arguments from the segment they were passed in anew (scalar loads).
#define MTP_PHASE                                                                                                          \
    [[maybe_unused]] auto& a = again(kernel_args<MtpArgs<T>>());                                                                \
    [[maybe_unused]] auto& p = a.p;                                                                                        \
    [[maybe_unused]] const bool seeded = (SEED || LOSS) && a.row_seed != nullptr;                                          \
    [[maybe_unused]] const bool no_tan = LOSS && a.no_tangent != 0;                 /* uniform over the launch */          \
    [[maybe_unused]] const AtomLds<T, LOSS> L(a, smem_raw);                                                            \
    [[maybe_unused]] T *const M = L.M, *const Tg = L.Tg, *const cf = L.cf, *const tab = L.tab, *const A = L.A, *const Bm = L.Bm; \
    [[maybe_unused]] T* const pw = TILED ? M : tab;                                                                        \
    [[maybe_unused]] const int NF = a.P + a.nghost, n_moms = p.n_moms, n_basic = p.n_basic, nmus = p.nmus, kmax = p.kmax,  \
                               K = a.K, E = a.E, MTP_NC = a.nc_cap;                                                        \
    [[maybe_unused]] const int OX = 0, OY = a.OY, OZ = a.OZ, OG = a.OG, ODG = a.ODG, OU = a.OU, OW = a.OW, OF = a.OF, ODF = a.ODF; \
    [[maybe_unused]] const size_t row = (size_t)b * a.P + ii;                                                              \
    [[maybe_unused]] const int* const first = a.bfirstneigh + row * a.U;                                                   \
    [[maybe_unused]] const T* const rcs = a.brcs + row * a.U * 3;                                                          \
    [[maybe_unused]] const int* const types = a.btypes + (size_t)b * NF

// NT threads per centre atom: 64 or 256 (wide_atoms).
// SEED: the instance of the energy / force / virial kernel that can start its adjoint sweep from per-row weights
// (row_seed, pair_out); the loss-gradient kernel tests the pointer at run time.  NET: the instances with a network read-out.
// TILES: the passes over the neighbours by matrix products, as many tiles to a wavefront, and nested polynomials (mtp_plan.h: ntiles),
// where the tables fit them; the others (0) go by basic moments and by polynomials in z, with 256 threads.  (Two tiles to a wavefront where
// one does, 32 registers of sums without use: the loss gradient of a network at level 10, 32 x 100 atoms 63 -> 62 us, fp32, level 16, 64 x
// 128 atoms 116 -> 104, fp32 energies and forces of level 8 29.5 -> 25.5.)
template <typename T, bool LOSS, int NT, bool SEED = false, bool NET = false, int TILES = 1>
__global__ void __launch_bounds__(NT, waves_of(sizeof(T) == 8, LOSS, NT)) mtp_atom_kernel(const MtpArgs<T>)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int lane = threadIdx.x;     // thread in the workgroup
    const int ii = blockIdx.x, b = blockIdx.y;
    int center, nn, ti;
    int nchunks, csize;               // the row is cut into equal chunks of at most nc_cap neighbours
    TableAhead<T> ahead;              // (energies and forces; the loss gradient's registers do not hold it: 166 -> 175 us)
    constexpr bool TILED = TILES > 0;
    constexpr int NTILE = TILED ? TILES : 1;
    unsigned tword[NTILE];        // the lane's rows and columns of the wavefront's tiles
    const int wave = __builtin_amdgcn_readfirstlane(lane >> 6), l64 = lane & 63;
    {
        MTP_PHASE;
        // (scalar loads, on their way while the plan's arrays are asked for; a padded row has places in the lists as well)
        const int inum = uniform_array(a.binum)[b];
        center = uniform_array(a.bilist)[row];
        nn = uniform_array(a.bnumneigh)[row];

        // Three trips to memory: the row's head with the plan's arrays, the row's entries with the species of the centre, the
        // coefficients with the neighbours' species.  (Five before, with the entries and their species behind the barrier: level 20, 8192
        // atoms 228.8 -> 226.4 us, the training step of level 16, 64 structures of 128 atoms, 272.8 -> 270.5, the linear solver there
        // 469 -> 462.)
        // (The number of rows was a trip of its own ahead of these: level 10, 216 atoms 29.5 -> 29.1 us, the solver 403 -> 401.)
        Staged<unsigned, NT, NT == 64 ? 4 : 2> basics;
        const int nwords = LOSS ? p.npoly : p.nrows + 1;
        const int* const wsrc = LOSS ? p.polys_mu : p.rows;
        Staged<int, NT, NT == 64 ? 2 : 1> words;
        if constexpr (TILED) {
            const TileShare ts = TileShare::of<NT>(p.ntiles, wave);
#pragma unroll
            for (int u = 0; u < NTILE; u++) tword[u] = tile_word<T>(p.tile_ops, min(ts.first + u * (NT / 64), p.ntiles - 1), l64);
        } else {
            basics.load(p.basic, n_basic, lane);
            words.load(wsrc, nwords, lane);
        }
        if (ii >= inum) {                  // padded row: contributes nothing
            if (!LOSS && a.partial && lane < 10) a.partial[ev_partial(a.P, b, ii, lane)] = 0.0;
            if (!LOSS && a.e_sites && lane == 0) a.e_sites[row] = (T)0;
            if (!LOSS && a.desc)
                for (int s = lane; s < p.n_scalar; s += NT) a.desc[row * p.n_scalar + s] = (T)0;
            return;                        // (its gradient row is not read)
        }
        if (nn > a.U) { if (lane == 0) atomicOr(a.status, ST_NEIGH_OVERFLOW); nn = a.U; }
        if ((unsigned)center >= (unsigned)NF) { if (lane == 0) atomicOr(a.status, ST_BAD_NEIGHBOR); center = 0; nn = 0; }
        ti = uniform_array(types)[center];
        {
            // (whole-number divisions: small_div cuts a row of two million and more into chunks longer than the table)
            const unsigned n = nn, cap = MTP_NC, cuts = (n + cap - 1) / cap;
            nchunks = (int)cuts;
            csize = cuts > 1 ? (int)((n + cuts - 1) / cuts) : max(nn, 1);
        }
        if (!LOSS && nn > 0) ahead.entries(rcs, first, lane, 0, min(csize, nn));
        if constexpr (!TILED) {
            for (int i = lane; i < n_moms; i += NT) {
                M[i] = (T)0;
                if (LOSS) Tg[i] = (T)0;
            }
            basics.store(L.bas, p.basic, n_basic, lane);
            words.store(L.rws, wsrc, nwords, lane);
            if (!LOSS)
                for (int i = lane; i < p.npoly; i += NT) L.rws[p.nrows + 1 + i] = p.polys[i];
            else
                for (int i = lane; i <= nmus; i += NT) L.rws[p.npoly + i] = p.polys_end[i];
        }
        if ((unsigned)ti >= (unsigned)a.ntypes) { if (lane == 0) atomicOr(a.status, ST_BAD_TYPE); ti = 0; nn = 0; }
        const T* const csrc = a.coeffs + (size_t)ti * a.ntypes * nmus * K;
        Staged<T, NT, NT == 64 ? 2 : 1> coefs;
        coefs.load(csrc, a.ntypes * nmus * K, lane);
        if (!LOSS && nn > 0) ahead.species(types, NF, center);
        coefs.store(cf, csrc, a.ntypes * nmus * K, lane);
        __syncthreads();
    }

    // ---- basic moments (and their tangents) --------------------------------------------------
    [[maybe_unused]] typename wave::Acc<T>::type msum[NTILE], dsum[NTILE];
    [[maybe_unused]] uint2 tplace[NTILE];
    auto table = [&](int c0, int nc) __attribute__((always_inline)) {
        MTP_PHASE;
        int nj; bool valid; T d[3];
        build_table<T, LOSS ? (TILED ? TAB_ALL : TAB_TANGENTS) : TAB_MOMENTS, NT>(a, tab, pw, cf, lane, nc, c0, rcs, first, types, center, b, NF, &nj, &valid,
                                                                              d, true, true, ahead, !LOSS);
        __syncthreads();
    };
    auto next_ahead = [&](int c0) __attribute__((always_inline)) {
        if (LOSS) return;              // (not held over the sums)
        MTP_PHASE;
        ahead.entries(rcs, first, lane, c0, min(csize, nn - c0));
        ahead.species(types, NF, center);
    };
    if constexpr (TILED) {
        {
            MTP_PHASE;
            const TileShare ts = TileShare::of<NT>(p.ntiles, wave);
#pragma unroll
            for (int u = 0; u < NTILE; u++) tplace[u] = p.tile_place[min(ts.first + u * (NT / 64), p.ntiles - 1) * 64 + l64];
        }
        auto products = [&](int nc) __attribute__((always_inline)) {
            MTP_PHASE;
            const TileShare ts = TileShare::of<NT>(p.ntiles, wave);
            if (LOSS && !no_tan) tile_products<T, LOSS, NT, NTILE>(a, tab, pw, lane, nc, ts, tword, msum, dsum);
            else tile_products<T, false, NT, NTILE>(a, tab, pw, lane, nc, ts, tword, msum, dsum);
            __syncthreads();
        };
        // (the first chunk, of most rows the only one, by itself: sums held over the table's phase do not fit the registers)
        if (nn > 0) table(0, min(csize, nn));
#pragma unroll
        for (int u = 0; u < NTILE; u++) msum[u] = dsum[u] = {0, 0, 0, 0};
        if (nn > 0) products(min(csize, nn));
#pragma unroll 1
        for (int c0 = csize; c0 < nn; c0 += csize) {
            next_ahead(c0);
            table(c0, min(csize, nn - c0));
            products(min(csize, nn - c0));
        }
    } else {
        for (int c0 = 0; c0 < nn; c0 += csize) {
            const int nc = min(csize, nn - c0);
            if (c0 > 0) next_ahead(c0);
            table(c0, nc);
            MTP_PHASE;
            for (int i = lane; i < n_basic; i += NT) {
                const unsigned bw = L.bas[i];
                const int mu = bw & 255, ea = (bw >> 8) & 255, eb = (bw >> 16) & 255, ec = bw >> 24;
                T acc = (T)0, tacc = (T)0;
                for (int j = 0; j < nc; j++) {
                    const T* t = tab + j * E;
                    const T g = t[OG + mu];
                    const T xa = t[OX + ea], yb = t[OY + eb], zc = t[OZ + ec];
                    const T m = xa * yb * zc;
                    acc += g * m;
                    if (LOSS && !no_tan) {
                        const T dg = t[ODG + mu], wu = t[OW + 3];
                        const T gm = (T)ea * t[OX + max(ea - 1, 0)] * yb * zc * t[OW + 0] +
                                     (T)eb * xa * t[OY + max(eb - 1, 0)] * zc * t[OW + 1] +
                                     (T)ec * xa * yb * t[OZ + max(ec - 1, 0)] * t[OW + 2];
                        tacc += wu * m * dg + g * gm;
                    }
                }
                M[i] += acc;
                if (LOSS) Tg[i] += tacc;
            }
            __syncthreads();
        }
    }
    if constexpr (TILED) {             // the powers are dead: the moments take their place
        MTP_PHASE;
        const TileShare ts = TileShare::of<NT>(p.ntiles, wave);
        const int per = LOSS ? 2 * n_basic : n_basic;
        tile_store<T, NT, NTILE>(p, ts.split == 0 ? M : L.part + (ts.split - 1) * per, ts, tplace, msum);
        if (LOSS) tile_store<T, NT, NTILE>(p, ts.split == 0 ? Tg : L.part + (ts.split - 1) * per + n_basic, ts, tplace, dsum);
        for (int i = n_basic + lane; i < n_moms; i += NT) {
            M[i] = (T)0;
            if (LOSS) Tg[i] = (T)0;
        }
        __syncthreads();
        if (ts.nsplit > 1) {
            for (int i = lane; i < n_basic; i += NT)
                for (int k = 0; k + 1 < ts.nsplit; k++) {
                    M[i] += L.part[k * per + i];
                    if (LOSS) Tg[i] += L.part[k * per + n_basic + i];
                }
            __syncthreads();
        }
    }

    // ---- products, energy, adjoint ------------------------------------------------------------
    {
        MTP_PHASE;
        if (LOSS && !no_tan) sweep_forward<T, LOSS>(p.fwd[NT / 256], M, Tg, lane);
        else sweep_forward<T, false>(p.fwd[NT / 256], M, Tg, lane);
    }
    T e_part = (T)0;
    {
        MTP_PHASE;
        for (int i = lane; i < n_moms; i += NT) {    // the table is dead: its place now holds the adjoints
            A[i] = (T)0;
            if (LOSS) Bm[i] = (T)0;
        }
        __syncthreads();
        // network buffers (H > 0): inputs q[S]; per neuron w1 tanh', and in loss mode tanh, tanh', tanh'', tau
        T* nnb = L.net;
        if constexpr (NET) {
            // one tanh layer of the centre's species on the shifted, scaled scalar moments; the
            // adjoint is seeded with dE_i/dM_k = sum_p w1_p tanh'(h_p) w0_pk / q_scaler_k
            // (nnMtp.h:470-507).  Loss mode also needs the derivative of that seed along the tangent:
            // tau_p = sum_k w0_pk Tg_k / q_scaler_k is the tangent of h_p, and the adjoint of
            // D_w E = sum_p w1_p tanh'(h_p) tau_p  w.r.t. M_k is  sum_p w1_p tanh''(h_p) tau_p w0_pk / q_scaler_k,
            // the seed of the mixed sweep (nnMtpLoss.h:216-610 computes the same quantities atom by atom).
            // A neuron's sum over the inputs, and an input's over the neurons, by 1, 2 .. 16 neighbouring lanes each, W weights
            // of a lane on their way together, the first of either sum ahead of what it waits for.  What bounds it is the trips to
            // the weights and the chain of their operations.  (A wavefront for four neurons at a time with sums over its 64 lanes,
            // then a lane for an input, against this, in us of the kernel: level 12, 20 neurons, 3000 atoms 37.6 and 33.9, 200 atoms
            // 25.6 and 23.5, the loss gradient of 16 structures of 64 atoms 45.5 and 41.4; level 20, 60 neurons, 152 and 143, 37.6
            // and 36.0, 221 and 197.)
            // At least two lanes to a neuron from 9 inputs on, four from 24 on, eight in fp32 from 128 on, in as many rounds as that
            // takes: fewer lanes read a few bytes of each of many rows at a time, whose lines are gone before they are used up
            // (one lane, two, four, eight; 3000 atoms: level 8, 9 inputs, 60 neurons 27.5, 27.2, 28.5, 32.0 us; level 10, 16
            // inputs, 100 neurons 42.8, 38.4, 39.2, 43.8; level 12, 29 inputs, 200 neurons 64.3, 56.0, 55.5, 64.6; level 20, 288
            // inputs, 200 neurons 463, 319, 250, 256, in fp32 383, 376, 179, 157).
            const int S = p.n_scalar, H = a.H;
            T* qv = nnb;                          // [S] network inputs
            T* hv = nnb + S;                      // [H] pre-activations, then w1 * tanh'
            T* n_th = hv + H;                     // loss mode: tanh, tanh', w1 tanh'' tau, tau   [H] each
            T* n_d1 = n_th + H;
            T* n_c2 = n_d1 + H;
            T* n_tau = n_c2 + H;
            // ... and the tangents of the inputs [S], where P and Q come in the last pass, or, when they do not fit there, where the
            // seeds come after them
            T* qt = mtp_tangents_at_pq(S, MTP_NC, nmus) ? L.pq : Bm;
            const T* w0 = a.w0 + (size_t)ti * H * S;
            const T* w1 = a.w1 + (size_t)ti * H;
            constexpr int W = LOSS ? 4 : 8;       // (eight: 8 more values spilled by the loss gradient)
            T w[W];
            const int lh = max(parts_log2(NT, H), S <= 8 ? 0 : S < 24 ? 1 : sizeof(T) == 4 && S >= 128 ? 3 : 2), ph = 1 << lh, ls = parts_log2(NT, S), ps = 1 << ls;
            const int hl = lane >> lh, hp = lane & (ph - 1), sl = lane >> ls, sp = lane & (ps - 1);
            // the wavefront's first neuron and input of a round
            const int hw = __builtin_amdgcn_readfirstlane(lane) >> lh, sw = __builtin_amdgcn_readfirstlane(lane) >> ls;
            // weights of neuron n and the inputs k0, k0 + ph ..; and of input k and the neurons n0, n0 + ps ..
            auto row_weights = [&](int n, int k0) __attribute__((always_inline)) {
                const unsigned at = __umul24(min(n, H - 1), S);
#pragma unroll
                for (int u = 0; u < W; u++) w[u] = w0[at + min(k0 + u * ph, S - 1)];
            };
            auto column_weights = [&](int k, int n0) __attribute__((always_inline)) {
                const unsigned at = min(k, S - 1);
#pragma unroll
                for (int u = 0; u < W; u++) w[u] = w0[__umul24(min(n0 + u * ps, H - 1), S) + at];
            };
            // W of the products of a sum: acc += w q[first + u step], below `end` (others may be infinite), and tac += w t[..]; by
            // halves, as the sums of the lanes (one after the other: energies in fp32 up to a tenth further from fp64)
            auto products = [&](T& acc, T& tac, const T* q, const T* t, int first, int step, int end, bool whole) __attribute__((always_inline)) {
                T v[W], d[LOSS ? W : 1];
                if (whole)                                     // wave-uniform
#pragma unroll
                    for (int u = 0; u < W; u++) {
                        v[u] = w[u] * q[first + u * step];
                        if constexpr (LOSS) d[u] = w[u] * t[first + u * step];
                    }
                else
#pragma unroll
                    for (int u = 0; u < W; u++) {
                        const int i = first + u * step, own = min(i, end - 1);
                        v[u] = w[u] * q[own];
                        if (i >= end) v[u] = (T)0;
                        if constexpr (LOSS) {
                            d[u] = w[u] * t[own];
                            if (i >= end) d[u] = (T)0;
                        }
                    }
#pragma unroll
                for (int n = W / 2; n > 0; n >>= 1)
#pragma unroll
                    for (int u = 0; u < n; u++) {
                        v[u] += v[u + n];
                        if constexpr (LOSS) d[u] += d[u + n];
                    }
                acc += v[0];
                if constexpr (LOSS) tac += d[0];
            };
            row_weights(hl, hp);
            const T w1_own = w1[min(lane, H - 1)];
            for (int s = lane; s < S; s += NT) {
                const int m = p.mapping[s];
                const T scaler = a.q_scaler[s];
                qv[s] = (M[m] - a.q_shift[s]) / scaler;
                if (LOSS) qt[s] = Tg[m] / scaler;
            }
            __syncthreads();
            for (int n0 = 0; n0 + hw < H; n0 += NT >> lh) {
                T acc = (T)0, tac = (T)0;
                for (int k0 = 0; k0 < S; k0 += W * ph) {
                    if (n0 + k0 > 0) row_weights(n0 + hl, k0 + hp);
                    products(acc, tac, qv, qt, k0 + hp, ph, S, k0 + W * ph <= S);
                }
                acc = parts_sum(acc, lh);
                if (LOSS) tac = parts_sum(tac, lh);
                if (hp == 0 && n0 + hl < H) {
                    hv[n0 + hl] = acc;
                    if (LOSS) n_tau[n0 + hl] = tac;
                }
            }
            column_weights(sl, sp);
            const int m_own = p.mapping[min(sl, S - 1)];
            const T scaler_own = a.q_scaler[min(sl, S - 1)];
            __syncthreads();
            for (int n = lane; n < H; n += NT) {
                const T th = tanh_t(hv[n]), w1n = n == lane ? w1_own : w1[n];
                const T d1 = (T)1 - th * th;
                e_part += w1n * th;
                hv[n] = w1n * d1;
                if (LOSS) {
                    n_th[n] = th; n_d1[n] = d1;
                    n_c2[n] = w1n * ((T)-2 * th * d1) * n_tau[n];
                }
            }
            if (LOSS && qt == Bm)
                for (int s = lane; s < S; s += NT) qt[s] = (T)0;
            __syncthreads();
            for (int i0 = 0; i0 + sw < S; i0 += NT >> ls) {
                const int k = i0 + sl;
                T acc = (T)0, bac = (T)0;
                for (int n0 = 0; n0 < H; n0 += W * ps) {
                    if (i0 + n0 > 0) column_weights(k, n0 + sp);
                    products(acc, bac, hv, n_c2, n0 + sp, ps, H, n0 + W * ps <= H);
                }
                acc = parts_sum(acc, ls);
                if (LOSS) bac = parts_sum(bac, ls);
                if (sp == 0 && k < S) {
                    const int m = i0 > 0 ? p.mapping[k] : m_own;
                    const T scaler = i0 > 0 ? a.q_scaler[k] : scaler_own;
                    A[m] = acc / scaler;
                    if (LOSS && a.nn_exact) Bm[m] = bac / scaler;
                }
            }
        } else if (seeded) {
            for (int s = lane; s < p.n_scalar; s += NT) A[p.mapping[s]] = a.row_seed[row * p.n_scalar + s];
        } else {
            for (int s = lane; s < p.n_scalar; s += NT) {
                const int mw = p.mapping_leaf[s], m = mw & 0xffff;
                const T w = a.lin[s] / a.q_scaler[s];
                if (!a.leaves_late || mw == m) e_part += w * M[m];
                A[m] = w;
            }
        }
        if (!LOSS && (a.e_sites || a.desc)) {
            if (a.desc)                                          // linearMtp.h:884-885: unscaled scalar moments
                for (int s = lane; s < p.n_scalar; s += NT) a.desc[row * p.n_scalar + s] = M[p.mapping[s]];
            const T e_row = block_sum<T, NT>(e_part, L.scratch, lane) + a.bias[ti];
            if (a.e_sites && lane == 0) a.e_sites[row] = e_row;  // linearMtp.h:594-599
            if (a.energy_only) return;
        }
        __syncthreads();
    }
    const int halves = csize <= 32 ? 2 : 1;       // lanes to a neighbour in the last passes
    [[maybe_unused]] int prog = 0;
    [[maybe_unused]] UnitSources<NT> sources;
    if constexpr (TILED) {
        MTP_PHASE;
        sources.load(p, halves, lane);
        prog = p.units[NT / 256][2 * (NT / 64) + lane];
    }
    {
        MTP_PHASE;
        // the leaves' moments: their part of the energy, or, for the loss gradient, the moments (and tangents) themselves;
        // mixed adjoints: linearMtpLoss.h:417-434; the reference's network backward has none (Bm stays zero)
        if (LOSS && !no_tan && (!NET || a.nn_exact))
            sweep_reverse<T, LOSS, !NET>(p.rev[NT / 256], M, A, Bm, (const T*)Tg, lane,
                [&](int m, T v, T t) __attribute__((always_inline)) { M[m] = v; Tg[m] = t; });
        else
            sweep_reverse<T, false, !NET>(p.rev[NT / 256], M, A, (T*)nullptr, (const T*)nullptr, lane,
                [&](int m, T v, T) __attribute__((always_inline)) {
                    if (LOSS) M[m] = v;
                    else e_part += A[m] * v;
                });
    }

    if (!LOSS) {
        // ---- pair derivatives ------------------------------------------------------------------
        // The adjoints of the basic moments as polynomial coefficients; the moments are dead.  Nested polynomials: two lanes to a neighbour
        // where a chunk has no more than 32, one otherwise; the wavefronts share the units.  General tables: within a chunk of nc
        // neighbours thread = group h * nc + neighbour j, and the groups (as many as fit, at most one per monomial row) share the rows.
        {
            MTP_PHASE;
            if constexpr (TILED) {
                sources.each(p, halves, lane, [&](int i, int m) __attribute__((always_inline)) { L.polys[i] = m == MTP_NO_MOMENT ? (T)0 : A[m]; });
            } else {
                scatter_polys<T, NT>(p, L.polys, A, lane);
            }
        }
        // Sums over the pairs, chunk by chunk, in wavefront 0's place in LDS (held by lane from chunk to chunk they cost the walk 24 registers).
        if (lane < 12) {
            MTP_PHASE;
            L.scratch[4 + lane] = (T)0;
        }
        for (int c0 = 0; c0 < nn; c0 += csize) {
            const int nc = min(csize, nn - c0);
            int nj; bool valid; T d[3] = {(T)0, (T)0, (T)0};
            __syncthreads();
            // (nested polynomials: a row of one chunk finds the table of the first pass still in place)
            {
                MTP_PHASE;
                build_table<T, TAB_MOMENTS, NT>(a, tab, pw, cf, lane, nc, c0, rcs, first, types, center, b, NF, &nj, &valid, d,
                                          !TILED || nchunks > 1, !TILED);
                if (!TILED || nchunks > 1) __syncthreads();
            }
            T gs = (T)0, wx = (T)0, wy = (T)0, wz = (T)0;
            T ux = (T)0, uy = (T)0, uz = (T)0, rinv = (T)0;
            // the pair claims an entry of its target's segment (zeros too: the count of a segment is the number of pairs
            // naming the target); claimed here, so that the walk covers the answer's way
            int rk = 0, ng, h, j;
            {
                MTP_PHASE;
                // (no load on its way beside the claims: a register of one, needed for something else, would wait for all of them.  vmcnt(0),
                // which the claims' addresses wait for anyway.  Level 10, 216 atoms 14.3 -> 13.6 us, level 16, 64 x 128 atoms 66.2 -> 64.7)
                __builtin_amdgcn_s_waitcnt(0x0f70);
                if (a.seg_cursor && lane < nc) rk = pair_claim_raw(&a.seg_cursor[b * NF + nj]);
                if constexpr (TILED) {
                    ng = NT / 64; h = wave; j = halves == 2 ? l64 & 31 : l64;
                    const T* t = tab + min(j, nc - 1) * E;
                    ux = t[OU + 0]; uy = t[OU + 1]; uz = t[OU + 2]; rinv = t[OU + 3];
                    const int n = uniform_array(p.units[NT / 256])[2 * wave], at = uniform_array(p.units[NT / 256])[2 * wave + 1];
                    T wt = (T)0;
                    auto add = [&](int mu, int, T r, T rx, T rt, T rz, T) __attribute__((always_inline)) {
                        const T g = t[OG + mu], dg = t[ODG + mu];
                        gs += dg * r;
                        wx += g * rx; wt += g * rt; wz += g * rz;
                    };
                    if (halves == 2) {
                        const bool up = l64 >= 32;
                        const T x = up ? uy : ux, y = up ? ux : uy;
                        nested<T, 2, false>(L.polys + (at >> 16) + (up ? p.half_at : 0), (const T*)nullptr, prog, n, x, y, uz, add);
                        wx += y * wt;
                        wy = x * wt;
                        const T sw = up ? wy : wx;
                        wy = up ? wx : wy;
                        wx = sw;
                        gs = wave::add_rows<32>(gs); wx = wave::add_rows<32>(wx); wy = wave::add_rows<32>(wy); wz = wave::add_rows<32>(wz);
                    } else {
                        nested<T, 1, false>(L.polys + (at & 0xffff), (const T*)nullptr, prog, n, ux, uy, uz, add);
                        wy = wt;
                    }
                } else {
                    ng = min(small_div(NT, nc), p.nrows);
                    h = small_div(lane, nc); j = lane - h * nc;
                    if (h < ng) {
                        const T* t = tab + j * E;
                        ux = t[OU + 0]; uy = t[OU + 1]; uz = t[OU + 2]; rinv = t[OU + 3];
                        pair_walk<T>(t, L.polys, L.rws, L.rws + p.nrows + 1, p.nrows, h, ng, OX, OY, OZ, OG, ODG, rinv, gs, wx, wy, wz);
                    }
                }
            }
            if (!TILED) __syncthreads();            // every thread has read its table row: the group sums take its place
            MTP_PHASE;
            // group sums in the order h = 0 .. ng-1
            if (!TILED) {
                T* gr = L.gred + lane * 4;
                gr[0] = gs; gr[1] = wx; gr[2] = wy; gr[3] = wz;
            } else if (NT > 64 && h > 0 && l64 < nc) {
                T* gr = L.gred + ((h - 1) * nc + l64) * 4;
                gr[0] = gs; gr[1] = wx; gr[2] = wy; gr[3] = wz;
            }
            if (!TILED || NT > 64) __syncthreads();
            T fv[12];
#pragma unroll
            for (int q = 0; q < 12; q++) fv[q] = (T)0;
            if (TILED ? lane < nc : h == 0) {
                if constexpr (TILED) {
#pragma unroll
                    for (int w = 0; w < NT / 64 - 1; w++) {
                        const T* gr = L.gred + (w * nc + j) * 4;
                        gs += gr[0]; wx += gr[1]; wy += gr[2]; wz += gr[3];
                    }
                    gs -= (ux * wx + uy * wy + uz * wz) * rinv;        // the monomials are homogeneous: k m = u . grad m
                } else {
                    for (int hh = 1; hh < ng; hh++) {
                        const T* gr = L.gred + (hh * nc + j) * 4;
                        gs += gr[0]; wx += gr[1]; wy += gr[2]; wz += gr[3];
                    }
                }
                T gx = gs * ux + wx * rinv;
                T gy = gs * uy + wy * rinv;
                T gz = gs * uz + wz * rinv;
                if (!valid) { gx = (T)0; gy = (T)0; gz = (T)0; }
                if (a.seg_cursor) {
                    asm volatile("" : "+v"(rk));         // (its bits taken apart here, not where the answer is on its way)
                    rk = pair_rank(rk);
                    const bool fits = (unsigned)rk < (unsigned)a.seg_cap;
                    T* dst = a.seg_g + (size_t)(fits ? (b * NF + nj) * a.seg_cap + rk : a.seg_spare) * 3;
                    if (!fits) atomicOr(a.status, ST_SEG_OVERFLOW);
                    dst[0] = gx; dst[1] = gy; dst[2] = gz;
                }
                if (SEED && a.pair_out) {         // padded layout of brcs; entries beyond the row stay zero
                    T* dst = a.pair_out + (row * a.U + c0 + j) * 3;
                    dst[0] = gx; dst[1] = gy; dst[2] = gz;
                }
                fv[0] = gx; fv[1] = gy; fv[2] = gz;
                fv[3] = -gx * d[0]; fv[4] = -gx * d[1]; fv[5] = -gx * d[2];
                fv[6] = -gy * d[0]; fv[7] = -gy * d[1]; fv[8] = -gy * d[2];
                fv[9] = -gz * d[0]; fv[10] = -gz * d[1]; fv[11] = -gz * d[2];
            }
            if (lane < 64) {
                T* const kept = L.scratch + 4;
#pragma unroll
                for (int q = 0; q < 12; q++) {
                    fv[q] = wave::all_sum(fv[q]) + kept[q];
                    kept[q] = fv[q];
                }
            }
        }
        MTP_PHASE;
        // only the threads of group 0 (inside wave 0) hold force and virial terms: the other wavefronts are done
        const double e_atom = (double)block_sum<T, NT>(e_part, L.scratch, lane);
        if (lane >= 64) return;
        const T* const fvsum = L.scratch + 4;
        double out[10];
        out[0] = e_atom + (seeded ? 0.0 : (double)a.bias[ti]);
#pragma unroll
        for (int q = 0; q < 9; q++) out[1 + q] = (double)fvsum[3 + q];
        if (lane == 0) {
            if (!SEED || a.force) {
                T* fo = a.force + ((size_t)b * NF + center) * 3;
                fo[0] = fvsum[0]; fo[1] = fvsum[1]; fo[2] = fvsum[2];
                if (a.seg_mark) pair_mark_own(&a.seg_cursor[b * NF + center]);
            }
            if (!SEED || a.partial) {
#pragma unroll
                for (int q = 0; q < 10; q++) a.partial[ev_partial(a.P, b, ii, q)] = out[q];
            }
        }
        return;
    }

    // ---- loss gradient ------------------------------------------------------------------------
    if (LOSS) {
        T cE;
        {
            MTP_PHASE;
            cE = seeded ? (T)1 : (a.cE_per_atom ? a.cE[row] : a.cE[b]);
        }
        {
            MTP_PHASE;
            // the last pass needs the adjoints of the basic moments while the table is back in its region
            if constexpr (TILED) {
                // (B's coefficients: cE times the adjoints plus the mixed ones)
                sources.each(p, halves, lane, [&](int i, int m) __attribute__((always_inline)) {
                    const T av = m == MTP_NO_MOMENT ? (T)0 : A[m];
                    L.Ab[i] = av;
                    L.Bb[i] = m == MTP_NO_MOMENT ? (T)0 : cE * av + Bm[m];
                });
            } else {
                scatter_polys<T, NT>(p, L.Ab, A, lane);
                scatter_polys<T, NT>(p, L.Bb, Bm, lane);
            }
            const int nblk = a.ntypes * nmus * K;
            T* const grow = a.gpart + row * a.ngrad;
            // everything but the coefficient block is written now: the pass over the neighbours below does
            // not read the moments or their tangents, and the group sums may take their place
            if constexpr (NET) {
                // coefficient block of the centre's species | w0[H, S] | w1[H] | bias
                const int S = p.n_scalar, H = a.H;
                const T* qv = L.net;
                const T* n_th = qv + S + H;
                const T* n_d1 = n_th + H;
                const T* n_tau = n_d1 + 2 * H;
                const T* w1 = a.w1 + (size_t)ti * H;
                const T* w0 = a.w0 + (size_t)ti * H * S;
                auto weight_gradient = [&](int q, int n, int k, T tk) __attribute__((always_inline)) {
                    const T d2 = (T)-2 * n_th[n] * n_d1[n];
                    if (a.nn_exact)
                        grow[nblk + q] = w1[n] * ((cE * n_d1[n] + d2 * n_tau[n]) * qv[k] + n_d1[n] * tk);
                    else        // nnMtpLoss.h:560-585: only the k' = k term of tau
                        grow[nblk + q] = w1[n] * (cE * n_d1[n] * qv[k] + tk * (n_d1[n] + d2 * w0[q] * qv[k]));
                };
                if (mtp_tangents_at_pq(S, MTP_NC, nmus))
                    for (int q = lane; q < H * S; q += NT) {
                        const int n = q / S, k = q - n * S;
                        weight_gradient(q, n, k, L.pq[k]);
                    }
                else        // (many inputs: a thread forms its input's tangent once; an entry at a time, level 22, 20 neurons: 328 -> 296 us)
                    for (int k = lane; k < S; k += NT) {
                        const T tk = Tg[p.mapping[k]] / a.q_scaler[k];
                        for (int n = 0; n < H; n++) weight_gradient(n * S + k, n, k, tk);
                    }
                for (int n = lane; n < H; n += NT) grow[nblk + H * S + n] = cE * n_th[n] + n_d1[n] * n_tau[n];
                if (lane == 0) grow[nblk + H * S + H] = cE;
            } else if (!seeded) {
                // linear coefficients and bias: linearMtpLoss.h:539-554
                for (int s = lane; s < p.n_scalar; s += NT)
                    grow[nblk + 1 + s] = (cE * M[p.mapping[s]] + Tg[p.mapping[s]]) / a.q_scaler[s];
                if (lane == 0) grow[nblk] = cE;
            }
            T* gacc = L.pq + 2 * MTP_NC * nmus + MTP_NC;          // [ntypes][nmus][K] for this centre type
            for (int q = lane; q < a.ntypes * nmus * K; q += NT) gacc[q] = (T)0;
        }
        for (int c0 = 0; c0 < nn; c0 += csize) {
            // equal chunks and as many thread groups per chunk as fit, as in the pair-derivative pass
            const int nc = min(csize, nn - c0);
            const int ng = min(small_div(NT, nc), MTP_NGMAX);
            const int h = TILED ? (lane < nc ? 0 : 1) : small_div(lane, nc), j = TILED ? lane : lane - h * nc;
            int nj; bool valid; T d[3];
            __syncthreads();
            {
                MTP_PHASE;
                build_table<T, TAB_GRADIENT, NT>(a, tab, pw, cf, lane, nc, c0, rcs, first, types, center, b, NF, &nj, &valid, d, !TILED || nchunks > 1, !TILED);
                if (!TILED || nchunks > 1) __syncthreads();
            }
            if constexpr (TILED) {
                MTP_PHASE;
                // P_mu(j), Q_mu(j): linearMtpLoss.h:438-536 with the k-sum factored out.  With A = sum adj m, B = sum (cE adj + mixed) m
                // over the basic moments of mu and k m = u . grad m (m is homogeneous),
                //   P_mu = B + (w - (w . u) u) . grad A / r,   Q_mu = (w . u) A.
                const T* t = tab + min(halves == 2 ? l64 & 31 : l64, nc - 1) * E;
                const T x = t[OU + 0], y = t[OU + 1], z = t[OU + 2];
                const T vx = no_tan ? (T)0 : t[OW + 0], vy = no_tan ? (T)0 : t[OW + 1], vz = no_tan ? (T)0 : t[OW + 2], wu = no_tan ? (T)0 : t[OW + 3];
                const bool up = halves == 2 && l64 >= 32, whole = p.nshares[NT / 256] == nmus && NT == 64;
                // along x (y in the upper half) at constant t, and along t
                const T hx = up ? vy : vx, ht = halves == 2 ? vx * y + vy * x : vy;
                const int n = uniform_array(p.units[NT / 256])[2 * wave], at = uniform_array(p.units[NT / 256])[2 * wave + 1];
                auto add = [&](int mu, int share, T r, T rx, T rt, T rz, T rb) __attribute__((always_inline)) {
                    T P = rb + hx * rx + ht * rt + vz * rz, Q = wu * r;
                    if (halves == 2) { P = wave::add_rows<32>(P); Q = wave::add_rows<32>(Q); }
                    if (l64 < nc) {
                        if (whole) {
                            L.pq[l64 * nmus + mu] = P;
                            L.pq[MTP_NC * nmus + l64 * nmus + mu] = Q;
                        } else {
                            T* o = L.gred + (share * nc + l64) * 2;
                            o[0] = P; o[1] = Q;
                        }
                    }
                };
                if (halves == 2) {
                    const int o = (at >> 16) + (up ? p.half_at : 0);
                    nested<T, 2, true>(L.Ab + o, L.Bb + o, prog, n, up ? y : x, up ? x : y, z, add);
                } else {
                    nested<T, 1, true>(L.Ab + (at & 0xffff), L.Bb + (at & 0xffff), prog, n, x, y, z, add);
                }
                __syncthreads();
                if (!whole) {
                    for (int q = lane; q < nc * nmus; q += NT) {
                        const int mu = small_div(q, nc), jn = q - mu * nc;
                        const unsigned long long shares = p.mu_shares[NT / 256];
                        int k0 = 0;
                        for (int m = 0; m < mu; m++) k0 += (int)(shares >> (8 * m)) & 255;
                        T P = (T)0, Q = (T)0;
                        for (int k = k0; k < k0 + ((int)(shares >> (8 * mu)) & 255); k++) {
                            P += L.gred[(k * nc + jn) * 2];
                            Q += L.gred[(k * nc + jn) * 2 + 1];
                        }
                        L.pq[jn * nmus + mu] = P;
                        L.pq[MTP_NC * nmus + jn * nmus + mu] = Q;
                    }
                    __syncthreads();
                }
            } else {
                MTP_PHASE;
                // P_mu(j), Q_mu(j): linearMtpLoss.h:438-536 with the k-sum factored out.  The groups take the polynomials in
                // turn, on from one mu to the next.  (All of a thread's sums kept to the end, with one round of group sums:
                // 100 registers instead of 70, so five wavefronts per SIMD instead of six, and the kernel 263 -> 320 us.)
                T* const Pm = L.pq;
                T* const Qm = L.pq + MTP_NC * nmus;
                int s = h < ng ? h : p.npoly;
                for (int mu = 0; mu < nmus; mu++) {
                    T Pv, Qv;
                    loss_walk<T>(tab + j * E, L.Ab, L.Bb, L.rws, s, L.rws[p.npoly + mu + 1], ng, OX, OY, OZ, OW, cE, no_tan, Pv, Qv);
                    {
                        T* gr = L.gred + lane * 2;
                        gr[0] = Pv; gr[1] = Qv;
                    }
                    __syncthreads();
                    if (h == 0) {
                        for (int hh = 1; hh < ng; hh++) {
                            const T* gr = L.gred + (hh * nc + j) * 2;
                            Pv += gr[0]; Qv += gr[1];
                        }
                        Pm[j * nmus + mu] = Pv; Qm[j * nmus + mu] = Qv;
                    }
                    __syncthreads();
                }
            }
            MTP_PHASE;
            const T* const Pm = L.pq;
            const T* const Qm = L.pq + MTP_NC * nmus;
            int* const tjs = (int*)(L.pq + 2 * MTP_NC * nmus);
            T* const gacc = L.pq + 2 * MTP_NC * nmus + MTP_NC;
            // The coefficient gradient: thread <- (part of the neighbours, mu, k), the parts' sums by species in the place of
            // the group sums.  (A thread per (mu, k) took 8.2 of the 77 thousand cycles an atom takes at level 16, this 3.3.)
            const int n1 = nmus * K, n2 = a.ntypes * n1;
            if (a.grad_parts > 1) {
                T* const part = L.gred;
                const int parts = a.grad_parts;
                for (int q = lane; q < parts * n2; q += NT) part[q] = (T)0;
                // tj of each neighbour of the chunk
                if (h == 0) tjs[j] = valid ? types[nj] : -1;
                __syncthreads();
                const int pt = small_div(lane, n1), q = lane - pt * n1;
                if (pt < parts) {
                    const int mu = small_div(q, K), k = q - mu * K;
                    T* const mine = part + pt * n2 + q;
                    for (int jn = pt; jn < nc; jn += parts) {
                        const int tj = tjs[jn];
                        const T* t = tab + jn * E;
                        const T g = t[OF + k] * Pm[jn * nmus + mu] + t[ODF + k] * Qm[jn * nmus + mu];
                        if (tj >= 0) mine[tj * n1] += g;
                    }
                }
                __syncthreads();
                for (int e = lane; e < n2; e += NT) gacc[e] += group_sum<T>(part + e, parts, n2);
            } else {
                // tj of each neighbour of the chunk, for the accumulation below
                if (h == 0) tjs[j] = valid ? types[nj] : -1;
                __syncthreads();
                // lanes <- (mu, k): sequential over neighbours keeps the sum order fixed
                for (int q = lane; q < n1; q += NT) {
                    const int mu = small_div(q, K), k = q - mu * K;
                    for (int jn = 0; jn < nc; jn++) {
                        const int tj = tjs[jn];
                        if (tj < 0) continue;
                        const T* t = tab + jn * E;
                        gacc[tj * n1 + q] += t[OF + k] * Pm[jn * nmus + mu] + t[ODF + k] * Qm[jn * nmus + mu];
                    }
                }
            }
        }
        __syncthreads();
        MTP_PHASE;
        const T* const gacc = L.pq + 2 * MTP_NC * nmus + MTP_NC;
        T* const grow = a.gpart + row * a.ngrad;
        for (int q = lane; q < a.ntypes * nmus * K; q += NT) grow[q] = gacc[q];
    }
}
#undef MTP_PHASE

// Sums of the gradient rows of a structure's atoms: a lane for an entry, a wavefront for each of four runs of the rows, which is summed in
// atom order, then the runs.  What bounds it is the trips to memory one after the other, then the rows' bytes: 64 x 128 atoms of three
// species at level 16 8.4 -> 6.6 us (and 131 -> 128.5 for the loss gradient, which writes half as much), of a network with 20 neurons
// 42 -> 24.6, 5 x 47 atoms at level 12 7.1 -> 4.0 (a thread for an entry and all rows, eight of them on their way, before; the rows of a
// linear potential with the blocks of all species).
constexpr int GRAD_RUNS = 4;
// Over the rows of species t (all for t < 0) entry `own`; the sum is in the threads of the first wavefront.
template <typename T>
__device__ __forceinline__ T grad_rows_sum(int P, int NF, int nrow, int own, int b, int t, const int* __restrict__ binum, const int* __restrict__ bilist,
                                           const int* __restrict__ btypes, const T* __restrict__ gpart)
{
    __shared__ T runs[GRAD_RUNS - 1][64];
    const int lane = threadIdx.x & 63, run = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int inum = max(min(binum[b], P), 0), i1 = (int)((long long)(run + 1) * inum / GRAD_RUNS);
    T acc = (T)0;
    // of 64 rows those of the species, sixteen on their way; the others are not read
    for (int i0 = (int)((long long)run * inum / GRAD_RUNS); i0 < i1; i0 += 64) {
        const int i = i0 + lane;
        bool mine = i < i1;
        if (t >= 0) {
            const int c = bilist[(size_t)b * P + min(i, i1 - 1)];
            const bool ok = mine && (unsigned)c < (unsigned)NF;
            mine = ok && btypes[(size_t)b * NF + (ok ? c : 0)] == t;
        }
        unsigned long long left = __ballot(mine);
        const T* const src = gpart + ((size_t)b * P + i0) * nrow + own;
        while (left) {
            T v[16];
            const int n = __popcll(left);
            int k = __builtin_ctzll(left);
#pragma unroll
            for (int u = 0; u < 16; u++) {
                v[u] = src[(size_t)k * nrow];
                left &= left - 1;                    // (the last one again where there are fewer)
                if (left) k = __builtin_ctzll(left);
            }
#pragma unroll
            for (int u = 0; u < 16; u++) acc += u < n ? v[u] : (T)0;
        }
    }
    if (run > 0) runs[run - 1][lane] = acc;
    __syncthreads();
#pragma unroll
    for (int k = 0; k + 1 < GRAD_RUNS; k++) acc += runs[k][lane];
    return acc;
}

// Linear potentials: row = [coefficient block of the centre's species | bias | linear coefficients], of which a launch without `dlin` and
// `dbias` may have the block alone.  Block x < ntypes * per takes the block and bias of a species, the others the linear coefficients.
template <typename T>
__global__ void __launch_bounds__(64 * GRAD_RUNS)
mtp_grad_reduce_kernel(int P, int NF, int nblk, int nlin, int ntypes, int nrow, const int* __restrict__ binum, const int* __restrict__ bilist,
                       const int* __restrict__ btypes, const T* __restrict__ gpart, T* __restrict__ dcoeffs, T* __restrict__ dlin,
                       T* __restrict__ dbias, const losskern::LossRmse<T> errors)
{
    const int b = blockIdx.y, per = (nblk + 64) / 64, x = blockIdx.x, lane = threadIdx.x & 63;
    if (x * 64 >= ntypes * per * 64 + nlin) {               // (a workgroup per structure too many, of which the first has the batch's errors)
        if (b == 0 && threadIdx.x < 64) losskern::loss_rmse(errors, lane);
        return;
    }
    const bool block = x < ntypes * per;
    const int t = block ? x / per : -1, q = (block ? x - t * per : x - ntypes * per) * 64 + lane;
    const int at = block ? q : nblk + 1 + q, end = block ? min(nblk + 1, nrow) : nblk + 1 + nlin;
    const T acc = grad_rows_sum<T>(P, NF, nrow, min(at, end - 1), b, t, binum, bilist, btypes, gpart);
    if (threadIdx.x >= 64 || at >= end) return;
    if (!block) { if (dlin) dlin[(size_t)b * nlin + q] = acc; }
    else if (q < nblk) { if (dcoeffs) dcoeffs[((size_t)b * ntypes + t) * nblk + q] = acc; }
    else if (dbias) dbias[(size_t)b * ntypes + t] = acc;
}

// Network potentials: row = [coefficient block of the centre's species | w0[H, S] | w1[H] | bias]; out[b] is laid out
// coeffs[ntypes^2 nmus K] | w0[ntypes H S] | w1[ntypes H] | bias[ntypes].  Block (x, t, b) sums the rows of species t.
template <typename T>
__global__ void __launch_bounds__(64 * GRAD_RUNS)
nnmtp_grad_reduce_kernel(int P, int NF, int nblk, int HS, int H, int ntypes, const int* __restrict__ binum,
                         const int* __restrict__ bilist, const int* __restrict__ btypes,
                         const T* __restrict__ gpart, T* __restrict__ dcoeffs, T* __restrict__ dw0,
                         T* __restrict__ dw1, T* __restrict__ dbias)
{
    const int b = blockIdx.z, t = blockIdx.y, nrow = nblk + HS + H + 1, q = blockIdx.x * 64 + (threadIdx.x & 63);
    const T acc = grad_rows_sum<T>(P, NF, nrow, min(q, nrow - 1), b, t, binum, bilist, btypes, gpart);
    if (threadIdx.x >= 64 || q >= nrow) return;
    if (q < nblk) { if (dcoeffs) dcoeffs[((size_t)b * ntypes + t) * nblk + q] = acc; }
    else if (q < nblk + HS) { if (dw0) dw0[((size_t)b * ntypes + t) * HS + q - nblk] = acc; }
    else if (q < nblk + HS + H) { if (dw1) dw1[((size_t)b * ntypes + t) * H + q - nblk - HS] = acc; }
    else if (dbias) dbias[(size_t)b * ntypes + t] = acc;
}
// Length of a linear potential's row, and its sums.
template <typename T>
int mtp_grad_row(const MtpArgs<T>& a, bool readout) { return a.ntypes * a.p.nmus * a.K + (readout ? 1 + a.p.n_scalar : 0); }
template <typename T>
int mtp_grad_reduce(const MtpArgs<T>& a, bool readout, T* dcoeffs, T* dlin, T* dbias, hipStream_t stream, const losskern::LossRmse<T>& errors = {})
{
    const int nblk = a.ntypes * a.p.nmus * a.K, nlin = readout ? a.p.n_scalar : 0;
    prof_begin("mtp_grad_reduce", stream);
    hipLaunchKernelGGL(mtp_grad_reduce_kernel<T>, dim3(a.ntypes * ((nblk + 64) / 64) + ceil_div(nlin, 64) + (errors.rmse ? 1 : 0), a.B), dim3(64 * GRAD_RUNS), 0, stream, a.P,
                       a.P + a.nghost, nblk, nlin, a.ntypes, a.ngrad, a.binum, a.bilist, a.btypes, a.gpart, dcoeffs, dlin, dbias, errors);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

// dst[(i * ncols) + col] = src[i] for i < n: one column of a row-major matrix
template <typename T>
__global__ void __launch_bounds__(256)
column_store_kernel(T* __restrict__ dst, const T* __restrict__ src, long long n, int ncols, int col)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i * ncols + col] = src[i];
}

// ---- linear-solver components, all scalar moments in one pass ------------------------------------------------
// Column s of the components is the E/F/V of the read-out e_s / q_scaler[s].  Its adjoint is non-zero on the
// ancestors of scalar moment s only (15 of 350 moments on average at level 16, 25 of 1352 at level 20), so the adjoints
// of all columns together are one reverse gather over the nodes (scalar moment, ancestor) of the plan, about as
// long as one ordinary reverse sweep, and a pair derivative sums over the basic ancestors of its column only.
// The kernel computes the moments once per atom, runs that gather, and writes the pair derivatives of every column
// to pb[pair][3][slots]; the kernels below add them up per atom (own pairs minus the pairs that name the atom, the
// latter in the fixed order of a sorted list) and per structure.
template <typename T>
struct CompArgs {
    T* pb;                  // [pairs of the structures from b0 on, 3, n_scalar]
    int b0;                 // first structure of the launch
    const int* pair_off;    // [rows + 1] first pair of each row
    const int* nnc;         // [rows] checked neighbour count of each row (0 for rows that are not evaluated)
    T* desc;                // [rows, n_scalar] scalar moments
    T* rowpart;             // [rows, 3, n_scalar] per row and column: sum of the pair derivatives
    int nc_cap, lds_basic_off;
    int node_region;        // entries of the node adjoints' place (even)
    int batch;              // neighbours whose D vectors are formed together (four or eight)
    int d_over_nodes;       // all groups of pieces are worked on at once, so the D vectors take the place of the node adjoints
};
template <typename T>
struct CompKernelArgs {
    MtpArgs<T> mtp;
    CompArgs<T> comp;
};

// six values from an even entry of LDS: 16-byte reads (8-byte in single precision)
__device__ __forceinline__ void load6(const double* p, double (&o)[6])
{
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double2 v = *reinterpret_cast<const double2*>(p + 2 * q);
        o[2 * q] = v.x; o[2 * q + 1] = v.y;
    }
}
__device__ __forceinline__ void load6(const float* p, float (&o)[6])
{
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const float2 v = *reinterpret_cast<const float2*>(p + 2 * q);
        o[2 * q] = v.x; o[2 * q + 1] = v.y;
    }
}

// Arguments anew in each phase, as in mtp_atom_kernel: 173 instead of 178 us for 32 structures of 128 atoms at level 16; with two
// places of D to a register, where sixteen of them and their adjoints had not fitted, 170.  (The basic moments by polynomials, as there:
// 173.  The pair derivatives as products of 16 x 16 tiles on the matrix cores, tiles without entries left out: 272; the fp64
// products take 41 us of that, the operands' chain of table, vector and gather the rest.)
#define COMP_PHASE                                                                                                         \
    [[maybe_unused]] auto& K_ = again(kernel_args<CompKernelArgs<T>>());                                                   \
    [[maybe_unused]] auto& a = K_.mtp;                                                                                     \
    [[maybe_unused]] auto& c = K_.comp;                                                                                    \
    [[maybe_unused]] auto& p = a.p;                                                                                        \
    [[maybe_unused]] const int NF = a.P, n_moms = p.n_moms, n_basic = p.n_basic, nmus = p.nmus, K = a.K, E = a.E,          \
                               S = p.n_scalar;                                                                             \
    [[maybe_unused]] const int OX = 0, OY = a.OY, OZ = a.OZ, OG = a.OG, ODG = a.ODG, OU = a.OU;                            \
    /* moments | node adjoints (+ the zero entry) | coefficients | neighbour table */                                      \
    [[maybe_unused]] T* const M = (T*)smem_raw;                                                                            \
    [[maybe_unused]] T* const X = M + ((n_moms + 1) & ~1);                                                                 \
    [[maybe_unused]] T* const cf = X + c.node_region;                                                                      \
    [[maybe_unused]] T* const tab = cf + a.ntypes * nmus * K;                                                              \
    [[maybe_unused]] unsigned* const bas = (unsigned*)(smem_raw + c.lds_basic_off);                                        \
    [[maybe_unused]] const size_t row = (size_t)b * a.P + ii;                                                              \
    [[maybe_unused]] const int* const first = a.bfirstneigh + row * a.U;                                                   \
    [[maybe_unused]] const T* const rcs = a.brcs + row * a.U * 3;                                                          \
    [[maybe_unused]] const int* const types = a.btypes + (size_t)b * NF

template <typename T, int NT>
__global__ void __launch_bounds__(NT, 4) mtp_components_kernel(const CompKernelArgs<T>)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int lane = threadIdx.x;
    const int ii = blockIdx.x, b = blockIdx.y + kernel_args<CompKernelArgs<T>>()->comp.b0;
    int nn, pair0, center, ti, nchunks, chunk;
    TableAhead<T> ahead;
    {
        COMP_PHASE;
        nn = uniform_array(c.nnc)[row];
        pair0 = uniform_array(c.pair_off)[row] - uniform_array(c.pair_off)[(size_t)c.b0 * a.P];     // of the structures of this launch
        center = uniform_array(a.bilist)[row];
        const int inum = uniform_array(a.binum)[b];
        Staged<unsigned, NT, 2> basics;
        basics.load(p.basic, n_basic, lane);
        if (ii >= inum || nn == 0) {                       // padded or refused row (k_rows flags the reasons)
            for (int s = lane; s < S; s += NT) c.desc[row * S + s] = (T)0;
            for (int q = lane; q < 3 * S; q += NT) c.rowpart[row * 3 * S + q] = (T)0;
            return;
        }
        nchunks = (nn + c.nc_cap - 1) / c.nc_cap;
        chunk = (nn + nchunks - 1) / nchunks;
        ahead.entries(rcs, first, lane, 0, min(chunk, nn));
        if ((unsigned)center >= (unsigned)NF) center = 0;
        ti = uniform_array(types)[center];
        if ((unsigned)ti >= (unsigned)a.ntypes) ti = 0;
        const T* const csrc = a.coeffs + (size_t)ti * a.ntypes * nmus * K;
        Staged<T, NT, 1> coefs;
        coefs.load(csrc, a.ntypes * nmus * K, lane);
        ahead.species(types, NF, center);
        for (int i = lane; i < n_moms; i += NT) M[i] = (T)0;
        for (int i = lane; i <= p.x_nodes; i += NT) X[i] = (T)0;
        basics.store(bas, p.basic, n_basic, lane);
        coefs.store(cf, csrc, a.ntypes * nmus * K, lane);
    }
    __syncthreads();

    // basic moments (as in mtp_atom_kernel)
    for (int c0 = 0;;) {
        COMP_PHASE;
        const int nc = min(chunk, nn - c0);
        int nj; bool valid; T d[3];
        build_table<T, TAB_MOMENTS, NT>(a, tab, tab, cf, lane, nc, c0, rcs, first, types, center, b, NF, &nj, &valid, d, true, true, ahead, true);
        __syncthreads();
        for (int i = lane; i < n_basic; i += NT) {
            const unsigned bw = bas[i];
            const int mu = bw & 255, ea = (bw >> 8) & 255, eb = (bw >> 16) & 255, ec = bw >> 24;
            T acc = (T)0;
            for (int j = 0; j < nc; j++) {
                const T* t = tab + j * E;
                acc += t[OG + mu] * (t[OX + ea] * t[OY + eb] * t[OZ + ec]);
            }
            M[i] += acc;
        }
        __syncthreads();
        c0 += chunk;
        if (c0 >= nn) break;
        ahead.entries(rcs, first, lane, c0, min(chunk, nn - c0));
        ahead.species(types, NF, center);
    }
    {
        COMP_PHASE;
        sweep_forward<T, false>(p.fwd[NT / 256], M, (T*)nullptr, lane);
    }
    {
        COMP_PHASE;
        for (int s = lane; s < S; s += NT) {
            c.desc[row * S + s] = M[p.mapping[s]];
            if (p.x_root[s] >= 0) X[p.x_root[s]] = (T)1 / a.q_scaler[s];       // (the columns of this launch)
        }
        if (p.x_polys)                                                        // (at most as many as basic moments)
            for (int i = lane; i < p.npoly; i += NT) bas[i] = p.polys_len[i];
        __syncthreads();
        sweep_reverse<T>(p.x, M, X, lane);
    }

    // Pair derivatives, four or eight neighbours at a time.  A thread forms, for one of them and the basic moments of a polynomial
    // (mu, a, b, z^0 .. z^(len-1)), the vectors
    //   D = d(g_mu x^a y^b z^c)/dr_j = m (g' - k g / r) u + g / r grad_u m
    // in LDS; then a lane owns a piece of a column's list of basic ancestors and sums adj * D over it for
    // pairs of neighbours (three 16-byte reads and six FMAs per ancestor, two ancestors' reads ahead).  The lane keeps its words and
    // their adjoints in registers over the whole row, and sums the column's force of the centre as it goes.  Up to four groups of 64
    // pieces are worked on at once; fewer groups share out the neighbours.
    // What bounds it: the latency and the number of the LDS reads of D, and the registers (128) that hold them.  Level 16, 64
    // structures of 128 atoms, thousands of a workgroup's cycles: 79 -> 66, of which D 16.9 -> 8.6 (a wavefront for a neighbour and a
    // lane for a basic moment before: ten reads of the table and 25 operations for each), the sums 24.1 -> 16.6 (the reads of one
    // ancestor at a time, the virial here instead of in comp_force_kernel, lists cut at sixteen words); the whole call 497 -> 467 us.
    // The words asked for ahead of the sweep, which they outlive: spilled, 544.
    const int l64 = lane & 63, wv = __builtin_amdgcn_readfirstlane(lane >> 6);
    constexpr int NW = NT / 64;
    int ngroups, at_once, shares, batch, log2_batch, plen;     // plen: D of a pair of neighbours
    T* D;
    {
        COMP_PHASE;
        ngroups = p.x_slots >> 6;
        at_once = min(ngroups, NW); shares = NW / at_once;
        batch = c.batch;
        plen = n_basic * 6 + 6;                                // (the banks of the pairs apart)
        log2_batch = batch == 8 ? 3 : 2;
        D = c.d_over_nodes ? X : (T*)smem_raw + (((tab - (T*)smem_raw) + (size_t)c.nc_cap * E + 1) & ~(size_t)1);
    }
    for (int g0 = 0; g0 < ngroups; g0 += NW) {
        const int g = g0 + wv % at_once, share = wv / at_once;
        const bool works = share < shares && g < ngroups;   // uniform over the wavefront
        int depth = 0, steps = 0;
        int off[MTP_SLOT_CAP / 2], col = -1, rem = 0;         // (two places of D to a register, 16 bits each)
        T adj[MTP_SLOT_CAP];
        if (works) {
            COMP_PHASE;
            depth = uniform_array(p.x_bdepth)[g];
            steps = uniform_array(p.x_bsteps)[g];
            const int* wp = p.x_bwords + p.x_bbase[g] + l64;
            col = p.x_seed[g * 64 + l64];
            rem = p.x_brem[g * 64 + l64];
            int w[MTP_SLOT_CAP];
#pragma unroll
            for (int k = 0; k < MTP_SLOT_CAP; k++) w[k] = k < depth ? wp[k * 64] : 0;
#pragma unroll
            for (int k = 0; k < MTP_SLOT_CAP; k++) adj[k] = k < depth ? X[(unsigned)w[k] & 0xffffu] : (T)0;
#pragma unroll
            for (int k = 0; k < MTP_SLOT_CAP; k += 2)
                off[k / 2] = (int)(((unsigned)w[k] >> 16) * 6 | ((unsigned)w[k + 1] >> 16) * 6 << 16);
        }
        T all[3] = {(T)0, (T)0, (T)0};                     // force of the centre
        for (int c0 = 0; c0 < nn; c0 += chunk) {
            const int nc = min(chunk, nn - c0);
            __syncthreads();                               // the adjoints, or the last batch of D, have been read
            if (nchunks > 1) {                             // (a single chunk's table is still in place)
                COMP_PHASE;
                int nj; bool valid; T d[3];
                build_table<T, TAB_MOMENTS, NT>(a, tab, tab, cf, lane, nc, c0, rcs, first, types, center, b, NF, &nj, &valid, d);
                __syncthreads();
            }
            for (int j0 = 0; j0 < nc; j0 += batch) {
                if (j0) __syncthreads();
                {
                    COMP_PHASE;
                    const int nb = min(batch, nc - j0);
                    if (p.x_polys) {
                        // thread <- (polynomial, neighbour of the batch): what its moments share is read and multiplied once
                        // (longest first, and the wavefronts in turn from either end)
                        for (int r = 0; r * NT < p.npoly * batch; r++) {
                            const int task = r * NT + (r & 1 ? (NT - 64 - wv * 64) + l64 : lane), jb = task & (batch - 1);
                            if (jb >= nb || task >= p.npoly * batch) continue;
                            const unsigned pw = bas[task >> log2_batch];
                            const T* t = tab + (j0 + jb) * E;
                            const int mu = pw & 7, ea = (pw >> 3) & 31, eb = (pw >> 8) & 31, len = (pw >> 13) & 31;
                            T* Dw = D + (jb >> 1) * plen + (jb & 1) * 3 + (int)(pw >> 18) * 6 + (len - 1) * 6;     // (highest power first)
                            const T ux = t[OU + 0], uy = t[OU + 1], uz = t[OU + 2], rinv = t[OU + 3];
                            const T gr = t[OG + mu] * rinv, xa = t[OX + ea], yb = t[OY + eb];
                            const T xy = xa * yb, hx = gr * ((T)ea * t[OX + max(ea - 1, 0)] * yb), hy = gr * ((T)eb * xa * t[OY + max(eb - 1, 0)]),
                                    hz = gr * xy, k0 = t[ODG + mu] - (T)(ea + eb) * gr;
                            T zc = (T)1, zd = (T)0, n = (T)0;                  // z^c, c z^(c-1), c
                            for (int i = 0; i < len; i++, Dw -= 6) {
                                const T gs = xy * zc * (k0 - n * gr);
                                Dw[0] = gs * ux + hx * zc;
                                Dw[1] = gs * uy + hy * zc;
                                Dw[2] = gs * uz + hz * zd;
                                n += (T)1;
                                zd = n * zc;
                                zc *= uz;
                            }
                        }
                    } else {
                        for (int jb = wv; jb < nb; jb += NW) {
                            const T* t = tab + (j0 + jb) * E;
                            T* Dw = D + (jb >> 1) * plen + (jb & 1) * 3;
                            const T ux = t[OU + 0], uy = t[OU + 1], uz = t[OU + 2], rinv = t[OU + 3];
                            for (int i = l64; i < n_basic; i += 64) {
                                const unsigned bw = bas[i];
                                const int mu = bw & 255, ea = (bw >> 8) & 255, eb = (bw >> 16) & 255, ec = bw >> 24;
                                const T gm = t[OG + mu], dg = t[ODG + mu];
                                const T xa = t[OX + ea], yb = t[OY + eb], zc = t[OZ + ec];
                                const T gs = xa * yb * zc * (dg - (T)(ea + eb + ec) * gm * rinv);
                                const T gr = gm * rinv;
                                Dw[i * 6 + 0] = gs * ux + gr * ((T)ea * t[OX + max(ea - 1, 0)] * yb * zc);
                                Dw[i * 6 + 1] = gs * uy + gr * ((T)eb * xa * t[OY + max(eb - 1, 0)] * zc);
                                Dw[i * 6 + 2] = gs * uz + gr * ((T)ec * xa * yb * t[OZ + max(ec - 1, 0)]);
                            }
                        }
                    }
                }
                __syncthreads();
                if (!works) continue;
                for (int jp = share * 2; jp < min(batch, nc - j0); jp += shares * 2) {
                    COMP_PHASE;
                    const T* Dp = D + (jp >> 1) * plen;
                    T gr[6], dv[2][2][6];
#pragma unroll
                    for (int q = 0; q < 6; q++) gr[q] = (T)0;
                    // (the next two vectors are on their way while two are worked on)
                    auto fetch = [&](T (&o)[2][6], int k) __attribute__((always_inline)) {
                        load6(Dp + ((unsigned)off[k / 2] & 0xffffu), o[0]);
                        load6(Dp + ((unsigned)off[k / 2] >> 16), o[1]);
                    };
                    fetch(dv[0], 0);
#pragma unroll
                    for (int k = 0; k < MTP_SLOT_CAP; k += 2) {
                        if (k < depth) {
                            if (k + 2 < MTP_SLOT_CAP) fetch(dv[k / 2 + 1 & 1], k + 2 < MTP_SLOT_CAP ? k + 2 : 0);
#pragma unroll
                            for (int u = 0; u < 2; u++)
#pragma unroll
                                for (int q = 0; q < 6; q++) gr[q] += adj[k + u] * dv[k / 2 & 1][u][q];
                        }
                    }
                    if (steps) piece_sums(gr, rem, steps);          // a long list's pieces sit in neighbouring lanes
                    T* dst = c.pb + ((size_t)(pair0 + c0 + j0 + jp) * 3) * S + col;
#pragma unroll
                    for (int o = 0; o < 2; o++) {
                        if (j0 + jp + o >= nc) continue;    // (the other half of D is not of this row)
#pragma unroll
                        for (int q = 0; q < 3; q++) {
                            all[q] += gr[o * 3 + q];
                            if (col >= 0) dst[(size_t)(o * 3 + q) * S] = gr[o * 3 + q];
                        }
                    }
                }
            }
        }
        // the shares of a group, through LDS
        if (shares > 1) {
            __syncthreads();
            if (works && share > 0)
#pragma unroll
                for (int q = 0; q < 3; q++) D[((wv - at_once) * 3 + q) * 64 + l64] = all[q];
            __syncthreads();
            if (share == 0)
                for (int o = wv; o < (shares - 1) * at_once; o += at_once)
#pragma unroll
                    for (int q = 0; q < 3; q++) all[q] += D[(o * 3 + q) * 64 + l64];
        }
        if (works && share == 0 && col >= 0) {
            COMP_PHASE;
            T* o = c.rowpart + row * 3 * S + col;
#pragma unroll
            for (int q = 0; q < 3; q++) o[(size_t)q * S] = all[q];
        }
    }
}
#undef COMP_PHASE

// rows that the components kernel evaluates, with the checks of mtp_atom_kernel; row_of1[b, atom] = 1 + the row whose
// centre the atom is
__global__ void __launch_bounds__(256)
comp_rows_kernel(int B, int P, int U, int ntypes, const int* __restrict__ binum, const int* __restrict__ bilist,
                 const int* __restrict__ bnumneigh, const int* __restrict__ btypes, int* __restrict__ nnc,
                 int* __restrict__ row_of1, int* __restrict__ status)
{
    const int row = blockIdx.x * 256 + threadIdx.x;
    if (row > B * P) return;
    if (row == B * P) { nnc[row] = 0; return; }
    const int b = row / P, ii = row - b * P;
    int nn = 0;
    if (ii < binum[b]) {
        nn = bnumneigh[row];
        if (nn > U) { atomicOr(status, ST_NEIGH_OVERFLOW); nn = U; }
        if (nn < 0) nn = 0;
        const int center = bilist[row];
        if ((unsigned)center >= (unsigned)P) { atomicOr(status, ST_BAD_NEIGHBOR); nn = 0; }
        else {
            if ((unsigned)btypes[(size_t)b * P + center] >= (unsigned)ntypes) { atomicOr(status, ST_BAD_TYPE); nn = 0; }
            row_of1[(size_t)b * P + center] = row + 1;
        }
    }
    nnc[row] = nn;
}

// The pairs that name each atom, by row * U + slot (B P U is below 2^31).  Each atom has room for `cap` of them (the row length
// of the list: enough for every list built with one cutoff), so one pass lists them; when an atom is named more often (spill[0]
// counts what found no room) the pass is repeated for counts only and then into segments of the right lengths (seg).
__global__ void __launch_bounds__(256)
comp_incoming_kernel(int B, int P, int U, const int* __restrict__ nnc, const int* __restrict__ bfirstneigh, int* __restrict__ cnt, const int* __restrict__ seg, int cap,
                     int* __restrict__ inc, int* __restrict__ spill)
{
    const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
    if (q >= (long long)B * P * U) return;
    const int row = (int)(q / U), j = (int)(q - (long long)row * U);
    if (j >= nnc[row]) return;
    const int nj = bfirstneigh[q];
    if ((unsigned)nj >= (unsigned)P) return;             // flagged by the components kernel's table
    const int tg = (row / P) * P + nj;
    const int place = atomicAdd(cnt + tg, 1);
    if (!inc) return;
    if (seg) inc[seg[tg] + place] = (int)q;
    else if (place < cap) inc[(size_t)tg * cap + place] = (int)q;
    else atomicAdd(spill, 1);
}

// Force column of every atom: its own row's sum minus the pairs that name it, in the order of their places in the lists; on the
// way these pairs' virial.  The pairs arrive in any order: a wavefront ranks those of its atom in LDS, up to COMP_SORT of them; a
// longer list is walked from each place to the next larger one.  Columns from S on (species counts) are zero.  A workgroup takes
// COMP_ROWS atoms in a row and sums up their virials, and the energies of as many rows, in order: written by each wavefront and
// summed by a kernel of its own they were 55 MB out and in at 64 structures of 128 atoms, 15 us beside 2 x 42, and the kernel that
// sums the workgroups took 8 with a thread to a column, now 5 with one to each of its ten values; the call 421 -> 402 us.  (Eight
// atoms to a workgroup: two of them fit no compute unit at the 156 registers of two columns in fp64, and at 128 112 bytes spill.)
// Bound by the reads of the pair derivatives, under which the virial's operations hide (in mtp_components_kernel they took a
// fifth of its instructions and the registers of four more reads in flight); sorting the lists by insertion, one thread per
// atom, used to take as long as they do (95 us beside 98 us at 64 structures of 128 atoms).
// With more than 64 columns a lane takes two of them, 64 apart, so that an atom's pairs are ranked once; the displacements of the
// first COMP_DISP pairs lie in LDS (of 256: 20 instead of 32 wavefronts to a compute unit).  2 x 50 -> 2 x 41 us there.  One column
// to a lane and two, 6,400 atoms: 53 columns 40.0 and 42.9 us, 65 67.6 and 56.4, 93 85.1 and 72.7, 127 109.5 and 97.5, 151 136.6 and
// 136.4, 261 243.6 and 249.3 (a last block half of which has no column); fp32 24.9 and 27.0, 38.2 and 28.5, 52.8 and 38.0, 65.5 and
// 52.6, 83.3 and 75.4, 130.5 and 122.7; 160 atoms, 93 columns 11.6 and 12.8.
constexpr int COMP_SORT = 256, COMP_DISP = 128, COMP_ROWS = 4;

template <typename T, int NC>
__global__ void __launch_bounds__(64 * COMP_ROWS, 3)
comp_force_kernel(int S, int n, int P, int cap, int U, int b0, const int* __restrict__ binum, const int* __restrict__ bilist,
                  const int* __restrict__ btypes, const int* __restrict__ pair_off, const int* __restrict__ row_of1, const int* __restrict__ cnt,
                  const int* __restrict__ seg, const int* __restrict__ inc, const T* __restrict__ brcs, const T* __restrict__ pb,
                  const T* __restrict__ rowpart, const T* __restrict__ desc, T* __restrict__ part, T* __restrict__ fcomp)
{
    struct Own { int list[COMP_SORT], order[COMP_SORT]; T disp[COMP_DISP][3]; };
    constexpr int COLS = 64 * NC;
    __shared__ union { Own own[COMP_ROWS]; T vir[COMP_ROWS][3][COLS]; } sh;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nblocks = (P + COMP_ROWS - 1) / COMP_ROWS, bb = blockIdx.x / nblocks, blk = blockIdx.x - bb * nblocks, b = b0 + bb;
    const int first = b * P + blk * COMP_ROWS, t = first + wave, col0 = blockIdx.y * COLS + lane;
    const bool there = blk * COMP_ROWS + wave < P;
    int* const list = sh.own[wave].list;
    int* const order = sh.own[wave].order;
    T (* const disp)[3] = sh.own[wave].disp;
    auto wave_sync = [&]() __attribute__((always_inline)) {           // (what a wavefront keeps in LDS is its own)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    T f[NC][3], vir[NC][9];
#pragma unroll
    for (int c = 0; c < NC; c++) {
#pragma unroll
        for (int i = 0; i < 9; i++) vir[c][i] = (T)0;
#pragma unroll
        for (int i = 0; i < 3; i++) f[c][i] = (T)0;
    }
    if (there) {
    const int* v = inc + (seg ? (size_t)seg[t] : (size_t)t * cap);
    const int m = seg ? seg[t + 1] - seg[t] : min(cnt[t], cap);
    const int r1 = row_of1[t], base = pair_off[(size_t)b0 * P];          // pb holds the pairs from structure b0 on
    const bool ranked = m <= COMP_SORT;
    int s[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) s[c] = min(col0 + c * 64, S - 1);
    auto pair_of = [&](int q) __attribute__((always_inline)) { const int row = q / U; return pair_off[row] + (q - row * U) - base; };
    if (ranked) {
        for (int k = lane; k < m; k += 64) list[k] = v[k];
        wave_sync();
        int place[COMP_SORT / 64];
#pragma unroll
        for (int u = 0; u < COMP_SORT / 64; u++) {
            const int k = u * 64 + lane;
            if (u * 64 >= m) break;
            if (k >= m) continue;
            const int x = list[k], pair = pair_of(x);
            T d[3];
#pragma unroll
            for (int q = 0; q < 3; q++) d[q] = brcs[(size_t)x * 3 + q];
            int r = 0;
            for (int i = 0; i < m; i++) r += list[i] < x;
            place[u] = r;
            order[r] = pair;
            if (r < COMP_DISP)
#pragma unroll
                for (int q = 0; q < 3; q++) disp[r][q] = d[q];
        }
        wave_sync();
        if (m > COMP_DISP) {                             // the places in the lists too, in order
            int x[COMP_SORT / 64];
#pragma unroll
            for (int u = 0; u < COMP_SORT / 64; u++)
                if (u * 64 + lane < m) x[u] = list[u * 64 + lane];
            wave_sync();
#pragma unroll
            for (int u = 0; u < COMP_SORT / 64; u++)
                if (u * 64 + lane < m) list[place[u]] = x[u];
            wave_sync();
        }
    }
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int i = 0; i < 3; i++) f[c][i] = r1 > 0 ? rowpart[((size_t)(r1 - 1) * 3 + i) * S + s[c]] : (T)0;
    auto take = [&](const T (&g)[NC][3], T d0, T d1, T d2) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
                f[c][i] -= g[c][i];
                vir[c][i * 3 + 0] -= g[c][i] * d0;
                vir[c][i * 3 + 1] -= g[c][i] * d1;
                vir[c][i * 3 + 2] -= g[c][i] * d2;
            }
    };
    auto fetch = [&](T (&g)[NC][3], int pair) __attribute__((always_inline)) {
        const T* src = pb + (size_t)pair * 3 * S;
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int i = 0; i < 3; i++) g[c][i] = src[(size_t)i * S + s[c]];
    };
    if (ranked) {
        for (int k0 = 0; k0 < m; k0 += 4) {              // twelve loads of a column in flight
            T g[4][NC][3];
#pragma unroll
            for (int u = 0; u < 4; u++) fetch(g[u], order[min(k0 + u, m - 1)]);
            if (k0 + 4 <= COMP_DISP || m <= COMP_DISP) {
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (k0 + u < m) take(g[u], disp[k0 + u][0], disp[k0 + u][1], disp[k0 + u][2]);
            } else {
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (k0 + u < m) {
                        const T* d = brcs + (size_t)list[k0 + u] * 3;
                        take(g[u], d[0], d[1], d[2]);
                    }
            }
        }
    } else {
        int last = -1;
        for (int k = 0; k < m; k++) {
            int next = 0x7fffffff;
            for (int i = lane; i < m; i += 64) {
                const int x = v[i];
                if (x > last && x < next) next = x;
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) next = min(next, __shfl_xor(next, off, 64));
            last = next;
            T g[NC][3];
            fetch(g, pair_of(next));
            const T* d = brcs + (size_t)next * 3;
            take(g, d[0], d[1], d[2]);
        }
    }
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int col = col0 + c * 64;
        if (col < n)
#pragma unroll
            for (int i = 0; i < 3; i++) fcomp[((size_t)t * 3 + i) * n + col] = col < S ? f[c][i] : (T)0;
    }
    }
    // the sums of the atoms of the workgroup, in order: three components at a time through the lists' place
    T* const out = part + ((size_t)b * nblocks + blk) * 10 * n;
    const int here = min(COMP_ROWS, P - blk * COMP_ROWS);
#pragma unroll
    for (int q = 0; q < 3; q++) {
        __syncthreads();
        if (there)
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int i = 0; i < 3; i++) sh.vir[wave][i][c * 64 + lane] = vir[c][q * 3 + i];
        __syncthreads();
        for (int o = threadIdx.x; o < 3 * COLS; o += 64 * COMP_ROWS) {
            const int i = o / COLS, c = o - i * COLS, col = blockIdx.y * COLS + c;
            if (col >= n) continue;
            T sum = (T)0;
            if (col < S)
                for (int w = 0; w < here; w++) sum += sh.vir[w][i][c];
            out[(size_t)(1 + q * 3 + i) * n + col] = sum;
        }
    }
    // ... and the energies of the rows; column S + t counts those whose centre has species t
    const int rows = min(here, binum[b] - blk * COMP_ROWS);
    for (int c = threadIdx.x; c < COLS; c += 64 * COMP_ROWS) {
        const int col = blockIdx.y * COLS + c;
        if (col >= n) continue;
        T e = (T)0;
        if (col < S) {
#pragma unroll
            for (int u = 0; u < COMP_ROWS; u++)
                if (u < rows) e += desc[(size_t)(first + u) * S + col];
        } else {
            for (int u = 0; u < rows; u++) {
                const int center = bilist[first + u];
                if ((unsigned)center < (unsigned)P && btypes[(size_t)b * P + center] == col - S) e += (T)1;
            }
        }
        out[col] = e;
    }
}

// Energy and virial columns per structure: the workgroups' sums (comp_force_kernel) in order; part[B][nblocks][10][n].
template <typename T>
__global__ void __launch_bounds__(64)
comp_structure_kernel(int n, int S, int nblocks, const T* __restrict__ q_scaler, const T* __restrict__ part,
                      T* __restrict__ ecomp, T* __restrict__ vcomp)
{
    const int b = blockIdx.x, s = blockIdx.y * 64 + threadIdx.x, i = blockIdx.z;        // (a component to a workgroup)
    if (s >= n) return;
    const T* const o = part + ((size_t)b * nblocks * 10 + i) * n + s;
    T acc = (T)0;
#pragma unroll 16
    for (int blk = 0; blk < nblocks; blk++) acc += o[(size_t)blk * 10 * n];
    if (i == 0) ecomp[(size_t)b * n + s] = s < S ? acc / q_scaler[s] : acc;
    else vcomp[((size_t)b * 9 + i - 1) * n + s] = acc;
}

// counts[b, t] += 1 for every evaluated row whose centre has species t (integer atomics: exact in any order)
__global__ void __launch_bounds__(256)
species_count_kernel(int B, int P, int ntypes, const int* __restrict__ binum, const int* __restrict__ bilist,
                     const int* __restrict__ btypes, int* __restrict__ counts)
{
    const int row = blockIdx.x * 256 + threadIdx.x;
    if (row >= B * P) return;
    const int b = row / P, ii = row - b * P;
    if (ii >= binum[b]) return;
    const int c = bilist[row];
    if ((unsigned)c >= (unsigned)P) return;
    const int t = btypes[(size_t)b * P + c];
    if ((unsigned)t < (unsigned)ntypes) atomicAdd(counts + b * ntypes + t, 1);
}

// eye[s * S + s] = 1 (the matrix is zero-filled before, may be null); ecomp[b, S + t] = counts[b, t]
template <typename T>
__global__ void __launch_bounds__(256)
lin_components_init_kernel(T* __restrict__ eye, int S, T* __restrict__ ecomp, int B, int ntypes,
                           const int* __restrict__ counts)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (eye && i < S) eye[(size_t)i * S + i] = (T)1;
    if (i < B * ntypes) {
        const int b = i / ntypes, t = i - b * ntypes;
        ecomp[(size_t)b * (S + ntypes) + S + t] = (T)counts[i];
    }
}

// Gram-Schmidt over the nmus radial functions, each the vector of its ntypes^2 * K coefficients
// (schmidt_orth.h:38-116), in the reference's summation order by one thread (the problem is tiny).
template <typename T>
__global__ void schmidt_orth_kernel(T* __restrict__ out, const T* __restrict__ in, int npairs, int nmus, int K)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const int n = npairs * nmus * K;
    for (int i = 0; i < n; i++) out[i] = in[i];
    for (int k1 = 0; k1 < nmus; k1++) {
        for (int k2 = 0; k2 < k1; k2++) {
            T norm2 = (T)0, scal = (T)0;
            for (int pr = 0; pr < npairs; pr++)
                for (int xi = 0; xi < K; xi++) {
                    const T v1 = out[(pr * nmus + k1) * K + xi], v2 = out[(pr * nmus + k2) * K + xi];
                    norm2 += v2 * v2;
                    scal += v1 * v2;
                }
            for (int pr = 0; pr < npairs; pr++)
                for (int xi = 0; xi < K; xi++)
                    out[(pr * nmus + k1) * K + xi] -= out[(pr * nmus + k2) * K + xi] * scal / norm2;
        }
        T norm2 = (T)1e-10;
        for (int pr = 0; pr < npairs; pr++)
            for (int xi = 0; xi < K; xi++) {
                const T v = out[(pr * nmus + k1) * K + xi];
                norm2 += v * v;
            }
        const T norm = sqrt_t(norm2);
        for (int pr = 0; pr < npairs; pr++)
            for (int xi = 0; xi < K; xi++) out[(pr * nmus + k1) * K + xi] /= norm;
    }
}

// ---- plan construction ---------------------------------------------------------------------------
std::mutex g_plan_mutex;
std::set<MtpPlan*> g_plans;

// Order in which 16 lanes read their vectors D_b (pairs of neighbours: three 16-byte reads 48 bytes apart): lists[q] are
// the words (node | basic << 16) of lane q, at most `depth` of them; out[k * stride + q] is the lane's word of step k, or
// a word of the node `zero_node` where it has none.  16 lanes read from the 64 banks at a time, and lanes that name basic
// moments of the same remainder mod 16 wait for each other unless they name the same one.  Greedy: the lanes with the
// fewest steps to spare choose first, each the moment whose banks are least taken.
void spread_over_banks(const std::vector<std::vector<int>>& lists, int depth, int zero_node, int* out, int stride)
{
    constexpr int LANES = 16;
    int left[LANES][MTP_SLOT_CAP], count[LANES];
    for (int q = 0; q < LANES; q++) {
        count[q] = (int)lists[q].size();
        std::copy(lists[q].begin(), lists[q].end(), left[q]);
    }
    for (int k = 0; k < depth; k++) {
        int order[LANES];                               // lanes by the steps they have to spare
        for (int q = 0; q < LANES; q++) {
            int at = q;
            for (; at > 0 && count[order[at - 1]] < count[q]; at--) order[at] = order[at - 1];
            order[at] = q;
        }
        int taken[LANES][LANES], ntaken[LANES] = {0}, most = 0, any = 0;
        bool waits[LANES] = {false};
        for (int o = 0; o < LANES; o++) {
            const int q = order[o];
            int pick = -1, load = 1 << 30;
            for (int i = 0; i < count[q] && load > 0; i++) {
                const int b = left[q][i] >> 16, bank = b % LANES;
                const bool same = std::find(taken[bank], taken[bank] + ntaken[bank], b) != taken[bank] + ntaken[bank];
                const int l = same ? 0 : ntaken[bank] + 1;
                if (l < load) { load = l; pick = i; }
            }
            if (pick < 0 || (depth - k > count[q] && load > 1 && load > most)) { waits[q] = true; continue; }
            const int w = left[q][pick], bank = (w >> 16) % LANES;
            left[q][pick] = left[q][--count[q]];
            out[(size_t)k * stride + q] = w;
            any = w >> 16;
            if (load > 0) taken[bank][ntaken[bank]++] = w >> 16;
            most = std::max(most, ntaken[bank]);
        }
        for (int q = 0; q < LANES; q++)
            if (waits[q]) out[(size_t)k * stride + q] = zero_node | (any << 16);
    }
}

// 256 threads per atom or 64 (the rule is at its definition), and whether a launch then goes by tiles and nested polynomials: others take
// 256 threads
bool wide_atoms(int n_moms, bool loss, bool network, bool fp64);
bool tiled_launch(int ntiles, bool loss, bool wide) { return ntiles > 0 && ntiles <= tiles_of(loss, wide ? 256 : 64) * (wide ? 4 : 1); }
bool wide_launch(int n_moms, int ntiles, bool loss, bool network, bool fp64)
{
    const bool wide = wide_atoms(n_moms, loss, network, fp64);
    return wide || !tiled_launch(ntiles, loss, wide);
}

int plan_create(int n_moms, int n_basic, const int* basic, int n_times, const int* times, int n_scalar,
                const int* mapping, MtpPlan** out)
{
    A2P_REQUIRE(n_moms > 0 && n_basic > 0 && n_basic <= n_moms && n_times >= 0 && n_scalar > 0,
                A2P_ERR_INVALID, "mtp plan: bad table sizes");
    A2P_REQUIRE(basic && mapping && (times || n_times == 0), A2P_ERR_INVALID, "mtp plan: null table");
    int nmus = 0, kmax = 0;
    for (int i = 0; i < n_basic; i++) {
        const int* q = basic + i * 4;
        A2P_REQUIRE(q[0] >= 0 && q[1] >= 0 && q[2] >= 0 && q[3] >= 0, A2P_ERR_INVALID,
                    "mtp plan: negative entry in alpha_index_basic");
        A2P_REQUIRE(i == 0 || q[0] >= basic[(i - 1) * 4], A2P_ERR_INVALID,
                    "mtp plan: alpha_index_basic is not grouped by radial function index");
        nmus = std::max(nmus, q[0] + 1);
        kmax = std::max(kmax, q[1] + q[2] + q[3]);
    }
    A2P_REQUIRE(nmus <= MTP_NMUS_MAX, A2P_ERR_INVALID, "mtp plan: more than %d radial functions", MTP_NMUS_MAX);
    A2P_REQUIRE(kmax <= 24, A2P_ERR_INVALID, "mtp plan: monomial degree %d too large", kmax);
    std::vector<int> level(n_moms, 0), last_write(n_moms, -1);
    for (int e = 0; e < n_times; e++) {
        const int* q = times + e * 4;
        A2P_REQUIRE(q[0] >= 0 && q[0] < n_moms && q[1] >= 0 && q[1] < n_moms && q[3] >= n_basic &&
                        q[3] < n_moms,
                    A2P_ERR_INVALID, "mtp plan: alpha_index_times entry %d out of range", e);
        last_write[q[3]] = e;
    }
    int n_levels = 0;
    for (int e = 0; e < n_times; e++) {
        const int* q = times + e * 4;
        for (int s = 0; s < 2; s++)
            A2P_REQUIRE(last_write[q[s]] < e, A2P_ERR_INVALID,
                        "mtp plan: moment %d is read by product %d before its last contribution (%d); "
                        "the table cannot be executed level by level", q[s], e, last_write[q[s]]);
        level[q[3]] = std::max(level[q[3]], 1 + std::max(level[q[0]], level[q[1]]));
        n_levels = std::max(n_levels, level[q[3]]);
    }
    std::vector<char> seen(n_moms, 0);
    for (int s = 0; s < n_scalar; s++) {
        A2P_REQUIRE(mapping[s] >= 0 && mapping[s] < n_moms, A2P_ERR_INVALID, "mtp plan: mapping out of range");
        A2P_REQUIRE(!seen[mapping[s]], A2P_ERR_INVALID, "mtp plan: alpha_moment_mapping repeats a moment");
        seen[mapping[s]] = 1;
    }
    A2P_REQUIRE(n_moms < 8192, A2P_ERR_INVALID, "mtp plan: more than 8191 moments");    // 16-bit byte offsets
    // Packed terms of each moment, in the order given; a list of products (mtp_plan.h) in pairs of the same multiplicity, whose
    // lower half as a double is zero: one that takes more than 21 bits is the sum of two.
    struct Term { int x; double mult; };
    struct Lists {
        std::vector<int> off;
        std::vector<Term> terms;
        int longest = 0;                                   // as given
        Lists(int n, const std::vector<std::pair<int, Term>>& given, bool products)
        {
            fill(n, given);
            for (int m = 0; m < n; m++) longest = std::max(longest, size(m));
            if (!products) return;
            auto low = [](const Term& t) { return std::fabs(t.mult) < 1 << 20 ? 0.0 : std::fmod(t.mult, 2048.0); };
            if (std::any_of(terms.begin(), terms.end(), [&](const Term& t) { return low(t) != 0.0; })) {
                std::vector<std::pair<int, Term>> cut;
                for (const auto& t : given) {
                    const double l = low(t.second);
                    cut.emplace_back(t.first, Term{t.second.x, t.second.mult - l});
                    if (l != 0.0) cut.emplace_back(t.first, Term{t.second.x, l});
                }
                fill(n, cut);
            }
            std::vector<Term> pairs;
            pairs.reserve(2 * terms.size());
            for (int m = 0; m < n; m++) {
                const auto begin = terms.begin() + off[m], end = terms.begin() + off[(size_t)m + 1];
                if (end - begin > 32) std::stable_sort(begin, end, [](const Term& x, const Term& y) { return x.mult < y.mult; });
                else                                       // (no buffer of its own)
                    for (auto t = begin; t != end; ++t)
                        for (auto u = t; u != begin && u->mult < (u - 1)->mult; --u) std::swap(*u, *(u - 1));
                off[m] = (int)pairs.size();
                for (auto t = begin; t != end; ++t) {
                    pairs.push_back(*t);
                    if ((pairs.size() - off[m]) % 2 == 0 || (t + 1 != end && (t + 1)->mult == t->mult)) continue;
                    pairs.back().mult *= 0.5;              // (alone: twice, each time half)
                    pairs.push_back(pairs.back());
                }
            }
            off[n] = off[(size_t)n + 1] = (int)pairs.size();
            terms = std::move(pairs);
        }
        void fill(int n, const std::vector<std::pair<int, Term>>& given)
        {
            off.assign((size_t)n + 2, 0);
            terms.resize(given.size());
            for (const auto& t : given) off[(size_t)t.first + 2]++;
            for (int m = 0; m < n; m++) off[(size_t)m + 2] += off[(size_t)m + 1];
            for (const auto& t : given) terms[(size_t)off[(size_t)t.first + 1]++] = t.second;
        }
        int size(int m) const { return off[(size_t)m + 1] - off[m]; }
        const Term* of(int m) const { return terms.data() + off[m]; }
    };
    // Interleaved gather lists (see mtp_plan.h).
    struct Ell {
        std::vector<int> level, slot, lead;                // lead: pieces behind
        std::vector<int4> group;                           // first term, depth, doubling steps, MTP_CTRL_LEAF or 0
        std::vector<Term> terms;
    };
    // Cuts the lists of one level into pieces of at most `cap` terms and lays them out in rows of sixteen lanes.
    struct Piece { int m, t0, n, rem; };
    struct Level {
        std::vector<Piece> lanes;                          // rows of sixteen, deepest first; whole groups of 64
        std::vector<int> depth, steps;                     // of each group
    };
    auto pieces_of = [](int n, int cap) { return n <= cap ? (n > 0 ? 1 : 0) : (n + cap - 1) / cap; };
    // (`placed` off: the groups' depths and doubling steps alone, all that the choice of a cut needs)
    auto pack_level = [&](const Lists& lists, const std::vector<int>& members, int cap, bool placed) {
        struct List { int m, n, np, len; };
        auto deep = [](int n) { return (n + 1) / 2 * 2; };
        // deepest pieces first, of those the lists of most pieces
        std::vector<List> given, ls(members.size());
        given.reserve(members.size());
        int most = 0;
        for (int m : members) {
            const int n = lists.size(m), np = pieces_of(n, cap);
            given.push_back({m, n, np, np > 1 ? deep((n + np - 1) / np) : n});        // pieces of equal length, of whole pairs
            most = std::max(most, np);
        }
        auto key = [&](const List& l) { return (cap - deep(l.len)) / 2 * (most + 1) + most - l.np; };
        std::vector<int> place((size_t)(cap / 2 + 1) * (most + 1) + 1, 0);
        for (const List& l : given) place[key(l) + 1]++;
        for (size_t k = 1; k < place.size(); k++) place[k] += place[k - 1];
        for (const List& l : given) ls[place[key(l)]++] = l;
        Level lv;
        std::vector<int> room;                             // free lanes of each row
        size_t from[17] = {0};                             // rows before from[n] have no room for n pieces (room only shrinks)
        auto steps_of = [](int pieces) { int k = 0; while ((1 << k) < pieces) k++; return k; };
        for (const List& l : ls) {
            if (l.np == 0) continue;
            size_t r;
            int at;
            if (l.np > 16) {                               // whole rows within a group (the last one has room left)
                const size_t need = (l.np + 15) / 16;
                while (room.size() % 4 + need > 4) room.push_back(16);
                r = room.size();
                for (size_t q = 0; q < need; q++) room.push_back(0);
                room.back() = (int)need * 16 - l.np;
                at = 0;
            } else {
                r = from[l.np];
                while (r < room.size() && room[r] < l.np) r++;
                from[l.np] = r;
                if (r == room.size()) room.push_back(16);
                at = 16 - room[r];
                room[r] -= l.np;
            }
            if (lv.depth.size() <= r / 4) { lv.depth.resize(r / 4 + 1, 0); lv.steps.resize(r / 4 + 1, 0); }
            lv.depth[r / 4] = std::max(lv.depth[r / 4], deep(l.len));
            lv.steps[r / 4] = std::max(lv.steps[r / 4], steps_of(l.np));
            if (!placed) continue;
            if (lv.lanes.size() < room.size() * 16) lv.lanes.resize(room.size() * 16, Piece{-1, 0, 0, 0});
            for (int q = 0; q < l.np; q++)
                lv.lanes[r * 16 + at + q] = {l.m, q * l.len, std::min(l.len, l.n - q * l.len), l.np - 1 - q};
        }
        while (lv.lanes.size() % 64) lv.lanes.push_back({-1, 0, 0, 0});
        return lv;
    };
    // what a wavefront issues: a step of four terms about twenty instructions, a group about 25, a doubling step about nine; the workgroup
    // waits for its slowest wavefront, and the others' share is what other workgroups can use meanwhile
    auto level_cost = [](const Level& lv, int waves) {
        std::vector<double> load(waves, 0.0);
        double all = 0;
        for (size_t g = 0; g < lv.depth.size(); g++) {
            const double c = 20.0 * ((lv.depth[g] + 3) / 4) + 25.0 + 9.0 * lv.steps[g];
            *std::min_element(load.begin(), load.end()) += c;
            all += c;
        }
        return *std::max_element(load.begin(), load.end()) + all / waves;
    };
    // A level as a workgroup of one wavefront and one of four walk it best.
    struct Best { Level lv[2]; };
    bool too_long = false;
    auto best_level = [&](const Lists& lists, const std::vector<int>& members) {
        std::vector<int> ms;
        int longest = 0;
        for (int m : members) {
            ms.push_back(m);
            longest = std::max(longest, lists.size(m));
        }
        double cost[2] = {-1, -1};
        int cut[2] = {MTP_SLOT_CAP, MTP_SLOT_CAP};
        long long pieces = -1;
        if (lists.longest > 64 * MTP_SLOT_CAP) { too_long = true; return Best(); }
        // (whole steps: between them a cut makes more pieces and no fewer steps; the longest lists hold more in pairs than as they
        // were given)
        for (int cap = MTP_DEPTH_STEP; cap <= MTP_SLOT_CAP || cost[0] < 0; cap += MTP_DEPTH_STEP) {
            if (longest > 64 * cap) continue;
            long long np = 0;
            for (int m : ms) np += pieces_of(lists.size(m), cap);
            if (np == pieces) continue;                    // (as many pieces of every list: the same layout)
            pieces = np;
            const Level lv = pack_level(lists, ms, cap, false);
            for (int i = 0; i < 2; i++) {
                const double c = level_cost(lv, i ? 4 : 1);
                if (cost[i] < 0 || c < cost[i]) { cut[i] = cap; cost[i] = c; }
            }
        }
        Best best;
        for (int i = 0; i < 2; i++) best.lv[i] = i && cut[1] == cut[0] ? best.lv[0] : pack_level(lists, ms, cut[i], true);
        return best;
    };
    auto best_levels = [&](const Lists& lists, const std::vector<std::vector<int>>& by_level) {
        std::vector<Best> out;
        for (const auto& members : by_level) out.push_back(best_level(lists, members));
        return out;
    };
    // (`leaves`: lists of another kind that go with the first level to be walked, the last of them)
    auto build_ell = [](const Lists& lists, const std::vector<Best>& levels, int wide,
                        const Lists* leaf_lists = nullptr, const Best* leaves = nullptr) {
        Ell e;
        size_t terms = 0, lanes = 0;
        auto count = [&](const Level& lv) { for (int d : lv.depth) { terms += (size_t)d * 64; lanes += 64; } };
        for (const Best& b : levels) count(b.lv[wide]);
        if (leaves) count(leaves->lv[wide]);
        e.terms.reserve(terms);
        e.slot.reserve(lanes);
        e.lead.reserve(lanes);
        auto append = [&](const Lists& lists, const Level& best, int kind) {
            for (size_t g = 0; g < best.depth.size(); g++) {
                e.group.push_back(make_int4((int)e.terms.size(), best.depth[g], best.steps[g], kind));
                e.terms.resize(e.terms.size() + (size_t)best.depth[g] * 64, Term{0, 0.0});
                for (size_t q = 0; q < 64; q++) {
                    const Piece& pc = best.lanes[g * 64 + q];
                    for (int k = 0; k < pc.n; k++)
                        e.terms[e.group.back().x + (size_t)k * 64 + q] = lists.of(pc.m)[pc.t0 + k];
                    e.slot.push_back(pc.n > 0 && pc.t0 == 0 ? pc.m : -1);      // the first piece of a list names the moment
                    e.lead.push_back(pc.rem);
                }
            }
        };
        for (size_t l = 0; l < levels.size(); l++) {
            e.level.push_back((int)e.slot.size());
            append(lists, levels[l].lv[wide], 0);
            if (leaves && l + 1 == levels.size()) append(*leaf_lists, leaves->lv[wide], MTP_CTRL_LEAF);
        }
        e.level.push_back((int)e.slot.size());
        return e;
    };
    struct Stream {
        std::vector<int4> head;
        std::vector<int> ctrl;
        std::vector<int4> words;
    };
    auto build_stream = [](const Ell& e, bool up, int waves) {
        Stream st;
        const int levels = (int)e.level.size() - 1;
        std::vector<std::vector<std::pair<int, int>>> seq(waves);        // (step of the level order, group) of each wavefront
        for (int q = 0; q < levels; q++) {
            const int l = up ? q : levels - 1 - q;
            std::vector<int> load(waves, 0);
            for (int g = e.level[l] / 64; g < e.level[l + 1] / 64; g++) {
                const int w = (int)(std::min_element(load.begin(), load.end()) - load.begin());
                load[w] += e.group[g].y + 4;
                seq[w].push_back({q, g});
            }
        }
        size_t steps = 2;
        for (const int4& info : e.group) steps += (info.y + MTP_DEPTH_STEP - 1) / MTP_DEPTH_STEP;
        st.words.reserve(steps * MTP_STEP_WORDS);
        st.ctrl.reserve(steps + 64);
        for (int w = 0; w < waves; w++) {
            const int first = (int)st.ctrl.size();
            for (size_t i = 0; i < seq[w].size(); i++) {
                const int q = seq[w][i].first, g = seq[w][i].second;
                const int barriers = (i + 1 < seq[w].size() ? seq[w][i + 1].first : levels) - q;
                const int4 info = e.group[g];
                // pairs of terms, two to a step, and the slots' moments
                for (int k = 0; k < info.y; k += MTP_DEPTH_STEP) {
                    for (int t = k; t < k + MTP_DEPTH_STEP; t += 2)
                        for (int l = 0; l < 64; l++) {
                            if (t >= info.y) { st.words.push_back(make_int4(0, 0, 0, 0)); continue; }
                            const Term &u = e.terms[info.x + (size_t)t * 64 + l], &v = e.terms[info.x + (size_t)(t + 1) * 64 + l];
                            unsigned long long bits;
                            std::memcpy(&bits, &u.mult, sizeof(bits));
                            st.words.push_back(make_int4(u.x, v.x, t == k ? ((e.slot[g * 64 + l] & 0xffff) | e.lead[g * 64 + l] << 16) + 1 : 0, (int)(bits >> 32)));
                        }
                    st.ctrl.push_back(info.w | (k + MTP_DEPTH_STEP < info.y ? 0 : 1 | info.z << 1 | barriers << 4));
                }
            }
            st.head.push_back(make_int4(first, (int)st.ctrl.size() - first, 0, seq[w].empty() ? levels : seq[w][0].first));
        }
        st.words.resize(st.words.size() + 2 * MTP_STEP_WORDS, make_int4(0, 0, 0, 0));      // requested ahead
        st.ctrl.resize(st.ctrl.size() + 64, 0);
        return st;
    };
    // forward: terms per destination in file order; level l >= 1 at index l - 1
    std::vector<std::pair<int, Term>> given;
    for (int e = 0; e < n_times; e++) {
        const int* q = times + e * 4;
        given.emplace_back(q[3], Term{(q[0] * 8) | ((q[1] * 8) << 16), (double)q[2]});
    }
    const Lists fl(n_moms, given, true);
    std::vector<std::vector<int>> f_by(n_levels), r_by(n_levels);
    for (int m = n_basic; m < n_moms; m++)
        if (level[m] >= 1 && fl.size(m)) f_by[level[m] - 1].push_back(m);
    // reverse: terms per source in reverse file order
    given.clear();
    for (int e = n_times - 1; e >= 0; e--) {
        const int* q = times + e * 4;
        given.emplace_back(q[1], Term{(q[3] * 8) | ((q[0] * 8) << 16), (double)q[2]});     // adj[m1] += adj[dst] mult M[m0]
        given.emplace_back(q[0], Term{(q[3] * 8) | ((q[1] * 8) << 16), (double)q[2]});     // adj[m0] += adj[dst] mult M[m1]
    }
    const Lists rl(n_moms, given, true);
    for (int m = 0; m < n_moms; m++)
        if (level[m] < n_levels && rl.size(m)) r_by[level[m]].push_back(m);
    // Leaves: scalar moments that no product reads.  Only the read-out needs them, so that the calls whose read-out is linear
    // form them in the first step of the reverse sweep; the levels of the forward sweep that held nothing else are gone.
    std::vector<char> is_source(n_moms, 0);
    for (int e = 0; e < n_times; e++) is_source[times[e * 4]] = is_source[times[e * 4 + 1]] = 1;
    std::vector<int> leaves, mapping_leaf(mapping, mapping + n_scalar);
    for (int s = 0; s < n_scalar; s++) {
        const int m = mapping[s];
        if (m < n_basic || is_source[m] || !fl.size(m)) continue;
        mapping_leaf[s] |= 1 << 16;
        leaves.push_back(m);
    }
    std::vector<std::vector<int>> core_by = f_by;
    for (auto& l : core_by)
        l.erase(std::remove_if(l.begin(), l.end(), [&](int m) { return !is_source[m]; }), l.end());
    while (!core_by.empty() && core_by.back().empty()) core_by.pop_back();
    const std::vector<Best> f_best = best_levels(fl, f_by), r_best = best_levels(rl, r_by);
    std::vector<Best> c_best;
    for (size_t l = 0; l < core_by.size(); l++)
        c_best.push_back(core_by[l].size() == f_by[l].size() ? f_best[l] : best_level(fl, core_by[l]));
    const Best leaf_best = best_level(fl, leaves);
    A2P_REQUIRE(!too_long, A2P_ERR_INVALID,
                "mtp plan: a moment takes part in more than %d products; this level is too large", 64 * MTP_SLOT_CAP);
    // monomial rows, their polynomials and the places of the basic moments among the coefficients (mtp_plan.h)
    std::vector<int> degree((size_t)(kmax + 1) * (kmax + 1) * nmus, 0);      // highest c + 1 of (a, b, mu), 0: none
    for (int i = 0; i < n_basic; i++) {
        const int* q = basic + i * 4;
        int& l = degree[((size_t)q[1] * (kmax + 1) + q[2]) * nmus + q[0]];
        l = std::max(l, q[3] + 1);
    }
    std::vector<std::pair<int, int>> row_ab;
    auto row_size = [&](const std::pair<int, int>& r) {
        int n = 0;
        for (int m = 0; m < nmus; m++) n += degree[((size_t)r.first * (kmax + 1) + r.second) * nmus + m];
        return n;
    };
    for (int a = 0; a <= kmax; a++)
        for (int b = 0; a + b <= kmax; b++)
            if (row_size({a, b})) row_ab.push_back({a, b});
    std::stable_sort(row_ab.begin(), row_ab.end(), [&](const std::pair<int, int>& x, const std::pair<int, int>& y) {
        return row_size(x) > row_size(y);                                       // longest rows first
    });
    std::vector<int> rows, polys, poly_off((size_t)(kmax + 1) * (kmax + 1) * nmus, 0);
    int n_poly_coef = 0;
    for (const auto& r : row_ab) {
        rows.push_back(r.first | (r.second << 8) | ((int)polys.size() << 16));
        for (int m = 0; m < nmus; m++) {
            const size_t e = ((size_t)r.first * (kmax + 1) + r.second) * nmus + m;
            if (!degree[e]) continue;
            poly_off[e] = n_poly_coef;
            polys.push_back(m | (degree[e] << 4) | (n_poly_coef << 12));
            n_poly_coef += degree[e];
        }
    }
    rows.push_back((int)polys.size() << 16);
    std::vector<int> polys_mu, polys_end(nmus + 1, 0);            // by mu, for the loss gradient
    for (int m = 0; m < nmus; m++) {
        for (const auto& r : row_ab) {
            const size_t e = ((size_t)r.first * (kmax + 1) + r.second) * nmus + m;
            if (degree[e]) polys_mu.push_back(r.first | (r.second << 5) | (degree[e] << 10) | (poly_off[e] << 15));
        }
        polys_end[m + 1] = (int)polys_mu.size();
    }
    std::vector<unsigned> polys_len;                              // longest first, for the sums of the basic moments
    const bool polys_fit = n_poly_coef < (1 << 14);               // (kmax <= 24, nmus <= 8)
    for (size_t r = 0; r < row_ab.size(); r++)
        for (int q = rows[r] >> 16; q < rows[r + 1] >> 16; q++) {
            const int mu = polys[q] & 15, len = (polys[q] >> 4) & 255, beg = polys[q] >> 12;
            polys_len.push_back((unsigned)mu | (unsigned)row_ab[r].first << 3 | (unsigned)row_ab[r].second << 8 |
                                (unsigned)len << 13 | (unsigned)beg << 18);
        }
    std::stable_sort(polys_len.begin(), polys_len.end(), [](unsigned x, unsigned y) { return (x >> 13 & 31) > (y >> 13 & 31); });
    std::vector<std::vector<int>> poly_lists(n_poly_coef);
    std::vector<int> poly_src(n_poly_coef), poly_items_off((size_t)n_poly_coef + 1, 0), poly_items, poly_pos(n_basic);
    int poly_unique = 1;
    for (int i = 0; i < n_basic; i++) {
        const int* q = basic + i * 4;
        const size_t e = ((size_t)q[1] * (kmax + 1) + q[2]) * nmus + q[0];
        poly_pos[i] = poly_off[e] + degree[e] - 1 - q[3];
        poly_lists[poly_pos[i]].push_back(i);
    }
    for (int e = 0; e < n_poly_coef; e++) {
        poly_src[e] = poly_lists[e].empty() ? -1 : (poly_lists[e].size() == 1 ? poly_lists[e][0] : -2);
        poly_items_off[e] = (int)poly_items.size();
        if (poly_lists[e].size() > 1) poly_unique = 0;
        poly_items.insert(poly_items.end(), poly_lists[e].begin(), poly_lists[e].end());
    }
    poly_items_off[n_poly_coef] = (int)poly_items.size();

    // tiles of the matrix products and units of the nested polynomials (mtp_plan.h)
    std::vector<unsigned> tile_ops;
    std::vector<uint2> tile_place;
    std::vector<unsigned short> stream_src[2];
    std::vector<int> units[2];
    int ntiles = 0, half_at = 0, nshares[2] = {0, 0};
    unsigned long long mu_shares[2] = {0, 0};
    std::vector<int> mu_degree(nmus, -1);
    for (int i = 0; i < n_basic; i++) {
        const int* q = basic + i * 4;
        mu_degree[q[0]] = std::max(mu_degree[q[0]], q[1] + q[2] + q[3]);
    }
    int nunits = 0;
    for (int m = 0; m < nmus; m++) nunits += mu_degree[m] + 1;
    if (poly_unique && kmax <= MTP_NEST_MAX && nunits <= MTP_UNITS_MAX && n_basic < MTP_NO_MOMENT) {
        std::map<std::array<int, 4>, int> at;                      // (mu, a, b, c) -> basic moment
        std::map<std::pair<int, int>, int> in_row, in_col;
        for (int i = 0; i < n_basic; i++) {
            const int* q = basic + i * 4;
            at[{q[0], q[1], q[2], q[3]}] = i;
            in_row[{q[1], q[2]}]++;
            in_col[{q[0], q[3]}]++;
        }
        auto moment = [&](int mu, int a, int b, int c) {
            const auto f = at.find({mu, a, b, c});
            return f == at.end() ? MTP_NO_MOMENT : f->second;
        };
        auto by_count = [](const std::map<std::pair<int, int>, int>& of) {
            std::vector<std::pair<int, int>> v;
            for (const auto& e : of) v.push_back(e.first);
            std::stable_sort(v.begin(), v.end(), [&](const auto& x, const auto& y) { return of.at(x) > of.at(y); });
            return v;
        };
        const std::vector<std::pair<int, int>> trow = by_count(in_row), tcol = by_count(in_col);
        for (size_t c0 = 0; c0 < tcol.size(); c0 += 16)
            for (size_t r0 = 0; r0 < trow.size(); r0 += 16) {
                std::vector<uint2> place(64);
                bool any = false;
                for (int l = 0; l < 64; l++) {
                    unsigned p[4];
                    for (int v = 0; v < 4; v++) {
                        const size_t r = r0 + 4 * v + l / 16, c = c0 + l % 16;
                        p[v] = r < trow.size() && c < tcol.size() ? moment(tcol[c].first, trow[r].first, trow[r].second, tcol[c].second) : MTP_NO_MOMENT;
                        any = any || p[v] != MTP_NO_MOMENT;
                    }
                    place[l] = make_uint2(p[0] | p[1] << 16, p[2] | p[3] << 16);
                }
                if (!any) continue;
                ntiles++;
                tile_place.insert(tile_place.end(), place.begin(), place.end());
                for (int l = 0; l < 64; l++) {
                    const auto& r = trow[std::min(r0 + l % 16, trow.size() - 1)];
                    const auto& c = tcol[std::min(c0 + l % 16, tcol.size() - 1)];
                    tile_ops.push_back((unsigned)r.first | (unsigned)r.second << 5 | (unsigned)c.first << 10 | (unsigned)c.second << 13);
                }
            }
        struct Unit { int mu, c, M, cost, at[2]; };
        std::vector<Unit> list;
        std::vector<unsigned short> half[2];
        for (int m = 0; m < nmus; m++)
            for (int c = mu_degree[m]; c >= 0; c--) {
                const int M = mu_degree[m] - c;
                list.push_back({m, c, M, 5 * (M + 1) * (M + 2) / 4 + 3 * (M + 1) + 9, {(int)stream_src[0].size(), (int)half[0].size()}});
                for (int b = M; b >= 0; b--)
                    for (int a = M - b; a >= 0; a--) stream_src[0].push_back((unsigned short)moment(m, a, b, c));
                for (int b = M / 2; b >= 0; b--)
                    for (int e = M - 2 * b; e >= 0; e--) {
                        half[0].push_back((unsigned short)moment(m, b + e, b, c));
                        half[1].push_back((unsigned short)(e > 0 ? moment(m, b, b + e, c) : MTP_NO_MOMENT));
                    }
            }
        // (lanes of the two halves read a coefficient each, and often the next one too: their banks apart)
        half_at = (int)half[0].size();
        while (half_at % 32 < 4 || half_at % 32 > 28) half_at++;
        stream_src[1] = half[0];
        stream_src[1].resize(half_at, MTP_NO_MOMENT);
        stream_src[1].insert(stream_src[1].end(), half[1].begin(), half[1].end());
        for (int w = 0; w < 2; w++) {
            const int waves = w ? 4 : 1;
            // runs of units, the dearest as cheap as can be: the smallest bound that needs no more wavefronts than there are
            std::vector<int> first(1, 0);
            int total = 0, bound = 0;
            for (const Unit& u : list) { total += u.cost; bound = std::max(bound, u.cost); }
            for (bound = std::max(bound, total / waves);; bound++) {
                first.assign(1, 0);
                int sum = 0;
                for (int i = 0; i < (int)list.size(); i++) {
                    if (sum + list[i].cost > bound) { first.push_back(i); sum = 0; }
                    sum += list[i].cost;
                }
                if ((int)first.size() <= waves) break;
            }
            first.resize(waves + 1, (int)list.size());
            std::vector<int> words((size_t)waves * 64, 0);
            int share = -1;
            for (int k = 0; k < waves; k++) {
                const int i0 = first[k], i1 = first[k + 1];
                units[w].push_back(i1 - i0);
                units[w].push_back(i0 < i1 ? list[i0].at[0] | list[i0].at[1] << 16 : 0);
                for (int i = i0; i < i1; i++) {
                    if (i == i0 || list[i].mu != list[i - 1].mu) {
                        share++;
                        mu_shares[w] += 1ull << (8 * list[i].mu);
                    }
                    const int end = i + 1 == i1 || list[i + 1].mu != list[i].mu;
                    words[(size_t)k * 64 + i - i0] = list[i].M | list[i].mu << 4 | end << 7 | list[i].c << 8 | share << 13;
                }
            }
            units[w].insert(units[w].end(), words.begin(), words.end());
            nshares[w] = share + 1;
        }
    }

    // The streams that a launch can ask for: those of the widths that wide_launch gives for as many moments, and the forward one
    // of four wavefronts for the components.  (Host time of a plan with all of them and every cut laid out for each by itself
    // 1.83 ms for level 16 and 14.2 for level 20, with the streams reached alone 0.78 and 4.2, in pairs of a multiplicity 0.77 and 4.1.)
    bool reached[2] = {false, false};
    for (int q = 0; q < 8; q++) reached[wide_launch(n_moms, ntiles, q & 1, q & 2, q & 4)] = true;
    Stream fs[2], rs[2], cs[2], vs[2];
    for (int i = 0; i < 2; i++) {
        const int waves = i ? 4 : 1;
        if (reached[i] || i == 1) fs[i] = build_stream(build_ell(fl, f_best, i), true, waves);
        if (!reached[i]) continue;
        rs[i] = build_stream(build_ell(rl, r_best, i), false, waves);
        cs[i] = build_stream(build_ell(fl, c_best, i), true, waves);
        vs[i] = build_stream(build_ell(rl, r_best, i, &fl, &leaf_best), false, waves);
    }

    const bool x_polys = polys_fit && n_poly_coef == n_basic;
    // nodes (scalar moment, ancestor) and their reverse gather (mtp_plan.h), for batches of scalar moments whose node
    // adjoints fit MTP_NODE_CAP entries of LDS
    struct XHost {
        std::vector<int> root, seed, brem, bsteps, bbase, bdepth, bwords;
        Stream stream;
        int nodes = 0;
    };
    std::vector<XHost> xhosts;
    if (n_basic < 64 * MTP_SLOT_CAP) {
        std::vector<std::vector<int>> terms_of(n_moms);
        for (int e = 0; e < n_times; e++) terms_of[times[e * 4 + 3]].push_back(e);
        std::vector<int> node_of(n_moms, -1), anc, stack, terms;
        auto ancestors = [&](int s, int first_node) {          // fills anc and node_of; returns the number of nodes
            anc.clear();
            stack.assign(1, mapping[s]);
            int nd = first_node;
            while (!stack.empty()) {
                const int m = stack.back();
                stack.pop_back();
                if (node_of[m] >= 0) continue;
                node_of[m] = nd++;
                anc.push_back(m);
                for (int e : terms_of[m]) { stack.push_back(times[e * 4]); stack.push_back(times[e * 4 + 1]); }
            }
            return nd - first_node;
        };
        // batches: scalar moments in table order, as many as fit
        std::vector<std::vector<int>> batches(1);
        int in_batch = 0;
        bool fits = true;
        for (int s = 0; s < n_scalar; s++) {
            const int cnt = ancestors(s, 0);
            for (int m : anc) node_of[m] = -1;
            if (cnt > MTP_NODE_CAP) fits = false;
            if (in_batch + cnt > MTP_NODE_CAP) { batches.emplace_back(); in_batch = 0; }
            batches.back().push_back(s);
            in_batch += cnt;
        }
        if (!fits) batches.clear();
        for (const auto& seeds : batches) {
            xhosts.emplace_back();
            XHost& h = xhosts.back();
            h.root.assign(n_scalar, -1);
            std::vector<std::pair<int, Term>> given, words;
            std::vector<std::pair<int, int>> by_level;
            for (int s : seeds) {
                const int cnt = ancestors(s, h.nodes);
                h.nodes += cnt;
                h.root[s] = node_of[mapping[s]];
                terms.clear();
                for (int m : anc) terms.insert(terms.end(), terms_of[m].begin(), terms_of[m].end());
                std::sort(terms.begin(), terms.end(), std::greater<int>());       // reverse file order, as in the reverse gather above
                for (int e : terms) {
                    const int* q = times + e * 4;
                    const int nd = node_of[q[3]];
                    given.emplace_back(node_of[q[1]], Term{(nd * 8) | ((q[0] * 8) << 16), (double)q[2]});
                    given.emplace_back(node_of[q[0]], Term{(nd * 8) | ((q[1] * 8) << 16), (double)q[2]});
                }
                bool any = false;
                for (int m : anc) {
                    if (level[m] < n_levels) by_level.emplace_back(level[m], node_of[m]);
                    if (m >= n_basic) continue;
                    words.emplace_back(s, Term{node_of[m] | (x_polys ? poly_pos[m] : m) << 16, 0.0});
                    any = true;
                }
                if (!any) words.emplace_back(s, Term{-1, 0.0});           // (a column of zeros)
                for (int m : anc) node_of[m] = -1;
            }
            const Lists xl(h.nodes, given, true);
            std::vector<std::vector<int>> x_by(n_levels);
            for (const auto& q : by_level)
                if (xl.size(q.second)) x_by[q.first].push_back(q.second);
            h.stream = build_stream(build_ell(xl, best_levels(xl, x_by), 1), false, 4);
            A2P_REQUIRE(!too_long, A2P_ERR_INVALID, "mtp plan: a moment takes part in more than %d products",
                        64 * MTP_SLOT_CAP);
            // The lists of basic ancestors, cut and placed as the gathers' are.  A group costs its reads of D and some ten more for
            // what it does once per pair of neighbours (and three for a doubling step); the groups of a round are worked on at the
            // same time, fewer than four by several wavefronts each, and the reads of all of them share the LDS.  (Lists cut at
            // sixteen words: 32 words deep instead of 24 at level 16.)
            for (auto& w : words)
                if (w.second.x < 0) w.second.x = h.nodes;
            const Lists columns(n_scalar, words, false);
            Level best;
            double best_cost = 0;
            for (int cap = MTP_SLOT_CAP; cap >= 2; cap -= 2) {
                bool fits = true;
                for (int s : seeds) fits &= columns.size(s) <= 64 * cap;
                if (!fits) break;
                Level lv = pack_level(columns, seeds, cap, true);
                const size_t n = lv.depth.size();
                double cost = 0;
                for (size_t g0 = 0; g0 < n; g0 += 4) {
                    const size_t at_once = std::min<size_t>(n - g0, 4);
                    double most = 0;
                    for (size_t g = g0; g < g0 + at_once; g++) {
                        const double one = lv.depth[g] + 10 + 3 * lv.steps[g];
                        most = std::max(most, one);
                        cost += 0.25 * one;
                    }
                    cost += most / (double)(4 / std::min<size_t>(n, 4));
                }
                if (best.depth.empty() || cost < best_cost) { best = std::move(lv); best_cost = cost; }
            }
            for (size_t g = 0; g < best.depth.size(); g++) {
                const int depth = best.depth[g];
                h.bbase.push_back((int)h.bwords.size());
                h.bdepth.push_back(depth);
                h.bsteps.push_back(best.steps[g]);
                h.bwords.resize(h.bwords.size() + (size_t)depth * 64, h.nodes);       // node `nodes` (a zero), basic moment 0
                for (size_t row = g * 64; row < g * 64 + 64; row += 16) {
                    std::vector<std::vector<int>> lists(16);
                    for (size_t q = 0; q < 16; q++) {
                        const Piece& pc = best.lanes[row + q];
                        for (int k = 0; k < pc.n; k++) lists[q].push_back(columns.of(pc.m)[pc.t0 + k].x);
                        h.seed.push_back(pc.n > 0 && pc.t0 == 0 ? pc.m : -1);
                        h.brem.push_back(pc.rem);
                    }
                    spread_over_banks(lists, depth, h.nodes, &h.bwords[h.bbase.back() + (row - g * 64)], 64);
                }
            }
            if (h.bwords.empty()) h.bwords.push_back(0);
        }
    }

    // one device block
    struct Seg { const void* src; size_t bytes; size_t off; };
    std::vector<Seg> segs;
    size_t total = 0;
    auto add = [&](const void* src, size_t bytes) {
        size_t off = total;
        segs.push_back({src, bytes, off});
        total += (bytes + 15) / 16 * 16;
        return off;
    };
    std::vector<unsigned> basic_words(n_basic);
    for (int i = 0; i < n_basic; i++)
        basic_words[i] = (unsigned)basic[i * 4] | ((unsigned)basic[i * 4 + 1] << 8) | ((unsigned)basic[i * 4 + 2] << 16) |
                         ((unsigned)basic[i * 4 + 3] << 24);
    const size_t o_basic = add(basic_words.data(), sizeof(unsigned) * n_basic);
    const size_t o_map = add(mapping, sizeof(int) * n_scalar);
    struct StreamOff { size_t head, ctrl, words; };
    auto add_stream = [&](const Stream& st) {
        return StreamOff{add(st.head.data(), sizeof(int4) * st.head.size()), add(st.ctrl.data(), sizeof(int) * st.ctrl.size()),
                         add(st.words.data(), sizeof(int4) * st.words.size())};
    };
    const size_t o_leaf = add(mapping_leaf.data(), sizeof(int) * n_scalar);
    StreamOff o_f[2], o_r[2], o_c[2], o_v[2];
    for (int i = 0; i < 2; i++) {
        o_f[i] = add_stream(fs[i]);
        o_r[i] = add_stream(rs[i]);
        o_c[i] = add_stream(cs[i]);
        o_v[i] = add_stream(vs[i]);
    }
    const size_t o_rows = add(rows.data(), sizeof(int) * rows.size());
    const size_t o_poly = add(polys.data(), sizeof(int) * polys.size());
    const size_t o_pmu = add(polys_mu.data(), sizeof(int) * polys_mu.size());
    const size_t o_pend = add(polys_end.data(), sizeof(int) * polys_end.size());
    const size_t o_psrc = add(poly_src.data(), sizeof(int) * poly_src.size());
    const size_t o_poff = add(poly_items_off.data(), sizeof(int) * poly_items_off.size());
    const size_t o_pit = add(poly_items.data(), sizeof(int) * poly_items.size());
    const size_t o_ppos = add(poly_pos.data(), sizeof(int) * poly_pos.size());
    const size_t o_plen = add(polys_len.data(), sizeof(unsigned) * polys_len.size());
    const size_t o_tops = add(tile_ops.data(), sizeof(unsigned) * tile_ops.size());
    const size_t o_tplace = add(tile_place.data(), sizeof(uint2) * tile_place.size());
    size_t o_ssrc[2], o_unit[2];
    for (int i = 0; i < 2; i++) {
        o_ssrc[i] = add(stream_src[i].data(), sizeof(unsigned short) * stream_src[i].size());
        o_unit[i] = add(units[i].data(), sizeof(int) * units[i].size());
    }
    struct XOff { size_t root, seed, bbase, bdepth, bsteps, brem, bwords; StreamOff x; };
    std::vector<XOff> xoffs;
    for (const XHost& h : xhosts) {
        XOff o;
        o.root = add(h.root.data(), sizeof(int) * h.root.size());
        o.seed = add(h.seed.data(), sizeof(int) * h.seed.size());
        o.x = add_stream(h.stream);
        o.bbase = add(h.bbase.data(), sizeof(int) * h.bbase.size());
        o.bdepth = add(h.bdepth.data(), sizeof(int) * h.bdepth.size());
        o.bsteps = add(h.bsteps.data(), sizeof(int) * h.bsteps.size());
        o.brem = add(h.brem.data(), sizeof(int) * h.brem.size());
        o.bwords = add(h.bwords.data(), sizeof(int) * h.bwords.size());
        xoffs.push_back(o);
    }
    std::vector<unsigned char> host(total + 16, 0);
    for (auto& s : segs)
        if (s.bytes) std::memcpy(host.data() + s.off, s.src, s.bytes);
    MtpPlan* plan = new MtpPlan();
    A2P_HIP_CHECK(hipGetDevice(&plan->device));
    A2P_HIP_CHECK(hipMalloc(&plan->device_block, total + 16));
    A2P_HIP_CHECK(hipMemcpy(plan->device_block, host.data(), total + 16, hipMemcpyHostToDevice));
    char* base = (char*)plan->device_block;
    MtpPlanDevice& d = plan->d;
    d.n_moms = n_moms; d.n_basic = n_basic; d.n_times = n_times; d.n_scalar = n_scalar;
    d.nmus = nmus; d.kmax = kmax; d.n_levels = n_levels;
    d.basic = (const unsigned*)(base + o_basic);
    d.mapping = (const int*)(base + o_map);
    auto stream_at = [&](const StreamOff& o) {
        return MtpStream{(const int4*)(base + o.head), (const int*)(base + o.ctrl), (const int4*)(base + o.words)};
    };
    for (int i = 0; i < 2; i++) { d.fwd[i] = stream_at(o_f[i]); d.rev[i] = stream_at(o_r[i]); }
    for (int i = 0; i < 2; i++) { d.fwd_core[i] = stream_at(o_c[i]); d.rev_leaf[i] = stream_at(o_v[i]); }
    d.mapping_leaf = (const int*)(base + o_leaf);
    d.x = MtpStream{nullptr, nullptr, nullptr};
    d.nrows = (int)rows.size() - 1; d.npoly = (int)polys.size(); d.ncoef_poly = n_poly_coef;
    d.rows = (const int*)(base + o_rows); d.polys = (const int*)(base + o_poly);
    d.polys_mu = (const int*)(base + o_pmu); d.polys_end = (const int*)(base + o_pend);
    d.poly_src = (const int*)(base + o_psrc); d.poly_off = (const int*)(base + o_poff);
    d.poly_items = (const int*)(base + o_pit); d.poly_pos = (const int*)(base + o_ppos);
    d.x_polys = x_polys;
    d.polys_len = polys_fit ? (const unsigned*)(base + o_plen) : nullptr;
    d.poly_unique = poly_unique;
    d.ntiles = ntiles; d.half_at = half_at;
    d.tile_ops = (const unsigned*)(base + o_tops);
    d.tile_place = (const uint2*)(base + o_tplace);
    for (int i = 0; i < 2; i++) {
        d.nstream[i] = (int)stream_src[i].size();
        d.stream_src[i] = (const unsigned short*)(base + o_ssrc[i]);
        d.units[i] = (const int*)(base + o_unit[i]);
        d.nshares[i] = nshares[i];
        d.mu_shares[i] = mu_shares[i];
    }
    d.x_nodes = 0; d.x_slots = 0;                // set per batch by the components call (MtpPlan::xbatches)
    for (size_t i = 0; i < xhosts.size(); i++) {
        const XOff& o = xoffs[i];
        MtpXBatch xb;
        xb.nodes = xhosts[i].nodes; xb.slots = (int)xhosts[i].seed.size();
        xb.root = (const int*)(base + o.root); xb.seed = (const int*)(base + o.seed);
        xb.x = stream_at(o.x);
        xb.bbase = (const int*)(base + o.bbase); xb.bdepth = (const int*)(base + o.bdepth);
        xb.bsteps = (const int*)(base + o.bsteps); xb.brem = (const int*)(base + o.brem);
        xb.bwords = (const int*)(base + o.bwords);
        plan->xbatches.push_back(xb);
    }
    {
        std::lock_guard<std::mutex> lock(g_plan_mutex);
        g_plans.insert(plan);
    }
    *out = plan;
    return A2P_OK;
}

int plan_check(void* handle, MtpPlan** out)
{
    std::lock_guard<std::mutex> lock(g_plan_mutex);
    A2P_REQUIRE(handle && g_plans.count((MtpPlan*)handle), A2P_ERR_INVALID, "mtp: invalid plan handle");
    *out = (MtpPlan*)handle;
    return A2P_OK;
}

// The entries of a row of the neighbour table, the powers among them (general tables, components).
template <typename T>
void table_layout(MtpArgs<T>& a, bool loss)
{
    const MtpPlanDevice& p = a.p;
    a.OY = p.kmax + 1;
    a.OZ = 2 * (p.kmax + 1);
    a.OG = 3 * (p.kmax + 1);
    a.ODG = a.OG + p.nmus; a.OU = a.ODG + p.nmus; a.OW = a.OU + 4; a.OF = a.OW + 4; a.ODF = a.OF + a.K;
    a.E = a.OU + 4 + (loss ? 4 + 2 * a.K : 0);
    a.E |= 1;                         // odd stride: neighbours land in different LDS banks
    a.PE = a.E;
}

// LDS of a workgroup of the atom kernel for tables of nc rows, in entries; sets the places in `a` (AtomLds).
// General tables: moments | (loss mode: their tangents) | coefficients | region of the neighbour table | ...
template <typename T>
size_t general_lds(MtpArgs<T>& a, bool loss, int nc)
{
    const MtpPlanDevice& p = a.p;
    const int nt = 256, ncf = a.ntypes * p.nmus * a.K;
    table_layout(a, loss);
    a.at_Tg = p.n_moms;
    a.at_cf = a.at_Tg + (loss ? p.n_moms : 0);
    a.at_tab = a.at_cf + ncf;
    a.at_A = a.at_tab;
    a.at_Bm = a.at_A + p.n_moms;
    // Partial sums of the thread groups, needed only in the last pass over the neighbours, when the moments (and, in
    // loss mode, their tangents) are dead: a long enough moment vector lends them its place.  Energy / force / virial
    // kernel: they are written over the table once it has been read.
    a.at_gred = !loss ? a.at_tab : mtp_gred_in_moments(loss, p.n_moms) ? 0 : a.at_tab + nc * a.E;
    a.at_Ab = a.at_tab + mtp_table_region(nc, a.E, loss, p.n_moms, nt);
    a.at_Bb = a.at_Ab + p.ncoef_poly;
    a.at_pq = loss ? a.at_Bb + p.ncoef_poly : a.at_Ab;
    a.at_net = a.at_pq + (loss ? 2 * nc * p.nmus + nc + ncf : 0);
    const int net = a.H > 0 ? p.n_scalar + (loss ? 5 : 1) * a.H : 0;
    const bool inside = mtp_polys_in_moments(p.ncoef_poly, p.n_moms);
    a.at_polys = inside ? 0 : a.at_net + net;
    a.at_part = 0;
    a.at_scratch = a.at_net + net + (!loss && !inside ? p.ncoef_poly : 0);
    if (loss) {
        // the group sums' place: the moments and their tangents, or 1024 entries behind the table
        const int n1 = p.nmus * a.K, place = mtp_gred_in_moments(true, p.n_moms) ? 2 * p.n_moms : 1024;
        a.grad_parts = std::max(1, std::min(nt / n1, place / (a.ntypes * n1)));
    }
    return (size_t)a.at_scratch + MTP_SCRATCH;
}
// moments | (tangents) | adjoints | (mixed adjoints), with the powers of the neighbours' unit vectors in their place before and sums of
// wavefronts over those already dead | coefficients | neighbour table | ...
template <typename T>
size_t tiled_lds(MtpArgs<T>& a, bool loss, bool wide, int nc)
{
    const MtpPlanDevice& p = a.p;
    const int vec = loss ? 2 : 1, n1 = p.nmus * a.K, ncf = a.ntypes * n1, stream = std::max(p.nstream[0], p.nstream[1]);
    const int shared = wide && p.ntiles < 4 ? 4 / p.ntiles : 1;          // wavefronts to a tile (TileShare)
    a.OU = 0; a.OG = 4; a.ODG = a.OG + p.nmus; a.OW = a.ODG + p.nmus; a.OF = a.OW + 4; a.ODF = a.OF + a.K;
    a.OY = a.OZ = 0;
    a.E = (loss ? a.ODF + a.K : a.OW) | 1;
    a.PE = 3 * (p.kmax + 1) | 1;
    a.at_Tg = p.n_moms;
    a.at_A = vec * p.n_moms;
    a.at_Bm = a.at_A + p.n_moms;
    a.at_part = a.at_gred = a.at_A;
    const int sums = loss ? 2 * nc * p.nshares[wide ? 1 : 0] : wide ? 3 * 4 * nc : 0;
    const int dead = std::max(vec * p.n_moms, std::max((shared - 1) * vec * p.n_basic, sums));
    const int region = std::max(vec * p.n_moms + dead, nc * a.PE);
    if (loss) a.grad_parts = std::max(1, std::min((wide ? 256 : 64) / n1, (region - a.at_gred) / ncf));
    a.at_cf = (region + 1) & ~1;
    a.at_tab = a.at_cf + ncf;
    a.at_Ab = a.at_tab + nc * a.E;
    a.at_Bb = a.at_Ab + stream;
    a.at_pq = loss ? a.at_Bb + stream : a.at_Ab;
    a.at_net = a.at_pq + (loss ? 2 * nc * p.nmus + nc + ncf : 0);
    const int net = a.H > 0 ? p.n_scalar + (loss ? 5 : 1) * a.H : 0;
    const bool inside = stream <= p.n_moms;
    a.at_polys = inside ? 0 : a.at_net + net;
    a.at_scratch = a.at_net + net + (!loss && !inside ? stream : 0);
    return (size_t)a.at_scratch + MTP_SCRATCH;
}

template <typename T>
int fill_args(MtpArgs<T>& a, MtpPlan* plan, int K, double scaling, const T* coeffs, const T* lin,
              const T* bias, int nmus, int ntypes, const T* q_scaler, double rmax, double rmin, int B, int P,
              int U, int nghost, const int* binum, const int* bilist, const int* bnumneigh,
              const int* bfirstneigh, const T* brcs, const int* btypes, bool readout = true)
{
    A2P_REQUIRE(K >= 1 && K <= MTP_KMAX, A2P_ERR_INVALID, "mtp: chebyshev_size %d outside [1, %d]", K, MTP_KMAX);
    A2P_REQUIRE(nmus == plan->d.nmus, A2P_ERR_INVALID, "mtp: nmus %d does not match the tables (%d)", nmus,
                plan->d.nmus);
    A2P_REQUIRE(ntypes >= 1 && B >= 0 && P >= 0 && U >= 1 && nghost >= 0, A2P_ERR_INVALID, "mtp: bad shape");
    A2P_REQUIRE(rmax > rmin && rmin >= 0, A2P_ERR_INVALID, "mtp: need 0 <= rmin < rmax");
    A2P_REQUIRE(coeffs && (!readout || (bias && q_scaler)) && binum && bilist && bnumneigh && bfirstneigh && brcs &&
                    btypes, A2P_ERR_INVALID, "mtp: null input pointer");
    A2P_REQUIRE((long long)B * P * U < (1ll << 31), A2P_ERR_INVALID, "mtp: batch too large");
    a.p = plan->d;
    a.K = K; a.ntypes = ntypes; a.scaling = (T)scaling; a.rmax = (T)rmax; a.rmin = (T)rmin;
    a.inv_span = (T)1 / (a.rmax - a.rmin);
    a.coeffs = coeffs; a.lin = lin; a.bias = bias; a.q_scaler = q_scaler;
    a.B = B; a.P = P; a.U = U; a.nghost = nghost;
    a.binum = binum; a.bilist = bilist; a.bnumneigh = bnumneigh; a.bfirstneigh = bfirstneigh;
    a.brcs = brcs; a.btypes = btypes;
    a.cE = nullptr; a.dFs = nullptr; a.dVs = nullptr; a.gpart = nullptr; a.ngrad = 0;
    a.force = nullptr; a.seg_cursor = nullptr; a.seg_g = nullptr; a.seg_spare = 0; a.seg_cap = 0; a.seg_mark = 0;
    a.partial = nullptr;
    a.e_sites = nullptr; a.desc = nullptr; a.energy_only = 0; a.cE_per_atom = 0; a.no_tangent = 0; a.leaves_late = 0; a.grad_parts = 1;
    a.nn_exact = 1;
    a.row_seed = nullptr; a.pair_out = nullptr;
    a.H = 0; a.w0 = nullptr; a.w1 = nullptr; a.q_shift = nullptr;
    void* ws = nullptr;
    int rc = ws_get(WS_FLAGS, 64, &ws);
    if (rc) return rc;
    a.status = (int*)ws;
    return A2P_OK;
}

// 256 threads per atom or 64: a rule on the tables alone, so that a structure's results do not depend on the batch it is
// in (the sums over neighbours are grouped by the threads).  Kernel times in us, 64 / 256 threads, fp64, energy / force /
// virial (8,000 atoms; 250 atoms) and loss gradient (8,000; 250):
//   level 8 (18 moments)   40 / 90    13.9 / 14.9    89 / 125   24 / 29
//   level 10 (41)          43 / 94    15.2 / 15.6   118 / 129   28 / 30
//   level 12 (84)          48 / 101   16.1 / 15.9   154 / 139   32 / 30
//   level 14 (174)         56 / 106   18.7 / 16.6   219 / 175   40 / 34
//   level 16 (350)         78 / 124   24 / 17.7     243 / 188   48 / 37
//   level 18 (718)        143 / 155   34 / 20       551 / 307   77 / 43
// With a network the loss gradient has a weight per neuron and scalar moment besides (64 x 125 atoms; 2 x 60; 30 neurons):
//   level 8  160 / 160, 28 / 24 (10 neurons: 112 / 139, 23 / 21)   level 10  185 / 168, 33 / 24   level 12  240 / 184, 38 / 25
// fp32, level 12: 84 / 126, 31 / 30; 14: 108 / 138, 38 / 33; 18: 275 / 212, 77 / 41.
// Those were the kernels that went by polynomials in z; the loss gradients by tiles and nested polynomials (64 x 128 atoms; 4 x 60):
//   level 10  86 / 103, 28 / 15   level 12  93 / 105, 27 / 15   level 12 in fp32  60 / 85
bool wide_atoms(int n_moms, bool loss, bool network, bool fp64)
{
    return n_moms >= (loss ? (network ? 40 : fp64 ? 80 : 150) : 600);
}

template <typename T, bool LOSS, bool SEED = false>
int launch_atoms(const MtpArgs<T>& args, hipStream_t stream)
{
    MtpArgs<T> a = args;         // (what belongs to this launch alone is set here)
    const bool tiled = tiled_launch(a.p.ntiles, LOSS, wide_atoms(a.p.n_moms, LOSS, a.H > 0, sizeof(T) == 8));
    const bool wide = wide_launch(a.p.n_moms, a.p.ntiles, LOSS, a.H > 0, sizeof(T) == 8);
    if (a.H == 0 && !a.row_seed && !a.e_sites && !a.desc && !a.energy_only) {
        a.leaves_late = 1;
        for (int i = 0; i < 2; i++) { a.p.fwd[i] = a.p.fwd_core[i]; a.p.rev[i] = a.p.rev_leaf[i]; }
    }
    auto lds_for = [&](int nc) {
        const size_t n = (tiled ? tiled_lds<T>(a, LOSS, wide, nc) : general_lds<T>(a, LOSS, nc)) * sizeof(T);
        if (tiled) return n;
        // the packed basic-moment table and the polynomials, with the monomial rows or the run of every mu
        a.lds_basic_off = (int)((n + 15) / 16 * 16);
        return a.lds_basic_off + ((size_t)a.p.n_basic + a.p.npoly + 1 + (LOSS ? a.p.nmus : a.p.nrows)) * sizeof(unsigned);
    };
    // Rows of the neighbour table: the kernel waits on dependent LDS reads and barriers, so workgroups per CU count first, and among the
    // tables that allow as many workgroups as the registers do, or as the shortest table does (loss gradient: one of MTP_NC rows), the
    // longest is taken.
    size_t lds = 0;
    {
        // LDS is handed out in pieces of 1280 bytes on this chip
        auto per_cu = [](size_t l) { return (size_t)(160 * 1024) / ((l + 1279) / 1280 * 1280); };
        const size_t by_registers = (wide ? 1 : 4) * waves_of(sizeof(T) == 8, LOSS, wide ? 256 : 64);
        const size_t want = std::min(by_registers, std::max<size_t>(1, per_cu(lds_for(LOSS ? MTP_NC : MTP_NC_MIN))));
        for (int nc : {MTP_NC_MAX, 40, MTP_NC, 24, 20, MTP_NC_MIN}) {
            lds = lds_for(nc);
            a.nc_cap = nc;
            if (per_cu(lds) >= want) break;
        }
    }
    A2P_REQUIRE(lds <= 160 * 1024, A2P_ERR_INVALID,
                "mtp: %d moments need %zu bytes of LDS per atom; this level is too large", a.p.n_moms, lds);
    auto kern = mtp_atom_kernel<T, LOSS, 256, SEED, false, 0>;
    if constexpr (!SEED)
        if (a.H > 0) kern = mtp_atom_kernel<T, LOSS, 256, false, true, 0>;
    if (tiled) {
        // (as many tiles to a wavefront as the tables take)
        const bool two = a.p.ntiles > (wide ? 4 : 1);
        auto pick = [&](auto net) {
            constexpr bool N = decltype(net)::value;
            auto narrow = mtp_atom_kernel<T, LOSS, 64, SEED, N, 1>;
            if constexpr (!LOSS)
                if (two) narrow = mtp_atom_kernel<T, LOSS, 64, SEED, N, 2>;
            return !wide ? narrow : two ? mtp_atom_kernel<T, LOSS, 256, SEED, N, 2> : mtp_atom_kernel<T, LOSS, 256, SEED, N, 1>;
        };
        kern = pick(std::false_type());
        if constexpr (!SEED)
            if (a.H > 0) kern = pick(std::true_type());
    }
    if (lds > 48 * 1024)
        A2P_HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                          (int)lds));
    prof_begin(LOSS ? "mtp_loss_bwd_kernel" : "mtp_efv_kernel", stream);
    hipLaunchKernelGGL(kern, dim3(a.P, a.B), dim3(wide ? 256 : 64), lds, stream, a);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

// network of the neural-network MTP: w0[ntypes, H, n_scalar], w1[ntypes, H], q_shift[n_scalar]
template <typename T>
struct MtpNet {
    int H;
    const T *w0, *w1, *q_shift;
};

template <typename T>
int set_net(MtpArgs<T>& a, const MtpNet<T>* net)
{
    if (!net) {
        A2P_REQUIRE(a.lin, A2P_ERR_INVALID, "mtp: null linear_coeffs");
        return A2P_OK;
    }
    A2P_REQUIRE(net->H >= 1 && net->w0 && net->w1 && net->q_shift, A2P_ERR_INVALID,
                "nnmtp: need num_neurons >= 1 and non-null w0, w1, q_shifter");
    a.H = net->H; a.w0 = net->w0; a.w1 = net->w1; a.q_shift = net->q_shift;
    return A2P_OK;
}

template <typename T>
int mtp_efv(void* handle, int K, double scaling, const T* coeffs, const T* lin, const T* bias, int nmus,
            int ntypes, const T* q_scaler, double rmax, double rmin, int B, int P, int U, int nghost,
            const int* binum, const int* bilist, const int* bnumneigh, const int* bfirstneigh, const T* brcs,
            const int* btypes, T* etot, T* force, T* virial, hipStream_t stream,
            const MtpNet<T>* net = nullptr, T* e_sites = nullptr)
{
    MtpPlan* plan = nullptr;
    int rc = plan_check(handle, &plan);
    if (rc) return rc;
    MtpArgs<T> a;
    rc = fill_args(a, plan, K, scaling, coeffs, lin, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U, nghost,
                   binum, bilist, bnumneigh, bfirstneigh, brcs, btypes);
    if (rc) return rc;
    rc = set_net(a, net);
    if (rc) return rc;
    if (B == 0 || P == 0) return A2P_OK;
    a.e_sites = e_sites;
    void* ws = nullptr;
    rc = ws_get(WS_PARTIAL, (size_t)B * P * 10 * sizeof(double), &ws);
    if (rc) return rc;
    a.partial = (double*)ws;
    const size_t force_bytes = (size_t)B * (P + nghost) * 3 * sizeof(T);
    a.force = force;
    if (!force) {
        rc = ws_get(WS_MISC, force_bytes, &ws);
        if (rc) return rc;
        a.force = (T*)ws;
    }
    PairCsr csr;
    if (force) {       // (atoms without a row start from zero, linearMtp.h:228-230)
        rc = pair_fixed_begin<T>(&csr, B, P, U, nghost, stream, a.force);
        if (rc) return rc;
        a.seg_cursor = csr.cursor;
        a.seg_g = (T*)csr.seg_g;
        a.seg_spare = csr.n * csr.seg_cap;
        a.seg_cap = csr.seg_cap;
        a.seg_mark = csr.mark;
    } else {
        rc = fill_zero(a.force, force_bytes, stream);
        if (rc) return rc;
    }
    rc = launch_atoms<T, false>(a, stream);
    if (rc) return rc;
    if (force)       // the segment sums and the energy / virial sums share a launch
        return pair_csr_finish<T>(force, csr, stream, etot, virial, a.partial, B, P);
    return finish_energy_virial<T>(etot, virial, a.partial, B, P, stream);
}

template <typename T>
int mtp_loss(void* handle, double e_w, double f_w, double v_w, const T* e_dft, const T* f_dft, const T* v_dft,
             int K, double scaling, const T* coeffs, const T* lin, const T* bias, int nmus, int ntypes,
             const T* q_scaler, double rmax, double rmin, int B, int P, int U, const int* binum,
             const int* bilist, const int* bnumneigh, const int* bfirstneigh, const T* brcs, const int* btypes,
             T* bloss, T* rmse, T* etot, T* force, T* virial, T* dcoeffs, T* dlin, T* dbias,
             hipStream_t stream)
{
    A2P_REQUIRE(e_dft && f_dft && v_dft && bloss && etot && force && virial && lin, A2P_ERR_INVALID,
                "mtp loss: null label, parameter or output pointer");
    int rc = mtp_efv<T>(handle, K, scaling, coeffs, lin, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U, 0,
                        binum, bilist, bnumneigh, bfirstneigh, brcs, btypes, etot, force, virial, stream);
    if (rc) return rc;
    if (B == 0 || P == 0) return A2P_OK;
    rc = status_post_early(stream);      // the gradient kernel looks at the same entries of the same lists
    if (rc) return rc;
    MtpPlan* plan = nullptr;
    rc = plan_check(handle, &plan);
    if (rc) return rc;
    MtpArgs<T> a;
    rc = fill_args(a, plan, K, scaling, coeffs, lin, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U, 0,
                   binum, bilist, bnumneigh, bfirstneigh, brcs, btypes);
    if (rc) return rc;
    const int ngrad = mtp_grad_row(a, true);
    const bool want_grad = dcoeffs || dlin || dbias;
    // workspace: cE[B] | dVs[B*9] | dFs[B*P*3] | gpart[B*P*ngrad] | sq[B*3] (double)
    size_t nT = (size_t)B + (size_t)B * 9 + (size_t)B * P * 3 + (want_grad ? (size_t)B * P * ngrad : 0);
    size_t bytesT = (nT * sizeof(T) + 15) / 16 * 16;
    void* ws = nullptr;
    rc = ws_get(WS_MTP, bytesT + (size_t)B * 3 * sizeof(double), &ws);
    if (rc) return rc;
    T* cE = (T*)ws;
    T* dVs = cE + B;
    T* dFs = dVs + (size_t)B * 9;
    T* gpart = dFs + (size_t)B * P * 3;
    double* sq = (double*)((char*)ws + bytesT);
    prof_begin("mtp_loss_forward", stream);
    hipLaunchKernelGGL(losskern::loss_forward_kernel<T>, dim3(B), dim3(256), 0, stream, P, binum, bilist, (T)e_w,
                       (T)f_w, (T)v_w, etot, e_dft, force, f_dft, virial, v_dft, bloss, cE, dFs, dVs, sq, 1);
    const losskern::LossRmse<T> errors{B, binum, sq, rmse};
    if (rmse && !want_grad) hipLaunchKernelGGL(losskern::loss_rmse_kernel<T>, dim3(1), dim3(64), 0, stream, errors);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    if (!want_grad) return A2P_OK;
    a.cE = cE; a.dFs = dFs; a.dVs = dVs; a.gpart = gpart; a.ngrad = ngrad;
    rc = launch_atoms<T, true>(a, stream);
    if (rc) return rc;
    return mtp_grad_reduce<T>(a, true, dcoeffs, dlin, dbias, stream, errors);
}

// Training loss of the neural-network MTP: E/F/V, per-structure loss and the per-structure gradients
// w.r.t. coeffs, w0, w1, type_bias (nnMtpLoss.h:141-181, 216-610; nnMtpOp.cc:1641-2780).
// exact = 0 evaluates the reference's backward formulas, which leave out two contributions of the
// force and virial terms: in d/dcoeffs the dependence of the adjoint on the moments (the mixed
// sweep of the linear MTP, linearMtpLoss.h:417-434, and the tanh'' term), and in d/dw0[p,k] the
// k' != k part of the tangent of the pre-activation (nnMtpLoss.h:497-529, 560-585).  exact = 1 is the
// complete derivative of the loss (it agrees with finite differences; the reference's does not).
template <typename T>
int nnmtp_loss(void* handle, double e_w, double f_w, double v_w, const T* e_dft, const T* f_dft, const T* v_dft,
               int K, const MtpNet<T>& net, const T* coeffs, const T* bias, int nmus, int ntypes,
               const T* q_scaler, double rmax, double rmin, int B, int P, int U, const int* binum,
               const int* bilist, const int* bnumneigh, const int* bfirstneigh, const T* brcs, const int* btypes,
               T* bloss, T* etot, T* force, T* virial, T* dcoeffs, T* dw0, T* dw1, T* dbias, int exact,
               hipStream_t stream)
{
    A2P_REQUIRE(e_dft && f_dft && v_dft && bloss && etot && force && virial, A2P_ERR_INVALID,
                "nnmtp loss: null label or output pointer");
    int rc = mtp_efv<T>(handle, K, 1.0, coeffs, nullptr, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U, 0, binum,
                        bilist, bnumneigh, bfirstneigh, brcs, btypes, etot, force, virial, stream, &net);
    if (rc) return rc;
    if (B == 0 || P == 0) return A2P_OK;
    rc = status_post_early(stream);      // the gradient kernel looks at the same entries of the same lists
    if (rc) return rc;
    MtpPlan* plan = nullptr;
    rc = plan_check(handle, &plan);
    if (rc) return rc;
    MtpArgs<T> a;
    rc = fill_args(a, plan, K, 1.0, coeffs, (const T*)nullptr, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U, 0,
                   binum, bilist, bnumneigh, bfirstneigh, brcs, btypes);
    if (rc) return rc;
    rc = set_net(a, &net);
    if (rc) return rc;
    const int S = a.p.n_scalar, H = net.H;
    const int nblk = ntypes * nmus * K;
    const int nrow = nblk + H * S + H + 1;
    const bool want_grad = dcoeffs || dw0 || dw1 || dbias;
    // workspace: cE[B] | dVs[B*9] | dFs[B*P*3] | gpart[B*P*nrow] | sq[B*3] (double)
    size_t nT = (size_t)B + (size_t)B * 9 + (size_t)B * P * 3 + (want_grad ? (size_t)B * P * nrow : 0);
    size_t bytesT = (nT * sizeof(T) + 15) / 16 * 16;
    void* ws = nullptr;
    rc = ws_get(WS_MTP, bytesT + (size_t)B * 3 * sizeof(double), &ws);
    if (rc) return rc;
    T* cE = (T*)ws;
    T* dVs = cE + B;
    T* dFs = dVs + (size_t)B * 9;
    T* gpart = dFs + (size_t)B * P * 3;
    double* sq = (double*)((char*)ws + bytesT);
    prof_begin("mtp_loss_forward", stream);
    hipLaunchKernelGGL(losskern::loss_forward_kernel<T>, dim3(B), dim3(256), 0, stream, P, binum, bilist, (T)e_w,
                       (T)f_w, (T)v_w, etot, e_dft, force, f_dft, virial, v_dft, bloss, cE, dFs, dVs, sq, 1);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    if (!want_grad) return A2P_OK;
    a.cE = cE; a.dFs = dFs; a.dVs = dVs; a.gpart = gpart; a.ngrad = nrow;
    a.nn_exact = exact ? 1 : 0;
    rc = launch_atoms<T, true>(a, stream);
    if (rc) return rc;
    prof_begin("mtp_grad_reduce", stream);
    hipLaunchKernelGGL(nnmtp_grad_reduce_kernel<T>, dim3(ceil_div(nrow, 64), ntypes, B), dim3(64 * GRAD_RUNS), 0, stream, P, P,
                       nblk, H * S, H, ntypes, binum, bilist, btypes, gpart, dcoeffs, dw0, dw1, dbias);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

// Site energies e_sites[B, P] (row order) and / or the scalar moments desc[B, P, n_scalar].
template <typename T>
int mtp_esites(void* handle, int K, double scaling, const T* coeffs, const T* lin, const T* bias, int nmus,
               int ntypes, const T* q_scaler, double rmax, double rmin, int B, int P, int U, int nghost,
               const int* binum, const int* bilist, const int* bnumneigh, const int* bfirstneigh, const T* brcs,
               const int* btypes, T* e_sites, T* desc, hipStream_t stream, const MtpNet<T>* net = nullptr)
{
    MtpPlan* plan = nullptr;
    int rc = plan_check(handle, &plan);
    if (rc) return rc;
    A2P_REQUIRE(e_sites || desc, A2P_ERR_INVALID, "mtp e_sites: no output requested");
    MtpArgs<T> a;
    rc = fill_args(a, plan, K, scaling, coeffs, lin, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U, nghost,
                   binum, bilist, bnumneigh, bfirstneigh, brcs, btypes);
    if (rc) return rc;
    rc = set_net(a, net);
    if (rc) return rc;
    if (B == 0 || P == 0) return A2P_OK;
    a.e_sites = e_sites; a.desc = desc; a.energy_only = 1;
    return launch_atoms<T, false>(a, stream);
}

// sum over rows of gout[b, ii] * d e_sites[b, ii] / d(coeffs, linear_coeffs, type_bias), per structure:
// the loss-gradient kernel with the per-row weight in place of cE and no force / virial residuals.
template <typename T>
int mtp_esites_bwd(void* handle, int K, double scaling, const T* coeffs, const T* lin, const T* bias, int nmus,
                   int ntypes, const T* q_scaler, double rmax, double rmin, int B, int P, int U, int nghost,
                   const int* binum, const int* bilist, const int* bnumneigh, const int* bfirstneigh,
                   const T* brcs, const int* btypes, const T* gout, T* dcoeffs, T* dlin, T* dbias,
                   hipStream_t stream)
{
    MtpPlan* plan = nullptr;
    int rc = plan_check(handle, &plan);
    if (rc) return rc;
    A2P_REQUIRE(gout && lin && (dcoeffs || dlin || dbias), A2P_ERR_INVALID, "mtp e_sites backward: null pointer");
    MtpArgs<T> a;
    rc = fill_args(a, plan, K, scaling, coeffs, lin, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U, nghost,
                   binum, bilist, bnumneigh, bfirstneigh, brcs, btypes);
    if (rc) return rc;
    if (B == 0 || P == 0) return A2P_OK;
    const int ngrad = mtp_grad_row(a, true);
    // workspace: dVs[B*9] | dFs[(B*P + nghost)*3] (both zero) | gpart[B*P*ngrad]
    const size_t nzero = (size_t)B * 9 + ((size_t)B * P + nghost) * 3;
    void* ws = nullptr;
    rc = ws_get(WS_MTP, (nzero + (size_t)B * P * ngrad) * sizeof(T), &ws);
    if (rc) return rc;
    T* dVs = (T*)ws;
    T* dFs = dVs + (size_t)B * 9;
    T* gpart = (T*)ws + nzero;
    rc = fill_zero(ws, ((nzero * sizeof(T) + 3) / 4) * 4, stream);
    if (rc) return rc;
    a.cE = gout; a.cE_per_atom = 1; a.no_tangent = 1; a.dFs = dFs; a.dVs = dVs; a.gpart = gpart; a.ngrad = ngrad;
    rc = launch_atoms<T, true>(a, stream);
    if (rc) return rc;
    return mtp_grad_reduce<T>(a, true, dcoeffs, dlin, dbias, stream);
}

// Backward of the legacy basis operator (mtpBasisOp.cc:220-326; mtpBasis.h:359-394 contracts the dense derivative
// arrays that find_val_der, :107-356, filled in the forward pass): with w = grad_desc[b, ii, :] the weights of
// the row's scalar moments,  drcs[b, ii, u, :] = sum_s w_s dM_s / d rcs[b, ii, u, :]  and
// dcoeffs[b, :] = sum_ii sum_s w_s dM_s / d coeffs.  Nothing dense is kept between the passes: the moments are
// recomputed and the adjoint sweep of the E/F/V kernel (pair derivatives) and of the loss-gradient kernel
// (coefficient gradient; with zero force and virial residuals its tangent vectors vanish) starts from w.
template <typename T>
int mtp_basis_bwd(void* handle, int K, double scaling, const T* coeffs, int nmus, int ntypes, double rmax,
                  double rmin, int B, int P, int U, int nghost, const int* binum, const int* bilist,
                  const int* bnumneigh, const int* bfirstneigh, const T* brcs, const int* btypes, const T* grad_desc,
                  T* drcs, T* dcoeffs, hipStream_t stream)
{
    MtpPlan* plan = nullptr;
    int rc = plan_check(handle, &plan);
    if (rc) return rc;
    A2P_REQUIRE(grad_desc && (drcs || dcoeffs), A2P_ERR_INVALID, "mtp basis backward: null pointer");
    MtpArgs<T> a;
    rc = fill_args(a, plan, K, scaling, coeffs, (const T*)nullptr, (const T*)nullptr, nmus, ntypes, (const T*)nullptr,
                   rmax, rmin, B, P, U, nghost, binum, bilist, bnumneigh, bfirstneigh, brcs, btypes, false);
    if (rc) return rc;
    if (B == 0 || P == 0) return A2P_OK;
    a.row_seed = grad_desc;
    if (drcs) {
        rc = fill_zero(drcs, (size_t)B * P * U * 3 * sizeof(T), stream);
        if (rc) return rc;
        MtpArgs<T> e = a;
        e.pair_out = drcs;
        rc = launch_atoms<T, false, true>(e, stream);
        if (rc) return rc;
    }
    if (dcoeffs) {
        const int ngrad = mtp_grad_row(a, false);
        // workspace: dVs[B*9] | dFs[(B*P + nghost)*3] (both zero) | gpart[B*P*ngrad]
        const size_t nzero = (size_t)B * 9 + ((size_t)B * P + nghost) * 3;
        void* ws = nullptr;
        rc = ws_get(WS_MTP, (nzero + (size_t)B * P * ngrad) * sizeof(T), &ws);
        if (rc) return rc;
        T* dVs = (T*)ws;
        T* dFs = dVs + (size_t)B * 9;
        T* gpart = (T*)ws + nzero;
        rc = fill_zero(ws, ((nzero * sizeof(T) + 3) / 4) * 4, stream);
        if (rc) return rc;
        MtpArgs<T> g = a;
        g.dFs = dFs; g.dVs = dVs; g.gpart = gpart; g.ngrad = ngrad; g.no_tangent = 1;
        rc = launch_atoms<T, true>(g, stream);
        if (rc) return rc;
        rc = mtp_grad_reduce<T>(g, false, dcoeffs, (T*)nullptr, (T*)nullptr, stream);
        if (rc) return rc;
    }
    return A2P_OK;
}

// Which route a2p_mtp_lin_components_* takes: 1 = all columns in one pass over the atoms (when the plan has the node
// graph and it fits in LDS), 0 = one E/F/V pass per column.  AI2POT_MTP_COMPONENTS=passes|nodes sets the initial value,
// a2p_mtp_components_route changes it at run time.
int g_components_route = -1;
int components_route()
{
    if (g_components_route < 0) {
        const char* e = getenv("AI2POT_MTP_COMPONENTS");
        g_components_route = (e && std::string(e) == "passes") ? 0 : 1;
    }
    return g_components_route;
}

template <typename T>
int mtp_lin_components_nodes(MtpPlan* plan, MtpArgs<T>& a, int S, int n, T* ecomp, T* fcomp, T* vcomp,
                             hipStream_t stream)
{
    const int B = a.B, P = a.P, U = a.U;
    const int rows = B * P;
    // integer scratch: nnc[rows+1] | pair_off[rows+1] | spill | cnt[rows+1] | row_of1[rows] | seg[rows+1] | scan tmp
    const int ntmp = scan_tmp_ints(rows + 1);
    void* wsI = nullptr;
    int rc = ws_get(WS_CSR, ((size_t)(rows + 1) * 4 + 1 + rows + ntmp) * sizeof(int), &wsI);
    if (rc) return rc;
    int* nnc = (int*)wsI;
    int* pair_off = nnc + rows + 1;
    int* spill = pair_off + rows + 1;        // (behind the number of pairs: read back together)
    int* cnt = spill + 1;
    int* row_of1 = cnt + rows + 1;
    int* seg = row_of1 + rows;
    int* tmp = seg + rows + 1;
    // the list of the pairs that name each atom has a place of its own: it is filled before the number of pairs is known
    void* wsL = nullptr;
    rc = ws_get(WS_NBL_A, (size_t)rows * U * sizeof(int), &wsL);
    if (rc) return rc;
    int* inc = (int*)wsL;
    rc = fill_zero(spill, (size_t)(2 * rows + 2) * sizeof(int), stream);       // spill, cnt, row_of1
    if (rc) return rc;
    prof_begin("mtp_components_lists", stream);
    hipLaunchKernelGGL(comp_rows_kernel, dim3(ceil_div(rows + 1, 256)), dim3(256), 0, stream, B, P, U, a.ntypes, a.binum,
                       a.bilist, a.bnumneigh, a.btypes, nnc, row_of1, a.status);
    prof_end(stream);
    rc = exclusive_scan_i32(nnc, pair_off, rows + 1, tmp, stream);
    if (rc) return rc;
    const long long nslots = (long long)rows * U;
    prof_begin("mtp_components_lists", stream);
    hipLaunchKernelGGL(comp_incoming_kernel, dim3(ceil_div(nslots, 256)), dim3(256), 0, stream, B, P, U, (const int*)nnc,
                       a.bfirstneigh, cnt, (const int*)nullptr, U, inc, spill);
    prof_end(stream);
    int found[2] = {0, 0};                  // the first sizes the pair buffer: one read-back per call
    rc = read_back(pair_off + rows, 2, found, stream);
    if (rc) return rc;
    A2P_HIP_CHECK(hipGetLastError());
    const int npairs = std::max(found[0], 0);
    const int* in_seg = nullptr;
    if (found[1] > 0) {                     // an atom is named by more pairs than a row has room for
        rc = exclusive_scan_i32(cnt, seg, rows + 1, tmp, stream);
        if (rc) return rc;
        rc = fill_zero(cnt, (size_t)(rows + 1) * sizeof(int), stream);
        if (rc) return rc;
        rc = ws_get(WS_NBL_A, (size_t)std::max(npairs, 1) * sizeof(int), &wsL);
        if (rc) return rc;
        inc = (int*)wsL;
        hipLaunchKernelGGL(comp_incoming_kernel, dim3(ceil_div(nslots, 256)), dim3(256), 0, stream, B, P, U,
                           (const int*)nnc, a.bfirstneigh, cnt, (const int*)seg, U, inc, spill);
        A2P_HIP_CHECK(hipGetLastError());
        in_seg = seg;
    }
    // pair derivatives | row sums | scalar moments
    const size_t n_pb = (size_t)std::max(npairs, 1) * 3 * S, n_rp = (size_t)rows * 3 * S, n_desc = (size_t)rows * S;
    void* wsT = nullptr;
    rc = ws_get(WS_MTP, (n_pb + n_rp + n_desc) * sizeof(T), &wsT);
    if (rc) return rc;
    T* pb = (T*)wsT;
    T* rowpart = pb + n_pb;
    T* desc = rowpart + n_rp;
    const int nblocks = ceil_div(P, COMP_ROWS);
    void* wsP = nullptr;
    rc = ws_get(WS_MISC, (size_t)B * nblocks * 10 * n * sizeof(T), &wsP);
    if (rc) return rc;

    CompArgs<T> c;
    c.pb = pb; c.pair_off = pair_off; c.nnc = nnc; c.desc = desc; c.rowpart = rowpart;
    auto kern = mtp_components_kernel<T, 256>;
    // The pair derivatives are written once and read once: structures are taken in chunks whose derivatives fit the
    // memory-side cache (256 MB) with what is read beside them, as long as a chunk fills the chip twice.  Level 16, 64
    // structures of 128 atoms, 390 MB: kernel + sums 370 + 124 us in one piece, 391 + 83 in two, 411 + 88 in four.
    const long long pair_bytes = (long long)npairs * 3 * S * (long long)sizeof(T);
    const int parts = (int)std::min<long long>(ceil_div(pair_bytes, 200ll << 20), std::max(1, rows / 2048));
    const int per = ceil_div(B, std::max(parts, 1));
    for (int b0 = 0; b0 < B; b0 += per) {
        const int nb = std::min(per, B - b0);
        c.b0 = b0;
        for (const MtpXBatch& xb : plan->xbatches) {
            MtpPlanDevice& p = a.p;
            p.x_nodes = xb.nodes; p.x_slots = xb.slots; p.x_root = xb.root; p.x_seed = xb.seed;
            p.x = xb.x;
            p.x_bbase = xb.bbase; p.x_bdepth = xb.bdepth; p.x_bsteps = xb.bsteps; p.x_brem = xb.brem; p.x_bwords = xb.bwords;
            // LDS: moments | node adjoints | coefficients | table of nc rows | D of a batch of neighbours (or three shares' sums, 192
            // values each); then the packed basic moments.  With at most four groups of pieces the adjoints are in registers
            // when the first D is formed, and D takes their place (level 16: 36 instead of 46 KB).
            // Workgroups per CU count first, then the longest table that still allows them.
            c.batch = p.x_slots <= 128 ? 8 : 4;         // a pair of neighbours for every wavefront that shares a group
            const int d_vals = std::max(c.batch * (3 * p.n_basic + 3), 576);
            c.d_over_nodes = p.x_slots <= 4 * 64;
            c.node_region = (std::max(p.x_nodes + 1, c.d_over_nodes ? d_vals : 0) + 1) & ~1;
            auto lds_for = [&](int nc, size_t* main) {
                const size_t vals = (size_t)((p.n_moms + 1) & ~1) + c.node_region + (size_t)a.ntypes * p.nmus * a.K +
                                    (size_t)nc * a.E + (c.d_over_nodes ? 0 : d_vals + 1);
                *main = (vals * sizeof(T) + 15) / 16 * 16;
                return *main + (size_t)p.n_basic * sizeof(unsigned);
            };
            auto per_cu = [](size_t l) { return (size_t)(160 * 1024) / ((l + 1279) / 1280 * 1280); };
            size_t m = 0;
            const size_t want = std::min<size_t>(per_cu(lds_for(MTP_NC_MIN, &m)), 4);
            A2P_REQUIRE(want >= 1, A2P_ERR_INVALID, "mtp components: %d moments need %zu bytes of LDS per atom", p.n_moms,
                        lds_for(MTP_NC_MIN, &m));
            int nc_cap = MTP_NC_MIN;
            for (int nc : {MTP_NC_MAX, 40, 32, 24, 20, MTP_NC_MIN})
                if (per_cu(lds_for(nc, &m)) >= want) { nc_cap = nc; break; }
            const size_t lds = lds_for(nc_cap, &m);
            c.nc_cap = nc_cap; c.lds_basic_off = (int)m;
            if (lds > 48 * 1024)
                A2P_HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            prof_begin("mtp_components_kernel", stream);
            hipLaunchKernelGGL(kern, dim3(P, nb), dim3(256), lds, stream, CompKernelArgs<T>{a, c});
            prof_end(stream);
        }
        prof_begin("mtp_components_sums", stream);
        auto sums = n > 64 ? comp_force_kernel<T, 2> : comp_force_kernel<T, 1>;
        hipLaunchKernelGGL(sums, dim3(nb * nblocks, ceil_div(n, n > 64 ? 128 : 64)), dim3(64 * COMP_ROWS), 0, stream, S, n, P, U, U, b0, a.binum, a.bilist,
                           a.btypes, (const int*)pair_off, (const int*)row_of1, (const int*)cnt, in_seg, (const int*)inc, a.brcs, (const T*)pb,
                           (const T*)rowpart, (const T*)desc, (T*)wsP, fcomp);
        prof_end(stream);
    }
    prof_begin("mtp_components_sums", stream);
    hipLaunchKernelGGL(comp_structure_kernel<T>, dim3(B, ceil_div(n, 64), 10), dim3(64), 0, stream, n, S, nblocks, a.q_scaler,
                       (const T*)wsP, ecomp, vcomp);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

// Energy, force and virial of every linear parameter taken alone (linear_mtp_gram_and_cross.h:125-374):
// ecomp[B, n], fcomp[B, P, 3, n], vcomp[B, 9, n] with n = n_scalar + ntypes.  Column s < n_scalar is the
// E/F/V of the model with linear_coeffs = e_s and no bias (the reference obtains the same numbers by
// differentiating each scalar moment along every pair displacement); column n_scalar + t counts the
// atoms of species t in the energy and is zero in force and virial.  All columns come from one pass over the
// atoms (mtp_components_kernel); levels whose node graph is too large take one E/F/V pass per scalar moment.
template <typename T>
int mtp_lin_components(void* handle, int K, double scaling, const T* coeffs, int nmus, int ntypes,
                       const T* q_scaler, double rmax, double rmin, int B, int P, int U, const int* binum,
                       const int* bilist, const int* bnumneigh, const int* bfirstneigh, const T* brcs,
                       const int* btypes, T* ecomp, T* fcomp, T* vcomp, hipStream_t stream)
{
    MtpPlan* plan = nullptr;
    int rc = plan_check(handle, &plan);
    if (rc) return rc;
    A2P_REQUIRE(ecomp && fcomp && vcomp, A2P_ERR_INVALID, "mtp components: null output pointer");
    A2P_REQUIRE(ntypes >= 1 && B >= 0 && P >= 0, A2P_ERR_INVALID, "mtp components: bad shape");
    const int S = plan->d.n_scalar, n = S + ntypes;
    if (B == 0 || P == 0) return A2P_OK;
    if (components_route() == 1 && !plan->xbatches.empty()) {
        MtpArgs<T> a;
        rc = fill_args(a, plan, K, scaling, coeffs, (const T*)nullptr, (const T*)nullptr, nmus, ntypes, q_scaler, rmax,
                       rmin, B, P, U, 0, binum, bilist, bnumneigh, bfirstneigh, brcs, btypes, false);
        if (rc) return rc;
        A2P_REQUIRE(q_scaler, A2P_ERR_INVALID, "mtp components: null q_scaler");
        table_layout(a, false);     // (the kernel forms derivatives of each basic moment)
        return mtp_lin_components_nodes<T>(plan, a, S, n, ecomp, fcomp, vcomp, stream);
    }
    rc = fill_zero(ecomp, (size_t)B * n * sizeof(T), stream);
    if (rc) return rc;
    rc = fill_zero(fcomp, (size_t)B * P * 3 * n * sizeof(T), stream);
    if (rc) return rc;
    rc = fill_zero(vcomp, (size_t)B * 9 * n * sizeof(T), stream);
    if (rc) return rc;
    // atoms of each species per structure (the bias columns of the energy)
    void* wsC = nullptr;
    rc = ws_get(WS_PARTIAL, (size_t)B * ntypes * sizeof(int), &wsC);
    if (rc) return rc;
    int* counts = (int*)wsC;
    rc = fill_zero(counts, (size_t)B * ntypes * sizeof(int), stream);
    if (rc) return rc;
    hipLaunchKernelGGL(species_count_kernel, dim3(ceil_div(B * P, 256)), dim3(256), 0, stream, B, P, ntypes, binum, bilist,
                       btypes, counts);
    A2P_HIP_CHECK(hipGetLastError());
    // one E/F/V pass per scalar moment with a one-hot read-out
    // workspace: eye[S*S] | zero bias[ntypes] | etot[B] | force[B*P*3] | virial[B*9]
    const size_t nT = (size_t)S * S + ntypes + B + (size_t)B * P * 3 + (size_t)B * 9;
    void* ws = nullptr;
    rc = ws_get(WS_MISC, nT * sizeof(T), &ws);
    if (rc) return rc;
    T* eye = (T*)ws;
    T* zero_bias = eye + (size_t)S * S;
    T* etot = zero_bias + ntypes;
    T* force = etot + B;
    T* virial = force + (size_t)B * P * 3;
    rc = fill_zero(ws, (((size_t)S * S + ntypes) * sizeof(T) + 3) / 4 * 4, stream);
    if (rc) return rc;
    hipLaunchKernelGGL(lin_components_init_kernel<T>, dim3(ceil_div(std::max(S, B * ntypes), 256)), dim3(256), 0,
                       stream, eye, S, ecomp, B, ntypes, (const int*)counts);
    A2P_HIP_CHECK(hipGetLastError());
    for (int s = 0; s < S; s++) {
        // force / virial go to WS_MISC, which mtp_efv does not touch when a force pointer is given
        rc = mtp_efv<T>(handle, K, scaling, coeffs, eye + (size_t)s * S, zero_bias, nmus, ntypes, q_scaler, rmax, rmin,
                        B, P, U, 0, binum, bilist, bnumneigh, bfirstneigh, brcs, btypes, etot, force, virial, stream);
        if (rc) return rc;
        hipLaunchKernelGGL(column_store_kernel<T>, dim3(ceil_div(B, 256)), dim3(256), 0, stream, ecomp, etot,
                           (long long)B, n, s);
        hipLaunchKernelGGL(column_store_kernel<T>, dim3(ceil_div((long long)B * P * 3, 256)), dim3(256), 0, stream,
                           fcomp, force, (long long)B * P * 3, n, s);
        hipLaunchKernelGGL(column_store_kernel<T>, dim3(ceil_div(B * 9, 256)), dim3(256), 0, stream, vcomp, virial,
                           (long long)B * 9, n, s);
        A2P_HIP_CHECK(hipGetLastError());
    }
    return A2P_OK;
}

template <typename T>
int mtp_schmidt_orth(int ntypes, int nmus, int K, const T* coeffs, T* out, hipStream_t stream)
{
    A2P_REQUIRE(ntypes >= 1 && nmus >= 1 && K >= 1 && coeffs && out && coeffs != out, A2P_ERR_INVALID,
                "schmidt orth: bad argument");
    hipLaunchKernelGGL(schmidt_orth_kernel<T>, dim3(1), dim3(64), 0, stream, out, coeffs, ntypes * ntypes, nmus, K);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

// The same for the neural-network MTP: gradients w.r.t. coeffs, w0, w1, type_bias
// (nnMtp.h:756-990, contracted with gout as nnMtpOp.cc does after find_e_sites_backward).
template <typename T>
int nnmtp_esites_bwd(void* handle, int K, const MtpNet<T>& net, const T* coeffs, const T* bias, int nmus,
                     int ntypes, const T* q_scaler, double rmax, double rmin, int B, int P, int U, int nghost,
                     const int* binum, const int* bilist, const int* bnumneigh, const int* bfirstneigh,
                     const T* brcs, const int* btypes, const T* gout, T* dcoeffs, T* dw0, T* dw1, T* dbias,
                     hipStream_t stream)
{
    MtpPlan* plan = nullptr;
    int rc = plan_check(handle, &plan);
    if (rc) return rc;
    A2P_REQUIRE(gout && (dcoeffs || dw0 || dw1 || dbias), A2P_ERR_INVALID, "nnmtp e_sites backward: null pointer");
    MtpArgs<T> a;
    rc = fill_args(a, plan, K, 1.0, coeffs, (const T*)nullptr, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U,
                   nghost, binum, bilist, bnumneigh, bfirstneigh, brcs, btypes);
    if (rc) return rc;
    rc = set_net(a, &net);
    if (rc) return rc;
    if (B == 0 || P == 0) return A2P_OK;
    const int S = a.p.n_scalar, H = net.H;
    const int nblk = ntypes * nmus * K;
    const int nrow = nblk + H * S + H + 1;
    // workspace: dVs[B*9] | dFs[(B*P + nghost)*3] (both zero) | gpart[B*P*nrow]
    const size_t nzero = (size_t)B * 9 + ((size_t)B * P + nghost) * 3;
    void* ws = nullptr;
    rc = ws_get(WS_MTP, (nzero + (size_t)B * P * nrow) * sizeof(T), &ws);
    if (rc) return rc;
    T* dVs = (T*)ws;
    T* dFs = dVs + (size_t)B * 9;
    T* gpart = (T*)ws + nzero;
    rc = fill_zero(ws, ((nzero * sizeof(T) + 3) / 4) * 4, stream);
    if (rc) return rc;
    a.cE = gout; a.cE_per_atom = 1; a.no_tangent = 1; a.dFs = dFs; a.dVs = dVs; a.gpart = gpart; a.ngrad = nrow;
    rc = launch_atoms<T, true>(a, stream);
    if (rc) return rc;
    prof_begin("mtp_grad_reduce", stream);
    hipLaunchKernelGGL(nnmtp_grad_reduce_kernel<T>, dim3(ceil_div(nrow, 64), ntypes, B), dim3(64 * GRAD_RUNS), 0, stream, P,
                       P + nghost, nblk, H * S, H, ntypes, binum, bilist, btypes, gpart, dcoeffs, dw0, dw1, dbias);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

}  // namespace
}  // namespace a2p

extern "C" {

int a2p_mtp_plan_create(int n_moms, int n_basic, const int* basic, int n_times, const int* times,
                        int n_scalar, const int* mapping, void** plan)
{
    A2P_REQUIRE(plan, A2P_ERR_INVALID, "mtp plan: null output");
    a2p::MtpPlan* p = nullptr;
    int rc = a2p::plan_create(n_moms, n_basic, basic, n_times, times, n_scalar, mapping, &p);
    if (rc) return rc;
    *plan = p;
    return A2P_OK;
}

int a2p_mtp_components_route(int route)
{
    const int before = a2p::components_route();
    if (route == 0 || route == 1) a2p::g_components_route = route;
    return before;
}

int a2p_mtp_plan_destroy(void* handle)
{
    a2p::MtpPlan* p = nullptr;
    int rc = a2p::plan_check(handle, &p);
    if (rc) return rc;
    {
        std::lock_guard<std::mutex> lock(a2p::g_plan_mutex);
        a2p::g_plans.erase(p);
    }
    A2P_HIP_CHECK(hipFree(p->device_block));
    delete p;
    return A2P_OK;
}

#define MTP_MODEL(T) int K, double scaling, const T* coeffs, const T* lin, const T* bias, int nmus, \
    int ntypes, const T* q_scaler, double rmax, double rmin
#define MTP_MODEL_PASS K, scaling, coeffs, lin, bias, nmus, ntypes, q_scaler, rmax, rmin
#define MTP_BATCH(T) const int* binum, const int* bilist, const int* bnumneigh, const int* bfirstneigh, \
    const T* brcs, const int* btypes
#define MTP_BATCH_PASS binum, bilist, bnumneigh, bfirstneigh, brcs, btypes

int a2p_mtp_efv_f64(void* plan, MTP_MODEL(double), int B, int P, int U, int nghost, MTP_BATCH(double),
                    double* etot, double* force, double* virial, void* stream)
{
    return a2p::mtp_efv<double>(plan, MTP_MODEL_PASS, B, P, U, nghost, binum, bilist, bnumneigh, bfirstneigh,
                                brcs, btypes, etot, force, virial, (hipStream_t)stream);
}

int a2p_mtp_efv_f32(void* plan, MTP_MODEL(float), int B, int P, int U, int nghost, MTP_BATCH(float),
                    float* etot, float* force, float* virial, void* stream)
{
    return a2p::mtp_efv<float>(plan, MTP_MODEL_PASS, B, P, U, nghost, binum, bilist, bnumneigh, bfirstneigh,
                               brcs, btypes, etot, force, virial, (hipStream_t)stream);
}

int a2p_mtp_loss_f64(void* plan, double e_weight, double f_weight, double v_weight, const double* e_dft,
                     const double* f_dft, const double* v_dft, MTP_MODEL(double), int B, int P, int U,
                     MTP_BATCH(double), double* bloss, double* rmse, double* etot, double* force,
                     double* virial, double* dcoeffs, double* dlinear, double* dbias, void* stream)
{
    return a2p::mtp_loss<double>(plan, e_weight, f_weight, v_weight, e_dft, f_dft, v_dft, MTP_MODEL_PASS, B, P,
                                 U, binum, bilist, bnumneigh, bfirstneigh, brcs, btypes, bloss, rmse, etot,
                                 force, virial, dcoeffs, dlinear, dbias, (hipStream_t)stream);
}

int a2p_mtp_loss_f32(void* plan, double e_weight, double f_weight, double v_weight, const float* e_dft,
                     const float* f_dft, const float* v_dft, MTP_MODEL(float), int B, int P, int U,
                     MTP_BATCH(float), float* bloss, float* rmse, float* etot, float* force, float* virial,
                     float* dcoeffs, float* dlinear, float* dbias, void* stream)
{
    return a2p::mtp_loss<float>(plan, e_weight, f_weight, v_weight, e_dft, f_dft, v_dft, MTP_MODEL_PASS, B, P,
                                U, binum, bilist, bnumneigh, bfirstneigh, brcs, btypes, bloss, rmse, etot, force,
                                virial, dcoeffs, dlinear, dbias, (hipStream_t)stream);
}

int a2p_mtp_esites_f64(void* plan, MTP_MODEL(double), int B, int P, int U, int nghost, MTP_BATCH(double),
                       double* e_sites, double* descriptors, void* stream)
{
    return a2p::mtp_esites<double>(plan, MTP_MODEL_PASS, B, P, U, nghost, MTP_BATCH_PASS, e_sites, descriptors,
                                   (hipStream_t)stream);
}
int a2p_mtp_esites_f32(void* plan, MTP_MODEL(float), int B, int P, int U, int nghost, MTP_BATCH(float),
                       float* e_sites, float* descriptors, void* stream)
{
    return a2p::mtp_esites<float>(plan, MTP_MODEL_PASS, B, P, U, nghost, MTP_BATCH_PASS, e_sites, descriptors,
                                  (hipStream_t)stream);
}
#define NNMTP_ENTRY(T, SUFFIX)                                                                                  \
    int a2p_nnmtp_efv_##SUFFIX(void* plan, int K, int H, const T* coeffs, const T* w0, const T* w1, const T* bias, \
                               int nmus, int ntypes, const T* q_shifter, const T* q_scaler, double rmax,          \
                               double rmin, int B, int P, int U, int nghost, MTP_BATCH(T), T* etot, T* force,      \
                               T* virial, T* e_sites, void* stream)                                               \
    {                                                                                                           \
        a2p::MtpNet<T> net{H, w0, w1, q_shifter};                                                                 \
        if (!etot && !force && !virial)                                                                           \
            return a2p::mtp_esites<T>(plan, K, 1.0, coeffs, nullptr, bias, nmus, ntypes, q_scaler, rmax, rmin, B, \
                                      P, U, nghost, MTP_BATCH_PASS, e_sites, nullptr, (hipStream_t)stream, &net); \
        return a2p::mtp_efv<T>(plan, K, 1.0, coeffs, nullptr, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U,   \
                               nghost, MTP_BATCH_PASS, etot, force, virial, (hipStream_t)stream, &net, e_sites);  \
    }
NNMTP_ENTRY(double, f64)
NNMTP_ENTRY(float, f32)

#define MTP_SOLVER_ENTRIES(T, SUFFIX)                                                                            \
    int a2p_mtp_lin_components_##SUFFIX(void* plan, int K, double scaling, const T* coeffs, int nmus, int ntypes,   \
                                        const T* q_scaler, double rmax, double rmin, int B, int P, int U,           \
                                        MTP_BATCH(T), T* ecomp, T* fcomp, T* vcomp, void* stream)                   \
    {                                                                                                             \
        return a2p::mtp_lin_components<T>(plan, K, scaling, coeffs, nmus, ntypes, q_scaler, rmax, rmin, B, P, U,    \
                                          MTP_BATCH_PASS, ecomp, fcomp, vcomp, (hipStream_t)stream);                \
    }                                                                                                             \
    int a2p_mtp_schmidt_orth_##SUFFIX(int ntypes, int nmus, int K, const T* coeffs, T* orth_coeffs, void* stream)   \
    {                                                                                                             \
        return a2p::mtp_schmidt_orth<T>(ntypes, nmus, K, coeffs, orth_coeffs, (hipStream_t)stream);                 \
    }
MTP_SOLVER_ENTRIES(double, f64)
MTP_SOLVER_ENTRIES(float, f32)

#define NNMTP_ESITES_BWD_ENTRY(T, SUFFIX)                                                                         \
    int a2p_nnmtp_esites_bwd_##SUFFIX(void* plan, int K, int H, const T* coeffs, const T* w0, const T* w1,          \
                                      const T* bias, int nmus, int ntypes, const T* q_shifter, const T* q_scaler,   \
                                      double rmax, double rmin, int B, int P, int U, int nghost, MTP_BATCH(T),      \
                                      const T* grad_e_sites, T* dcoeffs, T* dw0, T* dw1, T* dbias, void* stream)    \
    {                                                                                                             \
        a2p::MtpNet<T> net{H, w0, w1, q_shifter};                                                                   \
        return a2p::nnmtp_esites_bwd<T>(plan, K, net, coeffs, bias, nmus, ntypes, q_scaler, rmax, rmin, B, P, U,    \
                                        nghost, MTP_BATCH_PASS, grad_e_sites, dcoeffs, dw0, dw1, dbias,            \
                                        (hipStream_t)stream);                                                       \
    }
NNMTP_ESITES_BWD_ENTRY(double, f64)
NNMTP_ESITES_BWD_ENTRY(float, f32)

#define NNMTP_LOSS_ENTRY(T, SUFFIX)                                                                              \
    int a2p_nnmtp_loss_##SUFFIX(void* plan, double e_w, double f_w, double v_w, const T* e_dft, const T* f_dft,    \
                                const T* v_dft, int K, int H, const T* coeffs, const T* w0, const T* w1,           \
                                const T* bias, int nmus, int ntypes, const T* q_shifter, const T* q_scaler,        \
                                double rmax, double rmin, int B, int P, int U, MTP_BATCH(T), T* bloss, T* etot,    \
                                T* force, T* virial, T* dcoeffs, T* dw0, T* dw1, T* dbias, int exact_gradient,     \
                                void* stream)                                                                      \
    {                                                                                                            \
        a2p::MtpNet<T> net{H, w0, w1, q_shifter};                                                                  \
        return a2p::nnmtp_loss<T>(plan, e_w, f_w, v_w, e_dft, f_dft, v_dft, K, net, coeffs, bias, nmus, ntypes,    \
                                  q_scaler, rmax, rmin, B, P, U, MTP_BATCH_PASS, bloss, etot, force, virial,       \
                                  dcoeffs, dw0, dw1, dbias, exact_gradient, (hipStream_t)stream);                  \
    }
NNMTP_LOSS_ENTRY(double, f64)
NNMTP_LOSS_ENTRY(float, f32)

int a2p_mtp_esites_bwd_f64(void* plan, MTP_MODEL(double), int B, int P, int U, int nghost, MTP_BATCH(double),
                           const double* grad_e_sites, double* dcoeffs, double* dlinear, double* dbias, void* stream)
{
    return a2p::mtp_esites_bwd<double>(plan, MTP_MODEL_PASS, B, P, U, nghost, MTP_BATCH_PASS, grad_e_sites, dcoeffs,
                                       dlinear, dbias, (hipStream_t)stream);
}
int a2p_mtp_esites_bwd_f32(void* plan, MTP_MODEL(float), int B, int P, int U, int nghost, MTP_BATCH(float),
                           const float* grad_e_sites, float* dcoeffs, float* dlinear, float* dbias, void* stream)
{
    return a2p::mtp_esites_bwd<float>(plan, MTP_MODEL_PASS, B, P, U, nghost, MTP_BATCH_PASS, grad_e_sites, dcoeffs,
                                      dlinear, dbias, (hipStream_t)stream);
}

int a2p_mtp_basis_bwd_f64(void* plan, int K, double scaling, const double* coeffs, int nmus, int ntypes, double rmax,
                          double rmin, int B, int P, int U, int nghost, MTP_BATCH(double), const double* grad_desc,
                          double* drcs, double* dcoeffs, void* stream)
{
    return a2p::mtp_basis_bwd<double>(plan, K, scaling, coeffs, nmus, ntypes, rmax, rmin, B, P, U, nghost,
                                      MTP_BATCH_PASS, grad_desc, drcs, dcoeffs, (hipStream_t)stream);
}

int a2p_mtp_basis_bwd_f32(void* plan, int K, double scaling, const float* coeffs, int nmus, int ntypes, double rmax,
                          double rmin, int B, int P, int U, int nghost, MTP_BATCH(float), const float* grad_desc,
                          float* drcs, float* dcoeffs, void* stream)
{
    return a2p::mtp_basis_bwd<float>(plan, K, scaling, coeffs, nmus, ntypes, rmax, rmin, B, P, U, nghost,
                                     MTP_BATCH_PASS, grad_desc, drcs, dcoeffs, (hipStream_t)stream);
}
}
