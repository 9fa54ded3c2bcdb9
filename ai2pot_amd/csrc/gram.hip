// Normal equations of a weighted linear least-squares problem:
//     A = sum_k w_k X_k^T X_k  [n, n],     b = sum_k w_k X_k^T y_k  [n]
// for up to three tall row-major matrices X_k [N_k, n] (the energy, force and virial components of the linear parameters,
// source/descriptor/mtpr/include/linear_mtp_gram_and_cross.h:377-443).
//
// [X | y] is cut into blocks of rows; a workgroup takes a block, 32 rows at a time through LDS, and up to 24 of the 16 x 16
// tiles of the upper triangle of [X | y]^T [X | y], six per wavefront in the accumulators of the matrix instructions
// (16 x 16 x 4, the precision of X).  A second kernel adds the blocks' tiles in block order, in double, with the weights.
// Bound by the way of the rows through registers and LDS to the matrix instructions (24,640 rows, 95 columns, fp64: 21 tiles x 6,160
// instructions of 64 cycles on 1024 units, 3.4 us) and by the two launches; a batched library product per matrix with its
// concatenation, sum and scaling took 25 launches and about 100 us for the same.  Rows one pass ahead 27.8 -> 26.0 us, two blocks to
// a compute unit 19.5; the sum of the blocks 10 -> 6.4.
#include "a2p_common.h"
#include "wave_ops.h"

namespace a2p {
using namespace wave;
namespace {

constexpr int GR_ROWS = 32;                  // rows in LDS
constexpr int GR_TILES = 6;                  // tiles per wavefront
constexpr int GR_SETS = 3;

template <typename T>
struct GramArgs {
    const T *X[GR_SETS], *y[GR_SETS];
    long long rows[GR_SETS];
    double w[GR_SETS];
    int first_block[GR_SETS + 1];            // blocks of set k: [first_block[k], first_block[k + 1])
    int per_block;                           // rows of a block, a multiple of GR_ROWS
    int n, nc, stride, ntiles;               // columns of X, column tiles of [X | y], row of the LDS, tiles of the triangle
    T* part;                                 // [blocks][ntiles][256]
};

// tile t of the upper triangle of nc x nc: (i, j), i <= j, rows of the triangle in turn
__device__ __forceinline__ void tile_of(int t, int nc, int& i, int& j)
{
    i = 0;
    while (t >= nc - i) { t -= nc - i; i++; }
    j = i + t;
}

template <typename T, int AHEAD>
__global__ void __launch_bounds__(256) gram_kernel(const GramArgs<T> a)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* const tab = (T*)smem_raw;
    const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, k4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int blk = blockIdx.x, n = a.n, cols = a.nc * 16;
    int k = 0;
    while (k + 1 < GR_SETS && blk >= a.first_block[k + 1]) k++;
    const T* const X = a.X[k];
    const T* const y = a.y[k];
    const long long r0 = (long long)(blk - a.first_block[k]) * a.per_block;
    const int rows = (int)min((long long)a.per_block, a.rows[k] - r0);
    int ti[GR_TILES], tj[GR_TILES];
    typename Acc<T>::type acc[GR_TILES];
    const int t0 = (blockIdx.y * 4 + wave) * GR_TILES;
#pragma unroll
    for (int q = 0; q < GR_TILES; q++) {
        tile_of(min(t0 + q, a.ntiles - 1), a.nc, ti[q], tj[q]);
        acc[q] = {0, 0, 0, 0};
    }
    // Eight rows of a column per wavefront, all in flight (rows beyond the block and columns beyond y are zero).  Those of the
    // first AHEAD columns of a lane are on their way while the rows before them are multiplied.
    constexpr int PER = GR_ROWS / 4;
    auto fetch = [&](T (&v)[PER], int s0, int c) __attribute__((always_inline)) {
        const T* const src = c < n ? X + c : y;
        const long long step = c < n ? n : 1;
#pragma unroll
        for (int i = 0; i < PER; i++) v[i] = src[(r0 + min(s0 + wave * PER + i, rows - 1)) * step];
    };
    auto store = [&](T (&v)[PER], int s0, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int r = wave * PER + i;
            tab[r * a.stride + c] = s0 + r >= rows || c > n ? (T)0 : v[i];
        }
    };
    T ahead[AHEAD][PER];
#pragma unroll
    for (int u = 0; u < AHEAD; u++)
        if (lane + u * 64 < cols) fetch(ahead[u], 0, lane + u * 64);
    for (int s0 = 0; s0 < rows; s0 += GR_ROWS) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < AHEAD; u++)
            if (lane + u * 64 < cols) store(ahead[u], s0, lane + u * 64);
        for (int c = lane + AHEAD * 64; c < cols; c += 64) {
            T v[PER];
            fetch(v, s0, c);
            store(v, s0, c);
        }
        __syncthreads();
        if (s0 + GR_ROWS < rows)
#pragma unroll
            for (int u = 0; u < AHEAD; u++)
                if (lane + u * 64 < cols) fetch(ahead[u], s0 + GR_ROWS, lane + u * 64);
        for (int st = 0; st < GR_ROWS; st += 4) {
            const T* t = tab + (st + k4) * a.stride + c16;
#pragma unroll
            for (int q = 0; q < GR_TILES; q++)
                if (t0 + q < a.ntiles) acc[q] = mma(t[ti[q] * 16], t[tj[q] * 16], acc[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < GR_TILES; q++) {
        if (t0 + q >= a.ntiles) continue;
        T* o = a.part + ((size_t)blk * a.ntiles + t0 + q) * 256;
#pragma unroll
        for (int v = 0; v < 4; v++) o[mma_row<T>(v, lane) * 16 + c16] = acc[q][v];
    }
}

// A quarter of a tile per workgroup, GS_PARTS threads per entry, each for its share of the blocks.  Bound by its dependent loads
// while there are few tiles (sixteen threads per entry, four, and a workgroup per tile with four: 94 columns, 24,576 rows 8.7, 10.4 and
// 18.5 us; 127 columns 7.1, 7.7 and 12.0), and by the workgroups and what they write from a workgroup for every compute unit on,
// where four threads per entry suffice (164 columns, 66 tiles, 8.8, 7.4 and 10.6; 290 columns 9.2, 7.6 and 8.3; 503 columns, 3,072 rows
// 18.9, 8.7 and 11.1).
constexpr int GS_ENTRIES = 64, GS_MANY = 64;         // entries of a workgroup; tiles from which four threads per entry are taken
template <typename T, int GS_PARTS>
__global__ void __launch_bounds__(GS_PARTS * GS_ENTRIES)
gram_sum_kernel(const GramArgs<T> a, T* __restrict__ A, T* __restrict__ b)
{
    __shared__ double red[GS_PARTS][GS_ENTRIES];
    const int part = threadIdx.x / GS_ENTRIES, mine = threadIdx.x % GS_ENTRIES, e = blockIdx.y * GS_ENTRIES + mine, n = a.n;
    int ti, tj;
    tile_of(blockIdx.x, a.nc, ti, tj);
    const int blocks = a.first_block[GR_SETS], run = (blocks + GS_PARTS - 1) / GS_PARTS;
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < GR_SETS; k++) {
        const int q1 = min(a.first_block[k + 1], (part + 1) * run);
        double s = 0.0;
        for (int q0 = max(a.first_block[k], part * run); q0 < q1; q0 += 8) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = a.part[((size_t)min(q0 + u, q1 - 1) * a.ntiles + blockIdx.x) * 256 + e];
#pragma unroll
            for (int u = 0; u < 8; u++) s += q0 + u < q1 ? (double)v[u] : 0.0;
        }
        sum += a.w[k] * s;
    }
    red[part][mine] = sum;
    __syncthreads();
    if (part) return;
    sum = red[0][mine];
#pragma unroll
    for (int q = 1; q < GS_PARTS; q++) sum += red[q][mine];
    const T v = (T)sum;
    const int i = ti * 16 + (e >> 4), j = tj * 16 + (e & 15);
    if (i < n && j < n && i <= j) { A[(size_t)i * n + j] = v; A[(size_t)j * n + i] = v; }
    if (i < n && j == n) b[i] = v;
}

template <typename T>
int normal_equations(int n, const long long* rows, const double* w, const T* const* X, const T* const* y, T* A, T* b,
                     hipStream_t stream)
{
    A2P_REQUIRE(n >= 1 && rows && w && X && y && A && b, A2P_ERR_INVALID, "normal equations: bad argument");
    GramArgs<T> a;
    a.n = n;
    a.nc = ceil_div(n + 1, 16);
    a.ntiles = a.nc * (a.nc + 1) / 2;
    // an odd multiple of 16: the four rows of a matrix instruction's operand fall on all banks
    a.stride = a.nc * 16 + (a.nc & 1 ? 0 : 16);
    const size_t lds = (size_t)GR_ROWS * a.stride * sizeof(T);
    A2P_REQUIRE(n <= 575, A2P_ERR_INVALID, "normal equations: %d columns do not fit in LDS", n);
    long long total = 0;
    for (int k = 0; k < GR_SETS; k++) {
        A2P_REQUIRE(rows[k] >= 0 && (rows[k] == 0 || (X[k] && y[k])), A2P_ERR_INVALID, "normal equations: null matrix");
        total += rows[k];
    }
    // about two workgroups per compute unit over all tile groups (one: 26.0 + 4.6 us instead of 19.5 + 6.4 for 24,640 rows of 95
    // columns); never less than one pass through LDS
    const int groups = ceil_div(a.ntiles, 4 * GR_TILES);
    const long long want = std::max(32, 512 / groups);
    const long long per = std::max<long long>(GR_ROWS, (total / want + GR_ROWS - 1) / GR_ROWS * GR_ROWS);
    A2P_REQUIRE(per < (1ll << 30), A2P_ERR_INVALID, "normal equations: too many rows");
    a.per_block = (int)per;
    a.first_block[0] = 0;
    for (int k = 0; k < GR_SETS; k++) {
        a.X[k] = X[k]; a.y[k] = y[k]; a.rows[k] = rows[k]; a.w[k] = w[k];
        a.first_block[k + 1] = a.first_block[k] + (int)((rows[k] + per - 1) / per);
    }
    const int blocks = a.first_block[GR_SETS];
    void* ws = nullptr;
    int rc = ws_get(WS_MISC, (size_t)std::max(blocks, 1) * a.ntiles * 256 * sizeof(T), &ws);
    if (rc) return rc;
    a.part = (T*)ws;
    // columns of a lane that are asked for one pass ahead: two, and one beyond 256 columns, of which a lane has five or more (one and
    // two: 127 columns, 24,576 rows 32.2 and 31.7 us; 290, 120,000 rows 581 and 600; 503, 24,576 rows 618 and 634)
    auto kern = a.nc > 16 ? gram_kernel<T, 1> : gram_kernel<T, 2>;
    if (lds > 48 * 1024)
        A2P_HIP_CHECK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    prof_begin("gram", stream);
    if (blocks) hipLaunchKernelGGL(kern, dim3(blocks, groups), dim3(256), lds, stream, a);
    const int parts = a.ntiles < GS_MANY ? 16 : 4;
    auto sum = parts == 16 ? gram_sum_kernel<T, 16> : gram_sum_kernel<T, 4>;
    hipLaunchKernelGGL(sum, dim3(a.ntiles, 256 / GS_ENTRIES), dim3(parts * GS_ENTRIES), 0, stream, a, A, b);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

}  // namespace
}  // namespace a2p

extern "C" {

int a2p_normal_equations_f64(int n, const long long* rows, const double* weights, const double* const* X,
                             const double* const* y, double* A, double* b, void* stream)
{
    return a2p::normal_equations<double>(n, rows, weights, X, y, A, b, (hipStream_t)stream);
}

int a2p_normal_equations_f32(int n, const long long* rows, const double* weights, const float* const* X,
                             const float* const* y, float* A, float* b, void* stream)
{
    return a2p::normal_equations<float>(n, rows, weights, X, y, A, b, (hipStream_t)stream);
}
}
