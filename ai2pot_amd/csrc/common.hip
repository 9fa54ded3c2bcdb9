// Error state, per-device workspace and small utility kernels of libai2pot_hip.so.
#include "a2p_common.h"

#include <atomic>
#include <chrono>
#include <cstdlib>
#include <mutex>
#include <string>
#include <vector>

namespace a2p {

static thread_local std::string g_err;

void set_error(const char* fmt, ...)
{
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_err = buf;
}

const char* last_error() { return g_err.c_str(); }

// ---- pinned blocks -------------------------------------------------------------------------------------
// Copies from pageable memory are staged by the runtime (90 KB took 36 us down and up to 100 us up, 9 us from pinned
// memory) and pinning costs more than a small list: blocks are pinned once and kept.  A block belongs to one call, which
// gives it back with nothing queued that reads or writes it.  The library holds at most kPinnedMost bytes, in use and idle
// together, and no block above PINNED_BLOCK.
namespace {
constexpr size_t kPinnedMost = (size_t)256 << 20, kPinnedStep = 64 << 10;
struct PinnedBlock {
    char* ptr;
    size_t bytes;
    bool idle;
};
std::mutex g_pinned_mutex;
std::vector<PinnedBlock> g_pinned_blocks;
size_t g_pinned_bytes = 0;

// frees idle blocks until `want` more bytes fit the share (all of them with want = kPinnedMost)
void pinned_trim(size_t want)
{
    for (size_t i = 0; i < g_pinned_blocks.size() && g_pinned_bytes + want > kPinnedMost;) {
        if (!g_pinned_blocks[i].idle) { i++; continue; }
        (void)hipHostFree(g_pinned_blocks[i].ptr);
        g_pinned_bytes -= g_pinned_blocks[i].bytes;
        g_pinned_blocks.erase(g_pinned_blocks.begin() + i);
    }
}
}  // namespace

void* pinned_take(size_t bytes)
{
    if (bytes > PINNED_BLOCK) return nullptr;
    std::lock_guard<std::mutex> lock(g_pinned_mutex);
    PinnedBlock* best = nullptr;
    for (PinnedBlock& b : g_pinned_blocks)
        if (b.idle && b.bytes >= bytes && b.bytes <= 2 * bytes + kPinnedStep && (!best || b.bytes < best->bytes)) best = &b;
    if (best) {
        best->idle = false;
        return best->ptr;
    }
    const size_t want = (bytes + kPinnedStep - 1) / kPinnedStep * kPinnedStep;
    if (g_pinned_bytes + want > kPinnedMost) pinned_trim(want);
    if (g_pinned_bytes + want > kPinnedMost) return nullptr;
    void* p = nullptr;
    if (hipHostMalloc(&p, want, hipHostMallocPortable) != hipSuccess || !p) {
        (void)hipGetLastError();
        return nullptr;
    }
    g_pinned_blocks.push_back({(char*)p, want, false});
    g_pinned_bytes += want;
    return p;
}

void pinned_give(void* p)
{
    if (!p) return;
    std::lock_guard<std::mutex> lock(g_pinned_mutex);
    for (PinnedBlock& b : g_pinned_blocks)
        if (b.ptr == (char*)p) { b.idle = true; return; }
}

namespace {
struct Buf {
    void* ptr = nullptr;
    size_t bytes = 0;
};
struct DeviceWs {
    Buf slot[WS_NSLOTS];
};
std::mutex g_ws_mutex;
std::vector<DeviceWs> g_ws;
unsigned long long g_ws_generation = 0;   // bumped whenever a buffer is freed or replaced
}  // namespace

int ws_get(int slot, size_t bytes, void** out)
{
    int dev = 0;
    A2P_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    if ((int)g_ws.size() <= dev) g_ws.resize(dev + 1);
    Buf& b = g_ws[dev].slot[slot];
    if (bytes > b.bytes) {
        if (b.ptr) {
            A2P_HIP_CHECK(hipFree(b.ptr));          // synchronises: no kernel still uses it
            g_ws_generation++;                      // ... but a captured graph may still name it
        }
        b.ptr = nullptr;
        b.bytes = 0;
        size_t want = bytes + bytes / 8 + 256;      // head-room so small growth does not realloc
        A2P_HIP_CHECK(hipMalloc(&b.ptr, want));
        b.bytes = want;
        if (slot == WS_FLAGS || slot == WS_NEP_CLAIMS || slot == WS_CURSORS) {
            A2P_HIP_CHECK(hipMemset(b.ptr, 0, want));
            A2P_HIP_CHECK(hipStreamSynchronize(nullptr));      // callers' streams need not wait for the null stream
        }
    }
    *out = b.ptr;
    return A2P_OK;
}

int ws_drop(int slot)
{
    int dev = 0;
    A2P_HIP_CHECK(hipGetDevice(&dev));
    A2P_HIP_CHECK(hipDeviceSynchronize());
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    if ((int)g_ws.size() <= dev) return A2P_OK;
    Buf& b = g_ws[dev].slot[slot];
    if (b.ptr) {
        A2P_HIP_CHECK(hipFree(b.ptr));
        g_ws_generation++;
    }
    b.ptr = nullptr;
    b.bytes = 0;
    return A2P_OK;
}

size_t ws_bytes()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    if ((int)g_ws.size() <= dev) return 0;
    size_t total = 0;
    for (const Buf& b : g_ws[dev].slot) total += b.bytes;
    return total;
}

int ws_release()
{
    int dev = 0;
    A2P_HIP_CHECK(hipGetDevice(&dev));
    A2P_HIP_CHECK(hipDeviceSynchronize());          // no kernel of any stream still uses the buffers
    {
        std::lock_guard<std::mutex> pinned_lock(g_pinned_mutex);
        pinned_trim(kPinnedMost);
    }
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    if ((int)g_ws.size() <= dev) return A2P_OK;
    for (Buf& b : g_ws[dev].slot) {
        if (b.ptr) A2P_HIP_CHECK(hipFree(b.ptr));
        b.ptr = nullptr;
        b.bytes = 0;
    }
    g_ws_generation++;
    return A2P_OK;
}

// ---- small results read back to the host -----------------------------------------------------
// A status word or a dozen extents: one wavefront writes them to pinned host memory and then a sequence number, and
// the host polls that number.  Bound by latency alone.  A copy to pageable memory and a stream synchronisation cost
// 23 us behind a short kernel on an MI355X, the synchronisation alone 11.5 us, this 9.6 us: the write crosses the bus
// as the kernel ends, with no completion signal, interrupt or staging buffer behind it.
namespace {
constexpr int RB_SLOTS = 64, RB_WORDS = 32;          // words per slot; word 0 is the sequence number
std::mutex g_rb_mutex;
int* g_rb_page = nullptr;                            // one pinned allocation for the process (8 KiB)
std::atomic<unsigned long long> g_rb_used{0};        // slots in use, one bit each: a call holds one while it waits
std::atomic<int> g_rb_seq{0};

__global__ void read_back_kernel(const int* __restrict__ src, int nwords, int* host, int seq)
{
    const int l = (int)threadIdx.x;
    if (l < nwords) __hip_atomic_store(host + 1 + l, src[l], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();                          // the words of all lanes (one wavefront) before the number
    if (l == 0) __hip_atomic_store(host, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace

int* read_back_take(int nwords, hipStream_t stream, ReadBack* rb)
{
    rb->src = nullptr; rb->nwords = nwords; rb->stream = stream; rb->slot = -1;
    if (nwords < 1 || nwords >= RB_WORDS) return nullptr;
    {
        std::lock_guard<std::mutex> lock(g_rb_mutex);
        if (!g_rb_page) {
            void* p = nullptr;
            if (hipHostMalloc(&p, RB_SLOTS * RB_WORDS * sizeof(int), hipHostMallocPortable) != hipSuccess) return nullptr;
            for (int i = 0; i < RB_SLOTS * RB_WORDS; i++) ((int*)p)[i] = 0;
            g_rb_page = (int*)p;
        }
    }
    for (unsigned long long used = g_rb_used.load(); ~used != 0ull;) {
        const int free_slot = __builtin_ctzll(~used);
        if (g_rb_used.compare_exchange_weak(used, used | (1ull << free_slot))) { rb->slot = free_slot; break; }
    }
    if (rb->slot < 0) return nullptr;
    int* const word = g_rb_page + rb->slot * RB_WORDS;
    do rb->seq = g_rb_seq.fetch_add(1) + 1; while (rb->seq == 0 || rb->seq == __atomic_load_n(word, __ATOMIC_RELAXED));
    return word;
}

void read_back_drop(const ReadBack& rb)
{
    if (rb.slot >= 0) g_rb_used.fetch_and(~(1ull << rb.slot));
}

int read_back_post(const void* device_src, int nwords, hipStream_t stream, ReadBack* rb)
{
    A2P_REQUIRE(nwords > 0 && nwords < RB_WORDS, A2P_ERR_INVALID, "read_back: %d words", nwords);
    int* const word = read_back_take(nwords, stream, rb);
    rb->src = device_src;
    if (!word) return A2P_OK;                        // more waiters than slots: read_back_wait copies instead
    hipLaunchKernelGGL(read_back_kernel, dim3(1), dim3(64), 0, stream, (const int*)device_src, nwords, word, rb->seq);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) g_rb_used.fetch_and(~(1ull << rb->slot));
    A2P_HIP_CHECK(err);
    return A2P_OK;
}

int read_back_wait(const ReadBack& rb, void* host_dst)
{
    if (rb.slot < 0) {
        A2P_HIP_CHECK(hipMemcpyAsync(host_dst, rb.src, (size_t)rb.nwords * sizeof(int), hipMemcpyDeviceToHost, rb.stream));
        A2P_HIP_CHECK(hipStreamSynchronize(rb.stream));
        return A2P_OK;
    }
    // polling pays while the wait is short; behind a long queue (or after a fault, when the number never arrives) the
    // runtime's own wait takes over
    int* const word = g_rb_page + rb.slot * RB_WORDS;
    hipError_t err = hipSuccess;
    const auto began = std::chrono::steady_clock::now();
    bool there = false;
    while (!(there = __atomic_load_n(word, __ATOMIC_ACQUIRE) == rb.seq)) {
        for (int i = 0; i < 16; i++) __builtin_ia32_pause();
        if (std::chrono::steady_clock::now() - began > std::chrono::milliseconds(1)) break;
    }
    if (!there) {
        err = hipStreamSynchronize(rb.stream);
        if (err == hipSuccess && __atomic_load_n(word, __ATOMIC_ACQUIRE) != rb.seq) err = hipErrorUnknown;
    }
    if (err == hipSuccess) memcpy(host_dst, word + 1, (size_t)rb.nwords * sizeof(int));
    g_rb_used.fetch_and(~(1ull << rb.slot));
    A2P_HIP_CHECK(err);
    return A2P_OK;
}

int read_back(const void* device_src, int nwords, void* host_dst, hipStream_t stream)
{
    ReadBack rb;
    const int rc = read_back_post(device_src, nwords, stream, &rb);
    return rc ? rc : read_back_wait(rb, host_dst);
}

// The status word of a call that checks its inputs in its first kernels can be on its way to the host while the rest
// of the call runs: see a2p_status_early.
namespace {
thread_local bool g_early_asked = false, g_early_posted = false;
thread_local bool g_early_own = false;     // the posted word is the call's own (early_word), not the shared status word
thread_local int g_early_known = 0;        // ... and its value, where there is no slot to wait for
thread_local ReadBack g_early;

__global__ void early_word_kernel(int* slot, int seq)
{
    if (threadIdx.x == 0) __hip_atomic_store(slot, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace

int* early_word(hipStream_t stream, bool* no_slot)
{
    *no_slot = false;
    if (!g_early_asked || g_early_posted) return nullptr;
    int* const slot = read_back_take(1, stream, &g_early);
    *no_slot = slot == nullptr;
    if (!slot) return nullptr;
    __atomic_store_n(slot + 1, 0, __ATOMIC_RELAXED);
    return slot + 1;
}

int early_word_post(hipStream_t stream)
{
    // (kernels of a stream run in order, and what the one before stored to host memory is there when it has ended)
    hipLaunchKernelGGL(early_word_kernel, dim3(1), dim3(64), 0, stream, g_rb_page + g_early.slot * RB_WORDS, g_early.seq);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) read_back_drop(g_early);
    A2P_HIP_CHECK(err);
    g_early_posted = g_early_own = true;
    return A2P_OK;
}

void early_word_known(int word)
{
    g_early_known = word;
    g_early.slot = -1;
    g_early_posted = g_early_own = true;
}

void early_word_drop() { read_back_drop(g_early); }

int early_take(hipStream_t stream, EarlyPost* post)
{
    *post = EarlyPost{nullptr, 0, nullptr};
    if (!g_early_asked || g_early_posted) return A2P_OK;
    void* flags = nullptr;
    const int rc = ws_get(WS_FLAGS, 64, &flags);
    if (rc) return rc;
    post->flags = (const int*)flags;
    post->slot = read_back_take(1, stream, &g_early);
    post->seq = g_early.seq;
    g_early.src = flags;                 // more waiters than slots: read_back_wait copies instead
    if (!post->slot) g_early_posted = true;
    return A2P_OK;
}

void early_posted(const EarlyPost& post, bool launched)
{
    if (!post.slot) return;
    if (launched) g_early_posted = true;
    else read_back_drop(g_early);
}

int status_post_early(hipStream_t stream)
{
    if (!g_early_asked || g_early_posted) return A2P_OK;
    void* flags = nullptr;
    int rc = ws_get(WS_FLAGS, 64, &flags);
    if (rc) return rc;
    rc = read_back_post(flags, 1, stream, &g_early);
    g_early_posted = rc == A2P_OK;
    return rc;
}

// ---- per-kernel timing ---------------------------------------------------------------------
namespace {
struct ProfRec {
    const char* label;
    hipEvent_t start, stop;
};
bool g_prof_on = false;
std::mutex g_prof_mutex;
std::vector<ProfRec> g_prof_recs;
thread_local hipEvent_t g_prof_pending_stop = nullptr;
std::string g_prof_select;                 // ",label,label,": only these are timed; empty: all
std::vector<hipEvent_t> g_prof_pool;       // events of reported records, reused (one device's)
int g_prof_pool_dev = -1;

bool prof_event(hipEvent_t* e)
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    if (dev != g_prof_pool_dev) {
        for (hipEvent_t old : g_prof_pool) (void)hipEventDestroy(old);
        g_prof_pool.clear();
        g_prof_pool_dev = dev;
    }
    if (!g_prof_pool.empty()) {
        *e = g_prof_pool.back();
        g_prof_pool.pop_back();
        return true;
    }
    return hipEventCreate(e) == hipSuccess;
}
}  // namespace

// The workspace is shared by every call on a device, so work of this library on two streams must not overlap.
// Every launch passes through prof_begin, which calls enter_stream: when the stream differs from the one the
// previous launch on this device used, the device is synchronised first (callers that keep to one stream never
// pay for it).  Entry points whose launches are not bracketed by prof_begin call enter_stream themselves.  A
// stream that is being captured is left alone: a capture keeps to itself, and its replays are ordered by whoever
// launches them.
namespace {
std::mutex g_stream_mutex;
std::vector<hipStream_t> g_last_stream;
std::vector<char> g_have_stream;
}  // namespace

int enter_stream(hipStream_t stream)
{
    int dev = 0;
    A2P_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_stream_mutex);
    if ((int)g_last_stream.size() <= dev) { g_last_stream.resize(dev + 1, nullptr); g_have_stream.resize(dev + 1, 0); }
    if (g_have_stream[dev] && g_last_stream[dev] == stream) return A2P_OK;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &st) != hipSuccess) { (void)hipGetLastError(); return A2P_OK; }
    if (st != hipStreamCaptureStatusNone) return A2P_OK;
    if (g_have_stream[dev]) A2P_HIP_CHECK(hipDeviceSynchronize());
    g_last_stream[dev] = stream;
    g_have_stream[dev] = 1;
    return A2P_OK;
}

void prof_begin(const char* label, hipStream_t stream)
{
    (void)enter_stream(stream);        // a failed synchronisation stays pending and fails the call's own check
    if (!g_prof_on) return;
    std::lock_guard<std::mutex> lock(g_prof_mutex);
    if (!g_prof_select.empty() && g_prof_select.find("," + std::string(label) + ",") == std::string::npos) return;
    ProfRec r{label, nullptr, nullptr};
    if (!prof_event(&r.start) || !prof_event(&r.stop)) return;
    (void)hipEventRecord(r.start, stream);
    g_prof_pending_stop = r.stop;
    g_prof_recs.push_back(r);
}

void prof_end(hipStream_t stream)
{
    if (!g_prof_on || !g_prof_pending_stop) return;
    (void)hipEventRecord(g_prof_pending_stop, stream);
    g_prof_pending_stop = nullptr;
}

__global__ void fill_zero_kernel(uint32_t* p, size_t nwords)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < nwords; i += stride) p[i] = 0u;
}

__global__ void fill_zero2_kernel(uint32_t* p, size_t nwords, uint32_t* q, size_t mwords)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t k = i; k < nwords; k += stride) p[k] = 0u;
    for (size_t k = i; k < mwords; k += stride) q[k] = 0u;
}

int fill_zero2(void* ptr, size_t bytes, void* ptr2, size_t bytes2, hipStream_t stream)
{
    if (bytes == 0) return fill_zero(ptr2, bytes2, stream);
    if (bytes2 == 0) return fill_zero(ptr, bytes, stream);
    A2P_REQUIRE(bytes % 4 == 0 && bytes2 % 4 == 0, A2P_ERR_INVALID, "fill_zero: size not a multiple of 4");
    const size_t nwords = bytes / 4, mwords = bytes2 / 4;
    const int blocks = (int)std::min<size_t>((std::max(nwords, mwords) + 255) / 256, 256 * 32);
    prof_begin("fill_zero", stream);
    hipLaunchKernelGGL(fill_zero2_kernel, dim3(blocks), dim3(256), 0, stream, (uint32_t*)ptr, nwords,
                       (uint32_t*)ptr2, mwords);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

int fill_zero(void* ptr, size_t bytes, hipStream_t stream)
{
    if (bytes == 0) return A2P_OK;
    A2P_REQUIRE(bytes % 4 == 0, A2P_ERR_INVALID, "fill_zero: size not a multiple of 4");
    size_t nwords = bytes / 4;
    int blocks = (int)std::min<size_t>((nwords + 255) / 256, 256 * 32);
    prof_begin("fill_zero", stream);
    hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(256), 0, stream, (uint32_t*)ptr, nwords);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

// One block per (structure, component): sums the per-block partials in block order.
template <typename T>
__global__ void finish_partials_kernel(T* out, const double* partial, int nblocks, int src_stride,
                                       int out_stride)
{
    __shared__ double sh[4];
    const int b = blockIdx.y, c = blockIdx.x;
    const double* src = partial + ((size_t)b * nblocks) * src_stride + c;
    // fixed assignment of blocks to threads, fixed tree: the result does not depend on timing
    double acc = 0.0;
    for (int k = threadIdx.x; k < nblocks; k += 256) acc += src[(size_t)k * src_stride];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) out[(size_t)b * out_stride + c] = (T)((sh[0] + sh[1]) + (sh[2] + sh[3]));
}

template <typename T>
int finish_partials(T* out, const double* partial, int B, int nblocks, int ncomp, int src_stride,
                    int out_stride, hipStream_t stream, bool timed)
{
    if (timed) prof_begin("finish_partials", stream);
    hipLaunchKernelGGL(finish_partials_kernel<T>, dim3(ncomp, B), dim3(256), 0, stream, out, partial,
                       nblocks, src_stride, out_stride);
    if (timed) prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}
// Energy (component 0) and virial (components 1-9) of ev_partial's array in one launch; either output
// may be null.  Same summation per component as finish_partials.
template <typename T>
__global__ void finish_ev_kernel(T* etot, T* virial, const double* partial, int nblocks)
{
    __shared__ double sh[4];
    finish_ev_body<T>(etot, virial, partial, nblocks, blockIdx.y, blockIdx.x, sh);
}

template <typename T>
int finish_energy_virial(T* etot, T* virial, const double* partial, int B, int nblocks, hipStream_t stream)
{
    if (!etot && !virial) return A2P_OK;
    prof_begin("finish_partials", stream);
    hipLaunchKernelGGL(finish_ev_kernel<T>, dim3(10, B), dim3(256), 0, stream, etot, virial, partial, nblocks);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}
template int finish_energy_virial<float>(float*, float*, const double*, int, int, hipStream_t);
template int finish_energy_virial<double>(double*, double*, const double*, int, int, hipStream_t);
template int finish_partials<float>(float*, const double*, int, int, int, int, int, hipStream_t, bool);
template int finish_partials<double>(double*, const double*, int, int, int, int, int, hipStream_t, bool);

// Weighted sums of the per-structure gradient rows.  64 elements per workgroup, the structures in four runs (one per
// wavefront) whose sums are added in run order: a batch of 64 is sixteen loads per lane, eight of them in flight, and the
// few thousand parameters of a model still make dozens of workgroups.  Bound by the launch and one trip to the L2, where
// the rows lie (1.1 MB for a NEP model and 64 structures).
constexpr int WR_PARTS = 8;
template <typename T>
struct WeightedRows {
    const T* part[WR_PARTS];
    T* out[WR_PARTS];
    long long beg[WR_PARTS + 1];       // where each part begins among the elements of all
    int nparts;
};
template <typename T>
__global__ void __launch_bounds__(256)
weighted_rows_kernel(int B, const T* __restrict__ w, const WeightedRows<T> a)
{
    __shared__ double red[4][64];
    const int lane = threadIdx.x & 63, run = threadIdx.x >> 6;
    const long long e = (long long)blockIdx.x * 64 + lane, total = a.beg[a.nparts];
    double acc = 0.0;
    T* dst = a.out[0] + e;
    if (e < total) {
        const T* src = a.part[0];
        long long beg = 0, n = a.beg[1];
#pragma unroll
        for (int p = 1; p < WR_PARTS; p++)
            if (p < a.nparts && e >= a.beg[p]) { src = a.part[p]; beg = a.beg[p]; n = a.beg[p + 1] - beg; dst = a.out[p] + (e - beg); }
        src += e - beg;
        const int len = (B + 3) / 4, b1 = min(B, (run + 1) * len);
        for (int b0 = run * len; b0 < b1; b0 += 8) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = src[(long long)min(b0 + u, b1 - 1) * n];
#pragma unroll
            for (int u = 0; u < 8; u++)
                if (b0 + u < b1) acc += (double)w[b0 + u] * (double)v[u];
        }
    }
    red[run][lane] = acc;
    __syncthreads();
    if (run == 0 && e < total) *dst = (T)(((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane]);
}

template <typename T>
int weighted_rows(int B, const T* w, int nparts, const T* const* parts, const long long* sizes, T* const* outs,
                  hipStream_t stream)
{
    A2P_REQUIRE(B >= 1 && nparts >= 1 && nparts <= WR_PARTS && w && parts && sizes && outs, A2P_ERR_INVALID,
                "weighted_rows: need a batch, 1 to %d parts and non-null pointers", WR_PARTS);
    WeightedRows<T> a;
    a.nparts = nparts;
    a.beg[0] = 0;
    for (int p = 0; p < WR_PARTS; p++) {
        const bool have = p < nparts;
        A2P_REQUIRE(!have || (parts[p] && sizes[p] >= 0 && (outs[p] || sizes[p] == 0)), A2P_ERR_INVALID, "weighted_rows: part %d", p);
        a.part[p] = have ? parts[p] : nullptr;
        a.out[p] = have ? outs[p] : nullptr;
        a.beg[p + 1] = a.beg[p] + (have ? sizes[p] : 0);
    }
    const long long total = a.beg[nparts];
    if (total == 0) return A2P_OK;
    A2P_REQUIRE(total < (1ll << 36), A2P_ERR_INVALID, "weighted_rows: too many elements");
    prof_begin("weighted_rows", stream);
    hipLaunchKernelGGL(weighted_rows_kernel<T>, dim3(ceil_div(total, 64)), dim3(256), 0, stream, B, w, a);
    prof_end(stream);
    A2P_HIP_CHECK(hipGetLastError());
    return A2P_OK;
}

// the results behind one another
template <typename T>
int weighted_rows_joined(int B, const T* w, int nparts, const T* const* parts, const long long* sizes, T* out, hipStream_t stream)
{
    A2P_REQUIRE(nparts >= 1 && nparts <= WR_PARTS && sizes && out, A2P_ERR_INVALID,
                "weighted_rows: need 1 to %d parts and non-null pointers", WR_PARTS);
    T* outs[WR_PARTS];
    for (int p = 0; p < nparts; p++) { outs[p] = out; out += std::max(sizes[p], 0ll); }
    return weighted_rows<T>(B, w, nparts, parts, sizes, outs, stream);
}

}  // namespace a2p

extern "C" {

int a2p_weighted_rows_f32(int batch, const float* w, int nparts, const float* const* parts, const long long* sizes,
                          float* out, void* stream)
{
    return a2p::weighted_rows_joined<float>(batch, w, nparts, parts, sizes, out, (hipStream_t)stream);
}

int a2p_weighted_rows_split_f32(int batch, const float* w, int nparts, const float* const* parts, const long long* sizes,
                                float* const* outs, void* stream)
{
    return a2p::weighted_rows<float>(batch, w, nparts, parts, sizes, outs, (hipStream_t)stream);
}

int a2p_weighted_rows_f64(int batch, const double* w, int nparts, const double* const* parts, const long long* sizes,
                          double* out, void* stream)
{
    return a2p::weighted_rows_joined<double>(batch, w, nparts, parts, sizes, out, (hipStream_t)stream);
}

int a2p_weighted_rows_split_f64(int batch, const double* w, int nparts, const double* const* parts, const long long* sizes,
                                double* const* outs, void* stream)
{
    return a2p::weighted_rows<double>(batch, w, nparts, parts, sizes, outs, (hipStream_t)stream);
}

const char* a2p_last_error(void) { return a2p::last_error(); }

int a2p_abi_version(void) { return 1; }

size_t a2p_workspace_bytes(void) { return a2p::ws_bytes(); }

int a2p_workspace_release(void) { return a2p::ws_release(); }

unsigned long long a2p_workspace_generation(void)
{
    std::lock_guard<std::mutex> lock(a2p::g_ws_mutex);
    return a2p::g_ws_generation;
}

void a2p_profile_enable(int on)
{
    std::lock_guard<std::mutex> lock(a2p::g_prof_mutex);
    a2p::g_prof_on = on != 0;
}

void a2p_profile_select(const char* labels)
{
    std::lock_guard<std::mutex> lock(a2p::g_prof_mutex);
    a2p::g_prof_select.clear();
    if (labels && labels[0]) a2p::g_prof_select = "," + std::string(labels) + ",";
}

int a2p_profile_report(char* buf, size_t buflen)
{
    A2P_HIP_CHECK(hipDeviceSynchronize());
    std::lock_guard<std::mutex> lock(a2p::g_prof_mutex);
    struct Acc { const char* label; double ms; long count; };
    std::vector<Acc> acc;
    for (auto& r : a2p::g_prof_recs) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, r.start, r.stop) == hipSuccess) {
            bool found = false;
            for (auto& a : acc)
                if (std::string(a.label) == r.label) { a.ms += ms; a.count++; found = true; break; }
            if (!found) acc.push_back({r.label, (double)ms, 1});
        }
        int dev = -1;
        if (hipGetDevice(&dev) == hipSuccess && dev == a2p::g_prof_pool_dev && a2p::g_prof_pool.size() < 4096) {
            a2p::g_prof_pool.push_back(r.start);
            a2p::g_prof_pool.push_back(r.stop);
        } else {
            (void)hipEventDestroy(r.start);
            (void)hipEventDestroy(r.stop);
        }
    }
    a2p::g_prof_recs.clear();
    size_t used = 0;
    if (buf && buflen) buf[0] = 0;
    for (auto& a : acc) {
        int n = snprintf(buf + used, used < buflen ? buflen - used : 0, "%s %ld %.6f\n", a.label, a.count, a.ms);
        if (n < 0 || used + (size_t)n >= buflen) break;
        used += (size_t)n;
    }
    return A2P_OK;
}

static int a2p_report_status(int host, void* flags, hipStream_t stream);

int a2p_check_status(void* stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    void* flags = nullptr;
    int rc = a2p::ws_get(a2p::WS_FLAGS, 64, &flags);
    if (rc) return rc;
    int host = 0;
    rc = a2p::read_back(flags, 1, &host, stream);
    if (rc) return rc;
    return a2p_report_status(host, flags, stream);
}

void a2p_status_early(int on)
{
    if (a2p::g_early_posted) {          // left over from a call that failed: its slot is free once the word has arrived
        int word;
        if (!a2p::g_early_own || a2p::g_early.slot >= 0) (void)a2p::read_back_wait(a2p::g_early, &word);
        a2p::g_early_posted = a2p::g_early_own = false;
    }
    a2p::g_early_asked = on != 0;
}

int a2p_check_status_early(void* stream_)
{
    if (!a2p::g_early_posted) {         // the call had no early point
        a2p::g_early_asked = false;
        return a2p_check_status(stream_);
    }
    const bool own = a2p::g_early_own;
    int host = a2p::g_early_known;
    const int rc = own && a2p::g_early.slot < 0 ? A2P_OK : a2p::read_back_wait(a2p::g_early, &host);
    a2p::g_early_asked = a2p::g_early_posted = a2p::g_early_own = false;
    if (rc) return rc;
    if (host == 0) return A2P_OK;
    if (own) {
        a2p::set_error("a neighbour count exceeds umax_num_neigh_atoms");
        return A2P_ERR_OVERFLOW;
    }
    return a2p_check_status(stream_);   // behind the whole call: the word is cleared with nothing of the call to come
}

static int a2p_report_status(int host, void* flags, hipStream_t stream)
{
    if (host == 0) return A2P_OK;
    int rc = a2p::fill_zero(flags, 64, stream);
    if (rc) return rc;
    A2P_HIP_CHECK(hipStreamSynchronize(stream));
    if (host & a2p::ST_SEG_OVERFLOW) {
        a2p::set_error("an atom is named by more pairs than its reduction segment holds (the list is not symmetric, or "
                       "ghosts collect the pairs of several rows): forces of this call are incomplete; call again after "
                       "a2p_pair_segment_capacity(a2p_pair_incoming_max(...))");
        return A2P_ERR_SEGMENT;
    }
    if (host & a2p::ST_GRID_BOUND) {
        a2p::set_error("neighbour list: the bin box around the atoms outgrew the bound taken from the last synchronised "
                       "build (or the coordinates are not finite); the lists of this build are empty: build again "
                       "after a2p_nblist_sync_free(0)");
        return A2P_ERR_GRID;
    }
    if (host & a2p::ST_NEIGH_OVERFLOW) {
        a2p::set_error("a neighbour count exceeds umax_num_neigh_atoms");
        return A2P_ERR_OVERFLOW;
    }
    a2p::set_error("device-side input check failed:%s%s",
                   (host & a2p::ST_BAD_NEIGHBOR) ? " neighbour index outside [0, natoms_pad+nghost)" : "",
                   (host & a2p::ST_BAD_TYPE) ? " type index outside [0, ntypes)" : "");
    return A2P_ERR_INPUT;
}
}
