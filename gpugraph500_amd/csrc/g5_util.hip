// g5_util.hip -- library plumbing and device-wide primitives: error state,
// device memory helpers, exclusive scan, bitmap <-> sorted queue.
#include <cstdarg>
#include <cstring>
#include <mutex>

#include "g5_internal.hpp"

namespace g5 {

static thread_local char g_err[512] = "";

void set_error(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int fail_hip(hipError_t e, const char *what, const char *file, int line)
{
    set_error("%s failed: %s (%s:%d)", what, hipGetErrorString(e), file, line);
    (void)hipGetLastError();  // reported here, not by the next call's look after a launch
    return e == hipErrorOutOfMemory ? G5_E_NOMEM : G5_E_HIP;
}

int grid_for(int64_t n, int block, int max_grid)
{
    int64_t g = (n + block - 1) / block;
    if (g < 1) g = 1;
    if (g > max_grid) g = max_grid;
    return (int)g;
}

// ---------------------------------------------------------------- fills

template <typename T>
__global__ void k_fill(T *d, int64_t n, T v)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        d[i] = v;
}

hipError_t fill_u64(uint64_t *d, int64_t n, uint64_t v, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill<uint64_t>, grid_for(n, 256, 8192), 256, 0, s, d, n, v);
    return hipGetLastError();
}
hipError_t fill_u32(uint32_t *d, int64_t n, uint32_t v, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill<uint32_t>, grid_for(n, 256, 8192), 256, 0, s, d, n, v);
    return hipGetLastError();
}
hipError_t fill_i64(int64_t *d, int64_t n, int64_t v, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill<int64_t>, grid_for(n, 256, 8192), 256, 0, s, d, n, v);
    return hipGetLastError();
}
hipError_t fill_i32(int32_t *d, int64_t n, int32_t v, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill<int32_t>, grid_for(n, 256, 8192), 256, 0, s, d, n, v);
    return hipGetLastError();
}

// ---------------------------------------------------------------- scan
// Three-phase exclusive scan over 1024-element tiles (256 threads x 4):
// tile sums -> recursive scan of the sums -> tile scan plus offset.

constexpr int kScanBlock = 256;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanBlock * kScanItems;

__device__ __forceinline__ int64_t block_excl_scan(int64_t v, int64_t *lds_waves, int64_t *total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int64_t inc = g5_wave_incl_scan(v);
    if (lane == 63) lds_waves[wave] = inc;
    __syncthreads();
    int64_t off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kScanBlock / 64; ++w) {
        const int64_t t = lds_waves[w];
        off += (w < wave) ? t : 0;
        tot += t;
    }
    *total = tot;
    return off + inc - v;
}

__global__ void k_tile_sums(const int64_t *d, int64_t n, int64_t *sums)
{
    __shared__ int64_t lw[kScanBlock / 64];
    const int64_t base = blockIdx.x * (int64_t)kScanTile + threadIdx.x * kScanItems;
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i)
        if (base + i < n) s += d[base + i];
    int64_t tot;
    block_excl_scan(s, lw, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ void k_tile_scan(int64_t *d, int64_t n, const int64_t *offs, int64_t *d_total)
{
    __shared__ int64_t lw[kScanBlock / 64];
    const int64_t base = blockIdx.x * (int64_t)kScanTile + threadIdx.x * kScanItems;
    int64_t v[kScanItems];
    int64_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        v[i] = (base + i < n) ? d[base + i] : 0;
        s += v[i];
    }
    int64_t tot;
    int64_t run = block_excl_scan(s, lw, &tot) + (offs ? offs[blockIdx.x] : 0);
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        if (base + i < n) d[base + i] = run;
        run += v[i];
    }
    if (d_total && blockIdx.x == gridDim.x - 1 && threadIdx.x == kScanBlock - 1) *d_total = run;
}

size_t scan_scratch_words(int64_t n)
{
    size_t w = 0;
    while (n > kScanTile) {
        n = (n + kScanTile - 1) / kScanTile;
        w += (size_t)n + 1;
    }
    return w + 1;
}

hipError_t exclusive_scan_i64(int64_t *d, int64_t n, int64_t *d_total, int64_t *scratch,
                              hipStream_t s)
{
    if (n <= 0) return d_total ? fill_i64(d_total, 1, 0, s) : hipSuccess;
    const int64_t tiles = (n + kScanTile - 1) / kScanTile;
    if (tiles == 1) {
        hipLaunchKernelGGL(k_tile_scan, 1, kScanBlock, 0, s, d, n, (const int64_t *)nullptr,
                           d_total);
        return hipGetLastError();
    }
    int64_t *sums = scratch;
    hipLaunchKernelGGL(k_tile_sums, (unsigned)tiles, kScanBlock, 0, s, (const int64_t *)d, n, sums);
    hipError_t e = exclusive_scan_i64(sums, tiles, nullptr, scratch + tiles + 1, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_tile_scan, (unsigned)tiles, kScanBlock, 0, s, d, n,
                       (const int64_t *)sums, d_total);
    return hipGetLastError();
}

// ---------------------------------------------------------------- sums

// K arrays; all loads of a round are in flight at once
template <int K>
__global__ __launch_bounds__(1024) void k_fold(const int64_t *__restrict__ part, int64_t stride, int n, FoldOut out)
{
    __shared__ int64_t s_wave[K][16];
    int64_t c[K] = {};
    for (int i0 = 0; i0 < n; i0 += 4096) {
        int64_t x[K][4];
#pragma unroll
        for (int j = 0; j < K; ++j)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = i0 + k * 1024 + threadIdx.x;
                x[j][k] = i < n ? part[j * stride + i] : 0;
            }
#pragma unroll
        for (int j = 0; j < K; ++j) c[j] += (x[j][0] + x[j][1]) + (x[j][2] + x[j][3]);
    }
#pragma unroll
    for (int j = 0; j < K; ++j) {
        c[j] = g5_wave_sum(c[j]);
        if (__lane_id() == 0) s_wave[j][threadIdx.x >> 6] = c[j];
    }
    __syncthreads();
    if ((int)threadIdx.x < out.ncopy) out.to[threadIdx.x] = out.from[threadIdx.x];
    if (threadIdx.x >= 64) return;
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const int64_t t = g5_wave_sum(threadIdx.x < 16 ? s_wave[j][threadIdx.x] : 0);
        if (threadIdx.x == 0) {
            if (out.host[j]) *out.host[j] = t;
            if (out.dev[j]) *out.dev[j] = t;
        }
    }
}

bool in_memory_of(int device, const uint64_t *p, int64_t n)
{
    hipPointerAttribute_t a{};
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipPointerGetAttributes(&a, p) != hipSuccess || a.type != hipMemoryTypeDevice || a.device != device ||
        hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p) != hipSuccess) {
        (void)hipGetLastError();  // memory that the runtime does not know is no error here
        return false;
    }
    const size_t at = (size_t)((const char *)p - (const char *)base);
    return ((uintptr_t)p & 7) == 0 && at <= size && (size_t)n * 8 <= size - at;
}

hipError_t fold_parts(const int64_t *part, int64_t stride, int n, const FoldOut &out, hipStream_t s)
{
    const int k = out.host[3] ? 4 : out.host[2] ? 3 : out.host[1] ? 2 : 1;
    hipLaunchKernelGGL(k == 4 ? k_fold<4> : k == 3 ? k_fold<3> : k == 2 ? k_fold<2> : k_fold<1>, 1, 1024, 0, s, part,
                       stride, n, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------- bitmap <-> queue
//
// A tile's workgroup takes 64 words at a time, 16 to a wave (lane j holds
// word j); a word's vertices are then the wave's lanes, so that row offsets
// are read and the queue is written in order.  A workgroup finds its tile's
// place by adding up the tiles before it (at most kTiles) instead of waiting
// for a scan of them: two launches where counts, scan of one to three
// launches and write took three to five, and six to nine with a degree prefix
// (2^22 vertices: 26 us of kernels, now 12).
constexpr int kWordsWave = 16;

// the degrees of this wave's vertices whose bits (lane j: word w0 + j) are
// set, in d[j] of each word's lanes; returns the lane's sum
__device__ __forceinline__ int64_t wave_degrees(uint64_t bits, int64_t w0, const int64_t *__restrict__ rowptr,
                                                int lane, uint32_t (&d)[kWordsWave])
{
    int64_t sum = 0;
    int64_t lo[kWordsWave], hi[kWordsWave];
#pragma unroll
    for (int j = 0; j < kWordsWave; ++j) {
        const uint64_t b = g5_bcast64(bits, j);
        const int64_t v = (w0 + j) * 64 + lane;
        const bool set = b >> lane & 1;
        lo[j] = set ? rowptr[v] : 0;
        hi[j] = set ? rowptr[v + 1] : 0;
    }
#pragma unroll
    for (int j = 0; j < kWordsWave; ++j) {
        d[j] = (uint32_t)(hi[j] - lo[j]);
        sum += d[j];
    }
    return sum;
}

__global__ __launch_bounds__(256) void k_bm_sums(const uint64_t *__restrict__ bits, int64_t n_words, int64_t tile,
                                                 const int64_t *__restrict__ rowptr, int64_t *__restrict__ part)
{
    const int lane = __lane_id();
    const int64_t end = min(n_words, (blockIdx.x + 1) * tile);
    int64_t c = 0, e = 0;
    for (int64_t w0 = blockIdx.x * tile + (threadIdx.x >> 6) * kWordsWave; w0 < end; w0 += 64) {
        const uint64_t b = lane < kWordsWave && w0 + lane < end ? bits[w0 + lane] : 0ull;
        c += __popcll(b);
        if (rowptr && __ballot(b != 0)) {
            uint32_t d[kWordsWave];
            e += wave_degrees(b, w0, rowptr, lane, d);
        }
    }
    c = g5_block_sum256(c);
    if (threadIdx.x == 0) part[blockIdx.x] = c;
    if (!rowptr) return;
    e = g5_block_sum256(e);
    if (threadIdx.x == 0) part[kTiles + blockIdx.x] = e;
}

template <bool kOffsets>
__global__ __launch_bounds__(256) void k_bm_write(const uint64_t *__restrict__ bits, int64_t n_words, int64_t tile,
                                                  const int64_t *__restrict__ rowptr,
                                                  const int64_t *__restrict__ part, QueueOut out)
{
    __shared__ int64_t s_n[4], s_e[4];
    const int lane = __lane_id(), wave = threadIdx.x >> 6;
    for (int64_t w = blockIdx.x * 256ll + threadIdx.x; w < out.n_clear; w += gridDim.x * 256ll) out.clear[w] = 0;
    // tiles before this one
    int64_t pos = 0, eoff = 0;
    for (int t = threadIdx.x; t < (int)blockIdx.x; t += 256) {
        pos += part[t];
        if (kOffsets) eoff += part[kTiles + t];
    }
    pos = g5_block_sum256(pos);
    if (kOffsets) eoff = g5_block_sum256(eoff);
    const int64_t end = min(n_words, (blockIdx.x + 1) * tile);
    for (int64_t g = blockIdx.x * tile; g < end; g += 64) {
        const int64_t w0 = g + wave * kWordsWave;
        const uint64_t b = lane < kWordsWave && w0 + lane < end ? bits[w0 + lane] : 0ull;
        uint32_t d[kWordsWave] = {};
        int64_t n = __popcll(b), e = 0;
        const bool any = __ballot(b != 0) != 0;
        if (kOffsets && any) e = wave_degrees(b, w0, rowptr, lane, d);
        n = g5_wave_sum(n);
        if (kOffsets) e = g5_wave_sum(e);
        if (lane == 0) {
            s_n[wave] = n;
            if (kOffsets) s_e[wave] = e;
        }
        __syncthreads();
        int64_t at = pos, eat = eoff;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            at += k < wave ? s_n[k] : 0;
            pos += s_n[k];
            if (kOffsets) {
                eat += k < wave ? s_e[k] : 0;
                eoff += s_e[k];
            }
        }
        __syncthreads();
        if (!any) continue;
#pragma unroll
        for (int j = 0; j < kWordsWave; ++j) {
            const uint64_t word = g5_bcast64(b, j);
            if (!word) continue;
            const bool set = word >> lane & 1;
            const int64_t i = at + __popcll(word & ((1ull << lane) - 1));
            if (set) out.q[i] = (uint32_t)((w0 + j) * 64 + lane);
            at += __popcll(word);
            if (kOffsets) {
                const int64_t inc = g5_wave_incl_scan((int64_t)d[j]);
                if (set) out.qoff[i] = eat + inc - d[j];
                eat += (int64_t)g5_bcast64((uint64_t)inc, 63);
            }
        }
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        if (out.d_n) *out.d_n = pos;
        if (out.h_n) *out.h_n = pos;
        if (kOffsets && out.d_e) *out.d_e = eoff;
    }
}

hipError_t bitmap_to_queue(const uint64_t *bits, int64_t n_words, const int64_t *rowptr, const QueueOut &out,
                           int64_t *part, bool have_parts, hipStream_t s)
{
    const int64_t tile = tile_words(n_words);
    const int tiles = n_words > 0 ? tile_count(n_words) : 1;  // an empty bitmap: the counts
    if (!have_parts && n_words > 0)
        hipLaunchKernelGGL(k_bm_sums, tiles, 256, 0, s, bits, n_words, tile, rowptr, part);
    if (rowptr) hipLaunchKernelGGL(k_bm_write<true>, tiles, 256, 0, s, bits, n_words, tile, rowptr, part, out);
    else hipLaunchKernelGGL(k_bm_write<false>, tiles, 256, 0, s, bits, n_words, tile, rowptr, part, out);
    return hipGetLastError();
}

// A wave takes 64 consecutive ids (a dense level's queue at 2^21 vertices: 3 us;
// with an atomic per id 12).  Neighbours with the same word combine
// their bits (a lane takes in the lanes 1, 2, 4, ... further that hold its
// word; a bit more than once does no harm), and the first of each run of equal
// words writes them with one atomic: a queue in ascending order takes about
// one per word and wave, and any other order stays right.
__global__ __launch_bounds__(256) void k_q2bm(const uint32_t *__restrict__ q, int64_t n,
                                              uint64_t *__restrict__ bits, int64_t n_words, int64_t *h_bad)
{
    const int lane = __lane_id();
    const int64_t last = (n + 63) / 64 * 64;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < last; i += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t v = i < n ? q[i] : 0u;
        const bool ok = i < n && (int64_t)(v >> 6) < n_words;
        if (i < n && !ok && h_bad) *h_bad = 1;
        const uint32_t w = ok ? v >> 6 : ~0u;
        uint64_t acc = ok ? 1ull << (v & 63) : 0ull;
        const uint32_t before = __shfl_up(w, 1, 64);
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t ow = __shfl_down(w, d, 64);
            const uint64_t o = __shfl_down(acc, d, 64);
            if (lane + d < 64 && ow == w) acc |= o;
        }
        if (ok && (lane == 0 || before != w)) atomicOr((unsigned long long *)&bits[w], (unsigned long long)acc);
    }
}

hipError_t queue_to_bitmap(const uint32_t *q, int64_t n, uint64_t *bits, int64_t n_words, int64_t *h_bad,
                           hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_q2bm, grid_for(n, 256, 16384), 256, 0, s, q, n, bits, n_words, h_bad);
    return hipGetLastError();
}

}  // namespace g5

// ---------------------------------------------------------------- C ABI

extern "C" const char *g5_last_error(void) { return g5::g_err; }

// ---------------------------------------------------------------- exchange accounting

namespace {
std::mutex g_ex_mu;
bool g_ex_on = false;
double g_ex_ms[G5_UNIT_COUNT] = {}, g_ex_bytes[G5_UNIT_COUNT] = {};
int64_t g_ex_calls[G5_UNIT_COUNT] = {};
}  // namespace

namespace g5 {

ExchangeTimer::ExchangeTimer(hipStream_t s) : s_(s)
{
    {
        std::lock_guard<std::mutex> lk(g_ex_mu);
        if (!g_ex_on) return;
    }
    if (hipEventCreate(&e0_) != hipSuccess || hipEventCreate(&e1_) != hipSuccess) {
        if (e0_) (void)hipEventDestroy(e0_);
        if (e1_) (void)hipEventDestroy(e1_);
        e0_ = e1_ = nullptr;
    }
}

ExchangeTimer::~ExchangeTimer()
{
    if (e0_) (void)hipEventDestroy(e0_);
    if (e1_) (void)hipEventDestroy(e1_);
}

hipError_t ExchangeTimer::start() { return e0_ ? hipEventRecord(e0_, s_) : hipSuccess; }

hipError_t ExchangeTimer::stop() { return e1_ ? hipEventRecord(e1_, s_) : hipSuccess; }

hipError_t ExchangeTimer::commit(int unit, double bytes, int64_t calls)
{
    if (!e0_) return hipSuccess;
    hipError_t e = hipEventSynchronize(e1_);
    float ms = 0;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0_, e1_);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lk(g_ex_mu);
    g_ex_ms[unit] += ms;
    g_ex_bytes[unit] += bytes;
    g_ex_calls[unit] += calls;
    return hipSuccess;
}

}  // namespace g5

extern "C" int g5_exchange_profile(int enable)
{
    std::lock_guard<std::mutex> lk(g_ex_mu);
    g_ex_on = enable != 0;
    for (int u = 0; u < G5_UNIT_COUNT; ++u) {
        g_ex_ms[u] = g_ex_bytes[u] = 0;
        g_ex_calls[u] = 0;
    }
    return G5_OK;
}

extern "C" int g5_exchange_stats(int unit, double *ms, double *bytes, int64_t *calls)
{
    G5_REQUIRE(unit >= 0 && unit < G5_UNIT_COUNT, G5_E_ARG, "g5_exchange_stats: unit %d out of range", unit);
    std::lock_guard<std::mutex> lk(g_ex_mu);
    if (ms) *ms = g_ex_ms[unit];
    if (bytes) *bytes = g_ex_bytes[unit];
    if (calls) *calls = g_ex_calls[unit];
    return G5_OK;
}

extern "C" int g5_init(int device)
{
    G5_HIP(hipSetDevice(device));
    G5_HIP(hipFree(nullptr));
    // the device's address of the no-allocation round trip's scratch
    return g5::noalloc_setup(device);
}

extern "C" int g5_mem_info(int64_t *free_bytes, int64_t *total_bytes)
{
    size_t f = 0, t = 0;
    G5_HIP(hipMemGetInfo(&f, &t));
    if (free_bytes) *free_bytes = (int64_t)f;
    if (total_bytes) *total_bytes = (int64_t)t;
    return G5_OK;
}

extern "C" int g5_device_sync(void)
{
    G5_HIP(hipDeviceSynchronize());
    return G5_OK;
}

extern "C" int g5_dmalloc(void **p, size_t bytes)
{
    G5_REQUIRE(p != nullptr, G5_E_ARG, "g5_dmalloc: null output pointer");
    G5_HIP(hipMalloc(p, bytes ? bytes : 1));
    return G5_OK;
}

extern "C" int g5_dfree(void *p)
{
    if (p) G5_HIP(hipFree(p));
    return G5_OK;
}

extern "C" int g5_memcpy_h2d(void *dst, const void *src, size_t bytes)
{
    if (bytes) G5_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return G5_OK;
}

extern "C" int g5_memcpy_d2h(void *dst, const void *src, size_t bytes)
{
    if (bytes) G5_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return G5_OK;
}

extern "C" int g5_memcpy_d2d(void *d_dst, const void *d_src, size_t bytes)
{
    if (bytes) G5_HIP(hipMemcpy(d_dst, d_src, bytes, hipMemcpyDeviceToDevice));
    return G5_OK;
}

extern "C" int g5_fill_u64(uint64_t *d, int64_t n, uint64_t value)
{
    G5_REQUIRE(n >= 0 && (d || n == 0), G5_E_ARG, "g5_fill_u64: bad arguments");
    G5_HIP(g5::fill_u64(d, n, value, nullptr));
    G5_HIP(hipStreamSynchronize(nullptr));
    return G5_OK;
}

namespace {

// What the calls below need on a device: the tiles' sums and a few pinned
// words, 16 KiB.  A thread keeps one per device it has called them on (the
// first kDevices; on others a call allocates its own), so that a call
// neither allocates nor waits for a free; they go with the thread.
struct Work {
    int device = -1;
    int64_t *part = nullptr;  // 2 * kTiles, on the device
    int64_t *host = nullptr;  // 8, pinned
    Work() = default;
    Work(const Work &) = delete;
    Work &operator=(const Work &) = delete;
    ~Work()
    {
        if (part) (void)hipFree(part);
        if (host) (void)hipHostFree(host);
    }
    hipError_t get()
    {
        hipError_t e = hipSuccess;
        if (!part) e = hipMalloc(&part, 2 * g5::kTiles * 8);
        if (e == hipSuccess && !host) e = hipHostMalloc(&host, 8 * 8, hipHostMallocDefault);
        return e;
    }
};
constexpr int kDevices = 8;

// the calling thread's, for its current device; own: the caller's, for a
// device beyond those that are kept
hipError_t work_for(Work *&w, Work &own)
{
    static thread_local Work kept[kDevices];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    w = &own;
    for (Work &k : kept)
        if (k.device == dev || k.device < 0) {
            w = &k;
            break;
        }
    w->device = dev;
    return w->get();
}

// part[workgroup] = its positions where a and b differ
__global__ __launch_bounds__(256) void k_diff_u32(const uint32_t *__restrict__ a, const uint32_t *__restrict__ b,
                                                  int64_t n, int64_t *__restrict__ part)
{
    int64_t c = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        c += a[i] != b[i];
    c = g5_block_sum256(c);
    if (threadIdx.x == 0) part[blockIdx.x] = c;
}

// part[workgroup] = its ids at or beyond n_words * 64
__global__ __launch_bounds__(256) void k_beyond(const uint32_t *__restrict__ q, int64_t n, int64_t n_words,
                                                int64_t *__restrict__ part)
{
    int64_t c = 0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        c += (int64_t)(q[i] >> 6) >= n_words;
    c = g5_block_sum256(c);
    if (threadIdx.x == 0) part[blockIdx.x] = c;
}

__global__ __launch_bounds__(256) void k_popcount(const uint64_t *__restrict__ bits, int64_t n_words,
                                                  int64_t *__restrict__ part)
{
    int64_t c = 0;
    for (int64_t w = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; w < n_words; w += (int64_t)gridDim.x * blockDim.x)
        c += __popcll(bits[w]);
    c = g5_block_sum256(c);
    if (threadIdx.x == 0) part[blockIdx.x] = c;
}

// waits for the sum of w.part[0 .. n)
hipError_t sum_of(Work &w, int n, int64_t *sum)
{
    g5::FoldOut o{};
    o.host[0] = w.host;
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = g5::fold_parts(w.part, 0, n, o, nullptr);
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    if (e == hipSuccess) *sum = w.host[0];
    return e;
}

}  // namespace

extern "C" int g5_diff_u32(const uint32_t *d_a, const uint32_t *d_b, int64_t n, int64_t *ndiff)
{
    G5_REQUIRE(n >= 0 && ndiff && (n == 0 || (d_a && d_b)), G5_E_ARG, "g5_diff_u32: bad arguments");
    *ndiff = 0;
    if (n == 0) return G5_OK;
    Work own, *w = nullptr;
    G5_HIP(work_for(w, own));
    const int grid = g5::grid_for(n, 256, 2 * g5::kTiles);
    hipLaunchKernelGGL(k_diff_u32, grid, 256, 0, nullptr, d_a, d_b, n, w->part);
    G5_HIP(sum_of(*w, grid, ndiff));
    return G5_OK;
}

extern "C" int g5_bitmap_to_queue(const uint64_t *d_bits, int64_t n_words, uint32_t *d_queue, int64_t *n)
{
    G5_REQUIRE(n_words >= 0 && n && (n_words == 0 || (d_bits && d_queue)), G5_E_ARG,
               "g5_bitmap_to_queue: bad arguments");
    Work own, *w = nullptr;
    G5_HIP(work_for(w, own));
    g5::QueueOut o{};
    o.q = d_queue;
    o.h_n = w->host;
    G5_HIP(g5::bitmap_to_queue(d_bits, n_words, nullptr, o, w->part, false, nullptr));
    G5_HIP(hipStreamSynchronize(nullptr));
    *n = w->host[0];
    return G5_OK;
}

extern "C" int g5_bitmap_count(const uint64_t *d_bits, int64_t n_words, int64_t *count)
{
    G5_REQUIRE(n_words >= 0 && count && (n_words == 0 || d_bits), G5_E_ARG, "g5_bitmap_count: bad arguments");
    *count = 0;
    if (n_words == 0) return G5_OK;
    Work own, *w = nullptr;
    G5_HIP(work_for(w, own));
    const int grid = g5::grid_for(n_words, 256, 2 * g5::kTiles);
    hipLaunchKernelGGL(k_popcount, grid, 256, 0, nullptr, d_bits, n_words, w->part);
    G5_HIP(sum_of(*w, grid, count));
    return G5_OK;
}

extern "C" int g5_queue_to_bitmap(const uint32_t *d_queue, int64_t n, uint64_t *d_bits, int64_t n_words)
{
    G5_REQUIRE(n >= 0 && n_words >= 0 && (n == 0 || d_queue) && (n_words == 0 || d_bits), G5_E_ARG,
               "g5_queue_to_bitmap: bad arguments");
    Work own, *w = nullptr;
    G5_HIP(work_for(w, own));
    w->host[0] = 0;
    G5_HIP(g5::fill_u64(d_bits, n_words, 0, nullptr));
    G5_HIP(g5::queue_to_bitmap(d_queue, n, d_bits, n_words, w->host, nullptr));
    G5_HIP(hipStreamSynchronize(nullptr));
    if (w->host[0] == 0) return G5_OK;
    int64_t bad = 0;
    const int grid = g5::grid_for(n, 256, 2 * g5::kTiles);
    hipLaunchKernelGGL(k_beyond, grid, 256, 0, nullptr, d_queue, n, n_words, w->part);
    G5_HIP(sum_of(*w, grid, &bad));
    G5_REQUIRE(bad == 0, G5_E_ARG, "g5_queue_to_bitmap: %lld ids beyond %lld words", (long long)bad,
               (long long)n_words);
    return G5_OK;
}
