// Seeded synthetic column generators (device side) and the library runtime
// helpers (launch shape, scratch, last-error text).
//
// Generator: SplitMix64 (Steele, Lea, Flood, OOPSLA 2014) used as a counter
// hash of (seed, stream, row), reduced to [lo, hi] with Lemire's
// multiply-shift (TOMACS 2019).  Every value is a pure function of its row, so
// a table of any size is produced in one pass at HBM write speed.
#include "capi_util.hpp"

#include <atomic>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

namespace sdb {
namespace {

constexpr int BLOCK = 256;

__host__ __device__ __forceinline__ uint64_t splitmix64(uint64_t x)
{
    uint64_t z = x + 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

__host__ __device__ __forceinline__ uint64_t stream_key(uint64_t seed, uint64_t stream)
{
    return splitmix64(seed * 0x100000001B3ULL + stream);
}

__device__ __forceinline__ int32_t uniform(uint64_t key, uint64_t row, int32_t lo, uint64_t range)
{
    const uint64_t h = splitmix64(key + row);
    return (int32_t)((int64_t)lo + (int64_t)(((h >> 32) * range) >> 32));
}

__global__ void __launch_bounds__(BLOCK) k_gen_uniform(int32_t *out, int64_t n, uint64_t key, int64_t first,
                                                       int32_t lo, uint64_t range)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK)
        out[i] = uniform(key, (uint64_t)(first + i), lo, range);
}

__global__ void __launch_bounds__(BLOCK) k_gen_child(int32_t *out, const int32_t *base, int64_t n, uint64_t key,
                                                     int64_t first, int32_t mult, int32_t lo, uint64_t range)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK)
        out[i] = base[i] * mult + uniform(key, (uint64_t)(first + i), lo, range);
}

__global__ void __launch_bounds__(BLOCK) k_gen_lookup(int32_t *out, int64_t n, uint64_t key, int64_t first,
                                                      const int32_t *table, uint64_t len)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK)
        out[i] = table[uniform(key, (uint64_t)(first + i), 0, len)];
}

__global__ void __launch_bounds__(BLOCK) k_gen_rowid(int32_t *out, int64_t n, int64_t first)
{
    for (int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * BLOCK)
        out[i] = (int32_t)(first + i + 1);
}

thread_local std::string g_last_error;

std::mutex g_cu_mu;
std::vector<int> g_cu_count;      // per device, 0 = unknown

} // namespace

void set_last_error(const std::string &msg) { g_last_error = msg; }

int device_cu_count()
{
    int dev = 0;
    SDB_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_cu_mu);
    if ((int)g_cu_count.size() <= dev) g_cu_count.resize(dev + 1, 0);
    if (g_cu_count[dev] == 0) {
        int cus = 0;
        SDB_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        g_cu_count[dev] = cus > 0 ? cus : 256;
    }
    return g_cu_count[dev];
}

unsigned stream_grid(int64_t units, int64_t per_block, int blocks_per_cu)
{
    if (units <= 0) return 1;
    const int64_t need = (units + per_block - 1) / per_block;
    const int64_t cap = (int64_t)device_cu_count() * blocks_per_cu;
    return (unsigned)std::max<int64_t>(1, std::min(need, cap));
}

// ------------------------------------------------------------------ scratch

struct ScratchBuffer {
    std::mutex mu;   // held by the call that uses the buffer
    void *ptr = nullptr;
    size_t bytes = 0;
    uint64_t used = 0;     // when last asked for (under the pool's mutex)
    bool dropped = false;  // no longer in the pool (under both)
};

namespace {

// What a buffer belongs to.  A stream's handle names it: a destroyed stream's
// handle may come back for a new one, but only after its work is done
// (hipStreamDestroy waits for it).  hipStreamPerThread is one handle for every
// thread's own stream.
struct ScratchKey {
    int dev;
    hipStream_t stream;
    uint64_t thread; // 0 but for hipStreamPerThread
    bool captured;
    bool operator<(const ScratchKey &o) const
    {
        return std::tie(dev, stream, thread, captured) < std::tie(o.dev, o.stream, o.thread, o.captured);
    }
};

// At most SCRATCH_MAX_BUFFERS per device outside captures, and past
// SCRATCH_MAX_BYTES in all only the one in use: the longest unused go first.
constexpr size_t SCRATCH_MAX_BUFFERS = 32;
constexpr size_t SCRATCH_MAX_BYTES = size_t(1) << 30;
struct ScratchPool {
    std::mutex mu;
    std::map<ScratchKey, std::shared_ptr<ScratchBuffer>> buffers;
    uint64_t clock = 0;
};
// (never destroyed: the runtime may be gone before this library's statics)
ScratchPool &scratch_pool()
{
    static ScratchPool *p = new ScratchPool;
    return *p;
}

uint64_t thread_number()
{
    static std::atomic<uint64_t> next{1};
    thread_local const uint64_t n = next++;
    return n;
}

ScratchKey scratch_key(hipStream_t stream)
{
    ScratchKey k{0, stream, stream == hipStreamPerThread ? thread_number() : 0, false};
    SDB_HIP(hipGetDevice(&k.dev));
    if (stream) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &st) == hipSuccess) k.captured = st == hipStreamCaptureStatusActive;
        else (void)hipGetLastError(); // a stream that cannot be captured now
    }
    return k;
}

// While a stream is captured, allocations are refused unless the thread says
// that it means them.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { SDB_HIP(hipThreadExchangeStreamCaptureMode(&mode)); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// Drops buffers of the device (never `keep`, one in use or one of a capture)
// until `bytes` more stay within the pool's bounds.  hipFree waits for the
// device, so for the kernels that still use one.
void scratch_trim(ScratchPool &P, const ScratchKey &key, const ScratchBuffer *keep, size_t bytes)
{
    while (true) {
        size_t count = 0, total = bytes;
        auto oldest = P.buffers.end();
        for (auto it = P.buffers.begin(); it != P.buffers.end(); ++it) {
            if (it->first.dev != key.dev || it->first.captured) continue;
            count++;
            if (it->second.get() == keep) continue;
            total += it->second->bytes;
            if (it->second->mu.try_lock()) {
                if (oldest == P.buffers.end() || it->second->used < oldest->second->used) {
                    if (oldest != P.buffers.end()) oldest->second->mu.unlock();
                    oldest = it;
                } else {
                    it->second->mu.unlock();
                }
            }
        }
        if (oldest == P.buffers.end()) return;
        const std::shared_ptr<ScratchBuffer> b = oldest->second;
        const bool drop = count > SCRATCH_MAX_BUFFERS || total > SCRATCH_MAX_BYTES;
        if (drop) {
            b->dropped = true;
            P.buffers.erase(oldest);
            if (b->ptr) (void)hipFree(b->ptr);
            b->ptr = nullptr;
            b->bytes = 0;
        }
        b->mu.unlock();
        if (!drop) return;
    }
}

} // namespace

Scratch::Scratch(size_t bytes, hipStream_t stream)
{
    const ScratchKey key = scratch_key(stream);
    ScratchPool &P = scratch_pool();
    while (true) {
        {
            std::lock_guard<std::mutex> lk(P.mu);
            std::shared_ptr<ScratchBuffer> &b = P.buffers[key];
            if (!b) b = std::make_shared<ScratchBuffer>();
            b->used = ++P.clock;
            buf_ = b;
        }
        buf_->mu.lock();
        if (!buf_->dropped) break;
        buf_->mu.unlock();
    }
    if (buf_->bytes >= bytes) return;
    try {
        const size_t want = std::max<size_t>(bytes, 1 << 20);
        RelaxedCapture relaxed;
        std::lock_guard<std::mutex> lk(P.mu);
        if (!key.captured) {
            if (buf_->ptr) {
                SDB_HIP(hipStreamSynchronize(stream));
                SDB_HIP(hipFree(buf_->ptr));
            }
            buf_->ptr = nullptr;
            buf_->bytes = 0;
            scratch_trim(P, key, buf_.get(), want);
        }
        // (a captured buffer that has become too small stays for its graphs;
        // each new one is twice as large at least, so they add up to little)
        const size_t size = key.captured ? std::max(want, 2 * buf_->bytes) : want;
        void *p = nullptr;
        SDB_HIP(hipMalloc(&p, size));
        buf_->ptr = p;
        buf_->bytes = size;
    } catch (...) {
        buf_->mu.unlock();
        throw;
    }
}

Scratch::~Scratch() { buf_->mu.unlock(); }

uint8_t *Scratch::data() const { return static_cast<uint8_t *>(buf_->ptr); }

void scratch_release(hipStream_t stream)
{
    ScratchKey key{0, stream, 0, false};
    if (hipGetDevice(&key.dev) != hipSuccess) return;
    ScratchPool &P = scratch_pool();
    std::shared_ptr<ScratchBuffer> b;
    {
        std::lock_guard<std::mutex> lk(P.mu);
        auto it = P.buffers.find(key);
        if (it == P.buffers.end()) return;
        b = it->second;
    }
    std::lock_guard<std::mutex> own(b->mu); // (before the pool's, as a call that grows its buffer)
    std::lock_guard<std::mutex> lk(P.mu);
    if (b->dropped) return;
    b->dropped = true;
    P.buffers.erase(key);
    if (b->ptr) (void)hipFree(b->ptr);
    b->ptr = nullptr;
    b->bytes = 0;
}

} // namespace sdb

using namespace sdb;

extern "C" {

const char *sdb_last_error(void) { return g_last_error.c_str(); }

const char *sdb_version(void) { return "sycldb-mi355x 0.1"; }

int sdb_gen_uniform(int32_t *out, int64_t n, uint64_t seed, uint64_t stream_id, int64_t first_row, int32_t lo,
                    int32_t hi, sdb_stream stream)
{
    return guarded([&] {
        require(n >= 0 && (n == 0 || out), "bad output");
        require(hi >= lo, "hi < lo");
        if (n == 0) return;
        const uint64_t range = (uint64_t)((int64_t)hi - (int64_t)lo + 1);
        hipLaunchKernelGGL(k_gen_uniform, dim3(stream_grid(n, BLOCK)), dim3(BLOCK), 0, as_stream(stream), out, n,
                           stream_key(seed, stream_id), first_row, lo, range);
        hip_check(hipGetLastError(), "gen_uniform");
    });
}

int sdb_gen_child(int32_t *out, const int32_t *base, int64_t n, uint64_t seed, uint64_t stream_id,
                  int64_t first_row, int32_t mult, int32_t lo, int32_t hi, sdb_stream stream)
{
    return guarded([&] {
        require(n >= 0 && (n == 0 || (out && base)), "bad pointers");
        require(hi >= lo, "hi < lo");
        if (n == 0) return;
        const uint64_t range = (uint64_t)((int64_t)hi - (int64_t)lo + 1);
        hipLaunchKernelGGL(k_gen_child, dim3(stream_grid(n, BLOCK)), dim3(BLOCK), 0, as_stream(stream), out, base,
                           n, stream_key(seed, stream_id), first_row, mult, lo, range);
        hip_check(hipGetLastError(), "gen_child");
    });
}

int sdb_gen_lookup(int32_t *out, int64_t n, uint64_t seed, uint64_t stream_id, int64_t first_row,
                   const int32_t *table, int32_t table_len, sdb_stream stream)
{
    return guarded([&] {
        require(n >= 0 && (n == 0 || (out && table)), "bad pointers");
        require(table_len > 0, "empty lookup table");
        if (n == 0) return;
        hipLaunchKernelGGL(k_gen_lookup, dim3(stream_grid(n, BLOCK)), dim3(BLOCK), 0, as_stream(stream), out, n,
                           stream_key(seed, stream_id), first_row, table, (uint64_t)table_len);
        hip_check(hipGetLastError(), "gen_lookup");
    });
}

int sdb_device_alloc(void **ptr, uint64_t bytes)
{
    return guarded([&] {
        require(ptr != nullptr, "null output pointer");
        *ptr = nullptr;
        if (bytes == 0) return;
        const hipError_t e = hipMalloc(ptr, bytes);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            fail(SDB_ERR_OOM, "device allocation of " + std::to_string(bytes) + " bytes failed");
        }
        hip_check(e, "hipMalloc");
    });
}

int sdb_device_free(void *ptr)
{
    return guarded([&] {
        if (ptr) SDB_HIP(hipFree(ptr));
    });
}

int sdb_copy_to_device(void *dst, const void *host_src, uint64_t bytes, sdb_stream stream)
{
    return guarded([&] {
        if (bytes == 0) return;
        require(dst && host_src, "null pointer");
        SDB_HIP(hipMemcpyAsync(dst, host_src, bytes, hipMemcpyHostToDevice, as_stream(stream)));
        SDB_HIP(hipStreamSynchronize(as_stream(stream)));
    });
}

int sdb_copy_to_host(void *host_dst, const void *src, uint64_t bytes, sdb_stream stream)
{
    return guarded([&] {
        if (bytes == 0) return;
        require(host_dst && src, "null pointer");
        SDB_HIP(hipMemcpyAsync(host_dst, src, bytes, hipMemcpyDeviceToHost, as_stream(stream)));
        SDB_HIP(hipStreamSynchronize(as_stream(stream)));
    });
}

int sdb_stream_synchronize(sdb_stream stream)
{
    return guarded([&] { SDB_HIP(hipStreamSynchronize(as_stream(stream))); });
}

int sdb_gen_rowid(int32_t *out, int64_t n, int64_t first_row, sdb_stream stream)
{
    return guarded([&] {
        require(n >= 0 && (n == 0 || out), "bad output");
        if (n == 0) return;
        hipLaunchKernelGGL(k_gen_rowid, dim3(stream_grid(n, BLOCK)), dim3(BLOCK), 0, as_stream(stream), out, n,
                           first_row);
        hip_check(hipGetLastError(), "gen_rowid");
    });
}

} // extern "C"
