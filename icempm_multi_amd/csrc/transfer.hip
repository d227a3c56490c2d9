// transfer.hip -- points between HostSideSOA buffers and the device
// (GPU_Partition::transfer_points_from_soa_to_device and transfer_from_device,
// gpu_partition.cu:16-68).
//
// Chunks of points go through pinned staging memory that kernels read and
// write over the link, converting the mixed form's elements on the way, while
// the host copies the chunk before (or after) between staging and the
// caller's lines.  Before, each line was one copy from or to pageable memory
// (16 of them per call, 20 us each for any size, 18 GB/s for large ones) and
// one host thread converted the mixed form's elements.  Per call, before and
// after: download of 1.6k points 317 -> 29 us, of 4.0M points (512 MB) 30 -> 10
// ms, in the mixed form 172 -> 10 ms; upload of 4.0M points 17.7 -> 12.5 ms, of
// 410k points in the mixed form 13 -> 1.4 ms.  The large ones move 41 to 51
// GB/s over a link whose plain pinned copies reach 57.
//
// Built with -ffp-contract=off: the conversions round each operation, as the
// host code that they replace did.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstring>
#include <list>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "engine.h"
#include "icempm_host.h"

namespace icempm {

namespace {

constexpr int kBlock = 256;
constexpr int kStageDepth = 3;   // chunks in flight of a transfer
typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// The mixed form's position map: x/h = q*2^-frac_bits - origin.
struct PosMap {
    double h, hinv, scale, inv;   // scale = 2^frac_bits, inv = 2^-frac_bits
    int origin[2];
};

template <class To, class From>
__host__ __device__ __forceinline__ To bits_as(From v)
{
    static_assert(sizeof(To) == sizeof(From), "the same bits");
    return __builtin_bit_cast(To, v);
}

// One element of a line from the mixed form to FP64 bits.
__host__ __device__ __forceinline__ unsigned long long widen(int line, unsigned v, const PosMap &m)
{
    if (line == kLineUtility) return v;
    double d;
    if (line == kLinePosX || line == kLinePosX + 1) {
        d = ((double)v * m.inv - m.origin[line - kLinePosX]) * m.h;
    } else {
        d = (double)bits_as<float>(v);
        if (line == kLineJp || line == kLineFe00 || line == kLineFe00 + 3) d += 1.0;   // stored as the difference from 1
    }
    return bits_as<unsigned long long>(d);
}

// And back.
__host__ __device__ __forceinline__ unsigned narrow(int line, unsigned long long v, const PosMap &m)
{
    if (line == kLineUtility) return (unsigned)v;
    double d = bits_as<double>(v);
    if (line == kLinePosX || line == kLinePosX + 1) {
        const double q = rint((d * m.hinv + m.origin[line - kLinePosX]) * m.scale);
        return q > 0 ? (unsigned)fmin(q, 4294967295.0) : 0u;   // clamped to the fixed-point range (NaN: 0)
    }
    if (line == kLineJp || line == kLineFe00 || line == kLineFe00 + 3) d -= 1.0;
    return bits_as<unsigned>((float)d);
}

// Points [first, first + m) of the device lines to staging, line l at
// l * stage_pitch; a line per blockIdx.y, two points per thread (first and
// stage_pitch are even; a last odd point's neighbour lies in the scene's
// capacity, which is a multiple of 256, and in the staging line).
template <int EB>
__global__ void __launch_bounds__(kBlock) k_export(const void *pts, long long pitch, long long first, int m,
                                                   unsigned long long *stage, long long stage_pitch, PosMap map)
{
    const int i = 2 * (blockIdx.x * kBlock + threadIdx.x), line = blockIdx.y;
    if (i >= m) return;
    u64x2 out;
    if (EB == 8) {
        out = *(const u64x2 *)((const unsigned long long *)pts + line * pitch + first + i);
    } else {
        const u32x2 v = *(const u32x2 *)((const unsigned *)pts + line * pitch + first + i);
        out = u64x2{widen(line, v.x, map), widen(line, v.y, map)};
    }
    *(u64x2 *)(stage + line * stage_pitch + i) = out;
}

template <int EB>
__global__ void __launch_bounds__(kBlock) k_import(void *pts, long long pitch, long long first, int m,
                                                   const unsigned long long *stage, long long stage_pitch, PosMap map)
{
    const int i = 2 * (blockIdx.x * kBlock + threadIdx.x), line = blockIdx.y;
    if (i >= m) return;
    const u64x2 v = *(const u64x2 *)(stage + line * stage_pitch + i);
    const bool both = i + 1 < m;
    if (EB == 8) {
        unsigned long long *d = (unsigned long long *)pts + line * pitch + first + i;
        if (both) *(u64x2 *)d = v;
        else *d = v.x;
    } else {
        unsigned *d = (unsigned *)pts + line * pitch + first + i;
        const u32x2 w = {narrow(line, v.x, map), narrow(line, v.y, map)};
        if (both) *(u32x2 *)d = w;
        else *d = w.x;
    }
}

__global__ void __launch_bounds__(kBlock) k_read(const unsigned *src, unsigned *dst, int n)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

}  // namespace

// Pinned memory for the chunks in flight of one transfer, and an event per
// chunk, of one device.  The host reads a chunk after its event alone, and the
// next kernel reads what the host wrote, so the memory is coherent: without
// that flag it need not be, and an event need not make a kernel's stores
// visible to the host.  (It costs nothing: 4.0M points 12.24 ms up and 9.87
// down with it, 12.25 and 9.87 without.)
struct Staging {
    int device = 0;
    double *mem = nullptr;
    size_t bytes = 0;
    hipEvent_t ev[kStageDepth] = {nullptr, nullptr, nullptr};

    ~Staging()
    {
        if (mem) hipHostFree(mem);
        for (hipEvent_t e : ev)
            if (e) hipEventDestroy(e);
    }
};

// The line copies of one transfer.  The caller declares chunk after chunk
// ready and copies lines itself; pool threads take lines as they get a CPU.
// Nobody waits for a helper that has not started on a line: where other
// threads of the program keep the CPUs busy (an OpenMP pool that spins after
// its last loop), a fixed share per helper made the upload of 410k points 5
// times slower, and joining the helpers after the transfer 2 to 3 times.
struct CopyJob {
    double *stage;
    long long chunk, n;            // points per chunk, points in all
    int depth;
    double *host;                  // the caller's line 0, first point
    size_t capacity;
    bool to_host;
    std::atomic<long long> ready{0}, next{0};
    std::atomic<int> left[kStageDepth];
    std::atomic<bool> done{false};

    void copy(long long k, int line) const
    {
        const long long at = k * chunk, m = std::min(chunk, n - at);
        double *const s = stage + ((k % depth) * kNumPtsLines + line) * chunk, *const h = host + line * capacity + at;
        std::memcpy(to_host ? h : s, to_host ? s : h, sizeof(double) * m);
    }
    // one line of a ready chunk, if there is one left
    bool take()
    {
        long long i = next.load(std::memory_order_relaxed);
        do {
            if (i >= ready.load(std::memory_order_acquire)) return false;
        } while (!next.compare_exchange_weak(i, i + 1, std::memory_order_acq_rel));
        copy(i / kNumPtsLines, (int)(i % kNumPtsLines));
        left[(i / kNumPtsLines) % depth].fetch_sub(1, std::memory_order_acq_rel);
        return true;
    }
    // The caller's part: copies chunk k, the next one; returns when all of it is copied.
    void run_chunk(long long k)
    {
        left[k % depth].store(kNumPtsLines, std::memory_order_relaxed);
        ready.store((k + 1) * kNumPtsLines, std::memory_order_release);
        while (take()) {
        }
        while (left[k % depth].load(std::memory_order_acquire) > 0) std::this_thread::yield();
    }
};

// What the engines of the process share for their transfers, freed with the
// last engine that made one: the staging memory (making and freeing it per
// engine cost 0.8 ms each; a transfer takes a piece of its own for its time,
// and at most kIdleMost idle ones of at most 12 MB are kept) and the helper
// threads (started by the first large transfer, asleep unless one is under way).
class TransferPool {
public:
    static std::shared_ptr<TransferPool> get()
    {
        static std::mutex m;
        static std::weak_ptr<TransferPool> pool;
        std::lock_guard<std::mutex> lock(m);
        std::shared_ptr<TransferPool> p = pool.lock();
        if (!p) pool = p = std::make_shared<TransferPool>();
        return p;
    }
    ~TransferPool()
    {
        {
            std::lock_guard<std::mutex> lock(m_);
            stop_ = true;
        }
        cv_.notify_all();
        for (auto &t : threads_) t.join();
    }
    // Staging of at least `bytes` for a device; null if there is none to be had.
    std::unique_ptr<Staging> take(int device, size_t bytes)
    {
        {
            std::lock_guard<std::mutex> lock(m_);
            for (auto it = idle_.begin(); it != idle_.end(); ++it)
                if ((*it)->device == device && (*it)->bytes >= bytes) {
                    std::unique_ptr<Staging> st = std::move(*it);
                    idle_.erase(it);
                    return st;
                }
        }
        std::unique_ptr<Staging> st(new Staging);
        st->device = device;
        hipError_t e = hipHostMalloc((void **)&st->mem, bytes, hipHostMallocPortable | hipHostMallocCoherent);
        if (e != hipSuccess) st->mem = nullptr;
        st->bytes = bytes;
        const OnDevice here(device);
        for (hipEvent_t &ev : st->ev)
            if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e == hipSuccess) return st;
        hipGetLastError();   // the caller does without: not the error of its next launch
        return nullptr;
    }
    void give_back(std::unique_ptr<Staging> st)
    {
        std::unique_ptr<Staging> least;   // freed outside the lock
        std::lock_guard<std::mutex> lock(m_);
        idle_.push_back(std::move(st));
        if (idle_.size() > kIdleMost) {
            auto it = std::min_element(idle_.begin(), idle_.end(),
                                       [](const auto &x, const auto &y) { return x->bytes < y->bytes; });
            least = std::move(*it);
            idle_.erase(it);
        }
    }
    void begin(const std::shared_ptr<CopyJob> &job)
    {
        {
            std::lock_guard<std::mutex> lock(m_);
            if (threads_.empty()) {
                const unsigned hw = std::thread::hardware_concurrency();
                try {
                    for (int t = 0; t < (hw >= 8 ? 3 : hw >= 4 ? 1 : 0); t++) threads_.emplace_back([this] { work(); });
                } catch (const std::exception &) {
                    // fewer helpers, perhaps none
                }
            }
            jobs_.push_back(job);
        }
        cv_.notify_all();
    }
    void end(const std::shared_ptr<CopyJob> &job)
    {
        job->done.store(true, std::memory_order_release);
        std::lock_guard<std::mutex> lock(m_);
        jobs_.remove(job);
    }

private:
    void work()
    {
        std::unique_lock<std::mutex> lock(m_);
        for (;;) {
            cv_.wait(lock, [this] { return stop_ || !jobs_.empty(); });
            if (stop_) return;
            const std::shared_ptr<CopyJob> job = jobs_.front();
            lock.unlock();
            while (!job->done.load(std::memory_order_acquire))
                if (!job->take()) std::this_thread::yield();
            lock.lock();
        }
    }
    static constexpr size_t kIdleMost = 4;
    std::mutex m_;
    std::condition_variable cv_;
    std::list<std::unique_ptr<Staging>> idle_;
    std::list<std::shared_ptr<CopyJob>> jobs_;
    bool stop_ = false;
    std::vector<std::thread> threads_;
};

namespace {

// A transfer under way: its staging, and its job, known to the pool's helpers
// from a size on.  Ends at whatever point its scope is left: the stream has
// read or written the staging before it is given back.
// One thread copies about 20 GB/s between staging and memory that is not in
// its cache, three more keep up with the link; waking them pays from 16 MB on.
struct Transfer {
    std::shared_ptr<TransferPool> pool;
    hipStream_t stream;
    std::unique_ptr<Staging> st;
    std::shared_ptr<CopyJob> job = std::make_shared<CopyJob>();
    bool helped = false;

    Transfer(std::shared_ptr<TransferPool> p, hipStream_t s) : pool(std::move(p)), stream(s) {}
    void begin()
    {
        if (job->n < 128 * 1024) return;
        pool->begin(job);
        helped = true;
    }
    ~Transfer()
    {
        if (helped) pool->end(job);
        if (st) {
            hipStreamSynchronize(stream);
            pool->give_back(std::move(st));
        }
    }
};

// Chunks: at most 32k points (4 MB), and eight from 32k points on, so that the
// link and the host copies overlap and the staging of a small scene is small.
constexpr int kChunkMax = 32768, kChunkMin = 4096;
long long chunk_points(long long n)
{
    const long long q = ((n + 7) / 8 + 255) / 256 * 256;
    return std::min<long long>(std::max<long long>(q, kChunkMin), kChunkMax);
}

#define LAUNCH_EB(kernel, grid, ...)                                                       \
    do {                                                                                   \
        if (elem_bytes() == 8) hipLaunchKernelGGL(kernel<8>, grid, dim3(kBlock), 0, stream_, __VA_ARGS__); \
        else hipLaunchKernelGGL(kernel<4>, grid, dim3(kBlock), 0, stream_, __VA_ARGS__);   \
    } while (0)

}  // namespace

static PosMap position_map(const SceneConsts &c)
{
    PosMap m;
    m.h = c.h;
    m.hinv = c.hinv;
    m.scale = std::ldexp(1.0, c.frac_bits);
    m.inv = std::ldexp(1.0, -c.frac_bits);
    m.origin[0] = c.origin;
    m.origin[1] = c.origin_y;
    return m;
}

// A transfer without staging, where there is no pinned memory to be had: line
// by line from or to the caller's memory, the mixed form's elements converted
// by this thread.  Many times slower.
int Engine::copy_points(int scene, double *host, size_t capacity, long long n, bool to_host)
{
    const PosMap map = position_map(host_dev_[scene].c);
    const size_t eb = elem_bytes();
    std::vector<unsigned> words(eb == 4 ? n : 0);
    for (int line = 0; line < kNumPtsLines; line++) {
        char *const dev = (char *)pts_[0] + (line * pitch_ + scenes_[scene].pt_off) * eb;
        double *const h = host + line * capacity;
        void *const mem = eb == 4 ? (void *)words.data() : (void *)h;
        for (long long i = 0; i < (long long)words.size() && !to_host; i++)
            words[i] = narrow(line, bits_as<unsigned long long>(h[i]), map);
        hipError_t e = to_host ? hipMemcpyAsync(mem, dev, eb * n, hipMemcpyDeviceToHost, stream_)
                               : hipMemcpyAsync(dev, mem, eb * n, hipMemcpyHostToDevice, stream_);
        if (e == hipSuccess) e = hipStreamSynchronize(stream_);
        if (e != hipSuccess) return hipfail(e, "point transfer");
        for (long long i = 0; i < (long long)words.size() && to_host; i++)
            h[i] = bits_as<double>(widen(line, words[i], map));
    }
    return ICEMPM_OK;
}

int Engine::import_points(int scene, const double *hssoa, size_t capacity, long long offset, long long n)
{
    if (n <= 0) return ICEMPM_OK;
    hipError_t e = hipSuccess;
    Transfer t(transfer_pool(), stream_);
    CopyJob &job = *t.job;
    job.n = n;
    job.chunk = chunk_points(n);
    job.host = const_cast<double *>(hssoa) + offset;   // read only: to_host is false
    job.capacity = capacity;
    job.to_host = false;
    const long long chunk = job.chunk, n_chunks = (n + chunk - 1) / chunk, first = scenes_[scene].pt_off;
    const int depth = job.depth = (int)std::min<long long>(kStageDepth, n_chunks);
    t.st = t.pool->take(device_, (size_t)chunk * depth * kNumPtsLines * sizeof(double));
    if (!t.st) return copy_points(scene, job.host, capacity, n, job.to_host);
    job.stage = t.st->mem;
    const PosMap map = position_map(host_dev_[scene].c);
    t.begin();
    for (long long k = 0; k < n_chunks && e == hipSuccess; k++) {
        const int slot = (int)(k % depth), m = (int)std::min(chunk, n - k * chunk);
        if (k >= depth && (e = hipEventSynchronize(t.st->ev[slot])) != hipSuccess) break;   // read by its kernel
        job.run_chunk(k);
        LAUNCH_EB(k_import, dim3((m + 2 * kBlock - 1) / (2 * kBlock), kNumPtsLines), pts_[0], pitch_, first + k * chunk,
                  m, (const unsigned long long *)(job.stage + slot * chunk * kNumPtsLines), chunk, map);
        e = hipGetLastError();
        if (e == hipSuccess && n_chunks > depth) e = hipEventRecord(t.st->ev[slot], stream_);
    }
    const hipError_t es = hipStreamSynchronize(stream_);   // the staging is read
    if (e == hipSuccess) e = es;
    return e == hipSuccess ? ICEMPM_OK : hipfail(e, "point upload");
}

int Engine::export_points(int scene, double *hssoa, size_t capacity, long long offset, long long n)
{
    hipError_t e = hipSuccess;
    if (n <= 0) {
        e = hipStreamSynchronize(stream_);
        return e == hipSuccess ? ICEMPM_OK : hipfail(e, "point download");
    }
    Transfer t(transfer_pool(), stream_);
    CopyJob &job = *t.job;
    job.n = n;
    job.chunk = chunk_points(n);
    job.host = hssoa + offset;
    job.capacity = capacity;
    job.to_host = true;
    const long long chunk = job.chunk, n_chunks = (n + chunk - 1) / chunk, first = scenes_[scene].pt_off;
    const int depth = job.depth = (int)std::min<long long>(kStageDepth, n_chunks);
    t.st = t.pool->take(device_, (size_t)chunk * depth * kNumPtsLines * sizeof(double));
    if (!t.st) return copy_points(scene, job.host, capacity, n, job.to_host);
    job.stage = t.st->mem;
    const PosMap map = position_map(host_dev_[scene].c);
    auto launch = [&](long long k) {
        const int slot = (int)(k % depth), m = (int)std::min(chunk, n - k * chunk);
        LAUNCH_EB(k_export, dim3((m + 2 * kBlock - 1) / (2 * kBlock), kNumPtsLines), (const void *)pts_[0], pitch_,
                  first + k * chunk, m, (unsigned long long *)(job.stage + slot * chunk * kNumPtsLines), chunk, map);
        const hipError_t el = hipGetLastError();
        return el == hipSuccess ? hipEventRecord(t.st->ev[slot], stream_) : el;
    };
    for (long long k = 0; k < depth && e == hipSuccess; k++) e = launch(k);
    if (e == hipSuccess) t.begin();
    for (long long k = 0; k < n_chunks && e == hipSuccess; k++) {
        if ((e = hipEventSynchronize(t.st->ev[k % depth])) != hipSuccess) break;
        job.run_chunk(k);
        if (k + depth < n_chunks) e = launch(k + depth);
    }
    const hipError_t es = hipStreamSynchronize(stream_);
    if (e == hipSuccess) e = es;
    return e == hipSuccess ? ICEMPM_OK : hipfail(e, "point download");
}

// A copy of a few words to pageable memory takes 20 to 22 us;
// a kernel that writes them to pinned memory and the wait for it take 12 to 14.
int Engine::read_back(void *dst, const void *src, size_t bytes)
{
    constexpr size_t kMost = 64 * 1024;
    hipError_t e = hipSuccess;
    Transfer t(transfer_pool(), stream_);
    if (bytes <= kMost && bytes % sizeof(unsigned) == 0) t.st = t.pool->take(device_, kMost);
    if (!t.st) {
        e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream_);
        if (e == hipSuccess) e = hipStreamSynchronize(stream_);
        return e == hipSuccess ? ICEMPM_OK : hipfail(e, "read back");
    }
    if (bytes == 0) return ICEMPM_OK;
    const int n = (int)(bytes / sizeof(unsigned));
    hipLaunchKernelGGL(k_read, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, stream_, (const unsigned *)src,
                       (unsigned *)t.st->mem, n);
    e = hipGetLastError();
    const hipError_t es = hipStreamSynchronize(stream_);
    if (e == hipSuccess) e = es;
    if (e != hipSuccess) return hipfail(e, "read back");
    std::memcpy(dst, t.st->mem, bytes);
    return ICEMPM_OK;
}

const std::shared_ptr<TransferPool> &Engine::transfer_pool()
{
    if (!transfer_pool_) transfer_pool_ = TransferPool::get();
    return transfer_pool_;
}

}  // namespace icempm
