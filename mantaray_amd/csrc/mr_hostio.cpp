// mr_hostio.cpp -- staging for host-memory calls (mr_hostio.h).
//
// A host-memory trace returns its rows to pageable memory the caller has
// just allocated.  What bounds that is the host: a plain hipMemcpy into fresh
// pages runs at 4-8 GB/s, as one thread takes the page faults and copies out
// of the runtime's own staging, against 57 GB/s into pinned memory.  So rows
// come down in pinned chunks and several threads copy them on, each waiting
// for its own chunk while the others' are in flight and taking its share of
// the page faults: 8,191 rays x 1000 steps (262 MB) through ray_tracing took
// 60 ms before and takes 8.3 ms.  Memory belonging to the caller is not
// pinned in place (hipHostRegister), and no result lives in the pool.
//
// The chunks, the streams and the device buffer are kept between calls (small
// calls spent more on allocations and on one copy per array than on their
// copies).  The pool is bounded: at most kIdleStages idle stages a process,
// each with kChunk x kWorkers pinned bytes and at most kKeepDevice of device
// memory.  When the last field handle dies, the device memory beyond
// kKeepIdle goes; the rest stays, as a call on file paths opens and frees its
// fields each time and would otherwise make and free its chunks and streams as
// well.  All of it is given back by drop_idle_stages (mr_release_host_buffers),
// and by an allocation that fails.
#include "mr_hostio.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <utility>

namespace mr {

namespace {

// A pinned chunk: 75 us on the bus, long against a wait's overhead.  A thread
// is worth starting for each megabyte (about 100 us of copying into fresh
// pages, against 15 us to start it).  A chunk takes 50 us to make, but each of
// a process's first four streams 3 ms.  So a stage's first call copies on one
// stream, which its workers share, and the next one that has use for them makes
// a stream for each worker: with one stream repeated calls of 6 to 130 MB took 5
// to 9 % longer, with four those of 16 to 40 MB 5 %; made one a call, each
// cost its call 2 to 9 ms.  Calls of ray_tracing on NetCDF paths in a process,
// 1000 steps, the first / second / later ones (ms):
//                        500 rays          2000 rays         8191 rays
//   plain copies         20 / 11 / 11.5    30 / 22 / 20.8    77 / 64 / 61
//   all streams at first 31 / -  /  4.8    34 / -  /  6.2    41 / -  / 10.0
//   on the second call   17 / 19 /  4.6    20 / 19 /  6.3    23 / 25 /  9.8
// (A process's very first call still waits for that one stream, one ray 13 to
// 14 ms against 11.9.)
constexpr size_t kChunk = size_t(4) << 20;
constexpr size_t kLeastChunk = size_t(64) << 10;
constexpr size_t kPerThread = size_t(1) << 20;
constexpr int kWorkers = 12;
constexpr size_t kIdleStages = 2;
constexpr size_t kKeepDevice = size_t(512) << 20;
constexpr size_t kKeepIdle = size_t(16) << 20;

}  // namespace

struct HostStage {
    int device = 0;
    hipStream_t stream[kWorkers] = {};
    int streams = 0;                   // those made
    bool used = false;                 // by a call before this one
    char *pin[kWorkers] = {};
    size_t pin_bytes[kWorkers] = {};
    char *dev = nullptr;
    size_t dev_bytes = 0;

    hipError_t need_streams(int n)
    {
        hipError_t e = hipSuccess;
        for (; e == hipSuccess && streams < n; streams += e == hipSuccess)
            e = hipStreamCreateWithFlags(&stream[streams], hipStreamNonBlocking);
        return e;
    }
    // a pinned chunk of at least `bytes` (up to kChunk) for worker w, whose
    // chunk is not in use
    hipError_t need_chunk(int w, size_t bytes)
    {
        if (pin_bytes[w] >= bytes) return hipSuccess;
        size_t n = kLeastChunk;
        while (n < bytes) n *= 2;
        if (pin[w]) (void)hipHostFree(pin[w]);
        pin_bytes[w] = 0;
        const hipError_t e =
            hipHostMalloc(reinterpret_cast<void **>(&pin[w]), n, hipHostMallocDefault);
        if (e != hipSuccess) pin[w] = nullptr;
        else pin_bytes[w] = n;
        return e;
    }
    hipError_t grow(size_t bytes)
    {
        if (bytes <= dev_bytes) return hipSuccess;
        drop_device();
        const hipError_t e = hipMalloc(reinterpret_cast<void **>(&dev), bytes);
        if (e != hipSuccess) dev = nullptr;
        else dev_bytes = bytes;
        return e;
    }
    void drop_device()
    {
        if (dev) (void)hipFree(dev);
        dev = nullptr;
        dev_bytes = 0;
    }
    ~HostStage()
    {
        int prev = -1;
        const bool sw = hipGetDevice(&prev) == hipSuccess && prev != device &&
                        hipSetDevice(device) == hipSuccess;
        drop_device();
        for (int k = 0; k < streams; k++) (void)hipStreamDestroy(stream[k]);
        for (char *p : pin)
            if (p) (void)hipHostFree(p);
        if (sw) (void)hipSetDevice(prev);
    }
};

namespace {

struct Pool {
    std::mutex mu;
    HostStage *idle[kIdleStages] = {};
};
// never destroyed: the HIP runtime may be gone before static destructors run
Pool &pool()
{
    static Pool *p = new Pool;
    return *p;
}

}  // namespace

void StageReturn::operator()(HostStage *s) const
{
    if (!s) return;
    if (s->dev_bytes > kKeepDevice) s->drop_device();
    s->used = true;
    {
        Pool &p = pool();
        std::lock_guard<std::mutex> lk(p.mu);
        for (HostStage *&slot : p.idle)
            if (!slot) {
                slot = s;
                return;
            }
    }
    delete s;
}

StagePtr acquire_stage(size_t bytes, hipError_t *err)
{
    int device = 0;
    if ((*err = hipGetDevice(&device)) != hipSuccess) return nullptr;
    StagePtr s;
    {
        Pool &p = pool();
        std::lock_guard<std::mutex> lk(p.mu);
        for (HostStage *&slot : p.idle)
            if (!s && slot && slot->device == device) {
                s.reset(slot);
                slot = nullptr;
            }
    }
    if (!s) {
        s.reset(new HostStage);
        s->device = device;
    }
    *err = s->grow(bytes);
    if (*err == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        drop_idle_stages();
        *err = s->grow(bytes);
    }
    if (*err == hipSuccess) *err = s->need_streams(1);
    if (*err == hipSuccess) *err = s->need_chunk(0, std::min(kChunk, std::max(bytes, kLeastChunk)));
    return *err == hipSuccess ? std::move(s) : nullptr;
}

hipStream_t stage_stream(const HostStage &s) { return s.stream[0]; }
char *stage_device(const HostStage &s) { return s.dev; }

void trim_idle_stages()
{
    Pool &p = pool();
    std::lock_guard<std::mutex> lk(p.mu);
    for (HostStage *s : p.idle)
        if (s && s->dev_bytes > kKeepIdle) s->drop_device();
}

void drop_idle_stages()
{
    HostStage *gone[kIdleStages] = {};
    {
        Pool &p = pool();
        std::lock_guard<std::mutex> lk(p.mu);
        std::swap(gone, p.idle);
    }
    for (HostStage *s : gone) delete s;
}

void parallel_for(int64_t n, int threads, const std::function<void(int64_t)> &f)
{
    std::atomic<int64_t> next{0};
    auto work = [&] {
        for (int64_t i; (i = next.fetch_add(1)) < n;) f(i);
    };
    std::vector<std::thread> t;
    try {
        t.reserve((size_t)std::max(threads, 1));
        for (int k = 1; k < std::min<int64_t>(threads, n); k++) t.emplace_back(work);
    } catch (...) {
        // fewer threads then: those that started and this one do the work
    }
    work();
    for (std::thread &x : t) x.join();
}

int copy_threads(size_t bytes)
{
    const int cpus = std::max(1, (int)std::thread::hardware_concurrency());
    return (int)std::max<size_t>(1, std::min<size_t>({(size_t)kWorkers, (size_t)cpus,
                                                      bytes / kPerThread}));
}

namespace {

// The part of the pieces that lies in [lo, hi) of the device buffer, between
// the caller's arrays and a chunk that stands for that range.
template <bool IN>
void move_range(const std::vector<HostPiece> &pieces, size_t lo, size_t hi, char *chunk)
{
    auto it = std::partition_point(pieces.begin(), pieces.end(), [&](const HostPiece &p) {
        return p.offset + p.bytes <= lo;
    });
    for (; it != pieces.end() && it->offset < hi; ++it) {
        const size_t a = std::max(lo, it->offset), b = std::min(hi, it->offset + it->bytes);
        char *host = it->host + (a - it->offset);
        if (b <= a) continue;
        if (IN) std::memcpy(chunk + (a - lo), host, b - a);
        else std::memcpy(host, chunk + (a - lo), b - a);
    }
}

}  // namespace

hipError_t copy_in(HostStage &s, const std::vector<HostPiece> &pieces)
{
    if (pieces.empty()) return hipSuccess;
    const size_t end = pieces.back().offset + pieces.back().bytes, chunk = s.pin_bytes[0];
    for (size_t lo = pieces.front().offset; lo < end; lo += chunk) {
        const size_t hi = std::min(end, lo + chunk);
        move_range<true>(pieces, lo, hi, s.pin[0]);
        hipError_t e = hipMemcpyAsync(s.dev + lo, s.pin[0], hi - lo, hipMemcpyHostToDevice,
                                      s.stream[0]);
        // the last chunk is not written again before copy_out's wait
        if (e == hipSuccess && hi < end) e = hipStreamSynchronize(s.stream[0]);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t copy_out(HostStage &s, const std::vector<HostPiece> &pieces)
{
    if (pieces.empty()) return hipStreamSynchronize(s.stream[0]);
    const size_t begin = pieces.front().offset;
    const size_t bytes = pieces.back().offset + pieces.back().bytes - begin;
    int threads = copy_threads(bytes);
    // few bytes: one chunk for each thread
    const size_t step =
        std::min({kChunk, s.pin_bytes[0], (bytes / (size_t)threads + 4096) & ~size_t(4095)});
    // (without memory for a worker's chunk, or streams for them, the copy does
    // with what is there)
    for (int w = 1; w < threads; w++)
        if (s.need_chunk(w, step) != hipSuccess) {
            (void)hipGetLastError();
            threads = w;
        }
    if (s.used && s.need_streams(threads) != hipSuccess) (void)hipGetLastError();
    auto chunk = [&](int64_t c, int w) {
        const size_t lo = begin + (size_t)c * step, hi = std::min(begin + bytes, lo + step);
        const hipStream_t stream = s.stream[w % s.streams];
        hipError_t e = hipMemcpyAsync(s.pin[w], s.dev + lo, hi - lo, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (e == hipSuccess) move_range<false>(pieces, lo, hi, s.pin[w]);
        return e;
    };
    const int64_t chunks = (int64_t)((bytes + step - 1) / step);
    if (threads == 1) {
        for (int64_t c = 0; c < chunks; c++) {
            const hipError_t e = chunk(c, 0);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    hipError_t e0 = hipStreamSynchronize(s.stream[0]);
    if (e0 != hipSuccess) return e0;
    std::atomic<int64_t> next{0};
    std::atomic<int> err{(int)hipSuccess};
    parallel_for(threads, threads, [&](int64_t w) {
        hipError_t e = hipSetDevice(s.device);
        for (int64_t c; e == hipSuccess && (c = next.fetch_add(1)) < chunks;) e = chunk(c, (int)w);
        if (e != hipSuccess) err = (int)e;
    });
    return (hipError_t)err.load();
}

}  // namespace mr
