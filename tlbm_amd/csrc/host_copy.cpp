// host_copy.cpp -- see host_copy.h.
#include "host_copy.h"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <utility>
#include <vector>

namespace {

// A slot and what it widens to stay in a core's cache; 256 KiB to 1 MiB make
// no difference beyond the noise, and 8 MiB take half as long to pin as 16.
constexpr size_t kSlotBytes = size_t(512) << 10;
constexpr int kSlots = 16;
constexpr int kThreads = 8;
// Shorter copies go without ring and threads, whose start takes longer than
// they save.  Of FP32 values: 48^3 moments 178 us, through the ring 152 to 270,
// 64^3 (4 MiB) 415 and 300.  Of doubles, which the runtime puts straight into
// the caller's array: 17 MB 1.0 ms, through the ring 1.6; 40 MB 3.9 and 2.2.
constexpr size_t kRingFrom32 = size_t(4) << 20, kRingFrom64 = size_t(32) << 20;
constexpr size_t kKept = 2;

struct Ring {
    int device = -1;
    char *base = nullptr;
    hipEvent_t ev[kSlots] = {};
    Ring() = default;
    Ring(const Ring &) = delete;
    Ring &operator=(const Ring &) = delete;
    ~Ring() {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (base) (void)hipHostFree(base);
    }
    hipError_t create(int dev) {
        device = dev;
        hipError_t e = hipHostMalloc(reinterpret_cast<void **>(&base), kSlots * kSlotBytes, hipHostMallocPortable);
        for (int k = 0; k < kSlots && e == hipSuccess; ++k) e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
        return e;
    }
};

std::mutex g_mu;
Ring *g_kept[kKept] = {};
int g_users = 0;

// A ring of device dev, which need not be the calling thread's.
hipError_t take(int dev, Ring **out) {
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (Ring *&k : g_kept)
            if (k && k->device == dev) {
                *out = std::exchange(k, nullptr);
                return hipSuccess;
            }
    }
    Ring *r = new (std::nothrow) Ring;
    if (!r) return hipErrorOutOfMemory;
    int was = dev;
    hipError_t e = hipGetDevice(&was);
    if (e == hipSuccess) e = hipSetDevice(dev);
    if (e == hipSuccess) e = r->create(dev);
    (void)hipSetDevice(was);
    if (e != hipSuccess) {
        delete r;
        return e;
    }
    *out = r;
    return hipSuccess;
}

void give(Ring *r) {
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (g_users > 0)
            for (Ring *&k : g_kept)
                if (!k) {
                    k = r;
                    return;
                }
    }
    delete r;
}

struct Chunk {
    const char *dev;
    double *host;
    size_t count;
};

std::vector<Chunk> chunks_of(const tlbm::CopyPart *parts, int n, size_t esz) {
    std::vector<Chunk> out;
    const size_t most = kSlotBytes / esz;
    for (int k = 0; k < n; ++k)
        for (size_t at = 0; at < parts[k].count; at += most)
            out.push_back({parts[k].dev + at * esz, parts[k].host + at, std::min(most, parts[k].count - at)});
    return out;
}

void unpack(const Chunk &c, const void *from, bool widen) {
    if (!widen) {
        std::memcpy(c.host, from, c.count * sizeof(double));
        return;
    }
    const float *src = static_cast<const float *>(from);
    double *dst = c.host;
    for (size_t i = 0, n = c.count; i < n; ++i) dst[i] = double(src[i]);
}

// A copy through a ring.  Chunk i uses slot i % kSlots: the calling thread
// queues its DMA and an event, a worker waits for that and unpacks it, the
// slot is free.  Workers take chunks in order.
class Copier {
public:
    Copier(Ring &r, std::vector<Chunk> c, hipStream_t s, bool widen)
        : ring_(r), chunks_(std::move(c)), stream_(s), widen_(widen), stage_(chunks_.size(), 0) {}

    // false: no worker could be started, nothing was done
    bool run(hipError_t &result) {
        std::vector<std::thread> pool;
        const size_t n = std::min<size_t>(kThreads, chunks_.size() / 2);
        try {
            pool.reserve(n);
            while (pool.size() < n) pool.emplace_back([this] { work(); });
        } catch (const std::exception &) {
            // fewer threads
        }
        if (pool.empty()) return false;
        hipError_t e = hipSuccess;
        for (size_t i = 0; i < chunks_.size() && e == hipSuccess; ++i) {
            if (i >= size_t(kSlots)) {
                std::unique_lock<std::mutex> lock(mu_);
                cv_.wait(lock, [&] { return stage_[i - kSlots] == 2 || err_ != hipSuccess; });
                if ((e = err_) != hipSuccess) break;
            }
            e = queue(i);
            std::lock_guard<std::mutex> lock(mu_);
            if (e == hipSuccess)
                stage_[i] = 1;
            else
                err_ = e;
            cv_.notify_all();
        }
        for (auto &t : pool) t.join();
        const hipError_t s = hipStreamSynchronize(stream_);  // the ring's slots are free only now
        result = err_ != hipSuccess ? err_ : s;
        return true;
    }

private:
    char *slot(size_t i) { return ring_.base + (i % kSlots) * kSlotBytes; }

    hipError_t queue(size_t i) {
        const Chunk &c = chunks_[i];
        const hipError_t e = hipMemcpyAsync(slot(i), c.dev, c.count * (widen_ ? sizeof(float) : sizeof(double)),
                                            hipMemcpyDeviceToHost, stream_);
        return e != hipSuccess ? e : hipEventRecord(ring_.ev[i % kSlots], stream_);
    }

    void work() {
        (void)hipSetDevice(ring_.device);
        for (;;) {
            size_t i;
            {
                std::unique_lock<std::mutex> lock(mu_);
                i = next_++;
                if (i >= chunks_.size()) return;
                cv_.wait(lock, [&] { return stage_[i] == 1 || err_ != hipSuccess; });
                if (err_ != hipSuccess) return;
            }
            const hipError_t e = hipEventSynchronize(ring_.ev[i % kSlots]);
            if (e == hipSuccess) unpack(chunks_[i], slot(i), widen_);
            std::lock_guard<std::mutex> lock(mu_);
            if (e != hipSuccess) err_ = e;
            stage_[i] = 2;
            cv_.notify_all();
        }
    }

    Ring &ring_;
    std::vector<Chunk> chunks_;
    hipStream_t stream_;
    bool widen_;
    std::mutex mu_;
    std::condition_variable cv_;
    std::vector<char> stage_;  // 0: waiting, 1: queued, 2: unpacked
    size_t next_ = 0;
    hipError_t err_ = hipSuccess;
};

hipError_t direct(const tlbm::CopyPart *parts, int n, bool widen, hipStream_t stream) {
    if (!widen) {
        for (int k = 0; k < n; ++k) {
            const hipError_t e = hipMemcpyAsync(parts[k].host, parts[k].dev, parts[k].count * sizeof(double),
                                                hipMemcpyDeviceToHost, stream);
            if (e != hipSuccess) return e;
        }
        return hipStreamSynchronize(stream);
    }
    size_t most = 0, at = 0;
    for (int k = 0; k < n; ++k) most += parts[k].count;
    std::vector<float> tmp(most);
    for (int k = 0; k < n; at += parts[k++].count) {
        const hipError_t e = hipMemcpyAsync(tmp.data() + at, parts[k].dev, parts[k].count * sizeof(float),
                                            hipMemcpyDeviceToHost, stream);
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(stream);  // tmp is being written
            return e;
        }
    }
    const hipError_t e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return e;
    at = 0;
    for (int k = 0; k < n; at += parts[k++].count)
        unpack({parts[k].dev, parts[k].host, parts[k].count}, tmp.data() + at, true);
    return hipSuccess;
}

}  // namespace

namespace tlbm {

hipError_t copy_to_host(const CopyPart *parts, int n, bool widen, hipStream_t stream, int device) {
    try {
        const size_t esz = widen ? sizeof(float) : sizeof(double);
        size_t bytes = 0;
        for (int k = 0; k < n; ++k) bytes += parts[k].count * esz;
        if (bytes >= (widen ? kRingFrom32 : kRingFrom64)) {
            Ring *taken = nullptr;
            // no pinned memory left, or no thread: the direct copy
            if (take(device, &taken) == hipSuccess) {
                const std::unique_ptr<Ring, void (*)(Ring *)> ring(taken, give);
                hipError_t e = hipSuccess;
                if (Copier(*ring, chunks_of(parts, n, esz), stream, widen).run(e)) return e;
            } else {
                (void)hipGetLastError();
            }
        }
        return direct(parts, n, widen, stream);
    } catch (const std::bad_alloc &) {
        return hipErrorOutOfMemory;
    } catch (const std::exception &) {
        return hipErrorUnknown;
    }
}

void host_copy_retain() {
    std::lock_guard<std::mutex> lock(g_mu);
    ++g_users;
}

void host_copy_release() {
    Ring *drop[kKept] = {};
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (--g_users == 0) std::swap(drop, g_kept);
    }
    for (Ring *r : drop) delete r;
}

}  // namespace tlbm
