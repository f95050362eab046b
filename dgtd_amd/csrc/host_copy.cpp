#include "host_copy.hpp"

#include <algorithm>
#include <array>
#include <condition_variable>
#include <exception>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace dgtd {

namespace {

// Below kDirectBytes on the host a transfer takes the direct path; below
// kThreadBytes the calling thread converts the blocks itself.  Worker threads
// for less than that lose to threads a program keeps spinning (an OpenMP pool
// after a parallel region): 24 instances of 0.05-21 MB, read and converted in
// turn, took 9 ms directly and 12 ms with workers from 8 MB on.
constexpr int64_t kDirectBytes = int64_t(8) << 20;
constexpr int64_t kThreadBytes = int64_t(32) << 20;
constexpr int64_t kBytesPerWorker = int64_t(4) << 20;
constexpr int kMaxWorkers = 8;

constexpr int kMaxBlocks = 12;
constexpr size_t kBytes = size_t(1) << 20;
constexpr size_t kIdleRings = 2;

// Blocks of the ring a transfer uses, and so pins if nobody did before (85 us
// each, and up to 370 us at its first touch): two suffice while the calling
// thread converts (9 MB of FP32 unknowns, first and next download: 259 and 193
// us with two, 587 and 183 with twelve, 440 directly; the first in a process
// took 2-5 ms with twelve), eight and more keep the workers busy (38 MB: 1.7
// ms with eight or twelve, 2.1-2.8 with six or four).
int ring_blocks(int64_t host_bytes)
{
    return host_bytes < kThreadBytes ? 2 : (int)std::min<int64_t>(kMaxBlocks, host_bytes / (int64_t(4) << 20));
}

// Pinned blocks and the events that say when the copy engine is done with them.
struct Ring {
    int device = 0;
    void* block[kMaxBlocks] = {};
    hipEvent_t event[kMaxBlocks] = {};

    explicit Ring(int dev) : device(dev) {}
    Ring(const Ring&) = delete;
    Ring& operator=(const Ring&) = delete;
    ~Ring()
    {
        for (int b = 0; b < kMaxBlocks; ++b) {
            if (block[b]) (void)hipHostFree(block[b]);
            if (event[b]) (void)hipEventDestroy(event[b]);
        }
    }
    hipError_t prepare(int blocks)
    {
        for (int b = 0; b < blocks; ++b) {
            if (!block[b])
                if (const hipError_t e = hipHostMalloc(&block[b], kBytes, hipHostMallocDefault); e != hipSuccess) {
                    block[b] = nullptr;
                    return e;
                }
            if (!event[b])
                if (const hipError_t e = hipEventCreateWithFlags(&event[b], hipEventDisableTiming); e != hipSuccess) {
                    event[b] = nullptr;
                    return e;
                }
        }
        return hipSuccess;
    }
};

// The process's idle rings: at most kIdleRings, freed with the last HostCopy.
// A transfer borrows one for its duration, so transfers of any threads, on one
// operator too, never share blocks.
class Rings {
public:
    static Rings& get()
    {
        static Rings* r = new Rings;  // outlives every HostCopy
        return *r;
    }
    void add_owner()
    {
        std::lock_guard<std::mutex> lk(mu_);
        ++owners_;
    }
    void drop_owner()
    {
        std::array<std::unique_ptr<Ring>, kIdleRings> last;
        std::lock_guard<std::mutex> lk(mu_);
        if (--owners_ == 0) last.swap(idle_);
    }
    std::unique_ptr<Ring> take()
    {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return nullptr;
        {
            std::lock_guard<std::mutex> lk(mu_);
            for (auto& r : idle_)
                if (r && r->device == dev) return std::move(r);
        }
        return std::make_unique<Ring>(dev);
    }
    void give(std::unique_ptr<Ring> r)
    {
        std::lock_guard<std::mutex> lk(mu_);
        for (auto& slot : idle_)
            if (!slot) {
                slot = std::move(r);
                return;
            }
    }

private:
    std::mutex mu_;
    std::array<std::unique_ptr<Ring>, kIdleRings> idle_;
    int owners_ = 0;
};

// A ring for one transfer, with that many blocks (NULL: no pinned memory left).
class Borrowed {
public:
    explicit Borrowed(int blocks) : ring_(Rings::get().take())
    {
        if (ring_ && ring_->prepare(blocks) != hipSuccess) {
            (void)hipGetLastError();
            ring_.reset();
        }
    }
    ~Borrowed()
    {
        if (ring_) Rings::get().give(std::move(ring_));
    }
    Ring* get() const { return ring_.get(); }

private:
    std::unique_ptr<Ring> ring_;
};

// Progress of the blocks of one transfer, passed between the calling thread
// (which drives the copy engine) and the workers (which convert).
struct Progress {
    std::mutex mu;
    std::condition_variable cv;
    int64_t next = 0;             // next block a worker takes
    int64_t open = 0;             // blocks [0, open) may be taken
    std::vector<char> converted;  // per block
    bool stop = false;

    void set_open(int64_t n)
    {
        std::lock_guard<std::mutex> lk(mu);
        open = n;
        cv.notify_all();
    }
    void wait_converted(int64_t i)
    {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return converted[i] != 0; });
    }
};

// Worker threads that convert every block once it is open; joined (after a
// stop, when the transfer failed) before the progress they share goes away.
class Workers {
public:
    template <typename F>
    Workers(Progress& p, int count, int64_t blocks, F convert) : p_(p)
    {
        threads_.reserve(count);
        for (int w = 0; w < count; ++w) {
            try {
                threads_.emplace_back([&p, blocks, convert] {
                    for (;;) {
                        int64_t i;
                        {
                            std::unique_lock<std::mutex> lk(p.mu);
                            p.cv.wait(lk, [&] { return p.stop || p.next >= blocks || p.next < p.open; });
                            if (p.stop || p.next >= blocks) return;
                            i = p.next++;
                        }
                        convert(i);
                        std::lock_guard<std::mutex> lk(p.mu);
                        p.converted[i] = 1;
                        p.cv.notify_all();
                    }
                });
            } catch (const std::exception&) {
                break;  // no more threads or memory for one: those that started do the work
            }
        }
    }
    ~Workers()
    {
        {
            std::lock_guard<std::mutex> lk(p_.mu);
            p_.stop = true;
            p_.cv.notify_all();
        }
        for (auto& t : threads_) t.join();
    }
    bool empty() const { return threads_.empty(); }

private:
    Progress& p_;
    std::vector<std::thread> threads_;
};

int worker_count(int64_t bytes)
{
    const int hw = (int)std::max(1u, std::thread::hardware_concurrency());
    return (int)std::max<int64_t>(1, std::min<int64_t>({kMaxWorkers, hw, bytes / kBytesPerWorker}));
}

template <typename T>
hipError_t direct_to_host(const T* d, double* h, int64_t n, hipStream_t s)
{
    hipError_t e;
    if constexpr (sizeof(T) == sizeof(double)) {
        e = hipMemcpyAsync(h, d, sizeof(double) * n, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    } else {
        std::vector<T> tmp(n);
        e = hipMemcpyAsync(tmp.data(), d, sizeof(T) * n, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e == hipSuccess) std::copy(tmp.begin(), tmp.end(), h);
        return e;
    }
}

template <typename T>
hipError_t direct_to_device(const double* h, T* d, int64_t n, hipStream_t s)
{
    if constexpr (sizeof(T) == sizeof(double)) {
        return hipMemcpyAsync(d, h, sizeof(double) * n, hipMemcpyHostToDevice, s);
    } else {
        std::vector<T> tmp(h, h + n);
        const hipError_t e = hipMemcpyAsync(d, tmp.data(), sizeof(T) * n, hipMemcpyHostToDevice, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    }
}

}  // namespace

HostCopy::HostCopy() { Rings::get().add_owner(); }
HostCopy::~HostCopy() { Rings::get().drop_owner(); }

template <typename T>
hipError_t HostCopy::to_host(const T* d, double* h, int64_t n, hipStream_t s)
{
    const int64_t bytes = n * (int64_t)sizeof(double);
    if (bytes < kDirectBytes) return direct_to_host(d, h, n, s);
    const int nring = ring_blocks(bytes);
    const Borrowed borrowed(nring);
    Ring* const ring = borrowed.get();
    if (!ring) return direct_to_host(d, h, n, s);
    const int64_t per = (int64_t)(kBytes / sizeof(T)), blocks = (n + per - 1) / per;
    auto copy = [&](int64_t i) {
        const int b = (int)(i % nring);
        hipError_t e = hipMemcpyAsync(ring->block[b], d + i * per, sizeof(T) * std::min(per, n - i * per),
                                      hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipEventRecord(ring->event[b], s);
    };
    auto convert = [=](int64_t i) {
        const T* src = static_cast<const T*>(ring->block[i % nring]);
        std::copy(src, src + std::min(per, n - i * per), h + i * per);
    };
    // copies run ahead of the conversions by the ring's length
    hipError_t e = hipSuccess;
    int64_t issued = 0;
    if (bytes < kThreadBytes) {
        for (int64_t i = 0; i < blocks && e == hipSuccess; ++i) {
            while (e == hipSuccess && issued < std::min<int64_t>(blocks, i + nring)) e = copy(issued++);
            if (e == hipSuccess) e = hipEventSynchronize(ring->event[i % nring]);
            if (e == hipSuccess) convert(i);
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(s);
        return e;
    }
    Progress p;
    p.converted.assign(blocks, 0);
    Workers workers(p, worker_count(bytes), blocks, convert);
    if (workers.empty()) return direct_to_host(d, h, n, s);
    for (int64_t i = 0; i < blocks && e == hipSuccess; ++i) {
        while (e == hipSuccess && issued < blocks && issued < i + nring) {
            if (issued >= nring) {
                std::unique_lock<std::mutex> lk(p.mu);
                if (!p.converted[issued - nring] && issued > i) break;  // refill later
                p.cv.wait(lk, [&] { return p.converted[issued - nring] != 0; });
            }
            e = copy(issued);
            if (e == hipSuccess) ++issued;
        }
        if (e == hipSuccess) e = hipEventSynchronize(ring->event[i % nring]);
        if (e == hipSuccess) p.set_open(i + 1);
    }
    for (int64_t i = std::max<int64_t>(0, blocks - nring); i < blocks && e == hipSuccess; ++i) p.wait_converted(i);
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // no copy into the ring outlives the call
    return e;
}

template <typename T>
hipError_t HostCopy::to_device(const double* h, T* d, int64_t n, hipStream_t s)
{
    // FP64: nothing to convert, and the source's pages exist (a plain copy of 10-250
    // MB is as fast or up to a third faster than the ring)
    const int64_t bytes = n * (int64_t)sizeof(double);
    if (bytes < kDirectBytes || sizeof(T) == sizeof(double)) return direct_to_device(h, d, n, s);
    const int nring = ring_blocks(bytes);
    const Borrowed borrowed(nring);
    Ring* const ring = borrowed.get();
    if (!ring) return direct_to_device(h, d, n, s);
    const int64_t per = (int64_t)(kBytes / sizeof(T)), blocks = (n + per - 1) / per;
    auto copy = [&](int64_t i) {
        const int b = (int)(i % nring);
        hipError_t e = hipMemcpyAsync(d + i * per, ring->block[b], sizeof(T) * std::min(per, n - i * per),
                                      hipMemcpyHostToDevice, s);
        return e != hipSuccess ? e : hipEventRecord(ring->event[b], s);
    };
    auto convert = [=](int64_t i) {
        const double* src = h + i * per;
        std::copy(src, src + std::min(per, n - i * per), static_cast<T*>(ring->block[i % nring]));
    };
    hipError_t e = hipSuccess;
    if (bytes < kThreadBytes) {
        for (int64_t i = 0; i < blocks && e == hipSuccess; ++i) {
            if (i >= nring) e = hipEventSynchronize(ring->event[i % nring]);
            if (e != hipSuccess) break;
            convert(i);
            e = copy(i);
        }
        const hipError_t w = hipStreamSynchronize(s);
        return e != hipSuccess ? e : w;
    }
    Progress p;
    p.converted.assign(blocks, 0);
    p.open = std::min<int64_t>(blocks, nring);
    Workers workers(p, worker_count(bytes), blocks, convert);
    if (workers.empty()) return direct_to_device(h, d, n, s);
    for (int64_t i = 0; i < blocks && e == hipSuccess; ++i) {
        p.wait_converted(i);
        e = copy(i);
        // half a ring behind, the block is free again
        const int64_t done = i - nring / 2;
        if (e == hipSuccess && done >= 0) {
            e = hipEventSynchronize(ring->event[done % nring]);
            if (e == hipSuccess) p.set_open(std::min<int64_t>(blocks, done + 1 + nring));
        }
    }
    const hipError_t w = hipStreamSynchronize(s);
    return e != hipSuccess ? e : w;
}

template hipError_t HostCopy::to_host<double>(const double*, double*, int64_t, hipStream_t);
template hipError_t HostCopy::to_host<float>(const float*, double*, int64_t, hipStream_t);
template hipError_t HostCopy::to_device<double>(const double*, double*, int64_t, hipStream_t);
template hipError_t HostCopy::to_device<float>(const double*, float*, int64_t, hipStream_t);

}  // namespace dgtd
