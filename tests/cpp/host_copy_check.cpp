// Host part of the state transfers (dgtd_amd/csrc/host_copy.cpp) on the CPU,
// over a stand-in for the HIP calls it makes: one copy engine thread runs the
// asynchronous copies and event records of every stream in the order of their
// calls, some time after them, so a missing wait reads or overwrites a block
// too early.  "device" memory is host memory.  Run by tests/test_host_copy.py;
// prints the failing check, exit status 0 when all pass.
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "../../dgtd_amd/csrc/host_copy.hpp"

// ---- allocation failures: the countdown-th allocation of this thread throws ----
namespace {
thread_local int g_fail_new = -1;
std::atomic<int64_t> g_pinned{0}, g_pinned_peak{0};
std::atomic<int> g_fail_pinned{-1};  // pinned allocations that still succeed (-1: all)
std::atomic<int> g_fail_copy{-1};    // copies that still succeed (-1: all)
}  // namespace

void* operator new(size_t n)
{
    if (g_fail_new >= 0 && g_fail_new-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

// ---- stand-in for the HIP runtime ----
namespace {

struct Engine {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> queue;
    int64_t posted = 0, done = 0;
    bool quit = false;
    std::thread th;
    Engine() : th([this] { run(); }) {}
    ~Engine()
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            quit = true;
            cv.notify_all();
        }
        th.join();
    }
    void run()
    {
        for (;;) {
            std::function<void()> f;
            {
                std::unique_lock<std::mutex> lk(mu);
                cv.wait(lk, [&] { return quit || !queue.empty(); });
                if (queue.empty()) return;
                f = std::move(queue.front());
                queue.pop_front();
            }
            std::this_thread::sleep_for(std::chrono::microseconds(60));
            f();
            std::lock_guard<std::mutex> lk(mu);
            ++done;
            cv.notify_all();
        }
    }
    int64_t post(std::function<void()> f)
    {
        const int keep = g_fail_new;  // the stand-in's own allocations do not fail
        g_fail_new = -1;
        int64_t id;
        {
            std::lock_guard<std::mutex> lk(mu);
            queue.push_back(std::move(f));
            id = ++posted;
            cv.notify_all();
        }
        g_fail_new = keep;
        return id;
    }
    void wait(int64_t id)
    {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return done >= id; });
    }
    int64_t last()
    {
        std::lock_guard<std::mutex> lk(mu);
        return posted;
    }
};

Engine& engine()
{
    static Engine* e = new Engine;  // outlives every static
    return *e;
}

struct Event {
    std::atomic<int64_t> id{0};
};

std::mutex g_sizes_mu;
std::map<void*, size_t>& sizes()
{
    static auto* m = new std::map<void*, size_t>;
    return *m;
}

}  // namespace

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    if (g_fail_pinned >= 0 && g_fail_pinned-- <= 0) {
        g_fail_pinned = 0;
        return hipErrorOutOfMemory;
    }
    *p = std::malloc(n);
    const int keep = g_fail_new;
    g_fail_new = -1;
    {
        std::lock_guard<std::mutex> lk(g_sizes_mu);
        sizes()[*p] = n;
    }
    g_fail_new = keep;
    const int64_t now = g_pinned += (int64_t)n;
    if (now > g_pinned_peak) g_pinned_peak = now;
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::lock_guard<std::mutex> lk(g_sizes_mu);
    g_pinned -= (int64_t)sizes()[p];
    sizes().erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    const int keep = g_fail_new;
    g_fail_new = -1;
    *e = reinterpret_cast<hipEvent_t>(new Event);
    g_fail_new = keep;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    delete reinterpret_cast<Event*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    reinterpret_cast<Event*>(e)->id = engine().post([] {});
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    engine().wait(reinterpret_cast<Event*>(e)->id);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    engine().wait(engine().last());
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    if (g_fail_copy >= 0 && g_fail_copy-- <= 0) {
        g_fail_copy = 0;
        return hipErrorInvalidValue;
    }
    engine().post([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
}

namespace {

int g_failures = 0;
void check(bool ok, const std::string& what)
{
    if (ok) return;
    std::printf("FAILED: %s\n", what.c_str());
    ++g_failures;
}

template <typename T>
std::vector<T> device_values(int64_t n, int seed)
{
    std::vector<T> d(n);
    for (int64_t i = 0; i < n; ++i) d[i] = (T)(int32_t)((uint32_t)(i * 2654435761u) ^ (uint32_t)(seed * 40503));
    return d;
}

template <typename T>
bool same(const std::vector<T>& d, const std::vector<double>& h)
{
    for (size_t i = 0; i < d.size(); ++i)
        if ((double)d[i] != h[i]) return false;
    return true;
}

// doubles on the host: below 8 MB, 8-32 MB, above 32 MB, none whole blocks
const int64_t kSizes[] = {1, 1000, 1048575, 1048577, 2500001, 4194304, 5000003, 9000001};

template <typename T>
void round_trips()
{
    dgtd::HostCopy c;
    for (int64_t n : kSizes)
        for (int rep = 0; rep < 2; ++rep) {
            const auto d = device_values<T>(n, rep + 1);
            std::vector<double> h(n, -1.0);
            check(c.to_host(d.data(), h.data(), n, nullptr) == hipSuccess && same(d, h),
                  "to_host of " + std::to_string(n));
            std::vector<T> back(n, T(-1));
            check(c.to_device(h.data(), back.data(), n, nullptr) == hipSuccess, "to_device");
            (void)hipStreamSynchronize(nullptr);
            check(back == d, "to_device of " + std::to_string(n));
        }
}

// An allocation that fails anywhere in a transfer gives an exception or, where
// the work can go on, the right values; never an abort.
void failing_allocations()
{
    const int64_t n = 5000003;
    const auto d = device_values<float>(n, 3);
    for (int k = 0; k < 24; ++k) {
        dgtd::HostCopy c;
        std::vector<double> h(n, -1.0);
        bool threw = false;
        hipError_t e = hipSuccess;
        g_fail_new = k;
        try {
            e = c.to_host(d.data(), h.data(), n, nullptr);
        } catch (const std::bad_alloc&) {
            threw = true;
        }
        g_fail_new = -1;
        (void)hipStreamSynchronize(nullptr);
        check(threw || (e == hipSuccess && same(d, h)), "to_host with allocation " + std::to_string(k) + " failing");
        std::vector<float> back(n);
        threw = false;
        g_fail_new = k;
        const std::vector<double>& src = h;
        try {
            e = c.to_device(src.data(), back.data(), n, nullptr);
        } catch (const std::bad_alloc&) {
            threw = true;
        }
        g_fail_new = -1;
        (void)hipStreamSynchronize(nullptr);
        check(threw || e == hipSuccess, "to_device with allocation " + std::to_string(k) + " failing");
    }
}

// A copy that fails is reported, and the next transfer is right.
void failing_copies()
{
    for (int64_t n : {int64_t(2500001), int64_t(5000003)})
        for (int k : {0, 1, 3, 7}) {
            const auto d = device_values<float>(n, 4);
            dgtd::HostCopy c;
            std::vector<double> h(n, -1.0);
            g_fail_copy = k;
            check(c.to_host(d.data(), h.data(), n, nullptr) != hipSuccess, "failed copy to the host reported");
            g_fail_copy = -1;
            check(c.to_host(d.data(), h.data(), n, nullptr) == hipSuccess && same(d, h), "to_host after a failure");
            std::vector<float> back(n);
            g_fail_copy = k;
            check(c.to_device(h.data(), back.data(), n, nullptr) != hipSuccess, "failed copy to the device reported");
            g_fail_copy = -1;
            check(c.to_device(h.data(), back.data(), n, nullptr) == hipSuccess, "to_device after a failure");
            (void)hipStreamSynchronize(nullptr);
            check(back == d, "to_device after a failure");
        }
}

void no_pinned_memory()
{
    for (int64_t n : {int64_t(2500001), int64_t(5000003)})
        for (int k : {0, 2}) {
            const auto d = device_values<float>(n, 5);
            dgtd::HostCopy c;
            std::vector<double> h(n, -1.0);
            g_fail_pinned = k;
            check(c.to_host(d.data(), h.data(), n, nullptr) == hipSuccess && same(d, h), "to_host without pinned memory");
            g_fail_pinned = -1;
        }
}

// Transfers of several threads, through one object and through several: no
// block is shared, and at most 24 MB stay pinned between them.
void threads()
{
    std::vector<dgtd::HostCopy> c(3);
    for (const bool one : {true, false}) {
        std::vector<std::thread> th;
        for (int t = 0; t < 3; ++t)
            th.emplace_back([&, t] {
                for (int64_t n : {int64_t(2500001), int64_t(5000003)}) {
                    const auto d = device_values<float>(n, 10 + t);
                    std::vector<double> h(n, -1.0);
                    check(c[one ? 0 : t].to_host(d.data(), h.data(), n, nullptr) == hipSuccess && same(d, h),
                          "to_host of one of three threads");
                    std::vector<float> back(n);
                    check(c[one ? 0 : t].to_device(h.data(), back.data(), n, nullptr) == hipSuccess && back == d,
                          "to_device of one of three threads");
                }
            });
        for (auto& t : th) t.join();
        check(g_pinned <= 24 << 20, "pinned memory kept");
    }
}

// What a transfer pins: nothing below 8 MB or for an FP64 upload, 2 MB below
// 32 MB, at most 12 MB.
void pinned_memory()
{
    auto pins = [](int64_t n, auto value, bool up) {
        using T = decltype(value);
        std::vector<T> d(n);
        std::vector<double> h(n);
        dgtd::HostCopy c;
        check((up ? c.to_device(h.data(), d.data(), n, nullptr) : c.to_host(d.data(), h.data(), n, nullptr)) == hipSuccess,
              "transfer");
        (void)hipStreamSynchronize(nullptr);
        return (int64_t)g_pinned;
    };
    check(pins(1000000, 0.0f, false) == 0 && pins(1000000, 0.0, true) == 0, "nothing below 8 MB");
    check(pins(1500000, 0.0, true) == 0 && pins(9000001, 0.0, true) == 0, "nothing for an FP64 upload");
    for (const bool up : {false, true}) {
        check(pins(1500000, 0.0f, up) <= 2 << 20 && pins(4000000, 0.0f, up) <= 2 << 20, "2 MB below 32 MB");
        check(pins(9000001, 0.0f, up) <= 12 << 20 && pins(20000000, 0.0f, up) <= 12 << 20, "12 MB");
    }
    check(pins(4000000, 0.0, false) <= 2 << 20, "2 MB below 32 MB, FP64");
}

}  // namespace

int main(int argc, char** argv)
{
    const std::map<std::string, std::function<void()>> tests = {
        {"round_trips", [] { round_trips<float>(); round_trips<double>(); }},
        {"failing_allocations", failing_allocations},
        {"failing_copies", failing_copies},
        {"no_pinned_memory", no_pinned_memory},
        {"threads", threads},
        {"pinned_memory", pinned_memory},
    };
    const auto t = argc > 1 ? tests.find(argv[1]) : tests.end();
    if (t == tests.end()) return 2;
    t->second();
    check(g_pinned == 0, "pinned memory given back");
    if (g_failures == 0) std::printf("OK\n");
    std::fflush(stdout);
    return g_failures ? 1 : 0;
}
