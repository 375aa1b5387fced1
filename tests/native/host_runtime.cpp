#include "host_runtime.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <thread>

struct ihipStream_t {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> q;
    unsigned long long queued = 0, run = 0;
    bool stop = false;
    std::thread th{[this] { loop(); }};
    void loop();
    void put(std::function<void()> f) {
        {
            std::lock_guard<std::mutex> g(mu);
            q.push_back(std::move(f));
            queued++;
        }
        cv.notify_all();
    }
    void drain() {
        std::unique_lock<std::mutex> g(mu);
        const unsigned long long upto = queued;
        cv.wait(g, [&] { return run >= upto; });
    }
    bool idle() {
        std::lock_guard<std::mutex> g(mu);
        return run == queued;
    }
    ~ihipStream_t() {
        {
            std::lock_guard<std::mutex> g(mu);
            stop = true;
        }
        cv.notify_all();
        th.join();
    }
};
struct ihipEvent_t {
    std::mutex mu;
    std::condition_variable cv;
    unsigned long long recorded = 0, done = 0;
};

namespace host_runtime {
Faults faults;
size_t device_limit = ~size_t{0};
namespace {
std::mutex mu;
std::map<char*, size_t> device, pinned;
size_t used = 0;
std::atomic<int> n_copies{0}, n_mallocs{0}, delay{0};
bool fails(int& n) {
    std::lock_guard<std::mutex> g(mu);
    return n > 0 && --n == 0;
}
bool inside(const std::map<char*, size_t>& m, const void* p) {
    auto it = m.upper_bound(static_cast<char*>(const_cast<void*>(p)));
    return it != m.begin() && (--it, static_cast<const char*>(p) < it->first + it->second);
}
}  // namespace
void enqueue(ihipStream_t* s, std::function<void()> f) { s->put(std::move(f)); }
size_t device_bytes() {
    std::lock_guard<std::mutex> g(mu);
    return used;
}
int copies() { return n_copies; }
int mallocs() { return n_mallocs; }
void stream_delay_us(int us) { delay = us; }
}  // namespace host_runtime
using namespace host_runtime;

void ihipStream_t::loop() {
    std::unique_lock<std::mutex> g(mu);
    for (;;) {
        cv.wait(g, [&] { return stop || !q.empty(); });
        if (q.empty()) return;
        auto f = std::move(q.front());
        q.pop_front();
        g.unlock();
        if (delay) std::this_thread::sleep_for(std::chrono::microseconds(delay));
        f();
        f = nullptr;
        g.lock();
        run++;
        cv.notify_all();
    }
}

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> g(mu);
    n_mallocs++;
    if (used + n > device_limit) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    std::memset(*p, 0xA5, n);
    device[static_cast<char*>(*p)] = n;
    used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    std::lock_guard<std::mutex> g(mu);
    const auto it = device.find(static_cast<char*>(p));
    if (it == device.end()) std::abort();  // freed twice, or never allocated
    used -= it->second;
    device.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    std::lock_guard<std::mutex> g(mu);
    if (faults.pinned) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    pinned[static_cast<char*>(*p)] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> g(mu);
    pinned.erase(static_cast<char*>(p));
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    *d = h;
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    std::lock_guard<std::mutex> g(mu);
    const bool d = inside(device, p), h = inside(pinned, p);
    a->type = d ? hipMemoryTypeDevice : h ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return d || h ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
    n_copies++;
    if (fails(faults.copy)) return hipErrorUnknown;
    s->put([=] { std::memcpy(dst, src, n); });
    return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind) {
    std::memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
    s->put([=] { std::memset(p, v, n); });
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = new ihipStream_t;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    s->drain();
    delete s;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    s->drain();
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) { return s->idle() ? hipSuccess : hipErrorNotReady; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = new ihipEvent_t;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    {
        std::unique_lock<std::mutex> g(e->mu);
        e->cv.wait(g, [&] { return e->done == e->recorded; });
    }
    delete e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    unsigned long long k;
    {
        std::lock_guard<std::mutex> g(e->mu);
        k = ++e->recorded;
    }
    s->put([=] {
        std::lock_guard<std::mutex> g(e->mu);
        e->done = k;
        e->cv.notify_all();
    });
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (fails(faults.event_sync)) return hipErrorUnknown;
    std::unique_lock<std::mutex> g(e->mu);
    e->cv.wait(g, [&] { return e->done == e->recorded; });
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    std::lock_guard<std::mutex> g(e->mu);
    return e->done == e->recorded ? hipSuccess : hipErrorNotReady;
}
}
