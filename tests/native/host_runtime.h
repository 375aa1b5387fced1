// A HIP runtime of host memory for tests of the library's host code without a GPU: "device" memory is malloc'd, a
// stream is a thread that runs what is queued on it in order (so a copy is as asynchronous as on a GPU), and a test can
// limit the memory there is and make calls fail.
#pragma once

#include <cstddef>
#include <functional>

struct ihipStream_t;

namespace host_runtime {
void enqueue(ihipStream_t* s, std::function<void()> f);  // a kernel: f runs in stream order
// Calls from here on: the n-th (1 = the next) call of that kind fails, once; 0: none does.
struct Faults {
    int copy = 0;         // hipMemcpyAsync
    int event_sync = 0;   // hipEventSynchronize
    bool pinned = false;  // every hipHostMalloc fails
};
extern Faults faults;
extern size_t device_limit;   // bytes that hipMalloc hands out in all
size_t device_bytes();        // bytes in use
int copies(), mallocs();      // hipMemcpyAsync and hipMalloc calls so far
void stream_delay_us(int us);  // before each thing a stream runs
}  // namespace host_runtime
