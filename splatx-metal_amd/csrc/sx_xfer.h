// sx_xfer.h — copies between a caller's pageable host memory and the device, through a ring of pinned chunks.
//
// The runtime stages a pageable copy itself, one array and one chunk after another on the calling thread:
// measured 26 GB/s to the device and 16 GB/s back (708 MB, the rows and moments of 1 M Gaussians at SH3: 27 and
// 43 ms), where the link moves 56 GB/s, one thread's memcpy 29 GB/s and four threads' 56 GB/s; and 18 copies of
// a few kB each cost 0.5 ms. Here the chunks of a whole list of arrays run through one ring: neighbouring
// arrays share chunks, and a few threads copy between the caller's memory and the pinned chunks while the link
// moves others: the 708 MB take 18.3 ms to the device and 16 back.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>
#include <memory>
#include <vector>

namespace sxh {

// One array of a transfer, and the stream work that belongs to it: `stage` is called on the calling thread before
// the first of its device-to-host copies is queued (the kernel that packs it), or after the last of its
// host-to-device copies is (the kernel that unpacks it). May be empty.
struct XferItem {
    void* host = nullptr;
    void* dev = nullptr;
    size_t bytes = 0;
    std::function<void()> stage;
};

// The ring and its threads, made on first use and given back with the object: 32 MiB of pinned memory, at most
// four threads, which sleep between transfers. Without that memory the runtime copies the arrays. One transfer at a
// time (a lock held for its duration).
class HostXfer {
  public:
    explicit HostXfer(int device);
    ~HostXfer();
    HostXfer(const HostXfer&) = delete;
    HostXfer& operator=(const HostXfer&) = delete;

    // The items' copies on `s`, in order. A run of items that lie back to back in device memory is one block:
    // to the host all its stages come before its copies, to the device after them; blocks may use the same
    // device memory (the stream orders them). to_device returns when the host memory of the arrays it staged has
    // been read (their copies and the stages may still run; an array that the runtime copies is read once the
    // stream gets there); to_host when the host memory is written and the stream has drained.
    void to_device(const std::vector<XferItem>& items, hipStream_t s);
    void to_host(const std::vector<XferItem>& items, hipStream_t s);

  private:
    struct Impl;
    std::unique_ptr<Impl> p_;
};

}  // namespace sxh
