// xfer.cpp — the pinned ring of sx_xfer.h.
#include "sx_xfer.h"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <mutex>
#include <system_error>
#include <thread>

#include "sx_host.h"
#include "sx_kernels.h"

namespace sxh {
namespace {

constexpr size_t kMiB = size_t{1} << 20;
constexpr int kSlots = 8;
constexpr int kThreads = 4;
// Chunks: 4 MiB from 32 MiB on (75 us of the link each; queueing one takes about 15 us of the calling thread), 1 MiB
// below, 512 KiB below 2 MiB. Measured to the host: 256 MiB 15.9 ms by the runtime, 6.7 in chunks of 2 MiB, 5.9 of
// 4 MiB; 4.4 MB 0.27 ms by the runtime, 0.25 in chunks of 512 KiB, 0.21 of 1 MiB, and into pages not touched before
// 1.06, 0.55 and 0.62 ms; 100 kB 50 us and 20.
constexpr size_t kChunk = 4 * kMiB;
size_t chunk_bytes(size_t total) { return total >= 32 * kMiB ? kChunk : total >= 2 * kMiB ? kMiB : kMiB / 2; }
// Below this the calling thread copies alone: waking the others takes longer than they would save (with threads of
// their own for 128-KiB chunks, 1.2 MB took 0.56 ms instead of 0.27).
constexpr size_t kThreadedBytes = 2 * kMiB;
// Below this the chunks are moved by a kernel on the stream: a copy engine waits about 10 us for the kernel before it
// and the kernel after it for the engine.
constexpr size_t kKernelBytes = 8 * kMiB;
// A single array to the device between these is the runtime's own copy, which reads the caller's pages in place there
// (1.2 MB: 61 us against 74, 4.4 MB: 142 against 171-208, 13 MB: 378 against 438, 64 MB: 2.45 ms against 1.78).
constexpr size_t kDirectUpLo = kMiB, kDirectUpHi = 24 * kMiB;

// Whether the runtime knows the memory (pinned, managed or device memory): it then copies directly.
bool known_memory(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

// A part of one array within a chunk, at `at` bytes from the chunk's start.
struct Piece {
    char* host;
    size_t at, bytes;
};
struct Chunk {
    char* dev;
    size_t bytes;
    std::vector<Piece> pieces;
};
// Items back to back in device memory, as chunks; or one item the runtime copies (no chunks).
struct Block {
    size_t first, last;  // items [first, last)
    std::vector<Chunk> chunks;
};

std::vector<Block> blocks_of(const std::vector<XferItem>& items, size_t step, bool up, bool ring) {
    std::vector<Block> out;
    for (size_t k = 0; k < items.size();) {
        if (!ring || items[k].bytes == 0 || known_memory(items[k].host)) {
            out.push_back({k, k + 1, {}});
            k++;
            continue;
        }
        Block b{k, k + 1, {}};
        while (b.last < items.size() && items[b.last].bytes > 0 &&
               static_cast<char*>(items[b.last].dev) ==
                   static_cast<char*>(items[b.last - 1].dev) + items[b.last - 1].bytes &&
               !known_memory(items[b.last].host))
            b.last++;
        if (up && b.last == b.first + 1 && items[k].bytes >= kDirectUpLo && items[k].bytes < kDirectUpHi) {
            out.push_back(std::move(b));
            k++;
            continue;
        }
        for (size_t q = b.first; q < b.last; q++)
            for (size_t at = 0; at < items[q].bytes;) {
                if (b.chunks.empty() || b.chunks.back().bytes == step)
                    b.chunks.push_back({static_cast<char*>(items[q].dev) + at, 0, {}});
                Chunk& c = b.chunks.back();
                const size_t n = std::min(step - c.bytes, items[q].bytes - at);
                c.pieces.push_back({static_cast<char*>(items[q].host) + at, c.bytes, n});
                c.bytes += n;
                at += n;
            }
        k = b.last;
        out.push_back(std::move(b));
    }
    return out;
}

size_t total_bytes(const std::vector<XferItem>& items) {
    size_t n = 0;
    for (const auto& it : items) n += it.bytes;
    return n;
}

}  // namespace

struct HostXfer::Impl {
    // The host copies of one chunk, to the host after the slot's device copy.
    struct Job {
        const Chunk* c;
        int slot;
        bool to_host;
    };
    int device;
    std::mutex call;  // one transfer at a time
    std::mutex mu;    // everything below
    std::condition_variable work, changed;
    std::deque<Job> jobs;
    bool busy[kSlots] = {};  // a job of the slot is queued or running
    bool stop = false, threaded = false;
    hipError_t err = hipSuccess;
    std::vector<std::thread> threads;
    char* ring = nullptr;
    hipEvent_t ev[kSlots] = {};
    bool copying[kSlots] = {};  // a copy from the slot was queued and not seen done (calling thread only)
    int next = 0;               // the slot of the next chunk (calling thread only)

    explicit Impl(int d) : device(d) {}

    // The ring and its events; false where there is no pinned memory for it (asked for again with the next transfer).
    bool make_ring() {
        char* r = nullptr;
        bool ok = hipHostMalloc(reinterpret_cast<void**>(&r), kChunk * kSlots, hipHostMallocMapped) == hipSuccess;
        for (auto& e : ev)
            if (ok && !e) ok = hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            if (r) (void)hipHostFree(r);
            return false;
        }
        ring = r;
        return true;
    }

    // Before a transfer: whether there is a ring (without one the runtime copies every array).
    bool start(size_t total) {
        {
            std::lock_guard<std::mutex> g(mu);
            err = hipSuccess;  // (a transfer that threw may have left one; no job runs between transfers)
        }
        if (!ring && !make_ring()) return false;
        threaded = total >= kThreadedBytes;
        if (threaded && threads.empty()) {
            const int n = std::min<int>(kThreads, std::max(1u, std::thread::hardware_concurrency() / 2));
            try {
                while (static_cast<int>(threads.size()) < n) threads.emplace_back([this] { loop(); });
            } catch (const std::system_error&) {  // (the calling thread takes jobs as well)
            }
        }
        return true;
    }

    ~Impl() {
        {
            std::lock_guard<std::mutex> g(mu);
            stop = true;
        }
        work.notify_all();
        for (auto& t : threads) t.join();
        for (int k = 0; k < kSlots; k++) {
            if (copying[k]) (void)hipEventSynchronize(ev[k]);
            if (ev[k]) (void)hipEventDestroy(ev[k]);
        }
        if (ring) (void)hipHostFree(ring);
    }

    // One chunk between the device and the slot, either way.
    void copy_chunk(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, size_t total, hipStream_t s) {
        if (total >= kKernelBytes) {
            SXH_HIP(hipMemcpyAsync(dst, src, bytes, kind, s));
        } else {
            sxk::copy_bytes(dst, src, bytes, s);
            SXH_HIP(hipGetLastError());
        }
    }

    char* chunk(int slot) { return ring + static_cast<size_t>(slot) * kChunk; }

    // Runs the front job; `lk` holds mu and does so again afterwards.
    void run_one(std::unique_lock<std::mutex>& lk) {
        const Job j = jobs.front();
        jobs.pop_front();
        lk.unlock();
        const hipError_t e = j.to_host ? hipEventSynchronize(ev[j.slot]) : hipSuccess;
        if (e == hipSuccess)
            for (const Piece& p : j.c->pieces) {
                if (j.to_host) std::memcpy(p.host, chunk(j.slot) + p.at, p.bytes);
                else std::memcpy(chunk(j.slot) + p.at, p.host, p.bytes);
            }
        lk.lock();
        if (e != hipSuccess && err == hipSuccess) err = e;
        busy[j.slot] = false;
        changed.notify_all();
    }

    void loop() {
        (void)hipSetDevice(device);
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            work.wait(lk, [&] { return stop || !jobs.empty(); });
            if (stop) return;
            run_one(lk);
        }
    }

    void push(const Job& j) {
        {
            std::lock_guard<std::mutex> g(mu);
            busy[j.slot] = true;
            jobs.push_back(j);
        }
        if (threaded) work.notify_one();
    }

    // Until the slot's job is done; the calling thread takes queued jobs meanwhile.
    void wait_slot(int slot) {
        std::unique_lock<std::mutex> lk(mu);
        while (busy[slot]) {
            if (!jobs.empty()) run_one(lk);
            else changed.wait(lk);
        }
    }

    // Until no job is queued or running (also after an error, before the caller's memory goes away).
    void drain() {
        for (int k = 0; k < kSlots; k++) wait_slot(k);
    }

    void check() {
        hipError_t e;
        {
            std::lock_guard<std::mutex> g(mu);
            e = err;
            err = hipSuccess;
        }
        SXH_HIP(e);
    }

    void settle(int slot) {
        if (copying[slot]) SXH_HIP(hipEventSynchronize(ev[slot]));
        copying[slot] = false;
    }
};

HostXfer::HostXfer(int device) : p_(new Impl(device)) {}
HostXfer::~HostXfer() = default;

void HostXfer::to_device(const std::vector<XferItem>& items, hipStream_t s) {
    Impl& x = *p_;
    const size_t total = total_bytes(items);
    std::lock_guard<std::mutex> one(x.call);
    const bool ring = x.start(total);
    const std::vector<Block> blocks = blocks_of(items, chunk_bytes(total), true, ring);
    std::vector<const Chunk*> order;  // the chunks of every block
    for (const Block& b : blocks)
        for (const Chunk& c : b.chunks) order.push_back(&c);
    // the host copies run up to kSlots chunks ahead of the device copies, which are queued in order
    size_t filled = 0, sent = 0;
    const size_t base = static_cast<size_t>(x.next);
    try {
        for (const Block& b : blocks) {
            if (b.chunks.empty()) {
                const XferItem& it = items[b.first];
                if (it.bytes) SXH_HIP(hipMemcpyAsync(it.dev, it.host, it.bytes, hipMemcpyHostToDevice, s));
            }
            for (const Chunk& c : b.chunks) {
                for (; filled < order.size() && filled - sent < kSlots; filled++) {
                    const int slot = static_cast<int>((base + filled) % kSlots);
                    if (x.copying[slot]) {
                        if (filled > sent && hipEventQuery(x.ev[slot]) == hipErrorNotReady) break;  // send first
                        x.settle(slot);
                    }
                    x.push({order[filled], slot, false});
                }
                const int slot = static_cast<int>((base + sent) % kSlots);
                x.wait_slot(slot);
                x.copy_chunk(c.dev, x.chunk(slot), c.bytes, hipMemcpyHostToDevice, total, s);
                SXH_HIP(hipEventRecord(x.ev[slot], s));
                x.copying[slot] = true;
                sent++;
            }
            for (size_t k = b.first; k < b.last; k++)
                if (items[k].stage) items[k].stage();
        }
        x.next = static_cast<int>((base + sent) % kSlots);  // (a slot waits for its copy when it is used again)
    } catch (...) {
        x.drain();
        (void)hipStreamSynchronize(s);
        for (bool& c : x.copying) c = false;
        throw;
    }
    x.check();
}

void HostXfer::to_host(const std::vector<XferItem>& items, hipStream_t s) {
    Impl& x = *p_;
    const size_t total = total_bytes(items);
    std::lock_guard<std::mutex> one(x.call);
    const bool ring = x.start(total);
    const std::vector<Block> blocks = blocks_of(items, chunk_bytes(total), false, ring);
    try {
        for (const Block& b : blocks) {
            for (size_t k = b.first; k < b.last; k++)
                if (items[k].stage) items[k].stage();
            if (b.chunks.empty()) {
                const XferItem& it = items[b.first];
                if (it.bytes) SXH_HIP(hipMemcpyAsync(it.host, it.dev, it.bytes, hipMemcpyDeviceToHost, s));
            }
            for (const Chunk& c : b.chunks) {
                const int slot = x.next;
                x.next = (slot + 1) % kSlots;
                x.wait_slot(slot);
                x.settle(slot);
                x.copy_chunk(x.chunk(slot), c.dev, c.bytes, hipMemcpyDeviceToHost, total, s);
                SXH_HIP(hipEventRecord(x.ev[slot], s));
                x.push({&c, slot, true});
            }
        }
        x.drain();
        SXH_HIP(hipStreamSynchronize(s));
    } catch (...) {
        x.drain();
        (void)hipStreamSynchronize(s);
        throw;
    }
    x.check();
}

}  // namespace sxh
