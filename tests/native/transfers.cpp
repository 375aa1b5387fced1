// The executor's exchange of rows, the pinned ring and the device buffers' cache on a runtime of host memory
// (host_runtime.h). One check per argument; the kernels that move rows are written out here as their headers state them.
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <string>
#include <thread>
#include <vector>

#include "host_runtime.h"
#include "sx_exec.h"
#include "sx_host.h"
#include "sx_kernels.h"
#include "sx_step.h"

#define CHECK(x)                                                        \
    do {                                                                \
        if (!(x)) {                                                     \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);         \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

namespace sxh {
static thread_local std::string g_error;
void set_last_error(const std::string& m) { g_error = m; }
}  // namespace sxh

namespace sxk {
size_t scan_scratch_bytes(int64_t) { return 64; }
size_t sort_scratch_bytes(int64_t) { return 64; }
int step_preprocess_blocks(int64_t n) { return static_cast<int>((n + 255) / 256); }
void copy_bytes(void* dst, const void* src, size_t n, hipStream_t s) {
    host_runtime::enqueue(s, [=] { std::memcpy(dst, src, n); });
}
void soa_to_rows(const float* soa, float* aos, int n, int dim, int stride, hipStream_t s, const int32_t* dst_row, int n_perm,
                 int n_out) {
    host_runtime::enqueue(s, [=] {
        for (int k = 0; k < n; k++) {
            const int to = dst_row && k < n_perm ? dst_row[k] : k;
            if (to < (n_out < 0 ? n : n_out))
                for (int d = 0; d < dim; d++) aos[(size_t)to * dim + d] = soa[(size_t)d * stride + k];
        }
    });
}
void rows_to_soa(const float* aos, float* soa, int n, int dim, int stride, hipStream_t s, const int32_t* src_row) {
    host_runtime::enqueue(s, [=] {
        for (int k = 0; k < n; k++)
            for (int d = 0; d < dim; d++) soa[(size_t)d * stride + k] = aos[(size_t)(src_row ? src_row[k] : k) * dim + d];
    });
}
void arena_permute_rows(const Arena& A, const int dims[6], int count, const int32_t* src, float* tmp, hipStream_t s) {
    for (int g = 0; g < 6; g++)
        for (float* col : {A.p[g], A.m[g], A.v[g]}) {
            if (!col || dims[g] == 0) continue;
            soa_to_rows(col, tmp, count, dims[g], A.rows, s);
            rows_to_soa(tmp, col, count, dims[g], A.rows, s, src);
        }
}
}  // namespace sxk

namespace {

using sxh::DevBuf;
using sxh::DevCache;

struct Backend {
    sxh_backend* b = new sxh_backend;
    Backend() {
        SXH_HIP(hipStreamCreateWithFlags(&b->stream, 0));
        b->xfer = std::make_unique<sxh::HostXfer>(0);
    }
    ~Backend() {
        b->xfer.reset();
        b->cache.release();
        (void)hipStreamDestroy(b->stream);
        delete b;
    }
};

// Parameters and moments of `rows` rows at SH degree 1, every value its own; array `pin` (of 18) in pinned memory.
struct Rows {
    std::vector<float> a[3][6];
    float* pinned = nullptr;
    int pin;
    static constexpr int kDims[6] = {3, 4, 3, 1, 3, 9};
    Rows(int rows, float first, int pin_at = -1) : pin(pin_at) {
        for (int g = 0; g < 6; g++)
            for (int k = 0; k < 3; k++) {
                a[k][g].resize((size_t)rows * kDims[g]);
                for (size_t q = 0; q < a[k][g].size(); q++) a[k][g][q] = first + 1000.0f * (3 * g + k) + q * 0.25f;
                if (3 * g + k == pin) {
                    SXH_HIP(hipHostMalloc(reinterpret_cast<void**>(&pinned), a[k][g].size() * 4, 0));
                    std::memcpy(pinned, a[k][g].data(), a[k][g].size() * 4);
                }
            }
    }
    ~Rows() {
        if (pinned) (void)hipHostFree(pinned);
    }
    sxh_param_sync sync(int rows) {
        sxh_param_sync s{};
        for (int g = 0; g < 6; g++) {
            s.params[g] = 3 * g == pin ? pinned : a[0][g].data();
            s.exp_avg[g] = 3 * g + 1 == pin ? pinned : a[1][g].data();
            s.exp_avg_sq[g] = 3 * g + 2 == pin ? pinned : a[2][g].data();
        }
        s.rows = rows;
        return s;
    }
};

// The arena's first n rows as a training step leaves them in spatial order: internal row k holds row n - 1 - k.
void reverse_order(sxh_executor* e, int n) {
    e->row_orig.alloc(e->rows);
    e->row_int.alloc(e->rows);
    for (int k = 0; k < n; k++) e->row_orig.p[k] = e->row_int.p[k] = n - 1 - k;
    sxk::arena_permute_rows(e->arena(), e->dims, n, e->row_orig.p, e->staging.p, e->b->stream);
    SXH_HIP(hipStreamSynchronize(e->b->stream));
    e->permuted = true;
    e->perm_count = n;
}

sxh_executor* executor(sxh_backend* b, int rows) {
    sxh_exec_desc d{};
    d.arena_rows = rows;
    d.sh_degree = 1;
    d.isect_mode = SXH_ISECT_ACCUTILE;
    sxh_executor* e = nullptr;
    CHECK(sxh_exec_create(b, &d, &e) == SXH_OK);
    return e;
}

// An upload over every row of an arena in spatial order that fails at its eighth array: the seven before it hold the
// new rows, the others the old ones, all in the caller's order, and the next exchange sees them so. At 70,000 rows the
// arrays travel one by one, at 300 in one block up to the failing one.
void upload_fails_midway() {
    for (int n : {300, 70000}) {
        Backend B;
        sxh_executor* e = executor(B.b, n);
        Rows old(n, 0.0f), fresh(n, 0.5f, 7), got(n, -1.0f);
        auto so = old.sync(n), sf = fresh.sync(n), sg = got.sync(n);
        CHECK(sxh_exec_upload(e, &so) == SXH_OK);
        // (below 8 MiB only the array in pinned memory goes through a copy of the runtime's; above, every chunk does)
        const int before = host_runtime::copies();
        CHECK(sxh_exec_upload(e, &so) == SXH_OK);
        const int fail = n == 300 ? 1 : (host_runtime::copies() - before) / 2;
        for (const bool spatial : {true, false}) {
            if (spatial) reverse_order(e, n);
            host_runtime::faults.copy = fail;
            CHECK(sxh_exec_upload(e, &sf) == SXH_ERR_RUNTIME);
            CHECK(host_runtime::faults.copy == 0);
            CHECK(sxh_exec_download(e, &sg) == SXH_OK);
            int news = 0;
            for (int q = 0; q < 18; q++) {
                const auto& x = got.a[q % 3][q / 3];
                const bool is_new = x == fresh.a[q % 3][q / 3], is_old = x == old.a[q % 3][q / 3];
                CHECK(is_new != is_old);
                CHECK(!is_new || news == q);  // (the arrays before the failing one)
                news += is_new;
            }
            CHECK(n > 300 ? news > 0 && news < 18 : news == 7);
            CHECK(sxh_exec_upload(e, &so) == SXH_OK);
        }
        sxh_exec_destroy(e);
    }
}

// A transfer in which a wait fails on the way and then a copy: it reports an error, and the next one reports none.
void error_is_reported_once() {
    Backend B;
    const size_t n = size_t{64} << 20;  // 16 chunks of 4 MiB, twice around the ring
    DevBuf<char> dev(n);
    std::vector<char> host(n, 1), back(n);
    B.b->xfer->to_device({{host.data(), dev.p, n, {}}}, B.b->stream);
    B.b->xfer->to_host({{back.data(), dev.p, n, {}}}, B.b->stream);  // (waits for the upload's copies; only its own follow)
    host_runtime::faults.event_sync = 1;
    host_runtime::faults.copy = 15;
    bool threw = false;
    try {
        B.b->xfer->to_host({{back.data(), dev.p, n, {}}}, B.b->stream);
    } catch (const std::exception&) {
        threw = true;
    }
    CHECK(threw && host_runtime::faults.event_sync == 0 && host_runtime::faults.copy == 0);
    for (int k = 0; k < 2; k++) {
        back.assign(n, 0);
        B.b->xfer->to_host({{back.data(), dev.p, n, {}}}, B.b->stream);
        CHECK(back == host);
        host[5 + k] = 3;
        B.b->xfer->to_device({{host.data(), dev.p, n, {}}}, B.b->stream);
    }
    // a wait that fails by itself is reported by its own transfer
    B.b->xfer->to_host({{back.data(), dev.p, n, {}}}, B.b->stream);
    host_runtime::faults.event_sync = 3;
    threw = false;
    try {
        B.b->xfer->to_host({{back.data(), dev.p, n, {}}}, B.b->stream);
    } catch (const std::exception&) {
        threw = true;
    }
    CHECK(threw);
}

// Where there is no pinned memory for the ring the runtime copies the arrays; once there is, the ring does.
void without_the_ring() {
    for (int n : {300, 70000}) {
        Backend B;
        sxh_executor* e = executor(B.b, n);
        for (const bool none : {true, false}) {
            host_runtime::faults.pinned = none;
            Rows up(n, none ? 0.0f : 0.5f), got(n, -1.0f);
            auto su = up.sync(n), sg = got.sync(n);
            const int before = host_runtime::copies();
            CHECK(sxh_exec_upload(e, &su) == SXH_OK);
            CHECK(sxh_exec_download(e, &sg) == SXH_OK);
            CHECK(!none || host_runtime::copies() - before == 36);
            for (int k = 0; k < 3; k++)
                for (int g = 0; g < 6; g++) CHECK(got.a[k][g] == up.a[k][g]);
        }
        sxh_exec_destroy(e);
    }
}

// What the per-op calls left in a backend's cache is given back before an allocation fails: the executors' (uncached),
// another backend's, and a cached one that is only to be had without rounding.
void kept_memory_gives_way() {
    constexpr size_t kMiB = size_t{1} << 20;
    Backend A, B;
    host_runtime::device_limit = 200 * kMiB;
    { DevBuf<char> x(50 * kMiB, &A.b->cache), y(40 * kMiB, &B.b->cache); }
    CHECK(host_runtime::device_bytes() > 90 * kMiB);
    {
        DevBuf<char> arena(150 * kMiB);
        CHECK(arena.p && host_runtime::device_bytes() < 151 * kMiB);
    }
    { DevBuf<char> x(60 * kMiB, &A.b->cache); }
    {
        DevBuf<char> other(190 * kMiB, &B.b->cache);  // (with an eighth more it would pass the limit)
        CHECK(other.p);
    }
    bool threw = false;
    try {
        DevBuf<char> most(201 * kMiB);
    } catch (const std::exception&) {
        threw = true;
    }
    CHECK(threw);
    { DevBuf<char> x(8, &A.b->cache), y(8, &A.b->cache); }
    host_runtime::device_limit = ~size_t{0};
}

// After a burst of large sizes has filled the cache, the sizes of later calls are kept all the same, and no more than
// 256 MiB are.
void kept_memory_follows_use() {
    constexpr size_t kMiB = size_t{1} << 20;
    Backend B;
    const size_t before = host_runtime::device_bytes();
    { DevBuf<char> a(70 * kMiB, &B.b->cache), b(75 * kMiB, &B.b->cache), c(80 * kMiB, &B.b->cache); }
    for (int k = 0; k < 4; k++) {
        const int n = host_runtime::mallocs();
        { DevBuf<char> x(20 * kMiB, &B.b->cache), y(3 * kMiB, &B.b->cache), z(100, &B.b->cache); }
        CHECK(k == 0 || host_runtime::mallocs() == n);
        CHECK(host_runtime::device_bytes() - before <= 256 * kMiB);
    }
    { DevBuf<char> large(300 * kMiB, &B.b->cache); }  // larger than the cache: not kept, and nothing goes for it
    const int n = host_runtime::mallocs();
    { DevBuf<char> x(20 * kMiB, &B.b->cache); }
    CHECK(host_runtime::mallocs() == n);
    CHECK(host_runtime::device_bytes() - before <= 256 * kMiB);
    DevCache::release_all();
    CHECK(host_runtime::device_bytes() == before);
}

// Exchanges of many sizes from several threads at once, each thread with a backend of its own, and then all of them on
// one backend's ring, with streams that lag behind: every thread reads back its own rows.
void several_threads() {
    host_runtime::stream_delay_us(30);
    auto work = [](sxh_backend* b, int seed) {
        size_t n = 1000 + 4099 * seed;
        for (int k = 0; k < 12; k++, n = n * 3 + 1) {
            if (n > size_t{20} << 20) n = 77 + seed;
            std::vector<char> x(n), y(n), z(n / 2 + 1), w(n / 2 + 1);
            for (size_t q = 0; q < n; q++) x[q] = static_cast<char>(q * 7 + seed + k);
            for (size_t q = 0; q < z.size(); q++) z[q] = static_cast<char>(q * 5 - seed);
            DevBuf<char> d(n, &b->cache), e(z.size(), &b->cache);
            int staged = 0;
            b->xfer->to_device({{x.data(), d.p, n, [&] { staged++; }}, {z.data(), e.p, z.size(), [&] { staged++; }}},
                               b->stream);
            b->xfer->to_host({{y.data(), d.p, n, [&] { staged++; }}, {w.data(), e.p, w.size(), {}}}, b->stream);
            CHECK(x == y && z == w && staged == 3);
        }
    };
    std::vector<std::unique_ptr<Backend>> own;
    for (int k = 0; k < 3; k++) own.push_back(std::make_unique<Backend>());
    for (const bool one : {false, true}) {
        std::vector<std::thread> threads;
        for (int k = 0; k < 3; k++) threads.emplace_back([&, k] { work(own[one ? 0 : k]->b, k); });
        for (auto& t : threads) t.join();
    }
    host_runtime::stream_delay_us(0);
}

}  // namespace

int main(int argc, char** argv) {
    const std::map<std::string, std::function<void()>> all = {
        {"upload_fails_midway", upload_fails_midway},
        {"error_is_reported_once", error_is_reported_once},
        {"without_the_ring", without_the_ring},
        {"kept_memory_gives_way", kept_memory_gives_way},
        {"kept_memory_follows_use", kept_memory_follows_use},
        {"several_threads", several_threads},
    };
    for (int k = 1; k < argc; k++) {
        const auto it = all.find(argv[k]);
        CHECK(it != all.end());
        it->second();
        std::printf("%s: done\n", argv[k]);
    }
    return 0;
}
