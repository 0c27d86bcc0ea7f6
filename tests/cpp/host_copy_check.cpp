// CPU check of the copies of results into host arrays (host_copy.cpp), meant to
// run under AddressSanitizer or ThreadSanitizer: the HIP calls it makes are
// defined here, copy at once and are counted.  Argument: the check to run.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <thread>

#include "../../polyfem_amd/csrc/handle.hpp"

using namespace pfgpu;

static std::atomic<int> n_alloc{0}, n_free{0}, n_pageable{0};
static std::atomic<int> queued{0}, most_queued{0}; // copies into pageable memory since the last wait
static std::atomic<size_t> largest{0};
static std::atomic<bool> no_pinned{false}, bad_event{false};
static std::atomic<const char *> watch{nullptr}; // copies that end at this address are counted
static std::atomic<int> n_watched{0};
static std::mutex mutex;
static std::map<const char *, size_t> pinned; // pinned memory, the ring's and the caller's

static bool is_pinned(const void *p)
{
    std::lock_guard<std::mutex> lock(mutex);
    auto i = pinned.upper_bound(static_cast<const char *>(p));
    return i != pinned.begin() && (--i, static_cast<const char *>(p) < i->first + i->second);
}

extern "C" {
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
    if (no_pinned) return hipErrorOutOfMemory;
    ++n_alloc;
    for (size_t l = largest; l < bytes && !largest.compare_exchange_weak(l, bytes);) {}
    *p = std::malloc(bytes);
    std::lock_guard<std::mutex> lock(mutex);
    pinned[static_cast<char *>(*p)] = bytes;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    {
        std::lock_guard<std::mutex> lock(mutex);
        pinned.erase(static_cast<char *>(p));
    }
    ++n_free;
    std::free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    a->type = is_pinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t)
{
    if (to == watch) ++n_watched;
    if (!is_pinned(to)) {
        ++n_pageable;
        if (++queued > most_queued) most_queued = int(queued);
    }
    std::memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return queued = 0, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(std::malloc(1)), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(reinterpret_cast<void *>(e)), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return bad_event ? hipErrorUnknown : hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMalloc(void **, size_t) { std::abort(); }
hipError_t hipFree(void *) { std::abort(); }
}

pfgpu_handle::pfgpu_handle() { host_copy_handles(1); }
pfgpu_handle::~pfgpu_handle() { host_copy_handles(-1); }

static int fails = 0;
#define CHECK(c)                                                                  \
    do {                                                                          \
        if (!(c)) {                                                               \
            ++fails;                                                              \
            std::printf("CHECK failed line %d: %s\n", __LINE__, #c);              \
        }                                                                         \
    } while (0)

using Bytes = std::vector<char>;
// n bytes from place `seed` of a fixed sequence
static Bytes data(size_t n, unsigned seed)
{
    static const Bytes all = [] {
        Bytes b(size_t(32) << 20);
        uint64_t s = 1;
        for (size_t i = 0; i < b.size(); i += 8, s = s * 6364136223846793005u + 1442695040888963407u) std::memcpy(&b[i], &s, 8);
        return b;
    }();
    return Bytes(all.begin() + seed, all.begin() + seed + std::ptrdiff_t(n));
}

// results of the given sizes into host arrays, `times` times; what arrives is compared
static void copies(Handle &h, std::initializer_list<size_t> sizes, int times)
{
    std::vector<Bytes> dev, host;
    std::vector<HostCopy> items;
    for (size_t n : sizes) dev.push_back(data(n, unsigned(n % 65521))), host.emplace_back(n);
    for (size_t k = 0; k < dev.size(); ++k) items.push_back({host[k].data(), dev[k].data(), dev[k].size()});
    for (int t = 0; t < times; ++t) {
        for (Bytes &b : host) std::fill(b.begin(), b.end(), 0);
        CHECK(copy_to_host(h, items.data(), int(items.size())));
        for (size_t k = 0; k < dev.size(); ++k) CHECK(host[k] == dev[k]);
    }
}

// a flag and the values that it guards; false with the values untouched where it is set
static void guarded(Handle &h, int flag, size_t n)
{
    const Bytes dev = data(n, 3), before = data(n, 4);
    Bytes host = before;
    int bad = 0;
    const HostCopy items[2] = {{&bad, &flag, sizeof(flag)}, {host.data(), dev.data(), n}};
    const bool ok = copy_to_host(h, items, 2, &bad);
    CHECK(ok == (flag == 0) && bad == flag);
    CHECK(host == (flag ? before : dev));
}

constexpr size_t KB = 1024, MB = 1024 * KB;

static const std::map<std::string, std::function<void()>> checks = {
    // arrays that DMA reaches are copied to once and directly, the others around them as ever
    {"pinned_destination", [] {
        Handle h;
        copies(h, {4, 8 * MB, 100}, 9); // a handle in use
        void *p = nullptr;
        const Bytes dev = data(9 * MB, 5), small = data(300 * KB, 6), flag(4, 0);
        (void)hipHostMalloc(&p, dev.size(), 0);
        Bytes host(small.size());
        watch = static_cast<char *>(p);
        for (int bad_value : {0, 1}) {
            std::memset(p, 0, dev.size());
            int bad = 0;
            const HostCopy items[3] = {{&bad, &bad_value, 4}, {p, dev.data(), dev.size()}, {host.data(), small.data(), small.size()}};
            n_watched = 0;
            CHECK(copy_to_host(h, items, 3, &bad) == !bad_value);
            CHECK(n_watched == !bad_value && (bad_value || (std::memcmp(p, dev.data(), dev.size()) == 0 && host == small)));
        }
        watch = nullptr;
        (void)hipHostFree(p);
    }},
    // all sizes around the limits
    {"sizes", [] {
        Handle h;
        copies(h, {18 * MB, 3 * MB}, 5);
        for (size_t n : {size_t(1), size_t(16), 65 * KB, 1 * MB - 20, 1 * MB, 2 * MB - 1, 2 * MB, 4 * MB + 5, 17 * MB + 7}) {
            copies(h, {n}, 1);
            copies(h, {n, 5, n / 2 + 1}, 2);
            guarded(h, 0, n);
            guarded(h, 1, n);
        }
    }},
    // the runtime copies one result at a time; a handle in use takes several
    // results of any size through the ring, and a single one from 2 MB on
    {"small", [] {
        Handle h;
        copies(h, {4, 8, 3000, 20 * KB}, 1);
        CHECK(most_queued == 1 && n_pageable == 4);
        copies(h, {18 * MB}, 4);
        CHECK(n_pageable == 8 && n_alloc == 0);
        copies(h, {18 * MB}, 1);
        CHECK(n_pageable == 8 && n_alloc == 1);
        for (size_t n : {8 * KB, 70 * KB, 300 * KB, 1 * MB}) {
            n_pageable = 0;
            copies(h, {4, n}, 1);
            CHECK(n_pageable == 0);
            copies(h, {n}, 1);
            CHECK(n_pageable == 1);
        }
        copies(h, {2 * MB}, 1);
        CHECK(n_pageable == 1);
    }},
    // values that a flag keeps back, with helper threads started and copies in
    // flight, then the same ring under another handle
    {"kept_back", [] {
        Handle a, b;
        copies(a, {20 * MB}, 5);
        for (int k = 0; k < 4; ++k) {
            guarded(a, 1, (k % 2 ? 18 : 10) * MB);
            copies(b, {8, 300 * KB, 9 * MB}, 1);
        }
    }},
    // handles that are made, called a few times and dropped: no ring
    {"short_lived", [] {
        for (int k = 0; k < 4; ++k) {
            Handle h;
            copies(h, {8, 9 * MB}, 1);
            Handle g;
            copies(g, {8, 5000, 300 * KB}, 4);
            Handle twice;
            copies(twice, {20 * MB}, 2);
        }
        CHECK(n_alloc == 0);
    }},
    // a handle in use: one ring, as large as its copies need, given back with the last handle
    {"ring_size", [] {
        {
            Handle h;
            copies(h, {8, 20 * KB, 3000 * KB}, 20);
            CHECK(n_alloc == 1 && largest <= 4 * MB);
            copies(h, {8, 20 * KB, 300 * KB}, 20);
            copies(h, {3 * MB}, 20);
            CHECK(n_alloc == 1);
            {
                Handle g; // takes the idle ring at its first call
                const int waits = n_pageable;
                copies(g, {8, 20 * KB, 300 * KB}, 1);
                CHECK(n_pageable == waits);
            }
            copies(h, {18 * MB}, 5); // the ring is replaced
            CHECK(n_alloc == 2 && n_free == 1 && largest <= 16 * MB);
        }
        CHECK(n_free == 2 && pinned.empty());
    }},
    // more calls at once than idle rings were kept for: no ring is freed between them
    {"threads", [] {
        std::atomic<int> at{0};
        Handle keep;
        auto work = [&](int n) {
            return [&, n] {
                Handle h;
                for (int k = 0; k < 12; ++k) {
                    ++at;
                    for (int spins = 0; at < n * (k + 1) && spins < 1000; ++spins) std::this_thread::yield();
                    copies(h, {8, 3 * MB}, 1);
                }
            };
        };
        for (int n : {10, 24}) {
            std::vector<std::thread> threads;
            at = 0;
            for (int t = 0; t < n; ++t) threads.emplace_back(work(n));
            for (std::thread &t : threads) t.join();
            CHECK(n_alloc <= std::min(n, 16) && n_free == 0);
        }
    }},
    {"errors", [] {
        {
            Handle h;
            no_pinned = true;
            copies(h, {8, 100, 5 * MB}, 6);
            no_pinned = false;
            copies(h, {8, 100, 5 * MB}, 6);
            bad_event = true;
            Bytes dev = data(20 * MB, 1), host(dev.size());
            const HostCopy item{host.data(), dev.data(), dev.size()};
            for (int k = 0; k < 4; ++k) {
                bool thrown = false;
                try {
                    copy_to_host(h, &item, 1);
                } catch (const Error &) {
                    thrown = true;
                }
                CHECK(thrown);
            }
            bad_event = false;
            copies(h, {8, 100, 20 * MB}, 2);
        }
        CHECK(n_alloc == n_free && pinned.empty());
    }},
};

int main(int argc, char **argv)
{
    const auto c = checks.find(argc > 1 ? argv[1] : "");
    if (c == checks.end()) return 2;
    c->second();
    std::printf("%s: %d allocations, largest %zu\n%s\n", argv[1], int(n_alloc), size_t(largest), fails ? "FAIL" : "OK");
    return fails ? 1 : 0;
}
