// Results of the synchronous entry points: device memory into the caller's
// ordinary host arrays.
//
// The runtime copies into pageable memory at about 18 GB/s and waits 15 us for
// every result.  Pieces that go to pinned memory by DMA (56 GB/s) while earlier
// pieces are moved on to the caller's array end little after the DMA.  Energy,
// gradient and Hessian of P1 meshes with their kernels, by the runtime / through
// the ring, us: 40 KB of results 95 / 60, 2.1 MB 198 / 155, 9.3 MB 635 / 355,
// 31 MB 1,900 / 855; a projected Hessian of 24 MB 1,860 / 1,050.  These are calls
// of a handle in use: its first ones take the runtime's copies (RING_PAYS).
//
// The pinned memory is a ring of up to SLOTS pieces, as large as the copy needs.
// A call leases a ring for its own duration, so handles, threads and streams
// share no slot; idle rings wait for the next call and are freed with the last
// handle.  Arrays that DMA reaches by itself (pinned, managed) take the
// runtime's copy: a Hessian of 9.3 MB into pinned memory takes 234 us with its
// kernels, through the ring 325.
#include <algorithm>
#include <atomic>
#include <bit>
#include <cstring>
#include <exception>
#include <mutex>
#include <system_error>
#include <thread>

#include "handle.hpp"

namespace pfgpu {

namespace {

// A copy is cut into pieces of a quarter, so that the first one arrives early,
// but no larger than a slot and no smaller than what the launch of a piece and
// its event (13 us) cost in transfer time: 24 MB take 439 us in one piece, 514 in
// pieces of 4 MB, 769 in pieces of 1 MB.
constexpr int SLOTS = 4;
constexpr size_t SLOT_BYTES = size_t(4) << 20, PIECE_MIN = size_t(1) << 20;
// One array gains from here on (gradients with their kernels, by the runtime /
// through the ring, us: 0.7 MB 120 / 120, 1.9 MB 275 / 269, 5.5 MB 745 / 605);
// several arrays gain at any size, since their copies share one wait.
constexpr size_t SINGLE_MIN = size_t(2) << 20;
// A ring costs 0.1 to 0.2 ms per MB to allocate and first use (less where the
// process has freed pinned memory before), and gains 0.03 ms per MB copied.  A
// handle allocates one, for its largest copy so far, when its earlier copies (with
// RESULT_COST for every further result of a call) or the one at hand come to
// RING_PAYS times that.  Handles that are made, called once and dropped do not
// pay for it (0.7 MB of results: 1,690 us with a ring from the first call on, 1,510
// without; the first derivatives of a process, 25 MB: 3.8 ms and 2.3).
constexpr size_t RING_PAYS = 4, RESULT_COST = size_t(512) << 10;
// Rings of the process, leased and idle (256 MB); calls that find none take the
// runtime's copies.
constexpr int MAX_RINGS = 16;
// Threads that move a slot, the caller's own among them, and the copy from which
// there are more than one: a thread moves memory that the DMA has just written
// at about 28 GB/s, half of what the DMA brings, and costs about 20 us to start.
constexpr int MOVERS = 4;
constexpr size_t MOVERS_MIN = size_t(4) << 20;

struct Ring {
    char *mem = nullptr;
    size_t bytes = 0;
    hipEvent_t ev[SLOTS] = {};
    int device = -1;
    ~Ring()
    {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (mem) (void)hipHostFree(mem);
    }
};

std::mutex g_mutex;
// never destroyed: at the end of the process the runtime may be gone first
std::vector<std::unique_ptr<Ring>> &g_idle = *new std::vector<std::unique_ptr<Ring>>;
int g_handles = 0, g_rings = 0; // handles alive; rings, leased and idle

// null when pinned memory is not to be had
std::unique_ptr<Ring> new_ring(int device, size_t bytes)
{
    auto r = std::make_unique<Ring>();
    r->device = device;
    r->bytes = bytes;
    void *p = nullptr;
    bool ok = hipHostMalloc(&p, r->bytes, hipHostMallocDefault) == hipSuccess;
    r->mem = static_cast<char *>(p);
    for (hipEvent_t &e : r->ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (ok) return r;
    (void)hipGetLastError();
    return nullptr;
}

// An idle ring of the device with room for bytes; else, where allocate is not 0, a
// new one of so many in the place of a smaller idle one or within MAX_RINGS; else
// none.
struct Lease {
    std::unique_ptr<Ring> ring;
    hipStream_t stream;
    bool done = false; // every copy into the ring has ended
    Lease(int device, hipStream_t s, size_t bytes, size_t allocate) : stream(s)
    {
        std::unique_ptr<Ring> drop;
        {
            std::lock_guard<std::mutex> lock(g_mutex);
            auto take = [&](bool small) {
                auto r = std::find_if(g_idle.begin(), g_idle.end(), [&](auto &i) { return i->device == device && (i->bytes < bytes) == small; });
                if (r == g_idle.end()) return std::unique_ptr<Ring>();
                std::unique_ptr<Ring> taken = std::move(*r);
                g_idle.erase(r);
                return taken;
            };
            ring = take(false);
            if (ring || !allocate) return;
            drop = take(true);
            if (!drop && g_rings >= MAX_RINGS) return;
            g_rings += drop ? 0 : 1;
        }
        drop.reset();
        try {
            ring = new_ring(device, allocate);
        } catch (const std::bad_alloc &) {
        }
        if (!ring) {
            std::lock_guard<std::mutex> lock(g_mutex);
            --g_rings;
        }
    }
    Lease(const Lease &) = delete;
    ~Lease()
    {
        if (!ring) return;
        if (!done) (void)hipStreamSynchronize(stream);
        std::unique_ptr<Ring> drop; // freed outside the lock
        std::lock_guard<std::mutex> lock(g_mutex);
        if (g_handles > 0) { // g_idle has room for MAX_RINGS
            g_idle.push_back(std::move(ring));
        } else {
            drop = std::move(ring);
            --g_rings;
        }
    }
};

// whether the runtime's DMA reaches the array: pinned, managed or device memory
bool dma_reaches(const void *host)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}

void copy_plain(Handle &h, const HostCopy &c)
{
    PF_HIP(hipMemcpyAsync(c.host, c.dev, c.bytes, hipMemcpyDeviceToHost, h.stream));
    PF_HIP(hipStreamSynchronize(h.stream));
}

// the items by the runtime, one after the other: several copies into pageable
// memory queued at once take longer (95 us for four results of 37 KB, queued 114)
bool copy_plain(Handle &h, const HostCopy *items, int n_items, const int *stop)
{
    for (int i = 0; i < n_items; ++i) {
        copy_plain(h, items[i]);
        if (stop && items[i].host == stop && *stop) return false;
    }
    return true;
}

} // namespace

void host_copy_handles(int delta)
{
    std::vector<std::unique_ptr<Ring>> drop;
    std::lock_guard<std::mutex> lock(g_mutex);
    if (delta > 0) g_idle.reserve(MAX_RINGS); // a lease gives its ring back without allocating
    g_handles += delta;
    if (g_handles == 0) {
        g_rings -= int(g_idle.size());
        drop.swap(g_idle);
    }
}

bool copy_to_host(Handle &h, const HostCopy *all, int n_all, const int *stop)
{
    // through the ring, and past it
    std::vector<HostCopy> items, direct;
    size_t total = 0, padded = 0;
    for (int i = 0; i < n_all; ++i) {
        if (dma_reaches(all[i].host)) {
            direct.push_back(all[i]);
            continue;
        }
        items.push_back(all[i]);
        total += all[i].bytes;
        padded += (all[i].bytes + 15) & ~size_t(15);
    }
    const int n_items = int(items.size());
    const size_t piece = std::clamp((total / 4 + 4095) & ~size_t(4095), PIECE_MIN, SLOT_BYTES);
    std::unique_ptr<Lease> lease;
    if (n_items > 1 || total >= SINGLE_MIN) {
        const size_t pieces = padded / piece + 2; // the item that decides has its own
        const size_t need = padded <= piece ? padded : std::min(pieces, size_t(SLOTS)) * piece;
        h.host_ring = std::max(h.host_ring, std::bit_ceil(std::max(need, PIECE_MIN))); // few sizes: a ring is seldom replaced
        const bool pays = std::max(h.copied_to_host, total) >= RING_PAYS * h.host_ring;
        lease = std::make_unique<Lease>(h.device, h.stream, need, pays ? h.host_ring : 0);
        h.copied_to_host += total + size_t(n_items - 1) * RESULT_COST;
    }
    if (!lease || !lease->ring) return copy_plain(h, all, n_all, stop);
    Ring &ring = *lease->ring;
    // a single piece: nothing to overlap
    if (padded <= piece) {
        char *at = ring.mem;
        for (const HostCopy &c : items) {
            PF_HIP(hipMemcpyAsync(at, c.dev, c.bytes, hipMemcpyDeviceToHost, h.stream));
            at += (c.bytes + 15) & ~size_t(15);
        }
        PF_HIP(hipStreamSynchronize(h.stream));
        lease->done = true;
        at = ring.mem;
        for (const HostCopy &c : items) {
            std::memcpy(c.host, at, c.bytes);
            if (stop && c.host == stop && *stop) return false;
            at += (c.bytes + 15) & ~size_t(15);
        }
        return copy_plain(h, direct.data(), int(direct.size()), nullptr);
    }
    // pieces of the items, 16-byte aligned in their slots; batch b fills a slot
    // (the item that decides whether the others are written has its own)
    struct Piece {
        char *host;
        const char *dev;
        size_t at, bytes;
    };
    std::vector<Piece> pieces;
    std::vector<size_t> batch{0}; // first piece of every batch
    size_t at = 0;
    for (int i = 0; i < n_items; ++i)
        for (size_t o = 0; o < items[i].bytes;) {
            if (at >= piece) {
                batch.push_back(pieces.size());
                at = 0;
            }
            const size_t b = std::min(items[i].bytes - o, piece - at);
            pieces.push_back({static_cast<char *>(items[i].host) + o, static_cast<const char *>(items[i].dev) + o, at, b});
            at += (b + 15) & ~size_t(15);
            o += b;
            if (stop && items[i].host == stop) at = piece;
        }
    const int nb = int(batch.size());
    batch.push_back(pieces.size());
    auto issue = [&](int b) {
        char *slot = ring.mem + size_t(b % SLOTS) * piece;
        for (size_t k = batch[size_t(b)]; k < batch[size_t(b) + 1]; ++k)
            PF_HIP(hipMemcpyAsync(slot + pieces[k].at, pieces[k].dev, pieces[k].bytes, hipMemcpyDeviceToHost, h.stream));
        PF_HIP(hipEventRecord(ring.ev[b % SLOTS], h.stream));
    };
    const int ahead = std::min(nb, SLOTS);
    for (int b = 0; b < ahead; ++b) issue(b);
    // Every mover moves its share of every batch; the last to finish one refills
    // its slot.  It does so before it goes on to the next batch, so batches are
    // issued in order, and a mover waits for a batch to be issued before it
    // waits for the batch's event.
    std::atomic<int> issued{ahead}, n_movers{0};
    std::atomic<int> left[SLOTS];
    std::atomic<bool> failed{false};
    std::exception_ptr error;
    std::mutex error_mutex;
    auto finish = [&](int b, int n) {
        left[b % SLOTS] = n;
        if (b + SLOTS >= nb) return;
        issue(b + SLOTS);
        issued = b + SLOTS + 1;
        issued.notify_all();
    };
    auto move = [&](int b, int t, int n) { // share t of n of batch b
        PF_HIP(hipEventSynchronize(ring.ev[b % SLOTS]));
        const char *slot = ring.mem + size_t(b % SLOTS) * piece;
        const size_t end = pieces[batch[size_t(b) + 1] - 1].at + pieces[batch[size_t(b) + 1] - 1].bytes;
        const size_t lo = end * size_t(t) / size_t(n), hi = end * size_t(t + 1) / size_t(n);
        for (size_t k = batch[size_t(b)]; k < batch[size_t(b) + 1]; ++k) {
            const Piece &p = pieces[k];
            const size_t from = std::max(lo, p.at), to = std::min(hi, p.at + p.bytes);
            if (from < to) std::memcpy(p.host + (from - p.at), slot + from, to - from);
        }
    };
    auto mover = [&](int t, int first, int n) {
        try {
            for (int b = first; b < nb; ++b) {
                for (int i = issued; i <= b && !failed; i = issued) issued.wait(i);
                if (failed) return;
                move(b, t, n);
                if (left[b % SLOTS].fetch_sub(1) == 1) finish(b, n);
            }
        } catch (...) {
            {
                std::lock_guard<std::mutex> lock(error_mutex);
                if (!error) error = std::current_exception();
            }
            failed = true;
            issued = nb; // releases the movers that wait for a batch
            issued.notify_all();
        }
    };
    const int first = stop ? 1 : 0;
    std::vector<std::thread> helpers;
    struct Join {
        std::vector<std::thread> &threads;
        std::atomic<int> &go;
        ~Join()
        {
            if (go == 0) { // they never began
                go = -1;
                go.notify_all();
            }
            for (std::thread &t : threads) t.join();
        }
    };
    {
        Join join{helpers, n_movers};
        if (total >= MOVERS_MIN) {
            helpers.reserve(MOVERS - 1);
            try {
                for (int t = 1; t < MOVERS; ++t)
                    helpers.emplace_back([&, t] {
                        n_movers.wait(0);
                        const int n = n_movers;
                        if (n < 0) return;
                        if (hipSetDevice(h.device) != hipSuccess) (void)hipGetLastError();
                        mover(t, first, n);
                    });
            } catch (const std::system_error &) {
                // no more threads to be had: those that run share the work
            }
        }
        const int n = int(helpers.size()) + 1;
        for (std::atomic<int> &l : left) l = n;
        if (stop) {
            move(0, 0, 1);
            if (*stop) return false;
            finish(0, n);
        }
        n_movers = n;
        n_movers.notify_all();
        mover(0, first, n);
    }
    if (error) std::rethrow_exception(error);
    lease->done = true;
    return copy_plain(h, direct.data(), int(direct.size()), nullptr);
}

} // namespace pfgpu
