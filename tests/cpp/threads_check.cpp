// CPU check of the host loops that build the plans and tables: where threads or
// memory run out, or a table is refused, in one of their threads, the caller
// gets the plan or the exception.  Input: the binary mesh file of plan_check.cpp.
#include <dlfcn.h>
#include <pthread.h>

#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <thread>
#include <vector>

#include "../../polyfem_amd/csrc/fused.hpp"
#include "../../polyfem_amd/csrc/plans.hpp"

using namespace pfgpu;

static std::atomic<int> threads_left{1 << 30};
static std::atomic<bool> no_memory{false};
static thread_local bool in_thread = false;

struct Start {
    void *(*f)(void *);
    void *arg;
};
static void *started(void *p)
{
    const Start s = *static_cast<Start *>(p);
    std::free(p);
    in_thread = true;
    return s.f(s.arg);
}
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *attr, void *(*f)(void *), void *arg)
{
    if (threads_left.fetch_sub(1) <= 0) return EAGAIN;
    using Create = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static const Create create = reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"));
    Start *s = static_cast<Start *>(std::malloc(sizeof(Start)));
    *s = {f, arg};
    return create(t, attr, started, s);
}
void *operator new(size_t n)
{
    if (in_thread && no_memory) throw std::bad_alloc();
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

static int fails = 0;
#define CHECK(c)                                                     \
    do {                                                             \
        if (!(c)) {                                                  \
            ++fails;                                                 \
            std::printf("CHECK failed line %d: %s\n", __LINE__, #c); \
        }                                                            \
    } while (0)

int main(int argc, char **argv)
{
    FILE *f = argc < 2 ? nullptr : std::fopen(argv[1], "rb");
    int32_t hdr[4];
    if (!f || std::fread(hdr, 4, 4, f) != 4) return 2;
    const int order = hdr[0], E = hdr[1], N = hdr[2], Nv = hdr[3], NB = order == 1 ? 4 : 10;
    std::vector<int32_t> en(size_t(E) * NB), ev(size_t(E) * 4);
    std::vector<double> vx(size_t(Nv) * 3);
    if (std::fread(en.data(), 4, en.size(), f) != en.size() || std::fread(ev.data(), 4, ev.size(), f) != ev.size() ||
        std::fread(vx.data(), 8, vx.size(), f) != vx.size())
        return 2;
    std::fclose(f);
    struct Plans {
        Pattern pat;
        bool wave, unit;
        WavePlanHost w;
        UnitPlanHost u;
    };
    auto plans = [&] {
        Plans p;
        p.pat = build_pattern(E, NB, en.data(), N, Nv, ev.data());
        p.wave = plan_wave_gather(p.pat, order, 4, en.data(), 4, p.w);
        p.unit = make_unit_plan(p.pat, NB, en.data(), 64, 128, p.u);
        return p;
    };
    const Plans want = plans();
    for (int left : {0, 1, 3}) { // threads that can still be started
        threads_left = left;
        const Plans p = plans();
        CHECK(p.pat.bcol == want.pat.bcol && p.wave == want.wave && p.unit == want.unit);
        CHECK(p.w.dst == want.w.dst && p.w.desc == want.w.desc && p.w.long_desc == want.w.long_desc);
        CHECK(p.u.udst == want.u.udst && p.u.bq0 == want.u.bq0 && p.u.lanes == want.u.lanes);
    }
    threads_left = 1 << 30;
    auto throws = [&](auto &&call) {
        try {
            call();
        } catch (const std::bad_alloc &) {
            return true;
        }
        return false;
    };
    if (std::thread::hardware_concurrency() > 1) {
        no_memory = true;
        WavePlanHost w;
        UnitPlanHost u;
        if (want.wave) CHECK(throws([&] { plan_wave_gather(want.pat, order, 4, en.data(), 4, w); }));
        if (want.unit) CHECK(throws([&] { make_unit_plan(want.pat, NB, en.data(), 64, 128, u); }));
        no_memory = false;
    }
    FusedShape shape{}; // as in plan_check.cpp
    shape.groups = order == 1 ? 70 : 28;
    shape.chunk = order == 1 ? 128 : 32;
    shape.item_cap = shape.chunk * NB;
    shape.max_rows = 256;
    shape.acc_capacity = 30000;
    try {
        const FusedTables t = build_fused_tables(want.pat, NB, en.data(), E, vx.data(), ev.data(), shape);
        std::printf("fused tables: %d patches\n", t.n_patches);
    } catch (const Error &e) {
        std::printf("fused tables refused: %s\n", e.what());
    }
    std::printf("%s\n", fails ? "FAIL" : "OK");
    return fails ? 1 : 0;
}
