// The pool of page-locked host memory and the shared host copies (csrc/host_io.h) without a GPU: the two runtime calls
// behind the pool and the number of CPUs are this program's own.  One check per call, named by the argument; exit status 0: it holds.
#include <malloc.h>
#include <sys/sysinfo.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <thread>

#include "../../fyusenet_amd/csrc/host_io.h"

using namespace fynhip;

// Called in the place where the runtime may wait for the GPU.
static void (*g_runtime_waits)() = [] {};

extern "C" hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    g_runtime_waits();
    *p = aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
extern "C" hipError_t hipHostFree(void* p) {
    g_runtime_waits();
    free(p);
    return hipSuccess;
}

// What std::thread::hardware_concurrency asks.
static int g_cpus = 8;
extern "C" int get_nprocs() noexcept { return g_cpus; }

#define CHECK(x)                                              \
    do {                                                      \
        if (!(x)) {                                           \
            fprintf(stderr, "line %d: %s\n", __LINE__, #x);   \
            return 1;                                         \
        }                                                     \
    } while (0)

static constexpr size_t kArea = 1 << 20;

// A block that a launch uses is handed out again when the scope of the loan has ended and the launch has told so.
static int loans() {
    HostSignal signal;
    signal.create(nullptr);
    float* first;
    {
        HostLoan none(kArea);   // (no launch: back at once)
        first = none.floats();
    }
    HostDone done = signal.next();
    {
        HostLoan area(kArea);
        CHECK(area.floats() == first);
        area.used_until(signal, done.value);
        HostLoan other(kArea);
        CHECK(other.floats() != first);
        *done.flag = done.value;   // the launch has told, the scope has not ended
        HostLoan third(kArea);
        CHECK(third.floats() != first && third.floats() != other.floats());
    }
    done = signal.next();
    float* held;
    {
        HostLoan area(kArea);
        held = area.floats();
        area.used_until(signal, done.value);
    }
    {
        std::set<float*> seen;   // the scope has ended, the launch has not told
        HostLoan a(kArea), b(kArea), c(kArea), d(kArea);
        for (const HostLoan* l : {&a, &b, &c, &d}) seen.insert(l->floats());
        CHECK(seen.size() == 4 && !seen.count(held));
        CHECK(HostPool::contains(held, kArea));
    }
    *done.flag = done.value;
    bool again = false;
    HostLoan a(kArea), b(kArea), c(kArea), d(kArea), e(kArea);
    for (const HostLoan* l : {&a, &b, &c, &d, &e}) again = again || l->floats() == held;
    CHECK(again);
    signal.destroy();
    return 0;
}

// A thread inside one of the runtime's two calls, which may have to wait for the GPU, does not keep another one from
// the pool: what the GPU waits for may be that thread.
static std::atomic<int> g_inside{0}, g_other{0}, g_stuck{0};
static int runtime_calls_outside_the_lock() {
    HostPool::network_created();
    void* const idle = HostPool::acquire(kArea, false);
    void* const mine = HostPool::acquire(2 * kArea, false);
    HostPool::release(idle);
    g_runtime_waits = [] {
        g_inside++;
        const auto t0 = std::chrono::steady_clock::now();
        while (g_other.load() < g_inside.load())
            if (std::chrono::steady_clock::now() - t0 > std::chrono::seconds(5)) {
                g_stuck++;
                return;
            }
    };
    std::thread other([&] {
        for (int call = 1; call <= 2; call++) {
            while (g_inside.load() < call) {
            }
            (void)HostPool::contains(mine, kArea);
            g_other = call;
        }
    });
    void* const fresh = HostPool::acquire(4 * kArea, false);   // locks memory
    HostPool::network_gone();                                  // releases the idle block
    other.join();
    CHECK(g_inside.load() == 2 && g_stuck.load() == 0);
    g_runtime_waits = [] {};
    CHECK(HostPool::contains(mine, 2 * kArea) && HostPool::contains(fresh, 4 * kArea) && !HostPool::contains(idle, kArea));
    HostPool::release(mine);
    HostPool::release(fresh);
    CHECK(!HostPool::contains(mine, 1) && !HostPool::contains(fresh, 1));
    return 0;
}

// Copies on offer to helpers where the process has too few CPUs for any: they are made, and nothing is kept of them.
static int copies_without_helpers() {
    g_cpus = 3;
    CHECK(std::thread::hardware_concurrency() == 3);
    const int n = 20000;
    char from[256], to[256];
    for (size_t i = 0; i < sizeof(from); i++) from[i] = (char)(7 * i);
    auto in_use = [] { return mallinfo2().uordblks; };
    const size_t before = in_use();
    for (int i = 0; i < n; i++) {
        memset(to, 0, sizeof(to));
        {
            HostCopy copies;
            copies.add(to, from, sizeof(to));
            copies.start(0);   // (shared from no bytes on)
        }
        CHECK(!memcmp(to, from, sizeof(to)));
    }
    CHECK(in_use() < before + (64u << 10));
    return 0;
}

int main(int argc, char** argv) {
    const struct {
        const char* name;
        int (*run)();
    } checks[] = {{"loans", loans}, {"runtime_calls_outside_the_lock", runtime_calls_outside_the_lock},
                  {"copies_without_helpers", copies_without_helpers}};
    for (const auto& c : checks)
        if (argc == 2 && !strcmp(argv[1], c.name)) return c.run();
    fprintf(stderr, "no such check\n");
    return 2;
}
