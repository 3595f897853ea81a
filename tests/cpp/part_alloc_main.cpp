// A partitioned sweep's layout (ssgpu_parts.h) when the host runs out: every
// allocation of the layout, on whichever thread it is made, is made to fail in
// turn, and so is every thread that it starts.  Prints "ok" and the number of
// allocations if each failure reached the caller as std::bad_alloc, threads
// that could not be started changed nothing, and the layout afterwards is the
// one before.
#include <dlfcn.h>
#include <pthread.h>

#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <new>

static std::atomic<long> g_count{0}, g_fail_at{-1};
static std::atomic<long> g_threads{0}, g_most_threads{1L << 30};

void* operator new(size_t n) {
    if (g_count++ == g_fail_at) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) noexcept {
    using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    static Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
    if (g_threads++ >= g_most_threads) return EAGAIN;
    return real(t, a, f, arg);
}

#include "ssgpu_parts.h"

using namespace ssgpu;

int main() {
    const int m = 24, n = m * m * m;   // a 7-point grid
    std::vector<int> off(n + 1, 0), col, lev(n, 0);
    for (int i = 0; i < n; ++i) {
        const int x = i % m, y = i / m % m, z = i / m / m;
        if (z) col.push_back(i - m * m);
        if (y) col.push_back(i - m);
        if (x) col.push_back(i - 1);
        off[i + 1] = (int)col.size();
        lev[i] = x + y + z;
    }
    const PartChoice ch = part_intervals(n, true, 600);
    auto layout = [&]() { return part_layout(n, off.data(), col.data(), lev.data(), true, ch, 12); };
    const PartLayout ref = layout();
    auto same = [&](const PartLayout& L) {
        return L.order == ref.order && L.slot == ref.slot && L.src == ref.src && L.ext == ref.ext &&
               L.part_step == ref.part_step && L.steps.size() == ref.steps.size();
    };
    g_count = 0;
    if (!same(layout())) return std::puts("a second layout differs"), 1;
    const long total = g_count;
    for (long k = 0; k < total; k += k < 200 ? 1 : 7) {
        g_count = 0;
        g_fail_at = k;
        bool thrown = false;
        try {
            const PartLayout L = layout();
            if (!same(L)) return std::printf("layout differs after failure %ld\n", k), 1;
        } catch (const std::bad_alloc&) {
            thrown = true;
        }
        g_fail_at = -1;
        // a thread's own bookkeeping may fail instead: then one thread fewer, and the layout is whole
        if (!thrown && g_count <= k) return std::printf("failure %ld was not reached\n", k), 1;
    }
    for (long k = 0; k < 20; ++k) {
        g_threads = 0;
        g_most_threads = k;
        if (!same(layout())) return std::printf("layout differs with %ld threads\n", k), 1;
    }
    g_most_threads = 1L << 30;
    if (!same(layout())) return std::puts("the layout afterwards differs"), 1;
    std::printf("ok %ld\n", total);
    return 0;
}
