// Checks mg_hostpack.hpp with two buffers in turn, as the host-array entries use
// it: every thread count, and threads or memory refused after k threads.
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "mg_hostpack.hpp"

static thread_local int allocs_left = -1;  // -1: no limit
static int threads_left = -1;

void *operator new(std::size_t n) {
    if (allocs_left == 0) throw std::bad_alloc();
    if (allocs_left > 0) --allocs_left;
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) {
    using F = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static F real = (F)dlsym(RTLD_NEXT, "pthread_create");
    if (threads_left == 0) return EAGAIN;
    if (threads_left > 0) --threads_left;
    return real(t, a, f, x);
}

// nf fields of np pieces of 64 numbers packed into two buffers (in) or out of
// them; whether each arrived whole.  abandon: the owner leaves after that many
// fields; limit: allocations left while the threads are started.
static bool run(bool in, int nf, int np, int threads, int expect, int abandon = 1 << 20, int limit = -1) {
    const int n = np * 64;
    std::vector<std::vector<int>> host(nf, std::vector<int>(n)), dev(nf, std::vector<int>(n));
    std::vector<int> buf[2] = {std::vector<int>(n), std::vector<int>(n)};
    for (int f = 0; f < nf; ++f)
        for (int i = 0; i < n; ++i) (in ? host : dev)[f][i] = 1 + f * n + i;
    auto copy = [&](int f, int q) {
        for (int i = q * 64; i < (q + 1) * 64; ++i)
            if (in) buf[f & 1][i] = host[f][i];
            else host[f][i] = buf[f & 1][i];
    };
    {
        mf3d::PackTeam team(nf, np, copy);
        allocs_left = limit;
        const int got = team.start(threads);
        allocs_left = -1;
        if (got != expect) {
            std::printf("%d threads run, not %d (allocations %d)\n", got, expect, limit);
            return false;
        }
        if (!got) return true;
        if (in) team.open(2);
        for (int f = 0; !in && f < 2 && f < nf; ++f) buf[f] = dev[f];
        for (int f = 0; f < nf; ++f) {
            if (f == abandon) return true;  // the destructor ends threads that wait
            if (in) {
                team.wait(f);
                dev[f] = buf[f & 1];
                team.open(f + 3);
            } else {
                team.open(f + 1);
                team.wait(f);
                if (f + 2 < nf) buf[f & 1] = dev[f + 2];
            }
        }
    }
    return host == dev;
}

int main() {
    bool ok = true;
    for (int in = 0; in < 2; ++in)
        for (int nf : {1, 2, 4, 7, 8})
            for (int np : {1, 3, 50})
                for (int t = 1; t <= 8; ++t) ok = ok && run(in, nf, np, t, t);
    ok = ok && run(true, 7, 9, 12, 8);
    for (int k = 0; k < 6; ++k)
        for (int in = 0; in < 2; ++in) {
            threads_left = k;  // EAGAIN after k threads
            ok = ok && run(in, 7, 20, 6, k);
            threads_left = -1;
            ok = ok && run(in, 7, 20, 6, k, 1 << 20, k);  // a thread allocates once: its state
        }
    for (int in = 0; in < 2; ++in) ok = ok && run(in, 7, 20, 5, 5, 3);
    std::printf(ok ? "ok\n" : "failed\n");
    return ok ? 0 : 1;
}
