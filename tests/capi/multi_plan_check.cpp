// The multi-step plan when the system refuses threads or memory (test infrastructure, host only).
// make_multi over a grid of Quad4 tiles, with pthread_create and operator new of this program:
// thread refusals leave the plan as it is, allocation refusals in a worker end it with `false`.
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "svlg_tiles.hpp"

static int threads_left = 1 << 30;
static std::atomic<bool> refuse_in_workers{false};
static pthread_t main_thread;

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
    if (threads_left-- <= 0) return EAGAIN;
    return real(t, a, f, arg);
}

void *operator new(std::size_t n) {
    if (refuse_in_workers && !pthread_equal(pthread_self(), main_thread)) throw std::bad_alloc();
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

using namespace svlg;

int main() {
    main_thread = pthread_self();
    const int nx = 200, ny = 100, NX = nx + 1, NY = ny + 1, nn = NX * NY, ne = nx * ny;
    std::vector<double> X;
    std::vector<int32_t> conn, color;
    for (int j = 0; j < NY; ++j)
        for (int i = 0; i < NX; ++i) X.insert(X.end(), {double(i), double(j)});
    for (int j = 0; j < ny; ++j)
        for (int i = 0; i < nx; ++i) {
            const int n = j * NX + i;
            conn.insert(conn.end(), {n, n + 1, n + 1 + NX, n + NX});
            color.push_back((i & 1) | ((j & 1) << 1));
        }
    std::vector<uint8_t> special(nn, 0);
    HostTiles t;
    make_tiles(2, nn, ne, 4, X.data(), conn.data(), color.data(), 4, special.data(), 64, t);
    for (int32_t &c : conn) c = t.inv[c];
    auto plan = [&](HostMulti &h) { return make_multi(nn, ne, 4, conn.data(), special.data(), t.own_ptr, 4, 1024, h); };
    HostMulti a;
    if (!plan(a)) return std::puts("no plan"), 1;
    for (int allowed : {0, 1}) {  // refused at once, and after one thread has started
        HostMulti b;
        threads_left = allowed;
        const bool ok = plan(b);
        threads_left = 1 << 30;
        if (!ok || a.cnt != b.cnt || a.node != b.node || a.elem != b.elem || a.econn != b.econn || a.ncor != b.ncor)
            return std::puts("refused threads changed the plan"), 1;
    }
    HostMulti c;
    refuse_in_workers = true;
    const bool made = plan(c);
    refuse_in_workers = false;
    // (Whether a worker reaches an allocation before the first thread has built every tile is up to the
    // system: both answers are right, an abort is not.)
    std::printf("ok, %d tiles, plan with refused memory: %s\n", a.ntiles, made ? "made" : "left out");
    return 0;
}
