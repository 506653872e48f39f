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
    MultiInput in;
    in.special = special;
    in.own_ptr = t.own_ptr;
    in.n2e_ptr.assign(nn + 1, 0);
    for (int32_t c : conn) {
        in.conn.push_back(t.inv[c]);
        in.n2e_ptr[t.inv[c] + 1]++;
    }
    for (int n = 0; n < nn; ++n) in.n2e_ptr[n + 1] += in.n2e_ptr[n];
    in.n2e.resize(in.conn.size());
    std::vector<int32_t> at(in.n2e_ptr.begin(), in.n2e_ptr.end() - 1);
    for (int i = 0; i < int(in.conn.size()); ++i) in.n2e[at[in.conn[i]]++] = i;
    for (int e = 0; e < ne; ++e) {
        in.lam.push_back(1.0 + e);
        in.mu.push_back(2.0 + e);
    }
    // The plan and its arrays, as one list of numbers.
    auto plan = [&](std::vector<double> &v) {
        HostMulti h;
        if (!make_multi(in, 4, 4, 1024, h)) return false;
        const size_t k = h.tiles.size(), m = k * h.ne;
        std::vector<int32_t> cnt(k * 2 * 5), node(k * h.ns);
        std::vector<uint16_t> econn(m * 4), ncor(k * h.nu * 4), egeo(m);
        std::vector<double> lam(m), mu(m);
        fill_multi(h, in, 968, MultiArrays{cnt.data(), node.data(), econn.data(), ncor.data(), egeo.data(), lam.data(),
                                           mu.data()});
        v = {double(k), double(h.ns), double(h.ne), double(h.nu)};
        for (int32_t x : cnt) v.push_back(x);
        for (int32_t x : node) v.push_back(x);
        for (uint16_t x : econn) v.push_back(x);
        for (uint16_t x : ncor) v.push_back(x);
        for (uint16_t x : egeo) v.push_back(x);
        v.insert(v.end(), lam.begin(), lam.end());
        v.insert(v.end(), mu.begin(), mu.end());
        // Every owned node of every tile has all its corners, at its own slot.
        for (size_t ti = 0; ti < k; ++ti)
            for (int n = t.own_ptr[ti]; n < t.own_ptr[ti + 1]; ++n) {
                const int sl = n - t.own_ptr[ti];
                if (node[ti * h.ns + sl] != n) return false;
                int corners = 0;
                for (int a = 0; a < 4; ++a) {
                    const int e = ncor[(ti * h.nu + sl) * 4 + a];
                    if (e == 968) continue;
                    if (econn[(ti * h.ne + e) * 4 + a] != sl) return false;
                    ++corners;
                }
                if (corners != in.n2e_ptr[n + 1] - in.n2e_ptr[n]) return false;
            }
        return true;
    };
    std::vector<double> a, b;
    if (!plan(a)) return std::puts("no plan"), 1;
    for (int allowed : {0, 1}) {  // refused at once, and after one thread has started
        threads_left = allowed;
        const bool ok = plan(b);
        threads_left = 1 << 30;
        if (!ok || a != b) return std::puts("refused threads changed the plan"), 1;
    }
    refuse_in_workers = true;
    const bool made = plan(b);
    refuse_in_workers = false;
    // (Whether a worker reaches an allocation before the first thread has built every tile is up to the
    // system: both answers are right, an abort is not.)
    std::printf("ok, %d tiles, plan with refused memory: %s\n", t.ntiles, made ? "made" : "left out");
    return 0;
}
