// Host check of the contexts' device memory pools (csrc/graph.h) against a device
// of 64 MiB made here: hipMalloc counts and fails past it, hipFree takes only what it
// gave.  Prints "ok" or the first thing that is wrong.
#include "graph.h"

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <thread>

static std::mutex dev_mu;
static std::map<void *, size_t> dev;
static size_t dev_used = 0;
static const size_t DEV = (size_t)64 << 20;
static size_t dev_size = DEV;

extern "C" hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> lk(dev_mu);
    if (dev_used + n > dev_size) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    dev[*p] = n;
    dev_used += n;
    return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> lk(dev_mu);
    auto it = dev.find(p);
    if (it == dev.end()) std::printf("free of an unknown block\n"), std::exit(1);
    dev_used -= it->second;
    dev.erase(it);
    std::free(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError(void) { return hipSuccess; }
extern "C" const char *hipGetErrorString(hipError_t) { return "out of memory"; }

namespace vnm {
int set_error(int code, const char *, ...) { return code; }
}  // namespace vnm

using namespace vnm;
#define CHECK(x) \
    do { \
        if (!(x)) std::printf("line %d: %s\n", __LINE__, #x), std::exit(1); \
    } while (0)

constexpr size_t MB = 1 << 20;

int main() {
    {
        auto a = std::make_shared<DevPool>(), b = std::make_shared<DevPool>();
        {
            PoolScope s(a);
            DBuf<char> x, y;
            CHECK(x.alloc(30 * MB) == VNM_OK && y.alloc(30 * MB) == VNM_OK);
        }
        CHECK(dev_used == 60 * MB);  // idle in a
        {  // another context's call takes it
            PoolScope s(b);
            DBuf<char> x;
            CHECK(x.alloc(60 * MB) == VNM_OK);
            CHECK(x.alloc(50 * MB) == VNM_OK);  // and its own idle block serves a smaller one
        }
        CHECK(dev_used == 60 * MB);
        {  // so does a call outside any scope, of the very last byte
            DBuf<char> x;
            CHECK(x.alloc(DEV) == VNM_OK);
            CHECK(dev_used == DEV);
            DBuf<char> y;
            CHECK(y.alloc(1) == VNM_E_OOM && y.p == nullptr);
            PoolScope s(a);
            CHECK(y.alloc(1) == VNM_E_OOM && y.p == nullptr);
        }
        CHECK(dev_used == 0);
        {  // a size that fits as it is but not rounded up
            DBuf<char> x, y, z;
            CHECK(z.alloc(5) == VNM_OK);
            PoolScope s(a);
            CHECK(x.alloc(60 * MB) == VNM_OK && dev_used == 60 * MB + 5);
            CHECK(y.alloc(4 * MB - 5) == VNM_OK && dev_used == DEV);
        }
        CHECK(dev_used == DEV - 5);
        a->trim();
        CHECK(dev_used == 0);
        // a block goes back to the pool it came from, also without its scope and after a swap
        DBuf<int> u, v;
        {
            PoolScope s(a);
            CHECK(u.alloc(1000) == VNM_OK);
        }
        {
            PoolScope s(b);
            CHECK(v.alloc(9 * MB) == VNM_OK);
        }
        u.swap(v);
        u.release();
        v.release();
        a->trim();
        CHECK(dev_used >= 36 * MB);
        b->trim();
        CHECK(dev_used == 0);
    }
    {  // objects that outlive their context hold its pool
        auto a = std::make_shared<DevPool>();
        DBuf<char> x;
        {
            PoolScope s(a);
            DBuf<char> y;
            CHECK(x.alloc(MB) == VNM_OK && y.alloc(MB) == VNM_OK);
        }
        a.reset();
        CHECK(dev_used == 2 * MB);
        x.release();
        CHECK(dev_used == 0);
    }
    {  // no more than POOL_IDLE stays idle
        dev_size = 2 * POOL_IDLE;
        auto a = std::make_shared<DevPool>();
        {
            PoolScope s(a);
            DBuf<char> x[30];
            for (auto &q : x) CHECK(q.alloc(100 * MB) == VNM_OK);
        }
        CHECK(dev_used > POOL_IDLE / 2 && dev_used <= POOL_IDLE);
        a.reset();
        CHECK(dev_used == 0);
        dev_size = DEV;
    }
    {  // contexts in threads on a device that is nearly full: every call gets its memory
        bool ok[4] = {};
        std::vector<std::thread> ts;
        for (int t = 0; t < 4; ++t)
            ts.emplace_back([t, &ok] {
                unsigned r = 12345u * (t + 1);
                bool good = true;
                for (int round = 0; round < 20; ++round) {
                    auto a = std::make_shared<DevPool>();
                    PoolScope s(a);
                    for (int i = 0; i < 50; ++i) {
                        r = r * 1664525u + 1013904223u;
                        DBuf<char> x;
                        good &= x.alloc((r >> 8) % (15 * MB) + 1) == VNM_OK;
                    }
                }
                ok[t] = good;
            });
        for (auto &t : ts) t.join();
        for (bool o : ok) CHECK(o);
        CHECK(dev_used == 0);
    }
    std::printf("ok\n");
}
