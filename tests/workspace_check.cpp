// Compiled and run by tests/test_workspace.py: the pool of device blocks
// (nadvibs_amd/csrc/nv_workspace.hpp) over a counting allocator with a limit.
// Prints "ok" or what does not hold.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

#include "nv_workspace.hpp"

static std::mutex mu;
static std::map<void *, size_t> live;
static size_t held = 0, limit = 1000, calls = 0;

struct Counting {
    static int get(void **p, size_t bytes) {
        std::lock_guard<std::mutex> lock(mu);
        ++calls;
        if (held + bytes > limit) return 2;
        *p = std::malloc(1);
        live[*p] = bytes;
        held += bytes;
        return 0;
    }
    static void put(void *p) {
        std::lock_guard<std::mutex> lock(mu);
        held -= live.at(p);
        live.erase(p);
        std::free(p);
    }
};
using Pool = nv::BlockPool<Counting>;

#define CHECK(c)                                         \
    do {                                                 \
        if (!(c)) {                                      \
            std::printf("line %d: %s\n", __LINE__, #c);  \
            return 1;                                    \
        }                                                \
    } while (0)

int main() {
    {
        Pool pool(500);
        Pool::Block a, b, c;
        CHECK(pool.take(400, &a) == 0 && pool.take(100, &b) == 0 && held == 500);
        pool.give(a);
        pool.give(b);
        CHECK(held == 500);  // both kept
        const size_t before = calls;
        CHECK(pool.take(90, &c) == 0 && c.p == b.p && c.bytes == 100);  // the smallest that fits
        CHECK(pool.take(400, &b) == 0 && b.p == a.p && calls == before);
        pool.give(c);
        pool.give(b);
        // more than the cap in all: the longest idle goes
        CHECK(pool.take(450, &a) == 0 && held == 950);
        pool.give(a);
        CHECK(held == 450);
        // one above the cap is not kept
        CHECK(pool.take(501, &a) == 0);
        pool.give(a);
        CHECK(held == 450);
        // idle blocks make room
        CHECK(pool.take(800, &a) == 0 && held == 800);
        CHECK(pool.take(300, &b) != 0 && b.p == nullptr && held == 800);
        pool.give(a);
        pool.give(b);
        CHECK(held == 0 && !pool.trim());
        CHECK(pool.take(10, &a) == 0);
        pool.give(a);
        CHECK(pool.trim() && held == 0 && !pool.trim());
    }
    // threads: no block has two takers, and the kept bytes stay within the cap
    limit = (size_t)1 << 40;
    Pool pool(300);
    std::mutex um;
    std::set<void *> used;
    std::atomic<int> bad{0};
    std::vector<std::thread> th;
    for (int t = 0; t < 8; ++t)
        th.emplace_back([&, t] {
            unsigned x = 77 + t;
            for (int k = 0; k < 2000; ++k) {
                x = x * 1664525u + 1013904223u;
                Pool::Block b;
                if (pool.take(1 + (x >> 16) % 150, &b) != 0) ++bad;
                {
                    std::lock_guard<std::mutex> lock(um);
                    if (!used.insert(b.p).second) ++bad;
                }
                std::this_thread::yield();
                {
                    std::lock_guard<std::mutex> lock(um);
                    used.erase(b.p);
                }
                pool.give(b);
            }
        });
    for (auto &t : th) t.join();
    CHECK(bad == 0);
    CHECK(held <= 300);
    pool.trim();
    CHECK(held == 0 && live.empty());
    std::printf("ok\n");
    return 0;
}
