// Exercises csrc/uw_blocks.h on the host (tests/test_block_pool.py builds and runs it): random takes and
// gives against the pool's promises, with made-up addresses.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <set>

#include "../../underwaterworld_amd/csrc/uw_blocks.h"

#define CHECK(c)                                              \
    do {                                                      \
        if (!(c)) {                                           \
            std::printf("line %d: %s\n", __LINE__, #c);       \
            return 1;                                         \
        }                                                     \
    } while (0)

int main() {
    for (size_t n : {size_t(1), size_t(4096), size_t(65536), size_t(65537), size_t(1) << 20, (size_t(1) << 20) + 1, size_t(200) << 20}) {
        const size_t r = uw_block_pool::rounded(n);
        CHECK(r >= n && uw_block_pool::rounded(r) == r);
        CHECK(n < 65536 ? r - n < 8192 : r - n <= n / 8);
    }
    // slack: a block four times the request stays where it is, one a quarter above it serves
    {
        uw_block_pool pool;
        uw_block b;
        auto none = [](const uw_block&) { std::abort(); };
        pool.give({reinterpret_cast<void*>(1), size_t(40) << 20}, none);
        CHECK(!pool.take(size_t(10) << 20, &b) && !pool.take(size_t(31) << 20, &b) && !pool.take(size_t(41) << 20, &b));
        pool.give({reinterpret_cast<void*>(2), size_t(36) << 20}, none);
        CHECK(pool.take(size_t(35) << 20, &b) && b.p == reinterpret_cast<void*>(2));
        CHECK(pool.take(size_t(32) << 20, &b) && b.p == reinterpret_cast<void*>(1) && pool.count() == 0 && pool.bytes() == 0);
    }
    // a full pool lets the longest kept go, and keeps the new block
    {
        uw_block_pool pool;
        uintptr_t next = 1, dropped = 0;
        for (int i = 0; i < 100; ++i)
            pool.give({reinterpret_cast<void*>(next++), 8192}, [&](const uw_block& b) {
                ++dropped;
                if (b.p != reinterpret_cast<void*>(dropped)) std::abort();
            });
        CHECK(dropped == 36 && pool.count() == 64);
        pool.give({reinterpret_cast<void*>(next++), uw_block_pool::kMaxBytes}, [&](const uw_block&) { ++dropped; });
        CHECK(dropped == 100 && pool.count() == 1 && pool.bytes() == uw_block_pool::kMaxBytes);
        pool.give({reinterpret_cast<void*>(next++), uw_block_pool::kMaxBytes + 1}, [&](const uw_block& b) {
            if (b.bytes != uw_block_pool::kMaxBytes + 1) std::abort();
            ++dropped;
        });
        CHECK(dropped == 101 && pool.count() == 1);
    }
    // every block is with one owner at a time, and nothing is lost
    uw_block_pool pool;
    std::set<uintptr_t> kept, out;
    static uw_block held[256];
    int nheld = 0;
    uintptr_t next = 1;
    uint64_t x = 88172645463325252ull;
    auto rnd = [&] { return x ^= x << 13, x ^= x >> 7, x ^= x << 17, x; };
    bool bad = false;
    auto drop = [&](const uw_block& b) { bad = bad || kept.erase(reinterpret_cast<uintptr_t>(b.p)) == 0; };
    for (int i = 0; i < 200000; ++i) {
        if (nheld == 0 || (nheld < 256 && rnd() % 2)) {
            const size_t need = uw_block_pool::rounded(size_t(1) << (rnd() % 27) | rnd() % 5000);
            uw_block b;
            if (pool.take(need, &b)) {
                CHECK(kept.erase(reinterpret_cast<uintptr_t>(b.p)) == 1 && b.bytes >= need && b.bytes <= need + need / 4 + 8192);
            } else {
                b = {reinterpret_cast<void*>(next++), need};
            }
            CHECK(out.insert(reinterpret_cast<uintptr_t>(b.p)).second);
            held[nheld++] = b;
        } else {
            const int k = int(rnd() % uint64_t(nheld));
            const uw_block b = held[k];
            held[k] = held[--nheld];
            CHECK(out.erase(reinterpret_cast<uintptr_t>(b.p)) == 1);
            kept.insert(reinterpret_cast<uintptr_t>(b.p));
            pool.give(b, drop);
        }
        CHECK(!bad && pool.bytes() <= uw_block_pool::kMaxBytes && pool.count() <= uw_block_pool::kMaxCount && size_t(pool.count()) == kept.size());
    }
    pool.clear(drop);
    CHECK(!bad && kept.empty() && pool.count() == 0 && pool.bytes() == 0);
    std::printf("ok\n");
    return 0;
}
