// BlockCache over a memory of limited size: blocks are reused, bounded by the cap,
// and given back (by both siblings) when an allocation does not fit otherwise.
#include <cstdio>
#include <set>

#include "../signinum_amd/csrc/host/block_cache.hpp"

static uint64_t used = 0, limit = 1000 << 10;
static std::unordered_map<void *, uint64_t> held;
struct Memory {
    static int alloc(void **out, uint64_t bytes) {
        if (used + bytes > limit) return 2;
        *out = new char;
        held[*out] = bytes;
        used += bytes;
        return 0;
    }
    static void free(void *p) {
        used -= held.at(p);
        held.erase(p);
        delete static_cast<char *>(p);
    }
};

#define CHECK(x)                                            \
    if (!(x)) {                                             \
        std::printf("line %d: %s\n", __LINE__, #x);         \
        return 1;                                           \
    }

int main() {
    constexpr uint64_t kb = 1 << 10;
    {
        sgn::BlockCache<Memory> big(900 * kb), small(300 * kb, &big);
        void *a = nullptr, *b = nullptr, *c = nullptr, *d = nullptr;
        CHECK(!big.get(600 * kb, &a) && !small.get(200 * kb, &b));
        big.put(a);
        small.put(b);
        CHECK(big.cached() == 600 * kb && small.cached() == 200 * kb && used == 800 * kb);
        CHECK(!small.get(190 * kb, &c) && c == b);  // reused
        small.put(c);
        // does not fit beside the cached blocks of either
        CHECK(!small.get(900 * kb, &c) && used == 900 * kb && big.cached() == 0);
        // nothing cached any more: the error stands, nothing is lost
        CHECK(small.get(200 * kb, &d) == 2 && used == 900 * kb);
        small.put(c);  // over its cap: freed
        CHECK(small.cached() == 0 && used == 0);
        CHECK(!big.get(500 * kb, &a));
        CHECK(!small.get(300 * kb, &b));
        small.put(b);
        CHECK(!small.alloc(400 * kb, &d) && used == 900 * kb && small.cached() == 0);
        CHECK(small.alloc(200 * kb, &c) == 2);
        Memory::free(d);
        big.put(a);
    }
    CHECK(used == 0);
    std::printf("ok\n");
    return 0;
}
