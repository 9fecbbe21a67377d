// Host checks of parts of the library that need no GPU, run by
// test_host_units.py: each check is a name on the command line.
#include <cstdio>
#include <cstring>
#include <map>
#include <set>
#include <vector>

#include "sphk_buffers.hpp"
#include "sphk_spans.hpp"

#define CHECK(c)                                                        \
    do {                                                                \
        if (!(c)) {                                                     \
            std::printf("line %d: %s does not hold\n", __LINE__, #c);   \
            return 1;                                                   \
        }                                                               \
    } while (0)

namespace {

// Addresses without memory behind them; the allocation number `fail_at`
// (counted from 0) fails, and so does what would go beyond `most` bytes.
struct FakeAlloc {
    using Error = int;
    using Stream = int;
    static constexpr int ok = 0;
    static long fail_at, count, waits;
    static size_t next, held, most;
    static std::map<void *, size_t> live;

    static void reset(long fail = -1, size_t limit = SIZE_MAX)
    {
        fail_at = fail;
        count = waits = 0;
        most = limit;
    }
    static int alloc(void **p, size_t bytes)
    {
        if (count++ == fail_at || bytes > most - held) return 2;
        next += 4096;
        *p = reinterpret_cast<void *>(next);
        live[*p] = bytes;
        held += bytes;
        return ok;
    }
    static void free(void *p)
    {
        held -= live.at(p);   // throws for a block freed twice
        live.erase(p);
    }
    static int copy(void *, const void *, size_t, int) { return ok; }
    static int wait(int)
    {
        waits++;
        return ok;
    }
};
long FakeAlloc::fail_at, FakeAlloc::count, FakeAlloc::waits;
size_t FakeAlloc::next = 1 << 20, FakeAlloc::held, FakeAlloc::most;
std::map<void *, size_t> FakeAlloc::live;

struct Rec64 {
    char b[64];
};

// A build that runs out of memory at any of its node arrays, then builds of
// the same, a smaller and a larger size: every array holds what the handle
// says it does.
int node_buffers()
{
    using Nodes = sphk::NodeBuffers<FakeAlloc, Rec64, Rec64>;
    const long arrays = 20;
    for (long fail = 0; fail < arrays; fail++)
        for (size_t after : {900, 1000, 400, 3000}) {
            Nodes nb;
            FakeAlloc::reset();
            CHECK(nb.reserve_nodes(300, 500, 0) == 0);
            CHECK(FakeAlloc::count == arrays);
            FakeAlloc::reset(fail);
            CHECK(nb.reserve_nodes(1000, 700, 0) != 0);
            CHECK(nb.node_cap == 500);
            FakeAlloc::reset();
            CHECK(nb.reserve_nodes(after, 16, 0) == 0);
            CHECK(nb.node_cap >= after);
            for (auto *a : {&nb.begin, &nb.end, &nb.child, &nb.nchild, &nb.level, &nb.parent})
                CHECK(FakeAlloc::live.at(a->p) >= nb.node_cap * sizeof(int32_t));
            for (auto *a : {&nb.len, &nb.mm, &nb.mx, &nb.my, &nb.mz, &nb.me, &nb.sx, &nb.sy, &nb.sz, &nb.se})
                CHECK(FakeAlloc::live.at(a->p) >= nb.node_cap * sizeof(double));
            for (auto *a : {&nb.box_lo, &nb.box_hi}) CHECK(FakeAlloc::live.at(a->p) >= 3 * nb.node_cap * sizeof(double));
            for (auto *a : {&nb.brec, &nb.mrec}) CHECK(FakeAlloc::live.at(a->p) >= nb.node_cap * sizeof(Rec64));
            nb.release_nodes();
            CHECK(FakeAlloc::live.empty() && FakeAlloc::held == 0);
        }
    return 0;
}

// Builds of the three kinds in many orders and sizes, in memory and with a
// bound that do not always suffice.  A list lies where it was put until its
// array goes to another kind; then it has been packed.  What is held stays
// within the bound.
int list_rooms()
{
    unsigned seed = 1;
    auto rnd = [&](unsigned m) { return (seed = seed * 1664525u + 1013904223u) / 65536u % m; };
    long shared = 0, apart = 0, none = 0, failed = 0;
    for (int round = 0; round < 4000; round++) {
        const size_t bound = 4000;
        FakeAlloc::reset(-1, rnd(2) ? SIZE_MAX : 4 * (size_t)(500 + rnd(6000)));
        {
            sphk::ListRooms<FakeAlloc> rooms(bound);
            int packed[3] = {0, 0, 0}, refuse = rnd(4) == 0;
            auto pack = [&](int k) {
                if (refuse && rnd(8) == 0) return -5;
                packed[k]++;
                return 0;
            };
            for (int step = 0; step < 12; step++) {
                const int kind = (int)rnd(3);
                const size_t n = 1 + rnd(rnd(3) ? 600 : 2000), nn = kind == 2 ? 1 + rnd(rnd(3) ? 300 : 2000) : 0;
                int was[3], before[3], rc = 0;
                for (int k = 0; k < 3; k++) {
                    was[k] = rooms.lies[k];
                    before[k] = packed[k];
                }
                const int at = rooms.take(kind, n, nn, 0, pack, rc);
                CHECK(rooms.held() <= bound);
                CHECK(rooms.lies[kind] == -1 && packed[kind] == before[kind]);
                for (int k = 0; k < 3; k++) {
                    if (k == kind) continue;
                    if (rooms.lies[k] >= 0)        // where it was, and not where the new list goes
                        CHECK(rooms.lies[k] == was[k] && rooms.lies[k] != at && rooms.of[was[k]].cap > 0 && packed[k] == before[k]);
                    else                           // taken out once, if it lay anywhere
                        CHECK(packed[k] == before[k] + (was[k] >= 0));
                }
                if (rc) {
                    CHECK(at == -1 && rc == -5);
                    failed++;
                } else if (at < 0) {
                    CHECK(FakeAlloc::most != SIZE_MAX);
                    none++;
                } else {
                    CHECK(rooms.of[at].cap >= n && FakeAlloc::live.at(rooms.of[at].p) >= 4 * n);
                    CHECK(rooms.nodes.cap >= nn && (!nn || FakeAlloc::live.at(rooms.nodes.p) >= 4 * nn));
                    (at == kind ? apart : shared)++;
                    rooms.lies[kind] = at;
                }
            }
            rooms.release();
        }
        CHECK(FakeAlloc::live.empty() && FakeAlloc::held == 0);
    }
    CHECK(shared > 1000 && apart > 1000 && none > 100 && failed > 100);
    // sizes that fit: every kind keeps its own, nothing is packed or allocated again
    FakeAlloc::reset();
    sphk::ListRooms<FakeAlloc> rooms(4000);
    for (int step = 0; step < 9; step++) {
        int rc = 0;
        const int at = rooms.take(step % 3, 1000, step % 3 == 2 ? 500 : 0, 0, [](int) { return -1; }, rc);
        CHECK(at == step % 3 && rc == 0 && FakeAlloc::count == std::min(step + 1 + (step >= 2), 4));
        rooms.lies[at] = at;
    }
    rooms.release();
    return 0;
}

struct CountedKeys {
    const std::vector<uint64_t> &k;
    mutable long reads = 0;
    uint64_t operator[](size_t i) const
    {
        reads++;
        return k.at(i);   // throws beyond the array
    }
};

// The deepest level whose cell holds more than n_leaf particles against its
// definition (cells counted level by level), and the keys read for it: the
// logarithm of n_leaf, not n_leaf.
int leaf_levels()
{
    uint64_t seed = 7;
    auto rnd = [&]() {
        seed = seed * 6364136223846793005ull + 1442695040888963407ull;
        return seed >> 1;   // 63 bits
    };
    for (int n : {1, 2, 513, 3000, 20000})
        for (int kind = 0; kind < 4; kind++) {
            std::vector<uint64_t> key(n);
            for (auto &k : key) {
                k = rnd();
                if (kind == 1) k >>= k % 50;                  // few at the top, many in a corner
                if (kind == 2 && k % 3) k = 1234567;          // two thirds at one place
                if (kind == 3) k = k % 40 * 1000003;          // cells that cannot be split
            }
            std::sort(key.begin(), key.end());
            std::vector<std::vector<int>> held(sphk::kMaxLevel + 1, std::vector<int>(n));
            for (int L = 0; L <= sphk::kMaxLevel; L++)
                for (int b = 0; b < n;) {
                    const int shift = 3 * (sphk::kMaxLevel - L);
                    int e = b;
                    while (e < n && key[e] >> shift == key[b] >> shift) e++;
                    for (int i = b; i < e; i++) held[L][i] = e - b;
                    b = e;
                }
            for (int n_leaf : {1, 2, 8, 512, 513, 600, 2999, 3000, 3001, 10000, 30000}) {
                int log2 = 0;
                while ((1 << log2) < n_leaf) log2++;
                for (int i = 0; i < n; i += 1 + n / 700) {
                    int want = -1;
                    for (int L = 0; L <= sphk::kMaxLevel; L++)
                        if (held[L][i] > n_leaf) want = L;
                    CountedKeys counted{key};
                    CHECK(sphk::deepest_full_level(counted, n, n_leaf, i) == want);
                    CHECK(counted.reads <= 5 * (log2 + 3));
                }
            }
        }
    return 0;
}

}  // namespace

int main(int argc, char **argv)
{
    if (argc == 2 && !std::strcmp(argv[1], "node_buffers")) return node_buffers();
    if (argc == 2 && !std::strcmp(argv[1], "list_rooms")) return list_rooms();
    if (argc == 2 && !std::strcmp(argv[1], "leaf_levels")) return leaf_levels();
    std::printf("no such check\n");
    return 2;
}
