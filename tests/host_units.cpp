// Host checks of parts of the library that need no GPU, run by
// test_host_units.py: each check is a name on the command line.
#include <cstdio>
#include <cstring>
#include <map>
#include <set>
#include <vector>

#include "sphk_buffers.hpp"

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

}  // namespace

int main(int argc, char **argv)
{
    if (argc == 2 && !std::strcmp(argv[1], "node_buffers")) return node_buffers();
    std::printf("no such check\n");
    return 2;
}
