// sphk_buffers.hpp -- device arrays that grow, and two groups of them in a
// tree handle whose sizes belong together: the node arrays and the rooms of
// the lists.  The allocator is a parameter (A), so that allocations that fail
// can be tried on the host.
//
// A: Error (a type) and ok (its value for success), Stream (a type), and
//   static Error alloc(void **p, size_t bytes)   (a failure leaves no error behind)
//   static void free(void *p)
//   static Error copy(void *to, const void *from, size_t bytes, Stream st)
//   static Error wait(Stream st)
#ifndef SPHK_BUFFERS_HPP
#define SPHK_BUFFERS_HPP

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace sphk {

// Device array with capacity.
template <typename T, class A>
struct DeviceArray {
    T *p = nullptr;
    size_t cap = 0;

    // Room for n elements.  Where that fails the array is as it was.
    typename A::Error reserve(size_t n, bool keep, typename A::Stream st)
    {
        if (n <= cap) return A::ok;
        void *q = nullptr;
        typename A::Error e = A::alloc(&q, n * sizeof(T));
        if (e != A::ok) return e;
        if (keep && p && cap) e = A::copy(q, p, cap * sizeof(T), st);
        // queued work may still read the old block: wait before freeing it
        if (e == A::ok && p) e = A::wait(st);
        if (e != A::ok) {
            A::free(q);
            return e;
        }
        if (p) A::free(p);
        p = static_cast<T *>(q);
        cap = n;
        return A::ok;
    }
    void release()
    {
        if (p) A::free(p);
        p = nullptr;
        cap = 0;
    }
};

// The arrays with an entry per node (box_lo and box_hi: [3][node_cap]; Box and
// Mac: the node records of the list walks).  node_cap nodes fit in every one
// of them: it grows after the last array has, so a build that runs out of
// memory among them leaves no array that a later build takes for larger than
// it is.
template <class A, typename Box, typename Mac>
struct NodeBuffers {
    DeviceArray<int32_t, A> begin, end, child, nchild, level, parent;
    DeviceArray<double, A> len, box_lo, box_hi, mm, mx, my, mz, me, sx, sy, sz, se;
    DeviceArray<Box, A> brec;
    DeviceArray<Mac, A> mrec;
    size_t node_cap = 0;

    // Room for nn nodes (for at least `want` where the arrays have to grow);
    // the contents are not kept.
    typename A::Error reserve_nodes(size_t nn, size_t want, typename A::Stream st)
    {
        if (nn <= node_cap) return A::ok;
        const size_t cap = std::max(nn, want);
        typename A::Error e = A::ok;
        auto grow = [&](auto &a, size_t n) {
            if (e == A::ok) e = a.reserve(n, false, st);
        };
        for (auto *a : {&begin, &end, &child, &nchild, &level, &parent}) grow(*a, cap);
        for (auto *a : {&len, &mm, &mx, &my, &mz, &me, &sx, &sy, &sz, &se}) grow(*a, cap);
        for (auto *a : {&box_lo, &box_hi}) grow(*a, 3 * cap);
        grow(brec, cap);
        grow(mrec, cap);
        if (e == A::ok) node_cap = cap;
        return e;
    }
    void release_nodes()
    {
        for (auto *a : {&begin, &end, &child, &nchild, &level, &parent}) a->release();
        for (auto *a : {&len, &box_lo, &box_hi, &mm, &mx, &my, &mz, &me, &sx, &sy, &sz, &se}) a->release();
        brec.release();
        mrec.release();
        node_cap = 0;
    }
};

// Scratch of the one-pass list builds: an array of rooms for each of the three
// kinds of lists, so that a list stays in its rooms while another is built
// (packed first, wanted or not, the three lists of 10^6 particles took 3.54 ms
// against 3.48, for 0.2 GB less at 51463 walks), and one for the nodes of the
// long list.  All four hold at most `most` entries together.  Where another
// array would go beyond that, or does not fit in memory, the kinds share the
// largest one there is, and a list that lies in it is taken out first.
template <class A>
struct ListRooms {
    DeviceArray<int32_t, A> of[3], nodes;
    int lies[3] = {-1, -1, -1};   // the array in which a kind's list lies, -1: in none
    size_t most;

    explicit ListRooms(size_t most_) : most(most_) {}

    size_t held() const { return of[0].cap + of[1].cap + of[2].cap + nodes.cap; }

    // The array for n entries of `kind`, whose list before is given up, and
    // room for n_nodes; -1 if there is no memory for them.  pack(k) takes kind
    // k's list out of its rooms; if it fails its value is in rc, and -1 comes
    // back.
    template <class Pack>
    int take(int kind, size_t n, size_t n_nodes, typename A::Stream st, Pack &&pack, int &rc)
    {
        rc = 0;
        lies[kind] = -1;
        auto clear = [&](int a) {
            for (int k = 0; k < 3 && !rc; k++)
                if (lies[k] == a && !(rc = pack(k))) lies[k] = -1;
            return rc == 0;
        };
        const size_t more = (n > of[kind].cap ? n - of[kind].cap : 0) + (n_nodes > nodes.cap ? n_nodes - nodes.cap : 0);
        int use = kind;
        if (held() + more > most || of[kind].reserve(n, false, st) != A::ok) {
            use = 0;
            for (int k = 1; k < 3; k++)
                if (of[k].cap > of[use].cap) use = k;
            for (int k = 0; k < 3; k++) {
                if (k == use || !of[k].cap) continue;
                if (!clear(k) || A::wait(st) != A::ok) return -1;
                of[k].release();
            }
        }
        if (!clear(use)) return -1;
        if (of[use].reserve(n, false, st) != A::ok || nodes.reserve(n_nodes, false, st) != A::ok) return -1;
        return use;
    }
    void release()
    {
        for (int k = 0; k < 3; k++) {
            of[k].release();
            lies[k] = -1;
        }
        nodes.release();
    }
};

}  // namespace sphk

#endif
