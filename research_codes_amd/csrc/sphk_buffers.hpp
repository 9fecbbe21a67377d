// sphk_buffers.hpp -- device arrays that grow, and the node arrays of a tree
// handle, whose sizes belong together.  The allocator is a parameter (A), so
// that allocations that fail can be tried on the host.
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

}  // namespace sphk

#endif
