// sphk_dtree.hip -- device-resident octree, walk groups and interaction lists.
//
// The host builder (sphk_tree.cpp) and this one implement the same
// policies; this one keeps everything in HBM:
//   1. Morton keys over the bounding cube (block reduction, one key per
//      thread); sphk_morton_order_dev sorts (key, index) with a radix sort.
//   2. The octree's nodes, of all levels at once, from the sorted keys alone:
//      which cells begin at a particle follows from its key, its neighbour's
//      and those n_leaf places off (see span_kernel); nodes are counted per
//      block and level, scanned, and written to their places.  A level's
//      nodes are in key order, that is parent and octant order, as the host's
//      breadth-first loop numbers them.
//   3. Node boxes and monopoles bottom-up, one kernel per level (the top
//      levels in one), each node summing its particles (leaf) or children in
//      index order with FP contraction off, so the FP64 sums round as on the
//      host.
//   4. Groups: a node is a walk if it holds <= n_group particles (or is a
//      leaf) and its parent holds more; walks are ordered by first particle.
//   5. Lists, the host's element for element, each in one pass into a room
//      per walk: the host's depth-first traversal by one wave per walk, up
//      to 8 nodes opened at a time, a stack of pending entries in LDS; for
//      the short-range lists the reached leaves' particles are tested for
//      exact membership on the way.  A walk that overflows the stack is done
//      again with a larger one; one that overflows its room sends the build
//      through count and fill walks (8 lanes per walk) at scanned offsets.
#include <hip/hip_runtime.h>

#include <cstring>   // rocPRIM's iterator headers use memset without including it

#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <cstdint>
#include <limits>
#include <mutex>
#include <new>
#include <type_traits>
#include <vector>

#include "sphk.h"
#include "sphk_adjoint.h"
#include "sphk_buffers.hpp"
#include "sphk_device.hpp"
#include "sphk_dtree.h"
#include "sphk_internal.hpp"
#include "sphk_spans.hpp"

using sphk::kMaxLevel;
using sphk::set_error;
using sphk::shared_digits;

namespace {

constexpr int kBlock = 256;

#define SPHK_TRY(expr)                                                                          \
    do {                                                                                        \
        hipError_t e_ = (expr);                                                                 \
        if (e_ != hipSuccess) return set_error(SPHK_E_DEVICE, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

struct HipAlloc {
    using Error = hipError_t;
    using Stream = hipStream_t;
    static constexpr hipError_t ok = hipSuccess;
    static hipError_t alloc(void **p, size_t bytes)
    {
        const hipError_t e = hipMalloc(p, bytes);
        if (e != hipSuccess) (void)hipGetLastError();   // not left for the check of a later launch
        return e;
    }
    static void free(void *p) { (void)hipFree(p); }
    static hipError_t copy(void *to, const void *from, size_t bytes, hipStream_t st)
    {
        return hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToDevice, st);
    }
    static hipError_t wait(hipStream_t st) { return hipStreamSynchronize(st); }
};
template <typename T>
using DArr = sphk::DeviceArray<T, HipAlloc>;

struct DLists {
    DArr<int32_t> j_off, j_idx, s_off, s_idx;
    int64_t n_j = 0, n_s = 0;
    bool built = false;
    // of a list that was built in one walk and is not yet packed, whose
    // entries still lie in the handle's rooms: walk g's from g * room_j there,
    // the long list's nodes from g * room_s; j_off / s_off are final
    int64_t room_j = 0, room_s = 0;
};

__device__ __forceinline__ uint64_t spread3(uint64_t v)
{
    v &= 0x1fffff;
    v = (v | v << 32) & 0x1f00000000ffffULL;
    v = (v | v << 16) & 0x1f0000ff0000ffULL;
    v = (v | v << 8) & 0x100f00f00f00f00fULL;
    v = (v | v << 4) & 0x10c30c30c30c30c3ULL;
    v = (v | v << 2) & 0x1249249249249249ULL;
    return v;
}

// ---- bounding cube and keys ------------------------------------------------
// COPY: the positions go to cx, cy, cz on the way.
template <bool COPY>
__global__ __launch_bounds__(kBlock) void bbox_partial_kernel(int n, const double *__restrict__ x,
                                                              const double *__restrict__ y,
                                                              const double *__restrict__ z,
                                                              double *__restrict__ part, double *__restrict__ cx,
                                                              double *__restrict__ cy, double *__restrict__ cz)
{
    __shared__ double s[6][kBlock];
    const double inf = __builtin_inf();
    double lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf};
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const double p[3] = {x[i], y[i], z[i]};
        if (COPY) {
            cx[i] = p[0];
            cy[i] = p[1];
            cz[i] = p[2];
        }
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], p[d]);
            hi[d] = fmax(hi[d], p[d]);
        }
    }
    for (int d = 0; d < 3; d++) {
        s[d][threadIdx.x] = lo[d];
        s[3 + d][threadIdx.x] = hi[d];
    }
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int d = 0; d < 3; d++) {
                s[d][threadIdx.x] = fmin(s[d][threadIdx.x], s[d][threadIdx.x + w]);
                s[3 + d][threadIdx.x] = fmax(s[3 + d][threadIdx.x], s[3 + d][threadIdx.x + w]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int d = 0; d < 6; d++) part[6 * blockIdx.x + d] = s[d][0];
}

// frame = {origin x, y, z, side}: the bounding cube, side enlarged by 1e-9
// (the host's frame_of).
// One block combines the partial boxes (min and max are exact: any order
// gives the same box).
__global__ __launch_bounds__(kBlock) void bbox_final_kernel(int nb, const double *__restrict__ part,
                                                            double *__restrict__ frame)
{
    __shared__ double s[6][kBlock];
    const double inf = __builtin_inf();
    double lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf};
    for (int b = threadIdx.x; b < nb; b += kBlock)
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], part[6 * b + d]);
            hi[d] = fmax(hi[d], part[6 * b + 3 + d]);
        }
    for (int d = 0; d < 3; d++) {
        s[d][threadIdx.x] = lo[d];
        s[3 + d][threadIdx.x] = hi[d];
    }
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int d = 0; d < 3; d++) {
                s[d][threadIdx.x] = fmin(s[d][threadIdx.x], s[d][threadIdx.x + w]);
                s[3 + d][threadIdx.x] = fmax(s[3 + d][threadIdx.x], s[3 + d][threadIdx.x + w]);
            }
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    for (int d = 0; d < 3; d++) {
        lo[d] = s[d][0];
        hi[d] = s[3 + d][0];
    }
    double side = 0.;
    for (int d = 0; d < 3; d++) side = fmax(side, hi[d] - lo[d]);
    if (!(side > 0.)) side = 1.;
    side *= 1. + 1e-9;
    frame[0] = lo[0];
    frame[1] = lo[1];
    frame[2] = lo[2];
    frame[3] = side;
}

__device__ __forceinline__ uint64_t quant(double v, double o, double s)
{
    double t = (v - o) * s;
    if (!(t >= 0.)) t = 0.;
    const uint64_t u = (uint64_t)t;
    return u > 0x1fffff ? (uint64_t)0x1fffff : u;
}

__global__ __launch_bounds__(kBlock) void keys_kernel(int n, const double *__restrict__ x,
                                                      const double *__restrict__ y,
                                                      const double *__restrict__ z,
                                                      const double *__restrict__ frame,
                                                      uint64_t *__restrict__ key, int32_t *__restrict__ idx)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double s = double(1 << 21) / frame[3];
    key[i] = spread3(quant(x[i], frame[0], s)) << 2 | spread3(quant(y[i], frame[1], s)) << 1 |
             spread3(quant(z[i], frame[2], s));
    if (idx) idx[i] = i;
}

// Sets up the frame and keys of n particles (queued on st); with copies, the
// positions are copied to copies[0..2] first and the keys made from those.
int make_keys(int n, const double *x, const double *y, const double *z, hipStream_t st, DArr<double> &part,
              DArr<double> &frame, DArr<uint64_t> &key, int32_t *idx, double *const *copies = nullptr)
{
    const int nb = std::min(1024, (n + kBlock - 1) / kBlock);
    SPHK_TRY(part.reserve(6 * (size_t)nb, false, st));
    SPHK_TRY(frame.reserve(4, false, st));
    SPHK_TRY(key.reserve(n, false, st));
    if (copies) {
        hipLaunchKernelGGL(bbox_partial_kernel<true>, dim3(nb), dim3(kBlock), 0, st, n, x, y, z, part.p, copies[0],
                           copies[1], copies[2]);
        x = copies[0];
        y = copies[1];
        z = copies[2];
    } else {
        hipLaunchKernelGGL(bbox_partial_kernel<false>, dim3(nb), dim3(kBlock), 0, st, n, x, y, z, part.p, nullptr,
                           nullptr, nullptr);
    }
    hipLaunchKernelGGL(bbox_final_kernel, dim3(1), dim3(kBlock), 0, st, nb, part.p, frame.p);
    hipLaunchKernelGGL(keys_kernel, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, n, x, y, z,
                       frame.p, key.p, idx);
    SPHK_TRY(hipGetLastError());
    return SPHK_OK;
}

// ---- octree levels ---------------------------------------------------------
struct NodeArrays {
    int32_t *begin, *end, *child, *nchild, *level, *parent;
    double *len;
};

// A node is a cell (level L: equal first L key digits) that is the root or
// whose parent cell holds more than n_leaf particles; it begins at its first
// particle.  So the nodes that begin at particle i are those of the levels
//   c + 1 .. min(l + 1, kMaxLevel),
// c the digits key[i] shares with key[i - 1] (-1 for i = 0) and l the deepest
// level at which i's cell holds more than n_leaf particles: the most digits
// shared by the ends of any n_leaf + 1 consecutive particles with i among
// them (-1 if there are none).  All levels are built at once from these
// spans: a count kernel, scan kernels and a write kernel per level, each with
// a host read of the level's size, made a rebuild latency-bound (57 launches
// and 10 reads at 10^6 particles; rebuild and the three lists 6.5 -> 5.7 ms,
// a KDK step of 2x10^5 particles 5.2 -> 4.2 ms without them).
constexpr int kLevels = kMaxLevel + 1;
constexpr int kSpanTile = 1024;   // particles per block of the span, node and group kernels
// n_leaf up to this: window ends compared once per block, in LDS; larger: by
// bisection, as the windows' cost grows with n_leaf.  A build of 10^6
// particles in us, windows / bisection: n_leaf 8 366 / 395, 64 438 / 465, 128
// 576 / 577, 256 886 / 869, 512 1256 / 1202, and beyond (windows read from
// memory) 513 1648 / 1174, 2000 5462 / 3601, 10^4 18386 / 8944, most of which
// is the serial sums over such leaves.
constexpr int kSpanHalo = 512;

struct Span {
    int8_t lo, hi;
};

// Spans of all particles, the number of nodes that begin in each block per
// level (hist, level-major), and *unsorted set if the keys are not in order.
__global__ __launch_bounds__(kSpanTile) void span_kernel(int n, const uint64_t *__restrict__ key, int n_leaf,
                                                         Span *__restrict__ span, int32_t *__restrict__ hist,
                                                         int32_t *__restrict__ head, int *__restrict__ unsorted)
{
    __shared__ int8_t ends[kSpanTile + kSpanHalo];   // digits shared by the ends of window a
    __shared__ int cnt[kLevels];
    const int t = threadIdx.x, i0 = blockIdx.x * kSpanTile, i = i0 + t;
    auto window = [&](int a) { return a >= 0 && a + n_leaf < n ? shared_digits(key[a], key[a + n_leaf]) : -1; };
    if (t < kLevels) cnt[t] = 0;
    if (n_leaf <= kSpanHalo)
        for (int q = t; q < kSpanTile + n_leaf; q += kSpanTile) ends[q] = (int8_t)window(i0 - n_leaf + q);
    __syncthreads();
    int lo = kLevels, hi = -1;
    if (i < n) {
        int l = -1;
        if (n_leaf <= kSpanHalo)
            for (int q = 0; q <= n_leaf; q++) l = max(l, (int)ends[t + q]);
        else
            l = sphk::deepest_full_level(key, n, n_leaf, i);
        if (i > 0 && key[i] < key[i - 1]) atomicOr(unsorted, 1);
        lo = i == 0 ? 0 : shared_digits(key[i - 1], key[i]) + 1;
        hi = min(l + 1, kMaxLevel);
        span[i] = Span{(int8_t)lo, (int8_t)hi};
        head[i] = -1;
    }
    for (int L = 0; L < kLevels; L++) {
        const uint64_t b = __ballot(lo <= L && L <= hi);
        if ((t & 63) == 0 && b) atomicAdd(&cnt[L], __popcll(b));
    }
    __syncthreads();
    if (t < kLevels) hist[t * gridDim.x + blockIdx.x] = cnt[t];
}

// Exclusive scan of m counts in place by one block; total[0] the sum, and
// first[L] the value at L * stride (the starts of the levels) for L < nl.
constexpr int kScanThreads = 1024;

__global__ __launch_bounds__(kScanThreads) void block_scan_kernel(int m, int32_t *__restrict__ a, int nl, int stride,
                                                                  int64_t *__restrict__ first,
                                                                  int64_t *__restrict__ total)
{
    __shared__ int64_t wsum[kScanThreads / 64];
    const int t = threadIdx.x, lane = t & 63;
    const int per = (m + kScanThreads - 1) / kScanThreads;
    const int b = min(m, t * per), e = min(m, b + per);
    int64_t sum = 0;
    for (int k = b; k < e; k++) sum += a[k];
    int64_t incl = sum;
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t u = __shfl_up(incl, d, 64);
        if (lane >= d) incl += u;
    }
    if (lane == 63) wsum[t / 64] = incl;
    __syncthreads();
    int64_t at = incl - sum;
    for (int w = 0; w < t / 64; w++) at += wsum[w];
    for (int k = b; k < e; k++) {
        const int c = a[k];
        if (nl && k % stride == 0) first[k / stride] = at;
        a[k] = (int32_t)at;
        at += c;
    }
    if (t == kScanThreads - 1) *total = at;   // the last threads may own nothing: at is the sum
}

// First index past i whose key differs from key[i] in the first L digits
// (keys sorted): doubling steps, then bisection.
__device__ __forceinline__ int32_t cell_end(const uint64_t *__restrict__ key, int n, int i, int L)
{
    if (L == 0) return n;
    const int shift = 3 * (kMaxLevel - L);
    const uint64_t p = key[i] >> shift;
    int64_t step = 1;
    while (i + step < n && (key[i + step] >> shift) == p) step *= 2;
    int32_t b = (int32_t)(i + step / 2), e = (int32_t)(i + step < n ? i + step : n);   // key[b] inside, e outside
    while (e - b > 1) {
        const int32_t mid = b + (e - b) / 2;
        if ((key[mid] >> shift) == p)
            b = mid;
        else
            e = mid;
    }
    return e;
}

// The nodes that begin at each particle, at the places the scanned counts
// give.  A node's parent is the last node of the level above that begins at
// or before it; a parent counts its children (nchild zero before).
__global__ __launch_bounds__(kSpanTile) void node_kernel(int n, const uint64_t *__restrict__ key,
                                                         const Span *__restrict__ span,
                                                         const int32_t *__restrict__ hist, NodeArrays nd,
                                                         const double *__restrict__ frame)
{
    __shared__ int base[kSpanTile / 64][kLevels];
    const int t = threadIdx.x, lane = t & 63, wave = t / 64, i = blockIdx.x * kSpanTile + t;
    const Span sp = i < n ? span[i] : Span{(int8_t)kLevels, (int8_t)-1};
    for (int L = 0; L < kLevels; L++) {
        const uint64_t b = __ballot(sp.lo <= L && L <= sp.hi);
        if (lane == 0) base[wave][L] = __popcll(b);
    }
    __syncthreads();
    if (t < kLevels) {
        int at = hist[t * gridDim.x + blockIdx.x];
        for (int w = 0; w < kSpanTile / 64; w++) {
            const int c = base[w][t];
            base[w][t] = at;
            at += c;
        }
    }
    __syncthreads();
    int above = -1;   // the node of level L - 1 that holds i
    double len = frame[3];
    for (int L = 0; L < kLevels; L++, len *= 0.5) {
        const bool in = sp.lo <= L && L <= sp.hi;
        const uint64_t b = __ballot(in);
        const int a = base[wave][L] + __popcll(b & ((1ull << lane) - 1));
        if (in) {
            nd.begin[a] = i;
            nd.end[a] = cell_end(key, n, i, L);
            nd.level[a] = L;
            nd.parent[a] = above;
            nd.len[a] = len;
            if (L == sp.hi) nd.child[a] = -1;            // a leaf: its first particle heads no deeper node
            if (L > sp.lo) nd.child[above] = a;          // begins where its parent does
            if (L > 0) atomicAdd(&nd.nchild[above], 1);
        }
        above = in ? a : a - 1;
    }
}

// Node records for the list walks: the fields one visit reads, packed in
// one 64-byte record per node (one memory segment per visit instead of one
// per field array).  Values are copies of the node arrays, so the walks'
// comparisons and their results are unchanged.
struct alignas(64) BoxRec {     // gather and symmetry walks
    double lo[3], hi[3];        // tight box
    int32_t child, nchild, begin, end;
};
struct alignas(64) MacRec {     // long walk
    double mx, my, mz, mm, len;
    int32_t child, nchild, begin, end;
};
struct alignas(64) OboxRec {    // symmetry walk: box of the nodes' particle spheres, largest |h|
    double lo[3], hi[3], h;
};

// ---- boxes and monopoles, one level at a time (bottom-up) ------------------
struct Moments {
    double *lo, *hi;        // [3][cap] tight box
    double *mm, *mx, *my, *mz, *me;
    double *sx, *sy, *sz, *se;   // mass-weighted sums
    size_t cap;
};

__device__ __forceinline__ void node_moments(int a, const NodeArrays &nd, const Moments &mo, BoxRec *__restrict__ br,
                                             MacRec *__restrict__ mr, const double *__restrict__ x,
                                             const double *__restrict__ y, const double *__restrict__ z,
                                             const double *__restrict__ m, const double *__restrict__ eps2)
{
#pragma clang fp contract(off)
    const size_t C = mo.cap;
    const double inf = __builtin_inf();
    double lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf};
    double M = 0., X = 0., Y = 0., Z = 0., E = 0.;
    if (nd.child[a] < 0) {
        for (int i = nd.begin[a]; i < nd.end[a]; i++) {
            const double p[3] = {x[i], y[i], z[i]};
            for (int d = 0; d < 3; d++) {
                lo[d] = fmin(lo[d], p[d]);
                hi[d] = fmax(hi[d], p[d]);
            }
            const double e2 = eps2 ? eps2[i] : 0.;
            M += m[i];
            X += m[i] * x[i];
            Y += m[i] * y[i];
            Z += m[i] * z[i];
            E += m[i] * e2;
        }
    } else {
        for (int c = nd.child[a]; c < nd.child[a] + nd.nchild[a]; c++) {
            for (int d = 0; d < 3; d++) {
                lo[d] = fmin(lo[d], mo.lo[d * C + c]);
                hi[d] = fmax(hi[d], mo.hi[d * C + c]);
            }
            M += mo.mm[c];
            X += mo.sx[c];
            Y += mo.sy[c];
            Z += mo.sz[c];
            E += mo.se[c];
        }
    }
    for (int d = 0; d < 3; d++) {
        mo.lo[d * C + a] = lo[d];
        mo.hi[d * C + a] = hi[d];
    }
    mo.mm[a] = M;
    mo.sx[a] = X;
    mo.sy[a] = Y;
    mo.sz[a] = Z;
    mo.se[a] = E;
    double c[3], e = 0.;
    if (M > 0.) {
        c[0] = X / M;
        c[1] = Y / M;
        c[2] = Z / M;
        e = E / M;
    } else {
        for (int d = 0; d < 3; d++) c[d] = 0.5 * (lo[d] + hi[d]);
    }
    mo.mx[a] = c[0];
    mo.my[a] = c[1];
    mo.mz[a] = c[2];
    mo.me[a] = e;
    // the records the list walks read
    const int child = nd.child[a], nch = nd.nchild[a], begin = nd.begin[a], end = nd.end[a];
    br[a] = BoxRec{{lo[0], lo[1], lo[2]}, {hi[0], hi[1], hi[2]}, child, nch, begin, end};
    mr[a] = MacRec{c[0], c[1], c[2], M, nd.len[a], child, nch, begin, end};
}

__global__ __launch_bounds__(kBlock) void moments_kernel(int a0, int na, NodeArrays nd, Moments mo,
                                                         BoxRec *__restrict__ br, MacRec *__restrict__ mr,
                                                         const double *__restrict__ x, const double *__restrict__ y,
                                                         const double *__restrict__ z, const double *__restrict__ m,
                                                         const double *__restrict__ eps2)
{
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k < na) node_moments(a0 + k, nd, mo, br, mr, x, y, z, m, eps2);
}

// The top levels (starts in ls, `levels` of them) in one block, deepest first:
// a launch per level costs more than their few nodes.
struct TopLevels {
    int levels;
    int ls[kMaxLevel + 2];
};
constexpr int kTopThreads = 1024;
constexpr int kTopNodes = 512;   // levels are top while no level is wider than this

__global__ __launch_bounds__(kTopThreads) void moments_top_kernel(TopLevels tl, NodeArrays nd, Moments mo,
                                                                  BoxRec *br, MacRec *mr, const double *x,
                                                                  const double *y, const double *z, const double *m,
                                                                  const double *eps2)
{
    for (int L = tl.levels - 1; L >= 0; L--) {
        for (int a = tl.ls[L] + threadIdx.x; a < tl.ls[L + 1]; a += kTopThreads)
            node_moments(a, nd, mo, br, mr, x, y, z, m, eps2);
        __syncthreads();   // children's sums written before the parents read them
    }
}

// Box of x_j +- h_j per node (symmetry lists), bottom-up.
__device__ __forceinline__ void node_obox(int a, const NodeArrays &nd, OboxRec *orr, const double *__restrict__ x,
                                          const double *__restrict__ y, const double *__restrict__ z,
                                          const double *__restrict__ h)
{
    const double inf = __builtin_inf();
    double lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf}, hm = 0.;
    if (nd.child[a] < 0) {
        for (int i = nd.begin[a]; i < nd.end[a]; i++) {
            const double p[3] = {x[i], y[i], z[i]};
            hm = fmax(hm, fabs(h[i]));
            for (int d = 0; d < 3; d++) {
                lo[d] = fmin(lo[d], p[d] - h[i]);
                hi[d] = fmax(hi[d], p[d] + h[i]);
            }
        }
    } else {
        for (int c = nd.child[a]; c < nd.child[a] + nd.nchild[a]; c++) {
            const OboxRec o = orr[c];
            hm = fmax(hm, o.h);
            for (int d = 0; d < 3; d++) {
                lo[d] = fmin(lo[d], o.lo[d]);
                hi[d] = fmax(hi[d], o.hi[d]);
            }
        }
    }
    orr[a] = OboxRec{{lo[0], lo[1], lo[2]}, {hi[0], hi[1], hi[2]}, hm};
}

__global__ __launch_bounds__(kBlock) void obox_kernel(int a0, int na, NodeArrays nd, OboxRec *orr,
                                                      const double *__restrict__ x, const double *__restrict__ y,
                                                      const double *__restrict__ z, const double *__restrict__ h)
{
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k < na) node_obox(a0 + k, nd, orr, x, y, z, h);
}

__global__ __launch_bounds__(kTopThreads) void obox_top_kernel(TopLevels tl, NodeArrays nd, OboxRec *orr,
                                                               const double *x, const double *y, const double *z,
                                                               const double *h)
{
    for (int L = tl.levels - 1; L >= 0; L--) {
        for (int a = tl.ls[L] + threadIdx.x; a < tl.ls[L + 1]; a += kTopThreads) node_obox(a, nd, orr, x, y, z, h);
        __syncthreads();
    }
}

// ---- groups ------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void fill_kernel(int n, int32_t *__restrict__ a, int32_t v)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) a[i] = v;
}

__global__ __launch_bounds__(kBlock) void group_mark_kernel(int nn, NodeArrays nd, int n_group,
                                                            int32_t *__restrict__ head)
{
    const int a = blockIdx.x * kBlock + threadIdx.x;
    if (a >= nn) return;
    const bool small = nd.end[a] - nd.begin[a] <= n_group || nd.child[a] < 0;
    const int p = nd.parent[a];
    const bool opened = p < 0 || nd.end[p] - nd.begin[p] > n_group;
    if (small && opened) head[nd.begin[a]] = a;
}

// Groups that begin in each block of particles.
__global__ __launch_bounds__(kSpanTile) void group_count_kernel(int n, const int32_t *__restrict__ head,
                                                                int32_t *__restrict__ cnt)
{
    __shared__ int c;
    const int i = blockIdx.x * kSpanTile + threadIdx.x;
    if (threadIdx.x == 0) c = 0;
    __syncthreads();
    const uint64_t b = __ballot(i < n && head[i] >= 0);
    if ((threadIdx.x & 63) == 0) atomicAdd(&c, __popcll(b));
    __syncthreads();
    if (threadIdx.x == 0) cnt[blockIdx.x] = c;
}

__global__ __launch_bounds__(kSpanTile) void group_write_kernel(int n, const int32_t *__restrict__ head,
                                                                const int32_t *__restrict__ pos,
                                                                const int64_t *__restrict__ total,
                                                                int32_t *__restrict__ group,
                                                                int32_t *__restrict__ i_off)
{
    __shared__ int wc[kSpanTile / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t / 64, i = blockIdx.x * kSpanTile + t;
    const int a = i < n ? head[i] : -1;
    const uint64_t b = __ballot(a >= 0);
    if (lane == 0) wc[wave] = __popcll(b);
    __syncthreads();
    int at = pos[blockIdx.x] + __popcll(b & ((1ull << lane) - 1));
    for (int w = 0; w < wave; w++) at += wc[w];
    if (a >= 0) {
        group[at] = a;
        i_off[at] = i;
    }
    if (i == 0) i_off[*total] = n;
}

// ---- lists -------------------------------------------------------------------
// Walk of workgroup b: chunks of 64 consecutive walks dealt to the 8 XCDs in
// turn, so that an XCD's L2 serves the nodes and particles neighbours share.
__device__ __forceinline__ int xcd_chunk(int b, int n)
{
    constexpr int kX = 8, kC = 64;
    const int n_full = n / (kX * kC) * (kX * kC);
    if (b >= n_full) return b;
    const int x = b % kX, k = b / kX;
    return ((k / kC) * kX + x) * kC + k % kC;
}

struct TreeView {
    NodeArrays nd;
    Moments mo;
    const BoxRec *br;
    const MacRec *mr;
    const OboxRec *orr;
    const double *x, *y, *z;
    const int32_t *group, *i_off;
};

__device__ __forceinline__ bool box_overlaps(const double (&alo)[3], const double (&ahi)[3],
                                             const double (&blo)[3], const double (&bhi)[3])
{
    for (int d = 0; d < 3; d++)
        if (bhi[d] < alo[d] || blo[d] > ahi[d]) return false;
    return true;
}

// Box of the i search spheres of each walk (gather: rs, symmetry: h) and the
// largest |r| (rows 0-5 and 6 of wb).
__global__ __launch_bounds__(kBlock) void walk_box_kernel(int ng, const int32_t *__restrict__ i_off,
                                                          const double *__restrict__ x,
                                                          const double *__restrict__ y,
                                                          const double *__restrict__ z,
                                                          const double *__restrict__ r, double *__restrict__ wb)
{
    const int g = blockIdx.x * kBlock + threadIdx.x;
    if (g >= ng) return;
    const double inf = __builtin_inf();
    double lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf}, rm = 0.;
    for (int i = i_off[g]; i < i_off[g + 1]; i++) {
        const double p[3] = {x[i], y[i], z[i]};
        rm = fmax(rm, fabs(r[i]));
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], p[d] - r[i]);
            hi[d] = fmax(hi[d], p[d] + r[i]);
        }
    }
    for (int d = 0; d < 3; d++) {
        wb[d * ng + g] = lo[d];
        wb[(3 + d) * ng + g] = hi[d];
    }
    wb[6 * ng + g] = rm;
}

// What the depth-first walk does at node a: skip it (pruned, or massless for
// the long list), take it as one SPJ, emit its particles (leaf), or open it.
enum Visit { kSkip, kSpj, kLeaf, kOpen };

// Child range and particle range of the visited node, from its record.
struct NodeLinks {
    int32_t child, nchild, begin, end;
};

template <int MODE>
__device__ __forceinline__ Visit visit(const TreeView &t, int a, const double (&olo)[3],
                                       const double (&ohi)[3], const double (&glo)[3], const double (&ghi)[3],
                                       double inv_t2, NodeLinks &ln)
{
#pragma clang fp contract(off)
    if (MODE != 2) {
        const BoxRec b = t.br[a];
        OboxRec o{};
        if (MODE == 1) o = t.orr[a];   // loaded with b: one memory round trip per visit
        ln = NodeLinks{b.child, b.nchild, b.begin, b.end};
        const bool leaf = b.child < 0;
        if (MODE == 0) {
            if (!box_overlaps(olo, ohi, b.lo, b.hi)) return kSkip;
            return leaf ? kLeaf : kOpen;
        }
        if (!box_overlaps(olo, ohi, b.lo, b.hi)) {
            if (!box_overlaps(glo, ghi, o.lo, o.hi)) return kSkip;
        }
        return leaf ? kLeaf : kOpen;
    }
    const MacRec m = t.mr[a];
    ln = NodeLinks{m.child, m.nchild, m.begin, m.end};
    if (m.mm == 0.) return kSkip;
    const double c[3] = {m.mx, m.my, m.mz};
    double s = 0.;
    for (int d = 0; d < 3; d++) {
        double e = 0.;
        if (c[d] < glo[d])
            e = glo[d] - c[d];
        else if (c[d] > ghi[d])
            e = c[d] - ghi[d];
        s += e * e;
    }
    const double L = m.len;
    if (s > L * L * inv_t2) return kSpj;
    return m.child < 0 ? kLeaf : kOpen;
}

// ---- interaction lists: 8 lanes per walk -----------------------------------
// The host builder's depth-first walk of each group, 8 walks per wave and 8
// lanes per walk (an octree node has at most 8 children).  A walk keeps a
// stack of evaluated entries in LDS, the next one in preorder on top.  Each
// step evaluates the children of one opened node, a lane each: the finished
// children (SPJ, leaf) before the first child to open are emitted at once,
// the rest are pushed, first child on top.  Then the finished entries on top
// of the stack are popped and emitted, up to 8 at a time, down to the next
// node to open, whose children the next step evaluates.  Emitted in this
// order, the entries are the host's list element for element.  Each tree
// level leaves at most 7 siblings pending, so the stack never holds more
// than 7 (kMaxLevel + 1) + 8 entries (kListStack); walks run first with a
// stack of kListStackSmall entries (less LDS, more waves in flight) and,
// if one would overflow it, again with kListStack.
//
// Entry: word 0 the node (SPJ, and leaves in candidate-leaf mode), the first
// child (to open) or the first particle (leaf, particles listed); word 1 the
// type in bits 29-31 and the child or particle count below.
constexpr int kListWalks = 8;
constexpr int kListStack = 7 * (kMaxLevel + 1) + 8 + 2;   // 164 (even: 8-byte rows)
constexpr int kListStackSmall = 64;
constexpr uint32_t kTySpj = 1u << 29, kTyLeaf = 2u << 29, kTyOpen = 3u << 29, kTyMask = 7u << 29;
constexpr uint32_t kCountMask = (1u << 29) - 1;

// bits of the 8 lanes of this lane's walk
__device__ __forceinline__ unsigned walk_bits(bool p, int lane)
{
    return (unsigned)((__ballot(p) >> (lane & ~7)) & 0xffu);
}

__device__ __forceinline__ int walk_scan_incl(int v, int c)
{
    for (int d = 1; d < 8; d <<= 1) {
        const int u = __shfl_up(v, d, 8);
        if (c >= d) v += u;
    }
    return v;
}

// Exact membership of particle j of a reached leaf in a short-range list,
// as the host's leaf loop decides it: MODE 0 |x_j - x_i| < rs_i for some i of
// the walk; MODE 1 r_ij < max(H_i, H_j) for some i, after the box pre-tests
// (j inside the walk's search box, or j's sphere reaching the group's box).
// j's position is p (and its H hj in MODE 1).  The walk's i-particles
// (x, y, z, r) are read from si, the first nl of them staged in LDS.
constexpr int kWalkI = 256;

template <int MODE>
__device__ __forceinline__ bool member(const TreeView &t, const double *__restrict__ r, const double (&p)[3],
                                       double hj, int ib, int ni, int nl, const double4 *si,
                                       const double (&olo)[3], const double (&ohi)[3], const double (&glo)[3],
                                       const double (&ghi)[3])
{
#pragma clang fp contract(off)
    bool in = true, jov = MODE == 1;
    for (int d = 0; d < 3; d++) {
        in = in && !(p[d] < olo[d] || p[d] > ohi[d]);
        if (MODE == 1) jov = jov && !(ghi[d] < p[d] - hj || glo[d] > p[d] + hj);
    }
    if (!in && !jov) return false;
    auto hit = [&](double4 P) {
        const double dx = p[0] - P.x, dy = p[1] - P.y, dz = p[2] - P.z;
        const double rr = MODE == 1 ? (P.w > hj ? P.w : hj) : P.w;
        return dx * dx + dy * dy + dz * dz < rr * rr;
    };
    int q = 0;
    for (; q + 2 <= nl; q += 2) {   // LDS, two at a time
        const double4 P0 = si[q], P1 = si[q + 1];
        if (hit(P0) || hit(P1)) return true;
    }
    if (q < nl && hit(si[q])) return true;
    for (q = nl; q < ni; q++) {   // beyond the staged particles: from memory
        const int i = ib + q;
        if (hit(make_double4(t.x[i], t.y[i], t.z[i], r[i]))) return true;
    }
    return false;
}

// The particles of the leaves reached into jout (MODE 0 gather, 1 symmetry:
// the candidates of the short-range lists), and for MODE 2 (long) the SPJ
// nodes into sout.  FILL 0: the walk's counts go to cj/cs.  FILL 1: written
// from the walk's offsets oj/os.  Runs only when a room of room_list_kernel
// overflowed or does not fit in memory.
// Bit 1 of err is set if a stack of STACK entries would overflow.
template <int MODE, int FILL, int STACK>
__global__ __launch_bounds__(64) void walk_list_kernel(int ng, TreeView t, const double *__restrict__ wb,
                                                       const double *__restrict__ r, double inv_t2,
                                                       int64_t *__restrict__ cj, int64_t *__restrict__ cs,
                                                       const int64_t *__restrict__ oj, const int64_t *__restrict__ os,
                                                       int32_t *__restrict__ jout, int32_t *__restrict__ sout,
                                                       int *__restrict__ err)
{
#pragma clang fp contract(off)
    __shared__ uint2 stk[kListWalks][STACK];
    const int lane = threadIdx.x, sub = lane >> 3, c = lane & 7;
    const int g = blockIdx.x * kListWalks + sub;
    const bool live = g < ng;
    const unsigned below = (1u << c) - 1u, above = 0xffu & ~((2u << c) - 1u);
    const size_t C = t.mo.cap;
    double olo[3] = {0., 0., 0.}, ohi[3] = {0., 0., 0.}, glo[3] = {0., 0., 0.}, ghi[3] = {0., 0., 0.};
    int64_t nj = 0, ns = 0, j0 = 0, s0 = 0;
    if (live) {
        const int gn = t.group[g];
        for (int d = 0; d < 3; d++) {
            if (MODE != 2) {
                olo[d] = wb[d * ng + g];
                ohi[d] = wb[(3 + d) * ng + g];
            }
            glo[d] = t.mo.lo[d * C + gn];
            ghi[d] = t.mo.hi[d * C + gn];
        }
        if (FILL == 1) {
            j0 = oj[g];
            if (MODE == 2) s0 = os[g];
        }
    }
    // emit the entries (w0, w1) of the lanes with em set, in lane order
    auto emit = [&](bool em, uint32_t w0, uint32_t w1) {
        const uint32_t ty = w1 & kTyMask;
        if (MODE == 2) {
            const bool is_s = em && ty == kTySpj;
            const unsigned sb = walk_bits(is_s, lane);
            if (FILL == 1 && is_s) sout[s0 + ns + __popc(sb & below)] = (int32_t)w0;
            ns += __popc(sb);
        }
        const bool is_l = em && ty == kTyLeaf;
        const int sz = is_l ? (int)(w1 & kCountMask) : 0;
        const int incl = walk_scan_incl(sz, c);
        if (FILL == 1 && is_l) {
            const int64_t p0 = j0 + nj + incl - sz;
            for (int q = 0; q < sz; q++) jout[p0 + q] = (int32_t)w0 + q;
        }
        nj += __shfl(incl, 7, 8);
    };

    int sp = 0;                        // the walk's stack depth
    int first = 0, nch = live ? 1 : 0; // nodes evaluated by the next step: the root first
    bool bad = false;
    while (__ballot(nch > 0)) {
        // evaluate nodes first + c
        const bool ev = c < nch;
        uint32_t w0 = 0, w1 = 0;
        if (ev) {
            const int a = first + c;
            NodeLinks ln;
            const Visit v = visit<MODE>(t, a, olo, ohi, glo, ghi, inv_t2, ln);
            if (v == kSpj) {
                w0 = (uint32_t)a;
                w1 = kTySpj;
            } else if (v == kLeaf) {
                w0 = (uint32_t)ln.begin;
                w1 = kTyLeaf | (uint32_t)(ln.end - ln.begin);
            } else if (v == kOpen) {
                w0 = (uint32_t)ln.child;
                w1 = kTyOpen | (uint32_t)ln.nchild;
            }
        }
        const bool kept = ev && w1 != 0;
        const unsigned ob = walk_bits(kept && (w1 & kTyMask) == kTyOpen, lane);
        const int fo = ob ? __builtin_ctz(ob) : 8;
        emit(kept && c < fo, w0, w1);
        const bool push = kept && c >= fo;
        const unsigned pb = walk_bits(push, lane);
        if (sp + __popc(pb) > STACK) bad = true;
        if (push && !bad) stk[sub][sp + __popc(pb & above)] = make_uint2(w0, w1);
        if (!bad) sp += __popc(pb);
        // pop finished entries down to the next node to open
        nch = 0;
        while (sp > 0 && !bad) {
            const int avail = sp < 8 ? sp : 8;
            const uint2 e = c < avail ? stk[sub][sp - 1 - c] : make_uint2(0u, 0u);
            const unsigned ob2 = walk_bits(c < avail && (e.y & kTyMask) == kTyOpen, lane);
            const int k = ob2 ? __builtin_ctz(ob2) : avail;
            emit(c < k, e.x, e.y);
            if (ob2) {
                first = (int)__shfl((int)e.x, k, 8);
                nch = (int)(__shfl((int)e.y, k, 8) & kCountMask);
                sp -= k + 1;
                break;
            }
            sp -= k;
        }
    }
    if (bad && c == 0) atomicOr(err, 1);
    if (FILL == 0 && live && c == 0) {
        cj[g] = nj;
        if (MODE == 2) cs[g] = ns;
    }
}

// Exact membership of each walk's candidates (the particles of the leaves its
// walk reached, in the host's order), one wave per walk: the first n_si
// (<= kWalkI) i-particles of the walk sit in LDS (dynamic, n_si double4), any
// beyond are read from memory; lane l tests candidate c0 + l, and the members
// are compacted in place (in order) at the front of the walk's stretch of
// scr; their number goes to cnt.  Candidates are taken kMemberU * 64 at a
// time: their indices and positions are all loaded before any is tested.
constexpr int kMemberU = 4;

template <int MODE>
__global__ __launch_bounds__(64) void member_kernel(int ng, TreeView t, const double *__restrict__ wb,
                                                    const double *__restrict__ r, const int64_t *__restrict__ coff,
                                                    const int64_t *__restrict__ ccnt, int32_t *__restrict__ scr,
                                                    int64_t *__restrict__ cnt, int n_si)
{
    extern __shared__ double4 si[];
    const int g = blockIdx.x;
    if (g >= ng) return;
    const int lane = threadIdx.x;
    const size_t C = t.mo.cap;
    const int ib = t.i_off[g], ni = t.i_off[g + 1] - ib;
    const int nl = ni < n_si ? ni : n_si;
    for (int q = lane; q < nl; q += 64)
        si[q] = make_double4(t.x[ib + q], t.y[ib + q], t.z[ib + q], r[ib + q]);
    const int gn = t.group[g];
    double olo[3], ohi[3], glo[3], ghi[3];
    for (int d = 0; d < 3; d++) {
        olo[d] = wb[d * ng + g];
        ohi[d] = wb[(3 + d) * ng + g];
        glo[d] = t.mo.lo[d * C + gn];
        ghi[d] = t.mo.hi[d * C + gn];
    }
    __syncthreads();
    int32_t *s = scr + coff[g];
    const int64_t nc = ccnt[g];
    int64_t count = 0;
    for (int64_t c0 = 0; c0 < nc; c0 += 64 * kMemberU) {
        int j[kMemberU];
        double p[kMemberU][3], hj[kMemberU];
#pragma unroll
        for (int u = 0; u < kMemberU; u++) {
            const int64_t e = c0 + 64 * u + lane;
            j[u] = e < nc ? s[e] : -1;
        }
#pragma unroll
        for (int u = 0; u < kMemberU; u++) {
            const int k = j[u] < 0 ? 0 : j[u];
            p[u][0] = t.x[k];
            p[u][1] = t.y[k];
            p[u][2] = t.z[k];
            hj[u] = MODE == 1 ? r[k] : 0.;
        }
        // every slot of this stretch is read: writes land at or before them
#pragma unroll
        for (int u = 0; u < kMemberU; u++) {
            const bool acc = j[u] >= 0 && member<MODE>(t, r, p[u], hj[u], ib, ni, nl, si, olo, ohi, glo, ghi);
            const uint64_t bal = __ballot(acc);
            if (acc) s[count + __popcll(bal & ((1ull << lane) - 1ull))] = j[u];
            count += __popcll(bal);
        }
    }
    if (lane == 0) cnt[g] = count;
}

// ---- lists in one pass into rooms: one wave per walk --------------------------
// MODE 0 gather, 1 symmetry: the walk of the tree and the member test
// together; MODE 2 the long list.  The wave keeps the walk's pending entries
// in LDS in preorder, the next one on top.  A step looks at the top 64
// entries: finished ones on top (leaves, SPJ nodes) are taken off; otherwise
// up to 8 of the nodes to open among them are opened at once, 8 lanes each,
// and the entries from the top to the last opened one are written back with
// every opened node replaced by its kept children.  The order stays preorder,
// so entries come off in the host's order.  Long list: SPJ nodes and the
// leaves' particles go to the walk's two rooms.  Short-range lists: the
// leaves' particles are candidates; 256 or more of them are tested together
// (positions of four per lane loaded before any test) and the members written
// to the walk's room.
//
// One wave per walk because the walks differ: with 8 lanes per walk and 8
// walks per wave the short-range lists waited for a few walks in the
// outskirts that open nodes one after the other (VALU issue 16 %, 1.8 waves
// per SIMD), and the long list, issue-bound, paid two emissions per 8 nodes
// looked at.  10^6 particles, before and now: gather and symmetry with their
// member kernels 2.0 and 1.85 ms, 0.75 and 0.76; long 1.42, 0.90.
//
// A node of a short-range list is skipped if no particle of it can be a
// member: its tight box must meet the box of the walk's spheres (or its own
// spheres' box the walk's), as in the host's walk, and must lie within the
// largest radius that matters of the walk's box: the walk's largest r or, for
// symmetry, the node's.  The distance test (half the candidates: a sphere's
// share of its cube) leaves out only particles that the member test refuses,
// with 1e-9 to spare for rounding, so the lists do not change.
//
// A walk that opens several nodes at once may have many entries pending (a
// walk at the edge of a steep profile whose search box holds the centre).
// One that would have more than kRoomStack gives up (count -1, bit 8 of err)
// and is done again, alone, by the DEEP kernel with its larger stack.  That
// holds every walk: where a step would leave more than kDeepLoose entries it
// goes depth first until they are fewer again (every finished entry on top is
// taken, then one node opened, which leaves at most 7 entries per level beside
// those before).  Such walks sent every build through the count and fill walks
// as well: the long list of 3x10^4 particles spread evenly over four decades of
// radius took 1581 us, now 311 (8 lanes per walk, before: 931).  The larger stack
// for all walks costs waves: 576 entries took the lists of 10^6 particles from
// 3.21 to 3.47 ms.
constexpr int kRoomStack = 384;    // entries
constexpr int kDeepStack = 2048;
constexpr int kDeepLoose = kDeepStack - (7 * kMaxLevel + 1);
constexpr int kFlagStack = 1, kFlagRoom = 2, kFlagNodes = 4, kFlagDeep = 8;   // bits of err
constexpr int kRoomCand = 512;
constexpr int kRoomBatch = 256;    // candidates tested together
constexpr int kRoomTake = 32;      // finished entries on top that are worth taking before the next nodes are opened

template <int MODE, bool DEEP>
__global__ __launch_bounds__(64) void room_list_kernel(int ng, TreeView t, const double *__restrict__ wb,
                                                       const double *__restrict__ r, double inv_t2,
                                                       int64_t *__restrict__ cnt, int32_t *__restrict__ out,
                                                       int64_t room, int64_t *__restrict__ cnt_s,
                                                       int32_t *__restrict__ out_s, int64_t room_s, int n_si,
                                                       int *__restrict__ err)
{
#pragma clang fp contract(off)
    __shared__ uint2 stk[DEEP ? kDeepStack : kRoomStack];
    __shared__ int32_t cand[MODE == 2 ? 1 : kRoomCand];
    __shared__ uint32_t s_first[8], s_count[8], s_place[8];
    extern __shared__ double4 si[];
    if ((int)blockIdx.x >= ng) return;
    const int g = xcd_chunk(blockIdx.x, ng), lane = threadIdx.x;
    if (DEEP && cnt[g] >= 0) return;
    const uint64_t below = (1ull << lane) - 1ull;
    const size_t C = t.mo.cap;
    const int ib = t.i_off[g], ni = t.i_off[g + 1] - ib;
    const int nl = ni < n_si ? ni : n_si;
    if (MODE != 2) for (int q = lane; q < nl; q += 64)
        si[q] = make_double4(t.x[ib + q], t.y[ib + q], t.z[ib + q], r[ib + q]);
    const int gn = t.group[g];
    double olo[3], ohi[3], glo[3], ghi[3];
    for (int d = 0; d < 3; d++) {
        olo[d] = MODE == 2 ? 0. : wb[d * ng + g];
        ohi[d] = MODE == 2 ? 0. : wb[(3 + d) * ng + g];
        glo[d] = t.mo.lo[d * C + gn];
        ghi[d] = t.mo.hi[d * C + gn];
    }
    const double rm = MODE == 2 ? 0. : wb[6 * ng + g];
    int32_t *const room_out = out + (int64_t)g * room;
    int32_t *const room_spj = MODE == 2 ? out_s + (int64_t)g * room_s : nullptr;
    int64_t count = 0, spj = 0;
    int nc = 0;          // candidates waiting

    // node a: its entry (0 type if skipped)
    auto look = [&](int a) {
        if (MODE == 2) {
            NodeLinks ln;
            const Visit v = visit<2>(t, a, olo, ohi, glo, ghi, inv_t2, ln);
            return v == kSpj    ? make_uint2((uint32_t)a, kTySpj)
                   : v == kLeaf ? make_uint2((uint32_t)ln.begin, kTyLeaf | (uint32_t)(ln.end - ln.begin))
                   : v == kOpen ? make_uint2((uint32_t)ln.child, kTyOpen | (uint32_t)ln.nchild)
                                : make_uint2(0u, 0u);
        }
        const BoxRec b = t.br[a];
        OboxRec o{};
        if (MODE == 1) o = t.orr[a];
        uint2 e = make_uint2(0u, 0u);
        const bool near = box_overlaps(olo, ohi, b.lo, b.hi) || (MODE == 1 && box_overlaps(glo, ghi, o.lo, o.hi));
        double s = 0.;
        for (int d = 0; d < 3; d++) {
            const double e1 = glo[d] - b.hi[d], e2 = b.lo[d] - ghi[d];
            const double m = e1 > e2 ? e1 : e2;
            s += m > 0. ? m * m : 0.;
        }
        const double R = (MODE == 1 && o.h > rm ? o.h : rm) * (1. + 1e-9);
        if (near && !(s > R * R)) {
            e = b.child < 0 ? make_uint2((uint32_t)b.begin, kTyLeaf | (uint32_t)(b.end - b.begin))
                            : make_uint2((uint32_t)b.child, kTyOpen | (uint32_t)b.nchild);
        }
        return e;
    };
    // the members among candidates, n (<= 64 * U) of them, get(k) the k-th
    auto test = [&](auto &&get, int n) {
        int j[kMemberU];
        double p[kMemberU][3], hj[kMemberU];
#pragma unroll
        for (int u = 0; u < kMemberU; u++) {
            const int k = 64 * u + lane;
            j[u] = k < n ? get(k) : -1;
            const int jj = j[u] < 0 ? ib : j[u];
            p[u][0] = t.x[jj];
            p[u][1] = t.y[jj];
            p[u][2] = t.z[jj];
            hj[u] = MODE == 1 ? r[jj] : 0.;
        }
#pragma unroll
        for (int u = 0; u < kMemberU; u++) {
            if (64 * u >= n) break;
            const bool acc = j[u] >= 0 && member<MODE>(t, r, p[u], hj[u], ib, ni, nl, si, olo, ohi, glo, ghi);
            const uint64_t bal = __ballot(acc);
            const int64_t at = count + __popcll(bal & below);
            if (acc && at < room) room_out[at] = j[u];
            count += __popcll(bal);
        }
    };
    // candidates waiting: whole batches, or (all) every one
    auto drain = [&](bool all) {
        __syncthreads();
        int at = 0;
        while (nc - at >= (all ? 1 : kRoomBatch)) {
            const int n = min(kRoomBatch, nc - at);
            test([&](int k) { return cand[at + k]; }, n);
            at += n;
        }
        int32_t keep[(kRoomBatch + 63) / 64];
        const int left = nc - at;
#pragma unroll
        for (int u = 0; u < (kRoomBatch + 63) / 64; u++)
            keep[u] = at && 64 * u + lane < left ? cand[at + 64 * u + lane] : 0;
        __syncthreads();
        if (at)
#pragma unroll
            for (int u = 0; u < (kRoomBatch + 63) / 64; u++)
                if (64 * u + lane < left) cand[64 * u + lane] = keep[u];
        nc = left;
    };

    int sp = 0;
    {
        const uint2 e = look(0);
        if (lane == 0) stk[0] = e;
        sp = __builtin_amdgcn_readfirstlane(e.y) != 0u ? 1 : 0;
    }
    bool bad = false, tight = false;   // tight: depth first
    while (sp > 0) {
        __syncthreads();   // the entries of the last step are written
        const int W = sp < 64 ? sp : 64;
        const uint2 e = lane < W ? stk[sp - 1 - lane] : make_uint2(0u, 0u);
        const uint64_t ob = __ballot((e.y & kTyMask) == kTyOpen);
        const int P = ob ? __builtin_ctzll(ob) : W;    // finished entries on top
        if (!ob || P >= (tight ? 1 : kRoomTake)) {
            const int sz = lane < P && (e.y & kTyMask) == kTyLeaf ? (int)(e.y & kCountMask) : 0;
            if (MODE == 2) {
                const uint64_t sb = __ballot(lane < P && (e.y & kTyMask) == kTySpj);
                const int64_t at = spj + __popcll(sb & below);
                if (((sb >> lane) & 1) && at < room_s) room_spj[at] = (int32_t)e.x;
                spj += __popcll(sb);
                if (P < 64 ? sb == (1ull << P) - 1ull : sb == ~0ull) {   // no leaf among them
                    sp -= P;
                    continue;
                }
            }
            const int incl = sphk::wave_scan_incl(sz);
            if (MODE == 2) {
                for (int q = 0; q < sz; q++) {
                    const int64_t at = count + incl - sz + q;
                    if (at < room) room_out[at] = (int32_t)e.x + q;
                }
                count += __builtin_amdgcn_readlane(incl, 63);
                sp -= P;
                continue;
            }
            // the leading leaves that fit (nc < kRoomBatch here)
            const int take = __popcll(__ballot(lane < P && incl <= kRoomCand - nc));
            if (take > 0) {
                if (lane < take)
                    for (int q = 0; q < sz; q++) cand[nc + incl - sz + q] = (int32_t)e.x + q;
                nc += __builtin_amdgcn_readlane(incl, take - 1);
                sp -= take;
                if (nc >= kRoomBatch) drain(false);
            } else {   // one leaf of more particles than fit: from its range
                drain(true);
                const int b = __builtin_amdgcn_readlane((int)e.x, 0), n = __builtin_amdgcn_readlane(sz, 0);
                for (int c = 0; c < n; c += kRoomBatch) test([&](int k) { return b + c + k; }, min(kRoomBatch, n - c));
                sp -= 1;
            }
            continue;
        }
        // open the first (at most 8) nodes of the window
        const int rank = __popcll(ob & below);
        const bool sel = ((ob >> lane) & 1) && rank < (tight ? 1 : 8);
        const uint64_t sb = __ballot(sel);
        const int n_open = __popcll(sb), last = 63 - __builtin_clzll(sb);
        if (sel) {
            s_first[rank] = e.x;
            s_count[rank] = e.y & kCountMask;
            s_place[rank] = (uint32_t)lane;
        }
        __syncthreads();
        const int k = lane >> 3, c = lane & 7;
        uint2 w = make_uint2(0u, 0u);
        int place = 0;
        if (k < n_open) {
            place = (int)s_place[k];
            if (c < (int)s_count[k]) w = look((int)s_first[k] + c);
        }
        const uint64_t km = __ballot(w.y != 0u);
        const int T = last + 1 - n_open + __popcll(km), base = sp - 1 - last;
        if (DEEP && !tight && base + T > kDeepLoose) {
            tight = true;
            continue;
        }
        if (base + T > (DEEP ? kDeepStack : kRoomStack)) {
            bad = true;
            break;
        }
        // entry o of the rewritten window goes to stk[base + T - 1 - o]
        if (lane <= last && !sel) {
            const int before = __popcll(sb & below);   // <= 7: the last one opened lies behind
            stk[base + T - 1 - (lane - before + __popcll(km & ((1ull << (8 * before)) - 1ull)))] = e;
        }
        if (w.y != 0u) stk[base + T - 1 - (place - k + __popcll(km & below))] = w;
        sp = base + T;
        if (DEEP) tight = tight && sp > kDeepLoose - 64;
    }
    if (bad) {   // DEEP: not in a sound tree
        if (lane == 0) {
            cnt[g] = -1;
            if (MODE == 2) cnt_s[g] = 0;
            atomicOr(err, DEEP ? kFlagStack : kFlagDeep);
        }
        return;
    }
    if (MODE != 2) drain(true);
    if (lane == 0) {
        cnt[g] = count < room ? count : room;   // what the room holds (all of it unless err says so)
        if (MODE == 2) cnt_s[g] = spj < room_s ? spj : room_s;
        if (count > room) atomicOr(err, kFlagRoom);
        if (MODE == 2 && spj > room_s) atomicOr(err, kFlagNodes);
    }
}

// Members of each walk, from its stretch of the candidate scratch to its
// place in the list.
__global__ __launch_bounds__(64) void member_copy_kernel(int ng, const int64_t *__restrict__ soff,
                                                         const int32_t *__restrict__ j_off,
                                                         const int32_t *__restrict__ scr, int32_t *__restrict__ jout)
{
    const int g = blockIdx.x;
    if (g >= ng) return;
    const int64_t s0 = soff[g];
    const uint32_t b = j_off[g], n = j_off[g + 1] - b;
    for (uint32_t k = threadIdx.x; k < n; k += 64) jout[b + k] = scr[s0 + k];   // unsigned: n may be up to 2^31 - 1
}

// The lists' entries from their rooms (walk g's from g * room) to the walk
// offsets, a wave per walk.  A walk has a few hundred entries, so the copy is
// bound by the latency of a wave's rounds: eight loads are in flight per round
// (the lists of 10^6 particles 480 -> 410 us of copies against one).
constexpr int kCopyWalks = 4;
__global__ __launch_bounds__(64 * kCopyWalks) void room_copy_kernel(int ng, int64_t room,
                                                                    const int32_t *__restrict__ off,
                                                                    const int32_t *__restrict__ scr,
                                                                    int32_t *__restrict__ out)
{
    const int g = blockIdx.x * kCopyWalks + threadIdx.x / 64;
    if (g >= ng) return;
    const int32_t *src = scr + (int64_t)g * room;
    const int b = off[g], n = off[g + 1] - b;
    for (int k0 = threadIdx.x % 64; k0 < n; k0 += 8 * 64) {
        int32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (k0 + u * 64 < n) v[u] = src[k0 + u * 64];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (k0 + u * 64 < n) out[b + k0 + u * 64] = v[u];
    }
}

// Walk offsets from the scanned per-walk counts, and the total; with err the
// list walks' overflow flags, which start from 0 again.
__global__ void offsets_kernel(int ng, const int64_t *__restrict__ scan, const int64_t *__restrict__ cnt,
                               int32_t *__restrict__ off, int64_t *__restrict__ total, int *__restrict__ err,
                               int64_t *__restrict__ flags)
{
    const int g = blockIdx.x * kBlock + threadIdx.x;
    if (g < ng) off[g] = (int32_t)scan[g];
    if (g == ng - 1) {
        const int64_t t = scan[g] + cnt[g];
        *total = t;
        off[ng] = (int32_t)t;
        if (err) {
            *flags = *err;
            *err = 0;
        }
    }
}

// The same with the scan, for few walks: block 0 the counts a, block 1 b, one
// workgroup each (a thread's stretch of counts is summed, the sums scanned).
// All three lists of 10^4 particles (1007 walks) 650 -> 615 us against a
// library scan and offsets_kernel each, equal at 9198 walks, slower beyond.
constexpr int kScanWalks = 1 << 13;
__global__ __launch_bounds__(kScanThreads) void list_scan_kernel(int ng, const int64_t *__restrict__ a,
                                                                 int64_t *__restrict__ c, int32_t *__restrict__ off_a,
                                                                 const int64_t *__restrict__ b, int64_t *__restrict__ d,
                                                                 int32_t *__restrict__ off_b,
                                                                 int64_t *__restrict__ total, int *__restrict__ err)
{
    __shared__ int64_t wsum[kScanThreads / 64];
    const int64_t *const cnt = blockIdx.x ? b : a;
    int64_t *const scan = blockIdx.x ? d : c;
    int32_t *const off = blockIdx.x ? off_b : off_a;
    const int t = threadIdx.x, lane = t & 63;
    const int per = (ng + kScanThreads - 1) / kScanThreads;
    const int k0 = min(ng, t * per), k1 = min(ng, k0 + per);
    int64_t sum = 0;
    for (int k = k0; k < k1; k++) sum += cnt[k];
    int64_t incl = sum;
    for (int s = 1; s < 64; s <<= 1) {
        const int64_t u = __shfl_up(incl, s, 64);
        if (lane >= s) incl += u;
    }
    if (lane == 63) wsum[t / 64] = incl;
    __syncthreads();
    int64_t at = incl - sum;
    for (int w = 0; w < t / 64; w++) at += wsum[w];
    for (int k = k0; k < k1; k++) {
        scan[k] = at;
        off[k] = (int32_t)at;
        at += cnt[k];
    }
    if (t == kScanThreads - 1) {   // the last threads may own nothing: at is the sum
        total[blockIdx.x] = at;
        off[ng] = (int32_t)at;
        if (blockIdx.x == 0) {
            total[2] = *err;
            *err = 0;
        }
    }
}

}  // namespace

constexpr int64_t kRoomNearStart = 1024;      // short-range list entries per walk
constexpr int64_t kRoomStart = 2048;          // SPJ nodes per walk
constexpr int64_t kRoomLongStart = 8192;      // long-list particles per walk
constexpr int64_t kRoomMax = 1 << 16;
constexpr int64_t kRoomMaxEntries = 1ll << 31;  // entries of one kind's rooms (8 GiB)
constexpr size_t kRoomsHeld = 1ull << 32;       // of all rooms that a handle holds (16 GiB)

struct sphk_dtree : sphk::NodeBuffers<HipAlloc, BoxRec, MacRec> {
    int n = 0, n_leaf = 8, n_group = 16;
    hipStream_t st = nullptr;
    // a detached handle knows no stream: its last work is marked by `left`
    bool detached = false;
    hipEvent_t left = nullptr;
    DArr<double> x, y, z, part, frame;
    DArr<uint64_t> key;
    std::vector<int> level_start;   // node index of the first node of each level
    int n_node = 0;
    DArr<int32_t> head, group, i_off, hist;
    sphk::ListRooms<HipAlloc> rooms{kRoomsHeld};
    DArr<Span> span;
    DArr<int64_t> levels;   // starts of the levels and the node count; the group count; the unsorted flag
    int n_walk = 0;
    DArr<double> wbox;
    DArr<OboxRec> orec;
    DArr<int64_t> i64a, i64b, i64c, i64d;
    DArr<int64_t> total;
    int *err = nullptr;             // overflow flags of the list walks, 0 between builds (in levels)
    DArr<char> scratch;
    DLists lists[3];
    // per-walk rooms of the one-pass list builds (gather and symmetry
    // members; long-list EPJ and SPJ entries), doubled after a build that
    // overflowed them
    int64_t room[2] = {kRoomNearStart, kRoomNearStart};
    int64_t room_long[2] = {kRoomLongStart, kRoomStart};
    bool deep[3] = {false, false, false};   // whether a kind's last build had walks for the deep kernel

    // holds no tree and no lists
    void forget()
    {
        n_walk = 0;
        n_node = 0;
        for (int k = 0; k < 3; k++) {
            lists[k].built = false;
            rooms.lies[k] = -1;
        }
    }
    NodeArrays nodes() { return NodeArrays{begin.p, end.p, child.p, nchild.p, level.p, parent.p, len.p}; }
    Moments moments()
    {
        return Moments{box_lo.p, box_hi.p, mm.p, mx.p, my.p, mz.p, me.p, sx.p, sy.p, sz.p, se.p, node_cap};
    }
    void release()
    {
        release_nodes();
        for (auto *a : {&x, &y, &z, &part, &frame}) a->release();
        key.release();
        for (auto *a : {&head, &group, &i_off, &hist}) a->release();
        rooms.release();
        span.release();
        levels.release();
        wbox.release();
        orec.release();
        for (auto *a : {&i64a, &i64b, &i64c, &i64d, &total}) a->release();
        scratch.release();
        for (auto &L : lists) {
            L.j_off.release();
            L.j_idx.release();
            L.s_off.release();
            L.s_idx.release();
        }
    }
};

namespace {

// exclusive scan of n int64 counts (queued on st)
int scan64(sphk_dtree *t, const int64_t *in, int64_t *out, int n)
{
    size_t bytes = 0;
    SPHK_TRY(rocprim::exclusive_scan(nullptr, bytes, in, out, (int64_t)0, (size_t)n, rocprim::plus<int64_t>(),
                                     t->st));
    SPHK_TRY(t->scratch.reserve(bytes + 16, false, t->st));
    SPHK_TRY(rocprim::exclusive_scan(t->scratch.p, bytes, in, out, (int64_t)0, (size_t)n,
                                     rocprim::plus<int64_t>(), t->st));
    return SPHK_OK;
}

template <typename T>
int read1(hipStream_t st, const T *dev, T *host)
{
    SPHK_TRY(hipMemcpyAsync(host, dev, sizeof(T), hipMemcpyDeviceToHost, st));
    SPHK_TRY(hipStreamSynchronize(st));
    return SPHK_OK;
}

int grid(int n) { return (n + kBlock - 1) / kBlock; }

// Both totals of a list and the list walks' overflow flags, in one copy (each
// copy to the host waits for the one before it).
int read_totals(sphk_dtree *t, int64_t (&tot)[2], int &overflow)
{
    int64_t h[3] = {0, 0, 0};
    SPHK_TRY(hipMemcpyAsync(h, t->total.p, sizeof(h), hipMemcpyDeviceToHost, t->st));
    SPHK_TRY(hipStreamSynchronize(t->st));
    tot[0] = h[0];
    tot[1] = h[1];
    overflow = (int)h[2];
    return SPHK_OK;
}

// Per-walk counts -> offsets and totals: counts a (and b) are scanned into
// c (and d); off_a / off_b receive the walk offsets.
int walk_offsets(sphk_dtree *t, int ng, const int64_t *a, int64_t *c, int32_t *off_a, const int64_t *b,
                 int64_t *d, int32_t *off_b)
{
    if (ng <= kScanWalks) {
        hipLaunchKernelGGL(list_scan_kernel, dim3(b ? 2 : 1), dim3(kScanThreads), 0, t->st, ng, a, c, off_a, b, d,
                           off_b, t->total.p, t->err);
        SPHK_TRY(hipGetLastError());
        return SPHK_OK;
    }
    if (int rc = scan64(t, a, c, ng)) return rc;
    hipLaunchKernelGGL(offsets_kernel, dim3(grid(ng)), dim3(kBlock), 0, t->st, ng, c, a, off_a, t->total.p, t->err,
                       t->total.p + 2);
    if (b) {
        if (int rc = scan64(t, b, d, ng)) return rc;
        hipLaunchKernelGGL(offsets_kernel, dim3(grid(ng)), dim3(kBlock), 0, t->st, ng, d, b, off_b, t->total.p + 1,
                           nullptr, nullptr);
    }
    SPHK_TRY(hipGetLastError());
    return SPHK_OK;
}

// The walks of a list into their rooms, and the walk offsets: walks(false_type)
// queues the kernel for all of them, walks(true_type) the deep one.  A kind
// that had deep walks in its last build has both queued at once; else the deep
// kernel, the offsets and their read follow when the flags ask for them.
// flags: what is left for the counted build, 0 if the list is whole.
template <class Walks, class Offsets>
int room_walks(sphk_dtree *t, int kind, Walks &&walks, Offsets &&offsets, int64_t (&tot)[2], int &flags)
{
    const bool known = t->deep[kind];
    bool both = known;
    walks(std::false_type{});
    if (both) walks(std::true_type{});
    for (;;) {
        SPHK_TRY(hipGetLastError());
        if (int rc = offsets()) return rc;
        if (int rc = read_totals(t, tot, flags)) return rc;
        if (flags != kFlagDeep || both) break;
        t->deep[kind] = both = true;
        walks(std::true_type{});
    }
    if (known) t->deep[kind] = (flags & kFlagDeep) != 0;
    if (both) flags &= ~kFlagDeep;
    return SPHK_OK;
}

// A list still in the rooms of the scratch: packed to its offsets, into the
// caller's arrays (j_idx / s_idx non-NULL; the list stays in the rooms) or
// into the handle's own (the list leaves the rooms).
int pack_list(sphk_dtree *t, int kind, int32_t *j_idx, int32_t *s_idx)
{
    DLists &L = t->lists[kind];
    const int at = t->rooms.lies[kind];
    if (!L.built || at < 0) return SPHK_OK;
    const int ng = t->n_walk;
    const bool own = j_idx == nullptr;
    if (own) {
        SPHK_TRY(L.j_idx.reserve(std::max<int64_t>(L.n_j, 1), false, t->st));
        j_idx = L.j_idx.p;
        if (kind == 2) {
            SPHK_TRY(L.s_idx.reserve(std::max<int64_t>(L.n_s, 1), false, t->st));
            s_idx = L.s_idx.p;
        }
    }
    hipLaunchKernelGGL(room_copy_kernel, dim3((ng + kCopyWalks - 1) / kCopyWalks), dim3(64 * kCopyWalks), 0, t->st, ng,
                       L.room_j, L.j_off.p, t->rooms.of[at].p, j_idx);
    if (kind == 2 && s_idx)
        hipLaunchKernelGGL(room_copy_kernel, dim3((ng + kCopyWalks - 1) / kCopyWalks), dim3(64 * kCopyWalks), 0, t->st,
                           ng, L.room_s, L.s_off.p, t->rooms.nodes.p, s_idx);
    SPHK_TRY(hipGetLastError());
    if (own) t->rooms.lies[kind] = -1;
    return SPHK_OK;
}

// Interaction lists of every walk: one pass into rooms, and if a room
// overflowed (or does not fit in memory) the counted build.  That is, for the long list, the tree
// walk run as count, scan and fill; for the short-range lists (gather: r =
// rs, symmetry: r = H) the tree walk (count, scan, fill) writes the particles
// of the leaves reached into the walk's stretch of a scratch array,
// member_kernel keeps the members there, and they are copied to their offsets
// in the list.
template <int MODE>
int build_list(sphk_dtree *t, const double *r, double inv_t2)
{
    DLists &L = t->lists[MODE];
    L.built = false;
    t->rooms.lies[MODE] = -1;
    auto pack = [&](int kind) { return pack_list(t, kind, nullptr, nullptr); };   // another kind's list, where rooms are shared
    int rc_rooms = 0;
    const int ng = t->n_walk;
    // i-particles staged in LDS by the member test: a walk holds <= n_group
    // particles unless it is a leaf (<= n_leaf; more only at the deepest level)
    const int n_si = std::min(kWalkI, std::max(t->n_group, t->n_leaf));
    SPHK_TRY(t->i64a.reserve(ng, false, t->st));   // EPJ counts per walk
    SPHK_TRY(t->i64b.reserve(ng, false, t->st));   // SPJ counts
    SPHK_TRY(t->i64c.reserve(ng, false, t->st));   // EPJ offsets
    SPHK_TRY(t->i64d.reserve(ng, false, t->st));   // SPJ offsets
    SPHK_TRY(t->total.reserve(3, false, t->st));
    SPHK_TRY(L.j_off.reserve(ng + 1, false, t->st));
    if (MODE == 2) SPHK_TRY(L.s_off.reserve(ng + 1, false, t->st));
    if (MODE != 2) {
        SPHK_TRY(t->wbox.reserve(7 * (size_t)ng, false, t->st));
        hipLaunchKernelGGL(walk_box_kernel, dim3(grid(ng)), dim3(kBlock), 0, t->st, ng, t->i_off.p, t->x.p,
                           t->y.p, t->z.p, r, t->wbox.p);
    }
    TreeView v{t->nodes(), t->moments(), t->brec.p, t->mrec.p, t->orec.p, t->x.p, t->y.p, t->z.p, t->group.p,
               t->i_off.p};
    const double *wb = MODE == 2 ? nullptr : t->wbox.p;
    const dim3 lg((unsigned)((ng + kListWalks - 1) / kListWalks)), lb(64);
    if constexpr (MODE != 2) {
        // one pass into a room per walk: no count walk, one host read.  If a
        // walk overflows its room, the counted build below runs instead (and
        // later builds get twice the room), and so it does where the rooms do
        // not fit in memory.
        int64_t &room = t->room[MODE];
        const int at = (int64_t)ng * room <= kRoomMaxEntries
                           ? t->rooms.take(MODE, (size_t)ng * (size_t)room, 0, t->st, pack, rc_rooms)
                           : -1;
        if (rc_rooms) return rc_rooms;
        if (at >= 0) {
            auto walks = [&](auto deep) {
                hipLaunchKernelGGL((room_list_kernel<MODE, decltype(deep)::value>), dim3(ng), dim3(64),
                                   n_si * sizeof(double4), t->st, ng, v, wb, r, 0., t->i64b.p, t->rooms.of[at].p, room,
                                   nullptr, nullptr, 0, n_si, t->err);
            };
            auto offsets = [&]() { return walk_offsets(t, ng, t->i64b.p, t->i64d.p, L.j_off.p, nullptr, nullptr, nullptr); };
            int64_t tot1[2] = {0, 0};
            int flags = 0;
            if (int rc = room_walks(t, MODE, walks, offsets, tot1, flags)) return rc;
            if (flags == 0) {
                if (tot1[0] > std::numeric_limits<int32_t>::max())
                    return set_error(SPHK_E_CAPACITY, "dtree: list longer than 2^31 entries");
                // the members stay in their rooms until the list is read
                L.n_j = tot1[0];
                L.n_s = 0;
                t->rooms.lies[MODE] = at;
                L.room_j = room;
                L.room_s = 0;
                L.built = true;
                return SPHK_OK;
            }
            if (flags & kFlagRoom) room = std::min<int64_t>(room * 2, kRoomMax);
        }
    }
    if constexpr (MODE == 2) {
        // one walk into rooms per walk (EPJ and SPJ), then the entries packed
        // to the walk offsets: no count walk, one host read.  The counted
        // build below if a walk overflows a room (and later builds get twice
        // the room that overflowed).
        int64_t &rj = t->room_long[0], &rsp = t->room_long[1];
        const int at = (int64_t)ng * rj <= kRoomMaxEntries && (int64_t)ng * rsp <= kRoomMaxEntries
                           ? t->rooms.take(MODE, (size_t)ng * (size_t)rj, (size_t)ng * (size_t)rsp, t->st, pack, rc_rooms)
                           : -1;
        if (rc_rooms) return rc_rooms;
        if (at >= 0) {
            auto walks = [&](auto deep) {
                hipLaunchKernelGGL((room_list_kernel<2, decltype(deep)::value>), dim3(ng), dim3(64), 0, t->st, ng, v, wb,
                                   r, inv_t2, t->i64a.p, t->rooms.of[at].p, rj, t->i64b.p, t->rooms.nodes.p, rsp, 0,
                                   t->err);
            };
            auto offsets = [&]() {
                return walk_offsets(t, ng, t->i64a.p, t->i64c.p, L.j_off.p, t->i64b.p, t->i64d.p, L.s_off.p);
            };
            int64_t tot1[2] = {0, 0};
            int flags = 0;
            if (int rc = room_walks(t, MODE, walks, offsets, tot1, flags)) return rc;
            if (flags == 0) {
                if (tot1[0] > std::numeric_limits<int32_t>::max() || tot1[1] > std::numeric_limits<int32_t>::max())
                    return set_error(SPHK_E_CAPACITY, "dtree: list longer than 2^31 entries");
                // the entries stay in their rooms until the list is read
                L.n_j = tot1[0];
                L.n_s = tot1[1];
                t->rooms.lies[MODE] = at;
                L.room_j = rj;
                L.room_s = rsp;
                L.built = true;
                return SPHK_OK;
            }
            if (flags & kFlagRoom) rj = std::min<int64_t>(rj * 2, kRoomMax);
            if (flags & kFlagNodes) rsp = std::min<int64_t>(rsp * 2, kRoomMax);
        }
    }
    // count walk with the small stack, and with the worst-case one if a walk overflowed it
    int64_t tot[2] = {0, 0};
    int overflow = 0;
    bool big = false;
    for (;;) {
        if (big)
            hipLaunchKernelGGL((walk_list_kernel<MODE, 0, kListStack>), lg, lb, 0, t->st, ng, v, wb, r, inv_t2,
                               t->i64a.p, t->i64b.p, nullptr, nullptr, nullptr, nullptr, t->err);
        else
            hipLaunchKernelGGL((walk_list_kernel<MODE, 0, kListStackSmall>), lg, lb, 0, t->st, ng, v, wb, r,
                               inv_t2, t->i64a.p, t->i64b.p, nullptr, nullptr, nullptr, nullptr, t->err);
        SPHK_TRY(hipGetLastError());
        if (int rc = walk_offsets(t, ng, t->i64a.p, t->i64c.p, L.j_off.p, MODE == 2 ? t->i64b.p : nullptr,
                                  t->i64d.p, L.s_off.p))
            return rc;
        if (int rc = read_totals(t, tot, overflow)) return rc;
        if (!overflow) break;
        if (big) return set_error(SPHK_E_STATE, "dtree: list walk stack overflow (corrupt tree)");
        big = true;
    }
    if (MODE != 2) tot[1] = 0;
    if (tot[0] > std::numeric_limits<int32_t>::max() || tot[1] > std::numeric_limits<int32_t>::max())
        return set_error(SPHK_E_CAPACITY, "dtree: list longer than 2^31 entries");
    if constexpr (MODE == 2) {
        SPHK_TRY(L.j_idx.reserve(std::max<int64_t>(tot[0], 1), false, t->st));
        SPHK_TRY(L.s_idx.reserve(std::max<int64_t>(tot[1], 1), false, t->st));
        if (big)
            hipLaunchKernelGGL((walk_list_kernel<MODE, 1, kListStack>), lg, lb, 0, t->st, ng, v, wb, r, inv_t2,
                               nullptr, nullptr, t->i64c.p, t->i64d.p, L.j_idx.p, L.s_idx.p, t->err);
        else
            hipLaunchKernelGGL((walk_list_kernel<MODE, 1, kListStackSmall>), lg, lb, 0, t->st, ng, v, wb, r,
                               inv_t2, nullptr, nullptr, t->i64c.p, t->i64d.p, L.j_idx.p, L.s_idx.p, t->err);
        SPHK_TRY(hipGetLastError());
    } else {
        // tot[0] candidates into the scratch; the members compacted in place,
        // their counts to i64b
        const int at = t->rooms.take(MODE, (size_t)std::max<int64_t>(tot[0], 1), 0, t->st, pack, rc_rooms);
        if (rc_rooms) return rc_rooms;
        if (at < 0) return set_error(SPHK_E_DEVICE, "dtree: no memory for %lld candidates", (long long)tot[0]);
        int32_t *const cand = t->rooms.of[at].p;
        if (big)
            hipLaunchKernelGGL((walk_list_kernel<MODE, 1, kListStack>), lg, lb, 0, t->st, ng, v, wb, r, inv_t2,
                               nullptr, nullptr, t->i64c.p, nullptr, cand, nullptr, t->err);
        else
            hipLaunchKernelGGL((walk_list_kernel<MODE, 1, kListStackSmall>), lg, lb, 0, t->st, ng, v, wb, r,
                               inv_t2, nullptr, nullptr, t->i64c.p, nullptr, cand, nullptr, t->err);
        hipLaunchKernelGGL((member_kernel<MODE>), dim3(ng), dim3(64), n_si * sizeof(double4), t->st, ng, v, wb, r,
                           t->i64c.p, t->i64a.p, cand, t->i64b.p, n_si);
        SPHK_TRY(hipGetLastError());
        if (int rc = walk_offsets(t, ng, t->i64b.p, t->i64d.p, L.j_off.p, nullptr, nullptr, nullptr)) return rc;
        if (int rc = read_totals(t, tot, overflow)) return rc;
        if (overflow) return set_error(SPHK_E_STATE, "dtree: list walk stack overflow in the fill walk");
        tot[1] = 0;
        if (tot[0] > std::numeric_limits<int32_t>::max())
            return set_error(SPHK_E_CAPACITY, "dtree: list longer than 2^31 entries");
        SPHK_TRY(L.j_idx.reserve(std::max<int64_t>(tot[0], 1), false, t->st));
        hipLaunchKernelGGL(member_copy_kernel, dim3(ng), dim3(64), 0, t->st, ng, t->i64c.p, L.j_off.p, cand,
                           L.j_idx.p);
        SPHK_TRY(hipGetLastError());
    }
    L.n_j = tot[0];
    L.n_s = tot[1];
    L.built = true;
    return SPHK_OK;
}

// Workspace of sphk_morton_order_dev, one per device, grown as needed and
// kept until the process ends (no allocation once it has reached the run's
// size).  Calls on one device take it in turn; each call's stream first
// waits for the previous call's work (an event), so no host wait is needed.
struct MortonWork {
    std::mutex mu;
    DArr<double> part, frame;
    DArr<uint64_t> key, key2;
    DArr<int32_t> idx;
    DArr<char> tmp;
    hipEvent_t done = nullptr;
};
constexpr int kMortonDevices = 16;
MortonWork g_morton[kMortonDevices];

}  // namespace

extern "C" {

int sphk_morton_order_dev(int n, const double *x, const double *y, const double *z, int32_t *perm, void *stream)
{
    if (n < 0 || (n > 0 && (!x || !y || !z || !perm))) return set_error(SPHK_E_ARG, "morton_dev: bad args");
    if (n == 0) return SPHK_OK;
    hipStream_t st = (hipStream_t)stream;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMortonDevices)
        return set_error(SPHK_E_DEVICE, "morton_dev: no usable current device");
    MortonWork &w = g_morton[dev];
    std::lock_guard<std::mutex> lock(w.mu);
    // the previous call's kernels (maybe on another stream) finish before the workspace is reused
    if (!w.done) {
        if (hipEventCreateWithFlags(&w.done, hipEventDisableTiming) != hipSuccess) {
            w.done = nullptr;
            return set_error(SPHK_E_DEVICE, "morton_dev: event creation failed");
        }
    } else {
        SPHK_TRY(hipStreamWaitEvent(st, w.done, 0));
    }
    SPHK_TRY(w.idx.reserve(n, false, st));
    SPHK_TRY(w.key2.reserve(n, false, st));
    if (int rc = make_keys(n, x, y, z, st, w.part, w.frame, w.key, w.idx.p)) return rc;
    size_t bytes = 0;
    SPHK_TRY(rocprim::radix_sort_pairs(nullptr, bytes, w.key.p, w.key2.p, w.idx.p, perm, (size_t)n, 0, 63, st));
    SPHK_TRY(w.tmp.reserve(bytes + 16, false, st));
    SPHK_TRY(rocprim::radix_sort_pairs(w.tmp.p, bytes, w.key.p, w.key2.p, w.idx.p, perm, (size_t)n, 0, 63, st));
    SPHK_TRY(hipEventRecord(w.done, st));
    return SPHK_OK;
}

namespace {

// The levels that moments_top_kernel and obox_top_kernel take: from the root
// while none is wider than kTopNodes.
TopLevels top_levels(const sphk_dtree *t)
{
    TopLevels tl{};
    const int n = (int)t->level_start.size() - 1;
    while (tl.levels < n && t->level_start[tl.levels + 1] - t->level_start[tl.levels] <= kTopNodes) tl.levels++;
    for (int L = 0; L <= tl.levels; L++) tl.ls[L] = t->level_start[L];
    return tl;
}

// The build proper, into t's buffers (grown as needed).  On failure t holds
// no tree; its buffers stay allocated for a later build or sphk_dtree_free.
int build_tree(sphk_dtree *t, int n, const double *x, const double *y, const double *z, const double *m,
               const double *eps2, int n_leaf, int n_group, hipStream_t stream)
{
    // a previous user of the buffers may still be queued on the old stream
    if (t->detached ? hipStreamWaitEvent(stream, t->left, 0) != hipSuccess
                    : t->st != stream && hipStreamSynchronize(t->st) != hipSuccess)
        return set_error(SPHK_E_DEVICE, "dtree: stream synchronisation failed");
    t->detached = false;
    t->n = n;
    t->n_leaf = n_leaf;
    t->n_group = n_group;
    t->st = stream;
    t->forget();
    auto fail = [&](int rc) {
        t->n_walk = 0;
        t->n_node = 0;
        return rc;
    };
    hipStream_t st = t->st;
    const int nb = (n + kSpanTile - 1) / kSpanTile;
    // own copies of the positions (list builds read them later)
    for (auto *a : {&t->x, &t->y, &t->z})
        if (a->reserve(n, false, st) != hipSuccess) return fail(set_error(SPHK_E_DEVICE, "dtree: allocation failed"));
    if (t->span.reserve(n, false, st) != hipSuccess ||
        t->head.reserve(n, false, st) != hipSuccess || t->hist.reserve((size_t)kLevels * nb, false, st) != hipSuccess ||
        t->levels.reserve(kLevels + 4, false, st) != hipSuccess)
        return fail(set_error(SPHK_E_DEVICE, "dtree: allocation failed"));
    double *const copies[3] = {t->x.p, t->y.p, t->z.p};
    if (int rc = make_keys(n, x, y, z, st, t->part, t->frame, t->key, nullptr, copies)) return fail(rc);

    // nodes per level: one host read of the level starts and the order check
    int64_t *const lv = t->levels.p, *const n_group_dev = lv + kLevels + 1;
    int *const unsorted = reinterpret_cast<int *>(lv + kLevels + 2);
    t->err = unsorted + 2;
    hipLaunchKernelGGL(fill_kernel, dim3(1), dim3(kBlock), 0, st, 4, reinterpret_cast<int32_t *>(unsorted), 0);
    hipLaunchKernelGGL(span_kernel, dim3(nb), dim3(kSpanTile), 0, st, n, t->key.p, std::min(n_leaf, n), t->span.p, t->hist.p,
                       t->head.p, unsorted);
    hipLaunchKernelGGL(block_scan_kernel, dim3(1), dim3(kScanThreads), 0, st, kLevels * nb, t->hist.p, kLevels, nb, lv,
                       lv + kLevels);
    int64_t h[kLevels + 3];
    if (hipMemcpyAsync(h, lv, sizeof(h), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return fail(set_error(SPHK_E_DEVICE, "dtree: level sizes read failed"));
    if (h[kLevels + 2] != 0)
        return fail(set_error(SPHK_E_ARG, "dtree: particles are not in Morton order (use sphk_morton_order_dev)"));
    if (h[kLevels] >= (1 << 29))   // list walks pack node indices into 29 bits
        return fail(set_error(SPHK_E_CAPACITY, "dtree: too many nodes"));
    const size_t nn = (size_t)h[kLevels];
    t->n_node = (int)nn;
    t->level_start.clear();
    for (int L = 0; L <= kLevels && (L == 0 || h[L] > h[L - 1]); L++) t->level_start.push_back((int)h[L]);
    if (t->reserve_nodes(nn, 2 * (size_t)n / std::max(1, n_leaf) + 16, st) != hipSuccess)
        return fail(set_error(SPHK_E_DEVICE, "dtree: allocation failed"));
    hipLaunchKernelGGL(fill_kernel, dim3(grid((int)nn)), dim3(kBlock), 0, st, (int)nn, t->nchild.p, 0);
    hipLaunchKernelGGL(node_kernel, dim3(nb), dim3(kSpanTile), 0, st, n, t->key.p, t->span.p, t->hist.p, t->nodes(),
                       t->frame.p);

    // boxes and monopoles, deepest level first
    const TopLevels top = top_levels(t);
    for (int L = (int)t->level_start.size() - 2; L >= top.levels; L--) {
        const int a0 = t->level_start[L], na = t->level_start[L + 1] - a0;
        hipLaunchKernelGGL(moments_kernel, dim3(grid(na)), dim3(kBlock), 0, st, a0, na, t->nodes(), t->moments(),
                           t->brec.p, t->mrec.p, t->x.p, t->y.p, t->z.p, m, eps2);
    }
    hipLaunchKernelGGL(moments_top_kernel, dim3(1), dim3(kTopThreads), 0, st, top, t->nodes(), t->moments(), t->brec.p,
                       t->mrec.p, t->x.p, t->y.p, t->z.p, m, eps2);
    if (hipGetLastError() != hipSuccess) return fail(set_error(SPHK_E_DEVICE, "dtree: moments launch failed"));

    // groups (at most one per particle)
    if (t->group.reserve(n, false, st) != hipSuccess || t->i_off.reserve((size_t)n + 1, false, st) != hipSuccess)
        return fail(set_error(SPHK_E_DEVICE, "dtree: allocation failed"));
    hipLaunchKernelGGL(group_mark_kernel, dim3(grid((int)nn)), dim3(kBlock), 0, st, (int)nn, t->nodes(), n_group,
                       t->head.p);
    hipLaunchKernelGGL(group_count_kernel, dim3(nb), dim3(kSpanTile), 0, st, n, t->head.p, t->hist.p);
    hipLaunchKernelGGL(block_scan_kernel, dim3(1), dim3(kScanThreads), 0, st, nb, t->hist.p, 0, 1, nullptr, n_group_dev);
    hipLaunchKernelGGL(group_write_kernel, dim3(nb), dim3(kSpanTile), 0, st, n, t->head.p, t->hist.p, n_group_dev,
                       t->group.p, t->i_off.p);
    if (hipGetLastError() != hipSuccess) return fail(set_error(SPHK_E_DEVICE, "dtree: build failed"));
    int64_t groups = 0;
    if (int rc = read1(st, n_group_dev, &groups)) return fail(rc);
    const int ng = (int)groups;
    t->n_walk = ng;
    return SPHK_OK;
}

int check_build_args(int n, const double *x, const double *y, const double *z, const double *m, int n_leaf,
                     int n_group)
{
    if (n <= 0 || !x || !y || !z || !m) return set_error(SPHK_E_ARG, "dtree: bad particle arrays");
    // list walks pack node and particle indices into 29 bits
    if (n >= (1 << 29)) return set_error(SPHK_E_CAPACITY, "dtree: at most 2^29 - 1 particles per tree");
    if (n_leaf < 1 || n_group < 1) return set_error(SPHK_E_ARG, "dtree: n_leaf, n_group must be >= 1");
    return SPHK_OK;
}

}  // namespace

int sphk_dtree_build(int n, const double *x, const double *y, const double *z, const double *m,
                     const double *eps2, int n_leaf, int n_group, void *stream, sphk_dtree **out)
{
    if (!out) return set_error(SPHK_E_ARG, "dtree: null output");
    *out = nullptr;
    if (int rc = check_build_args(n, x, y, z, m, n_leaf, n_group)) return rc;
    sphk_dtree *t = new (std::nothrow) sphk_dtree();
    if (!t) return set_error(SPHK_E_CAPACITY, "dtree: out of memory");
    t->st = (hipStream_t)stream;
    if (int rc = build_tree(t, n, x, y, z, m, eps2, n_leaf, n_group, (hipStream_t)stream)) {
        t->release();
        delete t;
        return rc;
    }
    *out = t;
    return SPHK_OK;
}

int sphk_dtree_rebuild(sphk_dtree *t, int n, const double *x, const double *y, const double *z,
                       const double *m, const double *eps2, int n_leaf, int n_group, void *stream)
{
    if (!t) return set_error(SPHK_E_ARG, "dtree: null handle");
    if (int rc = check_build_args(n, x, y, z, m, n_leaf, n_group)) return rc;
    return build_tree(t, n, x, y, z, m, eps2, n_leaf, n_group, (hipStream_t)stream);
}

int sphk_dtree_detach(sphk_dtree *t)
{
    if (!t) return set_error(SPHK_E_ARG, "dtree detach: null handle");
    if (t->detached) return SPHK_OK;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(t->st, &cs);   // an event recorded into a graph marks nothing
    if (e == hipSuccess && cs != hipStreamCaptureStatusNone)
        return set_error(SPHK_E_STATE, "dtree detach: the stream is being captured");
    if (e == hipSuccess && !t->left) e = hipEventCreateWithFlags(&t->left, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(t->left, t->st);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return set_error(SPHK_E_DEVICE, "dtree detach: %s", hipGetErrorString(e));
    }
    t->detached = true;
    t->st = nullptr;
    t->forget();
    return SPHK_OK;
}

void sphk_dtree_free(sphk_dtree *t)
{
    if (!t) return;
    if (t->detached)
        (void)hipEventSynchronize(t->left);
    else
        (void)hipStreamSynchronize(t->st);
    if (t->left) (void)hipEventDestroy(t->left);
    t->release();
    delete t;
}

int sphk_dtree_n_walk(const sphk_dtree *t) { return t ? t->n_walk : -1; }
int sphk_dtree_n_node(const sphk_dtree *t) { return t ? t->n_node : -1; }
const int32_t *sphk_dtree_i_off(const sphk_dtree *t) { return t ? t->i_off.p : nullptr; }

int sphk_dtree_list_gather(sphk_dtree *t, const double *rs)
{
    if (!t || !rs) return set_error(SPHK_E_ARG, "dtree gather: null argument");
    if (t->n_walk <= 0) return set_error(SPHK_E_STATE, "dtree gather: no tree built");
    return build_list<0>(t, rs, 0.);
}

int sphk_dtree_list_symmetry(sphk_dtree *t, const double *h)
{
    if (!t || !h) return set_error(SPHK_E_ARG, "dtree symmetry: null argument");
    if (t->n_walk <= 0) return set_error(SPHK_E_STATE, "dtree symmetry: no tree built");
    if (t->orec.reserve((size_t)t->n_node, false, t->st) != hipSuccess)
        return set_error(SPHK_E_DEVICE, "dtree symmetry: allocation failed");
    const TopLevels top = top_levels(t);
    for (int L = (int)t->level_start.size() - 2; L >= top.levels; L--) {
        const int a0 = t->level_start[L], na = t->level_start[L + 1] - a0;
        hipLaunchKernelGGL(obox_kernel, dim3(grid(na)), dim3(kBlock), 0, t->st, a0, na, t->nodes(), t->orec.p, t->x.p,
                           t->y.p, t->z.p, h);
    }
    hipLaunchKernelGGL(obox_top_kernel, dim3(1), dim3(kTopThreads), 0, t->st, top, t->nodes(), t->orec.p, t->x.p,
                       t->y.p, t->z.p, h);
    SPHK_TRY(hipGetLastError());
    return build_list<1>(t, h, 0.);
}

int sphk_dtree_list_long(sphk_dtree *t, double theta)
{
    if (!t || !(theta >= 0.)) return set_error(SPHK_E_ARG, "dtree long: bad argument");
    if (t->n_walk <= 0) return set_error(SPHK_E_STATE, "dtree long: no tree built");
    const double inv_t2 = theta > 0. ? 1. / (theta * theta) : std::numeric_limits<double>::infinity();
    return build_list<2>(t, nullptr, inv_t2);
}

int sphk_dtree_list(sphk_dtree *t, int kind, const int32_t **j_off, const int32_t **j_idx,
                    const int32_t **s_off, const int32_t **s_idx, int64_t *n_j, int64_t *n_s)
{
    if (!t || kind < 0 || kind > 2) return set_error(SPHK_E_ARG, "dtree list: bad argument");
    DLists &L = t->lists[kind];
    if (!L.built) return set_error(SPHK_E_STATE, "dtree list kind %d not built", kind);
    if (int rc = pack_list(t, kind, nullptr, nullptr)) return rc;
    if (j_off) *j_off = L.j_off.p;
    if (j_idx) *j_idx = L.j_idx.p;
    if (s_off) *s_off = kind == 2 ? L.s_off.p : nullptr;
    if (s_idx) *s_idx = kind == 2 ? L.s_idx.p : nullptr;
    if (n_j) *n_j = L.n_j;
    if (n_s) *n_s = L.n_s;
    return SPHK_OK;
}

int sphk_dtree_list_size(const sphk_dtree *t, int kind, int64_t *n_j, int64_t *n_s)
{
    if (!t || kind < 0 || kind > 2) return set_error(SPHK_E_ARG, "dtree list size: bad argument");
    const DLists &L = t->lists[kind];
    if (!L.built) return set_error(SPHK_E_STATE, "dtree list kind %d not built", kind);
    if (n_j) *n_j = L.n_j;
    if (n_s) *n_s = L.n_s;
    return SPHK_OK;
}

int sphk_dtree_list_copy(sphk_dtree *t, int kind, int32_t *j_off, int32_t *j_idx, int32_t *s_off, int32_t *s_idx)
{
    if (!t || kind < 0 || kind > 2 || !j_off || (!j_idx && t->lists[kind].n_j > 0))
        return set_error(SPHK_E_ARG, "dtree list copy: bad argument");
    DLists &L = t->lists[kind];
    if (!L.built) return set_error(SPHK_E_STATE, "dtree list kind %d not built", kind);
    if (kind == 2 && (!s_off || (!s_idx && L.n_s > 0)))
        return set_error(SPHK_E_ARG, "dtree list copy: null SPJ array");
    const size_t no = (size_t)t->n_walk + 1;
    SPHK_TRY(hipMemcpyAsync(j_off, L.j_off.p, no * sizeof(int32_t), hipMemcpyDeviceToDevice, t->st));
    if (kind == 2) SPHK_TRY(hipMemcpyAsync(s_off, L.s_off.p, no * sizeof(int32_t), hipMemcpyDeviceToDevice, t->st));
    if (t->rooms.lies[kind] >= 0) return pack_list(t, kind, j_idx, kind == 2 ? s_idx : nullptr);
    if (L.n_j > 0)
        SPHK_TRY(hipMemcpyAsync(j_idx, L.j_idx.p, (size_t)L.n_j * sizeof(int32_t), hipMemcpyDeviceToDevice, t->st));
    if (kind == 2 && L.n_s > 0)
        SPHK_TRY(hipMemcpyAsync(s_idx, L.s_idx.p, (size_t)L.n_s * sizeof(int32_t), hipMemcpyDeviceToDevice, t->st));
    return SPHK_OK;
}

int sphk_dtree_moments(const sphk_dtree *t, const double **m, const double **x, const double **y,
                       const double **z, const double **eps2)
{
    if (!t) return set_error(SPHK_E_ARG, "dtree moments: null tree");
    if (m) *m = t->mm.p;
    if (x) *x = t->mx.p;
    if (y) *y = t->my.p;
    if (z) *z = t->mz.p;
    if (eps2) *eps2 = t->me.p;
    return SPHK_OK;
}

int sphk_dtree_nodes(const sphk_dtree *t, const int32_t **begin, const int32_t **end, const int32_t **child,
                     const int32_t **nchild, const int32_t **level, const double **len)
{
    if (!t) return set_error(SPHK_E_ARG, "dtree nodes: null tree");
    if (begin) *begin = t->begin.p;
    if (end) *end = t->end.p;
    if (child) *child = t->child.p;
    if (nchild) *nchild = t->nchild.p;
    if (level) *level = t->level.p;
    if (len) *len = t->len.p;
    return SPHK_OK;
}

}  // extern "C"

namespace {

// cotangent per unit mass of each node's centre of mass, summed over the node
// and its ancestors (at most 21 levels up)
__global__ __launch_bounds__(kBlock) void spread_node_kernel(int nn, NodeArrays nd, const double *__restrict__ M,
                                                             const double *__restrict__ nx,
                                                             const double *__restrict__ ny,
                                                             const double *__restrict__ nz, double *__restrict__ cx,
                                                             double *__restrict__ cy, double *__restrict__ cz)
{
    const int a = blockIdx.x * kBlock + threadIdx.x;
    if (a >= nn) return;
    double s[3] = {0., 0., 0.};
    for (int b = a; b >= 0; b = nd.parent[b])
        if (M[b] > 0.) {
            s[0] += nx[b] / M[b];
            s[1] += ny[b] / M[b];
            s[2] += nz[b] / M[b];
        }
    cx[a] = s[0];
    cy[a] = s[1];
    cz[a] = s[2];
}

__global__ __launch_bounds__(kBlock) void spread_leaf_kernel(int nn, NodeArrays nd, const double *__restrict__ m,
                                                             const double *__restrict__ cx,
                                                             const double *__restrict__ cy,
                                                             const double *__restrict__ cz, double *gx, double *gy,
                                                             double *gz)
{
    const int a = blockIdx.x * kBlock + threadIdx.x;
    if (a >= nn || nd.child[a] >= 0) return;
    for (int k = nd.begin[a]; k < nd.end[a]; k++) {
        gx[k] += m[k] * cx[a];
        gy[k] += m[k] * cy[a];
        gz[k] += m[k] * cz[a];
    }
}

}  // namespace

extern "C" int sphk_dtree_spread_dev(const sphk_dtree *t, const double *m, const double *nx, const double *ny,
                                     const double *nz, double *gx, double *gy, double *gz)
{
    if (!t || !m || !nx || !ny || !nz || !gx || !gy || !gz) return set_error(SPHK_E_ARG, "dtree spread: null argument");
    sphk_dtree *tt = const_cast<sphk_dtree *>(t);
    const int nn = t->n_node;
    if (nn <= 0) return set_error(SPHK_E_STATE, "dtree spread: no tree built");
    // three per-node sums, kept in the SPJ scratch of the tree
    SPHK_TRY(tt->sx.reserve(nn, false, t->st));
    SPHK_TRY(tt->sy.reserve(nn, false, t->st));
    SPHK_TRY(tt->sz.reserve(nn, false, t->st));
    hipLaunchKernelGGL(spread_node_kernel, dim3(grid(nn)), dim3(kBlock), 0, t->st, nn, tt->nodes(), t->mm.p, nx, ny,
                       nz, tt->sx.p, tt->sy.p, tt->sz.p);
    hipLaunchKernelGGL(spread_leaf_kernel, dim3(grid(nn)), dim3(kBlock), 0, t->st, nn, tt->nodes(), m, tt->sx.p,
                       tt->sy.p, tt->sz.p, gx, gy, gz);
    SPHK_TRY(hipGetLastError());
    return SPHK_OK;
}

namespace {

// ---- reorder and input comparison (host glue of the rebuilds) ----------------
constexpr int kPermCols = 64;
struct PermCols {
    char *col[kPermCols];
    char *tmp[kPermCols];
    int elem[kPermCols];
};

template <typename T>
__device__ __forceinline__ void gather_col(int n, const int32_t *__restrict__ perm, const char *src, char *dst)
{
    const T *s = reinterpret_cast<const T *>(src);
    T *d = reinterpret_cast<T *>(dst);
    for (int k = blockIdx.x * kBlock + threadIdx.x; k < n; k += gridDim.x * kBlock) d[k] = s[perm ? perm[k] : k];
}

// tmp_c[k] = col_c[perm[k]], or with perm == nullptr col_c[k] = tmp_c[k];
// grid row c handles column c
__global__ __launch_bounds__(kBlock) void permute_kernel(int n, const int32_t *__restrict__ perm, PermCols pc)
{
    const int c = blockIdx.y;
    const char *src = perm ? pc.col[c] : pc.tmp[c];
    char *dst = perm ? pc.tmp[c] : pc.col[c];
    if (!perm && ((uintptr_t)dst % 16) == 0) {
        // copy back 16 bytes per thread (the scratch is 256-byte aligned)
        const size_t bytes = (size_t)n * pc.elem[c];
        const size_t n16 = bytes / 16;
        const uint4 *s4 = reinterpret_cast<const uint4 *>(src);
        uint4 *d4 = reinterpret_cast<uint4 *>(dst);
        const size_t stride = (size_t)gridDim.x * kBlock;
        for (size_t k = blockIdx.x * kBlock + threadIdx.x; k < n16; k += stride) d4[k] = s4[k];
        for (size_t k = n16 * 16 + blockIdx.x * kBlock + threadIdx.x; k < bytes; k += stride) dst[k] = src[k];
        return;
    }
    // gather, or a copy back by elements into a column aligned to less than 16 bytes
    switch (pc.elem[c]) {
    case 8: gather_col<uint64_t>(n, perm, src, dst); break;
    case 4: gather_col<uint32_t>(n, perm, src, dst); break;
    case 2: gather_col<uint16_t>(n, perm, src, dst); break;
    default: gather_col<uint8_t>(n, perm, src, dst); break;
    }
}

constexpr int kEqualArrays = 8;
struct EqualArrays {
    const uint64_t *a[kEqualArrays];
    const uint64_t *b[kEqualArrays];
};

__global__ __launch_bounds__(kBlock) void equal_kernel(int n, EqualArrays ea, int32_t *__restrict__ flag)
{
    const int c = blockIdx.y;
    bool diff = false;
    for (int k = blockIdx.x * kBlock + threadIdx.x; k < n; k += gridDim.x * kBlock)
        diff = diff || ea.a[c][k] != ea.b[c][k];
    if (__any(diff) && threadIdx.x % 64 == 0) *flag = 1;   // every writer stores 1
}

__global__ void flag_zero_kernel(int32_t *flag) { *flag = 0; }

size_t permute_work(int n, int count, const int *elem)
{
    size_t w = 0;
    for (int c = 0; c < count; c++) w += (((size_t)n * (size_t)elem[c]) + 255) / 256 * 256;
    return w;
}

}  // namespace

extern "C" {

size_t sphk_permute_work_bytes(int n, int count, const int *elem)
{
    if (n <= 0 || count <= 0 || count > kPermCols || !elem) return 0;
    return permute_work(n, count, elem);
}

int sphk_permute_dev(int n, const int32_t *perm, int count, void *const *cols, const int *elem, void *work,
                     size_t work_bytes, void *stream)
{
    if (n < 0 || count < 0 || count > kPermCols) return set_error(SPHK_E_ARG, "permute_dev: bad sizes");
    if (n == 0 || count == 0) return SPHK_OK;
    if (!perm || !cols || !elem || !work) return set_error(SPHK_E_ARG, "permute_dev: null pointer");
    PermCols pc{};
    size_t off = 0;
    for (int c = 0; c < count; c++) {
        if (!cols[c]) return set_error(SPHK_E_ARG, "permute_dev: null column %d", c);
        if (elem[c] != 1 && elem[c] != 2 && elem[c] != 4 && elem[c] != 8)
            return set_error(SPHK_E_ARG, "permute_dev: element size %d of column %d", elem[c], c);
        if (((uintptr_t)cols[c]) % (uintptr_t)elem[c])
            return set_error(SPHK_E_ARG, "permute_dev: column %d misaligned", c);
        pc.col[c] = static_cast<char *>(cols[c]);
        pc.tmp[c] = static_cast<char *>(work) + off;
        pc.elem[c] = elem[c];
        off += (((size_t)n * (size_t)elem[c]) + 255) / 256 * 256;
    }
    if (work_bytes < off) return set_error(SPHK_E_CAPACITY, "permute_dev: work of %zu bytes, %zu needed", work_bytes, off);
    if (((uintptr_t)work) % 256) return set_error(SPHK_E_ARG, "permute_dev: work not 256-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid(std::min(1024, (n + kBlock - 1) / kBlock), count);
    hipLaunchKernelGGL(permute_kernel, grid, dim3(kBlock), 0, st, n, perm, pc);
    hipLaunchKernelGGL(permute_kernel, grid, dim3(kBlock), 0, st, n, nullptr, pc);
    SPHK_TRY(hipGetLastError());
    return SPHK_OK;
}

int sphk_equal_dev(int n, int count, const double *const *a, const double *const *b, int32_t *flag, void *stream)
{
    if (n < 0 || count < 0 || count > kEqualArrays) return set_error(SPHK_E_ARG, "equal_dev: bad sizes");
    if (!flag) return set_error(SPHK_E_ARG, "equal_dev: null flag");
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(flag_zero_kernel, dim3(1), dim3(1), 0, st, flag);
    if (n > 0 && count > 0) {
        if (!a || !b) return set_error(SPHK_E_ARG, "equal_dev: null array list");
        EqualArrays ea{};
        for (int c = 0; c < count; c++) {
            if (!a[c] || !b[c]) return set_error(SPHK_E_ARG, "equal_dev: null array %d", c);
            ea.a[c] = reinterpret_cast<const uint64_t *>(a[c]);
            ea.b[c] = reinterpret_cast<const uint64_t *>(b[c]);
        }
        const dim3 grid(std::min(512, (n + kBlock - 1) / kBlock), count);
        hipLaunchKernelGGL(equal_kernel, grid, dim3(kBlock), 0, st, n, ea, flag);
    }
    SPHK_TRY(hipGetLastError());
    return SPHK_OK;
}

int sphk_copy_dev(void *dst, const void *src, size_t bytes, void *stream)
{
    if (bytes == 0) return SPHK_OK;
    if (!dst || !src) return set_error(SPHK_E_ARG, "copy_dev: null pointer");
    SPHK_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream));
    return SPHK_OK;
}

}  // extern "C"
