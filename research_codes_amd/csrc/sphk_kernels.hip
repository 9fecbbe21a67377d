// sphk_kernels.hip -- gfx950 kernels for the SPH interaction functors.
//
// Launch shape (all three kernels): one workgroup per walk, of one 64-lane
// wavefront (several where walks are few or long, see WaveRule).  A walk's
// i-particles are processed in chunks of <= 64.  Inside a
// chunk of ni particles the wave is split into S = floor(64/ni) j-slices:
// lane l holds i = l mod ni and slice l / ni (lanes beyond S*ni idle), so a
// walk of 5 particles keeps 60 of 64 lanes busy.  j-entries are staged
// through LDS in tiles of 64 records: lane k gathers entry k through j_idx
// (coalesced where the list is a run of consecutive particles) and the tile
// is padded with inert records, so the sweep k = slice, slice+S, ... < 64
// has no bounds checks.  Records are packed as double4 / R4 so a lane reads
// an entry with 128-bit LDS loads.  Per-i partials are combined across
// slices through LDS in a fixed order (bitwise reproducible).
//
// Precision.  Positions are FP64; every pair displacement is formed in FP64.
// MIXED=false evaluates the pair term in FP64; MIXED=true casts the
// displacement to FP32, evaluates the pair term in FP32, sums a tile's
// partials in FP32 and folds them into FP64 per-i totals.  The three
// smoothing-length passes of the density functor are FP64 in both modes.

#include "sphk_device.hpp"
#include "sphk_internal.hpp"

namespace sphk {

template <bool MIXED>
using real_t = typename std::conditional<MIXED, float, double>::type;

template <typename R>
struct alignas(4 * sizeof(R)) R4 {
    R a, b, c, d;
};

// Positions in the lists: offsets run up to 2^31 - 1, and a position past a
// list's end (the next tile's, another wave's) may lie beyond that, so the
// kernels form them unsigned.

// Inert padding record: far away (q >> 1 for any realistic H), zero mass,
// id -1, very negative sound speed (cannot raise vsmx).
constexpr double kFar = 1e10;

// Walk of a workgroup.  Workgroups of a launch are dispatched round-robin
// over the 8 XCDs (block b runs on XCD b mod 8), each XCD with its own L2.
// Walks are Morton-ordered, so neighbouring walks share most of their
// j-records.  Chunks of kXcdChunk consecutive walks are dealt to the XCDs in
// turn: an XCD works through whole chunks (its L2 serves the shared
// records) while every XCD still sees a mix of dense and sparse regions
// (one contiguous range per XCD measured 20% slower from load imbalance).
// Walks past the last whole round of chunks keep their own index.
constexpr int kXcd = 8;
constexpr int kXcdChunk = 64;
static_assert(kQueueInts == (kXcd + 1) * kQueueStride, "walk queue layout");

__device__ __forceinline__ int xcd_walk(int b, int n_walk)
{
    const int n_full = n_walk / (kXcd * kXcdChunk) * (kXcd * kXcdChunk);
    if (b >= n_full) return b;
    const int x = b % kXcd, k = b / kXcd;
    return ((k / kXcdChunk) * kXcd + x) * kXcdChunk + k % kXcdChunk;
}

// Walk scheduling.  Ordinary launch: one workgroup per walk (grid = n_walk),
// workgroup b takes walk xcd_walk(b).  Persistent launch (a grid sized to the
// resident capacity of the chip): every workgroup repeatedly claims the next
// virtual index v = x + 8 k of its own XCD x (counter k of that XCD's queue)
// and runs walk xcd_walk(v), so an XCD works through the same walks as in
// the ordinary launch; it stops at the first v >= n_walk.  The last
// workgroup to finish zeroes the queue for its next use.  Queue layout:
// kXcd claim counters and one exit counter, kQueueStride ints apart.
template <bool PERSIST, typename F>
__device__ __forceinline__ void run_walks(int n_walk, int *queue, F &&walk)
{
    if (!PERSIST) {
        if ((int)blockIdx.x < n_walk) walk(xcd_walk(blockIdx.x, n_walk), (int)(threadIdx.x % kWave));
        return;
    }
    const int x = (int)(blockIdx.x % kXcd);
    int *ctr = queue + x * kQueueStride;
    for (;;) {
        int k = 0;
        if (threadIdx.x == 0) k = atomicAdd(ctr, 1);
        const int v = x + kXcd * __shfl(k, 0, kWave);
        if (v >= n_walk) break;
        walk(xcd_walk(v, n_walk), (int)threadIdx.x);
        __syncthreads();   // LDS of this walk no longer read
    }
    if (threadIdx.x == 0) {
        __threadfence();
        if (atomicAdd(queue + kXcd * kQueueStride, 1) == (int)gridDim.x - 1) {
            for (int c = 0; c < kXcd; c++) atomicExch(queue + c * kQueueStride, 0);
            atomicExch(queue + kXcd * kQueueStride, 0);
        }
    }
}

// LDS written by a wave's lanes before, read by them after (one wave's LDS
// operations complete in order; this keeps the compiler to it).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Waves per walk of the three functors.  A launch of few walks leaves SIMDs
// idle at one wave per walk, and each walk's list is a serial chain of tiles;
// so NW waves of one workgroup take a walk's tiles in turn.  Hydro and
// gravity: every wave sums its tile in the pair type as a single wave would,
// and the tiles' sums are folded into FP64 in list order (wave q keeps
// quantities q, q + NW, ...).  Density: see there.  The results do not depend
// on NW, bit for bit, so the choice may follow the launch.  It costs a walk's
// set-up once per wave, two barriers per NW tiles and LDS, so it pays where
// the walks are few or long.  Their length is known to the caller only as the
// mean number m of i-particles (a walk of more of them has a longer list too);
// without it one wave is taken.  The lines lie where both sides measured
// equal, in us for walks (m):
//   gravity, FP64, softening per particle, NW = 1 / 4 / 8: 635 (4.7) 29 / 18 /
//     16, 1000 (3.0) 28 / 17 / 16, 2144 (9.3) 155 / 87 / 86, 3852 (2.6) 48 /
//     47, 4127 (17) 480 / 281 / 280, 7585 (5.3) 148 / 141, 13487 (5.2) 229 /
//     224, 15589 (9.6) 530 / 496, 35089 (8.5) 904 / 884, 51463 (19) 1463 /
//     1518; mixed alike (13487: 135 / 133); FP64, uniform: 6885 (2.9) 63 / 67,
//     13487 (5.2) 165 / 177, 15589 (9.6) 370 / 334, 44603 (18) 1888 / 1808
//   gravity, mixed, uniform softening (blocks of 256 records), NW = 1 / 2 / 4:
//     635 (4.7) 16 / 13 / 11, 1000 (3.0) 12.6 / 14.1 / 11.1, 1958 (5.1) 26 / 21 /
//     21, 4477 (4.5) 34 / 32 / 33, 4660 (8.6) 76 / 60 / 60, 7464 (20) 254 / 206 /
//     200, 13487 (5.2) 87 / 88, 15589 (9.6) 173 / 170, 51463 (19) 479 / 513
//   hydro, mixed, NW = 1 / 4: 635 (4.7) 18 / 21, 1007 (9.9) 33 / 23, 2144 (9.3)
//     45 / 36, 4660 (8.6) 60 / 57, 7464 (20) 197 / 180, 15691 (19) 310 / 325;
//     FP64 (twice the LDS), NW = 1 / 2 / 4: 1007 (9.9) 50 / 47 / 40, 2144
//     (9.3) 71 / 65 / 65, 4127 (17) 244 / 199 / 206, 4660 (8.6) 94 / 98, 7464
//     (20) 326 / 335
//   density, FP64, NW = 1 / 2: 1000 (3.0) 29 / 25, 3852 (2.6) 42 / 61, 4477
//     (4.5) 71 / 69, 7165 (9.8) 200 / 171, 7585 (5.3) 112 / 117, 15589 (9.6)
//     324 / 325, 15691 (19) 906 / 845, 35089 (8.5) 534 / 565; mixed alike; 4
//     waves were slower than 2
struct WaveLine {
    double k, m0;   // up to k (m - m0) walks of m i-particles on average
};
struct WaveRule {
    WaveLine w8, w4, w2;   // lines for 8, 4 and 2 waves per walk
};
constexpr WaveLine kNever{0., 0.};
constexpr WaveRule kGravRule{{200., 0.}, {2500., 1.5}, kNever}, kGravRelRule{kNever, {500., 2.}, {3000., 3.}};
constexpr WaveRule kHydroRule{kNever, {600., 5.}, kNever}, kHydroF64Rule{kNever, {250., 4.}, {450., 4.5}};
constexpr WaveRule kDensRule{kNever, kNever, {2000., 2.2}};

int waves_per_walk(int n_walk, int64_t n_i, const WaveRule &r)
{
    const auto within = [&](const WaveLine &l) { return n_walk <= l.k * ((double)n_i / n_walk - l.m0); };
    return n_i <= 0 ? 1 : within(r.w8) ? 8 : within(r.w4) ? 4 : within(r.w2) ? 2 : 1;
}

// Lane map of one i-chunk: S = floor(64/ni) slices.
struct Map {
    int ni, S, il, slice;
    bool lead;  // slice 0 of a real i: owns the reduced result
    __device__ __forceinline__ Map(int ni_, int lane)
    {
        ni = ni_;
        S = kWave / ni;
        il = lane % ni;
        slice = lane / ni;
        if (slice >= S) slice = kTile;  // idle lane: its sweep is empty
        lead = lane < ni;
    }
};

// Sum (or max) of per-lane values over the slices of each i, through LDS.
// On return the lead lane of each i holds the result.  red has 64*NQ slots.
template <int NQ>
__device__ __forceinline__ void slice_reduce(double (&v)[NQ], double *red, const Map &m, int lane,
                                             int max_mask = 0)
{
    __syncthreads();
    for (int q = 0; q < NQ; q++) red[q * kWave + lane] = v[q];
    __syncthreads();
    if (m.lead) {
        for (int q = 0; q < NQ; q++) {
            double a = red[q * kWave + m.il];
            const bool is_max = (max_mask >> q) & 1;
            for (int t = 1; t < m.S; t++) {
                const double b = red[q * kWave + m.il + m.ni * t];
                a = is_max ? (a > b ? a : b) : a + b;
            }
            v[q] = a;
        }
    }
}

// ---------------------------------------------------------------------------
// Density: scalar calcDensity, sph_yamauchi/run/hdr_density.hpp:254-363.
// ---------------------------------------------------------------------------

// q = sqrt(r2) * hinv with the reference's FP64 rounding sequence (separate
// IEEE operations, correctly rounded sqrt): decides q < 1 for pairs within a
// few ulps of the kernel edge.
__device__ __attribute__((noinline)) double exact_q(double dx, double dy, double dz, double hinv)
{
#pragma clang fp contract(off)
    const double r2 = dx * dx + dy * dy + dz * dz;
    return __builtin_sqrt(r2) * hinv;
}

// r = sqrt(r2) with the reference's FP64 rounding sequence: q = r * (1/H)
// is then the reference's q bit for bit.
__device__ __forceinline__ double exact_r(double dx, double dy, double dz)
{
#pragma clang fp contract(off)
    const double r2 = dx * dx + dy * dy + dz * dz;
    return sqrt_ieee(r2);
}

struct Pass1 {
    double rh;
    int nj;
};

__device__ __forceinline__ void dens_pass1_pair(const double4 &j, double px, double py, double pz,
                                                double hi, double hi3, Pass1 &a)
{
    const double dx = px - j.x;
    const double dy = py - j.y;
    const double dz = pz - j.z;
    const double r2 = dx * dx + dy * dy + dz * dz;
    double q = r2 * rsqrt_f64(r2 > 1e-300 ? r2 : 1e-300) * hi;
    if (__builtin_fabs(q - 1.) < 1e-13) q = exact_q(dx, dy, dz, hi);
    a.rh += j.w * hi3 * kernel0th(q);
    a.nj += (q < 1.) ? 1 : 0;
}

template <typename R>
struct Pass2 {
    R g, dv, rx, ry, rz;
};

// The id of a j-record travels in the fourth slot of its velocity record:
// bit pattern in FP32, exact value in FP64.
__device__ __forceinline__ float pack_id(int32_t id, float) { return __int_as_float(id); }
__device__ __forceinline__ double pack_id(int32_t id, double) { return (double)id; }
__device__ __forceinline__ int32_t unpack_id(float v) { return __float_as_int(v); }
__device__ __forceinline__ int32_t unpack_id(double v) { return (int32_t)v; }

template <typename R>
__device__ __forceinline__ void dens_pass2_pair(const double4 &j, const R4<R> &v, double px, double py,
                                                double pz, R vx, R vy, R vz, int32_t id_i, R hi, R hi4,
                                                Pass2<R> &a)
{
    const R dpx = (R)(px - j.x);
    const R dpy = (R)(py - j.y);
    const R dpz = (R)(pz - j.z);
    const R dvx = vx - v.a;
    const R dvy = vy - v.b;
    const R dvz = vz - v.c;
    const R r2 = dpx * dpx + dpy * dpy + dpz * dpz;
    const R ri = (id_i != unpack_id(v.d)) ? rsqrt_r(r2) : R(0);
    const R q = r2 * ri * hi;
    // with t = (1-q)_+: W' = -5 C1 q t^3, 3W + qW' = C0 t^3 (3 + 9q - 32q^2),
    // and W'(q) / r = -5 C1 h t^3 (the self entry has d = 0: no div/curl term)
    R t = R(1) - q;
    t = t > R(0) ? t : R(0);
    const R t3 = t * t * t;
    const R mh = (R)j.w * hi4;
    a.g -= R(kCeff0) * t3 * (R(3) + q * (R(9) - R(32) * q)) * mh;
    const R dw = R(-5. * kCeff1) * mh * hi * t3;
    const R dwx = dw * dpx, dwy = dw * dpy, dwz = dw * dpz;
    a.dv -= dvx * dwx + dvy * dwy + dvz * dwz;
    a.rx += dvy * dwz - dvz * dwy;
    a.ry += dvz * dwx - dvx * dwz;
    a.rz += dvx * dwy - dvy * dwx;
}

// hdr_density.hpp:351-362: Omega^-1, div v and |rot v| from the grad-h sums.
__device__ __forceinline__ void dens_finish(const sphk_dens_out &out, int i, const double (&acc)[5],
                                            double dens, long long np, double hs, double rs)
{
    const double grdh = acc[0];
    double divv = acc[1];
    const double rot2 = acc[2] * acc[2] + acc[3] * acc[3] + acc[4] * acc[4];
    const double deni = 1. / dens;
    const double omgi = 1. / (1. + hs * deni * grdh / 3.);
    double rotv = rot2 != 0. ? __builtin_sqrt(rot2) : 0.;
    rotv *= deni * omgi;
    divv *= deni * omgi;
    out.dens[i] = dens;
    out.np[i] = np;
    out.ksr[i] = hs;
    out.itr[i] = (hs > rs) ? 1 : 0;
    out.divv[i] = divv;
    out.rotv[i] = rotv;
    out.grdh[i] = omgi;
}

// New H from rho: hdr_density.hpp:296-300 (eta * kappa * (m / rho)^(1/3), capped).
__device__ __forceinline__ double dens_next_h(double eta_ksrh, double m, double dens, double hmax)
{
    const double h = eta_ksrh * cbrt_f64(m / dens);
    return h < hmax ? h : hmax;
}

// Walks whose j-list holds at most kDensCap records keep the whole list in
// LDS for the four sweeps (three h-passes, grad-h pass); longer lists stream
// 64-record tiles.
//
// Resident lists are compacted per i-particle.  One FP64 sweep marks the
// records within R_i = max(rs_i, H_0,i) (times 1 + 1e-12) of i; every record
// outside contributes exactly zero to all four sweeps as long as H_k <= R_i,
// so the sweeps visit only the marked records (positions in LDS, one byte
// each).  The i-particles whose lists fit in kDensComp entries are taken
// together; the lanes are shared out so that every taken i needs at most
// T = ceil(C / (64 - n)) steps (C entries over n particles).  If an H_k of
// the iteration exceeds R_i the chunk continues with full sweeps.
//
// NW = 2: two waves per walk share the staging, the marking (a tile each in
// turn) and the h-passes (step or tile t belongs to wave t mod 2);
// per-particle work is wave 0's, and so is the mixed grad-h pass, whose FP32
// sums depend on their order.  FP64 sums that the waves share are formed by
// parity, the even steps (tiles) in order and the odd ones, and added, whatever
// NW is: results do not depend on it, bit for bit.
constexpr int kDensCap = 256;        // largest resident capacity (instantiated: 192, 256)
constexpr int kDensComp = 1728;
constexpr int kDensR = 12;           // members per lane held in registers for the h-passes
static_assert(kDensCap <= 256, "compacted positions are stored as bytes");

template <bool MIXED>
__device__ __forceinline__ void dens_stage(int e, int t0_abs, int nj_end, const int32_t *__restrict__ j_idx,
                                           const sphk_dens_src &pj, double4 *sp, R4<real_t<MIXED>> *sv,
                                           bool with_v)
{
    using R = real_t<MIXED>;
    const uint32_t k = (uint32_t)t0_abs + (uint32_t)e;
    if (k < (uint32_t)nj_end) {
        const int j = j_idx ? j_idx[k] : (int)k;
        sp[e] = make_double4(pj.x[j], pj.y[j], pj.z[j], pj.m[j]);
        if (with_v) sv[e] = R4<R>{(R)pj.vx[j], (R)pj.vy[j], (R)pj.vz[j], pack_id(pj.id[j], R(0))};
    } else {
        sp[e] = make_double4(kFar, kFar, kFar, 0.);
        if (with_v) sv[e] = R4<R>{R(0), R(0), R(0), pack_id(-1, R(0))};
    }
}

// The i-particle data one lane works with.
struct DensI {
    double x, y, z, m, ksr, rs, vx, vy, vz;
    int32_t id;
};

__device__ __forceinline__ DensI dens_load_i(const sphk_dens_src &pi, int i)
{
    return DensI{pi.x[i], pi.y[i], pi.z[i], pi.m[i], pi.ksr[i], pi.rs[i], pi.vx[i], pi.vy[i], pi.vz[i],
                 pi.id[i]};
}

// The parities that one of NW waves sums: kPar of them, wave wv's u-th is
// wv + u.
template <int NW>
constexpr int kPar = 2 / NW;

// Combination of the waves' values of one lane, kWave apart.
template <int NW>
__device__ __forceinline__ double wave_comb(const double *r)
{
    if constexpr (NW == 1) return r[0];
    return r[0] + r[kWave];
}

// An h-pass's sums and neighbour counts of the waves over lanes first, first +
// step, ... (cnt of them), in one loop: it is bound by the latency of its LDS
// reads (1.46 -> 1.44 ms mixed, 1.60 -> 1.54 FP64 at 10^6 particles against a
// loop each).
template <int NW>
__device__ __forceinline__ void lanes_pass(const double *r, const int *rn, int first, int cnt, int step, double &sum,
                                           long long &n)
{
    double s = wave_comb<NW>(r + first);
    int c = rn[first] + (NW == 2 ? rn[kWave + first] : 0);
#pragma unroll 4
    for (int t = 1; t < cnt; t++) {
        const int l = first + t * step;
        s += wave_comb<NW>(r + l);
        c += rn[l] + (NW == 2 ? rn[kWave + l] : 0);
    }
    sum = s;
    n = c;
}

// Per-particle sums of five quantities over the lanes of each particle; valid where `owner`.  ALL: both waves hold
// parts of them; else wave 0 alone.
template <int NW, bool ALL>
__device__ __forceinline__ void dens_sum5(const double (&part)[5], double (&acc)[5], double *red, int wv, int lane,
                                          bool owner, int cnt, int step)
{
    constexpr int kN = ALL ? NW : 1;
#pragma unroll
    for (int q0 = 0; q0 < 5; q0 += 2) {
        const bool two = q0 + 1 < 5;
        __syncthreads();
        if (ALL || wv == 0) {
            red[wv * kWave + lane] = part[q0];
            if (two) red[(NW + wv) * kWave + lane] = part[q0 + 1];
        }
        __syncthreads();
        if (owner) {
            const double *r = red + lane, *r2 = red + NW * kWave + lane;
            double a = wave_comb<kN>(r), b = two ? wave_comb<kN>(r2) : 0.;
#pragma unroll 4
            for (int t = 1; t < cnt; t++) {
                a += wave_comb<kN>(r + t * step);
                if (two) b += wave_comb<kN>(r2 + t * step);
            }
            acc[q0] = a;
            if (two) acc[q0 + 1] = b;
        }
    }
}

// Lists longer than kDensCap: every sweep streams the list through 64-record
// LDS tiles, one per wave.
template <bool MIXED, int NW>
__device__ void density_streaming(int lane, int wv, const Map &M, int i, int jb, int je,
                                  const int32_t *__restrict__ j_idx, const sphk_dens_src &pi,
                                  const sphk_dens_src &pj, const sphk_dens_out &out, double eta_ksrh,
                                  double hmax, double4 *sp, R4<real_t<MIXED>> *sv, double *red,
                                  double *shs)
{
    using R = real_t<MIXED>;
    const int ntile = (int)(((uint32_t)(je - jb) + kTile - 1) / kTile);
    const DensI I = dens_load_i(pi, i);
    const bool owner = M.lead && wv == 0;
    int *redn = reinterpret_cast<int *>(red + NW * kWave);
    double hs = I.ksr;
    double dens = 0.;
    long long np = 0;
    double4 *const tp = sp + wv * kTile;
    R4<R> *const tv = sv + wv * kTile;

    for (int rep = 0; rep < 3; rep++) {
        const double hi = 1. / hs;
        const double hi3 = hi * hi * hi;
        double sum = 0.;
        int nq = 0;
#pragma unroll
        for (int u = 0; u < kPar<NW>; u++) {
            double P = 0.;
            for (int t = wv + u; t < ntile; t += 2) {
                wave_sync();
                dens_stage<MIXED>(lane, jb + t * kTile, je, j_idx, pj, tp, tv, false);
                wave_sync();
                Pass1 a{0., 0};
                const int nt = min(kTile, je - jb - t * kTile);   // records of this tile
                int k = M.slice;
                for (; k + 3 * M.S < nt; k += 4 * M.S) {
                    const double4 j0 = tp[k], j1 = tp[k + M.S], j2 = tp[k + 2 * M.S], j3 = tp[k + 3 * M.S];
                    dens_pass1_pair(j0, I.x, I.y, I.z, hi, hi3, a);
                    dens_pass1_pair(j1, I.x, I.y, I.z, hi, hi3, a);
                    dens_pass1_pair(j2, I.x, I.y, I.z, hi, hi3, a);
                    dens_pass1_pair(j3, I.x, I.y, I.z, hi, hi3, a);
                }
                for (; k < nt; k += M.S) dens_pass1_pair(tp[k], I.x, I.y, I.z, hi, hi3, a);
                P += a.rh;
                nq += a.nj;
            }
            sum = u == 0 ? P : sum + P;
        }
        __syncthreads();
        red[wv * kWave + lane] = sum;
        redn[wv * kWave + lane] = nq;
        __syncthreads();
        if (owner) {
            lanes_pass<NW>(red, redn, M.il, M.S, M.ni, dens, np);
            shs[M.il] = dens_next_h(eta_ksrh, I.m, dens, hmax);
        }
        __syncthreads();
        hs = shs[M.il];
    }

    const double hi_d = 1. / hs;
    const R hi = (R)hi_d;
    const R hi4 = (R)(hi_d * (hi_d * hi_d * hi_d));
    const R vx = (R)I.vx, vy = (R)I.vy, vz = (R)I.vz;
    double part[5];
#pragma unroll
    for (int u = 0; u < kPar<NW>; u++) {
        double P[5] = {0., 0., 0., 0., 0.};
        for (int t = wv + u; t < ntile; t += 2) {
            wave_sync();
            dens_stage<MIXED>(lane, jb + t * kTile, je, j_idx, pj, tp, tv, true);
            wave_sync();
            Pass2<R> a{R(0), R(0), R(0), R(0), R(0)};
            const int nt = min(kTile, je - jb - t * kTile);
            int k = M.slice;
            for (; k + M.S < nt; k += 2 * M.S) {
                dens_pass2_pair<R>(tp[k], tv[k], I.x, I.y, I.z, vx, vy, vz, I.id, hi, hi4, a);
                dens_pass2_pair<R>(tp[k + M.S], tv[k + M.S], I.x, I.y, I.z, vx, vy, vz, I.id, hi, hi4, a);
            }
            for (; k < nt; k += M.S)
                dens_pass2_pair<R>(tp[k], tv[k], I.x, I.y, I.z, vx, vy, vz, I.id, hi, hi4, a);
            P[0] += (double)a.g;
            P[1] += (double)a.dv;
            P[2] += (double)a.rx;
            P[3] += (double)a.ry;
            P[4] += (double)a.rz;
        }
#pragma unroll
        for (int q = 0; q < 5; q++) part[q] = u == 0 ? P[q] : part[q] + P[q];
    }
    double acc[5];
    dens_sum5<NW, true>(part, acc, red, wv, lane, owner, M.S, M.ni);
    if (owner) dens_finish(out, i, acc, dens, np, hs, I.rs);
}

// Launch bound: OCC waves per SIMD, 3 for launches that fill the chip (at most
// 168 VGPRs; a few spill).  Between its sweeps the kernel is bound by latency,
// so scans go through DPP, lane sums run in one loop for all quantities, and
// distances take sqrt_ieee: 10^6 particles, one wave per walk, 1.38 -> 1.30 ms
// mixed and 1.67 -> 1.44 FP64 (there also 20 instead of 22 KB of LDS: 8 walks
// per CU).
// Mixed launches of few walks with a wave each wait for their longest walks,
// in which each spilled register is reloaded, and have no use for a third
// wave: OCC 2 (197 VGPRs, none spills).  Persistent mixed launches, whose loop
// over walks costs registers, take it always.  In us with 3 / 2, capacity 256
// (192), walks (particles on average): 572 (17) 213 / 198 (212 / 198), 1797
// (2.8) 53 / 46 (52 / 46), 3980 (5.0) 71 / 65 (70 / 66), 5385 (19) 998 / 921
// (987 / 935), 7358 (2.7) 83 / 76 (77 / 77), 10952 (9.1) 277 / 260 (274 / 264),
// 14449 (2.8) 106 / 110 (99 / 112), 42605 (9.4) 567 / 571 (546 / 614).  Where the
// mean is known, 8000 walks of more particles have two waves each; where it is
// not, walks may be long, and the line lies further out.  FP64 at capacity
// 256 is held to 2 waves by its LDS.
constexpr int kDensFew = 8192, kDensFewUnknown = 12288;

template <bool MIXED, int CAP, bool PERSIST, int NW, int OCC>
__global__ __launch_bounds__(kWave *NW, OCC) void density_kernel(
    int n_walk, const int32_t *__restrict__ i_off, const int32_t *__restrict__ j_off,
    const int32_t *__restrict__ j_idx, sphk_dens_src pi, sphk_dens_src pj, sphk_dens_out out,
    double eta_ksrh, double hmax, int *queue)
{
    using R = real_t<MIXED>;
    static_assert(CAP % kTile == 0 && CAP <= kDensCap && CAP >= NW * kTile, "list capacity");
    static_assert(!PERSIST || NW == 1, "persistent launches take one wave per walk");
    constexpr int kWords = CAP / kTile, kMine = (kWords + NW - 1) / NW;   // tiles, and those a wave marks
    constexpr int kDensPad = CAP;   // inert record after the list, target of idle steps
    constexpr int kRegs = kDensR / NW;
    static_assert((NW == 1 || NW == 2) && kDensR % 2 == 0, "steps are dealt to the waves by parity");
    __shared__ double4 sp[CAP + 1];     // x, y, z, m
    __shared__ R4<R> sv[CAP + 1];       // vx, vy, vz, id
    __shared__ uint8_t cidx[kDensComp];
    __shared__ double red[2 * NW * kWave];
    __shared__ double shs[kWave];
    __shared__ int s_own[kWave];
    __shared__ uint16_t s_ci[kWave], s_coff[kWave];
    int *const redn = reinterpret_cast<int *>(red + NW * kWave);
    uint8_t *const s_cnt = reinterpret_cast<uint8_t *>(red);   // membership counts [lane][tile], before any reduction
    const int wv = NW > 1 ? (int)threadIdx.x / kWave : 0;

    auto walk = [&](const int w, const int lane) {
        const int ib = i_off[w], ie = i_off[w + 1];
        const int jb = j_off[w], je = j_off[w + 1];
        const int nj = je - jb;
        const int ntile = (int)(((uint32_t)nj + kTile - 1) / kTile);

        if (nj > CAP) {
            for (int c0 = ib; c0 < ie; c0 += kWave) {
                const Map M(min(kWave, ie - c0), lane);
                density_streaming<MIXED, NW>(lane, wv, M, c0 + M.il, jb, je, j_idx, pi, pj, out, eta_ksrh, hmax,
                                             sp, sv, red, shs);
            }
            return;
        }

        // one burst: every record of the list, padded to whole tiles, plus the inert record
        for (int e = wv * kWave + lane; e < ntile * kTile; e += kWave * NW)
            dens_stage<MIXED>(e, jb, je, j_idx, pj, sp, sv, true);
        if (lane == 0 && wv == 0) dens_stage<MIXED>(kDensPad, 0, 0, j_idx, pj, sp, sv, true);

        for (int c0 = ib; c0 < ie;) {
            const Map M(min(kWave, ie - c0), lane);
            __syncthreads();   // staging done; LDS of the previous chunk no longer read

            // -- membership sweep: lane (i, slice) marks its records within R_i, tile by tile
            uint64_t wd[kMine];
            {
                const int i = c0 + M.il;
                const double px = pi.x[i], py = pi.y[i], pz = pi.z[i];
                const double h0 = pi.ksr[i], rs = pi.rs[i];
                const double rme = (h0 > rs ? h0 : rs) * (1. + 1e-12);
                const double rm2 = rme * rme;
#pragma unroll
                for (int u = 0; u < kMine; u++) {
                    const int t = wv + NW * u;
                    uint64_t b = 0;
                    if (t < ntile) {
                        const double4 *tp = sp + t * kTile;
                        const int nt = min(kTile, nj - t * kTile);
                        int k = M.slice;
                        for (; k + 3 * M.S < nt; k += 4 * M.S) {
                            const double4 j0 = tp[k], j1 = tp[k + M.S], j2 = tp[k + 2 * M.S], j3 = tp[k + 3 * M.S];
                            const double x0 = px - j0.x, y0 = py - j0.y, z0 = pz - j0.z;
                            const double x1 = px - j1.x, y1 = py - j1.y, z1 = pz - j1.z;
                            const double x2 = px - j2.x, y2 = py - j2.y, z2 = pz - j2.z;
                            const double x3 = px - j3.x, y3 = py - j3.y, z3 = pz - j3.z;
                            b |= (uint64_t)(x0 * x0 + y0 * y0 + z0 * z0 < rm2) << k;
                            b |= (uint64_t)(x1 * x1 + y1 * y1 + z1 * z1 < rm2) << (k + M.S);
                            b |= (uint64_t)(x2 * x2 + y2 * y2 + z2 * z2 < rm2) << (k + 2 * M.S);
                            b |= (uint64_t)(x3 * x3 + y3 * y3 + z3 * z3 < rm2) << (k + 3 * M.S);
                        }
                        for (; k < nt; k += M.S) {
                            const double dx = px - tp[k].x, dy = py - tp[k].y, dz = pz - tp[k].z;
                            b |= (uint64_t)(dx * dx + dy * dy + dz * dz < rm2) << k;
                        }
                    }
                    wd[u] = b;
                    if (t < 4) s_cnt[4 * lane + t] = (uint8_t)__popcll(b);
                }
                if (kWords < 4 && wv == 0) s_cnt[4 * lane + 3] = 0;
            }
            __syncthreads();
            // entries of a lane over its tiles (at most 256: four bytes summed)
            auto lane_cnt = [&](int l) {
                return (int)__builtin_amdgcn_sad_u8(reinterpret_cast<const uint32_t *>(s_cnt)[l], 0u, 0u);
            };
            int start = 0, ci = 0;
#pragma unroll 4
            for (int s2 = 0; s2 < M.S; s2++) {
                const int c = lane_cnt(M.il + M.ni * s2);
                start += s2 < M.slice ? c : 0;
                ci += c;
            }
            ci = M.lead ? ci : 0;
            const uint32_t own_cnt = reinterpret_cast<const uint32_t *>(s_cnt)[lane];
            // take the leading i-particles whose lists fit in kDensComp entries
            // (every single list fits: c_i <= kDensCap)
            const int incl = wave_scan_incl(ci);   // leads are lanes 0 .. ni-1
            const bool fits = M.lead && incl <= kDensComp;
            const int n_take = __popcll(__ballot(fits));
            const int total = __builtin_amdgcn_readlane(incl, n_take - 1);
            const bool take = M.il < n_take;             // lane works on a taken i

            if (wv == 0) {
                if (M.lead && take) {
                    s_coff[M.il] = (uint16_t)(incl - ci);
                    s_ci[M.il] = (uint16_t)ci;
                }
                s_own[lane] = -1;
            }
            __syncthreads();
            if (take && M.slice < M.S) {
                const int o0 = s_coff[M.il] + start;
#pragma unroll
                for (int u = 0; u < kMine; u++) {
                    const int t = wv + NW * u;
                    uint64_t b = t < kWords ? wd[u] : 0;
                    // entries of the lane's tiles before t
                    int o = o0 + (t == 0 ? 0 : (int)__builtin_amdgcn_sad_u8(own_cnt << (8 * (4 - min(t, 4))), 0u, 0u));
                    while (b) {
                        cidx[o++] = (uint8_t)(t * kTile + __builtin_ctzll(b));
                        b &= b - 1;
                    }
                }
            }
            // lanes per taken i: max(1, ceil(c_i / T)), T = ceil(C / (64 - n)); they sum to <= 64
            const int tsteps = n_take < kWave ? max(1, (total + (kWave - n_take) - 1) / (kWave - n_take)) : 1;
            const int si = (M.lead && take) ? (n_take < kWave ? max(1, (ci + tsteps - 1) / tsteps) : 1) : 0;
            const int lincl = wave_scan_incl(si);
            if (si > 0 && wv == 0)
                for (int s2 = 0; s2 < si; s2++) s_own[lincl - si + s2] = M.il | (s2 << 8) | (si << 16);
            __syncthreads();
            const int own = s_own[lane];

            // lane's particle and compacted range (the same in every wave);
            // every lane runs the wave's largest step count, idle steps read
            // the inert record
            int my = own >= 0 ? (own & 0xff) : 0;
            int e0 = 0, n_e = 0, stride = 1;
            const uint8_t *myidx = cidx;
            if (own >= 0) {
                e0 = (own >> 8) & 0xff;
                stride = own >> 16;
                n_e = s_ci[my];
                myidx = cidx + s_coff[my];
            }
            const int nsteps = wave_max(n_e > e0 ? (n_e - e0 + stride - 1) / stride : 0);
            bool compact = true;
            bool owner = own >= 0 && e0 == 0 && wv == 0;
            DensI I = dens_load_i(pi, c0 + my);
            const Map MF(n_take, lane);   // full sweeps over the taken i-particles
            double hs = I.ksr;
            double dens = 0.;
            long long np = 0;

            // After a pass's sums (in red, redn): rho, n and the next H of the
            // owners; with an H beyond R_i the compacted lists are incomplete:
            // full sweeps from the next pass on, wave 0's lead lanes of MF take
            // over ownership.
            auto pass_end = [&]() {
                int viol = 0;
                if (owner) {
                    const int first = compact ? lane : MF.il, cnt = compact ? stride : MF.S, step = compact ? 1 : MF.ni;
                    lanes_pass<NW>(red, redn, first, cnt, step, dens, np);
                    const double hnew = dens_next_h(eta_ksrh, I.m, dens, hmax);
                    shs[my] = hnew;
                    viol = compact && hnew > (I.ksr > I.rs ? I.ksr : I.rs);
                }
                if (__syncthreads_or(viol)) {
                    if (owner) {
                        red[my] = dens;
                        red[kWave + my] = (double)np;
                    }
                    __syncthreads();
                    compact = false;
                    my = MF.il;
                    owner = MF.lead && wv == 0;
                    I = dens_load_i(pi, c0 + my);
                    dens = red[my];
                    np = (long long)red[kWave + my];
                }
                hs = shs[my];
            };
            auto pass_put = [&](double sum, int nq) {
                __syncthreads();
                red[wv * kWave + lane] = sum;
                redn[wv * kWave + lane] = nq;
                __syncthreads();
            };

            // -- three fixed-point passes: rho(H_k), n(H_k), H_{k+1} (hdr_density.hpp:264-302).
            // When every lane has at most kDensR members, their exact distances
            // and masses are held in registers for the passes (one sqrt per
            // member instead of one rsqrt refinement per member and pass); the
            // passes that remain after an H beyond R_i run below.
            int rep0 = 0;
            if (nsteps <= kDensR) {
                double rr[kRegs], mm[kRegs];
#pragma unroll
                for (int u = 0; u < kRegs; u++) {
                    const int t = wv + NW * u;
                    if (t < nsteps) {
                        const int e = e0 + t * stride;
                        const double4 j = sp[e < n_e ? myidx[e] : kDensPad];
                        rr[u] = exact_r(I.x - j.x, I.y - j.y, I.z - j.z);
                        mm[u] = j.w;
                    }
                }
                for (; rep0 < 3 && compact; rep0++) {
                    const double hi = 1. / hs;
                    const double hi3 = hi * hi * hi;
                    double sum = 0.;
                    int nq = 0;
#pragma unroll
                    for (int v = 0; v < kPar<NW>; v++) {
                        double P = 0.;
#pragma unroll
                        for (int u = v; u < kRegs; u += kPar<NW>) {
                            if (wv + NW * u < nsteps) {
                                const double q = rr[u] * hi;
                                P += mm[u] * hi3 * kernel0th(q);
                                nq += (q < 1.) ? 1 : 0;
                            }
                        }
                        sum = v == 0 ? P : sum + P;
                    }
                    pass_put(sum, nq);
                    pass_end();
                }
            }
            for (int rep = rep0; rep < 3; rep++) {
                const double hi = 1. / hs;
                const double hi3 = hi * hi * hi;
                Pass1 a[kPar<NW>] = {};
                if (compact) {
                    // four members in flight, of both parities where the wave has both
                    for (int t0 = 0; t0 < nsteps; t0 += 4 * NW) {
                        double4 j[4];
#pragma unroll
                        for (int m = 0; m < 4; m++) {
                            const int e = e0 + (t0 + wv + m * NW) * stride;
                            j[m] = sp[e < n_e ? myidx[e] : kDensPad];
                        }
#pragma unroll
                        for (int m = 0; m < 4; m++)
                            if (t0 + m * NW < nsteps)
                                dens_pass1_pair(j[m], I.x, I.y, I.z, hi, hi3, a[m % kPar<NW>]);
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < kPar<NW>; u++)
                        for (int t = wv + u; t < ntile; t += 2) {
                            const double4 *tp = sp + t * kTile;
                            const int nt = min(kTile, nj - t * kTile);
                            for (int k = MF.slice; k < nt; k += MF.S)
                                dens_pass1_pair(tp[k], I.x, I.y, I.z, hi, hi3, a[u]);
                        }
                }
                const double sum = NW == 1 ? a[0].rh + a[kPar<NW> - 1].rh : a[0].rh;
                const int nq = NW == 1 ? a[0].nj + a[kPar<NW> - 1].nj : a[0].nj;
                pass_put(sum, nq);
                pass_end();
            }

            // -- grad-h, divergence, curl with H_3 (hdr_density.hpp:304-349)
            const double hi_d = 1. / hs;
            const R hi = (R)hi_d;
            const R hi4 = (R)(hi_d * (hi_d * hi_d * hi_d));
            const R vx = (R)I.vx, vy = (R)I.vy, vz = (R)I.vz;
            double part[5] = {0., 0., 0., 0., 0.}, acc[5];
            auto pair2 = [&](int e, Pass2<R> &a) {
                const int k = e < n_e ? myidx[e] : kDensPad;
                dens_pass2_pair<R>(sp[k], sv[k], I.x, I.y, I.z, vx, vy, vz, I.id, hi, hi4, a);
            };
            auto add2 = [&](double (&p)[5], const Pass2<R> &a) {
                p[0] += (double)a.g;
                p[1] += (double)a.dv;
                p[2] += (double)a.rx;
                p[3] += (double)a.ry;
                p[4] += (double)a.rz;
            };
            if (compact && MIXED) {
                // pair terms summed in FP32 over at most 16 entries, then folded
                // into FP64 (as the full sweep folds each 64-record tile)
                if (wv == 0) {
                    Pass2<R> a{R(0), R(0), R(0), R(0), R(0)};
                    int st = 0, e = e0;
                    for (; st + 2 <= nsteps; st += 2, e += 2 * stride) {
                        pair2(e, a);
                        pair2(e + stride, a);
                        if ((st & 14) == 14) {
                            add2(part, a);
                            a = Pass2<R>{R(0), R(0), R(0), R(0), R(0)};
                        }
                    }
                    if (st < nsteps) pair2(e, a);
                    add2(part, a);
                }
                dens_sum5<NW, false>(part, acc, red, wv, lane, owner, stride, 1);
            } else {
#pragma unroll
                for (int u = 0; u < kPar<NW>; u++) {
                    double P[5] = {0., 0., 0., 0., 0.};
                    Pass2<R> a{R(0), R(0), R(0), R(0), R(0)};
                    if (compact) {
                        for (int t = wv + u; t < nsteps; t += 2) pair2(e0 + t * stride, a);
                        add2(P, a);
                    } else {
                        for (int t = wv + u; t < ntile; t += 2) {
                            const double4 *tp = sp + t * kTile;
                            const R4<R> *tv = sv + t * kTile;
                            const int nt = min(kTile, nj - t * kTile);   // records of this tile
                            a = Pass2<R>{R(0), R(0), R(0), R(0), R(0)};
                            int k = MF.slice;
                            for (; k + MF.S < nt; k += 2 * MF.S) {
                                dens_pass2_pair<R>(tp[k], tv[k], I.x, I.y, I.z, vx, vy, vz, I.id, hi, hi4, a);
                                dens_pass2_pair<R>(tp[k + MF.S], tv[k + MF.S], I.x, I.y, I.z, vx, vy, vz, I.id, hi,
                                                   hi4, a);
                            }
                            for (; k < nt; k += MF.S)
                                dens_pass2_pair<R>(tp[k], tv[k], I.x, I.y, I.z, vx, vy, vz, I.id, hi, hi4, a);
                            add2(P, a);
                        }
                    }
#pragma unroll
                    for (int q = 0; q < 5; q++) part[q] = u == 0 ? P[q] : part[q] + P[q];
                }
                dens_sum5<NW, true>(part, acc, red, wv, lane, owner, compact ? stride : MF.S, compact ? 1 : MF.ni);
            }
            if (owner) dens_finish(out, c0 + my, acc, dens, np, hs, I.rs);
            c0 += n_take;
        }
    };
    run_walks<PERSIST>(n_walk, queue, walk);
}

// ---------------------------------------------------------------------------
// Hydro: scalar calcHydro, sph_yamauchi/run/hdr_hydro.hpp:320-421.
// ---------------------------------------------------------------------------
// Position record of a hydro j-entry: FP64 absolute in the FP64 path; in the
// mixed path FP32 offsets from the walk's first particle, formed in FP64 (as
// for gravity: 16-byte records, no FP64 arithmetic per pair).
template <typename R>
struct HPos;
template <>
struct HPos<double> {
    using rec = double4;
};
template <>
struct HPos<float> {
    using rec = float4;
};

template <typename R>
struct HydroI {
    double px, py, pz;   // FP64 path: absolute; mixed path: offsets (in the FP32 range)
    R vx, vy, vz, hi, h5, pp, pc, bs, dn, cs, al, au, eg, et;
    int32_t id;
};

template <typename R>
struct HydroAcc {
    R ax, ay, az, ud, df, gx, gy, gz, vs;
};

template <typename R>
__device__ __forceinline__ void hydro_pair(const typename HPos<R>::rec &p, const R4<R> &A, const R4<R> &B,
                                           const R4<R> &Cc, R eh_j, R h5_j, int32_t jid,
                                           const HydroI<R> &I, HydroAcc<R> &a)
{
    // p = {x, y, z, -5 C1 m}; A = {vx, vy, vz, hinv}; B = {pres, presc, bswt, dens};
    // Cc = {vsnd, alph, alphu, thrm}; eh_j = eta_j h_j^5, h5_j = h_j^5 (formed
    // per record when it is staged)
    const R dpx = (R)I.px - (R)p.x;
    const R dpy = (R)I.py - (R)p.y;
    const R dpz = (R)I.pz - (R)p.z;
    const R dvx = I.vx - A.a;
    const R dvy = I.vy - A.b;
    const R dvz = I.vz - A.c;
    const R r2 = dpx * dpx + dpy * dpy + dpz * dpz;
    const bool other = I.id != jid;
    const R ri = other ? rsqrt_r(r2) : R(0);
    const R r1 = r2 * ri;
    const R hj = A.d;
    const R q_i = r1 * I.hi;
    const R q_j = r1 * hj;
    // W'(q) = -5 C1 q (1-q)_+^3, so dW_k / r = h_k^4 W'(r h_k) / r = -5 C1 F_k
    // with F_k = h_k^5 (1 - q_k)_+^3: ka/r and the eta term need no kernel
    // evaluation beyond F (the self entry contributes nothing, as ri = 0
    // makes it in the reference's form)
    R ti = R(1) - q_i, tj = R(1) - q_j;
    ti = ti > R(0) ? ti : R(0);
    tj = tj > R(0) ? tj : R(0);
    const R tj3 = tj * tj * tj;
    const R Fi = I.h5 * (ti * ti * ti);
    const R Fj = h5_j * tj3;
    const R mk = other ? (R)p.w : R(0);
    const R kri = mk * (Fi + Fj);   // ka * ri, ka = (dW_i + dW_j) m_j
    const R ka = kri * r1;

    const R rv = dpx * dvx + dpy * dvy + dpz * dvz;
    const R w_ij = rv * ri;
    const R w0 = w_ij < R(0) ? w_ij : R(0);
    const R vs = I.cs + Cc.a - R(3) * w0;
    const R rhi = rcp_r(I.dn + B.d);
    const R av0 = (I.bs + B.c) * (I.al + Cc.b) * vs * w0;
    a.vs = a.vs > vs ? a.vs : vs;

    const R ta = (I.pc + B.b - R(0.5) * av0 * rhi) * kri;
    a.ax -= ta * dpx;
    a.ay -= ta * dpy;
    a.az -= ta * dpz;

    const R vsu2 = abs_r(I.pp - B.a) * rhi * R(2);
    const R vsu = vsu2 != R(0) ? vsu2 * rsqrt_r(vsu2) : R(0);
    const R du = I.eg - Cc.d;
    a.ud += ka * (I.pc * w_ij - rhi * (R(0.25) * av0 * w0 - (I.au + Cc.c) * vsu * du));
    a.df += rhi * du * kri;

    const R dg = mk * (I.et * Fi + eh_j * tj3);   // m_j ri (eta_i dW_i + eta_j dW_j)
    a.gx += dg * dpx;
    a.gy += dg * dpy;
    a.gz += dg * dpz;
}

// One j-record of the hydro functor as staged in LDS (R: the pair-term
// type; positions as offsets from the walk's first particle in mixed mode).
template <typename R>
struct HRec {
    typename HPos<R>::rec p;
    R4<R> a, b, c;
    R e, h5;
    int32_t id;
};

// Record k of the list, or an inert record for k >= end (beyond every
// support, zero mass, signal speed -1e20 so it never sets vsmx).  The
// per-record factors of the pair term are formed here in FP64: -5 C1 m_j,
// h_j^5 = hinv_j^5 and eta_j h_j^5.
template <typename R>
__device__ __forceinline__ HRec<R> hydro_load(const sphk_hydro_src &pj, const int32_t *__restrict__ j_idx, uint32_t k,
                                              uint32_t end, double cx, double cy, double cz)
{
    using PR = typename HPos<R>::rec;
    if (k < end) {
        const int j = j_idx ? j_idx[k] : (int)k;
        const double hid = pj.hinv[j];
        const double h5 = hid * (hid * hid * hid) * hid;
        return HRec<R>{PR{(R)(pj.x[j] - cx), (R)(pj.y[j] - cy), (R)(pj.z[j] - cz), (R)(-5. * kCeff1 * pj.m[j])},
                       R4<R>{(R)pj.vx[j], (R)pj.vy[j], (R)pj.vz[j], (R)hid},
                       R4<R>{(R)pj.pres[j], (R)pj.presc[j], (R)pj.bswt[j], (R)pj.dens[j]},
                       R4<R>{(R)pj.vsnd[j], (R)pj.alph[j], (R)pj.alphu[j], (R)pj.thrm[j]}, (R)(pj.eta[j] * h5),
                       (R)h5, pj.id[j]};
    }
    return HRec<R>{PR{(R)kFar, (R)kFar, (R)kFar, R(0)}, R4<R>{R(0), R(0), R(0), R(0)},
                   R4<R>{R(0), R(0), R(0), R(1)}, R4<R>{R(-1e20), R(0), R(0), R(0)}, R(0), R(0), -1};
}

// FP64: at most 168 VGPRs (3 waves per SIMD, a few spills): 11 % faster than
// 2 waves without spills at 10^6 particles.  But launches of few walks with a
// wave each wait for the longest of them and have no use for a third wave
// (OCC 2, none spills): in us with 3 / 2, walks (particles on average): 572
// (17) 124 / 98, 2079 (4.8) 38 / 34, 2592 (9.6) 107 / 88, 3085 (4.9) 59 / 49,
// 3518 (2.8) 33 / 34, 5368 (2.8) 42 / 46, 5385 (19) 298 / 237, 9189 (2.7) 60 /
// 68: the line lies where short walks lose.  Mixed needs 115 VGPRs (4 waves)
// as written.
constexpr int kHydroFew = 3072;

template <bool MIXED, bool PERSIST, int NW, int OCC = MIXED ? (PERSIST ? 4 : 1) : 3>
__global__ __launch_bounds__(kWave *NW) __attribute__((amdgpu_waves_per_eu(OCC))) void hydro_kernel(
    int n_walk, const int32_t *__restrict__ i_off, const int32_t *__restrict__ j_off,
    const int32_t *__restrict__ j_idx, sphk_hydro_src pi, sphk_hydro_src pj, sphk_hydro_out out, int *queue)
{
    using R = real_t<MIXED>;
    static_assert(!PERSIST || NW == 1, "persistent launches take one wave per walk");
    // tile records and the slice-reduction buffer share one LDS block (the
    // reduction runs after the last tile); NW > 1: the waves' sums beside it
    using PR = typename HPos<R>::rec;
    constexpr int kTileBytes = kTile * (sizeof(PR) + 3 * sizeof(R4<R>) + 2 * sizeof(R) + 4);
    constexpr int kRedBytes = 9 * kWave * sizeof(double);
    constexpr int kWaveBytes = (kTileBytes > kRedBytes ? kTileBytes : kRedBytes);
    __shared__ __attribute__((aligned(32))) char smem[NW * kWaveBytes];
    __shared__ R part[NW > 1 ? NW : 1][8][NW > 1 ? kWave : 1];
    const int wv = NW > 1 ? (int)threadIdx.x / kWave : 0;
    PR *sp = reinterpret_cast<PR *>(smem + wv * kWaveBytes);
    R4<R> *sa = reinterpret_cast<R4<R> *>(sp + kTile);
    R4<R> *sb = sa + kTile;
    R4<R> *sc = sb + kTile;
    R *se = reinterpret_cast<R *>(sc + kTile);
    R *sh = se + kTile;
    int32_t *sid = reinterpret_cast<int32_t *>(sh + kTile);
    double *red = reinterpret_cast<double *>(smem);

    auto walk = [&](const int w, const int lane) {
        const int ib = i_off[w], ie = i_off[w + 1];
        const uint32_t jb = j_off[w], je = j_off[w + 1];
        if (ib >= ie) return;   // a walk of no particles has no first one (ib may be past the last particle)

        // mixed: positions as offsets from the walk's first particle
        const double cx = MIXED ? pi.x[ib] : 0., cy = MIXED ? pi.y[ib] : 0., cz = MIXED ? pi.z[ib] : 0.;
        for (int c0 = ib; c0 < ie; c0 += kWave) {
            const Map M(min(kWave, ie - c0), lane);
            const int i = c0 + M.il;
            HydroI<R> I;
            I.px = pi.x[i] - cx;
            I.py = pi.y[i] - cy;
            I.pz = pi.z[i] - cz;
            I.vx = (R)pi.vx[i];
            I.vy = (R)pi.vy[i];
            I.vz = (R)pi.vz[i];
            const double hid = pi.hinv[i];
            I.hi = (R)hid;
            I.h5 = (R)(hid * (hid * hid * hid) * hid);
            I.pp = (R)pi.pres[i];
            I.pc = (R)pi.presc[i];
            I.bs = (R)pi.bswt[i];
            I.dn = (R)pi.dens[i];
            I.cs = (R)pi.vsnd[i];
            I.al = (R)pi.alph[i];
            I.au = (R)pi.alphu[i];
            I.eg = (R)pi.thrm[i];
            I.et = (R)pi.eta[i];
            I.id = pi.id[i];

            constexpr int kOwn = (8 + NW - 1) / NW;   // sums a wave keeps
            double acc[kOwn];
#pragma unroll
            for (int q = 0; q < kOwn; q++) acc[q] = 0.;
            R vsmx = R(0);
            // each lane loads its record of the tile into registers before the
            // barrier (loading the next tile's record during the sweep measured
            // 3 % slower in mixed mode, and its registers spill in FP64)
            for (uint32_t r0 = jb; r0 < je; r0 += NW * kTile) {
                const uint32_t t0 = r0 + wv * kTile;
                HydroAcc<R> a{R(0), R(0), R(0), R(0), R(0), R(0), R(0), R(0), vsmx};
                if (t0 < je) {
                    const int nt = (int)min((uint32_t)kTile, je - t0);
                    const HRec<R> nx = hydro_load<R>(pj, j_idx, t0 + lane, je, cx, cy, cz);
                    wave_sync();
                    sp[lane] = nx.p;
                    sa[lane] = nx.a;
                    sb[lane] = nx.b;
                    sc[lane] = nx.c;
                    se[lane] = nx.e;
                    sh[lane] = nx.h5;
                    sid[lane] = nx.id;
                    wave_sync();
                    int k = M.slice;
                    for (; k + M.S < nt; k += 2 * M.S) {
                        const int k1 = k + M.S;
                        const PR p0 = sp[k], p1 = sp[k1];
                        const R4<R> a0 = sa[k], a1 = sa[k1], b0 = sb[k], b1 = sb[k1], c0_ = sc[k], c1 = sc[k1];
                        const R e0 = se[k], e1 = se[k1], f0 = sh[k], f1 = sh[k1];
                        const int32_t d0 = sid[k], d1 = sid[k1];
                        hydro_pair<R>(p0, a0, b0, c0_, e0, f0, d0, I, a);
                        hydro_pair<R>(p1, a1, b1, c1, e1, f1, d1, I, a);
                    }
                    for (; k < nt; k += M.S) hydro_pair<R>(sp[k], sa[k], sb[k], sc[k], se[k], sh[k], sid[k], I, a);
                }
                vsmx = a.vs;
                const R sum[8] = {a.ax, a.ay, a.az, a.ud, a.df, a.gx, a.gy, a.gz};
                if (NW == 1) {
#pragma unroll
                    for (int q = 0; q < kOwn; q++) acc[q] += (double)sum[q];
                } else {
#pragma unroll
                    for (int q = 0; q < 8; q++) part[wv][q][lane] = sum[q];
                    __syncthreads();
#pragma unroll
                    for (int o = 0; o < kOwn; o++) {
                        const int q = wv + o * NW;
                        if (q < 8)
                            for (int v = 0; v < NW && r0 + v * kTile < je; v++) acc[o] += (double)part[v][q][lane];
                    }
                    __syncthreads();
                }
            }
            // hdr_hydro.hpp:402-419
            if (NW == 1) {
                double v[9] = {acc[0], acc[1 % kOwn], acc[2 % kOwn], acc[3 % kOwn], acc[4 % kOwn], acc[5 % kOwn],
                               acc[6 % kOwn], acc[7 % kOwn], (double)vsmx};
                slice_reduce<9>(v, red, M, lane, 1 << 8);
                if (M.lead) {
                    out.ax[i] = v[0] * 0.5;
                    out.ay[i] = v[1] * 0.5;
                    out.az[i] = v[2] * 0.5;
                    out.udot[i] = v[3] * 0.5;
                    out.diffu[i] = v[4] * 2.;
                    out.gx[i] = v[5] * 0.5;
                    out.gy[i] = v[6] * 0.5;
                    out.gz[i] = v[7] * 0.5;
                    out.vsmx[i] = v[8];
                }
            } else {
                double *const dst[9] = {out.ax, out.ay, out.az, out.udot, out.diffu, out.gx, out.gy, out.gz, out.vsmx};
                part[wv][0][lane] = vsmx;   // part and the tiles are no longer read
                __syncthreads();
#pragma unroll
                for (int o = 0; o < kOwn; o++)
                    if (wv + o * NW < 8) red[(wv + o * NW) * kWave + lane] = acc[o];
                if (wv == NW - 1) {
                    R m = part[0][0][lane];
                    for (int v = 1; v < NW; v++) m = m > part[v][0][lane] ? m : part[v][0][lane];
                    red[8 * kWave + lane] = (double)m;
                }
                __syncthreads();
                if (M.lead)
                    for (int q = wv; q < 9; q += NW) {
                        double a = red[q * kWave + M.il];
                        for (int t = 1; t < M.S; t++) {
                            const double b = red[q * kWave + M.il + M.ni * t];
                            a = q == 8 ? (a > b ? a : b) : a + b;
                        }
                        dst[q][i] = q == 8 ? a : q == 4 ? a * 2. : a * 0.5;
                    }
                __syncthreads();   // LDS of this chunk no longer read
            }
        }
    };
    run_walks<PERSIST>(n_walk, queue, walk);
}

// ---------------------------------------------------------------------------
// Gravity: scalar calcGravity<TJ>, sph_yamauchi/run/hdr_gravity.hpp:295-338,
// over the EPJ list and then the SPJ list of each walk.
// ---------------------------------------------------------------------------
// j-record staged in LDS: position FP64; mass and softening in the pair
// precision (one 32-byte record in the mixed path).
template <bool MIXED>
struct GRec;
template <>
struct alignas(16) GRec<true> {
    double x, y, z;
    float m, e;
};
template <>
struct alignas(8) GRec<false> {
    double x, y, z, m, e;
};

template <typename R>
struct GravAcc {
    R ax, ay, az, pt, et;
};

// General pair term (softening of i and of j may differ):
// acc -= m x (rei3_i + rei3_j), pot -= m (rei_i + rei_j), eta += m rei3_i;
// the per-particle totals are halved at the end (hdr_gravity.hpp:310-331).
template <bool MIXED, bool ETA>
__device__ __forceinline__ void gravity_pair(const GRec<MIXED> &p, double px, double py, double pz,
                                             real_t<MIXED> e2i, GravAcc<real_t<MIXED>> &a)
{
    using R = real_t<MIXED>;
    const R dpx = (R)(px - p.x);
    const R dpy = (R)(py - p.y);
    const R dpz = (R)(pz - p.z);
    const R r2 = dpx * dpx + dpy * dpy + dpz * dpz;
    const R rei_i = rsqrt_r(r2 + e2i);
    const R rei_j = rsqrt_r(r2 + (R)p.e);
    const R rei3_i = rei_i * rei_i * rei_i;
    const R rei3_j = rei_j * rei_j * rei_j;
    const R m_j = (R)p.m;
    const R dg2 = m_j * (rei3_i + rei3_j);
    a.pt -= m_j * (rei_i + rei_j);
    a.ax -= dpx * dg2;
    a.ay -= dpy * dg2;
    a.az -= dpz * dg2;
    if (ETA) a.et += m_j * rei3_i;
}

// Uniform softening (every eps2 equal, e.g. a constant gravitational
// softening): the two symmetrised terms coincide, one rsqrt per pair.
// Accumulates +m x rei3, +m rei, +m rei3; the caller finishes with the sign.
template <bool MIXED, bool ETA>
__device__ __forceinline__ void gravity_pair_uniform(const GRec<MIXED> &p, double px, double py,
                                                     double pz, real_t<MIXED> e2,
                                                     GravAcc<real_t<MIXED>> &a)
{
    using R = real_t<MIXED>;
    const R dpx = (R)(px - p.x);
    const R dpy = (R)(py - p.y);
    const R dpz = (R)(pz - p.z);
    // r^2 + eps^2 with the softening in the first FMA
    const R r2e = fma_r(dpz, dpz, fma_r(dpy, dpy, fma_r(dpx, dpx, e2)));
    const R rei = rsqrt_r(r2e);
    const R m_j = (R)p.m;
    const R mr = m_j * rei;
    const R w = mr * rei * rei;
    a.pt += mr;
    a.ax += dpx * w;
    a.ay += dpy * w;
    a.az += dpz * w;
    if (ETA) a.et += w;
}

// Records kb .. ke - 1 (at most kTile) of a list: the lane's sums over its slice.
template <bool MIXED, bool UNIFORM, bool ETA>
__device__ __forceinline__ GravAcc<real_t<MIXED>> gravity_tile(int lane, const Map &M, int kb, int ke,
                                                               const int32_t *__restrict__ idx,
                                                               const sphk_grav_src &src, double px, double py,
                                                               double pz, double e2_i, GRec<MIXED> *sp)
{
    using R = real_t<MIXED>;
    const R e2 = (R)e2_i;
    const int nt = ke - kb;
    wave_sync();
    if (lane < nt) {
        const int j = idx ? idx[kb + lane] : kb + lane;
        sp[lane] = GRec<MIXED>{src.x[j], src.y[j], src.z[j], (R)src.m[j], (R)src.eps2[j]};
    } else {
        sp[lane] = GRec<MIXED>{kFar, kFar, kFar, R(0), R(1)};
    }
    wave_sync();
    GravAcc<R> a{R(0), R(0), R(0), R(0), R(0)};
    int k = M.slice;
    for (; k + 3 * M.S < nt; k += 4 * M.S) {
        const GRec<MIXED> p0 = sp[k], p1 = sp[k + M.S], p2 = sp[k + 2 * M.S], p3 = sp[k + 3 * M.S];
        if (UNIFORM) {
            gravity_pair_uniform<MIXED, ETA>(p0, px, py, pz, e2, a);
            gravity_pair_uniform<MIXED, ETA>(p1, px, py, pz, e2, a);
            gravity_pair_uniform<MIXED, ETA>(p2, px, py, pz, e2, a);
            gravity_pair_uniform<MIXED, ETA>(p3, px, py, pz, e2, a);
        } else {
            gravity_pair<MIXED, ETA>(p0, px, py, pz, e2, a);
            gravity_pair<MIXED, ETA>(p1, px, py, pz, e2, a);
            gravity_pair<MIXED, ETA>(p2, px, py, pz, e2, a);
            gravity_pair<MIXED, ETA>(p3, px, py, pz, e2, a);
        }
    }
    for (; k < nt; k += M.S) {
        if (UNIFORM)
            gravity_pair_uniform<MIXED, ETA>(sp[k], px, py, pz, e2, a);
        else
            gravity_pair<MIXED, ETA>(sp[k], px, py, pz, e2, a);
    }
    return a;
}

// Mixed precision with uniform softening: the j-records of a walk are staged
// as FP32 offsets from a reference point of the walk (its first i-particle),
// formed in FP64, so the pair term needs no FP64 arithmetic.  The offset of
// a far record carries a relative rounding error of 2^-24 of its distance;
// for a near pair the error is 2^-24 of its distance from the reference point.
template <bool ETA>
__device__ __forceinline__ void gravity_pair_rel(const float4 &p, float xi, float yi, float zi, float e2,
                                                 GravAcc<float> &a)
{
    const float dx = xi - p.x;
    const float dy = yi - p.y;
    const float dz = zi - p.z;
    // r^2 + eps^2 with the softening in the first FMA
    const float rei = rsqrt_r(fma_r(dz, dz, fma_r(dy, dy, fma_r(dx, dx, e2))));
    const float mr = p.w * rei;
    const float w = mr * rei * rei;
    a.pt += mr;
    a.ax += dx * w;
    a.ay += dy * w;
    a.az += dz * w;
    if (ETA) a.et += w;
}

// Records are staged kGravBlock at a time (one barrier pair per block, four
// records in flight per lane); each lane's FP32 partial sums over a block
// (at most kGravBlock / S terms) are folded into FP64 once per block.
constexpr int kGravBlock = 4 * kTile;

// Records kb .. ke - 1 (at most kGravBlock) of a list, as gravity_tile.
template <bool ETA>
__device__ __forceinline__ GravAcc<float> gravity_block_rel(const Map &M, int lane, int kb, int ke,
                                                            const int32_t *__restrict__ idx,
                                                            const sphk_grav_src &src, double cx, double cy, double cz,
                                                            float xi, float yi, float zi, float e2, float4 *sp)
{
    const int nb = ke - kb;
    wave_sync();
    // all of a lane's indices, then all its records, are loaded before any is
    // written (past the end: the last record again): 955 -> 938 us at 10^6
    // particles against one record after the other
    constexpr int kPer = kGravBlock / kWave;
    int j[kPer];
    double4 v[kPer];
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const int e = min(u * kWave + lane, nb - 1);
        j[u] = idx ? idx[kb + e] : kb + e;
    }
#pragma unroll
    for (int u = 0; u < kPer; u++) v[u] = make_double4(src.x[j[u]], src.y[j[u]], src.z[j[u]], src.m[j[u]]);
#pragma unroll
    for (int u = 0; u < kPer; u++)
        sp[u * kWave + lane] = make_float4((float)(v[u].x - cx), (float)(v[u].y - cy), (float)(v[u].z - cz), (float)v[u].w);
    wave_sync();
    GravAcc<float> a{0.f, 0.f, 0.f, 0.f, 0.f};
    int k = M.slice < M.S ? M.slice : kGravBlock;   // idle lanes: empty sweeps
    for (; k + 3 * M.S < nb; k += 4 * M.S) {
        const float4 p0 = sp[k], p1 = sp[k + M.S], p2 = sp[k + 2 * M.S], p3 = sp[k + 3 * M.S];
        gravity_pair_rel<ETA>(p0, xi, yi, zi, e2, a);
        gravity_pair_rel<ETA>(p1, xi, yi, zi, e2, a);
        gravity_pair_rel<ETA>(p2, xi, yi, zi, e2, a);
        gravity_pair_rel<ETA>(p3, xi, yi, zi, e2, a);
    }
    for (; k < nb; k += M.S) gravity_pair_rel<ETA>(sp[k], xi, yi, zi, e2, a);
    return a;
}

// ETA false: the caller does not need the softening-gradient sum (out.eta
// NULL, e.g. under a constant softening, where it does not enter).
// Persistent mixed launches: at least 8 waves per SIMD, but 5 with uniform
// softening, whose four staged records would spill 29 registers at 8 (10^5
// particles: 208 us, 323 with the spills, 297 before the records were staged
// together).
template <bool MIXED, bool UNIFORM, bool ETA, bool PERSIST, int NW>
__global__ __launch_bounds__(kWave *NW) __attribute__((amdgpu_waves_per_eu(PERSIST && MIXED ? (UNIFORM ? 5 : 8) : 1))) void gravity_kernel(
    int n_walk, const int32_t *__restrict__ i_off, const int32_t *__restrict__ j_off,
    const int32_t *__restrict__ j_idx, sphk_grav_src pj, const int32_t *__restrict__ s_off,
    const int32_t *__restrict__ s_idx, sphk_grav_src ps, sphk_grav_src pi, sphk_grav_out out, int *queue)
{
    using R = real_t<MIXED>;
    static_assert(!PERSIST || NW == 1, "persistent launches take one wave per walk");
    constexpr bool kRel = MIXED && UNIFORM;
    constexpr int kBlk = kRel ? kGravBlock : kTile;
    constexpr int kBlkBytes = kRel ? kGravBlock * (int)sizeof(float4) : kTile * (int)sizeof(GRec<MIXED>);
    constexpr int kRedBytes = 5 * kWave * sizeof(double);
    constexpr int kWaveBytes = NW > 1 || kBlkBytes > kRedBytes ? kBlkBytes : kRedBytes;
    static_assert(NW == 1 || NW * kWaveBytes >= kRedBytes, "reduction buffer");
    __shared__ __attribute__((aligned(32))) char smem[NW * kWaveBytes];
    __shared__ R part[NW > 1 ? NW : 1][5][NW > 1 ? kWave : 1];   // the waves' block sums
    const int wv = NW > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave) : 0;
    char *mine = smem + wv * kWaveBytes;
    double *red = reinterpret_cast<double *>(smem);

    auto walk = [&](const int w, const int lane) {
        const int ib = i_off[w], ie = i_off[w + 1];

        for (int c0 = ib; c0 < ie; c0 += kWave) {
            const Map M(min(kWave, ie - c0), lane);
            const int i = c0 + M.il;
            const double px = pi.x[i], py = pi.y[i], pz = pi.z[i], e2 = pi.eps2[i];
            double cx = 0., cy = 0., cz = 0.;
            float xi = 0.f, yi = 0.f, zi = 0.f;
            if (kRel) {
                cx = pi.x[ib];
                cy = pi.y[ib];
                cz = pi.z[ib];
                xi = (float)(px - cx);
                yi = (float)(py - cy);
                zi = (float)(pz - cz);
            }
            constexpr int kOwn = (5 + NW - 1) / NW;   // sums a wave keeps
            double acc[kOwn];
#pragma unroll
            for (int q = 0; q < kOwn; q++) acc[q] = 0.;
            // the EPJ list, then the SPJ list; NW blocks at a time
            auto list = [&](uint32_t kb, uint32_t ke, const int32_t *idx, const sphk_grav_src &src) {
                for (uint32_t r0 = kb; r0 < ke; r0 += NW * kBlk) {
                    const uint32_t b0 = r0 + wv * kBlk;
                    GravAcc<R> a{R(0), R(0), R(0), R(0), R(0)};
                    if (b0 < ke) {
                        const uint32_t b1 = min(ke, b0 + kBlk);
                        if constexpr (kRel)
                            a = gravity_block_rel<ETA>(M, lane, b0, b1, idx, src, cx, cy, cz, xi, yi, zi, (float)e2,
                                                       reinterpret_cast<float4 *>(mine));
                        else
                            a = gravity_tile<MIXED, UNIFORM, ETA>(lane, M, b0, b1, idx, src, px, py, pz, e2,
                                                                  reinterpret_cast<GRec<MIXED> *>(mine));
                    }
                    const R sum[5] = {a.ax, a.ay, a.az, a.pt, a.et};
                    if (NW == 1) {
#pragma unroll
                        for (int q = 0; q < kOwn; q++) acc[q] += (double)sum[q];
                    } else {
#pragma unroll
                        for (int q = 0; q < 5; q++) part[wv][q][lane] = sum[q];
                        __syncthreads();
#pragma unroll
                        for (int o = 0; o < kOwn; o++) {
                            const int q = wv + o * NW;
                            if (q < 5)
                                for (int v = 0; v < NW && r0 + v * kBlk < ke; v++) acc[o] += (double)part[v][q][lane];
                        }
                        __syncthreads();
                    }
                }
            };
            list(j_off[w], j_off[w + 1], j_idx, pj);
            if (s_off) list(s_off[w], s_off[w + 1], s_idx, ps);
            // UNIFORM: 0.5 * (-2 sum m rei3 x) etc.
            constexpr double kf = UNIFORM ? -1. : 0.5;
            if (NW == 1) {
                double v[5] = {acc[0], acc[1 % kOwn], acc[2 % kOwn], acc[3 % kOwn], acc[4 % kOwn]};
                slice_reduce<5>(v, red, M, lane);
                if (M.lead) {
                    out.ax[i] = v[0] * kf;
                    out.ay[i] = v[1] * kf;
                    out.az[i] = v[2] * kf;
                    out.pot[i] = v[3] * kf;
                    if (ETA) out.eta[i] = v[4];
                }
            } else {
                double *const dst[5] = {out.ax, out.ay, out.az, out.pot, out.eta};
                __syncthreads();   // the last blocks are read
#pragma unroll
                for (int o = 0; o < kOwn; o++)
                    if (wv + o * NW < 5) red[(wv + o * NW) * kWave + lane] = acc[o];
                wave_sync();
                if (M.lead)
                    for (int q = wv; q < (ETA ? 5 : 4); q += NW) {
                        double a = red[q * kWave + M.il];
                        for (int t = 1; t < M.S; t++) a = a + red[q * kWave + M.il + M.ni * t];
                        dst[q][i] = q == 4 ? a : a * kf;
                    }
                __syncthreads();   // LDS of this chunk no longer read
            }
        }
    };
    run_walks<PERSIST>(n_walk, queue, walk);
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------
// Grid of a persistent launch: the workgroups of this kernel the chip holds
// at once (a multiple of kXcd), at most one per walk of each XCD queue.
template <typename K>
static int persistent_grid(K kernel, int n_walk)
{
    int dev = 0, n_cu = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kWave, 0) != hipSuccess)
        return -1;
    const int full = (per_cu > 0 ? per_cu : 1) * (n_cu > 0 ? n_cu : 1);
    const int g = (full + kXcd - 1) / kXcd * kXcd;
    const int need = (n_walk + kXcd - 1) / kXcd * kXcd;
    return g < need ? g : need;
}

// One launch: ordinary (grid = n_walk, waves waves per walk) or, with a queue,
// persistent.
#define SPHK_LAUNCH(KERNEL, KERNEL_P, waves, ...)                                                       \
    do {                                                                                                 \
        if (queue) {                                                                                     \
            const int g_ = persistent_grid(KERNEL_P, n_walk);                                            \
            if (g_ <= 0) return hipErrorInvalidValue;                                                    \
            hipLaunchKernelGGL(KERNEL_P, dim3(g_), dim3(kWave), 0, st, __VA_ARGS__, queue);              \
        } else {                                                                                         \
            hipLaunchKernelGGL(KERNEL, dim3(n_walk), dim3(kWave * (waves)), 0, st, __VA_ARGS__, nullptr); \
        }                                                                                                \
    } while (0)
hipError_t launch_density(hipStream_t st, int n_walk, int64_t n_i, const int32_t *i_off, const int32_t *j_off,
                          const int32_t *j_idx, const sphk_dens_src &pi, const sphk_dens_src &pj,
                          const sphk_dens_out &out, double eta_ksrh, double hmax, bool mixed, int list_cap,
                          int *queue)
{
    if (n_walk <= 0) return hipSuccess;
#define SPHK_LAUNCH_D(M, CAPV, W, OCC)                                                                    \
    SPHK_LAUNCH((density_kernel<M, CAPV, false, W, OCC>), (density_kernel<M, CAPV, true, 1, M ? 2 : 3>), W, \
                n_walk, i_off, j_off, j_idx, pi, pj, out, eta_ksrh, hmax)
#define SPHK_DENS(M, CAPV)                             \
    do {                                               \
        if (waves == 2)                                \
            SPHK_LAUNCH_D(M, CAPV, 2, 3);              \
        else if (M && few)                             \
            SPHK_LAUNCH_D(M, CAPV, 1, M ? 2 : 3);      \
        else                                           \
            SPHK_LAUNCH_D(M, CAPV, 1, 3);              \
    } while (0)
    const int waves = waves_per_walk(n_walk, n_i, kDensRule);
    const bool few = n_walk <= (n_i > 0 ? kDensFew : kDensFewUnknown);
    if (list_cap == 192) {
        if (mixed)
            SPHK_DENS(true, 192);
        else
            SPHK_DENS(false, 192);
    } else {
        if (mixed)
            SPHK_DENS(true, 256);
        else
            SPHK_DENS(false, 256);
    }
#undef SPHK_DENS
#undef SPHK_LAUNCH_D
    return hipGetLastError();
}

hipError_t launch_hydro(hipStream_t st, int n_walk, int64_t n_i, const int32_t *i_off, const int32_t *j_off,
                        const int32_t *j_idx, const sphk_hydro_src &pi, const sphk_hydro_src &pj,
                        const sphk_hydro_out &out, bool mixed, int *queue)
{
    if (n_walk <= 0) return hipSuccess;
#define SPHK_LAUNCH_H(M, W) \
    SPHK_LAUNCH((hydro_kernel<M, false, W>), (hydro_kernel<M, true, 1>), W, n_walk, i_off, j_off, j_idx, pi, pj, out)
    const int waves = waves_per_walk(n_walk, n_i, mixed ? kHydroRule : kHydroF64Rule);
    if (mixed) {
        if (waves == 4)
            SPHK_LAUNCH_H(true, 4);
        else
            SPHK_LAUNCH_H(true, 1);
    } else {
        switch (waves) {
        case 4: SPHK_LAUNCH_H(false, 4); break;
        case 2: SPHK_LAUNCH_H(false, 2); break;
        default:
            if (n_walk <= kHydroFew)
                SPHK_LAUNCH((hydro_kernel<false, false, 1, 2>), (hydro_kernel<false, true, 1>), 1, n_walk, i_off, j_off,
                            j_idx, pi, pj, out);
            else
                SPHK_LAUNCH_H(false, 1);
        }
    }
#undef SPHK_LAUNCH_H
    return hipGetLastError();
}

hipError_t launch_gravity(hipStream_t st, int n_walk, int64_t n_i, const int32_t *i_off, const int32_t *j_off,
                          const int32_t *j_idx, const sphk_grav_src &pj, const int32_t *s_off,
                          const int32_t *s_idx, const sphk_grav_src &ps, const sphk_grav_src &pi,
                          const sphk_grav_out &out, bool mixed, bool uniform, int *queue)
{
    if (n_walk <= 0) return hipSuccess;
#define SPHK_LAUNCH_G(M, U, E, W)                                                                            \
    SPHK_LAUNCH((gravity_kernel<M, U, E, false, W>), (gravity_kernel<M, U, E, true, 1>), W, n_walk, i_off, j_off, \
                j_idx, pj, s_off, s_idx, ps, pi, out)
    // the kernel of one (precision, softening, eta), by its waves per walk; the
    // rel path (mixed, uniform) has no use for 8
#define SPHK_REL(E)                               \
    switch (waves) {                              \
    case 4: SPHK_LAUNCH_G(true, true, E, 4); break; \
    case 2: SPHK_LAUNCH_G(true, true, E, 2); break; \
    default: SPHK_LAUNCH_G(true, true, E, 1); break; \
    }
#define SPHK_GEN(M, U, E)                      \
    switch (waves) {                           \
    case 8: SPHK_LAUNCH_G(M, U, E, 8); break;  \
    case 4: SPHK_LAUNCH_G(M, U, E, 4); break;  \
    default: SPHK_LAUNCH_G(M, U, E, 1); break; \
    }
    const bool eta = out.eta != nullptr;
    const int waves = waves_per_walk(n_walk, n_i, mixed && uniform ? kGravRelRule : kGravRule);
    if (mixed && uniform) {
        if (eta) SPHK_REL(true) else SPHK_REL(false)
    } else if (mixed) {
        if (eta) SPHK_GEN(true, false, true) else SPHK_GEN(true, false, false)
    } else if (uniform) {
        if (eta) SPHK_GEN(false, true, true) else SPHK_GEN(false, true, false)
    } else {
        if (eta) SPHK_GEN(false, false, true) else SPHK_GEN(false, false, false)
    }
#undef SPHK_REL
#undef SPHK_GEN
#undef SPHK_LAUNCH_G
    return hipGetLastError();
}
#undef SPHK_LAUNCH

}  // namespace sphk
