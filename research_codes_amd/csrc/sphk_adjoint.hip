// sphk_adjoint.hip -- vector-Jacobian products of the three functors in
// FP64: gravity (uniform softening, the reverse of gravity_pair_uniform),
// hydro and density.
//
// One wave per walk.  Hydro and density: layout as the forward kernels, S =
// floor(64/ni) j-slices, 64-record LDS tiles; the i-side cotangent of a lane
// stays in registers and is combined across slices through LDS at the end of
// the walk.  Gravity: one record per lane, the i-particles in LDS.  The
// j-side: a lane's own in gravity, collected per tile in LDS (atomic adds) in
// density, none in hydro (its symmetric lists hold both pair orders); it
// leaves with one HBM atomic add per record and component.
#include "sphk_adjoint.h"
#include "sphk_device.hpp"
#include "sphk_internal.hpp"

namespace sphk {
namespace {

// List positions are formed unsigned, as in the forward kernels: one past the
// end of a list may lie beyond 2^31 - 1.
__device__ __forceinline__ int xcd_walk_adj(int b, int n_walk)
{
    // as the forward kernels: chunks of 64 walks dealt to the 8 XCDs in turn
    constexpr int kX = 8, kC = 64;
    const int n_full = n_walk / (kX * kC) * (kX * kC);
    if (b >= n_full) return b;
    const int x = b % kX, k = b / kX;
    return ((k / kC) * kX + x) * kC + k % kC;
}

// Walk of workgroup b when each of the 8 XCDs takes one contiguous range.
__device__ __forceinline__ int xcd_walk_range(int b, int n_walk)
{
    constexpr int kX = 8;
    const int per = n_walk / kX;
    return b < per * kX ? (b % kX) * per + b / kX : b;
}

// Gravity VJP: one record per lane.  A walk's i-particles are taken kVjpI at
// a time; their positions and cotangents sit in LDS, read as broadcasts, and
// each lane keeps its share of their position cotangents in registers (three
// FP64 sums per i) over the whole list, so a pair is evaluated once for both
// sides and the i-sides are combined across the wave once per chunk.  A lane
// loads its next record before the j-side of the current one leaves with one
// global FP64 atomic per component: memory operations complete in order, and
// the next record must not wait behind the atomics.
//
// The atomics bound the kernel (2x10^5 particles, 2.5x10^7 records: 0.5 ms of
// 1.2 without them), by requests, not by values: PACKED sends the three
// components of a record from neighbouring lanes into one [n][3] array, and
// each XCD takes one contiguous range of walks, so that fewer lines move
// between the XCDs' caches (chunks of 8 to 1024 walks dealt in turn: 1.31 to
// 1.39 ms, one range each 1.19).  More chunks of i-particles mean more
// atomics: kVjpI = 8 / 12 / 16 take 2.4 / 1.9 / 1.6 ms unpacked, and 16 is
// what leaves 3 waves per SIMD (160 VGPRs).  Before, every pair was evaluated
// twice (a sweep per side, 64-record LDS tiles): 1.7 ms.  A walk of more than
// kVjpI particles sends its records' sums once per chunk and still gains: walk
// groups of 64 and 128 (17 and 35 particles a walk) 1.67 -> 1.48 and 2.89 ->
// 1.73 ms packed, 1.64 and 1.75 unpacked.
constexpr int kVjpI = 16;

struct alignas(16) VI {
    double x, y, z, ax, ay, az, pb, eb;
};

struct VRec {
    double x, y, z, m;
    int32_t j;
};

__device__ __forceinline__ VRec vjp_load(const sphk_grav_src &src, const int32_t *__restrict__ idx, uint32_t k, uint32_t ke)
{
    VRec r{0., 0., 0., 0., -1};   // past the end: j < 0
    if (k < ke) {
        r.j = idx ? idx[k] : (int32_t)k;
        r.x = src.x[r.j];
        r.y = src.y[r.j];
        r.z = src.z[r.j];
        r.m = src.m[r.j];
    }
    return r;
}

// One list of a walk chunk (n i-particles in sI).  The cotangent of record
// r's position from the pair (i, r) is the reverse of the uniform-softening
// pair term, m_r (T abar - pbar w^3 d + 3 ebar w^5 d) with T = w^3 I - 3 w^5
// d d^T and d = x_i - x_r; the i-side gets its negative.
template <bool PACKED>
__device__ __forceinline__ void vjp_list(int lane, int n, uint32_t kb, uint32_t ke, const int32_t *__restrict__ idx,
                                         const sphk_grav_src &src, const VI *sI, double *sv, int32_t *sj, double e2,
                                         double (&gi)[kVjpI][3], double *outx, double *outy, double *outz)
{
    VRec nx = vjp_load(src, idx, kb + lane, ke);
    for (uint32_t t0 = kb; t0 < ke; t0 += kWave) {
        const VRec r = nx;
        nx = vjp_load(src, idx, t0 + kWave + lane, ke);
        double jx = 0., jy = 0., jz = 0.;
        asm volatile("" ::: "memory");   // read sI per tile: hoisted, it would take every register
        if (r.j >= 0) {   // past the end a zero mass would not do: 0 times a cotangent that overflows is no 0
#pragma unroll
            for (int q = 0; q < kVjpI; q++) {
                if (q < n) {
                    const VI I = sI[q];
                    const double dx = I.x - r.x, dy = I.y - r.y, dz = I.z - r.z;
                    const double w = rsqrt_f64(__builtin_fma(dz, dz, __builtin_fma(dy, dy, __builtin_fma(dx, dx, e2))));
                    const double w2 = w * w;
                    const double mw3 = r.m * (w2 * w);
                    const double dot = __builtin_fma(dx, I.ax, __builtin_fma(dy, I.ay, __builtin_fma(dz, I.az, -I.eb)));
                    const double f = mw3 * __builtin_fma(3. * w2, dot, I.pb);
                    const double cx = mw3 * I.ax - f * dx, cy = mw3 * I.ay - f * dy, cz = mw3 * I.az - f * dz;
                    jx += cx;
                    jy += cy;
                    jz += cz;
                    gi[q][0] -= cx;
                    gi[q][1] -= cy;
                    gi[q][2] -= cz;
                }
            }
        }
        if (PACKED) {
            __syncthreads();   // values of the previous tile sent
            sj[lane] = r.j;
            sv[3 * lane] = jx;
            sv[3 * lane + 1] = jy;
            sv[3 * lane + 2] = jz;
            __syncthreads();
            for (int t = 0; t < 3; t++) {
                const int v = t * kWave + lane, q = v / 3;
                const int j = sj[q];
                if (j >= 0) atomicAdd(&outx[3 * (size_t)j + (v - 3 * q)], sv[v]);
            }
        } else if (r.j >= 0) {
            atomicAdd(&outx[r.j], jx);
            atomicAdd(&outy[r.j], jy);
            atomicAdd(&outz[r.j], jz);
        }
    }
}

template <bool PACKED>
__global__ __launch_bounds__(kWave) void gravity_vjp_kernel(
    int n_walk, const int32_t *__restrict__ i_off, const int32_t *__restrict__ j_off,
    const int32_t *__restrict__ j_idx, sphk_grav_src pj, const int32_t *__restrict__ s_off,
    const int32_t *__restrict__ s_idx, sphk_grav_src ps, sphk_grav_src pi, double e2,
    const double *__restrict__ abx, const double *__restrict__ aby, const double *__restrict__ abz,
    const double *__restrict__ pbar, const double *__restrict__ ebar, double *gx, double *gy, double *gz,
    double *nx, double *ny, double *nz)
{
    __shared__ VI sI[kVjpI];
    __shared__ double sv[PACKED ? 3 * kWave : 1];
    __shared__ int32_t sj[PACKED ? kWave : 1];
    if ((int)blockIdx.x >= n_walk) return;
    const int w = xcd_walk_range(blockIdx.x, n_walk);
    const int lane = threadIdx.x;
    const int ib = i_off[w], ie = i_off[w + 1];
    for (int c0 = ib; c0 < ie; c0 += kVjpI) {
        const int n = __builtin_amdgcn_readfirstlane(min(kVjpI, ie - c0));
        __syncthreads();   // sI of the previous chunk no longer read
        if (lane < n) {
            const int i = c0 + lane;
            sI[lane] = VI{pi.x[i], pi.y[i], pi.z[i], abx[i], aby[i], abz[i], pbar[i], ebar ? ebar[i] : 0.};
        }
        __syncthreads();
        double gi[kVjpI][3];
#pragma unroll
        for (int q = 0; q < kVjpI; q++) gi[q][0] = gi[q][1] = gi[q][2] = 0.;
        vjp_list<PACKED>(lane, n, j_off[w], j_off[w + 1], j_idx, pj, sI, sv, sj, e2, gi, gx, gy, gz);
        if (s_off)
            vjp_list<PACKED>(lane, n, s_off[w], s_off[w + 1], s_idx, ps, sI, sv, sj, e2, gi, nx, ny, nz);
        // the wave's sums of each i, in a fixed order
#pragma unroll
        for (int q = 0; q < kVjpI; q++) {
            if (q < n) {
                double s[3] = {gi[q][0], gi[q][1], gi[q][2]};
                for (int d = 1; d < kWave; d <<= 1)
                    for (int c = 0; c < 3; c++) s[c] += __shfl_xor(s[c], d, kWave);
                if (lane == 0) {
                    const size_t i = (size_t)(c0 + q);
                    atomicAdd(&gx[PACKED ? 3 * i : i], s[0]);
                    atomicAdd(&(PACKED ? gx + 1 : gy)[PACKED ? 3 * i : i], s[1]);
                    atomicAdd(&(PACKED ? gx + 2 : gz)[PACKED ? 3 * i : i], s[2]);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Hydro functor VJP (FP64).  The symmetric lists hold every interacting pair
// in both directions (r < max(H_i, H_j) puts j in the list of i's walk and i
// in the list of j's walk; pairs beyond both supports contribute exactly
// zero, with zero derivatives, as the kernel is C2 at q = 1).  So the
// cotangent of a particle's inputs is the sum, over its own list, of the
// i-side derivative of its pair terms and the j-side derivative of its
// neighbours' pair terms: one register accumulator per lane, no atomics,
// and a fixed summation order (bitwise reproducible).
//
// Both are derivatives of one scalar, the pair's terms in P's and in Q's
// outputs weighted by their cotangents, with respect to P's inputs.  The
// factors the two orders share (distance, F_P + F_Q, v_sig, 1/(rho_P +
// rho_Q), ...) are symmetric or change sign, so the scalar is
//   L = -5 C1 [ (F_P + F_Q) (-P_t (A.d)/2 + r B/2 + 2 rhi du D) + E (G.d)/2 ]
// with A = m_Q abar_P - m_P abar_Q (G the same of the accg cotangents), B and
// D the mass-weighted du/dt and diffu cotangents, and is reversed once per
// pair.  Bound by FP64 issue: an IEEE FP64 square root measures 86 cycles per
// wave and a division 59 against 4 for an FMA, so 1/r, 1/(rho_P + rho_Q) and
// the signal-speed root come from Newton-refined v_rsq / v_rcp.  2x10^5
// particles, 3.5x10^7 entries: 0.98 ms with two one-sided reverses per pair
// and IEEE roots and divisions, 0.53 ms so, 0.46 ms with the pairs of a tile
// that are not beyond both supports (about a third) marked first.  Against
// 80-bit values of the same sums each field's error is 1.96e-16 to 4.6e-16 of
// its norm (with IEEE roots and divisions 1.98e-16 to 5.1e-16).  205 VGPRs,
// 2 waves per SIMD; held to 168 (3 waves) it spills and takes 2.8 ms, and
// tiles of 32 or 48 records were 3 % slower.
// ---------------------------------------------------------------------------
struct HP {           // one particle's hydro inputs (hinv^5 derived)
    double x, y, z, vx, vy, vz, h, h5, p, pc, b, d, c, al, au, u, et, m;
};
struct HCot {         // cotangents of that particle's functor outputs
    double ax, ay, az, ud, df, gx, gy, gz;
};
constexpr int kHG = 16;   // x y z vx vy vz hinv pres presc bswt dens vsnd alph alphu thrm eta

__device__ __forceinline__ HP load_hp(const sphk_hydro_src &s, int k)
{
    const double h = s.hinv[k];
    const double h2 = h * h;
    return HP{s.x[k], s.y[k], s.z[k], s.vx[k], s.vy[k], s.vz[k], h, h2 * h2 * h, s.pres[k], s.presc[k],
              s.bswt[k], s.dens[k], s.vsnd[k], s.alph[k], s.alphu[k], s.thrm[k], s.eta[k], s.m[k]};
}

__device__ __forceinline__ HCot load_cot(const sphk_hydro_out &c, int k)
{
    return HCot{c.ax[k], c.ay[k], c.az[k], c.udot[k], c.diffu[k], c.gx[k], c.gy[k], c.gz[k]};
}

// Reverse of the pair (P, Q), hdr_hydro.hpp:352-399 in the closed form of the
// forward kernel: adds to g the derivative, with respect to P's inputs, of
// P's outputs weighted by cp plus Q's outputs weighted by cq.
__device__ __forceinline__ void hydro_pair_vjp(const HP &P, const HP &Q, const HCot &cp, const HCot &cq,
                                               double (&g)[kHG])
{
    constexpr double K = -5. * kCeff1;
    const double dx = P.x - Q.x, dy = P.y - Q.y, dz = P.z - Q.z;
    const double r2 = dx * dx + dy * dy + dz * dz;
    const double ri = rsqrt_f64(r2);
    const double r = r2 * ri;
    const double qp = r * P.h, qq = r * Q.h;
    const double tp = qp < 1. ? 1. - qp : 0., tq = qq < 1. ? 1. - qq : 0.;
    if (tp == 0. && tq == 0.) return;   // beyond both supports: value and derivatives vanish
    const double tp2 = tp * tp, tq2 = tq * tq;
    const double Fp = P.h5 * (tp2 * tp), Fq = Q.h5 * (tq2 * tq);
    const double KF = K * (Fp + Fq);
    const double dvx = P.vx - Q.vx, dvy = P.vy - Q.vy, dvz = P.vz - Q.vz;
    const double w = (dx * dvx + dy * dvy + dz * dvz) * ri;
    const double w0 = w < 0. ? w : 0.;
    const double vs = P.c + Q.c - 3. * w0;
    const double rhi = rcp_f64(P.d + Q.d);
    const double bs = P.b + Q.b, as = P.al + Q.al, aus = P.au + Q.au;
    const double bsas = bs * as;
    const double vsw = vs * w0;
    const double av0 = bsas * vsw;
    const double Pt = P.pc + Q.pc - 0.5 * av0 * rhi;
    const double dP = P.p - Q.p;
    const double vsu2 = __builtin_fabs(dP) * rhi * 2.;
    const double vsui = vsu2 > 0. ? rsqrt_f64(vsu2) : 0.;   // 1 / vsu
    const double vsu = vsu2 * vsui;
    const double du = P.u - Q.u;
    // the cotangents of the two orders of the pair, combined
    const double Ax = Q.m * cp.ax - P.m * cq.ax, Ay = Q.m * cp.ay - P.m * cq.ay, Az = Q.m * cp.az - P.m * cq.az;
    const double Gx = Q.m * cp.gx - P.m * cq.gx, Gy = Q.m * cp.gy - P.m * cq.gy, Gz = Q.m * cp.gz - P.m * cq.gz;
    const double D = Q.m * cp.df - P.m * cq.df;
    const double up = Q.m * cp.ud, uq = P.m * cq.ud;
    const double Us = up + uq, Ud = up - uq;
    const double Ad = Ax * dx + Ay * dy + Az * dz;
    const double hGd = 0.5 * (Gx * dx + Gy * dy + Gz * dz);
    const double vdu = vsu * du * Ud;
    const double Pw = up * P.pc + uq * Q.pc;
    const double T = 0.25 * av0 * w0 * Us - aus * vdu;
    const double B = w * Pw - rhi * T;
    const double M1 = -0.5 * Pt * Ad + 0.5 * r * B + 2. * rhi * du * D;
    // F_P, F_Q and eta
    const double KG = K * hGd;
    const double Fs_b = K * M1;
    const double Fp_b = Fs_b + KG * P.et, Fq_b = Fs_b + KG * Q.et;
    const double E = P.et * Fp + Q.et * Fq;
    const double Gd_b = 0.5 * K * E, Ad_b = -0.5 * KF * Pt;
    double dbx = Ad_b * Ax + Gd_b * Gx, dby = Ad_b * Ay + Gd_b * Gy, dbz = Ad_b * Az + Gd_b * Gz;
    // P_t, B and the conduction term
    const double Pt_b = -0.5 * KF * Ad;
    double r_b = 0.5 * KF * B;
    const double B_b = 0.5 * KF * r;
    double rhi_b = 2. * KF * du * D - B_b * T - 0.5 * av0 * Pt_b;
    double du_b = 2. * KF * rhi * D;
    const double T_b = -B_b * rhi;
    double w_b = B_b * Pw;
    const double pc_b = B_b * w * up + Pt_b;
    const double av0_b = 0.25 * w0 * Us * T_b - 0.5 * rhi * Pt_b;
    double w0_b = 0.25 * av0 * Us * T_b;
    const double aus_b = -vdu * T_b;
    const double vsu_b = -aus * du * Ud * T_b;
    du_b -= aus * vsu * Ud * T_b;
    // av0 = bs as vs w0, vs = c_P + c_Q - 3 w0, w0 = min(w, 0)
    const double avw = av0_b * vsw;
    const double bs_b = as * avw, as_b = bs * avw;
    const double abb = av0_b * bsas;
    const double vs_b = abb * w0;
    w0_b += abb * vs - 3. * vs_b;
    if (w < 0.) w_b += w0_b;
    // vsu = sqrt(2 |dP| rhi), rhi = 1 / (rho_P + rho_Q)
    const double vsu2_b = vsu_b * vsui;   // twice the derivative: the factors 2 and 1/2 cancel below
    const double p_b = vsu2_b * rhi * (dP > 0. ? 1. : (dP < 0. ? -1. : 0.));
    rhi_b += vsu2_b * __builtin_fabs(dP);
    const double d_b = -rhi_b * rhi * rhi;
    // w = (d . dv) / r
    const double rv_b = w_b * ri;
    dbx += rv_b * dvx;
    dby += rv_b * dvy;
    dbz += rv_b * dvz;
    r_b -= rv_b * w;
    // F = h^5 t^3, t = 1 - r h inside the support
    const double tp_b = Fp_b * 3. * P.h5 * tp2, tq_b = Fq_b * 3. * Q.h5 * tq2;
    const double ph2 = P.h * P.h;
    const double h_b = Fp_b * 5. * (ph2 * ph2) * (tp2 * tp) - tp_b * r;
    r_b -= tp_b * P.h + tq_b * Q.h;
    const double f = r_b * ri;
    g[0] += dbx + f * dx;
    g[1] += dby + f * dy;
    g[2] += dbz + f * dz;
    g[3] += rv_b * dx;
    g[4] += rv_b * dy;
    g[5] += rv_b * dz;
    g[6] += h_b;
    g[7] += p_b;
    g[8] += pc_b;
    g[9] += bs_b;
    g[10] += d_b;
    g[11] += vs_b;
    g[12] += as_b;
    g[13] += aus_b;
    g[14] += du_b;
    g[15] += KG * Fp;
}

struct HRecV {        // a staged j-record: inputs, its output cotangents, id
    HP p;
    HCot c;
    int32_t id;
};

__global__ __launch_bounds__(kWave) void hydro_vjp_kernel(int n_walk, const int32_t *__restrict__ i_off,
                                                          const int32_t *__restrict__ j_off,
                                                          const int32_t *__restrict__ j_idx, sphk_hydro_src src,
                                                          sphk_hydro_out cot, sphk_hydro_grad grad)
{
    __shared__ HRecV sp[kTile];
    __shared__ double red[kWave];
    if ((int)blockIdx.x >= n_walk) return;
    const int w = xcd_walk_adj(blockIdx.x, n_walk);
    const int lane = threadIdx.x;
    const int ib = i_off[w], ie = i_off[w + 1];
    const uint32_t kb = j_off[w], ke = j_off[w + 1];
    for (int c0 = ib; c0 < ie; c0 += kWave) {
        const int ni = min(kWave, ie - c0);
        const int S = kWave / ni, il = lane % ni;
        const int slice = lane / ni < S ? lane / ni : kTile;   // idle lanes sweep nothing
        const int i = c0 + il;
        const HP P = load_hp(src, i);
        const HCot cp = load_cot(cot, i);
        const int32_t id = src.id[i];
        double g[kHG];
#pragma unroll
        for (int q = 0; q < kHG; q++) g[q] = 0.;
        for (uint32_t t0 = kb; t0 < ke; t0 += kTile) {
            const int nt = (int)min((uint32_t)kTile, ke - t0);
            __syncthreads();
            if (lane < nt) {
                const int j = j_idx ? j_idx[t0 + lane] : (int)(t0 + lane);
                sp[lane] = HRecV{load_hp(src, j), load_cot(cot, j), src.id[j]};
            }
            __syncthreads();
            // the slice's records not beyond both supports, then their pairs
            uint64_t near = 0;
#pragma unroll 4
            for (int k = slice; k < nt; k += S) {
                const HP &q = sp[k].p;
                const double dx = P.x - q.x, dy = P.y - q.y, dz = P.z - q.z, h = fmin(P.h, q.h);
                const bool far = (dx * dx + dy * dy + dz * dz) * (h * h) >= 1. + 1e-12;
                near |= (uint64_t)(!far && sp[k].id != id) << k;
            }
            while (near) {
                const int k = __builtin_ctzll(near);
                near &= near - 1;
                hydro_pair_vjp(P, sp[k].p, cp, sp[k].c, g);
            }
        }
        // per i: the S slices' partials in slice order, then one plain add
        // per field (each particle is the i of exactly one walk lane group)
        double *outs[kHG] = {grad.x, grad.y, grad.z, grad.vx, grad.vy, grad.vz, grad.hinv, grad.pres,
                             grad.presc, grad.bswt, grad.dens, grad.vsnd, grad.alph, grad.alphu, grad.thrm,
                             grad.eta};
#pragma unroll
        for (int q = 0; q < kHG; q++) {
            __syncthreads();
            red[lane] = g[q];
            __syncthreads();
            if (lane < ni) {
                double s = 0.;
                for (int t = 0; t < S; t++) s += red[lane + ni * t];
                outs[q][i] += s;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Density functor VJP (FP64), hdr_density.hpp:254-363.  Per i-particle the
// forward is recomputed: three h-passes rho_k = h_k^3 sum m W(r h_k),
// H_{k+1} = min(eta kappa (m / rho_k)^(1/3), hmax), with S_k = sum m r^2 t^3
// (so that d rho_k / d h_k = 3 rho_k / h_k - 5 C1 h_k^4 S_k), then the grad-h
// sums at H_3.  The reverse runs the outputs' cotangents back through
// Omega, div v and |curl v| (per particle), down the chain H_3 -> rho_2 -> H_2
// -> rho_1 -> H_1 -> rho_0 -> H_0 (per particle; the derivative by h_3 comes
// from sums of the forward sweep), and through the pair sums of grad-h and of
// the h-passes (one sweep).  Gather lists are not symmetric, so the j-side
// position and velocity cotangents collect in LDS per tile (atomic adds) and
// leave with one global FP64 atomic per record and component.
// A list holds the neighbours of a whole walk, about a fifth of it within
// reach of any one particle: a lane first marks its records of a tile by
// distance and runs the pair terms over the marked ones.  Bound by the latency
// of the sweeps' loads and sums, so registers are held to 128 (4 waves per
// SIMD; 144 as the compiler chose, 5 waves spill) and the sums across slices
// take the tile's LDS.  2x10^5 particles: 0.99 ms with the terms of every
// listed pair and a reverse sweep each for grad-h and the h-passes, 0.68 with
// marks and one reverse sweep, 0.62 so.
// ---------------------------------------------------------------------------
// Square root of r2 >= 0 as sqrt_ieee, with 0 (self pairs) and r2 < 1e-300
// on the same path.
__device__ __forceinline__ double sqrt_r2(double r2)
{
    return sqrt_refine(r2, __builtin_amdgcn_rsq(r2 > 1e-300 ? r2 : 1e-300));
}

struct DRec {
    double x, y, z, m, vx, vy, vz;
};

// Per-i sums over the S slices (fixed order), visible to every lane of the i;
// one loop for all of them, as it is bound by the latency of its LDS reads.
template <int N>
__device__ __forceinline__ void slice_total(double (&v)[N], double *red, int lane, int il, int ni, int S)
{
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; q++) red[q * kWave + lane] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; q++) v[q] = red[q * kWave + il];
#pragma unroll 2
    for (int t = 1; t < S; t++) {
#pragma unroll
        for (int q = 0; q < N; q++) v[q] += red[q * kWave + il + ni * t];
    }
}

__global__ __launch_bounds__(kWave, 4) void density_vjp_kernel(int n_walk, const int32_t *__restrict__ i_off,
                                                            const int32_t *__restrict__ j_off,
                                                            const int32_t *__restrict__ j_idx, sphk_dens_src src,
                                                            double eta_ksrh, double hmax, sphk_dens_cot cot,
                                                            sphk_dens_grad grad)
{
    constexpr double C0 = kCeff0, k5 = -5. * kCeff1;
    // a tile and its cotangents; between sweeps the sums across slices
    __shared__ __attribute__((aligned(16))) char smem[kTile * (sizeof(DRec) + 6 * sizeof(double))];
    __shared__ int32_t sj[kTile];
    DRec *const sp = reinterpret_cast<DRec *>(smem);
    double *const jb = reinterpret_cast<double *>(sp + kTile), *const red = reinterpret_cast<double *>(smem);
    static_assert(10 * kWave * sizeof(double) <= sizeof(smem), "reduction buffer");
    if ((int)blockIdx.x >= n_walk) return;
    const int w = xcd_walk_adj(blockIdx.x, n_walk);
    const int lane = threadIdx.x;
    const int ib = i_off[w], ie = i_off[w + 1];
    const uint32_t kb = j_off[w], ke = j_off[w + 1];

    // one sweep over the walk's list: f(record, k-th slot) per pair of this
    // lane's slice that is not beyond sqrt(R2) of (px, py, pz); with FLUSH the
    // j-side cotangents in jb[0..5][k] go to grad
    auto sweep = [&](auto &&f, double px, double py, double pz, double R2, bool vel, bool flush, int slice, int S) {
        for (uint32_t t0 = kb; t0 < ke; t0 += kTile) {
            const int nt = (int)min((uint32_t)kTile, ke - t0);
            __syncthreads();
            if (lane < nt) {
                const int j = j_idx ? j_idx[t0 + lane] : (int)(t0 + lane);
                sp[lane].x = src.x[j];
                sp[lane].y = src.y[j];
                sp[lane].z = src.z[j];
                sp[lane].m = src.m[j];
                if (vel) {
                    sp[lane].vx = src.vx[j];
                    sp[lane].vy = src.vy[j];
                    sp[lane].vz = src.vz[j];
                }
                sj[lane] = j;
            }
            if (flush)
                for (int q = 0; q < 6; q++) jb[q * kTile + lane] = 0.;
            __syncthreads();
            uint64_t near = 0;
#pragma unroll 4
            for (int k = slice; k < nt; k += S) {
                const double dx = px - sp[k].x, dy = py - sp[k].y, dz = pz - sp[k].z;
                near |= (uint64_t)!(dx * dx + dy * dy + dz * dz >= R2) << k;
            }
            while (near) {
                const int k = __builtin_ctzll(near);
                near &= near - 1;
                f(sp[k], k);
            }
            if (flush) {
                __syncthreads();
                if (lane < nt) {
                    const int j = sj[lane];
                    double *dst[6] = {grad.x, grad.y, grad.z, grad.vx, grad.vy, grad.vz};
                    for (int q = 0; q < 6; q++) {
                        const double v = jb[q * kTile + lane];
                        if (v != 0.) atomicAdd(&dst[q][j], v);
                    }
                }
            }
        }
    };
    // squared radius of every pair that counts at a smoothing length H
    auto reach = [](double H) { return fmax(H * H * (1. + 1e-12), 1e-300); };

    for (int c0 = ib; c0 < ie; c0 += kWave) {
        const int ni = min(kWave, ie - c0);
        const int S = kWave / ni, il = lane % ni;
        const int slice = lane / ni < S ? lane / ni : kTile;   // idle lanes sweep nothing
        const bool lead = lane < ni;
        const int i = c0 + il;
        const double px = src.x[i], py = src.y[i], pz = src.z[i];
        const double pvx = src.vx[i], pvy = src.vy[i], pvz = src.vz[i];
        const double mi = src.m[i];

        // -- forward: three h-passes (rho_k, S_k) and H_{k+1}
        double H[4], rho[3], Sk[3];
        bool capped[4] = {false, false, false, false};
        H[0] = src.ksr[i];
        for (int k = 0; k < 3; k++) {
            const double h = 1. / H[k];
            double v[2] = {0., 0.};
            sweep([&](const DRec &r, int) {
                const double dx = px - r.x, dy = py - r.y, dz = pz - r.z;
                const double r2 = dx * dx + dy * dy + dz * dz;
                const double q = sqrt_r2(r2) * h;
                const double t = q < 1. ? 1. - q : 0.;
                const double t2 = t * t;
                v[0] += r.m * (C0 * t2 * t2 * (1. + 4. * q));
                v[1] += r.m * r2 * (t2 * t);
            }, px, py, pz, reach(H[k]), false, false, slice, S);
            slice_total<2>(v, red, lane, il, ni, S);
            rho[k] = v[0] * (h * h * h);
            Sk[k] = v[1];
            const double hn = eta_ksrh * cbrt_f64(mi / rho[k]);
            capped[k + 1] = !(hn < hmax);
            H[k + 1] = hn < hmax ? hn : hmax;
        }
        // -- forward grad-h sums at H_3
        const double h3 = 1. / H[3];
        const double h3_4 = (h3 * h3) * (h3 * h3), h3_5 = h3_4 * h3;
        // gsum, dvsum, rot x, y, z (dw folded in); then the sums of which
        // d L / d h_3 is made: its weights are known per particle below, so
        // that one reverse sweep serves the grad-h sums and the h-passes
        double fg[10] = {0., 0., 0., 0., 0., 0., 0., 0., 0., 0.};
        sweep([&](const DRec &r, int) {
            const double dx = px - r.x, dy = py - r.y, dz = pz - r.z;
            const double dvx = pvx - r.vx, dvy = pvy - r.vy, dvz = pvz - r.vz;
            const double r2 = dx * dx + dy * dy + dz * dz;
            const double rr = sqrt_r2(r2);
            const double q = rr * h3;
            const double t = q < 1. ? 1. - q : 0.;
            const double t2 = t * t, t3 = t2 * t;
            const double dw = k5 * r.m * h3_5 * t3;
            const double P = 3. + q * (9. - 32. * q), Pp = 9. - 64. * q;
            const double dd = dvx * dx + dvy * dy + dvz * dz;
            const double cx = dvy * dz - dvz * dy, cy = dvz * dx - dvx * dz, cz = dvx * dy - dvy * dx;
            fg[0] += r.m * t3 * P;
            fg[1] += dd * dw;
            fg[2] += cx * dw;
            fg[3] += cy * dw;
            fg[4] += cz * dw;
            const double mt2 = r.m * t2, u = mt2 * (5. * t - 3. * q);
            fg[5] += mt2 * (t * Pp - 3. * P) * rr;
            fg[6] += dd * u;
            fg[7] += cx * u;
            fg[8] += cy * u;
            fg[9] += cz * u;
        }, px, py, pz, reach(H[3]), true, false, slice, S);
        slice_total<10>(fg, red, lane, il, ni, S);
        const double g = -C0 * h3_4 * fg[0];
        const double dvv = -fg[1];
        const double rho2 = rho[2];
        const double B = 1. + H[3] * g / (3. * rho2);
        const double Om = 1. / B;
        const double rotm2 = fg[2] * fg[2] + fg[3] * fg[3] + fg[4] * fg[4];
        const double rotm = rotm2 > 0. ? __builtin_sqrt(rotm2) : 0.;

        // -- reverse through the outputs (per particle)
        const double cD = cot.dens[i], cK = cot.ksr[i], cV = cot.divv[i], cR = cot.rotv[i], cG = cot.grdh[i];
        // a particle whose outputs carry no cotangent contributes nothing;
        // it is skipped outright, so that outputs it does not own (e.g. an
        // empty sum over a list built for other particles: 0 * inf) cannot
        // turn into NaN cotangents of its neighbours
        const bool live = cD != 0. || cK != 0. || cV != 0. || cR != 0. || cG != 0.;
        const double Omb = cG + (cV * dvv + cR * rotm) / rho2;
        double rho2b = cD - (cV * dvv + cR * rotm) * Om / (rho2 * rho2);
        const double A = Om / rho2;
        const double dvsb = -cV * A;   // d L / d dvsum (dv = -dvsum)
        double rb[3] = {0., 0., 0.};
        if (rotm > 0.)
            for (int q = 0; q < 3; q++) rb[q] = cR * A * fg[2 + q] / rotm;
        const double Bb = -Omb * Om * Om;
        double H3b = cK + Bb * g / (3. * rho2);
        const double gb = Bb * H[3] / (3. * rho2);
        rho2b -= Bb * H[3] * g / (3. * rho2 * rho2);
        const double gsb = -C0 * h3_4 * gb;            // d L / d gsum
        double h3b = gb * (-4. * C0 * h3 * h3 * h3 * fg[0]);

        h3b += gsb * fg[5] + k5 * h3_4 * (dvsb * fg[6] + rb[0] * fg[7] + rb[1] * fg[8] + rb[2] * fg[9]);
        H3b += h3b * (-h3 * h3);

        // -- reverse down the smoothing-length chain (per particle)
        double rhob[3];
        rhob[2] = rho2b + (capped[3] ? 0. : H3b * (-H[3] / (3. * rho2)));
        double Hb = 0.;
        for (int k = 2; k >= 0; k--) {
            const double h = 1. / H[k];
            const double drho_dh = 3. * rho[k] / h + k5 * (h * h) * (h * h) * Sk[k];
            Hb = rhob[k] * drho_dh * (-h * h);
            if (k > 0) rhob[k - 1] = capped[k] ? 0. : Hb * (-H[k] / (3. * rho[k - 1]));
        }
        // Hb is now d L / d H_0

        // -- reverse of the pair sums: grad-h, and the three h-passes
        // (positions only)
        double wk[3], hk[3];
        for (int k = 0; k < 3; k++) {
            hk[k] = 1. / H[k];
            const double h2 = hk[k] * hk[k];
            wk[k] = rhob[k] * k5 * (h2 * h2 * hk[k]);   // rho_bar h^5 (-5 C1)
        }
        double gi[6] = {0., 0., 0., 0., 0., 0.};   // x, y, z, vx, vy, vz of i
        sweep([&](const DRec &r, int k) {
            if (!live) return;
            const double dx = px - r.x, dy = py - r.y, dz = pz - r.z;
            const double rr = sqrt_r2(dx * dx + dy * dy + dz * dz);
            double c = 0.;   // along d
            for (int q = 0; q < 3; q++) {
                const double qq = rr * hk[q];
                if (qq < 1.) {
                    const double t = 1. - qq;
                    c += wk[q] * (t * t * t);
                }
            }
            c *= r.m;
            double db[3] = {0., 0., 0.};
            const double q = rr * h3;
            if (q < 1.) {
                const double dvx = pvx - r.vx, dvy = pvy - r.vy, dvz = pvz - r.vz;
                const double t = 1. - q;
                const double t2 = t * t, t3 = t2 * t;
                const double dw = k5 * r.m * h3_5 * t3;
                const double P = 3. + q * (9. - 32. * q), Pp = 9. - 64. * q;
                const double cx = dvy * dz - dvz * dy, cy = dvz * dx - dvx * dz, cz = dvx * dy - dvy * dx;
                const double Sdw = dvsb * (dvx * dx + dvy * dy + dvz * dz) + rb[0] * cx + rb[1] * cy + rb[2] * cz;
                // explicit d and dv terms
                db[0] = dw * (dvsb * dvx + (rb[1] * dvz - rb[2] * dvy));
                db[1] = dw * (dvsb * dvy + (rb[2] * dvx - rb[0] * dvz));
                db[2] = dw * (dvsb * dvz + (rb[0] * dvy - rb[1] * dvx));
                const double vb[3] = {dw * (dvsb * dx + (dy * rb[2] - dz * rb[1])),
                                      dw * (dvsb * dy + (dz * rb[0] - dx * rb[2])),
                                      dw * (dvsb * dz + (dx * rb[1] - dy * rb[0]))};
                // d L / d q: through gsum's m t^3 P(q) and through dw (t = 1 - q)
                const double qb = gsb * r.m * t2 * (t * Pp - 3. * P) - 3. * Sdw * k5 * r.m * h3_5 * t2;
                if (rr > 0.) c += qb * h3 * rcp_f64(rr);
                gi[3] += vb[0];
                gi[4] += vb[1];
                gi[5] += vb[2];
                atomicAdd(&jb[3 * kTile + k], -vb[0]);
                atomicAdd(&jb[4 * kTile + k], -vb[1]);
                atomicAdd(&jb[5 * kTile + k], -vb[2]);
            }
            db[0] += c * dx;
            db[1] += c * dy;
            db[2] += c * dz;
            gi[0] += db[0];
            gi[1] += db[1];
            gi[2] += db[2];
            atomicAdd(&jb[0 * kTile + k], -db[0]);
            atomicAdd(&jb[1 * kTile + k], -db[1]);
            atomicAdd(&jb[2 * kTile + k], -db[2]);
        }, px, py, pz, live ? reach(fmax(fmax(H[0], H[1]), fmax(H[2], H[3]))) : -1., true, true, slice, S);

        // -- i-side totals
        slice_total<6>(gi, red, lane, il, ni, S);
        if (lead && live) {
            atomicAdd(&grad.x[i], gi[0]);
            atomicAdd(&grad.y[i], gi[1]);
            atomicAdd(&grad.z[i], gi[2]);
            atomicAdd(&grad.vx[i], gi[3]);
            atomicAdd(&grad.vy[i], gi[4]);
            atomicAdd(&grad.vz[i], gi[5]);
            grad.ksr[i] += Hb;
        }
    }
}

}  // namespace
}  // namespace sphk

extern "C" int sphk_density_vjp_dev(sphk_ctx *ctx, int n_walk, const int32_t *i_off, const int32_t *j_off,
                                    const int32_t *j_idx, sphk_dens_src src, sphk_dens_cot cot,
                                    sphk_dens_grad grad, void *stream)
{
    using sphk::set_error;
    if (!ctx) return set_error(SPHK_E_ARG, "density_vjp: null context");
    if (n_walk < 0 || (n_walk > 0 && (!i_off || !j_off))) return set_error(SPHK_E_ARG, "density_vjp: bad walks");
    if (n_walk == 0) return SPHK_OK;
    const void *in[] = {src.id, src.m, src.x, src.y, src.z, src.vx, src.vy, src.vz, src.ksr,
                        cot.dens, cot.ksr, cot.divv, cot.rotv, cot.grdh,
                        grad.x, grad.y, grad.z, grad.vx, grad.vy, grad.vz, grad.ksr};
    for (const void *q : in)
        if (!q) return set_error(SPHK_E_ARG, "density_vjp: null pointer");
    sphk_params p;
    const int rc = sphk_get_params(ctx, &p);
    if (rc) return rc;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(sphk::density_vjp_kernel, dim3(n_walk), dim3(sphk::kWave), 0, st, n_walk, i_off, j_off,
                       j_idx, src, p.eta * p.ksrh, p.hmax, cot, grad);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(SPHK_E_DEVICE, "density_vjp: %s", hipGetErrorString(e));
    return SPHK_OK;
}

extern "C" int sphk_hydro_vjp_dev(sphk_ctx *ctx, int n_walk, const int32_t *i_off, const int32_t *j_off,
                                  const int32_t *j_idx, sphk_hydro_src src, sphk_hydro_out cot,
                                  sphk_hydro_grad grad, void *stream)
{
    using sphk::set_error;
    if (!ctx) return set_error(SPHK_E_ARG, "hydro_vjp: null context");
    if (n_walk < 0 || (n_walk > 0 && (!i_off || !j_off))) return set_error(SPHK_E_ARG, "hydro_vjp: bad walks");
    if (n_walk == 0) return SPHK_OK;
    const void *in[] = {src.id, src.m, src.x, src.y, src.z, src.vx, src.vy, src.vz, src.hinv, src.pres,
                        src.presc, src.bswt, src.dens, src.vsnd, src.alph, src.alphu, src.thrm, src.eta,
                        cot.ax, cot.ay, cot.az, cot.udot, cot.diffu, cot.gx, cot.gy, cot.gz,
                        grad.x, grad.y, grad.z, grad.vx, grad.vy, grad.vz, grad.hinv, grad.pres, grad.presc,
                        grad.bswt, grad.dens, grad.vsnd, grad.alph, grad.alphu, grad.thrm, grad.eta};
    for (const void *q : in)
        if (!q) return set_error(SPHK_E_ARG, "hydro_vjp: null pointer");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(sphk::hydro_vjp_kernel, dim3(n_walk), dim3(sphk::kWave), 0, st, n_walk, i_off, j_off, j_idx,
                       src, cot, grad);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(SPHK_E_DEVICE, "hydro_vjp: %s", hipGetErrorString(e));
    return SPHK_OK;
}

namespace {
// Checks and launch of both gravity VJP entries; packed: gx and nx are [.][3]
// arrays and the other four outputs are not used.
int gravity_vjp(bool packed, sphk_ctx *ctx, int n_walk, const int32_t *i_off, const int32_t *j_off,
                const int32_t *j_idx, const sphk_grav_src &pj, const int32_t *s_off, const int32_t *s_idx,
                const sphk_grav_src &ps, const sphk_grav_src &pi, double e2, const double *abx, const double *aby,
                const double *abz, const double *pbar, const double *ebar, double *gx, double *gy, double *gz,
                double *nx, double *ny, double *nz, void *stream)
{
    using sphk::set_error;
    if (!ctx) return set_error(SPHK_E_ARG, "gravity_vjp: null context");
    if (n_walk < 0 || (n_walk > 0 && (!i_off || !j_off))) return set_error(SPHK_E_ARG, "gravity_vjp: bad walks");
    if (n_walk == 0) return SPHK_OK;
    if (!pi.x || !pi.y || !pi.z || !pj.m || !pj.x || !pj.y || !pj.z || !abx || !aby || !abz || !pbar || !gx ||
        (!packed && (!gy || !gz)))
        return set_error(SPHK_E_ARG, "gravity_vjp: null pointer");
    if (s_off && (!ps.m || !ps.x || !ps.y || !ps.z || !nx || (!packed && (!ny || !nz))))
        return set_error(SPHK_E_ARG, "gravity_vjp: null SPJ pointer");
    if (!(e2 > 0.)) return set_error(SPHK_E_ARG, "gravity_vjp: softening must be positive");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (packed)
        hipLaunchKernelGGL(sphk::gravity_vjp_kernel<true>, dim3(n_walk), dim3(sphk::kWave), 0, st, n_walk, i_off,
                           j_off, j_idx, pj, s_off, s_idx, ps, pi, e2, abx, aby, abz, pbar, ebar, gx, gy, gz, nx, ny,
                           nz);
    else
        hipLaunchKernelGGL(sphk::gravity_vjp_kernel<false>, dim3(n_walk), dim3(sphk::kWave), 0, st, n_walk, i_off,
                           j_off, j_idx, pj, s_off, s_idx, ps, pi, e2, abx, aby, abz, pbar, ebar, gx, gy, gz, nx, ny,
                           nz);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(SPHK_E_DEVICE, "gravity_vjp: %s", hipGetErrorString(e));
    return SPHK_OK;
}
}  // namespace

extern "C" int sphk_gravity_vjp_dev(sphk_ctx *ctx, int n_walk, const int32_t *i_off, const int32_t *j_off,
                                    const int32_t *j_idx, sphk_grav_src pj, const int32_t *s_off,
                                    const int32_t *s_idx, sphk_grav_src ps, sphk_grav_src pi, double e2,
                                    const double *abx, const double *aby, const double *abz,
                                    const double *pbar, const double *ebar, double *gx, double *gy,
                                    double *gz, double *nx, double *ny, double *nz, void *stream)
{
    return gravity_vjp(false, ctx, n_walk, i_off, j_off, j_idx, pj, s_off, s_idx, ps, pi, e2, abx, aby, abz, pbar,
                       ebar, gx, gy, gz, nx, ny, nz, stream);
}

extern "C" int sphk_gravity_vjp_packed_dev(sphk_ctx *ctx, int n_walk, const int32_t *i_off, const int32_t *j_off,
                                           const int32_t *j_idx, sphk_grav_src pj, const int32_t *s_off,
                                           const int32_t *s_idx, sphk_grav_src ps, sphk_grav_src pi, double e2,
                                           const double *abx, const double *aby, const double *abz,
                                           const double *pbar, const double *ebar, double *g3, double *n3,
                                           void *stream)
{
    return gravity_vjp(true, ctx, n_walk, i_off, j_off, j_idx, pj, s_off, s_idx, ps, pi, e2, abx, aby, abz, pbar,
                       ebar, g3, nullptr, nullptr, n3, nullptr, nullptr, stream);
}
