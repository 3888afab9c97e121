// pme.hip -- smooth PME reciprocal space on the device.
//
// Follows NonbondedForce::ReciprocalPMEcalculateForcesAndEnergy
// (core/baseline/src/Forces/NonbondedForce.cpp:467-499): fractional index
// and offset from the origin (:51-71), order-5 B-splines by the standard
// recursion (:150-181), charge spreading (:220-260), forward 3D FFT, the
// influence-function convolution and energy (:323-388), backward FFT and the
// force gather (:407-461).
//
// The reference runs a full complex-to-complex FFTW transform of a real grid.
// Here the spread grid is real, so the forward transform is real-to-complex
// onto the half spectrum [Kx][Ky][Kz/2+1] and the backward one complex-to-
// real; by Hermitian symmetry this is the same result (the reference keeps
// only the real part after its backward transform).  Five passes:
//   Z  : the charges spread to rows in LDS (there is no charge grid in memory),
//        R2C along z;
//   Y  : C2C along y on tiles of consecutive kz (coalesced rows);
//   X  : C2C along x, multiply by the influence function eta(k) and sum the
//        energy, inverse C2C along x -- fused so the spectrum makes one trip;
//   Y' : inverse C2C along y;
//   Z' : C2R along z into the real potential grid.
// Z with Y, and Y' with Z', are one kernel each where planes fit in LDS.  Each
// line FFT is a Stockham autosort transform in LDS (fft_lines) with twiddles from
// a per-axis table exp(-2 pi i t / K) computed on the host in FP64.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "nx_terms.h"

namespace nx {

template <typename real>
__device__ __forceinline__ void bspline5(real dr, real* th, real* dth) {
    // NonbondedForce.cpp:150-181 with pmeOrder = 5
    th[4] = 0;
    th[1] = dr;
    th[0] = 1 - dr;
#pragma unroll
    for (int k = 3; k < 5; ++k) {
        const real div = (real)1.0 / (real)(k - 1.0);
        th[k - 1] = div * dr * th[k - 2];
#pragma unroll
        for (int l = 1; l < (k - 1); ++l)
            th[k - l - 1] = div * ((dr + l) * th[k - l - 2] + (k - l - dr) * th[k - l - 1]);
        th[0] = div * (1 - dr) * th[0];
    }
    dth[0] = -th[0];
#pragma unroll
    for (int k = 1; k < 5; ++k) dth[k] = th[k - 1] - th[k];
    const real div = (real)1.0 / (real)4.0;
    th[4] = div * dr * th[3];
#pragma unroll
    for (int l = 1; l < 4; ++l) th[4 - l] = div * ((dr + l) * th[4 - l - 1] + (5 - l - dr) * th[4 - l]);
    th[0] = div * (1 - dr) * th[0];
}

template <typename real>
__device__ __forceinline__ void grid_index(real x, double invL, int K, int& idx, real& fr) {
    real t = x * (real)invL;
    t = (t - floor(t)) * (real)K;
    if (!(t >= (real)0)) t = 0;
    int ti = (int)t;
    fr = t - (real)ti;
    idx = ti >= K ? ti - K : ti;     // t is in [0, K]
}

// The charge grid is fixed point in both paths (exact, order-free sums): 2^32
// in the mixed path (FP32 contributions), 2^48 in the FP64 path.  A grid
// value is a sum of q w over the atoms within 2.5 grid spacings, a few units
// at most, far inside the FP64 range of +-32768; the resolution, 3.6e-15 per
// contribution, keeps the reciprocal forces within ~1e-12 of their double
// sums (at 2^40 positive and negative charges cancelling on a point left
// 2e-10 relative RMS in the total force).
__device__ __forceinline__ long long grid_fixed(float v) { return to_fixed(v); }
__device__ __forceinline__ long long grid_fixed(double v) {
    double s = v * PrecFP64::grid_scale;
    s = fmin(fmax(s, -9.2e18), 9.2e18);
    return (long long)rint(s);
}
// LDS accumulation (a ds_add_u64)
__device__ __forceinline__ void lds_add(long long* g, long long v) {
    atomicAdd(reinterpret_cast<unsigned long long*>(g), static_cast<unsigned long long>(v));
}
// grid_fixed(v) for |v| below grid_fixed_small: v scaled and added to 1.5 2^52 in
// FP64 is rounded to an integer in the low bits of the sum, three instructions
// where the 64-bit conversion takes about 18.  The same integer: both round to
// nearest, ties to even.
template <class P>
constexpr double grid_fixed_small = 2251799813685248.0 / P::grid_scale;     // 2^51 units
template <class P>
__device__ __forceinline__ long long grid_fixed_fast(typename P::real v) {
    return __double_as_longlong(fma((double)v, P::grid_scale, 6755399441055744.0)) - 0x4338000000000000ll;
}

// Quotient of non-negative integers n, d with n + d < 2^22 through a float
// reciprocal: (n + 0.5) / d is at least 0.5 / d away from an integer, and the
// two roundings (of 1/d and of the product) move it by at most
// (n / d + 1) 2^-23, which is less.
__device__ __forceinline__ int qdiv(int n, float inv_d) { return (int)(((float)n + 0.5f) * inv_d); }

// Charge spreading by ownership.  A workgroup owns ny rows (y0, y0 + 1, ..) of
// one x plane of the grid, every z: it finds the atoms whose stencils touch
// them, adds their points in LDS (fixed point: exact, whatever the order) and
// goes on to the z transform with the sums in place.  No charge grid in global
// memory: nothing is cleared, added atomically or read back.  Each atom is
// visited by the five planes of its stencil, 25 points in each.  (Tiles that
// owned atoms, with every tile's halo added to a global grid, took 35 us alone
// on 100,000 atoms at 96^3 and 565 us at 128^3, where the halos made 20 million
// global atomics; the transform then read and cleared the grid.)
//
// The candidates are the slots of the neighbour-list columns the rows' atoms
// were binned into at the last build, widened by the distance an atom may have
// moved since: column cx of x is a contiguous range of slots, and so is a range
// of columns cy in it.  A wavefront takes 64 candidates at a time, keeps those
// that touch its rows in a queue of its own, and spreads 64 of them at once.
struct SpreadArgs {
    const SysCount* sc;     // by system
    const int* col_count;
    const int* col_slot;
};

template <class P>
__device__ __forceinline__ void spread_rows(const SysDev& d, const SpreadArgs& a,
                                            const typename P::real4* __restrict__ pos, int x, int y0, int ny, int* lds,
                                            long long* g) {
    using real = typename P::real;
    const int Kx = d.grid[0], Ky = d.grid[1], Kz = d.grid[2];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    int* seg_slot = lds;                          // first slot of each segment
    int* seg_end = lds + kSpreadSegs;             // past its last slot
    int* seg_chunk = lds + 2 * kSpreadSegs;       // its first chunk of 64 slots; the total at [n_seg]
    int* n_seg = lds + 3 * kSpreadSegs + 1;
    int* queue = lds + 3 * kSpreadSegs + 2 + wv * 128;
    // rows are Kz + 4 long: a stencil runs past the end, and the reader folds the
    // last four points onto the first (no wrapped index in the inner loop)
    const int ls = Kz + 4;
    for (int i = threadIdx.x; i < ny * ls; i += blockDim.x) g[i] = 0ll;
    if (wv == 0) {
        // columns of x (and y) that can hold an atom of these rows: stencils start
        // at most four points before a row
        const double hx = d.L[0] / Kx, hy = d.L[1] / Ky, m = d.sp_margin;
        int xa = (int)floor(((x - 4) * hx - m) / d.colw[0]), nx = (int)floor(((x + 1) * hx + m) / d.colw[0]) - xa + 1;
        int ya = (int)floor(((y0 - 4) * hy - m) / d.colw[1]), nyc = (int)floor(((y0 + ny) * hy + m) / d.colw[1]) - ya + 1;
        if (nx >= d.ncx) { xa = 0; nx = d.ncx; }
        // whole columns of x when the rows need them (or there are too many for the table)
        const bool whole = nyc >= d.ncy || nx * 2 > kSpreadSegs;
        if (xa < 0) xa += d.ncx;
        if (ya < 0) ya += d.ncy;
        int slot = 0, len = 0, n;
        if (whole) {
            // lane 0: columns xa .. of x, lane 1: those past the last, wrapped
            n = xa + nx > d.ncx ? 2 : 1;
            const int c0 = lane == 0 ? xa : 0, c1 = lane == 0 ? min(xa + nx, d.ncx) : xa + nx - d.ncx;
            if (lane < n) {
                const int last = d.col_off + c1 * d.ncy - 1;
                slot = a.col_slot[d.col_off + c0 * d.ncy];
                len = a.col_slot[last] + ((a.col_count[last] + 7) & ~7) - slot;
            }
        } else {
            const int parts = ya + nyc > d.ncy ? 2 : 1;
            n = nx * parts;
            if (lane < n) {
                int cx = xa + lane / parts;
                if (cx >= d.ncx) cx -= d.ncx;
                const int c0 = lane % parts == 0 ? ya : 0;
                const int c1 = lane % parts == 0 ? min(ya + nyc, d.ncy) : ya + nyc - d.ncy;
                const int first = d.col_off + cx * d.ncy + c0, last = d.col_off + cx * d.ncy + c1 - 1;
                slot = a.col_slot[first];
                len = a.col_slot[last] + ((a.col_count[last] + 7) & ~7) - slot;
            }
        }
        const int chunks = (len + 63) >> 6;
        int incl = chunks;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o);
            if (lane >= o) incl += t;
        }
        if (lane < n) {
            seg_slot[lane] = slot;
            seg_end[lane] = slot + len;
            seg_chunk[lane] = incl - chunks;
        }
        if (lane == n - 1) {
            seg_chunk[n] = incl;
            *n_seg = n;
        }
    }
    __syncthreads();
    const int ns = *n_seg, total = seg_chunk[ns];
    auto spread = [&](int slot) {
        const typename P::real4 p = pos[slot];
        // every weight is below 1, so a charge below the bound keeps its products so
        const bool small = fabs(p.w) < (real)grid_fixed_small<P>;
        int i0, i1, i2;
        real f0, f1, f2;
        grid_index<real>(p.x, d.invL[0], Kx, i0, f0);
        grid_index<real>(p.y, d.invL[1], Ky, i1, f1);
        grid_index<real>(p.z, d.invL[2], Kz, i2, f2);
        real tx[5], ty[5], tz[5], dt[5];
        bspline5<real>(f0, tx, dt);
        bspline5<real>(f1, ty, dt);
        bspline5<real>(f2, tz, dt);
        int ix = x - i0;
        if (ix < 0) ix += Kx;
        real qx = p.w * tx[0];
#pragma unroll
        for (int k = 1; k < 5; ++k)
            if (ix == k) qx = p.w * tx[k];
        int y = i1 - y0;
        if (y < 0) y += Ky;
        long long* row = g + y * ls + i2;
#pragma unroll
        for (int iy = 0; iy < 5; ++iy) {
            if (y < ny) {
                const real qxy = qx * ty[iy];
                if (small) {
#pragma unroll
                    for (int iz = 0; iz < 5; ++iz) lds_add(row + iz, grid_fixed_fast<P>(qxy * tz[iz]));
                } else {
                    for (int iz = 0; iz < 5; ++iz) lds_add(row + iz, grid_fixed(qxy * tz[iz]));
                }
            }
            const bool last = y + 1 == Ky;
            y = last ? 0 : y + 1;
            row += last ? (1 - Ky) * ls : ls;
        }
    };
    int nq = 0;
    // the slot of this lane's candidate in chunk c (-1: none) and, loaded while the
    // chunk before it is worked on, its position
    auto candidate = [&](int c) {
        if (c >= total) return -1;
        int s = 0;
        while (s + 1 < ns && seg_chunk[s + 1] <= c) ++s;
        const int slot = seg_slot[s] + (c - seg_chunk[s]) * 64 + lane;
        return slot < seg_end[s] ? slot : -1;
    };
    int slot_n = candidate(wv);
    typename P::real4 p_n;
    if (slot_n >= 0) p_n = pos[slot_n];
    for (int c = wv; c < total; c += nw) {
        const int slot = slot_n;
        const typename P::real4 p = p_n;
        slot_n = candidate(c + nw);
        if (slot_n >= 0) p_n = pos[slot_n];
        bool hit = false;
        if (slot >= 0) {
            int i0, i1;
            real f;
            grid_index<real>(p.x, d.invL[0], Kx, i0, f);
            grid_index<real>(p.y, d.invL[1], Ky, i1, f);
            int ix = x - i0, y = i1 - y0;
            if (ix < 0) ix += Kx;
            if (y < 0) y += Ky;
            hit = p.x < (real)(0.5 * kPadPos) && ix < 5 && (y < ny || y + 4 >= Ky);
        }
        const unsigned long long m = __ballot(hit);
        if (hit) queue[nq + __popcll(m & ((1ull << lane) - 1ull))] = slot;
        nq += __popcll(m);
        wave_lds_sync();
        if (nq >= 64) {
            spread(queue[lane]);
            nq -= 64;
            if (lane < nq) queue[lane] = queue[64 + lane];
            wave_lds_sync();
        }
    }
    if (lane < nq) spread(queue[lane]);
    __syncthreads();
}

// Force from the potential grid (NonbondedForce.cpp:407-461).  A block of
// 5 wavefronts covers 64 slots: wavefront ix takes stencil plane i0 + ix of
// every slot (25 points per lane instead of 125, five times the loads in
// flight), and the five partial gradients are summed in LDS in plane order.
// The loads bound it: the lanes' stencils start anywhere, so a load costs by the
// cache lines its lanes touch, not by the bytes.  A row of the stencil is
// therefore read as four points and one instead of point by point, which the
// rows' copied first points (kPhiPad) allow at any start: on 10^6 atoms, 200^3
// points, 165 -> 92 us; on 10^5 atoms and 96^3, 24 -> 15 us (FP64 29 -> 26 us).
// Staging the points under a super-cluster in LDS first cost more than it saved.
constexpr int kGatherSlots = 64;

// Five consecutive points of a row of the potential, at the alignment of one.
template <typename real>
struct Row5 {
    using V = typename std::conditional<sizeof(real) == 4, float, double>::type __attribute__((ext_vector_type(4)));
    struct __attribute__((packed, aligned(sizeof(real)))) { V v; } head;
    real tail;
    __device__ __forceinline__ real at(int k) const { return k < 4 ? head.v[k] : tail; }
};

template <class P>
__global__ __launch_bounds__(5 * kGatherSlots, 5) void pme_gather_kernel(const SysDev* __restrict__ sd,
                                                                     const SysCount* __restrict__ sc,
                                                                     const int* __restrict__ slot_sys,
                                                                     const int* __restrict__ atom_of_slot,
                                                                     const typename P::real4* __restrict__ pos,
                                                                     const typename P::real* __restrict__ phi,
                                                                     typename P::facc* FX, typename P::facc* FY,
                                                                     typename P::facc* FZ, int n_slots_total,
                                                                     int atom_blocks, TermArgs<P> terms) {
    side_priority();
    // the atom forces' blocks first: theirs is the longer chain of loads (the last
    // ones, FP64, 100,000 atoms: a step 5 us longer)
    if ((int)blockIdx.x < atom_blocks) {
        const int a = (int)blockIdx.x * (5 * kGatherSlots) + (int)threadIdx.x;
        atom_force<P, false>(terms, a, nullptr);
        return;
    }
    using real = typename P::real;
    __shared__ real part[3][5][kGatherSlots];
    const int ix = threadIdx.x / kGatherSlots, l = threadIdx.x - ix * kGatherSlots;
    const int slot = ((int)blockIdx.x - atom_blocks) * kGatherSlots + l;
    bool on = slot < n_slots_total;
    int s = 0;
    if (on) {
        s = slot_sys[slot];
        on = slot - sd[s].slot_off < sc[s].n_slots && !sc[s].overflow && atom_of_slot[slot] >= 0 &&
             sd[s].grid[0] != 0;
    }
    real fx = 0, fy = 0, fz = 0;
    typename P::real4 p;
    if (on) {
        const SysDev& d = sd[s];
        p = pos[slot];
        const int Kx = d.grid[0], Ky = d.grid[1], Kz = d.grid[2];
        int i0, i1, i2;
        real f0, f1, f2;
        grid_index<real>(p.x, d.invL[0], Kx, i0, f0);
        grid_index<real>(p.y, d.invL[1], Ky, i1, f1);
        grid_index<real>(p.z, d.invL[2], Kz, i2, f2);
        real tx[5], dtx[5], ty[5], dty[5], tz[5], dtz[5];
        bspline5<real>(f0, tx, dtx);
        bspline5<real>(f1, ty, dty);
        bspline5<real>(f2, tz, dtz);
        // stencil indices, periodic (i + t < 2K: one conditional subtraction, no division)
        const int xi = (i0 + ix >= Kx) ? i0 + ix - Kx : i0 + ix;
        const int pitch = Kz + kPhiPad;
        const real* g = phi + d.rgrid_off + (long long)xi * Ky * pitch + i2;
        real tix = tx[0], dtix = dtx[0];
#pragma unroll
        for (int k = 1; k < 5; ++k)
            if (ix == k) { tix = tx[k]; dtix = dtx[k]; }
#pragma unroll
        for (int iy = 0; iy < 5; ++iy) {
            const int yi = (i1 + iy >= Ky) ? i1 + iy - Ky : i1 + iy;
            const Row5<real> v = *reinterpret_cast<const Row5<real>*>(g + yi * pitch);
            const real a = dtix * ty[iy], b = tix * dty[iy], c = tix * ty[iy];
            real s = 0, ds = 0;
#pragma unroll
            for (int iz = 0; iz < 5; ++iz) {
                s += tz[iz] * v.at(iz);
                ds += dtz[iz] * v.at(iz);
            }
            fx += a * s;
            fy += b * s;
            fz += c * ds;
        }
    }
    part[0][ix][l] = fx;
    part[1][ix][l] = fy;
    part[2][ix][l] = fz;
    __syncthreads();
    if (ix == 0 && on) {
        const SysDev& d = sd[s];
        real gx = 0, gy = 0, gz = 0;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            gx += part[0][k][l];
            gy += part[1][k][l];
            gz += part[2][k][l];
        }
        const real q = p.w;
        facc_add(&FX[slot], -q * (gx * (real)d.grid[0] * (real)d.invL[0]));
        facc_add(&FY[slot], -q * (gy * (real)d.grid[1] * (real)d.invL[1]));
        facc_add(&FZ[slot], -q * (gz * (real)d.grid[2] * (real)d.invL[2]));
    }
}

// ------------------------------------------------------------------ FFT

template <typename R2>
__device__ __forceinline__ R2 cmul(R2 a, R2 b) {
    R2 r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    return r;
}

// DFT of R points in registers; SIGN -1 forward, +1 backward.
template <int R, int SIGN, typename R2>
__device__ __forceinline__ void dft(R2* v) {
    using real = decltype(v->x);
    constexpr real sg = (real)SIGN;
    if constexpr (R == 2) {
        const R2 a = v[0], b = v[1];
        v[0].x = a.x + b.x; v[0].y = a.y + b.y;
        v[1].x = a.x - b.x; v[1].y = a.y - b.y;
    } else if constexpr (R == 3) {
        constexpr real c1 = (real)-0.5, s1 = sg * (real)0.86602540378443864676;
        const R2 a0 = v[0], a1 = v[1], a2 = v[2];
        const R2 sm = {a1.x + a2.x, a1.y + a2.y}, df = {a1.x - a2.x, a1.y - a2.y};
        const R2 t = {a0.x + c1 * sm.x, a0.y + c1 * sm.y};
        // i * s1 * df = (-s1 df.y, s1 df.x)
        v[0].x = a0.x + sm.x; v[0].y = a0.y + sm.y;
        v[1].x = t.x - s1 * df.y; v[1].y = t.y + s1 * df.x;
        v[2].x = t.x + s1 * df.y; v[2].y = t.y - s1 * df.x;
    } else if constexpr (R == 4) {
        const R2 s02 = {v[0].x + v[2].x, v[0].y + v[2].y}, d02 = {v[0].x - v[2].x, v[0].y - v[2].y};
        const R2 s13 = {v[1].x + v[3].x, v[1].y + v[3].y}, d13 = {v[1].x - v[3].x, v[1].y - v[3].y};
        const R2 wd = {-sg * d13.y, sg * d13.x};         // +-i (v1 - v3)
        v[0].x = s02.x + s13.x; v[0].y = s02.y + s13.y;
        v[2].x = s02.x - s13.x; v[2].y = s02.y - s13.y;
        v[1].x = d02.x + wd.x;  v[1].y = d02.y + wd.y;
        v[3].x = d02.x - wd.x;  v[3].y = d02.y - wd.y;
    } else if constexpr (R == 5) {
        constexpr real c1 = (real)0.30901699437494742410, c2 = (real)-0.80901699437494742410;
        constexpr real s1 = sg * (real)0.95105651629515357212, s2 = sg * (real)0.58778525229247312917;
        const R2 a0 = v[0], a1 = v[1], a2 = v[2], a3 = v[3], a4 = v[4];
        const R2 b1 = {a1.x + a4.x, a1.y + a4.y}, b4 = {a1.x - a4.x, a1.y - a4.y};
        const R2 b2 = {a2.x + a3.x, a2.y + a3.y}, b3 = {a2.x - a3.x, a2.y - a3.y};
        const R2 t1 = {a0.x + c1 * b1.x + c2 * b2.x, a0.y + c1 * b1.y + c2 * b2.y};
        const R2 t2 = {a0.x + c2 * b1.x + c1 * b2.x, a0.y + c2 * b1.y + c1 * b2.y};
        // u1 = s1 b4 + s2 b3, u2 = s2 b4 - s1 b3 ; X1 = t1 + i u1, X4 = t1 - i u1, X2 = t2 + i u2, X3 = t2 - i u2
        const R2 u1 = {s1 * b4.x + s2 * b3.x, s1 * b4.y + s2 * b3.y};
        const R2 u2 = {s2 * b4.x - s1 * b3.x, s2 * b4.y - s1 * b3.y};
        v[0].x = a0.x + b1.x + b2.x; v[0].y = a0.y + b1.y + b2.y;
        v[1].x = t1.x - u1.y; v[1].y = t1.y + u1.x;
        v[4].x = t1.x + u1.y; v[4].y = t1.y - u1.x;
        v[2].x = t2.x - u2.y; v[2].y = t2.y + u2.x;
        v[3].x = t2.x + u2.y; v[3].y = t2.y - u2.x;
    } else {
        static_assert(R == 8, "radix");
        constexpr real h = (real)0.70710678118654752440;
        R2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        dft<4, SIGN>(e);
        dft<4, SIGN>(o);
        // o[k] times exp(SIGN i pi k / 4)
        const R2 o1 = {h * (o[1].x - sg * o[1].y), h * (o[1].y + sg * o[1].x)};
        const R2 o2 = {-sg * o[2].y, sg * o[2].x};
        const R2 o3 = {-h * (o[3].x + sg * o[3].y), h * (sg * o[3].x - o[3].y)};
        v[0].x = e[0].x + o[0].x; v[0].y = e[0].y + o[0].y;
        v[4].x = e[0].x - o[0].x; v[4].y = e[0].y - o[0].y;
        v[1].x = e[1].x + o1.x;   v[1].y = e[1].y + o1.y;
        v[5].x = e[1].x - o1.x;   v[5].y = e[1].y - o1.y;
        v[2].x = e[2].x + o2.x;   v[2].y = e[2].y + o2.y;
        v[6].x = e[2].x - o2.x;   v[6].y = e[2].y - o2.y;
        v[3].x = e[3].x + o3.x;   v[3].y = e[3].y + o3.y;
        v[7].x = e[3].x - o3.x;   v[7].y = e[3].y - o3.y;
    }
}

// Copies the N twiddles of an axis into LDS (all threads of the block).
template <typename R2>
__device__ __forceinline__ void load_twiddles(R2* dst, const R2* __restrict__ src, int N) {
    for (int i = threadIdx.x; i < N; i += blockDim.x) dst[i] = src[i];
}

// FFTs of `lines` lines of N points by a block: Stockham autosort, unnormalised,
// the radices in `plan` (fft_plan).  `tw` holds exp(-2 pi i m / N), m < N, in LDS.
//
// The passes are bound by their trips through LDS and by the barriers between
// them, so the radices go up to 8 (64 points in two stages, 96 in three), the
// first stage takes its points from load(m, l) -- global memory, mostly -- and the
// last one gives them to store(buf, m, l, v), and between stages point m of line l
// stands at [m * pitch + l] with the threads running over the lines: no bank
// conflicts, and one twiddle read serves all lines.  (Radices up to 5, every line's
// points side by side, and copies into and out of LDS before: the passes after the
// spread's took 23.4 us alone at 64^3, 36.8 at 96^3, 209 at 200^3, FP64 57 at 96^3;
// now 15.0, 21.7, 122 and 39.6.)  FAST_IN / FAST_OUT run the
// threads of the first / last stage over the points instead, where those are
// consecutive in memory; an odd pitch then keeps the LDS side free of conflicts.
//
// Buffers: stages alternate, the first into b0, the next into b1; store gets the
// one that would be next.  With Ns > 1 (a power product of radices already done)
// the points stand in b1 and `load` is not called.  Returns the buffer after the
// last stage, without a barrier.
template <int R, int SIGN, bool FAST_IN, bool FAST_OUT, typename R2, class Load, class Store>
__device__ __forceinline__ void fft_stage(int Ns, int step, int lines, int pitch, bool first, bool last, const R2* tw,
                                          const R2* src, R2* dst, Load& load, Store& store) {
    const int nb = step * Ns, total = nb * lines;      // nb butterflies a line
    const bool fast = (FAST_IN && first) || (FAST_OUT && last);
    const int inner = fast ? nb : lines;
    const float inv_inner = 1.0f / (float)inner, inv_ns = 1.0f / (float)Ns;
    for (int w = threadIdx.x; w < total; w += blockDim.x) {
        const int outer = qdiv(w, inv_inner), in = w - outer * inner;
        const int j = fast ? in : outer, l = fast ? outer : in;
        R2 v[R];
        int k = 0, base = j * R;
        if (first) {
#pragma unroll
            for (int q = 0; q < R; ++q) v[q] = load(j + q * nb, l);
        } else {
            const int jq = qdiv(j, inv_ns);
            k = j - jq * Ns;
            base = jq * Ns * R + k;
#pragma unroll
            for (int q = 0; q < R; ++q) v[q] = src[(j + q * nb) * pitch + l];
#pragma unroll
            for (int q = 1; q < R; ++q) {
                R2 t = tw[k * q * step];     // k q step < N
                if (SIGN > 0) t.y = -t.y;
                v[q] = cmul(v[q], t);
            }
        }
        dft<R, SIGN>(v);
        if (last) {
#pragma unroll
            for (int q = 0; q < R; ++q) store(dst, base + q * Ns, l, v[q]);
        } else {
#pragma unroll
            for (int q = 0; q < R; ++q) dst[(base + q * Ns) * pitch + l] = v[q];
        }
    }
}

// fn(radix) with the radix a compile-time constant.
template <class Fn>
__device__ __forceinline__ void with_radix(int r, Fn&& fn) {
    if (r == 8) fn(std::integral_constant<int, 8>{});
    else if (r == 4) fn(std::integral_constant<int, 4>{});
    else if (r == 5) fn(std::integral_constant<int, 5>{});
    else if (r == 3) fn(std::integral_constant<int, 3>{});
    else fn(std::integral_constant<int, 2>{});
}

template <int SIGN, bool FAST_IN, bool FAST_OUT, typename R2, class Load, class Store>
__device__ __forceinline__ R2* fft_lines(int N, unsigned plan, int lines, int pitch, const R2* tw, R2* b0, R2* b1, int Ns,
                                         Load load, Store store) {
    R2* src = b1;
    R2* dst = b0;
    int rem = N / Ns;
    while (plan) {
        const int r = plan & 15;
        plan >>= 4;
        const bool first = Ns == 1, last = plan == 0;
        int step = 0;
        with_radix(r, [&](auto R) {
            step = rem / R.value;
            fft_stage<R.value, SIGN, FAST_IN, FAST_OUT>(Ns, step, lines, pitch, first, last, tw, src, dst, load, store);
        });
        Ns *= r;
        rem = step;
        R2* t = src;
        src = dst;
        dst = t;
        if (!last) __syncthreads();
    }
    return src;
}

// store() of a last stage whose result stays in LDS
template <typename R2>
struct KeepLine {
    int pitch;
    __device__ __forceinline__ void operator()(R2* buf, int m, int l, R2 v) const { buf[m * pitch + l] = v; }
};

__device__ __forceinline__ float fixed_to_real(long long v, float) { return (float)((double)v * (1.0 / PrecMixed::grid_scale)); }
__device__ __forceinline__ double fixed_to_real(long long v, double) { return (double)v * (1.0 / PrecFP64::grid_scale); }

// Point (row y, z) of a grid plane: rows of Kz points in memory, of Kz + 4 as the
// spread leaves them in LDS.
template <bool SPREAD>
__device__ __forceinline__ long long grid_value(const long long* g, int y, int z, int Kz) {
    if constexpr (!SPREAD) return g[y * Kz + z];
    const long long* row = g + y * (Kz + 4);
    return z < 4 ? row[z] + row[z + Kz] : row[z];
}

// Point m of the real rows at o and o + second, and the copies past their ends.
template <typename real, typename R2>
__device__ __forceinline__ void store_rows(real* o, int second, bool both, int m, int Kz, int pad, R2 v) {
    o[m] = v.x;
    if (m < pad) o[Kz + m] = v.x;
    if (both) {
        o[second + m] = v.y;
        if (m < pad) o[second + Kz + m] = v.y;
    }
}

// First z stage of `rows` rows of the spread's sums g, rows 2p and 2p + 1 as one
// complex line: the sums take the room of the line buffers, so every thread holds
// its butterflies over the barrier (at most `Points` points of all lines in
// THREADS threads).
template <int R, int THREADS, int Points, typename R2>
__device__ __forceinline__ void fft_sums_stage(const long long* g, int rows, int np, int Kz, int pitch, R2* out) {
    using real = decltype(out->x);
    constexpr int U = (Points / R + THREADS - 1) / THREADS;
    const int nb = Kz / R, total = nb * np;
    const float inv_nb = 1.0f / (float)nb;
    R2 v[U][R];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int w = threadIdx.x + u * THREADS;
        if (w < total) {
            const int p = qdiv(w, inv_nb), j = w - p * nb;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int z = j + q * nb;
                v[u][q].x = fixed_to_real(grid_value<true>(g, 2 * p, z, Kz), (real)0);
                v[u][q].y = 2 * p + 1 < rows ? fixed_to_real(grid_value<true>(g, 2 * p + 1, z, Kz), (real)0) : (real)0;
            }
            dft<R, -1>(v[u]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int w = threadIdx.x + u * THREADS;
        if (w < total) {
            const int p = qdiv(w, inv_nb), j = w - p * nb;
#pragma unroll
            for (int q = 0; q < R; ++q) out[(j * R + q) * pitch + p] = v[u][q];
        }
    }
    __syncthreads();
}

// Wave number k of row y, from the transform Z of the complex lines that rows 2p
// and 2p + 1 make:  A_k = (Z_k + conj Z_{N-k}) / 2,  B_k = (Z_k - conj Z_{N-k}) / 2i.
template <typename R2>
__device__ __forceinline__ R2 paired_row(const R2* Z, int pitch, int Kz, int y, int k) {
    using real = decltype(Z->x);
    const bool second = y & 1;
    const int p = y >> 1;
    const R2 zk = Z[k * pitch + p], zn = Z[(k == 0 ? 0 : Kz - k) * pitch + p];
    R2 r;
    r.x = (real)0.5 * (second ? zk.y + zn.y : zk.x + zn.x);
    r.y = (real)0.5 * (second ? zn.x - zk.x : zk.y - zn.y);
    return r;
}

// Point m of the complex line a + ib whose inverse transform holds two real rows,
// from the half spectra: row(ks, 0) of the first, row(ks, 1) of the second.
template <typename R2, class Row>
__device__ __forceinline__ R2 paired_point(int m, int Kz, Row&& row) {
    const bool hi = 2 * m > Kz;               // upper half from the Hermitian symmetry
    const int ks = hi ? Kz - m : m;
    R2 a = row(ks, 0), b = row(ks, 1);
    if (ks == 0 || 2 * ks == Kz) { a.y = 0; b.y = 0; }      // DC and Nyquist terms are real
    if (hi) { a.y = -a.y; b.y = -b.y; }
    R2 z;
    z.x = a.x - b.y;
    z.y = a.y + b.x;
    return z;
}

// Z pass forward with the spread: rows y0 .. y0 + ny - 1 of plane x, two rows as
// one complex line (see fft_plane_fwd).  item = (sys, x, y0, ny)
template <class P>
__global__ __launch_bounds__(kSpreadZThreads) void fft_z_spread(const SysDev* __restrict__ sd,
                                                               const int4* __restrict__ items, SpreadArgs sp,
                                                               const typename P::real4* __restrict__ pos,
                                                               typename P::real2* cgrid,
                                                               const typename P::real2* __restrict__ tw) {
    side_priority();
    using R2 = typename P::real2;
    extern __shared__ unsigned char smem_raw[];
    const int4 it = items[blockIdx.x];
    const SysDev& d = sd[it.x];
    if (no_list(sp.sc[it.x])) return;      // the system is frozen
    const int x = it.y, y0 = it.z, ny = it.w;
    const int Ky = d.grid[1], Kz = d.grid[2], Kzh = Kz / 2 + 1, np = (ny + 1) >> 1, pz = np | 1, cap = pz * Kz;
    R2* TW = reinterpret_cast<R2*>(smem_raw);
    R2* A = TW + Kz;
    R2* B = A + cap;
    load_twiddles(TW, tw + d.tw_off[2], Kz);
    long long* g = reinterpret_cast<long long*>(A);
    spread_rows<P>(d, sp, pos, x, y0, ny, reinterpret_cast<int*>(A + spread_points<R2>(cap, ny, Kz)), g);
    const unsigned plan = d.fft_plan[2];
    const int r0 = plan & 15;
    with_radix(r0, [&](auto R) { fft_sums_stage<R.value, kSpreadZThreads, kSpreadZPoints>(g, ny, np, Kz, pz, A); });
    const R2* Z = fft_lines<-1, false, false>(Kz, plan >> 4, np, pz, TW, B, A, r0, [](int, int) { return R2{}; },
                                              KeepLine<R2>{pz});
    __syncthreads();
    R2* c = cgrid + d.cgrid_off + ((long long)x * Ky + y0) * Kzh;
    const float inv_kzh = 1.0f / (float)Kzh;
    for (int i = threadIdx.x; i < ny * Kzh; i += kSpreadZThreads) {
        const int y = qdiv(i, inv_kzh), k = i - y * Kzh;
        c[i] = paired_row(Z, pz, Kz, y, k);
    }
}

// Z pass forward: R2C.  item = (sys, first line, n lines)
template <class P>
__global__ __launch_bounds__(256) void fft_z_fwd(const SysDev* __restrict__ sd, const int4* __restrict__ items,
                                                 const typename P::gacc* __restrict__ rgrid,
                                                 typename P::real2* cgrid, const typename P::real2* __restrict__ tw) {
    side_priority();
    using real = typename P::real;
    using R2 = typename P::real2;
    extern __shared__ unsigned char smem_raw[];
    const int4 it = items[blockIdx.x];
    const SysDev& d = sd[it.x];
    const int Kz = d.grid[2], Kzh = Kz / 2 + 1;
    const int line0 = it.y, nl = it.z;
    R2* A = reinterpret_cast<R2*>(smem_raw);
    R2* B = A + nl * Kz;
    R2* TW = B + nl * Kz;
    load_twiddles(TW, tw + d.tw_off[2], Kz);
    __syncthreads();
    const typename P::gacc* g = rgrid + d.rgrid_off + (long long)line0 * Kz;
    R2* c = cgrid + d.cgrid_off + (long long)line0 * Kzh;
    fft_lines<-1, false, false>(
        Kz, d.fft_plan[2], nl, nl, TW, A, B, 1,
        [=](int m, int l) { return R2{fixed_to_real(g[l * Kz + m], (real)0), (real)0}; },
        [=](R2*, int m, int l, R2 v) { if (m < Kzh) c[l * Kzh + m] = v; });
}

// Z pass inverse: C2R into the potential grid, two rows as one complex line.
// item = (sys, x, p0, n): rows p0 .. p0 + n - 1 of the plane and their partners half a
// plane on, as in fft_plane_inv
template <class P>
__global__ __launch_bounds__(256) void fft_z_inv(const SysDev* __restrict__ sd, const int4* __restrict__ items,
                                                 const typename P::real2* __restrict__ cgrid, typename P::real* phi,
                                                 const typename P::real2* __restrict__ tw, int pad) {
    side_priority();
    using real = typename P::real;
    using R2 = typename P::real2;
    extern __shared__ unsigned char smem_raw[];
    const int4 it = items[blockIdx.x];
    const SysDev& d = sd[it.x];
    const int Ky = d.grid[1], Kz = d.grid[2], Kzh = Kz / 2 + 1;
    const int np = it.w, pz = np | 1, half = (Ky + 1) >> 1;
    R2* A = reinterpret_cast<R2*>(smem_raw);
    R2* B = A + pz * Kz;
    R2* TW = B + pz * Kz;
    load_twiddles(TW, tw + d.tw_off[2], Kz);
    __syncthreads();
    const long long line0 = (long long)it.y * Ky + it.z;
    const int past = Ky - it.z - half;      // pairs of the item with a second row
    const R2* c = cgrid + d.cgrid_off + line0 * Kzh;
    const int pitch = Kz + pad;
    real* o = phi + d.rgrid_off + line0 * pitch;
    fft_lines<+1, true, true>(
        Kz, d.fft_plan[2], np, pz, TW, A, B, 1,
        [=](int m, int p) {
            return paired_point<R2>(m, Kz, [=](int ks, int second) {
                return !second || p < past ? c[(p + second * half) * Kzh + ks] : R2{};
            });
        },
        [=](R2*, int m, int p, R2 v) { store_rows(o + p * pitch, half * pitch, p < past, m, Kz, pad, v); });
}

// Y pass: tile (sys, x, kz0) of TZ consecutive kz columns, lines along y.
template <class P, int SIGN>
__global__ __launch_bounds__(256) void fft_y(const SysDev* __restrict__ sd, const int4* __restrict__ items,
                                             typename P::real2* cgrid, const typename P::real2* __restrict__ tw,
                                             int TZ) {
    side_priority();
    using R2 = typename P::real2;
    extern __shared__ unsigned char smem_raw[];
    const int4 it = items[blockIdx.x];
    const SysDev& d = sd[it.x];
    const int Ky = d.grid[1], Kzh = d.grid[2] / 2 + 1;
    const int x = it.y, kz0 = it.z, nt = min(TZ, Kzh - kz0);
    R2* A = reinterpret_cast<R2*>(smem_raw);
    R2* B = A + nt * Ky;
    R2* TW = B + nt * Ky;
    load_twiddles(TW, tw + d.tw_off[1], Ky);
    __syncthreads();
    R2* c = cgrid + d.cgrid_off + (long long)x * Ky * Kzh + kz0;
    fft_lines<SIGN, false, false>(
        Ky, d.fft_plan[1], nt, nt, TW, A, B, 1, [=](int m, int l) { return c[m * Kzh + l]; },
        [=](R2*, int m, int l, R2 v) { c[m * Kzh + l] = v; });
}

// ---------------------------------------------------------- plane FFT passes
//
// Whole x-planes in LDS (gfx950 gives a workgroup up to 160 KiB): the forward
// pass transforms along z and then y in one kernel, the x pass transforms
// along x, multiplies by the influence function and transforms back, and the
// inverse pass runs y and then z.  Three launches per step instead of five.
// The real-to-complex z transform handles two real rows (2p and 2p + 1) as one
// complex line a + ib and separates them as the y transform reads them
// (paired_row); the complex-to-real inverse packs two rows (p and p + np: the
// reads of neighbouring p then meet no bank twice) the same way, Z_k = A_k + i B_k
// over the Hermitian extension (paired_point), then a = Re, b = Im.  The pairs are
// the same ones in the line passes, however those deal the rows to workgroups: a
// system's numbers do not depend on which passes its batch takes.

// Forward: plane x of the charge grid -> plane x of the half spectrum (z then y).
// The grid's plane is spread here (SPREAD) or read from `rgrid`.
// item = (sys, x)
template <class P, bool SPREAD>
__global__ __launch_bounds__(kPlaneThreads<typename P::real2>) void fft_plane_fwd(const SysDev* __restrict__ sd,
                                                              const int4* __restrict__ items,
                                                              const typename P::gacc* __restrict__ rgrid, SpreadArgs sp,
                                                              const typename P::real4* __restrict__ pos,
                                                              typename P::real2* cgrid,
                                                              const typename P::real2* __restrict__ tw) {
    side_priority();
    using real = typename P::real;
    using R2 = typename P::real2;
    extern __shared__ unsigned char smem_raw[];
    const int4 it = items[blockIdx.x];
    const SysDev& d = sd[it.x];
    const int x = it.y;
    const int Ky = d.grid[1], Kz = d.grid[2], Kzh = Kz / 2 + 1, np = (Ky + 1) >> 1;
    const int pz = np | 1, py = Kzh | 1, cap = plane_cap(Ky, Kz);
    R2* TWy = reinterpret_cast<R2*>(smem_raw);
    R2* TWz = TWy + Ky;
    R2* A = TWz + Kz;
    R2* B = A + cap;
    const unsigned plan = d.fft_plan[2];
    const R2* Z;
    if constexpr (SPREAD) {
        if (no_list(sp.sc[it.x])) return;      // the system is frozen
        long long* g = reinterpret_cast<long long*>(A);
        spread_rows<P>(d, sp, pos, x, 0, Ky, reinterpret_cast<int*>(A + spread_points<R2>(cap, Ky, Kz)), g);
        load_twiddles(TWy, tw + d.tw_off[1], Ky);
        load_twiddles(TWz, tw + d.tw_off[2], Kz);
        const int r0 = plan & 15;
        with_radix(r0, [&](auto R) {
            fft_sums_stage<R.value, kPlaneThreads<R2>, (int)(kPlaneSpreadLds<R2> / (2 * sizeof(R2)))>(g, Ky, np, Kz, pz, A);
        });
        Z = fft_lines<-1, false, false>(Kz, plan >> 4, np, pz, TWz, B, A, r0, [](int, int) { return R2{}; },
                                        KeepLine<R2>{pz});
    } else {
        load_twiddles(TWy, tw + d.tw_off[1], Ky);
        load_twiddles(TWz, tw + d.tw_off[2], Kz);
        __syncthreads();
        const typename P::gacc* g = rgrid + d.rgrid_off + (long long)x * Ky * Kz;
        Z = fft_lines<-1, true, false>(
            Kz, plan, np, pz, TWz, B, A, 1,
            [=](int m, int p) {
                return R2{fixed_to_real(g[2 * p * Kz + m], (real)0),
                          2 * p + 1 < Ky ? fixed_to_real(g[(2 * p + 1) * Kz + m], (real)0) : (real)0};
            },
            KeepLine<R2>{pz});
    }
    __syncthreads();
    R2* c = cgrid + d.cgrid_off + (long long)x * Ky * Kzh;
    fft_lines<-1, false, false>(
        Ky, d.fft_plan[1], Kzh, py, TWy, Z == A ? B : A, Z == A ? A : B, 1,
        [=](int m, int l) { return paired_row(Z, pz, Kz, m, l); },
        [=](R2*, int m, int l, R2 v) { c[m * Kzh + l] = v; });
}

// Inverse: plane x of the half spectrum -> plane x of the potential (y then z).
template <class P>
__global__ __launch_bounds__(kPlaneThreads<typename P::real2>) void fft_plane_inv(const SysDev* __restrict__ sd,
                                                              const int4* __restrict__ items,
                                                              const typename P::real2* __restrict__ cgrid,
                                                              typename P::real* phi,
                                                              const typename P::real2* __restrict__ tw, int pad) {
    side_priority();
    using real = typename P::real;
    using R2 = typename P::real2;
    extern __shared__ unsigned char smem_raw[];
    const int4 it = items[blockIdx.x];
    const SysDev& d = sd[it.x];
    const int x = it.y;
    const int Ky = d.grid[1], Kz = d.grid[2], Kzh = Kz / 2 + 1, np = (Ky + 1) >> 1;
    const int pz = np | 1, py = Kzh | 1, cap = plane_cap(Ky, Kz);
    R2* TWy = reinterpret_cast<R2*>(smem_raw);
    R2* TWz = TWy + Ky;
    R2* A = TWz + Kz;
    R2* B = A + cap;
    load_twiddles(TWy, tw + d.tw_off[1], Ky);
    load_twiddles(TWz, tw + d.tw_off[2], Kz);
    __syncthreads();
    const R2* c = cgrid + d.cgrid_off + (long long)x * Ky * Kzh;
    R2* Y = fft_lines<+1, false, false>(Ky, d.fft_plan[1], Kzh, py, TWy, A, B, 1,
                                        [=](int m, int l) { return c[m * Kzh + l]; }, KeepLine<R2>{py});
    __syncthreads();
    const int pitch = Kz + pad;
    real* o = phi + d.rgrid_off + (long long)x * Ky * pitch;
    fft_lines<+1, false, true>(
        Kz, d.fft_plan[2], np, pz, TWz, Y == A ? B : A, Y, 1,
        [=](int m, int p) {
            return paired_point<R2>(m, Kz, [=](int ks, int second) {
                return !second || p + np < Ky ? Y[(p + second * np) * py + ks] : R2{};
            });
        },
        [=](R2*, int m, int p, R2 v) { store_rows(o + p * pitch, np * pitch, p + np < Ky, m, Kz, pad, v); });
}

// fft_x's terms: in MODE 2 alone
struct NoTerms {};
template <class P, int MODE>
using XTerms = typename std::conditional<MODE == 2, TermArgs<P>, NoTerms>::type;

// X pass over nr consecutive (y, kz) lines from r0 = y Kzh + kz on (they stand
// side by side in memory, whatever Kzh): MODE 0 forward, 1 inverse, 2 forward /
// influence function / inverse, 3 the same with the energy.  The inverse takes
// the radices in reverse, so its first stage needs the very points that the
// forward's last one leaves in a thread's registers: the product and both stages
// are one (64 points: two trips through LDS for both transforms).
// item = (sys, r0, nr)
//
// A step's bonded terms ride along (MODE 2): the blocks past the items' are a
// thread a term, and the forces per atom follow in the gather's launch.  On a small
// system a launch costs the step about as much as its kernel, on the device and on
// the host, which needs 5 us for a node of the two-branch step graph (as kernels of
// their own, before the spread, the two made the 1,500-bead chain's step 64.6 us
// instead of 51.2).
template <class P, int MODE>
__global__ __launch_bounds__(kXPassThreads) void fft_x(const SysDev* __restrict__ sd, const int4* __restrict__ items,
                                                      int n_items, typename P::real2* cgrid,
                                                      const typename P::real* __restrict__ eta,
                                                      const typename P::real2* __restrict__ tw, long long* energy,
                                                      XTerms<P, MODE> terms) {
    side_priority();
    if constexpr (MODE == 2) {
        if ((int)blockIdx.x >= n_items) {
            bonded_term<P, false>(terms, ((int)blockIdx.x - n_items) * (int)blockDim.x + (int)threadIdx.x, nullptr);
            return;
        }
    }
    using R2 = typename P::real2;
    extern __shared__ unsigned char smem_raw[];
    const int4 it = items[blockIdx.x];
    const int s = it.x, r0 = it.y, nr = it.z;
    const SysDev& d = sd[s];
    const int Kx = d.grid[0], Ky = d.grid[1], Kz = d.grid[2], Kzh = Kz / 2 + 1;
    R2* TW = reinterpret_cast<R2*>(smem_raw);
    R2* A = TW + Kx;
    R2* B = A + nr * Kx;
    load_twiddles(TW, tw + d.tw_off[0], Kx);
    __syncthreads();
    const int sx = Ky * Kzh;
    R2* c = cgrid + d.cgrid_off + r0;
    auto from_grid = [=](int m, int l) { return c[(long long)m * sx + l]; };
    auto to_grid = [=](R2*, int m, int l, R2 v) { c[(long long)m * sx + l] = v; };
    const unsigned plan = d.fft_plan[0];
    if constexpr (MODE < 2) {
        fft_lines<(MODE == 0 ? -1 : +1), false, false>(Kx, plan, nr, nr, TW, A, B, 1, from_grid, to_grid);
    } else {
        const auto* et = eta + d.cgrid_off + r0;
        // the radices before the last, and the same in reverse
        unsigned head = 0, back = 0, rest = plan;
        int at = 0;
        for (; rest >> 4; rest >>= 4, at += 4) {
            head |= (rest & 15) << at;
            back = back << 4 | (rest & 15);
        }
        const R2* src = fft_lines<-1, false, false>(Kx, head, nr, nr, TW, A, B, 1, from_grid, KeepLine<R2>{nr});
        if (head) __syncthreads();
        R2* dst = src == A ? B : A;
        long long e = 0;   // fixed point per element: independent of the tiling
        with_radix((int)rest, [&](auto RC) {
            constexpr int R = RC.value;
            const int nb = Kx / R;
            const float inv_nr = 1.0f / (float)nr, inv_kzh = 1.0f / (float)Kzh;
            for (int w = threadIdx.x; w < nb * nr; w += blockDim.x) {
                const int j = qdiv(w, inv_nr), l = w - j * nr;
                typename P::real wt[R];
#pragma unroll
                for (int q = 0; q < R; ++q) wt[q] = et[(long long)(j + q * nb) * sx + l];
                R2 v[R];
                if (!head) {
#pragma unroll
                    for (int q = 0; q < R; ++q) v[q] = from_grid(j + q * nb, l);
                } else {
#pragma unroll
                    for (int q = 0; q < R; ++q) v[q] = src[(j + q * nb) * nr + l];
#pragma unroll
                    for (int q = 1; q < R; ++q) v[q] = cmul(v[q], TW[j * q]);      // j q < Kx
                }
                dft<R, -1>(v);
                if constexpr (MODE == 3) {
                    const int kz = (r0 + l) - qdiv(r0 + l, inv_kzh) * Kzh;
                    const double half = (kz == 0 || 2 * kz == Kz) ? 0.5 : 1.0;
#pragma unroll
                    for (int q = 0; q < R; ++q)
                        e += energy_fixed(half * (double)wt[q] * ((double)v[q].x * v[q].x + (double)v[q].y * v[q].y));
                }
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    v[q].x *= wt[q];
                    v[q].y *= wt[q];
                }
                dft<R, +1>(v);
                if (!head) {
#pragma unroll
                    for (int q = 0; q < R; ++q) to_grid(nullptr, j * R + q, l, v[q]);
                } else {
#pragma unroll
                    for (int q = 0; q < R; ++q) dst[(j * R + q) * nr + l] = v[q];
                }
            }
        });
        if (head) {
            __syncthreads();
            fft_lines<+1, false, false>(Kx, back, nr, nr, TW, dst == A ? B : A, dst, (int)rest, from_grid, to_grid);
        }
        if constexpr (MODE == 3) block_energy_add(energy, s, E_RECIP, e);
    }
}

// NEXUSMD_FFT_PLANE=0 selects the five line passes even where planes fit.
bool fft_plane_enabled() {
    const char* e = std::getenv("NEXUSMD_FFT_PLANE");
    return !(e && std::string(e) == "0");
}

// Raises the dynamic-LDS limit of the plane kernels to what the batch needs.
template <class P>
hipError_t prepare_fft(Batch<P>& B) {
    const int sl = (int)B.fft_spread_lds, pl = (int)B.fft_plane_lds, xl = (int)B.fft_x_lds;
    const hipFuncAttribute a = hipFuncAttributeMaxDynamicSharedMemorySize;
    hipError_t e = hipFuncSetAttribute(
        !B.fft_plane ? (const void*)fft_z_spread<P> : (const void*)fft_plane_fwd<P, true>, a, sl);
    if (e == hipSuccess) e = hipFuncSetAttribute((const void*)fft_x<P, 2>, a, xl);
    if (e == hipSuccess) e = hipFuncSetAttribute((const void*)fft_x<P, 3>, a, xl);
    if (e == hipSuccess && B.fft_plane) e = hipFuncSetAttribute((const void*)fft_plane_inv<P>, a, pl);
    return e;
}

template <class P>
void launch_pme_spread(Batch<P>& B) {
    if (!B.pme_any) return;
    const SpreadArgs sp{B.d_cnt, B.col_count, B.col_slot};
    if (B.fft_plane)
        fft_plane_fwd<P, true><<<B.n_fftz, kPlaneThreads<typename P::real2>, B.fft_spread_lds, B.stream>>>(
            B.d_sys, B.fftz_items, nullptr, sp, B.pos, B.cgrid, B.twiddle);
    else
        fft_z_spread<P><<<B.n_fftz, kSpreadZThreads, B.fft_spread_lds, B.stream>>>(B.d_sys, B.fftz_items, sp, B.pos,
                                                                                 B.cgrid, B.twiddle);
}

template <class P>
void launch_fft_forward(Batch<P>& B) {
    if (!B.pme_any || B.fft_plane) return;      // the spread's launch ran the plane pass
    fft_y<P, -1><<<B.n_ffty, 256, B.fft_y_lds, B.stream>>>(B.d_sys, B.ffty_items, B.cgrid, B.twiddle, B.fft_tile);
}

template <class P>
void launch_fft_convolve(Batch<P>& B, bool energy, int term_mask) {
    if (!B.pme_any) return;
    const int T = B.fft_x_threads;
    if (energy) {
        fft_x<P, 3><<<B.n_fftx, T, B.fft_x_lds, B.stream>>>(B.d_sys, B.fftx_items, B.n_fftx, B.cgrid, B.eta, B.twiddle,
                                                           B.energy, {});
    } else {
        const int blocks = (bonded_count(B, term_mask) + T - 1) / T;
        fft_x<P, 2><<<B.n_fftx + blocks, T, B.fft_x_lds, B.stream>>>(B.d_sys, B.fftx_items, B.n_fftx, B.cgrid, B.eta,
                                                                    B.twiddle, B.energy, term_args(B, term_mask));
    }
}

template <class P>
void launch_fft_inverse(Batch<P>& B) {
    if (!B.pme_any) return;
    if (B.fft_plane) {
        fft_plane_inv<P><<<B.n_fftp, B.fft_plane_threads, B.fft_plane_lds, B.stream>>>(B.d_sys, B.fftp_items, B.cgrid,
                                                                                      B.phi, B.twiddle, kPhiPad);
        return;
    }
    fft_y<P, +1><<<B.n_ffty, 256, B.fft_y_lds, B.stream>>>(B.d_sys, B.ffty_items, B.cgrid, B.twiddle, B.fft_tile);
    fft_z_inv<P><<<B.n_fftl, 256, B.fft_z_lds, B.stream>>>(B.d_sys, B.fftl_items, B.cgrid, B.phi, B.twiddle, kPhiPad);
}

template <class P>
void launch_pme_gather(Batch<P>& B, int atom_mask) {
    if (!B.pme_any) return;
    const int T = 5 * kGatherSlots, atom_blocks = atom_mask >= 0 ? (B.n_atoms + T - 1) / T : 0;
    pme_gather_kernel<P><<<(unsigned)(atom_blocks + (B.n_slots_cap + kGatherSlots - 1) / kGatherSlots), T, 0, B.stream>>>(
        B.d_sys, B.d_cnt, B.slot_sys, B.atom_of_slot, B.pos, B.phi, B.FSx, B.FSy, B.FSz, B.n_slots_cap, atom_blocks,
        term_args(B, atom_force_mask(B, std::max(0, atom_mask))));
}

template void launch_pme_spread<PrecFP64>(Batch<PrecFP64>&);
template void launch_pme_spread<PrecMixed>(Batch<PrecMixed>&);
template hipError_t prepare_fft<PrecFP64>(Batch<PrecFP64>&);
template hipError_t prepare_fft<PrecMixed>(Batch<PrecMixed>&);
template void launch_fft_forward<PrecFP64>(Batch<PrecFP64>&);
template void launch_fft_forward<PrecMixed>(Batch<PrecMixed>&);
template void launch_fft_convolve<PrecFP64>(Batch<PrecFP64>&, bool, int);
template void launch_fft_convolve<PrecMixed>(Batch<PrecMixed>&, bool, int);
template void launch_fft_inverse<PrecFP64>(Batch<PrecFP64>&);
template void launch_fft_inverse<PrecMixed>(Batch<PrecMixed>&);
template void launch_pme_gather<PrecFP64>(Batch<PrecFP64>&, int);
template void launch_pme_gather<PrecMixed>(Batch<PrecMixed>&, int);

// Standalone 3D transform of one real grid through the same pass kernels.
template <class P>
void fft3d_roundtrip(int nx, int ny, int nz, const double* in, double* out, bool forward, hipStream_t st) {
    using R2 = typename P::real2;
    using real = typename P::real;
    const int nzh = nz / 2 + 1;
    SysDev d{};
    d.grid[0] = nx; d.grid[1] = ny; d.grid[2] = nz;
    d.rgrid_off = 0; d.cgrid_off = 0;
    d.tw_off[0] = 0; d.tw_off[1] = nx; d.tw_off[2] = nx + ny;
    for (int a = 0; a < 3; ++a) d.fft_plan[a] = fft_plan(d.grid[a]);
    std::vector<R2> tw(nx + ny + nz);
    const int K[3] = {nx, ny, nz};
    for (int a = 0, o = 0; a < 3; o += K[a], ++a)
        for (int t = 0; t < K[a]; ++t) {
            const double ang = -2.0 * kPi * (double)t / (double)K[a];
            tw[o + t].x = (real)cos(ang);
            tw[o + t].y = (real)sin(ang);
        }
    const int maxK = std::max(nx, std::max(ny, nz));
    const int T = std::max(1, std::min(8, (int)((61440 / (int)sizeof(R2) - maxK) / (2 * maxK))));
    std::vector<int4> zi, yi, xi;
    if (forward) {
        for (int l = 0; l < nx * ny; l += T) zi.push_back(make_int4(0, l, std::min(T, nx * ny - l), 0));
    } else {
        const int half = (ny + 1) / 2, pairs = (T - 1) | 1;
        for (int x = 0; x < nx; ++x)
            for (int p = 0; p < half; p += pairs) zi.push_back(make_int4(0, x, p, std::min(pairs, half - p)));
    }
    for (int x = 0; x < nx; ++x)
        for (int k = 0; k < nzh; k += T) yi.push_back(make_int4(0, x, k, 0));
    for (int y = 0; y < ny; ++y)
        for (int k = 0; k < nzh; k += T) xi.push_back(make_int4(0, y * nzh + k, std::min(T, nzh - k), 0));
    SysDev* dd; R2* dtw; int4 *dz, *dy, *dx; typename P::gacc* rg; R2* cg; real* ph;
    const size_t G = (size_t)nx * ny * nz, Gh = (size_t)nx * ny * nzh;
    hipMalloc(&dd, sizeof(SysDev));
    hipMalloc(&dtw, tw.size() * sizeof(R2));
    hipMalloc(&dz, zi.size() * sizeof(int4));
    hipMalloc(&dy, yi.size() * sizeof(int4));
    hipMalloc(&dx, xi.size() * sizeof(int4));
    hipMalloc(&rg, G * sizeof(typename P::gacc));
    hipMalloc(&cg, Gh * sizeof(R2));
    hipMalloc(&ph, G * sizeof(real));
    hipMemcpyAsync(dd, &d, sizeof(SysDev), hipMemcpyHostToDevice, st);
    hipMemcpyAsync(dtw, tw.data(), tw.size() * sizeof(R2), hipMemcpyHostToDevice, st);
    hipMemcpyAsync(dz, zi.data(), zi.size() * sizeof(int4), hipMemcpyHostToDevice, st);
    hipMemcpyAsync(dy, yi.data(), yi.size() * sizeof(int4), hipMemcpyHostToDevice, st);
    hipMemcpyAsync(dx, xi.data(), xi.size() * sizeof(int4), hipMemcpyHostToDevice, st);
    const size_t sm = (size_t)(2 * T + 1) * maxK * sizeof(R2);
    // plane passes (as the engine uses them) when the planes fit
    const bool plane = fft_plane_enabled() && plane_lds_bytes<R2>(ny, nz) <= kMaxBlockLds &&
                       line_lds_bytes<R2>(nx, nzh) <= kMaxBlockLds;
    std::vector<int4> pi, bi;
    int4 *dp = nullptr, *db = nullptr;
    const size_t pl = plane_lds_bytes<R2>(ny, nz), xl = line_lds_bytes<R2>(nx, nzh);
    if (plane) {
        for (int x = 0; x < nx; ++x) pi.push_back(make_int4(0, x, 0, 0));
        for (int y = 0; y < ny; ++y) bi.push_back(make_int4(0, y * nzh, nzh, 0));
        hipMalloc(&dp, pi.size() * sizeof(int4));
        hipMalloc(&db, bi.size() * sizeof(int4));
        hipMemcpyAsync(dp, pi.data(), pi.size() * sizeof(int4), hipMemcpyHostToDevice, st);
        hipMemcpyAsync(db, bi.data(), bi.size() * sizeof(int4), hipMemcpyHostToDevice, st);
        hipFuncSetAttribute((const void*)fft_plane_fwd<P, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl);
        hipFuncSetAttribute((const void*)fft_plane_inv<P>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl);
        hipFuncSetAttribute((const void*)fft_x<P, 0>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)xl);
        hipFuncSetAttribute((const void*)fft_x<P, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)xl);
    }
    if (forward) {
        std::vector<typename P::gacc> h(G);
        for (size_t i = 0; i < G; ++i) {
            h[i] = (long long)llrint(in[i] * P::grid_scale);
        }
        hipMemcpyAsync(rg, h.data(), G * sizeof(typename P::gacc), hipMemcpyHostToDevice, st);
        if (plane) {
            fft_plane_fwd<P, false><<<(unsigned)pi.size(), kPlaneThreads<R2>, pl, st>>>(dd, dp, rg, {}, nullptr, cg, dtw);
            fft_x<P, 0><<<(unsigned)bi.size(), kXPassThreads, xl, st>>>(dd, db, (int)bi.size(), cg, nullptr, dtw, nullptr, {});
        } else {
            fft_z_fwd<P><<<(unsigned)zi.size(), 256, sm, st>>>(dd, dz, rg, cg, dtw);
            fft_y<P, -1><<<(unsigned)yi.size(), 256, sm, st>>>(dd, dy, cg, dtw, T);
            fft_x<P, 0><<<(unsigned)xi.size(), 256, sm, st>>>(dd, dx, (int)xi.size(), cg, nullptr, dtw, nullptr, {});
        }
        std::vector<R2> hc(Gh);
        hipMemcpyAsync(hc.data(), cg, Gh * sizeof(R2), hipMemcpyDeviceToHost, st);
        hipStreamSynchronize(st);
        for (size_t i = 0; i < Gh; ++i) { out[2 * i] = hc[i].x; out[2 * i + 1] = hc[i].y; }
    } else {
        std::vector<R2> hc(Gh);
        for (size_t i = 0; i < Gh; ++i) { hc[i].x = (real)in[2 * i]; hc[i].y = (real)in[2 * i + 1]; }
        hipMemcpyAsync(cg, hc.data(), Gh * sizeof(R2), hipMemcpyHostToDevice, st);
        if (plane) {
            fft_x<P, 1><<<(unsigned)bi.size(), kXPassThreads, xl, st>>>(dd, db, (int)bi.size(), cg, nullptr, dtw, nullptr, {});
            fft_plane_inv<P><<<(unsigned)pi.size(), kPlaneThreads<R2>, pl, st>>>(dd, dp, cg, ph, dtw, 0);
        } else {
            fft_x<P, 1><<<(unsigned)xi.size(), 256, sm, st>>>(dd, dx, (int)xi.size(), cg, nullptr, dtw, nullptr, {});
            fft_y<P, +1><<<(unsigned)yi.size(), 256, sm, st>>>(dd, dy, cg, dtw, T);
            fft_z_inv<P><<<(unsigned)zi.size(), 256, sm, st>>>(dd, dz, cg, ph, dtw, 0);
        }
        std::vector<real> hr(G);
        hipMemcpyAsync(hr.data(), ph, G * sizeof(real), hipMemcpyDeviceToHost, st);
        hipStreamSynchronize(st);
        for (size_t i = 0; i < G; ++i) out[i] = hr[i];
    }
    hipFree(dd); hipFree(dtw); hipFree(dz); hipFree(dy); hipFree(dx); hipFree(rg); hipFree(cg); hipFree(ph);
    if (dp) hipFree(dp);
    if (db) hipFree(db);
}

template void fft3d_roundtrip<PrecFP64>(int, int, int, const double*, double*, bool, hipStream_t);
template void fft3d_roundtrip<PrecMixed>(int, int, int, const double*, double*, bool, hipStream_t);

// ------------------------------------------------------ no-allocation FFT
//
// The forward transform of fft3d_roundtrip with every device buffer carved
// out of one file-scope array, `scratch`, so that a call allocates nothing.
// Each GPU holds its own copy of the array from the library's load until the
// process ends.  Layout (256-byte aligned regions):
//   [SysDev][twiddles, 3 x kNoAllocMaxK][work items, kNoAllocItems int4]
//   [real grid, 8 B per point][half spectrum, sizeof(real2) per point]
// The input is copied straight into the real-grid region (the mixed path
// then converts it to fixed point in place, element by element), and the
// FP64 spectrum is copied straight out of its region; the mixed spectrum
// (float pairs) is copied into the caller's output and widened there in
// place, from the last element backwards.  The host side uses the device
// address returned by hipGetSymbolAddress, never the array's name.
constexpr int kNoAllocMaxK = 256;
constexpr long long kNoAllocMaxPoints = 1LL << 20;
constexpr int kNoAllocItems = 32768;
constexpr size_t kNoAllocBytes = 20u << 20;
constexpr int kNoAllocMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

namespace {

std::mutex g_noalloc_mu[kNoAllocMaxDevices];     // one call at a time per device
void* g_noalloc_ptr[kNoAllocMaxDevices] = {};    // device address of each device's array

constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Work items of the forward passes, in fft3d_roundtrip's order.  Plane passes:
// x planes, then the x pass's lines of one y.  Line passes: groups of T z
// lines, then (x, kz block) items and the x pass's lines of a (y, kz block).
__global__ void noalloc_items_kernel(int4* it, int nx, int ny, int nzh, int T, int plane, int n0, int n1, int n2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n0 + n1 + n2) return;
    if (plane) {
        if (i < n0) it[i] = make_int4(0, i, 0, 0);
        else it[i] = make_int4(0, (i - n0) * nzh, nzh, 0);
        return;
    }
    const int nkb = (nzh + T - 1) / T;
    if (i < n0) {
        const int l = i * T;
        it[i] = make_int4(0, l, min(T, nx * ny - l), 0);
    } else if (i < n0 + n1) {
        const int j = i - n0;
        it[i] = make_int4(0, j / nkb, (j % nkb) * T, 0);
    } else {
        const int j = i - n0 - n1, k = (j % nkb) * T;
        it[i] = make_int4(0, j / nkb * nzh + k, min(T, nzh - k), 0);
    }
}

// In place: the doubles of the input become 2^32 fixed point (as the host
// conversion of fft3d_roundtrip: round to nearest, ties to even).
__global__ void noalloc_to_fixed_kernel(void* g, long long n, double scale) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double v = reinterpret_cast<const double*>(g)[i];
    reinterpret_cast<long long*>(g)[i] = __double2ll_rn(v * scale);
}

}  // namespace

template <class P>
nx_status fft3d_r2c_noalloc(int device, int nx, int ny, int nz, const double* in, double* out, std::string& err) {
    using R2 = typename P::real2;
    using real = typename P::real;
    if (device < 0 || device >= kNoAllocMaxDevices) { err = "device index out of range"; return NX_ERR_ARG; }
    const int nzh = nz / 2 + 1;
    const long long G = (long long)nx * ny * nz, Gh = (long long)nx * ny * nzh;
    if (nx > kNoAllocMaxK || ny > kNoAllocMaxK || nz > kNoAllocMaxK || G > kNoAllocMaxPoints) {
        err = "grid " + std::to_string(nx) + "x" + std::to_string(ny) + "x" + std::to_string(nz) +
              " exceeds the no-allocation maximum (each dimension <= " + std::to_string(kNoAllocMaxK) + ", at most " +
              std::to_string(kNoAllocMaxPoints) + " points)";
        return NX_ERR_CAPACITY;
    }
    const int maxK = std::max(nx, std::max(ny, nz));
    const int T = std::max(1, std::min(8, (int)((61440 / (int)sizeof(R2) - maxK) / (2 * maxK))));
    const bool plane = fft_plane_enabled() && plane_lds_bytes<R2>(ny, nz) <= kMaxBlockLds &&
                       line_lds_bytes<R2>(nx, nzh) <= kMaxBlockLds;
    const int nkb = (nzh + T - 1) / T;
    const int n0 = plane ? nx : (nx * ny + T - 1) / T;
    const int n1 = plane ? ny : nx * nkb;
    const int n2 = plane ? 0 : ny * nkb;
    const size_t o_tw = align256(sizeof(SysDev));
    const size_t o_it = o_tw + align256(3 * kNoAllocMaxK * sizeof(R2));
    const size_t o_rg = o_it + align256((size_t)kNoAllocItems * sizeof(int4));
    const size_t o_cg = o_rg + align256((size_t)G * 8);
    const size_t need = o_cg + (size_t)Gh * sizeof(R2);
    if (n0 + n1 + n2 > kNoAllocItems || need > kNoAllocBytes) {
        err = "grid " + std::to_string(nx) + "x" + std::to_string(ny) + "x" + std::to_string(nz) + " needs " +
              std::to_string(need) + " bytes of scratch; the no-allocation array holds " + std::to_string(kNoAllocBytes);
        return NX_ERR_CAPACITY;
    }
    std::lock_guard<std::mutex> lock(g_noalloc_mu[device]);
    auto fail = [&](hipError_t e, const char* what) {
        err = std::string(what) + ": " + hipGetErrorString(e);
        return NX_ERR_HIP;
    };
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) return fail(e, "hipSetDevice");
    if (!g_noalloc_ptr[device]) {
        // once per device, with that device current: the address of its copy
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return fail(e, "hipGetSymbolAddress(scratch)");
        g_noalloc_ptr[device] = p;
    }
    unsigned char* base = static_cast<unsigned char*>(g_noalloc_ptr[device]);
    SysDev* dd = reinterpret_cast<SysDev*>(base);
    R2* dtw = reinterpret_cast<R2*>(base + o_tw);
    int4* items = reinterpret_cast<int4*>(base + o_it);
    typename P::gacc* rg = reinterpret_cast<typename P::gacc*>(base + o_rg);
    R2* cg = reinterpret_cast<R2*>(base + o_cg);
    const hipStream_t st = nullptr;
    // the per-call tables, from host values on the stack
    SysDev d{};
    d.grid[0] = nx; d.grid[1] = ny; d.grid[2] = nz;
    d.tw_off[0] = 0; d.tw_off[1] = nx; d.tw_off[2] = nx + ny;
    for (int a = 0; a < 3; ++a) d.fft_plan[a] = fft_plan(d.grid[a]);
    R2 tw[3 * kNoAllocMaxK];
    const int K[3] = {nx, ny, nz};
    for (int a = 0, o = 0; a < 3; o += K[a], ++a)
        for (int t = 0; t < K[a]; ++t) {
            const double ang = -2.0 * kPi * (double)t / (double)K[a];
            tw[o + t].x = (real)cos(ang);
            tw[o + t].y = (real)sin(ang);
        }
    if ((e = hipMemcpyAsync(dd, &d, sizeof(SysDev), hipMemcpyHostToDevice, st)) != hipSuccess) return fail(e, "copy");
    if ((e = hipMemcpyAsync(dtw, tw, (size_t)(nx + ny + nz) * sizeof(R2), hipMemcpyHostToDevice, st)) != hipSuccess)
        return fail(e, "copy");
    noalloc_items_kernel<<<(n0 + n1 + n2 + 255) / 256, 256, 0, st>>>(items, nx, ny, nzh, T, plane ? 1 : 0, n0, n1, n2);
    if ((e = hipMemcpyAsync(rg, in, (size_t)G * sizeof(double), hipMemcpyHostToDevice, st)) != hipSuccess)
        return fail(e, "copy");
    noalloc_to_fixed_kernel<<<(unsigned)((G + 255) / 256), 256, 0, st>>>(rg, G, P::grid_scale);
    if (plane) {
        const size_t pl = plane_lds_bytes<R2>(ny, nz), xl = line_lds_bytes<R2>(nx, nzh);
        if ((e = hipFuncSetAttribute((const void*)fft_plane_fwd<P, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)pl)) != hipSuccess ||
            (e = hipFuncSetAttribute((const void*)fft_x<P, 0>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)xl)) != hipSuccess)
            return fail(e, "hipFuncSetAttribute");
        fft_plane_fwd<P, false><<<(unsigned)n0, kPlaneThreads<R2>, pl, st>>>(dd, items, rg, {}, nullptr, cg, dtw);
        fft_x<P, 0><<<(unsigned)n1, kXPassThreads, xl, st>>>(dd, items + n0, n1, cg, nullptr, dtw, nullptr, {});
    } else {
        const size_t sm = (size_t)(2 * T + 1) * maxK * sizeof(R2);
        fft_z_fwd<P><<<(unsigned)n0, 256, sm, st>>>(dd, items, rg, cg, dtw);
        fft_y<P, -1><<<(unsigned)n1, 256, sm, st>>>(dd, items + n0, cg, dtw, T);
        fft_x<P, 0><<<(unsigned)n2, 256, sm, st>>>(dd, items + n0 + n1, n2, cg, nullptr, dtw, nullptr, {});
    }
    if ((e = hipGetLastError()) != hipSuccess) return fail(e, "kernel launch");
    if ((e = hipMemcpyAsync(out, cg, (size_t)Gh * sizeof(R2), hipMemcpyDeviceToHost, st)) != hipSuccess)
        return fail(e, "copy");
    if ((e = hipStreamSynchronize(st)) != hipSuccess) return fail(e, "hipStreamSynchronize");
    if constexpr (P::mixed) {
        // float pairs at the front of `out` widened to doubles in place, last first:
        // element i is read from bytes [8i, 8i + 8) before bytes [16i, 16i + 16) are
        // written, and no element below i is read from at or above byte 8i
        unsigned char* ob = reinterpret_cast<unsigned char*>(out);
        for (long long i = Gh - 1; i >= 0; --i) {
            float v[2];
            std::memcpy(v, ob + 8 * i, sizeof(v));
            const double w[2] = {(double)v[0], (double)v[1]};
            std::memcpy(ob + 16 * i, w, sizeof(w));
        }
    }
    return NX_OK;
}

template nx_status fft3d_r2c_noalloc<PrecFP64>(int, int, int, int, const double*, double*, std::string&);
template nx_status fft3d_r2c_noalloc<PrecMixed>(int, int, int, int, const double*, double*, std::string&);

}  // namespace nx
