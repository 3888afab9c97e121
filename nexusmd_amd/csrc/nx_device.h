// nx_device.h -- device-side types and helpers shared by the HIP kernels.
//
// Data layout (all systems of a batch packed back to back):
//   atom order  : FP64 master state x/y/z, vx/vy/vz, 1/m (SoA), per-atom
//                 force accumulators F_atom (bonded terms, exclusion
//                 correction), atom_sys, slot_of_atom.
//   slot order  : atoms binned into xy columns, sorted by z inside a column and
//                 cut into super-clusters of 64, each split into 8 clusters of
//                 8 (padded).  Per slot: packed (x,y,z,q), (sig/2, 2*sqrt(eps)),
//                 atom_of_slot (-1 = padding), force accumulators F_slot
//                 (pair, PME).
//   PME         : per system a half-spectrum complex grid [Kx][Ky][Kz/2+1] and
//                 a real potential grid (rows of Kz + kPhiPad points); the
//                 charge grid stands in LDS only.
// Forces: each contribution is converted to fixed point (mixed: 64 bits, 2^32
// units per kJ/mol/nm; FP64: two parts, Fix2), so sums are exact integers and
// independent of order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nx {

constexpr double kOne4PiEps0 = 138.93545764446428693393;   // kJ nm / (mol e^2)
constexpr double kPi = 3.14159265358979323846;
constexpr double kSqrtPi = 1.77245385090551602729;
constexpr double kTwoOverSqrtPi = 1.1283791670955126;
constexpr double kForceScale = 4294967296.0;               // 2^32 fixed-point units
constexpr double kEnergyScale = 1073741824.0;              // 2^30 fixed-point units
constexpr int kClusterSize = 8;
constexpr int kSuperClusters = 8;                           // clusters per super-cluster
constexpr int kPmeOrder = 5;

constexpr int NX_FORCE_NONBONDED_BIT = 8;   // the nonbonded bit of a force mask

enum EnergyTerm { E_BOND = 0, E_ANGLE, E_TORSION, E_COUL, E_LJ, E_RECIP, E_EXCL, E_KIN, E_NTERMS };

// Per-system constants (device copy; written once per topology/box).
struct SysDev {
    double L[3], invL[3], lb[3], ub[3];
    double rc, rc2, rlist, alpha, skin_half2;
    double sw_on, sw_inv;        // switching: r_switch, 1/(rc - r_switch); sw_on < 0 = off
    double ew_exp, ew_exp_lo;    // FP64 direct space: alpha^2 / ln 2 in two parts,
    double ew_u, ew_q;           // alpha / sqrt(2), 2 alpha / sqrt(pi) (pair_fp64_series)
    int n_atoms, atom_off;
    int slot_off, slot_cap;
    int col_off, ncx, ncy, col_cap;   // columns: ncx*ncy, each of 2 x 2 quarters
    int super_off, super_cap;
    int chunk_off, chunk_cap;    // pair-kernel work items (list chunks)
    int chunk_entries;           // pair-list entries per chunk (chunk_entries_for)
    int list_off, list_cap;
    int emask_off, emask_cap;
    double colw[2];              // column widths
    int grid[3];
    int pair_image;              // mixed path: per-entry periodic images in the list (0: pair by pair)
    long long rgrid_off, cgrid_off;   // offsets into the real / complex grids
    int excl_off, n_excl;        // excluded pair list
    int bond_off, n_bonds, angle_off, n_angles, tors_off, n_tors;
    int tw_off[3];               // twiddle-table offsets per axis
    unsigned fft_plan[3];        // radices of the axes' transforms (fft_plan)
    double sp_margin;            // distance an atom may move between rebuilds
};

// Per-system counters written by the device.
struct SysCount {
    int n_slots, n_clusters, n_super, list_count;
    int emask_count, rebuild, overflow, rebuilds;
    int n_chunks, steps_done, pad1, pad2;   // steps_done: leapfrog steps the system completed
};
// overflow bit of a system that ran a step without the list kernels although
// its list was due for a build: the update froze it for that step (the host
// runs the step again with the list kernels; not a failure)
constexpr int kStaleList = 8;
// No list to work on: the system is empty or its last build failed.  Every bit of
// this was written before the work that asks for it was queued, so all wavefronts
// of a workgroup see the same answer and may leave it on it, barriers or not.  Not
// so kStaleList: nl_waves sets it while the kernels of the side stream run.  They
// go through such a step on the last build's list (the update drops what they sum).
__device__ __forceinline__ bool no_list(const SysCount& sc) {
    return sc.n_slots == 0 || (sc.overflow & ~kStaleList) != 0;
}

// What nl_waves of a one-system batch reports to host memory early in every
// step, for the host's choice between the step graphs with and without the
// list kernels: the report count, the largest displacement of an atom from
// its build position after the last update, the steps done, whether this
// step's list is due, and the overflow flags.
struct __align__(16) StepInfo {
    unsigned seq;               // reports so far (modulo 2^32)
    float dmax;                 // nm
    int steps_done;
    int flags;                  // bit 0: the list is due; bits 1..: the overflow flags
};
// slots of the update's largest squared displacement (block b adds to slot b % 64)
constexpr int kStepMaxSlots = 64;

constexpr int kChunkEntries = 32;       // most pair-list entries per chunk, the pair kernel's unit of work
// Pair-list entries one super-cluster may hold (the list build keeps them in
// LDS).  A super-cluster is 64 atoms, about a 0.9 nm cube at water density, with
// ~150 j clusters of higher index within rlist = 1.1 nm.
constexpr int kSuperListCap = 2048;
constexpr int kPairWaves = 4;           // independent wavefronts per 256-thread pair-kernel block
// The pair kernel's chunk ranges, one per XCD, 128 bytes apart: the next chunk
// to hand out, and the range's first and end chunk.
constexpr int kPoolStride = 32, kPoolInts = 8 * kPoolStride;
constexpr int kPoolFirst = 1, kPoolEnd = 2;

// Second word of a pair-list entry: the exclusion-mask id in the low 26 bits
// (kNoMask: the tile has no listed exclusion) and the j-cluster's periodic
// image in the high 6 bits, two per axis (0: none, 1: +L, 2: -L), for which
// every atom pair of the entry that can come within the cutoff before the next
// build is at its nearest image; kImgPerPair (all six bits set): the entry's
// pairs need the nearest image pair by pair.
constexpr unsigned kNoMask = 0x3ffffffu;
constexpr unsigned kImgShift = 26u;
constexpr unsigned kImgPerPair = 0x3fu;

// Slot position of a padding slot.  Finite, so that the pair kernel's force
// products stay finite, and far outside every box, so that a padding slot
// fails every cutoff test; the pair kernel moves padding j slots to -kPadPos
// so that two padding slots are far apart as well.
constexpr double kPadPos = 1e15;

// Issue priority of a wavefront of the kernels that run beside the pair kernel
// (PME, bonded terms), above the pair kernel's default 0: the sequencer
// otherwise issues for the oldest wavefront first, and the pair kernel's
// persistent wavefronts are older than every kernel launched after it.
__device__ __forceinline__ void side_priority() { __builtin_amdgcn_s_setprio(2); }

// ------------------------------------------------------------ precision

// FP64 force accumulator: v = hi 2^-20 + lo 2^-74, each part summed exactly
// in a 64-bit integer, so a sum of contributions is the same whatever their
// order (the reference sums serially and is reproducible; double atomics are
// not).  Range |v| < 8.7e12, resolution 2^-74 (5e-23) per contribution.
struct Fix2 {
    long long hi, lo;
};

struct PrecFP64 {
    using real = double;
    using real2 = double2;
    using real4 = double4;
    using facc = Fix2;            // force accumulator element
    using gacc = long long;       // PME charge grid element, 2^48 fixed point
    static constexpr double grid_scale = 281474976710656.0;
    static constexpr bool mixed = false;
    static constexpr int pair_waves_per_simd = 1;   // minimum pair-kernel waves per SIMD the registers must allow
};

struct PrecMixed {
    using real = float;
    using real2 = float2;
    using real4 = float4;
    using facc = long long;       // 2^32 fixed point
    using gacc = long long;       // PME charge grid element, 2^32 fixed point
    static constexpr double grid_scale = 4294967296.0;
    static constexpr bool mixed = true;
    static constexpr int pair_waves_per_simd = 4;
    // Three pair-kernel waves per SIMD (the persistent grid's three blocks per
    // CU) at 112 VGPRs leave 176 of a SIMD's 512 to the PME kernels beside
    // them: a 768-thread plane-FFT block (three waves per SIMD at 56 VGPRs)
    // then fits; at 120 it does not, and PME waits for the pair kernel.
    static constexpr int pair_max_vgpr = 112;
};

__device__ __forceinline__ long long to_fixed(float v) {
    float s = v * 4294967296.0f;
    s = fminf(fmaxf(s, -9.2e18f), 9.2e18f);
    return __float2ll_rn(s);
}
__device__ __forceinline__ long long to_fixed(double v) {
    double s = v * kForceScale;
    s = fmin(fmax(s, -9.2e18), 9.2e18);
    return __double2ll_rn(s);
}

// the two parts of v: hi = v 2^20 rounded, lo = the rest times 2^74 rounded
// (v - hi 2^-20 is exact: the low bits of v)
__device__ __forceinline__ void fix2_parts(double v, long long& hi, long long& lo) {
    double s = v * 1048576.0;
    s = fmin(fmax(s, -9.2e18), 9.2e18);
    const double h = rint(s);
    hi = (long long)h;
    lo = (long long)rint((s - h) * 18014398509481984.0);     // (v - hi 2^-20) 2^74 = (s - h) 2^54
}
__device__ __forceinline__ void facc_add(Fix2* p, double v) {
    long long hi, lo;
    fix2_parts(v, hi, lo);
    atomicAdd(reinterpret_cast<unsigned long long*>(&p->hi), static_cast<unsigned long long>(hi));
    atomicAdd(reinterpret_cast<unsigned long long*>(&p->lo), static_cast<unsigned long long>(lo));
}
__device__ __forceinline__ void facc_add(long long* p, float v) {
    atomicAdd(reinterpret_cast<unsigned long long*>(p), static_cast<unsigned long long>(to_fixed(v)));
}
__device__ __forceinline__ void facc_add(long long* p, double v) {
    atomicAdd(reinterpret_cast<unsigned long long*>(p), static_cast<unsigned long long>(to_fixed(v)));
}
// Non-atomic add / store, for a location that no other thread writes meanwhile.
__device__ __forceinline__ void facc_set_add(Fix2* p, double v) {
    long long hi, lo;
    fix2_parts(v, hi, lo);
    p->hi += hi;
    p->lo += lo;
}
__device__ __forceinline__ void facc_set_add(long long* p, float v) { *p += to_fixed(v); }
__device__ __forceinline__ void facc_set(Fix2* p, double v) {
    long long hi, lo;
    fix2_parts(v, hi, lo);
    p->hi = hi;
    p->lo = lo;
}
__device__ __forceinline__ void facc_set(long long* p, float v) { *p = to_fixed(v); }
__device__ __forceinline__ double fix2_value(long long hi, long long lo) {
    return (double)hi * (1.0 / 1048576.0) + (double)lo * (1.0 / 18889465931478580854784.0);   // 2^-20, 2^-74
}
__device__ __forceinline__ double facc_get(const Fix2* p) { return fix2_value(p->hi, p->lo); }
__device__ __forceinline__ double facc_get(const long long* p) { return static_cast<double>(*p) * (1.0 / kForceScale); }

// Energy accumulation in 2^30 fixed point.  Every contribution is rounded to
// an integer on its own lane before any summation, so a system's energy is the
// same integer whatever the grouping of its terms into waves and blocks (alone
// or inside any batch).
__device__ __forceinline__ long long energy_fixed(double v) {
    double s = v * kEnergyScale;
    s = fmin(fmax(s, -9.2e18), 9.2e18);
    return __double2ll_rn(s);
}
// A system's sums are spread over kEnergySlots copies, by block: a million
// atoms' terms are 16,000 wavefronts, and that many atomics on one address took
// 1.8 ms where the kernel needs 30 us.  energy_sum_kernel adds the copies up.
constexpr int kEnergySlots = 64;
__device__ __forceinline__ void energy_add_fixed(long long* energy, int s, int term, long long v) {
    long long* e = energy + ((size_t)s * kEnergySlots + blockIdx.x % kEnergySlots) * E_NTERMS + term;
    atomicAdd(reinterpret_cast<unsigned long long*>(e), static_cast<unsigned long long>(v));
}

// ---------------------------------------------------------- wave helpers

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ long long wave_sum(long long v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Block-wide (<=1024 threads) sum of fixed-point energies into system s's term (one atomic per block).
__device__ __forceinline__ void block_energy_add(long long* energy, int s, int term, long long v) {
    __shared__ long long part[16];
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) part[w] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        long long t = 0;
        const int nw = (blockDim.x + 63) >> 6;
        for (int i = 0; i < nw; ++i) t += part[i];
        energy_add_fixed(energy, s, term, t);
    }
    __syncthreads();
}

// Adds v of the valid lanes to system s's term with one atomic per
// wavefront when all valid lanes belong to one system.  Every lane must call it.
__device__ __forceinline__ void wave_energy_add(long long* energy, int s, int term, double v, bool valid) {
    const unsigned long long m = __ballot(valid);
    if (m == 0ull) return;
    const long long q = valid ? energy_fixed(v) : 0ll;
    const int lead = __ffsll((long long)m) - 1;
    const int s0 = __shfl(s, lead, 64);
    if (__all(!valid || s == s0)) {
        const long long t = wave_sum(q);
        if ((int)(threadIdx.x & 63) == lead) energy_add_fixed(energy, s0, term, t);
    } else if (valid) {
        energy_add_fixed(energy, s, term, q);
    }
}

// Wave-local ordering of LDS traffic (lanes of one wavefront exchanging data
// through LDS; the other wavefronts of the block run independently).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Reference minimum image: one +-L correction (PeriodicBoundaryCondition.cpp:93-104),
// written with selects so that it compiles without branches.
__device__ __forceinline__ double min_image1(double d, double L) {
    // d - L, d + L or d, as one subtraction of +-L or 0
    const double n = fabs(d) > 0.5 * L ? copysign(L, d) : 0.0;
    return d - n;
}
__device__ __forceinline__ float min_image1(float d, float L) {
    const float h = 0.5f * L;
    const float up = d - L, dn = d + L;
    return d > h ? up : (d < -h ? dn : d);
}

// The slot position the mixed path's pair and PME kernels read: the build-time
// wrapped position plus the displacement since the build, continuous between
// builds (an atom's wrapped position jumps by L when it crosses the box), so
// that a j-cluster's periodic image found at the build holds until the next
// one.  (The FP64 path reads the positions themselves and takes the nearest
// image pair by pair with the reference's arithmetic.)
__device__ __forceinline__ void continuous_position(const SysDev& d, double x, double y, double z, double xb,
                                                    double yb, double zb, double* p) {
    p[0] = xb + min_image1(x - xb, d.L[0]);
    p[1] = yb + min_image1(y - yb, d.L[1]);
    p[2] = zb + min_image1(z - zb, d.L[2]);
}

// The FP64 direct-space term, x = alpha r: erfc(x) / r and its force factor
// (erfc(x) + 2 x exp(-x^2) / sqrt(pi)) / r^3 with
//     erfc(x) = exp(-x^2) E(x),  E(x) = exp(x^2) erfc(x),
// so that the force's bracket is exp(-x^2) (E(x) + 2 x / sqrt(pi)): positive terms
// throughout, as accurate at the cutoff, where the bracket is 1e-3, as near it.
// kErfcx: E over x^2 <= kErfSeriesMax in powers of u = x / sqrt(2) - 1; kExp2m1:
// (2^f - 1) / f over |f| <= 1/2 in powers of f; both Chebyshev interpolants computed
// with 60 digits, off by 7e-17 of E + 2 x / sqrt(pi) and 2e-17 of 2^f.  RMS error on
// the device by ranges of r from 0.1 to 1 nm at alpha = 2.63 and 2.82 / nm, of the
// force factor 1.3e-16 to 1.7e-16 of itself, of the energy 1.2e-16 to 2.9e-16.  The
// library's erfc, exp, sqrt and division: 2.0e-16 to 7.5e-16 and 1.2e-16 to 7.9e-16.
// The difference 1 / r^3 - alpha^3 B(x^2) (B below) takes 17 instructions less, and
// near the cutoff it is off by 5e-14 to 2.5e-13 of itself, its energy by 1e-12.
constexpr double kErfSeriesMax = 8.0;
constexpr double kErfcx[25] = {
    3.36204002446341188e-01, -2.50953111820364894e-01, 1.70501781251950396e-01, -1.07268440757989941e-01,
    6.32333404940961935e-02, -3.52280802078909563e-02, 1.86701735210091091e-02, -9.46166101025903983e-03,
    4.60425629257135618e-03, -2.15884616869028599e-03, 9.78163787719972793e-04, -4.29340898122935783e-04,
    1.82942140905975538e-04, -7.58089997705473317e-05, 3.06059328780922143e-05, -1.20672317082442645e-05,
    4.64191805310459557e-06, -1.72783460106342884e-06, 6.37418316159805450e-07, -2.48576005282112033e-07,
    8.73588365632618443e-08, -1.87243078346221425e-08, 6.64889187949806792e-09, -6.46832001623310008e-09,
    2.09039891445411742e-09,
};
constexpr double kExp2m1[11] = {
    6.93147180559945286e-01, 2.40226506959100972e-01, 5.55041086648215970e-02, 9.61812910760688825e-03,
    1.33335581464169356e-03, 1.54035304417360499e-04, 1.52527338298361192e-05, 1.32154425879216893e-06,
    1.01780624458457737e-07, 7.07258594926922339e-09, 4.45496059818651856e-10,
};
// erf(x) / x and (erf(x) - 2 x exp(-x^2) / sqrt(pi)) / x^3, entire functions of x^2,
// in powers of x^2 / 4 - 1: the same two quantities by another route, which the
// coefficients above are checked against as this header is compiled.
constexpr double kErfA[22] = {
    4.97661132509476356e-01, -2.38497073577692176e-01, 1.58205819829175892e-01, -1.04282202718857353e-01,
    6.36909469069244089e-02, -3.52770678385127892e-02, 1.76407892660984562e-02, -7.98271979410423126e-03,
    3.28479326482311422e-03, -1.23607961382126200e-03, 4.27785551802345595e-04, -1.36889844490136983e-04,
    4.07025421452981889e-05, -1.12958817428514669e-05, 2.93769052661021184e-06, -7.18648852211750148e-07,
    1.66084339812328716e-07, -3.62878189045594433e-08, 7.39320016599416468e-09, -1.46104235443290689e-09,
    3.30946272093021783e-10, -5.91195428737397584e-11,
};
constexpr double kErfB[23] = {
    1.19248536788846074e-01, -1.58205819829177086e-01, 1.56423304078287251e-01, -1.27381893813754754e-01,
    8.81926695962295254e-02, -5.29223678004963477e-02, 2.79395192802459787e-02, -1.31391730358153547e-02,
    5.56235825464281540e-03, -2.13892789596149347e-03, 7.52894182292228559e-04, -2.44214774792607923e-04,
    7.34231151212477582e-05, -2.05648756537177909e-05, 5.39009625215538716e-06, -1.32724573457226400e-06,
    3.08155303970224502e-07, -6.77366262557539614e-08, 1.41082605777249840e-08, -2.74907686745350267e-09,
    5.19796833377220498e-10, -1.12077170695342987e-10, 1.92301651041994177e-11,
};
constexpr double poly(const double* c, int n, double u) {
    double r = 0.0;
    for (int k = n - 1; k >= 0; --k) r = r * u + c[k];
    return r;
}
constexpr double poly_difference(double x) {       // of 1 - x A and 1 - x^3 B from exp(-x^2) times E and E + 2 x / sqrt(pi)
    const double s = x * x, t = -s / 0.69314718055994530942;
    const int k = (int)(t - 0.5);
    double ex = 1.0 + (t - k) * poly(kExp2m1, 11, t - k);
    for (int i = 0; i > k; --i) ex *= 0.5;
    const double e = poly(kErfcx, 25, x / 1.41421356237309504880 - 1.0), u = 0.25 * s - 1.0;
    const double energy = 1.0 - x * poly(kErfA, 22, u) - ex * e;
    const double force = 1.0 - x * s * poly(kErfB, 23, u) - ex * (e + kTwoOverSqrtPi * x);
    const double a = energy < 0 ? -energy : energy, b = force < 0 ? -force : force;
    return a > b ? a : b;
}
static_assert(poly_difference(0.01) < 4e-15 && poly_difference(0.6) < 4e-15 && poly_difference(1.3) < 4e-15 &&
                  poly_difference(2.0) < 4e-15 && poly_difference(2.8) < 4e-15,
              "the two routes to the direct-space term differ");
// a b + c with the constant c in scalar registers.  Written out because the
// compiler otherwise picks the two-address form, whose addend is its result: a
// copy of the constant, kept in vector registers, before every step.
__device__ __forceinline__ double fma_const(double a, double b, double c) {
    double r;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
    return r;
}
// 2^f - 1 and E at u: three chains of multiply-adds (E's even and odd powers), a step
// of each in turn
__device__ __forceinline__ void direct_space_series(double f, double u, double& fp, double& e) {
    const double u2 = u * u;
    double p = kExp2m1[10], o = kErfcx[23];
    e = kErfcx[24];
#pragma unroll
    for (int k = 11; k >= 0; --k) {
        e = fma_const(e, u2, kErfcx[2 * k]);
        if (k > 0) o = fma_const(o, u2, kErfcx[2 * k - 1]);
        if (k < 10) p = fma_const(p, f, kExp2m1[k]);
    }
    e = fma(o, u, e);
    fp = p * f;
}

// r^2 without contraction, left-to-right as Coords3D::dot (Coords3D.h:116-124).
__device__ __forceinline__ double dot_rn(double x, double y, double z) {
    return __dadd_rn(__dadd_rn(__dmul_rn(x, x), __dmul_rn(y, y)), __dmul_rn(z, z));
}

// Cross-lane sums on a 64-wide wavefront without LDS: DPP row rotate for
// lane^8, permlane16/32 swaps for lane^16 and lane^32, DPP quad permutes and
// the half-row mirror for lane^1, lane^2 and the 8-lane halves.
__device__ __forceinline__ int dpp_ror8(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, false); }
__device__ __forceinline__ int dpp_xor1(int v) { return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false); }
__device__ __forceinline__ int dpp_xor2(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false); }
__device__ __forceinline__ int dpp_hmirror(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false); }

// x, y and z summed over the lanes with the same l & 7 (by 8, 16, then 32 lanes
// apart): the sum of x on lanes 0-15, of y on 16-31, of z on 32-63 (each at every
// lane of its l & 7).  Two of them share a swap and an addition where one alone
// wastes half: 10 instructions, where three sums of their own take 21.
template <typename real>
__device__ __forceinline__ void swap16(real& a, real& b);      // odd rows of 16 lanes of a with even ones of b
template <typename real>
__device__ __forceinline__ void swap32(real& a, real& b);      // upper half of a with the lower one of b
template <>
__device__ __forceinline__ void swap16(float& a, float& b) {
    auto p = __builtin_amdgcn_permlane16_swap(__float_as_int(a), __float_as_int(b), false, false);
    a = __int_as_float(p[0]);
    b = __int_as_float(p[1]);
}
template <>
__device__ __forceinline__ void swap32(float& a, float& b) {
    auto p = __builtin_amdgcn_permlane32_swap(__float_as_int(a), __float_as_int(b), false, false);
    a = __int_as_float(p[0]);
    b = __int_as_float(p[1]);
}
template <>
__device__ __forceinline__ void swap16(double& a, double& b) {
    auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    a = __hiloint2double(h[0], l[0]);
    b = __hiloint2double(h[1], l[1]);
}
template <>
__device__ __forceinline__ void swap32(double& a, double& b) {
    auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    a = __hiloint2double(h[0], l[0]);
    b = __hiloint2double(h[1], l[1]);
}
__device__ __forceinline__ float add_ror8(float v) { return v + __int_as_float(dpp_ror8(__float_as_int(v))); }
__device__ __forceinline__ double add_ror8(double v) {
    return v + __hiloint2double(dpp_ror8(__double2hiint(v)), dpp_ror8(__double2loint(v)));
}
template <typename real>
__device__ __forceinline__ real sum3_stride8(real x, real y, real z) {
    x = add_ror8(x);
    y = add_ror8(y);
    z = add_ror8(z);
    swap16(x, y);           // x: rows 0, 2 of x in rows 0, 2, of y in 1, 3; y: rows 1, 3
    real xy = x + y, z2 = z;
    swap16(z, z2);
    z += z2;
    swap32(xy, z);          // xy: rows 0, 1 of both; z: rows 2, 3
    return xy + z;
}
// sum over the 8 lanes l & ~7 .. l | 7
__device__ __forceinline__ float sum_group8(float v) {
    v += __int_as_float(dpp_xor1(__float_as_int(v)));
    v += __int_as_float(dpp_xor2(__float_as_int(v)));
    v += __int_as_float(dpp_hmirror(__float_as_int(v)));
    return v;
}
__device__ __forceinline__ double sum_group8(double v) {
    v += __hiloint2double(dpp_xor1(__double2hiint(v)), dpp_xor1(__double2loint(v)));
    v += __hiloint2double(dpp_xor2(__double2hiint(v)), dpp_xor2(__double2loint(v)));
    v += __hiloint2double(dpp_hmirror(__double2hiint(v)), dpp_hmirror(__double2loint(v)));
    return v;
}

// Before a pair kernel of nb blocks, threads x < 8: XCD x's range of the n
// chunks, in proportion to its blocks (b % 8 == x), and its counter past the
// first chunk of each of its wavefronts.
__device__ __forceinline__ void pool_begin(int x, int n, int* pool, int nb) {
    if (x >= 8) return;
    auto first = [&](int y) {
        const int b = y * (nb >> 3) + min(y, nb & 7);      // blocks of the XCDs below y
        return (n / nb) * b + (n % nb) * b / nb;
    };
    int* p = pool + x * kPoolStride;
    p[kPoolFirst] = first(x);
    p[kPoolEnd] = first(x + 1);
    p[0] = first(x) + ((nb >> 3) + (x < (nb & 7) ? 1 : 0)) * kPairWaves;
}

// XCD-aware block order: consecutive work items land on one XCD (8 XCDs,
// round-robin dispatch), so neighbouring super-clusters share an L2.
__device__ __forceinline__ int xcd_remap(int b, int nblocks) {
    const int per = (nblocks + 7) >> 3;
    const int xcd = b & 7, k = b >> 3;
    const int full = nblocks & 7 ? (nblocks & 7) : 8;   // XCDs that get `per` blocks
    int base = (xcd < full) ? xcd * per : full * per + (xcd - full) * (per - 1);
    int r = base + k;
    return r < nblocks ? r : b;
}

}  // namespace nx
