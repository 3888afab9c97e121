// nonbonded.hip -- real-space LJ + erfc-Coulomb pair kernel, exclusion
// correction, and the explicit pair-set export.
//
// Physics follows NonbondedForce::DirectForcesAndEnergy and
// CalculateExclusionEnergyAndForces (core/baseline/src/Forces/
// NonbondedForce.cpp:530-585, :590-630) with the modified parameters of
// NonbondedParamsModifier (:504-513): sigma_ij = sig_i/2 + sig_j/2 and
// eps'_i = 2 sqrt(eps_i), so E_LJ = eps'_i eps'_j (s^6 - 1) s^6.
//
// Work decomposition: the list is cut into chunks of up to kChunkEntries
// entries of one super-cluster (up to 8 clusters of 8 atoms); wavefronts claim
// chunks one at a time from their XCD's range.  Lane l = 8*ia + ja holds i-atom
// ia of the current i-cluster and j-atom ja of the current j-cluster, so one
// (i-cluster, j-cluster) tile is 64 pairs in one VALU pass.  i-forces stay in
// registers over the chunk; j-forces are reduced across the 8 lanes sharing ja
// and added once per entry.  The FP64 path tests r^2 < rc^2 with the
// reference's minimum image and an uncontracted left-to-right dot product, so
// its pair set is bit-identical to the reference's.
#include <algorithm>

#include "nx_device.h"
#include "nx_engine.h"

namespace nx {

// Abramowitz & Stegun 7.1.26: erfc(x) ~ t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) exp(-x^2),
// t = 1 / (1 + p x), |error| <= 1.5e-7 for x >= 0.
constexpr double kAsP = 0.3275911;
__device__ __forceinline__ float erfc_as_t(float t, float expmx2) {
    const float a1 = 0.254829592f, a2 = -0.284496736f, a3 = 1.421413741f, a4 = -1.453152027f,
                a5 = 1.061405429f;
    return t * (a1 + t * (a2 + t * (a3 + t * (a4 + t * a5)))) * expmx2;
}

constexpr double kLog2E = 1.4426950408889634;   // log2(e)

// Per-system constants of the mixed pair function, formed once per chunk so
// that the per-pair work starts from r and r^2 directly.
struct MixedPair {
    float ap;       // p alpha: the A&S variable is t = 1 / (1 + p alpha r)
    float ek;       // -alpha^2 log2(e): exp(-(alpha r)^2) = 2^(ek r^2)
    float cg;       // 2 alpha / sqrt(pi)
    float sw_on;    // switch start, < 0 without a switch
    float sw_inv;   // 1 / (rc - r_switch)
    float sw_rc;    // the cutoff: 1 - t = (rc - r) sw_inv
    float sw_d;     // -30 / (rc - r_switch): dsv/dr = sw_d t^2 (1 - t)^2
};

__device__ __forceinline__ MixedPair mixed_pair_const(const SysDev& d) {
    MixedPair c;
    c.ap = (float)(kAsP * d.alpha);
    c.ek = (float)(-d.alpha * d.alpha * kLog2E);
    c.cg = (float)(kTwoOverSqrtPi * d.alpha);
    c.sw_on = (float)d.sw_on;
    c.sw_inv = (float)d.sw_inv;
    c.sw_rc = (float)d.rc;
    c.sw_d = (float)(-30.0 * d.sw_inv);
    return c;
}

// Mixed path: FP32 pair math.  Returns dE/dr / r (force = d * value on i).
// With erfc(alpha r) = ex u (ex = exp(-(alpha r)^2), u the A&S polynomial in
// t), the Coulomb part qq (cg ex + erfc / r) / r^2 is qq ex (cg + u / r) / r^2,
// so that it joins the LJ part in one multiply-add before the common 1/r^2.
__device__ __forceinline__ float pair_mixed(float r2, float qq, float sig, float epsij, const MixedPair& c,
                                            float& ecoul, float& elj) {
    const float inv_r = __builtin_amdgcn_rsqf(r2);
    const float r = r2 * inv_r;
    const float inv_r2 = inv_r * inv_r;
    const float ex = __builtin_amdgcn_exp2f(c.ek * r2);                  // exp(-(alpha r)^2)
    const float u = erfc_as_t(__builtin_amdgcn_rcpf(fmaf(c.ap, r, 1.0f)), 1.0f);
    const float cy = ex * fmaf(inv_r, u, c.cg);
    const float s2 = sig * sig * inv_r2;
    const float s6 = s2 * s2 * s2;
    float le = epsij * (s6 - 1.0f) * s6;
    float dl = epsij * (12.0f * s6 - 6.0f) * s6;                          // r^2 times its dE/dr / r
    if (c.sw_on >= 0.f) {   // uniform per system
        // sv = 1 - 10 t^3 + 15 t^4 - 6 t^5 = w^3 (1 + 3 t + 6 t^2) with w = 1 - t,
        // dsv/dt = -30 t^2 w^2.  The factored form keeps FP32 accuracy where sv
        // is small (r near rc); w = 1 inside r_switch gives sv = 1, sd = 0.
        const float w = fminf((c.sw_rc - r) * c.sw_inv, 1.0f);
        const float t = 1.0f - w;
        const float sv = w * w * w * fmaf(t, fmaf(t, 6.0f, 3.0f), 1.0f);
        const float uw = t * w;
        const float sd = c.sw_d * uw * uw;
        dl = sv * dl - le * sd * r;
        le *= sv;
    }
    ecoul = qq * inv_r * ex * u;
    elj = le;
    return fmaf(qq, cy, dl) * inv_r2;
}

// FP64 path inside the range of kErfcx: the direct-space term as exp(-(alpha r)^2)
// times a polynomial (nx_device.h), without a library function or a division.  1/r
// is the hardware's reciprocal square root with one third-order step (its first
// error, 2^-26 or less, goes to the third power), 1/r^2 its square with one
// second-order step.  The kernel is bound by its vector instructions.  Its launch on
// 100,000 atoms alone: 307 us; with library erfc, exp, sqrt and division 469; with
// the difference 1/r^3 - alpha^3 B, which loses two digits near the cutoff, 260
// (24,000 atoms: 98, 165, 84; a step 133, 199, 118).
struct EwaldFit {
    double ex, ex_lo, u, q;      // as SysDev::ew_*
};
template <bool ENERGY>
__device__ __forceinline__ double pair_fp64_series(double r2, double qq, double sig, double epsij, const EwaldFit& w,
                                                   double sw_on, double sw_inv, double& ecoul, double& elj) {
#pragma clang fp contract(off)      // the same operations in both kernels below
    double y = __builtin_amdgcn_rsq(r2);
    const double err = fma(-(r2 * y), y, 1.0);
    y = fma(y * err, fma(0.375, err, 0.5), y);
    double y2 = y * y;
    y2 = fma(y2, fma(-r2, y2, 1.0), y2);
    const double r = r2 * y;
    // exp(-(alpha r)^2) = 2^k (1 + fp): k the integer nearest to the exponent in base
    // two, in the low bits of the sum with 1.5 2^52; the rest of it, rounded once
    const double big = fma(r2, -w.ex, 6755399441055744.0);
    const double f = fma(r2, -w.ex_lo, fma(r2, -w.ex, -(big - 6755399441055744.0)));
    double fp, e;
    direct_space_series(f, fma(r, w.u, -1.0), fp, e);
    const double q = fma(r, w.q, e);
    auto scaled = [&](double v) {      // v of 0.1 to 6 times 2^k, k of -12 to 0
        return __hiloint2double(__double2hiint(v) + (__double2loint(big) << 20), __double2loint(v));
    };
    const double cf = qq * (scaled(fma(fp, q, q)) * (y2 * y));
    double s2 = sig * y;
    s2 *= s2;
    const double s6 = s2 * s2 * s2;
    const double es = epsij * s6;
    double lf = es * fma(12.0, s6, -6.0) * y2;
    double le = es * (s6 - 1.0);
    if (sw_on >= 0.0) {
        const double t = r > sw_on ? (r - sw_on) * sw_inv : 0.0;
        const double sv = fma(t * t * t, fma(t, fma(-6.0, t, 15.0), -10.0), 1.0);
        const double sd = t * t * fma(t, fma(-30.0, t, 60.0), -30.0) * sw_inv;
        lf = fma(sv, lf, -(le * sd * y));
        le *= sv;
    }
    if constexpr (ENERGY) ecoul = qq * (scaled(fma(fp, e, e)) * y);
    elj = le;
    return cf + lf;
}

// FP64 path: the reference's formulas with library erfc/exp.
__device__ __forceinline__ double pair_fp64(double r2, double qq, double sig, double epsij, double alpha,
                                            double sw_on, double sw_inv, double& ecoul, double& elj) {
    const double r = sqrt(r2);
    const double inv_r = 1.0 / r;
    const double ar = alpha * r;
    const double erfcv = erfc(ar);
    const double ex = exp(-ar * ar);
    double dEdR = qq * inv_r * inv_r * inv_r * (erfcv + 2.0 * ar * ex / kSqrtPi);
    double s2 = sig * inv_r;
    s2 *= s2;
    const double s6 = s2 * s2 * s2;
    double le = epsij * (s6 - 1.0) * s6;
    double sv = 1.0, sd = 0.0;
    if (sw_on >= 0.0 && r > sw_on) {
        const double t = (r - sw_on) * sw_inv;
        sv = 1.0 + t * t * t * (-10.0 + t * (15.0 - t * 6.0));
        sd = t * t * (-30.0 + t * (60.0 - t * 30.0)) * sw_inv;
    }
    dEdR += sv * epsij * (12.0 * s6 - 6.0) * s6 * inv_r * inv_r;
    if (sw_on >= 0.0) {
        dEdR -= le * sd * inv_r;
        le *= sv;
    }
    ecoul = qq * inv_r * erfcv;
    elj = le;
    return dEdR;
}

// Lanes l = 8 * ia + ja with ja <= ia: on a diagonal tile (i and j the same
// cluster) these are the self pairs and the half counted from the other side.
constexpr unsigned long long lower_triangle_mask() {
    unsigned long long m = 0ull;
    for (int l = 0; l < 64; ++l)
        if ((l & 7) <= (l >> 3)) m |= 1ull << l;
    return m;
}
constexpr unsigned long long kLowerTriangle = lower_triangle_mask();

template <class P, bool ENERGY, bool ALL_SERIES>
__device__ __forceinline__ void pair_body(const SysDev* __restrict__ sd, const int* __restrict__ prefix,
                                                   int nsys, const int4* __restrict__ chunks,
                                                   const uint2* __restrict__ list,
                                                   const unsigned long long* __restrict__ emask,
                                                   const typename P::real4* __restrict__ pos,
                                                   const typename P::real2* __restrict__ lj, typename P::facc* FX,
                                                   typename P::facc* FY, typename P::facc* FZ, long long* energy,
                                                   int* __restrict__ pool) {
    using real = typename P::real;
    using real4 = typename P::real4;
    using real2 = typename P::real2;
    // the wavefront index is the same on every lane: in a scalar register, the
    // chunk and list-entry indices derived from it are scalar too, and so are
    // the loads of chunk records and list words
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, ia = lane >> 3,
              ja = lane & 7;
    __shared__ real4 ipos_s[kPairWaves][64];
    __shared__ real2 ilj_s[kPairWaves][64];
    __shared__ real jf_s[kPairWaves][kChunkEntries * 3 * 8];
    __shared__ uint2 jw_s[kPairWaves][kChunkEntries];
    real4* ipos = ipos_s[w];
    real2* ilj = ilj_s[w];
    real* jf = jf_s[w];
    const bool j_out = lane < 48 && (lane & 8) == 0;     // lanes that hold a j force (sum3_stride8)
    uint2* jw = jw_s[w];

    // Each XCD's wavefronts (blocks b with b % 8 equal, as the hardware hands
    // them out) share a contiguous range of the batch's chunks, in proportion to
    // their number, and claim chunks one at a time from an XCD counter.  A fixed
    // range per wavefront finished 1.3x apart on one CU: the sequencer issues
    // for its oldest wavefront first, so the first block placed on a CU ran
    // ahead of the third.  Adjacent chunks are spatial neighbours, so an XCD's
    // L2 sees one region.  A wavefront's first chunk is fixed (the counters start
    // past those), which keeps the first claims' round trip out of the small
    // systems' time.  Every chunk is done whole by one wavefront: its arithmetic
    // does not depend on who does it or when.
    int* counter = pool + (blockIdx.x & 7) * kPoolStride;
    const int hi = __builtin_amdgcn_readfirstlane(counter[kPoolEnd]);
    // lane 0 claims the next chunk; the result is read (and waited for) later.  An
    // increment, not an addition of 1: the compiler aggregates additions over the
    // wavefront, and the code it makes for that waits for the result at once.
    auto claim = [&]() {
        int t = 0;
        if (lane == 0) t = (int)atomicInc(reinterpret_cast<unsigned*>(counter), 0xffffffffu);
        return t;
    };
    auto claimed = [&](int t) { return __builtin_amdgcn_readfirstlane(t); };
    const real ke = (real)kOne4PiEps0;

    // Everything a chunk needs from memory before its first pair: the chunk
    // record, the i data of its clusters and its first list entry.  The next
    // chunk's copy is loaded before this chunk's force atomics are issued, so
    // the wait for it does not sit behind them (one in-order vmem counter).
    struct Pre {
        int s;
        int4 ch;
        real4 p;
        real2 l;
        uint2 words;     // lane l < kChunkEntries: the chunk's list word l
        uint2 ent;
        real4 pj;
        real2 ljj;
    };
    auto fetch = [&](int g) {
        Pre q;
        int lo = 0, hi = nsys - 1;     // largest s with prefix[s] <= g
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (prefix[mid] <= g) lo = mid; else hi = mid - 1;
        }
        q.s = lo;
        q.ch = chunks[sd[lo].chunk_off + (g - prefix[lo])];
        if ((lane >> 3) < q.ch.y) {
            q.p = pos[q.ch.x * 8 + lane];
            q.l = lj[q.ch.x * 8 + lane];
        } else {
            q.p.x = q.p.y = q.p.z = q.p.w = 0;
            q.l.x = q.l.y = 0;
        }
        // the first entry and its j data (none for a chunk without entries)
        q.words = make_uint2(0u, kNoMask);
        if (lane < q.ch.w - q.ch.z) q.words = list[q.ch.z + lane];
        q.ent = make_uint2(0u, kNoMask);
        q.pj.x = q.pj.y = q.pj.z = q.pj.w = 0;
        q.ljj.x = q.ljj.y = 0;
        if (q.ch.w > q.ch.z) {
            q.ent = list[q.ch.z];
            const int sj = (int)(q.ent.x & 0xffffffu) * 8 + ja;
            q.pj = pos[sj];
            q.ljj = lj[sj];
        }
        return q;
    };

    int e_sys = -1;
    long long ec_sum = 0, el_sum = 0;
    auto flush_energy = [&]() {
        if (e_sys < 0) return;
        ec_sum = wave_sum(ec_sum);
        el_sum = wave_sum(el_sum);
        if (lane == 0) {
            energy_add_fixed(energy, e_sys, E_COUL, ec_sum);
            energy_add_fixed(energy, e_sys, E_LJ, el_sum);
        }
        ec_sum = el_sum = 0;
    };
    // The mixed path prefetches the next chunk across the flush below; the FP64
    // kernel is register-bound and fetches at the top of each chunk.
    int g = __builtin_amdgcn_readfirstlane(counter[kPoolFirst]) + (int)(blockIdx.x >> 3) * kPairWaves + w;
    Pre cur;
    if (P::mixed && g < hi) cur = fetch(g);
    while (g < hi) {
        if constexpr (!P::mixed) cur = fetch(g);
        // chunk values are the same on every lane: keep them in scalar registers
        const int s = __builtin_amdgcn_readfirstlane(cur.s);
        const int fc = __builtin_amdgcn_readfirstlane(cur.ch.x), ncl = __builtin_amdgcn_readfirstlane(cur.ch.y);
        const int e0 = __builtin_amdgcn_readfirstlane(cur.ch.z), e1 = __builtin_amdgcn_readfirstlane(cur.ch.w);
        // the claim of the chunk after this one: inside the entry loop, or here for
        // a chunk without entries (the loop below then does not run)
        int tk = 0;
        if (e1 <= e0) tk = claim();
        const real Lx = (real)sd[s].L[0], Ly = (real)sd[s].L[1], Lz = (real)sd[s].L[2];
        const real iLx = (real)sd[s].invL[0], iLy = (real)sd[s].invL[1], iLz = (real)sd[s].invL[2];
        const real rc2 = (real)sd[s].rc2;
        const real alpha = (real)sd[s].alpha;
        const real sw_on = (real)sd[s].sw_on, sw_inv = (real)sd[s].sw_inv;
        const bool series = (double)alpha * (double)alpha * (double)rc2 <= kErfSeriesMax;   // FP64 path only
        EwaldFit ew = {sd[s].ew_exp, sd[s].ew_exp_lo, sd[s].ew_u, sd[s].ew_q};
        // in a vector register: an instruction takes one scalar operand, and the first
        // one that reads it adds a constant
        if constexpr (!P::mixed) asm("" : "+v"(ew.ex));
        const MixedPair mpc = mixed_pair_const(sd[s]);   // mixed path only
        {
            real4 p = cur.p;
            p.w *= ke;
            ipos[lane] = p;
            ilj[lane] = cur.l;
            if (lane < kChunkEntries) jw[lane] = cur.words;
        }
        wave_lds_sync();
        real fxi[8], fyi[8], fzi[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) fxi[k] = fyi[k] = fzi[k] = 0;
        double ec_acc = 0.0, el_acc = 0.0;

        // software pipeline: the j data of entry e+1 loads while entry e computes.
        // The chunk's list words sit in LDS (written above with the i data); the
        // word of entry e+1 is read at the end of entry e-1.  A scalar load of it
        // would be simpler, but scalar loads return out of order, so every wait
        // for an LDS read issued after one would also wait for it.
        unsigned ex_n = __builtin_amdgcn_readfirstlane(cur.ent.x), ey_n = __builtin_amdgcn_readfirstlane(cur.ent.y);
        uint2 wv = jw[1];
        real4 pj = cur.pj;
        real2 lj_j = cur.ljj;
        for (int e = e0; e < e1; ++e) {
            // the list word is the same on every lane: in scalar registers, the
            // per-cluster tests below are scalar branches
            const unsigned ex = ex_n;
            const unsigned ey = ey_n;
            ex_n = __builtin_amdgcn_readfirstlane(wv.x);
            ey_n = __builtin_amdgcn_readfirstlane(wv.y);
            const int cj = (int)(ex & 0xffffffu);
            const unsigned im = ex >> 24;
            const unsigned eid = ey & kNoMask, img = ey >> kImgShift;
            // exclusion bits of the 8 cluster pairs, one load before the cluster loop
            unsigned long long em[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) em[k] = 0ull;
            if (eid != kNoMask) {
#pragma unroll
                for (int k = 0; k < 8; ++k) em[k] = emask[(size_t)eid * 8 + k];
            }
            // mixed path: the j cluster at the entry's periodic image (the list build
            // checked that it is the nearest image of every pair that can be within
            // the cutoff), or, for an entry whose pairs need it, the nearest image
            // pair by pair below; the FP64 path takes it pair by pair with the
            // reference's arithmetic, so that its cutoff test is the reference's bit
            // for bit.  Padding j slots move to -kPadPos, far from every i slot
            // (padding ones at +kPadPos included).
            const bool per_pair = !P::mixed || img == kImgPerPair;
            real4 pjs;
            {
                // +1, -1 or 0 boxes, selected in scalar registers (the pair-by-pair
                // marker has both bits of an axis: 0)
                auto boxes = [&](unsigned both, unsigned plus) {
                    const unsigned b = img & both;
                    const unsigned one = b == plus ? 0x3f800000u : (b == 2u * plus ? 0xbf800000u : 0u);
                    return __uint_as_float(one);
                };
                real x = pj.x;
                pjs.y = pj.y;
                pjs.z = pj.z;
                if constexpr (P::mixed) {
                    x = fmaf(boxes(3u, 1u), Lx, x);
                    pjs.y = fmaf(boxes(12u, 4u), Ly, pjs.y);
                    pjs.z = fmaf(boxes(48u, 16u), Lz, pjs.z);
                }
                pjs.x = (pj.x > (real)(0.5 * kPadPos)) ? (real)(-kPadPos) : x;
                pjs.w = pj.w;
            }
            real4 pj_n = pj;
            real2 lj_n = lj_j;
            if (e + 1 < e1) {
                const int sjn = (int)(ex_n & 0xffffffu) * 8 + ja;
                pj_n = pos[sjn];
                lj_n = lj[sjn];
            }
            // claim the next chunk two entries before this chunk's end, after the
            // loads above: the waits for them then do not wait for the atomic (the
            // vector memory counter drains in issue order), and its round trip
            // overlaps the last entries' pairs
            if (e == max(e0, e1 - 2)) tk = claim();
            real fxj = 0, fyj = 0, fzj = 0;
            // i data of each cluster is read from LDS at its tile (reading it one
            // tile ahead cost 6 registers and measured slower; the other waves on
            // the SIMD hide the read).  The empty asm makes the LDS index opaque per
            // entry: otherwise the compiler hoists all 8 clusters' reads out of the
            // entry loop and holds them in 48 more registers, which spills.
            int io = ia;
            asm volatile("" : "+v"(io));
            const real4* ipe = ipos + io;
            const real2* ile = ilj + io;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (im & (1u << k)) {
                    const real4 pi = ipe[k * 8];
                    const real2 li = ile[k * 8];
                    // excluded lanes, as a wave-wide bit mask: listed exclusions, and on
                    // the diagonal tile the pairs with ja <= ia (self pairs and the other half)
                    const unsigned long long xm = em[k] | (cj == fc + k ? kLowerTriangle : 0ull);
                    real dx = pi.x - pjs.x, dy = pi.y - pjs.y, dz = pi.z - pjs.z;
                    if (per_pair) {     // a uniform branch
                        if constexpr (P::mixed) {
                            // nearest image by rounding (equal to the one-correction rule for
                            // |d| < 1.5 L); a padding slot keeps its distance of ~kPadPos in x
                            const real cx = dx - Lx * rintf(dx * iLx);
                            dx = fabsf(dx) < (real)(0.5 * kPadPos) ? cx : dx;
                            dy -= Ly * rintf(dy * iLy);
                            dz -= Lz * rintf(dz * iLz);
                        } else {
                            dx = min_image1(dx, Lx);
                            dy = min_image1(dy, Ly);
                            dz = min_image1(dz, Lz);
                        }
                    }
                    real r2;
                    if constexpr (P::mixed) r2 = dx * dx + dy * dy + dz * dz;
                    else r2 = dot_rn(dx, dy, dz);
                    // lane l is on when bit l of the cutoff ballot is set and bit l of the
                    // exclusion mask is clear: the mask logic runs in scalar registers
                    const unsigned long long onm = __builtin_amdgcn_ballot_w64(r2 < rc2) & ~xm;
                    // a tile with no pair inside the cutoff (kept by the list's outer
                    // radius) skips the pair arithmetic: a uniform branch
                    if constexpr (P::mixed) {
                        if (onm == 0ull) continue;
                    }
                    const bool on = __builtin_amdgcn_inverse_ballot_w64(onm);
                    real ecv, elv, dEdR;
                    if constexpr (P::mixed) {
                        // evaluated on every lane; lanes that are off (incl. r2 = 0) select zero
                        dEdR = pair_mixed(r2, pi.w * pjs.w, li.x + lj_j.x, li.y * lj_j.y, mpc, ecv, elv);
                        dEdR = on ? dEdR : 0.0f;
                    } else {
                        dEdR = 0;
                        ecv = elv = 0;
                        if (on) {
                            const real qq = pi.w * pjs.w, sg = li.x + lj_j.x, ep = li.y * lj_j.y;
                            if (ALL_SERIES || series) dEdR = pair_fp64_series<ENERGY>(r2, qq, sg, ep, ew, sw_on, sw_inv, ecv, elv);
                            else dEdR = pair_fp64(r2, qq, sg, ep, alpha, sw_on, sw_inv, ecv, elv);
                        }
                    }
                    // every displacement is finite (padding slots included), so the
                    // zero of an off lane gives zero force
                    const real fx = dx * dEdR, fy = dy * dEdR, fz = dz * dEdR;
                    fxi[k] += fx; fyi[k] += fy; fzi[k] += fz;
                    fxj -= fx; fyj -= fy; fzj -= fz;
                    if constexpr (ENERGY) {
                        if (on) { ec_acc += (double)ecv; el_acc += (double)elv; }
                    }
                }
            }
            const real fj = sum3_stride8(fxj, fyj, fzj);
            // staged in LDS: no global atomics inside the loop, so waiting for the
            // prefetched loads never waits behind atomics
            const int el = e - e0;
            if (j_out) jf[el * 24 + (lane >> 4) * 8 + ja] = fj;
            if (e + 2 < e1) wv = jw[el + 2];
            pj = pj_n;
            lj_j = lj_n;
        }
        const int gn = claimed(tk);
        if constexpr (P::mixed) {
            if (gn < hi) cur = fetch(gn);
        }
        wave_lds_sync();
        {
            // j-forces of the chunk, 8 entries (64 lanes) per atomic instruction
            const int n = e1 - e0;
            for (int b = 0; b < n; b += 8) {
                const int el = b + ia;
                if (el < n) {
                    const int sj = (int)(jw[el].x & 0xffffffu) * 8 + ja;
                    facc_add(&FX[sj], jf[(el * 3 + 0) * 8 + ja]);
                    facc_add(&FY[sj], jf[(el * 3 + 1) * 8 + ja]);
                    facc_add(&FZ[sj], jf[(el * 3 + 2) * 8 + ja]);
                }
            }
        }
        // i-forces: sums over the 8 j lanes, transposed through LDS so that one
        // full-wave atomic per component covers the chunk's 64 i atoms
        wave_lds_sync();   // the j flush has read jf
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const real fx = sum_group8(fxi[k]), fy = sum_group8(fyi[k]), fz = sum_group8(fzi[k]);
            if (ja == 0) {
                jf[0 * 64 + k * 8 + ia] = fx;
                jf[1 * 64 + k * 8 + ia] = fy;
                jf[2 * 64 + k * 8 + ia] = fz;
            }
        }
        wave_lds_sync();
        if ((lane >> 3) < ncl) {
            const int slot = fc * 8 + lane;
            facc_add(&FX[slot], jf[0 * 64 + lane]);
            facc_add(&FY[slot], jf[1 * 64 + lane]);
            facc_add(&FZ[slot], jf[2 * 64 + lane]);
        }
        if constexpr (ENERGY) {
            // each lane's share of the chunk is rounded; the integers add up over the
            // wavefront's chunks of one system before they leave it
            if (s != e_sys) flush_energy();
            e_sys = s;
            ec_sum += energy_fixed(ec_acc);
            el_sum += energy_fixed(el_acc);
        }
        wave_lds_sync();   // LDS of this wave is reused by its next chunk
        g = gn;
    }
    if constexpr (ENERGY) flush_energy();
}

#define NX_PAIR_PARAMS(P)                                                                                      \
    const SysDev *__restrict__ sd, const int *__restrict__ prefix, int nsys, const int4 *__restrict__ chunks, const uint2 *__restrict__ list, const unsigned long long *__restrict__ emask, \
        const typename P::real4 *__restrict__ pos, const typename P::real2 *__restrict__ lj, typename P::facc *FX,    \
        typename P::facc *FY, typename P::facc *FZ, long long *energy, int *__restrict__ pool
#define NX_PAIR_ARGS sd, prefix, nsys, chunks, list, emask, pos, lj, FX, FY, FZ, energy, pool

// The pair kernels.  The mixed one without energies must stay within
// PrecMixed::pair_max_vgpr VGPRs (the compiler offers no cap short of a higher
// occupancy target, which spills; a test of the build checks the count), so
// that the PME kernels still find room beside its persistent grid.
template <bool ENERGY>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PrecMixed::pair_waves_per_simd))) void
pair_kernel_mixed(NX_PAIR_PARAMS(PrecMixed)) {
    pair_body<PrecMixed, ENERGY, true>(NX_PAIR_ARGS);
}
// The FP64 kernel with the series alone, for batches whose every system is in
// its range, needs 156 VGPRs; with the library functions beside it (chosen per
// system) 226.
template <bool ENERGY, bool ALL_SERIES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PrecFP64::pair_waves_per_simd))) void
pair_kernel_fp64(NX_PAIR_PARAMS(PrecFP64)) {
    pair_body<PrecFP64, ENERGY, ALL_SERIES>(NX_PAIR_ARGS);
}
#undef NX_PAIR_ARGS
#undef NX_PAIR_PARAMS

template <class P, bool ENERGY>
static auto pair_kernel_of(bool all_series) {
    if constexpr (P::mixed) return pair_kernel_mixed<ENERGY>;
    else return all_series ? pair_kernel_fp64<ENERGY, true> : pair_kernel_fp64<ENERGY, false>;
}

// Explicit pair set (atom ids, first > second) with the FP64 test of the pair kernel.
template <class P>
__global__ __launch_bounds__(64) void export_pairs_kernel(const SysDev* sd, const SysCount* sc, const int* super_sys,
                                                          const int4* super_item, const uint2* list,
                                                          const unsigned long long* emask, const int* atom_of_slot,
                                                          const double* X, const double* Y, const double* Z,
                                                          int2* out, long long cap, unsigned long long* count,
                                                          int n_items) {
    const int item = blockIdx.x;
    if (item >= n_items) return;
    const int s = super_sys[item];
    if (item - sd[s].super_off >= sc[s].n_super) return;
    const int4 it = super_item[item];
    const int fc = it.x, ncl = it.y, lstart = it.z, llen = it.w;
    const int lane = threadIdx.x, ia = lane >> 3, ja = lane & 7;
    const double Lx = sd[s].L[0], Ly = sd[s].L[1], Lz = sd[s].L[2], rc2 = sd[s].rc2;
    for (int e = 0; e < llen; ++e) {
        const uint2 ent = list[lstart + e];
        const int cj = (int)(ent.x & 0xffffffu);
        const unsigned im = ent.x >> 24;
        const int aj = atom_of_slot[cj * 8 + ja];
        for (int k = 0; k < ncl; ++k) {
            if (!(im & (1u << k))) continue;
            const int ai = atom_of_slot[(fc + k) * 8 + ia];
            bool excl = (cj == fc + k) && (ja <= ia);
            const unsigned eid = ent.y & kNoMask;
            if (eid != kNoMask) excl |= ((emask[(size_t)eid * 8 + k] >> lane) & 1ull) != 0ull;
            if (excl || ai < 0 || aj < 0) continue;
            const double dx = min_image1(X[ai] - X[aj], Lx);
            const double dy = min_image1(Y[ai] - Y[aj], Ly);
            const double dz = min_image1(Z[ai] - Z[aj], Lz);
            if (dot_rn(dx, dy, dz) < rc2) {
                unsigned long long w = atomicAdd(count, 1ull);
                if ((long long)w < cap) out[w] = make_int2(max(ai, aj), min(ai, aj));
            }
        }
    }
}

// Blocks of the pair kernel one CU holds at once (its occupancy limit), for the
// kernel that a batch takes.
template <class P, bool ALL_SERIES>
static int pair_blocks_per_cu() {
    static const int v = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, pair_kernel_of<P, false>(ALL_SERIES), 256, 0) != hipSuccess || n <= 0)
            n = 2;
        return n;
    }();
    return v;
}
template <class P>
int pair_blocks_occupancy(bool all_series) {
    return all_series ? pair_blocks_per_cu<P, true>() : pair_blocks_per_cu<P, false>();
}

// Persistent grid of the pair kernel, all blocks resident at once, at most
// three per CU: the rest of a CU's wave slots go to the bonded and PME kernels
// running beside it.  Measured on the 100k-atom step (mixed, five
// resident blocks possible): 3 per CU 261 us, 4 per CU 303 us, 2 per CU 268 us.
// FP64 takes two, which leave PME room, and three (all it can have) up to 50,000
// atoms, where two waves per SIMD's worth of chunks end too unevenly: us a step with
// 2 and 3 per CU on water of 3,000 to 12,000 atoms the same, 18,000 125 117, 24,000
// 143 133, 30,000 161 149, 36,000 179 168, 48,000 215 198, 54,000 245 250, 81,000 331
// 334; solvated chains of 100,000 386 387.  The FP64 kernel with library functions in
// it has room for two only: a third would start its first chunks when another ends
// (24,000 atoms 222 us a step, with two 199).
// Fixed per batch layout: the claim counters are set for it.
template <class P>
int pair_grid_blocks(int n_cu, int n_chunk_cap, int n_atoms, bool all_series, int per_cu_request) {
    // a requested count (the autotuner's) is capped by what a CU can hold at once
    const int occ = pair_blocks_occupancy<P>(all_series);
    const int per_cu = per_cu_request > 0 ? std::min(per_cu_request, occ) : std::min(occ, P::mixed || n_atoms <= 50000 ? 3 : 2);
    return std::max(1, std::min((n_chunk_cap + kPairWaves - 1) / kPairWaves, per_cu * std::max(1, n_cu)));
}

// Ends the step's list work before the pair kernel: clears the rebuild flags
// (every list kernel that reads them ran before) and counts the builds.  As a
// separate launch it also gives the kernels forked to the side stream (bonded
// terms, PME) a head start on the CUs before the pair kernel's persistent grid
// takes its slots; without it the step measured about 10% slower.
__global__ void pair_begin_kernel(SysCount* sc, int nsys, const int* prefix, int* pool, int pair_blocks) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    pool_begin(s, prefix[nsys], pool, pair_blocks);
    if (s >= nsys) return;
    if (sc[s].rebuild) {
        sc[s].rebuild = 0;
        sc[s].rebuilds += 1;
    }
}

template <class P>
void launch_pair_begin(Batch<P>& B) {
    pair_begin_kernel<<<(B.nsys + 63) / 64, 64, 0, B.stream>>>(B.d_cnt, B.nsys, B.chunk_prefix, B.pair_pool,
                                                               B.pair_blocks);
}

template <class P>
void launch_pair_kernel(Batch<P>& B, bool energy) {
    if (B.n_chunk_cap == 0) return;
    const unsigned blocks = (unsigned)B.pair_blocks;
    if (energy)
        pair_kernel_of<P, true>(B.all_series)<<<blocks, 256, 0, B.stream>>>(B.d_sys, B.chunk_prefix, B.nsys, B.chunks, B.list,
                                                           B.emask, B.pos, B.lj, B.FSx, B.FSy, B.FSz, B.energy,
                                                           B.pair_pool);
    else
        pair_kernel_of<P, false>(B.all_series)<<<blocks, 256, 0, B.stream>>>(B.d_sys, B.chunk_prefix, B.nsys, B.chunks, B.list,
                                                            B.emask, B.pos, B.lj, B.FSx, B.FSy, B.FSz, B.energy,
                                                            B.pair_pool);
}

template <class P>
void launch_pair(Batch<P>& B, bool energy) {
    launch_pair_begin<P>(B);
    launch_pair_kernel<P>(B, energy);
}

template <class P>
void launch_export_pairs(Batch<P>& B, int2* out, long long cap, long long* d_count) {
    export_pairs_kernel<P><<<B.n_super_cap, 64, 0, B.stream>>>(B.d_sys, B.d_cnt, B.super_sys, B.super_item, B.list,
                                                               B.emask, B.atom_of_slot, B.X, B.Y, B.Z, out, cap,
                                                               reinterpret_cast<unsigned long long*>(d_count),
                                                               B.n_super_cap);
}

template int pair_grid_blocks<PrecFP64>(int, int, int, bool, int);
template int pair_grid_blocks<PrecMixed>(int, int, int, bool, int);
template int pair_blocks_occupancy<PrecFP64>(bool);
template int pair_blocks_occupancy<PrecMixed>(bool);
template void launch_pair<PrecFP64>(Batch<PrecFP64>&, bool);
template void launch_pair<PrecMixed>(Batch<PrecMixed>&, bool);
template void launch_pair_begin<PrecFP64>(Batch<PrecFP64>&);
template void launch_pair_begin<PrecMixed>(Batch<PrecMixed>&);
template void launch_pair_kernel<PrecFP64>(Batch<PrecFP64>&, bool);
template void launch_pair_kernel<PrecMixed>(Batch<PrecMixed>&, bool);
template void launch_export_pairs<PrecFP64>(Batch<PrecFP64>&, int2*, long long, long long*);
template void launch_export_pairs<PrecMixed>(Batch<PrecMixed>&, int2*, long long, long long*);

}  // namespace nx
