// nx_engine.h -- host-side batch of systems resident on one GPU.
//
// A Batch holds every device buffer for one or more independent systems
// packed back to back (a single-system context is a batch of one).  Kernels
// take the packed arrays plus per-item system tables, so one launch advances
// every system of the batch.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/nexusmd.h"

#include "nx_device.h"

namespace nx {

struct HostSystem;   // engine.hip

// Threads of a plane pass: what the pair kernel's blocks leave of a SIMD's 512 VGPRs
// holds three waves of 56 VGPRs in the mixed path (R2 float2; three blocks a CU of
// 112), two of 96 in FP64 (two blocks of 160; with three waves the pass waited for the
// pair kernel: 24,000 atoms at 64^3 130.3 us a step, with two 125.1).
template <typename R2>
constexpr int kPlaneThreads = sizeof(R2) == 8 ? 768 : 512;
// Most LDS of a plane pass with the spread: what those blocks leave of a CU's 160 KB.
// Beside the three blocks that FP64 takes up to 50,000 atoms (pair_grid_blocks) a
// plane pass finds neither the registers nor the LDS and waits for one of them to
// end.  So would the line passes, and planes are still the faster ones: us a step,
// planes and lines, 12,000 atoms 98.2, 100.7; 24,000 132.8, 136.9.
template <typename R2>
constexpr size_t kPlaneSpreadLds = (sizeof(R2) == 8 ? 100 : 82) * 1024;
constexpr int kXPassThreads = 256;
// Bytes of a row that the y and x passes take at a time: a cache line.
constexpr int kPassRowBytes = 128;
// Points by which each row of the potential runs on past its end (its first
// ones again): the gather reads five consecutive points from any of the row's.
constexpr int kPhiPad = 4;
// LDS of one workgroup on gfx950, less the kernels' static LDS.
constexpr size_t kMaxBlockLds = 160 * 1024 - 1024;

// LDS bytes of the spread in a block of `threads`: its table of slot segments
// and 128 queued slots per wavefront.
constexpr int kSpreadSegs = 64;
constexpr size_t spread_lds_bytes(int threads) { return (size_t)(3 * kSpreadSegs + 2 + threads / 64 * 128) * sizeof(int); }
// Complex points that two line buffers of cap points, or ny rows of the spread's
// sums (Kz + 4 long, 8 bytes each) in their place, take.
template <typename R2>
__host__ __device__ constexpr int spread_points(int cap, int ny, int Kz) {
    const int sums = (int)(((size_t)ny * (Kz + 4) * 8 + sizeof(R2) - 1) / sizeof(R2));
    return 2 * cap > sums ? 2 * cap : sums;
}
// Spread and z pass of the line FFT: threads per block, and the complex points
// one of them moves (two rows of the grid make one complex line).
constexpr int kSpreadZThreads = 512;
constexpr int kSpreadZPerThread = 6;
constexpr int kSpreadZPoints = kSpreadZThreads * kSpreadZPerThread;

// The radices of a transform of N = 2^a 3^b 5^c points, four bits each, the first
// stage's lowest: as few stages as radices up to 8 allow.
__host__ __device__ inline unsigned fft_plan(int N) {
    int twos = 0, m = N;
    for (; m % 2 == 0; m /= 2) ++twos;
    unsigned plan = 0;
    int at = 0;
    auto add = [&](unsigned r) { plan |= r << at; at += 4; };
    if (twos == 1) add(2);
    else if (twos % 3 == 1) { add(4); add(4); twos -= 4; }
    else if (twos % 3 == 2) { add(4); twos -= 2; }
    for (; twos >= 3; twos -= 3) add(8);
    for (; m % 3 == 0; m /= 3) add(3);
    for (; m % 5 == 0; m /= 5) add(5);
    return plan;
}

// Complex points of a line buffer of a plane pass: row pairs by z or, the other
// way, wave numbers by y, the inner extent made odd.
__host__ __device__ constexpr int plane_cap(int Ky, int Kz) {
    const int z = Kz * (((Ky + 1) / 2) | 1), y = Ky * ((Kz / 2 + 1) | 1);
    return z > y ? z : y;
}

// LDS bytes of a plane pass (two buffers, the y and z twiddles).
template <typename R2>
inline size_t plane_lds_bytes(int Ky, int Kz) {
    return (size_t)(Ky + Kz + 2 * plane_cap(Ky, Kz)) * sizeof(R2);
}

// The same with the spread in it.
template <typename R2>
inline size_t plane_spread_lds_bytes(int Ky, int Kz) {
    return (size_t)(Ky + Kz + spread_points<R2>(plane_cap(Ky, Kz), Ky, Kz)) * sizeof(R2) + spread_lds_bytes(kPlaneThreads<R2>);
}

// Lines of a workgroup of the x pass: a cache line's width (`row` of them), half of
// one for more workgroups only on request (the passes after the spread, us alone,
// whole and half: 64^3 15.1, 15.4; 50 x 50 x 75 17.9, 18.1; unaligned widths between
// them are worse: 96^3 21.6 with 16 lines, 25.3 with 10).
constexpr int kXPassHalfLines = 65536;      // as the request: half lines on any grid, the one other shape to try
constexpr int x_pass_lines(long long x_lines, int row, int workgroups) {
    return workgroups < kXPassHalfLines && x_lines > (long long)row * workgroups ? row : row / 2;
}
static_assert(x_pass_lines(1, 8, 0) == 8 && x_pass_lines(1024 * 513, 8, 0) == 8 &&
                  x_pass_lines(1, 8, kXPassHalfLines) == 4 && x_pass_lines(1024 * 513, 8, kXPassHalfLines) == 4,
              "two shapes on the smallest grid and on the largest");

// LDS bytes of `lines` lines of K points (two buffers, the twiddles).
template <typename R2>
inline size_t line_lds_bytes(int K, int lines) {
    return (size_t)(K + 2 * lines * K) * sizeof(R2);
}

template <class P>
struct Batch {
    using real = typename P::real;
    using real2 = typename P::real2;
    using real4 = typename P::real4;
    using facc = typename P::facc;

    int nsys = 0;
    std::vector<SysDev> sys;             // host copy of the descriptors
    SysDev* d_sys = nullptr;
    SysCount* d_cnt = nullptr;
    hipStream_t stream = nullptr;

    int n_atoms = 0, n_slots_cap = 0, n_cols = 0, n_super_cap = 0;
    long long n_list_cap = 0, n_emask_cap = 0;

    // atom order (FP64 master state)
    double *X = nullptr, *Y = nullptr, *Z = nullptr;
    double *VX = nullptr, *VY = nullptr, *VZ = nullptr;
    double *invm = nullptr, *mass = nullptr, *q = nullptr, *sig = nullptr, *eps = nullptr;
    double *XB = nullptr, *YB = nullptr, *ZB = nullptr;
    int *atom_sys = nullptr, *slot_of_atom = nullptr, *atom_col = nullptr;
    facc *FAx = nullptr, *FAy = nullptr, *FAz = nullptr;

    // slot order
    int *slot_sys = nullptr, *atom_of_slot = nullptr, *slot_tmp = nullptr;
    real4* pos = nullptr;
    real2* lj = nullptr;
    facc *FSx = nullptr, *FSy = nullptr, *FSz = nullptr;

    // columns / clusters / pair list
    int *col_sys = nullptr, *col_count = nullptr, *col_fill = nullptr, *col_slot = nullptr, *col_super = nullptr;
    int* col_tmp = nullptr;         // counts of the columns' quarters during a build (zero between builds)
    float4 *cl_ctr = nullptr, *cl_half = nullptr;     // cluster boxes at the last build
    float4 *sup_ctr = nullptr, *sup_half = nullptr;   // super-cluster boxes
    float4* slot_wpos = nullptr;    // build-time wrapped position of each slot, w = 1 (atom) or 0 (padding)
    int* super_sys = nullptr;
    int4* super_item = nullptr;
    int4* chunks = nullptr;         // (first cluster, n clusters, first entry, end entry)
    int* chunk_prefix = nullptr;    // [nsys + 1] running total of chunks over systems
    int* pair_pool = nullptr;       // [kPoolInts] per XCD: chunks handed out so far by the running pair kernel
    // one-system batches: nl_waves' report to the host (host memory, mapped),
    // the report count (device) and the update's largest squared displacement
    // (device, kStepMaxSlots float bit patterns)
    StepInfo* step_info = nullptr;
    unsigned* step_seq = nullptr;
    unsigned* step_max = nullptr;
    int pair_blocks = 0;
    bool all_series = true;         // every system's alpha^2 rc^2 is within kErfSeriesMax
    int n_cu = 0;                   // compute units of the device
    int n_chunk_cap = 0;
    uint2* list = nullptr;
    unsigned long long* emask = nullptr;
    int *excl_off = nullptr, *excl_idx = nullptr;
    int2* excl_pairs = nullptr;
    int n_excl_pairs = 0;

    // bonded terms (global atom indices)
    int2* bond_idx = nullptr;
    double2* bond_par = nullptr;
    int n_bonds = 0;
    int4* angle_idx = nullptr;
    double2* angle_par = nullptr;
    int n_angles = 0;
    real* tF = nullptr;             // per-term forces [3][n_tslots]: bonds 2, angles 3, torsions 4 slots each
    int n_tslots = 0;
    int* at_off = nullptr;          // per atom: CSR of the term-force slots that act on it
    int* at_idx = nullptr;
    int4* tors_idx = nullptr;
    double4* tors_par = nullptr;   // k, phase, periodicity, unused
    int n_tors = 0;

    // PME
    using gacc = typename P::gacc;
    real2* cgrid = nullptr;         // half spectrum [sum Kx*Ky*(Kz/2+1)]
    real* phi = nullptr;            // potential grid [sum Kx*Ky*(Kz + kPhiPad)]
    real* eta = nullptr;            // influence function on the half spectrum
    real2* twiddle = nullptr;       // per system, per axis exp(-2 pi i t / K)
    long long rgrid_total = 0, cgrid_total = 0, tw_total = 0;
    int4* fftz_items = nullptr;     // spread: (sys, x, y0, ny), or whole planes (sys, x)
    int4* fftp_items = nullptr;     // inverse plane pass: (sys, x)
    int4* fftl_items = nullptr;     // inverse z pass: (sys, x, first pair of rows, n pairs)
    int4* ffty_items = nullptr;     // (sys, x, kz0, 0)
    int4* fftx_items = nullptr;     // (sys, first (y, kz) line, n lines, 0)
    int n_fftz = 0, n_fftp = 0, n_fftl = 0, n_ffty = 0, n_fftx = 0;
    int fft_tile = 1;               // columns of a y pass's tile
    int fft_plane_threads = 0, fft_x_threads = 0;
    int fft_plane = 0;              // 1: plane passes (fftp_items); 0: y and z passes over lines
    size_t fft_spread_lds = 0, fft_plane_lds = 0, fft_x_lds = 0, fft_y_lds = 0, fft_z_lds = 0;
    int pme_any = 0;

    // energies [nsys][kEnergySlots][E_NTERMS] in 2^30 fixed point
    long long* energy = nullptr;

    // flags
    int timing = 0;                 // NX_TIMING_* mode
};

// part 0: the whole list work; 1: all but its last kernel; 2: the last kernel
// alone, which then also does the pair kernel's set-up (launch_pair_begin); 3: the
// same in a step without the other list kernels (a due list is marked stale)
template <class P> void launch_nlist(Batch<P>& B, bool clear_flags, int part = 0);
// persistent pair-kernel grid: per_cu_request blocks per CU (0: the built-in count), capped by occupancy
template <class P> int pair_grid_blocks(int n_cu, int n_chunk_cap, int n_atoms, bool all_series, int per_cu_request);
template <class P> int pair_blocks_occupancy(bool all_series);     // pair-kernel blocks one CU holds at once
template <class P> void launch_pack(Batch<P>& B);
template <class P> void launch_pair(Batch<P>& B, bool energy);
// the two launches of launch_pair: the per-system set-up kernel, then the pair kernel
template <class P> void launch_pair_begin(Batch<P>& B);
template <class P> void launch_pair_kernel(Batch<P>& B, bool energy);
template <class P> void launch_bonded(Batch<P>& B, int mask, bool energy);
template <class P> void launch_atom_forces(Batch<P>& B, int mask, bool energy);
template <class P> void launch_pme_spread(Batch<P>& B);
bool fft_plane_enabled();
template <class P> hipError_t prepare_fft(Batch<P>& B);
template <class P> void launch_fft_forward(Batch<P>& B);
// without energies also the bonded terms of the kinds in term_mask
template <class P> void launch_fft_convolve(Batch<P>& B, bool energy, int term_mask = 0);
template <class P> void launch_fft_inverse(Batch<P>& B);
// also the atom forces of a step with force mask atom_mask (launch_atom_forces), unless it is negative
template <class P> void launch_pme_gather(Batch<P>& B, int atom_mask = -1);
// the systems' energies [nsys][E_NTERMS] into total and their counters into counts (may be NULL)
template <class P> void launch_energy_sum(Batch<P>& B, long long* total, SysCount* counts);
template <class P> void launch_kinetic(Batch<P>& B, double dt);
template <class P> void launch_integrate(Batch<P>& B, double dt);
// positions, velocities and total forces (each may be NULL) of n atoms from a0 on, [n][3] each
template <class P> void launch_report_snapshot(Batch<P>& B, double* pos, double* vel, double* force, int a0, int n);
// positions and velocities (NULL: zeros) [n][3] into the state (pos NULL: it stays), every list due
template <class P> void launch_set_state(Batch<P>& B, const double* pos, const double* vel);
// Writes up to cap pairs to out and their total count to *d_count, which must be zero before the launch.
template <class P> void launch_export_pairs(Batch<P>& B, int2* out, long long cap, long long* d_count);
// standalone FFT (verification)
template <class P> void fft3d_roundtrip(int nx, int ny, int nz, const double* in, double* out, bool forward,
                                        hipStream_t st);
// the forward transform of fft3d_roundtrip in the library's static device
// scratch array (no allocation); err receives the reason of a failure
template <class P> nx_status fft3d_r2c_noalloc(int device, int nx, int ny, int nz, const double* in, double* out,
                                               std::string& err);

}  // namespace nx
