// bonded.hip -- the kernels of the bonded terms and of the per-atom force gather
// (nx_terms.h has the terms).
//
// bonded_kernel: one thread per term (bonds, then angles, then torsions, in
// one launch).  Each term writes the force on each of its atoms into its own
// slots of the per-term force buffer tF (plain stores).
// atom_force_kernel: one thread per atom sums the term forces acting on it
// (per-atom CSR of slots, fixed order) and its exclusion corrections, and
// stores the atom-order force.  No force is added atomically.
#include "nx_terms.h"

namespace nx {

template <class P, bool ENERGY>
__global__ void bonded_kernel(TermArgs<P> g, long long* energy) {
    side_priority();
    bonded_term<P, ENERGY>(g, blockIdx.x * blockDim.x + threadIdx.x, energy);
}

template <class P, bool ENERGY>
__global__ void atom_force_kernel(TermArgs<P> g, long long* energy) {
    side_priority();
    atom_force<P, ENERGY>(g, blockIdx.x * blockDim.x + threadIdx.x, energy);
}

template <class P>
void launch_bonded(Batch<P>& B, int mask, bool energy) {
    const int n = bonded_count(B, mask);
    if (n == 0) return;
    const int T = 256;
    (energy ? bonded_kernel<P, true> : bonded_kernel<P, false>)<<<(unsigned)((n + T - 1) / T), T, 0, B.stream>>>(
        term_args(B, mask), B.energy);
}

template <class P>
void launch_atom_forces(Batch<P>& B, int mask, bool energy) {
    const int T = 256;
    (energy ? atom_force_kernel<P, true> : atom_force_kernel<P, false>)<<<(unsigned)((B.n_atoms + T - 1) / T), T, 0,
                                                                         B.stream>>>(
        term_args(B, atom_force_mask(B, mask)), B.energy);
}

template void launch_bonded<PrecFP64>(Batch<PrecFP64>&, int, bool);
template void launch_bonded<PrecMixed>(Batch<PrecMixed>&, int, bool);
template void launch_atom_forces<PrecFP64>(Batch<PrecFP64>&, int, bool);
template void launch_atom_forces<PrecMixed>(Batch<PrecMixed>&, int, bool);

}  // namespace nx
