// Arguments of the shell-class kernels of the nuclear gradient.
#pragma once
#include <hip/hip_runtime.h>
#include "mmd_types.h"

namespace mmd {

// bra primitive pairs of a work unit of the lane kernels, by pair class (ss,
// ps, pp, ds, dp, dd): the staged tables of a d pair are up to 4 KB each
__host__ __device__ constexpr int grad_pslice(int pc) { return pc <= 2 ? 16 : (pc <= 4 ? 8 : 4); }
constexpr int GRAD_REPLICAS = 64;   // copies of the gradient the workgroups add to (summed at the end):
                                    // a few dozen addresses would serialise the atomics of a large molecule

struct GradArgs {
    const ShellPair* pairs;
    const PrimPair* pp;
    const double* ppa;      // exponent of the pair's first function, per primitive pair
    const double* boys;
    const double* gcomp;
    const double* P;        // half density, N x N
    const int* bf_atom;
    double* grad;           // GRAD_REPLICAS x natom x 3
    int N, natom;
    int lds_atoms;          // the workgroup sums its atoms in LDS
};

// Work of one quartet class.
struct GradClass {
    const int4* slices;     // bra: {pair, first, end primitive, end of the pair's own primitives in flat}
    int nslice;
    const int2* flat;       // the ket class's primitive pairs, pair by pair: {pair, primitive}
    int nflat, nkc;         // their number, and in blocks of 256
    int tri;                // same pair class: ket pair <= bra pair (flat entries below the slice's w)
};

// Two-electron gradient of one quartet class (mmd_grad_class.hip): the
// workgroup-per-primitive-quartet classes take slices of one primitive pair.
hipError_t launch_grad_class(int qc, const GradArgs& A, const GradClass& C, hipStream_t st);
struct OneeArgs;
// One-electron gradient of the n shell pairs of pair class pc at list.
hipError_t launch_grad_onee(int pc, const OneeArgs& A, const int2* list, int n, const int* bf_atom, const double* P,
                            const double* W, double* grad, hipStream_t st);
// grad (natom x 3) = the sum of the nrep copies at rep, plus the nuclear
// repulsion gradient of the nuclei nuc (natom x 4: Z, x, y, z) when given.
hipError_t launch_grad_sum(int natom, int nrep, const double* rep, const double* nuc, double* grad, hipStream_t st);

}  // namespace mmd
