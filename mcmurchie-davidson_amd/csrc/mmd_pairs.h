// Shell-pair tables and Fock work units, built on the device (mmd_pairs.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "mmd_device.h"
#include "mmd_kernels.h"
#include "mmd_types.h"

namespace mmd {

constexpr int UNIT_BUCKETS = 128;    // cost classes of the work units (quarter octaves)
constexpr int QMAX_BLOCK = 32;       // kets per running maximum of the pair factors

// What the build reads: the shells, the shell pairs of every molecule grouped
// by pair class (list[off[pc] .. off[pc+1]), by molecule inside a class), the
// class-local range {first, end} of each molecule's pairs (ranges[pc * nmol +
// m]), and the Schwarz diagonal (N x N, or null: factors 1).
struct PairInput {
    const OneeShell* shells;
    const double* exps;
    const double* wts;
    const int2* list;
    const int2* ranges;
    const int4* mol_blocks;          // {first function, ...} per molecule, or null for one molecule
    const double* diag;
    int off[NPAIRCLASS + 1];
    int nmol, N;
};

// 64-bit words of keep bits per pair (PairWork), for shells of at most maxnp
// primitives.
inline int pair_keep_words(int maxnp) { return (int)(((int64_t)maxnp * maxnp + 63) / 64); }

// Work buffers, npairs entries each but for the last three.
struct PairWork {
    int* count;                      // surviving primitive pairs, list order
    int* entry;                      // list entry of each sorted pair
    double* q;                       // pair factors, list order
    int* scan;                       // npairs + npairs / 1024 + 2
    unsigned long long* qmax;        // largest primitive-pair bound
    unsigned long long* keep;        // per primitive pair whether it survives: word w of list entry e at w * npairs + e
};

// Results on the host: largest and total primitive-pair count per class.
struct PairStats {
    int maxpp[NPAIRCLASS];
    int total[NPAIRCLASS];
};

// Primitive pairs counted and screened, the pairs sorted inside each class by
// (molecule, primitive pairs descending, factor descending, list order) into
// `pairs` with their ranges in the primitive-pair table, class by class.
hipError_t launch_pair_sort(const PairInput& I, const PairWork& W, ShellPair* pairs, PairStats* stats, hipStream_t st);
// The primitive-pair table of the sorted pairs (the W of the sort), and each
// entry's first exponent (ppa), and the row kernels' ket tables of both.
struct KetTables {
    KetScreen* scr;
    KetRef* ref;
    double* pp;
    int64_t stride;
};
hipError_t launch_pair_fill(const PairInput& I, const PairWork& W, const ShellPair* pairs, PrimPair* pp, double* ppa,
                            const KetTables& K, hipStream_t st);

// Work units of the row kernels.  One per (bra pair, slice of at most PSLICE
// of its primitive pairs, segment of seg[qc] kets of its molecule), in
// decreasing order of cost (bra x ket primitive pairs, by quarter octaves).
struct UnitInput {
    const ShellPair* pairs;
    const int2* ranges;
    int off[NPAIRCLASS + 1];
    int seg[NQCLASS];
    int nmol;
};
// hist: NQCLASS x UNIT_BUCKETS counters; counts[qc]: units of class qc;
// qrun: npairs running maxima.  The scatter takes the cursors that the count
// left in hist, and writes class qc at units + (sum of the counts before it).
hipError_t launch_unit_count(const UnitInput& I, int* hist, int* counts, double* qrun, hipStream_t st);
hipError_t launch_unit_scatter(const UnitInput& I, int* hist, const double* qrun, int4* units, UnitBound* bounds,
                               hipStream_t st);

// Of each class's units [off[qc], off[qc + 1]) those that hold a quartet which
// can pass the screen: pair factors q_P q_Q <= the unit's bound, and density
// weights at most 4 max |dP| of the molecule (0 once it has converged).  Their
// class-local numbers, roughly in order, to live + off[qc]; nlive[qc] of them
// (cleared before).
struct UnitLive {
    int64_t off[NQCLASS + 1];
    const UnitBound* bound;
    const double* mol_dmax;
    double tol;
    int* live;
    int* nlive;
};
hipError_t launch_unit_live(const UnitLive& I, hipStream_t st);

}  // namespace mmd
