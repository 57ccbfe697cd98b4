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

// Results per class: the largest and total primitive-pair count; and units.
struct PairStats {
    int maxpp[NPAIRCLASS];
    int total[NPAIRCLASS];
};
constexpr int PAIR_STATS = (int)(sizeof(PairStats) / sizeof(int));
constexpr int PAIR_REPORT = PAIR_STATS + NQCLASS;   // ints: PairStats, units of each quartet class
constexpr int UNIT_HIST = NQCLASS * UNIT_BUCKETS;

// Keep bits of a pair's primitive pairs come in pieces of 16; the pieces of a
// pair of shells of at most maxnp primitives.
constexpr int PAIR_KEEP_BITS = 16;
inline size_t pair_keep_pieces(int maxnp) { return ((size_t)maxnp * maxnp + PAIR_KEEP_BITS - 1) / PAIR_KEEP_BITS; }

// Work buffers, npairs entries each but for the last four.
struct PairWork {
    int* count;                      // surviving primitive pairs, list order
    int* entry;                      // list entry of each sorted pair
    double* q;                       // pair factors, list order; then the units' running maxima
    uint16_t* keep;                  // piece t of list entry e at t * npairs + e (pair_keep_pieces)
    int* scan;                       // npairs + npairs / 1024 + 2
    // nclear ints one after the other, cleared together:
    int* report;                     // PAIR_REPORT
    int* hist;                       // UNIT_HIST counters of the units' cost buckets, then their cursors
    unsigned long long* qmax;        // largest primitive-pair bound
    int nclear;
};

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

// Primitive pairs counted and screened, the pairs sorted inside each class by
// (molecule, primitive pairs descending, factor descending, list order) into
// `pairs` with their ranges in the primitive-pair table, class by class; and
// the units counted, where asked for.
hipError_t launch_pair_sort(const PairInput& I, const PairWork& W, const UnitInput& U, bool units, ShellPair* pairs,
                            hipStream_t st);

// The tables of the sorted pairs (the W of the sort): their primitive pairs,
// each entry's first exponent (ppa), and the row kernels' ket tables of both;
// the units (T.units null: none), class qc after the classes before it.  The
// report goes to pinned host memory.
struct KetTables {
    KetScreen* scr;
    KetRef* ref;
    double* pp;
    int64_t stride;
};
struct UnitTables {
    int4* units;
    UnitBound* bounds;
};
hipError_t launch_pair_tables(const PairInput& I, const PairWork& W, const ShellPair* pairs, PrimPair* pp, double* ppa,
                              const KetTables& K, const UnitInput& U, const UnitTables& T, int* host_report,
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
