// Data layout shared by the host runtime and the gfx950 kernels.
#pragma once
#include <stdint.h>

namespace mmd {

// A contracted shell pair in canonical orientation (la >= lb).  Shell pairs
// are grouped by angular-momentum pair class and, inside a class, sorted by
// primitive-pair count and Schwarz factor (descending) so that the quartets a
// wavefront enumerates have similar cost and similar screening fate.
struct ShellPair {
    int32_t sa, sb;      // shell indices (sa carries la >= lb)
    int32_t bfa, bfb;    // first basis-function index of each shell
    int32_t pp0, npp;    // range in the primitive-pair table
    int32_t same;        // sa == sb
    int32_t mol;         // molecule of the pair (a basis can hold several, block-diagonally)
    int32_t c0;          // first basis function of that molecule
    int32_t class_pp0;   // its first primitive pair's position among those of its pair class
    double q;            // max over the pair's functions of sqrt((ab|ab))
};

// A primitive pair: exponent sum, Gaussian-product prefactor including both
// contraction coefficients, product centre and its offsets from A and B,
// 1/(2p) and 1/p.
struct PrimPair {
    double p, K;
    double Px, Py, Pz;
    double PAx, PAy, PAz;
    double PBx, PBy, PBz;
    double inv2p, invp;
};

// What the row kernels read of a ket pair: its screen, and its functions and
// primitive pairs.  16 bytes each in the order of the pair table, so that
// consecutive lanes read consecutive records.
struct KetScreen {
    double q;
    int32_t sa, sb;
};
struct KetRef {
    int32_t bfa, bfb, pp0, npp;
};
// Fields of the primitive pairs field by field (KET_FIELDS arrays of the
// table's length), for lanes that take consecutive primitive pairs.
enum KetField { KF_P, KF_KQ, KF_X, KF_Y, KF_Z, KF_INV2P, KF_PAX, KF_PAY, KF_PAZ, KF_PBX, KF_PBY, KF_PBZ, KET_FIELDS };

// Arguments of the quartet-class kernels (passed by value).
struct ClassArgs {
    const int2* quart;          // surviving (bra pair, ket pair) for this class
    const int* count;           // number of survivors (device)
    const ShellPair* pairs;     // all shell pairs
    const PrimPair* pp;         // primitive pairs
    const double* boys;         // Boys table [BOYS_ROWS][BOYS_NT]
    const float* boysf;         // the same table in float (FP32-tier kernels)
    const double* gcomp;        // per-basis-function component scale
    const double* D;            // density (difference) N x N
    const double* absD;         // |dP| N x N (screening)
    const double* sqS;          // sqrt((ij|ij)) N x N (screening)
    double tol;                 // screening threshold
    int N;
    double* G;                  // Fock accumulation N x N
};

// Ket primitive pairs per lane item of the sliced classes, unless set per
// class (mmd_set_ket_slices): short slices keep the lanes of a wavefront
// even when a batch mixes contraction lengths (a 64-molecule 6-31G batch
// pass measured 369, 341 and 334 ms for slices of 8, 4 and 2; (H2O)8
// cc-pVDZ builds were the same for all three).
constexpr int KSLICE_DEFAULT = 2;
constexpr int KSLICE_MAX = 16;

// Row decomposition of one quartet class for the Fock kernels.
// Primitive pairs per slice of the Fock-build class kernels: a work unit
// takes at most PSLICE bra primitive pairs (a 64-molecule 6-31G batch pass
// measured 372, 336, 313 and 313 ms for 4, 8, 16 and 32; (H2O)8 cc-pVDZ
// builds 1.95, 1.99 and 2.02 ms for 8, 16 and 32).
#ifndef MMD_PSLICE
#define MMD_PSLICE 16
#endif
constexpr int PSLICE = MMD_PSLICE;

// Per work unit: an upper bound of the pair factors q_P q_Q over the unit's
// quartets (rounded up to float) and the molecule of its bra pair, so that a
// unit whose every quartet fails the density-weighted screen is skipped
// before anything else of it is read.
struct UnitBound {
    float q;
    int32_t mol;
};

// Queues of work units per class: workgroup b draws from queue b % ROW_QUEUES,
// which holds every ROW_QUEUES-th unit of the list (costs are sorted, so the
// queues are alike).  One counter served a draw every 11 to 13 ns whoever
// asked, 300 us for the (ps|ss) and (ss|ss) units of a 45-molecule batch;
// counters in cache lines of their own are served side by side.
constexpr int ROW_QUEUES = 8;
constexpr int ROW_QUEUE_PAD = 32;      // ints: 128 bytes

struct RowArgs {
    int boff, nb;               // bra pairs of the class: pairs[boff .. boff+nb)
    int koff, nk;               // ket pairs of the class
    int tri;                    // same pair class: ket index <= bra index
    int rw;                     // width of the LDS rows: the largest molecule of the basis
    const int4* units;          // work units: {bra pair, first | end << 16 bra primitive pair, first ket, end ket}
    int nunits;
    int maxpp;                  // largest primitive-pair count of the class's bra pairs
    int kj;                     // LDS holds the ket-side Coulomb buffer (classes that have one)
    int kslice;                 // ket primitive pairs per lane item of the sliced classes (1 .. 16)
    int nshell;
    const double* Dsh;          // shell-block maxima of |dP| (nshell x nshell)
    const int* live;            // batches: the units that this build's density leaves alive; or null for all
    const int* nlive;           // their number
    double tier_lo, tier_hi;    // this launch takes quartets with tier_lo <= bound < tier_hi
    int* row_counter;           // ROW_QUEUES counters, ROW_QUEUE_PAD apart (zeroed before the launch)
    unsigned long long* stat_nquart;   // optional statistics
    unsigned long long* stat_nprim;
    const KetScreen* kscr;      // all pairs
    const KetRef* kref;
    const double* kpp;          // field f of primitive pair i at kpp[f * kstride + i]
    int64_t kstride;
};

// Work of one quartet class of the integral-block kernels: the stored tensor
// (raw = 0, A.G the N^4 output) or formPT's unsymmetrised build (raw = 1,
// A.G nrep copies of the real and imaginary N x N matrices).
constexpr int BLOCK_GROUPS = 16;     // quartets of a wavefront at most (groups of at least 4 lanes)
struct BlockArgs {
    int boff, nb, koff, nk;     // bra and ket pairs of the class
    int tri;                    // same pair class: ket <= bra
    int lgb, lgk;               // a group is 2^lgb x 2^lgk lanes: bra x ket primitive pairs
    const double* table;        // staged bra data of the bra's pair class
    int raw, nrep;
    const double* Dim;          // raw: imaginary part of dP, or null
    const double* Dsh;          // raw: shell-block maxima of |dP|
    const double* qraw;         // raw: per pair the largest square root of its Schwarz values
    int nshell;
};

}  // namespace mmd
