#pragma once
// Shell-quartet Fock-build kernel for gfx950, one instantiation per
// angular-momentum class (la lb | lc ld), la >= lb, lc >= ld,
// pair_class(bra) >= pair_class(ket).
//
// Work decomposition: one lane per (contracted shell quartet, chunk of bra
// Cartesian components); the chunk index is uniform across a wavefront, so
// every lane of a wave runs the same compile-time specialised code.
//
// All lanes of a work unit share the bra shell pair, whose primitive pairs
// (with their Hermite tables) are staged in LDS; per ket primitive pair the
// lane loops over them: Boys function from the LDS-staged Taylor table, R_tuv
// recursion in registers, and the bra contraction accumulated in the ket's
// Hermite space,
//   V_{tau nu phi}(ab) += sum_tuv E^{ab}_tuv R_{t+tau,u+nu,v+phi}.
// The ket expansion is applied once per ket primitive pair,
//   (ab|cd) += sum (-1)^{tau+nu+phi} E^{cd}_{tau nu phi} V_{tau nu phi}(ab),
// so the dense ket contraction is not repeated per primitive quartet.  All
// loops are unrolled at compile time (sfor) so that every array lives in
// registers.  The epilogue digests the block into the Fock matrix: Coulomb
// and exchange with the incremental density after the Schwarz x |dP| test.
//
// Reference semantics: cython/twoe.pyx:52-94 (primitive ERI),
// cython/twoe.pyx:34-50 (contraction), cython/fock.pyx:38-85 (screening,
// degeneracy, Coulomb/exchange scatter).
//
// This header is instantiated once per class by mmd_eri_class.hip.
#include <hip/hip_runtime.h>
#include "mmd_eri_core.h"
#include "mmd_kernels.h"

namespace mmd {

// Stage primitive pairs ip0 .. ip0+np-1 of the bra pair in LDS: p,
// 2 pi^{5/2} K / p, P and the three 1-D Hermite tables E^{ab}_t
// (cython/util.pxi:13-28).
template <int LA, int LB, int LC, int LD, typename T>
__device__ __forceinline__ void stage_bra(const ClassArgs& A, const ShellPair& bra, int ip0, int np, T* bp)
{
    using S = ClassShape<LA, LB, LC, LD>;
    for (int idx = threadIdx.x; idx < 3 * np; idx += blockDim.x) {
        const int ip = idx / 3, x = idx - 3 * ip;
        const PrimPair* P = A.pp + bra.pp0 + ip0 + ip;
        T* b = bp + ip * S::BPS;
        if (x == 0) {
            b[0] = (T)P->p;
            b[1] = (T)(TWO_PI_2_5 * P->K * P->invp);
            b[2] = (T)P->Px;
            b[3] = (T)P->Py;
            b[4] = (T)P->Pz;
        }
        double E[S::EB];
        hermite_E<LA, LB, 1>(P->inv2p, x == 0 ? P->PAx : (x == 1 ? P->PAy : P->PAz),
                             x == 0 ? P->PBx : (x == 1 ? P->PBy : P->PBz), E);
        sfor<S::EB>([&](auto k) { b[8 + x * S::EB + k] = (T)E[k]; });
    }
}

// Sum of v over the wavefront, in lane 63 (all 64 lanes active): four steps in
// the rows of 16 lanes, then across them, by DPP.
__device__ __forceinline__ double wave_sum63(double v)
{
    auto step = [](double x, auto ctrl, auto rows) {
        const long long b = __double_as_longlong(x);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)b, decltype(ctrl)::value, decltype(rows)::value, 0xf, true);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), decltype(ctrl)::value, decltype(rows)::value, 0xf, true);
        return x + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
    };
    using std::integral_constant;
    v = step(v, integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});   // row_shr:1
    v = step(v, integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});   // row_shr:2
    v = step(v, integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});   // row_shr:4
    v = step(v, integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});   // row_shr:8
    v = step(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});   // row_bcast:15
    v = step(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});   // row_bcast:31
    return v;
}

// Digest the integrals acc of a quartet (bra components A0..A1-1) into G.
// Called by whole wavefronts; lanes without a quartet pass on = false.
// rowA / rowB: rows of G for the bra shells' functions accumulated in LDS,
// row x holding column `col` of G at rowA[x * RW + col] (the caller offsets
// the pointers by the first column of the molecule); the ket-side Coulomb
// block goes to G.
template <int LA, int LB, int LC, int LD, int A0, int A1>
__device__ __forceinline__ void quartet_digest(const ClassArgs& A, int2 qd, const ShellPair& bra,
                                               const KetRef& ket, double* acc, double* rowA, double* rowB,
                                               int RW, bool on, double* kj = nullptr)
{
    using S = ClassShape<LA, LB, LC, LD>;
    constexpr int NCH = A1 - A0;
    constexpr int NCD = S::NCD;
    auto AI = [](int ab, int cd) { return (ab - A0) * NCD + cd; };
    // -----------------------------------------------------------------------
    // Epilogue: component scales, shell-level degeneracy, basis-function-level
    // Schwarz x |dP| test (cython/fock.pyx:46-57), then Coulomb and exchange.
    // Every component combination of the unique shell quartet is digested
    // with the shell degeneracy; the symmetrised result equals formPT's
    // symmetrised result for a real symmetric density difference.
    // -----------------------------------------------------------------------
    const int N = A.N;
    const int bfa = bra.bfa, bfb = bra.bfb, bfc = ket.bfa, bfd = ket.bfb;
    double ga[S::NA], gb[S::NB], gc[S::NC], gd[S::ND];
    sfor<S::NA>([&](auto i) { ga[i] = A.gcomp[bfa + i]; });
    sfor<S::NB>([&](auto i) { gb[i] = A.gcomp[bfb + i]; });
    sfor<S::NC>([&](auto i) { gc[i] = A.gcomp[bfc + i]; });
    sfor<S::ND>([&](auto i) { gd[i] = A.gcomp[bfd + i]; });
    const double deg = (bra.same ? 1.0 : 2.0) * (ket.bfa == ket.bfb ? 1.0 : 2.0) * (qd.x == qd.y ? 1.0 : 2.0);
    const double* D = A.D;
    double* G = A.G;
    const double* sq = A.sqS;
    const double tol = A.tol;
    // |dP| of the test is the absolute value of the D read for the updates
    // (one gathered read instead of two)
    auto aD = [&](int i, int j) { return fabs(D[(size_t)i * N + j]); };
    if (on) sfor<NCH>([&](auto ii) {
        constexpr int ab = A0 + decltype(ii)::value;
        constexpr int a = ab / S::NB, b = ab % S::NB;
        const int p = bfa + a, q = bfb + b;
        const double sab = sq[(size_t)p * N + q];
        const double dab = 4.0 * aD(p, q);
        sfor<NCD>([&](auto icd) {
            constexpr int cd = decltype(icd)::value;
            constexpr int c = cd / S::ND, d = cd % S::ND;
            const int r = bfc + c, s = bfd + d;
            const double bound = sab * sq[(size_t)r * N + s]
                * dmax6(dab, 4.0 * aD(r, s), aD(p, r), aD(p, s), aD(q, r), aD(q, s));
            const double v = acc[AI(ab, cd)] * deg * ga[a] * gb[b] * gc[c] * gd[d];
            acc[AI(ab, cd)] = (bound < tol) ? 0.0 : v;
        });
    });
    // Coulomb: G_ab += sum_cd (ab|cd) D_cd (bra rows): the same element for
    // every lane of the wavefront, so it is summed across the lanes first (64
    // LDS atomics on one address took 2.0 of the 2.5 ms of (dp|ss) at (H2O)16
    // cc-pVDZ, 0.9 of 1.2 of (dd|ss))
    sfor<NCH>([&](auto ii) {
        constexpr int ab = A0 + decltype(ii)::value;
        constexpr int a = ab / S::NB, b = ab % S::NB;
        double s = 0.0;
        if (on) sfor<NCD>([&](auto icd) {
            constexpr int cd = decltype(icd)::value;
            constexpr int c = cd / S::ND, d = cd % S::ND;
            s = fma(acc[AI(ab, cd)], D[(size_t)(bfc + c) * N + bfd + d], s);
        });
        s = wave_sum63(s);
        if ((threadIdx.x & 63) == 63) atomicAdd(&rowA[a * RW + bfb + b], s);
    });
    if (!on) return;
    // Coulomb: G_cd += sum_ab (ab|cd) D_ab   (ket block: to G, or to the
    // quartet's LDS row kj when given, added to G after the batch)
    sfor<NCD>([&](auto icd) {
        constexpr int cd = decltype(icd)::value;
        constexpr int c = cd / S::ND, d = cd % S::ND;
        double s = 0.0;
        sfor<NCH>([&](auto ii) {
            constexpr int ab = A0 + decltype(ii)::value;
            constexpr int a = ab / S::NB, b = ab % S::NB;
            s = fma(acc[AI(ab, cd)], D[(size_t)(bfa + a) * N + bfb + b], s);
        });
        if (kj)
            atomicAdd(&kj[cd], s);
        else
            atomicAdd(&G[(size_t)(bfc + c) * N + bfd + d], s);
    });
    // Exchange (cython/fock.pyx:82-85): G_bd -= 1/4 (ab|cd) D_ac ;
    // G_bc -= 1/4 (ab|cd) D_ad ; G_ac -= 1/4 (ab|cd) D_bd ; G_ad -= 1/4 (ab|cd) D_bc.
    // Each target element sums the item's contributions in registers first.
    sfor<S::NB>([&](auto ix) {
        constexpr int x = decltype(ix)::value;
        sfor<S::ND>([&](auto iy) {        // (b,d) block
            constexpr int y = decltype(iy)::value;
            double s = 0.0;
            bool any = false;
            sfor<S::NA>([&](auto ia) {
                constexpr int a = decltype(ia)::value;
                constexpr int ab = a * S::NB + x;
                if constexpr (ab >= A0 && ab < A1) {
                    any = true;
                    sfor<S::NC>([&](auto icc) {
                        constexpr int c = decltype(icc)::value;
                        s = fma(acc[AI(ab, c * S::ND + y)], D[(size_t)(bfa + a) * N + bfc + c], s);
                    });
                }
            });
            if (any) atomicAdd(&rowB[x * RW + bfd + y], -0.25 * s);
        });
        sfor<S::NC>([&](auto iy) {        // (b,c) block
            constexpr int y = decltype(iy)::value;
            double s = 0.0;
            bool any = false;
            sfor<S::NA>([&](auto ia) {
                constexpr int a = decltype(ia)::value;
                constexpr int ab = a * S::NB + x;
                if constexpr (ab >= A0 && ab < A1) {
                    any = true;
                    sfor<S::ND>([&](auto idd) {
                        constexpr int d = decltype(idd)::value;
                        s = fma(acc[AI(ab, y * S::ND + d)], D[(size_t)(bfa + a) * N + bfd + d], s);
                    });
                }
            });
            if (any) atomicAdd(&rowB[x * RW + bfc + y], -0.25 * s);
        });
    });
    sfor<S::NA>([&](auto ix) {
        constexpr int x = decltype(ix)::value;
        sfor<S::NC>([&](auto iy) {        // (a,c) block
            constexpr int y = decltype(iy)::value;
            double s = 0.0;
            bool any = false;
            sfor<S::NB>([&](auto ib) {
                constexpr int b = decltype(ib)::value;
                constexpr int ab = x * S::NB + b;
                if constexpr (ab >= A0 && ab < A1) {
                    any = true;
                    sfor<S::ND>([&](auto idd) {
                        constexpr int d = decltype(idd)::value;
                        s = fma(acc[AI(ab, y * S::ND + d)], D[(size_t)(bfb + b) * N + bfd + d], s);
                    });
                }
            });
            if (any) atomicAdd(&rowA[x * RW + bfc + y], -0.25 * s);
        });
        sfor<S::ND>([&](auto iy) {        // (a,d) block
            constexpr int y = decltype(iy)::value;
            double s = 0.0;
            bool any = false;
            sfor<S::NB>([&](auto ib) {
                constexpr int b = decltype(ib)::value;
                constexpr int ab = x * S::NB + b;
                if constexpr (ab >= A0 && ab < A1) {
                    any = true;
                    sfor<S::NC>([&](auto icc) {
                        constexpr int c = decltype(icc)::value;
                        s = fma(acc[AI(ab, c * S::ND + y)], D[(size_t)(bfb + b) * N + bfc + c], s);
                    });
                }
            });
            if (any) atomicAdd(&rowA[x * RW + bfd + y], -0.25 * s);
        });
    });
}

// ---------------------------------------------------------------------------
// Class kernel.  A work unit is one bra shell pair ("row"), a slice of at
// most PSLICE of its primitive pairs and a segment of its ket pairs (a
// table built at set-up, heaviest first); workgroups draw units from the
// queues of ROW_QUEUES.  The unit's ket pairs are screened a workgroup at a time;
// survivors are appended to an LDS list that is digested whenever it holds
// a full batch, as wave items of (bra-component chunk, 64 consecutive
// (ket primitive slice, quartet) lane items).  Classes with an integral
// buffer (IBUF) slice the ket primitives too, add each item's partial
// integrals into LDS and digest every quartet once, after the batch; the
// others contract a quartet's whole ket side in one lane and digest it.  Coulomb G_ab and the four exchange
// blocks, all in the rows of the bra shells, are accumulated in LDS
// (ds_add_f64) and their nonzero entries added to G once per unit; only the
// ket-side Coulomb block is added to G directly.  (The host sends a class
// whose bra rows do not fit in LDS to the wavefront-per-quartet kernel.)
// ---------------------------------------------------------------------------
constexpr int CLASS_BLOCK = 256;           // threads per workgroup

#ifndef MMD_BOYS_LDS_MIN_L
#define MMD_BOYS_LDS_MIN_L 0
#endif
constexpr int BOYS_LDS_MIN_L = MMD_BOYS_LDS_MIN_L;   // classes with L below it read Boys rows from L1

template <int QB>
struct ClassList {
    static constexpr int QLIST = QB + CLASS_BLOCK;   // batch + one screening step
};

// Least wavefronts per SIMD that the compiler plans the registers for, class
// by class as measured.  The row kernels wait more than they compute (at
// (H2O)16 cc-pVDZ the vector units are busy 30% of the time), so a second or
// third wavefront can pay for the registers it spills: (pp|pp) 0.385 -> 0.284, (ds|pp) 0.451 -> 0.321, (ds|ds)
// 0.332 -> 0.281 ms for two instead of one (2-15 registers spilled), (ps|ps)
// 1.21 -> 1.10 ms for three instead of two (none).  (pp|ps), (dp|ss), (dp|ps)
// and (dd|ss) were slower with more.
template <int LA, int LB, int LC, int LD, typename T>
constexpr int row_min_waves()
{
    constexpr int c = LA * 1000 + LB * 100 + LC * 10 + LD;
    if (!std::is_same<T, double>::value) return 1;
    if (c == 1111 || c == 2011 || c == 2020) return 2;
    return c == 1010 ? 3 : 1;
}

// T is the arithmetic type of the integrals (double, or float for the
// FP32 tier); screening, digestion and all accumulation into G are FP64.
template <int LA, int LB, int LC, int LD, typename T>
__global__ void __launch_bounds__(CLASS_BLOCK, (row_min_waves<LA, LB, LC, LD, T>())) eri_fock_class_kernel(ClassArgs A, RowArgs R)
{
    using S = ClassShape<LA, LB, LC, LD>;
    constexpr int QB = S::QB;
    static_assert(QB <= CLASS_BLOCK, "one thread per batch entry in the slice-count scan");
    extern __shared__ double dyn[];
    double* rows = dyn;
    const int RW = R.rw;
    double* ibuf = rows + (S::NA + S::NB) * RW;
    // ket-side Coulomb buffer (KJ classes, when the launch has room for it)
    const bool kj = S::KJ && R.kj;
    const int nbuf = S::IBUF_DOUBLES + (kj ? S::KJ_DOUBLES : 0);
    // the class's Boys rows in LDS, or read from the global table (L1) for
    // the classes below BOYS_LDS_MIN_L, which leaves their workgroups the LDS
    // for more of them per CU (the default keeps every class in LDS: reading
    // the rows through L1 made the (ps|ss) class 20% slower)
    constexpr bool boys_lds = S::L >= BOYS_LDS_MIN_L;
    T* lds_boys = reinterpret_cast<T*>(ibuf + nbuf);
    T* bp = boys_lds ? lds_boys + BOYS_TAYLOR * BOYS_NT : lds_boys;
    int* qlist = reinterpret_cast<int*>(bp + (size_t)(R.maxpp < PSLICE ? R.maxpp : PSLICE) * S::BPS);
    int* misc = qlist + ClassList<QB>::QLIST;
    int* pre = misc + 4;         // IBUF classes: prefix sums of the batch's ket slice counts
    int* wsum = pre + QB + 1;    // per-wavefront partial sums of that scan
    const T* boys_tab;
    if constexpr (std::is_same<T, float>::value) {
        if constexpr (boys_lds) boys_stage_lds<S::L, float>(lds_boys, A.boysf);
        boys_tab = boys_lds ? lds_boys : A.boysf + (size_t)S::L * BOYS_NT;
    } else {
        if constexpr (boys_lds) boys_stage_lds<S::L, double>(lds_boys, A.boys);
        boys_tab = boys_lds ? lds_boys : A.boys + (size_t)S::L * BOYS_NT;
    }
    for (int i = threadIdx.x; i < nbuf; i += blockDim.x) ibuf[i] = 0.0;
    const int N = A.N;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nwv = (int)(blockDim.x >> 6);
    const int nunits = R.live ? *R.nlive : R.nunits;
    const int nqueue = min(ROW_QUEUES, (int)gridDim.x), queue = (int)blockIdx.x % nqueue;
    const size_t ns = (size_t)R.nshell;
    unsigned long long my_nprim = 0;   // primitive quartets of this lane (statistics)
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) misc[0] = atomicAdd(&R.row_counter[queue * ROW_QUEUE_PAD], 1) * nqueue + queue;
        __syncthreads();
        const int iu = misc[0];
        if (iu >= nunits) {
            if (R.stat_nprim) {   // one atomic per wavefront
                for (int off = 32; off > 0; off >>= 1) my_nprim += __shfl_xor(my_nprim, off);
                if (lane == 0 && my_nprim) atomicAdd(R.stat_nprim, my_nprim);
            }
            break;
        }
        // unit: bra pair P, its primitive pairs [ip0, ip1) and the ket
        // pairs [k0, k1) of its molecule
        const int u = R.live ? R.live[iu] : iu;
        const int4 U = R.units[u];
        const int P = U.x, k0 = U.z;
        const int ip0u = U.y & 0xffff, ip1u = U.y >> 16;
        const int segn = U.w - U.z;
        const int bnp = ip1u - ip0u;   // bra primitive pairs of the unit (<= PSLICE)
        const ShellPair bra = A.pairs[R.boff + P];
        const int nrows = bra.same ? S::NA : S::NA + S::NB;
        const int c0 = bra.c0;       // the rows hold the molecule's columns c0 .. c0+RW-1
        double* rowA = rows - c0;
        double* rowB = rows + (bra.same ? 0 : S::NA * RW) - c0;
        for (int i = threadIdx.x; i < nrows * RW; i += blockDim.x) rows[i] = 0.0;
        stage_bra<LA, LB, LC, LD, T>(A, bra, ip0u, bnp, bp);
        if (threadIdx.x == 0) misc[1] = 0;   // survivors in the list
        __syncthreads();
        for (int t0 = 0;; t0 += (int)blockDim.x) {
            // screen the next kets and append the survivors
            if (t0 < segn) {
                const int t = t0 + threadIdx.x;
                bool keep = false;
                if (t < segn) {
                    const KetScreen ket = R.kscr[R.koff + k0 + t];
                    const double* Dsh = R.Dsh;
                    const double dm = fmax(fmax(fmax(4.0 * Dsh[bra.sa * ns + bra.sb], 4.0 * Dsh[ket.sa * ns + ket.sb]),
                                                fmax(Dsh[bra.sa * ns + ket.sa], Dsh[bra.sa * ns + ket.sb])),
                                           fmax(Dsh[bra.sb * ns + ket.sa], Dsh[bra.sb * ns + ket.sb]));
                    const double bound = bra.q * ket.q * dm;
                    keep = bound >= A.tol && bound >= R.tier_lo && bound < R.tier_hi;
                }
                const unsigned long long m = __ballot(keep);
                int pos = 0;
                if (lane == 0 && m) pos = atomicAdd(&misc[1], __popcll(m));
                pos = __shfl(pos, 0);
                if (keep) qlist[pos + __popcll(m & ((1ull << lane) - 1ull))] = k0 + t;
            }
            __syncthreads();
            const int cnt0 = misc[1];
            const bool last = t0 + (int)blockDim.x >= segn;
            for (int b0 = 0; b0 < cnt0 && (cnt0 - b0 >= QB || last); b0 += QB) {
                // digest the batch qlist[b0, b0+cnt): a wavefront takes one
                // chunk of bra components and 64 consecutive lane items.
                // Classes that add partial integrals into the LDS buffer
                // split each ket's primitives into slices of R.kslice; their
                // lane items are the (quartet, ket slice) pairs that exist,
                // numbered through the prefix sums pre[] of the quartets'
                // slice counts, so that lanes stay busy however the batch
                // mixes contraction lengths.  The other classes take a
                // quartet's whole ket contraction in one lane and digest it.
                const int cnt = min(QB, cnt0 - b0);
                if (R.stat_nquart && threadIdx.x == 0) atomicAdd(R.stat_nquart, (unsigned long long)cnt);
                int nflat = cnt;
                if constexpr (S::KSL) {
                    const int j = threadIdx.x;   // cnt <= QB <= CLASS_BLOCK
                    int x = 0;
                    if (j < cnt) x = (R.kref[R.koff + qlist[b0 + j]].npp + R.kslice - 1) / R.kslice;
                    for (int off = 1; off < 64; off <<= 1) {
                        const int y = __shfl_up(x, off);
                        if (lane >= off) x += y;
                    }
                    if (lane == 63) wsum[wv] = x;
                    __syncthreads();
                    for (int k = 0; k < wv; ++k) x += wsum[k];
                    if (j < cnt) pre[j + 1] = x;
                    if (j == 0) pre[0] = 0;
                    __syncthreads();
                    nflat = pre[cnt];
                }
                const int total = ((nflat + 63) / 64) * S::NCHUNK;
                for (int w = wv; w < total; w += nwv) {
                    const int chunk = w % S::NCHUNK;
                    // lanes beyond the last item repeat it with no primitives
                    const int item = (w / S::NCHUNK) * 64 + lane;
                    const bool on = item < nflat;
                    const int flat = on ? item : nflat - 1;
                    int idx = flat, ks = 0;
                    if constexpr (S::KSL) {
                        // the quartet whose slices cover item flat: pre[idx] <= flat < pre[idx + 1]
                        int lo = 0, hi = cnt - 1;
                        while (lo < hi) {
                            const int mid = (lo + hi + 1) >> 1;
                            if (pre[mid] <= flat) lo = mid;
                            else hi = mid - 1;
                        }
                        idx = lo;
                        ks = flat - pre[lo];
                    }
                    const int Q = qlist[b0 + idx];
                    const int2 qd = make_int2(R.boff + P, R.koff + Q);
                    const KetRef ket = R.kref[qd.y];
                    const int jq0 = ks * R.kslice;
                    const int jq1 = on ? (S::KSL ? min(ket.npp, jq0 + R.kslice) : ket.npp) : jq0;
                    const int ip0 = 0, ip1 = bnp;
                    if (chunk == 0) my_nprim += (unsigned long long)(ip1 - ip0) * (unsigned long long)(jq1 - jq0);
                    static_switch<0, S::NCHUNK>(chunk, [&](auto ic) {
                        constexpr int C = decltype(ic)::value;
                        constexpr int A0 = C * S::CH, A1 = (C + 1) * S::CH;
                        T acc[(A1 - A0) * S::NCD];
                        quartet_compute<LA, LB, LC, LD, A0, A1, T>(KetArrays{R.kpp, R.kstride}, boys_tab, bp, ip0, ip1,
                                                                   ket.pp0 + jq0, ket.pp0 + jq1, acc);
                        if constexpr (S::IBUF) {
                            double* dst = ibuf + (size_t)idx * S::NABCD + A0 * S::NCD;
                            if (on) sfor<(A1 - A0) * S::NCD>(
                                [&](auto k) { atomicAdd(&dst[decltype(k)::value], (double)acc[k]); });
                        } else {
                            double accd[(A1 - A0) * S::NCD];
                            sfor<(A1 - A0) * S::NCD>([&](auto k) { accd[k] = (double)acc[k]; });
                            quartet_digest<LA, LB, LC, LD, A0, A1>(A, qd, bra, ket, accd, rowA, rowB, RW, on,
                                                                   kj ? ibuf + (size_t)idx * S::NCD : nullptr);
                        }
                    });
                }
                if (kj) {
                    // the summed ket-side Coulomb blocks of the batch into G
                    // (kj is uniform across the workgroup)
                    __syncthreads();
                    for (int i = threadIdx.x; i < cnt * S::NCD; i += blockDim.x) {
                        const double v = ibuf[i];
                        if (v == 0.0) continue;
                        ibuf[i] = 0.0;
                        const int idx = i / S::NCD, cd = i - idx * S::NCD;
                        const KetRef ket = R.kref[R.koff + qlist[b0 + idx]];
                        atomicAdd(&A.G[(size_t)(ket.bfa + cd / S::ND) * N + ket.bfb + cd % S::ND], v);
                    }
                }
                if constexpr (S::IBUF) {
                    // every quartet of the batch once: its summed integrals into G
                    __syncthreads();
                    const int total2 = ((cnt + 63) / 64) * S::NCHUNK;
                    for (int w = wv; w < total2; w += nwv) {
                        const int chunk = w % S::NCHUNK;
                        const int item = (w / S::NCHUNK) * 64 + lane;
                        const bool on = item < cnt;
                        const int idx = on ? item : cnt - 1;
                        const int Q = qlist[b0 + idx];
                        const int2 qd = make_int2(R.boff + P, R.koff + Q);
                        const KetRef ket = R.kref[qd.y];
                        static_switch<0, S::NCHUNK>(chunk, [&](auto ic) {
                            constexpr int C = decltype(ic)::value;
                            constexpr int A0 = C * S::CH, A1 = (C + 1) * S::CH;
                            double acc[(A1 - A0) * S::NCD];
                            double* src = ibuf + (size_t)idx * S::NABCD + A0 * S::NCD;
                            if (on) sfor<(A1 - A0) * S::NCD>([&](auto k) {
                                acc[k] = src[decltype(k)::value];
                                src[decltype(k)::value] = 0.0;
                            });
                            quartet_digest<LA, LB, LC, LD, A0, A1>(A, qd, bra, ket, acc, rowA, rowB, RW, on);
                        });
                    }
                }
                __syncthreads();
            }
            if (last) break;
            // keep the survivors that did not fill a batch at the front of the list
            const int done = (cnt0 / QB) * QB;
            const int rest = cnt0 - done;
            if (done > 0) {
                int v = 0;
                if ((int)threadIdx.x < rest) v = qlist[done + threadIdx.x];
                __syncthreads();
                if ((int)threadIdx.x < rest) qlist[threadIdx.x] = v;
                if (threadIdx.x == 0) misc[1] = rest;
            }
            __syncthreads();
        }
        __syncthreads();
        for (int i = threadIdx.x; i < nrows * RW; i += blockDim.x) {
            const double v = rows[i];
            const int x = i / RW, col = c0 + i - x * RW;
            const int g = x < S::NA ? bra.bfa + x : bra.bfb + (x - S::NA);
            if (v != 0.0) atomicAdd(&A.G[(size_t)g * N + col], v);
        }
    }
}

template <int LA, int LB, int LC, int LD, typename T>
inline size_t fock_class_lds_bytes(int RW, int maxpp, int kj)
{
    using S = ClassShape<LA, LB, LC, LD>;
    return sizeof(double) * ((size_t)(S::NA + S::NB) * RW + S::IBUF_DOUBLES + (kj ? S::KJ_DOUBLES : 0))
         + sizeof(T) * ((S::L >= BOYS_LDS_MIN_L ? BOYS_TAYLOR * BOYS_NT : 0)
                        + (size_t)(maxpp < PSLICE ? maxpp : PSLICE) * S::BPS)
         + sizeof(int) * (ClassList<S::QB>::QLIST + 4 + S::QB + 1 + CLASS_BLOCK / 64);
}

}  // namespace mmd
