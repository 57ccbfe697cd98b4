// Shell-pair and primitive-pair tables and the Fock build's work units, on
// the device.  A group of 128 clusters of six waters in 6-31G has 190 thousand
// shell pairs, 1.1 million primitive pairs and 150 thousand work units; on one
// host thread they took 102 ms, the iterations of the group 74 ms.
//
// A group of lanes per pair: the largest Schwarz-type bound of its primitive
// pairs, the number that survive the primitive screen, its factor
// q = max sqrt((ab|ab)).  A pair's place in its class is the number of pairs of
// its molecule that sort before it (molecules have at most a few thousand
// pairs of a class, and the lanes of a wavefront read the same ones), its
// place in the primitive table a prefix sum.  Units are counted into cost
// buckets and scattered through the buckets' cursors.
//
// Every step needs all of the one before it.  A table of up to PAIR_ONE pairs
// (two waters in 6-31G) takes them in one workgroup and one launch; more pairs
// keep more than one compute unit busy.  Tables and units after a new Schwarz
// diagonal, one workgroup against ten launches: 45 pairs ((H2O) 6-31G) 39 and
// 78 us, 171 60 and 76, 300 86 and 83, 465 130 and 109, 666 160 and 119.  A
// host thread took 67, 118, 160, 178 and 260 to 290 us, 441 for 1035 pairs
// (146 here).
#include <hip/hip_runtime.h>
#include "mmd_pairs.h"

namespace mmd {

namespace {

constexpr double PRIM_DROP = 1e-20;
constexpr int SCAN_BLOCK = 1024;
constexpr int PAIR_ONE = 256;         // pairs that one workgroup sorts (at most SCAN_BLOCK)
static_assert(PAIR_ONE <= SCAN_BLOCK, "a thread per pair");
constexpr int GL = 16;                // lanes of a pair's primitive loops (PAIR_KEEP_BITS)
static_assert(GL == PAIR_KEEP_BITS, "a round of the group's lanes is a piece of keep bits");

// Schwarz-type bound of a primitive pair's product function (any component):
// sqrt([ab|ab]) of an s-type pair, 2 pi^{5/2} / (p^2 sqrt(2p)) K^2, times
// (1 + |AB| + 1/sqrt(p))^{la+lb} 4^{la+lb} to cover the Hermite expansion of
// higher angular momenta.
__device__ double prim_bound(double p, double K, double AB2, int lab)
{
    const double s = sqrt(34.98683665524972497 / (p * p * sqrt(2.0 * p))) * fabs(K);
    const double f = 4.0 * (1.0 + sqrt(AB2) + 1.0 / sqrt(p));
    double m = 1.0;
    for (int i = 0; i < lab; ++i) m *= f;
    return s * m;
}

__device__ double dist2(const OneeShell& a, const OneeShell& b)
{
    return (a.x - b.x) * (a.x - b.x) + (a.y - b.y) * (a.y - b.y) + (a.z - b.z) * (a.z - b.z);
}

__device__ int class_of_entry(const int* off, int e)
{
    int c = 0;
    while (e >= off[c + 1]) ++c;
    return c;
}

// Largest bound among the primitive pairs of lane li of pair e.
__device__ double pair_bound(const PairInput& I, int e, int li)
{
    const int2 pr = I.list[e];
    const OneeShell a = I.shells[pr.x], b = I.shells[pr.y];
    const double AB2 = dist2(a, b);
    double m = 0.0;
    for (int k = li; k < a.np * b.np; k += GL) {
        const int i = k / b.np, j = k - i * b.np;
        const double ea = I.exps[a.p0 + i], eb = I.exps[b.p0 + j], p = ea + eb;
        m = fmax(m, prim_bound(p, I.wts[a.p0 + i] * I.wts[b.p0 + j] * exp(-ea * eb / p * AB2), AB2, a.l + b.l));
    }
    return m;
}

__device__ void add_bound(double m, unsigned long long* qmax)
{
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
    // positive doubles order like their bits; most wavefronts find theirs below
    // the maximum so far and need no turn at the one address
    const unsigned long long bits = (unsigned long long)__double_as_longlong(m);
    if ((threadIdx.x & 63) == 0 && m > 0.0 && bits > __hip_atomic_load(qmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(qmax, bits);
}

// A primitive pair whose bound, times the largest bound of any pair, is below
// PRIM_DROP contributes less than that to every primitive quartet and is
// left out of the table.  Decided here once, as a bit of the pair's keep pieces:
// the count sizes the pair's range of the table and the fill writes it, and a
// pair at the threshold that each decided for itself, in code that the
// compiler contracts in its own way, could be one record more than the range.
__device__ void pair_count(const PairInput& I, const PairWork& W, double qmax, int e, int li)
{
    const int npairs = I.off[NPAIRCLASS];
    const int2 pr = I.list[e];
    const OneeShell a = I.shells[pr.x], b = I.shells[pr.y];
    const double AB2 = dist2(a, b);
    const int np = a.np * b.np, shift = threadIdx.x & 63 & ~(GL - 1);
    int n = 0;
    for (int k0 = 0, t = 0; k0 < np; k0 += GL, ++t) {   // the group's lanes together
        const int k = k0 + li;
        bool keep = false;
        if (k < np) {
            const int i = k / b.np, j = k - i * b.np;
            const double ea = I.exps[a.p0 + i], eb = I.exps[b.p0 + j], p = ea + eb;
            const double K = I.wts[a.p0 + i] * I.wts[b.p0 + j] * exp(-ea * eb / p * AB2);
            keep = !(prim_bound(p, K, AB2, a.l + b.l) * qmax < PRIM_DROP);
        }
        const unsigned piece = (unsigned)(__ballot(keep) >> shift) & ((1u << GL) - 1u);
        n += __popc(piece);
        if (li == 0) W.keep[(size_t)t * npairs + e] = (uint16_t)piece;
    }
    double q = 1.0;
    if (I.diag) {
        q = 0.0;
        const int nb = ncart(b.l);
        for (int c = li; c < ncart(a.l) * nb; c += GL) {
            const int x = c / nb, y = c - x * nb;
            const double v = I.diag[(size_t)(a.bf0 + x) * I.N + b.bf0 + y];
            q = fmax(q, v > 0.0 ? sqrt(v) : 0.0);
        }
        for (int off = GL / 2; off > 0; off >>= 1) q = fmax(q, __shfl_xor(q, off));
    }
    if (li == 0) {
        W.count[e] = n;
        W.q[e] = n == 0 ? 0.0 : q;   // no primitive pair survives: never screened in
    }
}

// Place of pair e among those of its molecule and class, and its record.
__device__ void pair_rank(const PairInput& I, const PairWork& W, ShellPair* pairs, int e)
{
    const int c = class_of_entry(I.off, e);
    const int2 pr = I.list[e];
    const OneeShell a = I.shells[pr.x], b = I.shells[pr.y];
    const int2 seg = I.ranges[(size_t)c * I.nmol + a.mol];
    const int s0 = I.off[c] + seg.x, s1 = I.off[c] + seg.y;
    const int n = W.count[e];
    const double q = W.q[e];
    int rank = 0;
    auto before = [&](int nj, double qj, int j) {
        rank += (nj > n || (nj == n && (qj > q || (qj == q && j < e)))) ? 1 : 0;
    };
    int j = s0;
    for (; j + 8 <= s1; j += 8) {   // eight loads in flight: one at a time took 220 ns
        int nj[8];
        double qj[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            nj[u] = W.count[j + u];
            qj[u] = W.q[j + u];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) before(nj[u], qj[u], j + u);
    }
    for (; j < s1; ++j) before(W.count[j], W.q[j], j);
    ShellPair sp;
    sp.sa = pr.x;
    sp.sb = pr.y;
    sp.bfa = a.bf0;
    sp.bfb = b.bf0;
    sp.pp0 = 0;
    sp.npp = n;
    sp.same = pr.x == pr.y ? 1 : 0;
    sp.mol = a.mol;
    sp.c0 = I.mol_blocks ? I.mol_blocks[a.mol].x : 0;
    sp.class_pp0 = 0;
    sp.q = q;
    pairs[s0 + rank] = sp;
    W.entry[s0 + rank] = e;
}

// Exclusive prefix sum over the SCAN_BLOCK threads; all: the total.
__device__ int block_scan(int v, int* part, int* all)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int x = v;
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) part[wv] = x;
    __syncthreads();
    int before = 0, sum = 0;
    for (int k = 0; k < SCAN_BLOCK / 64; ++k) {
        if (k < wv) before += part[k];
        sum += part[k];
    }
    __syncthreads();
    *all = sum;
    return before + x - v;
}

__device__ int pair_start(const int* scan, const int* sums, int i) { return scan[i] + sums[i / SCAN_BLOCK]; }

// Table range of sorted pair i, and per class the largest and total count.
__device__ void pair_place(const PairInput& I, const int* scan, const int* sums, ShellPair* pairs, PairStats* stats,
                           int i)
{
    const int c = class_of_entry(I.off, i);
    const int p0 = pair_start(scan, sums, i);
    const int at = p0 - pair_start(scan, sums, I.off[c]);
    const int n = pairs[i].npp;
    pairs[i].pp0 = p0;
    pairs[i].class_pp0 = at;
    // the first pair of a molecule holds its largest count
    if (i == I.off[c] + I.ranges[(size_t)c * I.nmol + pairs[i].mol].x) atomicMax(&stats->maxpp[c], n);
    if (i == I.off[c + 1] - 1) stats->total[c] = at + n;
}

// The primitive-pair records of sorted pair e: lane li takes every GL-th
// primitive pair, and its place among the kept ones.
__device__ void pair_fill(const PairInput& I, const PairWork& W, const ShellPair* __restrict__ pairs,
                          PrimPair* __restrict__ pp, double* __restrict__ ppa, const KetTables& K, int e, int li)
{
    const int npairs = I.off[NPAIRCLASS];
    const ShellPair sp = pairs[e];
    const OneeShell a = I.shells[sp.sa], b = I.shells[sp.sb];
    const double AB2 = dist2(a, b);
    const uint16_t* keep = W.keep + W.entry[e];
    if (li == 0) {
        K.scr[e] = KetScreen{sp.q, sp.sa, sp.sb};
        K.ref[e] = KetRef{sp.bfa, sp.bfb, sp.pp0, sp.npp};
    }
    int base = sp.pp0;
    for (int k = li; k < a.np * b.np; k += GL, keep += npairs) {
        const unsigned piece = *keep;
        const int o = base + __popc(piece & ((1u << li) - 1u));
        base += __popc(piece);
        if (!(piece >> li & 1u)) continue;
        const int i = k / b.np, j = k - i * b.np;
        const double ea = I.exps[a.p0 + i], eb = I.exps[b.p0 + j];
        PrimPair pq;
        pq.p = ea + eb;
        pq.K = I.wts[a.p0 + i] * I.wts[b.p0 + j] * exp(-ea * eb / pq.p * AB2);
        pq.Px = (ea * a.x + eb * b.x) / pq.p;
        pq.Py = (ea * a.y + eb * b.y) / pq.p;
        pq.Pz = (ea * a.z + eb * b.z) / pq.p;
        pq.PAx = pq.Px - a.x;
        pq.PAy = pq.Py - a.y;
        pq.PAz = pq.Pz - a.z;
        pq.PBx = pq.Px - b.x;
        pq.PBy = pq.Py - b.y;
        pq.PBz = pq.Pz - b.z;
        pq.inv2p = 0.5 / pq.p;
        pq.invp = 1.0 / pq.p;
        pp[o] = pq;
        ppa[o] = ea;
        const double f[KET_FIELDS] = {pq.p, pq.K * pq.invp, pq.Px, pq.Py, pq.Pz, pq.inv2p,
                                      pq.PAx, pq.PAy, pq.PAz, pq.PBx, pq.PBy, pq.PBz};
        for (int u = 0; u < KET_FIELDS; ++u) K.pp[u * K.stride + o] = f[u];
    }
}

// ---------------------------------------------------------------------------
// Work units
// ---------------------------------------------------------------------------

// Running maximum of the pair factors over the QMAX_BLOCK pairs that pair i
// lies in, counted from its molecule's first pair of the class.
__device__ void unit_qrun(const UnitInput& I, double* qrun, int i)
{
    const int c = class_of_entry(I.off, i);
    const int first = I.off[c] + I.ranges[(size_t)c * I.nmol + I.pairs[i].mol].x;
    double m = 0.0;
#pragma unroll 8
    for (int k = first + (i - first) / QMAX_BLOCK * QMAX_BLOCK; k <= i; ++k) m = fmax(m, I.pairs[k].q);
    qrun[i] = m;
}

__device__ int unit_bucket(long long cost)   // 0 for the heaviest
{
    const float f = (float)(cost > 1 ? cost : 1);
    const int b = (__float_as_int(f) >> 21) - (127 << 2);   // quarter octaves
    return UNIT_BUCKETS - 1 - (b < UNIT_BUCKETS ? b : UNIT_BUCKETS - 1);
}

struct UnitRange {
    int P, npp, kfirst, kend, nfull, rest;   // nfull slices of PSLICE primitive pairs, and one of `rest`
};

// Bra pair `entry` of quartet class qc and the kets of its units.
__device__ UnitRange unit_range(const UnitInput& I, int pcb, int pck, int entry)
{
    const ShellPair& sp = I.pairs[I.off[pcb] + entry];
    const int2 r = I.ranges[(size_t)pck * I.nmol + sp.mol];
    UnitRange u;
    u.P = entry;
    u.npp = sp.npp;
    u.kfirst = r.x;
    u.kend = pcb == pck ? entry + 1 : r.y;
    u.nfull = sp.npp / PSLICE;
    u.rest = sp.npp - u.nfull * PSLICE;
    return u;
}

// primitive pairs of the kets [k0, k1) of a class
__device__ long long ket_prims(const UnitInput& I, int pck, int k0, int k1)
{
    const ShellPair& a = I.pairs[I.off[pck] + k0];
    const ShellPair& z = I.pairs[I.off[pck] + k1 - 1];
    return (long long)z.pp0 + z.npp - a.pp0;
}

__device__ void qclass_pairs(int qc, int* pcb, int* pck)
{
    int b = 0;
    while ((b + 1) * (b + 2) / 2 <= qc) ++b;
    *pcb = b;
    *pck = qc - b * (b + 1) / 2;
}

// Bra pair e of class qc into the class's cost buckets h.
__device__ void unit_count(const UnitInput& I, int qc, int pcb, int pck, int e, int* h)
{
    const UnitRange u = unit_range(I, pcb, pck, e);
    for (int k0 = u.kfirst; k0 < u.kend; k0 += I.seg[qc]) {
        const long long kc = ket_prims(I, pck, k0, min(u.kend, k0 + I.seg[qc]));
        if (u.nfull) atomicAdd(&h[unit_bucket(PSLICE * kc)], u.nfull);
        if (u.rest) atomicAdd(&h[unit_bucket(u.rest * kc)], 1);
    }
}

// Bucket counts to cursors (positions in the table of all classes; one
// workgroup of SCAN_BLOCK threads, three counters each) and the classes'
// totals.  in may be out.
__device__ void unit_scan(const int* in, int* out, int* counts, int* part)
{
    constexpr int HIST = NQCLASS * UNIT_BUCKETS;
    static_assert(HIST <= 3 * SCAN_BLOCK, "three counters per thread");
    __shared__ int start[NQCLASS];
    int v[3], sum = 0, all;
    for (int u = 0; u < 3; ++u) {
        const int i = 3 * threadIdx.x + u;
        v[u] = i < HIST ? in[i] : 0;
        sum += v[u];
    }
    int pos = block_scan(sum, part, &all);
    for (int u = 0; u < 3; ++u) {
        const int i = 3 * threadIdx.x + u;
        if (i >= HIST) break;
        if (i % UNIT_BUCKETS == 0) start[i / UNIT_BUCKETS] = pos;
        out[i] = pos;
        pos += v[u];
    }
    __syncthreads();
    if (threadIdx.x < NQCLASS)
        counts[threadIdx.x] = (threadIdx.x + 1 < NQCLASS ? start[threadIdx.x + 1] : all) - start[threadIdx.x];
}

__device__ void unit_scatter(const UnitInput& I, int* __restrict__ hist, const double* __restrict__ qrun,
                             int4* __restrict__ units, UnitBound* __restrict__ bounds, int qc, int pcb, int pck, int e)
{
    const UnitRange u = unit_range(I, pcb, pck, e);
    const double q = I.pairs[I.off[pcb] + e].q;
    const int mol = I.pairs[I.off[pcb] + e].mol;
    const int seg = I.seg[qc], koff = I.off[pck];
    for (int k0 = u.kfirst; k0 < u.kend; k0 += seg) {
        const int k1 = min(u.kend, k0 + seg);
        // segments start at multiples of QMAX_BLOCK from kfirst
        double qm = qrun[koff + k1 - 1];
        for (int k = k0 + QMAX_BLOCK - 1; k < k1 - 1; k += QMAX_BLOCK) qm = fmax(qm, qrun[koff + k]);
        const double qb = q * qm;
        float qf = (float)qb;
        if ((double)qf < qb) qf = __int_as_float(__float_as_int(qf) + 1);   // rounded up (qb > 0 here)
        const UnitBound ub{qf, mol};
        const long long kc = ket_prims(I, pck, k0, k1);
        if (u.nfull) {
            const int at = atomicAdd(&hist[qc * UNIT_BUCKETS + unit_bucket(PSLICE * kc)], u.nfull);
            for (int s = 0; s < u.nfull; ++s) {
                units[at + s] = make_int4(u.P, s * PSLICE | ((s + 1) * PSLICE << 16), k0, k1);
                bounds[at + s] = ub;
            }
        }
        if (u.rest) {
            const int at = atomicAdd(&hist[qc * UNIT_BUCKETS + unit_bucket(u.rest * kc)], 1);
            units[at] = make_int4(u.P, u.nfull * PSLICE | (u.npp << 16), k0, k1);
            bounds[at] = ub;
        }
    }
}

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

// All steps up to the units' cursors for at most PAIR_ONE pairs.  (U.pairs is
// `pairs`: no __restrict__, what one step writes the next one reads.)
__global__ void __launch_bounds__(SCAN_BLOCK) pair_sort_small_kernel(PairInput I, PairWork W, UnitInput U,
                                                                     ShellPair* pairs, int units)
{
    constexpr int HIST = NQCLASS * UNIT_BUCKETS;
    __shared__ unsigned long long qm;
    __shared__ int part[SCAN_BLOCK / 64], hist[HIST];
    const int n = I.off[NPAIRCLASS], tid = threadIdx.x, grp = tid / GL, li = tid & (GL - 1);
    if (tid == 0) qm = 0;
    for (int i = tid; i < HIST; i += SCAN_BLOCK) hist[i] = 0;
    if (tid < PAIR_REPORT) W.report[tid] = 0;
    __syncthreads();
    double m = 0.0;
    for (int e = grp; e < n; e += SCAN_BLOCK / GL) m = fmax(m, pair_bound(I, e, li));
    add_bound(m, &qm);
    __syncthreads();
    const double qmax = __longlong_as_double((long long)qm);
    for (int e = grp; e < n; e += SCAN_BLOCK / GL) pair_count(I, W, qmax, e, li);
    __syncthreads();
    if (tid < n) pair_rank(I, W, pairs, tid);
    __syncthreads();
    int all;
    const int p0 = block_scan(tid < n ? pairs[tid].npp : 0, part, &all);
    int* sums = W.scan + n;
    if (tid < n) W.scan[tid] = p0;
    if (tid == 0) sums[0] = 0;
    __syncthreads();
    if (tid < n) pair_place(I, W.scan, sums, pairs, reinterpret_cast<PairStats*>(W.report), tid);
    if (!units) return;
    __syncthreads();
    if (tid < n) unit_qrun(U, W.q, tid);
    for (int qc = tid >> 6; qc < NQCLASS; qc += SCAN_BLOCK / 64) {   // a wavefront per class
        int pcb, pck;
        qclass_pairs(qc, &pcb, &pck);
        if (U.off[pck + 1] == U.off[pck]) continue;
        for (int e = tid & 63; e < U.off[pcb + 1] - U.off[pcb]; e += 64)
            unit_count(U, qc, pcb, pck, e, hist + qc * UNIT_BUCKETS);
    }
    __syncthreads();
    unit_scan(hist, W.hist, W.report + PAIR_STATS, part);
}

// The same steps over many workgroups.
__global__ void __launch_bounds__(256) pair_bound_kernel(PairInput I, unsigned long long* qmax)
{
    const int e = (blockIdx.x * blockDim.x + threadIdx.x) / GL;
    add_bound(e < I.off[NPAIRCLASS] ? pair_bound(I, e, threadIdx.x & (GL - 1)) : 0.0, qmax);
}

__global__ void __launch_bounds__(256) pair_count_kernel(PairInput I, PairWork W)
{
    const int e = (blockIdx.x * blockDim.x + threadIdx.x) / GL;
    if (e >= I.off[NPAIRCLASS]) return;
    pair_count(I, W, __longlong_as_double((long long)*W.qmax), e, threadIdx.x & (GL - 1));
}

__global__ void __launch_bounds__(256) pair_rank_kernel(PairInput I, PairWork W, ShellPair* __restrict__ pairs)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < I.off[NPAIRCLASS]) pair_rank(I, W, pairs, e);
}

// Exclusive prefix sums of the pairs' primitive counts: inside blocks, then of
// the block sums.
__global__ void __launch_bounds__(SCAN_BLOCK) pair_scan_kernel(int n, const ShellPair* __restrict__ pairs, int* scan,
                                                               int* sums)
{
    __shared__ int part[SCAN_BLOCK / 64];
    const int i = blockIdx.x * SCAN_BLOCK + threadIdx.x;
    int all;
    const int x = block_scan(i < n ? pairs[i].npp : 0, part, &all);
    if (i < n) scan[i] = x;
    if (threadIdx.x == 0) sums[blockIdx.x] = all;
}

__global__ void __launch_bounds__(SCAN_BLOCK) pair_scan_sums_kernel(int n, int* sums)
{
    __shared__ int part[SCAN_BLOCK / 64];
    int base = 0;
    for (int i0 = 0; i0 < n; i0 += SCAN_BLOCK) {
        const int i = i0 + threadIdx.x;
        int all;
        const int x = block_scan(i < n ? sums[i] : 0, part, &all);
        if (i < n) sums[i] = base + x;
        base += all;
    }
}

__global__ void __launch_bounds__(256) pair_place_kernel(PairInput I, const int* __restrict__ scan,
                                                         const int* __restrict__ sums, ShellPair* __restrict__ pairs,
                                                         PairStats* stats)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < I.off[NPAIRCLASS]) pair_place(I, scan, sums, pairs, stats, i);
}

__global__ void __launch_bounds__(256) unit_qrun_kernel(UnitInput I, double* __restrict__ qrun)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < I.off[NPAIRCLASS]) unit_qrun(I, qrun, i);
}

__global__ void __launch_bounds__(256) unit_count_kernel(UnitInput I, int* __restrict__ hist)
{
    __shared__ int h[UNIT_BUCKETS];
    int pcb, pck;
    const int qc = blockIdx.y;
    qclass_pairs(qc, &pcb, &pck);
    const int nb = I.off[pcb + 1] - I.off[pcb];
    if (I.off[pck + 1] == I.off[pck] || (int)(blockIdx.x * blockDim.x) >= nb) return;   // uniform
    for (int i = threadIdx.x; i < UNIT_BUCKETS; i += blockDim.x) h[i] = 0;
    __syncthreads();
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < nb) unit_count(I, qc, pcb, pck, e, h);
    __syncthreads();
    for (int i = threadIdx.x; i < UNIT_BUCKETS; i += blockDim.x)
        if (h[i]) atomicAdd(&hist[qc * UNIT_BUCKETS + i], h[i]);
}

__global__ void __launch_bounds__(SCAN_BLOCK) unit_scan_kernel(int* hist, int* counts)
{
    __shared__ int part[SCAN_BLOCK / 64];
    unit_scan(hist, hist, counts, part);
}

// The tables themselves: fill_blocks workgroups for the primitive pairs, then
// unit_blocks per quartet class for the units; the report to the host by the
// way, which saves it a copy of its own.
__global__ void __launch_bounds__(256) pair_tables_kernel(PairInput I, PairWork W, const ShellPair* __restrict__ pairs,
                                                          PrimPair* __restrict__ pp, double* __restrict__ ppa,
                                                          KetTables K, UnitInput U, UnitTables T, int fill_blocks,
                                                          int unit_blocks, int* __restrict__ host_report)
{
    int b = blockIdx.x;
    if (b < fill_blocks) {
        const int e = (b * (int)blockDim.x + (int)threadIdx.x) / GL;
        if (b == 0 && threadIdx.x < PAIR_REPORT) host_report[threadIdx.x] = W.report[threadIdx.x];
        if (e < I.off[NPAIRCLASS]) pair_fill(I, W, pairs, pp, ppa, K, e, threadIdx.x & (GL - 1));
        return;
    }
    b -= fill_blocks;
    int pcb, pck;
    const int qc = b / unit_blocks;
    qclass_pairs(qc, &pcb, &pck);
    const int e = (b - qc * unit_blocks) * (int)blockDim.x + (int)threadIdx.x;
    if (e >= U.off[pcb + 1] - U.off[pcb] || U.off[pck + 1] == U.off[pck]) return;
    unit_scatter(U, W.hist, W.q, T.units, T.bounds, qc, pcb, pck, e);
}

int largest_class(const UnitInput& I)
{
    int m = 1;
    for (int pc = 0; pc < NPAIRCLASS; ++pc) m = m > I.off[pc + 1] - I.off[pc] ? m : I.off[pc + 1] - I.off[pc];
    return m;
}

}  // namespace

hipError_t launch_pair_sort(const PairInput& I, const PairWork& W, const UnitInput& U, bool units, ShellPair* pairs,
                            hipStream_t st)
{
    const int n = I.off[NPAIRCLASS];
    if (n <= 0) return hipSuccess;
    if (n <= PAIR_ONE) {
        hipLaunchKernelGGL(pair_sort_small_kernel, dim3(1), dim3(SCAN_BLOCK), 0, st, I, W, U, pairs, units ? 1 : 0);
        return hipGetLastError();
    }
    const dim3 g((n + 255) / 256), gl((unsigned)(((int64_t)n * GL + 255) / 256)), b(256);
    const int nsum = (n + SCAN_BLOCK - 1) / SCAN_BLOCK;
    int* sums = W.scan + n;
    const hipError_t e = launch_fill_int(W.nclear, W.report, 0, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(pair_bound_kernel, gl, b, 0, st, I, W.qmax);
    hipLaunchKernelGGL(pair_count_kernel, gl, b, 0, st, I, W);
    hipLaunchKernelGGL(pair_rank_kernel, g, b, 0, st, I, W, pairs);
    hipLaunchKernelGGL(pair_scan_kernel, dim3(nsum), dim3(SCAN_BLOCK), 0, st, n, pairs, W.scan, sums);
    hipLaunchKernelGGL(pair_scan_sums_kernel, dim3(1), dim3(SCAN_BLOCK), 0, st, nsum, sums);
    hipLaunchKernelGGL(pair_place_kernel, g, b, 0, st, I, W.scan, sums, pairs, reinterpret_cast<PairStats*>(W.report));
    if (units) {   // the factors are in the pairs now, and W.q is free
        hipLaunchKernelGGL(unit_qrun_kernel, g, b, 0, st, U, W.q);
        hipLaunchKernelGGL(unit_count_kernel, dim3((largest_class(U) + 255) / 256, NQCLASS), b, 0, st, U, W.hist);
        hipLaunchKernelGGL(unit_scan_kernel, dim3(1), dim3(SCAN_BLOCK), 0, st, W.hist, W.report + PAIR_STATS);
    }
    return hipGetLastError();
}

hipError_t launch_pair_tables(const PairInput& I, const PairWork& W, const ShellPair* pairs, PrimPair* pp, double* ppa,
                              const KetTables& K, const UnitInput& U, const UnitTables& T, int* host_report,
                              hipStream_t st)
{
    const int n = I.off[NPAIRCLASS];
    if (n <= 0) return hipSuccess;
    const int fill = (int)(((int64_t)n * GL + 255) / 256), per = (largest_class(U) + 255) / 256;
    hipLaunchKernelGGL(pair_tables_kernel, dim3((unsigned)(fill + (T.units ? per * NQCLASS : 0))), dim3(256), 0, st, I, W,
                       pairs, pp, ppa, K, U, T, fill, per, host_report);
    return hipGetLastError();
}

namespace {
// One thread per unit, a row of blocks per class.  A row kernel that drew and
// dropped the dead units itself spent 0.3 of 0.4 ms on them late in a batch's
// SCF, when most molecules have converged; this pass takes 6 us (65 to 100 on average
// where it shares the GPU with the other groups of a large batch).
__global__ void __launch_bounds__(256) unit_live_kernel(UnitLive I)
{
    const int qc = blockIdx.y;
    const int64_t n = I.off[qc + 1] - I.off[qc];
    const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if ((int64_t)blockIdx.x * blockDim.x >= n) return;
    __shared__ int base[4], total;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    bool keep = false;
    if (u < n) {
        const UnitBound b = I.bound[I.off[qc] + u];
        keep = !((double)b.q * 4.0 * I.mol_dmax[b.mol] < 0.999999 * I.tol);
    }
    const unsigned long long m = __ballot(keep);
    if (lane == 0) base[wv] = __popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        const int c = base[0] + base[1] + base[2] + base[3];
        total = c ? atomicAdd(&I.nlive[qc], c) : 0;
    }
    __syncthreads();
    int pos = total;
    for (int w = 0; w < wv; ++w) pos += base[w];
    if (keep) I.live[I.off[qc] + pos + __popcll(m & ((1ull << lane) - 1ull))] = (int)u;
}
}  // namespace

hipError_t launch_unit_live(const UnitLive& I, hipStream_t st)
{
    int64_t most = 0;
    for (int qc = 0; qc < NQCLASS; ++qc) most = I.off[qc + 1] - I.off[qc] > most ? I.off[qc + 1] - I.off[qc] : most;
    if (most == 0) return hipSuccess;
    hipLaunchKernelGGL(unit_live_kernel, dim3((unsigned)((most + 255) / 256), NQCLASS), dim3(256), 0, st, I);
    return hipGetLastError();
}

}  // namespace mmd
