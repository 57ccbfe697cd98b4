// Shell-pair and primitive-pair tables and the Fock build's work units, on
// the device.  A group of 128 clusters of six waters in 6-31G has 190 thousand
// shell pairs, 1.1 million primitive pairs and 150 thousand work units; on one
// host thread they took 102 ms, the iterations of the group 74 ms.
//
// Per pair (one thread each): the largest Schwarz-type bound of its primitive
// pairs, the number that survive the primitive screen, its factor
// q = max sqrt((ab|ab)).  A pair's place in its class is the number of pairs of
// its molecule that sort before it (molecules have at most a few thousand
// pairs of a class, and the lanes of a wavefront read the same ones), its
// place in the primitive table a prefix sum.  Units are counted into cost
// buckets and scattered through the buckets' cursors.
#include <hip/hip_runtime.h>
#include "mmd_pairs.h"

namespace mmd {

namespace {

constexpr double PRIM_DROP = 1e-20;
constexpr int SCAN_BLOCK = 1024;

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

__global__ void __launch_bounds__(256) pair_bound_kernel(PairInput I, unsigned long long* qmax)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    double m = 0.0;
    if (e < I.off[NPAIRCLASS]) {
        const int2 pr = I.list[e];
        const OneeShell a = I.shells[pr.x], b = I.shells[pr.y];
        const double AB2 = dist2(a, b);
        for (int i = 0; i < a.np; ++i)
            for (int j = 0; j < b.np; ++j) {
                const double ea = I.exps[a.p0 + i], eb = I.exps[b.p0 + j], p = ea + eb;
                m = fmax(m, prim_bound(p, I.wts[a.p0 + i] * I.wts[b.p0 + j] * exp(-ea * eb / p * AB2), AB2, a.l + b.l));
            }
    }
    for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
    // positive doubles order like their bits
    if ((threadIdx.x & 63) == 0 && m > 0.0) atomicMax(qmax, (unsigned long long)__double_as_longlong(m));
}

// A primitive pair whose bound, times the largest bound of any pair, is below
// PRIM_DROP contributes less than that to every primitive quartet and is
// left out of the table.  Decided here once, as a bit of the pair's keep words:
// the count sizes the pair's range of the table and the fill writes it, and a
// pair at the threshold that each decided for itself, in code that the
// compiler contracts in its own way, could be one record more than the range.
__global__ void __launch_bounds__(256) pair_count_kernel(PairInput I, PairWork W)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    const int npairs = I.off[NPAIRCLASS];
    if (e >= npairs) return;
    const double qmax = __longlong_as_double((long long)*W.qmax);
    const int2 pr = I.list[e];
    const OneeShell a = I.shells[pr.x], b = I.shells[pr.y];
    const double AB2 = dist2(a, b);
    int n = 0, bit = 0;
    unsigned long long word = 0, *keep = W.keep + e;
    for (int i = 0; i < a.np; ++i)
        for (int j = 0; j < b.np; ++j) {
            const double ea = I.exps[a.p0 + i], eb = I.exps[b.p0 + j], p = ea + eb;
            const double K = I.wts[a.p0 + i] * I.wts[b.p0 + j] * exp(-ea * eb / p * AB2);
            if (!(prim_bound(p, K, AB2, a.l + b.l) * qmax < PRIM_DROP)) {
                word |= 1ull << bit;
                ++n;
            }
            if (++bit == 64) {
                *keep = word;
                keep += npairs;
                word = 0;
                bit = 0;
            }
        }
    if (bit) *keep = word;
    double q = 1.0;
    if (I.diag) {
        q = 0.0;
        for (int x = 0; x < ncart(a.l); ++x)
            for (int y = 0; y < ncart(b.l); ++y) {
                const double v = I.diag[(size_t)(a.bf0 + x) * I.N + b.bf0 + y];
                q = fmax(q, v > 0.0 ? sqrt(v) : 0.0);
            }
    }
    W.count[e] = n;
    W.q[e] = n == 0 ? 0.0 : q;   // no primitive pair survives: never screened in
}

// Place of every pair among those of its molecule and class, and its record.
__global__ void __launch_bounds__(256) pair_rank_kernel(PairInput I, PairWork W, ShellPair* __restrict__ pairs)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= I.off[NPAIRCLASS]) return;
    const int c = class_of_entry(I.off, e);
    const int2 pr = I.list[e];
    const OneeShell a = I.shells[pr.x], b = I.shells[pr.y];
    const int2 seg = I.ranges[(size_t)c * I.nmol + a.mol];
    const int s0 = I.off[c] + seg.x, s1 = I.off[c] + seg.y;
    const int n = W.count[e];
    const double q = W.q[e];
    int rank = 0;
    for (int j = s0; j < s1; ++j) {
        const int nj = W.count[j];
        const double qj = W.q[j];
        rank += (nj > n || (nj == n && (qj > q || (qj == q && j < e)))) ? 1 : 0;
    }
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
    sp.pad = 0;
    sp.q = q;
    pairs[s0 + rank] = sp;
    W.entry[s0 + rank] = e;
}

// Exclusive prefix sums of the pairs' primitive counts: inside blocks, then of
// the block sums.
__global__ void __launch_bounds__(SCAN_BLOCK) pair_scan_kernel(int n, const ShellPair* __restrict__ pairs, int* scan,
                                                               int* sums)
{
    __shared__ int part[SCAN_BLOCK / 64];
    const int i = blockIdx.x * SCAN_BLOCK + threadIdx.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int v = i < n ? pairs[i].npp : 0;
    int x = v;
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) part[wv] = x;
    __syncthreads();
    for (int k = 0; k < wv; ++k) x += part[k];
    if (i < n) scan[i] = x - v;
    if (threadIdx.x == SCAN_BLOCK - 1) sums[blockIdx.x] = x;
}

__global__ void __launch_bounds__(SCAN_BLOCK) pair_scan_sums_kernel(int n, int* sums)
{
    __shared__ int part[SCAN_BLOCK / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int base = 0;
    for (int i0 = 0; i0 < n; i0 += SCAN_BLOCK) {
        const int i = i0 + threadIdx.x;
        const int v = i < n ? sums[i] : 0;
        int x = v;
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(x, off);
            if (lane >= off) x += y;
        }
        if (lane == 63) part[wv] = x;
        __syncthreads();
        int before = base, all = 0;
        for (int k = 0; k < SCAN_BLOCK / 64; ++k) {
            if (k < wv) before += part[k];
            all += part[k];
        }
        if (i < n) sums[i] = before + x - v;
        base += all;
        __syncthreads();
    }
}

__device__ int pair_start(const int* scan, const int* sums, int i) { return scan[i] + sums[i / SCAN_BLOCK]; }

// Table ranges of the sorted pairs, and per class the largest and total count.
__global__ void __launch_bounds__(256) pair_place_kernel(PairInput I, const int* __restrict__ scan,
                                                         const int* __restrict__ sums, ShellPair* __restrict__ pairs,
                                                         PairStats* stats)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= I.off[NPAIRCLASS]) return;
    const int c = class_of_entry(I.off, i);
    const int p0 = pair_start(scan, sums, i);
    pairs[i].pp0 = p0;
    pairs[i].pad = p0 - pair_start(scan, sums, I.off[c]);
    const int n = pairs[i].npp;
    // the first pair of a molecule holds its largest count
    if (i == I.off[c] + I.ranges[(size_t)c * I.nmol + pairs[i].mol].x) atomicMax(&stats->maxpp[c], n);
    if (i == I.off[c + 1] - 1) stats->total[c] = pairs[i].pad + n;
}

__global__ void __launch_bounds__(256) pair_fill_kernel(PairInput I, PairWork W, const ShellPair* __restrict__ pairs,
                                                        PrimPair* __restrict__ pp, double* __restrict__ ppa,
                                                        KetTables K)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    const int npairs = I.off[NPAIRCLASS];
    if (e >= npairs) return;
    const ShellPair sp = pairs[e];
    const OneeShell a = I.shells[sp.sa], b = I.shells[sp.sb];
    const double AB2 = dist2(a, b);
    int o = sp.pp0, bit = 0;
    const unsigned long long* keep = W.keep + W.entry[e];
    unsigned long long word = 0;
    K.scr[e] = KetScreen{sp.q, sp.sa, sp.sb};
    K.ref[e] = KetRef{sp.bfa, sp.bfb, sp.pp0, sp.npp};
    for (int i = 0; i < a.np; ++i)
        for (int j = 0; j < b.np; ++j) {
            if (bit == 0) {
                word = *keep;
                keep += npairs;
            }
            const bool kept = word >> bit & 1;
            bit = (bit + 1) & 63;
            if (!kept) continue;
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
            for (int k = 0; k < KET_FIELDS; ++k) K.pp[k * K.stride + o] = f[k];
            ++o;
        }
}

// ---------------------------------------------------------------------------
// Work units
// ---------------------------------------------------------------------------

// Running maximum of the pair factors over the QMAX_BLOCK pairs that a pair
// lies in, counted from its molecule's first pair of the class.
__global__ void __launch_bounds__(256) unit_qrun_kernel(UnitInput I, double* __restrict__ qrun)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= I.off[NPAIRCLASS]) return;
    const int c = class_of_entry(I.off, i);
    const int first = I.off[c] + I.ranges[(size_t)c * I.nmol + I.pairs[i].mol].x;
    double m = 0.0;
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
    if (e < nb) {
        const UnitRange u = unit_range(I, pcb, pck, e);
        for (int k0 = u.kfirst; k0 < u.kend; k0 += I.seg[qc]) {
            const long long kc = ket_prims(I, pck, k0, min(u.kend, k0 + I.seg[qc]));
            if (u.nfull) atomicAdd(&h[unit_bucket(PSLICE * kc)], u.nfull);
            if (u.rest) atomicAdd(&h[unit_bucket(u.rest * kc)], 1);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < UNIT_BUCKETS; i += blockDim.x)
        if (h[i]) atomicAdd(&hist[qc * UNIT_BUCKETS + i], h[i]);
}

// Bucket counts to cursors: positions in the table of all classes, and the
// classes' totals.
__global__ void unit_scan_kernel(int* hist, int* counts)
{
    if (threadIdx.x != 0) return;
    int pos = 0;
    for (int qc = 0; qc < NQCLASS; ++qc) {
        const int start = pos;
        for (int b = 0; b < UNIT_BUCKETS; ++b) {
            const int n = hist[qc * UNIT_BUCKETS + b];
            hist[qc * UNIT_BUCKETS + b] = pos;
            pos += n;
        }
        counts[qc] = pos - start;
    }
}

__global__ void __launch_bounds__(256) unit_scatter_kernel(UnitInput I, int* __restrict__ hist,
                                                           const double* __restrict__ qrun, int4* __restrict__ units,
                                                           UnitBound* __restrict__ bounds)
{
    int pcb, pck;
    const int qc = blockIdx.y;
    qclass_pairs(qc, &pcb, &pck);
    const int nb = I.off[pcb + 1] - I.off[pcb];
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nb || I.off[pck + 1] == I.off[pck]) return;
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

}  // namespace

hipError_t launch_pair_sort(const PairInput& I, const PairWork& W, ShellPair* pairs, PairStats* stats, hipStream_t st)
{
    const int n = I.off[NPAIRCLASS];
    if (n <= 0) return hipSuccess;
    const dim3 g((n + 255) / 256), b(256);
    const int nsum = (n + SCAN_BLOCK - 1) / SCAN_BLOCK;
    int* sums = W.scan + n;
    hipError_t e = launch_fill_int(2, reinterpret_cast<int*>(W.qmax), 0, st);
    if (e == hipSuccess) e = launch_fill_int((int)(sizeof(PairStats) / sizeof(int)), reinterpret_cast<int*>(stats), 0, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(pair_bound_kernel, g, b, 0, st, I, W.qmax);
    hipLaunchKernelGGL(pair_count_kernel, g, b, 0, st, I, W);
    hipLaunchKernelGGL(pair_rank_kernel, g, b, 0, st, I, W, pairs);
    hipLaunchKernelGGL(pair_scan_kernel, dim3(nsum), dim3(SCAN_BLOCK), 0, st, n, pairs, W.scan, sums);
    hipLaunchKernelGGL(pair_scan_sums_kernel, dim3(1), dim3(SCAN_BLOCK), 0, st, nsum, sums);
    hipLaunchKernelGGL(pair_place_kernel, g, b, 0, st, I, W.scan, sums, pairs, stats);
    return hipGetLastError();
}

hipError_t launch_pair_fill(const PairInput& I, const PairWork& W, const ShellPair* pairs, PrimPair* pp, double* ppa,
                            const KetTables& K, hipStream_t st)
{
    const int n = I.off[NPAIRCLASS];
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(pair_fill_kernel, dim3((n + 255) / 256), dim3(256), 0, st, I, W, pairs, pp, ppa, K);
    return hipGetLastError();
}

namespace {
int largest_class(const UnitInput& I)
{
    int m = 1;
    for (int pc = 0; pc < NPAIRCLASS; ++pc) m = m > I.off[pc + 1] - I.off[pc] ? m : I.off[pc + 1] - I.off[pc];
    return m;
}
}  // namespace

hipError_t launch_unit_count(const UnitInput& I, int* hist, int* counts, double* qrun, hipStream_t st)
{
    const int n = I.off[NPAIRCLASS];
    if (n <= 0) return hipSuccess;
    const hipError_t e = launch_fill_int(NQCLASS * UNIT_BUCKETS, hist, 0, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(unit_qrun_kernel, dim3((n + 255) / 256), dim3(256), 0, st, I, qrun);
    hipLaunchKernelGGL(unit_count_kernel, dim3((largest_class(I) + 255) / 256, NQCLASS), dim3(256), 0, st, I, hist);
    hipLaunchKernelGGL(unit_scan_kernel, dim3(1), dim3(64), 0, st, hist, counts);
    return hipGetLastError();
}

hipError_t launch_unit_scatter(const UnitInput& I, int* hist, const double* qrun, int4* units, UnitBound* bounds,
                               hipStream_t st)
{
    if (I.off[NPAIRCLASS] <= 0) return hipSuccess;
    hipLaunchKernelGGL(unit_scatter_kernel, dim3((largest_class(I) + 255) / 256, NQCLASS), dim3(256), 0, st, I, hist,
                       qrun, units, bounds);
    return hipGetLastError();
}

namespace {
// One thread per unit, a row of blocks per class.  A row kernel that drew and
// dropped the dead units itself spent 0.3 of 0.4 ms on them late in a batch's
// SCF, when most molecules have converged; this pass takes 6 us.
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
