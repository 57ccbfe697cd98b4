#pragma once
// Contracted integral blocks of the unscreened or raw entry points, by
// shell-quartet class: the stored tensor (doERIs, cython/twoe.pyx:9-31) and
// formPT's unsymmetrised build (cython/fock.pyx:10-87).
//
// A group of 4 to 16 lanes takes one shell quartet and one chunk of its bra
// components: the lanes split the quartet's bra and ket primitive pairs as a
// gb x gk grid (quartet_compute, mmd_eri_core.h), sum their blocks across the
// group, and share the component quartets of the epilogue through LDS.  One
// lane per quartet left the lanes of a wavefront waiting for a core quartet of
// up to 1296 primitive quartets while the others had one; a whole wavefront
// per quartet would idle on the uncontracted ones.  Bound by FP64 VALU issue
// and latency of the primitive loops; the tensor's stores are scattered 8-byte
// ones that the L2s merge.
// (H2O)2 6-31G, formPT with a complex density: 22.5 ms with one lane per
// canonical function quartet, tables in scratch, and one pass per part; 0.205
// ms here (six classes of 24 to 58 us side by side).  (H2O)4 6-31G, the
// tensor's kernels: 2.0 ms one after the other with one lane per shell
// quartet, about 0.3 ms here.
#include "mmd_eri_core.h"

namespace mmd {

// Adds one function quartet's integral (pq|rs) (component scales applied) to
// formPT's unsymmetrised G as the canonical quartet i >= j, k >= l, ij >= kl:
// its Schwarz x |dP| test, degeneracy and the six updates
// (cython/fock.pyx:38-85); the imaginary part of dP, when given, goes to the
// second matrix of the same replica.
__device__ __forceinline__ void raw_digest(const ClassArgs& A, const BlockArgs& B, double* G, double eri, int p, int q,
                                           int r, int s)
{
    const size_t n = (size_t)A.N;
    size_t i = p > q ? p : q, j = p > q ? q : p, k = r > s ? r : s, l = r > s ? s : r;
    if (i * (i + 1) / 2 + j < k * (k + 1) / 2 + l) {
        size_t t = i; i = k; k = t;
        t = j; j = l; l = t;
    }
    const double* aD = A.absD;
    const double bound = A.sqS[i * n + j] * A.sqS[k * n + l]
        * fmax(fmax(fmax(4.0 * aD[i * n + j], 4.0 * aD[k * n + l]), fmax(aD[i * n + k], aD[i * n + l])),
               fmax(aD[j * n + k], aD[j * n + l]));
    if (bound < A.tol) return;
    eri *= (i == j ? 1.0 : 2.0) * (k == l ? 1.0 : 2.0) * (i == k && j == l ? 1.0 : 2.0);
    for (int part = 0; part < (B.Dim ? 2 : 1); ++part) {
        const double* D = part ? B.Dim : A.D;
        double* g = G + part * n * n;
        atomicAdd(&g[i * n + j], D[k * n + l] * eri);
        atomicAdd(&g[k * n + l], D[i * n + j] * eri);
        atomicAdd(&g[i * n + k], -0.25 * D[j * n + l] * eri);
        atomicAdd(&g[j * n + l], -0.25 * D[i * n + k] * eri);
        atomicAdd(&g[i * n + l], -0.25 * D[j * n + k] * eri);
        atomicAdd(&g[k * n + j], -0.25 * D[i * n + l] * eri);
    }
}

// Stores (pq|rs) at its eight index permutations (cython/twoe.pyx:23-30).
__device__ __forceinline__ void tensor_store(double* __restrict__ out, size_t n, double v, size_t p, size_t q,
                                             size_t r, size_t s)
{
    const size_t pq = p * n + q, qp = q * n + p, rs = r * n + s, sr = s * n + r, nn = n * n;
    out[pq * nn + rs] = v;
    out[qp * nn + rs] = v;
    out[pq * nn + sr] = v;
    out[qp * nn + sr] = v;
    out[rs * nn + pq] = v;
    out[sr * nn + pq] = v;
    out[rs * nn + qp] = v;
    out[sr * nn + qp] = v;
}

// Component quartet (a b | c d) of a unique shell quartet: exactly one of the
// components that are permutations of each other (functions of one shell on
// both sides of a pair, or one pair on both sides) is produced.
__device__ __forceinline__ bool unique_component(const ShellPair& bra, const ShellPair& ket, bool same_pair, int a,
                                                 int b, int c, int d)
{
    if ((bra.same && a < b) || (ket.same && c < d)) return false;
    return !same_pair || a > c || (a == c && b >= d);
}

// The q-th shell quartet of a class: bra pair P, ket pair Q (global indices).
__device__ __forceinline__ void block_quartet(const BlockArgs& B, int64_t q, int& P, int& Q)
{
    if (B.tri) {
        int64_t r = (int64_t)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
        while (r * (r + 1) / 2 > q) --r;
        while ((r + 1) * (r + 2) / 2 <= q) ++r;
        P = B.boff + (int)r;
        Q = B.koff + (int)(q - r * (r + 1) / 2);
    } else {
        const int64_t r = q / B.nk;
        P = B.boff + (int)r;
        Q = B.koff + (int)(q - r * B.nk);
    }
}

// Shell-level form of raw_digest's test for the pairs P and Q: qraw is the
// largest root of a pair's Schwarz values and Dsh the largest |dP| of a shell
// block, infinity where a value is not a number (the test above keeps what
// does not compare as small), so a quartet that fails it has no component that
// passes.  A pair without primitive pairs has integrals that are zero to 1e-20,
// and takes part only where |dP| is not finite.
__device__ __forceinline__ bool raw_keeps(const ClassArgs& A, const BlockArgs& B, int P, int Q, const ShellPair& bra,
                                          const ShellPair& ket)
{
    const size_t ns = (size_t)B.nshell;
    const double* D = B.Dsh;
    const double dm = fmax(fmax(fmax(4.0 * D[bra.sa * ns + bra.sb], 4.0 * D[ket.sa * ns + ket.sb]),
                                fmax(D[bra.sa * ns + ket.sa], D[bra.sa * ns + ket.sb])),
                           fmax(D[bra.sb * ns + ket.sa], D[bra.sb * ns + ket.sb]));
    if ((bra.npp == 0 || ket.npp == 0) && dm < HUGE_VAL) return false;
    return !(B.qraw[P] * B.qraw[Q] * dm < A.tol);
}

template <int LA, int LB, int LC, int LD>
__global__ void __launch_bounds__(256) eri_block_kernel(ClassArgs A, BlockArgs B)
{
    using S = ClassShape<LA, LB, LC, LD>;
    constexpr int NV = S::CH * S::NCD;
    __shared__ double boys[BOYS_TAYLOR * BOYS_NT];
    __shared__ double blk[4][BLOCK_GROUPS * NV];
    boys_stage_lds<S::L, double>(boys, A.boys);
    __syncthreads();
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int gb = 1 << B.lgb, gk = 1 << B.lgk, lg = B.lgb + B.lgk, G = 1 << lg, NG = 64 >> lg;
    const int grp = lane >> lg, li = lane & (G - 1), lib = li & (gb - 1), lik = li >> B.lgb;
    const int64_t nq = B.tri ? (int64_t)B.nb * (B.nb + 1) / 2 : (int64_t)B.nb * B.nk;
    const int64_t items = ((nq + NG - 1) / NG) * S::NCHUNK;
    double* mine = blk[wv] + grp * NV;
    double* Grep = A.G + (B.raw ? (size_t)(blockIdx.x % B.nrep) * 2 * A.N * A.N : 0);
    for (int64_t w = (int64_t)blockIdx.x * 4 + wv; w < items; w += (int64_t)gridDim.x * 4) {   // uniform
        const int chunk = (int)(w % S::NCHUNK);
        const int64_t q = (w / S::NCHUNK) * NG + grp;
        int P = B.boff, Q = B.koff;
        bool on = q < nq;
        if (on) block_quartet(B, q, P, Q);
        const ShellPair bra = A.pairs[P], ket = A.pairs[Q];
        if (B.raw) on = on && raw_keeps(A, B, P, Q, bra, ket);
        if (!__any(on)) continue;
        const int nb_ = on ? bra.npp : 0, nk_ = on ? ket.npp : 0;
        const int ip0 = nb_ * lib / gb, ip1 = nb_ * (lib + 1) / gb;
        const int jq0 = nk_ * lik / gk, jq1 = nk_ * (lik + 1) / gk;
        static_switch<0, S::NCHUNK>(chunk, [&](auto ic) {
            constexpr int A0 = decltype(ic)::value * S::CH, A1 = A0 + S::CH;
            double acc[NV];
            quartet_compute<LA, LB, LC, LD, A0, A1, double>(KetRecords{A.pp}, boys, B.table + (size_t)bra.class_pp0 * S::BPS,
                                                            ip0, ip1, ket.pp0 + jq0, ket.pp0 + jq1, acc);
            for (int off = 1; off < G; off <<= 1)
                sfor<NV>([&](auto k) { acc[decltype(k)::value] += __shfl_xor(acc[decltype(k)::value], off); });
            sfor<NV>([&](auto k) {
                if ((decltype(k)::value & (G - 1)) == li) mine[decltype(k)::value] = acc[decltype(k)::value];
            });
        });
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (on)
            for (int k = li; k < NV; k += G) {
                const int ab = chunk * S::CH + k / S::NCD, cd = k % S::NCD;
                const int a = ab / S::NB, b = ab % S::NB, c = cd / S::ND, d = cd % S::ND;
                if (!unique_component(bra, ket, P == Q, a, b, c, d)) continue;
                const int i = bra.bfa + a, j = bra.bfb + b, kk = ket.bfa + c, l = ket.bfb + d;
                const double v = mine[k] * A.gcomp[i] * A.gcomp[j] * A.gcomp[kk] * A.gcomp[l];
                if (B.raw) raw_digest(A, B, Grep, v, i, j, kk, l);
                else tensor_store(A.G, (size_t)A.N, v, i, j, kk, l);
            }
        __builtin_amdgcn_wave_barrier();   // the block is rewritten by the next quartet
    }
}

}  // namespace mmd
