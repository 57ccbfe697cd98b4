// Device side of the batched RHF driver (mmd_batch_rhf): many molecules
// stepped together, one workgroup per molecule.
//
// The molecules of a batch form one block-diagonal basis: molecule m owns
// basis functions [f0, f0 + n) and the n x n diagonal block of every N x N
// matrix (S, H, X, F, P, P_old, dP, G; N = all functions of the batch).  The
// Fock build (the class kernels) runs once per iteration for the whole
// batch; these kernels do the per-molecule rest of the reference's loop
// (mmd/scf.py:10-80) in the block: the F update, the DIIS extrapolation
// (mmd/scf.py:146-180), FO = X^T F X, the symmetric eigensolver
// (scipy.linalg.eigh at mmd/scf.py:47, here a cyclic Jacobi method), the
// density, the energy (mmd/scf.py:118-121) and the convergence test on
// ||P - P_old||_F.  A molecule that has converged keeps its state and
// contributes dP = 0 to later Fock builds, so it costs the builds no work.
#include <hip/hip_runtime.h>
#include <math.h>
#include "mmd_batch.h"

namespace mmd {

namespace {

constexpr int BT = 256;   // threads per molecule workgroup

__device__ __forceinline__ double* blk(double* M, int N, int f0) { return M + (size_t)f0 * N + f0; }
__device__ __forceinline__ const double* blk(const double* M, int N, int f0) { return M + (size_t)f0 * N + f0; }

// C (n x n, leading dimension ldc) = op(A) op(B), A and B n x n with leading
// dimensions lda, ldb; the workgroup's threads share the output elements.
__device__ void wg_gemm(int n, bool tA, const double* A, int lda, bool tB, const double* B, int ldb, double* C,
                        int ldc)
{
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
        const int i = e / n, j = e - i * n;
        double s = 0.0;
        for (int k = 0; k < n; ++k) {
            const double a = tA ? A[(size_t)k * lda + i] : A[(size_t)i * lda + k];
            const double b = tB ? B[(size_t)j * ldb + k] : B[(size_t)k * ldb + j];
            s = fma(a, b, s);
        }
        C[(size_t)i * ldc + j] = s;
    }
    __syncthreads();
}

// Workgroup sum of v (all threads get the result); red: BT/64 doubles of LDS.
__device__ double wg_sum(double v, double* red)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wv] = v;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
    __syncthreads();
    return s;
}

typedef double dbl4_t __attribute__((ext_vector_type(4)));

constexpr int BTL = 1024;   // threads of the all-LDS molecule workgroups

// Pointers that say which memory they are in: the routines below are called
// from many places and not inlined (a step runs each of its twenty products
// once, and inlined copies spent their time on instruction fetches), and a
// plain pointer argument would make every access a flat one.
typedef __attribute__((address_space(3))) double lds_d;
typedef __attribute__((address_space(1))) double gbl_d;

// Leading dimension of an n x n matrix in LDS: odd, so that a column of
// doubles touches every bank pair once (at n = 52 a column of leading
// dimension 52 falls on 16 of the 64 banks).
__host__ __device__ constexpr int lds_ld(int n) { return n | 1; }

// f(u, i, j, in) for this thread's elements e = tid + 1024 u of an n x n
// matrix, u in [u0, u1) a compile-time range: unrolled, so that the loads of
// all u are in flight before the first is used (a loop that stores each
// element before it loads the next waits for memory up to eight times).  The
// empty asm keeps the compiler from holding every call's indices in registers
// for the whole kernel (200 of them spilled).
template <int u0 = 0, int u1 = 8, class F>
__device__ __forceinline__ void elems(int n, F&& f)
{
    static_assert(BATCH_MAX_NBF * BATCH_MAX_NBF <= 8 * BTL, "eight elements per thread cover a matrix");
    int e = threadIdx.x + u0 * BTL;
    asm volatile("" : "+v"(e));
    int i = e / n, j = e - i * n;
    const int di = BTL / n, dj = BTL - di * n;
#pragma unroll
    for (int u = u0; u < u1; ++u) {
        f(u, i, j, e < n * n);
        e += BTL;
        i += di;
        j += dj;
        if (j >= n) {
            j -= n;
            ++i;
        }
    }
}

// f(i, j) for the same elements in a loop, where nothing is loaded from memory
// (unrolled, the step kernel outgrew the instruction cache).
template <class F>
__device__ __forceinline__ void elems_loop(int n, F&& f)
{
    int i = (int)threadIdx.x / n, j = (int)threadIdx.x - i * n;
    const int di = BTL / n, dj = BTL - di * n;
#pragma unroll 1
    while (i < n) {
        f(i, j);
        i += di;
        j += dj;
        if (j >= n) {
            j -= n;
            ++i;
        }
    }
}

// load the n x n block at M (leading dimension N) into LDS
__device__ __noinline__ void lds_load(int n, const gbl_d* M, int N, lds_d* L)
{
    const int ld = lds_ld(n);
    double v[8];
    elems(n, [&](int u, int i, int j, bool in) {
        if (in) v[u] = M[(size_t)i * N + j];
    });
    elems(n, [&](int u, int i, int j, bool in) {
        if (in) L[i * ld + j] = v[u];
    });
    __syncthreads();
}

// C = op(A) op(B), contracted over the first kn indices, with A, B and C in
// LDS (leading dimension lds_ld(n)) or, where Cg is given, the result in
// global memory (leading dimension ldg) instead; on the matrix cores: each
// wavefront takes 16 x 16 output tiles and runs v_mfma_f64_16x16x4_f64 over k
// in steps of 4.  Operand layout (wave64): A[i][k] in lane i + 16k, B[k][j]
// in lane j + 16k; the accumulator holds D[i][j] in lane j + 16g, element r,
// with i = g + 4r.  Rows and columns past n are read from the last one
// (D[i][j] uses row i and column j only, and those are not stored), so the
// loop has no conditions and its loads run four steps ahead of the products;
// only k past kn is zeroed.
__device__ __noinline__ void lds_gemm(int n, bool tA, const lds_d* A, bool tB, const lds_d* B, lds_d* C, int kn,
                                      gbl_d* Cg, int ldg)
{
    const int ld = lds_ld(n);
    const int nt = (n + 15) >> 4;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nw = (int)(blockDim.x >> 6);
    const int l16 = lane & 15, l4 = lane >> 4;
    for (int tile = wave; tile < nt * nt; tile += nw) {
        const int ti = tile / nt, tj = tile - ti * nt;
        const int i = min(ti * 16 + l16, n - 1), j = min(tj * 16 + l16, n - 1);
        const lds_d* pa = tA ? A + i + l4 * ld : A + i * ld + l4;
        const lds_d* pb = tB ? B + j * ld + l4 : B + j + l4 * ld;
        const int sa = tA ? 4 * ld : 4, sb = tB ? 4 : 4 * ld;
        dbl4_t acc = {0.0, 0.0, 0.0, 0.0};
        int k0 = 0;
        for (; k0 + 16 <= kn; k0 += 16) {
            double a[4], b[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                a[u] = pa[u * sa];
                b[u] = pb[u * sb];
            }
            pa += 4 * sa;
            pb += 4 * sb;
#pragma unroll
            for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[u], acc, 0, 0, 0);
        }
        for (; k0 < kn; k0 += 4) {
            const bool in = k0 + l4 < kn;
            const double a = in ? *pa : 0.0;
            const double b = in ? *pb : 0.0;
            pa += sa;
            pb += sb;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
        }
        const int jc = tj * 16 + l16;
        for (int r = 0; r < 4; ++r) {
            const int ir = ti * 16 + l4 + 4 * r;
            if (ir < n && jc < n) {
                if (Cg) Cg[(size_t)ir * ldg + jc] = acc[r];
                else C[ir * ld + jc] = acc[r];
            }
        }
    }
    __syncthreads();
}
__device__ __forceinline__ void lds_gemm(int n, bool tA, const lds_d* A, bool tB, const lds_d* B, lds_d* C)
{
    lds_gemm(n, tA, A, tB, B, C, n, nullptr, 0);
}

// Symmetric eigendecomposition A = V diag(w) V^T of the n x n matrix in LDS
// (A, leading dimension lda; destroyed) by the cyclic Jacobi method with a
// round-robin ordering: each round applies n/2 disjoint rotations at once.
// V (n x n, leading dimension ldv, global memory) receives the eigenvectors
// as columns and w the eigenvalues, both in ascending order of w (the order
// of LAPACK's drivers).  perm, cs: LDS scratch of n + 1 ints and 2 (n + 1)
// doubles; red: BT/64 doubles.
__device__ void wg_jacobi(int n, double* A, int lda, double* V, int ldv, double* w, int* perm, double* cs,
                          double* red)
{
    const int m = (n + 1) & ~1;   // even: an odd n takes a dummy index n that stays decoupled
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
        const int i = e / n, j = e - i * n;
        V[(size_t)i * ldv + j] = (i == j) ? 1.0 : 0.0;
    }
    double fro = 0.0;
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) fro += A[(e / n) * lda + e % n] * A[(e / n) * lda + e % n];
    fro = wg_sum(fro, red);
    double* c = cs;
    double* s = cs + (m / 2);
    for (int sweep = 0; sweep < 60; ++sweep) {
        double off = 0.0;
        for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
            const int i = e / n, j = e - i * n;
            if (i != j) off += A[i * lda + j] * A[i * lda + j];
        }
        off = wg_sum(off, red);
        if (!(off > 1e-30 * fro) ) break;
        for (int round = 0; round < m - 1; ++round) {
            // round-robin pairs: index 0 fixed, the others rotate
            for (int k = threadIdx.x; k < m / 2; k += blockDim.x) {
                auto slot = [&](int pos) { return pos == 0 ? 0 : 1 + (pos - 1 + round) % (m - 1); };
                int p = slot(k), q = slot(m - 1 - k);
                if (p > q) { const int t = p; p = q; q = t; }
                perm[2 * k] = p;
                perm[2 * k + 1] = q;
                double cc = 1.0, ss = 0.0;
                if (q < n) {
                    const double apq = A[p * lda + q];
                    if (apq != 0.0) {
                        const double app = A[p * lda + p], aqq = A[q * lda + q];
                        const double theta = (aqq - app) / (2.0 * apq);
                        const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
                        cc = 1.0 / sqrt(t * t + 1.0);
                        ss = t * cc;
                    }
                }
                c[k] = cc;
                s[k] = ss;
            }
            __syncthreads();
            // rows: (A_p., A_q.) <- (c A_p. - s A_q., s A_p. + c A_q.)
            for (int e = threadIdx.x; e < (m / 2) * n; e += blockDim.x) {
                const int k = e / n, j = e - k * n;
                const int p = perm[2 * k], q = perm[2 * k + 1];
                if (q >= n || s[k] == 0.0) continue;
                const double ap = A[p * lda + j], aq = A[q * lda + j];
                A[p * lda + j] = c[k] * ap - s[k] * aq;
                A[q * lda + j] = s[k] * ap + c[k] * aq;
            }
            __syncthreads();
            // columns of A and of V
            for (int e = threadIdx.x; e < (m / 2) * n; e += blockDim.x) {
                const int k = e / n, i = e - k * n;
                const int p = perm[2 * k], q = perm[2 * k + 1];
                if (q >= n || s[k] == 0.0) continue;
                const double ap = A[i * lda + p], aq = A[i * lda + q];
                A[i * lda + p] = c[k] * ap - s[k] * aq;
                A[i * lda + q] = s[k] * ap + c[k] * aq;
                double* vr = V + (size_t)i * ldv;
                const double vp = vr[p], vq = vr[q];
                vr[p] = c[k] * vp - s[k] * vq;
                vr[q] = s[k] * vp + c[k] * vq;
            }
            __syncthreads();
        }
    }
    // ascending order: rank of each eigenvalue (ties by index)
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const double di = A[i * lda + i];
        int r = 0;
        for (int j = 0; j < n; ++j) {
            const double dj = A[j * lda + j];
            if (dj < di || (dj == di && j < i)) ++r;
        }
        perm[i] = r;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) w[perm[i]] = A[i * lda + i];
    __syncthreads();
    // permute the columns of V row by row through LDS (A is free now)
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
        const int i = e / n, j = e - i * n;
        A[i * lda + perm[j]] = V[(size_t)i * ldv + j];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
        const int i = e / n, j = e - i * n;
        V[(size_t)i * ldv + j] = A[i * lda + j];
    }
    __syncthreads();
}

// LDS vectors of a molecule workgroup (the matrices are dynamic LDS).
struct WgSmall {
    double w[BATCH_MAX_NBF];
    double cs[2][BATCH_MAX_NBF];      // (c, s) of a round's rotations, two rounds
    int pq[2][BATCH_MAX_NBF];         // (p, q), p < q
    int perm[BATCH_MAX_NBF];
    double red[BTL / 64];
    double dots[8 * (BTL / 64)];
    double Bm[9 * 9];
    double rhs[9];
};
static_assert(BATCH_MAX_NBF <= 88, "a round's blocks (h (h + 1) / 2, h = n / 2) take one thread each");

// V <- V J for one round's rotations (thread t of nt): a group of threads
// per rotation, so (c, s) and (p, q) are read once for several rows.
__device__ __forceinline__ void jacobi_rotate_v(int n, int ld, int h, lds_d* V, const double* cs, const int* pq,
                                                int k, int i0, int tk)
{
    if (k >= h) return;
    const int p = pq[2 * k], q = pq[2 * k + 1];
    const double c = cs[2 * k], s = cs[2 * k + 1];
    if (q >= n || s == 0.0) return;
    for (int i = i0; i < n; i += tk) {
        lds_d* vr = V + i * ld;
        const double vp = vr[p], vq = vr[q];
        vr[p] = c * vp - s * vq;
        vr[q] = s * vp + c * vq;
    }
}

// Cyclic Jacobi eigensolver with A (destroyed, only its upper triangle is
// read) and V both in LDS (leading dimension lds_ld(n)).  V holds the
// starting basis on entry: the identity, or the eigenvectors of a nearby
// matrix, in which case A must be V^T A0 V; on exit A0 = V diag(w) V^T with
// V's columns in ascending order of w.  A round applies the h = m/2 disjoint
// rotations of the round-robin ordering (m = n rounded up to even).
//
// Bound by the latency of the m - 1 rounds of each sweep (a barrier, a chain
// of two reciprocal square roots, a barrier, an LDS round trip), and by LDS
// bandwidth at the largest n.  So: one wavefront computes the angles of round
// r while the others apply round r - 1 to V (nothing else needs V); a thread
// owns one 2 x 2 block (rows of one rotation, columns of another) of the
// upper triangle for the whole run, so no index is divided inside the loops
// and half the matrix is neither read nor written; (c, s) come from
// rsqrt(d^2 + 4 a^2) and rsqrt(cos^2), without a division.  A and V
// say that they are in LDS: through plain pointers every access took the flat
// path (S^-1/2 of 45 clusters of up to 65 functions 1.30 ms against 0.78).
// Convergence: sum of squared off-diagonal elements at most 1e-30 of the
// squared Frobenius norm.
//
// Once all angles are small together, near the end and often from the start
// when V comes from the last SCF step, one product with Q = I + E + E^2/2 +
// E^3/8 takes the place of a sweep and has the same quadratic convergence;
// E_ij is the angle of the rotation of (i, j).  Q Q^T = I - E^6/64 for any
// antisymmetric E: I to 1e-18 where ||E||_F <= 2e-3, else after one or two
// Newton-Schulz steps Q (3 - Q^T Q)/2, up to ||E||_F = 0.39.  That is five to
// nine products on the matrix cores instead of m - 1 rounds with two barriers
// each.  Elements that are negligible together (a^2 <= 1e-30 ||A||^2 / n^2)
// are left out of E, so degenerate pairs do not matter; where E is larger, or
// a product did not halve the sum, sweeps go on.  At n = 65 a sweep takes
// 75 us, a product 45-58 us (5 us per matrix product: 6800 cycles of the FP64
// matrix cores), the last one 25 us.  products: E is a third
// matrix in LDS (else sweeps only); W: 2 n^2 doubles in global memory.
__device__ __forceinline__ void lds_jacobi(int n, lds_d* A, lds_d* V, bool products, lds_d* E, gbl_d* W, WgSmall& L)
{
    const int ld = lds_ld(n);
    const int m = (n + 1) & ~1;
    const int h = m / 2;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nwave = (int)(blockDim.x >> 6);
    double* w = L.w;
    int* perm = L.perm;
    // this thread's block (k1 <= k2) of A
    int k1 = -1, k2 = 0;
    if (tid < h * (h + 1) / 2) {
        k2 = (int)((sqrtf(8.0f * tid + 1.0f) - 1.0f) * 0.5f);
        while (k2 * (k2 + 1) / 2 > tid) --k2;
        while ((k2 + 1) * (k2 + 2) / 2 <= tid) ++k2;
        k1 = tid - k2 * (k2 + 1) / 2;
    }
    // rows of V: threads 64.. inside the rounds, all of them after the last
    const int tk = max(1, ((int)blockDim.x - 64) / h);
    const int vk = tid >= 64 ? (tid - 64) / tk : h, vi = tid >= 64 ? (tid - 64) - vk * tk : 0;
    // positions of rotation `lane` in the round-robin (first wavefront)
    int s1 = lane, s2 = m - 1 - lane;
    double diag = 0.0, norm = 0.0;
    for (int i = wave; i < n; i += nwave)
        for (int j = i + lane; j < n; j += 64) {
            const double a = A[i * ld + j];
            if (j == i) diag = fma(a, a, diag);
            else norm = fma(2.0 * a, a, norm);
        }
    const double fro = wg_sum(diag + norm, L.red);
    const double small = 1e-30 * fro / ((double)n * n);
    double last = HUGE_VAL;   // the off-diagonal sum before the last product
    // angle of the rotation that zeroes a between diagonal elements d apart
    auto angle = [](double a, double d) { return copysign(0.5, d) * atan2(2.0 * a, fabs(d)); };
    int buf = 0;
    bool pending = false;
    for (int sweep = 0; sweep < 60; ++sweep) {
        double off = 0.0, e2 = 0.0;
        for (int i = wave; i < n; i += nwave)
            for (int j = i + 1 + lane; j < n; j += 64) {
                const double a = A[i * ld + j];
                off = fma(2.0 * a, a, off);
                if (products && a * a > small) {
                    const double e = angle(a, A[j * ld + j] - A[i * ld + i]);
                    e2 = fma(2.0 * e, e, e2);
                }
            }
        off = wg_sum(off, L.red);
        if (!(off > 1e-30 * fro)) break;
        if (off > 0.5 * last) products = false;
        if (products) {
            e2 = wg_sum(e2, L.red);
            if (e2 <= 0.15) {
                last = off;
                if (pending) {
                    if (wave > 0) jacobi_rotate_v(n, ld, h, V, L.cs[buf ^ 1], L.pq[buf ^ 1], vk, vi, tk);
                    pending = false;
                }
                gbl_d* W1 = W;
                gbl_d* W2 = W + (size_t)n * n;
                elems_loop(n, [&](int i, int j) {
                    const int p = min(i, j), q = max(i, j);
                    const double a = A[p * ld + q];
                    W1[i * n + j] = a;
                    const double e = p != q && a * a > small ? angle(a, A[q * ld + q] - A[p * ld + p]) : 0.0;
                    E[i * ld + j] = i < j ? e : -e;
                });
                __syncthreads();
                double v[8];
                auto from_w2 = [&] {
                    elems(n, [&](int u, int i, int j, bool in) {
                        if (in) v[u] = W2[i * n + j];
                    });
                };
                // what is left off the diagonal after this product is at most
                // e2 off; where that converges, V is all that is needed, and
                // the eigenvalues are the diagonal to second order
                const bool final = 4.0 * e2 * off <= 1e-30 * fro;
                double wi = 0.0;
                if (final && tid < n) {
                    wi = A[tid * ld + tid];
                    for (int j = 0; j < n; ++j)
                        if (j != tid) wi = fma(-A[min(tid, j) * ld + max(tid, j)], E[tid * ld + j], wi);
                }
                __syncthreads();
                lds_gemm(n, false, E, false, E, A);
                if (e2 > 4e-9) {   // without E^3/8 Q Q^T = I + E^4/4: I to 4e-18 otherwise
                    lds_gemm(n, false, E, false, A, E, n, W2, n);
                    from_w2();
                } else {
                    for (int u = 0; u < 8; ++u) v[u] = 0.0;
                }
                elems(n, [&](int u, int i, int j, bool in) {
                    if (in) A[i * ld + j] = (i == j ? 1.0 : 0.0) + E[i * ld + j] + 0.5 * A[i * ld + j] + 0.125 * v[u];
                });
                __syncthreads();
                for (int ns = e2 <= 4e-6 ? 0 : (e2 <= 5.8e-3 ? 1 : 2); ns > 0; --ns) {
                    lds_gemm(n, true, A, false, A, E);
                    lds_gemm(n, false, A, false, E, E, n, W2, n);
                    from_w2();
                    elems(n, [&](int u, int i, int j, bool in) {
                        if (in) A[i * ld + j] = 1.5 * A[i * ld + j] - 0.5 * v[u];
                    });
                    __syncthreads();
                }
                lds_gemm(n, false, V, false, A, E);
                for (int e = tid; e < n * ld; e += blockDim.x) V[e] = E[e];
                if (final && tid < n) A[tid * ld + tid] = wi;
                __syncthreads();
                if (final) break;
                lds_load(n, W1, n, E);
                lds_gemm(n, false, E, false, A, E, n, W2, n);
                lds_load(n, W2, n, E);
                lds_gemm(n, true, A, false, E, E, n, W1, n);
                lds_load(n, W1, n, A);
                continue;
            }
        }
        for (int round = 0; round < m - 1; ++round) {
            double* cs = L.cs[buf];
            int* pq = L.pq[buf];
            if (wave == 0) {
                if (lane < h) {
                    const int p = min(s1, s2), q = max(s1, s2);
                    double cc = 1.0, ss = 0.0;
                    if (q < n) {
                        const double apq = A[p * ld + q];
                        const double d = A[q * ld + q] - A[p * ld + p];
                        const double r2 = fma(d, d, 4.0 * apq * apq);
                        if (apq != 0.0 && r2 > 1e-290) {
                            const double ri = rsqrt(r2);
                            const double x = fma(0.5 * fabs(d), ri, 0.5);   // cos^2 of the smaller angle
                            const double rc = rsqrt(x);
                            cc = x * rc;
                            ss = copysign(apq * ri * rc, (d >= 0.0) == (apq >= 0.0) ? 1.0 : -1.0);
                            // c^2 + s^2 = 1 to rounding, whatever the two roots' last bits
                            const double f = -0.5 * fma(ss, ss, fma(cc, cc, -1.0));
                            cc = fma(cc, f, cc);
                            ss = fma(ss, f, ss);
                        }
                    }
                    cs[2 * lane] = cc;
                    cs[2 * lane + 1] = ss;
                    pq[2 * lane] = p;
                    pq[2 * lane + 1] = q;
                    if (s1 != 0 && ++s1 == m) s1 = 1;
                    if (++s2 == m) s2 = 1;
                }
            } else if (pending) {
                jacobi_rotate_v(n, ld, h, V, L.cs[buf ^ 1], L.pq[buf ^ 1], vk, vi, tk);
            }
            __syncthreads();
            // A <- J^T A J, block (k1, k2) = rows p1, q1 x columns p2, q2
            if (k1 >= 0) {
                const double c1 = cs[2 * k1], t1 = cs[2 * k1 + 1], c2 = cs[2 * k2], t2 = cs[2 * k2 + 1];
                if (t1 != 0.0 || t2 != 0.0) {
                    const int p1 = pq[2 * k1], q1 = pq[2 * k1 + 1], p2 = pq[2 * k2], q2 = pq[2 * k2 + 1];
                    const bool r1 = q1 < n, r2 = q2 < n;   // the dummy index n has no row or column
                    auto at = [&](int i, int j) { return min(i, j) * ld + max(i, j); };
                    const int ia = at(p1, p2), ib = at(p1, q2), id = at(q1, p2), ie = at(q1, q2);
                    const double a = A[ia];
                    const double b = r2 ? A[ib] : 0.0;
                    const double d = r1 ? A[id] : 0.0;
                    const double e = (r1 && r2) ? A[ie] : 0.0;
                    const double a1 = c1 * a - t1 * d, b1 = c1 * b - t1 * e;
                    const double d1 = t1 * a + c1 * d, e1 = t1 * b + c1 * e;
                    A[ia] = c2 * a1 - t2 * b1;
                    if (r2) A[ib] = t2 * a1 + c2 * b1;
                    if (r1 && k1 != k2) A[id] = c2 * d1 - t2 * e1;
                    if (r1 && r2) A[ie] = t2 * d1 + c2 * e1;
                }
            }
            __syncthreads();
            buf ^= 1;
            pending = true;
        }
    }
    if (pending) {
        if (wave > 0) jacobi_rotate_v(n, ld, h, V, L.cs[buf ^ 1], L.pq[buf ^ 1], vk, vi, tk);
        __syncthreads();
    }
    // ascending order: rank of each eigenvalue (ties by index)
    for (int i = tid; i < n; i += blockDim.x) {
        const double di = A[i * ld + i];
        int r = 0;
        for (int j = 0; j < n; ++j) {
            const double dj = A[j * ld + j];
            if (dj < di || (dj == di && j < i)) ++r;
        }
        perm[i] = r;
    }
    __syncthreads();
    for (int i = tid; i < n; i += blockDim.x) w[perm[i]] = A[i * ld + i];
    __syncthreads();
    for (int i = wave; i < n; i += nwave)
        for (int j = lane; j < n; j += 64) A[i * ld + perm[j]] = V[i * ld + j];
    __syncthreads();
    for (int e = tid; e < n * ld; e += blockDim.x) V[e] = A[e];
    __syncthreads();
}

// LDS of a molecule workgroup: one n x n matrix (leading dimension n) plus
// small vectors; n <= BATCH_MAX_NBF.
struct WgLds {
    double A[BATCH_MAX_NBF * BATCH_MAX_NBF];
    double w[BATCH_MAX_NBF];
    double cs[BATCH_MAX_NBF + 2];
    int perm[BATCH_MAX_NBF + 2];
    double red[BT / 64];
    double Bm[9 * 9];
    double rhs[9];
};

// X = S^-1/2 and U = S^1/2 of each molecule's overlap block (mmd/molecule.py:284-286).
__global__ void __launch_bounds__(BT) batch_overlap_kernel(BatchArgs B)
{
    __shared__ WgLds L;
    const BatchMol M = B.mol[blockIdx.x];
    const int n = M.n, N = B.N;
    double* V = B.work + M.wo;   // n x n eigenvectors
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) L.A[e] = blk(B.S, N, M.f0)[(size_t)(e / n) * N + e % n];
    __syncthreads();
    wg_jacobi(n, L.A, n, V, n, L.w, L.perm, L.cs, L.red);
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
        const int i = e / n, j = e - i * n;
        double x = 0.0, u = 0.0;
        for (int k = 0; k < n; ++k) {
            const double vv = V[(size_t)i * n + k] * V[(size_t)j * n + k];
            x = fma(vv, 1.0 / sqrt(L.w[k]), x);
            u = fma(vv, sqrt(L.w[k]), u);
        }
        blk(B.X, N, M.f0)[(size_t)i * N + j] = x;
        blk(B.U, N, M.f0)[(size_t)i * N + j] = u;
    }
    if (threadIdx.x == 0 && !(L.w[0] > 0.0)) B.flag[blockIdx.x] = -1;   // not positive definite
}

// batch_overlap_kernel with S and its eigenvectors in LDS (two n x n
// matrices of dynamic shared memory, and a third for the eigensolver where
// it fits).
__global__ void __launch_bounds__(BTL) batch_overlap_lds_kernel(BatchArgs B, int three)
{
    extern __shared__ double dyn[];
    __shared__ WgSmall L;
    const BatchMol M = B.mol[blockIdx.x];
    const int n = M.n, N = B.N, ld = lds_ld(n);
    lds_d* A = (lds_d*)dyn;
    lds_d* V = A + n * ld;
    elems_loop(n, [&](int i, int j) { V[i * ld + j] = i == j ? 1.0 : 0.0; });
    lds_load(n, (const gbl_d*)blk(B.S, N, M.f0), N, A);
    lds_jacobi(n, A, V, three != 0, V + n * ld, (gbl_d*)(B.work + M.wo), L);
    // X = V w^-1/2 V^T and U = V w^1/2 V^T: the scaled eigenvectors in A, then
    // one product each straight into the molecule's blocks
    for (int u = 0; u < 2; ++u) {
        elems_loop(n, [&](int i, int j) {
            A[i * ld + j] = u ? V[i * ld + j] * sqrt(L.w[j]) : V[i * ld + j] / sqrt(L.w[j]);
        });
        __syncthreads();
        lds_gemm(n, false, A, true, V, A, n, (gbl_d*)blk(u ? B.U : B.X, N, M.f0), N);
    }
    if (threadIdx.x == 0 && !(L.w[0] > 0.0)) B.flag[blockIdx.x] = -1;   // not positive definite
}

// One iteration of the reference's loop for each unconverged molecule.
// build = 0: step 0 (FO = X^T F X); build = 1: after a Fock build into G:
// F += G, P_old = P, DIIS (window 8), FO = X^T F_diis X.  Then eigh(FO),
// C = X C', P = C_occ C_occ^T, the energy sum (H + F)_pq P_qp, ||P - P_old||,
// dP = P - P_old for the next build, and the convergence flag.
__global__ void __launch_bounds__(BT) batch_step_kernel(BatchArgs B, int build, int diis, double conver)
{
    __shared__ WgLds L;
    const int mi = blockIdx.x;
    const BatchMol M = B.mol[mi];
    BatchState& Sx = B.state[mi];
    const int n = M.n, N = B.N, f0 = M.f0;
    if (Sx.converged) return;
    double* F = blk(B.F, N, f0);
    double* P = blk(B.P, N, f0);
    double* Po = blk(B.Pold, N, f0);
    double* dP = blk(B.dP, N, f0);
    const double* G = blk(B.G, N, f0);
    const double* H = blk(B.H, N, f0);
    const double* S = blk(B.S, N, f0);
    const double* X = blk(B.X, N, f0);
    double* T1 = B.work + M.wo;                 // n x n work matrices (packed)
    double* T2 = T1 + (size_t)n * n;
    double* Fd = T2 + (size_t)n * n;
    double* Eset = B.diis + M.d8;               // 8 error matrices, then 8 Fock matrices
    double* Fset = Eset + (size_t)8 * n * n;
    const double* Fuse = F;
    int ld_use = N;
    if (build) {
        for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
            const size_t o = (size_t)(e / n) * N + e % n;
            F[o] += G[o];
            Po[o] = P[o];
        }
        __syncthreads();
        if (diis) {
            // error X (F P S - S P F) X of the new F (mmd/scf.py:146-150)
            const int cnt = Sx.ndiis;
            const int slot = cnt == 8 ? Sx.order[0] : cnt;   // a full window drops its oldest entry
            __syncthreads();
            if (cnt == 8 && threadIdx.x == 0) {
                for (int i = 0; i < 7; ++i) Sx.order[i] = Sx.order[i + 1];
                for (int i = 0; i < 7; ++i)
                    for (int j = 0; j < 7; ++j) Sx.Bm[i * 8 + j] = Sx.Bm[(i + 1) * 8 + (j + 1)];
            }
            __syncthreads();
            const int nw = cnt == 8 ? 8 : cnt + 1;
            double* Es = Eset + (size_t)slot * n * n;
            wg_gemm(n, false, P, N, false, S, N, T1, n);          // P S
            wg_gemm(n, false, F, N, false, T1, n, T2, n);         // F P S
            for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
                const int i = e / n, j = e - i * n;
                T1[e] = T2[i * n + j] - T2[j * n + i];            // FPS - SPF
            }
            __syncthreads();
            wg_gemm(n, false, X, N, false, T1, n, T2, n);
            wg_gemm(n, false, T2, n, false, X, N, Es, n);
            for (int e = threadIdx.x; e < n * n; e += blockDim.x)
                Fset[(size_t)slot * n * n + e] = F[(size_t)(e / n) * N + e % n];
            if (threadIdx.x == 0) Sx.order[nw - 1] = slot;
            __syncthreads();
            // new row of B: tr(e_k^T e_new) (mmd/scf.py:163-167)
            for (int k = 0; k < nw; ++k) {
                const double* Ek = Eset + (size_t)Sx.order[k] * n * n;
                double d = 0.0;
                for (int e = threadIdx.x; e < n * n; e += blockDim.x) d = fma(Ek[e], Es[e], d);
                d = wg_sum(d, L.red);
                if (threadIdx.x == 0) Sx.Bm[(nw - 1) * 8 + k] = Sx.Bm[k * 8 + (nw - 1)] = d;
            }
            if (threadIdx.x == 0) {
                Sx.ndiis = nw;
                // [B -1; -1 0] c = [0 .. 0 -1] (mmd/scf.py:160-170), Gaussian
                // elimination with partial pivoting
                const int mm = nw + 1;
                double* a = L.Bm;
                double* r = L.rhs;
                for (int i = 0; i < mm; ++i) {
                    for (int j = 0; j < mm; ++j)
                        a[i * 9 + j] = (i < nw && j < nw) ? Sx.Bm[i * 8 + j] : ((i == nw && j == nw) ? 0.0 : -1.0);
                    r[i] = i == nw ? -1.0 : 0.0;
                }
                bool ok = true;
                for (int col = 0; col < mm; ++col) {
                    int piv = col;
                    for (int i = col + 1; i < mm; ++i)
                        if (fabs(a[i * 9 + col]) > fabs(a[piv * 9 + col])) piv = i;
                    if (a[piv * 9 + col] == 0.0) { ok = false; break; }
                    if (piv != col) {
                        for (int j = 0; j < mm; ++j) { const double t = a[col * 9 + j]; a[col * 9 + j] = a[piv * 9 + j]; a[piv * 9 + j] = t; }
                        const double t = r[col]; r[col] = r[piv]; r[piv] = t;
                    }
                    for (int i = col + 1; i < mm; ++i) {
                        const double f = a[i * 9 + col] / a[col * 9 + col];
                        for (int j = col; j < mm; ++j) a[i * 9 + j] -= f * a[col * 9 + j];
                        r[i] -= f * r[col];
                    }
                }
                for (int i = mm - 1; i >= 0 && ok; --i) {
                    double v = r[i];
                    for (int j = i + 1; j < mm; ++j) v -= a[i * 9 + j] * r[j];
                    r[i] = v / a[i * 9 + i];
                }
                if (!ok) B.flag[mi] = -2;
            }
            __syncthreads();
            // F_diis = sum_k c_k F_k (mmd/scf.py:175-178)
            for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
                double v = 0.0;
                for (int k = 0; k < nw; ++k) v = fma(L.rhs[k], Fset[(size_t)Sx.order[k] * n * n + e], v);
                Fd[e] = v;
            }
            __syncthreads();
            Fuse = Fd;
            ld_use = n;
        }
    }
    // FO = X^T F X into LDS
    wg_gemm(n, true, X, N, false, Fuse, ld_use, T1, n);
    wg_gemm(n, false, T1, n, false, X, N, T2, n);
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) L.A[e] = T2[e];
    __syncthreads();
    double* CO = T1;   // eigenvectors C' (n x n)
    wg_jacobi(n, L.A, n, CO, n, L.w, L.perm, L.cs, L.red);
    // C = X C'  (T2); P = C_occ C_occ^T
    wg_gemm(n, false, X, N, false, CO, n, T2, n);
    const int nocc = M.nocc;
    double e_el = 0.0, rms = 0.0;
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
        const int i = e / n, j = e - i * n;
        double v = 0.0;
        for (int k = 0; k < nocc; ++k) v = fma(T2[i * n + k], T2[j * n + k], v);
        const size_t o = (size_t)i * N + j;
        P[o] = v;
        const double d = v - Po[o];
        dP[o] = d;
        rms = fma(d, d, rms);
        // sum_pq (H + F)_pq P_qp, P symmetric (mmd/scf.py:118-121)
        e_el = fma(H[o] + F[o], v, e_el);
    }
    e_el = wg_sum(e_el, L.red);
    rms = wg_sum(rms, L.red);
    // a molecule that converges here adds nothing to later builds
    if (Sx.iterations > 0 && sqrt(rms) < conver)
        for (int e = threadIdx.x; e < n * n; e += blockDim.x) dP[(size_t)(e / n) * N + e % n] = 0.0;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double energy = e_el + M.enuc;
        const int step = Sx.iterations;
        Sx.delta_energy = step > 0 ? energy - Sx.energy : 1e20;
        Sx.energy = energy;
        Sx.prms = step > 0 ? sqrt(rms) : 1e20;
        if (step > 0 && Sx.prms < conver) Sx.converged = 1;
        else Sx.iterations = step + 1;
    }
    for (int k = threadIdx.x; k < n; k += blockDim.x) B.mo[M.f0 + k] = L.w[k];
}

// Solves the DIIS equations [B -1; -1 0] c = [0 .. 0 -1] (mmd/scf.py:160-170)
// of nw errors by Gaussian elimination with partial pivoting in one
// wavefront, a lane per row: c in r, false if singular.  a, r: LDS, leading
// dimension 9; Bw: the window's error overlaps.
__device__ bool diis_solve(int nw, const double* Bw, double* a, double* r)
{
    const int mm = nw + 1, i = threadIdx.x;
    if (i < mm) {
        for (int j = 0; j < mm; ++j)
            a[i * 9 + j] = (i < nw && j < nw) ? Bw[i * 8 + j] : ((i == nw && j == nw) ? 0.0 : -1.0);
        r[i] = i == nw ? -1.0 : 0.0;
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    for (int col = 0; col < mm; ++col) {
        int piv = col;
        for (int k = col + 1; k < mm; ++k)
            if (fabs(a[k * 9 + col]) > fabs(a[piv * 9 + col])) piv = k;
        if (a[piv * 9 + col] == 0.0) return false;
        __threadfence_block();
        if (piv != col && i <= mm) {   // lane j swaps column j, lane mm the right side
            double* x = i < mm ? a + col * 9 + i : r + col;
            double* y = i < mm ? a + piv * 9 + i : r + piv;
            const double t = *x;
            *x = *y;
            *y = t;
        }
        __threadfence_block();
        if (i > col && i < mm) {
            const double f = a[i * 9 + col] / a[col * 9 + col];
            for (int j = col; j < mm; ++j) a[i * 9 + j] -= f * a[col * 9 + j];
            r[i] -= f * r[col];
        }
        __threadfence_block();
    }
    if (i == 0)
        for (int k = mm - 1; k >= 0; --k) {
            double v = r[k];
            for (int j = k + 1; j < mm; ++j) v -= a[k * 9 + j] * r[j];
            r[k] = v / a[k * 9 + k];
        }
    return true;
}

// The step of batch_step_kernel with its matrices in LDS: three n x n
// matrices (dynamic shared memory) hold P S, F P S, the error, X, F_diis, FO
// and the eigenvectors in turn, so the products and the eigensolver run from
// LDS.  Same operations as batch_step_kernel.  One molecule is one serial
// chain on one compute unit, so what bounds it is latency: barriers, rounds
// trips to memory (issued together, see elems) and the eigensolver's rounds.
__global__ void __launch_bounds__(BTL) batch_step_lds_kernel(BatchArgs B, int build, int diis, double conver)
{
    extern __shared__ double dyn[];
    __shared__ WgSmall L;
    const int mi = blockIdx.x;
    const BatchMol M = B.mol[mi];
    BatchState& Sx = B.state[mi];
    const int n = M.n, N = B.N, f0 = M.f0, ld = lds_ld(n);
    if (Sx.converged) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = (int)(blockDim.x >> 6);
    const size_t nn = (size_t)n * n;
    lds_d* M0 = (lds_d*)dyn;
    lds_d* M1 = M0 + n * ld;
    lds_d* M2 = M1 + n * ld;
    gbl_d* F = (gbl_d*)blk(B.F, N, f0);
    gbl_d* P = (gbl_d*)blk(B.P, N, f0);
    gbl_d* Po = (gbl_d*)blk(B.Pold, N, f0);
    gbl_d* dP = (gbl_d*)blk(B.dP, N, f0);
    const gbl_d* G = (const gbl_d*)blk(B.G, N, f0);
    const gbl_d* H = (const gbl_d*)blk(B.H, N, f0);
    const gbl_d* S = (const gbl_d*)blk(B.S, N, f0);
    const gbl_d* X = (const gbl_d*)blk(B.X, N, f0);
    gbl_d* Eset = (gbl_d*)(B.diis + M.d8);
    gbl_d* Fset = Eset + (size_t)8 * nn;
    bool fo_from_lds = false;   // F_diis in M1
    if (build) {
        double v[8], g[8];
        elems(n, [&](int u, int i, int j, bool in) {   // F += G
            if (in) {
                v[u] = F[(size_t)i * N + j];
                g[u] = G[(size_t)i * N + j];
            }
        });
        elems(n, [&](int u, int i, int j, bool in) {
            v[u] += g[u];
            if (in) F[(size_t)i * N + j] = v[u];
        });
        if (diis) {
            const int cnt = Sx.ndiis;
            const int slot = cnt == 8 ? Sx.order[0] : cnt;
            const int nw = cnt == 8 ? 8 : cnt + 1;
            gbl_d* Es = Eset + (size_t)slot * nn;
            gbl_d* Fs = Fset + (size_t)slot * nn;
            lds_load(n, P, N, M0);
            lds_load(n, S, N, M1);
            if (cnt == 8 && threadIdx.x == 0) {   // every thread has read cnt and order[0]
                for (int i = 0; i < 7; ++i) Sx.order[i] = Sx.order[i + 1];
                for (int i = 0; i < 7; ++i)
                    for (int j = 0; j < 7; ++j) Sx.Bm[i * 8 + j] = Sx.Bm[(i + 1) * 8 + (j + 1)];
            }
            if (threadIdx.x == 0) Sx.order[nw - 1] = slot;
            lds_gemm(n, false, M0, false, M1, M2);                 // P S
            elems(n, [&](int u, int i, int j, bool in) {
                if (!in) return;
                Po[(size_t)i * N + j] = M0[i * ld + j];
                Fs[i * n + j] = v[u];
                M0[i * ld + j] = v[u];
            });
            __syncthreads();
            lds_gemm(n, false, M0, false, M2, M1);                 // F P S
            elems_loop(n, [&](int i, int j) { M2[i * ld + j] = M1[i * ld + j] - M1[j * ld + i]; });   // FPS - SPF
            lds_load(n, X, N, M0);
            lds_gemm(n, false, M0, false, M2, M1);                 // X (FPS - SPF)
            lds_gemm(n, false, M1, false, M0, M2);                 // ... X: the error
            // the error into the window and its overlaps with the others
            elems_loop(n, [&](int i, int j) { Es[i * n + j] = M2[i * ld + j]; });
            for (int k = 0; k < nw; ++k) {
                const gbl_d* Ek = Eset + (size_t)Sx.order[k] * nn;   // this thread wrote its own elements of the last
                double d = 0.0;
                elems(n, [&](int u, int i, int j, bool in) {
                    if (in) g[u] = Ek[i * n + j];
                });
                elems(n, [&](int u, int i, int j, bool in) {
                    if (in) d = fma(g[u], M2[i * ld + j], d);
                });
                for (int o = 32; o > 0; o >>= 1) d += __shfl_xor(d, o);
                if (lane == 0) L.dots[k * (BTL / 64) + wave] = d;
            }
            __syncthreads();
            if (wave == 0) {
                if (lane < nw) {
                    double d = 0.0;
                    for (int w = 0; w < nwave; ++w) d += L.dots[lane * (BTL / 64) + w];
                    Sx.Bm[(nw - 1) * 8 + lane] = d;
                    Sx.Bm[lane * 8 + (nw - 1)] = d;
                }
                __threadfence_block();
                const bool ok = diis_solve(nw, Sx.Bm, L.Bm, L.rhs);
                if (lane == 0) {
                    Sx.ndiis = nw;
                    if (!ok) B.flag[mi] = -2;
                }
            }
            __syncthreads();
            double f[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};   // F_diis into M1
            for (int k = 0; k < nw - 1; ++k) {
                const gbl_d* Fk = Fset + (size_t)Sx.order[k] * nn;
                const double ck = L.rhs[k];
                elems(n, [&](int u, int i, int j, bool in) {
                    if (in) g[u] = Fk[i * n + j];
                });
                elems(n, [&](int u, int, int, bool in) {
                    if (in) f[u] = fma(ck, g[u], f[u]);
                });
            }
            elems(n, [&](int u, int i, int j, bool in) {
                if (in) M1[i * ld + j] = fma(L.rhs[nw - 1], v[u], f[u]);
            });
            __syncthreads();
            fo_from_lds = true;                                    // X still in M0
        } else {
            elems(n, [&](int u, int i, int j, bool in) {
                if (in) g[u] = P[(size_t)i * N + j];
            });
            elems(n, [&](int u, int i, int j, bool in) {
                if (in) Po[(size_t)i * N + j] = g[u];
            });
            __syncthreads();
        }
    }
    // FO = X^T F X  (X in M0, F in M1)
    if (!fo_from_lds) {
        lds_load(n, X, N, M0);
        lds_load(n, F, N, M1);
    }
    lds_gemm(n, true, M0, false, M1, M2);
    lds_gemm(n, false, M2, false, M0, M1);                         // FO in M1
    // eigenvectors of FO, started from the last step's (kept in the work
    // area): A = V^T FO V is nearly diagonal once the SCF settles
    gbl_d* Vkeep = (gbl_d*)(B.work + M.wo);
    if (Sx.warm) {
        lds_load(n, Vkeep, n, M0);
        lds_gemm(n, false, M1, false, M0, M2);                     // FO V
        lds_gemm(n, true, M0, false, M2, M1);                      // V^T FO V
    } else {
        elems_loop(n, [&](int i, int j) { M0[i * ld + j] = i == j ? 1.0 : 0.0; });
        __syncthreads();
    }
    lds_jacobi(n, M1, M0, true, M2, Vkeep + nn, L);                // C' in M0
    elems_loop(n, [&](int i, int j) { Vkeep[i * n + j] = M0[i * ld + j]; });
    lds_load(n, X, N, M2);
    lds_gemm(n, false, M2, false, M0, M1);                         // C = X C' in M1
    lds_gemm(n, false, M1, true, M1, M2, M.nocc, nullptr, 0);      // P = C_occ C_occ^T in M2
    double e_el = 0.0, rms = 0.0;
    {
        double po[8], hf[8], ff[8];
        elems(n, [&](int u, int i, int j, bool in) {
            if (!in) return;
            const size_t o = (size_t)i * N + j;
            po[u] = Po[o];
            hf[u] = H[o];
            ff[u] = F[o];
        });
        elems(n, [&](int u, int i, int j, bool in) {
            if (!in) return;
            const double p = M2[i * ld + j];
            const size_t o = (size_t)i * N + j;
            P[o] = p;
            const double d = p - po[u];
            dP[o] = d;
            rms = fma(d, d, rms);
            e_el = fma(hf[u] + ff[u], p, e_el);
        });
    }
    e_el = wg_sum(e_el, L.red);
    rms = wg_sum(rms, L.red);
    const int step = Sx.iterations;
    // a molecule that converges here adds nothing to later builds
    if (step > 0 && sqrt(rms) < conver)
        elems_loop(n, [&](int i, int j) { dP[(size_t)i * N + j] = 0.0; });
    __syncthreads();
    if (threadIdx.x == 0) {
        const double energy = e_el + M.enuc;
        Sx.warm = 1;
        Sx.delta_energy = step > 0 ? energy - Sx.energy : 1e20;
        Sx.energy = energy;
        Sx.prms = step > 0 ? sqrt(rms) : 1e20;
        if (step > 0 && Sx.prms < conver) Sx.converged = 1;
        else Sx.iterations = step + 1;
    }
    for (int k = threadIdx.x; k < n; k += blockDim.x) B.mo[M.f0 + k] = L.w[k];
}

// Number of unconverged molecules into *out.
__global__ void batch_count_kernel(int nmol, const BatchState* state, int* out)
{
    int c = 0;
    for (int i = threadIdx.x; i < nmol; i += blockDim.x) c += state[i].converged ? 0 : 1;
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off);
    __shared__ int part[16];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += part[w];
        *out = t;
    }
}

// Copies each molecule's n x n block between the N x N block-diagonal
// matrix and the packed array (unpack: packed -> full).
__global__ void batch_pack_kernel(BatchArgs B, double* full, double* packed, int unpack)
{
    const BatchMol M = B.mol[blockIdx.x];
    const int n = M.n;
    for (int e = threadIdx.x; e < n * n; e += blockDim.x) {
        const size_t o = (size_t)(M.f0 + e / n) * B.N + M.f0 + e % n;
        if (unpack)
            full[o] = packed[M.po + e];
        else
            packed[M.po + e] = full[o];
    }
}

}  // namespace

hipError_t launch_batch_pack(const BatchArgs& B, const double* full, double* packed, hipStream_t st)
{
    hipLaunchKernelGGL(batch_pack_kernel, dim3(B.nmol), dim3(256), 0, st, B, const_cast<double*>(full), packed, 0);
    return hipGetLastError();
}

hipError_t launch_batch_unpack(const BatchArgs& B, const double* packed, double* full, hipStream_t st)
{
    hipLaunchKernelGGL(batch_pack_kernel, dim3(B.nmol), dim3(256), 0, st, B, full, const_cast<double*>(packed), 1);
    return hipGetLastError();
}

hipError_t launch_batch_overlap(const BatchArgs& B, hipStream_t st)
{
    const size_t mat = (size_t)B.maxn * lds_ld(B.maxn) * sizeof(double);
    if (B.lds_bytes >= 2 * mat + sizeof(WgSmall)) {
        const int three = B.lds_bytes >= 3 * mat + sizeof(WgSmall);
        hipLaunchKernelGGL(batch_overlap_lds_kernel, dim3(B.nmol), dim3(BTL), (2 + three) * mat, st, B, three);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(batch_overlap_kernel, dim3(B.nmol), dim3(BT), 0, st, B);
    return hipGetLastError();
}

hipError_t launch_batch_step(const BatchArgs& B, int build, int diis, double conver, hipStream_t st)
{
    // the all-LDS step where three n x n matrices of the largest molecule fit
    // beside the small vectors; the global-memory step otherwise
    const size_t dyn = 3 * (size_t)B.maxn * lds_ld(B.maxn) * sizeof(double);
    if (B.lds_bytes >= dyn + sizeof(WgSmall)) {
        hipLaunchKernelGGL(batch_step_lds_kernel, dim3(B.nmol), dim3(BTL), dyn, st, B, build, diis, conver);
    } else {
        hipLaunchKernelGGL(batch_step_kernel, dim3(B.nmol), dim3(BT), 0, st, B, build, diis, conver);
    }
    return hipGetLastError();
}

hipError_t launch_batch_count(const BatchArgs& B, int* out, hipStream_t st)
{
    hipLaunchKernelGGL(batch_count_kernel, dim3(1), dim3(1024), 0, st, B.nmol, B.state, out);
    return hipGetLastError();
}

}  // namespace mmd
