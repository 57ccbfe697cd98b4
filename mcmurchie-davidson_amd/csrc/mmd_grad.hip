// Nuclear gradient of the converged RHF energy (mmd/forces.py:8-97) with the
// derivative integrals of cython/grad.pyx, on the device:
//
//   dE/dX = sum_pq P_pq (2 dH_pq/dX) + sum_pqrs Gamma_pqrs d(pq|rs)/dX
//           - 2 sum_pq W_pq dS_pq/dX            (+ dV_NN/dX on the host)
//
// with P the half density (C_occ C_occ^T), W = P F P and, for the
// two-electron part, the density products of the positions a canonical
// quartet occupies in the reference's derivative tensor (forces.py:73-84):
// Gamma = sum over the distinct permutations (a,b,c,d) of the quartet of
// 2 P_ba P_dc - P_ca P_bd.  The derivative of a Gaussian with respect to its
// centre raises and lowers its Cartesian power: in Hermite form the 1-D
// coefficient E^{ij}_t becomes 2a E^{i+1,j}_t - i E^{i-1,j}_t (first centre)
// or 2b E^{i,j+1}_t - j E^{i,j-1}_t (second centre), cython/grad.pyx:97-103.
// The fourth centre of an ERI follows from translational invariance,
// d/dD = -(d/dA + d/dB + d/dC).
//
// Bases of whole shells take the kernels by shell class (the pair kernels
// below and mmd_grad_class.h); the per-function kernels with runtime angular
// momenta, whose tables lie in scratch, serve the other bases.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "mmd_device.h"
#include "mmd_grad.h"
#include "mmd_kernels.h"

namespace mmd {

namespace {

// 1-D Hermite table of a primitive pair (divided by K_AB), i <= LI, j <= LJ.
struct Tab1 {
    const double* E;
    int LI, LJ;
    __device__ double e(int i, int j, int t) const
    {
        if (i < 0 || j < 0 || t < 0 || t > i + j || i > LI || j > LJ) return 0.0;
        return E[(i * (LJ + 1) + j) * (LI + LJ + 1) + t];
    }
    // mode 0: E^{ij}_t; 1: derivative for the first centre; 2: for the second
    __device__ double c(int i, int j, int t, int mode, double a, double b) const
    {
        if (mode == 1) return 2.0 * a * e(i + 1, j, t) - (double)i * e(i - 1, j, t);
        if (mode == 2) return 2.0 * b * e(i, j + 1, t) - (double)j * e(i, j - 1, t);
        return e(i, j, t);
    }
};

constexpr int GERI_TAB = (MAX_L + 2) * (MAX_L + 2) * (2 * MAX_L + 3);   // LI, LJ <= MAX_L + 1
constexpr int GONE_TAB = (MAX_L + 2) * (MAX_L + 4) * (2 * MAX_L + 5);   // LI <= MAX_L + 1, LJ <= MAX_L + 3
constexpr int GMAX_LTOT = MAX_LTOT + 1;

// A primitive pair with tables one order above its functions on both indices.
struct GPair {
    double a, b, p, w, P[3];
    double E[3][GERI_TAB];
};

__device__ void gpair(const BFDesc& fa, const BFDesc& fb, int ia, int ib, const double* __restrict__ pexp,
                      const double* __restrict__ pw, GPair& o)
{
    const double A[3] = {fa.x, fa.y, fa.z}, B[3] = {fb.x, fb.y, fb.z};
    const int la[3] = {fa.l, fa.m, fa.n}, lb[3] = {fb.l, fb.m, fb.n};
    o.a = pexp[fa.p0 + ia];
    o.b = pexp[fb.p0 + ib];
    o.p = o.a + o.b;
    double k = 1.0;
    for (int x = 0; x < 3; ++x) {
        o.P[x] = (o.a * A[x] + o.b * B[x]) / o.p;
        k *= exp(-o.a * o.b / o.p * (A[x] - B[x]) * (A[x] - B[x]));
        etab_rt(la[x] + 1, lb[x] + 1, 0.5 / o.p, o.P[x] - A[x], o.P[x] - B[x], o.E[x]);
    }
    o.w = pw[fa.p0 + ia] * pw[fb.p0 + ib] * k;
}

// d[ab|cd]/d(centre, axis) of one primitive quartet for the nine
// directions A x,y,z, B x,y,z, C x,y,z (cython/grad.pyx:107-350).
__device__ void prim_quartet_grad(const int* la, const int* lb, const int* lc, const int* ld, const GPair& P,
                                  const GPair& Q, const double* __restrict__ boys, double* out)
{
    const int L = la[0] + la[1] + la[2] + lb[0] + lb[1] + lb[2] + lc[0] + lc[1] + lc[2] + ld[0] + ld[1] + ld[2] + 1;
    const double alpha = P.p * Q.p / (P.p + Q.p);
    const double X = P.P[0] - Q.P[0], Y = P.P[1] - Q.P[1], Z = P.P[2] - Q.P[2];
    double F[GMAX_LTOT + 1];
    boys_runtime(L, alpha * (X * X + Y * Y + Z * Z), boys, F);
    double s = 1.0;
    for (int m = 0; m <= L; ++m) { F[m] *= s; s *= -2.0 * alpha; }
    double R[nherm(GMAX_LTOT)];
    hermite_R_rt(L, X, Y, Z, F, R);
    const double pref = 34.98683665524972497 / (P.p * Q.p * sqrt(P.p + Q.p)) * P.w * Q.w;
    Tab1 tb[3], tk[3];
    for (int x = 0; x < 3; ++x) {
        tb[x] = Tab1{P.E[x], la[x] + 1, lb[x] + 1};
        tk[x] = Tab1{Q.E[x], lc[x] + 1, ld[x] + 1};
    }
    for (int dir = 0; dir < 9; ++dir) {
        const int ax = dir % 3;
        const int cb = dir < 3 ? 1 : (dir < 6 ? 2 : 0);
        const int ck = dir >= 6 ? 1 : 0;
        int nb[3], nk[3], mb[3], mk[3];
        for (int x = 0; x < 3; ++x) {
            mb[x] = x == ax ? cb : 0;
            mk[x] = x == ax ? ck : 0;
            nb[x] = la[x] + lb[x] + (mb[x] ? 1 : 0);
            nk[x] = lc[x] + ld[x] + (mk[x] ? 1 : 0);
        }
        double val = 0.0;
        for (int t = 0; t <= nb[0]; ++t) {
            const double e0 = tb[0].c(la[0], lb[0], t, mb[0], P.a, P.b);
            if (e0 == 0.0) continue;
            for (int u = 0; u <= nb[1]; ++u) {
                const double e1 = e0 * tb[1].c(la[1], lb[1], u, mb[1], P.a, P.b);
                if (e1 == 0.0) continue;
                for (int v = 0; v <= nb[2]; ++v) {
                    const double eb = e1 * tb[2].c(la[2], lb[2], v, mb[2], P.a, P.b);
                    if (eb == 0.0) continue;
                    double inner = 0.0;
                    for (int tau = 0; tau <= nk[0]; ++tau) {
                        const double k0 = tk[0].c(lc[0], ld[0], tau, mk[0], Q.a, Q.b);
                        for (int nu = 0; nu <= nk[1]; ++nu) {
                            const double k1 = k0 * tk[1].c(lc[1], ld[1], nu, mk[1], Q.a, Q.b);
                            for (int phi = 0; phi <= nk[2]; ++phi) {
                                const double kk = k1 * tk[2].c(lc[2], ld[2], phi, mk[2], Q.a, Q.b);
                                const double sg = ((tau + nu + phi) & 1) ? -kk : kk;
                                inner = fma(sg, R[hidx(t + tau, u + nu, v + phi)], inner);
                            }
                        }
                    }
                    val = fma(eb, inner, val);
                }
            }
        }
        out[dir] = fma(val, pref, out[dir]);
    }
}

__device__ inline void tri_decode_g(int64_t idx, int64_t* r, int64_t* c)
{
    int64_t x = (int64_t)((sqrt(8.0 * (double)idx + 1.0) - 1.0) * 0.5);
    while (x * (x + 1) / 2 > idx) --x;
    while ((x + 1) * (x + 2) / 2 <= idx) ++x;
    *r = x;
    *c = idx - x * (x + 1) / 2;
}

// Two-electron part: one wavefront per canonical quartet i>=j, k>=l, ij>=kl
// (forces.py:62-80), its primitive quartets spread over the lanes and summed
// by a wavefront reduction; the workgroup sums the quartets' contributions
// per atom in LDS and adds them to grad once.
__global__ void __launch_bounds__(256) grad_eri_kernel(int N, const BFDesc* __restrict__ bfs,
                                                       const double* __restrict__ pexp,
                                                       const double* __restrict__ pw,
                                                       const double* __restrict__ boys,
                                                       const int* __restrict__ bf_atom, int natom,
                                                       const double* __restrict__ P, double* grad)
{
    extern __shared__ double gl[];   // 3 * natom
    for (int i = threadIdx.x; i < 3 * natom; i += blockDim.x) gl[i] = 0.0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t npair = (int64_t)N * (N + 1) / 2;
    const int64_t total = npair * (npair + 1) / 2;
    const size_t n = (size_t)N;
    const int64_t wave0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwave = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (int64_t idx = wave0; idx < total; idx += nwave) {   // uniform across the wavefront
        int64_t ij, kl, i, j, k, l;
        tri_decode_g(idx, &ij, &kl);
        tri_decode_g(ij, &i, &j);
        tri_decode_g(kl, &k, &l);
        // density weight of the quartet's distinct positions
        const int64_t pm[8][4] = {{i, j, k, l}, {k, l, i, j}, {j, i, l, k}, {l, k, j, i},
                                  {j, i, k, l}, {l, k, i, j}, {i, j, l, k}, {k, l, j, i}};
        double wgt = 0.0;
        for (int s = 0; s < 8; ++s) {
            bool dup = false;
            for (int r = 0; r < s && !dup; ++r)
                dup = pm[r][0] == pm[s][0] && pm[r][1] == pm[s][1] && pm[r][2] == pm[s][2] && pm[r][3] == pm[s][3];
            if (dup) continue;
            const int64_t a = pm[s][0], b = pm[s][1], c = pm[s][2], d = pm[s][3];
            wgt += 2.0 * P[b * n + a] * P[d * n + c] - P[c * n + a] * P[b * n + d];
        }
        if (wgt == 0.0) continue;
        const BFDesc fa = bfs[i], fb = bfs[j], fc = bfs[k], fd = bfs[l];
        const int la[3] = {fa.l, fa.m, fa.n}, lb[3] = {fb.l, fb.m, fb.n};
        const int lc[3] = {fc.l, fc.m, fc.n}, ld[3] = {fd.l, fd.m, fd.n};
        double g[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        const int nab = fa.np * fb.np, ncd = fc.np * fd.np;
        GPair Pp, Qp;
        for (int q = lane; q < nab * ncd; q += 64) {
            const int pab = q / ncd, pcd = q - pab * ncd;
            gpair(fa, fb, pab / fb.np, pab % fb.np, pexp, pw, Pp);
            gpair(fc, fd, pcd / fd.np, pcd % fd.np, pexp, pw, Qp);
            prim_quartet_grad(la, lb, lc, ld, Pp, Qp, boys, g);
        }
        for (int off = 32; off > 0; off >>= 1)
            for (int d = 0; d < 9; ++d) g[d] += __shfl_xor(g[d], off);
        if (lane == 0) {
            const int at[4] = {bf_atom[i], bf_atom[j], bf_atom[k], bf_atom[l]};
            for (int x = 0; x < 3; ++x) {
                const double dA = g[x], dB = g[3 + x], dC = g[6 + x];
                atomicAdd(&gl[3 * at[0] + x], wgt * dA);
                atomicAdd(&gl[3 * at[1] + x], wgt * dB);
                atomicAdd(&gl[3 * at[2] + x], wgt * dC);
                atomicAdd(&gl[3 * at[3] + x], -wgt * (dA + dB + dC));
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 3 * natom; i += blockDim.x)
        if (gl[i] != 0.0) atomicAdd(&grad[i], gl[i]);
}

// One-electron part: one wavefront per basis-function pair i >= j; a lane
// item is a primitive pair with a share of the nuclei (every G-th), as in
// the one-electron integrals.  For centre A (function i) and B (function j)
// along each axis: the overlap and kinetic derivatives (overlapX,
// kineticX) and the nuclear attraction of every nucleus with a
// differentiated function (nuclear_attractionXb); for each nucleus C the
// derivative of its operator (nuclear_attractionXa), added to C's gradient.
__global__ void __launch_bounds__(256) grad_one_electron_kernel(int nbf, const BFDesc* __restrict__ bfs,
                                                                const double* __restrict__ pexp,
                                                                const double* __restrict__ pw, int natom,
                                                                const double* __restrict__ atoms,
                                                                const double* __restrict__ boys,
                                                                const int* __restrict__ bf_atom,
                                                                const double* __restrict__ P,
                                                                const double* __restrict__ W, double* grad)
{
    const int64_t idx = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    const int64_t npair = (int64_t)nbf * (nbf + 1) / 2;
    if (idx >= npair) return;   // uniform across the wavefront
    int64_t ii, jj;
    tri_decode_g(idx, &ii, &jj);
    const int i = (int)ii, j = (int)jj;
    const BFDesc a = bfs[i], b = bfs[j];
    const double A[3] = {a.x, a.y, a.z}, B[3] = {b.x, b.y, b.z};
    const int l1[3] = {a.l, a.m, a.n}, l2[3] = {b.l, b.m, b.n};
    const double f = (i == j) ? 1.0 : 2.0;
    const double pij = 2.0 * f * P[(size_t)i * nbf + j];
    const double wij = 2.0 * f * W[(size_t)i * nbf + j];
    double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0};
    const int npp = a.np * b.np;
    const int G = npp >= 64 ? 1 : 64 / npp;
    const int nitem = npp * G;
    for (int it = lane; it < nitem; it += 64) {
        const int ipp = it % npp, g = it / npp;
        const int ia = ipp / b.np, ib = ipp % b.np;
        const double ea = pexp[a.p0 + ia], eb = pexp[b.p0 + ib];
        const double p = ea + eb;
        const double w = pw[a.p0 + ia] * pw[b.p0 + ib];
        double Pc[3], kab = 1.0;
        double E[3][GONE_TAB];
        Tab1 tb[3];
        for (int x = 0; x < 3; ++x) {
            Pc[x] = (ea * A[x] + eb * B[x]) / p;
            kab *= exp(-ea * eb / p * (A[x] - B[x]) * (A[x] - B[x]));
            etab_rt(l1[x] + 1, l2[x] + 3, 0.5 / p, Pc[x] - A[x], Pc[x] - B[x], E[x]);
            tb[x] = Tab1{E[x], l1[x] + 1, l2[x] + 3};
        }
        if (g == 0) {
            // overlap and kinetic derivatives (cython/grad.pyx:352-507)
            const double pre = pow(3.141592653589793238462643383279 / p, 1.5) * kab * w;
            for (int ctr = 1; ctr <= 2; ++ctr)
                for (int ax = 0; ax < 3; ++ax) {
                    double S0[3], Tk[3];
                    for (int x = 0; x < 3; ++x) {
                        const int m = x == ax ? ctr : 0;
                        const double jq = (double)l2[x];
                        S0[x] = tb[x].c(l1[x], l2[x], 0, m, ea, eb);
                        Tk[x] = (2.0 * jq + 1.0) * eb * tb[x].c(l1[x], l2[x], 0, m, ea, eb)
                              - 2.0 * eb * eb * tb[x].c(l1[x], l2[x] + 2, 0, m, ea, eb)
                              - 0.5 * jq * (jq - 1.0) * (l2[x] >= 2 ? tb[x].c(l1[x], l2[x] - 2, 0, m, ea, eb) : 0.0);
                    }
                    const double ds = S0[0] * S0[1] * S0[2] * pre;
                    const double dt = (Tk[0] * S0[1] * S0[2] + Tk[1] * S0[0] * S0[2] + Tk[2] * S0[0] * S0[1]) * pre;
                    double& gc = ctr == 1 ? gA[ax] : gB[ax];
                    gc += pij * dt - wij * ds;
                }
        }
        // nuclear attraction (cython/grad.pyx:509-)
        const int Lv = l1[0] + l2[0] + l1[1] + l2[1] + l1[2] + l2[2] + 1;
        const double vpre = 2.0 * 3.141592653589793238462643383279 / p * kab * w;
        for (int at = g; at < natom; at += G) {
            const double* nuc = atoms + 4 * at;
            const double Z = nuc[0];
            const double X = Pc[0] - nuc[1], Y = Pc[1] - nuc[2], Wd = Pc[2] - nuc[3];
            double F[2 * MAX_L + 2];
            boys_runtime(Lv, p * (X * X + Y * Y + Wd * Wd), boys, F);
            double sc = 1.0;
            for (int m = 0; m <= Lv; ++m) { F[m] *= sc; sc *= -2.0 * p; }
            double R[nherm(2 * MAX_L + 1)];
            hermite_R_rt(Lv, X, Y, Wd, F, R);
            double opd[3] = {0, 0, 0};
            for (int ctr = 1; ctr <= 2; ++ctr)
                for (int ax = 0; ax < 3; ++ax) {
                    double val = 0.0;
                    const int m0 = ax == 0 ? ctr : 0, m1 = ax == 1 ? ctr : 0, m2 = ax == 2 ? ctr : 0;
                    for (int t = 0; t <= l1[0] + l2[0] + (m0 ? 1 : 0); ++t)
                        for (int u = 0; u <= l1[1] + l2[1] + (m1 ? 1 : 0); ++u)
                            for (int v = 0; v <= l1[2] + l2[2] + (m2 ? 1 : 0); ++v)
                                val += tb[0].c(l1[0], l2[0], t, m0, ea, eb) * tb[1].c(l1[1], l2[1], u, m1, ea, eb)
                                     * tb[2].c(l1[2], l2[2], v, m2, ea, eb) * R[hidx(t, u, v)];
                    double& gc = ctr == 1 ? gA[ax] : gB[ax];
                    gc += pij * (-Z) * val * vpre;
                }
            for (int t = 0; t <= l1[0] + l2[0]; ++t)
                for (int u = 0; u <= l1[1] + l2[1]; ++u)
                    for (int v = 0; v <= l1[2] + l2[2]; ++v) {
                        const double e3 = tb[0].e(l1[0], l2[0], t) * tb[1].e(l1[1], l2[1], u)
                                        * tb[2].e(l1[2], l2[2], v);
                        opd[0] -= e3 * R[hidx(t + 1, u, v)];
                        opd[1] -= e3 * R[hidx(t, u + 1, v)];
                        opd[2] -= e3 * R[hidx(t, u, v + 1)];
                    }
            for (int x = 0; x < 3; ++x) atomicAdd(&grad[3 * at + x], pij * (-Z) * opd[x] * vpre);
        }
    }
    for (int off = 32; off > 0; off >>= 1)
        for (int x = 0; x < 3; ++x) {
            gA[x] += __shfl_xor(gA[x], off);
            gB[x] += __shfl_xor(gB[x], off);
        }
    if (lane != 0) return;
    for (int x = 0; x < 3; ++x) {
        atomicAdd(&grad[3 * bf_atom[i] + x], gA[x]);
        atomicAdd(&grad[3 * bf_atom[j] + x], gB[x]);
    }
}

// ---------------------------------------------------------------------------
// One-electron part by shell pair, compile-time pair classes: one wavefront
// per pair (a, b), l_a >= l_b; a lane item is a primitive pair with every
// G-th nucleus.  With w_ab = 2 P_ab times the pair's degeneracy, the pair's
// weights enter the Hermite space first, D_k = sum_ab w_ab E^{ab}_k and
// DR_x,k = sum_ab w_ab dE^{ab}_k/dR_x (R = A - B), so that a nucleus costs
// one R_tuv table of order l_a + l_b + 1 and 6 H(l_a + l_b) products:
//   d/dP = sum_k D_k R_{k+x},  A: (a/p) d/dP + d/dR,  B: (b/p) d/dP - d/dR,
//   the nucleus: -d/dP.
// Overlap and kinetic energy need 1-D overlaps only, and d/dB = -d/dA.
// Bound by FP64 latency; the per-function kernel, its tables in scratch,
// took 1182 us at (H2O)4 6-31G.
// ---------------------------------------------------------------------------
template <int LA, int LB>
__global__ void __launch_bounds__(256) grad_onee_pair_kernel(OneeArgs A, const int2* __restrict__ list, int npairs,
                                                             const int* __restrict__ bf_atom,
                                                             const double* __restrict__ P,
                                                             const double* __restrict__ W, double* grad)
{
    constexpr int NA = ncart(LA), NB = ncart(LB), NAB = NA * NB, L = LA + LB, H = nherm(L), NT = L + 2;
    const int wid = (int)(((size_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const int lane = threadIdx.x & 63;
    if (wid >= npairs) return;   // uniform across the wavefront
    double* g = grad + (size_t)(wid % GRAD_REPLICAS) * 3 * A.natom;
    const int2 pr = list[wid];
    const OneeShell a = A.shells[pr.x], b = A.shells[pr.y];
    const double Ac[3] = {a.x, a.y, a.z}, Bc[3] = {b.x, b.y, b.z};
    const double AB2 = (a.x - b.x) * (a.x - b.x) + (a.y - b.y) * (a.y - b.y) + (a.z - b.z) * (a.z - b.z);
    const double deg = pr.x == pr.y ? 1.0 : 2.0;
    const size_t n = (size_t)A.nbf;
    const int npp = a.np * b.np;
    int G = npp >= 64 ? 1 : 64 / npp;
    if (G > A.natom) G = A.natom;
    // weight of component pair (ca, cb) in M (the lower triangle counts)
    auto wgt = [&](const double* __restrict__ M, int ca, int cb) {
        const size_t i = (size_t)a.bf0 + ca, j = (size_t)b.bf0 + cb;
        return 2.0 * deg * A.gcomp[i] * A.gcomp[j] * M[(i > j ? i : j) * n + (i > j ? j : i)];
    };
    double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0};
    for (int it = lane; it < npp * G; it += 64) {
        const int ipp = it % npp, grp = it / npp;
        const int ia = ipp / b.np, ib = ipp - ia * b.np;
        const double ea = A.exps[a.p0 + ia], eb = A.exps[b.p0 + ib];
        const double p = ea + eb, ip = 1.0 / p;
        const double w = A.wts[a.p0 + ia] * A.wts[b.p0 + ib] * exp(-ea * eb * ip * AB2);
        const double Pc[3] = {(ea * a.x + eb * b.x) * ip, (ea * a.y + eb * b.y) * ip, (ea * a.z + eb * b.z) * ip};
        if (grp == 0) {
            // overlap and kinetic energy (cython/grad.pyx:352-507) from the 1-D
            // overlaps s_ij = E^{ij}_0: s_{i+1,j} = PA s_ij + (i s_{i-1,j} + j s_{i,j-1}) / 2p
            constexpr int SJ = LB + 3;
            double s[3][(LA + 2) * SJ];
            const double h = 0.5 * ip;
            sfor<3>([&](auto xx) {
                constexpr int x = decltype(xx)::value;
                const double pa = Pc[x] - Ac[x], pb = Pc[x] - Bc[x];
                s[x][0] = 1.0;
                sfor<SJ - 1>([&](auto jj) {
                    constexpr int j = decltype(jj)::value;
                    double v = pb * s[x][j];
                    if constexpr (j > 0) v = fma((double)j * h, s[x][j - 1], v);
                    s[x][j + 1] = v;
                });
                sfor<LA + 1>([&](auto ii) {
                    sfor<SJ>([&](auto jj) {
                        constexpr int i = decltype(ii)::value, j = decltype(jj)::value;
                        double v = pa * s[x][i * SJ + j];
                        if constexpr (i > 0) v = fma((double)i * h, s[x][(i - 1) * SJ + j], v);
                        if constexpr (j > 0) v = fma((double)j * h, s[x][i * SJ + j - 1], v);
                        s[x][(i + 1) * SJ + j] = v;
                    });
                });
            });
            const double pre = 3.141592653589793238462643383279 * ip * sqrt(3.141592653589793238462643383279 * ip) * w;
            sfor<NAB>([&](auto kk) {
                constexpr int k = decltype(kk)::value, ca = k / NB, cb = k % NB;
                constexpr int li[3] = {comp_lx(LA, ca), comp_ly(LA, ca), comp_lz(LA, ca)};
                constexpr int lj[3] = {comp_lx(LB, cb), comp_ly(LB, cb), comp_lz(LB, cb)};
                const double wp = wgt(P, ca, cb) * pre, ws = wgt(W, ca, cb) * pre;
                double S0[3], S1[3], T0[3], T1[3];   // plain and d/dA
                sfor<3>([&](auto xx) {
                    constexpr int x = decltype(xx)::value, i = li[x], j = lj[x];
                    auto kin = [&](auto i_) {   // (2j+1) b s_ij - 2 b^2 s_{i,j+2} - j (j-1)/2 s_{i,j-2}
                        constexpr int q = decltype(i_)::value;
                        double v = (2.0 * j + 1.0) * eb * s[x][q * SJ + j] - 2.0 * eb * eb * s[x][q * SJ + j + 2];
                        if constexpr (j >= 2) v -= 0.5 * j * (j - 1.0) * s[x][q * SJ + j - 2];
                        return v;
                    };
                    S0[x] = s[x][i * SJ + j];
                    T0[x] = kin(std::integral_constant<int, i>{});
                    S1[x] = 2.0 * ea * s[x][(i + 1) * SJ + j];
                    T1[x] = 2.0 * ea * kin(std::integral_constant<int, i + 1>{});
                    if constexpr (i > 0) {
                        S1[x] -= (double)i * s[x][(i - 1) * SJ + j];
                        T1[x] -= (double)i * kin(std::integral_constant<int, i - 1>{});
                    }
                });
                sfor<3>([&](auto xx) {
                    constexpr int x = decltype(xx)::value, y = (x + 1) % 3, z = (x + 2) % 3;
                    const double dt = T1[x] * S0[y] * S0[z] + S1[x] * (T0[y] * S0[z] + S0[y] * T0[z]);
                    const double v = wp * dt - ws * S1[x] * S0[y] * S0[z];
                    gA[x] += v;
                    gB[x] -= v;
                });
            });
        }
        // nuclear attraction (cython/grad.pyx:509-)
        double D[H], DR[3][H];
        {
            double e0[3][(LA + 1) * (LB + 1) * (L + 1)], e1[3][(LA + 1) * (LB + 1) * (L + 1)];
            sfor<3>([&](auto xx) {
                constexpr int x = decltype(xx)::value;
                double E[(LA + 2) * (LB + 1) * NT];
                hermite_E<LA + 1, LB, 1>(0.5 * ip, Pc[x] - Ac[x], Pc[x] - Bc[x], E);
                sfor<LA + 1>([&](auto ii) {
                    sfor<LB + 1>([&](auto jj) {
                        constexpr int i = decltype(ii)::value, j = decltype(jj)::value;
                        sfor<i + j + 1>([&](auto tt) {
                            constexpr int t = decltype(tt)::value;
                            auto e = [&](int i_, int k) { return E[(i_ * (LB + 1) + j) * NT + k]; };
                            double dv = 2.0 * ea * e(i + 1, t);
                            if constexpr (i > 0) dv -= (double)i * e(i - 1, t);
                            if constexpr (t > 0) dv -= ea * ip * e(i, t - 1);
                            e0[x][(i * (LB + 1) + j) * (L + 1) + t] = e(i, t);
                            e1[x][(i * (LB + 1) + j) * (L + 1) + t] = dv;
                        });
                    });
                });
            });
            sfor<H>([&](auto k) { D[k] = DR[0][k] = DR[1][k] = DR[2][k] = 0.0; });
            sfor<NAB>([&](auto kk) {
                constexpr int k = decltype(kk)::value, ca = k / NB, cb = k % NB;
                constexpr int ix = comp_lx(LA, ca), iy = comp_ly(LA, ca), iz = comp_lz(LA, ca);
                constexpr int jx = comp_lx(LB, cb), jy = comp_ly(LB, cb), jz = comp_lz(LB, cb);
                constexpr int ox = (ix * (LB + 1) + jx) * (L + 1), oy = (iy * (LB + 1) + jy) * (L + 1),
                              oz = (iz * (LB + 1) + jz) * (L + 1);
                const double wp = wgt(P, ca, cb);
                sfor<ix + jx + 1>([&](auto t_) {
                    constexpr int t = decltype(t_)::value;
                    sfor<iy + jy + 1>([&](auto u_) {
                        constexpr int u = decltype(u_)::value;
                        sfor<iz + jz + 1>([&](auto v_) {
                            constexpr int v = decltype(v_)::value, m = hidx(t, u, v);
                            const double x0 = wp * e0[0][ox + t], yz = e0[1][oy + u] * e0[2][oz + v];
                            D[m] = fma(x0, yz, D[m]);
                            DR[0][m] = fma(wp * e1[0][ox + t], yz, DR[0][m]);
                            DR[1][m] = fma(x0 * e1[1][oy + u], e0[2][oz + v], DR[1][m]);
                            DR[2][m] = fma(x0 * e0[1][oy + u], e1[2][oz + v], DR[2][m]);
                        });
                    });
                });
            });
        }
        const double vpre = -2.0 * 3.141592653589793238462643383279 * ip * w;
        for (int at = grp; at < A.natom; at += G) {
            const double* nuc = A.atoms + 4 * (size_t)at;
            const double X = Pc[0] - nuc[1], Y = Pc[1] - nuc[2], Z = Pc[2] - nuc[3];
            double F[L + 2];
            boys_seeds<L + 1, double>(p * (X * X + Y * Y + Z * Z), p, nuc[0] * vpre, A.boys + (size_t)(L + 1) * BOYS_NT,
                                      F);
            double R[nherm(L + 1)];
            hermite_R<L + 1, double>(X, Y, Z, F, R);
            double gP[3] = {0, 0, 0}, gR[3] = {0, 0, 0};
            sfor<H>([&](auto kk) {
                constexpr int k = decltype(kk)::value;
                constexpr Herm3 h = hdecode(k);
                gP[0] = fma(D[k], R[hidx(h.t + 1, h.u, h.v)], gP[0]);
                gP[1] = fma(D[k], R[hidx(h.t, h.u + 1, h.v)], gP[1]);
                gP[2] = fma(D[k], R[hidx(h.t, h.u, h.v + 1)], gP[2]);
                sfor<3>([&](auto x) { gR[x] = fma(DR[x][k], R[k], gR[x]); });
            });
            sfor<3>([&](auto x) {
                gA[x] += fma(ea * ip, gP[x], gR[x]);
                gB[x] += fma(eb * ip, gP[x], -gR[x]);
                atomicAdd(&g[3 * at + x], -gP[x]);
            });
        }
    }
    for (int off = 32; off > 0; off >>= 1)
        sfor<3>([&](auto x) {
            gA[x] += __shfl_xor(gA[x], off);
            gB[x] += __shfl_xor(gB[x], off);
        });
    if (lane != 0) return;
    const int ta = bf_atom[a.bf0], tb = bf_atom[b.bf0];
    sfor<3>([&](auto x) {
        atomicAdd(&g[3 * ta + x], gA[x]);
        atomicAdd(&g[3 * tb + x], gB[x]);
    });
}

// out[3a + x] = sum of the replicas, plus the nuclear repulsion term
// -sum_b Z_a Z_b (r_a - r_b)_x / R^3 (mmd/forces.py:52-60; coinciding nuclei
// are left out as there) when nuc is given
__global__ void grad_sum_kernel(int natom, int nrep, const double* __restrict__ rep, const double* __restrict__ nuc,
                                double* __restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, n = 3 * natom;
    if (i >= n) return;
    double s = 0.0;
    for (int r = 0; r < nrep; ++r) s += rep[(size_t)r * n + i];
    if (nuc) {
        const int a = i / 3, x = i - 3 * a;
        double v = 0.0;
        for (int b = 0; b < natom; ++b) {
            const double dx = nuc[4 * a + 1] - nuc[4 * b + 1], dy = nuc[4 * a + 2] - nuc[4 * b + 2],
                         dz = nuc[4 * a + 3] - nuc[4 * b + 3];
            const double r2 = dx * dx + dy * dy + dz * dz, r = sqrt(r2);
            if (r <= 1e-8) continue;
            v -= (x == 0 ? dx : (x == 1 ? dy : dz)) * nuc[4 * a] * nuc[4 * b] / (r2 * r);
        }
        s += v;
    }
    out[i] = s;
}

template <int LA, int LB>
hipError_t launch_grad_onee_pc(const OneeArgs& A, const int2* list, int n, const int* bf_atom, const double* P,
                               const double* W, double* grad, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL((grad_onee_pair_kernel<LA, LB>), dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st, A, list, n,
                       bf_atom, P, W, grad);
    return hipGetLastError();
}

}  // namespace

#define MMD_GRAD_CLASSES(X)                                                                              \
    X(0, 0, 0, 0) X(1, 0, 0, 0) X(1, 0, 1, 0) X(1, 1, 0, 0) X(1, 1, 1, 0) X(1, 1, 1, 1) X(2, 0, 0, 0)   \
    X(2, 0, 1, 0) X(2, 0, 1, 1) X(2, 0, 2, 0) X(2, 1, 0, 0) X(2, 1, 1, 0) X(2, 1, 1, 1) X(2, 1, 2, 0)   \
    X(2, 1, 2, 1) X(2, 2, 0, 0) X(2, 2, 1, 0) X(2, 2, 1, 1) X(2, 2, 2, 0) X(2, 2, 2, 1) X(2, 2, 2, 2)
#define DECL(a, b, c, d) \
    hipError_t grad_class_launch_##a##b##c##d(const GradArgs& A, const GradClass& C, hipStream_t st);
MMD_GRAD_CLASSES(DECL)
#undef DECL

hipError_t launch_grad_class(int qc, const GradArgs& A, const GradClass& C, hipStream_t st)
{
    int la, lb, lc, ld;
    qclass_decode(qc, &la, &lb, &lc, &ld);
#define CASE(a, b, c, d) \
    if (la == a && lb == b && lc == c && ld == d) return grad_class_launch_##a##b##c##d(A, C, st);
    MMD_GRAD_CLASSES(CASE)
#undef CASE
    return hipErrorInvalidValue;
}

hipError_t launch_grad_onee(int pc, const OneeArgs& A, const int2* list, int n, const int* bf_atom, const double* P,
                            const double* W, double* grad, hipStream_t st)
{
    switch (pc) {
    case 0: return launch_grad_onee_pc<0, 0>(A, list, n, bf_atom, P, W, grad, st);
    case 1: return launch_grad_onee_pc<1, 0>(A, list, n, bf_atom, P, W, grad, st);
    case 2: return launch_grad_onee_pc<1, 1>(A, list, n, bf_atom, P, W, grad, st);
    case 3: return launch_grad_onee_pc<2, 0>(A, list, n, bf_atom, P, W, grad, st);
    case 4: return launch_grad_onee_pc<2, 1>(A, list, n, bf_atom, P, W, grad, st);
    default: return launch_grad_onee_pc<2, 2>(A, list, n, bf_atom, P, W, grad, st);
    }
}

hipError_t launch_grad_sum(int natom, int nrep, const double* rep, const double* nuc, double* grad, hipStream_t st)
{
    hipLaunchKernelGGL(grad_sum_kernel, dim3((3 * natom + 63) / 64), dim3(64), 0, st, natom, nrep, rep, nuc, grad);
    return hipGetLastError();
}

hipError_t launch_rhf_gradient(int nbf, const BFDesc* bfs, const double* pexp, const double* pw, int natom,
                               const double* atoms, const double* boys, const int* bf_atom, const double* P,
                               const double* W, double* grad, hipStream_t st)
{
    if (nbf <= 0 || natom <= 0) return hipSuccess;
    const int64_t npair = (int64_t)nbf * (nbf + 1) / 2;
    hipLaunchKernelGGL(grad_one_electron_kernel, dim3((unsigned)((npair + 3) / 4)), dim3(256), 0, st, nbf, bfs, pexp,
                       pw, natom, atoms, boys, bf_atom, P, W, grad);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t total = npair * (npair + 1) / 2;   // quartets: one wavefront each, four per workgroup
    const int64_t grid = std::min<int64_t>(std::max<int64_t>(1, (total + 3) / 4), 16384);
    hipLaunchKernelGGL(grad_eri_kernel, dim3((unsigned)grid), dim3(256), sizeof(double) * 3 * natom, st, nbf, bfs,
                       pexp, pw, boys, bf_atom, natom, P, grad);
    return hipGetLastError();
}

}  // namespace mmd
