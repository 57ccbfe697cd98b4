#pragma once
// Two-electron part of the RHF nuclear gradient by shell-quartet class
// (la lb | lc ld): sum over quartets of Gamma_abcd d(ab|cd)/dX with
//   Gamma_abcd = deg (2 P_ab P_cd - (P_ac P_bd + P_ad P_bc) / 2)
// (mmd/forces.py:62-84: the density products of the positions a quartet
// fills in the derivative tensor, for a unique shell quartet of degeneracy
// deg).  The derivative of a function with respect to its centre raises and
// lowers its Cartesian power, 2a E^{i+1,j}_t - i E^{i-1,j}_t in Hermite form
// (cython/grad.pyx:97-103); what the two centres of a pair share is the
// derivative with respect to the product centre, which only raises the
// Hermite index, so that with R = A - B
//   d/dA = (a/p) d/dP + d/dR,   d/dB = (b/p) d/dP - d/dR,
//   dE^{ij}_t/dR = 2a E^{i+1,j}_t - i E^{i-1,j}_t - (a/p) E^{ij}_{t-1}
// and d/dQ = -d/dP.  Contracting Gamma with the expansions before the
// derivative integrals exist leaves one R_tuv table of order L + 1 and a few
// dot products per primitive quartet.
#include <hip/hip_runtime.h>
#include "mmd_device.h"
#include "mmd_grad.h"
#include "mmd_types.h"

namespace mmd {

constexpr double GRAD_TWO_PI_2_5 = 34.98683665524972497;   // 2 pi^{5/2}
constexpr int GRAD_BLOCK = 256;

// Density weight of component quartet (i j | k l) of a unique shell quartet,
// averaged over the eight index orders, so that a P that is not symmetric
// gives what the sum over all positions gives.
__device__ __forceinline__ double grad_gamma(const double* __restrict__ P, size_t n, int i, int j, int k, int l)
{
    const double pij = P[i * n + j] + P[j * n + i], pkl = P[k * n + l] + P[l * n + k];
    const double x = fma(P[k * n + i], P[j * n + l], P[i * n + k] * P[l * n + j])
                   + fma(P[k * n + j], P[i * n + l], P[l * n + i] * P[j * n + k]);
    return 0.5 * pij * pkl - 0.25 * x;
}

// Adds to the gradient of one atom: the workgroup's LDS array, or the global
// replica for molecules whose atoms do not fit there.
__device__ __forceinline__ void grad_add3(double* g, int atom, double x, double y, double z)
{
    atomicAdd(&g[3 * atom], x);
    atomicAdd(&g[3 * atom + 1], y);
    atomicAdd(&g[3 * atom + 2], z);
}

__device__ __forceinline__ double wave_sum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

template <int I, int N, class F>
__device__ __forceinline__ void grad_switch(int i, F&& f)
{
    if constexpr (I < N) {
        if (i == I) f(std::integral_constant<int, I>{});
        else grad_switch<I + 1, N>(i, f);
    }
}

template <int LA, int LB, int LC, int LD>
struct GradShape {
    static constexpr int LAB = LA + LB, LCD = LC + LD, L1 = LAB + LCD + 1;
    static constexpr int HCD = nherm(LCD);
    static constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
    static constexpr int NAB = NA * NB, NCD = NC * ND;
    // bra components per pass: the weights y and the integrals V of a pass
    // (2 H(cd) doubles per component) in up to 40 doubles beside R_tuv
    static constexpr int chunk()
    {
        int best = 1;
        for (int c = 1; c <= NAB; ++c)
            if (NAB % c == 0 && 2 * HCD * c <= 40) best = c;
        return best;
    }
    static constexpr int CH = chunk(), NCHUNK = NAB / CH;
    static constexpr int NT = LAB + 2;                        // Hermite indices of a differentiated pair
    static constexpr int ET = (LA + 1) * (LB + 1) * NT;       // one 1-D table
    static constexpr int REC = 8 + 9 * ET;                    // staged bra primitive: E, dE/dA, dE/dB per axis
};

// Lane-per-ket-primitive kernel.  A work unit is a slice of at most grad_pslice
// primitive pairs of one bra pair (staged in LDS with their plain and
// differentiated 1-D tables) against GRAD_BLOCK consecutive ket primitive
// pairs of the class; a lane takes one ket primitive pair and loops over
// the staged bra primitives.  Per bra primitive: Boys, R_tuv (order L + 1),
// the ket-contracted potentials q_tuv = sum_k y_k R_{tuv+k} (y: Gamma times
// the ket expansion, fixed per lane), their dot products with the bra's
// differentiated tables (the forces on A and B), and V_k = sum_tuv E_tuv
// R_{tuv+k} for the ket's own relative derivative after the loop.
// Bound by FP64 VALU issue (R_tuv and the dot products): lanes are whole
// primitive pairs, so contraction lengths do not unbalance a wavefront.
// (H2O)4 6-31G: the two-electron part took 119.2 ms with a wavefront per
// function quartet and its tables in scratch; here the six classes take 35
// to 90 us each, side by side.
template <int LA, int LB, int LC, int LD>
__global__ void __launch_bounds__(GRAD_BLOCK) grad_class_kernel(GradArgs A, GradClass C)
{
    using S = GradShape<LA, LB, LC, LD>;
    constexpr int NT = S::NT, ET = S::ET, HCD = S::HCD, L1 = S::L1;
    __shared__ double boys[BOYS_TAYLOR * BOYS_NT];
    __shared__ double bp[grad_pslice(pair_class(LA, LB)) * S::REC];
    extern __shared__ double gl[];   // 3 natom, when A.lds_atoms
    boys_stage_lds<L1, double>(boys, A.boys);
    double* rep = A.grad + (size_t)(blockIdx.x % GRAD_REPLICAS) * 3 * A.natom;
    double* g = A.lds_atoms ? gl : rep;
    if (A.lds_atoms)
        for (int i = threadIdx.x; i < 3 * A.natom; i += GRAD_BLOCK) gl[i] = 0.0;
    const size_t N = (size_t)A.N;
    const int64_t nunits = (int64_t)C.nslice * C.nkc;
    for (int64_t u = blockIdx.x; u < nunits; u += gridDim.x) {
        const int4 sl = C.slices[u / C.nkc];
        const int f0 = (int)(u % C.nkc) * GRAD_BLOCK;
        const int fend = C.tri ? sl.w : C.nflat;
        if (f0 >= fend) continue;              // uniform: the triangular classes' empty corner
        const ShellPair bra = A.pairs[sl.x];
        const int np = sl.z - sl.y;
        __syncthreads();
        for (int idx = threadIdx.x; idx < 3 * np; idx += GRAD_BLOCK) {
            const int ip = idx / 3, x = idx - 3 * ip;
            const int gi = bra.pp0 + sl.y + ip;
            const PrimPair* P = A.pp + gi;
            double* b = bp + ip * S::REC;
            const double ea = A.ppa[gi], eb = P->p - ea;
            if (x == 0) {
                b[0] = P->p;
                b[1] = GRAD_TWO_PI_2_5 * P->K * P->invp;
                b[2] = P->Px;
                b[3] = P->Py;
                b[4] = P->Pz;
            }
            const double PA = x == 0 ? P->PAx : (x == 1 ? P->PAy : P->PAz);
            const double PB = x == 0 ? P->PBx : (x == 1 ? P->PBy : P->PBz);
            double E[(LA + 2) * (LB + 2) * (LA + LB + 3)];
            hermite_E<LA + 1, LB + 1, 1>(P->inv2p, PA, PB, E);
            double* t = b + 8 + 3 * x * ET;
            sfor<LA + 1>([&](auto ii) {
                sfor<LB + 1>([&](auto jj) {
                    sfor<NT>([&](auto tt) {
                        constexpr int i = decltype(ii)::value, j = decltype(jj)::value, k = decltype(tt)::value;
                        auto e = [&](int i_, int j_) { return E[(i_ * (LB + 2) + j_) * (LA + LB + 3) + k]; };
                        constexpr int o = (i * (LB + 1) + j) * NT + k;
                        t[o] = e(i, j);
                        double dA = 2.0 * ea * e(i + 1, j), dB = 2.0 * eb * e(i, j + 1);
                        if constexpr (i > 0) dA -= (double)i * e(i - 1, j);
                        if constexpr (j > 0) dB -= (double)j * e(i, j - 1);
                        t[ET + o] = dA;
                        t[2 * ET + o] = dB;
                    });
                });
            });
        }
        __syncthreads();
        double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0};   // over the unit
        const int f = f0 + (int)threadIdx.x;
        if (f < fend) {
            const int2 kp = C.flat[f];
            const ShellPair ket = A.pairs[kp.x];
            const int qi = ket.pp0 + kp.y;
            const PrimPair* Q = A.pp + qi;
            const double Qp = Q->p, QK = Q->K * Q->invp, Qx = Q->Px, Qy = Q->Py, Qz = Q->Pz;
            const double qc = A.ppa[qi], cq = qc * Q->invp;
            const double deg = (bra.same ? 1.0 : 2.0) * (ket.same ? 1.0 : 2.0) * (sl.x == kp.x ? 1.0 : 2.0);
            constexpr int KT0 = LC + LD + 1, KE0 = (LC + 1) * (LD + 1) * KT0;
            constexpr int KT = LC + LD + 2, KE = (LC + 2) * (LD + 1) * KT;
            auto gam = [&](int a, int b, int c, int d) {
                const int i = bra.bfa + a, j = bra.bfb + b, k = ket.bfa + c, l = ket.bfb + d;
                return deg * A.gcomp[i] * A.gcomp[j] * A.gcomp[k] * A.gcomp[l] * grad_gamma(A.P, N, i, j, k, l);
            };
            double kA[3] = {0, 0, 0}, kB[3] = {0, 0, 0}, kR[3] = {0, 0, 0};   // over this ket primitive
            // one pass per chunk of bra components, as a loop over a switch, so
            // that nothing of one pass is kept in registers for the next
            for (int chunk = 0; chunk < S::NCHUNK; ++chunk) grad_switch<0, S::NCHUNK>(chunk, [&](auto ic) {
                constexpr int A0 = decltype(ic)::value * S::CH;
                double y[S::CH * HCD], V[S::CH * HCD];
                sfor<S::CH * HCD>([&](auto k) { y[k] = 0.0; V[k] = 0.0; });
                const double PC[3] = {Q->PAx, Q->PAy, Q->PAz}, PD[3] = {Q->PBx, Q->PBy, Q->PBz};
                double E0[3][KE0];   // ket tables, signed
                sfor<3>([&](auto x) { hermite_E<LC, LD, -1>(Q->inv2p, PC[x], PD[x], E0[x]); });
                sfor<S::CH>([&](auto ii) {
                    constexpr int ab = A0 + decltype(ii)::value;
                    sfor<S::NCD>([&](auto icd) {
                        constexpr int cd = decltype(icd)::value, c = cd / S::ND, d = cd % S::ND;
                        const double w = gam(ab / S::NB, ab % S::NB, c, d);
                        constexpr int cx = comp_lx(LC, c), cy = comp_ly(LC, c), cz = comp_lz(LC, c);
                        constexpr int dx = comp_lx(LD, d), dy = comp_ly(LD, d), dz = comp_lz(LD, d);
                        sfor<cx + dx + 1>([&](auto t_) {
                            constexpr int t = decltype(t_)::value;
                            sfor<cy + dy + 1>([&](auto u_) {
                                constexpr int u = decltype(u_)::value;
                                sfor<cz + dz + 1>([&](auto v_) {
                                    constexpr int v = decltype(v_)::value;
                                    const double e = E0[0][(cx * (LD + 1) + dx) * KT0 + t] * E0[1][(cy * (LD + 1) + dy) * KT0 + u]
                                                   * E0[2][(cz * (LD + 1) + dz) * KT0 + v];
                                    constexpr int k = decltype(ii)::value * HCD + hidx(t, u, v);
                                    y[k] = fma(w, e, y[k]);
                                });
                            });
                        });
                    });
                });
                for (int ip = 0; ip < np; ++ip) {
                    const double* b = bp + ip * S::REC;
                    const double Pp = b[0];
                    const double rs = rsqrt(Pp + Qp);
                    const double alpha = Pp * Qp * rs * rs;
                    const double X = b[2] - Qx, Y = b[3] - Qy, Z = b[4] - Qz;
                    double F[L1 + 1];
                    boys_seeds<L1, double>(alpha * (X * X + Y * Y + Z * Z), alpha, b[1] * QK * rs, boys, F);
                    double R[nherm(L1)];
                    hermite_R<L1, double>(X, Y, Z, F, R);
                    const double* T = b + 8;
                    sfor<S::CH>([&](auto ii) {
                        __builtin_amdgcn_sched_barrier(0);   // table reads stay with their component
                        constexpr int ab = A0 + decltype(ii)::value, a = ab / S::NB, bb = ab % S::NB;
                        constexpr int mx = comp_lx(LA, a) + comp_lx(LB, bb), my = comp_ly(LA, a) + comp_ly(LB, bb),
                                      mz = comp_lz(LA, a) + comp_lz(LB, bb);
                        constexpr int ox = (comp_lx(LA, a) * (LB + 1) + comp_lx(LB, bb)) * NT;
                        constexpr int oy = (comp_ly(LA, a) * (LB + 1) + comp_ly(LB, bb)) * NT + 3 * ET;
                        constexpr int oz = (comp_lz(LA, a) * (LB + 1) + comp_lz(LB, bb)) * NT + 6 * ET;
                        sfor<mx + 2>([&](auto t_) {
                            constexpr int t = decltype(t_)::value;
                            sfor<my + 2>([&](auto u_) {
                                constexpr int u = decltype(u_)::value;
                                sfor<mz + 2>([&](auto v_) {
                                    constexpr int v = decltype(v_)::value;
                                    constexpr int over = (t > mx) + (u > my) + (v > mz);
                                    if constexpr (over <= 1) {
                                        double q = 0.0;
                                        sfor<HCD>([&](auto k_) {
                                            constexpr Herm3 h = hdecode(decltype(k_)::value);
                                            q = fma(y[decltype(ii)::value * HCD + decltype(k_)::value],
                                                    R[hidx(t + h.t, u + h.u, v + h.v)], q);
                                        });
                                        if constexpr (u <= my && v <= mz) {
                                            const double s = T[oy + u] * T[oz + v] * q;
                                            kA[0] = fma(T[ox + ET + t], s, kA[0]);
                                            kB[0] = fma(T[ox + 2 * ET + t], s, kB[0]);
                                        }
                                        if constexpr (t <= mx && v <= mz) {
                                            const double s = T[ox + t] * T[oz + v] * q;
                                            kA[1] = fma(T[oy + ET + u], s, kA[1]);
                                            kB[1] = fma(T[oy + 2 * ET + u], s, kB[1]);
                                        }
                                        if constexpr (t <= mx && u <= my) {
                                            const double s = T[ox + t] * T[oy + u] * q;
                                            kA[2] = fma(T[oz + ET + v], s, kA[2]);
                                            kB[2] = fma(T[oz + 2 * ET + v], s, kB[2]);
                                        }
                                        if constexpr (over == 0) {
                                            const double e = T[ox + t] * T[oy + u] * T[oz + v];
                                            sfor<HCD>([&](auto k_) {
                                                constexpr Herm3 h = hdecode(decltype(k_)::value);
                                                constexpr int k = decltype(ii)::value * HCD + decltype(k_)::value;
                                                V[k] = fma(e, R[hidx(t + h.t, u + h.u, v + h.v)], V[k]);
                                            });
                                        }
                                    }
                                });
                            });
                        });
                    });
                }
                // relative derivative of the ket: sum Gamma dE^{cd}_k/dR_x V_k;
                // its tables to (lc + 1, ld) are made here, after the loop, so
                // that they do not hold registers through it
                asm volatile("" ::: "memory");   // P and the ket's data are read again
                const double PC2[3] = {Q->PAx, Q->PAy, Q->PAz}, PD2[3] = {Q->PBx, Q->PBy, Q->PBz};
                double Ek[3][KE];
                sfor<3>([&](auto x) { hermite_E<LC + 1, LD, 1>(Q->inv2p, PC2[x], PD2[x], Ek[x]); });
                sfor<S::NCD>([&](auto icd) {
                    constexpr int cd = decltype(icd)::value, c = cd / S::ND, d = cd % S::ND;
                    constexpr int cl[3] = {comp_lx(LC, c), comp_ly(LC, c), comp_lz(LC, c)};
                    constexpr int dl[3] = {comp_lx(LD, d), comp_ly(LD, d), comp_lz(LD, d)};
                    double VG[HCD];   // sum over the chunk's bra components of Gamma V
                    sfor<HCD>([&](auto k) { VG[k] = 0.0; });
                    sfor<S::CH>([&](auto ii) {
                        constexpr int ab = A0 + decltype(ii)::value;
                        const double w = gam(ab / S::NB, ab % S::NB, c, d);
                        sfor<HCD>([&](auto k) {
                            VG[k] = fma(w, V[decltype(ii)::value * HCD + decltype(k)::value], VG[k]);
                        });
                    });
                    // 1-D factors: plain and dE/dR, signed
                    double e0[3][KT], e1[3][KT];
                    sfor<3>([&](auto xx) {
                        constexpr int x = decltype(xx)::value;
                        sfor<cl[x] + dl[x] + 1>([&](auto tt) {
                            constexpr int t = decltype(tt)::value;
                            auto e = [&](int i, int j, int k) { return Ek[x][(i * (LD + 1) + j) * KT + k]; };
                            double dv = 2.0 * qc * e(cl[x] + 1, dl[x], t);
                            if constexpr (cl[x] > 0) dv -= (double)cl[x] * e(cl[x] - 1, dl[x], t);
                            if constexpr (t > 0) dv -= cq * e(cl[x], dl[x], t - 1);
                            e0[x][t] = (t & 1) ? -e(cl[x], dl[x], t) : e(cl[x], dl[x], t);
                            e1[x][t] = (t & 1) ? -dv : dv;
                        });
                    });
                    sfor<cl[0] + dl[0] + 1>([&](auto t_) {
                        constexpr int t = decltype(t_)::value;
                        sfor<cl[1] + dl[1] + 1>([&](auto u_) {
                            constexpr int u = decltype(u_)::value;
                            sfor<cl[2] + dl[2] + 1>([&](auto v_) {
                                constexpr int v = decltype(v_)::value;
                                const double s = VG[hidx(t, u, v)];
                                kR[0] = fma(e1[0][t] * e0[1][u] * e0[2][v], s, kR[0]);
                                kR[1] = fma(e0[0][t] * e1[1][u] * e0[2][v], s, kR[1]);
                                kR[2] = fma(e0[0][t] * e0[1][u] * e1[2][v], s, kR[2]);
                            });
                        });
                    });
                });
            });
            double gC[3], gD[3];
            sfor<3>([&](auto x) {
                const double gQ = -(kA[x] + kB[x]);   // d/dQ = -d/dP
                gC[x] = fma(cq, gQ, kR[x]);
                gD[x] = gQ - gC[x];
                gA[x] = kA[x];
                gB[x] = kB[x];
            });
            grad_add3(g, A.bf_atom[ket.bfa], gC[0], gC[1], gC[2]);
            grad_add3(g, A.bf_atom[ket.bfb], gD[0], gD[1], gD[2]);
        }
        sfor<3>([&](auto x) {
            gA[x] = wave_sum(gA[x]);
            gB[x] = wave_sum(gB[x]);
        });
        if ((threadIdx.x & 63) == 0) {
            grad_add3(g, A.bf_atom[bra.bfa], gA[0], gA[1], gA[2]);
            grad_add3(g, A.bf_atom[bra.bfb], gB[0], gB[1], gB[2]);
        }
    }
    if (A.lds_atoms) {
        __syncthreads();
        for (int i = threadIdx.x; i < 3 * A.natom; i += GRAD_BLOCK)
            if (gl[i] != 0.0) atomicAdd(&rep[i], gl[i]);
    }
}

// Workgroup-per-primitive-quartet kernel for the classes whose weights do
// not fit a lane (a bra with a d shell against (ds), (pp) and higher).  The
// quartet's Gamma, the dense bra expansion (plain and dE/dR per axis) and
// Gamma times the ket expansion (plain and per axis) lie in LDS; the threads
// share the Hermite pairs (k, k'), each of which meets R_{k+k'} and its
// three neighbours.  These classes are few quartets of short contractions
// (one (dd|dd) quartet in a water molecule), so the work of one primitive
// quartet is spread as wide as it goes: bound by LDS reads and the latency
// of the R recursion's L + 1 levels.  One water in cc-pVDZ: 12 to 40 us per
// class against 90 to 226 us with one wavefront per quartet and its ket
// primitives in turn (13.6 ms for the whole two-electron part with the
// per-function kernel).
template <int LA, int LB, int LC, int LD>
struct GradBlockShape {
    static constexpr int LAB = LA + LB, LCD = LC + LD, L1 = LAB + LCD + 1, HL = nherm(L1);
    static constexpr int NAB = ncart(LA) * ncart(LB), NCD = ncart(LC) * ncart(LD);
    static constexpr int HAB = nherm(LAB), HCD = nherm(LCD);
    static constexpr int TB = (LA + 1) * (LB + 1) * (LAB + 1), TK = (LC + 1) * (LD + 1) * (LCD + 1);
    static constexpr int DOUBLES = NAB * NCD + 4 * NAB * HAB + 4 * NAB * HCD + 2 * HL + 6 * TB + 6 * TK + L1 + 1;
    static constexpr int HM = HAB > HCD ? HAB : HCD;
    static constexpr size_t LDS = sizeof(double) * DOUBLES + sizeof(int) * (HL + NAB + NCD + HM);
};

// plain and d/dR 1-D tables of one primitive pair along one axis, signed by
// (-1)^t where SIGN < 0: e0, e1 [(i (LJ+1) + j) (LI+LJ+1) + t]
template <int LI, int LJ, int SIGN>
__device__ inline void grad_tables(double a, double ap, double inv2p, double PA, double PB, double* e0, double* e1)
{
    constexpr int NT = LI + LJ + 1, NX = LI + LJ + 2;
    double E[(LI + 2) * (LJ + 1) * NX];
    hermite_E<LI + 1, LJ, 1>(inv2p, PA, PB, E);
    sfor<LI + 1>([&](auto ii) {
        sfor<LJ + 1>([&](auto jj) {
            sfor<NT>([&](auto tt) {
                constexpr int i = decltype(ii)::value, j = decltype(jj)::value, t = decltype(tt)::value;
                auto e = [&](int i_, int j_, int k) { return E[(i_ * (LJ + 1) + j_) * NX + k]; };
                double p0 = 0.0, dv = 0.0;
                if constexpr (t <= i + j) {
                    p0 = e(i, j, t);
                    dv = 2.0 * a * e(i + 1, j, t);
                    if constexpr (i > 0) dv -= (double)i * e(i - 1, j, t);
                    if constexpr (t > 0) dv -= ap * e(i, j, t - 1);
                }
                constexpr bool neg = SIGN < 0 && (t & 1);
                e0[(i * (LJ + 1) + j) * NT + t] = neg ? -p0 : p0;
                e1[(i * (LJ + 1) + j) * NT + t] = neg ? -dv : dv;
            });
        });
    });
}

template <int LA, int LB, int LC, int LD>
__global__ void __launch_bounds__(GRAD_BLOCK) grad_block_kernel(GradArgs A, GradClass C)
{
    using S = GradBlockShape<LA, LB, LC, LD>;
    constexpr int NAB = S::NAB, NCD = S::NCD, HAB = S::HAB, HCD = S::HCD, HL = S::HL, L1 = S::L1;
    constexpr int NB = ncart(LB), ND = ncart(LD);
    constexpr int NTB = S::LAB + 1, NTK = S::LCD + 1;
    extern __shared__ double lds[];
    double* Gm = lds;                        // Gamma [ab][cd]
    double* Eb = Gm + NAB * NCD;             // [4][ab][k]
    double* Y = Eb + 4 * NAB * HAB;          // [4][ab][k']
    double* Rb = Y + 4 * NAB * HCD;          // two levels of R
    double* Tb = Rb + 2 * HL;                // [2][3][TB]
    double* Tk = Tb + 6 * S::TB;             // [2][3][TK]
    double* Fs = Tk + 6 * S::TK;
    int* rtab = reinterpret_cast<int*>(Fs + L1 + 1);
    // offsets of a component's three 1-D tables (8 bits each), and (t, u, v)
    // of a Hermite index (4 bits each)
    int* bofs = rtab + HL;
    int* kofs = bofs + NAB;
    int* htuv = kofs + NCD;
    const int tid = threadIdx.x;
    // R_tuv = X_dir R(i1) + c R(i2): dir | i1 << 2 | i2 << 10 | c << 18, i2 = 255 without the second term
    for (int k = tid; k < HL; k += GRAD_BLOCK) {
        const Herm3 h = hdecode(k);
        int dir = 0, i1 = 0, i2 = 255, c = 0;
        if (h.t > 0) {
            i1 = hidx(h.t - 1, h.u, h.v);
            if (h.t > 1) { i2 = hidx(h.t - 2, h.u, h.v); c = h.t - 1; }
        } else if (h.u > 0) {
            dir = 1;
            i1 = hidx(h.t, h.u - 1, h.v);
            if (h.u > 1) { i2 = hidx(h.t, h.u - 2, h.v); c = h.u - 1; }
        } else if (h.v > 0) {
            dir = 2;
            i1 = hidx(h.t, h.u, h.v - 1);
            if (h.v > 1) { i2 = hidx(h.t, h.u, h.v - 2); c = h.v - 1; }
        }
        rtab[k] = dir | (i1 << 2) | (i2 << 10) | (c << 18);
    }
    for (int e = tid; e < NAB; e += GRAD_BLOCK) {
        const int a = e / NB, b = e % NB;
        bofs[e] = ((comp_lx(LA, a) * (LB + 1) + comp_lx(LB, b)) * NTB)
                | ((S::TB + (comp_ly(LA, a) * (LB + 1) + comp_ly(LB, b)) * NTB) << 8)
                | ((2 * S::TB + (comp_lz(LA, a) * (LB + 1) + comp_lz(LB, b)) * NTB) << 16);
    }
    for (int e = tid; e < NCD; e += GRAD_BLOCK) {
        const int c = e / ND, d = e % ND;
        kofs[e] = ((comp_lx(LC, c) * (LD + 1) + comp_lx(LD, d)) * NTK)
                | ((S::TK + (comp_ly(LC, c) * (LD + 1) + comp_ly(LD, d)) * NTK) << 8)
                | ((2 * S::TK + (comp_lz(LC, c) * (LD + 1) + comp_lz(LD, d)) * NTK) << 16);
    }
    for (int e = tid; e < S::HM; e += GRAD_BLOCK) {
        const Herm3 h = hdecode(e);
        htuv[e] = h.t | (h.u << 4) | (h.v << 8);
    }
    double* rep = A.grad + (size_t)(blockIdx.x % GRAD_REPLICAS) * 3 * A.natom;
    const size_t N = (size_t)A.N;
    const int64_t nunits = (int64_t)C.nslice * C.nflat;   // slices of one primitive pair here
    for (int64_t u = blockIdx.x; u < nunits; u += gridDim.x) {
        const int4 sl = C.slices[u / C.nflat];
        const int f = (int)(u % C.nflat);
        if (C.tri && f >= sl.w) continue;      // uniform
        const int kq = C.flat[f].x;
        const ShellPair bra = A.pairs[sl.x], ket = A.pairs[kq];
        const int gi = bra.pp0 + sl.y;
        const PrimPair* P = A.pp + gi;
        const double ea = A.ppa[gi], ap = ea * P->invp;
        const int qi = ket.pp0 + C.flat[f].y;
        const PrimPair* Q = A.pp + qi;
        const double qc = A.ppa[qi], cq = qc * Q->invp;
        const double rs = rsqrt(P->p + Q->p);
        const double alpha = P->p * Q->p * rs * rs;
        const double X[3] = {P->Px - Q->Px, P->Py - Q->Py, P->Pz - Q->Pz};
        const double deg = (bra.same ? 1.0 : 2.0) * (ket.same ? 1.0 : 2.0) * (sl.x == kq ? 1.0 : 2.0);
        __syncthreads();
        for (int e = tid; e < NAB * NCD; e += GRAD_BLOCK) {
            const int ab = e / NCD, cd = e % NCD;
            const int i = bra.bfa + ab / NB, j = bra.bfb + ab % NB, k = ket.bfa + cd / ND, l = ket.bfb + cd % ND;
            Gm[e] = deg * A.gcomp[i] * A.gcomp[j] * A.gcomp[k] * A.gcomp[l] * grad_gamma(A.P, N, i, j, k, l);
        }
        if (tid < 3) {
            const int x = tid;
            grad_tables<LA, LB, 1>(ea, ap, P->inv2p, x == 0 ? P->PAx : (x == 1 ? P->PAy : P->PAz),
                                   x == 0 ? P->PBx : (x == 1 ? P->PBy : P->PBz), Tb + x * S::TB, Tb + (3 + x) * S::TB);
        } else if (tid >= 64 && tid < 67) {
            const int x = tid - 64;
            grad_tables<LC, LD, -1>(qc, cq, Q->inv2p, x == 0 ? Q->PAx : (x == 1 ? Q->PAy : Q->PAz),
                                    x == 0 ? Q->PBx : (x == 1 ? Q->PBy : Q->PBz), Tk + x * S::TK,
                                    Tk + (3 + x) * S::TK);
        } else if (tid == 128) {
            double F[L1 + 1];
            boys_runtime(L1, alpha * (X[0] * X[0] + X[1] * X[1] + X[2] * X[2]), A.boys, F);
            double s = GRAD_TWO_PI_2_5 * P->K * P->invp * Q->K * Q->invp * rs;
            for (int m = 0; m <= L1; ++m) {
                Fs[m] = s * F[m];
                s *= -2.0 * alpha;
            }
            Rb[(L1 & 1) * HL] = Fs[L1];
        }
        __syncthreads();
        for (int e = tid; e < NAB * HAB; e += GRAD_BLOCK) {
            const int o = bofs[e / HAB], h = htuv[e % HAB];
            const int i[3] = {(o & 255) + (h & 15), ((o >> 8) & 255) + ((h >> 4) & 15), (o >> 16) + (h >> 8)};
            double p0[3], p1[3];
            for (int x = 0; x < 3; ++x) {
                p0[x] = Tb[i[x]];       // zero for t > i + j
                p1[x] = Tb[3 * S::TB + i[x]];
            }
            Eb[e] = p0[0] * p0[1] * p0[2];
            Eb[NAB * HAB + e] = p1[0] * p0[1] * p0[2];
            Eb[2 * NAB * HAB + e] = p0[0] * p1[1] * p0[2];
            Eb[3 * NAB * HAB + e] = p0[0] * p0[1] * p1[2];
        }
        for (int e = tid; e < NAB * HCD; e += GRAD_BLOCK) {
            const int ab = e / HCD, h = htuv[e % HCD];
            const int t = h & 15, u = (h >> 4) & 15, v = h >> 8;
            double y[4] = {0, 0, 0, 0};
            for (int cd = 0; cd < NCD; ++cd) {
                const int o = kofs[cd];
                const int i[3] = {(o & 255) + t, ((o >> 8) & 255) + u, (o >> 16) + v};
                double p0[3], p1[3];
                for (int x = 0; x < 3; ++x) {
                    p0[x] = Tk[i[x]];
                    p1[x] = Tk[3 * S::TK + i[x]];
                }
                const double w = Gm[ab * NCD + cd];
                y[0] = fma(w, p0[0] * p0[1] * p0[2], y[0]);
                y[1] = fma(w, p1[0] * p0[1] * p0[2], y[1]);
                y[2] = fma(w, p0[0] * p1[1] * p0[2], y[2]);
                y[3] = fma(w, p0[0] * p0[1] * p1[2], y[3]);
            }
            for (int m = 0; m < 4; ++m) Y[m * NAB * HCD + e] = y[m];
        }
        for (int n = L1 - 1; n >= 0; --n) {
            const double* prev = Rb + ((n + 1) & 1) * HL;
            double* cur = Rb + (n & 1) * HL;
            for (int k = tid; k < nherm(L1 - n); k += GRAD_BLOCK) {
                double val = Fs[n];
                if (k > 0) {
                    const int e = rtab[k], i2 = (e >> 10) & 255, dir = e & 3;
                    val = (dir == 0 ? X[0] : (dir == 1 ? X[1] : X[2])) * prev[(e >> 2) & 255];
                    if (i2 != 255) val = fma((double)(e >> 18), prev[i2], val);
                }
                cur[k] = val;
            }
            __syncthreads();
        }
        const double* R = Rb;
        double gP[3] = {0, 0, 0}, gb[3] = {0, 0, 0}, gk[3] = {0, 0, 0};
        for (int e = tid; e < HAB * HCD; e += GRAD_BLOCK) {
            const int k = e / HCD, kk = e % HCD;
            const int h = htuv[k] + htuv[kk];
            double z = 0.0, zb[3] = {0, 0, 0}, zk[3] = {0, 0, 0};
            for (int ab = 0; ab < NAB; ++ab) {
                const double e0 = Eb[ab * HAB + k], y0 = Y[ab * HCD + kk];
                z = fma(e0, y0, z);
                for (int x = 0; x < 3; ++x) {
                    zb[x] = fma(Eb[(x + 1) * NAB * HAB + ab * HAB + k], y0, zb[x]);
                    zk[x] = fma(e0, Y[(x + 1) * NAB * HCD + ab * HCD + kk], zk[x]);
                }
            }
            const int t = h & 15, uu = (h >> 4) & 15, v = h >> 8;
            const double r = R[hidx(t, uu, v)];
            gP[0] = fma(z, R[hidx(t + 1, uu, v)], gP[0]);
            gP[1] = fma(z, R[hidx(t, uu + 1, v)], gP[1]);
            gP[2] = fma(z, R[hidx(t, uu, v + 1)], gP[2]);
            for (int x = 0; x < 3; ++x) {
                gb[x] = fma(zb[x], r, gb[x]);
                gk[x] = fma(zk[x], r, gk[x]);
            }
        }
        double gA[3], gB[3], gC[3], gD[3];
        for (int x = 0; x < 3; ++x) {
            const double p = wave_sum(gP[x]), b = wave_sum(gb[x]), k = wave_sum(gk[x]);
            gA[x] = fma(ap, p, b);
            gB[x] = fma(1.0 - ap, p, -b);
            gC[x] = fma(-cq, p, k);
            gD[x] = fma(cq - 1.0, p, -k);
        }
        if ((tid & 63) == 0) {
            grad_add3(rep, A.bf_atom[bra.bfa], gA[0], gA[1], gA[2]);
            grad_add3(rep, A.bf_atom[bra.bfb], gB[0], gB[1], gB[2]);
            grad_add3(rep, A.bf_atom[ket.bfa], gC[0], gC[1], gC[2]);
            grad_add3(rep, A.bf_atom[ket.bfb], gD[0], gD[1], gD[2]);
        }
    }
}

}  // namespace mmd
