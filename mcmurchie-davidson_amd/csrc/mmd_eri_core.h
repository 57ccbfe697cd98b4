#pragma once
// Contracted integrals of one shell quartet in registers, shared by the
// Fock-build row kernels (mmd_eri_impl.h) and the integral-block kernels
// (mmd_eri_block.h): class shapes and the primitive loops.
//
// Reference semantics: cython/twoe.pyx:52-94 (primitive ERI),
// cython/twoe.pyx:34-50 (contraction).
#include <hip/hip_runtime.h>
#include <type_traits>
#include <utility>
#include "mmd_device.h"
#include "mmd_types.h"

namespace mmd {

constexpr double TWO_PI_2_5 = 34.98683665524972497;   // 2 pi^{5/2}

// Largest divisor of nab whose chunk of bra components keeps the per-lane
// accumulators (ket Hermite intermediate + contracted block) within `limit`
// doubles.
__host__ __device__ constexpr int chunk_size(int nab, int hcd, int ncd, int limit)
{
    int best = 1;
    for (int c = 1; c <= nab; ++c)
        if (nab % c == 0 && (hcd + ncd) * c <= limit) best = c;
    return best;
}
constexpr int ACC_LIMIT = 40;
#ifndef MMD_IBUF_CAP
#define MMD_IBUF_CAP 2048
#endif
constexpr int IBUF_CAP = MMD_IBUF_CAP;     // doubles of the LDS integral buffer that set its batch size
constexpr int ACC_LIMIT_HIGH = 64;

template <int LA, int LB, int LC, int LD>
struct ClassShape {
    static constexpr int L = LA + LB + LC + LD;
    static constexpr int LAB = LA + LB, LCD = LC + LD;
    static constexpr int HCD = nherm(LCD);
    static constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
    static constexpr int NAB = NA * NB, NCD = NC * ND;
    // bra components per item: accumulators (ket Hermite + ket Cartesian
    // per component) up to ACC_LIMIT doubles, or ACC_LIMIT_HIGH for L >= 4,
    // whose R_tuv dominates the registers anyway and whose chunks each
    // recompute Boys and R
    static constexpr int CH = chunk_size(NAB, HCD, NCD, L >= 4 ? ACC_LIMIT_HIGH : ACC_LIMIT);
    static constexpr int NCHUNK = NAB / CH;
    static constexpr int NTB = LA + LB + 1, NTK = LC + LD + 1;
    static constexpr int EB = (LA + 1) * (LB + 1) * NTB;   // 1-D bra E table
    static constexpr int BPS = 8 + 3 * EB;                 // staged bra primitive stride (doubles)
    // Classes with few integrals per quartet (the heavily contracted low-L
    // ones) add the primitive-slice partials of a batch into an LDS buffer
    // and digest each quartet once; QB is their batch size (buffer <= 16 KB).
    static constexpr int NABCD = NAB * NCD;
    static constexpr bool IBUF = NABCD <= 36;
    // Items are (quartet, ket primitive slice) pairs, not whole quartets,
    // for the buffered classes and for the classes whose ket pairs are the
    // heavily contracted (ss) and (ps) pairs (up to 81 primitive pairs per
    // ket in cc-pVDZ): there a whole-ket lane would carry up to 81 primitive
    // quartets alone and set the length of its batch.  Unbuffered classes
    // digest each slice's partial block directly (the digestion is linear).
    // (pp|pp) is sliced too: its units hold few surviving kets in batches of
    // small molecules, and slices multiply its lane items (a 6-31G batch
    // pass measured 285 against 298 ms; (H2O)8 cc-pVDZ builds unchanged).
    // (ds|pp) likewise: a lane with a whole (pp) ket set the length of the build
    // of a small molecule ((H2O)3 6-31G* 98 us alone, 35 sliced; (H2O)8
    // cc-pVDZ 146 and 111; (H2O)16, where lanes abound, 300 and 354).
    static constexpr bool KSL = IBUF || (LC <= 1 && LD == 0) || (LA <= 1 && LC <= 1)
                             || (LA == 2 && LB == 0 && LC == 1 && LD == 1);
    // The other classes digest each (quartet, chunk) item; when a quartet
    // has several chunks, their ket-side Coulomb blocks are summed in an LDS
    // buffer per batch (KJ) and added to G once per quartet.
    static constexpr bool KJ = !IBUF && NCHUNK > 1;
    static constexpr int QB = IBUF ? (IBUF_CAP / NABCD >= 256 ? 256 : (IBUF_CAP / NABCD >= 128 ? 128 : 64))
                                   : (KJ ? (2048 / NCD >= 256 ? 256 : (2048 / NCD >= 128 ? 128 : 64)) : 256);
    static constexpr int IBUF_DOUBLES = IBUF ? QB * NABCD : 0;
    static constexpr int KJ_DOUBLES = KJ ? QB * NCD : 0;   // used when the launch has LDS for it
};

__device__ __forceinline__ double dmax6(double a, double b, double c, double d, double e, double f)
{
    return fmax(fmax(fmax(a, b), fmax(c, d)), fmax(e, f));
}

// ---------------------------------------------------------------------------
// One work item: a quartet, a chunk of its bra components, and a slice of its
// bra and ket primitive pairs (the contributions of the slices add up, and
// so do their digestions).  Outer loop: the lane's ket primitive pairs jq
// (global memory, indices of the primitive-pair table).  Inner loop: the bra primitive pairs staged in LDS (the
// same for every lane of the work unit).  Per inner step: Boys,
// R_tuv, and the bra contraction accumulated in the ket's Hermite space,
//   V_{tau nu phi}(ab) += sum_tuv E^{ab}_tuv R_{t+tau,u+nu,v+phi};
// per ket primitive: (ab|cd) += sum (-1)^{tau+nu+phi} E^{cd}_{tau nu phi} V(ab).
// The integrals of the item (its bra components x all ket components) are
// returned in acc; quartet_digest adds them to the Fock matrix.
// ---------------------------------------------------------------------------
// Ket primitive pairs as the table of records, or field by field: a lane that
// reads a 104-byte record touches two cache lines alone, where the arrays let
// consecutive lanes share them.
struct KetRecords {
    const PrimPair* pp;
    __device__ __forceinline__ double operator()(int i, KetField f) const
    {
        const PrimPair& Q = pp[i];
        switch (f) {
            case KF_P: return Q.p;
            case KF_KQ: return Q.K * Q.invp;
            case KF_X: return Q.Px;
            case KF_Y: return Q.Py;
            case KF_Z: return Q.Pz;
            case KF_INV2P: return Q.inv2p;
            case KF_PAX: return Q.PAx;
            case KF_PAY: return Q.PAy;
            case KF_PAZ: return Q.PAz;
            case KF_PBX: return Q.PBx;
            case KF_PBY: return Q.PBy;
            default: return Q.PBz;
        }
    }
};
struct KetArrays {
    const double* p;
    int64_t stride;
    __device__ __forceinline__ double operator()(int i, KetField f) const { return p[f * stride + i]; }
};

template <int LA, int LB, int LC, int LD, int A0, int A1, typename T, class KET>
__device__ __forceinline__ void quartet_compute(const KET& Q, const T* lds, const T* bp, int ip0, int ip1, int jq0,
                                                int jq1, T* acc)
{
    using S = ClassShape<LA, LB, LC, LD>;
    constexpr int NCH = A1 - A0;
    constexpr int NCD = S::NCD;
    constexpr int L = S::L;
    constexpr int HCD = S::HCD;
    sfor<NCH * NCD>([&](auto k) { acc[k] = T(0); });

    for (int jq = jq0; jq < jq1; ++jq) {
        const T Qp = (T)Q(jq, KF_P), QK = (T)Q(jq, KF_KQ), Qx = (T)Q(jq, KF_X), Qy = (T)Q(jq, KF_Y),
                Qz = (T)Q(jq, KF_Z);
        T V[HCD * NCH];
        sfor<HCD * NCH>([&](auto k) { V[k] = T(0); });
        for (int ip = ip0; ip < ip1; ++ip) {
            const T* b = bp + ip * S::BPS;
            const T Pp = b[0];
            const T rs = dev_rsqrt(Pp + Qp);
            const T alpha = Pp * Qp * rs * rs;
            const T X = b[2] - Qx, Y = b[3] - Qy, Z = b[4] - Qz;
            const T Targ = alpha * (X * X + Y * Y + Z * Z);
            const T pref = b[1] * QK * rs;   // 2 pi^{5/2} / (p q sqrt(p+q)) K_ab K_cd
            T F[L + 1];
            boys_seeds<L, T>(Targ, alpha, pref, lds, F);
            T R[nherm(L)];
            hermite_R<L, T>(X, Y, Z, F, R);
            const T* Ebx = b + 8;
            const T* Eby = b + 8 + S::EB;
            const T* Ebz = b + 8 + 2 * S::EB;
            sfor<NCH>([&](auto ii) {
                constexpr int ab = A0 + decltype(ii)::value;
                constexpr int a = ab / S::NB, bb = ab % S::NB;
                constexpr int ax = comp_lx(LA, a), ay = comp_ly(LA, a), az = comp_lz(LA, a);
                constexpr int bx = comp_lx(LB, bb), by = comp_ly(LB, bb), bz = comp_lz(LB, bb);
                constexpr int ix = (ax * (LB + 1) + bx) * S::NTB;
                constexpr int iy = (ay * (LB + 1) + by) * S::NTB;
                constexpr int iz = (az * (LB + 1) + bz) * S::NTB;
                sfor<HCD>([&](auto ik) {
                    constexpr Herm3 h = hdecode(decltype(ik)::value);
                    T v = V[decltype(ik)::value * NCH + decltype(ii)::value];
                    sfor<ax + bx + 1>([&](auto it) {
                        constexpr int t = decltype(it)::value;
                        sfor<ay + by + 1>([&](auto iu) {
                            constexpr int u = decltype(iu)::value;
                            const T exy = Ebx[ix + t] * Eby[iy + u];
                            sfor<az + bz + 1>([&](auto iw) {
                                constexpr int w = decltype(iw)::value;
                                v = fma(exy * Ebz[iz + w], R[hidx(t + h.t, u + h.u, w + h.v)], v);
                            });
                        });
                    });
                    V[decltype(ik)::value * NCH + decltype(ii)::value] = v;
                });
            });
        }
        // ket expansion, once per ket primitive pair
        T Ekx[(LC + 1) * (LD + 1) * S::NTK], Eky[(LC + 1) * (LD + 1) * S::NTK],
            Ekz[(LC + 1) * (LD + 1) * S::NTK];
        if constexpr (LC + LD > 0) {
            const T qinv2 = (T)Q(jq, KF_INV2P);
            hermite_E<LC, LD, -1, T>(qinv2, (T)Q(jq, KF_PAX), (T)Q(jq, KF_PBX), Ekx);
            hermite_E<LC, LD, -1, T>(qinv2, (T)Q(jq, KF_PAY), (T)Q(jq, KF_PBY), Eky);
            hermite_E<LC, LD, -1, T>(qinv2, (T)Q(jq, KF_PAZ), (T)Q(jq, KF_PBZ), Ekz);
        } else {
            Ekx[0] = Eky[0] = Ekz[0] = T(1);
        }
        sfor<NCD>([&](auto icd) {
            constexpr int cd = decltype(icd)::value;
            constexpr int c = cd / S::ND, d = cd % S::ND;
            constexpr int cx = comp_lx(LC, c), cy = comp_ly(LC, c), cz = comp_lz(LC, c);
            constexpr int dx = comp_lx(LD, d), dy = comp_ly(LD, d), dz = comp_lz(LD, d);
            constexpr int kx = (cx * (LD + 1) + dx) * S::NTK;
            constexpr int ky = (cy * (LD + 1) + dy) * S::NTK;
            constexpr int kz = (cz * (LD + 1) + dz) * S::NTK;
            sfor<NCH>([&](auto ii) {
                T sacc = acc[decltype(ii)::value * NCD + cd];
                sfor<cx + dx + 1>([&](auto itau) {
                    constexpr int tau = decltype(itau)::value;
                    sfor<cy + dy + 1>([&](auto inu) {
                        constexpr int nu = decltype(inu)::value;
                        const T exy = Ekx[kx + tau] * Eky[ky + nu];
                        sfor<cz + dz + 1>([&](auto iphi) {
                            constexpr int phi = decltype(iphi)::value;
                            sacc = fma(exy * Ekz[kz + phi], V[hidx(tau, nu, phi) * NCH + decltype(ii)::value], sacc);
                        });
                    });
                });
                acc[decltype(ii)::value * NCD + cd] = sacc;
            });
        });
    }
}

template <int I, int N, class F>
__device__ __forceinline__ void static_switch(int i, F&& f)
{
    if constexpr (I < N) {
        if (i == I) f(std::integral_constant<int, I>{});
        else static_switch<I + 1, N>(i, f);
    }
}

}  // namespace mmd
