// Dispatch table over the shell-quartet classes of the Fock-build kernel
// (each compiled in its own objects from mmd_eri_class.hip, in FP64 and in
// the FP32 tier).
#include "mmd_eri_core.h"
#include "mmd_kernels.h"

namespace mmd {

#define MMD_CLASSES(X)                                                                                   \
    X(0, 0, 0, 0) X(1, 0, 0, 0) X(1, 0, 1, 0) X(1, 1, 0, 0) X(1, 1, 1, 0) X(1, 1, 1, 1) X(2, 0, 0, 0)   \
    X(2, 0, 1, 0) X(2, 0, 1, 1) X(2, 0, 2, 0) X(2, 1, 0, 0) X(2, 1, 1, 0) X(2, 1, 1, 1) X(2, 1, 2, 0)   \
    X(2, 1, 2, 1) X(2, 2, 0, 0) X(2, 2, 1, 0) X(2, 2, 1, 1) X(2, 2, 2, 0) X(2, 2, 2, 1)

#define DECL(a, b, c, d)                                                                                         \
    hipError_t fock_class_launch_##a##b##c##d##_d(const ClassArgs& A, const RowArgs& R, int grid, hipStream_t st); \
    hipError_t fock_class_launch_##a##b##c##d##_f(const ClassArgs& A, const RowArgs& R, int grid, hipStream_t st); \
    size_t fock_class_lds_##a##b##c##d##_d(int N, int maxpp, int kj);                                            \
    size_t fock_class_lds_##a##b##c##d##_f(int N, int maxpp, int kj);
MMD_CLASSES(DECL)
#undef DECL

// Staged bra data of stage_bra for every primitive pair of a pair class, in
// class order: table + (pair's position) * BPS.
namespace {
template <int LA, int LB>
__global__ void __launch_bounds__(64) bra_table_kernel(const ShellPair* __restrict__ pairs,
                                                       const PrimPair* __restrict__ pp, int boff, double* table)
{
    using S = ClassShape<LA, LB, 0, 0>;
    const ShellPair bra = pairs[boff + blockIdx.x];
    for (int idx = threadIdx.x; idx < 3 * bra.npp; idx += blockDim.x) {
        const int ip = idx / 3, x = idx - 3 * ip;
        const PrimPair* P = pp + bra.pp0 + ip;
        double* b = table + (size_t)(bra.class_pp0 + ip) * S::BPS;
        if (x == 0) {
            b[0] = P->p;
            b[1] = TWO_PI_2_5 * P->K * P->invp;
            b[2] = P->Px;
            b[3] = P->Py;
            b[4] = P->Pz;
        }
        double E[S::EB];
        hermite_E<LA, LB, 1>(P->inv2p, x == 0 ? P->PAx : (x == 1 ? P->PAy : P->PAz),
                             x == 0 ? P->PBx : (x == 1 ? P->PBy : P->PBz), E);
        sfor<S::EB>([&](auto k) { b[8 + x * S::EB + k] = E[k]; });
    }
}
}  // namespace

int bra_table_stride(int pc)
{
    constexpr int bps[NPAIRCLASS] = {ClassShape<0, 0, 0, 0>::BPS, ClassShape<1, 0, 0, 0>::BPS,
                                     ClassShape<1, 1, 0, 0>::BPS, ClassShape<2, 0, 0, 0>::BPS,
                                     ClassShape<2, 1, 0, 0>::BPS, ClassShape<2, 2, 0, 0>::BPS};
    return bps[pc];
}

hipError_t launch_bra_table(int pc, const ShellPair* pairs, const PrimPair* pp, int boff, int nb, double* table,
                            hipStream_t st)
{
    if (nb <= 0) return hipSuccess;
#define CASE(i, a, b) \
    case i: hipLaunchKernelGGL((bra_table_kernel<a, b>), dim3(nb), dim3(64), 0, st, pairs, pp, boff, table); break;
    switch (pc) {
        CASE(0, 0, 0) CASE(1, 1, 0) CASE(2, 1, 1) CASE(3, 2, 0) CASE(4, 2, 1) CASE(5, 2, 2)
    default: return hipErrorInvalidValue;
    }
#undef CASE
    return hipGetLastError();
}

#define DECLB(a, b, c, d) \
    hipError_t block_class_launch_##a##b##c##d(const ClassArgs& A, const BlockArgs& B, hipStream_t st);
MMD_CLASSES(DECLB)
#undef DECLB

hipError_t launch_block_class(int qc, const ClassArgs& A, const BlockArgs& B, hipStream_t st)
{
    int la, lb, lc, ld;
    qclass_decode(qc, &la, &lb, &lc, &ld);
#define CASE(a, b, c, d) \
    if (la == a && lb == b && lc == c && ld == d) return block_class_launch_##a##b##c##d(A, B, st);
    MMD_CLASSES(CASE)
#undef CASE
    return launch_block_dddd(A, B, st);
}

hipError_t launch_fock_class(int qc, int fp32, const ClassArgs& A, const RowArgs& R, int grid, hipStream_t st)
{
    int la, lb, lc, ld;
    qclass_decode(qc, &la, &lb, &lc, &ld);
#define CASE(a, b, c, d)                                                                               \
    if (la == a && lb == b && lc == c && ld == d)                                                      \
        return fp32 ? fock_class_launch_##a##b##c##d##_f(A, R, grid, st)                               \
                    : fock_class_launch_##a##b##c##d##_d(A, R, grid, st);
    MMD_CLASSES(CASE)
#undef CASE
    return hipErrorInvalidValue;  // wavefront-per-quartet classes are launched separately
}

#define MMD_MFMA_CLASSES(X) X(2, 2, 2, 2) X(2, 2, 2, 1) X(2, 2, 1, 1) X(2, 2, 2, 0) X(2, 1, 2, 1) X(2, 1, 1, 1) X(2, 1, 2, 0)

#define DECLM(a, b, c, d)                                                                                    \
    hipError_t fock_mfma_launch_##a##b##c##d##_d(const ClassArgs& A, int64_t max_quartets, hipStream_t st); \
    hipError_t fock_mfma_launch_##a##b##c##d##_f(const ClassArgs& A, int64_t max_quartets, hipStream_t st);
MMD_MFMA_CLASSES(DECLM)
#undef DECLM

hipError_t launch_fock_mfma_class(int la, int lb, int lc, int ld, int fp32, const ClassArgs& A, int64_t max_quartets,
                                  hipStream_t st)
{
#define CASE(a, b, c, d)                                                                    \
    if (la == a && lb == b && lc == c && ld == d)                                           \
        return fp32 ? fock_mfma_launch_##a##b##c##d##_f(A, max_quartets, st)                \
                    : fock_mfma_launch_##a##b##c##d##_d(A, max_quartets, st);
    MMD_MFMA_CLASSES(CASE)
#undef CASE
    return hipErrorInvalidValue;
}

size_t fock_class_lds(int qc, int fp32, int N, int maxpp, int kj)
{
    int la, lb, lc, ld;
    qclass_decode(qc, &la, &lb, &lc, &ld);
#define CASE(a, b, c, d)                          \
    if (la == a && lb == b && lc == c && ld == d) \
        return fp32 ? fock_class_lds_##a##b##c##d##_f(N, maxpp, kj) : fock_class_lds_##a##b##c##d##_d(N, maxpp, kj);
    MMD_CLASSES(CASE)
#undef CASE
    return 0;
}

}  // namespace mmd
