// One quartet class of the integral-block kernels per translation unit
// (QC_LA .. QC_LD), so that the classes compile in parallel.
#include <algorithm>
#include "mmd_eri_block.h"

#define MMD_PASTE5(p, a, b, c, d) p##a##b##c##d
#define MMD_NAME(p, a, b, c, d) MMD_PASTE5(p, a, b, c, d)

namespace mmd {

hipError_t MMD_NAME(block_class_launch_, QC_LA, QC_LB, QC_LC, QC_LD)(const ClassArgs& A, const BlockArgs& B,
                                                                     hipStream_t st)
{
    const int64_t nq = B.tri ? (int64_t)B.nb * (B.nb + 1) / 2 : (int64_t)B.nb * B.nk;
    if (nq <= 0) return hipSuccess;
    const int64_t waves = ((nq << (B.lgb + B.lgk)) + 63) / 64 * ClassShape<QC_LA, QC_LB, QC_LC, QC_LD>::NCHUNK;
    hipLaunchKernelGGL((eri_block_kernel<QC_LA, QC_LB, QC_LC, QC_LD>),
                       dim3((unsigned)std::min<int64_t>((waves + 3) / 4, 4096)), dim3(256), 0, st, A, B);
    return hipGetLastError();
}

}  // namespace mmd
