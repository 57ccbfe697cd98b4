// One quartet class of the two-electron gradient per translation unit
// (QC_LA .. QC_LD), so that the classes compile in parallel.  QC_BLOCK: the
// workgroup-per-primitive-quartet kernel.
#include <algorithm>
#include "mmd_grad_class.h"

#define MMD_PASTE5(p, a, b, c, d) p##a##b##c##d
#define MMD_NAME(p, a, b, c, d) MMD_PASTE5(p, a, b, c, d)

namespace mmd {

hipError_t MMD_NAME(grad_class_launch_, QC_LA, QC_LB, QC_LC, QC_LD)(const GradArgs& A, const GradClass& C,
                                                                    hipStream_t st)
{
#ifdef QC_BLOCK
    const int64_t units = (int64_t)C.nslice * C.nflat;
    if (units <= 0) return hipSuccess;
    hipLaunchKernelGGL((grad_block_kernel<QC_LA, QC_LB, QC_LC, QC_LD>), dim3((unsigned)std::min<int64_t>(units, 4096)),
                       dim3(GRAD_BLOCK), (GradBlockShape<QC_LA, QC_LB, QC_LC, QC_LD>::LDS), st, A, C);
#else
    const int64_t units = (int64_t)C.nslice * C.nkc;
    if (units <= 0) return hipSuccess;
    hipLaunchKernelGGL((grad_class_kernel<QC_LA, QC_LB, QC_LC, QC_LD>), dim3((unsigned)std::min<int64_t>(units, 2048)),
                       dim3(GRAD_BLOCK), A.lds_atoms ? sizeof(double) * 3 * A.natom : 0, st, A, C);
#endif
    return hipGetLastError();
}

}  // namespace mmd
