// One shell-quartet class of the Fock-build kernel per translation unit; the
// build sets QC_LA, QC_LB, QC_LC, QC_LD, and QC_F32 for the FP32-tier
// instantiation.  Splitting the classes over separate objects lets them
// compile in parallel.
#include <algorithm>
#include "mmd_eri_impl.h"

#define MMD_PASTE6(p, a, b, c, d, s) p##a##b##c##d##s
#define MMD_NAME(p, a, b, c, d, s) MMD_PASTE6(p, a, b, c, d, s)

#ifdef QC_F32
#define QC_T float
#define QC_SUFFIX _f
#else
#define QC_T double
#define QC_SUFFIX _d
#endif

namespace mmd {

hipError_t MMD_NAME(fock_class_launch_, QC_LA, QC_LB, QC_LC, QC_LD, QC_SUFFIX)(const ClassArgs& A, const RowArgs& R,
                                                                               int grid, hipStream_t st)
{
    const size_t lds = fock_class_lds_bytes<QC_LA, QC_LB, QC_LC, QC_LD, QC_T>(R.rw, R.maxpp, R.kj);
    hipLaunchKernelGGL((eri_fock_class_kernel<QC_LA, QC_LB, QC_LC, QC_LD, QC_T>), dim3(grid), dim3(CLASS_BLOCK), lds,
                       st, A, R);
    return hipGetLastError();
}

size_t MMD_NAME(fock_class_lds_, QC_LA, QC_LB, QC_LC, QC_LD, QC_SUFFIX)(int rw, int maxpp, int kj)
{
    return fock_class_lds_bytes<QC_LA, QC_LB, QC_LC, QC_LD, QC_T>(rw, maxpp, kj);
}

}  // namespace mmd
