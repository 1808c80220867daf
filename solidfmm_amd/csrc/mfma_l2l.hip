// Instantiations of the MFMA translation kernels for L2L (square orders
// kMfmaMin..kMfmaKernelMax, uniform orders).
#include "translate_mfma.hpp"

namespace sfmm {
namespace mfma {

template hipError_t launch_op<SFMM_L2L, false>(uint32_t, const sfmm_item *, size_t, const double *, double *,
                                                   const double *, hipStream_t, int);

}  // namespace mfma
}  // namespace sfmm
