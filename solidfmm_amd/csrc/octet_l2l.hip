// L2L octet kernels (octet.hpp).
#include "octet.hpp"

namespace sfmm {
namespace octet {

template hipError_t launch_op<SFMM_L2L>(uint32_t, const sfmm_item *, size_t, const double *, double *, hipStream_t, int,
                                           bool);

}  // namespace octet
}  // namespace sfmm
