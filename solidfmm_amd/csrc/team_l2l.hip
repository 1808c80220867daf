// Instantiations of the team kernel for L2L.
#include "team.hpp"

namespace sfmm {
namespace team {

template <>
const Kernels &kernels<SFMM_L2L>()
{
    static const Kernels k{&k_team<SFMM_L2L, 2, 4, 4, 2>, &k_team<SFMM_L2L, 3, 4, 4, 2>, &k_team<SFMM_L2L, 2, 4, 8, 2>,
                           &k_team<SFMM_L2L, 3, 4, 8, 2>, &k_team<SFMM_L2L, 4, 4, 8, 2>, &k_team<SFMM_L2L, 6, -1, 8, 2>};
    return k;
}

}  // namespace team
}  // namespace sfmm
