// Instantiations of the team kernel for M2M.
#include "team.hpp"

namespace sfmm {
namespace team {

template <>
const Kernels &kernels<SFMM_M2M>()
{
    static const Kernels k{&k_team<SFMM_M2M, 2, 4, 4, 2>, &k_team<SFMM_M2M, 3, 4, 4, 2>, &k_team<SFMM_M2M, 2, 4, 8, 2>,
                           &k_team<SFMM_M2M, 3, 4, 8, 2>, &k_team<SFMM_M2M, 4, 4, 8, 2>, &k_team<SFMM_M2M, 6, -1, 8, 2>};
    return k;
}

}  // namespace team
}  // namespace sfmm
