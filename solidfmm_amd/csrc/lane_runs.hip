// Instantiations of the one-lane-per-translation kernels for lists whose
// targets repeat in long runs.
#include <utility>

#include "lane_kernel.hpp"

namespace sfmm {
namespace lane {

const Table &runs_table()
{
    static const Table t = make_table<true, true>();
    return t;
}

}  // namespace lane
}  // namespace sfmm
