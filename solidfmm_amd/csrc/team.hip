// Launches of the team kernels (team.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/solidfmm_gpu.h"
#include "team.hpp"

namespace sfmm {
namespace team {

template <>
const Kernels &kernels<SFMM_M2M>();
template <>
const Kernels &kernels<SFMM_M2L>();
template <>
const Kernels &kernels<SFMM_L2L>();

static_assert(kTeamMax == uint32_t(team::kMaxOrder));

namespace {

// LDS of a workgroup of 2^tl translations of orders up to pc: the weights,
// the triangle and the rotation factors.
size_t lds_bytes(int op, int njx, int pc, int tl)
{
    return sizeof(double) *
           (size_t(weight_size(op, pc)) + (size_t(pc) * (pc + 1) << tl) + size_t(rot_size(njx, pc, 1 << tl)));
}
constexpr size_t kLds = 160 * 1024;

}  // namespace
}  // namespace team

hipError_t launch_team(int op, uint32_t pc, const sfmm_item *items, size_t n, const double *src, double *dst,
                       hipStream_t stream, int mode)
{
    using namespace team;
    if (op < 0 || op > 2 || pc < 1 || pc > kTeamMax) return hipErrorInvalidValue;
    if (n == 0) return hipSuccess;
    if (n > 0xFFFFFFFFull) return hipErrorInvalidValue;
    const double *table = team::device_table();
    const double *fac = mfma::device_factorials();
    if (!table || !fac) return hipErrorOutOfMemory;
    const Kernels &ks = op == SFMM_M2M   ? kernels<SFMM_M2M>()
                        : op == SFMM_M2L ? kernels<SFMM_M2L>()
                                         : kernels<SFMM_L2L>();
    const int njx = pc > 32 ? 6 : pc > 24 ? 4 : pc > 16 ? 3 : 2;
    // as many translations as the triangle leaves room for: 16 up to order
    // 32 (fixed in that kernel), 8 up to 48
    int tl = 4;
    while (lds_bytes(op, njx, int(pc), tl) > kLds) --tl;
    const size_t lds = lds_bytes(op, njx, int(pc), tl);
    const size_t groups = (n + (size_t(1) << tl) - 1) >> tl;
    // Eight waves while every group has a CU of its own (the shortest chain
    // of degrees a wave), four beyond: two or three groups share a CU and one
    // group's waits for memory and barriers cover another's (order 16, 4,000
    // items: 14 us with eight waves, 16 with four; 8,000: 24 and 22; 24,000:
    // 60 and 52).
    const int waves = pc > 24 || groups <= 256 ? 8 : 4;
    const fn_t f = njx == 6   ? ks.upto48
                   : njx == 4 ? ks.upto32
                   : njx == 3 ? (waves == 8 ? ks.upto24w : ks.upto24)
                             : (waves == 8 ? ks.upto16w : ks.upto16);
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(f),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(kLds));
        if (e != hipSuccess) return e;
    }
    // a launch holds fewer than 2^32 threads
    constexpr size_t kMost = size_t(1) << 22;
    for (size_t g = 0; g < groups; g += kMost) {
        const size_t first = g << tl;
        hipLaunchKernelGGL(f, dim3(uint32_t(std::min(groups - g, kMost))), dim3(64 * waves), lds, stream, src, dst,
                           items + first, uint32_t(n - first), table, fac, int(pc), tl, mode);
    }
    return hipGetLastError();
}

}  // namespace sfmm
