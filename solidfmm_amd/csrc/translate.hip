// Dispatch of the translation kernels: (op, kernel choice) -> launch.
//
// The kernels themselves live in lane_kernel.hpp (one lane per
// translation), translate_mfma.hpp (16 translations per wave on the FP64
// matrix cores), team.hpp (up to 16 translations per workgroup, orders 25 to
// 48), generic.hip (one workgroup per translation, any order) and,
// for the reduced-precision modes, lane_prec.hpp, mfma_prec.hpp (FP32
// matrix cores) and prec_generic.hip.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <utility>
#include <vector>

#include "../../include/solidfmm_gpu.h"
#include "lane_kernel.hpp"
#include "mfma_tables.hpp"
#include "translate.hpp"

namespace sfmm {

size_t max_kernel_order() { return size_t(mfma::kMaxOrder); }

bool family_covers(int family, uint32_t pb)
{
    if (pb < 1) return false;
    switch (family) {
    case kLaneKernels: return pb <= kLaneMax;
    case kMfmaKernels: return pb >= uint32_t(mfma::kMfmaMin) && pb <= uint32_t(mfma::kMfmaMax);
    case kGenericKernel: return pb <= uint32_t(mfma::kMaxOrder);
    default: return false;
    }
}

int default_family(uint32_t pb)
{
    if (pb <= kLaneAutoMax) return kLaneKernels;
    if (pb <= uint32_t(mfma::kMfmaMax)) return kMfmaKernels;
    return kGenericKernel;
}

// The straight-line MFMA kernels give a wave 16 translations from start to
// end, so a list takes whole rounds of 16,384 (one wave per SIMD): 20 us a
// round at order 12, 35 at 16, 72 at 20, most of it one wave's chain of
// degrees and, above order 17, code that outgrows the instruction cache. The
// team kernel walks the degrees of a group side by side: 9 us for one group
// and 11 for 4,000 translations at order 12, 11 and 14 at 16, 15 and 21 at 20.
// It needs more instructions per translation, so the straight-line kernels
// keep the long lists up to order 20. M2M, straight-line against team (us):
//   order 12:  8,000 19.1, 15.6;  12,000 20.5, 23.0;  120,000 144, 175
//   order 16:  12,000 34.3, 32.2;  16,000 35.3, 37.3;  120,000 288, 281
//   order 18:  12,000 50.6, 45.9;  16,000 51.4, 52.0;  120,000 360, 430
//   order 20:  24,000 121, 80;  50,000 229, 204;  120,000 452, 472
//   order 21:  120,000 817, 523;  order 24: 1565, 609
// (M2L and L2L of order 20 at 120,000: 470, 435 and 450, 428).
size_t team_items(int op, uint32_t pb)
{
    constexpr size_t kAll = ~size_t(0);
    if (pb <= 14) return 8192;
    if (pb <= 19) return 12288;
    if (pb == 20) return op == SFMM_M2M ? 65536 : kAll;
    return kAll;
}

// At orders 8 to 11 a team is faster than one lane per translation while the
// lanes leave most of the chip idle (M2L: order 8, 1,000 items 11.9 -> 8.1
// us, 4,000 12.4 -> 8.6; order 10 13.9 -> 9.5 and 14.3 -> 10.2; at 8,000 order
// 10 takes 14.8 and 14.0, L2L 12.4 and 14.0). Below, a lane's chain is as short
// as a team's (order 7, 4,000: 8.2 and 8.4).
size_t lane_team_items(uint32_t pb)
{
    return pb >= 8 && pb <= kLaneAutoMax ? 4096 : 0;
}

uint32_t generic_bucket(uint32_t pb)
{
    if (pb <= uint32_t(mfma::kMfmaMax) || pb > kTeamMax) return kGenericRest;
    return pb <= 32 ? 32 : kTeamMax;
}

bool have_kernel(int op, uint32_t p_in, uint32_t p_out, int family)
{
    if (op < 0 || op > 2 || p_in < 1 || p_out < 1) return false;
    const uint32_t pb = p_in > p_out ? p_in : p_out;
    if (family == kAuto) return pb <= uint32_t(mfma::kMaxOrder);
    return family_covers(family, pb);
}

uint32_t persistent_grid(const void *kernel, int block, size_t work)
{
    struct Key {
        const void *k;
        int dev;
    };
    static std::mutex mu;
    static std::vector<std::pair<Key, uint32_t>> cache;
    int dev = 0;
    (void)hipGetDevice(&dev);
    uint32_t resident = 0;
    {
        std::lock_guard<std::mutex> lock(mu);
        for (auto &e : cache)
            if (e.first.k == kernel && e.first.dev == dev) resident = e.second;
        if (!resident) {
            int per_cu = 0, cus = 0;
            // a failed query falls back to one workgroup per CU; its error
            // is cleared so the launch that follows does not report it
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess || per_cu < 1) {
                (void)hipGetLastError();
                per_cu = 1;
            }
            if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) {
                (void)hipGetLastError();
                cus = 1;
            }
            resident = uint32_t(per_cu) * uint32_t(cus);
            cache.push_back({{kernel, dev}, resident});
        }
    }
    if (work < resident) return uint32_t(work < 1 ? 1 : work);
    return resident;
}

// Items per wave of a lane launch of n items: 64, unless the last round of
// resident waves would be partly empty -- then the items are spread evenly
// over whole rounds (1e5 items on 1,024 resident waves: 2,041 waves of 49
// instead of 1,563 of 64, two full rounds either way).
uint32_t lane_items_per_wave(const void *kernel, size_t n)
{
    const size_t slots = persistent_grid(kernel, 64, size_t(1) << 40);
    const size_t waves = (n + 63) / 64;
    if (slots == 0 || waves <= slots) return 64;
    const size_t rounds = (waves + slots - 1) / slots;
    const size_t ipw = (n + rounds * slots - 1) / (rounds * slots);
    return uint32_t(ipw < 1 ? 1 : ipw > 64 ? 64 : ipw);
}

namespace {

template <bool RT>
hipError_t launch_mfma(int op, uint32_t pk, const sfmm_item *items, size_t n, const double *src, double *dst,
                       const double *table, hipStream_t stream, int acc)
{
    switch (op) {
    case SFMM_M2M: return mfma::launch_op<SFMM_M2M, RT>(pk, items, n, src, dst, table, stream, acc);
    case SFMM_M2L: return mfma::launch_op<SFMM_M2L, RT>(pk, items, n, src, dst, table, stream, acc);
    default: return mfma::launch_op<SFMM_L2L, RT>(pk, items, n, src, dst, table, stream, acc);
    }
}

}  // namespace

hipError_t launch_kernel(int op, const KernelChoice &k, const sfmm_item *items, size_t n, const double *src,
                         double *dst, hipStream_t stream)
{
    const int acc = k.acc ? 1 : 0;
    if (k.precision != SFMM_FP64) {
        if (k.family == kLaneKernels && op == SFMM_M2L && !k.rt)
            return launch_prec_lane_m2l(k.precision, k.pk, items, n, src, dst, stream, acc);
        if (k.family == kMfmaKernels && op == SFMM_M2L && !k.rt && k.precision == SFMM_FP32)
            return launch_prec_mfma_m2l(k.pk, items, n, src, dst, stream, acc);
        if (k.family == kGenericKernel)
            return launch_prec_generic(k.precision, op, k.pk, items, n, src, dst, stream, acc);
        return hipErrorInvalidValue;
    }
    if (op < 0 || op > 2 || !family_covers(k.family, k.pk)) return hipErrorInvalidValue;
    if (n == 0) return hipSuccess;
    if (n > 0xFFFFFFFFull) return hipErrorInvalidValue;
    switch (k.family) {
    case kLaneKernels: {
        // scratch launches with runs use the per-item-order kernels (the
        // fixed-order ones have no code for runs)
        const bool runs = !k.acc && k.seg;
        const lane::Table &t = (k.rt || runs) ? lane::rt_table() : lane::fixed_table();
        lane::kernel_fn f = t.f[op][k.pk - 1];
        const uint32_t block = 64;
        uint32_t ipw = lane_items_per_wave(reinterpret_cast<const void *>(f), n);
        if (runs) ipw = 64;  // the plan lays runs out in 64-item waves
        const uint32_t grid = static_cast<uint32_t>((n + ipw - 1) / ipw);
        hipLaunchKernelGGL(f, dim3(grid), dim3(block), 0, stream, src, dst, items, static_cast<uint32_t>(n),
                           runs ? 2 : acc, ipw);
        return hipGetLastError();
    }
    case kMfmaKernels: {
        const int mode = (!k.acc && k.seg) ? 2 : acc;
        if (n <= team_items(op, k.pk)) return launch_team(op, k.pk, items, n, src, dst, stream, mode);
        const double *table = mfma::device_table();
        if (!table) return hipErrorOutOfMemory;
        return k.rt ? launch_mfma<true>(op, k.pk, items, n, src, dst, table, stream, mode)
                    : launch_mfma<false>(op, k.pk, items, n, src, dst, table, stream, mode);
    }
    default:
        // Orders above the MFMA kernels' 24 run on the team kernels as far
        // as their LDS triangle reaches (M2L, 2,000 items: order 25 340 ->
        // 27 us, 32 577 -> 40, 40 895 -> 84, 48 2500 -> 121; a single group
        // of 7 items: order 32 488 -> 31).
        if (generic_bucket(k.pk) != kGenericRest) return launch_team(op, k.pk, items, n, src, dst, stream, acc);
        return launch_generic(op, k.pk, items, n, src, dst, stream, acc);
    }
}

hipError_t launch_translate(int op, uint32_t p_in, uint32_t p_out, const sfmm_item *items, size_t n,
                            const double *src, double *dst, hipStream_t stream, int family)
{
    if (!have_kernel(op, p_in, p_out, family)) return hipErrorInvalidValue;
    const uint32_t pb = p_in > p_out ? p_in : p_out;
    const int fam = family == kAuto ? default_family(pb) : family;
    return launch_kernel(op, KernelChoice{fam, pb, p_in != p_out}, items, n, src, dst, stream);
}

}  // namespace sfmm
