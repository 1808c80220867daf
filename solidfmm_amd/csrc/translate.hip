// Dispatch of the translation kernels: (op, kernel choice) -> launch.
//
// The kernels themselves live in lane_kernel.hpp (one lane per
// translation), octet.hpp (a wave per 8 translations on the FP64 matrix
// cores) and team.hpp (several waves per 16, short lists and orders to 48),
// generic.hip (one workgroup per translation, any order) and, for the
// reduced-precision modes, lane_prec.hpp, mfma_prec.hpp (FP32 matrix cores)
// and prec_generic.hip.
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
    case kMfmaKernels: return pb <= uint32_t(mfma::kMfmaMax);
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

// An octet kernel walks a group's degrees in one wave, a team kernel side by
// side in four or eight: 9 us against 8 for a lone group of order 8, 22
// against 12 at 16, 42 against 20 at 24. The octet kernel does the same work
// in fewer cycles, so it takes over once groups fill the chip.  Up to order 13
// that is where team groups begin to share CUs: 4,096 items are 256 groups of
// 16, and the next one costs all of them a quarter (order 9, 4,000 items 7.8,
// 4,200 9.9; octets 7.8 and 7.5, from HBM).  Above, the team's shorter chain
// carries it further. M2L, team against octet (us):
//   order  8: 4,000 6.5, 7.1;   5,000 8.1, 7.2;    120,000 99, 46
//   order 10: 4,000 8.4, 9.2;   5,000 12.2, 9.7;   6,000 12.6, 10.0
//   order 12: 4,000 10.3, 11.6; 5,000 13.8, 11.8;  120,000 178, 101
//   order 16: 8,192 22.6, 25.7; 12,288 33.2, 26.4; 120,000 288, 204
//   order 18: 8,192 27.9, 27.3; 12,288 41.8, 41.8; 120,000 378, 288
//   order 20: 12,288 45.7, 53.0; 24,000 76.5, 76.1; 120,000 425, 365
//   order 22: 30,011 122, 123;  60,000 266, 242
//   order 24: 60,000 299, 344;  120,000 584, 626
// M2M and L2L keep one operand table instead of two and cross over earlier
// from order 19 (M2M of order 20: 8,192 29.9, 29.0; 12,288 44.8, 45.5;
// 16,384 51.8, 46.5; order 24: 16,384 67.8, 68.1; 24,000 96.6, 94.4).  L2L of
// orders 8 to 12 as M2L within 5 %.
size_t team_items(int op, uint32_t pb)
{
    if (pb <= 13) return 4096;
    if (pb <= 18) return 8192;
    if (op != SFMM_M2L) return 12288;
    if (int(pb) > octet::max_order(op)) return ~size_t(0);
    return pb <= 20 ? 24576 : 32768;
}

// The tree of shuffles costs the same for any runs, the sums through LDS some
// 15 instructions a run and degree and an LDS copy of the wave's results.  M2L
// with its reduction, tree against LDS (us), by items and length of the runs:
//   order  6, 250,000: 16 52, 49; 20 51, 51; 32 50, 42; 140 47, 41
//   order  8, 250,000: 16 98, 83; 32 92, 74; 140 89, 70;  50,000: 32, 31 at any
//   order 10, 250,000: 16 180, 151; 140 171, 122;  20,000: 35, 37 at any
// and at 200,000 items in runs of 8: order 6 50, 65; 9 128, 156; 11 220, 236.
bool long_runs(uint32_t pb, size_t n, size_t runs)
{
    return n >= 65536 && n >= (pb >= 7 ? 16 : 24) * runs;
}

// Octet times go up in steps of 8,192 items, a wave of eight for each SIMD;
// lanes spread any number of items over theirs.  L2L, whose lane kernels need
// the fewest registers, is faster on lanes after such a step where few waves
// are in flight: lanes against octets (us, from HBM)
//   order  9:  8,256 9.6, 10.2;  12,296 10.7, 11.7; 16,384 11.9, 13.0; 16,904 16.5, 16.6
//             20,000 17.6, 17.5; 25,096 19.0, 20.9; 32,768 22.0, 22.8; 40,000 29.2, 27.2
//   order 10:  8,256 11.7, 11.8; 12,296 12.9, 13.3; 16,384 14.3, 14.7; 18,000 20.8, 19.9
//   order 11:  8,256 13.3, 13.9; 12,296 14.7, 15.2; 16,384 16.5, 17.1; 18,000 23.9, 23.1
// and M2M and M2L of order 9 at 12,000 items: 11.7, 11.5 and 12.0, 10.9.
// Children that share their parent's expansion read it from the caches, and the
// lanes' single accesses cost less: lanes ahead at any length from there on, with
// the pools in HBM (8 children; order 9 12,000 9.5, 10.7; 100,000 56, 61; 300,000
// 157, 178; order 10 12,000 11.4, 12.5; 200,000 136, 140; order 11 25,000 21.7,
// 24.9; 300,000 230, 245) as in the last-level cache (order 10, 100,000 47, 60).
bool lanes_ahead(int op, uint32_t pb, size_t n, bool shared)
{
    constexpr size_t step = 8192;
    if (op != SFMM_L2L || pb < 9 || pb > 11) return false;
    return n > step && (shared || n <= 2 * step || (pb == 9 && n > 3 * step && n <= 4 * step));
}

// A lane wave adds runs of up to 64 items before it stores, an octet group runs
// of up to 8, and a lane takes one translation's latency for 64 of them; but 64
// items a wave need long lists to fill the chip.  The lists from which lanes are
// ahead, by order and by mean length of the runs; M2L with its reduction, lanes
// against octets (us) by items and length:
//   order  8: 100,000  5 60, 58;   16 45, 50;   140 42, 51;  500,000  5 220, 258; 140 113, 204
//   order  9: 100,000 20 67, 62;   32 58, 62;   200,000 16 105, 113;  500,000  5 284, 313
//   order 10: 100,000 32 74, 73;   64 71, 72;   200,000 16 126, 136;  500,000 12 320, 321
//   order 11: 300,000 16 239, 228; 32 215, 226; 200,000 140 129, 154; 500,000 12 431, 376
//   order 12: 300,000 64 271, 248; 140 236, 254; 500,000 140 342, 408; 200,000 140 176, 175
// M2M, whose runs are the up to eight children of a cell: order 8, 500,000
// 238, 248; order 9 300,000 177, 186; order 12 616, 478.  The lane kernels of
// L2L are slower at any length (order 8, 500,000: 5 395, 274; 140 287, 215).
// One round of lane waves, 65,536 items, takes the same time from 40,000 on:
// M2L of order 9, 60,000: 16 37, 43; order 10: 16 45, 50; order 11: 140 54, 60;
// and two waves fit a SIMD at order 8, 130,000: 5 69, 72; 12 58, 63.
//
// Launches of one plan run side by side and fill each other's last rounds, so
// what counts is the plan's `total`, as long as the launch itself has work for
// most SIMDs: M2L of an FMM, 75,000 of its 997,000 items of order 11, 823 us
// with that bucket on lanes, 847 on octets; 30,000 of order 12 869 and 847.
bool lanes_for_runs(int op, uint32_t pb, size_t n, size_t runs, size_t total)
{
    constexpr size_t no = ~size_t(0);
    struct Row {
        size_t len4, len16, len24, len40;  // items from which lanes are ahead
        size_t round, full, round_len;     // one round of M2L: items from, to, length
    };
    constexpr Row rows[] = {{200000, 100000, 100000, 70000, 110000, 131072, 4},
                            {300000, 200000, 100000, 100000, 43000, 65536, 10},
                            {450000, 200000, 150000, 100000, 48000, 65536, 16},
                            {no, 500000, 250000, 150000, 57000, 65536, 40},
                            {no, no, no, 300000, no, 0, 0}};
    if (op == SFMM_L2L || pb < 8 || pb > kLaneMax || n <= 40000) return false;
    const Row &r = rows[pb - 8];
    if (op == SFMM_M2L && total == n && n >= r.round && n <= r.full && n >= r.round_len * runs) return true;
    return total >= (n >= 40 * runs   ? r.len40
                     : n >= 24 * runs ? r.len24
                     : n >= 16 * runs ? r.len16
                     : n >= 4 * runs  ? r.len4
                                      : no);
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

uint32_t persistent_grid(const void *kernel, int block, size_t work, size_t lds)
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
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, lds) != hipSuccess || per_cu < 1) {
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
        const lane::Table &t = k.long_runs     ? lane::runs_table()
                               : k.rt || runs ? lane::rt_table()
                                              : lane::fixed_table();
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
        if (k.team) return launch_team(op, k.pk, items, n, src, dst, stream, mode);
        switch (op) {
        case SFMM_M2M: return octet::launch_op<SFMM_M2M>(k.pk, items, n, src, dst, stream, mode, k.pairs);
        case SFMM_M2L: return octet::launch_op<SFMM_M2L>(k.pk, items, n, src, dst, stream, mode, k.pairs);
        default: return octet::launch_op<SFMM_L2L>(k.pk, items, n, src, dst, stream, mode, k.pairs);
        }
    }
    default:
        // Orders above the MFMA kernels' 24 run on the team kernels as far
        // as their LDS triangle reaches (M2L, 2,000 items: order 25 340 ->
        // 27 us, 32 577 -> 40, 40 895 -> 84, 48 2500 -> 121; a single group
        // of 7 items: order 32 488 -> 31).
        if (k.team) return launch_team(op, k.pk, items, n, src, dst, stream, acc);
        return launch_generic(op, k.pk, items, n, src, dst, stream, acc);
    }
}

}  // namespace sfmm
