// Internal launcher interface of the translation kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "../../include/solidfmm_gpu.h"

namespace sfmm {

// Kernel families:
//   lane     one lane per translation, FP64 VALU, orders up to 12
//            (lane_kernel.hpp);
//   MFMA     swaps on the FP64 matrix cores, orders up to 24: one wave per
//            eight translations (octet.hpp, long lists) or several waves per
//            sixteen (team.hpp);
//   generic  any orders up to 86, one workgroup per translation
//            (generic.hip); orders 25 to 48 run on the team kernels (team.hpp)
//            unless the context asks for this family.
// Lane and octet kernels are instantiated per order bound PB.  Lane kernels
// take items of orders (PB, PB), their RT variants any p_in, p_out <= PB, as
// all other kernels do.
enum Family { kAuto = 0, kLaneKernels = 1, kMfmaKernels = 2, kGenericKernel = 3 };

inline constexpr uint32_t kLaneMax = 12;
// lane kernels by default up to this order: at 7 they are level with the
// octet kernels on long lists (M2L of 200,000: 63.1 us on lanes, 62.9), at 8
// and from 10 up behind (8: 137 against 71; 9: 105, 104; 10: 156, 129; 11:
// 211, 149), and on short lists of order 8 behind the team kernels (1,000:
// 11.9 against 8.1; order 7, 4,000: 8.2, 8.4)
inline constexpr uint32_t kLaneAutoMax = 7;
// Whether a lane launch of n items in `runs` runs adds them through LDS
// (run_sums) instead of by a tree of shuffles (translate.hip has the figures).
bool long_runs(uint32_t pb, size_t n, size_t runs);

// M2L lists of at most kLaneSmallM2L items keep orders 9 to 11 on lanes by
// default.  Small batches are where single results are compared with the
// reference, and the lanes' sums follow its order: 256 items of order 10
// differ from the oracle by 5.9e-14 at the 99th percentile on lanes and 1.1e-13
// on the team kernel, whose distance from exact results is the same.  The
// price is 11.1 us against 7.1.
inline constexpr size_t kLaneSmallM2L = 512;

namespace mfma {
inline constexpr int kMfmaMax = 24;
}  // namespace mfma

// Highest order with a kernel.
size_t max_kernel_order();

// True when `family` (not kAuto) has a kernel for items whose larger order
// is pb.
bool family_covers(int family, uint32_t pb);

// The family kAuto picks for items whose larger order is pb.
int default_family(uint32_t pb);

// True when the library has a kernel for (op, p_in, p_out) in `family`.
bool have_kernel(int op, uint32_t p_in, uint32_t p_out, int family = kAuto);

// Workgroups for a persistent kernel: as many as can be resident on the
// current device at once, but no more than `work` (one per unit of work).
// `lds` is the dynamic LDS of a workgroup.
uint32_t persistent_grid(const void *kernel, int block, size_t work, size_t lds = 0);

// Reduced-precision kernels (arithmetic policies of prec.hpp): a lane
// kernel for square M2L up to kPrecLaneMax and a generic kernel for every
// operator and order up to kPrecMaxOrder.
inline constexpr uint32_t kPrecLaneMax = 16;    // FP32
inline constexpr uint32_t kPrecLaneMaxDW = 10;  // double-word FP32
inline constexpr uint32_t kPrecMaxOrder = 24;
hipError_t launch_prec_lane_m2l(int precision, uint32_t P, const sfmm_item *items, size_t n, const double *src,
                                double *dst, hipStream_t stream, int acc);
hipError_t launch_prec_generic(int precision, int op, uint32_t pc, const sfmm_item *items, size_t n,
                               const double *src, double *dst, hipStream_t stream, int acc);
// FP32 square M2L on the matrix cores, orders 1..kPrecMaxOrder
// (mfma_prec.hip).  FP32 contexts use it above kPrecLaneAutoMax.
inline constexpr uint32_t kPrecLaneAutoMax = 16;
hipError_t launch_prec_mfma_m2l(uint32_t P, const sfmm_item *items, size_t n, const double *src, double *dst,
                                hipStream_t stream, int acc);

// Team kernels (team.hpp): items of any orders up to pc <= kTeamMax; mode as
// there.
inline constexpr uint32_t kTeamMax = 48;
hipError_t launch_team(int op, uint32_t pc, const sfmm_item *items, size_t n, const double *src, double *dst,
                       hipStream_t stream, int mode);

// Octet kernels (octet.hpp): items of any orders up to pb <= max_order(OP);
// mode as there.
namespace octet {
// M2L lists above it all go to the team kernels (team_items)
constexpr int max_order(int op) { return op == SFMM_M2L ? 22 : 24; }
template <int OP>
hipError_t launch_op(uint32_t pb, const sfmm_item *items, size_t n, const double *src, double *dst,
                     hipStream_t stream, int mode, bool pairs);
// Orders whose kernels have a variant with runs of up to two groups (`pairs`).
inline constexpr uint32_t kPairsMin = 13, kPairsMax = 17;
}  // namespace octet

// Largest list of orders up to pb that the MFMA family sends to the team
// kernel instead of the octet kernel (translate.hip has the figures).
size_t team_items(int op, uint32_t pb);

// Launches above kLaneAutoMax that stay on lanes: n items of distinct targets
// (shared: whose list reads a source twice or more on average), and n of the
// `total` items of a plan of repeated targets that are `runs` runs in lane
// waves.
bool lanes_ahead(int op, uint32_t pb, size_t n, bool shared);
bool lanes_for_runs(int op, uint32_t pb, size_t n, size_t runs, size_t total);

// Kernels of the plans of the fewest scratch blocks: up to order 12 lanes, with
// runs of 64, above it team kernels or octets in pairs, with runs of 16.  Pairs
// take lists that fill the chip twice over where a team takes longer than the
// former one-wave-per-16 kernel did: M2L of 300,000 items in runs of 24, that
// kernel, team, pairs, octets (us): order 14 487, 552, 349, 326; 16 601, 597,
// 434, 412; 18 992, 820, 720, 700.
inline constexpr uint32_t kLaneSmallPlan = kLaneMax;
constexpr bool octet_pairs(uint32_t pb, size_t n)
{
    return pb >= octet::kPairsMin && pb <= octet::kPairsMax && n > 32768;
}

// Launch bucket of an FP64 item of the generic family, by its larger order:
// 32 (orders 25 to 32) and kTeamMax (33 to 48) run on team kernels of their
// own registers and LDS, everything else together on the generic kernel (all
// of them in a context that asks for it: then the team kernels have a path of
// other steps to be compared with).
inline constexpr uint32_t kGenericRest = 0;
uint32_t generic_bucket(uint32_t pb);

// One launch of a plan: family (not kAuto), the kernel's order bound pk,
// whether items carry their own orders (rt), the arithmetic (SFMM_FP64,
// SFMM_FP32, SFMM_SPLIT32) and whether targets accumulate (acc) or are
// overwritten with the translation (scratch blocks of a segmented
// reduction).  The generic kernels always read per-item orders; pk is then
// the largest order of the group.
struct KernelChoice {
    int family;
    uint32_t pk;
    bool rt;
    int precision = SFMM_FP64;
    bool acc = true;
    // scratch mode with runs of one target's items sharing a block (FP64
    // lane, team and octet kernels; the plan lays the runs out)
    bool seg = false;
    // lane kernels: the runs are long_runs
    bool long_runs = false;
    // MFMA and generic families: the team kernels, not the octet and generic
    // ones.  Decided with the runs, which are as long as the kernel's groups.
    bool team = false;
    // octet kernels: the variant with runs of up to two groups
    bool pairs = false;
};

// Segmented reduction: target block t += sum of its items' scratch blocks,
// in list order.  Both arrays are device memory.
struct RedTarget {
    uint64_t dst;    // offset (reals) of the target block in the target pool
    uint32_t first;  // first entry of the target's items in RedItem[]
    uint32_t count;  // number of items
    uint32_t len;    // reals to add (the longest of the items' blocks)
    uint32_t pad;
};
struct RedItem {
    uint64_t off;  // offset (reals) of the item's block in the scratch pool
    uint32_t len;  // reals the translation wrote
    uint32_t pad;
};
hipError_t launch_reduce(const RedTarget *targets, size_t n_targets, const RedItem *items, const double *scratch,
                         double *dst, hipStream_t stream);

// Enqueue dst += T(src) for n device-resident items with pairwise distinct
// targets and orders within `k`.
hipError_t launch_kernel(int op, const KernelChoice &k, const sfmm_item *items, size_t n, const double *src,
                         double *dst, hipStream_t stream);

// The generic kernel: items of any orders up to `pc`.
hipError_t launch_generic(int op, uint32_t pc, const sfmm_item *items, size_t n, const double *src, double *dst,
                          hipStream_t stream, int acc = 1);

// Particle-side operators over device-resident cells (particles.hip).
// dim: values per point and blocks per cell, 1..kMaxParticleDim.
inline constexpr int kMaxParticleDim = 4;
// What the launches need to know of a set's cells.
struct CellCounts {
    size_t cells = 0;
    uint32_t max_order = 0;
    uint32_t most = 0;                // points of the largest cell
    uint64_t points = 0, chunks = 0;  // sums of count and ceil(count / 64)
    bool mixed = false;               // cells of several orders
    double walk = 0.0, single = 0.0;  // L2P's work by runs and by cells (particles.hip)
};
CellCounts count_cells(const sfmm_cell *cells, size_t n, int dim);
hipError_t launch_p2m(const double *pts, const sfmm_cell *cells, const CellCounts &counts, double *pool, int dim,
                      hipStream_t stream);
hipError_t launch_l2p(const double *pts, const sfmm_cell *cells, const CellCounts &counts, const double *pool,
                      double *phi, double *grad, int dim, hipStream_t stream);

}  // namespace sfmm
