// Particle-side operators on either side of the translations, batched over
// cells, for D-valued expansions (D blocks per cell, D charges per point):
//   P2M  M_{c,d} += sum_{i in c} q_{i,d} R(P_c, p_i - c)
//   L2P  phi_{i,d} += dot(L_{c,d}, R(P_c, p_i - c)),
//        grad_{i,d} += dot(L_{c,d}, dR(...))
// In the reference these are user code over harmonics::R / dR and
// solid::fmadd / dot (harmonics.cpp:31-174, solid.cpp:40-105, the pattern of
// tests/test_m2l.cpp:70-116).
//
// R follows the reference's recurrences: the diagonal R_m^m from
// R_{m-1}^{m-1} (x + iy)/(2m), then down each column R_{m+1}^m = z R_m^m and
// (n+m)(n-m) R_n^m = (2n-1) z R_{n-1}^m - |x|^2 R_{n-2}^m; dR is the same
// recurrence differentiated term by term.
//
// Both kernels: one wave per run of up to kRun consecutive cells.  The cells'
// points follow each other in quads of lanes (a cell starts a new quad, so
// every quad belongs to one cell), 64 lanes to a chunk.  Each lane walks the
// columns of R once for its own point, O(P^2) steps, and leaves the values
// in LDS, two rows (re, im) a coefficient; after every kGroup coefficients
// the contraction over them runs on v_mfma_f64_4x4x4_4b_f64:
//   P2M  M[row][d] = sum_points R[row][point] q[point][d]: 16 rows by the
//        (up to four) charges, four points of one cell a step;
//   L2P  out[point][j] = sum_rows R[row][point] H[row][j]: 16 points by
//        (phi, d/dx, d/dy, d/dz), four rows a step, H the cell's
//        coefficients rearranged by
//          d/dz R_n^m = R_{n-1}^m,
//          (d/dx -+ i d/dy) R_n^m = +-R_{n-1}^{m-+1},
//        so the gradient needs no recurrence of its own.  The instruction's
//        four blocks are four quads, each with the H of its own cell.
// What bounds them: the FP64 pipe and the latency of a wave's chunk (the
// registers leave three waves per SIMD, two of L2P with more than one charge).
// The kernels per cell (one lane per coefficient with its own O(n) recurrence
// per point, P2M; one lane per point with the gradient's recurrences, L2P) take
// longer where a cell's points are no match for their lanes: P2M of 250,000
// points, order 8, three charges, 24 a cell 157 and 42 us (the multiplications
// would take 4 us, the bytes 10), L2P of 500,000 points, order 10, 32 a cell
// on average 115 and 75 us (11 and 12 us).  They stay for the sets that
// per_cell_p2m and per_cell_l2p name.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/solidfmm_gpu.h"
#include "tables.hpp"
#include "translate.hpp"

namespace sfmm {
namespace {

constexpr int kRun = 8;            // cells per wave at most
constexpr int kGroup = 8;          // coefficients per contraction
constexpr int kRows = 2 * kGroup;
constexpr int kWalkMax = 32;       // largest order with a walk table
// Below this order (the largest of a set) L2P's few columns do not pay for the
// exchange through LDS: 300,000 points of order 3, 128 a cell, take 16 us a
// point per lane and 21 us on the walk; 1,000,000 of order 4, 8 a cell, 158
// and 72.
constexpr int kWalkMinL2P = 4;
// Row strides (doubles) of R in LDS that spread the operands' lanes over all
// banks: 16 rows by 4 points (P2M), 4 rows by 16 points (L2P).
constexpr int kStrideP2M = 68, kStrideL2P = 72;

// 1/k for the recurrences' divisors (2j on the diagonal, (n+m)(n-m) =
// (n+m) times (n-m) down a column), so the inner loops multiply instead of
// divide.
constexpr int kInvSize = 2 * 88;  // n + m < 2 * 86 for every order the library takes
struct InvTable {
    double v[kInvSize];
};
constexpr InvTable make_inv()
{
    InvTable t{};
    for (int k = 1; k < kInvSize; ++k) t.v[k] = 1.0 / k;
    return t;
}
__constant__ constexpr InvTable kInv = make_inv();

// Orders the LDS writes and reads of the wave's lanes (they run in program
// order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double mfma4(double a, double b, double c)
{
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// The cells of a wave: lane g holds cell g of the run.
struct Run {
    sfmm_cell cell;
    int start, quads;    // first quad of the cell in the run, number of them
    int first[kRun + 1];  // the same, wave-uniform; cells past the run are empty
    int order;           // largest order of the run
    bool mixed;          // cells of several orders

    __device__ __forceinline__ void load(const sfmm_cell *__restrict__ cells, uint32_t c0, uint32_t n)
    {
        const int lane = threadIdx.x;
        cell = sfmm_cell{};
        if (uint32_t(lane) < n) cell = cells[c0 + lane];
        quads = int(cell.count / 4 + (cell.count % 4 != 0));
        int sum = quads, p = cell.count ? int(cell.order) : 0;
        for (int d = 1; d < kRun; d *= 2) {
            const int v = __shfl_up(sum, d, 64);
            sum += lane >= d ? v : 0;
        }
        start = sum - quads;
        order = 0;
        for (int g = 0; g < kRun; ++g) {
            first[g] = __builtin_amdgcn_readlane(start, g);
            order = max(order, __builtin_amdgcn_readlane(p, g));
        }
        mixed = __ballot(cell.count != 0 && p != order) != 0;
        first[kRun] = __builtin_amdgcn_readlane(sum, kRun - 1);
    }
    // cell of quad k (the last non-empty one at or before it)
    __device__ __forceinline__ int of_quad(int k) const
    {
        int g = 0;
#pragma unroll
        for (int j = 1; j < kRun; ++j) g += k >= first[j] ? 1 : 0;
        return g;
    }
    // point of quad k, lane i of it, in cell g; -1: none
    __device__ __forceinline__ int64_t point(int k, int i, int g) const
    {
        const uint32_t j = 4u * uint32_t(k - __shfl(start, g, 64)) + uint32_t(i);
        const uint32_t n = __shfl(cell.count, g, 64), f = __shfl(cell.first, g, 64);
        return k < first[kRun] && j < n ? int64_t(f) + j : -1;
    }
};

// P2M without a walk, one wave per cell: one lane per coefficient, which goes
// over the points and evaluates its own R_n^m.
template <int D>
__global__ void __launch_bounds__(64)
    k_p2m_cell(const double *__restrict__ pts, const sfmm_cell *__restrict__ cells, uint32_t n_cells,
               double *__restrict__ pool)
{
    constexpr int W = 3 + D;  // doubles per point
    for (uint32_t c = blockIdx.x; c < n_cells; c += gridDim.x) {
        const sfmm_cell cell = cells[c];
        const int P = int(cell.order);
        const int ncoef = P * (P + 1) / 2;
        double *__restrict__ M = pool + cell.offset;
        for (int k = threadIdx.x; k < ncoef; k += 64) {
            int n = int((sqrt(8.0 * k + 1.0) - 1.0) * 0.5);
            while (n * (n + 1) / 2 > k) --n;
            while ((n + 1) * (n + 2) / 2 <= k) ++n;
            const int m = k - n * (n + 1) / 2;
            double sr[D], si[D];
            for (int d = 0; d < D; ++d) sr[d] = si[d] = 0.0;
            for (uint32_t i = 0; i < cell.count; ++i) {
                const double *p = pts + W * size_t(cell.first + i);
                const double x = p[0] - cell.x, y = p[1] - cell.y, z = p[2] - cell.z;
                // diagonal: R_0^0 = 1, R_1^1 = (x + iy)/2, R_j^j = R_{j-1}^{j-1} (x + iy)/(2j)
                double dr = 1.0, di = 0.0;
                if (m >= 1) {
                    dr = x / 2;
                    di = y / 2;
                }
                for (int j = 2; j <= m; ++j) {
                    const double f = kInv.v[2 * j];
                    const double a = dr, b = di;
                    dr = (a * x - b * y) * f;
                    di = (a * y + b * x) * f;
                }
                double ar = dr, ai = di;  // R_n^m, walking down column m
                if (n > m) {
                    double br = ar, bi = ai;  // R_{n-2}^m, R_{n-1}^m
                    ar = z * ar;
                    ai = z * ai;
                    const double r2 = x * x + y * y + z * z;
                    for (int nn = m + 2; nn <= n; ++nn) {
                        const double f = kInv.v[nn + m] * kInv.v[nn - m];
                        const double tr = (ar * z * (2 * nn - 1) - r2 * br) * f;
                        const double ti = (ai * z * (2 * nn - 1) - r2 * bi) * f;
                        br = ar;
                        bi = ai;
                        ar = tr;
                        ai = ti;
                    }
                }
                for (int d = 0; d < D; ++d) {
                    sr[d] = fma(p[3 + d], ar, sr[d]);
                    si[d] = fma(p[3 + d], ai, si[d]);
                }
            }
            const int kr = n * (n + 1) + m, ki = (n + 1) * (n + 1) + m;
            for (int d = 0; d < D; ++d) {
                double *Md = M + d * P * (P + 1);
                Md[kr] = Md[kr] + sr[d];
                Md[ki] = Md[ki] + si[d];
            }
        }
    }
}

// L2P without a walk, one wave per cell: one lane per point, which goes down
// the columns with running values of R and its gradient.
template <int D>
__global__ void __launch_bounds__(64)
    k_l2p_cell(const double *__restrict__ pts, const sfmm_cell *__restrict__ cells, uint32_t n_cells,
               const double *__restrict__ pool, double *__restrict__ phi, double *__restrict__ grad)
{
    constexpr int W = 3 + D;  // doubles per point
    for (uint32_t c = blockIdx.x; c < n_cells; c += gridDim.x) {
        const sfmm_cell cell = cells[c];
        const int P = int(cell.order);
        const double *__restrict__ L = pool + cell.offset;
        for (uint32_t i0 = 0; i0 < cell.count; i0 += 64) {
            const uint32_t i = i0 + threadIdx.x;
            const bool valid = i < cell.count;
            const double *p = pts + W * size_t(cell.first + (valid ? i : 0));
            const double x = p[0] - cell.x, y = p[1] - cell.y, z = p[2] - cell.z;
            const double r2 = x * x + y * y + z * z;
            // running diagonal value and gradient: R_m^m, d/dx, d/dy, d/dz
            double dr = 1.0, di = 0.0, gdr[3] = {0.0, 0.0, 0.0}, gdi[3] = {0.0, 0.0, 0.0};
            double f0[D], g[D][3];
            for (int d = 0; d < D; ++d) f0[d] = g[d][0] = g[d][1] = g[d][2] = 0.0;
            for (int m = 0; m < P; ++m) {
                if (m == 1) {
                    dr = x / 2;
                    di = y / 2;
                    gdr[0] = 0.5;
                    gdi[1] = 0.5;
                } else if (m >= 2) {
                    const double f = kInv.v[2 * m];
                    const double a = dr, b = di;
                    const double ax = gdr[0], ay = gdr[1], az = gdr[2], bx = gdi[0], by = gdi[1], bz = gdi[2];
                    dr = (a * x - b * y) * f;
                    gdr[0] = (ax * x + a - bx * y) * f;
                    gdr[1] = (ay * x - by * y - b) * f;
                    gdr[2] = (az * x - bz * y) * f;
                    di = (a * y + b * x) * f;
                    gdi[0] = (ax * y + bx * x + b) * f;
                    gdi[1] = (ay * y + a + by * x) * f;
                    gdi[2] = (az * y + bz * x) * f;
                }
                // dot weight: 2 for m >= 1, 1 for m == 0 (solid.cpp:51-66)
                const double w = m ? 2.0 : 1.0;
                // column m: a = R_n^m, b = R_{n-1}^m (with gradients)
                double ar = dr, ai = di, gar[3] = {gdr[0], gdr[1], gdr[2]}, gai[3] = {gdi[0], gdi[1], gdi[2]};
                double br = 0.0, bi = 0.0, gbr[3] = {0.0, 0.0, 0.0}, gbi[3] = {0.0, 0.0, 0.0};
                for (int n = m; n < P; ++n) {
                    if (n == m + 1) {  // R_{m+1}^m = z R_m^m
                        br = ar;
                        bi = ai;
                        for (int d = 0; d < 3; ++d) {
                            gbr[d] = gar[d];
                            gbi[d] = gai[d];
                        }
                        ar = z * br;
                        ai = z * bi;
                        for (int d = 0; d < 3; ++d) {
                            gar[d] = z * gbr[d];
                            gai[d] = z * gbi[d];
                        }
                        gar[2] += br;
                        gai[2] += bi;
                    } else if (n >= m + 2) {
                        const double f = kInv.v[n + m] * kInv.v[n - m];
                        const double k2 = 2.0 * n - 1.0;
                        const double tr = (ar * z * k2 - r2 * br) * f;
                        const double ti = (ai * z * k2 - r2 * bi) * f;
                        double tgr[3], tgi[3];
                        for (int d = 0; d < 3; ++d) {
                            const double r2d = d == 0 ? 2 * x : d == 1 ? 2 * y : 2 * z;
                            tgr[d] = gar[d] * z * k2 - r2d * br - r2 * gbr[d];
                            tgi[d] = gai[d] * z * k2 - r2d * bi - r2 * gbi[d];
                        }
                        tgr[2] += ar * k2;
                        tgi[2] += ai * k2;
                        br = ar;
                        bi = ai;
                        ar = tr;
                        ai = ti;
                        for (int d = 0; d < 3; ++d) {
                            gbr[d] = gar[d];
                            gbi[d] = gai[d];
                            gar[d] = tgr[d] * f;
                            gai[d] = tgi[d] * f;
                        }
                    }
                    for (int d = 0; d < D; ++d) {
                        const double *Ld = L + d * P * (P + 1);
                        const double lr = Ld[n * (n + 1) + m], li = Ld[(n + 1) * (n + 1) + m];
                        f0[d] = fma(w * lr, ar, fma(w * li, ai, f0[d]));
                        for (int k = 0; k < 3; ++k) g[d][k] = fma(w * lr, gar[k], fma(w * li, gai[k], g[d][k]));
                    }
                }
            }
            if (valid) {
                const size_t j = cell.first + i;
                for (int d = 0; d < D; ++d) {
                    phi[j * D + d] += f0[d];
                    if (grad) {
                        grad[3 * (j * D + d)] += g[d][0];
                        grad[3 * (j * D + d) + 1] += g[d][1];
                        grad[3 * (j * D + d) + 2] += g[d][2];
                    }
                }
            }
        }
    }
}

// The walk over the coefficients of an order-P block: degrees m..P-1 of order
// m, column by column, in groups of kGroup.  A step that starts a column
// takes R_m^m and makes R_{m+1}^{m+1} = c (x + iy) R_m^m, c = 1/(2m+2); the
// others are R_n^m = z c R_{n-1}^m - |x|^2 f R_{n-2}^m with
// f = 1/((n+m)(n-m)) and c = (2n-1) f (c = 1 at n = m+1, where R_{n-2}^m is
// zero).  Past the last coefficient c = f = 0 and nm has n = P.
struct Step {
    double c, f;
};
constexpr int walk_groups(int P) { return (P * (P + 1) / 2 + kGroup - 1) / kGroup; }
constexpr int walk_offset(int P)  // one group of padding each, read ahead
{
    int s = 0;
    for (int p = 1; p < P; ++p) s += (walk_groups(p) + 1) * kGroup;
    return s;
}
struct Walks {
    Step step[walk_offset(kWalkMax + 1)];
    uint16_t nm[walk_offset(kWalkMax + 1)];  // (n << 8) | m
    uint32_t starts[walk_offset(kWalkMax + 1) / kGroup];  // bit k: the group's step k starts a column
    int offset[kWalkMax + 1];
};
constexpr Walks make_walks()
{
    Walks w{};
    int at = 0;
    for (int P = 1; P <= kWalkMax; ++P) {
        w.offset[P] = at;
        const int end = at + (walk_groups(P) + 1) * kGroup;
        for (int m = 0; m < P; ++m)
            for (int n = m; n < P; ++n, ++at) {
                w.nm[at] = uint16_t((n << 8) | m);
                if (n == m) w.starts[at / kGroup] |= 1u << (at % kGroup);
                if (n == m) w.step[at] = {1.0 / (2 * m + 2), 0.0};
                else w.step[at] = {double(2 * n - 1) / double((n + m) * (n - m)), 1.0 / double((n + m) * (n - m))};
            }
        for (; at < end; ++at) w.nm[at] = uint16_t(P << 8);
    }
    return w;
}
__constant__ constexpr Walks kWalks = make_walks();

// R of (x, y, z) along the walk of order P into rows 2k, 2k + 1 of `rows`
// (this lane's column of them); full(G) once group G is complete.  Degrees
// p.. of a lane are zero where MIXED.  A group's steps are straight-line
// code with their factors in scalar registers, loaded a group ahead: a loop
// over the degrees spent more time on branches and waits than on arithmetic.
template <int STRIDE, bool MIXED, class Full>
__device__ __forceinline__ void regular(double x, double y, double z, int p, int P, double *rows, Full &&full)
{
    const double r2 = x * x + y * y + z * z;
    const int off = kWalks.offset[P], groups = walk_groups(P);
    const Step *step = kWalks.step + off;
    const uint32_t *starts = kWalks.starts + off / kGroup;
    double dr = 1.0, di = 0.0, ar = 0.0, ai = 0.0, br = 0.0, bi = 0.0;
    int n = 0, m = 0;  // the step's degree, the next column
    Step next[kGroup];
    uint32_t next_starts = starts[0];
#pragma unroll
    for (int k = 0; k < kGroup; ++k) next[k] = step[k];
    for (int G = 0; G < groups; ++G) {
        Step now[kGroup];
        const uint32_t now_starts = next_starts;
        next_starts = starts[G + 1];
#pragma unroll
        for (int k = 0; k < kGroup; ++k) {
            now[k] = next[k];
            next[k] = step[kGroup * (G + 1) + k];
        }
#pragma unroll
        for (int k = 0; k < kGroup; ++k) {
            const double zc = z * now[k].c, rf = r2 * now[k].f;
            const double tr = ar * zc - br * rf, ti = ai * zc - bi * rf;
            br = ar;
            bi = ai;
            ar = tr;
            ai = ti;
            if (__builtin_expect((now_starts >> k) & 1, 0)) {
                ar = dr;
                ai = di;
                br = bi = 0.0;
                const double a = dr * now[k].c, b = di * now[k].c;
                dr = a * x - b * y;
                di = a * y + b * x;
            }
            double vr = ar, vi = ai;
            if constexpr (MIXED) {
                n = (now_starts >> k) & 1 ? m++ : n + 1;
                vr = n < p ? ar : 0.0;
                vi = n < p ? ai : 0.0;
            }
            rows[(2 * k) * STRIDE] = vr;
            rows[(2 * k + 1) * STRIDE] = vi;
        }
        full(G);
    }
}

// Doubles of one staged block per charge: the walk's rows, whole groups.
__host__ __device__ constexpr int staged_rows(int P) { return kRows * walk_groups(P); }

// Row of pool real e of a block in a walk of order P.
__device__ __forceinline__ int staged_row(int e, int P)
{
    int n = int((sqrtf(4.0f * float(e) + 1.0f) - 1.0f) * 0.5f);
    while (n * (n + 1) > e) --n;
    while ((n + 1) * (n + 2) <= e) ++n;
    const int r = e - n * (n + 1);
    const int part = r > n ? 1 : 0, m = part ? r - n - 1 : r;
    return 2 * (m * P - m * (m - 1) / 2 + n - m) + part;
}

// P2M of a run.
template <int D>
__device__ __forceinline__ void p2m_run(const double *__restrict__ pts, double *__restrict__ pool, const Run &cr,
                                        double *R, double *Q, double *stage)
{
    constexpr int W = 3 + D;  // doubles per point
    const int lane = threadIdx.x;
    const int row = lane & 15, k4 = lane >> 4;                  // operand: row, point of the quad
    const int orow = 4 * ((lane >> 2) & 3) + k4, d = lane & 3;  // result: row, charge
    const int rows = staged_rows(cr.order);
    for (int q0 = 0; q0 < cr.first[kRun]; q0 += 16) {
        const int g = cr.of_quad(q0 + (lane >> 2));
        const int64_t i = cr.point(q0 + (lane >> 2), lane & 3, g);
        double x = 0.0, y = 0.0, z = 0.0;
        const double ox = __shfl(cr.cell.x, g, 64), oy = __shfl(cr.cell.y, g, 64), oz = __shfl(cr.cell.z, g, 64);
        const int p = __shfl(cr.cell.order, g, 64);
#pragma unroll
        for (int c = 0; c < 4; ++c) Q[c * kStrideP2M + lane] = i >= 0 && c < D ? pts[W * i + 3 + c] : 0.0;
        if (i >= 0) {
            x = pts[W * i] - ox;
            y = pts[W * i + 1] - oy;
            z = pts[W * i + 2] - oz;
        }
        // quads that end their cell's part of the chunk, and those of them
        // whose cell began in an earlier chunk
        const int after = __shfl(g, (lane + 4) & 63, 64);  // every lane takes part
        const uint64_t ends =
            __ballot((lane & 3) == 0 && q0 + (lane >> 2) < cr.first[kRun] &&
                     (lane == 60 || q0 + (lane >> 2) + 1 == cr.first[kRun] || after != g));
        const uint64_t more = ends & __ballot(__shfl(cr.start, g, 64) < q0);
        wave_sync();
        double qv[16];  // the charges' operands
#pragma unroll
        for (int k = 0; k < 16; ++k) qv[k] = Q[d * kStrideP2M + 4 * k + k4];
        auto sums = [&](int G) {
            wave_sync();
            double *to = stage + d * rows + kRows * G + orow;
            // the quads' products first: they are independent, a chain of
            // products into one sum waits 45 clocks a link
            double part[16], sum = 0.0;
#pragma unroll
            for (int k = 0; k < 16; ++k) part[k] = R[row * kStrideP2M + 4 * k + k4];
#pragma unroll
            for (int k = 0; k < 16; ++k) part[k] = mfma4(part[k], qv[k], 0.0);
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                sum += part[k];
                if ((ends >> (4 * k)) & 1) {
                    double *at = to + __builtin_amdgcn_readlane(g, 4 * k) * (D * rows);
                    if (d < D) *at = ((more >> (4 * k)) & 1) ? *at + sum : sum;
                    sum = 0.0;
                }
            }
            wave_sync();
        };
        if (cr.mixed) regular<kStrideP2M, true>(x, y, z, p, cr.order, R + lane, sums);
        else regular<kStrideP2M, false>(x, y, z, p, cr.order, R + lane, sums);
        // the blocks of the cells that end here go to the pool
        for (uint64_t left = ends; left; left &= left - 1) {
            const int c = __builtin_amdgcn_readlane(g, __builtin_ctzll(left));
            if (__shfl(cr.start, c, 64) + __shfl(cr.quads, c, 64) > q0 + 16) continue;
            const int P = __builtin_amdgcn_readlane(int(cr.cell.order), c), len = P * (P + 1);
            double *M = pool + __shfl(cr.cell.offset, c, 64);
            for (int e = lane; e < len; e += 64) {
                const double *from = stage + c * (D * rows) + staged_row(e, cr.order);
                double old[D];
                static_for<0, D>([&](auto bc) { old[decltype(bc)::value] = M[decltype(bc)::value * len + e]; });
                static_for<0, D>([&](auto bc) {
                    constexpr int b = decltype(bc)::value;
                    M[b * len + e] = old[b] + from[b * rows];
                });
            }
        }
        wave_sync();
    }
}

// Doubles of a cell's H, [d][row][phi, d/dx, d/dy, d/dz], off a multiple of the
// banks' width so that blocks of two cells read different banks.
template <int D>
constexpr int kCellH = D * kRows * 4 + 16;

// L2P of a run.
template <int D>
__device__ __forceinline__ void l2p_run(const double *__restrict__ pts, const double *__restrict__ pool,
                                        double *__restrict__ phi, double *__restrict__ grad, const Run &cr, double *R,
                                        double *H, int64_t *at)
{
    constexpr int W = 3 + D;  // doubles per point
    const int lane = threadIdx.x;
    // operands and results: tile u is points 16 u.., the lane's block of it
    // is quad 4 u + block
    const int block = (lane >> 2) & 3, k4 = lane >> 4, col = lane & 3;
    for (int q0 = 16 * int(blockIdx.y); q0 < cr.first[kRun]; q0 += 16 * int(gridDim.y)) {
        const int g = cr.of_quad(q0 + (lane >> 2));
        const int64_t i = cr.point(q0 + (lane >> 2), lane & 3, g);
        double x = 0.0, y = 0.0, z = 0.0;
        const double ox = __shfl(cr.cell.x, g, 64), oy = __shfl(cr.cell.y, g, 64), oz = __shfl(cr.cell.z, g, 64);
        const int p = __shfl(cr.cell.order, g, 64);
        if (i >= 0) {
            x = pts[W * i] - ox;
            y = pts[W * i + 1] - oy;
            z = pts[W * i + 2] - oz;
        }
        at[lane] = i;
        // H is filled by eight cells (from the chunk's first) by eight
        // coefficients
        const int gmin = __builtin_amdgcn_readlane(g, 0);
        const int hc = min(gmin + (lane >> 3), kRun - 1), k = lane & 7;
        const int hstart = __shfl(cr.start, hc, 64);
        const bool hon = gmin + (lane >> 3) < kRun && hstart < q0 + 16;
        const int hp = __shfl(cr.cell.order, hc, 64);
        const double *L = pool + __shfl(cr.cell.offset, hc, 64);
        const int stride = hp * (hp + 1);
        int hb[4];
        double acc[4][D];
        static_for<0, 4>([&](auto uc) {
            constexpr int u = decltype(uc)::value;
            hb[u] = (__shfl(g, 4 * (4 * u + block), 64) - gmin) * kCellH<D> + k4 * 4 + col;
            static_for<0, D>([&](auto dc) { acc[u][decltype(dc)::value] = 0.0; });
        });
        // the cell's coefficients that a group needs, fetched a group ahead
        double2 c[D], up[D], right[D], left[D];  // L_n^m, L_{n+1}^m, L_{n+1}^{m+1}, L_{n+1}^{m-1}
        int m = 0;
        const uint16_t *nms = kWalks.nm + kWalks.offset[cr.order] + k;
        int nm = nms[0];
        auto fetch = [&](int G) {
            const int n = nm >> 8;
            m = nm & 255;
            nm = nms[kGroup * (G + 1)];
            const bool here = hon && n < hp, above = hon && n + 1 < hp;
            const double *re = L + (n * (n + 1) + m);
            const int nu = 2 * (n + 1);  // from L_n^m to L_{n+1}^m
            static_for<0, D>([&](auto dc) {
                constexpr int d = decltype(dc)::value;
                const double *b = re + d * stride;
                c[d] = up[d] = right[d] = left[d] = double2{0.0, 0.0};
                if (here) c[d] = double2{b[0], b[n + 1]};
                if (above) {
                    up[d] = double2{b[nu], b[nu + n + 2]};
                    right[d] = double2{b[nu + 1], b[nu + n + 3]};
                    if (m > 0) left[d] = double2{b[nu - 1], b[nu + n + 1]};
                }
            });
        };
        const int groups = walk_groups(cr.order);
        fetch(0);
        auto sums = [&](int G) {
            const double w = m ? 2.0 : 1.0;  // dot weight (solid.cpp:51-66)
            static_for<0, D>([&](auto dc) {
                constexpr int d = decltype(dc)::value;
                const double im = m == 1 ? 0.0 : left[d].y;  // Im L_n^0 does not count
                double2 *h = reinterpret_cast<double2 *>(H + (lane >> 3) * kCellH<D> + d * kRows * 4 + 2 * k * 4);
                h[0] = double2{w * c[d].x, right[d].x - left[d].x};
                h[1] = double2{right[d].y + im, w * up[d].x};
                h[2] = double2{w * c[d].y, right[d].y - im};
                h[3] = double2{-(right[d].x + left[d].x), w * up[d].y};
            });
            wave_sync();
            if (G + 1 < groups) fetch(G + 1);
            static_for<0, 4>([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                double a[4];
                static_for<0, 4>([&](auto uc) {
                    a[decltype(uc)::value] = R[(4 * s + k4) * kStrideL2P + 16 * decltype(uc)::value + (lane & 15)];
                });
                static_for<0, D>([&](auto dc) {
                    constexpr int d = decltype(dc)::value;
                    static_for<0, 4>([&](auto uc) {  // four independent chains
                        constexpr int u = decltype(uc)::value;
                        acc[u][d] = mfma4(a[u], H[hb[u] + d * kRows * 4 + 16 * s], acc[u][d]);
                    });
                });
            });
            wave_sync();
        };
        // D > 1: one instance, two would cost registers and so waves in flight
        if (D > 1 || cr.mixed) regular<kStrideL2P, true>(x, y, z, p, cr.order, R + lane, sums);
        else regular<kStrideL2P, false>(x, y, z, p, cr.order, R + lane, sums);
        static_for<0, 4>([&](auto uc) {
            constexpr int u = decltype(uc)::value;
            const int64_t j = at[16 * u + 4 * block + k4];
            if (j >= 0 && (col == 0 || grad)) {
                static_for<0, D>([&](auto dc) {
                    constexpr int d = decltype(dc)::value;
                    double *o = col == 0 ? phi + (j * D + d) : grad + 3 * (j * D + d) + col - 1;
                    *o += acc[u][d];
                });
            }
        });
        wave_sync();
    }
}

template <int D>
__global__ void __launch_bounds__(64)
    k_p2m(const double *__restrict__ pts, const sfmm_cell *__restrict__ cells, uint32_t n_cells,
          double *__restrict__ pool, uint32_t run)
{
    __shared__ double R[kRows * kStrideP2M], Q[4 * kStrideP2M];
    extern __shared__ double stage[];  // [cell][charge][row]
    const uint32_t c0 = blockIdx.x * run, n = min(run, n_cells - c0);
    Run cr;
    cr.load(cells, c0, n);
    p2m_run<D>(pts, pool, cr, R, Q, stage);
}

template <int D>
__global__ void __launch_bounds__(64)
    k_l2p(const double *__restrict__ pts, const sfmm_cell *__restrict__ cells, uint32_t n_cells,
          const double *__restrict__ pool, double *__restrict__ phi, double *__restrict__ grad, uint32_t run)
{
    __shared__ double R[kRows * kStrideL2P];
    __shared__ double H[kRun * kCellH<D>];
    __shared__ int64_t at[64];
    const uint32_t c0 = blockIdx.x * run, n = min(run, n_cells - c0);
    Run cr;
    cr.load(cells, c0, n);
    l2p_run<D>(pts, pool, phi, grad, cr, R, H, at);
}

// Calls launch(first cell, cells, workgroups) for n_cells cells, `run` a
// workgroup of 64 threads, in launches of fewer than 2^32 threads.
template <class F>
void launch_runs(size_t n_cells, uint32_t run, F &&launch)
{
    const size_t most = (size_t(1) << 24) * run;
    for (size_t first = 0; first < n_cells; first += most) {
        const size_t n = std::min(n_cells - first, most);
        launch(first, uint32_t(n), uint32_t((n + run - 1) / run));
    }
}

// Cells per wave: about `waves` waves.  Over orders 4 to 16, 8 to 128 points a
// cell and 2,000 to 500,000 points, half as many take 0.61 to 1.25 of P2M's
// time (the least where 4,000 cells go two to a wave) and 0.85 to 1.38 of
// L2P's, twice as many 0.90 to 1.15 and 0.83 to 1.45.
uint32_t run_length(size_t n_cells, size_t waves)
{
    const size_t r = (n_cells + waves - 1) / waves;
    return r < 1 ? 1 : r > size_t(kRun) ? kRun : uint32_t(r);
}
constexpr size_t kWavesP2M = 5632, kWavesL2P = 1792;

// LDS (bytes) of P2M's staged blocks that leaves room for eight waves a CU.
constexpr size_t kStageBytes = 9 * 1024;

// P2M takes a wave per cell where the cells have so few points that the walk
// would mostly be for lanes without one: up to `few` and a half on average,
// four times `few` in the largest, which a wave goes through by itself.  Where
// the kernel per cell was no slower, in us against the walk's:
//   orders to 10, a cell's coefficients one pass of a wave: up to 6 while the
//   cells are in flight at once (30,000 points of order 8, one charge: 17 and
//   22 at 4 a cell, 21 and 14 at 12), 4 of very few cells; of many cells 2 or
//   3 from order 8 on, below it 1 and only up to two charges, since one
//   more charge costs the walk less;
//   above: 2 of few cells; of many 3 or 4, with one charge 1 and from order 20
//   on 2 to 4, as the staged blocks leave the walk fewer waves (200,000 points
//   of order 24, one charge: 1126 and 1634 at 3 a cell, 997 and 821 at 6).
// The walk takes every cell of a run to the largest order, so 2 are always few
// in sets of several (1,000,000 points, a quarter of the cells of order 16,
// the others of 5, one charge, 2 a cell: 1001 and 1721).
bool per_cell_p2m(const CellCounts &c, int dim)
{
    const uint32_t P = c.max_order;
    size_t few;
    if (P <= 10) {
        if (c.cells <= 512) few = 4;
        else if (c.cells <= 32768) few = 6;
        else if (P >= 8) few = dim >= 3 && P > 8 ? 3 : 2;
        else few = dim <= 2 ? 1 : 0;
    } else if (c.cells < 1024) few = 2;
    else if (dim == 1) few = P >= 24 ? 4 : P >= 20 ? 2 : 1;
    else few = P >= 16 || dim == 4 ? 4 : 3;
    if (c.mixed) few = std::max(few, size_t(2));
    return 2 * c.points <= (2 * few + 1) * c.cells && c.most <= 4 * few;
}

// L2P takes a wave per cell where cells fill their own chunks of 64 lanes so
// well that the walk, whose runs share chunks, has few less to go through, or
// where it would take cells of low orders to the run's largest.  A chunk's
// work by its order is chunk_work in the kernel per cell and as much over
// (share + slope (order - 4)) on the walk; CellCounts holds the sums of both.
// The cells must fill the chip as well, from `cells` times the order on for
// cells of one chunk.  The lines are fitted to the times of both kernels at
// orders 4 to 32, 1 to 1,000 points a cell and 2,000 to 1,000,000 points,
// where the chosen one is on average 0.4 % behind the faster, 0.7 % in sets of
// two orders.  1,000,000 points of order 8, three charges, per cell and on the
// walk: 131 and 210 us at 64 points a cell, 311 and 164 at 24; of order 10,
// one charge, 123 and 97 at 64; a quarter of the cells of order 10, the
// others of 3, three charges, 64 a cell on average, 191 and 313.
struct Line {
    double share, slope;
    uint32_t cells;
};
constexpr Line kLine[kMaxParticleDim] = {{0.40, 0.15, 375}, {0.45, 0.06, 256}, {0.35, 0.08, 192}, {0.40, 0.03, 128}};
double chunk_work(uint32_t order) { return double(order) * (order + 1) + 20.0; }

// Order 4 with all chunks in flight at once gains nothing from the exchange
// through LDS with more than one charge (30,000 points, three charges, 24 a
// cell: 8.8 and 10.9; 60,000 points, one charge, 12 a cell: 10.0 and 9.0).
bool per_cell_l2p(const CellCounts &c, int dim)
{
    if (c.max_order <= 4 && dim > 1 && c.most <= 64 && c.cells <= 5120) return true;
    const uint64_t deepest = c.most / 64 + (c.most % 64 != 0);
    return c.walk >= c.single && c.chunks >= deepest * kLine[dim - 1].cells * c.max_order;
}

template <int D>
hipError_t p2m_d(const double *pts, const sfmm_cell *cells, const CellCounts &c, double *pool, hipStream_t stream)
{
    if (c.max_order > kWalkMax || per_cell_p2m(c, D)) {
        const uint32_t grid = persistent_grid(reinterpret_cast<const void *>(&k_p2m_cell<D>), 64, c.cells);
        hipLaunchKernelGGL(k_p2m_cell<D>, dim3(grid), dim3(64), 0, stream, pts, cells, uint32_t(c.cells), pool);
        return hipGetLastError();
    }
    const size_t block = size_t(staged_rows(int(c.max_order))) * D * sizeof(double);
    const size_t fit = std::max(block ? kStageBytes / block : kRun, size_t(1));
    const uint32_t run = std::min(run_length(c.cells, kWavesP2M), uint32_t(fit));
    launch_runs(c.cells, run, [&](size_t first, uint32_t n, uint32_t groups) {
        hipLaunchKernelGGL(k_p2m<D>, dim3(groups), dim3(64), run * block, stream, pts, cells + first, n, pool, run);
    });
    return hipGetLastError();
}

template <int D>
hipError_t l2p_d(const double *pts, const sfmm_cell *cells, const CellCounts &c, const double *pool, double *phi,
                 double *grad, hipStream_t stream)
{
    if (c.max_order < kWalkMinL2P || c.max_order > kWalkMax || per_cell_l2p(c, D)) {
        const uint32_t grid = persistent_grid(reinterpret_cast<const void *>(&k_l2p_cell<D>), 64, c.cells);
        hipLaunchKernelGGL(k_l2p_cell<D>, dim3(grid), dim3(64), 0, stream, pts, cells, uint32_t(c.cells), pool, phi,
                           grad);
        return hipGetLastError();
    }
    const uint32_t run = run_length(c.cells, kWavesL2P);
    // few cells: a run's chunks side by side, 30,000 points of order 10, 128 a
    // cell, 10.9 us, one after the other 28.9
    const uint32_t split = c.cells < 2048 ? 4 : 1;
    launch_runs(c.cells, run, [&](size_t first, uint32_t n, uint32_t groups) {
        hipLaunchKernelGGL(k_l2p<D>, dim3(groups, split), dim3(64), 0, stream, pts, cells + first, n, pool, phi, grad,
                           run);
    });
    return hipGetLastError();
}

}  // namespace

CellCounts count_cells(const sfmm_cell *cells, size_t n, int dim)
{
    CellCounts c;
    c.cells = n;
    const Line &line = kLine[dim - 1];
    const uint32_t run = run_length(n, kWavesL2P);
    uint32_t some = 0;  // order of a cell with points
    for (size_t first = 0; first < n; first += run) {
        uint64_t quads = 0;
        uint32_t order = 0;
        for (size_t i = first; i < std::min(n, first + run); ++i) {
            const sfmm_cell &cell = cells[i];
            c.max_order = std::max(c.max_order, cell.order);
            if (cell.count == 0) continue;
            const uint32_t chunks = cell.count / 64 + (cell.count % 64 != 0);
            c.most = std::max(c.most, cell.count);
            c.points += cell.count;
            c.chunks += chunks;
            c.single += chunks * chunk_work(cell.order);
            c.mixed = c.mixed || (some && some != cell.order);
            some = cell.order;
            quads += cell.count / 4 + (cell.count % 4 != 0);
            order = std::max(order, cell.order);
        }
        c.walk += double((quads + 15) / 16) * chunk_work(order) /
                  (line.share + line.slope * double(std::max(order, 4u) - 4));
    }
    return c;
}

hipError_t launch_p2m(const double *pts, const sfmm_cell *cells, const CellCounts &counts, double *pool, int dim,
                      hipStream_t stream)
{
    if (counts.cells == 0) return hipSuccess;
    if (counts.cells > 0xFFFFFFFFull) return hipErrorInvalidValue;
    switch (dim) {
    case 1: return p2m_d<1>(pts, cells, counts, pool, stream);
    case 2: return p2m_d<2>(pts, cells, counts, pool, stream);
    case 3: return p2m_d<3>(pts, cells, counts, pool, stream);
    case 4: return p2m_d<4>(pts, cells, counts, pool, stream);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_l2p(const double *pts, const sfmm_cell *cells, const CellCounts &counts, const double *pool,
                      double *phi, double *grad, int dim, hipStream_t stream)
{
    if (counts.cells == 0) return hipSuccess;
    if (counts.cells > 0xFFFFFFFFull) return hipErrorInvalidValue;
    switch (dim) {
    case 1: return l2p_d<1>(pts, cells, counts, pool, phi, grad, stream);
    case 2: return l2p_d<2>(pts, cells, counts, pool, phi, grad, stream);
    case 3: return l2p_d<3>(pts, cells, counts, pool, phi, grad, stream);
    case 4: return l2p_d<4>(pts, cells, counts, pool, phi, grad, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace sfmm
