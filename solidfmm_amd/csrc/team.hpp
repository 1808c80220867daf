// FP64 translation kernel of a team of waves: one workgroup takes up to 16
// translations of any orders, its waves share the work by degree.
//
//   forward    wave w transforms its degrees n (scale, rotate by alpha, swap,
//              rotate by beta, swap) and leaves them in the triangle in LDS;
//   z          wave w translates its orders m along z, in place: column m of
//              the triangle (degrees K) becomes the column of output degrees
//              N, a matrix product with the weights (N+K)!, 1/(N-K)! or
//              1/(K-N)! on the matrix cores;
//   backward   wave w transforms its output degrees N back and adds them into
//              the targets.
//
// Algorithm: Dehnen's rotation scheme as in translations.cpp:36-471.  Lane
// (q, t) = t + 16 q holds translation t (a column of the matrix cores'
// operands) and the orders m = 2 (q + 4 j) + e of a degree, e the parity
// class: in the result registers of both FP64 matrix instructions lane
// (q, t) holds outputs q, q + 4, ..., which are the next product's input
// rows, so a degree stays in the same lanes from load to store.  A swap
// couples one class of inputs with one class of outputs per part, i.e. four
// dense blocks of half the degree's size instead of two half-empty ones of
// its full size (team_tables.hpp).
//
// Degrees are a run-time loop over a body per chunk count NJ = n/8 + 1 and
// parity of n, so code does not grow with the order (45 kB at order 32; the
// straight-line kernel would have 159 kB at order 24, more than the 64 kB
// instruction cache).  A lone group is bound by its chain of degrees, which
// the waves walk side by side; a full chip by the FP64 pipe that matrix and
// vector instructions share.  M2L of order 32: 2,003 translations 577 us on
// the one-workgroup-per-translation kernel, 38 us here; 30,000 7.7 ms and
// 0.34 ms (97 us would be the FP64 pipe's time at its measured 47 TFLOP/s).
// Orders up to 24 come here on lists too short to fill the chip with
// octet.hpp's groups (team_items): M2L of order 8, 500 translations took 8.8
// us on lanes and 5.2 here.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/solidfmm_gpu.h"
#include "tables.hpp"
#include "team_tables.hpp"
#include "translate.hpp"

namespace sfmm {
namespace team {

typedef double dbl4 __attribute__((ext_vector_type(4)));
// 16 bytes at 8-byte alignment
typedef double dbl2 __attribute__((ext_vector_type(2), aligned(8)));

// 16 outputs by 4 inputs: operand lane (q, r) = r + 16 q holds output r of
// input q, result element i of lane (q, t) is output q + 4 i.
__device__ __forceinline__ dbl4 mfma16(double a, double b, dbl4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// 4 outputs by 4 inputs for all 16 translations: operand lane l holds output
// l % 4 of input l / 16 (repeated for the instruction's four blocks, which
// are translations 0-3, 4-7, ...), lane (q, t) of the result is output q.
__device__ __forceinline__ double mfma4(double a, double b, double c)
{
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// Read in place of a block that a column does not load.
inline __device__ double kZeroBlock[kMaxOrder * (kMaxOrder + 1)];

// Largest value of v over the wave (0 <= v < 128), wave-uniform.
__device__ __forceinline__ int wave_max7(uint32_t v)
{
    uint32_t m = 0;
    for (int b = 6; b >= 0; --b) {
        const uint32_t cand = m | (1u << b);
        if (__ballot(v >= cand)) m = cand;
    }
    return int(m);
}

// The triangle in LDS is stored by order: column m holds degrees m..pc-1.
// Index of degree K of order m, less K.
__device__ __forceinline__ int column(int pc, int m) { return m * pc - m * (m - 1) / 2 - m; }

// Weight table of the z-translation in LDS, for orders up to pc: entry
// weight_pad + d holds the weight of d = N + K (M2L), N - K (M2M) or K - N
// (L2L), zero where there is none (operands reach 18 below the smallest d of
// M2M and L2L, and 18 above the largest).
constexpr int weight_pad(int op) { return op == SFMM_M2L ? 0 : 18; }
__host__ __device__ constexpr int weight_size(int op, int pc)
{
    return ((op == SFMM_M2L ? 2 * pc + 17 : pc + 33) + 1) & ~1;
}
// Kernels of this many chunks or more keep the rotation factors in LDS.
inline constexpr int kRotLds = 4;
__host__ __device__ constexpr int rot_size(int njx, int pc, int T) { return njx >= kRotLds ? 4 * pc * T : 0; }

struct cplx {
    double c, s;
};
__device__ __forceinline__ cplx mul(cplx a, cplx b) { return {a.c * b.c - a.s * b.s, a.s * b.c + a.c * b.s}; }

// Values in twice the precision (hi + lo).  A power of a rounded value is off
// by its error times the exponent, and by as much again where it comes from
// squarings: with angles in 64 bits, M2L of order 25 had a median error of
// 1.08e-14 a degree, 28 of 1.72e-14, where the one-workgroup kernel, which
// multiplies up, has 9.2e-15 and 1.42e-14; with these 8.7e-15 and 1.24e-14.
struct Wide {
    double hi, lo;
};
__device__ __forceinline__ Wide normal(double hi, double lo)
{
    const double h = hi + lo;
    return {h, lo - (h - hi)};
}
__device__ __forceinline__ Wide two_sum(double a, double b)
{
    const double s = a + b, bb = s - a;
    return {s, (a - (s - bb)) + (b - bb)};
}
__device__ __forceinline__ Wide two_prod(double a, double b)
{
    const double p = a * b;
    return {p, __builtin_fma(a, b, -p)};
}
__device__ __forceinline__ Wide mul(Wide a, Wide b)
{
    const Wide p = two_prod(a.hi, b.hi);
    return normal(p.hi, __builtin_fma(a.hi, b.lo, __builtin_fma(a.lo, b.hi, p.lo)));
}

// |(x, y, z)| and its inverse.
struct Distance {
    Wide r, inv;
};
__device__ __forceinline__ Distance distance(double x, double y, double z)
{
    const Wide xx = two_prod(x, x), yy = two_prod(y, y), zz = two_prod(z, z);
    const Wide s = two_sum(xx.hi, yy.hi), t = two_sum(s.hi, zz.hi);
    const double lo = t.lo + s.lo + (xx.lo + yy.lo + zz.lo);  // r^2 = t.hi + lo
    const double inv = 1.0 / sqrt(t.hi);
    Wide r = two_prod(t.hi, inv);
    r.lo += lo * inv;
    const Wide v = two_prod(r.hi, inv);
    const double e = (1.0 - v.hi) - v.lo - r.lo * inv;  // 1 - r^2 inv^2
    return {normal(r.hi, r.lo + 0.5 * e * r.hi), normal(inv, 0.5 * e * inv)};
}

// e^{i theta}, squared and once more.
struct Turn {
    Wide c, s;
};
__device__ __forceinline__ Turn square(const Turn &a)
{
    const Wide cc = two_prod(a.c.hi, a.c.hi), ss = two_prod(a.s.hi, a.s.hi), cs = two_prod(a.c.hi, a.s.hi);
    const Wide d = two_sum(cc.hi, -ss.hi);
    const double dl = d.lo + (cc.lo - ss.lo) + 2.0 * (a.c.hi * a.c.lo - a.s.hi * a.s.lo);
    const double sl = cs.lo + a.c.hi * a.s.lo + a.s.hi * a.c.lo;
    return {normal(d.hi, dl), normal(2.0 * cs.hi, 2.0 * sl)};
}
__device__ __forceinline__ cplx rounded(const Turn &a) { return {a.c.hi, a.s.hi}; }

// Kernels of this many chunks or more have Wide angles: orders above 24, at 1
// to 4 % of their time (M2L of order 32, 2,003 items 37.4 -> 37.8 us).  Up to 24
// the errors are those of the kernels before, and short lists would take 8 %
// longer.
inline constexpr int kWide = 4;

// e^{i m theta} for m = 2 (q + 4 j) + e: squares for e^{2i}, e^{4i}, e^{8i},
// then one product per slot.
template <int NJX>
__device__ __forceinline__ void powers(const Turn &t1, int q, double (&c)[2][NJX], double (&s)[2][NJX])
{
    const cplx one = rounded(t1);
    cplx two, four, eight;
    if constexpr (NJX >= kWide) {
        const Turn t2 = square(t1), t4 = square(t2);
        two = rounded(t2);
        four = rounded(t4);
        eight = rounded(square(t4));
    } else {
        two = mul(one, one);
        four = mul(two, two);
        eight = mul(four, four);
    }
    cplx p{1.0, 0.0};
    if (q & 1) p = two;
    if (q & 2) p = (q & 1) ? mul(two, four) : four;
    cplx r = mul(p, one);
    static_for<0, NJX>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        if constexpr (j > 0) {
            p = mul(p, eight);
            r = mul(r, eight);
        }
        c[0][j] = p.c;
        s[0][j] = p.s;
        c[1][j] = r.c;
        s[1][j] = r.s;
    });
}

// b^e for a wave-uniform 0 <= e < 2^BITS, from sq[k] = b^(2^k).
template <int BITS>
__device__ __forceinline__ double ipow(const double (&sq)[BITS], int e)
{
    double v = 1.0;
    static_for<0, BITS>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if (e & (1 << k)) v *= sq[k];
    });
    return v;
}

// The swap operands of one degree.  Held in registers for both swaps of a
// transform where they are few, re-read from the cache otherwise.
template <int NJ>
struct Operands {
    static constexpr int NB = row_blocks(NJ);
    static constexpr bool kPairs = NJ <= kSmall;
    static constexpr int kCount = kPairs ? 4 * NJ * NJ : 4 * NB * NJ;
    static constexpr bool kHeld = NJ <= 2;
    double v[kHeld ? kCount : 1];
    const double *p;
    __device__ __forceinline__ void load(const double *tab, int n, int lane)
    {
        p = tab + base_of(NJ) + (n - 8 * (NJ - 1)) * degree_size(NJ);
        p += kPairs ? 2 * ((lane & 3) + 4 * (lane >> 4)) : lane;
        if constexpr (kHeld)
            static_for<0, kCount / 2>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const double2 w = *reinterpret_cast<const double2 *>(p + 32 * i);
                v[2 * i] = w.x;
                v[2 * i + 1] = w.y;
            });
    }
    // operands [first, first + COUNT) of a block
    template <int FIRST, int COUNT>
    __device__ __forceinline__ void get(double (&a)[COUNT]) const
    {
        static_for<0, COUNT>([&](auto ic) {
            constexpr int i = FIRST + decltype(ic)::value;
            if constexpr (kHeld) a[i - FIRST] = v[i];
            else if constexpr (kPairs) a[i - FIRST] = p[32 * (i / 2) + i % 2];
            else a[i - FIRST] = p[64 * i];
        });
    }
};

// One swap of a degree whose parity is ODD: x[class][slot] in place.
template <int NJ, int ODD>
__device__ __forceinline__ void swap(const Operands<NJ> &A, double (&xr)[2][NJ], double (&xi)[2][NJ])
{
    constexpr int NB = row_blocks(NJ);
    double d[4][NJ];
    if constexpr (NJ <= kSmall) {
        static_for<0, 4>([&](auto kc) {  // independent chains
            constexpr int k = decltype(kc)::value;
            double a[NJ * NJ];
            A.template get<k * NJ * NJ, NJ * NJ>(a);
            static_for<0, NJ>([&](auto oc) { d[k][decltype(oc)::value] = 0.0; });
            static_for<0, NJ>([&](auto cc) {
                constexpr int c = decltype(cc)::value;
                static_for<0, NJ>([&](auto oc) {
                    constexpr int o = decltype(oc)::value;
                    d[k][o] = mfma4(a[o * NJ + c], k < 2 ? xr[k][c] : xi[k - 2][c], d[k][o]);
                });
            });
        });
    } else {
        static_for<0, 4>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            dbl4 f[NB];
            static_for<0, NB>([&](auto bc) {
                constexpr int b = decltype(bc)::value;
                __builtin_amdgcn_sched_barrier(0);  // one row block's operands in flight
                double a[NJ];
                A.template get<(k * NB + b) * NJ, NJ>(a);
                f[b] = dbl4{0.0, 0.0, 0.0, 0.0};
                static_for<0, NJ>([&](auto cc) {
                    constexpr int c = decltype(cc)::value;
                    f[b] = mfma16(a[c], k < 2 ? xr[k][c] : xi[k - 2][c], f[b]);
                });
            });
            static_for<0, NJ>([&](auto jc) { d[k][decltype(jc)::value] = f[decltype(jc)::value / 4][decltype(jc)::value % 4]; });
        });
    }
    static_for<0, NJ>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        static_for<0, 2>([&](auto ec) {
            constexpr int e = decltype(ec)::value;
            xr[(e + ODD) & 1][j] = d[e][j];
            xi[(e + ODD + 1) & 1][j] = d[2 + e][j];
        });
    });
}

// x <- scale e^{+-i m theta} x
template <int NJ, bool FWD, int NJX>
__device__ __forceinline__ void rotate(const double (&c)[2][NJX], const double (&s)[2][NJX], double (&xr)[2][NJ],
                                       double (&xi)[2][NJ])
{
    static_for<0, 2 * NJ>([&](auto ic) {
        constexpr int e = decltype(ic)::value & 1, j = decltype(ic)::value >> 1;
        const double a = xr[e][j], b = xi[e][j];
        if constexpr (FWD) {
            xr[e][j] = c[e][j] * a - s[e][j] * b;
            xi[e][j] = s[e][j] * a + c[e][j] * b;
        } else {
            xr[e][j] = c[e][j] * a + s[e][j] * b;
            xi[e][j] = c[e][j] * b - s[e][j] * a;
        }
    });
}

template <int NJ>
__device__ __forceinline__ void scale_by(double f, double (&xr)[2][NJ], double (&xi)[2][NJ])
{
    static_for<0, 2 * NJ>([&](auto ic) {
        constexpr int e = decltype(ic)::value & 1, j = decltype(ic)::value >> 1;
        xr[e][j] *= f;
        xi[e][j] *= f;
    });
}

// Bands of W items are dealt to the waves in alternating order, so every
// wave gets nearly the same total: position of wave w's k-th item.
__device__ __forceinline__ int dealt(int k, int w, int W) { return k * W + ((k & 1) ? W - 1 - w : w); }

// NJX: largest chunk count (orders up to 8 NJX).  TL: log2 of the
// translations per workgroup (columns t >= 2^TL repeat column t mod 2^TL and
// store nothing), or -1 to take it from `tl`.  mode 1: target += T(source);
// 0: target block = T(source); 2: as 0, with the items of a run (consecutive
// translations of one group of 16 with one block) added across lanes and
// stored by the run's first.
template <int OP, int NJX, int TL, int WAVES, int PER_SIMD>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(PER_SIMD)))
    k_team(const double *__restrict__ src_pool, double *__restrict__ dst_pool, const sfmm_item *__restrict__ items,
           uint32_t n_items, const double *__restrict__ tables, const double *__restrict__ facs, int pc, int tl,
           int mode)
{
    extern __shared__ double sh[];
    constexpr bool kLFwd = OP == SFMM_L2L;  // L-type: transposed blocks
    constexpr bool kLBwd = OP != SFMM_M2M;
    constexpr int kBits = NJX <= 1 ? 4 : NJX <= 3 ? 5 : NJX <= 7 ? 6 : 7;  // 8 NJX < 2^kBits
    const int tlog = TL >= 0 ? TL : tl;
    const int T = 1 << tlog;
    // (re, im) of coefficient c, translation t at tri[c T + t]
    double2 *tri = reinterpret_cast<double2 *>(sh + weight_size(OP, pc));
    // e^{i m alpha} and e^{i m beta} of translation t at rot[2 m T + t] and
    // rot[(2 m + 1) T + t]
    double2 *rot = tri + (pc * (pc + 1) / 2) * T;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const int W = int(blockDim.x >> 6);
    const int q = lane >> 4, t = lane & 15;
    const int tt = TL == 4 ? t : t & (T - 1);

    const uint32_t idx = blockIdx.x * uint32_t(T) + uint32_t(tt);
    const bool valid = idx < n_items;
    const bool writer = valid && (TL == 4 || t < T);
    sfmm_item it{};
    if (valid) it = items[idx];
    double x = it.x, y = it.y, z = it.z;
    bool zero_shift = false;
    if constexpr (OP != SFMM_M2L) zero_shift = valid && (x * x + y * y + z * z == 0.0);
    if constexpr (OP == SFMM_M2M) {  // translations.cpp:331-333
        x = -x;
        y = -y;
        z = -z;
    }
    if (!valid || zero_shift) {  // harmless geometry for idle columns
        x = 0.0;
        y = 0.0;
        z = 1.0;
    }
    const bool active = valid && !zero_shift;
    const double *__restrict__ S = src_pool + it.src;
    double *__restrict__ D = dst_pool + it.dst;
    const int pin = active ? int(it.p_in) : 0;
    const int pend = it.p_in < it.p_out ? int(it.p_in) : int(it.p_out);
    // outputs of L2L stop at min(p_in, p_out) (translations.cpp:412)
    const int pout = !active ? 0 : OP == SFMM_L2L ? pend : int(it.p_out);
    const int pin_w = wave_max7(uint32_t(pin)), pout_w = wave_max7(uint32_t(pout));

    // runs: bit j of `same` says translation t + 2^j is in t's run
    uint32_t same = 0;
    bool head = true;
    if (mode == 2) {
        const uint64_t key = valid ? it.dst : ~uint64_t(lane);
        const uint32_t lo = uint32_t(key), hi = uint32_t(key >> 32);
        static_for<0, 4>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const uint32_t olo = __shfl_down(lo, 1u << j, 64), ohi = __shfl_down(hi, 1u << j, 64);
            if (t + (1 << j) < T && olo == lo && ohi == hi) same |= 1u << j;
        });
        const uint32_t plo = __shfl_up(lo, 1u, 64), phi = __shfl_up(hi, 1u, 64);
        head = t == 0 || plo != lo || phi != hi;
    }

    // A degree's coefficients as pairs of orders (2i, 2i + 1), i = q + 4 j;
    // lanes past the degree repeat its last pair, which the swap's zero
    // entries drop.  Where the last order is even, the lanes that hold it read
    // the imaginary pair one double lower, inside the block, and take its
    // upper half; their second order is dropped too.
    auto load_degree = [&](const double *blk, int n, dbl2(&re)[NJX], dbl2(&im)[NJX]) {
        const double *row = blk + n * (n + 1);
        static_for<0, NJX>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            re[j] = dbl2{0.0, 0.0};
            im[j] = dbl2{0.0, 0.0};
            if (8 * j <= n) {
                const int m = min(2 * (q + 4 * j), n & ~1);
                re[j] = *reinterpret_cast<const dbl2 *>(row + m);
                im[j] = *reinterpret_cast<const dbl2 *>(row + (m + n + (m == n ? 0 : 1)));
            }
        });
    };

    // One degree of sources, later of targets, is on its way while the one
    // before is worked on, where the registers allow it.
    constexpr bool kAhead = NJX <= 4;
    dbl2 pr[NJX], pi[NJX];
    auto load_source = [&](int n) {
        if (n >= 0) load_degree(n < pin ? S : kZeroBlock, n, pr, pi);
    };
    auto load_target = [&](int N) {
        if (N >= 0 && mode == 1) load_degree(writer && N < pout ? D : kZeroBlock, N, pr, pi);
    };
    auto take = [&](dbl2(&cr)[NJX], dbl2(&ci)[NJX]) {
        static_for<0, NJX>([&](auto jc) {
            cr[decltype(jc)::value] = pr[decltype(jc)::value];
            ci[decltype(jc)::value] = pi[decltype(jc)::value];
        });
    };
    int n = pin_w - 1 - dealt(0, wave, W);
    if constexpr (kAhead) load_source(n);

    // weights of the z-translation
    for (int i = threadIdx.x; i < weight_size(OP, pc); i += blockDim.x) {
        const int d = i - weight_pad(OP);
        double w = 0.0;
        if (d >= 0 && d <= (OP == SFMM_M2L ? 2 * pc - 2 : pc - 1))
            w = facs[(OP == SFMM_M2L ? 0 : 2 * mfma::kMaxOrder) + d];
        sh[i] = w;
    }

    // Euler data (microkernel_generic.cpp:61-74).
    const double rho2 = x * x + y * y;
    const double rho = sqrt(rho2);
    const double r = sqrt(rho2 + z * z);
    const double rinv = 1.0 / r;  // of the rounded r: M2M and L2L multiply by powers of both
    Turn ea{{1.0, 0.0}, {0.0, 0.0}}, eb{{z * rinv, 0.0}, {-rho * rinv, 0.0}};
    if constexpr (NJX >= kWide) {
        const Distance xyz = distance(x, y, z), xy = distance(x, y, 0.0);
        eb.c = mul({z, 0.0}, xyz.inv);
        if (rho != 0.0) {
            ea = {mul({y, 0.0}, xy.inv), mul({x, 0.0}, xy.inv)};
            eb.s = mul({-xy.r.hi, -xy.r.lo}, xyz.inv);
        }
    } else if (rho != 0.0) {
        const double qq = 1.0 / rho;
        ea = {{y * qq, 0.0}, {x * qq, 0.0}};
    }
    constexpr bool kInLds = NJX >= kRotLds;
    double ca[2][NJX], sa[2][NJX], cb[2][NJX], sb[2][NJX];
    if constexpr (kInLds) {
        if (wave < 2) {
            powers<NJX>(wave ? eb : ea, q, ca, sa);
            static_for<0, 2 * NJX>([&](auto ic) {
                constexpr int e = decltype(ic)::value & 1, j = decltype(ic)::value >> 1;
                const int m = 2 * (q + 4 * j) + e;
                if (m < pc) rot[(2 * m + wave) * T + tt] = double2{ca[e][j], sa[e][j]};
            });
        }
        __syncthreads();
    } else {
        powers<NJX>(ea, q, ca, sa);
        powers<NJX>(eb, q, cb, sb);
    }
    // x <- e^{+-i m theta} x; angle 0 alpha, 1 beta
    auto turn = [&](auto fwdc, auto anglec, auto &xr, auto &xi) {
        constexpr bool FWD = decltype(fwdc)::value != 0;
        constexpr int angle = decltype(anglec)::value, NJ = int(sizeof(xr[0]) / sizeof(double));
        if constexpr (kInLds) {
            double c[2][NJ], s[2][NJ];
            static_for<0, 2 * NJ>([&](auto ic) {
                constexpr int e = decltype(ic)::value & 1, j = decltype(ic)::value >> 1;
                const double2 v = rot[(2 * min(2 * (q + 4 * j) + e, pc - 1) + angle) * T + tt];
                c[e][j] = v.x;
                s[e][j] = v.y;
            });
            rotate<NJ, FWD, NJ>(c, s, xr, xi);
        } else if constexpr (angle == 0) {
            rotate<NJ, FWD, NJX>(ca, sa, xr, xi);
        } else {
            rotate<NJ, FWD, NJX>(cb, sb, xr, xi);
        }
    };
    int col[2][NJX];  // triangle columns of the lane's orders
    static_for<0, 2 * NJX>([&](auto ic) {
        constexpr int e = decltype(ic)::value & 1, j = decltype(ic)::value >> 1;
        col[e][j] = column(pc, 2 * (q + 4 * j) + e);
    });
    double sq[kBits];
    auto squares = [&](double b) {
        sq[0] = b;
        static_for<1, kBits>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            sq[k] = sq[k - 1] * sq[k - 1];
        });
    };
    squares(kLFwd ? r : rinv);

    // ---- forward: scale r^-(n+1) (translations.cpp:45), L2L r^n (:198)
    // Loads return in order.  Where the operands are held in registers they
    // are requested before the next degree, so that no swap waits for it;
    // where they are read again and again it comes first and has the longest
    // way (order 20 measured 5-8 % slower the other way round).
    constexpr bool kHeldAll = NJX <= 2;
    auto forward = [&](auto njc, auto oddc, int n, double f, const dbl2(&cr)[NJX], const dbl2(&ci)[NJX], int next) {
        constexpr int NJ = decltype(njc)::value, ODD = decltype(oddc)::value;
        Operands<NJ> A;
        A.load(tables + (kLFwd ? table_size() : 0), n, lane);
        if constexpr (kAhead && kHeldAll) load_source(next);
        double xr[2][NJ], xi[2][NJ];
        static_for<0, NJ>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            xr[0][j] = cr[j].x;
            xr[1][j] = cr[j].y;
            xi[0][j] = ODD || 2 * (q + 4 * j) < n ? ci[j].x : ci[j].y;
            xi[1][j] = ci[j].y;
        });
        scale_by<NJ>(f, xr, xi);
        turn(ic<1>{}, ic<0>{}, xr, xi);
        swap<NJ, ODD>(A, xr, xi);
        turn(ic<1>{}, ic<1>{}, xr, xi);
        swap<NJ, ODD>(A, xr, xi);
        static_for<0, 2 * NJ>([&](auto ic) {
            constexpr int e = decltype(ic)::value & 1, j = decltype(ic)::value >> 1;
            const int m = 2 * (q + 4 * j) + e;
            if (m <= n) tri[(col[e][j] + n) * T + tt] = double2{xr[e][j], xi[e][j]};
        });
    };
    // run body(ic<NJ>, ic<parity>) for degree n
    auto by_degree = [&](int n, auto &&body) {
        static_for<1, NJX + 1>([&](auto njc) {
            if ((n >> 3) + 1 == decltype(njc)::value) {
                if (n & 1) body(njc, ic<1>{});
                else body(njc, ic<0>{});
            }
        });
    };
    for (int k = 0; n >= 0; ++k) {
        const int next = pin_w - 1 - dealt(k + 1, wave, W);
        dbl2 cr[NJX], ci[NJX];
        if constexpr (!kAhead) load_source(n);
        take(cr, ci);
        if constexpr (kAhead && !kHeldAll) load_source(next);
        // a degree that a translation does not have is zero, whatever the
        // power of r that only longer translations of the group reach
        const double f = n < pin ? ipow<kBits>(sq, kLFwd ? n : n + 1) : 0.0;
        by_degree(n, [&](auto njc, auto oddc) { forward(njc, oddc, n, f, cr, ci, next); });
        n = next;
    }
    // the first target degree is on its way during the z-translation
    int N = pout_w - 1 - dealt(0, wave, W);
    static_for<0, NJX>([&](auto jc) { pr[decltype(jc)::value] = pi[decltype(jc)::value] = dbl2{0.0, 0.0}; });
    if constexpr (kAhead) load_target(N);
    __syncthreads();

    // ---- z-translation, column by column in place:
    // L_N^m = (-1)^(N+m) sum_K (N+K)! T_K^m (translations.cpp:283-296),
    // M_N^m = sum_{K<=N} T_K^m / (N-K)! (:363-377),
    // L_N^m = sum_{K>=N} T_K^m / (K-N)! (:440-451)
    for (int k = 0;; ++k) {
        const int m = dealt(k, wave, W);
        if (k * W >= pout_w) break;
        if (m >= pout_w) continue;
        const int nk = pin_w - m, nn = pout_w - m;  // input and output degrees
        double2 *top = tri + (column(pc, m) + m) * T + tt;  // degree m
        const bool flip = OP == SFMM_M2L && (q & 1);  // (-1)^(N+m) of the lane's rows
        auto put = [&](int row, double re, double im) {
            if (row < nn) top[row * T] = double2{flip ? -re : re, flip ? -im : im};
        };
        // M2M and L2L couple a degree with the degrees on one side of it.
        // The matrix product has zero weights for the others, which an
        // infinity or a NaN would turn into NaN: such columns are summed
        // degree by degree.  Looking for them costs 0.5 us of the 8 to 14 of
        // a short launch (FMM of 100,000 points 872 -> 880 us).
        auto one_sided = [&] {
            for (int k4 = 0; 4 * k4 < nn; ++k4) {
                const int N0 = OP == SFMM_M2M ? 4 * ((nn - 1) / 4 - k4) : 4 * k4;  // read before it is replaced
                const int N = N0 + q, end = OP == SFMM_M2M ? min(nk, N0 + 4) : nk;
                double re = 0.0, im = 0.0;
                for (int K = OP == SFMM_M2M ? 0 : N0; K < end; ++K) {
                    const double2 v = top[K * T];
                    const double w = sh[weight_pad(OP) + (OP == SFMM_M2M ? N - K : K - N)];
                    const bool on = OP == SFMM_M2M ? K <= N : K >= N;
                    re = on ? __builtin_fma(w, v.x, re) : re;
                    im = on ? __builtin_fma(w, v.y, im) : im;
                }
                __builtin_amdgcn_wave_barrier();
                put(N, re, im);
            }
        };
        // true where any value of the column is infinite or NaN; integer
        // instructions between the products, which have the FP64 pipe
        auto unbounded = [&](const auto &re, const auto &im) {
            uint32_t top_bits = 0;
            static_for<0, int(sizeof(re) / sizeof(double))>([&](auto cc) {
                const double v[2] = {re[decltype(cc)::value], im[decltype(cc)::value]};
                for (int i = 0; i < 2; ++i)
                    top_bits = max(top_bits, uint32_t(__builtin_bit_cast(uint64_t, v[i]) >> 32) & 0x7fffffffu);
            });
            return OP != SFMM_M2L && __ballot(top_bits >= 0x7ff00000u) != 0;
        };
        if constexpr (NJX <= kSmall) {
            const int chunks = (max(nk, nn) + 3) / 4;
            bool slow = false;
            static_for<1, 2 * NJX + 1>([&](auto ncc) {
                constexpr int NC = decltype(ncc)::value;
                if (chunks == NC) {
                    double br[NC], bi[NC], dr[NC], di[NC], w[2 * NC];
                    static_for<0, NC>([&](auto cc) {
                        constexpr int c = decltype(cc)::value;
                        const bool ok = 4 * c + q < nk;
                        const double2 v = top[(ok ? 4 * c + q : 0) * T];
                        br[c] = ok ? v.x : 0.0;
                        bi[c] = ok ? v.y : 0.0;
                    });
                    const int i = t & 3;
                    const double *wt =
                        sh + weight_pad(OP) + (OP == SFMM_M2L ? 2 * m + (i + q) : OP == SFMM_M2M ? i - q : q - i);
                    static_for<0, OP == SFMM_M2L ? 2 * NC - 1 : NC>(
                        [&](auto uc) { w[decltype(uc)::value] = wt[4 * decltype(uc)::value]; });
                    static_for<0, NC>([&](auto cc) {  // 2 NC independent chains
                        constexpr int c = decltype(cc)::value;
                        static_for<0, NC>([&](auto oc) {
                            constexpr int o = decltype(oc)::value;
                            constexpr int u = OP == SFMM_M2L ? o + c : OP == SFMM_M2M ? o - c : c - o;
                            if constexpr (u >= 0) {
                                constexpr bool fresh = OP == SFMM_L2L ? c == o : c == 0;
                                dr[o] = mfma4(w[u], br[c], fresh ? 0.0 : dr[o]);
                                di[o] = mfma4(w[u], bi[c], fresh ? 0.0 : di[o]);
                            }
                        });
                    });
                    if constexpr (OP != SFMM_M2L) slow = unbounded(br, bi);
                    if (!slow)
                        static_for<0, NC>([&](auto oc) { put(4 * decltype(oc)::value + q, dr[decltype(oc)::value], di[decltype(oc)::value]); });
                }
            });
            if constexpr (OP != SFMM_M2L) {
                if (slow) one_sided();
            }
        } else {
            double br[2 * NJX], bi[2 * NJX];
            static_for<0, 2 * NJX>([&](auto cc) {
                constexpr int c = decltype(cc)::value;
                br[c] = 0.0;
                bi[c] = 0.0;
                if (4 * c < nk) {
                    const bool ok = 4 * c + q < nk;
                    const double2 v = top[(ok ? 4 * c + q : 0) * T];
                    br[c] = ok ? v.x : 0.0;
                    bi[c] = ok ? v.y : 0.0;
                }
            });
            if (unbounded(br, bi)) {
                one_sided();
                continue;
            }
            const double *wt = sh + weight_pad(OP) + (OP == SFMM_M2L ? 2 * m + (t + q) : OP == SFMM_M2M ? t - q : q - t);
            static_for<0, (NJX + 1) / 2>([&](auto bc) {
                constexpr int b = decltype(bc)::value;
                if (16 * b < nn) {
                    dbl4 dr{0.0, 0.0, 0.0, 0.0}, di{0.0, 0.0, 0.0, 0.0};
                    static_for<0, 2 * NJX>([&](auto cc) {
                        constexpr int c = decltype(cc)::value;
                        constexpr bool none = (OP == SFMM_M2M && 4 * c > 16 * b + 15) ||
                                              (OP == SFMM_L2L && 4 * c + 3 < 16 * b);
                        if constexpr (!none) {
                            if (4 * c < nk) {
                                const double w = wt[OP == SFMM_M2L   ? 16 * b + 4 * c
                                                    : OP == SFMM_M2M ? 16 * b - 4 * c
                                                                     : 4 * c - 16 * b];
                                dr = mfma16(w, br[c], dr);
                                di = mfma16(w, bi[c], di);
                            }
                        }
                    });
                    static_for<0, 4>([&](auto ec) {
                        constexpr int e = decltype(ec)::value;
                        put(16 * b + 4 * e + q, dr[e], di[e]);
                    });
                }
            });
        }
    }
    __syncthreads();

    // ---- backward: scale r^-N (translations.cpp:180), M2M r^(N+1) (:129)
    squares(OP == SFMM_M2M ? r : rinv);
    auto backward = [&](auto njc, auto oddc, int N, double f, const dbl2(&cr)[NJX], const dbl2(&ci)[NJX], int next) {
        constexpr int NJ = decltype(njc)::value, ODD = decltype(oddc)::value;
        Operands<NJ> A;
        A.load(tables + (kLBwd ? table_size() : 0), N, lane);
        if constexpr (kAhead && kHeldAll) load_target(next);
        double xr[2][NJ], xi[2][NJ];
        static_for<0, 2 * NJ>([&](auto ic) {
            constexpr int e = decltype(ic)::value & 1, j = decltype(ic)::value >> 1;
            const int m = 2 * (q + 4 * j) + e;
            const bool ok = m <= N;
            const double2 v = tri[(ok ? col[e][j] + N : 0) * T + tt];
            xr[e][j] = ok ? v.x : 0.0;
            xi[e][j] = ok ? v.y : 0.0;
        });
        swap<NJ, ODD>(A, xr, xi);
        turn(ic<0>{}, ic<1>{}, xr, xi);
        swap<NJ, ODD>(A, xr, xi);
        turn(ic<0>{}, ic<0>{}, xr, xi);
        scale_by<NJ>(f, xr, xi);
        bool on = writer && N < pout;
        if (mode == 2) {  // fixed tree over the run's translations
            static_for<0, 4>([&](auto jc) {
                constexpr int b = decltype(jc)::value;
                const bool take = (same >> b) & 1u;
                static_for<0, 2 * NJ>([&](auto ic) {
                    constexpr int e = decltype(ic)::value & 1, j = decltype(ic)::value >> 1;
                    const double u = __shfl_down(xr[e][j], 1u << b, 64), v = __shfl_down(xi[e][j], 1u << b, 64);
                    xr[e][j] += take ? u : 0.0;
                    xi[e][j] += take ? v : 0.0;
                });
            });
            on = on && head;
        }
        static_for<0, NJ>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const int m = 2 * (q + 4 * j);
            const double r0 = cr[j].x + xr[0][j], r1 = cr[j].y + xr[1][j];
            const double i0 = (ODD || m < N ? ci[j].x : ci[j].y) + xi[0][j], i1 = ci[j].y + xi[1][j];
            double *pr = D + N * (N + 1) + m, *pi = pr + N + 1;
            if (on && m < N) {
                *reinterpret_cast<dbl2 *>(pr) = dbl2{r0, r1};
                *reinterpret_cast<dbl2 *>(pi) = dbl2{i0, i1};
            }
            if constexpr (!ODD) {
                if (on && m == N) {
                    *pr = r0;
                    *pi = i0;
                }
            }
        });
    };
    for (int k = 0; N >= 0; ++k) {
        const int next = pout_w - 1 - dealt(k + 1, wave, W);
        dbl2 cr[NJX], ci[NJX];
        if constexpr (!kAhead) load_target(N);
        take(cr, ci);
        if constexpr (kAhead && !kHeldAll) load_target(next);
        const double f = ipow<kBits>(sq, OP == SFMM_M2M ? N + 1 : N);
        by_degree(N, [&](auto njc, auto oddc) { backward(njc, oddc, N, f, cr, ci, next); });
        N = next;
    }

    if (zero_shift && writer) {
        // M2M / L2L with zero shift: target += source over the common
        // degrees (translations.cpp:539-547, 596-604)
        for (int i = wave * 4 + q; i < pend * (pend + 1); i += 4 * W) D[i] = (mode == 1 ? D[i] : 0.0) + S[i];
    }
}

using fn_t = void (*)(const double *, double *, const sfmm_item *, uint32_t, const double *, const double *, int, int,
                      int);

// Kernels of one operator, by largest chunk count (team_{m2m,m2l,l2l}.hip).
struct Kernels {
    fn_t upto16, upto24;    // four waves
    fn_t upto16w, upto24w;  // eight waves
    fn_t upto32, upto48;
};
template <int OP>
const Kernels &kernels();

}  // namespace team
}  // namespace sfmm
