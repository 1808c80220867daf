// FP64 translation kernel of one wave per eight translations of any orders
// up to a bound, for long lists of orders 8 to 24 (M2L to 22).
//
//   forward, per input degree n:   scale, rotate by alpha, swap, rotate by
//                                  beta, swap; the degree stays in registers
//   z-translation, per order m:    sums over the registers of a lane
//   backward, per output degree N: swap, rotate, swap, rotate, scale, add
//
// Algorithm: Dehnen's rotation scheme as in translations.cpp:36-471.  Lane
// (q, part, t) = t + 8 part + 16 q holds the real (part 0) or imaginary part
// of the orders m = 2 (q + 4 j) + e of translation t, e the parity class.
// Half the wave for each part halves a translation's registers per lane: the
// rotated triangle of order 16 takes 92, where a wave of 16 translations
// with both parts in a lane needs 184 and its SIMD has no room for a second
// wave.  One v_mfma_f64_4x4x4_4b_f64 does a block of four orders by four of
// both parts, each with its own operand (octet_tables.hpp).  The class of an
// output order differs between the parts, so after one swap register e holds
// class e in the lanes of one part and 1 - e in the other's ("crossed"), and
// after two it does not: the rotation in between has its factors stored
// crossed and takes a coefficient's other part from the other register of
// lane u ^ 8.
//
// Memory moves in 16-byte pieces, eight lanes for 128 consecutive bytes of a
// translation, and changes lanes through a staging buffer in LDS.  Read in
// the layout of the computation, every 8-byte piece was an access of its
// own, 13,500 for 16 translations of order 16; now it is 3,300.
//
// What bounds it: order 8 the memory (M2L of 200,000 translations in 72 us,
// 4.8 of the 5.2 TB/s that a large copy reaches; lane kernel 137, a wave of
// 16 translations 94); from order 9 latency, with 8 waves a CU and then 4
// (210,000 VALU and 100,000 LDS cycles of 740,000 at order 16): order 10 130
// us (156, 181), 12 180 (333, 250), 16 330 (16 translations: 457), 20 580
// (752).
//
// Orders 9 to 14 and from 17 up run two degrees side by side, as far as the
// registers reach (order 10: 146 -> 130 us, 12: 194 -> 180); from 17 on with
// one wave per SIMD (order 20 at two: 1,008 us from spills, at one 580; three
// degrees side by side 606).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

#include "../../include/solidfmm_gpu.h"
#include "octet_tables.hpp"
#include "tables.hpp"
#include "translate.hpp"

namespace sfmm {
namespace octet {

// 16 bytes at 8-byte alignment: a piece may start at any coefficient of its
// block
typedef double dbl2 __attribute__((ext_vector_type(2), aligned(8)));

inline constexpr int kItems = 8;  // translations per wave

// Read in place of a block that a lane does not load.
inline __device__ double kZeroBlock[kMaxOrder * (kMaxOrder + 1)];

__device__ __forceinline__ void sched_fence() { __builtin_amdgcn_sched_barrier(0); }
// Lanes of the wave see each other's LDS writes: the hardware keeps a wave's
// LDS accesses in order, the fence keeps the compiler's.
__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Operand lane l holds output l % 4 of input l / 16 for block (l / 4) % 4,
// i.e. for translations 4 (l / 4 % 4) ... of the 16 columns; result lane
// (q, u) is output q of column u.
__device__ __forceinline__ double mfma4(double a, double b, double c)
{
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// Value of the lane that `CTRL` names within the row of 16.
template <int CTRL>
__device__ __forceinline__ double dpp(double v)
{
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_mov_dpp(int(uint32_t(b)), CTRL, 0xf, 0xf, true);
    const uint32_t hi = __builtin_amdgcn_mov_dpp(int(uint32_t(b >> 32)), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, uint64_t(hi) << 32 | lo);
}
// The other part of the same coefficient: lane u ^ 8 (row_ror:8).
__device__ __forceinline__ double other_part(double v) { return dpp<0x128>(v); }

// Largest value of v over the wave (0 <= v < 32), wave-uniform.
__device__ __forceinline__ int wave_max5(uint32_t v)
{
    uint32_t m = 0;
    for (int b = 4; b >= 0; --b) {
        const uint32_t cand = m | (1u << b);
        if (__ballot(v >= cand)) m = cand;
    }
    return int(m);
}

struct cplx {
    double c, s;
};
__device__ __forceinline__ cplx mul(cplx a, cplx b) { return {a.c * b.c - a.s * b.s, a.s * b.c + a.c * b.s}; }

// e^{i m theta}, register e of chunk j for m = 2 (q + 4 j) + e, or for the
// other class where `cross` is set.
template <int NJX>
__device__ __forceinline__ void powers(cplx one, int q, bool cross, double (&c)[2][NJX], double (&s)[2][NJX])
{
    const cplx two = mul(one, one), four = mul(two, two), eight = mul(four, four);
    cplx p{1.0, 0.0};
    if (q & 1) p = two;
    if (q & 2) p = (q & 1) ? mul(two, four) : four;
    const cplx o = mul(p, one);
    cplx r{cross ? p.c : o.c, cross ? p.s : o.s};
    p = {cross ? o.c : p.c, cross ? o.s : p.s};
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

// One swap of degree N.  CROSS: on entry register i holds class i in the
// lanes of the real part and 1 - i in those of the imaginary part, and class
// i in all lanes on return; otherwise the other way round.
template <int N, bool CROSS, int NJX>
__device__ __forceinline__ void swap(const double *tab, int lo, int part, double (&x)[2][NJX])
{
    constexpr int NJ = chunks(N);
    constexpr int CS = class_size(NJ);
    const double *lane_tab = tab + (NJ == 1 ? lo : 2 * lo);
    const double *a[2] = {lane_tab + (CROSS ? part * CS : 0) + degree_base(N),
                          lane_tab - (CROSS ? part * CS : 0) + (degree_base(N) + CS)};
    double d[2][NJ];
    static_for<0, NJ>([&](auto oc) {
        constexpr int o = decltype(oc)::value;
        d[0][o] = 0.0;
        d[1][o] = 0.0;
    });
    double op[2][NJ * NJ + (NJ > 1 ? NJ * NJ % 2 : 0)];
    static_for<0, 2>([&](auto ic_) {
        constexpr int i = decltype(ic_)::value;
        if constexpr (NJ == 1) {
            op[i][0] = a[i][0];
        } else {
            static_for<0, (NJ * NJ + 1) / 2>([&](auto pc) {
                constexpr int p = decltype(pc)::value;
                const double2 w = *reinterpret_cast<const double2 *>(a[i] + 64 * p);
                op[i][2 * p] = w.x;
                op[i][2 * p + 1] = w.y;
            });
        }
    });
    static_for<0, NJ>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        static_for<0, NJ>([&](auto oc) {
            constexpr int o = decltype(oc)::value;
            d[0][o] = mfma4(op[0][o * NJ + c], x[0][c], d[0][o]);
            d[1][o] = mfma4(op[1][o * NJ + c], x[1][c], d[1][o]);
        });
    });
    static_for<0, NJ>([&](auto oc) {
        constexpr int o = decltype(oc)::value;
        x[N & 1][o] = d[0][o];
        x[(N + 1) & 1][o] = d[1][o];
    });
}

// Rotation factors: the sines carry the sign of the part (minus for real).
// Those of beta are stored as the swap in between leaves the registers.
template <int NJX>
struct Rot {
    double ca[2][NJX], sa[2][NJX], cb[2][NJX], sb[2][NJX];
};

template <int N, bool FWD, int NJX>
__device__ __forceinline__ void rotate_alpha(const Rot<NJX> &R, double (&x)[2][NJX])
{
    static_for<0, 2 * chunks(N)>([&](auto ic_) {
        constexpr int e = decltype(ic_)::value & 1, j = decltype(ic_)::value >> 1;
        const double p = other_part(x[e][j]) * R.sa[e][j];
        x[e][j] = FWD ? __builtin_fma(R.ca[e][j], x[e][j], p) : __builtin_fma(R.ca[e][j], x[e][j], -p);
    });
}
template <int N, bool FWD, int NJX>
__device__ __forceinline__ void rotate_beta(const Rot<NJX> &R, double (&x)[2][NJX])
{
    static_for<0, chunks(N)>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const double p0 = other_part(x[1][j]) * R.sb[0][j], p1 = other_part(x[0][j]) * R.sb[1][j];
        x[0][j] = FWD ? __builtin_fma(R.cb[0][j], x[0][j], p0) : __builtin_fma(R.cb[0][j], x[0][j], -p0);
        x[1][j] = FWD ? __builtin_fma(R.cb[1][j], x[1][j], p1) : __builtin_fma(R.cb[1][j], x[1][j], -p1);
    });
}

template <int N, int NJX>
__device__ __forceinline__ void scale_by(double f, double (&x)[2][NJX])
{
    static_for<0, 2 * chunks(N)>([&](auto ic_) { x[decltype(ic_)::value & 1][decltype(ic_)::value >> 1] *= f; });
}

// Degrees N0 .. N0 + U - 1 side by side.
template <int N0, int U, int NJX>
__device__ __forceinline__ void forward(const double *tab, int lo, int part, const Rot<NJX> &R,
                                        const double (&scale)[U], double (&x)[U][2][NJX])
{
    static_for<0, U>([&](auto uc) { scale_by<N0 + decltype(uc)::value>(scale[decltype(uc)::value], x[decltype(uc)::value]); });
    static_for<0, U>([&](auto uc) { rotate_alpha<N0 + decltype(uc)::value, true>(R, x[decltype(uc)::value]); });
    static_for<0, U>([&](auto uc) { swap<N0 + decltype(uc)::value, false>(tab, lo, part, x[decltype(uc)::value]); });
    static_for<0, U>([&](auto uc) { rotate_beta<N0 + decltype(uc)::value, true>(R, x[decltype(uc)::value]); });
    static_for<0, U>([&](auto uc) { swap<N0 + decltype(uc)::value, true>(tab, lo, part, x[decltype(uc)::value]); });
}
template <int N0, int U, int NJX>
__device__ __forceinline__ void backward(const double *tab, int lo, int part, const Rot<NJX> &R,
                                         const double (&scale)[U], double (&x)[U][2][NJX])
{
    static_for<0, U>([&](auto uc) { swap<N0 + decltype(uc)::value, false>(tab, lo, part, x[decltype(uc)::value]); });
    static_for<0, U>([&](auto uc) { rotate_beta<N0 + decltype(uc)::value, false>(R, x[decltype(uc)::value]); });
    static_for<0, U>([&](auto uc) { swap<N0 + decltype(uc)::value, true>(tab, lo, part, x[decltype(uc)::value]); });
    static_for<0, U>([&](auto uc) { rotate_alpha<N0 + decltype(uc)::value, false>(R, x[decltype(uc)::value]); });
    static_for<0, U>([&](auto uc) { scale_by<N0 + decltype(uc)::value>(scale[decltype(uc)::value], x[decltype(uc)::value]); });
}

// What a lane knows of a group's items: the block offsets and orders of the
// translation whose coefficients it moves (lane / 8), the shift of the one
// it computes on (lane % 8).
struct Group {
    uint64_t src, dst;
    uint32_t p_in, p_out;
    double x, y, z;
    __device__ __forceinline__ void load(const sfmm_item *__restrict__ items, uint32_t n_items, uint32_t g, int lane)
    {
        const uint32_t last = n_items - 1;
        const uint32_t i = kItems * g + uint32_t(lane >> 3), k = kItems * g + uint32_t(lane & 7);
        const sfmm_item &a = items[i < last ? i : last];
        const sfmm_item &b = items[k < last ? k : last];
        src = a.src;
        dst = a.dst;
        p_in = a.p_in;
        p_out = a.p_out;
        x = b.x;
        y = b.y;
        z = b.z;
    }
};

// doubles of a translation in a wave's staging buffer: a degree of up to
// 8 NJX pieces and 8 for values that are not kept, at a stride that spreads
// the lanes' reads over the banks (12 modulo 16)
constexpr int stage_stride(int njx) { return 16 * njx + 12; }

// degrees of a step
constexpr int side_by_side(int pb) { return pb <= 8 || pb == 15 || pb == 16 ? 1 : 2; }

// The eight translations of group g.  Degrees above the group's largest
// orders are skipped, a missing source degree is a zero, and output degrees
// >= p_out (L2L: >= min(p_in, p_out), translations.cpp:412) are not stored.
// mode 1: target += T(source); 0: target block = T(source); 2: as 0, with
// the items of a run (consecutive translations of the group with one block)
// added across lanes and stored by the run's first.  PAIRS: mode 2 with runs
// that may go on from an even group into the odd one after it; bit 0 of such a
// group's first block offset says that the block has the run's beginning
// already.  `late` is called once the registers of the triangle are free.
template <int OP, int PB, bool PAIRS, class F>
__device__ __forceinline__ void translate_group(const double *__restrict__ src_pool, double *__restrict__ dst_pool,
                                                const Group &G, uint32_t n_items, uint32_t g, const double *tab,
                                                double *buf, int lane, int mode, F &&late)
{
    constexpr int NJX = chunks(PB - 1);
    constexpr int ST = stage_stride(NJX);
    const bool acc = mode == 1;
    const int q = lane >> 4, part = (lane >> 3) & 1, t = lane & 7;  // computing
    const int tp = lane >> 3, c = lane & 7;                         // moving coefficients
    const int lo = (lane & 3) + 4 * part + 8 * q;
    // the L-type table follows where both are used
    const double *tab_f = tab, *tab_b = tab + (OP == SFMM_M2L ? table_size(PB) : 0);

    double x = G.x, y = G.y, z = G.z;
    const bool is_zero = OP != SFMM_M2L && x * x + y * y + z * z == 0.0;
    const bool zero_shift =
        OP != SFMM_M2L && ((__ballot(is_zero) >> tp) & 1u) && uint32_t(kItems) * g + uint32_t(tp) < n_items;
    const bool active = uint32_t(kItems) * g + uint32_t(tp) < n_items && !zero_shift;
    const uint32_t p_end = G.p_in < G.p_out ? G.p_in : G.p_out;
    const uint32_t p_src = G.p_in, p_dst = OP == SFMM_L2L ? p_end : G.p_out;
    const int pin_w = wave_max5(active ? p_src : 0u);
    const int pout_w = wave_max5(active ? p_dst : 0u);

    const double *__restrict__ S = active ? src_pool + G.src + 2 * c : kZeroBlock;
    const uint64_t block = PAIRS ? G.dst & ~uint64_t(1) : G.dst;
    const bool joins = PAIRS && (G.dst & 1);
    // the group before has stored to the CU's cache before this one loads
    if (__ballot(joins)) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    double *__restrict__ D = dst_pool + block + 2 * c;
    const double *__restrict__ O = active && (acc || joins) ? D : kZeroBlock;

    // pieces c + 8 i of degree n, zeros beyond the degree or the order
    auto fetch = [&](auto nc, const double *p, uint32_t order, auto &v) {
        constexpr int n = decltype(nc)::value;
        static_for<0, chunks(n)>([&](auto ic_) {
            constexpr int i = decltype(ic_)::value;
            bool on = uint32_t(n) < order;
            if constexpr (8 * i + 7 > n) on = on && c <= n - 8 * i;
            const double *a = on ? p : kZeroBlock;  // of the same extent
            v[i] = *reinterpret_cast<const dbl2 *>(a + n * (n + 1) + 16 * i);
        });
    };
    // Steps of U degrees; sources are requested two degrees ahead.
    constexpr int U = side_by_side(PB);
    constexpr int kIn = U + 2, kOld = OP == SFMM_M2L ? 2 * U : U;
    dbl2 in[kIn][NJX], old[kOld][NJX];
    auto fetch_src = [&](auto nc) {
        if constexpr (decltype(nc)::value >= 0 && decltype(nc)::value < PB)
            fetch(nc, S, p_src, in[decltype(nc)::value % kIn]);
    };
    auto fetch_old = [&](auto Nc) {
        if constexpr (decltype(Nc)::value >= 0 && decltype(Nc)::value < PB)
            fetch(Nc, O, p_dst, old[decltype(Nc)::value % kOld]);
    };
    static_for<0, 2>([&](auto ic_) {
        if constexpr (OP == SFMM_L2L) fetch_src(ic<PB - 1 - decltype(ic_)::value>{});
        else fetch_src(ic_);
    });

    // runs: bit j of `same` says translation t + 2^j shares t's block
    uint32_t same = 0;
    bool store = active;
    if (mode == 2) {
        const uint64_t key = active ? block : ~uint64_t(tp);
        const uint32_t lo32 = uint32_t(key), hi32 = uint32_t(key >> 32);
        static_for<0, 3>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const uint32_t ol = __shfl_down(lo32, 8u << j, 64), oh = __shfl_down(hi32, 8u << j, 64);
            const uint64_t m = __ballot(tp + (1 << j) < kItems && ol == lo32 && oh == hi32);
            same |= uint32_t((m >> (8 * t)) & 1u) << j;
        });
        const uint32_t pl = __shfl_up(lo32, 8u, 64), ph = __shfl_up(hi32, 8u, 64);
        store = active && (tp == 0 || pl != lo32 || ph != hi32);
    }

    if constexpr (OP == SFMM_M2M) {  // translations.cpp:331-333
        x = -x;
        y = -y;
        z = -z;
    }
    if (is_zero) z = 1.0;  // harmless geometry

    // Euler data (microkernel_generic.cpp:61-74)
    const double rho2 = x * x + y * y;
    const double rho = sqrt(rho2);
    const double r = sqrt(rho2 + z * z);
    const double rinv = 1.0 / r;
    Rot<NJX> R;
    {
        const double qq = 1.0 / rho;
        const bool up = rho == 0.0;
        const double ca = up ? 1.0 : y * qq, sa = up ? 0.0 : x * qq;
        const double cb = z * rinv, sb = -rho * rinv;
        powers<NJX>({ca, part ? sa : -sa}, q, false, R.ca, R.sa);
        powers<NJX>({cb, part ? sb : -sb}, q, part != 0, R.cb, R.sb);
    }

    double *put = buf + tp * ST + 2 * c;
    double *get = buf + t * ST + 2 * q;
    const int pstep = part;  // the imaginary part of degree n is n + 1 further
    auto to_lanes = [&](auto nc, auto &xs) {
        constexpr int n = decltype(nc)::value;
        wave_fence();
        static_for<0, chunks(n)>([&](auto ic_) {
            constexpr int i = decltype(ic_)::value;
            const dbl2 v = in[n % kIn][i];
            *reinterpret_cast<double2 *>(put + 16 * i) = double2{v.x, v.y};
        });
        wave_fence();
        const double *b = get + pstep * (n + 1);
        static_for<0, 2 * chunks(n)>([&](auto ic_) {
            constexpr int e = decltype(ic_)::value & 1, j = decltype(ic_)::value >> 1;
            xs[e][j] = b[8 * j + e];
        });
    };
    auto to_target = [&](auto Nc, auto &xs) {
        constexpr int N = decltype(Nc)::value;
        if (mode == 2) {
            static_for<0, 2 * chunks(N)>([&](auto ic_) {
                constexpr int e = decltype(ic_)::value & 1, j = decltype(ic_)::value >> 1;
                const double a = dpp<0x101>(xs[e][j]);
                xs[e][j] += (same & 1u) ? a : 0.0;
                const double b = dpp<0x102>(xs[e][j]);
                xs[e][j] += (same & 2u) ? b : 0.0;
                const double d = dpp<0x104>(xs[e][j]);
                xs[e][j] += (same & 4u) ? d : 0.0;
            });
        }
        wave_fence();
        double *b = get + pstep * (N + 1);
        static_for<0, 2 * chunks(N)>([&](auto ic_) {
            constexpr int e = decltype(ic_)::value & 1, j = decltype(ic_)::value >> 1;
            if constexpr (8 * j + e + 6 <= N) {
                b[8 * j + e] = xs[e][j];
            } else if constexpr (8 * j + e <= N) {
                double *a = 2 * q + 8 * j + e <= N ? b + 8 * j + e : buf + t * ST + 16 * NJX + 4 * part + q;
                *a = xs[e][j];
            }
        });
        wave_fence();
        static_for<0, chunks(N)>([&](auto ic_) {
            constexpr int i = decltype(ic_)::value;
            const double2 w = *reinterpret_cast<const double2 *>(put + 16 * i);
            const dbl2 v = old[N % kOld][i] + dbl2{w.x, w.y};
            bool on = store && uint32_t(N) < p_dst;
            if constexpr (8 * i + 7 > N) on = on && c <= N - 8 * i;
            if (on) *reinterpret_cast<dbl2 *>(D + N * (N + 1) + 16 * i) = v;
        });
    };

    // The rotated triangle: T[e][j][K], order m = 2 (q + 4 j) + e of degree K
    // (entries with K below 8 j + e do not exist, those with K < m are zero).
    double T[2][NJX][PB];
    auto keep = [&](auto nc, const auto &xs) {
        constexpr int n = decltype(nc)::value;
        static_for<0, 2 * chunks(n)>([&](auto ic_) {
            constexpr int e = decltype(ic_)::value & 1, j = decltype(ic_)::value >> 1;
            if constexpr (8 * j + e <= n) T[e][j][n] = xs[e][j];
        });
    };
    auto clear = [&](auto nc) {
        constexpr int n = decltype(nc)::value;
        static_for<0, 2 * chunks(n)>([&](auto ic_) {
            constexpr int e = decltype(ic_)::value & 1, j = decltype(ic_)::value >> 1;
            if constexpr (8 * j + e <= n) T[e][j][n] = 0.0;
        });
    };
    // output degree N along z
    auto along_z = [&](auto Nc, auto &ys) {
        constexpr int N = decltype(Nc)::value;
        static_for<0, 2 * chunks(N)>([&](auto ic_) {
            constexpr int e = decltype(ic_)::value & 1, j = decltype(ic_)::value >> 1, m0 = 8 * j + e;
            double a = 0.0;
            if constexpr (m0 <= N) {
                constexpr int KB = OP == SFMM_L2L && N > m0 ? N : m0;
                constexpr int KE = OP == SFMM_M2M && N + 1 < PB ? N + 1 : PB;
                static_for<KB, KE>([&](auto Kc) {
                    constexpr int K = decltype(Kc)::value;
                    constexpr double f = OP == SFMM_M2L   ? ((N + e) & 1 ? -kFac.fac[N + K] : kFac.fac[N + K])
                                         : OP == SFMM_M2M ? kFac.inv[N - K]
                                                          : kFac.inv[K - N];
                    if constexpr (K == KB) a = f * T[e][j][K];
                    else a = __builtin_fma(f, T[e][j][K], a);
                });
            }
            ys[e][j] = a;
        });
    };

    // source degrees n0 .. n0 + C - 1
    auto take_in = [&](auto nc, auto cc, const auto &scale) {
        constexpr int n0 = decltype(nc)::value, C = decltype(cc)::value;
        if (n0 < pin_w) {
            double xs[C][2][NJX];
            static_for<0, C>([&](auto uc) { to_lanes(ic<n0 + decltype(uc)::value>{}, xs[decltype(uc)::value]); });
            forward<n0, C>(tab_f, lo, part, R, scale, xs);
            static_for<0, C>([&](auto uc) { keep(ic<n0 + decltype(uc)::value>{}, xs[decltype(uc)::value]); });
        } else {
            static_for<0, C>([&](auto uc) { clear(ic<n0 + decltype(uc)::value>{}); });
        }
    };
    auto give_out = [&](auto Nc, auto cc, const auto &scale) {
        constexpr int N0 = decltype(Nc)::value, C = decltype(cc)::value;
        if (N0 < pout_w) {
            double ys[C][2][NJX];
            static_for<0, C>([&](auto uc) { along_z(ic<N0 + decltype(uc)::value>{}, ys[decltype(uc)::value]); });
            backward<N0, C>(tab_b, lo, part, R, scale, ys);
            static_for<0, C>([&](auto uc) { to_target(ic<N0 + decltype(uc)::value>{}, ys[decltype(uc)::value]); });
        }
    };
    constexpr int kSteps = (PB + U - 1) / U;
    if constexpr (OP == SFMM_M2L) {
        double sc = rinv;  // r^-(n+1) (translations.cpp:45)
        static_for<0, kSteps>([&](auto kc) {
            constexpr int n0 = decltype(kc)::value * U, C = n0 + U < PB ? U : PB - n0;
            double scale[C];
            static_for<0, C>([&](auto uc) {
                scale[decltype(uc)::value] = sc;
                sc *= rinv;
                fetch_src(ic<n0 + 2 + decltype(uc)::value>{});
            });
            if constexpr (n0 + C == PB) static_for<0, U>(fetch_old);
            sched_fence();
            take_in(ic<n0>{}, ic<C>{}, scale);
        });
        double rp = 1.0;
        static_for<0, kSteps>([&](auto kc) {
            constexpr int N0 = decltype(kc)::value * U, C = N0 + U < PB ? U : PB - N0;
            double scale[C];
            static_for<0, C>([&](auto uc) {
                scale[decltype(uc)::value] = rp;
                rp *= rinv;
            });
            static_for<0, U>([&](auto uc) { fetch_old(ic<N0 + U + decltype(uc)::value>{}); });
            sched_fence();
            give_out(ic<N0>{}, ic<C>{}, scale);
        });
    } else if constexpr (OP == SFMM_M2M) {
        // output degree n needs source degrees up to n only
        double sc = rinv, sb = r;  // r^-(n+1); r^(N+1) (translations.cpp:129)
        static_for<0, kSteps>([&](auto kc) {
            constexpr int n0 = decltype(kc)::value * U, C = n0 + U < PB ? U : PB - n0;
            double fs[C], bs[C];
            static_for<0, C>([&](auto uc) {
                constexpr int u = decltype(uc)::value;
                fs[u] = sc;
                bs[u] = sb;
                sc *= rinv;
                sb *= r;
                fetch_src(ic<n0 + 2 + u>{});
                fetch_old(ic<n0 + u>{});
            });
            sched_fence();
            take_in(ic<n0>{}, ic<C>{}, fs);
            give_out(ic<n0>{}, ic<C>{}, bs);
        });
    } else {
        // forward r^n (translations.cpp:198), backward r^-n (:180),
        // descending: output degree n needs source degrees from n up
        double rf[PB], rb[PB];
        rf[0] = 1.0;
        rb[0] = 1.0;
        static_for<1, PB>([&](auto nc) {
            constexpr int n = decltype(nc)::value;
            rf[n] = rf[n - 1] * r;
            rb[n] = rb[n - 1] * rinv;
        });
        static_for<0, kSteps>([&](auto kc) {
            constexpr int top = PB - decltype(kc)::value * U, C = top < U ? top : U, n0 = top - C;
            double fs[C], bs[C];
            static_for<0, C>([&](auto uc) {
                constexpr int u = decltype(uc)::value;
                fs[u] = rf[n0 + u];
                bs[u] = rb[n0 + u];
                fetch_src(ic<n0 + u - 2>{});
                fetch_old(ic<n0 + u>{});
            });
            sched_fence();
            take_in(ic<n0>{}, ic<C>{}, fs);
            give_out(ic<n0>{}, ic<C>{}, bs);
        });
    }

    late();
    if (zero_shift) {
        // target += source over the common degrees (translations.cpp:539-547,
        // 596-604)
        const double *s = src_pool + G.src;
        double *d = dst_pool + block;
        const int len = int(p_end * (p_end + 1));
        for (int i = c; i < len; i += kItems) d[i] = (acc ? d[i] : 0.0) + s[i];
    }
}

constexpr int waves(int pb) { return pb <= 12 || pb >= 17 ? 4 : 8; }
constexpr int per_simd(int pb) { return pb <= 8 ? 3 : pb <= 16 ? 2 : 1; }
constexpr int tables(int op) { return op == SFMM_M2L ? 2 : 1; }
constexpr size_t lds_bytes(int op, int pb)
{
    return sizeof(double) * size_t(tables(op) * table_size(pb) + waves(pb) * kItems * stage_stride(chunks(pb - 1)));
}

// Persistent workgroups: stage the swap operands in LDS, then each wave takes
// groups of eight translations.
template <int OP, int PB, bool PAIRS>
__global__ void __launch_bounds__(64 * waves(PB)) __attribute__((amdgpu_waves_per_eu(per_simd(PB))))
    k_octet(const double *__restrict__ src_pool, double *__restrict__ dst_pool, const sfmm_item *__restrict__ items,
            uint32_t n_items, const double *__restrict__ tables_m, const double *__restrict__ tables_l, int mode)
{
    extern __shared__ __align__(16) double lds[];
    constexpr int W = waves(PB), SIZE = table_size(PB);
    const int lane = int(threadIdx.x & 63), wave = int(threadIdx.x >> 6);
    const uint32_t groups = (n_items + kItems - 1) / kItems;
    constexpr uint32_t kPair = PAIRS ? 1 : 0;  // a wave takes two groups in a row
    uint32_t g = (blockIdx.x * W + uint32_t(wave)) << kPair;
    Group next{};
    if (g < groups) next.load(items, n_items, g, lane);
    const double2 *from_m = reinterpret_cast<const double2 *>(OP == SFMM_L2L ? tables_l : tables_m);
    for (int i = int(threadIdx.x); i < SIZE / 2; i += 64 * W) reinterpret_cast<double2 *>(lds)[i] = from_m[i];
    if constexpr (tables(OP) == 2)
        for (int i = int(threadIdx.x); i < SIZE / 2; i += 64 * W)
            reinterpret_cast<double2 *>(lds + SIZE)[i] = reinterpret_cast<const double2 *>(tables_l)[i];
    __syncthreads();

    double *buf = lds + tables(OP) * SIZE + wave * kItems * stage_stride(chunks(PB - 1));
    // the next group's items are requested before a group where registers
    // allow (14 of them), after it otherwise
    constexpr bool kEarly = PB <= 12 || PB >= 17;
    while (g < groups) {
        const Group G = next;
        const uint32_t cur = g;
        g += (cur & kPair) == kPair ? ((gridDim.x * W) << kPair) - kPair : 1;
        if (kEarly && g < groups) next.load(items, n_items, g, lane);
        // an opaque zero offset per group keeps the compiler from holding
        // operands in registers across groups
        int base = 0;
        asm volatile("" : "+s"(base));
        translate_group<OP, PB, PAIRS>(src_pool, dst_pool, G, n_items, cur, lds + base, buf, lane, mode, [&] {
            if (!kEarly && g < groups) next.load(items, n_items, g, lane);
        });
    }
}

using fn_t = void (*)(const double *, double *, const sfmm_item *, uint32_t, const double *, const double *, int);

template <int OP, bool PAIRS, int FIRST, int... Ps>
constexpr auto make_table(std::integer_sequence<int, Ps...>)
{
    struct T {
        fn_t f[sizeof...(Ps)];
    } t{{&k_octet<OP, FIRST + Ps, PAIRS>...}};
    return t;
}

template <int OP>
hipError_t launch_op(uint32_t pb, const sfmm_item *items, size_t n, const double *src, double *dst,
                     hipStream_t stream, int mode, bool pairs)
{
    static const auto single = make_table<OP, false, 1>(std::make_integer_sequence<int, max_order(OP)>{});
    static const auto paired =
        make_table<OP, true, kPairsMin>(std::make_integer_sequence<int, kPairsMax - kPairsMin + 1>{});
    if (pb < 1 || pb > uint32_t(max_order(OP))) return hipErrorInvalidValue;
    if (pairs && (mode != 2 || pb < kPairsMin || pb > kPairsMax)) return hipErrorInvalidValue;
    const double *table = device_table();
    if (!table) return hipErrorOutOfMemory;
    const fn_t f = pairs ? paired.f[pb - kPairsMin] : single.f[pb - 1];
    const size_t lds = lds_bytes(OP, int(pb));
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(f),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return e;
    }
    const size_t w = size_t(waves(int(pb))), groups = (n + kItems - 1) / kItems;
    const size_t units = pairs ? (groups + 1) / 2 : groups;  // what a wave takes at a time
    const uint32_t grid = persistent_grid(reinterpret_cast<const void *>(f), int(64 * w), (units + w - 1) / w, lds);
    hipLaunchKernelGGL(f, dim3(grid), dim3(uint32_t(64 * w)), uint32_t(lds), stream, src, dst, items, uint32_t(n),
                       table, table + table_size(kMaxOrder), mode);
    return hipGetLastError();
}

}  // namespace octet
}  // namespace sfmm
