// Host construction of the folded swap blocks for any degree, and of the
// dense device table (layout in mfma_tables.hpp) that the MFMA and generic
// kernels read.
//
// B_n^{m,l} by Dehnen's recurrence (swap_matrix.cpp:148-171): B_0 = 1; the
// row m = 0 of degree n from 0.5 (b(0,l-1) - b(0,l+1)) of degree n-1; rows
// m+1 and -m-1 from rows m and -m of degree n-1.  The folded real and
// imaginary blocks over the stored orders m, l >= 0 follow
// operator_data.cpp:47-147.  Same double operations in the same order as
// the compile-time tables of tables.hpp, so the values agree bit for bit
// (checked by the test-suite through sfmm_swap_block).
#include <hip/hip_runtime.h>

#include <cstring>
#include <mutex>
#include <vector>

#include "../../include/solidfmm_gpu.h"
#include "mfma_tables.hpp"
#include "octet_tables.hpp"
#include "team_tables.hpp"

namespace sfmm {

namespace {

// B_n for n < nmax, each as a (2n+1)^2 array indexed [(m+n) + (l+n)(2n+1)].
struct SwapRecurrence {
    std::vector<std::vector<double>> B;

    double get(int n, int m, int l) const
    {
        if (m < -n || m > n || l < -n || l > n) return 0.0;
        return B[n][(m + n) + (l + n) * (2 * n + 1)];
    }

    void extend(int nmax)
    {
        for (int n = int(B.size()); n < nmax; ++n) {
            std::vector<double> a(size_t(2 * n + 1) * (2 * n + 1), 0.0);
            auto at = [n](int m, int l) { return size_t((m + n) + (l + n) * (2 * n + 1)); };
            if (n == 0) {
                a[0] = 1.0;
            } else {
                for (int l = -n; l <= n; ++l) a[at(0, l)] = 0.5 * (get(n - 1, 0, l - 1) - get(n - 1, 0, l + 1));
                for (int m = 0; m < n; ++m)
                    for (int l = -n; l <= n; ++l) {
                        a[at(m + 1, l)] = 0.5 * (get(n - 1, m, l - 1) + get(n - 1, m, l + 1)) + get(n - 1, m, l);
                        a[at(-m - 1, l)] =
                            0.5 * (get(n - 1, -m, l - 1) + get(n - 1, -m, l + 1)) - get(n - 1, -m, l);
                    }
            }
            B.push_back(std::move(a));
        }
    }

    // Folded block entry [m][l] of degree n; part 0 real, 1 imaginary.
    double folded(int n, int part, int m, int l) const
    {
        const bool odd = ((l + m + n) & 1) != 0;
        if (part == 0 ? odd : !odd) return 0.0;
        const double bp = get(n, l, m), bm = get(n, -l, m);
        if (part == 0) {
            if (l == 0) return get(n, 0, m);
            return (l & 1) ? bp - bm : bp + bm;
        }
        return (l & 1) ? bp + bm : bp - bm;
    }
};

// Built once for every tabulated degree, then only read.
const SwapRecurrence &recurrence()
{
    static const SwapRecurrence rec = [] {
        SwapRecurrence r;
        r.extend(mfma::kMaxOrder);
        return r;
    }();
    return rec;
}

// One device copy per device of a table built on the host.
class DeviceCopies {
    std::mutex mu;
    std::vector<double *> per_device;

public:
    const double *get(std::vector<double> (*build)())
    {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return nullptr;
        std::lock_guard<std::mutex> lock(mu);
        if (per_device.size() <= size_t(dev)) per_device.resize(dev + 1, nullptr);
        if (!per_device[dev]) {
            const std::vector<double> h = build();
            double *d = nullptr;
            if (hipMalloc(&d, h.size() * sizeof(double)) != hipSuccess) return nullptr;
            if (hipMemcpy(d, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
                (void)hipFree(d);
                return nullptr;
            }
            per_device[dev] = d;
        }
        return per_device[dev];
    }
};

}  // namespace

namespace mfma {

void build_table(double *out)
{
    const SwapRecurrence &rec = recurrence();
    for (int n = 0; n < kMaxOrder; ++n) {
        const int st = dense_stride(n);
        double *sr = out + dense_base(n);
        double *si = sr + dense_part(n);
        for (int m = 0; m <= n; ++m)
            for (int l = 0; l < st; ++l) {
                sr[size_t(m) * st + l] = (l <= n) ? rec.folded(n, 0, m, l) : 0.0;
                si[size_t(m) * st + l] = (l <= n) ? rec.folded(n, 1, m, l) : 0.0;
            }
    }
}

namespace {
struct DeviceTables {
    std::mutex mu;
    std::vector<double *> per_device;
};
DeviceTables &tables_state()
{
    static DeviceTables s;
    return s;
}
}  // namespace

const double *device_table()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    DeviceTables &st = tables_state();
    std::lock_guard<std::mutex> lock(st.mu);
    if (st.per_device.size() <= size_t(dev)) st.per_device.resize(dev + 1, nullptr);
    if (!st.per_device[dev]) {
        std::vector<double> host(table_doubles());
        build_table(host.data());
        double *d = nullptr;
        if (hipMalloc(&d, host.size() * sizeof(double)) != hipSuccess) return nullptr;
        if (hipMemcpy(d, host.data(), host.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipFree(d);
            return nullptr;
        }
        st.per_device[dev] = d;
    }
    return st.per_device[dev];
}

const double *device_factorials()
{
    static std::mutex mu;
    static std::vector<double *> per_device;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    if (per_device.size() <= size_t(dev)) per_device.resize(dev + 1, nullptr);
    if (!per_device[dev]) {
        std::vector<double> h(4 * size_t(kMaxOrder));
        h[0] = 1.0;
        // (2 kMaxOrder - 1)! overflows to inf; the kernels read n! only for
        // n <= 2 kMaxOrder - 2.
        for (int i = 1; i < 2 * kMaxOrder; ++i) h[i] = double(i) * h[i - 1];
        for (int i = 0; i < 2 * kMaxOrder; ++i) h[2 * kMaxOrder + i] = 1.0 / h[i];
        double *d = nullptr;
        if (hipMalloc(&d, h.size() * sizeof(double)) != hipSuccess) return nullptr;
        if (hipMemcpy(d, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipFree(d);
            return nullptr;
        }
        per_device[dev] = d;
    }
    return per_device[dev];
}

}  // namespace mfma

namespace team {

namespace {

// Both tables of team_tables.hpp.
std::vector<double> build_tables()
{
    const SwapRecurrence &rec = recurrence();
    std::vector<double> out(2 * size_t(table_size()), 0.0);
    for (int n = 0; n < kMaxOrder; ++n) {
        const int nj = chunks(n);
        double *deg = out.data() + base_of(nj) + size_t(n - 8 * (nj - 1)) * degree_size(nj);
        for (int block = 0; block < 4; ++block) {
            const int part = block / 2, e = block % 2;
            const int o = (e + n + part) & 1;  // class of the outputs
            for (int i = 0; 2 * i + o <= n; ++i)
                for (int j = 0; 2 * j + e <= n; ++j) {
                    size_t at;
                    if (nj <= kSmall) {
                        const int p = (block * nj + i / 4) * nj + j / 4;  // operand
                        at = size_t(p / 2) * 32 + (i % 4 + 4 * (j % 4)) * 2 + p % 2;
                    } else {
                        const int p = (block * row_blocks(nj) + i / 16) * nj + j / 4;
                        at = size_t(p) * 64 + i % 16 + 16 * (j % 4);
                    }
                    const int m = 2 * i + o, l = 2 * j + e;
                    deg[at] = rec.folded(n, part, m, l);
                    deg[table_size() + at] = (l ? 2.0 : 1.0) * (m ? 0.5 : 1.0) * rec.folded(n, part, l, m);
                }
        }
    }
    return out;
}

}  // namespace

const double *device_table()
{
    static DeviceCopies copies;
    return copies.get(build_tables);
}

}  // namespace team

namespace octet {

namespace {

// Both tables of octet_tables.hpp.
std::vector<double> build_tables()
{
    const SwapRecurrence &rec = recurrence();
    const int size = table_size(kMaxOrder);
    std::vector<double> out(2 * size_t(size), 0.0);
    for (int n = 0; n < kMaxOrder; ++n)
        for (int part = 0; part < 2; ++part)
            for (int e = 0; e < 2; ++e) {
                const int o = (e + n + part) & 1;  // class of the outputs
                for (int i = 0; 2 * i + o <= n; ++i)
                    for (int j = 0; 2 * j + e <= n; ++j) {
                        const int at = entry(n, part, e, i / 4, j / 4, i % 4, j % 4);
                        const int m = 2 * i + o, l = 2 * j + e;
                        out[at] = rec.folded(n, part, m, l);
                        out[size + at] = (l ? 2.0 : 1.0) * (m ? 0.5 : 1.0) * rec.folded(n, part, l, m);
                    }
            }
    return out;
}

}  // namespace

const double *device_table()
{
    static DeviceCopies copies;
    return copies.get(build_tables);
}

}  // namespace octet
}  // namespace sfmm

extern "C" int sfmm_swap_block(int n, int part, double *out)
{
    if (n < 0 || n >= sfmm::mfma::kMaxOrder || (part != 0 && part != 1) || !out) return SFMM_ERR_LOGIC;
    const auto &rec = sfmm::recurrence();
    for (int m = 0; m <= n; ++m)
        for (int l = 0; l <= n; ++l) out[size_t(m) * (n + 1) + l] = rec.folded(n, part, m, l);
    return SFMM_OK;
}
