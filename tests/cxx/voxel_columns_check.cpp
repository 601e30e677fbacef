// voxel_columns_check.cpp -- the voxel kernels' footprints by columns on the CPU.
//
// Built with g++ against elsa_amd/csrc/ehp_voxel.hpp (the functions the HIP kernels call): random
// footprints of scalings in [smin, smax]. Every footprint must fit the columns, the FP64 weights must
// be those of visit() and tap_weight bit for bit, the FP32 weights theirs within the rounding of the
// table index, columns past the footprint must weigh 0 and every table index must lie in the span that
// the kernels lay out. Used by tests/test_voxel_columns.py.
#include "ehp_voxel.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <type_traits>
#include <vector>

using namespace ehp;

namespace
{
    template <int NC, bool TZ>
    int run(const std::vector<double>& lut, float support, double smin, double smax, bool diff, int count)
    {
        const int n = (int) lut.size();
        std::vector<float> lut32(lut.begin(), lut.end());
        std::vector<double> ref(lut32.begin(), lut32.end()), tab64(lut);
        tab64.push_back(0.0);
        const int span = (int) column_table_span(n, support, smin, NC);
        std::vector<float> tab(2 * (size_t) span, NAN);
        for (int i = 0; i < span; ++i)
            lerp_table_entry(lut32.data(), n, i, tab.data());
        double step = 0.0, top = 0.0;
        for (int i = 0; i < n; ++i) {
            top = std::max(top, std::fabs(ref[i]));
            if (i > 0)
                step = std::max(step, std::fabs(ref[i] - ref[i - 1]));
        }
        const double reach = diff ? support : 1.0;
        std::mt19937 gen(5);
        std::uniform_real_distribution<double> uni(0.0, 1.0);
        for (int k = 0; k < count; ++k) {
            Footprint fp{};
            fp.scaling = (float) (smin + (smax - smin) * (k == 0 ? 0.0 : (k == 1 ? 1.0 : uni(gen))));
            const float rod = fp.scaling * support;
            fp.center[0] = (float) (100.0 * uni(gen) + 20.0);
            fp.center[1] = (float) (100.0 * uni(gen) + 20.0);
            if (k % 4 == 1)
                fp.center[0] = std::floor(fp.center[0]) + rod; // the first column at the very rim
            const int l0 = (int) std::ceil(fp.center[0] - rod), h0 = (int) std::floor(fp.center[0] + rod);
            const int j0 = (int) std::ceil(fp.center[1] - rod), j1 = (int) std::floor(fp.center[1] + rod);
            if (h0 - l0 + 1 > NC)
                return 1;
            const float rs = 1.0f / fp.scaling, rsk = rs * ((float) (n - 1) / support);
            float d0k[NC], du[NC], w[NC], d0[NC];
            double w64[NC];
            column_units<NC, TZ>(fp.center[0], l0, h0, rs, rsk, diff, d0k, du);
            column_units64<NC>(fp.center[0], l0, h0, fp.scaling, 1.0f / fp.scaling, d0);
            for (int j = j0; j <= j1; ++j) {
                row_units<NC, TZ>(tab.data(), n, fp.center[1], j, rsk, d0k, du, diff, w);
                row_units64<NC>(tab64.data(), n, support, 1.0f / support, fp.center[1], j, fp.scaling,
                                1.0f / fp.scaling, d0, diff, w64);
                // clipped to columns of the footprint's middle (the detector's edge): the same weights
                // inside, 0 past the last from entries of the pair table
                float dc[NC], uc[NC], wc[NC];
                const int lo = l0 + (k & 1), last = h0 - lo - (k >> 1 & 1);
                column_units_clipped<NC>(fp.center[0], lo, last, n, rs, rsk, diff, dc, uc);
                row_units<NC, TZ>(tab.data(), n, fp.center[1], j, rsk, dc, uc, diff, wc);
                for (int i = 0; i < NC; ++i) {
                    const float d1c = (fp.center[1] - (float) j) * rsk;
                    if ((int) std::sqrt(std::fma(dc[i], dc[i], d1c * d1c)) >= lerp_table_size(n))
                        return 6;
                    if (i <= last ? wc[i] != w[i + (k & 1)] : wc[i] != 0.0f)
                        return 7;
                }
                for (int i = 0; i < NC; ++i) {
                    const float d1k = (fp.center[1] - (float) j) * rsk;
                    if (TZ && (int) std::sqrt(std::fma(d0k[i], d0k[i], d1k * d1k)) >= span)
                        return 2;
                    if (l0 + i > h0) {
                        if (w[i] != 0.0f || w64[i] != 0.0)
                            return 3;
                        continue;
                    }
                    // as visit() has them
                    const float e0 = (fp.center[0] - (float) (l0 + i)) / fp.scaling;
                    const float e1 = (fp.center[1] - (float) j) / fp.scaling;
                    const float dist = std::sqrt(e0 * e0 + e1 * e1);
                    if (w64[i] != tap_weight<3, double>(lut.data(), n, support, dist, e0, diff))
                        return 4;
                    const double index = (double) dist / support * (n - 1);
                    if (!TZ && std::fabs(index - (n - 1)) < 1.0e-5 * n)
                        continue; // the table's jump to 0
                    const double want = tap_weight<3, double>(ref.data(), n, support, dist, e0, diff);
                    // a handful of roundings of the index (half an ulp each) and of the weight
                    if (std::fabs(w[i] - want) > reach * (step * index * 8 * 6.0e-8 + top * 4 * 6.0e-8))
                        return 5;
                }
            }
        }
        return 0;
    }
} // namespace

extern "C" int voxel_columns(int n, float support, double smin, double smax, double tail, int diff, int count,
                             int* cols_out)
{
    std::vector<double> lut(n);
    for (int i = 0; i < n; ++i) {
        const double t = (double) i / (n - 1);
        lut[i] = (1.0 - t * t) * std::exp(-3.0 * t) + tail;
    }
    lut[n - 1] = tail;
    const int cols = footprint_cols(support, smax);
    *cols_out = cols;
    if (cols > kVoxMaxCols)
        return 0;
    auto go = [&](auto tz) {
        constexpr bool TZ = decltype(tz)::value;
        switch (kernel_cols(cols)) {
            case 4: return run<4, TZ>(lut, support, smin, smax, diff != 0, count);
            case 5: return run<5, TZ>(lut, support, smin, smax, diff != 0, count);
            case 6: return run<6, TZ>(lut, support, smin, smax, diff != 0, count);
            default: return run<8, TZ>(lut, support, smin, smax, diff != 0, count);
        }
    };
    return tail == 0.0 ? go(std::true_type{}) : go(std::false_type{});
}
