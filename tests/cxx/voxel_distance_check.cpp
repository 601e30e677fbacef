// voxel_distance_check.cpp -- the FP32 voxel kernels' distance from the source on the CPU.
//
// Built with g++ against elsa_amd/csrc/ehp_voxel.hpp (source_dist2, the function the HIP kernels call):
// its errors and those of elsa's FP32 order over random voxels, against 64-bit arithmetic on the same
// matrices. Used by tests/test_voxel_distance.py.
#include "ehp_voxel.hpp"

#include <cmath>
#include <random>

using namespace ehp;

namespace
{
    template <int D>
    int run(const int* vol, int nposes, const float* ext, int count, double* rms)
    {
        std::mt19937 gen(7);
        double sum[2] = {0.0, 0.0};
        for (int p = 0; p < nposes; ++p) {
            PoseGeom g{};
            for (int i = 0; i < D * (D + 1); ++i)
                g.ext[i] = ext[p * D * (D + 1) + i];
            for (int k = 0; k < count; ++k) {
                int v[3] = {0, 0, 0};
                double exact = 0.0;
                for (int i = 0; i < D; ++i)
                    v[i] = (int) (gen() % (unsigned) vol[i]);
                for (int i = 0; i < D; ++i) {
                    double c = g.ext[i + D * D];
                    for (int j = 0; j < D; ++j)
                        c += (double) g.ext[i + j * D] * (v[j] + 0.5);
                    exact += c * c;
                }
                float pc[3], ce[3];
                voxel_project<D>(g, v[0], v[1], v[2], pc, ce);
                float elsa = ce[0] * ce[0];
                for (int i = 1; i < D; ++i)
                    elsa = elsa + ce[i] * ce[i];
                const float got = source_dist2<D>(g, v[0], v[1], v[2]);
                if (D == 2 && got != elsa)
                    return 1;
                const double e0 = got / exact - 1.0, e1 = elsa / exact - 1.0;
                sum[0] += e0 * e0;
                sum[1] += e1 * e1;
            }
        }
        for (int i = 0; i < 2; ++i)
            rms[i] = std::sqrt(sum[i] / ((double) nposes * count));
        return 0;
    }
} // namespace

// rms[0]: the relative RMS error of source_dist2, rms[1]: of elsa's order
extern "C" int voxel_distance(int dim, const int* vol, int nposes, const float* ext, int count, double* rms)
{
    return dim == 2 ? run<2>(vol, nposes, ext, count, rms) : run<3>(vol, nposes, ext, count, rms);
}
