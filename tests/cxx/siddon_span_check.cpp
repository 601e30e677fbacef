// siddon_span_check.cpp -- runs the plane-by-plane Siddon forward on the CPU.
//
// Built with g++ against elsa_amd/csrc/ehp_siddon.hpp (the functions the HIP kernel calls): rays
// given by origin and direction walk a zero-padded plane-major view (sid_span_init, sid_plane_add)
// of a volume whose voxels off the ray are NaN. The sum must equal siddon_traverse's bit for bit,
// and every read must lie in the ray's plane. The same rays through the tiles of the back
// projection (sid_tile_ray) must give each of the traversal's crossings of nonzero length once, in
// its slot and with its length. Used by tests/test_siddon_span.py.
#include "ehp_siddon.hpp"

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <map>
#include <vector>

using namespace ehp;

namespace
{
    template <int D, int A, bool FB2, class T>
    int run(const Dims& dims, const SidRec& r, const std::vector<T>& vol)
    {
        constexpr uint32_t lg = sizeof(T) == 8 ? 3u : 2u;
        const int f = D == 2 ? 1 - A : (FB2 ? TileAxes<D, A>::b2 : TileAxes<D, A>::b1);
        const PadLayout L = pad_layout(dims, A, f);
        std::vector<T> view(L.size, T(0));
        for (int z = 0; z < dims.vol[2]; ++z)
            for (int y = 0; y < dims.vol[1]; ++y)
                for (int x = 0; x < dims.vol[0]; ++x)
                    view[pad_index(L, x, y, z)] = std::numeric_limits<T>::quiet_NaN();
        T ref = T(0);
        int crossings = 0;
        siddon_traverse<D>(r, dims.vol, [&](int c0, int c1, int c2, float w) {
            const T v = vol[c0 + c1 * dims.strides[1] + c2 * dims.strides[2]];
            view[pad_index(L, c0, c1, c2)] = v;
            ref += v * (T) w;
            ++crossings;
        });
        T acc = T(0);
        bool bad = false;
        if (sid_hit(r)) {
            SidSpan s = sid_span_init<D, A, FB2>(r, dims.vol, (uint32_t) (L.RS << lg), lg);
            const int dir = sid_step(r, A);
            const bool twice = sid_may_cross_twice<D, A>(r, s.tend);
            auto add = [&](const SidRec& rr, SidSpan& ss, T sum, auto ld) {
                return twice ? sid_plane_add<D, A, T>(rr, ss, sum, ld)
                             : sid_segments_add<D>(sid_plane_segments<D, A, T>(rr, ss, ld), sum);
            };
            for (int p = r.cur0[A]; p >= 0 && p < dims.vol[A] && s.t < s.tend; p += dir)
                acc = add(r, s, acc, [&](uint32_t off) {
                    if ((off & (sizeof(T) - 1)) || (off >> lg) >= L.PS) {
                        bad = true;
                        return T(0);
                    }
                    return view[(int64_t) p * L.PS + (off >> lg)];
                });
        }
        if (bad)
            return 2;
        if (std::memcmp(&acc, &ref, sizeof(T)) != 0) {
            std::fprintf(stderr, "sum %.17g, traversal %.17g over %d crossings (axis %d)\n", (double) acc, (double) ref,
                         crossings, A);
            return 3;
        }
        return 0;
    }

    // every tile of the pass along A: the crossings of ray r by voxel
    template <int D, int A>
    int tiles(const Dims& dims, const SidRec& r, const TileCfg& tc)
    {
        constexpr int b1 = TileAxes<D, A>::b1, b2 = TileAxes<D, A>::b2;
        std::map<int64_t, float> full, got;
        siddon_traverse<D>(r, dims.vol, [&](int c0, int c1, int c2, float w) {
            if (w != 0.0f)
                full[c0 + c1 * dims.strides[1] + c2 * dims.strides[2]] = w;
        });
        int ntA, ntB, ntC, rc = 0;
        tile_counts(dims, tc, A, ntA, ntB, ntC);
        const int row = sid_row_slots(tc, D);
        for (int tile = 0; tile < ntA * ntB * ntC && !rc; ++tile) {
            const TileBox t = make_tile<D, A>(dims, tc, tile % ntA, (tile / ntA) % ntB, tile / (ntA * ntB));
            sid_tile_ray<D, A>(r, t, sid_tile_offsets<D>(t, tc), [&](uint32_t off, float w) {
                const int slot = (int) (off / 8), xb = slot % row, rest = slot / row;
                const int xc = D == 3 ? rest % tc.TC : 0, xa = D == 3 ? rest / tc.TC : rest;
                int c[3] = {0, 0, 0};
                c[A] = t.A0 + xa;
                c[b1] = t.B0 + xb;
                if (D == 3)
                    c[b2] = t.C0 + xc;
                if (off % 8 || xa >= t.A1 - t.A0 || c[b1] >= t.B1 || (D == 3 && c[b2] >= t.C1)) {
                    rc = 4; // outside the tile
                    return;
                }
                const int64_t lin = c[0] + c[1] * dims.strides[1] + c[2] * dims.strides[2];
                if (!got.emplace(lin, w).second)
                    rc = 5; // a voxel twice
            });
        }
        if (!rc && got != full) {
            std::fprintf(stderr, "%zu crossings in the tiles, %zu in the traversal (axis %d)\n", got.size(), full.size(), A);
            rc = 6;
        }
        return rc;
    }

    template <int D, class T>
    int all(const int64_t* n, const float* od, int nrays, const T* data, int64_t* per_axis)
    {
        Dims d{};
        d.dim = D;
        for (int i = 0; i < 3; ++i)
            d.vol[i] = i < D ? (int) n[i] : 1;
        d.strides[0] = 1;
        d.strides[1] = d.vol[0];
        d.strides[2] = (int64_t) d.vol[0] * d.vol[1];
        d.nvox = (int64_t) d.vol[0] * d.vol[1] * d.vol[2];
        const std::vector<T> vol(data, data + d.nvox);
        for (int k = 0; k < nrays; ++k) {
            const SidRec r = siddon_setup<D>(od + 6 * k, od + 6 * k + 3, d.vol);
            const int a = sid_axis(r);
            int rc = 0;
            if (a == 0) {
                rc = run<D, 0, false, T>(d, r, vol);
                if (!rc && D == 3)
                    rc = run<D, 0, true, T>(d, r, vol);
            } else if (a == 1) {
                rc = run<D, 1, false, T>(d, r, vol);
                if (!rc && D == 3)
                    rc = run<D, 1, true, T>(d, r, vol);
            } else {
                rc = run<D, D - 1, false, T>(d, r, vol);
                if (!rc && D == 3)
                    rc = run<D, D - 1, true, T>(d, r, vol);
            }
            const TileCfg cfgs[] = {{8, 16, 16}, {3, 5, 4}, {1, 2, 1}, {64, 64, 64}};
            for (const TileCfg& tc : cfgs)
                if (!rc && sid_hit(r))
                    rc = a == 0 ? tiles<D, 0>(d, r, tc) : (a == 1 ? tiles<D, 1>(d, r, tc) : tiles<D, D - 1>(d, r, tc));
            if (rc) {
                std::fprintf(stderr, "ray %d\n", k);
                return rc;
            }
            per_axis[a] += sid_hit(r);
        }
        return 0;
    }
} // namespace

// od: nrays x 6, origin and direction (dim 2: the first two of each)
extern "C" int siddon_span32(int dim, const int64_t* n, const float* od, int nrays, const float* vol, int64_t* axes)
{
    return dim == 2 ? all<2, float>(n, od, nrays, vol, axes) : all<3, float>(n, od, nrays, vol, axes);
}

extern "C" int siddon_span64(int dim, const int64_t* n, const float* od, int nrays, const double* vol, int64_t* axes)
{
    return dim == 2 ? all<2, double>(n, od, nrays, vol, axes) : all<3, double>(n, od, nrays, vol, axes);
}
