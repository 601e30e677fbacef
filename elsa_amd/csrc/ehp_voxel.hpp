// ehp_voxel.hpp -- footprint arithmetic of the voxel-driven projectors, shared by the GPU
// kernels and the CPU checks.
//
// elsa/projectors/VoxelComputation.h:40-107 (projectAndScaleVoxelOnDetector,
// visitDetector): the voxel centre projected to the detector (minus 0.5), the scaling
// sdd / |ext x|, and the detector pixels within radius * scaling of the centre -- the full
// rectangle [ceil(c - r s), floor(c + r s)] (elsa's CPU loop visits it correctly only for
// square footprints, VoxelComputation.h:90-105) -- each weighted with the projected basis
// function at the distance |c - pixel| / scaling, read from a table by Luts.hpp:60-78.
#pragma once

#include "ehp_joseph_tile.hpp"

namespace ehp
{
    // Largest table of the LDS-table kernels (tiled forward, FP32 gather back projection)
    constexpr int kVoxMaxLut = 1024;

    // Entries of the FP32 kernels' pair table of an n-entry table: the entries and zeros past
    // sqrt(2) (n - 1), the largest index a tap of a footprint rectangle reaches (|d0|, |d1| at most
    // the radius, up to rounding), plus the entry after it.
    EHP_HD inline int lerp_table_size(int n)
    {
        return (int) (1.4143f * (float) (n - 1)) + 3;
    }
    constexpr int kVoxLutSpan = (int) (1.4143f * (float) (kVoxMaxLut - 1)) + 3;

    template <class T>
    EHP_HD inline T lut_eval(const T* __restrict__ lut, int n, float support, float distance)
    {
        const float index = (distance / support) * (float) (n - 1);
        if (index < 0.0f || index > (float) (n - 1))
            return T(0);
        const int a = (int) floorf(index);
        const int b = (int) ceilf(index);
        const T fa = lut[a];
        const T fb = lut[b];
        const T t = (T) (index - (float) a);
        return t * fb + (T(1) - t) * fa;
    }

    // Footprint of voxel (x, y, z) in one pose (VoxelComputation.h:40-107, full rectangle).
    struct Footprint {
        float center[2];
        float scaling;
        int lo[2];
        int hi[2];
    };

    // P (x + 0.5) and ext (x + 0.5) of voxel (x, y, z), homogeneous (VoxelComputation.h:40-60)
    template <int D>
    EHP_HD inline void voxel_project(const PoseGeom& g, int x, int y, int z, float* pc, float* ce)
    {
        float hv[4];
        hv[0] = (float) x + 0.5f;
        hv[1] = (float) y + 0.5f;
        hv[2] = (float) z + 0.5f;
        hv[D] = 1.0f;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            float acc = g.P[i] * hv[0];
            float acc2 = g.ext[i] * hv[0];
#pragma unroll
            for (int j = 1; j <= D; ++j) {
                acc = acc + g.P[i + j * D] * hv[j];
                acc2 = acc2 + g.ext[i + j * D] * hv[j];
            }
            pc[i] = acc;
            ce[i] = acc2;
        }
    }

    // The pixel rectangle [ceil(c - r s), floor(c + r s)] of a footprint, clipped to the detector
    template <int D>
    EHP_HD inline void footprint_rect(const Dims& dims, float radius, Footprint& fp)
    {
        const float rod = fp.scaling * radius;
#pragma unroll
        for (int i = 0; i < D - 1; ++i) {
            const int l = (int) ceilf(fp.center[i] - rod);
            const int h = (int) floorf(fp.center[i] + rod);
            fp.lo[i] = l < 0 ? 0 : l;
            fp.hi[i] = h > dims.det[i] - 1 ? dims.det[i] - 1 : h;
        }
        if (D == 2) {
            fp.lo[1] = 0;
            fp.hi[1] = 0;
        }
    }

    template <int D>
    EHP_HD inline void footprint(const PoseGeom& g, const Dims& dims, int x, int y, int z, float radius,
                                     Footprint& fp)
    {
        float pc[3], ce[3];
        voxel_project<D>(g, x, y, z, pc, ce);
#pragma unroll
        for (int i = 0; i < D - 1; ++i)
            fp.center[i] = pc[i] / pc[D - 1] - 0.5f;
        float n2 = ce[0] * ce[0];
#pragma unroll
        for (int i = 1; i < D; ++i)
            n2 = n2 + ce[i] * ce[i];
        fp.scaling = g.sdd / sqrtf(n2);
        footprint_rect<D>(dims, radius, fp);
    }

    // |ext x|^2 of voxel (x, y, z) for the FP32 kernels. 2D: elsa's order. 3D: the rotated coordinates by
    // FMAs with the translation (the source's distance, up to a hundred times the volume) added last, so that
    // only the last addition rounds at that size, and the squares by FMAs: eight instructions a voxel less than
    // elsa's order, and an RMS error of the scaling against 64 bits of 4.9e-8 instead of 5.1e-8 (36 to 400 voxels
    // a side, source 100 sides away; 4.6e-8 and 4.85e-8 at a source 1.2 sides away). An FMA chain that
    // starts with the translation rounds at its size at every step: 5.3e-8 to 5.7e-8.
    template <int D>
    EHP_HD inline float source_dist2(const PoseGeom& g, int x, int y, int z)
    {
        if constexpr (D == 2) {
            float pc[3], ce[3];
            voxel_project<2>(g, x, y, z, pc, ce);
            return ce[0] * ce[0] + ce[1] * ce[1];
        } else {
            const float h[3] = {(float) x + 0.5f, (float) y + 0.5f, (float) z + 0.5f};
            float n2 = 0.0f;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                float c = g.ext[i] * h[0];
                c = __builtin_fmaf(g.ext[i + 3], h[1], c);
                c = __builtin_fmaf(g.ext[i + 6], h[2], c);
                c = c + g.ext[i + 9];
                n2 = i == 0 ? c * c : __builtin_fmaf(c, c, n2);
            }
            return n2;
        }
    }

    // Reciprocal and reciprocal square root in one instruction each (v_rcp_f32, v_rsq_f32, within
    // 1 ulp); correctly rounded on the CPU.
    EHP_HD inline float fast_rcp(float x)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        return __builtin_amdgcn_rcpf(x);
#else
        return 1.0f / x;
#endif
    }

    EHP_HD inline float fast_rsq(float x)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        return __builtin_amdgcn_rsqf(x);
#else
        return 1.0f / sqrtf(x);
#endif
    }

    // The FP32 kernels' footprint (tiled forward, gather back projection): footprint()'s
    // projection with the hardware's reciprocal and reciprocal square root in place of three
    // correctly rounded divisions and a square root (about 45 VALU instructions fewer per
    // footprint). The homogeneous division is the quotient q = p rcp(w) with one correction,
    // q + (p - q w) rcp(w) (two FMAs): within about half an ulp of p / w, as the centre, a
    // coordinate of hundreds of pixels from which the taps' pixel indices are subtracted, needs.
    // The scaling sdd / |ext x| = sdd rsq(|ext x|^2) (source_dist2) and rs = 1 / scaling come within an ulp or
    // two (relative errors of 1e-7 in the tap distances). Forward and back projection share it, so
    // they stay each other's adjoint.
    template <int D>
    EHP_HD inline void footprint_fast(const PoseGeom& g, const Dims& dims, int x, int y, int z, float radius,
                                      Footprint& fp, float& rs)
    {
        float pc[3], unused[3];
        voxel_project<D>(g, x, y, z, pc, unused);
        const float w = pc[D - 1];
        const float rw = fast_rcp(w);
#pragma unroll
        for (int i = 0; i < D - 1; ++i) {
            const float q = pc[i] * rw;
            fp.center[i] = __builtin_fmaf(__builtin_fmaf(-q, w, pc[i]), rw, q) - 0.5f;
        }
        fp.scaling = g.sdd * fast_rsq(source_dist2<D>(g, x, y, z));
        rs = fast_rcp(fp.scaling);
        footprint_rect<D>(dims, radius, fp);
    }

    // fn(pixel, |d|, d_u) for every pixel of the footprint, d = (centre - pixel) / scaling
    template <int D, class T, class Fn>
    EHP_HD inline void visit(const Footprint& fp, const Dims& dims, Fn fn)
    {
        for (int j = fp.lo[1]; j <= fp.hi[1]; ++j)
            for (int i = fp.lo[0]; i <= fp.hi[0]; ++i) {
                const float d0 = (fp.center[0] - (float) i) / fp.scaling;
                float dist;
                if (D == 2) {
                    dist = sqrtf(d0 * d0);
                } else {
                    const float d1 = (fp.center[1] - (float) j) / fp.scaling;
                    dist = sqrtf(d0 * d0 + d1 * d1);
                }
                fn((int64_t) j * dims.det[0] + i, dist, d0);
            }
    }

    // Weight of one footprint tap: the table at |d| (VoxelComputation.h:20-24), or for the
    // phase-contrast projectors (diff) times sgn(d_u) in 2D and d_u in 3D (VoxelComputation.h:
    // 26-38, ProjectVoxelsCUDA.cu:73-76, :160-165).
    template <int D, class T>
    EHP_HD inline T tap_weight(const T* __restrict__ lut, int n, float support, float dist, float d0, bool diff)
    {
        const T w = lut_eval<T>(lut, n, support, dist);
        if (!diff)
            return w;
        if (D == 2)
            return d0 > 0.0f ? w : (d0 < 0.0f ? -w : T(0));
        return w * (T) d0;
    }

    // Square root for the FP32 taps: the hardware's v_sqrt_f32 (within 1 ulp; the correctly
    // rounded sqrtf adds a dozen instructions per tap on this part); sqrtf on the CPU.
    EHP_HD inline float tap_sqrt(float x)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        return __builtin_amdgcn_sqrtf(x);
#else
        return sqrtf(x);
#endif
    }

    // The FP32 kernels' table (tiled forward, gather back projection): entry i < lerp_table_size(n)
    // of a table of n values as the pair (lut[i], lut[i + 1] - lut[i]) in tab[2 i], tab[2 i + 1],
    // with lut[i] = 0 for i >= n, so that one aligned 8-byte read gives an interpolation's two
    // operands.
    EHP_HD inline void lerp_table_entry(const float* __restrict__ lut, int n, int i, float* __restrict__ tab)
    {
        const float cur = i < n ? lut[i] : 0.0f;
        const float next = i + 1 < n ? lut[i + 1] : 0.0f;
        tab[2 * i] = cur;
        tab[2 * i + 1] = next - cur;
    }

    // The FP32 kernels' tap weight from the squared distance d2 = |d|^2 (d0 * d0 + d1 * d1 with one
    // rounding): the table index as |d| * k, k = (n - 1) / support (one multiplication instead of
    // a division per tap), and with a = floor(index), t = index - a the interpolation
    // lut[a] + t * (lut[a + 1] - lut[a]) in one FMA over the pair table (lerp_table_entry; lut_eval
    // forms t * lut[b] + (1 - t) * lut[a], b = ceil(index): the same up to FP32 rounding, and
    // exactly lut[a] at an integer index), 0 outside [0, n - 1]. Branch-free. TZ: the table's last
    // entry is 0 (blob and B-spline tables vanish at the support), so that past n - 1 the zero
    // pairs of the padded table give 0 by themselves and the clamp and range test drop out.
    template <int D, bool TZ = false>
    EHP_HD inline float tap_weight_fast(const float* __restrict__ tab, int n, float k, float d2, float d0, bool diff)
    {
        // index >= 0, and below sqrt(2) (n - 1) for a tap of the footprint rectangle (|d0|, |d1| at
        // most the radius in table units), so its integer part fits an int. In 2D |d| is |d0|,
        // which the correctly rounded sqrt(d0 * d0) equals (d0 * d0 normal).
        const float index = (D == 2 ? fabsf(d0) : tap_sqrt(d2)) * k;
        const float last = (float) (n - 1);
        const int ia = (int) index;
        const int a = TZ ? ia : (ia < n - 1 ? ia : n - 1); // floor(index) where index <= n - 1
        const float t = fract_pos(index);                  // index - a there (exact)
        float w = __builtin_fmaf(t, tab[2 * a + 1], tab[2 * a]);
        if (!TZ)
            w = index <= last ? w : 0.0f;
        if (!diff)
            return w;
        if (D == 2)
            return d0 > 0.0f ? w : (d0 < 0.0f ? -w : 0.0f);
        return w * d0;
    }

    // ---------------------------------------------------------------------------------
    // The 3D kernels' footprints by columns: a footprint is at most `cols` pixels wide (a property of
    // the operator), so a voxel's column distances are formed once and every row of taps is straight
    // code over them, with no loop over columns.

    // Most columns of the 3D kernels' footprints; wider ones take the general kernels.
    constexpr int kVoxMaxCols = 8;

    // Pixels across the widest footprint: floor(2 r s) + 1 for the radius r and the largest scaling s,
    // with room for the rounding of its ends.
    inline int footprint_cols(double support, double smax)
    {
        const double w = 2.0 * support * smax * (1.0 + 1.0e-5) + 1.0e-4;
        return w < 1.0e6 ? (int) w + 1 : 1 << 20;
    }

    // Detector tile of the general 3D forward
    constexpr TileCfg kVoxGeneralTile{32, 32, 1};

    // The kernels' column counts: the next of 4, 5, 6 and 8
    inline int kernel_cols(int cols)
    {
        return cols <= 4 ? 4 : (cols <= 6 ? cols : 8);
    }

    // Entries of the pair table (lerp_table_entry) that taps reach when columns past the footprint's end
    // are not masked: the first of nc columns lies at least r s - 1 before the centre, so the last less
    // than nc - r s past it: (nc / (r s) - 1) (n - 1) in table units, and at least n - 1; rows at most n - 1.
    inline double column_table_span(int n, double support, double smin, int nc)
    {
        const double far = nc / (support * smin) - 1.0, e = far > 1.0 ? far : 1.0;
        return sqrt(e * e + 1.0) * 1.0001 * (n - 1) + 4.0;
    }

    // What fixes an operator's columns: its footprints' (0: none), its table and its least scaling
    struct ColumnNeeds {
        int cols, n_lut;
        double support, smin;
    };

    // Entries of the pair table in the reach of a kernel of nc columns (as a number that may be too large)
    inline double column_table_span(const ColumnNeeds& c, int nc)
    {
        return column_table_span(c.n_lut, c.support, c.smin, nc);
    }

    // Columns of the kernel that takes all of n operators: the widest one's (the further columns of the others
    // add nothing where their tables reach as far), 0 if one has none or its table would not fit.
    inline int common_cols(const ColumnNeeds* ops, int n)
    {
        int nc = 0;
        for (int j = 0; j < n; ++j)
            nc = kernel_cols(ops[j].cols) > nc ? kernel_cols(ops[j].cols) : nc;
        for (int j = 0; j < n; ++j)
            if (ops[j].cols <= 0 || !(column_table_span(ops[j], nc) <= kVoxLutSpan))
                return 0;
        return nc;
    }

    // Parts that a voxel's poses are summed in by the gather, added in order (a property of the operator: its launches
    // alone and in a batch give the same sums): as many (a power of two, at most 16, at least four poses each) as
    // bring a launch with a wavefront for each part to six wavefronts a SIMD of a device of 1024.
    inline int gather_part_count(const Dims& dims)
    {
        int parts = 1;
        while (parts < 16 && dims.nvox * parts < (int64_t) 6144 * 64 && dims.nposes >= 8 * parts)
            parts *= 2;
        return parts;
    }

    // Wavefronts that share a voxel's parts: all of them apart, which one sum a voxel would leave most of the
    // device idle for on small volumes: 92 x 80 blobs, 70 poses 48.3 -> 11.9 us, 300 x 380 / 524 poses 319 -> 147,
    // 36 x 33 x 40 / 40 poses 125 -> 25. In 3D wide footprints (`width` pixels at most) fill the caches: further
    // wavefronts, at other poses, displace the detector rows that a wavefront comes back to. Up to four a SIMD past eight
    // pixels, 2.4 past sixteen, 1.5 past 24. (FP64's divisions weigh more than its loads: blobs 64^3 / 60 poses, width 13
    // 2782 us with one, 2493 with two wavefronts.) Blobs in FP32, us, with 1 / 2 / 4 / 8 wavefronts over 360 degrees (and,
    // as neighbouring poses share rows, 45; columns beside the parts empty):
    //              width 16                              width 23                              width 31
    //   64^3 / 60   964 1121 (1551 1722)                 2437 3634 (3886 4231)                 5487 8081 (9121 9016)
    //   56^3 / 40   525  483  598 (707 570 514)          1243 1561 1979 (1729 1458 1576)       2393 3862 4406 (3186 3581 3663)
    //   48^3 / 60   635  474  500 (1031 647 485)         1467 1169 1636 (2318 1546 1418)       2759 2992 3911 (4180 2859 3437)
    //   40^3 / 40   424  228  208  185 (621 366 241 213)  909  495  472  577 (1400 817 552 503) 1580  917 1165 1289
    inline int gather_waves(const Dims& dims, int width, bool f64)
    {
        const int64_t simd = 1024 * 64; // a wavefront each
        const int parts = gather_part_count(dims);
        if (f64 || dims.dim == 2 || width <= kVoxMaxCols)
            return parts;
        int waves = 1;
        while (waves < parts && 10 * dims.nvox * waves < (width <= 16 ? 40 : (width <= 24 ? 24 : 15)) * simd)
            waves *= 2;
        return waves;
    }

    // a / b, correctly rounded, from rb = 1 / b correctly rounded: the quotient estimate with one
    // correction (Markstein, Computation of elementary functions on the IBM RISC System/6000, 1990,
    // theorem on division); b's mantissa is not all ones, quotients far from underflow.
    EHP_HD inline float div_rounded(float a, float b, float rb)
    {
        const float q = a * rb;
        return __builtin_fmaf(__builtin_fmaf(-b, q, a), rb, q);
    }

    // The FP64 weight at table position index (tap_weight's interpolation t fb + (1 - t) fa), 0 past
    // n - 1; tab holds n entries and a zero.
    EHP_HD inline double lut_weight64(const double* __restrict__ tab, int n, float index)
    {
        const int ia = (int) index; // index >= 0
        const int a = ia < n - 1 ? ia : n - 1;
        const double t = (double) (index - (float) a);
        const double w = t * tab[a + 1] + (1.0 - t) * tab[a];
        return index <= (float) (n - 1) ? w : 0.0;
    }

    // The weight of an FP32 tap as every FP32 kernel forms it, from the distances in table units: d0k =
    // (c0 - i) rsk and d1s = ((c1 - j) rsk)^2 (2D: 0) with rsk = (n - 1) / (support scaling), so that
    // the square root is the table index; du = d0 in footprint radii (diff in 3D only).
    template <int D, bool TZ>
    EHP_HD inline float tap_weight_units(const float* __restrict__ tab, int n, float d0k, float d1s, float du,
                                         bool diff)
    {
        if (D == 2)
            return tap_weight_fast<2, TZ>(tab, n, 1.0f, 0.0f, d0k, diff);
        const float w = tap_weight_fast<3, TZ>(tab, n, 1.0f, __builtin_fmaf(d0k, d0k, d1s), 0.0f, false);
        return diff ? w * du : w;
    }

    // Columns l0 .. l0 + NC - 1 of an FP32 footprint of columns l0 .. h0: the distances in table units and,
    // for the phase-contrast weights, in footprint radii. A table that ends in 0 (TZ) gives the columns
    // past h0 weight 0 by itself (column_table_span); others put them past its end.
    template <int NC, bool TZ>
    EHP_HD inline void column_units(float c0, int l0, int h0, float rs, float rsk, bool diff, float* d0k, float* du)
    {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const float d = c0 - (float) (l0 + i);
            d0k[i] = d * rsk;
            if (!TZ)
                d0k[i] = l0 + i <= h0 ? d0k[i] : 1.0e6f;
            du[i] = diff ? d * rs : 1.0f;
        }
    }

    // The same for NC columns from lo, of which those past the last lie just past the end of the table
    // (index at least n - 1 + 1/16, below lerp_table_size(n) on every row), so that every table gives them 0.
    template <int NC>
    EHP_HD inline void column_units_clipped(float c0, int lo, int last, int n, float rs, float rsk, bool diff,
                                            float* d0k, float* du)
    {
        const float past = (float) (n - 1) + 0.0625f;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const float d = c0 - (float) (lo + i);
            d0k[i] = i <= last ? d * rsk : past;
            du[i] = diff ? d * rs : 1.0f;
        }
    }

    // The weights of row j over those columns
    template <int NC, bool TZ>
    EHP_HD inline void row_units(const float* __restrict__ tab, int n, float c1, int j, float rsk, const float* d0k,
                                 const float* du, bool diff, float* w)
    {
        const float d1 = (c1 - (float) j) * rsk;
        const float d1s = d1 * d1;
#pragma unroll
        for (int i = 0; i < NC; ++i)
            w[i] = tap_weight_units<3, TZ>(tab, n, d0k[i], d1s, du[i], diff);
    }

    // The same for FP64 tables: the distances and weights of visit() and tap_weight bit for bit, their
    // divisions from correctly rounded reciprocals (rsc = 1 / scaling, rsupport = 1 / support).
    template <int NC>
    EHP_HD inline void column_units64(float c0, int l0, int h0, float scaling, float rsc, float* d0)
    {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            d0[i] = div_rounded(c0 - (float) (l0 + i), scaling, rsc);
            d0[i] = l0 + i <= h0 ? d0[i] : 1.0e6f;
        }
    }

    template <int NC>
    EHP_HD inline void row_units64(const double* __restrict__ tab, int n, float support, float rsupport, float c1,
                                   int j, float scaling, float rsc, const float* d0, bool diff, double* w)
    {
        const float d1 = div_rounded(c1 - (float) j, scaling, rsc);
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const float dist = sqrtf(d0[i] * d0[i] + d1 * d1);
            w[i] = lut_weight64(tab, n, div_rounded(dist, support, rsupport) * (float) (n - 1));
            if (diff)
                w[i] = w[i] * (double) d0[i];
        }
    }

    // Row stride (slots) of a detector tile's LDS sums in the tiled voxel forward: odd in 3D, so
    // that the 8-byte slots of neighbouring detector rows fall on different LDS banks.
    EHP_HD inline int vox_acc_stride(int TU, int TV)
    {
        return TV > 1 ? (TU | 1) : TU;
    }

    // What one detector pixel of the tiled voxel forward can receive, in units of max|x|: at most
    // (2 r s + 2)^(dim-1) voxels per plane (s the largest footprint scaling), each with a
    // weight of at most ls (a power of two at least the largest |weight|), over the longest
    // axis of planes; at least 4096 ls, so that one term x * w stays below 2^51 units (the range
    // of fixed_round).
    inline double voxel_slot_bound(const Dims& dims, double support, double smax, double ls)
    {
        int maxdim = 0;
        for (int i = 0; i < dims.dim; ++i)
            maxdim = dims.vol[i] > maxdim ? dims.vol[i] : maxdim;
        const double per_plane = 2.0 * support * smax + 2.0;
        const double b = (double) maxdim * (dims.dim == 3 ? per_plane * per_plane : per_plane) * ls;
        return b > 4096.0 * ls ? b : 4096.0 * ls;
    }

    // Least (sign -1) or largest (+1) stretch of the extrinsic matrix' linear part: |ext x| lies between
    // these times the distance, in voxels, from the source to the voxel centre x. Bounds of its singular
    // values from M^T M (Gershgorin): the voxel spacings for a rotation of them, 1 for unit spacing.
    inline double ext_stretch(const PoseGeom& g, const Dims& dims, int sign)
    {
        double best = 0.0;
        for (int i = 0; i < dims.dim; ++i) {
            double diag = 0.0, off = 0.0;
            for (int j = 0; j < dims.dim; ++j) {
                double dot = 0.0;
                for (int k = 0; k < dims.dim; ++k)
                    dot += (double) g.ext[k + i * dims.dim] * g.ext[k + j * dims.dim];
                if (i == j)
                    diag = dot;
                else
                    off += fabs(dot);
            }
            const double b = diag + sign * off;
            best = i == 0 || sign * b > sign * best ? b : best;
        }
        if (fabs(best - 1.0) < 1.0e-5) // the rounding of a rotation
            return 1.0;
        return best > 0.0 ? sqrt(best) : 0.0;
    }

    // Largest footprint scaling of a pose over the volume, sdd / |ext x|: from the smallest distance from the
    // source to the volume box (the source inside, or ext singular: -1).
    inline double voxel_max_scaling(const PoseGeom& g, const Dims& dims)
    {
        double dist2 = 0.0;
        for (int i = 0; i < dims.dim; ++i) {
            const double c = g.C[i];
            const double e = c < 0.0 ? -c : (c > dims.vol[i] ? c - dims.vol[i] : 0.0);
            dist2 += e * e;
        }
        const double least = ext_stretch(g, dims, -1) * sqrt(dist2);
        return least > 0.0 ? (double) g.sdd / least : -1.0;
    }

    // Smallest footprint scaling of a pose over the volume, from the largest distance from the source to a
    // corner of the volume.
    inline double voxel_min_scaling(const PoseGeom& g, const Dims& dims)
    {
        double dist2 = 0.0;
        for (int i = 0; i < dims.dim; ++i) {
            const double c = g.C[i], far = c < 0.5 * dims.vol[i] ? dims.vol[i] - c : c;
            dist2 += far * far;
        }
        const double most = ext_stretch(g, dims, 1) * sqrt(dist2);
        return most > 0.0 ? (double) g.sdd / most : -1.0;
    }

    // Driving axis of a pose for the tiled forward: the largest component of the central ray.
    template <int D>
    EHP_HD inline int pose_axis(const PoseGeom& g, const Dims& dims)
    {
        float o[3], d[3];
        make_ray<D>(g, dims.det[0] / 2, D == 3 ? dims.det[1] / 2 : 0, o, d);
        int a = 0;
        float m = fabsf(d[0]);
        for (int i = 1; i < D; ++i)
            if (fabsf(d[i]) > m) {
                m = fabsf(d[i]);
                a = i;
            }
        return a;
    }

    // Voxels of plane `pa` (along axis A) whose footprint can reach the detector rectangle
    // [u0, u1] x [v0, v1]: the footprint centre c = (P x)_hom - 0.5 of such a voxel lies within
    // margin m of the rectangle, i.e. P x lies in [u0 + 0.5 - m, u1 + 0.5 + m] x ..., the
    // frustum through the source spanned by the rays of those four corners. Its cross-section
    // with the plane of voxel centres pa + 0.5 is the quadrilateral of the corner rays' hits;
    // the voxel ranges cover its bounding rectangle with one voxel to spare. Returns false
    // when no voxel qualifies; falls back to the whole plane when a corner ray does not reach
    // the plane in front of the source.
    template <int D>
    EHP_HD inline bool frustum_plane_range(const PoseGeom& g, const Dims& dims, int A, int pa, const float* cdir,
                                           int ncorners, int& blo, int& bhi, int& clo, int& chi)
    {
        const int b1 = (D == 2) ? 1 - A : (A == 0 ? 1 : 0);
        const int b2 = (D == 2) ? -1 : (A == 2 ? 1 : 2);
        const float X = (float) pa + 0.5f;
        const float CA = pick<D>(g.C, A);
        float bmin = 3.0e38f, bmax = -3.0e38f, cmin = 3.0e38f, cmax = -3.0e38f;
        bool ok = true;
        for (int k = 0; k < ncorners; ++k) {
            const float* dk = cdir + 3 * k;
            const float da = pick<D>(dk, A);
            const float t = (X - CA) / da;
            ok = ok && (da != 0.0f) && (t > 0.0f) && (t < 3.0e38f);
            const float pb = pick<D>(g.C, b1) + t * pick<D>(dk, b1);
            bmin = pb < bmin ? pb : bmin;
            bmax = pb > bmax ? pb : bmax;
            if (D == 3) {
                const float pc = pick<D>(g.C, b2) + t * pick<D>(dk, b2);
                cmin = pc < cmin ? pc : cmin;
                cmax = pc > cmax ? pc : cmax;
            }
        }
        const int nb = dims.vol[b1], nc = D == 3 ? dims.vol[b2] : 1;
        if (!ok) {
            blo = 0;
            bhi = nb - 1;
            clo = 0;
            chi = nc - 1;
            return true;
        }
        // voxel centres b + 0.5 in [bmin, bmax], one voxel to spare
        bmin = bmin < -2.0f ? -2.0f : (bmin > (float) nb + 2.0f ? (float) nb + 2.0f : bmin);
        bmax = bmax < -2.0f ? -2.0f : (bmax > (float) nb + 2.0f ? (float) nb + 2.0f : bmax);
        blo = (int) floorf(bmin - 0.5f) - 1;
        bhi = (int) ceilf(bmax - 0.5f) + 1;
        blo = blo < 0 ? 0 : blo;
        bhi = bhi > nb - 1 ? nb - 1 : bhi;
        if (D == 3) {
            cmin = cmin < -2.0f ? -2.0f : (cmin > (float) nc + 2.0f ? (float) nc + 2.0f : cmin);
            cmax = cmax < -2.0f ? -2.0f : (cmax > (float) nc + 2.0f ? (float) nc + 2.0f : cmax);
            clo = (int) floorf(cmin - 0.5f) - 1;
            chi = (int) ceilf(cmax - 0.5f) + 1;
            clo = clo < 0 ? 0 : clo;
            chi = chi > nc - 1 ? nc - 1 : chi;
        } else {
            clo = chi = 0;
        }
        return blo <= bhi && clo <= chi;
    }

    // Directions of the corner rays of the detector rectangle [u0, u1] x [v0, v1] widened by
    // margin m (unnormalised: Pinv applied to the homogeneous detector point).
    template <int D>
    EHP_HD inline int frustum_corners(const PoseGeom& g, int u0, int u1, int v0, int v1, float m, float* cdir)
    {
        const float us[2] = {(float) u0 + 0.5f - m, (float) u1 + 0.5f + m};
        const float vs[2] = {(float) v0 + 0.5f - m, (float) v1 + 0.5f + m};
        int n = 0;
        for (int jv = 0; jv < (D == 3 ? 2 : 1); ++jv)
            for (int ju = 0; ju < 2; ++ju) {
                const float h[3] = {us[ju], D == 3 ? vs[jv] : 1.0f, 1.0f};
                for (int i = 0; i < 3; ++i)
                    cdir[3 * n + i] = 0.0f;
                for (int i = 0; i < D; ++i) {
                    float acc = 0.0f;
                    for (int j = 0; j < D; ++j)
                        acc += g.Pinv[i + j * (D + 1)] * h[j];
                    cdir[3 * n + i] = acc;
                }
                ++n;
            }
        return n;
    }
} // namespace ehp
