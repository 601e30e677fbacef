// ehp_voxel_tiled.hip -- voxel-driven forward projection with LDS-privatised detector tiles
// (FP32 arithmetic with the volume and sinogram stored in FP32 or bfloat16; FP64).
//
// The forward of elsa's voxel projectors (VoxelComputation.h:110-152: every voxel adds
// x * basis(distance) to the detector pixels of its footprint) without global atomics. One
// workgroup owns one detector tile of one pose and accumulates it in LDS: it walks the planes
// of the volume along the pose's driving axis, takes on each plane the voxels whose footprint
// can reach the tile (frustum_plane_range), computes each one's footprint exactly as the
// one-thread-per-voxel kernels do and adds the taps that fall in the tile. Every pixel then
// belongs to one tile and is written once, so the output needs no clearing. Tiles are ordered
// tile first, pose second: the poses of a tile, which read nearly the same column of the
// volume, run together on one XCD.
//
// Sums are 64-bit fixed point as in the tiled back projections: one exponent per call from
// max|x| and a bound on what one pixel can receive, each tap's x * weight rounded once to the
// unit (fixed_round; exact product in FP64 for FP32 data). With bfloat16 storage the voxels
// are widened exactly and each pixel's sum is rounded to bfloat16 once, so the result is the
// FP32 operator's on the same (bfloat16) volume, rounded once. FP64 operators take an FP64
// table and form each weight as the one-thread-per-voxel FP64 kernel does (tap_weight, the
// divisions of VoxelComputation.h), so their terms are that kernel's.
#include "ehp_kernels.hpp"

#include <type_traits>

namespace ehp
{
    namespace
    {
        constexpr int kThreads = 256;
        constexpr int kMaxLut = kVoxMaxLut;
        // LDS (address space 3) pointers: 32-bit byte addresses
        typedef __attribute__((address_space(3))) unsigned long long lds_u64;
        typedef __attribute__((address_space(3))) char lds_char;

        // The frustum rectangle of one plane: first voxel along b1 and b2, width along b1 and its
        // reciprocal (rect_split), and the linear index of its first voxel (volumes below 2^31
        // voxels with strides below 2^24, whose indices are formed with 24-bit multiplications)
        struct PlaneRect {
            int blo, clo, nb;
            float rnb;
            uint32_t base;
        };
        // LDS of the plane tables of a chunk of kThreads planes: rectangles, counts and their prefix
        constexpr size_t kPlaneLds = kThreads * (sizeof(PlaneRect) + sizeof(int)) + (kThreads + 1) * sizeof(int);
    } // namespace

    // Tile-pose id (tile * nposes + pose) of one operator's forward, whose pose has driving axis
    // A; LT = float (FP32 and bfloat16 storage) or double (FP64) is the table's type.
    // The static LDS of the forward, declared once per kernel (each instantiation of a function
    // declaring its own would get its own copy): FP64 the table, FP32 its pair table
    // (lerp_table_entry, tap_weight_fast); the plane tables of a chunk.
    template <class LT>
    struct VoxFwdLds {
        LT* lut;
        PlaneRect* pr;
        int* cnt;
        int* pref;
    };

    template <int D, int A, class ST, class LT>
    __device__ __forceinline__ void vox_fwd_tiled_axis(const PoseGeom* __restrict__ geo, const Dims& dims,
                                                       const LT* __restrict__ lut, const int n_lut,
                                                       const float support, const int diff,
                                                       const float* __restrict__ pose_margin, const int TU,
                                                       const int TV, const int ntu, const int64_t id,
                                                       const int* __restrict__ fixexp,
                                                       const ST* __restrict__ vol, ST* __restrict__ sino,
                                                       const VoxFwdLds<LT>& L)
    {
        extern __shared__ long long lds[];
        LT* s_lut = L.lut;
        PlaneRect* s_pr = L.pr;
        int* s_cnt = L.cnt;
        int* s_pref = L.pref;
        const int tid = threadIdx.x;
        // id = tile * nposes + pose
        const int pose = (int) (id % dims.nposes);
        const int tile = (int) (id / dims.nposes);
        const int tu = tile % ntu, tv = tile / ntu;
        const int u0 = tu * TU, v0 = tv * TV;
        const int u1 = (u0 + TU < dims.det[0] ? u0 + TU : dims.det[0]) - 1;
        const int v1 = (v0 + TV < dims.det[1] ? v0 + TV : dims.det[1]) - 1;
        long long* acc = lds;
        const int RS = vox_acc_stride(TU, TV); // slot (v - v0, u - u0) at (v - v0) * RS + u - u0
        for (int i = tid; i < RS * TV; i += kThreads)
            acc[i] = 0;
        for (int i = tid; i < (sizeof(LT) == 8 ? n_lut : lerp_table_size(n_lut)); i += kThreads) {
            if constexpr (sizeof(LT) == 8)
                s_lut[i] = lut[i];
            else
                lerp_table_entry(lut, n_lut, i, s_lut);
        }
        const int eg = fixexp[0];
        const float lut_index_scale = (float) (n_lut - 1) / support;
        const bool lut_tail_zero = lut[n_lut - 1] == LT(0); // tap_weight_fast's TZ (FP32)
        const PoseGeom& g = geo[pose];
        float cdir[12];
        const int ncorner = frustum_corners<D>(g, u0, u1, v0, v1, pose_margin[pose], cdir);
        __syncthreads();

        constexpr int b1 = (D == 2) ? 1 - A : (A == 0 ? 1 : 0);
        constexpr int b2 = (D == 2) ? 2 : (A == 2 ? 1 : 2);
        const bool small = dims.nvox < (1ll << 31) && dims.strides[1] < (1 << 24) && dims.strides[2] < (1 << 24);
        const uint32_t sA = (uint32_t) dims.strides[A], s1 = (uint32_t) dims.strides[b1];
        const uint32_t s2 = D == 3 ? (uint32_t) dims.strides[b2] : 0u;
        // The planes in chunks of up to kThreads: one thread per plane computes the plane's frustum
        // rectangle (frustum_plane_range) into LDS, then every thread walks its candidates
        // k = tid, tid + kThreads, ... over all planes of the chunk in order, keeping its plane jp in
        // registers (candidate k is entry k - pref[jp] of plane jp's rectangle, jp the last plane with
        // pref[jp] <= k). A chunk holds fewer planes when its candidates could pass 2^31 - 1.
        const int64_t psz = (int64_t) dims.vol[b1] * (D == 3 ? dims.vol[b2] : 1);
        int pch = kThreads;
        while (pch > 1 && (int64_t) pch * psz > 0x7fffffffll)
            pch >>= 1;
        for (int pc0 = 0; eg != kNonFinite && pc0 < dims.vol[A]; pc0 += pch) {
            const int npl = dims.vol[A] - pc0 < pch ? dims.vol[A] - pc0 : pch;
            if (tid < npl) {
                int blo, bhi, clo, chi, cnt = 0;
                if (frustum_plane_range<D>(g, dims, A, pc0 + tid, cdir, ncorner, blo, bhi, clo, chi))
                    cnt = (bhi - blo + 1) * (chi - clo + 1);
                const int nb = cnt > 0 ? bhi - blo + 1 : 1;
                const uint32_t base = small && cnt > 0
                                          ? (uint32_t) (pc0 + tid) * sA + (uint32_t) blo * s1 + (uint32_t) clo * s2
                                          : 0u;
                s_pr[tid] = PlaneRect{blo, clo, nb, 1.0f / (float) nb, base};
                s_cnt[tid] = cnt;
            }
            __syncthreads();
            if (tid == 0) {
                s_pref[0] = 0;
                for (int q = 0; q < npl; ++q)
                    s_pref[q + 1] = s_pref[q] + s_cnt[q];
            }
            __syncthreads();
            const int total = s_pref[npl];
            int jp = 0, pj = 0, pn = s_pref[1];
            PlaneRect pr = s_pr[0];
            // candidate k's voxel c and its linear index (k increasing from call to call)
            auto locate = [&](int k, int* c) -> int64_t {
                while (k >= pn) {
                    ++jp;
                    pj = pn;
                    pn = s_pref[jp + 1];
                    pr = s_pr[jp];
                }
                int row, col;
                rect_split(k - pj, pr.nb, pr.rnb, row, col);
                c[A] = pc0 + jp;
                c[b1] = pr.blo + col;
                if (D == 3)
                    c[b2] = pr.clo + row;
                return small ? (int64_t) (pr.base + mul24((uint32_t) col, s1) + mul24((uint32_t) row, s2))
                             : c[0] + c[1] * dims.strides[1] + (int64_t) c[2] * dims.strides[2];
            };
            using XT = decltype(up(vol[0]));
            // the taps of voxel c with value xv
            auto visit = [&](const int* c, const XT xv) {
                if (xv == 0)
                    return;
                // FP64: footprint()'s divisions, as the one-thread-per-voxel FP64 kernel; FP32:
                // footprint_fast, as the gather back projection
                Footprint fp;
                float rs = 0.0f;
                if constexpr (sizeof(LT) == 8)
                    footprint<D>(g, dims, c[0], c[1], c[2], support, fp);
                else
                    footprint_fast<D>(g, dims, c[0], c[1], c[2], support, fp, rs);
                const int lo0 = fp.lo[0] > u0 ? fp.lo[0] : u0, hi0 = fp.hi[0] < u1 ? fp.hi[0] : u1;
                const int lo1 = fp.lo[1] > v0 ? fp.lo[1] : v0, hi1 = fp.hi[1] < v1 ? fp.hi[1] : v1;
                if (lo0 > hi0 || lo1 > hi1)
                    return;
                // x in units of q (a power-of-two scaling, exact); each tap adds x * w rounded once
                // (|x w| < 2^51 units: the pixel bound is at least 4096 times the table's bound)
                const double xq = ldexp((double) xv, 62 - eg);
                if constexpr (sizeof(LT) == 8) {
                    // FP64: the weights of visit() and tap_weight, as the one-thread-per-voxel kernel
                    for (int j = lo1; j <= hi1; ++j) {
                        const float d1 = D == 3 ? (fp.center[1] - (float) j) / fp.scaling : 0.0f;
                        for (int i = lo0; i <= hi0; ++i) {
                            const float d0 = (fp.center[0] - (float) i) / fp.scaling;
                            const float dist = D == 2 ? sqrtf(d0 * d0) : sqrtf(d0 * d0 + d1 * d1);
                            const double w = tap_weight<D, double>(s_lut, n_lut, support, dist, d0, diff != 0);
                            if (w != 0.0)
                                atomicAdd(reinterpret_cast<unsigned long long*>(acc + (j - v0) * RS + (i - u0)),
                                          fixed_round(xq, w));
                        }
                    }
                } else {
                    // the distance as visit() forms it, with the reciprocal rs of the scaling per
                    // voxel instead of a division per tap (and tap_weight_fast's square root and
                    // table index): within a few ulp of the one-thread-per-voxel kernels' weights,
                    // and the gather back projection's weights bit for bit. Two columns per step, so
                    // that their table reads are in flight together (the second is skipped past hi0).
                    // A table ending in 0 takes tap_weight_fast's TZ form.
                    const float rsk = rs * lut_index_scale;
                    auto taps = [&](auto tzc) {
                        constexpr bool TZ = decltype(tzc)::value;
                        for (int j = lo1; j <= hi1; ++j) {
                            const float d1 = D == 3 ? (fp.center[1] - (float) j) * rsk : 0.0f;
                            const float d1s = d1 * d1;
                            unsigned long long* row = reinterpret_cast<unsigned long long*>(acc + (j - v0) * RS);
                            float fi = (float) lo0; // i as a float (exact), without a conversion per tap
                            for (int i = lo0; i <= hi0; i += 2, fi += 2.0f) {
                                const float da = fp.center[0] - fi, db = fp.center[0] - (fi + 1.0f);
                                const float wa =
                                    tap_weight_units<D, TZ>(s_lut, n_lut, da * rsk, d1s, da * rs, diff != 0);
                                const float wb =
                                    tap_weight_units<D, TZ>(s_lut, n_lut, db * rsk, d1s, db * rs, diff != 0);
                                if (wa != 0.0f)
                                    atomicAdd(row + (i - u0), fixed_round(xq, (double) wa));
                                if (i < hi0 && wb != 0.0f)
                                    atomicAdd(row + (i + 1 - u0), fixed_round(xq, (double) wb));
                            }
                        }
                    };
                    if (lut_tail_zero)
                        taps(std::true_type{});
                    else
                        taps(std::false_type{});
                }
            };
            // each lane loads its next candidate's value before it visits the current one, so that
            // the load's latency is spent on that visit
            int cur[3] = {0, 0, 0};
            XT xcur = 0;
            if (tid < total)
                xcur = up(vol[locate(tid, cur)]);
            for (int k = tid; k < total; k += kThreads) {
                int nxt[3] = {0, 0, 0};
                XT xnxt = 0;
                if (k + kThreads < total)
                    xnxt = up(vol[locate(k + kThreads, nxt)]);
                visit(cur, xcur);
                cur[0] = nxt[0];
                cur[1] = nxt[1];
                cur[2] = nxt[2];
                xcur = xnxt;
            }
            __syncthreads(); // the next chunk rewrites the plane tables
        }
        const double q = eg == kNonFinite ? __longlong_as_double(0x7ff8000000000000ll) : ldexp(1.0, eg - 62);
        ST* sp = sino + (int64_t) pose * dims.pix_per_pose;
        for (int i = tid; i < TU * TV; i += kThreads) {
            const int u = u0 + i % TU, v = v0 + i / TU;
            if (u <= u1 && v <= v1)
                sp[(int64_t) v * dims.det[0] + u] =
                    down<ST>((typename Acc<ST>::type) ((double) acc[(v - v0) * RS + (u - u0)] * q));
        }
    }

    // Tile-pose id of one operator's forward: the pose's driving axis as a template parameter
    template <int D, class ST, class LT = float>
    __device__ __forceinline__ void vox_fwd_tiled_block(const PoseGeom* __restrict__ geo, const Dims& dims,
                                                        const LT* __restrict__ lut, const int n_lut,
                                                        const float support, const int diff,
                                                        const int* __restrict__ pose_axis,
                                                        const float* __restrict__ pose_margin, const int TU,
                                                        const int TV, const int ntu, const int64_t id,
                                                        const int* __restrict__ fixexp,
                                                        const ST* __restrict__ vol, ST* __restrict__ sino)
    {
        __shared__ LT s_lut[sizeof(LT) == 8 ? kMaxLut : 2 * kVoxLutSpan];
        __shared__ PlaneRect s_pr[kThreads];
        __shared__ int s_cnt[kThreads];
        __shared__ int s_pref[kThreads + 1];
        const VoxFwdLds<LT> L{s_lut, s_pr, s_cnt, s_pref};
        const int A = pose_axis[(int) (id % dims.nposes)];
        if (A == 0)
            vox_fwd_tiled_axis<D, 0, ST, LT>(geo, dims, lut, n_lut, support, diff, pose_margin, TU, TV, ntu, id,
                                             fixexp, vol, sino, L);
        else if (D == 2 || A == 1)
            vox_fwd_tiled_axis<D, 1, ST, LT>(geo, dims, lut, n_lut, support, diff, pose_margin, TU, TV, ntu, id,
                                             fixexp, vol, sino, L);
        else
            vox_fwd_tiled_axis<D, D == 3 ? 2 : 1, ST, LT>(geo, dims, lut, n_lut, support, diff, pose_margin, TU, TV,
                                                          ntu, id, fixexp, vol, sino, L);
    }

    // ---------------------------------------------------------------------------------
    // 3D forward by columns. As above, but a voxel's taps are rows of NC columns in straight code: the
    // tile's LDS sums have NC - 1 columns to spare on either side, so no column needs a test against
    // the tile or the detector, and the column distances are formed once per voxel. Where the table
    // ends in 0 (TZ) columns past the footprint's end weigh 0 by themselves (column_table_span); else they are
    // moved out of the table's reach. A wavefront's lanes run along the axis that fans out over detector
    // columns (VoxFan), as lanes whose voxels fall on one pixel add to one LDS word in turn.
    //
    // Bound by vector instructions and LDS together: a tap is 13 instructions (the square root counts as
    // four issues) and two LDS operations, a voxel another 140 (projection, scaling, rectangle). At
    // 131 x 125 x 119 blobs on 193 x 187, 180 poses: 2.69e9 wavefront instructions (0.78 a cycle and CU), the
    // LDS active 0.65 of the time; 5.48 ms against 11.42 ms for loops over the
    // clipped rectangle in 32 x 32 tiles, which ran 26 instructions a tap and left lanes idle in the
    // loops over columns. FP64 B-splines 96^3 on 144^2, 90 poses: 2.39 ms against 5.33 ms (correctly rounded
    // divisions from reciprocals that are formed once, div_rounded).

    // Row stride in slots
    __host__ __device__ inline int cols_stride(int TU, int NC)
    {
        return (TU + 2 * (NC - 1)) | 1;
    }

    // The volume as a launch reads it along driving axis A: element (ca, cf, cm) at ca sA + cf sf +
    // cm sm, f the axis that a wavefront's lanes run along.
    struct VoxFan {
        int f[3]; // per driving axis
    };

    template <int NC, class ST, class LT, int DIFF>
    __device__ __forceinline__ void vox_fwd_cols_block(const PoseGeom* __restrict__ geo, const Dims& dims,
                                                       const LT* __restrict__ lut, const int n_lut, const int span,
                                                       const float support, const int diff,
                                                       const int* __restrict__ pose_axis,
                                                       const float* __restrict__ pose_margin, const VoxFan& fan,
                                                       const int TU, const int TV, const int ntu, const int64_t id,
                                                       const int* __restrict__ fixexp, const ST* __restrict__ vol,
                                                       ST* __restrict__ sino)
    {
        constexpr bool F64 = sizeof(LT) == 8;
        extern __shared__ long long lds[];
        __shared__ PlaneRect s_pr[kThreads];
        __shared__ int s_cnt[kThreads];
        __shared__ int s_pref[kThreads + 1];
        const int tid = threadIdx.x;
        const int pose = (int) (id % dims.nposes);
        const int tile = (int) (id / dims.nposes);
        const int u0 = (tile % ntu) * TU, v0 = (tile / ntu) * TV;
        const int u1 = (u0 + TU < dims.det[0] ? u0 + TU : dims.det[0]) - 1;
        const int v1 = (v0 + TV < dims.det[1] ? v0 + TV : dims.det[1]) - 1;
        const int RS = cols_stride(TU, NC);
        long long* acc = lds;
        LT* s_lut = reinterpret_cast<LT*>(lds + RS * TV);
        for (int i = tid; i < RS * TV; i += kThreads)
            acc[i] = 0;
        for (int i = tid; i < span; i += kThreads) {
            if constexpr (F64)
                s_lut[i] = i < n_lut ? lut[i] : 0.0;
            else
                lerp_table_entry(lut, n_lut, i, s_lut);
        }
        const int eg = fixexp[0];
        const bool tail_zero = lut[n_lut - 1] == LT(0);
        const float kidx = (float) (n_lut - 1) / support;
        const float rsupport = 1.0f / support;
        const PoseGeom& g = geo[pose];
        float cdir[12];
        const int ncorner = frustum_corners<3>(g, u0, u1, v0, v1, pose_margin[pose], cdir);
        const int A = pose_axis[pose];
        const int b1 = A == 0 ? 1 : 0, b2 = A == 2 ? 1 : 2;
        const int f = A == 0 ? fan.f[0] : (A == 1 ? fan.f[1] : fan.f[2]);
        const bool fb2 = f == b2;
        const int m = fb2 ? b1 : b2;
        const uint32_t str[3] = {1u, (uint32_t) dims.strides[1], (uint32_t) dims.strides[2]};
        const uint32_t sA = A == 0 ? str[0] : (A == 1 ? str[1] : str[2]);
        const uint32_t sf = f == 0 ? str[0] : (f == 1 ? str[1] : str[2]);
        const uint32_t sm = m == 0 ? str[0] : (m == 1 ? str[1] : str[2]);
        const int nA = A == 0 ? dims.vol[0] : (A == 1 ? dims.vol[1] : dims.vol[2]);
        const uint32_t acc0 = (uint32_t) (uintptr_t) (lds_char*) acc;
        __syncthreads();

        const int64_t psz = (int64_t) dims.nvox / nA;
        int pch = kThreads;
        while (pch > 1 && (int64_t) pch * psz > 0x7fffffffll)
            pch >>= 1;
        for (int pc0 = 0; eg != kNonFinite && pc0 < nA; pc0 += pch) {
            const int npl = nA - pc0 < pch ? nA - pc0 : pch;
            if (tid < npl) {
                int blo, bhi, clo, chi, cnt = 0;
                if (frustum_plane_range<3>(g, dims, A, pc0 + tid, cdir, ncorner, blo, bhi, clo, chi))
                    cnt = (bhi - blo + 1) * (chi - clo + 1);
                const int flo = fb2 ? clo : blo, mlo = fb2 ? blo : clo;
                const int nf = cnt > 0 ? (fb2 ? chi - clo + 1 : bhi - blo + 1) : 1;
                const uint32_t base = cnt > 0 ? (uint32_t) (pc0 + tid) * sA + (uint32_t) flo * sf + (uint32_t) mlo * sm : 0u;
                s_pr[tid] = PlaneRect{flo, mlo, nf, 1.0f / (float) nf, base};
                s_cnt[tid] = cnt;
            }
            __syncthreads();
            if (tid == 0) {
                s_pref[0] = 0;
                for (int q = 0; q < npl; ++q)
                    s_pref[q + 1] = s_pref[q] + s_cnt[q];
            }
            __syncthreads();
            const int total = s_pref[npl];
            int jp = 0, pj = 0, pn = s_pref[1];
            PlaneRect pr = s_pr[0];
            // candidate k's voxel (x, y, z) and its index in the volume (k increasing from call to call)
            auto locate = [&](int k, int* c) -> uint32_t {
                while (k >= pn) {
                    ++jp;
                    pj = pn;
                    pn = s_pref[jp + 1];
                    pr = s_pr[jp];
                }
                int row, col;
                rect_split(k - pj, pr.nb, pr.rnb, row, col);
                const int ca = pc0 + jp, cf = pr.blo + col, cm = pr.clo + row;
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    c[i] = A == i ? ca : (f == i ? cf : cm);
                return pr.base + mul24((uint32_t) col, sf) + mul24((uint32_t) row, sm);
            };
            using XT = decltype(up(vol[0]));
            auto visit = [&](const int* c, const XT xv) {
                if (xv == 0)
                    return;
                Footprint fp;
                float rs = 0.0f;
                if constexpr (F64)
                    footprint<3>(g, dims, c[0], c[1], c[2], support, fp);
                else
                    footprint_fast<3>(g, dims, c[0], c[1], c[2], support, fp, rs);
                // the pixel rectangle as footprint_rect has it, the columns not clipped to the detector
                const float rod = fp.scaling * support;
                const int l0 = (int) ceilf(fp.center[0] - rod), h0 = (int) floorf(fp.center[0] + rod);
                int j0 = (int) ceilf(fp.center[1] - rod), j1 = (int) floorf(fp.center[1] + rod);
                j0 = j0 > v0 ? j0 : v0;
                j1 = j1 < v1 ? j1 : v1;
                if (l0 > u1 || h0 < u0 || l0 < u0 - (NC - 1) || j0 > j1)
                    return;
                // x in units of q (a power-of-two scaling, exact); each tap adds x * w rounded once
                // (|x w| < 2^51 units: the pixel bound is at least 4096 times the table's bound)
                const double xq = ldexp((double) xv, 62 - eg);
                lds_u64* at = (lds_u64*) (uintptr_t) (acc0 + 8u * (uint32_t) ((j0 - v0) * RS + (l0 - u0 + NC - 1)));
                // a row's weights are formed before any is added (the table reads and the atomics of a row
                // apart: 3 % of the kernel)
                auto add_row = [&](const auto* w) {
#pragma unroll
                    for (int i = 0; i < NC; ++i)
                        __hip_atomic_fetch_add(at + i, fixed_round(xq, (double) w[i]), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                    at += RS;
                };
                const bool df = DIFF == 1 || (DIFF == 2 && diff);
                if constexpr (F64) {
                    const float rsc = 1.0f / fp.scaling;
                    float d0[NC];
                    column_units64<NC>(fp.center[0], l0, h0, fp.scaling, rsc, d0);
                    for (int j = j0; j <= j1; ++j) {
                        double w[NC];
                        row_units64<NC>(s_lut, n_lut, support, rsupport, fp.center[1], j, fp.scaling, rsc, d0, df, w);
                        add_row(w);
                    }
                } else {
                    const float rsk = rs * kidx;
                    auto taps = [&](auto tzc) {
                        constexpr bool TZ = decltype(tzc)::value;
                        float d0k[NC], du[NC];
                        column_units<NC, TZ>(fp.center[0], l0, h0, rs, rsk, df, d0k, du);
                        for (int j = j0; j <= j1; ++j) {
                            float w[NC];
                            row_units<NC, TZ>(s_lut, n_lut, fp.center[1], j, rsk, d0k, du, df, w);
                            add_row(w);
                        }
                    };
                    if (tail_zero)
                        taps(std::true_type{});
                    else
                        taps(std::false_type{});
                }
            };
            // each lane loads its next candidate's value before it visits the current one
            int cur[3] = {0, 0, 0};
            XT xcur = 0;
            if (tid < total)
                xcur = up(vol[locate(tid, cur)]);
            for (int k = tid; k < total; k += kThreads) {
                int nxt[3] = {0, 0, 0};
                XT xnxt = 0;
                if (k + kThreads < total)
                    xnxt = up(vol[locate(k + kThreads, nxt)]);
                visit(cur, xcur);
                cur[0] = nxt[0];
                cur[1] = nxt[1];
                cur[2] = nxt[2];
                xcur = xnxt;
            }
            __syncthreads(); // the next chunk rewrites the plane tables
        }
        const double q = eg == kNonFinite ? __longlong_as_double(0x7ff8000000000000ll) : ldexp(1.0, eg - 62);
        ST* sp = sino + (int64_t) pose * dims.pix_per_pose;
        for (int i = tid; i < TU * TV; i += kThreads) {
            const int u = u0 + i % TU, v = v0 + i / TU;
            if (u <= u1 && v <= v1)
                sp[(int64_t) v * dims.det[0] + u] =
                    down<ST>((typename Acc<ST>::type) ((double) acc[(v - v0) * RS + (u - u0) + NC - 1] * q));
        }
    }

    template <int NC, class ST, class LT, int DIFF>
    __global__ void __launch_bounds__(kThreads)
        voxel_fwd_cols_kernel(const PoseGeom* __restrict__ geo, const Dims dims, const LT* __restrict__ lut,
                              const int n_lut, const int span, const float support, const int* __restrict__ pose_axis,
                              const float* __restrict__ pose_margin, const VoxFan fan, const int TU, const int TV,
                              const int ntu, const int per_xcd, const int64_t total, const int* __restrict__ fixexp,
                              const ST* __restrict__ vol, ST* __restrict__ sino)
    {
        const int64_t id = (int64_t) (blockIdx.x % 8u) * per_xcd + (blockIdx.x / 8u);
        if (id >= total)
            return;
        vox_fwd_cols_block<NC, ST, LT, DIFF>(geo, dims, lut, n_lut, span, support, DIFF, pose_axis, pose_margin, fan, TU,
                                             TV, ntu, id, fixexp, vol, sino);
    }

    // DIFF: the phase-contrast projectors' weights (a compile-time flag, so that the taps of the
    // others carry no select)
    template <int D, class ST, class LT, bool DIFF>
    __global__ void __launch_bounds__(kThreads)
        voxel_fwd_tiled_kernel(const PoseGeom* __restrict__ geo, const Dims dims, const LT* __restrict__ lut,
                               const int n_lut, const float support, const int* __restrict__ pose_axis,
                               const float* __restrict__ pose_margin, const int TU, const int TV, const int ntu,
                               const int per_xcd, const int64_t total, const int* __restrict__ fixexp,
                               const ST* __restrict__ vol, ST* __restrict__ sino)
    {
        const int64_t id = (int64_t) (blockIdx.x % 8u) * per_xcd + (blockIdx.x / 8u);
        if (id >= total)
            return;
        vox_fwd_tiled_block<D, ST, LT>(geo, dims, lut, n_lut, support, DIFF ? 1 : 0, pose_axis, pose_margin, TU, TV,
                                       ntu, id, fixexp, vol, sino);
    }

    // the forwards of many operators in one launch (block b: tile-pose b - job.block0 of job
    // block_job[b], as that operator's own launch would run it)
    template <int D>
    __global__ void __launch_bounds__(kThreads)
        voxel_fwd_tiled_batch_kernel(const VoxFwdJob* __restrict__ jobs, const int* __restrict__ block_job,
                                     const int per_xcd, const int64_t total, const int* __restrict__ fixexp,
                                     const float* __restrict__ vols, float* __restrict__ sinos)
    {
        const int64_t id = (int64_t) (blockIdx.x % 8u) * per_xcd + (blockIdx.x / 8u);
        if (id >= total)
            return;
        const VoxFwdJob& J = jobs[block_job[id]];
        vox_fwd_tiled_block<D, float>(J.geo, J.dims, J.lut, J.n_lut, J.support, J.diff, J.pose_axis, J.pose_margin,
                                      J.TU, J.TV, J.ntu, id - J.block0, fixexp + J.item,
                                      vols + J.vol_off, sinos + J.sino_off);
    }

    // the same for 3D operators whose footprints all take NC columns
    template <int NC>
    __global__ void __launch_bounds__(kThreads)
        voxel_fwd_cols_batch_kernel(const VoxFwdJob* __restrict__ jobs, const int* __restrict__ block_job,
                                    const int per_xcd, const int64_t total, const int* __restrict__ fixexp,
                                    const float* __restrict__ vols, float* __restrict__ sinos)
    {
        const int64_t id = (int64_t) (blockIdx.x % 8u) * per_xcd + (blockIdx.x / 8u);
        if (id >= total)
            return;
        const VoxFwdJob& J = jobs[block_job[id]];
        const VoxFan fan{{J.plan.fan[0], J.plan.fan[1], J.plan.fan[2]}};
        vox_fwd_cols_block<NC, float, float, 2>(J.geo, J.dims, J.lut, J.n_lut, J.plan.span, J.support, J.diff,
                                                J.pose_axis, J.pose_margin, fan, J.TU, J.TV, J.ntu, id - J.block0,
                                                fixexp + J.item, vols + J.vol_off, sinos + J.sino_off);
    }

    // dynamic LDS (the tile's sums) plus the table: FP64 entries (lut_bytes 8) or the FP32 pair
    // table (lut_bytes 4), 8 bytes per entry either way
    size_t voxel_tile_lds_bytes(const TileCfg& tc, size_t lut_bytes)
    {
        return (size_t) vox_acc_stride(tc.LA, tc.TB) * tc.TB * sizeof(long long) +
               (lut_bytes == 8 ? (size_t) kMaxLut * 8 : (size_t) kVoxLutSpan * 2 * lut_bytes) + kPlaneLds;
    }

    // Dynamic LDS of the forward by columns: the sums and the table, 8 bytes per entry; with the static
    // plane tables it has to fit 64 KB.
    constexpr size_t kColsLds = 65536 - kPlaneLds;

    size_t cols_lds_bytes(int nc, int span, const TileCfg& tc)
    {
        return ((size_t) cols_stride(tc.LA, nc) * tc.TB + (size_t) span) * 8;
    }

    int voxel_max_lut()
    {
        return kMaxLut;
    }

    // tc.LA x tc.TB: tile width x height in pixels (height 1 in 2D); LT: the table's type (FP64
    // for FP64 operators, else FP32)
    template <class ST, class LT>
    hipError_t voxel_forward_tiled(const PoseGeom* geo, const Dims& dims, const LT* lut, int n_lut, float support,
                                   int diff, const int* pose_axis, const float* pose_margin, const VoxPlan& plan,
                                   const TileCfg& tc, double slot_bound, unsigned int* d_maxbits, int* d_fixexp,
                                   const ST* vol, ST* sino, hipStream_t s)
    {
        if (n_lut < 2 || n_lut > kMaxLut)
            return hipErrorInvalidValue;
        hipError_t e = fixed_point_exponent_launch(vol, dims.nvox, slot_bound, d_maxbits, d_fixexp, s);
        if (e != hipSuccess)
            return e;
        const int TU = tc.LA, TV = dims.dim == 3 ? tc.TB : 1;
        const int ntu = (dims.det[0] + TU - 1) / TU, ntv = (dims.det[1] + TV - 1) / TV;
        const int64_t total = (int64_t) ntu * ntv * dims.nposes;
        const int64_t per_xcd = (total + 7) / 8;
        if (per_xcd * 8 > (int64_t) 0x7fffffff)
            return hipErrorInvalidValue;
        const dim3 grid((unsigned) (per_xcd * 8));
        const size_t clds = plan.cols > 0 ? cols_lds_bytes(kernel_cols(plan.cols), plan.span, tc) : 0;
        if (clds > 0 && clds <= kColsLds) {
            const VoxFan fan{{plan.fan[0], plan.fan[1], plan.fan[2]}};
            auto cols = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, grid, dim3(kThreads), clds, s, geo, dims, lut, n_lut, plan.span, support,
                                   pose_axis, pose_margin, fan, TU, TV, ntu, (int) per_xcd, total, d_fixexp, vol, sino);
            };
            auto pick = [&](auto nc) {
                constexpr int NC = decltype(nc)::value;
                if (diff)
                    cols(voxel_fwd_cols_kernel<NC, ST, LT, 1>);
                else
                    cols(voxel_fwd_cols_kernel<NC, ST, LT, 0>);
            };
            if (plan.cols <= 4)
                pick(std::integral_constant<int, 4>{});
            else if (plan.cols == 5)
                pick(std::integral_constant<int, 5>{});
            else if (plan.cols == 6)
                pick(std::integral_constant<int, 6>{});
            else
                pick(std::integral_constant<int, 8>{});
            return hipGetLastError();
        }
        const size_t lds = (size_t) vox_acc_stride(TU, TV) * TV * sizeof(long long);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(kThreads), lds, s, geo, dims, lut, n_lut, support, pose_axis,
                               pose_margin, TU, TV, ntu, (int) per_xcd, total, d_fixexp, vol, sino);
        };
        if (dims.dim == 2)
            diff ? launch(voxel_fwd_tiled_kernel<2, ST, LT, true>) : launch(voxel_fwd_tiled_kernel<2, ST, LT, false>);
        else
            diff ? launch(voxel_fwd_tiled_kernel<3, ST, LT, true>) : launch(voxel_fwd_tiled_kernel<3, ST, LT, false>);
        return hipGetLastError();
    }

    template hipError_t voxel_forward_tiled<float, float>(const PoseGeom*, const Dims&, const float*, int, float,
                                                          int, const int*, const float*, const VoxPlan&,
                                                          const TileCfg&, double,
                                                          unsigned int*, int*, const float*, float*, hipStream_t);
    template hipError_t voxel_forward_tiled<bf16, float>(const PoseGeom*, const Dims&, const float*, int, float,
                                                         int, const int*, const float*, const VoxPlan&,
                                                          const TileCfg&, double,
                                                         unsigned int*, int*, const bf16*, bf16*, hipStream_t);
    template hipError_t voxel_forward_tiled<double, double>(const PoseGeom*, const Dims&, const double*, int, float,
                                                            int, const int*, const float*, const VoxPlan&,
                                                          const TileCfg&, double,
                                                            unsigned int*, int*, const double*, double*,
                                                            hipStream_t);

    // Jobs of a batched voxel forward: one per operator, its tile-pose blocks back to back; the
    // launch's dynamic LDS is the largest tile's. cols: the columns of the widest operator's kernel by columns
    // (the further columns of the others add nothing; their tables reach as far), or 0 where one has none: all
    // take the general kernel, in its tiles unless the caller chose others. A batch of 96^3 blobs and B-splines,
    // 90 poses each, us: general kernel in 96 x 16 tiles 5017, in 32 x 32 4172, by columns 2502.
    void voxel_forward_batch_jobs(const VoxBatchItem* items, int n, std::vector<VoxFwdJob>& jobs,
                                  std::vector<int>& blocks, size_t& lds, int& cols)
    {
        jobs.clear();
        blocks.clear();
        lds = 0;
        std::vector<ColumnNeeds> needs(n);
        for (int j = 0; j < n; ++j)
            needs[j] = ColumnNeeds{items[j].plan.cols, items[j].n_lut, items[j].support, items[j].plan.smin};
        cols = common_cols(needs.data(), n);
        for (int j = 0; j < n && cols > 0; ++j)
            if (cols_lds_bytes(cols, (int) column_table_span(needs[j], cols), items[j].tile) > kColsLds)
                cols = 0;
        for (int j = 0; j < n; ++j) {
            const VoxBatchItem& it = items[j];
            VoxFwdJob J{};
            J.geo = it.geo;
            J.dims = it.dims;
            J.lut = it.lut;
            J.n_lut = it.n_lut;
            J.support = it.support;
            J.diff = it.diff;
            J.pose_axis = it.pose_axes;
            J.pose_margin = it.pose_margin;
            J.plan = it.plan;
            TileCfg tile = it.tile;
            if (cols > 0)
                J.plan.span = (int) column_table_span(needs[j], cols);
            else if (it.dims.dim == 3 && !it.tile_set)
                tile = kVoxGeneralTile;
            J.TU = tile.LA;
            J.TV = it.dims.dim == 3 ? tile.TB : 1;
            J.ntu = (it.dims.det[0] + J.TU - 1) / J.TU;
            const int ntv = (it.dims.det[1] + J.TV - 1) / J.TV;
            J.item = j;
            J.vol_off = it.vol_off;
            J.sino_off = it.sino_off;
            J.block0 = (int64_t) blocks.size();
            blocks.insert(blocks.end(), (size_t) J.ntu * ntv * it.dims.nposes, (int) jobs.size());
            jobs.push_back(J);
            const size_t need = cols > 0 ? cols_lds_bytes(cols, J.plan.span, tile)
                                         : (size_t) vox_acc_stride(J.TU, J.TV) * J.TV * sizeof(long long);
            lds = need > lds ? need : lds;
        }
    }

    // The tile launch of a batched voxel forward (the exponents d_fixexp[item] computed from
    // each operator's volume by fixed_point_exponent_batch).
    hipError_t voxel_forward_batch(int dim, int cols, const VoxFwdJob* jobs, const int* blocks, int64_t nblocks,
                                   size_t lds, const int* d_fixexp, const float* vols, float* sinos, hipStream_t s)
    {
        const int64_t per_xcd = (nblocks + 7) / 8;
        if (per_xcd * 8 > (int64_t) 0x7fffffff)
            return hipErrorInvalidValue;
        if (nblocks == 0)
            return hipSuccess;
        const dim3 grid((unsigned) (per_xcd * 8));
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(kThreads), lds, s, jobs, blocks, (int) per_xcd, nblocks, d_fixexp,
                               vols, sinos);
        };
        if (dim == 2)
            launch(voxel_fwd_tiled_batch_kernel<2>);
        else if (cols == 0)
            launch(voxel_fwd_tiled_batch_kernel<3>);
        else if (cols == 4)
            launch(voxel_fwd_cols_batch_kernel<4>);
        else if (cols == 5)
            launch(voxel_fwd_cols_batch_kernel<5>);
        else if (cols == 6)
            launch(voxel_fwd_cols_batch_kernel<6>);
        else
            launch(voxel_fwd_cols_batch_kernel<8>);
        return hipGetLastError();
    }
} // namespace ehp
