// ehp_siddon_planes.hip -- Siddon forward projection over plane-major volume views (FP32, FP64).
//
// The forward of Siddon's method (elsa/projectors/SiddonsMethod.cpp:76-124, forward :115-117;
// traversal of TraverseAABB.cpp:6-184) with one lane per ray, reading the zero-padded
// plane-major views of the Joseph forward (that axis slowest, the fan-out axis fastest). A
// wavefront holds 16 x 4 neighbouring pixels; its rays are grouped by driving axis A (their
// largest |d|) and step direction along it, and each group walks the planes of A together:
// on plane p every ray takes the segments of its traversal that lie on p, so all lanes read the
// same plane at neighbouring positions. One loop per lane would put rays that enter through a
// side face, each at its own plane, on a cache line of their own at every step.
//
// On a plane a ray crosses each transverse axis at most once, so its segments follow from sorting
// two crossing parameters below the plane's exit (sid_plane_segments): about 37 vector
// instructions and three 4-byte loads a plane for every lane alike, where taking the steps one by
// one cost 80 (47 a crossing, 1.4 crossings a plane, with the lanes of a wavefront waiting for the one that
// crosses most). 256^3, 360 poses, 384^2 pixels, FP32: 12.3 -> 7.3 ms (of which the step-free
// plane 9.2, buffer loads and unquieted minima 8.1, 16 x 4 instead of 8 x 8 wavefronts 7.5 (32 x 2:
// 7.8), two planes in flight 7.3); VALU issue bounds it (0.8 of the rate). The segments are
// siddon_traverse's, in its order, so the sum is the one-thread-per-ray kernel's bit for bit, in FP32 and in FP64 (SiddonsMethodCUDA<double>: FP64
// views and sums, the FP32 lengths of the FP32 traversal, as that kernel forms them). The
// traversal state of every ray comes from the per-operator table of the tiled back projection.
#include "ehp_waves.hpp"

namespace ehp
{
    namespace
    {
        // Wavefront width in pixels (3D): three loads a plane make the rows a wavefront touches count
        // more than the lanes that idle at its ends (7.34 ms; 8 wide 8.05 ms, 32 wide 7.69 ms).
        constexpr int kSidWU = 16;

        // 32-bit offsets from a view's base through a buffer resource: the plane's offset goes into
        // the load's scalar operand and the ray's into its vector operand, with no address arithmetic.
        typedef __amdgpu_buffer_rsrc_t buf_t;

        __device__ __forceinline__ buf_t view_resource(const PadView& V, uint32_t esize)
        {
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(V.base), 0, (int) ((uint32_t) V.size * esize),
                                                     0x00020000);
        }

        template <class T>
        __device__ __forceinline__ T view_load(buf_t rsrc, uint32_t off, uint32_t poff)
        {
            if constexpr (sizeof(T) == 8) {
                const auto w = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int) off, (int) poff, 0);
                T v;
                __builtin_memcpy(&v, &w, 8);
                return v;
            } else {
                const int w = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int) off, (int) poff, 0);
                T v;
                __builtin_memcpy(&v, &w, 4);
                return v;
            }
        }

        // The group's rays walk the planes of axis A together (sid_plane_add) from plane p0 on, dir up
        // or down: start is the iteration of the ray's first plane and full0 the last of these in the
        // group. FB2: the view's fastest axis is b2 (else b1). T: the view's element type, in which the
        // sum runs. TWICE: some ray of the group may cross an axis twice on a plane.
        template <int D, int A, bool TWICE, class T>
        __device__ inline T sid_planes(const SidRec& r, SidSpan s, const Dims& dims, const PadView& V, int p0,
                                       int dir, int start, int full0)
        {
            const buf_t rsrc = view_resource(V, (uint32_t) sizeof(T));
            T acc = T(0);
            // the plane's offset, the same for the whole group (in scalar registers)
            uint32_t poff = (uint32_t) p0 * V.PS4;
            const uint32_t dp = dir < 0 ? 0u - V.PS4 : V.PS4;
            auto at = [&](uint32_t pl) { return [=](uint32_t off) { return view_load<T>(rsrc, off, pl); }; };
            const int np = dir < 0 ? p0 + 1 : dims.vol[A] - p0; // planes up to the volume's end
            int it = 0;
            for (; it < full0 && it < np; ++it, poff += dp)
                if (it >= start && s.t < s.tend)
                    acc = sid_plane_add<D, A, T>(r, s, acc, at(poff));
            if constexpr (!TWICE) {
                // two planes per step, both fetched before either is added
                for (; it + 1 < np && s.t < s.tend; it += 2, poff += 2u * dp) {
                    const SidSegments<T> ga = sid_plane_segments<D, A, T>(r, s, at(poff));
                    const bool more = s.t < s.tend;
                    SidSegments<T> gb{};
                    if (more)
                        gb = sid_plane_segments<D, A, T>(r, s, at(poff + dp));
                    acc = sid_segments_add<D>(ga, acc);
                    if (more)
                        acc = sid_segments_add<D>(gb, acc);
                }
            }
            for (; it < np && s.t < s.tend; ++it, poff += dp)
                acc = sid_plane_add<D, A, T>(r, s, acc, at(poff));
            return acc;
        }

        // The rays of group K = 2 * axis + direction of a wavefront (every lane active here); t: the
        // traversal coordinate of the ray's first plane (the plane, or its negative downwards).
        template <int D, int K, class T>
        __device__ __forceinline__ void sid_group(int keys, int key, const SidRec& r, const Dims& dims,
                                                  const ViewSet& vs, int t, T& val)
        {
            if (!((keys >> K) & 1))
                return;
            constexpr int A = K / 2, dir = (K & 1) ? -1 : 1;
            constexpr uint32_t lg = sizeof(T) == 8 ? 3u : 2u;
            const bool mine = key == K;
            const int t0 = wave_min(mine ? t : 0x7fffffff);
            const int full0 = wave_max(mine ? t : -0x7fffffff) - t0;
            if (mine) {
                const PadView& V = vs.v[A];
                const SidSpan s = (D == 3 && ((vs.fb2 >> A) & 1)) ? sid_span_init<D, A, true>(r, dims.vol, V.RS4, lg)
                                                                  : sid_span_init<D, A, false>(r, dims.vol, V.RS4, lg);
                val = __any(sid_may_cross_twice<D, A>(r, s.tend))
                          ? sid_planes<D, A, true, T>(r, s, dims, V, dir * t0, dir, t - t0, full0)
                          : sid_planes<D, A, false, T>(r, s, dims, V, dir * t0, dir, t - t0, full0);
            }
        }

        // Block id of the forward's tiles (fwd_pixel's order): the rays of its wavefronts, grouped
        // by driving axis and direction, each group walking its planes together.
        template <int D, class T>
        __device__ __forceinline__ void sid_fwd_block(const SidRec* __restrict__ table, const Dims& dims,
                                                      const ViewSet& views, const int tiles_u, const int64_t id,
                                                      T* __restrict__ sino)
        {
            int u, v, pose;
            fwd_pixel<D, kSidWU>(dims, tiles_u, id, u, v, pose);
            const bool inside = u < dims.det[0] && v < dims.det[1];
            const int64_t ray = (int64_t) pose * dims.pix_per_pose + (int64_t) v * dims.det[0] + u;
            SidRec r{};
            int key = -1, t = 0;
            if (inside) {
                r = table[ray];
                if (sid_hit(r)) {
                    const int a = sid_axis(r);
                    const bool neg = sid_step(r, a) < 0;
                    key = 2 * a + (neg ? 1 : 0);
                    const int c = a == 0 ? r.cur0[0] : (a == 1 ? r.cur0[1] : r.cur0[2]); // in registers
                    t = neg ? -c : c;
                }
            }
            const int keys = wave_or(key >= 0 ? 1 << key : 0);
            T val = T(0);
            sid_group<D, 0>(keys, key, r, dims, views, t, val);
            sid_group<D, 1>(keys, key, r, dims, views, t, val);
            sid_group<D, 2>(keys, key, r, dims, views, t, val);
            sid_group<D, 3>(keys, key, r, dims, views, t, val);
            if (D == 3) {
                sid_group<D, 2 * D - 2>(keys, key, r, dims, views, t, val);
                sid_group<D, 2 * D - 1>(keys, key, r, dims, views, t, val);
            }
            if (inside)
                sino[ray] = val;
        }

        template <int D, class T>
        __global__ void __launch_bounds__(kFwdThreads)
            siddon_fwd_planes_kernel(const SidRec* __restrict__ table, const Dims dims, const ViewSet views,
                                     const int tiles_u, const int per_xcd, const int64_t total,
                                     T* __restrict__ sino)
        {
            const int64_t id = (int64_t) (blockIdx.x % 8u) * per_xcd + (blockIdx.x / 8u);
            if (id >= total)
                return;
            sid_fwd_block<D, T>(table, dims, views, tiles_u, id, sino);
        }

        // the forwards of many operators in one launch (block b: block b - job.block0 of job
        // block_job[b], as that operator's own launch would run it)
        template <int D>
        __global__ void __launch_bounds__(kFwdThreads)
            siddon_fwd_planes_batch_kernel(const SidFwdJob* __restrict__ jobs, const int* __restrict__ block_job,
                                           const int per_xcd, const int64_t total, float* __restrict__ sinos)
        {
            const int64_t id = (int64_t) (blockIdx.x % 8u) * per_xcd + (blockIdx.x / 8u);
            if (id >= total)
                return;
            const SidFwdJob& J = jobs[block_job[id]];
            sid_fwd_block<D, float>(J.table, J.dims, J.views, J.tiles_u, id - J.block0, sinos + J.sino_off);
        }
    } // namespace

    template <class T>
    hipError_t siddon_forward_planes(const SidRec* table, const Dims& dims, const PadLayout* layouts,
                                     void* const* views, int axes_present, const T* vol, T* sino, hipStream_t s)
    {
        constexpr uint32_t es = sizeof(T);
        ViewSet vs{};
        for (int a = 0; a < dims.dim; ++a) {
            if (!(axes_present & (1 << a)))
                continue;
            const PadLayout& L = layouts[a];
            if (L.pairs)
                return hipErrorInvalidValue; // the Siddon walk reads single voxels of plain views
            vs.v[a] = PadView{views[a], L.PS * es, L.RS * es, L.size};
            const int b2 = dims.dim == 3 ? (a == 2 ? 1 : 2) : -1;
            if (L.f == b2)
                vs.fb2 |= 1 << a;
        }
        hipError_t e = joseph_view_copies<T>(dims, layouts, views, axes_present, vol, s);
        if (e != hipSuccess)
            return e;
        const FwdGrid fg = fwd_grid(dims, kSidWU);
        if (fg.per_xcd * 8 > (int64_t) 0x7fffffff)
            return hipErrorInvalidValue;
        const dim3 grid((unsigned) (fg.per_xcd * 8));
        if (dims.dim == 2)
            hipLaunchKernelGGL((siddon_fwd_planes_kernel<2, T>), grid, dim3(kFwdThreads), 0, s, table, dims, vs,
                               fg.tiles_u, (int) fg.per_xcd, fg.total, sino);
        else
            hipLaunchKernelGGL((siddon_fwd_planes_kernel<3, T>), grid, dim3(kFwdThreads), 0, s, table, dims, vs,
                               fg.tiles_u, (int) fg.per_xcd, fg.total, sino);
        return hipGetLastError();
    }

    template hipError_t siddon_forward_planes<float>(const SidRec*, const Dims&, const PadLayout*, void* const*, int,
                                                     const float*, float*, hipStream_t);
    template hipError_t siddon_forward_planes<double>(const SidRec*, const Dims&, const PadLayout*, void* const*, int,
                                                      const double*, double*, hipStream_t);

    // Jobs of a batched Siddon forward: the view copies of every operator (one job per view)
    // and the forward blocks (one job per operator).
    void siddon_forward_batch_jobs(const JosephBatchItem* items, int n, std::vector<CopyJob>& cjobs,
                                   std::vector<int>& cblocks, std::vector<SidFwdJob>& fjobs, std::vector<int>& fblocks)
    {
        cjobs.clear();
        cblocks.clear();
        fjobs.clear();
        fblocks.clear();
        for (int j = 0; j < n; ++j) {
            const JosephBatchItem& it = items[j];
            SidFwdJob fj{};
            fj.table = it.sidtable;
            fj.dims = it.dims;
            fj.sino_off = it.sino_off;
            for (int a = 0; a < it.dims.dim; ++a) {
                if (!(it.axes_present & (1 << a)))
                    continue;
                const PadLayout& L = it.layouts[a];
                CopyJob cj{};
                cj.view = it.views[a];
                cj.dims = it.dims;
                cj.L = L;
                cj.vol_off = it.vol_off;
                cj.block0 = (int64_t) cblocks.size();
                const int64_t nb = view_copy_blocks(it.dims, L, cj.gx, cj.gy);
                cblocks.insert(cblocks.end(), (size_t) nb, (int) cjobs.size());
                cjobs.push_back(cj);
                fj.views.v[a] = PadView{it.views[a], L.PS * 4u, L.RS * 4u, L.size};
                const int b2 = it.dims.dim == 3 ? (a == 2 ? 1 : 2) : -1;
                if (L.f == b2)
                    fj.views.fb2 |= 1 << a;
            }
            const FwdGrid fg = fwd_grid(it.dims, kSidWU);
            fj.tiles_u = fg.tiles_u;
            fj.block0 = (int64_t) fblocks.size();
            fblocks.insert(fblocks.end(), (size_t) fg.total, (int) fjobs.size());
            fjobs.push_back(fj);
        }
    }

    hipError_t siddon_forward_batch(int dim, const CopyJob* cjobs, const int* cblocks, int64_t ncblocks,
                                    const SidFwdJob* fjobs, const int* fblocks, int64_t nfblocks, const float* vols,
                                    float* sinos, hipStream_t s)
    {
        hipError_t e = view_copy_batch(cjobs, cblocks, ncblocks, vols, s);
        if (e != hipSuccess)
            return e;
        const int64_t per_xcd = (nfblocks + 7) / 8;
        if (per_xcd * 8 > (int64_t) 0x7fffffff)
            return hipErrorInvalidValue;
        if (nfblocks > 0) {
            const dim3 grid((unsigned) (per_xcd * 8));
            if (dim == 2)
                hipLaunchKernelGGL((siddon_fwd_planes_batch_kernel<2>), grid, dim3(kFwdThreads), 0, s, fjobs, fblocks,
                                   (int) per_xcd, nfblocks, sinos);
            else
                hipLaunchKernelGGL((siddon_fwd_planes_batch_kernel<3>), grid, dim3(kFwdThreads), 0, s, fjobs, fblocks,
                                   (int) per_xcd, nfblocks, sinos);
        }
        return hipGetLastError();
    }
} // namespace ehp
