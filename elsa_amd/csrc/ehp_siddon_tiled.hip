// ehp_siddon_tiled.hip -- Siddon back projection with LDS-privatised volume tiles (FP32, FP64).
//
// The adjoint of Siddon's method (elsa/projectors/SiddonsMethod.cpp:76-124, adjoint
// :119-120) without global atomics, on the scheme of the tiled Joseph back projection: the
// volume is cut into tiles long along one driving axis, one workgroup owns a tile for all
// poses and sums in LDS every crossing of every ray (driving along that axis) that passes
// through it, then adds the tile to the volume once; one launch for the tiles of two driving axes
// (siddon_adj_pair_kernel) where rays enough pay for it (pair_launch), one per axis otherwise.
//
// A ray takes the tile's planes in its own order (sid_tile_ray): its state at the first plane
// follows from the step counts there, and each plane's segments from sorting two crossing
// parameters, as in the forward, with every lane doing the same work. Restarting the traversal at
// the tile's boundary and stepping through it crossing by crossing (siddon_box, kept for rays that may cross an axis
// twice on a plane) took 111 vector instructions a crossing, most of them masked updates of the three axes:
// 256^3, 360 poses, 384^2 pixels 20.0 -> 10.6 ms; 128^3 2.12 -> 0.94 ms; 2D 256^2 0.131 -> 0.078 ms.
// The crossings, voxels and lengths are the forward's. Rows of slots are an odd number long
// (sid_row_slots). VALU issue and the 64-bit LDS atomics (three a plane) bound it.
//
// Both axes in one launch and 512 threads in 64 VGPRs, against one launch of 256 threads per axis:
// 256^3 10.6 -> 9.96 ms, 128^3 0.94 -> 0.79, FP64 96 x 64 x 112 / 77 poses 0.23 -> 0.185; 2D (256
// threads) 256^2 78 -> 54 us.
//
// Sums are 64-bit fixed point as in the Joseph kernel: one exponent per call from max|y|
// and the slot bound, each contribution y * length rounded once to the unit (fixed_round; in
// FP32 the product is exact in FP64).
#include "ehp_kernels.hpp"
#include "ehp_tile_pair.hpp"

namespace ehp
{
    namespace
    {
        // threads of a workgroup
        template <int D>
        constexpr int kNT = D == 3 ? 512 : 256;
        // LDS (address space 3) pointers: 32-bit byte addresses
        typedef __attribute__((address_space(3))) unsigned long long lds_u64;
        typedef __attribute__((address_space(3))) char lds_char;
    } // namespace

    template <int D>
    __global__ void __launch_bounds__(256)
        siddon_table_kernel(const PoseGeom* __restrict__ geo, const Dims dims, SidRec* __restrict__ table)
    {
        const int pose = blockIdx.y;
        const int64_t pix = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
        if (pix >= dims.pix_per_pose)
            return;
        const int u = (int) (pix % dims.det[0]);
        const int v = (int) (pix / dims.det[0]);
        float o[3], d[3];
        make_ray_px<D>(geo[pose], dims, u, v, o, d);
        table[(int64_t) pose * dims.pix_per_pose + pix] = siddon_setup<D>(o, d, dims.vol);
    }

    __global__ void __launch_bounds__(256)
        siddon_pose_axes_kernel(const SidRec* __restrict__ table, const Dims dims, int* __restrict__ pose_axes)
    {
        const int pose = blockIdx.y;
        const int64_t pix = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
        if (pix >= dims.pix_per_pose)
            return;
        const SidRec r = table[(int64_t) pose * dims.pix_per_pose + pix];
        if (sid_hit(r))
            atomicOr(pose_axes + pose, 1 << sid_axis(r));
    }

    hipError_t siddon_ray_table(const PoseGeom* geo, const Dims& dims, SidRec* table, int* pose_axes, hipStream_t s)
    {
        const dim3 grid((unsigned) ((dims.pix_per_pose + 255) / 256), (unsigned) dims.nposes);
        if (dims.dim == 2)
            hipLaunchKernelGGL((siddon_table_kernel<2>), grid, dim3(256), 0, s, geo, dims, table);
        else
            hipLaunchKernelGGL((siddon_table_kernel<3>), grid, dim3(256), 0, s, geo, dims, table);
        hipError_t e = launch_fill<int>(pose_axes, dims.nposes, 0, s);
        if (e != hipSuccess)
            return e;
        hipLaunchKernelGGL(siddon_pose_axes_kernel, grid, dim3(256), 0, s, table, dims, pose_axes);
        return hipGetLastError();
    }

    size_t siddon_tile_lds_bytes(const Dims& dims, const TileCfg& tc, int batch)
    {
        return (size_t) tc.LA * sid_row_slots(tc, dims.dim) * (dims.dim == 3 ? tc.TC : 1) * sizeof(long long) +
               batch_lds_bytes(batch);
    }

    // One tile of the back projection along driving axis A (tile < ntA * ntB * ntC); T = float or
    // double (sinogram and volume).
    // PAIR: the other axis' tiles may add to the volume now
    template <int D, int A, bool PAIR, class T>
    __device__ __forceinline__ void sid_adj_tiled_block(const PoseGeom* __restrict__ geo,
                                                        const SidRec* __restrict__ table, const Dims& dims,
                                                        const int* __restrict__ pose_axes, const TileCfg& tc,
                                                        const int ntA, const int ntB, const int tile, const int batch,
                                                        const int* __restrict__ fixexp, const T* __restrict__ sino,
                                                        T* __restrict__ vol)
    {
        constexpr int b1 = TileAxes<D, A>::b1, b2 = TileAxes<D, A>::b2;
        constexpr int kThreads = kNT<D>;
        extern __shared__ long long lds[];

        const int tid = threadIdx.x;
        const TileBox t = make_tile<D, A>(dims, tc, tile % ntA, (tile / ntA) % ntB, tile / (ntA * ntB));
        const SidTileOff to = sid_tile_offsets<D>(t, tc, (uint32_t) (uintptr_t) (lds_char*) lds);
        const int row = to.cs / 8; // slots per row
        const int nslots = tc.LA * row * (D == 3 ? tc.TC : 1);
        long long* iacc = lds;
        const BatchLds bl = batch_lds(lds, nslots, batch);
        CandRect* s_rect = bl.rect;
        int *s_cnt = bl.cnt, *s_pref = bl.pref;
        for (int i = tid; i < nslots; i += kThreads)
            iacc[i] = 0;
        // the tile's voxel box
        float flo[3] = {0.0f, 0.0f, 0.0f}, fhi[3] = {0.0f, 0.0f, 0.0f};
        flo[A] = (float) t.A0;
        fhi[A] = (float) t.A1;
        flo[b1] = (float) t.B0;
        fhi[b1] = (float) t.B1;
        if (D == 3) {
            flo[b2] = (float) t.C0;
            fhi[b2] = (float) t.C1;
        }
        const int eg = fixexp[0];
        __syncthreads();

        for (int pbase = 0; eg != kNonFinite && pbase < dims.nposes; pbase += batch) {
            if (tid < batch) {
                const int p = pbase + tid;
                int u0 = 0, u1 = -1, v0 = 0, v1 = -1;
                int cnt = 0;
                if (p < dims.nposes && (pose_axes[p] & (1 << A))) {
                    if (box_bbox<D>(geo[p], flo, fhi, dims, u0, u1, v0, v1))
                        cnt = (u1 - u0 + 1) * (v1 - v0 + 1);
                }
                CandRect cr;
                cr.nu = u1 - u0 + 1;
                cr.rnu = 1.0f / (float) (u1 - u0 + 1);
                cr.base = (long long) p * dims.pix_per_pose + (long long) v0 * dims.det[0] + u0;
                s_rect[tid] = cr;
                s_cnt[tid] = cnt;
            }
            __syncthreads();
            if (tid == 0) {
                s_pref[0] = 0;
                for (int j = 0; j < batch; ++j)
                    s_pref[j + 1] = s_pref[j] + s_cnt[j];
            }
            __syncthreads();
            const int total = s_pref[batch];
            // Candidate k of this batch is entry k - pref[j] of pose j's rectangle, j the last pose with
            // pref[j] <= k; each lane takes k = tid, tid + kThreads, ... in order, keeping j in
            // registers. The next candidate is loaded while the current one is added (two register
            // sets taken in turn).
            int j = 0, pj = 0, pn = s_pref[1];
            CandRect cr = s_rect[0];
            auto fetch = [&](int k, SidRec& r, T& yv) {
                while (k >= pn) {
                    ++j;
                    pj = pn;
                    pn = s_pref[j + 1];
                    cr = s_rect[j];
                }
                int rrow, col;
                rect_split(k - pj, cr.nu, cr.rnu, rrow, col);
                const int64_t ray = cr.base + (int64_t) (mul24((uint32_t) rrow, (uint32_t) dims.det[0]) + (uint32_t) col);
                yv = sino[ray];
                r = table[ray];
            };
            auto process = [&](const SidRec& r, T yv) {
                if (yv == T(0) || !sid_hit(r) || sid_axis(r) != A)
                    return;
                // y in units of q (a power-of-two scaling, exact); each crossing adds
                // y * length rounded once to an integer (|y * length| < 2^51 units: the slot
                // bound is at least 4096 and lengths are below 2)
                const double yq = ldexp((double) yv, 62 - eg);
                sid_tile_ray<D, A>(r, t, to, [&](uint32_t off, float w) {
                    __hip_atomic_fetch_add((lds_u64*) (uintptr_t) off, fixed_round(yq, (double) w), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                });
            };
            SidRec ra{}, rb{};
            T ya = T(0), yb = T(0);
            if (tid < total)
                fetch(tid, ra, ya);
            for (int k = tid; k < total; k += 2 * kThreads) {
                const int k1 = k + kThreads, k2 = k + 2 * kThreads;
                if (k1 < total)
                    fetch(k1, rb, yb);
                process(ra, ya);
                if (k2 < total)
                    fetch(k2, ra, ya);
                if (k1 < total)
                    process(rb, yb);
            }
            __syncthreads();
        }

        // add the tile to the volume
        const double q = eg == kNonFinite ? __longlong_as_double(0x7ff8000000000000ll) : ldexp(1.0, eg - 62);
        const int TCe = D == 3 ? tc.TC : 1;
        for (int i = tid; i < nslots; i += kThreads) {
            const int xb = i % row;
            const int rest = i / row;
            const int xc = rest % TCe;
            const int xa = rest / TCe;
            const int ca = t.A0 + xa, cb = t.B0 + xb, cc = t.C0 + xc;
            if (ca >= t.A1 || cb >= t.B1 || (D == 3 && cc >= t.C1))
                continue;
            int c[3] = {0, 0, 0};
            c[A] = ca;
            c[b1] = cb;
            if (D == 3)
                c[b2] = cc;
            const int64_t lin = c[0] + c[1] * dims.strides[1] + (int64_t) c[2] * dims.strides[2];
            const T sum = (T) ((double) iacc[i] * q);
            if (PAIR)
                add_second(vol + lin, sum);
            else
                vol[lin] += sum;
        }
    }

    template <int D, int A, class T>
    __global__ void __launch_bounds__(kNT<D>, 8)
        siddon_adj_tiled_kernel(const PoseGeom* __restrict__ geo, const SidRec* __restrict__ table, const Dims dims,
                                const int* __restrict__ pose_axes, const TileCfg tc, const TileCounts c,
                                const int batch, const int* __restrict__ fixexp, const T* __restrict__ sino,
                                T* __restrict__ vol)
    {
        // consecutive workgroups land on different XCDs: give each XCD a contiguous block of tiles
        const int tile = (int) (blockIdx.x % 8u) * c.per_xcd + (int) (blockIdx.x / 8u);
        if (tile < c.n)
            sid_adj_tiled_block<D, A, false, T>(geo, table, dims, pose_axes, tc, c.nA, c.nB, tile, batch, fixexp, sino,
                                                vol);
    }

    // the tiles of two driving axes
    template <int D, int A0, int A1, class T>
    __global__ void __launch_bounds__(kNT<D>, 8)
        siddon_adj_pair_kernel(const PoseGeom* __restrict__ geo, const SidRec* __restrict__ table, const Dims dims,
                               const int* __restrict__ pose_axes, const TileCfg tc, const TileCounts c0,
                               const TileCounts c1, const int batch, const int* __restrict__ fixexp,
                               const T* __restrict__ sino, T* __restrict__ vol)
    {
        const int xcd = (int) (blockIdx.x % 8u), k = (int) (blockIdx.x / 8u);
        if (k < c0.per_xcd) {
            const int tile = xcd * c0.per_xcd + k;
            if (tile < c0.n)
                sid_adj_tiled_block<D, A0, true, T>(geo, table, dims, pose_axes, tc, c0.nA, c0.nB, tile, batch, fixexp,
                                                    sino, vol);
        } else {
            const int tile = xcd * c1.per_xcd + k - c0.per_xcd;
            if (tile < c1.n)
                sid_adj_tiled_block<D, A1, true, T>(geo, table, dims, pose_axes, tc, c1.nA, c1.nB, tile, batch, fixexp,
                                                    sino, vol);
        }
    }

    // the tiles of many operators in one launch (block b: tile b - job.block0 of job block_job[b])
    template <int D, int A, bool PAIR>
    __device__ __forceinline__ void sid_batch_block(const SidAdjJob* __restrict__ jobs,
                                                    const int* __restrict__ block_job, const int64_t id,
                                                    const int* __restrict__ fixexp, const float* __restrict__ sinos,
                                                    float* __restrict__ vols)
    {
        const SidAdjJob& J = jobs[block_job[id]];
        sid_adj_tiled_block<D, A, PAIR, float>(J.geo, J.table, J.dims, J.pose_axes, J.tc, J.ntA, J.ntB,
                                               (int) (id - J.block0), J.batch, fixexp + J.item, sinos + J.sino_off,
                                               vols + J.vol_off);
    }

    template <int D, int A>
    __global__ void __launch_bounds__(kNT<D>, 8)
        siddon_adj_tiled_batch_kernel(const BatchTiles<SidAdjJob> t, const int* __restrict__ fixexp,
                                      const float* __restrict__ sinos, float* __restrict__ vols)
    {
        const int64_t id = (int64_t) (blockIdx.x % 8u) * t.per_xcd + (blockIdx.x / 8u);
        if (id < t.total)
            sid_batch_block<D, A, false>(t.jobs, t.block_job, id, fixexp, sinos, vols);
    }

    template <int D, int A0, int A1>
    __global__ void __launch_bounds__(kNT<D>, 8)
        siddon_adj_pair_batch_kernel(const BatchTiles<SidAdjJob> t0, const BatchTiles<SidAdjJob> t1,
                                     const int* __restrict__ fixexp, const float* __restrict__ sinos,
                                     float* __restrict__ vols)
    {
        const int64_t xcd = blockIdx.x % 8u;
        const int k = (int) (blockIdx.x / 8u);
        if (k < t0.per_xcd) {
            const int64_t id = xcd * t0.per_xcd + k;
            if (id < t0.total)
                sid_batch_block<D, A0, true>(t0.jobs, t0.block_job, id, fixexp, sinos, vols);
        } else {
            const int64_t id = xcd * t1.per_xcd + k - t0.per_xcd;
            if (id < t1.total)
                sid_batch_block<D, A1, true>(t1.jobs, t1.block_job, id, fixexp, sinos, vols);
        }
    }

    // fn(D, axis) or fn(D, first, second) as constants
    template <class Fn>
    void with_axis(int dim, int a, Fn fn)
    {
        using std::integral_constant;
        if (dim == 2) {
            if (a == 0)
                fn(integral_constant<int, 2>{}, integral_constant<int, 0>{});
            else
                fn(integral_constant<int, 2>{}, integral_constant<int, 1>{});
        } else {
            if (a == 0)
                fn(integral_constant<int, 3>{}, integral_constant<int, 0>{});
            else if (a == 1)
                fn(integral_constant<int, 3>{}, integral_constant<int, 1>{});
            else
                fn(integral_constant<int, 3>{}, integral_constant<int, 2>{});
        }
    }

    template <class Fn>
    void with_pair(int dim, int axes, Fn fn)
    {
        using std::integral_constant;
        if (dim == 2)
            fn(integral_constant<int, 2>{}, integral_constant<int, 0>{}, integral_constant<int, 1>{});
        else
            with_axis_pair(axes, [&](auto a0, auto a1) { fn(integral_constant<int, 3>{}, a0, a1); });
    }

    template <class T>
    hipError_t siddon_adjoint_tiled(const PoseGeom* geo, const SidRec* table, const Dims& dims, const int* pose_axes,
                                    int axes_present, const TileCfg& tc, int batch, double slot_bound, double wait,
                                    unsigned int* d_maxbits, int* d_fixexp, const T* sino, T* vol, hipStream_t s)
    {
        if (batch < 1 || batch > kMaxPoseBatch)
            return hipErrorInvalidValue;
        hipError_t e = launch_fill<T>(vol, dims.nvox, T(0), s);
        if (e == hipSuccess)
            e = fixed_point_exponent_launch(sino, dims.nrays, slot_bound, d_maxbits, d_fixexp, s);
        if (e != hipSuccess)
            return e;
        const size_t lds = siddon_tile_lds_bytes(dims, tc, batch);
        if (pair_launch(axes_present, dims.nvox, wait)) {
            with_pair(dims.dim, axes_present, [&](auto d, auto a0, auto a1) {
                constexpr int D = decltype(d)::value;
                const TileCounts c0 = axis_tiles(dims, tc, a0), c1 = axis_tiles(dims, tc, a1);
                if ((int64_t) (c0.per_xcd + c1.per_xcd) * 8 > (int64_t) 0x7fffffff) {
                    e = hipErrorInvalidValue;
                    return;
                }
                hipLaunchKernelGGL((siddon_adj_pair_kernel<D, decltype(a0)::value, decltype(a1)::value, T>),
                                   dim3((unsigned) (c0.per_xcd + c1.per_xcd) * 8), dim3(kNT<D>), lds, s, geo, table,
                                   dims, pose_axes, tc, c0, c1, batch, d_fixexp, sino, vol);
                e = hipGetLastError();
            });
            return e;
        }
        for (int a = 0; e == hipSuccess && a < dims.dim; ++a) {
            if (!(axes_present & (1 << a)))
                continue;
            with_axis(dims.dim, a, [&](auto d, auto ax) {
                constexpr int D = decltype(d)::value;
                const TileCounts c = axis_tiles(dims, tc, a);
                hipLaunchKernelGGL((siddon_adj_tiled_kernel<D, decltype(ax)::value, T>),
                                   dim3((unsigned) c.per_xcd * 8), dim3(kNT<D>), lds, s, geo, table, dims, pose_axes, tc,
                                   c, batch, d_fixexp, sino, vol);
                e = hipGetLastError();
            });
        }
        return e;
    }

    template hipError_t siddon_adjoint_tiled<float>(const PoseGeom*, const SidRec*, const Dims&, const int*, int,
                                                    const TileCfg&, int, double, double, unsigned int*, int*, const float*,
                                                    float*, hipStream_t);
    template hipError_t siddon_adjoint_tiled<double>(const PoseGeom*, const SidRec*, const Dims&, const int*, int,
                                                     const TileCfg&, int, double, double, unsigned int*, int*,
                                                     const double*, double*, hipStream_t);

    // The tiles of every operator per driving axis (one job per operator that has rays of that
    // axis).
    void siddon_adjoint_batch_jobs(const JosephBatchItem* items, int n, std::vector<SidAdjJob> ajobs[3],
                                   std::vector<int> ablocks[3], size_t lds[3])
    {
        for (int a = 0; a < 3; ++a) {
            ajobs[a].clear();
            ablocks[a].clear();
            lds[a] = 0;
        }
        for (int j = 0; j < n; ++j) {
            const JosephBatchItem& it = items[j];
            for (int a = 0; a < it.dims.dim; ++a) {
                if (!(it.axes_present & (1 << a)))
                    continue;
                SidAdjJob aj{};
                aj.geo = it.geo;
                aj.table = it.sidtable;
                aj.pose_axes = it.pose_axes;
                aj.dims = it.dims;
                aj.tc = it.tile;
                aj.batch = it.batch;
                aj.item = j;
                aj.sino_off = it.sino_off;
                aj.vol_off = it.vol_off;
                int ntC;
                tile_counts(it.dims, it.tile, a, aj.ntA, aj.ntB, ntC);
                aj.block0 = (int64_t) ablocks[a].size();
                ablocks[a].insert(ablocks[a].end(), (size_t) aj.ntA * aj.ntB * ntC, (int) ajobs[a].size());
                ajobs[a].push_back(aj);
                const size_t need = siddon_tile_lds_bytes(it.dims, it.tile, it.batch);
                lds[a] = need > lds[a] ? need : lds[a];
            }
        }
    }

    // The tile launches of a batched back projection (the volumes already cleared and the
    // exponents d_fixexp[item] computed by fixed_point_exponent_batch).
    hipError_t siddon_adjoint_batch(int dim, const SidAdjJob* const ajobs[3], const int* const ablocks[3],
                                    const int64_t nablocks[3], const size_t lds[3], int64_t nvol_total, double wait,
                                    const int* d_fixexp, const float* sinos, float* vols, hipStream_t s)
    {
        hipError_t e = hipSuccess;
        auto tiles = [&](int a) {
            return BatchTiles<SidAdjJob>{ajobs[a], ablocks[a], nablocks[a], (int) ((nablocks[a] + 7) / 8)};
        };
        int axes = 0;
        int64_t most = 0;
        for (int a = 0; a < dim; ++a) {
            axes |= nablocks[a] > 0 ? 1 << a : 0;
            most += nablocks[a] + 8;
        }
        if (most > (int64_t) 0x7fffffff)
            return hipErrorInvalidValue;
        if (pair_launch(axes, nvol_total, wait)) {
            with_pair(dim, axes, [&](auto d, auto a0, auto a1) {
                constexpr int D = decltype(d)::value;
                const BatchTiles<SidAdjJob> t0 = tiles(a0), t1 = tiles(a1);
                const size_t need = lds[a0] > lds[a1] ? lds[a0] : lds[a1];
                hipLaunchKernelGGL((siddon_adj_pair_batch_kernel<D, decltype(a0)::value, decltype(a1)::value>),
                                   dim3((unsigned) (t0.per_xcd + t1.per_xcd) * 8), dim3(kNT<D>), need, s, t0, t1,
                                   d_fixexp, sinos, vols);
                e = hipGetLastError();
            });
            return e;
        }
        for (int a = 0; e == hipSuccess && a < dim; ++a) {
            if (nablocks[a] == 0)
                continue;
            with_axis(dim, a, [&](auto d, auto ax) {
                constexpr int D = decltype(d)::value;
                const BatchTiles<SidAdjJob> t = tiles(a);
                hipLaunchKernelGGL((siddon_adj_tiled_batch_kernel<D, decltype(ax)::value>),
                                   dim3((unsigned) t.per_xcd * 8), dim3(kNT<D>), lds[a], s, t, d_fixexp, sinos, vols);
                e = hipGetLastError();
            });
        }
        return e;
    }
} // namespace ehp
