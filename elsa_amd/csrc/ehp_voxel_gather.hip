// ehp_voxel_gather.hip -- voxel-driven back projection as a gather (FP32 arithmetic with the sinogram
// and volume stored in FP32 or bfloat16; FP64).
//
// The adjoint of elsa's voxel projectors (VoxelComputation.h:110-152): every voxel sums weight x pixel
// over the pixels of its footprint in every pose, in registers, and is written once. Footprints and taps
// are those of the tiled forward (FP32: footprint_fast and the pair table; FP64: the weights of the
// one-thread-per-voxel kernel).
#include "ehp_kernels.hpp"

#include <type_traits>

namespace ehp
{
    namespace
    {
        constexpr int kMaxThreads = 1024;

        // Threads of a block: 256, or one wavefront for each of a voxel's
        int gather_threads(int waves)
        {
            return waves > 4 ? 64 * waves : 256;
        }

        typedef __amdgpu_buffer_rsrc_t buf_t;

        // a pixel at a byte offset of one pose's detector, 0 past its end
        template <class ST>
        __device__ __forceinline__ auto pixel_load(buf_t rsrc, uint32_t off)
        {
            if constexpr (sizeof(ST) == 8) {
                const auto w = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int) off, 0, 0);
                double v;
                __builtin_memcpy(&v, &w, 8);
                return v;
            } else if constexpr (sizeof(ST) == 4) {
                const int w = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int) off, 0, 0);
                float v;
                __builtin_memcpy(&v, &w, 4);
                return v;
            } else {
                const auto w = __builtin_amdgcn_raw_buffer_load_b16(rsrc, (int) off, 0, 0);
                ST v;
                __builtin_memcpy(&v, &w, 2);
                return up(v);
            }
        }
    } // namespace

    // The voxels of a block: threads / waves (at least 64), lane t taking parts (t / voxels) * parts / waves onwards of
    // voxel t % voxels; one part unless MORE. gather(p0, p1, x, y, z): the sum over poses p0 .. p1 - 1, the same in a
    // wavefront. sums: LDS for the parts of each of the block's voxels (waves > 1). YSLOW: voxels are counted with y
    // slowest (x fastest, then z), else in the volume's order.
    template <bool YSLOW, bool MORE, class AT, class ST, class Fn>
    __device__ __forceinline__ void gather_parts(const Dims& dims, const int parts, const int waves, const int64_t blk,
                                                 AT* sums, ST* __restrict__ vol, Fn gather)
    {
        const int nv = (int) blockDim.x / waves;
        const int wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x / nv);
        const int64_t vox = blk * nv + (int) threadIdx.x % nv;
        const bool in = vox < dims.nvox;
        int x = 0, y = 0, z = 0;
        AT acc = AT(0);
        if (in) {
            x = (int) (vox % dims.vol[0]);
            if (YSLOW) {
                z = (int) ((vox / dims.vol[0]) % dims.vol[2]);
                y = (int) (vox / ((int64_t) dims.vol[0] * dims.vol[2]));
            } else {
                y = (int) ((vox / dims.vol[0]) % dims.vol[1]);
                z = (int) (vox / ((int64_t) dims.vol[0] * dims.vol[1]));
            }
            if constexpr (MORE) {
                const int each = parts / waves;
                for (int q = wave * each; q < (wave + 1) * each; ++q) {
                    const AT sum = gather((int) ((int64_t) dims.nposes * q / parts),
                                          (int) ((int64_t) dims.nposes * (q + 1) / parts), x, y, z);
                    acc = q == wave * each ? sum : acc + sum;
                    if (waves > 1)
                        sums[q * nv + (int) threadIdx.x % nv] = sum;
                }
            } else {
                acc = gather((int) ((int64_t) dims.nposes * wave / parts),
                             (int) ((int64_t) dims.nposes * (wave + 1) / parts), x, y, z);
            }
        }
        if (waves > 1) {
            if (!MORE)
                sums[threadIdx.x] = acc;
            __syncthreads();
            if (wave == 0) // whose own parts are added already
                for (int q = MORE ? parts / waves : 1; q < parts; ++q)
                    acc = acc + sums[threadIdx.x + q * nv];
        }
        if (in && wave == 0)
            vol[x + (int64_t) y * dims.strides[1] + (int64_t) z * dims.strides[2]] = down<ST>(acc);
    }

    // The general gather, a loop over the clipped rectangle of every footprint. FP32 tables (at most
    // kVoxMaxLut entries) are read as pairs from LDS.
    template <int D, class ST, class LT, bool YSLOW, bool MORE>
    __device__ __forceinline__ void vox_gather_block(const PoseGeom* __restrict__ geo, const Dims& dims,
                                                     const LT* __restrict__ lut, const int n_lut, const float support,
                                                     const int diff, const int parts, const int waves, const int64_t blk,
                                                     const ST* __restrict__ sino, ST* __restrict__ vol)
    {
        extern __shared__ long long lds[];
        if constexpr (sizeof(LT) == 8) {
            auto gather = [&](int p0, int p1, int x, int y, int z) {
                double acc = 0.0;
                for (int p = p0; p < p1; ++p) {
                    Footprint fp;
                    footprint<D>(geo[p], dims, x, y, z, support, fp);
                    const ST* sp = sino + (int64_t) p * dims.pix_per_pose;
                    visit<D, double>(fp, dims, [&](int64_t pix, float dist, float d0) {
                        acc += tap_weight<D, double>(lut, n_lut, support, dist, d0, diff != 0) * up(sp[pix]);
                    });
                }
                return acc;
            };
            gather_parts<YSLOW, MORE>(dims, parts, waves, blk, reinterpret_cast<double*>(lds), vol, gather);
        } else {
            float* s_lut = reinterpret_cast<float*>(lds);
            for (int i = threadIdx.x; i < lerp_table_size(n_lut); i += blockDim.x)
                lerp_table_entry(lut, n_lut, i, s_lut);
            __syncthreads();
            const float kidx = (float) (n_lut - 1) / support;
            const bool tail_zero = lut[n_lut - 1] == 0.0f;
            auto gather = [&](int p0, int p1, int x, int y, int z) {
                // a table ending in 0 takes tap_weight_fast's TZ form
                auto sum = [&](auto tzc) {
                    constexpr bool TZ = decltype(tzc)::value;
                    float acc = 0.0f;
                    for (int p = p0; p < p1; ++p) {
                        Footprint fp;
                        float rs;
                        footprint_fast<D>(geo[p], dims, x, y, z, support, fp, rs);
                        const float rsk = rs * kidx;
                        const ST* sp = sino + (int64_t) p * dims.pix_per_pose;
                        for (int j = fp.lo[1]; j <= fp.hi[1]; ++j) {
                            const float d1 = D == 3 ? (fp.center[1] - (float) j) * rsk : 0.0f;
                            const float d1s = d1 * d1;
                            float fi = (float) fp.lo[0]; // i as a float (exact), without a conversion per tap
                            for (int i = fp.lo[0]; i <= fp.hi[0]; ++i, fi += 1.0f) {
                                const float d0 = fp.center[0] - fi;
                                // one FMA per tap: the sum of the taps in pose and pixel order, each product
                                // unrounded
                                acc = __builtin_fmaf(
                                    tap_weight_units<D, TZ>(s_lut, n_lut, d0 * rsk, d1s, d0 * rs, diff != 0),
                                    up(sp[(int64_t) j * dims.det[0] + i]), acc);
                            }
                        }
                    }
                    return acc;
                };
                return tail_zero ? sum(std::true_type{}) : sum(std::false_type{});
            };
            float* sums = s_lut + 2 * lerp_table_size(n_lut);
            gather_parts<YSLOW, MORE>(dims, parts, waves, blk, sums, vol, gather);
        }
    }

    // The 3D gather by columns: rows of NC taps in straight code. Columns past the footprint or the detector
    // lie past the table's end and read past the pose's detector (0 by the buffer's bounds), so that
    // they add nothing to the sum, whatever the sinogram holds.
    //
    // Bound by vector instructions (1.17 a cycle and CU) and the L1 (9 accesses a load, 0.75 a cycle): 14
    // wavefront instructions a tap against 19 in the general loops, all of a row's pixels in flight.
    // 131 x 125 x 119 blobs on 193 x 187, 180 poses: 2.29 ms against 3.05 ms; FP64 B-splines 96^3 on
    // 144^2, 90 poses: 1.15 ms against 2.00 ms (two divisions a tap).
    template <int NC, class ST, class LT, int DIFF, bool YSLOW>
    __device__ __forceinline__ void vox_gather_cols_block(const PoseGeom* __restrict__ geo, const Dims& dims,
                                                          const LT* __restrict__ lut, const int n_lut,
                                                          const float support, const int diff, const int parts,
                                                          const int64_t blk, const ST* __restrict__ sino,
                                                          ST* __restrict__ vol)
    {
        constexpr bool F64 = sizeof(LT) == 8;
        constexpr uint32_t es = sizeof(ST);
        constexpr uint32_t kPast = 0x40000000u; // past any detector (pix_per_pose * es < 2^30)
        extern __shared__ long long lds[];
        LT* s_lut = reinterpret_cast<LT*>(lds);
        if constexpr (F64) {
            for (int i = threadIdx.x; i <= n_lut; i += blockDim.x)
                s_lut[i] = i < n_lut ? lut[i] : 0.0;
        } else {
            for (int i = threadIdx.x; i < lerp_table_size(n_lut); i += blockDim.x)
                lerp_table_entry(lut, n_lut, i, s_lut);
        }
        __syncthreads();
        const bool df = DIFF == 1 || (DIFF == 2 && diff);
        const bool tail_zero = lut[n_lut - 1] == LT(0);
        const float kidx = (float) (n_lut - 1) / support;
        const float rsupport = 1.0f / support;
        const uint32_t rowb = (uint32_t) dims.det[0] * es;
        typedef typename std::conditional<F64, double, float>::type AT;
        AT* sums = s_lut + (F64 ? n_lut + 1 : 2 * lerp_table_size(n_lut));
        gather_parts<YSLOW, false, AT>(dims, parts, parts, blk, sums, vol, [&](const int p0, const int p1, int x, int y, int z) {
            auto sum = [&](auto tzc) {
                constexpr bool TZ = decltype(tzc)::value;
                AT acc = AT(0);
                for (int p = p0; p < p1; ++p) {
                    const buf_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
                        const_cast<ST*>(sino + (int64_t) p * dims.pix_per_pose), 0,
                        (int) ((uint32_t) dims.pix_per_pose * es), 0x00020000);
                    Footprint fp;
                    float rs = 0.0f;
                    if constexpr (F64)
                        footprint<3>(geo[p], dims, x, y, z, support, fp);
                    else
                        footprint_fast<3>(geo[p], dims, x, y, z, support, fp, rs);
                    const int lo = fp.lo[0], last = fp.hi[0] - lo;
                    uint32_t off[NC];
                    const uint32_t base = ((uint32_t) fp.lo[1] * (uint32_t) dims.det[0] + (uint32_t) lo) * es;
#pragma unroll
                    for (int i = 0; i < NC; ++i)
                        off[i] = i <= last ? base + i * es : kPast;
                    if constexpr (F64) {
                        const float rsc = 1.0f / fp.scaling;
                        float d0[NC];
                        column_units64<NC>(fp.center[0], lo, fp.hi[0], fp.scaling, rsc, d0);
                        for (int j = fp.lo[1]; j <= fp.hi[1]; ++j) {
                            double w[NC], v[NC];
#pragma unroll
                            for (int i = 0; i < NC; ++i) {
                                v[i] = pixel_load<ST>(rsrc, off[i]);
                                off[i] += rowb;
                            }
                            row_units64<NC>(s_lut, n_lut, support, rsupport, fp.center[1], j, fp.scaling, rsc, d0, df, w);
#pragma unroll
                            for (int i = 0; i < NC; ++i)
                                acc += w[i] * v[i];
                        }
                    } else {
                        const float rsk = rs * kidx;
                        float d0k[NC], du[NC];
                        column_units_clipped<NC>(fp.center[0], lo, last, n_lut, rs, rsk, df, d0k, du);
                        for (int j = fp.lo[1]; j <= fp.hi[1]; ++j) {
                            float w[NC], v[NC];
#pragma unroll
                            for (int i = 0; i < NC; ++i) {
                                v[i] = pixel_load<ST>(rsrc, off[i]);
                                off[i] += rowb;
                            }
                            row_units<NC, TZ>(s_lut, n_lut, fp.center[1], j, rsk, d0k, du, df, w);
#pragma unroll
                            for (int i = 0; i < NC; ++i)
                                acc = __builtin_fmaf(w[i], v[i], acc);
                        }
                    }
                }
                return acc;
            };
            if constexpr (F64)
                return sum(std::false_type{});
            else
                return tail_zero ? sum(std::true_type{}) : sum(std::false_type{});
        });
    }

    // NC 0: the general gather. DIFF: the phase-contrast projectors' weights (a compile-time flag, so
    // that the taps of the others carry no select). split: the parts of a voxel's sum, a wavefront each; MORE: a
    // wavefront takes more than one (gather_waves), their number is in split's upper bits. In 3D the voxels are taken with y slowest and each
    // XCD gets a contiguous run of blocks (consecutive blocks land on different XCDs): a slab of y, whose
    // detector rows over all poses stay in that XCD's L2 when the trajectory turns about y.
    template <int D, int NC, class ST, class LT, int DIFF, bool MORE = false>
    __global__ void __launch_bounds__(kMaxThreads)
        voxel_gather_kernel(const PoseGeom* __restrict__ geo, const Dims dims, const LT* __restrict__ lut,
                            const int n_lut, const float support, const int split, const int per_xcd,
                            const ST* __restrict__ sino, ST* __restrict__ vol)
    {
        const int64_t blk = (int64_t) (blockIdx.x % 8u) * per_xcd + (blockIdx.x / 8u);
        const int parts = MORE ? split & 255 : split, waves = MORE ? split >> 8 : split;
        if (blk * ((int) blockDim.x / waves) >= dims.nvox)
            return; // the whole block
        if constexpr (NC == 0)
            vox_gather_block<D, ST, LT, D == 3, MORE>(geo, dims, lut, n_lut, support, DIFF, parts, waves, blk, sino, vol);
        else
            vox_gather_cols_block<NC, ST, LT, DIFF, true>(geo, dims, lut, n_lut, support, DIFF, parts, blk, sino, vol);
    }

    // the gathers of many operators in one launch (block b: block b - job.block0 of job block_job[b]);
    // NC: the columns of the widest operator's kernel (a wider kernel's extra columns add nothing), 0: the general one
    template <int D, int NC, bool MORE = false>
    __global__ void __launch_bounds__(kMaxThreads)
        voxel_gather_batch_kernel(const VoxAdjJob* __restrict__ jobs, const int* __restrict__ block_job,
                                  const float* __restrict__ sinos, float* __restrict__ vols)
    {
        const VoxAdjJob& J = jobs[block_job[blockIdx.x]];
        const int64_t blk = (int64_t) blockIdx.x - J.block0;
        if constexpr (NC == 0)
            vox_gather_block<D, float, float, false, MORE>(J.geo, J.dims, J.lut, J.n_lut, J.support, J.diff, J.parts,
                                                           MORE ? J.waves : J.parts, blk,
                                                     sinos + J.sino_off, vols + J.vol_off);
        else
            vox_gather_cols_block<NC, float, float, 2, false>(J.geo, J.dims, J.lut, J.n_lut, J.support, J.diff,
                                                              J.parts, blk, sinos + J.sino_off, vols + J.vol_off);
    }

    namespace
    {
        // dynamic LDS: the table and the sums of a block's voxels' parts
        template <class LT>
        size_t gather_lds(int n_lut, bool cols, int parts, int waves, int threads)
        {
            const size_t sums = waves > 1 ? (size_t) threads / waves * parts * sizeof(LT) : 0;
            if (sizeof(LT) == 8)
                return (cols ? (size_t) (n_lut + 1) * 8 : 0) + sums;
            return (size_t) lerp_table_size(n_lut) * 8 + sums;
        }

        // fn(the kernel's column count as a constant)
        template <class Fn>
        void with_columns(int cols, Fn fn)
        {
            switch (cols > 0 ? kernel_cols(cols) : 0) {
                case 0: return fn(std::integral_constant<int, 0>{});
                case 4: return fn(std::integral_constant<int, 4>{});
                case 5: return fn(std::integral_constant<int, 5>{});
                case 6: return fn(std::integral_constant<int, 6>{});
                default: return fn(std::integral_constant<int, 8>{});
            }
        }
    } // namespace

    void voxel_gather_batch_jobs(const VoxBatchItem* items, int n, std::vector<VoxAdjJob>& jobs,
                                 std::vector<int>& blocks, size_t& lds, int& cols, int& threads)
    {
        jobs.clear();
        blocks.clear();
        lds = 0;
        threads = 256;
        for (int j = 0; j < n; ++j) {
            const int t = gather_threads(gather_waves(items[j].dims, items[j].plan.width, false));
            threads = t > threads ? t : threads;
        }
        cols = kVoxMaxCols;
        for (int j = 0; j < n; ++j)
            cols = items[j].plan.cols <= 0 ? 0 : cols;
        if (cols > 0) {
            cols = 0;
            for (int j = 0; j < n; ++j)
                cols = items[j].plan.cols > cols ? items[j].plan.cols : cols;
        }
        for (int j = 0; j < n; ++j) {
            const VoxBatchItem& it = items[j];
            VoxAdjJob J{};
            J.geo = it.geo;
            J.dims = it.dims;
            J.lut = it.lut;
            J.n_lut = it.n_lut;
            J.support = it.support;
            J.diff = it.diff;
            J.parts = gather_part_count(it.dims);
            J.waves = gather_waves(it.dims, it.plan.width, false);
            J.vol_off = it.vol_off;
            J.sino_off = it.sino_off;
            J.block0 = (int64_t) blocks.size();
            const int nv = threads / J.waves;
            blocks.insert(blocks.end(), (size_t) ((it.dims.nvox + nv - 1) / nv), (int) jobs.size());
            jobs.push_back(J);
            if (J.waves < J.parts)
                cols = -1; // the general kernel in any case: its footprints are too wide for columns
            const size_t need = gather_lds<float>(it.n_lut, cols > 0, J.parts, J.waves, threads);
            lds = need > lds ? need : lds;
        }
    }

    hipError_t voxel_gather_batch(int dim, int cols, const VoxAdjJob* jobs, const int* blocks, int64_t nblocks,
                                  size_t lds, int threads, const float* sinos, float* vols, hipStream_t s)
    {
        if (nblocks > 0x7fffffff)
            return hipErrorInvalidValue;
        if (nblocks == 0)
            return hipSuccess;
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned) nblocks), dim3((unsigned) threads), lds, s, jobs, blocks, sinos, vols);
        };
        if (dim == 2)
            launch(voxel_gather_batch_kernel<2, 0>);
        else if (cols < 0)
            launch(voxel_gather_batch_kernel<3, 0, true>);
        else
            with_columns(cols, [&](auto nc) { launch(voxel_gather_batch_kernel<3, decltype(nc)::value>); });
        return hipGetLastError();
    }

    template <class ST, class LT>
    hipError_t voxel_gather(const PoseGeom* geo, const Dims& dims, const LT* lut, int n_lut, float support, int diff,
                            const VoxPlan& plan, const ST* sino, ST* vol, hipStream_t s)
    {
        if (n_lut < 2 || n_lut > kVoxMaxLut)
            return hipErrorInvalidValue;
        const int parts = gather_part_count(dims), waves = gather_waves(dims, plan.width, sizeof(LT) == 8);
        const int threads = gather_threads(waves), nv = threads / waves;
        const int64_t per_xcd = ((dims.nvox + nv - 1) / nv + 7) / 8;
        if (per_xcd * 8 > (int64_t) 0x7fffffff)
            return hipErrorInvalidValue;
        const dim3 grid((unsigned) (per_xcd * 8));
        const int split = waves < parts ? waves << 8 | parts : parts;
        const size_t lds = gather_lds<LT>(n_lut, plan.cols > 0, parts, waves, threads);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3((unsigned) threads), lds, s, geo, dims, lut, n_lut, support, split,
                               (int) per_xcd, sino, vol);
        };
        if (dims.dim == 2) {
            diff ? launch(voxel_gather_kernel<2, 0, ST, LT, 1>) : launch(voxel_gather_kernel<2, 0, ST, LT, 0>);
            return hipGetLastError();
        }
        if constexpr (sizeof(LT) == 4)
            if (waves < parts) { // footprints too wide for columns
                diff ? launch(voxel_gather_kernel<3, 0, ST, LT, 1, true>) : launch(voxel_gather_kernel<3, 0, ST, LT, 0, true>);
                return hipGetLastError();
            }
        with_columns(plan.cols, [&](auto nc) {
            constexpr int NC = decltype(nc)::value;
            diff ? launch(voxel_gather_kernel<3, NC, ST, LT, 1>) : launch(voxel_gather_kernel<3, NC, ST, LT, 0>);
        });
        return hipGetLastError();
    }

    template hipError_t voxel_gather<float, float>(const PoseGeom*, const Dims&, const float*, int, float, int,
                                                   const VoxPlan&, const float*, float*, hipStream_t);
    template hipError_t voxel_gather<bf16, float>(const PoseGeom*, const Dims&, const float*, int, float, int,
                                                  const VoxPlan&, const bf16*, bf16*, hipStream_t);
    template hipError_t voxel_gather<double, double>(const PoseGeom*, const Dims&, const double*, int, float, int,
                                                     const VoxPlan&, const double*, double*, hipStream_t);
} // namespace ehp
