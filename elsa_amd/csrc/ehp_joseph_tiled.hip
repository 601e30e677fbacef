// ehp_joseph_tiled.hip -- Joseph back projection with LDS-privatised volume tiles (FP32).
//
// The matched adjoint of the Joseph forward (elsa/projectors/JosephsMethod.cpp:140-198,
// adjoint branch :180-186) without global atomics. The volume is cut into tiles that are
// long along one driving axis a (LA planes) and TB x TC voxels across. One workgroup owns a
// tile for all poses: it accumulates in LDS every sample of every ray whose driving axis is
// a and whose bilinear footprint touches the tile, then adds the tile to the volume once.
// Each voxel is owned by exactly one tile per driving axis that occurs in the trajectory. With two
// such axes, as about any axis of rotation, and rays enough to pay for it (pair_launch), one launch runs the
// tiles of both (joseph_adj_pair_kernel: a voxel gets two sums, added by whichever workgroup comes second);
// otherwise one launch per axis adds to the volume in plain read-modify-write. In 2D a tile takes the rays of both axes
// (adj2d_block) and one launch writes the volume.
//
// Accumulation: LDS float atomics are slow on this part (a ds_add_f32 wave operation costs
// about 15 times a ds_add_u64), so the tile is summed with 64-bit integer atomics in fixed
// point: units of q = 2^(eg - 62), eg chosen per call from max|y| and a bound on what one slot
// can receive, so that no sum can overflow, each contribution rounded once (fixed_round). Integer sums do not depend on the order of the additions, so the result is
// bitwise reproducible, whatever the tile shape, and more accurate than a sequential FP32
// accumulation. A non-finite y makes the whole output NaN (the fixed-point sums cannot carry
// it to just the voxels it touches).
//
// The per-ray state comes from a table built once per operator from the same functions as
// the one-thread-per-ray kernels (make_ray, joseph_setup), and the per-sample weights use the
// same arithmetic as joseph_sample, so they are bit-identical to the forward's.
#include "ehp_kernels.hpp"
#include "ehp_last_block.hpp"
#include "ehp_tile_pair.hpp"

#include <type_traits>

namespace ehp
{
    namespace
    {
        constexpr int kThreads = 512; // of the 3D back projection's workgroups
        // LDS (address space 3) pointers: 32-bit byte addresses
        typedef __attribute__((address_space(3))) unsigned long long lds_u64;
        typedef __attribute__((address_space(3))) char lds_char;
    } // namespace

    // ---------------------------------------------------------------------------------
    // per-ray table

    template <int D>
    __global__ void __launch_bounds__(256)
        joseph_ray_table_kernel(const PoseGeom* __restrict__ geo, const Dims dims, RayRec* __restrict__ table)
    {
        const int pose = blockIdx.y;
        const int64_t pix = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
        if (pix >= dims.pix_per_pose)
            return;
        const int u = (int) (pix % dims.det[0]);
        const int v = (int) (pix / dims.det[0]);
        float o[3], d[3];
        make_ray_px<D>(geo[pose], dims, u, v, o, d);
        JRay jr;
        joseph_setup<D>(o, d, dims.vol, jr);
        table[(int64_t) pose * dims.pix_per_pose + pix] = make_ray_rec<D>(jr);
    }

    hipError_t joseph_ray_table(const PoseGeom* geo, const Dims& dims, RayRec* table, hipStream_t s)
    {
        const dim3 grid((unsigned) ((dims.pix_per_pose + 255) / 256), (unsigned) dims.nposes);
        if (dims.dim == 2)
            hipLaunchKernelGGL((joseph_ray_table_kernel<2>), grid, dim3(256), 0, s, geo, dims, table);
        else
            hipLaunchKernelGGL((joseph_ray_table_kernel<3>), grid, dim3(256), 0, s, geo, dims, table);
        return hipGetLastError();
    }

    // ---------------------------------------------------------------------------------
    // fixed-point scale of one back projection

    // Largest |y| in two stages: each block writes the maximum of its share as the bit pattern of
    // |y| (for non-negative floats, and NaN above infinity, the integer order of the bits is the
    // order of the values), the block that finishes last (counts_last) reduces those.
    template <class U>
    __device__ inline U block_max_bits(U m)
    {
        for (int off = 32; off > 0; off >>= 1) {
            const U o = __shfl_down(m, off, 64);
            m = o > m ? o : m;
        }
        __shared__ U red[16]; // at most 1024 threads
        if ((threadIdx.x & 63) == 0)
            red[threadIdx.x >> 6] = m;
        __syncthreads();
        if (threadIdx.x == 0)
            for (int w = 1; w < (int) (blockDim.x >> 6); ++w)
                m = red[w] > m ? red[w] : m;
        return m; // valid in thread 0
    }

    // Bit pattern of |x| (FP32 and bfloat16: of its FP32 value), whose integer order is the values'
    template <class T>
    __device__ __forceinline__ auto abs_bits(T x)
    {
        if constexpr (sizeof(T) == 8)
            return (unsigned long long) __double_as_longlong(fabs(x));
        else
            return __float_as_uint(fabsf(up(x)));
    }

    __device__ inline double bits_value(unsigned int u) { return __uint_as_float(u); }
    __device__ inline double bits_value(unsigned long long u) { return __longlong_as_double((long long) u); }

    // Max of the |x| bits over a thread's share of n elements (thread t of threads): 16 bytes at a time,
    // four of them in flight, from the first aligned element on.
    template <class T>
    __device__ __forceinline__ auto max_share(const T* __restrict__ x, int64_t n, int64_t t, int64_t threads)
    {
        using U = decltype(abs_bits(x[0]));
        constexpr int W = 16 / sizeof(T);
        struct alignas(16) Vec {
            T v[W];
        };
        U m = 0;
        auto take = [&](T v) {
            const U u = abs_bits(v);
            m = u > m ? u : m;
        };
        int64_t head = (int64_t) ((16u - (uint32_t) (uintptr_t) x % 16u) % 16u / sizeof(T));
        head = head < n ? head : n;
        const int64_t nvec = (n - head) / W, tail = head + nvec * W;
        if (t < head)
            take(x[t]);
        if (t < n - tail)
            take(x[tail + t]);
        const Vec* xv = reinterpret_cast<const Vec*>(x + head);
        int64_t i = t;
        for (; i + 3 * threads < nvec; i += 4 * threads) {
            const Vec a = xv[i], b = xv[i + threads], c = xv[i + 2 * threads], d = xv[i + 3 * threads];
#pragma unroll
            for (int k = 0; k < W; ++k) {
                take(a.v[k]);
                take(b.v[k]);
                take(c.v[k]);
                take(d.v[k]);
            }
        }
        for (; i < nvec; i += threads) {
            const Vec a = xv[i];
#pragma unroll
            for (int k = 0; k < W; ++k)
                take(a.v[k]);
        }
        return m;
    }

    // fixexp[0] = the fixed-point exponent eg for the slot bound of the operator. Each block reduces its
    // share of x; the block that finishes last (fixexp[1] counts them, wraps and so is 0 between launches)
    // reduces the blocks' maxima, so that the exponent takes one launch. A block's count releases its
    // maximum to the other XCDs, which costs more than a small block's share: at most one block a CU, of 1024
    // threads. 6.6 million FP32 values: 43 us with 1620 blocks of 256 threads and 4-byte loads, 10.7 with 256
    // blocks, 8.6 with 128; 53 million 106, 44.5, 49.6.
    template <class T>
    __global__ void __launch_bounds__(1024)
        absmax_scale_kernel(const T* __restrict__ x, int64_t n, double bound, unsigned long long* __restrict__ partial,
                            int* __restrict__ fixexp)
    {
        using U = decltype(abs_bits(x[0]));
        U m = max_share(x, n, (int64_t) blockIdx.x * blockDim.x + threadIdx.x, (int64_t) gridDim.x * blockDim.x);
        m = block_max_bits(m);
        __shared__ bool last;
        if (gridDim.x > 1) {
            if (threadIdx.x == 0) {
                __hip_atomic_store(partial + blockIdx.x, (unsigned long long) m, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
                last = counts_last(reinterpret_cast<unsigned int*>(fixexp + 1), gridDim.x);
            }
            __syncthreads();
            if (!last)
                return;
            m = 0;
            for (int i = threadIdx.x; i < (int) gridDim.x; i += blockDim.x) {
                const U u = (U) __hip_atomic_load(partial + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                m = u > m ? u : m;
            }
            __syncthreads(); // block_max_bits' LDS is read again
            m = block_max_bits(m);
        }
        if (threadIdx.x == 0)
            fixexp[0] = fixed_point_exponent(bits_value(m), bound);
    }

    // d_maxbits holds kAbsmaxBlocks 64-bit partial maxima, d_fixexp the exponent and a counter that is
    // 0 between launches
    template <class T>
    hipError_t fixed_point_exponent_launch(const T* y, int64_t n, double slot_bound, unsigned int* d_maxbits,
                                           int* d_fixexp, hipStream_t s)
    {
        // 16 elements per thread at least, past 16 blocks 64
        int64_t blocks = (n + 1024 * 16 - 1) / (1024 * 16);
        if (blocks > 16)
            blocks = n / (1024 * 64) > 16 ? n / (1024 * 64) : 16;
        blocks = blocks > kAbsmaxBlocks ? kAbsmaxBlocks : (blocks < 1 ? 1 : blocks);
        hipLaunchKernelGGL((absmax_scale_kernel<T>), dim3((unsigned) blocks), dim3(1024), 0, s, y, n, slot_bound,
                           reinterpret_cast<unsigned long long*>(d_maxbits), d_fixexp);
        return hipGetLastError();
    }

    template hipError_t fixed_point_exponent_launch<float>(const float*, int64_t, double, unsigned int*, int*,
                                                           hipStream_t);
    template hipError_t fixed_point_exponent_launch<bf16>(const bf16*, int64_t, double, unsigned int*, int*,
                                                          hipStream_t);
    template hipError_t fixed_point_exponent_launch<double>(const double*, int64_t, double, unsigned int*, int*,
                                                            hipStream_t);

    // ---------------------------------------------------------------------------------
    // the tiled back projection

    // The ray value in units of the fixed-point unit q = 2^(eg - 62): FP64 y * len as elsa's FP64
    // operator forms it, else elsa's FP32 product (both scaled by a power of two, exactly).
    template <class YT>
    __device__ __forceinline__ double ray_units(YT yv, float len, int eg)
    {
        if constexpr (sizeof(YT) == 8)
            return ldexp(yv * (double) len, 62 - eg);
        else
            return ldexp((double) (yv * len), 62 - eg);
    }

    __device__ __forceinline__ void lds_add(uint32_t off, unsigned long long v)
    {
        __hip_atomic_fetch_add((lds_u64*) (uintptr_t) off, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    // The candidate rays of one pose batch of one 3D tile, all added into the tile's slots.
    // Candidate k (k < total) is pixel k - pref[j] of pose j's rectangle, j the last pose with
    // pref[j] <= k. Each lane walks its candidates k = tid, tid + kThreads, ... in order, so it keeps
    // its pose j (and j's rectangle) in registers and moves on when k passes pref[j + 1]. The
    // ray state and y of the next candidate are loaded while the current one is added (two
    // register sets taken in turn).
    template <int A, bool LOW, class ST>
    __device__ __forceinline__ void adj_tile_batch(const RayRec* __restrict__ table, const ST* __restrict__ sino,
                                                   const int det0, const CandRect* s_rect, const int* s_pref,
                                                   const int total, const TileBox& t, const TileOff& to,
                                                   const int eg)
    {
        using YT = typename Acc<ST>::type; // FP64 for FP64 sinograms, else FP32
        const int tid = threadIdx.x;
        int j = 0, pj = 0, pn = s_pref[1];
        CandRect cr = s_rect[0];
        auto fetch = [&](int k, RayRec& r, YT& yv) {
            while (k >= pn) {
                ++j;
                pj = pn;
                pn = s_pref[j + 1];
                cr = s_rect[j];
            }
            int row, col;
            rect_split(k - pj, cr.nu, cr.rnu, row, col);
            const int64_t ray = cr.base + (int64_t) (mul24((uint32_t) row, (uint32_t) det0) + (uint32_t) col);
            yv = up(sino[ray]);
            r = table[ray];
        };
        auto process = [&](const RayRec& r, YT yv) {
            const double yq = ray_units(yv, r.len, eg);
            if constexpr (sizeof(YT) == 8) {
                // FP64: each contribution is elsa's (y * len) * weight in FP64 (the weight in FP32,
                // as the one-thread-per-ray FP64 kernel forms it), rounded to the nearest multiple of
                // q; yq is y * len in units of q (a power-of-two scaling, exact)
                tile_candidate_fx<3, A, LOW, TAP_WEIGHT>(
                    r, t, to, yq, [&](uint32_t off, float w) { lds_add(off, fixed_round(yq, (double) w)); });
            } else {
                // FP32 (and bfloat16, widened): elsa's FP32 product y * len in units of q (exact),
                // times the exact weights, rounded once to the nearest multiple of q
                // off: the slot's LDS byte address (the tile's base included)
                tile_candidate_fx<3, A, LOW, TAP_FIXED>(r, t, to, yq, lds_add);
            }
        };
        RayRec ra{}, rb{};
        YT ya = 0, yb = 0;
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
    }

    // ---------------------------------------------------------------------------------
    // 2D: a workgroup owns LA x TB voxels (x by y) for the rays of both driving axes, each with its own
    // slots, and writes each voxel once: one launch per back projection, with no volume to clear and
    // none to add to. Few rays of a pose meet a tile, so one step takes many poses at once; while a
    // launch has few tiles its workgroups are large, as nothing but the number of
    // wavefronts per tile hides the latency of the ray table and the LDS. Latency bounds the small
    // problems, the 64-bit LDS atomics and VALU the large ones. Against one launch per axis over 4 x 15 tiles (the pass with the
    // exponent's launch): 64^2 / 90 poses 42 -> 19 us, 256^2 / 180 73 -> 34, 512^2 / 360 309 -> 109; 64 problems
    // of 128^2..512^2 in one launch 4635 -> 1129 us.

    template <int NT, class ST>
    __device__ __forceinline__ void adj2d_block(const PoseGeom* __restrict__ geo, const RayRec* __restrict__ table,
                                                const Dims& dims, const int* __restrict__ pose_axes, const TileCfg& tc,
                                                const int ntx, const int tile, const int steps, const int eg,
                                                const ST* __restrict__ sino, typename Acc<ST>::type* __restrict__ vol)
    {
        using YT = typename Acc<ST>::type;
        extern __shared__ long long lds[];
        const int tid = threadIdx.x;
        const int ix = tile % ntx, iy = tile / ntx;
        const TileBox t0 = make_tile<2, 0>(dims, tc, ix, iy, 0);
        const TileBox t1 = make_tile<2, 1>(dims, TileCfg{tc.TB, tc.LA, 1}, iy, ix, 0);
        const uint32_t lds0 = (uint32_t) (uintptr_t) (lds_char*) lds;
        const TileOff o0 = tile_offsets(t0, lds0), o1 = tile_offsets(t1, lds0 + 8u * (uint32_t) t0.nslots);
        Rays2d* rays = reinterpret_cast<Rays2d*>(lds + t0.nslots + t1.nslots);
        for (int i = tid; i < t0.nslots + t1.nslots; i += NT)
            lds[i] = 0;
        const bool low = tile_low_face<2>(t0) || tile_low_face<2>(t1);

        for (int pbase = 0; eg != kNonFinite && pbase < dims.nposes; pbase += steps) {
            __syncthreads();
            for (int i = tid; i < steps; i += NT) {
                const int p = pbase + i;
                int u0 = dims.det[0], u1 = -1;
                if (p < dims.nposes) {
                    int a0, a1, v0, v1;
                    if ((pose_axes[p] & 1) && tile_bbox<2, 0>(geo[p], t0, dims, a0, a1, v0, v1)) {
                        u0 = a0;
                        u1 = a1;
                    }
                    if ((pose_axes[p] & 2) && tile_bbox<2, 1>(geo[p], t1, dims, a0, a1, v0, v1)) {
                        u0 = a0 < u0 ? a0 : u0;
                        u1 = a1 > u1 ? a1 : u1;
                    }
                }
                rays[i].base = (long long) p * dims.pix_per_pose + u0;
                rays[i].cnt = u1 >= u0 ? u1 - u0 + 1 : 0;
            }
            __syncthreads();
            if (tid < 64) {
                // exclusive prefix of the counts, kPoses2d / 64 consecutive ones a lane
                constexpr int per = kPoses2d / 64;
                int sum = 0;
                for (int i = 0; i < per; ++i)
                    sum += tid * per + i < steps ? rays[tid * per + i].cnt : 0;
                int pre = sum;
                for (int o = 1; o < 64; o <<= 1) {
                    const int v = __shfl_up(pre, o, 64);
                    pre += tid >= o ? v : 0;
                }
                pre -= sum;
                for (int i = 0; i < per; ++i)
                    if (tid * per + i < steps) {
                        rays[tid * per + i].pref = pre;
                        pre += rays[tid * per + i].cnt;
                    }
                if (tid == 63)
                    rays[steps].pref = pre;
            }
            __syncthreads();
            const int total = rays[steps].pref;
            // ray k is pixel k - pref[j] of pose j's pixels, j the last pose with pref[j] <= k; each lane
            // takes k = tid, tid + NT, ... in order, keeping j in registers
            int j = 0, pj = 0, pn = rays[1].pref;
            int64_t base = rays[0].base;
            auto fetch = [&](int k, RayRec& r, YT& yv) {
                while (k >= pn) {
                    ++j;
                    pj = pn;
                    pn = rays[j + 1].pref;
                    base = rays[j].base;
                }
                const int64_t ray = base + (k - pj);
                yv = up(sino[ray]);
                r = table[ray];
            };
            auto walk = [&](auto lw) {
                constexpr bool LOW = decltype(lw)::value;
                auto process = [&](const RayRec& r, YT yv) {
                    const double yq = ray_units(yv, r.len, eg);
                    if constexpr (sizeof(YT) == 8) {
                        auto add = [&](uint32_t off, float w) { lds_add(off, fixed_round(yq, (double) w)); };
                        if ((r.meta & 3) == 0)
                            tile_candidate_fx<2, 0, LOW, TAP_WEIGHT>(r, t0, o0, yq, add);
                        else
                            tile_candidate_fx<2, 1, LOW, TAP_WEIGHT>(r, t1, o1, yq, add);
                    } else if ((r.meta & 3) == 0) {
                        tile_candidate_fx<2, 0, LOW, TAP_FIXED>(r, t0, o0, yq, lds_add);
                    } else {
                        tile_candidate_fx<2, 1, LOW, TAP_FIXED>(r, t1, o1, yq, lds_add);
                    }
                };
                RayRec ra{}, rb{};
                YT ya = 0, yb = 0;
                if (tid < total)
                    fetch(tid, ra, ya);
                for (int k = tid; k < total; k += 2 * NT) {
                    const int k1 = k + NT, k2 = k + 2 * NT;
                    if (k1 < total)
                        fetch(k1, rb, yb);
                    process(ra, ya);
                    if (k2 < total)
                        fetch(k2, ra, ya);
                    if (k1 < total)
                        process(rb, yb);
                }
            };
            if (low)
                walk(TagTrue{});
            else
                walk(TagFalse{});
        }
        __syncthreads();

        // the voxels: the sum of both axes' slots (each axis keeps its own halo)
        const double q = eg == kNonFinite ? __longlong_as_double(0x7ff8000000000000ll) : ldexp(1.0, eg - 62);
        const int nx = t0.A1 - t0.A0, ny = t0.B1 - t0.B0;
        for (int i = tid; i < nx * ny; i += NT) {
            const int x = i % nx, y = i / nx;
            const long long sum = lds[x * t0.PB + y + 1] + lds[t0.nslots + y * t1.PB + x + 1];
            vol[(int64_t) (t0.B0 + y) * dims.strides[1] + t0.A0 + x] = (YT) ((double) sum * q);
        }
    }

    // OWN: every workgroup finds the exponent itself from the whole sinogram, instead of reading it from
    // fixexp after a launch in the chain. Up to this many rays that is faster (the pass, us with the
    // launch / without): 64^2 / 90 poses (8190 rays) 19.0 / 15.8, 100^2 / 100 (14100) 20.6 / 18.4, 128^2 /
    // 180 (32760) 26.0 / 23.7.
    constexpr int64_t kOwnExponent = 32768;

    template <int NT, class ST, bool OWN>
    __global__ void __launch_bounds__(NT)
        joseph_adj2d_kernel(const PoseGeom* __restrict__ geo, const RayRec* __restrict__ table, const Dims dims,
                            const int* __restrict__ pose_axes, const TileCfg tc, const int ntx, const int steps,
                            const int* __restrict__ fixexp, const double bound, const ST* __restrict__ sino,
                            typename Acc<ST>::type* __restrict__ vol)
    {
        int eg;
        if constexpr (OWN) {
            __shared__ int s_eg;
            const auto m = block_max_bits(max_share(sino, dims.nrays, threadIdx.x, NT));
            if (threadIdx.x == 0)
                s_eg = fixed_point_exponent(bits_value(m), bound);
            __syncthreads();
            eg = s_eg;
        } else {
            eg = fixexp[0];
        }
        adj2d_block<NT, ST>(geo, table, dims, pose_axes, tc, ntx, (int) blockIdx.x, steps, eg, sino, vol);
    }

    // the tiles of many 2D operators in one launch (block b: tile b - job.block0 of job block_job[b])
    __global__ void __launch_bounds__(256)
        joseph_adj2d_batch_kernel(const AdjJob* __restrict__ jobs, const int* __restrict__ block_job,
                                  const int per_xcd, const int64_t total, const int* __restrict__ fixexp,
                                  const float* __restrict__ sinos, float* __restrict__ vols)
    {
        const int64_t id = (int64_t) (blockIdx.x % 8u) * per_xcd + (blockIdx.x / 8u);
        if (id >= total)
            return;
        const AdjJob& J = jobs[block_job[id]];
        adj2d_block<256, float>(J.geo, J.table, J.dims, J.pose_axes, J.tc, J.ntA, (int) (id - J.block0), J.batch,
                                fixexp[J.item], sinos + J.sino_off, vols + J.vol_off);
    }

    // One tile of the back projection along driving axis A (tile < ntA * ntB * ntC).
    template <int D, int A, bool PAIR, class ST = float>
    __device__ __forceinline__ void adj_tiled_block(const PoseGeom* __restrict__ geo,
                                                    const RayRec* __restrict__ table, const Dims& dims,
                                                    const int* __restrict__ pose_axes, const TileCfg& tc,
                                                    const int ntA, const int ntB, const int tile, const int batch,
                                                    const int* __restrict__ fixexp, const ST* __restrict__ sino,
                                                    typename Acc<ST>::type* __restrict__ vol)
    {
        extern __shared__ long long lds[];

        const int tid = threadIdx.x;
        const TileBox t = make_tile<D, A>(dims, tc, tile % ntA, (tile / ntA) % ntB, tile / (ntA * ntB));
        const TileOff to = tile_offsets(t, (uint32_t) (uintptr_t) (lds_char*) lds);
        const bool low = tile_low_face<D>(t);
        long long* iacc = lds;
        const BatchLds bl = batch_lds(lds, t.nslots, batch);
        CandRect* s_rect = bl.rect;
        int *s_cnt = bl.cnt, *s_pref = bl.pref;
        for (int i = tid; i < t.nslots; i += kThreads)
            iacc[i] = 0;
        const int eg = fixexp[0];
        __syncthreads();

        for (int pbase = 0; eg != kNonFinite && pbase < dims.nposes; pbase += batch) {
            if (tid < batch) {
                const int p = pbase + tid;
                int u0 = 0, u1 = -1, v0 = 0, v1 = -1;
                int cnt = 0;
                if (p < dims.nposes && (pose_axes[p] & (1 << A))) {
                    if (tile_bbox<D, A>(geo[p], t, dims, u0, u1, v0, v1))
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
            if (low)
                adj_tile_batch<A, true>(table, sino, dims.det[0], s_rect, s_pref, total, t, to, eg);
            else
                adj_tile_batch<A, false>(table, sino, dims.det[0], s_rect, s_pref, total, t, to, eg);
            __syncthreads();
        }

        // add the owned voxels of the tile to the volume (PAIR: the other axis' tiles may add theirs now)
        const double q = eg == kNonFinite ? __longlong_as_double(0x7ff8000000000000ll) : ldexp(1.0, eg - 62);
        for (int i = tid; i < t.nslots; i += kThreads) {
            const int64_t lin = tile_slot_voxel<D, A>(t, dims, i);
            if (lin < 0)
                continue;
            const typename Acc<ST>::type sum = (typename Acc<ST>::type) ((double) iacc[i] * q);
            if (PAIR)
                add_second(vol + lin, sum);
            else
                vol[lin] += sum;
        }
    }

    template <int D, int A, class ST>
    __global__ void __launch_bounds__(kThreads, 8)
        joseph_adj_tiled_kernel(const PoseGeom* __restrict__ geo, const RayRec* __restrict__ table, const Dims dims,
                                const int* __restrict__ pose_axes, const TileCfg tc, const int ntA, const int ntB,
                                const int ntC, const int tiles_per_xcd, const int batch,
                                const int* __restrict__ fixexp, const ST* __restrict__ sino,
                                typename Acc<ST>::type* __restrict__ vol)
    {
        // consecutive workgroups land on different XCDs: give each XCD a contiguous block of tiles
        const int tile = (int) (blockIdx.x % 8u) * tiles_per_xcd + (int) (blockIdx.x / 8u);
        if (tile >= ntA * ntB * ntC)
            return;
        adj_tiled_block<D, A, false, ST>(geo, table, dims, pose_axes, tc, ntA, ntB, tile, batch, fixexp, sino, vol);
    }

    // One launch leaves the device waiting for its last workgroups once instead of twice. Bound by the
    // LDS and VALU together (64-bit atomics, four a sample: the LDS is busy 0.97 of the time, vector
    // instructions 0.85 a cycle and CU), close to the card's power limit: after it the next kernel's clock is a few
    // percent lower. Workgroups of 512 threads in 64 VGPRs over tiles of 8 x 26 x 26 (53 KB of LDS: three of them,
    // 24 wavefronts, a CU) or 4 x 32 x 32 and less (four, 32 wavefronts), against one launch of 256 threads per axis over 8 x 17 x 17 and 4 x 17 x 17 tiles:
    // 256^3 / 360 poses 8.9 -> 8.0 ms, 192^3 / 270 3.05 -> 2.56, 128^3 / 180 0.79 -> 0.61, 96^3 / 120 0.33 -> 0.23,
    // 64^3 / 90 0.142 -> 0.081, FP64 97 x 61 x 113 / 77 0.195 -> 0.17.
    template <int A0, int A1, class ST>
    __global__ void __launch_bounds__(kThreads, 8)
        joseph_adj_pair_kernel(const PoseGeom* __restrict__ geo, const RayRec* __restrict__ table, const Dims dims,
                               const int* __restrict__ pose_axes, const TileCfg tc, const TileCounts c0,
                               const TileCounts c1, const int batch, const int* __restrict__ fixexp,
                               const ST* __restrict__ sino, typename Acc<ST>::type* __restrict__ vol)
    {
        const int xcd = (int) (blockIdx.x % 8u), k = (int) (blockIdx.x / 8u);
        if (k < c0.per_xcd) {
            const int tile = xcd * c0.per_xcd + k;
            if (tile < c0.n)
                adj_tiled_block<3, A0, true, ST>(geo, table, dims, pose_axes, tc, c0.nA, c0.nB, tile, batch, fixexp,
                                                 sino, vol);
        } else {
            const int tile = xcd * c1.per_xcd + k - c0.per_xcd;
            if (tile < c1.n)
                adj_tiled_block<3, A1, true, ST>(geo, table, dims, pose_axes, tc, c1.nA, c1.nB, tile, batch, fixexp,
                                                 sino, vol);
        }
    }

    // the tiles of axis A of many operators in one launch (block b: tile b - job.block0 of job
    // block_job[b])
    template <int A, bool PAIR>
    __device__ __forceinline__ void adj_batch_block(const AdjJob* __restrict__ jobs, const int* __restrict__ block_job,
                                                    const int64_t id, const int* __restrict__ fixexp,
                                                    const float* __restrict__ sinos, float* __restrict__ vols)
    {
        const AdjJob& J = jobs[block_job[id]];
        adj_tiled_block<3, A, PAIR, float>(J.geo, J.table, J.dims, J.pose_axes, J.tc, J.ntA, J.ntB,
                                           (int) (id - J.block0), J.batch, fixexp + J.item, sinos + J.sino_off,
                                           vols + J.vol_off);
    }

    template <int A>
    __global__ void __launch_bounds__(kThreads, 8)
        joseph_adj_tiled_batch_kernel(const AdjJob* __restrict__ jobs, const int* __restrict__ block_job,
                                      const int per_xcd, const int64_t total, const int* __restrict__ fixexp,
                                      const float* __restrict__ sinos, float* __restrict__ vols)
    {
        const int64_t id = (int64_t) (blockIdx.x % 8u) * per_xcd + (blockIdx.x / 8u);
        if (id < total)
            adj_batch_block<A, false>(jobs, block_job, id, fixexp, sinos, vols);
    }

    template <int A0, int A1>
    __global__ void __launch_bounds__(kThreads, 8)
        joseph_adj_pair_batch_kernel(const BatchTiles<AdjJob> t0, const BatchTiles<AdjJob> t1, const int* __restrict__ fixexp,
                                     const float* __restrict__ sinos, float* __restrict__ vols)
    {
        const int64_t xcd = blockIdx.x % 8u;
        const int k = (int) (blockIdx.x / 8u);
        if (k < t0.per_xcd) {
            const int64_t id = xcd * t0.per_xcd + k;
            if (id < t0.total)
                adj_batch_block<A0, true>(t0.jobs, t0.block_job, id, fixexp, sinos, vols);
        } else {
            const int64_t id = xcd * t1.per_xcd + k - t0.per_xcd;
            if (id < t1.total)
                adj_batch_block<A1, true>(t1.jobs, t1.block_job, id, fixexp, sinos, vols);
        }
    }

    // max|y| per operator of a batch: block b writes the maximum of its share of segment
    // block_seg[b] to partial[b]; then one block per segment reduces its partials
    __global__ void __launch_bounds__(256)
        absmax_batch_kernel(const float* __restrict__ y, const SegJob* __restrict__ segs,
                            const int* __restrict__ block_seg, unsigned int* __restrict__ partial)
    {
        const SegJob& S = segs[block_seg[blockIdx.x]];
        const int64_t b = (int64_t) blockIdx.x - S.block0;
        unsigned int m = 0u;
        const int64_t stride = (int64_t) S.nblocks * 256;
        for (int64_t i = b * 256 + threadIdx.x; i < S.n; i += stride) {
            const unsigned int u = __float_as_uint(fabsf(y[S.off + i]));
            m = u > m ? u : m;
        }
        m = block_max_bits(m);
        if (threadIdx.x == 0)
            partial[blockIdx.x] = m;
    }

    __global__ void __launch_bounds__(256)
        scale_batch_kernel(const unsigned int* __restrict__ partial, const SegJob* __restrict__ segs,
                           const double* __restrict__ bounds, int* __restrict__ fixexp)
    {
        const int j = blockIdx.x;
        const SegJob& S = segs[j];
        unsigned int m = 0u;
        for (int i = threadIdx.x; i < S.nblocks; i += blockDim.x) {
            const unsigned int u = partial[S.block0 + i];
            m = u > m ? u : m;
        }
        m = block_max_bits(m);
        if (threadIdx.x == 0)
            fixexp[j] = fixed_point_exponent(__uint_as_float(m), bounds[j]);
    }

    // Which driving axes occur among the rays of each pose (bit a set when some ray that hits
    // the volume drives along a).
    __global__ void __launch_bounds__(256)
        pose_axes_kernel(const RayRec* __restrict__ table, const Dims dims, int* __restrict__ pose_axes)
    {
        const int pose = blockIdx.y;
        const int64_t pix = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
        if (pix >= dims.pix_per_pose)
            return;
        const RayRec r = table[(int64_t) pose * dims.pix_per_pose + pix];
        if (r.nsteps > 0)
            atomicOr(pose_axes + pose, 1 << (r.meta & 3));
    }

    hipError_t joseph_pose_axes(const RayRec* table, const Dims& dims, int* pose_axes, hipStream_t s)
    {
        hipError_t e = launch_fill<int>(pose_axes, dims.nposes, 0, s);
        if (e != hipSuccess)
            return e;
        const dim3 grid((unsigned) ((dims.pix_per_pose + 255) / 256), (unsigned) dims.nposes);
        hipLaunchKernelGGL(pose_axes_kernel, grid, dim3(256), 0, s, table, dims, pose_axes);
        return hipGetLastError();
    }

    size_t joseph_tile_lds_bytes(const Dims& dims, const TileCfg& tc, int batch)
    {
        const int PC = dims.dim == 3 ? tc.TC + 2 : 1;
        return (size_t) tc.LA * PC * tile_row_slots(dims.dim, tc) * sizeof(long long) + batch_lds_bytes(batch);
    }

    // ST: the sinogram's storage type (float, or bf16 for bfloat16 operators); the volume is
    // FP32 either way.
    template <class ST>
    hipError_t joseph_adjoint_tiled(const PoseGeom* geo, const RayRec* table, const Dims& dims, const int* pose_axes,
                                    int axes_present, const TileCfg& tc, int batch, double slot_bound, double wait,
                                    unsigned int* d_maxbits, int* d_fixexp, const ST* sino,
                                    typename Acc<ST>::type* vol, hipStream_t s)
    {
        using VT = typename Acc<ST>::type;
        if (batch < 1 || batch > kMaxPoseBatch)
            return hipErrorInvalidValue;
        auto exponent = [&] {
            return fixed_point_exponent_launch(sino, dims.nrays, slot_bound, d_maxbits, d_fixexp, s);
        };
        hipError_t e = hipSuccess;
        if (dims.dim == 2) {
            const TileCfg t = tile2d(tc);
            const int ntx = (dims.vol[0] + t.LA - 1) / t.LA;
            const int64_t tiles = (int64_t) ntx * ((dims.vol[1] + t.TB - 1) / t.TB);
            if (tiles > 0x7fffffff)
                return hipErrorInvalidValue;
            const int steps = steps2d(dims, batch);
            const size_t lds = lds2d(t, steps);
            // up to two tiles per CU: large workgroups
            const int nt = tiles <= 512 ? 1024 : 256;
            const bool own = nt == 1024 && dims.nrays <= kOwnExponent && lds + 1024 <= 65536;
            if (!own) {
                e = exponent();
                if (e != hipSuccess)
                    return e;
            }
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3((unsigned) tiles), dim3((unsigned) nt), lds, s, geo, table, dims,
                                   pose_axes, t, ntx, steps, d_fixexp, slot_bound, sino, vol);
            };
            if (own)
                launch(joseph_adj2d_kernel<1024, ST, true>);
            else if (nt == 1024)
                launch(joseph_adj2d_kernel<1024, ST, false>);
            else
                launch(joseph_adj2d_kernel<256, ST, false>);
            return hipGetLastError();
        }
        e = exponent();
        if (e != hipSuccess)
            return e;
        e = launch_fill<VT>(vol, dims.nvox, VT(0), s);
        if (e != hipSuccess)
            return e;
        const size_t lds = joseph_tile_lds_bytes(dims, tc, batch);
        if (pair_launch(axes_present, dims.nvox, wait)) {
            with_axis_pair(axes_present, [&](auto a0, auto a1) {
                const TileCounts c0 = axis_tiles(dims, tc, a0), c1 = axis_tiles(dims, tc, a1);
                if ((int64_t) (c0.per_xcd + c1.per_xcd) * 8 > (int64_t) 0x7fffffff) {
                    e = hipErrorInvalidValue;
                    return;
                }
                hipLaunchKernelGGL((joseph_adj_pair_kernel<decltype(a0)::value, decltype(a1)::value, ST>),
                                   dim3((unsigned) (c0.per_xcd + c1.per_xcd) * 8), dim3(kThreads), lds, s, geo, table,
                                   dims, pose_axes, tc, c0, c1, batch, d_fixexp, sino, vol);
                e = hipGetLastError();
            });
            return e;
        }
        for (int a = 0; a < dims.dim; ++a) {
            if (!(axes_present & (1 << a)))
                continue;
            int ntA, ntB, ntC;
            tile_counts(dims, tc, a, ntA, ntB, ntC);
            const int per_xcd = (ntA * ntB * ntC + 7) / 8;
            const dim3 grid((unsigned) (per_xcd * 8));
#define EHP_ADJ_TILED(Av)                                                                                          \
    hipLaunchKernelGGL((joseph_adj_tiled_kernel<3, Av, ST>), grid, dim3(kThreads), lds, s, geo, table, dims, pose_axes, \
                       tc, ntA, ntB, ntC, per_xcd, batch, d_fixexp, sino, vol)
            if (a == 0)
                EHP_ADJ_TILED(0);
            else if (a == 1)
                EHP_ADJ_TILED(1);
            else
                EHP_ADJ_TILED(2);
#undef EHP_ADJ_TILED
            e = hipGetLastError();
            if (e != hipSuccess)
                return e;
        }
        return hipSuccess;
    }

    template hipError_t joseph_adjoint_tiled<float>(const PoseGeom*, const RayRec*, const Dims&, const int*, int,
                                                    const TileCfg&, int, double, double, unsigned int*, int*, const float*,
                                                    float*, hipStream_t);
    template hipError_t joseph_adjoint_tiled<bf16>(const PoseGeom*, const RayRec*, const Dims&, const int*, int,
                                                   const TileCfg&, int, double, double, unsigned int*, int*, const bf16*,
                                                   float*, hipStream_t);
    template hipError_t joseph_adjoint_tiled<double>(const PoseGeom*, const RayRec*, const Dims&, const int*, int,
                                                     const TileCfg&, int, double, double, unsigned int*, int*, const double*,
                                                     double*, hipStream_t);

    // Segments of a batch's sinograms (absmax) and the tiles of every operator per driving
    // axis (one job per operator that has rays of that axis).
    // One segment per operator (offset and size in a packed vector), each reduced by up to 256
    // blocks of the batched absmax.
    void batch_segments(const int64_t* offs, const int64_t* sizes, int n, std::vector<SegJob>& segs,
                        std::vector<int>& sblocks)
    {
        segs.clear();
        sblocks.clear();
        for (int j = 0; j < n; ++j) {
            SegJob sg{};
            sg.off = offs[j];
            sg.n = sizes[j];
            int64_t nb = (sg.n + 256 * 16 - 1) / (256 * 16);
            nb = nb > 256 ? 256 : (nb < 1 ? 1 : nb);
            sg.nblocks = (int) nb;
            sg.block0 = (int64_t) sblocks.size();
            sblocks.insert(sblocks.end(), (size_t) nb, j);
            segs.push_back(sg);
        }
    }

    hipError_t fixed_point_exponent_batch(int nitems, const SegJob* segs, const int* sblocks, int64_t nsblocks,
                                          const double* bounds, unsigned int* d_maxbits, int* d_fixexp,
                                          const float* y, hipStream_t s)
    {
        if (nsblocks > 0x7fffffff)
            return hipErrorInvalidValue;
        hipLaunchKernelGGL(absmax_batch_kernel, dim3((unsigned) nsblocks), dim3(256), 0, s, y, segs, sblocks,
                           d_maxbits);
        hipLaunchKernelGGL(scale_batch_kernel, dim3((unsigned) nitems), dim3(256), 0, s, d_maxbits, segs, bounds,
                           d_fixexp);
        return hipGetLastError();
    }

    void joseph_adjoint_batch_jobs(const JosephBatchItem* items, int n, std::vector<SegJob>& segs,
                                   std::vector<int>& sblocks, std::vector<AdjJob> ajobs[3],
                                   std::vector<int> ablocks[3], size_t lds[3])
    {
        std::vector<int64_t> offs(n), sizes(n);
        for (int j = 0; j < n; ++j) {
            offs[j] = items[j].sino_off;
            sizes[j] = items[j].dims.nrays;
        }
        batch_segments(offs.data(), sizes.data(), n, segs, sblocks);
        for (int a = 0; a < 3; ++a) {
            ajobs[a].clear();
            ablocks[a].clear();
            lds[a] = 0;
        }
        for (int j = 0; j < n; ++j) {
            const JosephBatchItem& it = items[j];
            if (it.dims.dim == 2) {
                // one list for both axes
                AdjJob aj{};
                aj.geo = it.geo;
                aj.table = it.table;
                aj.pose_axes = it.pose_axes;
                aj.dims = it.dims;
                aj.tc = tile2d(it.tile);
                aj.batch = steps2d(it.dims, it.batch);
                aj.item = j;
                aj.sino_off = it.sino_off;
                aj.vol_off = it.vol_off;
                aj.ntA = (it.dims.vol[0] + aj.tc.LA - 1) / aj.tc.LA;
                const int nty = (it.dims.vol[1] + aj.tc.TB - 1) / aj.tc.TB;
                aj.block0 = (int64_t) ablocks[0].size();
                ablocks[0].insert(ablocks[0].end(), (size_t) aj.ntA * nty, (int) ajobs[0].size());
                ajobs[0].push_back(aj);
                const size_t need = lds2d(aj.tc, aj.batch);
                lds[0] = need > lds[0] ? need : lds[0];
                continue;
            }
            for (int a = 0; a < it.dims.dim; ++a) {
                if (!(it.axes_present & (1 << a)))
                    continue;
                AdjJob aj{};
                aj.geo = it.geo;
                aj.table = it.table;
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
                const size_t need = joseph_tile_lds_bytes(it.dims, it.tile);
                lds[a] = need > lds[a] ? need : lds[a];
            }
        }
    }

    hipError_t joseph_adjoint_batch(int dim, int nitems, const SegJob* segs, const int* sblocks, int64_t nsblocks,
                                    const double* bounds, const AdjJob* const ajobs[3], const int* const ablocks[3],
                                    const int64_t nablocks[3], const size_t lds[3], int64_t nvol_total, double wait,
                                    unsigned int* d_maxbits, int* d_fixexp, const float* sinos, float* vols,
                                    hipStream_t s)
    {
        hipError_t e = dim == 2 ? hipSuccess : launch_fill<float>(vols, nvol_total, 0.0f, s); // 2D tiles write every voxel
        if (e == hipSuccess)
            e = fixed_point_exponent_batch(nitems, segs, sblocks, nsblocks, bounds, d_maxbits, d_fixexp, sinos, s);
        if (e != hipSuccess)
            return e;
        int axes = 0;
        for (int a = 0; a < dim; ++a)
            axes |= nablocks[a] > 0 ? 1 << a : 0;
        if (dim == 3 && pair_launch(axes, nvol_total, wait)) {
            with_axis_pair(axes, [&](auto a0, auto a1) {
                const int64_t p0 = (nablocks[a0] + 7) / 8, p1 = (nablocks[a1] + 7) / 8;
                if ((p0 + p1) * 8 > (int64_t) 0x7fffffff) {
                    e = hipErrorInvalidValue;
                    return;
                }
                const BatchTiles<AdjJob> t0{ajobs[a0], ablocks[a0], nablocks[a0], (int) p0};
                const BatchTiles<AdjJob> t1{ajobs[a1], ablocks[a1], nablocks[a1], (int) p1};
                const size_t need = lds[a0] > lds[a1] ? lds[a0] : lds[a1];
                hipLaunchKernelGGL((joseph_adj_pair_batch_kernel<decltype(a0)::value, decltype(a1)::value>),
                                   dim3((unsigned) (p0 + p1) * 8), dim3(kThreads), need, s, t0, t1, d_fixexp, sinos,
                                   vols);
                e = hipGetLastError();
            });
            return e;
        }
        for (int a = 0; a < dim; ++a) {
            const int64_t total = nablocks[a];
            if (total == 0)
                continue;
            const int64_t per_xcd = (total + 7) / 8;
            if (per_xcd * 8 > (int64_t) 0x7fffffff)
                return hipErrorInvalidValue;
            const dim3 grid((unsigned) (per_xcd * 8));
#define EHP_ADJ_BATCH(Av)                                                                                          \
    hipLaunchKernelGGL((joseph_adj_tiled_batch_kernel<Av>), grid, dim3(kThreads), lds[a], s, ajobs[a], ablocks[a],   \
                       (int) per_xcd, total, d_fixexp, sinos, vols)
            if (dim == 2)
                hipLaunchKernelGGL(joseph_adj2d_batch_kernel, grid, dim3(256), lds[a], s, ajobs[a], ablocks[a],
                                   (int) per_xcd, total, d_fixexp, sinos, vols);
            else if (a == 0)
                EHP_ADJ_BATCH(0);
            else if (a == 1)
                EHP_ADJ_BATCH(1);
            else
                EHP_ADJ_BATCH(2);
#undef EHP_ADJ_BATCH
            e = hipGetLastError();
            if (e != hipSuccess)
                return e;
        }
        return hipGetLastError();
    }
} // namespace ehp
