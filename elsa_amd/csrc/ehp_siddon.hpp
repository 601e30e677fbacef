// ehp_siddon.hpp -- Siddon traversal shared by the GPU kernels and the CPU checks.
//
// The traversal of elsa's TraverseAABB (elsa/projectors/TraverseAABB.cpp:6-184): the voxel
// containing the entry point (a coordinate on a voxel face counts to the lower voxel when the
// ray runs downwards, :136-147), the parameters T[i] of the next face crossing per axis, and
// per step the axes whose T is smallest -- ties step several axes at once (:59-69) -- with the
// segment length tExit - tEntry, tExit starting at 0 (TraverseAABB.h). The crossing
// parameters use the direct rule T[i](k) = fma(k, tDelta[i], T0[i]) after k steps along axis i
// (the oracle's MODE_DIRECT; elsa adds tDelta repeatedly). The state at any point of a ray
// then follows from its step counts, so a tile can restart a ray exactly where it enters.
#pragma once

#include "ehp_joseph_tile.hpp"

namespace ehp
{
    constexpr float kSidMax = 3.4028234663852886e+38f; // numeric_limits<float>::max()

    // Traversal state of one ray after set-up, 32 bytes (one record of the per-operator table).
    struct alignas(16) SidRec {
        float T0[3];     // T of the first face crossing per axis (kSidMax: axis never steps)
        float dt[3];     // tDelta per axis (kSidMax: axis never steps)
        short cur0[3];   // first voxel
        unsigned short meta; // bits 2i..2i+1: step of axis i (0: none, 1: +1, 2: -1); bit 6: the
                             // ray traverses the volume; bits 7-8: driving axis (largest |d|)
    };
    static_assert(sizeof(SidRec) == 32, "SidRec must be 32 bytes");

    EHP_HD inline int sid_step(const SidRec& r, int i)
    {
        const int s = (r.meta >> (2 * i)) & 3;
        return s == 1 ? 1 : (s == 2 ? -1 : 0);
    }
    EHP_HD inline bool sid_hit(const SidRec& r)
    {
        return (r.meta >> 6) & 1;
    }
    EHP_HD inline int sid_axis(const SidRec& r)
    {
        return (r.meta >> 7) & 3;
    }

    // T of axis i after k steps
    EHP_HD inline float sid_T(const SidRec& r, int i, int k)
    {
        return r.dt[i] == kSidMax ? kSidMax : __builtin_fmaf((float) k, r.dt[i], r.T0[i]);
    }

    // Set-up of TraverseAABB for the ray o + t d (d normalised) against [0, vol).
    template <int D>
    EHP_HD inline SidRec siddon_setup(const float* o, const float* d, const int* vol)
    {
        SidRec r;
        for (int i = 0; i < 3; ++i) {
            r.T0[i] = kSidMax;
            r.dt[i] = kSidMax;
            r.cur0[i] = 0;
        }
        int a = 0;
        float m = fabsf(d[0]);
        if (fabsf(d[1]) > m) {
            m = fabsf(d[1]);
            a = 1;
        }
        if (D == 3 && fabsf(d[D - 1]) > m)
            a = 2;
        unsigned meta = (unsigned) a << 7;
        float tmin, tmax;
        bool inbox = intersect<D>(o, d, vol, tmin, tmax);
        if (inbox) {
            float entry[3], cur[3];
            int stepdir[3];
#pragma unroll
            for (int i = 0; i < D; ++i) {
                const float hi = (float) vol[i];
                entry[i] = o[i] + tmin * d[i];
                entry[i] = entry[i] < 0.0f ? 0.0f : entry[i];
                entry[i] = entry[i] > hi ? hi : entry[i];
                stepdir[i] = (int) sgnf(d[i]);
            }
#pragma unroll
            for (int i = 0; i < D; ++i) {
                float lower = floorf(entry[i]);
                if (lower == entry[i] && stepdir[i] < 0)
                    lower = lower - 1.0f;
                cur[i] = lower;
                if (cur[i] >= (float) vol[i] || cur[i] < 0.0f)
                    inbox = false;
            }
            const float EPS = 1.1920928955078125e-07f; // numeric_limits<float>::epsilon()
#pragma unroll
            for (int i = 0; i < D; ++i) {
                const bool moves = fabsf(d[i]) > EPS;
                r.dt[i] = moves ? (float) stepdir[i] / d[i] : kSidMax;
                r.T0[i] = moves ? ((d[i] > 0.0f ? cur[i] + 1.0f : cur[i]) - entry[i]) / d[i] : kSidMax;
                r.cur0[i] = inbox ? (short) cur[i] : (short) 0;
                const int st = moves ? stepdir[i] : 0;
                meta |= (unsigned) (st == 1 ? 1 : (st == -1 ? 2 : 0)) << (2 * i);
            }
        }
        if (inbox)
            meta |= 1u << 6;
        r.meta = (unsigned short) meta;
        return r;
    }

    // The whole traversal: fn(c0, c1, c2, w) per crossed voxel (c2 = 0 in 2D), in ray order.
    // An axis whose |d| <= epsilon never steps (its T stays kSidMax), as in elsa.
    template <int D, class Fn>
    EHP_HD inline void siddon_traverse(const SidRec& r, const int* vol, Fn fn)
    {
        if (!sid_hit(r))
            return;
        int cur[3] = {r.cur0[0], r.cur0[1], D == 3 ? r.cur0[2] : 0};
        int k[3] = {0, 0, 0};
        float Tn[3] = {r.T0[0], r.T0[1], D == 3 ? r.T0[2] : kSidMax};
        float tExit = 0.0f;
        // a ray crosses at most vol[0] + vol[1] + vol[2] voxels; the cap only matters for
        // degenerate (non-finite) rays
        int guard = vol[0] + vol[1] + (D == 3 ? vol[2] : 0) + 2;
        bool inbox = true;
        while (inbox && guard-- > 0) {
            const float tEntry = tExit;
            float tm = Tn[0];
#pragma unroll
            for (int i = 1; i < D; ++i)
                tm = fminf(tm, Tn[i]);
            tExit = tm;
            bool mask[3];
#pragma unroll
            for (int i = 0; i < D; ++i) {
                bool mi = true;
#pragma unroll
                for (int j = 0; j < D; ++j)
                    if (j != i)
                        mi = mi && (Tn[i] <= Tn[j]);
                mask[i] = mi;
            }
            fn(cur[0], cur[1], cur[2], tExit - tEntry);
#pragma unroll
            for (int i = 0; i < D; ++i) {
                if (mask[i]) {
                    cur[i] += sid_step(r, i);
                    k[i] += 1;
                    Tn[i] = sid_T(r, i, k[i]);
                }
            }
#pragma unroll
            for (int i = 0; i < D; ++i)
                inbox = inbox && cur[i] < vol[i] && cur[i] >= 0;
        }
    }

    // The traversal plane by plane in single steps, which the CPU checks of the views run; the kernels form a
    // plane's segments by sorting (sid_plane_segments). It can pause between the planes of one axis: the state of
    // siddon_traverse after some of its steps (voxel, step direction and count per axis as a
    // float -- exact, as counts stay below 2^24 -- next crossing per axis, the last crossing).
    struct SidWalk {
        int cur[3];
        int st[3];
        float fk[3];
        float Tn[3];
        float tExit;
        bool alive;
    };

    template <int D>
    EHP_HD inline void sid_walk_init(const SidRec& r, SidWalk& w)
    {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            w.cur[i] = i < D ? r.cur0[i] : 0;
            w.st[i] = i < D ? sid_step(r, i) : 0;
            w.fk[i] = 0.0f;
            w.Tn[i] = i < D ? r.T0[i] : kSidMax;
        }
        w.tExit = 0.0f;
        w.alive = sid_hit(r);
    }

    // Steps of one plane: a ray crossing plane p of its driving axis A (the largest |d|) in it
    // moves less than one voxel along every other axis, so it visits at most D voxels there.
    constexpr int kSidPlaneSteps = 8;

    // The steps of siddon_traverse whose voxel lies on plane p of axis A, fn(c0, c1, c2, w) for
    // each in ray order, leaving the walk at the first voxel beyond that plane (or ended). The
    // same arithmetic as siddon_traverse step by step, so walking plane after plane gives its
    // crossings bit for bit. (Only an axis that moves can have the smallest T, as the driving
    // axis moves, so the update needs no test for a non-moving one.) At most kSidPlaneSteps steps
    // per call, which also stops a degenerate ray.
    template <int D, class Fn>
    EHP_HD inline void sid_walk_plane(const SidRec& r, const int* vol, int A, int p, SidWalk& w, Fn fn)
    {
        for (int g = 0; g < kSidPlaneSteps && w.alive && w.cur[A] == p; ++g) {
            const float tEntry = w.tExit;
            float tm = w.Tn[0];
#pragma unroll
            for (int i = 1; i < D; ++i)
                tm = fminf(tm, w.Tn[i]);
            w.tExit = tm;
            bool mask[3];
#pragma unroll
            for (int i = 0; i < D; ++i) {
                bool mi = true;
#pragma unroll
                for (int j = 0; j < D; ++j)
                    if (j != i)
                        mi = mi && (w.Tn[i] <= w.Tn[j]);
                mask[i] = mi;
            }
            fn(w.cur[0], w.cur[1], w.cur[2], w.tExit - tEntry);
            bool in = true;
#pragma unroll
            for (int i = 0; i < D; ++i) {
                if (mask[i]) {
                    w.cur[i] += w.st[i];
                    w.fk[i] += 1.0f;
                    w.Tn[i] = __builtin_fmaf(w.fk[i], r.dt[i], r.T0[i]);
                }
                in = in && (uint32_t) w.cur[i] < (uint32_t) vol[i];
            }
            w.alive = in;
        }
    }

    // ---------------------------------------------------------------------------------
    // The forward kernel's traversal: plane by plane of the driving axis A, without a loop over the crossings. On a
    // plane the ray crosses each transverse axis at most once (the driving axis has the largest
    // |d|), so its crossings there are the sorted values of at most two parameters below the plane's
    // exit T_A, and three segments (2D: two) cover them. The same parameters, segments and order as
    // siddon_traverse, so the same crossings bit for bit.

    // State of a ray between two planes: the exit parameter of the last plane, the parameter at
    // which the ray leaves the volume, per axis the steps taken (as a float: exact below 2^24) and
    // the next crossing, and the byte offset of the current voxel in a plane of the view with its
    // changes per step along b1 and b2.
    struct SidSpan {
        float t, tend;
        float ka, kb, kc;
        float Tb, Tc;
        uint32_t off;
        uint32_t db, dc;
    };

    // The parameter of the crossing by which axis i leaves [0, n): its step number n - cur0 upwards,
    // cur0 + 1 downwards (T_i rises with the step number)
    EHP_HD inline float sid_exit_T(const SidRec& r, int i, int n)
    {
        const int st = sid_step(r, i);
        return st == 0 ? kSidMax : sid_T(r, i, st > 0 ? n - 1 - (int) r.cur0[i] : (int) r.cur0[i]);
    }

    // V: the plane-major view of driving axis A (bytes per row RS4, elements of 2^lg bytes); FB2: its
    // fastest axis is b2 (else b1).
    template <int D, int A, bool FB2>
    EHP_HD inline SidSpan sid_span_init(const SidRec& r, const int* vol, uint32_t RS4, uint32_t lg)
    {
        constexpr int b1 = TileAxes<D, A>::b1, b2 = TileAxes<D, A>::b2;
        SidSpan s;
        s.t = 0.0f;
        s.tend = fminf(sid_exit_T(r, 0, vol[0]), sid_exit_T(r, 1, vol[1]));
        if (D == 3)
            s.tend = fminf(s.tend, sid_exit_T(r, D - 1, vol[D - 1]));
        s.ka = s.kb = s.kc = 0.0f;
        s.Tb = r.T0[b1];
        s.Tc = D == 3 ? r.T0[b2] : kSidMax;
        const uint32_t e = 1u << lg;
        if (D == 3) {
            const int m = FB2 ? b1 : b2, f = FB2 ? b2 : b1;
            s.off = mul24((uint32_t) (r.cur0[m] + 2), RS4) + ((uint32_t) (r.cur0[f] + 2) << lg);
            s.db = (uint32_t) sid_step(r, b1) * (FB2 ? RS4 : e);
            s.dc = (uint32_t) sid_step(r, b2) * (FB2 ? e : RS4);
        } else {
            s.off = (uint32_t) (r.cur0[b1] + 2) << lg;
            s.db = (uint32_t) sid_step(r, b1) * e;
            s.dc = 0;
        }
        return s;
    }

    // Smallest and middle of three crossing parameters and the smaller of two, one instruction each
    // (crossing parameters are never NaN: fminf would first quiet one)
    EHP_HD inline float sid_min3(float a, float b, float c)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        float r;
        asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
        return r;
#else
        return fminf(fminf(a, b), c);
#endif
    }
    EHP_HD inline float sid_min(float a, float b)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        float r;
        asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
        return r;
#else
        return fminf(a, b);
#endif
    }
    EHP_HD inline float sid_med3(float a, float b, float c)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        float r;
        asm("v_med3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
        return r;
#else
        return fmaxf(fminf(a, b), fminf(fmaxf(a, b), c));
#endif
    }

    // Whether the ray may cross a transverse axis twice on one plane of its driving axis A: the
    // crossings of an axis lie dt apart up to the roundings of two parameters, a plane is dt[A] long up
    // to the same, and no parameter inside the volume passes tend.
    template <int D, int A>
    EHP_HD inline bool sid_may_cross_twice(const SidRec& r, float tend)
    {
        constexpr int b1 = TileAxes<D, A>::b1, b2 = TileAxes<D, A>::b2;
        const float least = D == 3 ? fminf(r.dt[b1], r.dt[b2]) : r.dt[b1];
        return !(least > r.dt[A] + 4.0f * 1.1920929e-7f * (tend + 2.0f * r.dt[A]));
    }

    // The values and lengths of the segments of one plane, in ray order (2D: two)
    template <class T>
    struct SidSegments {
        T v1, v2, v3;
        float w1, w2, w3;
    };

    template <int D, class T>
    EHP_HD inline T sid_segments_add(const SidSegments<T>& g, T acc)
    {
        acc += g.v1 * (T) g.w1;
        acc += g.v2 * (T) g.w2;
        if (D == 3)
            acc += g.v3 * (T) g.w3;
        return acc;
    }

    // The next plane of a ray that crosses each transverse axis at most once on it (ta: its exit;
    // kb, kc, Tb, Tc: the state after it): its segments (ld(off): the view's element at byte offset off
    // of the plane), and the ray's state moved past it. Off-path elements are never read: a segment
    // that is not there reads offset 0, a zero of the padding.
    template <int D, class T, class Ld>
    EHP_HD inline SidSegments<T> sid_plane_once(SidSpan& s, float ta, float kb, float kc, float Tb, float Tc, Ld ld)
    {
        SidSegments<T> g;
        const bool sb = s.Tb <= ta, sc = D == 3 && s.Tc <= ta;
        if (D == 3) {
            const float first = sid_min3(s.Tb, s.Tc, ta);
            const float second = sid_min(sid_med3(s.Tb, s.Tc, ta), ta);
            const uint32_t o2 = s.off + (s.Tb <= s.Tc ? s.db : s.dc), o3 = s.off + (s.db + s.dc);
            g.v1 = ld(s.off);
            g.v2 = ld(first < second ? o2 : 0u);
            g.v3 = ld(second < ta ? o3 : 0u);
            g.w1 = first - s.t;
            g.w2 = second - first;
            g.w3 = ta - second;
        } else {
            const float first = sid_min(s.Tb, ta);
            g.v1 = ld(s.off);
            g.v2 = ld(first < ta ? s.off + s.db : 0u);
            g.v3 = T(0);
            g.w1 = first - s.t;
            g.w2 = ta - first;
            g.w3 = 0.0f;
        }
        s.off += (sb ? s.db : 0u) + (sc ? s.dc : 0u);
        s.kb = kb;
        s.kc = kc;
        s.Tb = Tb;
        s.Tc = Tc;
        s.t = ta;
        s.ka += 1.0f;
        return g;
    }

    // The exit of the ray's next plane and its crossing state after the plane, one crossing per
    // transverse axis. (An axis that does not move has kb = 0 and dt = T0 = kSidMax: its T stays kSidMax.)
    template <int D, int A>
    EHP_HD inline void sid_plane_next(const SidRec& r, const SidSpan& s, float& ta, float& kb, float& kc, float& Tb,
                                      float& Tc)
    {
        constexpr int b1 = TileAxes<D, A>::b1, b2 = TileAxes<D, A>::b2;
        ta = __builtin_fmaf(s.ka, r.dt[A], r.T0[A]);
        kb = s.kb + (s.Tb <= ta ? 1.0f : 0.0f);
        kc = D == 3 ? s.kc + (s.Tc <= ta ? 1.0f : 0.0f) : 0.0f;
        Tb = __builtin_fmaf(kb, r.dt[b1], r.T0[b1]);
        Tc = D == 3 ? __builtin_fmaf(kc, r.dt[b2], r.T0[b2]) : kSidMax;
    }

    // The segments of the next plane of a ray that crosses no axis twice on it (sid_may_cross_twice
    // says so). After the ray has left the volume (t >= tend) the caller stops; until the end of that
    // plane it reads the padding's zeros.
    template <int D, int A, class T, class Ld>
    EHP_HD inline SidSegments<T> sid_plane_segments(const SidRec& r, SidSpan& s, Ld ld)
    {
        float ta, kb, kc, Tb, Tc;
        sid_plane_next<D, A>(r, s, ta, kb, kc, Tb, Tc);
        return sid_plane_once<D, T>(s, ta, kb, kc, Tb, Tc, ld);
    }

    // acc plus the crossings of the next plane of any ray: a plane with two crossings of one axis
    // (rays at 45 degrees, by rounding) is walked step by step.
    template <int D, int A, class T, class Ld>
    EHP_HD inline T sid_plane_add(const SidRec& r, SidSpan& s, T acc, Ld ld)
    {
        constexpr int b1 = TileAxes<D, A>::b1, b2 = TileAxes<D, A>::b2;
        float ta, kb, kc, Tb, Tc;
        sid_plane_next<D, A>(r, s, ta, kb, kc, Tb, Tc);
        if (sid_min(Tb, Tc) > ta)
            return sid_segments_add<D>(sid_plane_once<D, T>(s, ta, kb, kc, Tb, Tc, ld), acc);
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll 1
#endif
        for (int g = 0; g < kSidPlaneSteps; ++g) {
            const float tm = sid_min3(s.Tb, s.Tc, ta);
            const bool mb = s.Tb <= tm, mc = D == 3 && s.Tc <= tm;
            acc += ld(s.off) * (T) (tm - s.t);
            s.t = tm;
            if (mb) {
                s.kb += 1.0f;
                s.Tb = __builtin_fmaf(s.kb, r.dt[b1], r.T0[b1]);
                s.off += s.db;
            }
            if (mc) {
                s.kc += 1.0f;
                s.Tc = __builtin_fmaf(s.kc, r.dt[b2], r.T0[b2]);
                s.off += s.dc;
            }
            if (ta <= tm)
                break;
        }
        s.t = ta;
        s.ka += 1.0f;
        return acc;
    }

    // The part of the traversal inside the voxel box lo[i] <= c[i] <= hi[i]: fn(c0, c1, c2, w)
    // for exactly the crossings of siddon_traverse whose voxel lies in the box, with the same
    // w. The ray is restarted at the last face crossing before the box: for each axis the step
    // counts keeping it inside the box form a range [a_i, b_i]; the crossing that brings the
    // last axis into its range happens at t_lo = max_i T_i(a_i - 1), and at t_lo axis i has
    // taken every step whose T_i(k) <= t_lo.
    template <int D, class Fn>
    EHP_HD inline void siddon_box(const SidRec& r, const int* lo, const int* hi, Fn fn)
    {
        if (!sid_hit(r))
            return;
        int a[3], st[3];
        float t_lo = 0.0f;
#pragma unroll
        for (int i = 0; i < D; ++i) {
            st[i] = sid_step(r, i);
            const int c0 = r.cur0[i];
            int ai, bi;
            if (st[i] == 0) {
                if (c0 < lo[i] || c0 > hi[i])
                    return;
                ai = 0;
                bi = 0x7fffffff;
            } else if (st[i] > 0) {
                ai = lo[i] - c0;
                bi = hi[i] - c0;
            } else {
                ai = c0 - hi[i];
                bi = c0 - lo[i];
            }
            if (bi < 0)
                return;
            ai = ai > 0 ? ai : 0;
            a[i] = ai;
            if (ai > 0) {
                const float te = sid_T(r, i, ai - 1);
                t_lo = te > t_lo ? te : t_lo;
            }
        }
        int cur[3] = {0, 0, 0};
        float fk[3] = {0.0f, 0.0f, 0.0f}; // step counts (exact below 2^24)
        float Tn[3] = {kSidMax, kSidMax, kSidMax};
#pragma unroll
        for (int i = 0; i < D; ++i) {
            int j = 0;
            if (st[i] != 0 && t_lo > 0.0f) {
                // smallest j with T_i(j) > t_lo: estimate (an approximate reciprocal will do),
                // then step to it
                const float est = (t_lo - r.T0[i]) * ehp_rcp(r.dt[i]);
                j = est < 0.0f ? 0 : (est > 1.0e7f ? 10000000 : (int) est);
                j = j > a[i] ? a[i] : j;
                while (sid_T(r, i, j) <= t_lo)
                    ++j;
                while (j > 0 && sid_T(r, i, j - 1) > t_lo)
                    --j;
            }
            fk[i] = (float) j;
            cur[i] = r.cur0[i] + st[i] * j;
            Tn[i] = sid_T(r, i, j);
        }
        float tEntry = t_lo;
        int guard = 0;
#pragma unroll
        for (int i = 0; i < D; ++i)
            guard += hi[i] - lo[i] + 1;
        while (guard-- > 0) {
            bool in = true;
#pragma unroll
            for (int i = 0; i < D; ++i)
                in = in && (uint32_t) (cur[i] - lo[i]) <= (uint32_t) (hi[i] - lo[i]);
            if (!in)
                return;
            float tm = Tn[0];
#pragma unroll
            for (int i = 1; i < D; ++i)
                tm = fminf(tm, Tn[i]);
            bool mask[3];
#pragma unroll
            for (int i = 0; i < D; ++i) {
                bool mi = true;
#pragma unroll
                for (int j = 0; j < D; ++j)
                    if (j != i)
                        mi = mi && (Tn[i] <= Tn[j]);
                mask[i] = mi;
            }
            fn(cur[0], cur[1], cur[2], tm - tEntry);
            tEntry = tm;
            // only an axis that moves can have the smallest T (the driving axis moves)
#pragma unroll
            for (int i = 0; i < D; ++i) {
                if (mask[i]) {
                    cur[i] += st[i];
                    fk[i] += 1.0f;
                    Tn[i] = __builtin_fmaf(fk[i], r.dt[i], r.T0[i]);
                }
            }
        }
    }

    // ---------------------------------------------------------------------------------
    // The back projection's traversal of a tile: the planes of the driving axis in ray order, each
    // with its segments from the sorted crossing parameters as in the forward, restarted at the
    // tile's first plane.

    // Number of steps of axis i up to parameter t (T_i(k) <= t), as a float: estimated with an
    // approximate reciprocal, then stepped to the exact count.
    EHP_HD inline float sid_steps_until(const SidRec& r, int i, float t)
    {
        const float est = (t - r.T0[i]) * ehp_rcp(r.dt[i]);
        float k = floorf(est) + 1.0f;
        k = k > 0.0f ? (k < 1.0e7f ? k : 1.0e7f) : 0.0f;
        // (an axis that does not move has T = kSidMax at k = 0)
        while (__builtin_fmaf(k, r.dt[i], r.T0[i]) <= t)
            k += 1.0f;
        while (k > 0.0f && __builtin_fmaf(k - 1.0f, r.dt[i], r.T0[i]) > t)
            k -= 1.0f;
        return k;
    }

    // Bytes per row of a tile's slots along b1 (8 bytes each): an odd number of slots where the LDS
    // allows it, so that neighbouring rows fall on different banks.
    EHP_HD inline int sid_row_slots(const TileCfg& tc, int dim)
    {
        const int rows = tc.LA * (dim == 3 ? tc.TC : 1);
        return dim == 3 && (int64_t) rows * (tc.TB | 1) * 8 + (int64_t) batch_lds_bytes(kMaxPoseBatch) <= 65536
                   ? (tc.TB | 1)
                   : tc.TB;
    }

    // Slot offsets of a tile in bytes: voxel (a, b, c) of the tile's axes at base + (a - A0) plane +
    // oc + ob with ob = 8 b + nb < maxb and oc = c cs + nc < maxc as unsigned numbers (2D: ob only).
    struct SidTileOff {
        uint32_t nb, maxb;
        int nc, cs;
        uint32_t maxc, plane, base;
    };

    template <int D>
    EHP_HD inline SidTileOff sid_tile_offsets(const TileBox& t, const TileCfg& tc, uint32_t base = 0)
    {
        SidTileOff o;
        o.cs = 8 * sid_row_slots(tc, D);
        o.nb = (uint32_t) (-8 * t.B0);
        o.maxb = (uint32_t) (8 * (t.B1 - t.B0));
        o.nc = -t.C0 * o.cs;
        o.maxc = (uint32_t) ((t.C1 - t.C0) * o.cs);
        o.plane = (uint32_t) (o.cs * (D == 3 ? tc.TC : 1));
        o.base = base;
        return o;
    }

    // add(off, w) for exactly the crossings of siddon_traverse whose voxel lies in the tile and whose
    // length w is not 0, off the byte offset of the voxel's slot. r drives along A and hits the volume.
    // A ray that has left the volume is outside every tile, as no voxel it would meet comes back.
    template <int D, int A, class Add>
    EHP_HD inline void sid_tile_ray(const SidRec& r, const TileBox& t, const SidTileOff& to, Add add)
    {
        constexpr int b1 = TileAxes<D, A>::b1, b2 = TileAxes<D, A>::b2;
        const bool neg = sid_step(r, A) < 0;
        const int cA = r.cur0[A];
        // steps along A before the tile's first plane in ray order (negative: the ray starts later)
        const int d = neg ? cA - (t.A1 - 1) : t.A0 - cA;
        const int ja = d > 0 ? d : 0;
        const int p = (neg ? cA - ja : cA + ja) - t.A0; // the first plane to visit, in the tile
        int n = neg ? p + 1 : t.A1 - t.A0 - p;
        if (n <= 0)
            return;
        float ka = (float) ja;
        const float tlast = __builtin_fmaf(ka + (float) (n - 1), r.dt[A], r.T0[A]);
        if (sid_may_cross_twice<D, A>(r, tlast)) {
            int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
            lo[A] = t.A0;
            hi[A] = t.A1 - 1;
            lo[b1] = t.B0;
            hi[b1] = t.B1 - 1;
            if (D == 3) {
                lo[b2] = t.C0;
                hi[b2] = t.C1 - 1;
            }
            siddon_box<D>(r, lo, hi, [&](int c0, int c1, int c2, float w) {
                const int ca = A == 0 ? c0 : (A == 1 ? c1 : c2), cb = b1 == 0 ? c0 : c1;
                const int cc = D == 3 ? (b2 == 1 ? c1 : c2) : 0;
                if (w != 0.0f)
                    add(to.base + (uint32_t) (ca - t.A0) * to.plane + (uint32_t) (8 * cb) + to.nb +
                            (D == 3 ? (uint32_t) (cc * to.cs + to.nc) : 0u),
                        w);
            });
            return;
        }
        float t0 = 0.0f, kb = 0.0f, kc = 0.0f;
        if (ja > 0) {
            t0 = __builtin_fmaf(ka - 1.0f, r.dt[A], r.T0[A]);
            kb = sid_steps_until(r, b1, t0);
            if (D == 3)
                kc = sid_steps_until(r, b2, t0);
        }
        const int sb1 = sid_step(r, b1), sb2 = D == 3 ? sid_step(r, b2) : 0;
        uint32_t ob = (uint32_t) (8 * ((int) r.cur0[b1] + sb1 * (int) kb)) + to.nb;
        uint32_t oc = D == 3 ? (uint32_t) (((int) r.cur0[b2] + sb2 * (int) kc) * to.cs + to.nc) : 0u;
        const uint32_t db = (uint32_t) (8 * sb1), dc = (uint32_t) (sb2 * to.cs);
        uint32_t poff = to.base + (uint32_t) p * to.plane;
        const uint32_t dp = neg ? 0u - to.plane : to.plane;
        float Tb = __builtin_fmaf(kb, r.dt[b1], r.T0[b1]);
        float Tc = D == 3 ? __builtin_fmaf(kc, r.dt[b2], r.T0[b2]) : kSidMax;
        for (; n > 0; --n, poff += dp) {
            const float ta = __builtin_fmaf(ka, r.dt[A], r.T0[A]);
            const bool sb = Tb <= ta, sc = D == 3 && Tc <= ta;
            const float first = D == 3 ? sid_min3(Tb, Tc, ta) : sid_min(Tb, ta);
            const float second = D == 3 ? sid_min(sid_med3(Tb, Tc, ta), ta) : ta;
            const float w1 = first - t0, w2 = second - first, w3 = ta - second;
            if (ob < to.maxb && (D == 2 || oc < to.maxc) && w1 != 0.0f)
                add(poff + ob + oc, w1);
            // the second segment lies past the axis crossed first, the third past both
            const bool bf = D == 2 || Tb <= Tc;
            const uint32_t ob2 = ob + (bf ? db : 0u), oc2 = oc + (bf ? 0u : dc);
            if (ob2 < to.maxb && (D == 2 || oc2 < to.maxc) && w2 != 0.0f)
                add(poff + ob2 + oc2, w2);
            if (D == 3) {
                const uint32_t ob3 = ob + db, oc3 = oc + dc;
                if (ob3 < to.maxb && oc3 < to.maxc && w3 != 0.0f)
                    add(poff + ob3 + oc3, w3);
            }
            ob += sb ? db : 0u;
            oc += sc ? dc : 0u;
            kb += sb ? 1.0f : 0.0f;
            Tb = __builtin_fmaf(kb, r.dt[b1], r.T0[b1]);
            if (D == 3) {
                kc += sc ? 1.0f : 0.0f;
                Tc = __builtin_fmaf(kc, r.dt[b2], r.T0[b2]);
            }
            t0 = ta;
            ka += 1.0f;
        }
    }

    // Slot of voxel c in a tile of the Siddon back projection with unpadded rows (no halo: the tile's own voxels,
    // b1 fastest, then b2, then the driving axis), for the CPU checks; the kernels' rows are sid_row_slots long.
    template <int D, int A>
    EHP_HD inline int sid_slot(const TileBox& t, const TileCfg& tc, int c0, int c1, int c2)
    {
        constexpr int b1 = TileAxes<D, A>::b1, b2 = TileAxes<D, A>::b2;
        const int c[3] = {c0, c1, c2};
        const int xa = (A == 0 ? c[0] : (A == 1 ? c[1] : c[2])) - t.A0;
        const int xb = (b1 == 0 ? c[0] : (b1 == 1 ? c[1] : c[2])) - t.B0;
        const int xc = D == 3 ? (b2 == 0 ? c[0] : (b2 == 1 ? c[1] : c[2])) - t.C0 : 0;
        return (int) (mul24((uint32_t) xa, (uint32_t) (tc.TB * (D == 3 ? tc.TC : 1))) +
                      mul24((uint32_t) xc, (uint32_t) tc.TB)) +
               xb;
    }
} // namespace ehp
