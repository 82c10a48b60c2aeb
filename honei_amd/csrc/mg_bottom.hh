// mg_bottom.hh -- the V-cycle's bottom levels in one workgroup per slot.
// Included by mg_engine.hip.
//
// Levels minl .. top (top <= 6, below the finest) of a V-cycle on Q1 bands:
// two sweeps from zero, defect and restriction down to minl, the coarse CG,
// then prolongation with the correction factor and two sweeps back up, the
// same operations per node as the one-pass kernels and the coarse solve run
// there.  It reads the rhs of level top and leaves top's smoothed iterate in
// its F_TMP, where the one-pass post-smoother above reads it.
#pragma once

namespace
{
    constexpr int kBottomMax = 6;
    constexpr int kBottomLanes = 1024;
    template <int L> constexpr int kSide = (1 << L) + 1;
    template <int L> constexpr int kSize = kSide<L> * kSide<L>;
    template <int L> constexpr int kRowsPerLane = (kSize<L> + kBottomLanes - 1) / kBottomLanes;
    // LDS floats before level L's three vectors (rhs, x, tmp); a stencil row
    // at a level's ends reads up to a side + 1 floats outside its vector and
    // selects the value away
    template <int L> constexpr int kBottomOff = kBottomOff<L - 1> + 3 * kSize<L - 1>;
    template <> constexpr int kBottomOff<1> = kSide<kBottomMax> + 1;
    template <int L> constexpr int kBottomFloats = kBottomOff<L> + 3 * kSize<L> + kSide<L> + 1;

    struct BottomArgs
    {
        LevelArgs lv[kBottomMax + 1];
        int top;
        float alpha;
        k::Mask mk;
        double konv_rad;
        uint64_t max_iters;
    };

    // Row i of A v on level L, v in LDS, the row's bands in registers: q1_row's
    // order and index guards.
    template <int L, int ORD>
    __device__ __forceinline__ float bottom_row(const float (&b)[10], const float * v, int i)
    {
        constexpr int m = kSide<L>, n = kSize<L>;
        float s = ORD == 1 ? 0.0f : b[4] * v[i];
        auto put = [&](bool on, float w, float x) {
            const float t = s + w * x;
            s = on ? t : s;
        };
        put(i - m - 1 >= 0, b[0], v[i - m - 1]);
        put(i - m >= 0, b[1], v[i - m]);
        put(i - m + 1 >= 0, b[2], v[i - m + 1]);
        put(i - 1 >= 0, b[3], v[i - 1]);
        if (ORD == 1)
            put(true, b[4], v[i]);
        put(i + 1 < n, b[5], v[i + 1]);
        put(i + m - 1 < n, b[6], v[i + m - 1]);
        put(i + m < n, b[7], v[i + m]);
        put(i + m + 1 < n, b[8], v[i + m + 1]);
        return s;
    }

    // ConjugateGradients<NONE>(A, rhs, x, konv_rad) on a level of at most 64
    // nodes in one wave, lane i holding node i of every vector: the steps of
    // k::cg_konv_body_op, whose sums run over the lanes in index order.  (Its
    // step's first sum, g.g, is the last step's ng.ng: the same terms in the
    // same order.)  A step is a chain of about 1300 cycles; with the vectors
    // in LDS, whose sums and rows waited on LDS round trips, it took 3.2 us.
    template <int L, int ORD>
    __device__ __forceinline__ float bottom_cg(const float (&b)[10], float rhs, double konv_rad, uint64_t max_iters,
                                               uint64_t * iters_out)
    {
        constexpr int m = kSide<L>, n = kSize<L>;
        static_assert(n <= 64, "one lane per node");
        constexpr float eps = k::Eps<float>::v;
        const int i = threadIdx.x & 63;
        auto row = [&](float v) {
            float s = ORD == 1 ? 0.0f : b[4] * v;
            auto put = [&](int off, float w) {
                const float x = __shfl(v, i + off, 64);
                const float t = s + w * x;
                s = (i + off >= 0 && i + off < n) ? t : s;
            };
            put(-m - 1, b[0]);
            put(-m, b[1]);
            put(-m + 1, b[2]);
            put(-1, b[3]);
            if (ORD == 1)
                s += b[4] * v;
            put(1, b[5]);
            put(m - 1, b[6]);
            put(m, b[7]);
            put(m + 1, b[8]);
            return s;
        };
        auto dot = [&](float p, float q) {
            const float t = p * q;
            float r = 0.0f;
#pragma unroll
            for (int j = 0; j < n; ++j)
                r += k::lane_value(t, j);
            return r;
        };
        float x = 0.0f;
        float g = row(x) - rhs;
        float u = g * -1.0f;
        float upper = dot(g, g);
        float norm_x = dot(x, x), norm_x_last = norm_x - 1.0f;
        uint64_t it = 0;
        while ((double)(norm_x - norm_x_last) > konv_rad && it < max_iters)
        {
            float lower = dot(row(u), u);
            const float f1 = fabs(lower) >= eps ? upper / lower : upper / eps;
            const float en = u * f1 + x;
            lower = upper;
            const float ng = row(en) - rhs;
            upper = dot(ng, ng);
            const float f2 = fabs(lower) >= eps ? upper / lower : upper / eps;
            u = u * f2 - ng;
            x = en;
            ++it;
            norm_x_last = norm_x;
            norm_x = dot(x, x);
        }
        if (iters_out && i == 0)
            *iters_out = it;
        return x;
    }

    // MINL: the coarsest level (1 or 2: a lane per node in the CG).  Each lane
    // owns rows tid, tid + 1024, ... of every level and keeps their bands and
    // dinv in registers; LDS holds the vectors.  Up to level 5 every band is
    // loaded in one round trip.  TOP6 (top is 6): level 6 takes 50 registers
    // for its five rows, so its bands are loaded twice, for the way down with
    // level 5's and for the way up before or after the coarse solve, which with
    // the levels between hides them.
    // With level 6 here a cycle saves two launches of 7 to 10 us (measured on
    // MI355X, a solve: 129^2 661 -> 598 us, 1025^2 1655 -> 1583 us, 4097^2
    // 4957 -> 4887 us, 64 of 513^2 1.03x).  Level 7 would need 17 rows a lane.
    template <int MK, int MINL, bool TOP6>
    __global__ __launch_bounds__(kBottomLanes) void v_bottom_kernel(BottomArgs ba, const Slot * T)
    {
        const VB vb = vblock();
        const Slot & sl = T[vb.z];
        if (! live(sl) || sl.s->run == 0)
            return;
        constexpr int ORD = kOrd<MK>;
        __shared__ float lds[kBottomFloats<TOP6 ? 6 : 5>];
        const int tid = threadIdx.x;
        float b6[TOP6 ? kRowsPerLane<6> : 1][10], b5[2][10], b4[10], b3[10], b2[10], b1[10];
        auto load_from = [&](auto l_tag, int r, int k0, float (&b)[10]) {
            constexpr int L = decltype(l_tag)::value;
            const LevelArgs & a = ba.lv[L];
            const int i = min(tid + r * kBottomLanes, kSize<L> - 1) + k0;
#pragma unroll
            for (int k = 0; k < 10; ++k)
                b[k] = as_global<const float>(k < 9 ? (const float *)a.B.b[k] : a.dinv)[i];
        };
        auto load = [&](auto l_tag, int r, float (&b)[10]) { load_from(l_tag, r, 0, b); };
        auto load6 = [&]() {
            int zero = 0;
            asm volatile("" : "+v"(zero));   // a second load, not the first one's registers kept
#pragma unroll
            for (int r = 0; r < kRowsPerLane<6>; ++r)
                load_from(IntC<6>{}, r, zero, b6[TOP6 ? r : 0]);
        };
        auto load_low = [&](int top) {
            if (top >= 4)
                load(IntC<4>{}, 0, b4);
            if (top >= 3)
                load(IntC<3>{}, 0, b3);
            load(IntC<2>{}, 0, b2);
            if (MINL == 1)
                load(IntC<1>{}, 0, b1);
        };
        const int top = TOP6 ? 6 : ba.top;
        if constexpr (TOP6)
            load6();
        if (top >= 5)
        {
            load(IntC<5>{}, 0, b5[0]);
            load(IntC<5>{}, 1, b5[1]);
        }
        if (! TOP6)
            load_low(top);
        {
            auto take = [&](auto l_tag) {
                constexpr int L = decltype(l_tag)::value;
                const gptr<const float> g = as_global<const float>(sl.v[L][F_RHS]);
                for (int i = tid; i < kSize<L>; i += kBottomLanes)
                    lds[kBottomOff<L> + i] = g[i];
            };
            if constexpr (TOP6)
                take(IntC<6>{});
            else if (top == 5)
                take(IntC<5>{});
            else if (top == 4)
                take(IntC<4>{});
            else if (top == 3)
                take(IntC<3>{});
            else if (top == 2)
                take(IntC<2>{});
        }
        lds_barrier();
        // the rows' bands of level L
        auto bands = [&](auto l_tag, int r) -> const float (&)[10] {
            constexpr int L = decltype(l_tag)::value;
            if constexpr (L == 6)
                return b6[TOP6 ? r : 0];
            else if constexpr (L == 5)
                return b5[r];
            else if constexpr (L == 4)
                return b4;
            else if constexpr (L == 3)
                return b3;
            else
                return b2;
        };
        auto each = [&](auto l_tag, auto && f) {
            constexpr int L = decltype(l_tag)::value;
#pragma unroll
            for (int r = 0; r < kRowsPerLane<L>; ++r)
            {
                const int i = tid + r * kBottomLanes;
                if (i < kSize<L>)
                    f(i, bands(l_tag, r));
            }
            lds_barrier();
        };
        // x = c1 + dinv (rhs - A c1) with c1 = dinv rhs, d' = rhs - A x, rhs of L - 1 = R d'
        auto down = [&](auto l_tag) {
            constexpr int L = decltype(l_tag)::value, n = kSize<L>, m = kSide<L>, Nc = kSide<L - 1>;
            float * rhs = lds + kBottomOff<L>;
            float * x = rhs + n;
            float * tmp = x + n;
            each(l_tag, [&](int i, const float (&b)[10]) { tmp[i] = b[9] * rhs[i]; });
            each(l_tag, [&](int i, const float (&b)[10]) {
                const float t = rhs[i] - bottom_row<L, ORD>(b, tmp, i);
                x[i] = tmp[i] + t * b[9];
            });
            each(l_tag, [&](int i, const float (&b)[10]) { tmp[i] = rhs[i] - bottom_row<L, ORD>(b, x, i); });
            float * crhs = lds + kBottomOff<L - 1>;
            for (int c = tid; c < Nc * Nc; c += kBottomLanes)
            {
                const int r = c / Nc, s = c - r * Nc;
                crhs[c] = k::restrict_node<float>(
                    [&](int dr, int ds) { return tmp[min(max((2 * r + dr) * m + 2 * s + ds, 0), n - 1)]; }, r, s, Nc,
                    ba.mk);
            }
            lds_barrier();
        };
        // x_in = x + alpha P(coarse iterate), then two sweeps into tmp
        auto up = [&](auto l_tag) {
            constexpr int L = decltype(l_tag)::value, n = kSize<L>, m = kSide<L>;
            const float * rhs = lds + kBottomOff<L>;
            float * x = lds + kBottomOff<L> + n;
            float * tmp = x + n;
            // the coarse solve's x, or the level below's tmp
            const float * cf = lds + kBottomOff<L - 1> + (L - 1 == MINL ? 1 : 2) * kSize<L - 1>;
            each(l_tag, [&](int i, const float (&)[10]) {
                const int R = i / m, S = i - R * m, Nc = kSide<L - 1>;
                const int ra = (R >> 1) * Nc, rb = ((R + 1) >> 1) * Nc, j = S >> 1, j1 = min(j + 1, Nc - 1);
                const float c[4] = {cf[ra + j], cf[ra + j1], cf[rb + j], cf[rb + j1]};
                tmp[i] = x[i] + ba.alpha * k::prolongation_node_v<float>(c, m, ba.mk, R, S);
            });
            each(l_tag, [&](int i, const float (&b)[10]) {
                const float t = rhs[i] - bottom_row<L, ORD>(b, tmp, i);
                x[i] = tmp[i] + t * b[9];
            });
            each(l_tag, [&](int i, const float (&b)[10]) {
                const float t = rhs[i] - bottom_row<L, ORD>(b, x, i);
                tmp[i] = x[i] + t * b[9];
            });
        };
        if constexpr (TOP6)
        {
            down(IntC<6>{});
            load_low(6);
        }
        if (top >= 5) down(IntC<5>{});
        if (top >= 4) down(IntC<4>{});
        if (top >= 3) down(IntC<3>{});
        if (MINL == 1 && top >= 2) down(IntC<2>{});
        if constexpr (TOP6 && MINL == 2)
            load6();
        if (tid < 64)
        {
            constexpr int n = kSize<MINL>;
            const float rhs = lds[kBottomOff<MINL> + min(tid, n - 1)];
            const float x = bottom_cg<MINL, ORD>(MINL == 1 ? b1 : b2, rhs, ba.konv_rad, ba.max_iters, &sl.s->cg_iters);
            if (tid < n)
                lds[kBottomOff<MINL> + n + tid] = x;
        }
        lds_barrier();
        if (MINL == 1 && top >= 2) up(IntC<2>{});
        if constexpr (TOP6 && MINL == 1)
            load6();
        if (top >= 3) up(IntC<3>{});
        if (top >= 4) up(IntC<4>{});
        if (top >= 5) up(IntC<5>{});
        if constexpr (TOP6)
            up(IntC<6>{});
        {
            auto leave = [&](auto l_tag) {
                constexpr int L = decltype(l_tag)::value;
                float * g = sl.v[L][F_TMP];
                for (int i = tid; i < kSize<L>; i += kBottomLanes)
                    g[i] = lds[kBottomOff<L> + 2 * kSize<L> + i];
            };
            if constexpr (TOP6)
                leave(IntC<6>{});
            else if (top == 5)
                leave(IntC<5>{});
            else if (top == 4)
                leave(IntC<4>{});
            else if (top == 3)
                leave(IntC<3>{});
            else if (top == 2)
                leave(IntC<2>{});
        }
    }
}
