// mg_march.hh -- the V-cycle's one-pass level kernels of the MG engine: the
// first two sweeps with defect and restriction (v_pre2r), and prolongation
// with two sweeps and the defect (v_post2).  Included by mg_engine.hip.
//
// A wave owns a tile: kW<V> columns of th grid rows, V columns per lane, with
// a halo of kHalo<V> columns on either side, and marches down its rows with
// everything in registers: three-row rings of each stage's values, the
// horizontal neighbours read from the next lanes by DPP wave shifts that the
// multiplications take as an operand.  Waves share nothing, so there is no
// barrier and no LDS traffic between the stages.
//
// What bounds them: on large levels HBM, and the post-smoothing the vector
// units as well (finest 4097^2, 302 MB each and the tiles' halos: pre-smoothing
// 66 us for 364 MB, 5.4 TB/s, vector units busy 64% of the time; post-smoothing
// 74 us for 352 MB, 4.6 TB/s, 88%), on levels below 1025^2 the chain of th + 6
// steps (8 to 13 us a launch).  The form before, 256 columns per workgroup with
// the rings in LDS and two or three barriers a step, took 118 and 159 us there,
// 44 us a kernel at 2049^2 (now 20), 13 to 23 us from 65^2 to 513^2, and with
// plain bands and 64 slots at 513^2 204 and 235 us (now 105 and 114).
//
// A tile's lanes hold linear node indices i = r m + c for columns c0 - kHalo
// .. c0 + W + kHalo - 1, so columns past a grid row's ends are the
// neighbouring rows' nodes, exactly as q1_row's linear offsets are.  EDGE
// tiles (the first strip and those that reach the last column) treat them;
// other tiles have every column strictly inside the grid row.
#pragma once

namespace
{
    constexpr int kMarchWaves = 4;                       // waves (tiles) per workgroup
    template <int V> constexpr int kHalo = V == 2 ? 4 : 3;
    template <int V> constexpr int kW = 64 * V - 2 * kHalo<V>;   // 120 or 58 columns, even

    typedef float MarchF2 __attribute__((ext_vector_type(2), aligned(4)));
    typedef uint16_t MarchU2 __attribute__((aligned(1)));

    // The lane's value as held by the lane to the left / right (0 past the
    // wave's ends, which only halo columns see).  Every lane of the wave must
    // be active.
    __device__ __forceinline__ float from_left(float v)
    {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
    }
    __device__ __forceinline__ float from_right(float v)
    {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
    }

    // Tap o of a row for a lane: o = 0 the left neighbour of its first
    // column, 1 .. V its columns, V + 1 the right neighbour of its last.
    template <int V> __device__ __forceinline__ float tap(const float (&row)[V], int o)
    {
        return o == 0 ? from_left(row[V - 1]) : (o == V + 1 ? from_right(row[0]) : row[o - 1]);
    }

    // Row sum of A x at the lane's column o (0 .. V - 1) from the rows above,
    // at and below it, in q1_row's order.  G: each neighbour's index is tested
    // against [0, n) as q1_row does (i: the node's index); without it every
    // neighbour must lie in the matrix.
    template <int ORD, bool G, int V>
    __device__ __forceinline__ float march_sum(const float (&b)[10], const float (&up)[V], const float (&mid)[V],
                                               const float (&dn)[V], int o, int i, int n, int m)
    {
        float s = ORD == 1 ? 0.0f : b[4] * mid[o];
        auto put = [&](bool on, float w, float v) {
            const float t = s + w * v;
            s = (! G || on) ? t : s;
        };
        put(i - m - 1 >= 0, b[0], tap<V>(up, o));
        put(i - m >= 0, b[1], tap<V>(up, o + 1));
        put(i - m + 1 >= 0, b[2], tap<V>(up, o + 2));
        put(i - 1 >= 0, b[3], tap<V>(mid, o));
        if (ORD == 1)
            put(true, b[4], mid[o]);
        put(i + 1 < n, b[5], tap<V>(mid, o + 2));
        put(i + m - 1 < n, b[6], tap<V>(dn, o));
        put(i + m < n, b[7], tap<V>(dn, o + 1));
        put(i + m + 1 < n, b[8], tap<V>(dn, o + 2));
        return s;
    }

    // A wave's tile.
    template <int V> struct MarchTile
    {
        int n, m, r0, H, c0;
        int lane, c;         // c: the lane's first column offset, c0 - kHalo + V lane
        bool edge;
        __device__ __forceinline__ MarchTile(int n_, int m_, unsigned t, int th)
        {
            n = n_;
            m = m_;
            const int nst = (m + kW<V> - 1) / kW<V>;
            c0 = (int)(t % (unsigned)nst) * kW<V>;
            r0 = (int)(t / (unsigned)nst) * th;
            H = min(th, m - r0);
            lane = threadIdx.x & 63;
            c = c0 - kHalo<V> + V * lane;
            edge = c0 == 0 || c0 + kW<V> + kHalo<V> >= m;
        }
        // column o of the lane is one the tile stores
        __device__ __forceinline__ bool own(int o) const
        {
            const int q = V * lane + o;
            return q >= kHalo<V> && q < kHalo<V> + kW<V> && c + o < m;
        }
        // Index of the lane's first node in row r, clamped so that a load of V
        // elements there stays inside the arrays (which hold at least one
        // element of padding before and after; a pair may start at -1, whose
        // second node is node 0).
        __device__ __forceinline__ int at(int r) const { return min(max(r * m + c, V == 2 ? -1 : 0), n - 1); }
    };

    template <int V, bool EDGE>
    __device__ __forceinline__ void march_load(const MarchTile<V> & t, gptr<const float> p, int r, float (&out)[V])
    {
        if constexpr (EDGE)
        {
            const int i = t.at(r);
            if constexpr (V == 2)
            {
                const MarchF2 v = *(gptr<const MarchF2>)(p + i);
                out[0] = v.x;
                out[1] = v.y;
            }
            else
                out[0] = p[i];
        }
        else
        {
            // a wave-uniform base and a constant lane offset
            gptr<const float> q = p + (min(max(r, 0), t.m - 1) * t.m + t.c0 - kHalo<V>);
            if constexpr (V == 2)
            {
                const MarchF2 v = *((gptr<const MarchF2>)q + t.lane);
                out[0] = v.x;
                out[1] = v.y;
            }
            else
                out[0] = q[t.lane];
        }
    }

    // Stores the owned columns of row r (0 <= r < m).
    template <int V, bool EDGE>
    __device__ __forceinline__ void march_store(const MarchTile<V> & t, gptr<float> p, int r, const float (&v)[V])
    {
        if constexpr (EDGE || V == 1)
        {
#pragma unroll
            for (int o = 0; o < V; ++o)
                if (t.own(o))
                    p[r * t.m + t.c + o] = v[o];
        }
        else
        {
            // the halo is two whole lanes on either side
            if (t.own(0))
            {
                gptr<float> q = p + (r * t.m + t.c0 - kHalo<V>);
                MarchF2 w;
                w.x = v[0];
                w.y = v[1];
                *((gptr<MarchF2>)q + t.lane) = w;
            }
        }
    }

    // A tile's matrix rows.  CB 1: row codes (one byte per node, an index into
    // a table of the level's distinct rows of nine bands and dinv, held in
    // LDS).  `keep` holds the coefficients of the lane's columns while the
    // codes of the last rows stay the same in every lane, as they do in the
    // interior of a constant-coefficient level; other rows look theirs up.
    // CB 2: value codes (one 64-bit word per node, ten 4-bit indices), decoded
    // through their ten 16-entry tables in LDS.  CB 0: the bands and dinv
    // themselves, a three-row ring.
    template <int V, int CB> struct MarchRows;

    template <int V> struct MarchRows<V, 1>
    {
        uint32_t ring[3] = {}, next[3];   // the lane's V codes of a row
        float keep[V][10];
        int run = 0;                      // rows in a row whose codes are those of the row before
        const float * tab;                // LDS
        gptr<const uint8_t> code;

        template <bool EDGE> __device__ __forceinline__ void load(const MarchTile<V> & t, int I, int r)
        {
            gptr<const uint8_t> q = EDGE ? code + t.at(r)
                                         : code + (min(max(r, 0), t.m - 1) * t.m + t.c0 - kHalo<V> + V * t.lane);
            if constexpr (V == 2)
                next[I] = *(gptr<const MarchU2>)q;
            else
                next[I] = *q;
        }
        // the row of ring entry I in the lane's column o
        __device__ __forceinline__ void row(int I, int o, float (&b)[10]) const
        {
            typedef float F4 __attribute__((ext_vector_type(4)));
            const F4 * e = (const F4 *)(tab + 12 * ((ring[I] >> (8 * o)) & 255u));
            const F4 e0 = e[0], e1 = e[1], e2 = e[2];
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                b[k] = e0[k];
                b[4 + k] = e1[k];
            }
            b[8] = e2[0];
            b[9] = e2[1];
        }
        // row I enters; true when the codes of it and of the two rows before are the same
        __device__ __forceinline__ bool enter(int I)
        {
            ring[I] = next[I];
            const bool same = __ballot(ring[I] != ring[(I + 2) % 3]) == 0;
            run = same ? run + 1 : 0;
            if (run == 2)
#pragma unroll
                for (int o = 0; o < V; ++o)
                    row(I, o, keep[o]);
            return run >= 2;
        }
    };

    template <int V> struct MarchRows<V, 2>
    {
        uint64_t ring[3][V] = {}, next[3][V];
        const float * tab;                // LDS
        gptr<const uint64_t> code;

        template <bool EDGE> __device__ __forceinline__ void load(const MarchTile<V> & t, int I, int r)
        {
#pragma unroll
            for (int o = 0; o < V; ++o)
                next[I][o] = code[min(max(r * t.m + t.c + o, 0), t.n - 1)];
        }
        __device__ __forceinline__ void row(int I, int o, float (&b)[10]) const
        {
#pragma unroll
            for (int k = 0; k < 10; ++k)
                b[k] = tab[16 * k + (int)((ring[I][o] >> (4 * k)) & 15u)];
        }
        __device__ __forceinline__ bool enter(int I)
        {
#pragma unroll
            for (int o = 0; o < V; ++o)
                ring[I][o] = next[I][o];
            return false;
        }
    };

    template <int V> struct MarchRows<V, 0>
    {
        float ring[3][V][10], next[3][V][10];
        gptr<const float> bands, dinv;
        int64_t bs;
        template <bool EDGE> __device__ __forceinline__ void load(const MarchTile<V> & t, int I, int r)
        {
            float w[V];
#pragma unroll
            for (int k = 0; k < 10; ++k)
            {
                march_load<V, EDGE>(t, k < 9 ? bands + k * bs : dinv, r, w);
#pragma unroll
                for (int o = 0; o < V; ++o)
                    next[I][o][k] = w[o];
            }
        }
        __device__ __forceinline__ void row(int I, int o, float (&b)[10]) const
        {
#pragma unroll
            for (int k = 0; k < 10; ++k)
                b[k] = ring[I][o][k];
        }
        __device__ __forceinline__ bool enter(int I)
        {
#pragma unroll
            for (int o = 0; o < V; ++o)
#pragma unroll
                for (int k = 0; k < 10; ++k)
                    ring[I][o][k] = next[I][o][k];
            return true;
        }
    };

    // alpha P(coarse) around a tile's nodes (Prolongation<NONE>), formed as
    // the rows enter.  A lane keeps the coarse value(s) of the last row and
    // loads those of the next: coarse row (R + 1) >> 1 of fine row R, so an
    // odd R has its upper coarse row from the step before.  General form (V
    // = 1 or EDGE): two coarse columns J, J + 1 per lane (J = S >> 1 of the
    // first column S) and, where the lane's columns lie past the grid row's
    // ends, the row that they wrap to.  Other tiles: one coarse column per
    // lane, the next from the next lane; S is even.
    template <int V, bool EDGE> struct MarchProl
    {
        static constexpr bool kGen = EDGE || V == 1;
        gptr<const float> p;
        int Nc, dr, dr1, J, J1;
        bool flip;                        // the lane's first column is odd
        bool over;                        // V = 2: the lane's second column is column 0 of the next row
        int S;
        float cur[2] = {}, next[3][2];

        __device__ __forceinline__ void init(const MarchTile<V> & t, gptr<const float> coarse)
        {
            p = coarse;
            Nc = (t.m + 1) / 2;
            dr = 0;
            S = t.c;
            if (S < 0)
            {
                S += t.m;
                dr = -1;
            }
            else if (S >= t.m)
            {
                S -= t.m;
                dr = 1;
            }
            S = min(max(S, 0), t.m - 1);      // (lanes past the halo)
            over = V == 2 && S == t.m - 1;
            dr1 = over ? dr + 1 : dr;
            J = S >> 1;
            J1 = over ? 0 : min(J + 1, Nc - 1);
            flip = (S & 1) != 0;
            // the first row (r0 - 3, odd) also takes the coarse row above it
            load(t, 0, t.r0 - 4);
            cur[0] = next[0][0];
            cur[1] = kGen ? next[0][1] : 0.0f;
        }
        __device__ __forceinline__ void load(const MarchTile<V> & t, int I, int R)
        {
            if constexpr (kGen)
            {
                next[I][0] = p[((min(max(R + dr, 0), t.m - 1) + 1) >> 1) * Nc + J];
                next[I][1] = p[((min(max(R + dr1, 0), t.m - 1) + 1) >> 1) * Nc + J1];
            }
            else
            {
                const int q = ((min(max(R, 0), t.m - 1) + 1) >> 1) * Nc;
                next[I][0] = (p + (q + ((t.c0 - kHalo<V>) >> 1)))[t.lane];
            }
        }
        // x += alpha P at row R (the row that load(I, R) fetched for)
        __device__ __forceinline__ void add(const MarchTile<V> & t, int I, int R, float alpha, const k::Mask & mk,
                                            float (&x)[V])
        {
            const float a0 = cur[0], b0 = next[I][0];
            cur[0] = b0;
            if constexpr (kGen)
            {
                const float a1 = cur[1], b1 = next[I][1];
                cur[1] = b1;
                const int Rl = R + dr;
                const bool ro = (Rl & 1) != 0;
                // at an even column: the coarse value, or the mean of two rows'
                auto even = [&](float a, float b, bool odd) {
                    const float h = k::add_d(k::add_d(0.0f, 0.5, a), 0.5, b);
                    return odd ? h : b;
                };
                // between the columns: two terms on an even row, four on an odd one
                const float e2 = k::add_d(k::add_d(0.0f, 0.5, b0), 0.5, b1);
                const float o4 = k::add_d(k::add_d(k::add_d(k::add_d(0.0f, 0.25, a0), 0.25, a1), 0.25, b0), 0.25, b1);
                const float between = ro ? o4 : e2;
                float q[2];
                q[0] = flip ? between : even(a0, b0, ro);
                q[1] = (flip || over) ? even(a1, b1, ((R + dr1) & 1) != 0) : between;
#pragma unroll
                for (int o = 0; o < V; ++o)
                {
                    const bool w = o == 1 && over;
                    const int Rc = min(max(w ? R + dr1 : Rl, 0), t.m - 1);
                    if (k::dirichlet_rs(Rc, w ? 0 : S + o, t.m, mk))
                        q[o] = 0.0f;
                    x[o] = x[o] + alpha * q[o];
                }
            }
            else
            {
                const float a1 = from_right(a0), b1 = from_right(b0);
                float q0, q1;
                if ((R & 1) == 0)
                {
                    q0 = b0;
                    q1 = k::add_d(k::add_d(0.0f, 0.5, b0), 0.5, b1);
                }
                else
                {
                    q0 = k::add_d(k::add_d(0.0f, 0.5, a0), 0.5, b0);
                    q1 = k::add_d(k::add_d(k::add_d(k::add_d(0.0f, 0.25, a0), 0.25, a1), 0.25, b0), 0.25, b1);
                }
                // the first and last grid row (columns 0 and m - 1 lie in
                // EDGE tiles)
                if ((R == 0 && mk.dir[4]) || (R == t.m - 1 && mk.dir[6]))
                    q0 = q1 = 0.0f;
                x[0] = x[0] + alpha * q0;
                x[V - 1] = x[V - 1] + alpha * q1;
            }
        }
    };

    // The slots of a workgroup: K consecutive table entries from z K, which
    // share its matrix loads.  A slot that is not running borrows the arrays
    // of one that is for its loads and stores nothing.
    template <int K> struct MarchSlots
    {
        bool on[K];
        int at[K];
        __device__ __forceinline__ bool find(const Slot * T, unsigned z, int nslots)
        {
            int pick = -1;
#pragma unroll
            for (int q = 0; q < K; ++q)
            {
                const int s = (int)z * K + q;
                on[q] = s < nslots && live(T[s]) && T[s].s->run != 0;
                if (on[q] && pick < 0)
                    pick = s;
            }
#pragma unroll
            for (int q = 0; q < K; ++q)
                at[q] = on[q] ? (int)z * K + q : pick;
            return pick >= 0;
        }
    };

    // the level's table (CB 1: its distinct rows; CB 2: its values) in LDS
    template <int CB> constexpr int kTabFloats = CB == 1 ? 12 * kRowCodes : (CB == 2 ? 160 : 4);
    // (fetch: the lane's first entry, loaded while the slot's pointers are
    // still on their way; store: to LDS)
    template <int CB> __device__ __forceinline__ int tab_count(const LevelArgs & a)
    {
        return CB == 1 ? 12 * a.rows : (CB == 2 ? 160 : 0);
    }
    template <int CB> __device__ __forceinline__ float march_table_fetch(const LevelArgs & a)
    {
        if constexpr (CB == 0)
            return 0.0f;
        else
            return as_global<const float>(CB == 1 ? a.rtab : a.ctab)[min((int)threadIdx.x, tab_count<CB>(a) - 1)];
    }
    template <int CB> __device__ __forceinline__ void march_table_store(const LevelArgs & a, float first, float * tab)
    {
        if constexpr (CB != 0)
        {
            const gptr<const float> src = as_global<const float>(CB == 1 ? a.rtab : a.ctab);
            const int cnt = tab_count<CB>(a);
            if ((int)threadIdx.x < cnt)
                tab[threadIdx.x] = first;
            for (int q = threadIdx.x + 64 * kMarchWaves; q < cnt; q += 64 * kMarchWaves)
                tab[q] = src[q];
            lds_barrier();
        }
    }
    template <int V, int CB>
    __device__ __forceinline__ void march_matrix(MarchRows<V, CB> & rows, const LevelArgs & a, const float * tab)
    {
        if constexpr (CB == 0)
        {
            rows.bands = as_global<const float>((const float *)a.B.b[0]);
            rows.dinv = as_global<const float>(a.dinv);
            rows.bs = a.bs;
        }
        else
        {
            rows.tab = tab;
            if constexpr (CB == 1)
                rows.code = as_global<const uint8_t>(a.rcode);
            else
                rows.code = as_global<const uint64_t>(a.codes);
        }
    }

    // Restriction<NONE> of three rows 2r - 1, 2r, 2r + 1 of d' to coarse row r
    // (the lanes' even columns), in restrict_node's order.
    template <int V, bool EDGE>
    __device__ __forceinline__ void restrict_row(const MarchTile<V> & t, const float (&up)[V], const float (&mid)[V],
                                                 const float (&dn)[V], int r, int Nc, const k::Mask & mk,
                                                 gptr<float> co, bool on)
    {
        const float f[3][3] = {{tap<V>(up, 0), tap<V>(up, 1), tap<V>(up, 2)},
                               {tap<V>(mid, 0), tap<V>(mid, 1), tap<V>(mid, 2)},
                               {tap<V>(dn, 0), tap<V>(dn, 1), tap<V>(dn, 2)}};
        const int sc = t.c >> 1;
        const int lo = t.c0 >> 1, hi = lo + kW<V> / 2 - 1;    // the tile's coarse columns
        float v;
        if (! EDGE && r >= 1 && r <= Nc - 2 && (hi < r - 1 || lo > r + 1))
        {
            // away from the border and from the diagonal every column's
            // additions come in one order (restrict_node: s < r-1, s > r+1)
            v = f[1][1];
            if (hi < r - 1)
            {
                v = k::add_d(v, 0.5, f[1][0]);
                v = k::add_d(v, 0.5, f[1][2]);
            }
            v = k::add_d(v, 0.5, f[0][1]);
            v = k::add_d(v, 0.25, f[0][2]);
            v = k::add_d(v, 0.25, f[0][0]);
            v = k::add_d(v, 0.5, f[2][1]);
            v = k::add_d(v, 0.25, f[2][2]);
            v = k::add_d(v, 0.25, f[2][0]);
            if (hi >= r - 1)
            {
                v = k::add_d(v, 0.5, f[1][0]);
                v = k::add_d(v, 0.5, f[1][2]);
            }
        }
        else
            v = k::restrict_node<float>([&](int ddr, int dds) { return f[ddr + 1][dds + 1]; }, r, sc, Nc, mk);
        if (on && t.own(0) && (V == 2 || (t.c & 1) == 0))
            co[r * Nc + sc] = v;
    }

    // ------------------------------------------- post-smoothing in one pass
    // Two damped-Jacobi sweeps x1 = x + dinv (rhs - A x), x2 = x1 + dinv (rhs
    // - A x1) and, with DEFECT, d = rhs - A x2 and the tile's |d|^2 (a partial
    // sum of the slot).  PROL: x is first corrected
    // by alpha P(level L-1's field fcoarse).  x2 goes to field fout (not fx:
    // neighbouring tiles read x around their own rows).  Every value is the
    // one the separate kernels form.
    //
    // Step s takes x at row r0 + s - 3 and the matrix and rhs at the row
    // before it (loaded three steps ahead), and forms x1 at row s - 4, x2 at
    // s - 5 and d at s - 6.
    template <int MK, int DEFECT, int PROL, int K, int V, int CB>
    __global__ __launch_bounds__(64 * kMarchWaves) void v_post2_kernel(LevelArgs a, const Slot * T, int L, int fx,
            int fout, int fcoarse, float alpha, k::Mask mk, int th, unsigned tiles, int nslots)
    {
        const VB vb = vblock();
        const float tab0 = march_table_fetch<CB>(a);
        MarchSlots<K> sl;
        if (! sl.find(T, vb.z, nslots))
            return;
        __shared__ __align__(16) float tab[kTabFloats<CB>];
        march_table_store<CB>(a, tab0, tab);
        const unsigned blk = gridDim.z == 1 ? k::xcd_block(vb.x, gridDim.x) : vb.x;
        const unsigned tile = blk * kMarchWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (tile >= tiles)
            return;
        const MarchTile<V> t((int)a.n, (int)a.m, tile, th);
        const int n = t.n, m = t.m, r0 = t.r0, H = t.H;
        gptr<const float> x[K], rhs[K], xc[K];
        gptr<float> out[K], dout[K];
#pragma unroll
        for (int q = 0; q < K; ++q)
        {
            const Slot & z = T[sl.at[q]];
            x[q] = as_global<const float>(z.v[L][fx]);
            rhs[q] = as_global<const float>(z.v[L][F_RHS]);
            out[q] = as_global<float>(z.v[L][fout]);
            dout[q] = as_global<float>(z.v[L][F_D]);
            xc[q] = as_global<const float>(PROL ? z.v[L - 1][fcoarse] : z.v[L][fx]);
        }
        auto march = [&](auto edge_tag) {
            constexpr bool EDGE = decltype(edge_tag)::value;
            constexpr int ORD = kOrd<MK>;
            MarchRows<V, CB> rows;
            march_matrix<V, CB>(rows, a, tab);
            MarchProl<V, EDGE> prol[K];
            float xr[K][3][V] = {}, x1r[K][3][V] = {}, x2r[K][3][V] = {}, rr[K][3][V] = {};
            float xn[K][3][V], rn[K][3][V];
            double dd[K] = {};                // |d|^2 over the lane's stored nodes
            auto load = [&](int I, int s) {
#pragma unroll
                for (int q = 0; q < K; ++q)
                {
                    march_load<V, EDGE>(t, x[q], r0 + s - 3, xn[q][I]);
                    if (PROL)
                        prol[q].load(t, I, r0 + s - 3);
                    march_load<V, EDGE>(t, rhs[q], r0 + s - 4, rn[q][I]);
                }
                rows.template load<EDGE>(t, I, r0 + s - 4);
            };
#pragma unroll
            for (int q = 0; q < K; ++q)
                if (PROL)
                    prol[q].init(t, xc[q]);
            auto step = [&](auto i_tag, int s) {
                constexpr int I = decltype(i_tag)::value, P = (I + 2) % 3, O = (I + 1) % 3;
                const bool same = rows.enter(I);
#pragma unroll
                for (int q = 0; q < K; ++q)
                {
#pragma unroll
                    for (int o = 0; o < V; ++o)
                    {
                        xr[q][I][o] = xn[q][I][o];
                        rr[q][I][o] = rn[q][I][o];
                    }
                    if (PROL)
                        prol[q].add(t, I, r0 + s - 3, alpha, mk, xr[q][I]);
                }
                load(I, s + 3);
                const int r1 = r0 + s - 4, r2 = r1 - 1, r3 = r1 - 2;
                // stage rows 2 .. m - 3: every neighbour of every lane's node
                // lies in the matrix (a first step's stages whose rows have
                // not entered yet form values that no stored one depends on)
                const bool inside = r3 >= 2 && r1 <= m - 3;
                // coef(J, o, b): the matrix row of ring entry J in column o
                auto stage = [&](auto g_tag, auto && coef) {
                    constexpr bool G = decltype(g_tag)::value;
                    auto ok = [&](int r, int o) { return ! G || (uint32_t)(r * m + t.c + o) < (uint32_t)n; };
#pragma unroll
                    for (int q = 0; q < K; ++q)
                    {
                        if (! G || s >= 2)
#pragma unroll
                            for (int o = 0; o < V; ++o)
                            {
                                float b[10];
                                coef(I, o, b);
                                const float sum = march_sum<ORD, G, V>(b, xr[q][O], xr[q][P], xr[q][I], o,
                                                                       r1 * m + t.c + o, n, m);
                                const float tt = rr[q][I][o] - sum;
                                const float v = xr[q][P][o] + tt * b[9];
                                x1r[q][I][o] = ok(r1, o) ? v : 0.0f;
                            }
                        if (! G || s >= 4)
                        {
#pragma unroll
                            for (int o = 0; o < V; ++o)
                            {
                                float b[10];
                                coef(P, o, b);
                                const float sum = march_sum<ORD, G, V>(b, x1r[q][O], x1r[q][P], x1r[q][I], o,
                                                                       r2 * m + t.c + o, n, m);
                                const float tt = rr[q][P][o] - sum;
                                const float v = x1r[q][P][o] + tt * b[9];
                                x2r[q][I][o] = ok(r2, o) ? v : 0.0f;
                            }
                            if (sl.on[q] && r2 >= r0 && r2 < r0 + H)
                                march_store<V, EDGE>(t, out[q], r2, x2r[q][I]);
                        }
                        if (DEFECT && (! G || s >= 6))
                        {
                            float d[V];
#pragma unroll
                            for (int o = 0; o < V; ++o)
                            {
                                float b[10];
                                coef(O, o, b);
                                const float sum = march_sum<ORD, G, V>(b, x2r[q][O], x2r[q][P], x2r[q][I], o,
                                                                       r3 * m + t.c + o, n, m);
                                d[o] = rr[q][O][o] - sum;
                            }
                            if (sl.on[q] && r3 >= r0 && r3 < r0 + H)
                            {
                                march_store<V, EDGE>(t, dout[q], r3, d);
#pragma unroll
                                for (int o = 0; o < V; ++o)
                                    if (t.own(o))
                                        dd[q] += (double)d[o] * (double)d[o];
                            }
                        }
                    }
                };
                auto look_up = [&](int J, int o, float (&b)[10]) { rows.row(J, o, b); };
                if (same && inside)
                {
                    if constexpr (CB == 1)
                        stage(std::false_type{}, [&](int, int o, float (&b)[10]) {
#pragma unroll
                            for (int k = 0; k < 10; ++k)
                                b[k] = rows.keep[o][k];
                        });
                    else
                        stage(std::false_type{}, look_up);
                }
                else
                    stage(std::true_type{}, look_up);
            };
            load(0, 0);
            load(1, 1);
            load(2, 2);
            const int steps = H + (DEFECT ? 6 : 5);
            for (int s = 0; s < steps; s += 3)
            {
                step(IntC<0>{}, s);
                step(IntC<1>{}, s + 1);
                step(IntC<2>{}, s + 2);
            }
            if (DEFECT)
#pragma unroll
                for (int q = 0; q < K; ++q)
                {
                    const double sum = k::wave_sum(dd[q]);
                    if (sl.on[q] && t.lane == 0)
                        T[sl.at[q]].partials[kCyclePartials + tile] = sum;
                }
        };
        if (t.edge)
            march(std::true_type{});
        else
            march(std::false_type{});
    }

    // ---------------------- pre-smoothing, defect and restriction in one pass
    // The first two damped-Jacobi sweeps from zero (c1 = dinv d, c2 = c1 +
    // dinv (d - A c1)), x = c2 (ACC: x = (field facc) + c2), the defect d' =
    // rhs - A x and the coarse right-hand side Restriction<NONE>(d') with the
    // Dirichlet mask.  Every value is the one the separate kernels form; d'
    // is never stored.  th is even, so a tile's first row is even and it owns
    // the coarse rows r with 2r in its rows.
    //
    // Step s takes d and the matrix at row r0 + s - 3 (loaded three steps
    // ahead), forms c1 there, x at row s - 4 and d' at s - 5, and, when that
    // row is 2r + 1, coarse row r.
    template <int MK, int ACC, int K, int V, int CB>
    __global__ __launch_bounds__(64 * kMarchWaves) void v_pre2r_kernel(LevelArgs a, const Slot * T, int L, int facc,
            int64_t Nc64, k::Mask mk, int th, unsigned tiles, int nslots, int fold)
    {
        const VB vb = vblock();
        const float tab0 = march_table_fetch<CB>(a);
        MarchSlots<K> sl;
        if (! sl.find(T, vb.z, nslots))
            return;
        __shared__ __align__(16) float tab[kTabFloats<CB>];
        march_table_store<CB>(a, tab0, tab);
        const unsigned blk = gridDim.z == 1 ? k::xcd_block(vb.x, gridDim.x) : vb.x;
        const unsigned tile = blk * kMarchWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (tile >= tiles)
            return;
        const MarchTile<V> t((int)a.n, (int)a.m, tile, th);
        const int n = t.n, m = t.m, r0 = t.r0, H = t.H, Nc = (int)Nc64;
        gptr<const float> d[K], rhs[K], acc[K];
        gptr<float> xo[K], co[K];
#pragma unroll
        for (int q = 0; q < K; ++q)
        {
            const Slot & z = T[sl.at[q]];
            // d is field F_D on the finest level (ACC), but rhs itself in an
            // inner solve's first cycle where no F_D was written (fold)
            const bool from_rhs = ! ACC || (fold && z.s->inner_last == 0);
            d[q] = as_global<const float>(z.v[L][from_rhs ? F_RHS : F_D]);
            rhs[q] = as_global<const float>(z.v[L][F_RHS]);
            acc[q] = as_global<const float>(z.v[L][facc]);
            xo[q] = as_global<float>(z.v[L][F_X]);
            co[q] = as_global<float>(z.v[L - 1][F_RHS]);
        }
        auto march = [&](auto edge_tag) {
            constexpr bool EDGE = decltype(edge_tag)::value;
            constexpr int ORD = kOrd<MK>;
            MarchRows<V, CB> rows;
            march_matrix<V, CB>(rows, a, tab);
            float cr[K][3][V] = {}, xr[K][3][V] = {}, er[K][3][V] = {}, dr[K][3][V] = {};
            float dn[K][3][V], an[K][3][V], rn[K][3][V];
            auto load = [&](int I, int s) {
#pragma unroll
                for (int q = 0; q < K; ++q)
                {
                    march_load<V, EDGE>(t, d[q], r0 + s - 3, dn[q][I]);
                    if (ACC)
                    {
                        march_load<V, EDGE>(t, acc[q], r0 + s - 4, an[q][I]);
                        march_load<V, EDGE>(t, rhs[q], r0 + s - 5, rn[q][I]);
                    }
                }
                rows.template load<EDGE>(t, I, r0 + s - 3);
            };
            auto step = [&](auto i_tag, int s) {
                constexpr int I = decltype(i_tag)::value, P = (I + 2) % 3, O = (I + 1) % 3;
                const bool same = rows.enter(I);
                float av[K][V], rv[K][V];
#pragma unroll
                for (int q = 0; q < K; ++q)
#pragma unroll
                    for (int o = 0; o < V; ++o)
                    {
                        dr[q][I][o] = dn[q][I][o];
                        av[q][o] = ACC ? an[q][I][o] : 0.0f;
                        rv[q][o] = ACC ? rn[q][I][o] : dr[q][O][o];
                    }
                load(I, s + 3);
                const int rc = r0 + s - 3, r1 = rc - 1, r2 = rc - 2;
                // rows r1 and r2 within 2 .. m - 3 (as v_post2_kernel) and row
                // rc in the grid
                const bool inside = r2 >= 2 && r1 <= m - 3;
                // coef(J, o, b): the matrix row of ring entry J in column o
                auto stage = [&](auto g_tag, auto && coef) {
                    constexpr bool G = decltype(g_tag)::value;
                    auto ok = [&](int r, int o) { return ! G || (uint32_t)(r * m + t.c + o) < (uint32_t)n; };
#pragma unroll
                    for (int q = 0; q < K; ++q)
                    {
#pragma unroll
                        for (int o = 0; o < V; ++o)
                        {
                            float b[10];
                            coef(I, o, b);
                            const float v = b[9] * dr[q][I][o];
                            cr[q][I][o] = ok(rc, o) ? v : 0.0f;
                        }
                        if (! G || s >= 2)
                        {
#pragma unroll
                            for (int o = 0; o < V; ++o)
                            {
                                float b[10];
                                coef(P, o, b);
                                const float sum = march_sum<ORD, G, V>(b, cr[q][O], cr[q][P], cr[q][I], o,
                                                                       r1 * m + t.c + o, n, m);
                                const float tt = dr[q][P][o] - sum;
                                const float c2 = cr[q][P][o] + tt * b[9];
                                const float v = ACC ? av[q][o] + c2 : c2;
                                xr[q][I][o] = ok(r1, o) ? v : 0.0f;
                            }
                            if (sl.on[q] && r1 >= r0 && r1 < r0 + H)
                                march_store<V, EDGE>(t, xo[q], r1, xr[q][I]);
                        }
                        if (! G || s >= 4)
                        {
#pragma unroll
                            for (int o = 0; o < V; ++o)
                            {
                                float b[10];
                                coef(O, o, b);
                                const float sum = march_sum<ORD, G, V>(b, xr[q][O], xr[q][P], xr[q][I], o,
                                                                       r2 * m + t.c + o, n, m);
                                const float v = rv[q][o] - sum;
                                er[q][I][o] = ok(r2, o) ? v : 0.0f;
                            }
                            if ((r2 & 1) != 0 && r2 > r0 && r2 <= r0 + H)
                                restrict_row<V, EDGE>(t, er[q][O], er[q][P], er[q][I], (r2 - 1) >> 1, Nc, mk, co[q],
                                                      sl.on[q]);
                        }
                    }
                };
                auto look_up = [&](int J, int o, float (&b)[10]) { rows.row(J, o, b); };
                if (same && inside)
                {
                    if constexpr (CB == 1)
                        stage(std::false_type{}, [&](int, int o, float (&b)[10]) {
#pragma unroll
                            for (int k = 0; k < 10; ++k)
                                b[k] = rows.keep[o][k];
                        });
                    else
                        stage(std::false_type{}, look_up);
                }
                else
                    stage(std::true_type{}, look_up);
            };
            load(0, 0);
            load(1, 1);
            load(2, 2);
            const int steps = H + 6;
            for (int s = 0; s < steps; s += 3)
            {
                step(IntC<0>{}, s);
                step(IntC<1>{}, s + 1);
                step(IntC<2>{}, s + 2);
            }
        };
        if (t.edge)
            march(std::true_type{});
        else
            march(std::false_type{});
    }
}
