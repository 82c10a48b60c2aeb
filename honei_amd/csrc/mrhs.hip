// mrhs.hip -- many right-hand sides on one ELL matrix.
//
// A *column-blocked multivector* of R <= 64 columns keeps row i's R entries
// contiguous at [i * R, i * R + R): a wavefront owns one row at a time with
// lane j on column j, so every gather of x[col] is one 8 R-byte coalesced
// load and every matrix entry is read once for all columns.
//
//   hsolve_ell_spmm    Y = A X or Y = RHS - A X (Product / Defect,
//                      product.hh:148-206, defect.hh:357-384, per column)
//   hsolve_cg_ell_multi CGSolver<Tag, NONE | VAR> (cg.hh:63-219) on every
//                      column at once: each column follows the reference's
//                      scalar recurrences and stopping test step for step
//                      (its own alpha, lambda, iteration count and
//                      convergence flag); converged columns stop loading.
//   hsolve_rhs_uniform_multi  seeded U[-1, 1] right-hand sides with zeros on
//                      the Dirichlet nodes of a macro border mask.
//
// Work split: rows are cut into tiles of 64; each block takes a contiguous
// range of tiles (in XCD-contiguous block order, so the rows +-side away
// that a Q1 row gathers stay in one XCD's L2) and its 4 waves take every
// 4th tile of the range.  A wave loads a tile's ELL slots with one
// coalesced load per slot (lane l on row base + l) and hands them to the
// row loop by readlane.  Per-column reductions accumulate per lane in
// double in the wave's row order, then over the 4 waves, then over the
// blocks in block order (a one-block finish launch), so results are
// deterministic.
#include "ell_handle.hh"
#include "kernels_mg.hh"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace hsolve
{
namespace
{
    constexpr int kMaxCols = 64;           // columns of a multivector (one per lane)
    constexpr int kTileK = 16;             // most ELL slots per row a tile keeps in registers
    constexpr unsigned kMvBlocks = 2048;   // grid cap of the multivector kernels
    constexpr int kFinThreads = 256;       // threads of the finish launches (one block per column)

    template <typename DT, typename IT, typename LT> struct MvEll
    {
        const IT * Aj;
        const DT * Ax;
        const LT * Arl;
        uint64_t stride;
        int64_t n;
        uint32_t ncpr;
        int64_t q1_side;       // hsolve_ell_s::q1_side
    };

    __device__ __forceinline__ uint32_t rlane(uint32_t v, int l)
    {
        return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
    }
    __device__ __forceinline__ float rlane(float v, int l)
    {
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
    }
    __device__ __forceinline__ double rlane(double v, int l)
    {
        const long long b = __double_as_longlong(v);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
        return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
    }

    // The tiles of the calling wave: block range in XCD-contiguous order,
    // every 4th tile of it.
    struct TileRange
    {
        int64_t first, end, step;
    };
    __device__ __forceinline__ TileRange wave_tiles(int64_t tiles)
    {
        const uint32_t b = k::xcd_block(blockIdx.x, gridDim.x);
        const int64_t per = (tiles + gridDim.x - 1) / gridDim.x;
        const int64_t lo = (int64_t)b * per;
        const int64_t hi = lo + per < tiles ? lo + per : tiles;
        const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        return TileRange{lo + wid, hi, (int64_t)(blockDim.x >> 6)};
    }

    // Calls f(row, sum_j) for every row of the tile at `base`, sum_j = row
    // of A times column j of X (lane j), the row's slots summed from zero in
    // ascending slot order (product.hh:192-202), and own_j = OWN[row][j]
    // (0 when OWN is null).  K >= num_cols_per_row: the tile keeps K slots
    // per row in registers (unused slots point at the row itself), and each
    // row issues all K gathers and the OWN load before the first add, so a
    // row costs one memory round trip.
    template <int K, typename DT, typename IT, typename LT, typename F>
    __device__ __forceinline__ void tile_rows(const MvEll<DT, IT, LT> & A, const DT * __restrict__ X,
                                              const DT * __restrict__ OWN, unsigned R, int64_t base, bool on, F && f)
    {
        const int lane = threadIdx.x & 63;
        const int64_t myrow = base + lane;
        const int rows = (int)(A.n - base < 64 ? A.n - base : 64);
        uint32_t len = 0;
        if (myrow < A.n)
            len = (uint32_t)A.Arl[myrow];
        const uint32_t self = myrow < A.n ? (uint32_t)myrow : 0u;
        // every stored slot (k < num_cols_per_row) of the tile's rows in one
        // batch of coalesced loads, then the row lengths applied
        IT rc[K];
        DT ra[K];
#pragma unroll
        for (int kk = 0; kk < K; ++kk)
        {
            rc[kk] = IT(0);
            ra[kk] = DT(0);
            if ((uint32_t)kk < A.ncpr)
            {
                const uint64_t at = (uint64_t)kk * A.stride + (uint64_t)self;
                rc[kk] = k::ld_stream(A.Aj + at);
                ra[kk] = k::ld_stream(A.Ax + at);
            }
        }
        uint32_t c[K];
        DT a[K];
#pragma unroll
        for (int kk = 0; kk < K; ++kk)
        {
            const bool in = (uint32_t)kk < len;
            c[kk] = in ? (uint32_t)k::col_of<IT>(rc[kk], (uint64_t)myrow) : self;
            a[kk] = in ? ra[kk] : DT(0);
        }
        for (int r = 0; r < rows; ++r)
        {
            DT xv[K];
#pragma unroll
            for (int kk = 0; kk < K; ++kk)
            {
                const uint32_t col = rlane(c[kk], r);
                xv[kk] = on ? X[(uint64_t)col * R + lane] : DT(0);
            }
            const DT ov = (on && OWN) ? OWN[(uint64_t)(base + r) * R + lane] : DT(0);
            const uint32_t lr = rlane(len, r);
            DT sum = DT(0);
#pragma unroll
            for (int kk = 0; kk < K; ++kk)
            {
                if ((uint32_t)kk < lr)
                    sum += rlane(a[kk], r) * xv[kk];
            }
            f(base + r, sum, ov);
        }
    }

    // The slots of a tile's rows (lane l: row base + l) of a Q1-structured
    // matrix in their 9 neighbour positions: values and presence bits.
    template <typename DT, typename IT, typename LT>
    __device__ __forceinline__ void q1_slots(const MvEll<DT, IT, LT> & A, int64_t base, DT (&ap)[9], uint32_t & mask)
    {
        const int lane = threadIdx.x & 63;
        const int64_t n = A.n, M = A.q1_side;
        const int64_t myrow = base + lane;
        const uint32_t self = myrow < n ? (uint32_t)myrow : 0u;
        const uint32_t len = myrow < n ? (uint32_t)A.Arl[myrow] : 0u;
        IT rc[9];
        DT ra[9];
#pragma unroll
        for (int kk = 0; kk < 9; ++kk)
        {
            rc[kk] = IT(0);
            ra[kk] = DT(0);
            if ((uint32_t)kk < A.ncpr)
            {
                const uint64_t at = (uint64_t)kk * A.stride + (uint64_t)self;
                rc[kk] = k::ld_stream(A.Aj + at);
                ra[kk] = k::ld_stream(A.Ax + at);
            }
        }
        mask = 0;
#pragma unroll
        for (int q = 0; q < 9; ++q)
            ap[q] = DT(0);
#pragma unroll
        for (int kk = 0; kk < 9; ++kk)
        {
            if ((uint32_t)kk < len)
            {
                const int64_t d = (int64_t)k::col_of<IT>(rc[kk], (uint64_t)myrow) - myrow;
                const int p = d < -1 ? (int)(d + M) + 1 : (d > 1 ? (int)(d - M) + 7 : (int)d + 4);
#pragma unroll
                for (int q = 0; q < 9; ++q)
                    ap[q] = (p == q) ? ra[kk] : ap[q];
                mask |= 1u << p;
            }
        }
    }

    // The same for Q1-structured matrices (every stored column of row
    // (y, x) is a neighbour (y + dy, x + dx), |dy|, |dx| <= 1, ascending, on
    // a side-M grid).  The tile's slots are first sorted into their 9
    // neighbour positions (value, presence bit) per lane.  The wave then
    // walks the rows in order keeping the 3 x 3 window of X rows around the
    // current row in registers: one step right along a grid line drops the
    // window's left column and gathers the 3 entries of its new right column,
    // so a row costs 3 gathers instead of 9; 4 rows of one grid line issue
    // their 12 gathers together.  Present entries are summed in
    // position order, which is the slot order, so the result is the same
    // bits as tile_rows.  Window entries off the grid are read at a clamped
    // (valid) address and never summed.
    template <typename DT, typename IT, typename LT, typename F>
    __device__ __forceinline__ void tile_rows_q1(const MvEll<DT, IT, LT> & A, const DT * __restrict__ X,
                                                 const DT * __restrict__ OWN, unsigned R, int64_t base, bool on,
                                                 F && f)
    {
        const int lane = threadIdx.x & 63;
        const int64_t n = A.n, M = A.q1_side;
        const int rows = (int)(n - base < 64 ? n - base : 64);
        DT ap[9];
        uint32_t mask;
        q1_slots(A, base, ap, mask);
        auto at = [&](int64_t c) { return X[(uint64_t)(c < 0 ? 0 : (c >= n ? n - 1 : c)) * R + lane]; };
        auto row_sum = [&](int r, const DT (&w)[9]) {
            const uint32_t mr = rlane(mask, r);
            DT sum = DT(0);
#pragma unroll
            for (int q = 0; q < 9; ++q)
            {
                if ((mr >> q) & 1u)
                    sum += rlane(ap[q], r) * w[q];
            }
            return sum;
        };
        // c0[b], c1[b]: window columns x - 1 and x of the next row, band b
        // (grid line y - 1, y, y + 1); valid after a row of the same line
        DT c0[3], c1[3];
        bool have = false;
        int64_t x = base % M;
        int r = 0;
        while (r < rows)
        {
            const int64_t i = base + r;
            if (x == 0 || ! have)
            {
#pragma unroll
                for (int b = 0; b < 3; ++b)
                {
                    c0[b] = on ? at(i + (b - 1) * M - 1) : DT(0);
                    c1[b] = on ? at(i + (b - 1) * M) : DT(0);
                }
            }
            if (r + 4 <= rows && x + 3 < M)
            {
                // 4 rows of one grid line: their 12 new gathers in flight at once
                DT v[3][4], ov[4];
#pragma unroll
                for (int b = 0; b < 3; ++b)
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        v[b][u] = on ? at(i + (b - 1) * M + 1 + u) : DT(0);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    ov[u] = (on && OWN && OWN != X) ? OWN[(uint64_t)(i + u) * R + lane] : DT(0);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    DT w[9];
#pragma unroll
                    for (int b = 0; b < 3; ++b)
#pragma unroll
                        for (int d = 0; d < 3; ++d)
                        {
                            const int k = u + d;       // column x - 1 + k of band b
                            w[b * 3 + d] = k == 0 ? c0[b] : (k == 1 ? c1[b] : v[b][k - 2]);
                        }
                    f(i + u, row_sum(r + u, w), OWN == X ? w[4] : ov[u]);
                }
#pragma unroll
                for (int b = 0; b < 3; ++b)
                {
                    c0[b] = v[b][2];
                    c1[b] = v[b][3];
                }
                r += 4;
                x += 4;
            }
            else
            {
                DT w[9];
#pragma unroll
                for (int b = 0; b < 3; ++b)
                {
                    w[b * 3] = c0[b];
                    w[b * 3 + 1] = c1[b];
                    w[b * 3 + 2] = on ? at(i + (b - 1) * M + 1) : DT(0);
                }
                const DT ov = OWN == X ? w[4] : ((on && OWN) ? OWN[(uint64_t)i * R + lane] : DT(0));
                f(i, row_sum(r, w), ov);
#pragma unroll
                for (int b = 0; b < 3; ++b)
                {
                    c0[b] = w[b * 3 + 1];
                    c1[b] = w[b * 3 + 2];
                }
                r += 1;
                x += 1;
            }
            if (x >= M)
                x -= M;
            have = true;
        }
    }

    // The same for matrices with more than kTileK slots per row: the row's
    // slots are read with wave-uniform addresses.
    template <typename DT, typename IT, typename LT, typename F>
    __device__ __forceinline__ void tile_rows_long(const MvEll<DT, IT, LT> & A, const DT * __restrict__ X,
                                                   const DT * __restrict__ OWN, unsigned R, int64_t base, bool on,
                                                   F && f)
    {
        const int lane = threadIdx.x & 63;
        const int rows = (int)(A.n - base < 64 ? A.n - base : 64);
        for (int r = 0; r < rows; ++r)
        {
            const int64_t row = base + r;
            const uint32_t len = (uint32_t)A.Arl[row];
            DT sum = DT(0);
            for (uint32_t kk = 0; kk < len; ++kk)
            {
                const uint64_t at = (uint64_t)kk * A.stride + (uint64_t)row;
                const uint64_t col = k::col_of<IT>(A.Aj[at], (uint64_t)row);
                const DT val = A.Ax[at];
                if (on)
                    sum += val * X[col * R + lane];
            }
            f(row, sum, (on && OWN) ? OWN[(uint64_t)row * R + lane] : DT(0));
        }
    }

    // K: slots per row kept in registers (9 or 16), 0 for longer rows, -1
    // for Q1-structured matrices
    template <typename DT, typename IT, typename LT, int K, typename F>
    __device__ __forceinline__ void for_rows_spmv(const MvEll<DT, IT, LT> & A, const DT * __restrict__ X,
                                                  const DT * __restrict__ OWN, unsigned R, bool on, F && f)
    {
        const TileRange t = wave_tiles((A.n + 63) / 64);
        for (int64_t tile = t.first; tile < t.end; tile += t.step)
        {
            if constexpr (K == 0)
                tile_rows_long(A, X, OWN, R, tile * 64, on, f);
            else if constexpr (K < 0)
                tile_rows_q1(A, X, OWN, R, tile * 64, on, f);
            else
                tile_rows<K>(A, X, OWN, R, tile * 64, on, f);
        }
    }

    // f(row0, cnt) for the wave's rows in groups of G (cnt < G only at the
    // end of the matrix), in ascending row order: the callers issue the loads
    // of a group before its first store.
    template <int G, typename F>
    __device__ __forceinline__ void for_rows(int64_t n, F && f)
    {
        const TileRange t = wave_tiles((n + 63) / 64);
        for (int64_t tile = t.first; tile < t.end; tile += t.step)
        {
            const int64_t base = tile * 64;
            const int rows = (int)(n - base < 64 ? n - base : 64);
            for (int r = 0; r < rows; r += G)
                f(base + r, rows - r < G ? rows - r : G);
        }
    }

    // Y = A X (MODE 0) or Y = RHS - A X (MODE 1), every column
    template <typename DT, typename IT, typename LT, int K, int MODE>
    __global__ __launch_bounds__(256) void spmm_kernel(MvEll<DT, IT, LT> A, const DT * __restrict__ X,
                                                       DT * __restrict__ Y, const DT * __restrict__ RHS, unsigned R)
    {
        const unsigned lane = threadIdx.x & 63;
        const bool on = lane < R;
        for_rows_spmv<DT, IT, LT, K>(A, X, MODE == 0 ? nullptr : RHS, R, on, [&](int64_t row, DT sum, DT rhs) {
            if (! on)
                return;
            const uint64_t e = (uint64_t)row * R + lane;
            Y[e] = MODE == 0 ? sum : rhs - sum;
        });
    }

    // ------------------------------------------------------------ CG state
    template <typename DT> struct MState
    {
        DT alpha[kMaxCols], alpha_old[kMaxCols], alpha_new[kMaxCols], lambda[kMaxCols], talpha[kMaxCols];
        DT initial_defect[kMaxCols], current_defect[kMaxCols];
        uint64_t iters[kMaxCols];
        int run[kMaxCols], converged[kMaxCols];
        int pbuf[kMaxCols];  // the direction buffer of the column's last step (run_mcg's fused steps)
        DT eps_relative;
        uint64_t max_iters;
        int active;          // columns still iterating
    };

    template <typename DT> struct Eps;
    template <> struct Eps<float> { static constexpr float v = 1.19209290e-07F; };
    template <> struct Eps<double> { static constexpr double v = 2.2204460492503131e-16; };

    template <typename DT> __device__ __forceinline__ DT guard(DT v)
    {
        return (fabs(v) > Eps<DT>::v) ? v : Eps<DT>::v;
    }
    template <typename DT> __device__ __forceinline__ DT guard_signed(DT v)
    {
        return (fabs(v) > Eps<DT>::v) ? v : Eps<DT>::v * (v / (DT)fabs(v));
    }

    // Per-column reductions in two launches.  Each block stores, per column,
    // the sum of its 4 waves' lane sums in wave order (mput, no fence and no
    // atomic; column after column, so that a column's partials lie together);
    // a following launch of one block per column sums them (msum: 16 sums
    // over blocks w, w + 16, ..., then those in order) and applies the scalar
    // step on thread 0.  The kernel boundary orders the stores.  (One block for
    // all columns read its 0.5 to 1 MB of partials in 10 to 18 us.)
    template <int V>
    __device__ __forceinline__ void mput(const double (&acc)[V], double * partials)
    {
        __shared__ double lds[4][V][64];
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
        for (int v = 0; v < V; ++v)
            lds[wid][v][lane] = acc[v];
        __syncthreads();
        if (wid == 0)
        {
#pragma unroll
            for (int v = 0; v < V; ++v)
            {
                double s = lds[0][v][lane];
                s += lds[1][v][lane];
                s += lds[2][v][lane];
                s += lds[3][v][lane];
                partials[(uint64_t)(v * kMaxCols + lane) * gridDim.x + blockIdx.x] = s;
            }
        }
    }

    // block blockIdx.x sums column blockIdx.x's nb partials (kFinThreads threads)
    template <int V, typename F>
    __device__ __forceinline__ void msum(const double * partials, unsigned nb, F && fin)
    {
        constexpr int W = 16;
        __shared__ double lds[V][kMvBlocks];
        __shared__ double sums[V][W];
        const unsigned j = blockIdx.x;
#pragma unroll
        for (int v = 0; v < V; ++v)
            for (unsigned b = threadIdx.x; b < nb; b += kFinThreads)
                lds[v][b] = partials[(uint64_t)(v * kMaxCols + j) * nb + b];
        __syncthreads();
        if (threadIdx.x < (unsigned)(V * W))
        {
            const unsigned v = threadIdx.x / W, w = threadIdx.x % W;
            double t = 0.0;
#pragma unroll 8
            for (unsigned b = w; b < nb; b += W)
                t += lds[v][b];
            sums[v][w] = t;
        }
        __syncthreads();
        if (threadIdx.x == 0)
        {
            double tot[V];
#pragma unroll
            for (int v = 0; v < V; ++v)
            {
                double s = sums[v][0];
                for (int w = 1; w < W; ++w)
                    s += sums[v][w];
                tot[v] = s;
            }
            fin((int)j, tot);
        }
    }

    // R = B - A X; P = Pc * R (VAR) or R (NONE); per column r.r, r.p
    template <typename DT, typename IT, typename LT, int K, bool VAR>
    __global__ __launch_bounds__(256) void mcg_init_kernel(MvEll<DT, IT, LT> A, const DT * __restrict__ Bv,
            const DT * __restrict__ X, DT * __restrict__ Rv, DT * __restrict__ Pv, const DT * __restrict__ Pc,
            unsigned R, double * partials)
    {
        const unsigned lane = threadIdx.x & 63;
        const bool on = lane < R;
        double acc[2] = {0.0, 0.0};
        for_rows_spmv<DT, IT, LT, K>(A, X, Bv, R, on, [&](int64_t row, DT sum, DT bi) {
            if (! on)
                return;
            const uint64_t e = (uint64_t)row * R + lane;
            const DT ri = bi - sum;
            Rv[e] = ri;
            const DT pi = VAR ? Pc[row] * ri : ri;
            Pv[e] = pi;
            acc[0] += (double)ri * (double)ri;
            acc[1] += (double)ri * (double)pi;
        });
        mput<2>(acc, partials);
    }

    template <typename DT, bool VAR>
    __global__ __launch_bounds__(kFinThreads) void mcg_init_finish(const double * partials, unsigned nb, unsigned R,
            MState<DT> * s)
    {
        msum<2>(partials, nb, [&](int j, const double (&t)[2]) {
            s->iters[j] = 0;
            s->converged[j] = 0;
            s->run[j] = (s->max_iters > 0) ? 1 : 0;
            if (VAR)
            {
                s->initial_defect[j] = (DT)sqrt((DT)t[0]);
                s->alpha_new[j] = (DT)t[1];
            }
            else
            {
                s->alpha[j] = (DT)t[0];
                s->initial_defect[j] = (DT)sqrt((DT)t[0]);
            }
            s->current_defect[j] = s->initial_defect[j];
            if (j == 0)
                s->active = (s->max_iters > 0) ? (int)R : 0;
        });
    }

    // V = A P; per column temp = v.p and lambda
    template <typename DT, typename IT, typename LT, int K>
    __global__ __launch_bounds__(256) void mcg_spmv_kernel(MvEll<DT, IT, LT> A, const DT * __restrict__ Pv,
            DT * __restrict__ Vv, unsigned R, double * partials, const MState<DT> * s)
    {
        if (s->active == 0)
            return;
        const unsigned lane = threadIdx.x & 63;
        const bool on = lane < R && s->run[lane] != 0;
        double acc[1] = {0.0};
        for_rows_spmv<DT, IT, LT, K>(A, Pv, Pv, R, on, [&](int64_t row, DT sum, DT pi) {
            if (! on)
                return;
            Vv[(uint64_t)row * R + lane] = sum;
            acc[0] += (double)sum * (double)pi;
        });
        mput<1>(acc, partials);
    }

    template <typename DT, bool VAR>
    __global__ __launch_bounds__(kFinThreads) void mcg_spmv_finish(const double * partials, unsigned nb, unsigned R,
            MState<DT> * s)
    {
        if (s->run[blockIdx.x] == 0)
            return;
        msum<1>(partials, nb, [&](int j, const double (&t)[1]) {
            const DT temp = (DT)t[0];
            if (VAR)
                s->lambda[j] = s->alpha_new[j] / guard_signed<DT>(temp);
            else
                s->lambda[j] = s->alpha[j] / guard<DT>(temp);
        });
    }

    // X += lambda P; R += (-lambda) V; per column r.r (and r.(Pc r)); stopping test
    template <typename DT, bool VAR>
    __global__ __launch_bounds__(256) void mcg_update_kernel(DT * __restrict__ X, DT * __restrict__ Rv,
            const DT * __restrict__ Pv, const DT * __restrict__ Vv, const DT * __restrict__ Pc, int64_t n,
            unsigned R, double * partials, const MState<DT> * s)
    {
        if (s->active == 0)
            return;
        const unsigned lane = threadIdx.x & 63;
        const bool on = lane < R && s->run[lane] != 0;
        const DT lambda = on ? s->lambda[lane] : DT(0);
        const DT mlambda = -lambda;
        double acc[2] = {0.0, 0.0};
        if (on)
        {
            for_rows<4>(n, [&](int64_t row0, int cnt) {
                DT xv[4], pv[4], rv[4], vv[4], pc[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    const int64_t row = row0 + (u < cnt ? u : 0);
                    const uint64_t e = (uint64_t)row * R + lane;
                    xv[u] = X[e];
                    pv[u] = Pv[e];
                    rv[u] = Rv[e];
                    vv[u] = Vv[e];
                    pc[u] = VAR ? Pc[row] : DT(0);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                {
                    if (u < cnt)
                    {
                        const uint64_t e = (uint64_t)(row0 + u) * R + lane;
                        X[e] = xv[u] + lambda * pv[u];
                        const DT ri = rv[u] + mlambda * vv[u];
                        Rv[e] = ri;
                        acc[0] += (double)ri * (double)ri;
                        if (VAR)
                            acc[1] += (double)ri * (double)(pc[u] * ri);
                    }
                }
            });
        }
        mput<2>(acc, partials);
    }

    template <typename DT, bool VAR>
    __global__ __launch_bounds__(kFinThreads) void mcg_update_finish(const double * partials, unsigned nb, unsigned R,
            MState<DT> * s, int pbuf)
    {
        if (s->run[blockIdx.x] == 0)
            return;
        msum<2>(partials, nb, [&](int j, const double (&t)[2]) {
            const DT eps = s->eps_relative;
            s->pbuf[j] = pbuf;
            bool stop = false;
            if (VAR)
            {
                ++s->iters[j];
                const DT cur = (DT)sqrt((DT)t[0]);
                s->current_defect[j] = cur;
                if (cur < eps * s->initial_defect[j] || cur < eps)
                {
                    s->converged[j] = 1;
                    stop = true;
                }
                else if (s->iters[j] == s->max_iters)
                    stop = true;
                else
                {
                    s->alpha[j] = s->alpha_new[j];
                    s->alpha_new[j] = (DT)t[1];
                    s->talpha[j] = s->alpha_new[j] / guard_signed<DT>(s->alpha[j]);
                }
            }
            else
            {
                s->alpha_old[j] = s->alpha[j];
                s->alpha[j] = (DT)t[0];
                s->talpha[j] = s->alpha[j] / guard<DT>(s->alpha_old[j]);
                ++s->iters[j];
                const DT cur = (DT)sqrt(s->alpha[j]);
                s->current_defect[j] = cur;
                if (cur < eps * s->initial_defect[j] || cur < eps)
                {
                    s->converged[j] = 1;
                    stop = true;
                }
                else if (s->iters[j] == s->max_iters)
                    stop = true;
            }
            if (stop)
            {
                s->run[j] = 0;
                atomicSub(&s->active, 1);
            }
        });
    }

    // One step of every running column on a Q1-structured matrix, in one
    // pass: the update of X that the last step left (X += lambda P), the next
    // direction P' = P * talpha + Pc * R (VAR) or P * talpha + R, V = A P' and
    // the partials of v.p'.  The window of tile_rows_q1 holds P', formed
    // wherever it is read with the operations of mcg_direction_kernel; each
    // row stores its own into the other direction buffer.  With the update of
    // R alone in mcg_residual_kernel, a step moves nine vectors instead of
    // eleven and launches four kernels instead of five (513^2, 64 columns:
    // 221 + 72 us instead of 97 + 183 + 83).  X, V and P' pass the caches by
    // (non-temporal: the window's lines of P and R stay in L2, 496 instead of
    // 561 MB read; V and X are not read again before they would be evicted).
    // It moves 0.90 GB at 4.1 TB/s.
    template <typename DT, typename IT, typename LT, bool VAR>
    __global__ __launch_bounds__(256) void mcg_step_kernel(MvEll<DT, IT, LT> A, const DT * __restrict__ Pold,
            const DT * __restrict__ Rv, const DT * __restrict__ Pc, DT * __restrict__ Pnew, DT * __restrict__ Vv,
            DT * __restrict__ X, unsigned R, double * partials, const MState<DT> * s)
    {
        if (s->active == 0)
            return;
        const unsigned lane = threadIdx.x & 63;
        const bool on = lane < R && s->run[lane] != 0;
        const DT talpha = on ? s->talpha[lane] : DT(0), lambda = on ? s->lambda[lane] : DT(0);
        const int64_t n = A.n, M = A.q1_side;
        double acc[1] = {0.0};
        // P and Pc * R (or R) at row c, clamped to the matrix; dir: P'
        auto old_at = [&](int64_t c) { return on ? Pold[(uint64_t)c * R + lane] : DT(0); };
        auto res_at = [&](int64_t c) { return on ? Rv[(uint64_t)c * R + lane] : DT(0); };
        auto dir = [&](DT p, DT r, DT pc) {
            const DT t = p * talpha;
            return t + (VAR ? pc * r : r);
        };
        auto clamp = [&](int64_t c) { return c < 0 ? (int64_t)0 : (c >= n ? n - 1 : c); };
        // the tile's matrix values per wave, read back row by row (kept in
        // registers they leave room for four waves per SIMD instead of five,
        // and 1029 blocks of four waves then run in two rounds)
        __shared__ DT slots[4][64][9];
        DT (*const sl)[9] = slots[threadIdx.x >> 6];
        const TileRange t = wave_tiles((n + 63) / 64);
        for (int64_t tile = t.first; tile < t.end; tile += t.step)
        {
            const int64_t base = tile * 64;
            const int rows = (int)(n - base < 64 ? n - base : 64);
            uint32_t mask;
            {
                DT ap[9];
                q1_slots(A, base, ap, mask);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int q = 0; q < 9; ++q)
                    sl[lane][q] = ap[q];
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
            auto row_out = [&](int r, const DT (&w)[9], DT po, DT xv) {
                const uint32_t mr = rlane(mask, r);
                DT sum = DT(0);
#pragma unroll
                for (int q = 0; q < 9; ++q)
                {
                    if ((mr >> q) & 1u)
                        sum += sl[r][q] * w[q];
                }
                if (on)
                {
                    const uint64_t e = (uint64_t)(base + r) * R + lane;
                    __builtin_nontemporal_store(xv + lambda * po, X + e);
                    __builtin_nontemporal_store(w[4], Pnew + e);
                    __builtin_nontemporal_store(sum, Vv + e);
                    acc[0] += (double)sum * (double)w[4];
                }
            };
            // window columns x - 1 and x of the next row (P'), and P at (y, x)
            DT c0[3], c1[3], c1o = DT(0);
            bool have = false;
            int64_t x = base % M;
            int r = 0;
            while (r < rows)
            {
                const int64_t i = base + r;
                if (x == 0 || ! have)
                {
                    DT p[3][2], rr[3][2], pc[3][2];
#pragma unroll
                    for (int b = 0; b < 3; ++b)
#pragma unroll
                        for (int d = 0; d < 2; ++d)
                        {
                            const int64_t c = clamp(i + (b - 1) * M - 1 + d);
                            p[b][d] = old_at(c);
                            rr[b][d] = res_at(c);
                            pc[b][d] = VAR ? Pc[c] : DT(0);
                        }
#pragma unroll
                    for (int b = 0; b < 3; ++b)
                    {
                        c0[b] = dir(p[b][0], rr[b][0], pc[b][0]);
                        c1[b] = dir(p[b][1], rr[b][1], pc[b][1]);
                    }
                    c1o = p[1][1];
                }
                const bool four = r + 4 <= rows && x + 3 < M;
                const int cnt = four ? 4 : 1;
                DT p[3][4], rr[3][4], pc[3][4], xv[4];
                if (four)
                {
                    // 4 rows of one grid line: their 28 loads in flight at once
#pragma unroll
                    for (int b = 0; b < 3; ++b)
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                        {
                            const int64_t c = clamp(i + (b - 1) * M + 1 + u);
                            p[b][u] = old_at(c);
                            rr[b][u] = res_at(c);
                            pc[b][u] = VAR ? Pc[c] : DT(0);
                        }
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        xv[u] = on ? k::ld_stream(X + (uint64_t)(i + u) * R + lane) : DT(0);
                    DT v[3][4];
#pragma unroll
                    for (int b = 0; b < 3; ++b)
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            v[b][u] = dir(p[b][u], rr[b][u], pc[b][u]);
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                    {
                        DT w[9];
#pragma unroll
                        for (int b = 0; b < 3; ++b)
#pragma unroll
                            for (int d = 0; d < 3; ++d)
                            {
                                const int k = u + d;       // column x - 1 + k of band b
                                w[b * 3 + d] = k == 0 ? c0[b] : (k == 1 ? c1[b] : v[b][k - 2]);
                            }
                        row_out(r + u, w, u == 0 ? c1o : p[1][u > 0 ? u - 1 : 0], xv[u]);
                    }
#pragma unroll
                    for (int b = 0; b < 3; ++b)
                    {
                        c0[b] = v[b][2];
                        c1[b] = v[b][3];
                    }
                    c1o = p[1][3];
                }
                else
                {
#pragma unroll
                    for (int b = 0; b < 3; ++b)
                    {
                        const int64_t c = clamp(i + (b - 1) * M + 1);
                        p[b][0] = old_at(c);
                        rr[b][0] = res_at(c);
                        pc[b][0] = VAR ? Pc[c] : DT(0);
                    }
                    xv[0] = on ? k::ld_stream(X + (uint64_t)i * R + lane) : DT(0);
                    DT w[9];
#pragma unroll
                    for (int b = 0; b < 3; ++b)
                    {
                        w[b * 3] = c0[b];
                        w[b * 3 + 1] = c1[b];
                        w[b * 3 + 2] = dir(p[b][0], rr[b][0], pc[b][0]);
                    }
                    row_out(r, w, c1o, xv[0]);
#pragma unroll
                    for (int b = 0; b < 3; ++b)
                    {
                        c0[b] = w[b * 3 + 1];
                        c1[b] = w[b * 3 + 2];
                    }
                    c1o = p[1][0];
                }
                r += cnt;
                x += cnt;
                if (x >= M)
                    x -= M;
                have = true;
            }
        }
        mput<1>(acc, partials);
    }

    // R += (-lambda) V; per column r.r (and r.(Pc r)): mcg_update_kernel
    // without its update of X, which mcg_step_kernel or mcg_flush_kernel makes
    template <typename DT, bool VAR>
    __global__ __launch_bounds__(256) void mcg_residual_kernel(DT * __restrict__ Rv, const DT * __restrict__ Vv,
            const DT * __restrict__ Pc, int64_t n, unsigned R, double * partials, const MState<DT> * s)
    {
        if (s->active == 0)
            return;
        const unsigned lane = threadIdx.x & 63;
        const bool on = lane < R && s->run[lane] != 0;
        const DT mlambda = on ? -s->lambda[lane] : DT(0);
        double acc[2] = {0.0, 0.0};
        if (on)
        {
            for_rows<16>(n, [&](int64_t row0, int cnt) {
                DT rv[16], vv[16], pc[16];
#pragma unroll
                for (int u = 0; u < 16; ++u)
                {
                    const int64_t row = row0 + (u < cnt ? u : 0);
                    const uint64_t e = (uint64_t)row * R + lane;
                    rv[u] = Rv[e];
                    vv[u] = k::ld_stream(Vv + e);
                    pc[u] = VAR ? Pc[row] : DT(0);
                }
#pragma unroll
                for (int u = 0; u < 16; ++u)
                {
                    if (u < cnt)
                    {
                        const DT ri = rv[u] + mlambda * vv[u];
                        Rv[(uint64_t)(row0 + u) * R + lane] = ri;
                        acc[0] += (double)ri * (double)ri;
                        if (VAR)
                            acc[1] += (double)ri * (double)(pc[u] * ri);
                    }
                }
            });
        }
        mput<2>(acc, partials);
    }

    // The update of X that each column's last step left: X += lambda P, P in
    // the direction buffer of that step.
    template <typename DT>
    __global__ __launch_bounds__(256) void mcg_flush_kernel(DT * __restrict__ X, const DT * __restrict__ P0,
            const DT * __restrict__ P1, int64_t n, unsigned R, const MState<DT> * s)
    {
        const unsigned lane = threadIdx.x & 63;
        if (! (lane < R && s->iters[lane] != 0))
            return;
        const DT lambda = s->lambda[lane];
        const DT * P = s->pbuf[lane] ? P1 : P0;
        for_rows<4>(n, [&](int64_t row0, int cnt) {
            DT xv[4], pv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const uint64_t e = (uint64_t)(row0 + (u < cnt ? u : 0)) * R + lane;
                xv[u] = X[e];
                pv[u] = P[e];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (u < cnt)
                    X[(uint64_t)(row0 + u) * R + lane] = xv[u] + lambda * pv[u];
        });
    }

    // P = P * talpha + Pc * R (VAR) or P * talpha + R (NONE)
    template <typename DT, bool VAR>
    __global__ __launch_bounds__(256) void mcg_direction_kernel(DT * __restrict__ Pv, const DT * __restrict__ Rv,
            const DT * __restrict__ Pc, int64_t n, unsigned R, const MState<DT> * s)
    {
        if (s->active == 0)
            return;
        const unsigned lane = threadIdx.x & 63;
        if (! (lane < R && s->run[lane] != 0))
            return;
        const DT talpha = s->talpha[lane];
        for_rows<4>(n, [&](int64_t row0, int cnt) {
            DT pv[4], rv[4], pc[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                const int64_t row = row0 + (u < cnt ? u : 0);
                const uint64_t e = (uint64_t)row * R + lane;
                pv[u] = Pv[e];
                rv[u] = Rv[e];
                pc[u] = VAR ? Pc[row] : DT(0);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                if (u < cnt)
                {
                    const DT t = pv[u] * talpha;
                    Pv[(uint64_t)(row0 + u) * R + lane] = t + (VAR ? pc[u] * rv[u] : rv[u]);
                }
            }
        });
    }

    unsigned mv_grid(uint64_t n)
    {
        const uint64_t tiles = (n + 63) / 64;
        return (unsigned)std::min<uint64_t>(kMvBlocks, std::max<uint64_t>(1, (tiles + 3) / 4));
    }

    template <typename F>
    void with_mv(const hsolve_ell_s * m, F && f)
    {
        require(m->threads == 1, HSOLVE_ERR_INVALID, "multivector kernels need an ELL handle with threads == 1");
        require(m->rows < (1ull << 32) && m->cols < (1ull << 32), HSOLVE_ERR_SIZE, "multivector: rows >= 2^32");
        with_ell_types(m, [&](auto Aj, auto Arl) {
            using IT = std::remove_const_t<std::remove_pointer_t<decltype(Aj)>>;
            using LT = std::remove_const_t<std::remove_pointer_t<decltype(Arl)>>;
            auto run = [&](auto dt_tag) {
                using DT = decltype(dt_tag);
                MvEll<DT, IT, LT> A{Aj, (const DT *)m->Ax, Arl, m->stride, (int64_t)m->rows, (uint32_t)m->ncpr,
                                    (int64_t)m->q1_side};
                if (m->q1_side != 0 && m->ncpr <= 9 && (m->variant & HSOLVE_ELL_SET) == 0)
                    f(A, std::integral_constant<int, -1>());
                else if (m->ncpr <= 9)
                    f(A, std::integral_constant<int, 9>());
                else if (m->ncpr <= (uint64_t)kTileK)
                    f(A, std::integral_constant<int, kTileK>());
                else
                    f(A, std::integral_constant<int, 0>());
            };
            if (m->dtype)
                run(double(0));
            else
                run(float(0));
        });
    }

    template <typename DT, typename IT, typename LT, int K, bool VAR>
    void run_mcg(const MvEll<DT, IT, LT> & A, unsigned R, const DT * Bv, DT * X, const DT * Pc, uint64_t max_iters,
                 double eps, uint64_t * used, double * defect, int * converged, hipStream_t st)
    {
        const uint64_t n = (uint64_t)A.n;
        const size_t vb = ((sizeof(DT) * n * R + 255) / 256) * 256;
        const unsigned grid = mv_grid(n);
        const size_t pb = sizeof(double) * 2 * 64 * grid;
        // Q1-structured matrices: fused steps with a second direction buffer
        // (a step's gathers read P and R, three of each per row through the
        // window; other matrices would gather both for every entry)
        const size_t rest = pb + sizeof(MState<DT>) + 256;
        void * block = nullptr;
        // FP32 with a preconditioner: on small multivectors the fused step's
        // longer chain costs more than the vectors it saves.  Measured on MI355X,
        // us an iteration, fused and separate: 65^2 64 columns 70.8 / 67.0, 161^2
        // 80.9 / 73.1, 193^2 82.6 / 83.6, 257^2 90.1 / 97.8; 16 columns 65^2 72.5 / 70.5,
        // 321^2 87.7 / 82.7, 513^2 123.0 / 123.4; 2 columns 513^2 116.6 / 111.4.  (Without
        // one 65.5 / 66.3, 75.5 / 72.4, 77.3 / 82.3; FP64 71.5 / 79.1, 86.5 / 95.2, 90.4 /
        // 99.8.)
        const bool small = sizeof(DT) == 4 && VAR && n * R < (uint64_t)1 << 21;
        bool fused = K < 0 && ! small;
        if (fused && hipMalloc(&block, 4 * vb + rest) != hipSuccess)
        {
            (void)hipGetLastError();
            block = nullptr;
            fused = false;
        }
        if (! block && hipMalloc(&block, 3 * vb + rest) != hipSuccess)
            throw Error(HSOLVE_ERR_ALLOC, "cg_ell_multi: workspace allocation failed");
        struct Free
        {
            void * p;
            ~Free() { (void)hipFree(p); }
        } guard_block{block};
        char * c = (char *)block;
        DT * Rv = (DT *)c; c += vb;
        DT * Pv = (DT *)c; c += vb;
        DT * Vv = (DT *)c; c += vb;
        DT * pv[2] = {Pv, Pv};
        if (fused)
        {
            pv[1] = (DT *)c;
            c += vb;
        }
        double * partials = (double *)c; c += pb;
        MState<DT> * s = (MState<DT> *)c;

        MState<DT> h;
        std::memset(&h, 0, sizeof(h));
        h.eps_relative = (DT)eps;
        h.max_iters = max_iters;
        HIP_CHECK(hipMemcpyAsync(s, &h, sizeof(h), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL((mcg_init_kernel<DT, IT, LT, K, VAR>), dim3(grid), dim3(kBlock), 0, st, A, Bv,
                           (const DT *)X, Rv, Pv, Pc, R, partials);
        hipLaunchKernelGGL((mcg_init_finish<DT, VAR>), dim3(R), dim3(kFinThreads), 0, st, (const double *)partials, grid,
                           R, s);
        HIP_CHECK(hipGetLastError());
        uint64_t enqueued = 0, chunk = 8;
        int cp = 0;             // pv[cp] holds the current direction
        while (true)
        {
            for (uint64_t i = 0; i < chunk && enqueued < max_iters; ++i, ++enqueued)
            {
                bool step = false;
                if constexpr (K < 0)
                {
                    if (fused && enqueued > 0)
                    {
                        hipLaunchKernelGGL((mcg_step_kernel<DT, IT, LT, VAR>), dim3(grid), dim3(kBlock), 0, st, A,
                                           (const DT *)pv[cp], (const DT *)Rv, Pc, pv[cp ^ 1], Vv, X, R, partials,
                                           (const MState<DT> *)s);
                        cp ^= 1;
                        step = true;
                    }
                }
                if (! step)
                    hipLaunchKernelGGL((mcg_spmv_kernel<DT, IT, LT, K>), dim3(grid), dim3(kBlock), 0, st, A,
                                       (const DT *)pv[cp], Vv, R, partials, (const MState<DT> *)s);
                hipLaunchKernelGGL((mcg_spmv_finish<DT, VAR>), dim3(R), dim3(kFinThreads), 0, st,
                                   (const double *)partials, grid, R, s);
                if (fused)
                    hipLaunchKernelGGL((mcg_residual_kernel<DT, VAR>), dim3(grid), dim3(kBlock), 0, st, Rv,
                                       (const DT *)Vv, Pc, (int64_t)n, R, partials, (const MState<DT> *)s);
                else
                    hipLaunchKernelGGL((mcg_update_kernel<DT, VAR>), dim3(grid), dim3(kBlock), 0, st, X, Rv,
                                       (const DT *)Pv, (const DT *)Vv, Pc, (int64_t)n, R, partials,
                                       (const MState<DT> *)s);
                hipLaunchKernelGGL((mcg_update_finish<DT, VAR>), dim3(R), dim3(kFinThreads), 0, st,
                                   (const double *)partials, grid, R, s, cp);
                if (! fused)
                    hipLaunchKernelGGL((mcg_direction_kernel<DT, VAR>), dim3(grid), dim3(kBlock), 0, st, Pv,
                                       (const DT *)Rv, Pc, (int64_t)n, R, (const MState<DT> *)s);
            }
            HIP_CHECK(hipGetLastError());
            HIP_CHECK(hipMemcpyAsync(&h, s, sizeof(h), hipMemcpyDeviceToHost, st));
            HIP_CHECK(hipStreamSynchronize(st));
            if (h.active == 0 || enqueued >= max_iters)
                break;
            if (chunk < 64)
                chunk *= 2;
        }
        if (fused)
        {
            hipLaunchKernelGGL((mcg_flush_kernel<DT>), dim3(grid), dim3(kBlock), 0, st, X, (const DT *)pv[0],
                               (const DT *)pv[1], (int64_t)n, R, (const MState<DT> *)s);
            HIP_CHECK(hipGetLastError());
            HIP_CHECK(hipStreamSynchronize(st));
        }
        for (unsigned j = 0; j < R; ++j)
        {
            if (used)
                used[j] = h.iters[j];
            if (defect)
                defect[j] = (h.initial_defect[j] > 0) ? (double)h.current_defect[j] / (double)h.initial_defect[j]
                                                     : (double)h.current_defect[j];
            if (converged)
                converged[j] = h.converged[j];
        }
    }

    // b[i * rs + j * cs] = U[-1, 1] from (seed + j, stream) counter i, 0 on
    // the Dirichlet nodes of the side-M grid
    __global__ __launch_bounds__(256) void rhs_multi_kernel(double * b, int64_t n, int M, uint64_t rs, uint64_t cs,
                                                            uint64_t seed, uint64_t stream_id, k::Mask mk)
    {
        const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
        if (i >= n)
            return;
        const uint64_t j = blockIdx.y;
        const int r = (int)(i / M), c = (int)(i - (int64_t)r * M);
        double v = 0.0;
        if (! k::dirichlet_rs(r, c, M, mk))
        {
            const uint64_t key = mix64(seed + j + kGolden * (stream_id + 1));
            const uint64_t bits = mix64(key + kGolden * ((uint64_t)i + 1));
            const double u = (double)(bits >> 11) * 0x1.0p-53;
            v = -1.0 + 2.0 * u;
        }
        b[(uint64_t)i * rs + j * cs] = v;
    }
}  // namespace
}  // namespace hsolve

using namespace hsolve;

extern "C" {

int hsolve_ell_spmm(hsolve_ell m, uint64_t nrhs, const void * X, void * Y, const void * RHS, void * stream)
{
    HSOLVE_API_BEGIN
    require(m && X && Y, HSOLVE_ERR_INVALID, "ell_spmm: null pointer");
    require(nrhs >= 1 && nrhs <= (uint64_t)kMaxCols, HSOLVE_ERR_INVALID, "ell_spmm: nrhs in [1, 64]");
    hipStream_t st = as_stream(stream);
    const unsigned R = (unsigned)nrhs;
    with_mv(m, [&](auto A, auto k_tag) {
        using MV = decltype(A);
        using DT = std::remove_const_t<std::remove_pointer_t<decltype(MV::Ax)>>;
        constexpr int K = decltype(k_tag)::value;
        using IT = std::remove_const_t<std::remove_pointer_t<decltype(MV::Aj)>>;
        using LT = std::remove_const_t<std::remove_pointer_t<decltype(MV::Arl)>>;
        const unsigned grid = mv_grid(m->rows);
        if (RHS)
            hipLaunchKernelGGL((spmm_kernel<DT, IT, LT, K, 1>), dim3(grid), dim3(kBlock), 0, st, A,
                               (const DT *)X, (DT *)Y, (const DT *)RHS, R);
        else
            hipLaunchKernelGGL((spmm_kernel<DT, IT, LT, K, 0>), dim3(grid), dim3(kBlock), 0, st, A,
                               (const DT *)X, (DT *)Y, (const DT *)nullptr, R);
        HIP_CHECK(hipGetLastError());
    });
    HSOLVE_API_END
}

int hsolve_cg_ell_multi(hsolve_ell m, uint64_t nrhs, const void * P, const void * B, void * X, uint64_t max_iters,
                        double eps, uint64_t * used_iters, double * defect_out, void * stream)
{
    HSOLVE_API_BEGIN
    require(m && B && X, HSOLVE_ERR_INVALID, "cg_ell_multi: null pointer");
    require(m->rows == m->cols, HSOLVE_ERR_SIZE, "cg_ell_multi: matrix is not square");
    require(nrhs >= 1 && nrhs <= (uint64_t)kMaxCols, HSOLVE_ERR_INVALID, "cg_ell_multi: nrhs in [1, 64]");
    hipStream_t st = as_stream(stream);
    const unsigned R = (unsigned)nrhs;
    std::vector<int> conv(R, 0);
    with_mv(m, [&](auto A, auto k_tag) {
        using MV = decltype(A);
        using DT = std::remove_const_t<std::remove_pointer_t<decltype(MV::Ax)>>;
        constexpr int K = decltype(k_tag)::value;
        using IT = std::remove_const_t<std::remove_pointer_t<decltype(MV::Aj)>>;
        using LT = std::remove_const_t<std::remove_pointer_t<decltype(MV::Arl)>>;
        if (P)
            run_mcg<DT, IT, LT, K, true>(A, R, (const DT *)B, (DT *)X, (const DT *)P, max_iters, eps, used_iters,
                                            defect_out, conv.data(), st);
        else
            run_mcg<DT, IT, LT, K, false>(A, R, (const DT *)B, (DT *)X, nullptr, max_iters, eps, used_iters,
                                             defect_out, conv.data(), st);
    });
    if (max_iters > 0)
        for (unsigned j = 0; j < R; ++j)
            if (! conv[j])
            {
                set_last_error("cg_ell_multi: max_iters reached on column " + std::to_string(j));
                return HSOLVE_ERR_NOT_CONVERGED;
            }
    HSOLVE_API_END
}

int hsolve_rhs_uniform_multi(void * b, uint64_t side, uint64_t count, uint64_t row_stride, uint64_t col_stride,
                             const uint64_t * macro_border_mask, uint64_t seed, uint64_t stream_id, void * stream)
{
    HSOLVE_API_BEGIN
    require(b != nullptr, HSOLVE_ERR_INVALID, "rhs_uniform_multi: null vector");
    require(side >= 2 && side <= 65536, HSOLVE_ERR_SIZE, "rhs_uniform_multi: side in [2, 65536]");
    require(count >= 1 && count <= 65535, HSOLVE_ERR_INVALID, "rhs_uniform_multi: count in [1, 65535]");
    k::Mask mk;
    for (int i = 0; i < 8; ++i)
        mk.dir[i] = macro_border_mask ? (macro_border_mask[i] == 2) : 1;
    const uint64_t n = side * side;
    hipLaunchKernelGGL(rhs_multi_kernel, dim3(grid_for(n, kBlock), (unsigned)count), dim3(kBlock), 0,
                       as_stream(stream), (double *)b, (int64_t)n, (int)side, row_stride, col_stride, seed,
                       stream_id, mk);
    HIP_CHECK(hipGetLastError());
    HSOLVE_API_END
}

}  // extern "C"
