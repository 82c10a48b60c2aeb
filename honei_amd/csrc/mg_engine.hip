// mg_engine.hip -- kernels and tick sequence of the FP32-MG / FP64-IR engine
// (declarations and the slot/tick model: mg_engine.hh).
//
// Reference: Multigrid<Tag, OuterTag, NONE, JAC, CYCLE::V, MIXED>::value
// (honei/math/multigrid.hh:2245-2393) around the FP32 V-cycle
// (multigrid.hh:1616-1905):
//   outer: x0 with b's Dirichlet values injected (:2277-2298); result = 0;
//          d = b - A x0 (FP64); loop { rhs32 = (float)(d / |d|) (unscaled
//          the first time); inner FP32 MG solve; result += |d| * x32;
//          d = b - A result; stop when |d| < eps |d0| }
//   inner: |d| of the initial FP32 defect, V-cycles until
//          |d_k| <= tol |d_0| or n_max_iter cycles
//   cycle: per level down: Jacobi sweeps from zero (x = dinv*d, then
//          n_pre_smooth-1 sweeps), defect, restriction; coarse
//          ConjugateGradients<NONE> (konv_rad form); per level up:
//          prolongation + correction, n_pre_smooth post-sweeps, defect on
//          the finest level.
#include "mg_engine.hh"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <type_traits>
#include <unordered_map>
#include <vector>

namespace hsolve
{
namespace mg
{
namespace
{
    __device__ __forceinline__ bool live(const Slot & sl) { return sl.s != nullptr; }

    // Virtual block coordinates of a slot launch (grid x [, y] per slot,
    // blockIdx.z = slot).  The hardware hands out workgroups in linear order
    // (x fastest), dealing consecutive ones to the 8 XCDs in turn.  Logical
    // blocks are ordered row block major, slot fastest, and every XCD gets
    // one contiguous range of them (k::xcd_block): all slots of a row block
    // run on one XCD, one after another, so the level matrix that they
    // share is fetched into that XCD's L2 once per row block, and the rows
    // +-side away that a stencil row gathers stay in the same L2.
    struct VB
    {
        unsigned x, y, z;
    };
    __device__ __forceinline__ VB vblock()
    {
        if (gridDim.z == 1)     // one slot: the hardware order
            return VB{blockIdx.x, blockIdx.y, 0u};
        const unsigned lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
        const unsigned L = k::xcd_block(lin, gridDim.x * gridDim.y * gridDim.z);
        const unsigned z = L % gridDim.z, r = L / gridDim.z;
        return VB{r % gridDim.x, r / gridDim.x, z};
    }

    // Row i of y = A x' for an engine ELL matrix, x'_c = gx(c), in the
    // reference's order (slots ascending, summed from zero:
    // honei/la/product.hh:148-206).  With 9 stored slots per row (the Q1
    // stencils) every slot load and gather is issued before the first add;
    // padding slots hold valid columns (checked at upload) and are loaded but
    // not summed.
    template <typename DT, typename GX>
    __device__ __forceinline__ DT ell_row_g(const EllMat<DT> & E, int64_t i, GX && gx)
    {
        const uint32_t l = E.len[i];
        DT s = DT(0);
        if (E.ncpr == 9)
        {
            uint32_t c[9];
            DT v[9], xv[9];
#pragma unroll
            for (int k = 0; k < 9; ++k)
            {
                const uint64_t j = (uint64_t)i + (uint64_t)k * E.stride;
                c[k] = E.col[j];
                v[k] = E.val[j];
            }
#pragma unroll
            for (int k = 0; k < 9; ++k)
                xv[k] = gx(c[k]);
#pragma unroll
            for (int k = 0; k < 9; ++k)
                if ((uint32_t)k < l)
                    s += v[k] * xv[k];
            return s;
        }
        uint64_t j = (uint64_t)i;
        for (uint32_t k = 0; k < l; ++k, j += E.stride)
            s += E.val[j] * gx(E.col[j]);
        return s;
    }

    template <typename DT>
    __device__ __forceinline__ DT ell_row(const EllMat<DT> & E, const DT * __restrict__ x, int64_t i)
    {
        return ell_row_g<DT>(E, i, [&](uint32_t c) { return x[c]; });
    }

    struct LevelSizes
    {
        int64_t n[kMaxLevels];
    };

    // One level's matrix and smoother data for the kernels: Q1 bands (B, m =
    // grid side) or an ELL matrix (E), chosen by the kernels' MK argument.
    struct LevelArgs
    {
        k::Bands B;          // B.b[k] = B.b[0] + k * bs
        EllMat32 E;
        const float * dinv;
        int64_t n, m;
        int64_t bs;          // band stride in elements
        const uint8_t * rcode = nullptr;    // row codes (HierLevel::rcode), or null
        const float * rtab = nullptr;       // their rows (12 floats each)
        int rows = 0;                       // how many
        const uint64_t * codes = nullptr;   // value codes of bands and dinv, or null
        const float * ctab = nullptr;       // their tables (16 per array)
    };

    // Matrix kinds of the level kernels: MK 0 Q1 bands (Product<Q1>'s sum
    // order), MK 1 ELL matrices, MK 2 bands holding 9-point structured ELL
    // matrices (ascending-column order, the same bits as MK 1).
    template <int MK> constexpr bool kBands = MK != 1;
    template <int MK> constexpr int kOrd = MK == 2 ? 1 : 0;

    template <int MK>
    __device__ __forceinline__ float level_row(const LevelArgs & a, const float * __restrict__ x, int64_t i)
    {
        if (kBands<MK>)
            return k::q1_row<float, kOrd<MK>>(a.B, x, i, a.n, a.m);
        return ell_row<float>(a.E, x, i);
    }

    // the level operator for the one-workgroup coarse CG
    template <int MK> struct LevelRowOp
    {
        LevelArgs a;
        __device__ __forceinline__ float row(const float * __restrict__ x, int64_t i) const
        {
            return level_row<MK>(a, x, i);
        }
    };

    // ------------------------------------------------------------ tick gates
    // What a tick does for a slot before its V-cycle follows from the phase
    // and need_outer, which hold still until outer_defect_finish_kernel: a
    // start, the FP64 outer step that closes an inner solve, or nothing.
    __device__ __forceinline__ bool starts(const Scalars * s) { return s->phase == PH_START; }
    __device__ __forceinline__ bool closes(const Scalars * s) { return s->phase == PH_SOLVE && s->need_outer != 0; }

    // Start of a solve: result = initial guess (0 or the caller's) with b
    // injected on the first row, the last row and the first column
    // (multigrid.hh:2282-2297), x32 of the finest level = (float)result.
    // Outer step: result += scale * (double)x32.
    __global__ __launch_bounds__(256) void tick_begin_kernel(const Slot * T, int L, int64_t n, int64_t sq, int fx)
    {
        const VB vb = vblock();
        const Slot & sl = T[vb.z];
        if (! live(sl))
            return;
        const Scalars * s = sl.s;
        const int64_t i0 = (int64_t)vb.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
        if (starts(s))
        {
            const bool zero = s->zero_guess != 0;
            for (int64_t i = i0; i < n; i += stride)
            {
                double g = zero ? 0.0 : sl.result[i];
                if (i < sq || i >= n - sq || (i % sq) == 0)
                    g = sl.b[i];
                sl.result[i] = g;
                sl.v[L][fx][i] = (float)g;
            }
        }
        else if (closes(s))
        {
            // four rows a lane where there is more than one (result is the
            // caller's, 8-byte aligned; x32 is the slot's): a workgroup's accesses cover 8 KB of every array
            // (measured on MI355X, 64 slots of 513^2: 92 -> 70 us, one row a
            // lane before; one slot of 4097^2: 48 us both ways)
            typedef double D4 __attribute__((ext_vector_type(4), aligned(8)));
            typedef float F4 __attribute__((ext_vector_type(4)));
            const double scale = s->scale;
            const gptr<double> x = as_global(sl.result);
            const gptr<const float> c = as_global<const float>(sl.v[L][fx]);
            if (n <= stride)
            {
                if (i0 < n)
                    x[i0] = x[i0] + scale * (double)c[i0];
                return;
            }
            for (int64_t i = 4 * i0; i < n; i += 4 * stride)
            {
                if (i + 4 <= n)
                {
                    D4 v = *(gptr<const D4>)(x + i);
                    const F4 w = *(gptr<const F4>)(c + i);
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        v[q] = v[q] + scale * (double)w[q];
                    *(gptr<D4>)(x + i) = v;
                }
                else
                    for (int64_t j = i; j < n; ++j)
                        x[j] = x[j] + scale * (double)c[j];
            }
        }
    }

    // iterates of the coarser levels start at zero
    __global__ __launch_bounds__(256) void start_zero_kernel(const Slot * T, int minl, int L, LevelSizes sz)
    {
        const VB vb = vblock();
        const Slot & sl = T[vb.z];
        if (! live(sl) || ! starts(sl.s))
            return;
        for (int l = minl; l < L; ++l)
            for (int64_t i = (int64_t)vb.x * blockDim.x + threadIdx.x; i < sz.n[l]; i += (int64_t)gridDim.x * blockDim.x)
                sl.v[l][F_X][i] = 0.0f;
    }

    // ------------------------------------------------------- FP64 outer step
    // od = b - A64 result and its norm; opens the next inner solve or ends
    // the outer loop.  On a start: the initial defect.  MK 0: Q1 bands B
    // (two rows per lane, 16-byte loads inside); MK 1: the ELL matrix E.
    //
    // CB: the interior rows read the bands as codes and look the values up in a
    // table copied to LDS; the same values, the same sums.  CB 1: row codes
    // (one byte per row; ctab: the nine values of each of `rows` rows), 2:
    // value codes (one 64-bit word per row, band k in bits 4k .. 4k + 3; ctab:
    // 16 values per band).  Bound by HBM: measured on MI355X, one slot of
    // 4097^2, value codes 91 us (32 bytes a node, 5.9 TB/s), row codes
    // 84 us (25 bytes, 5.0 TB/s).
    //
    // KS: slots per workgroup.  The bands are 72 bytes a node where a slot's
    // vectors are 24, so with several slots one load of them serves KS (bands
    // without codes).  Bound by the L2: measured on MI355X, 64 slots of 513^2,
    // one slot a workgroup 172 us (9.4 TB/s of L2 and HBM together), four 133.
    template <int MK, int CB = 0, int KS = 1>
    __global__ __launch_bounds__(256) void outer_defect_kernel(k::Bands B, EllMat64 E, const Slot * T, int64_t n,
            int64_t m, const void * __restrict__ codes, const double * __restrict__ ctab, int rows, int S)
    {
        static_assert(KS == 1 || (kBands<MK> && CB == 0), "several slots: plain bands");
        __shared__ double tab[CB == 1 ? 9 * kRowCodes : (CB == 2 ? 144 : 1)];
        // (the table's first entries are on their way while the gate is read)
        const int entries = CB == 1 ? 9 * rows : 144;
        double entry = 0.0;
        if (CB != 0)
            entry = ctab[min((int)threadIdx.x, entries - 1)];
        const VB vb = vblock();
        bool on[KS], any = false;
        const double * b[KS];
        const double * x[KS];
        double * od[KS];
        double acc[KS];
#pragma unroll
        for (int q = 0; q < KS; ++q)
        {
            const int z = (int)vb.z * KS + q;
            const Slot & sl = T[z < S ? z : 0];
            on[q] = z < S && live(sl) && (starts(sl.s) || closes(sl.s));
            any = any || on[q];
            b[q] = (const double *)as_global<const double>(sl.b);
            x[q] = (const double *)as_global<const double>(sl.result);
            od[q] = (double *)as_global(sl.od);
            acc[q] = 0.0;
        }
        if (! any)
            return;
        if constexpr (CB != 0)
        {
            for (int i = threadIdx.x; i < entries; i += 256)
                tab[i] = i < 256 ? entry : ctab[i];
            __syncthreads();
        }
        if (MK == 1)
        {
            // one row per lane and pass, lanes on consecutive rows
            const int64_t stride1 = (int64_t)gridDim.x * blockDim.x;
            for (int64_t i = (int64_t)vb.x * blockDim.x + threadIdx.x; i < n; i += stride1)
            {
                const double di = b[0][i] - ell_row<double>(E, x[0], i);
                od[0][i] = di;
                acc[0] += di * di;
            }
        }
        const int64_t stride = (int64_t)gridDim.x * blockDim.x * 2;
        for (int64_t i0 = ((int64_t)vb.x * blockDim.x + threadIdx.x) * 2; kBands<MK> && i0 < n; i0 += stride)
        {
            if (i0 - m - 1 >= 0 && i0 + 2 + m < n)
            {
                // b and x are the caller's arrays (8-byte aligned), od is the slot's
                typedef k::Vec16<double>::type V2;
                typedef double U2 __attribute__((ext_vector_type(2), aligned(8)));
                V2 bv[9];
                if constexpr (CB == 0)
                    k::q1_bands_v<double>(B, i0, bv);
#pragma unroll
                for (int q = 0; q < KS; ++q)
                {
                    if (! on[q])
                        continue;
                    const U2 bb = __builtin_nontemporal_load((const U2 *)(b[q] + i0));
                    double prod[2];
                    if constexpr (CB != 0)
                    {
                        // q1_sums_v's sums (Product<Q1>'s order: dd first) with
                        // the band values from the codes of rows i0, i0 + 1
                        typedef uint64_t C2 __attribute__((ext_vector_type(2)));
                        C2 cw = {0, 0};
                        uint32_t rw = 0;
                        if constexpr (CB == 1)
                            rw = __builtin_nontemporal_load((const uint16_t *)((const uint8_t *)codes + i0));
                        else
                            cw = __builtin_nontemporal_load((const C2 *)((const uint64_t *)codes + i0));
                        double xm[4], xc[4], xp[4];
                        k::ld_window<4>(x[q] + i0 - m - 1, xm);
                        k::ld_window<4>(x[q] + i0 - 1, xc);
                        k::ld_window<4>(x[q] + i0 + m - 1, xp);
#pragma unroll
                        for (int v = 0; v < 2; ++v)
                        {
                            const uint64_t w = cw[v];
                            const double * row = tab + 9 * ((rw >> (8 * v)) & 255u);
                            auto bk = [&](int k) {
                                return CB == 1 ? row[k] : tab[16 * k + (int)((w >> (4 * k)) & 15u)];
                            };
                            double sum = bk(4) * xc[v + 1];
                            sum += bk(0) * xm[v];
                            sum += bk(1) * xm[v + 1];
                            sum += bk(2) * xm[v + 2];
                            sum += bk(3) * xc[v];
                            sum += bk(5) * xc[v + 2];
                            sum += bk(6) * xp[v];
                            sum += bk(7) * xp[v + 1];
                            sum += bk(8) * xp[v + 2];
                            prod[v] = sum;
                        }
                    }
                    else
                        k::q1_sums_v<double, kOrd<MK>>(bv, x[q], i0, m, prod);
                    V2 o;
                    o[0] = bb[0] - prod[0];
                    o[1] = bb[1] - prod[1];
                    *(V2 *)(od[q] + i0) = o;
                    acc[q] += o[0] * o[0];
                    acc[q] += o[1] * o[1];
                }
            }
            else
            {
                for (int64_t i = i0; i < i0 + 2 && i < n; ++i)
#pragma unroll
                    for (int q = 0; q < KS; ++q)
                    {
                        if (! on[q])
                            continue;
                        const double prod = k::q1_row<double, kOrd<MK>>(B, x[q], i, n, m);
                        const double di = b[q][i] - prod;
                        od[q][i] = di;
                        acc[q] += di * di;
                    }
            }
        }
#pragma unroll
        for (int q = 0; q < KS; ++q)
            if (on[q])
                k::put_partials2(acc[q], 0.0, T[vb.z * KS + q].partials, vb.x);
    }

    // |od| from the partials of outer_defect_kernel (nb blocks per slot), then
    // the outer step's decisions; one block per slot (blockIdx.z).  Opening an
    // inner solve starts its V-cycles (run) and, with `fold` (no separate
    // opening kernels), its cycle count.
    __global__ __launch_bounds__(256) void outer_defect_finish_kernel(const Slot * T, unsigned nb, double outer_eps,
                                                                      uint64_t max_outer, int fold)
    {
        const Slot & sl = T[blockIdx.z];
        if (! live(sl))
            return;
        Scalars * s = sl.s;
        const bool start = starts(s);
        if (! start && ! closes(s))
        {
            if (threadIdx.x == 0)
            {
                s->open = 0;
                s->clear = 0;
                if (s->phase == PH_SOLVE)
                    s->ticks += 1;
            }
            return;
        }
        double dd, unused;
        k::sum_partials2(sl.partials, nb, dd, unused);
        if (threadIdx.x != 0)
            return;
        {
            const double nrm = sqrt(dd);
            s->ticks += 1;
            s->open = 0;
            s->clear = start ? 1 : 0;
            if (start)
            {
                s->initial_defect = nrm;
                s->def_norm = nrm;
                s->scale = 1.0;
                s->inv = 1.0;
                s->outer_iters = 0;
                s->inner_total = 0;
                s->phase = PH_SOLVE;
                s->open = 1;
            }
            else
            {
                s->def_norm = nrm;
                s->outer_iters += 1;
                s->inner_total += s->inner_last;
                s->need_outer = 0;
                if (nrm < outer_eps * s->initial_defect)
                {
                    s->outer_active = 0;
                    s->phase = PH_DONE;
                }
                else
                {
                    s->scale = nrm;
                    s->inv = 1.0 / nrm;
                    if (max_outer != 0 && s->outer_iters >= max_outer)
                    {
                        s->outer_active = 0;
                        s->status = 1;
                        s->phase = PH_DONE;
                    }
                    else
                        s->open = 1;
                }
            }
            if (s->open)
            {
                s->run = 1;
                if (fold)
                    s->inner_last = 0;
            }
        }
    }

    // rhs32 = (float)(od * inv) (inv == 1 on the first step, so the cast of
    // the unscaled defect); a start also clears the result array.  NORM: block
    // partials of |rhs32|^2, the initial defect of an inner solve from zero
    // (four entries per lane; od and rhs32 are the slot's, 16-byte aligned).
    template <bool NORM>
    __global__ __launch_bounds__(256) void to_inner_kernel(const Slot * T, int L, int64_t n)
    {
        const VB vb = vblock();
        const Slot & sl = T[vb.z];
        if (! live(sl) || sl.s->open == 0)
            return;
        typedef k::Vec16<double>::type D2;
        typedef k::Vec16<float>::type F4;
        const double inv = sl.s->inv;
        const bool clear = sl.s->clear != 0;
        const gptr<const double> od = as_global<const double>(sl.od);
        const gptr<float> rhs = as_global(sl.v[L][F_RHS]);
        const gptr<double> res = as_global(sl.result);
        double acc = 0.0;
        for (int64_t i0 = ((int64_t)vb.x * blockDim.x + threadIdx.x) * 4; i0 < n;
             i0 += (int64_t)gridDim.x * blockDim.x * 4)
        {
            const int cnt = (int)min((int64_t)4, n - i0);
            if (cnt == 4)
            {
                const D2 a = *(gptr<const D2>)(od + i0), b = *(gptr<const D2>)(od + i0 + 2);
                F4 v;
                v[0] = (float)(a[0] * inv);
                v[1] = (float)(a[1] * inv);
                v[2] = (float)(b[0] * inv);
                v[3] = (float)(b[1] * inv);
                *(gptr<F4>)(rhs + i0) = v;
                if (NORM)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        acc += (double)v[q] * (double)v[q];
            }
            else
                for (int q = 0; q < cnt; ++q)
                {
                    const float v = (float)(od[i0 + q] * inv);
                    rhs[i0 + q] = v;
                    acc += (double)v * (double)v;
                }
            if (clear)
                for (int q = 0; q < cnt; ++q)
                    res[i0 + q] = 0.0;
        }
        if (NORM)
        {
            __shared__ double lds[16];
            const double t = k::block_sum(acc, lds);
            if (threadIdx.x == 0)
                sl.partials[kOpenPartials + vb.x] = t;
        }
    }

    // Opens the inner solve: its initial defect d is rhs itself when
    // initial_zero (multigrid.hh:1626-1628), else rhs - A x.
    template <int INITIAL_ZERO, int MK>
    __global__ __launch_bounds__(256) void open_inner_kernel(LevelArgs a, const Slot * T, int L, int fx)
    {
        const VB vb = vblock();
        const Slot & sl = T[vb.z];
        if (! live(sl) || sl.s->open == 0)
            return;
        const int64_t n = a.n;
        const int64_t lane0 = (int64_t)vb.x * blockDim.x + threadIdx.x;
        const int64_t lanes = (int64_t)gridDim.x * blockDim.x;
        const float * rhs = sl.v[L][F_RHS];
        float * d = sl.v[L][F_D];
        if (INITIAL_ZERO)
        {
            typedef k::Vec16<float>::type F4;
            for (int64_t i0 = lane0 * 4; i0 < n; i0 += lanes * 4)
            {
                if (i0 + 4 <= n)
                    *(F4 *)(d + i0) = *(const F4 *)(rhs + i0);
                else
                    for (int64_t i = i0; i < n; ++i)
                        d[i] = rhs[i];
            }
        }
        else if (kBands<MK>)
        {
            for (int64_t lane = lane0; lane * 4 < n; lane += lanes)
                k::q1_body_v<float, 1, kOrd<MK>>(a.B, sl.v[L][fx], d, rhs, nullptr, n, a.m, lane);
        }
        else
        {
            const float * x = sl.v[L][fx];
            for (int64_t i = lane0; i < n; i += lanes)
                d[i] = rhs[i] - ell_row<float>(a.E, x, i);
        }
    }

    // |d| of the finest FP32 defect.  MODE 0: start of an inner solve (gate
    // `open`); MODE 1: end of a V-cycle (gate `run`): count it, stop on
    // |d| <= tol |d_0| or after n_max_iter cycles.
    template <int MODE>
    __global__ __launch_bounds__(256) void inner_norm_kernel(const Slot * T, int L, int64_t n)
    {
        const VB vb = vblock();
        const Slot & sl = T[vb.z];
        if (! live(sl))
            return;
        Scalars * s = sl.s;
        if (MODE == 0 ? s->open == 0 : s->run == 0)
            return;
        const float * __restrict__ d = sl.v[L][F_D];
        double acc = 0.0;
        typedef k::Vec16<float>::type F4;
        const int64_t stride = (int64_t)gridDim.x * blockDim.x;
        const int64_t tid = (int64_t)vb.x * blockDim.x + threadIdx.x;
        const int64_t n4 = n >> 2;
        const F4 * d4 = reinterpret_cast<const F4 *>(d);
        int64_t i = tid;
        for (; i + 3 * stride < n4; i += 4 * stride)
        {
            F4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                v[u] = __builtin_nontemporal_load(d4 + i + u * stride);
#pragma unroll
            for (int u = 0; u < 4; ++u)
            {
                acc += (double)v[u].x * (double)v[u].x;
                acc += (double)v[u].y * (double)v[u].y;
                acc += (double)v[u].z * (double)v[u].z;
                acc += (double)v[u].w * (double)v[u].w;
            }
        }
        for (; i < n4; i += stride)
        {
            const F4 v = __builtin_nontemporal_load(d4 + i);
            acc += (double)v.x * (double)v.x;
            acc += (double)v.y * (double)v.y;
            acc += (double)v.z * (double)v.z;
            acc += (double)v.w * (double)v.w;
        }
        for (int64_t t = 4 * n4 + tid; t < n; t += stride)
        {
            const double v = (double)d[t];
            acc += v * v;
        }
        k::put_partials2(acc, 0.0, sl.partials, vb.x);
    }

    // the inner stopping test from inner_norm_kernel's partials (nb blocks
    // per slot); one block per slot (blockIdx.z)
    template <int MODE>
    __global__ __launch_bounds__(256) void inner_norm_finish_kernel(const Slot * T, unsigned nb, float tol,
            int convergence_check, uint64_t n_max_iter)
    {
        const Slot & sl = T[blockIdx.z];
        if (! live(sl))
            return;
        Scalars * s = sl.s;
        if (MODE == 0 ? s->open == 0 : s->run == 0)
            return;
        double ss, unused;
        k::sum_partials2(sl.partials, nb, ss, unused);
        if (threadIdx.x != 0)
            return;
        {
            const float nrm = sqrtf((float)ss);
            if (MODE == 0)
            {
                s->inner_initial = nrm;
                s->inner_defect = nrm;
                if (convergence_check && nrm <= tol)
                {
                    // nothing to do; the count keeps the previous solve's value
                    s->run = 0;
                    s->need_outer = 1;
                }
                else
                    s->inner_last = 0;
            }
            else
            {
                s->inner_defect = nrm;
                s->inner_last += 1;
                if (nrm <= s->inner_initial * tol || s->inner_last >= n_max_iter)
                {
                    s->run = 0;
                    s->need_outer = 1;
                }
            }
        }
    }

    // The inner stopping test after a V-cycle whose post-smoothing left the
    // partials of |d|^2 (nd of them); FOLD: the inner solve's initial defect
    // comes from to_inner_kernel's partials (nr) after its first cycle.
    // One block per slot (blockIdx.z).
    //
    // How the partials group the nodes depends on the number of slots, the
    // matrix form and the device.  Their totals differ in the last bits, which
    // decide nothing unless |d| comes within kTie of its limit (rounding to
    // float and n sums in double stay below a tenth of that): then the test is
    // made on sums over the arrays in an order of their own.  So a solve stops
    // at the same cycle alone, in any batch and from codes or plain bands.  (One
    // block over n nodes: measured 2.3 ms at 4097^2, for one test in 30,000.)
    constexpr float kTie = 0x1p-16f;
    template <bool FOLD>
    __global__ __launch_bounds__(1024) void inner_end_kernel(const Slot * T, int L, int64_t n, unsigned nd,
                                                             unsigned nr, float tol, uint64_t n_max_iter)
    {
        const Slot & sl = T[blockIdx.z];
        if (! live(sl))
            return;
        Scalars * s = sl.s;
        if (s->run == 0)
            return;
        __shared__ double lds[32];
        __shared__ int tie;
        const uint64_t count = s->inner_last + 1;
        const bool first = FOLD && count == 1;
        const gptr<const double> pd = as_global<const double>(sl.partials + kCyclePartials);
        const gptr<const double> pr = as_global<const double>(sl.partials + kOpenPartials);
        double d = 0.0, r = 0.0;
        for (unsigned i = threadIdx.x; i < nd; i += blockDim.x)
            d += pd[i];
        if (first)
            for (unsigned i = threadIdx.x; i < nr; i += blockDim.x)
                r += pr[i];
        k::block_sum2(d, r, lds);
        float initial = 0.0f, nrm = 0.0f;
        if (threadIdx.x == 0)
        {
            initial = first ? sqrtf((float)r) : s->inner_initial;
            nrm = sqrtf((float)d);
            const float limit = initial * tol;
            tie = nrm != 0.0f && fabsf(nrm - limit) <= kTie * limit;
            s->inner_initial = initial;
        }
        // (the last cycle ends the solve whatever the test says)
        if (count < n_max_iter)
            __syncthreads();
        if (count < n_max_iter && tie)
        {
            const gptr<const float> fd = as_global<const float>(sl.v[L][F_D]);
            const gptr<const float> fr = as_global<const float>(sl.v[L][F_RHS]);
            d = r = 0.0;
#pragma unroll 8
            for (int64_t i = threadIdx.x; i < n; i += blockDim.x)
            {
                d += (double)fd[i] * (double)fd[i];
                if (FOLD)
                    r += (double)fr[i] * (double)fr[i];
            }
            k::block_sum2(d, r, lds);
            nrm = sqrtf((float)d);
            if (FOLD)
                initial = sqrtf((float)r);
        }
        if (threadIdx.x != 0)
            return;
        s->inner_defect = nrm;
        s->inner_last = count;
        if (nrm <= initial * tol || count >= n_max_iter)
        {
            s->run = 0;
            s->need_outer = 1;
        }
    }

    // one-level hierarchy: the cycle loop is left after the coarse solve
    __global__ void one_level_end_kernel(const Slot * T, unsigned nslots)
    {
        const unsigned z = blockIdx.x * blockDim.x + threadIdx.x;
        if (z >= nslots)
            return;
        Scalars * s = T[z].s;
        if (s == nullptr || s->run == 0)
            return;
        s->inner_last += 1;
        s->run = 0;
        s->need_outer = 1;
    }

    // --------------------------------------------------------------- V-cycle
#define HS_GATE_RUN                                     \
    const Slot & sl = T[vb.z];                          \
    if (! live(sl) || sl.s->run == 0)                   \
        return;

    // x (+)= dinv * d: the single first sweep when n_pre_smooth == 1
    template <int ACC>
    __global__ __launch_bounds__(256) void v_zero1_kernel(LevelArgs a, const Slot * T, int L, int fsrc, int fout)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        const int64_t i = (int64_t)vb.x * blockDim.x + threadIdx.x;
        if (i >= a.n)
            return;
        const float * d = sl.v[L][fsrc];
        float * out = sl.v[L][fout];
        const float c = a.dinv[i] * d[i];
        out[i] = ACC ? out[i] + c : c;
    }

    // The row kernels below cover 4 rows per lane: on Q1 bands 4 consecutive
    // rows as 16-byte vectors (kernels_la.hh / kernels_mg.hh bodies), on ELL
    // one row per pass of a grid-stride loop (lanes on consecutive rows, so
    // every slot load of a wave is one coalesced access).

    // the first two sweeps from zero (c1 = dinv*d, c2 = c1 + dinv*(d - A c1));
    // ACC: out = (field facc) + c2 (facc may be fout), else out = c2
    template <int ACC, int MK>
    __global__ __launch_bounds__(256) void v_zero2_kernel(LevelArgs a, const Slot * T, int L, int fsrc, int fout,
                                                          int facc)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        const int64_t lane = (int64_t)vb.x * blockDim.x + threadIdx.x;
        const float * d = sl.v[L][fsrc];
        float * out = sl.v[L][fout];
        const float * accin = sl.v[L][facc];
        if (kBands<MK>)
        {
            k::jacobi_zero2_body<float, ACC, kOrd<MK>>(a.B, d, a.dinv, out, a.n, a.m, lane, accin);
            return;
        }
        for (int64_t i = lane; i < a.n; i += (int64_t)gridDim.x * blockDim.x)
        {
            const float s = ell_row_g<float>(a.E, i, [&](uint32_t c) { return a.dinv[c] * d[c]; });
            const float di = a.dinv[i];
            const float c1 = di * d[i];
            const float t = d[i] - s;
            const float c2 = c1 + t * di;
            out[i] = ACC ? accin[i] + c2 : c2;
        }
    }

    // workgroups (over all slots) of the per-tick gate kernels' capped grids
    constexpr unsigned kGateBlocks = 4096;
    template <int N> using IntC = std::integral_constant<int, N>;

#include "mg_march.hh"

    // Tiles of a level of side m with th rows each, V columns per lane.
    template <int V> unsigned march_tiles(int64_t m, int th)
    {
        return (unsigned)(((m + kW<V> - 1) / kW<V>) * ((m + th - 1) / th));
    }

    // Tile rows of the one-pass kernels: a tile's steps are sequential (th + 6
    // of them), so the height is the even th <= 128 with the fewest rounds of
    // steps, ceil(tiles / resident) * (th + 6), where `resident` tiles fit on
    // the device at once (the larger th on a tie: fewer halo rows).
    // At most kMaxTiles tiles (a slot's room for their partial sums).
    template <int V> int march_rows(int64_t m, unsigned slots, unsigned resident)
    {
        int best = 2;
        uint64_t best_cost = ~(uint64_t)0;
        for (int th = 2; th <= 128; th += 2)
        {
            const uint64_t tiles = (uint64_t)march_tiles<V>(m, th) * slots;
            if (tiles > (uint64_t)slots * kMaxTiles)
                continue;
            const uint64_t rounds = (tiles + resident - 1) / resident;
            const uint64_t cost = rounds * (uint64_t)(th + 6);
            if (cost <= best_cost)
            {
                best_cost = cost;
                best = th;
            }
            if (th >= m)
                break;
        }
        return best;
    }

    // Workgroups of kernel `fn` (256 lanes) resident on the current device at
    // once: CUs x the occupancy its registers and LDS allow (cached).
    inline unsigned post_resident(const void * fn)
    {
        static std::mutex mu;
        static std::map<std::pair<int, const void *>, unsigned> cache;
        int dev = 0;
        HIP_CHECK(hipGetDevice(&dev));
        std::lock_guard<std::mutex> lock(mu);
        auto it = cache.find(std::make_pair(dev, fn));
        if (it != cache.end())
            return it->second;
        int cus = 0, per_cu = 0;
        HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, 0));
        const unsigned r = (unsigned)std::max(1, cus * std::max(1, per_cu));
        cache.emplace(std::make_pair(dev, fn), r);
        return r;
    }

    // y = x + dinv * (rhs - A x)
    template <int MK>
    __global__ __launch_bounds__(256) void v_sweep_kernel(LevelArgs a, const Slot * T, int L, int fx, int fy, int frhs)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        const int64_t lane = (int64_t)vb.x * blockDim.x + threadIdx.x;
        const float * x = sl.v[L][fx];
        float * y = sl.v[L][fy];
        const float * rhs = sl.v[L][frhs];
        if (kBands<MK>)
        {
            k::q1_body_v<float, 2, kOrd<MK>>(a.B, x, y, rhs, a.dinv, a.n, a.m, lane);
            return;
        }
        for (int64_t i = lane; i < a.n; i += (int64_t)gridDim.x * blockDim.x)
        {
            const float t = rhs[i] - ell_row<float>(a.E, x, i);
            y[i] = x[i] + t * a.dinv[i];
        }
    }

    // d = rhs - A x
    template <int MK>
    __global__ __launch_bounds__(256) void v_defect_kernel(LevelArgs a, const Slot * T, int L)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        const int64_t lane = (int64_t)vb.x * blockDim.x + threadIdx.x;
        const float * x = sl.v[L][F_X];
        float * d = sl.v[L][F_D];
        const float * rhs = sl.v[L][F_RHS];
        if (kBands<MK>)
        {
            k::q1_body_v<float, 1, kOrd<MK>>(a.B, x, d, rhs, nullptr, a.n, a.m, lane);
            return;
        }
        for (int64_t i = lane; i < a.n; i += (int64_t)gridDim.x * blockDim.x)
            d[i] = rhs[i] - ell_row<float>(a.E, x, i);
    }

    // Product<PROLMAT>: level Ldst's fdst = E * (level Lsrc's fsrc)
    __global__ __launch_bounds__(256) void v_apply_ell_kernel(EllMat32 E, const Slot * T, int Lsrc, int fsrc, int Ldst,
                                                              int fdst)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        const float * x = sl.v[Lsrc][fsrc];
        float * y = sl.v[Ldst][fdst];
        const int64_t lane = (int64_t)vb.x * blockDim.x + threadIdx.x;
        for (int64_t i = lane; i < (int64_t)E.rows; i += (int64_t)gridDim.x * blockDim.x)
            y[i] = ell_row<float>(E, x, i);
    }

    // x += alpha * c (ScaledSum with the constant correction factor)
    __global__ __launch_bounds__(256) void v_axpy_const_kernel(const Slot * T, int L, int64_t n, float alpha)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        const int64_t i = (int64_t)vb.x * blockDim.x + threadIdx.x;
        if (i >= n)
            return;
        float * x = sl.v[L][F_X];
        x[i] = x[i] + alpha * sl.v[L][F_C][i];
    }

    // dst = src (ADD 0) or dst += src (ADD 1), four entries per lane
    template <int ADD>
    __global__ __launch_bounds__(256) void v_move_kernel(const Slot * T, int L, int64_t n, int fsrc, int fdst)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        typedef k::Vec16<float>::type F4;
        const float * src = sl.v[L][fsrc];
        float * dst = sl.v[L][fdst];
        const int64_t i0 = ((int64_t)vb.x * blockDim.x + threadIdx.x) * 4;
        if (i0 + 4 <= n)
        {
            const F4 s = *(const F4 *)(src + i0);
            if (ADD)
            {
                F4 d = *(const F4 *)(dst + i0);
                d.x = d.x + s.x;
                d.y = d.y + s.y;
                d.z = d.z + s.z;
                d.w = d.w + s.w;
                *(F4 *)(dst + i0) = d;
            }
            else
                *(F4 *)(dst + i0) = s;
        }
        else
            for (int64_t i = i0; i < n; ++i)
                dst[i] = ADD ? dst[i] + src[i] : src[i];
    }

    // rhs of level L-1 = restriction of d of level L
    __global__ __launch_bounds__(256) void v_restrict_kernel(const Slot * T, int L, int64_t Nc, k::Mask mk)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        k::restriction_body<float>(sl.v[L - 1][F_RHS], sl.v[L][F_D], Nc, mk, vb.y,
                                   (int64_t)vb.x * blockDim.x + threadIdx.x);
    }

    // ConjugateGradients<NONE> (konv_rad form) on the coarsest level
    template <int MK>
    __global__ __launch_bounds__(256) void v_coarse_kernel(LevelArgs a, const Slot * T, int L, int frhs,
                                                           double konv_rad, uint64_t max_iters)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        LevelRowOp<MK> A{a};
        k::cg_konv_body_op<float>(A, sl.v[L][frhs], sl.v[L][F_X], sl.cg_work, a.n, konv_rad, max_iters,
                                  &sl.s->cg_iters);
    }

    // v_coarse_kernel with the vectors and (Q1 bands) the level's nine bands
    // copied to LDS, for coarsest levels up to 17^2: the CG's sequential
    // sums then wait on LDS, not on a memory round trip per step.  It runs
    // k::cg_konv_body_op itself on the copies, so every operation and its
    // order are unchanged and so are the bits.  One wave per slot.
    constexpr int kCoarseLdsMax = 289;
    template <int MK>
    __global__ __launch_bounds__(64) void v_coarse_lds_kernel(LevelArgs a, const Slot * T, int L, int frhs,
                                                              double konv_rad, uint64_t max_iters)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        __shared__ float vec[6 * kCoarseLdsMax];                  // rhs, x, then the 4n of work
        __shared__ float bnd[kBands<MK> ? 9 * kCoarseLdsMax : 1];
        const int n = (int)a.n;
        float * rhs = vec;
        float * x = vec + kCoarseLdsMax;
        float * work = vec + 2 * kCoarseLdsMax;
        const float * rg = sl.v[L][frhs];
        for (int i = threadIdx.x; i < n; i += blockDim.x)
            rhs[i] = rg[i];
        if constexpr (kBands<MK>)
        {
            for (int k = 0; k < 9; ++k)
            {
                const float * b = (const float *)a.B.b[k];
                for (int i = threadIdx.x; i < n; i += blockDim.x)
                    bnd[k * kCoarseLdsMax + i] = b[i];
                a.B.b[k] = bnd + k * kCoarseLdsMax;
            }
        }
        __syncthreads();
        LevelRowOp<MK> A{a};
        k::cg_konv_body_op<float>(A, rhs, x, work, a.n, konv_rad, max_iters, &sl.s->cg_iters);
        __syncthreads();
        float * xg = sl.v[L][F_X];
        for (int i = threadIdx.x; i < n; i += blockDim.x)
            xg[i] = x[i];
    }

#include "mg_bottom.hh"

    // The same for a coarsest level too large for one wave (minl 3 or 4):
    // every vector and band of the levels in LDS, the coarse CG on the first
    // wave with its vectors there.
    struct BottomLdsArgs
    {
        BottomArgs b;
        int off[kBottomMax + 1];   // float offset of each level's block in the dynamic LDS
        int minl;
    };

    // Row i of A x on a level held in LDS (band k at b + k n): q1_row's
    // order and index guards
    template <int ORD>
    __device__ __forceinline__ float lds_row(const float * b, const float * x, int i, int n, int m)
    {
        if (ORD == 1)
        {
            float s = 0.0f;
            if (i - m - 1 >= 0) s += b[i] * x[i - m - 1];
            if (i - m >= 0)     s += b[n + i] * x[i - m];
            if (i - m + 1 >= 0) s += b[2 * n + i] * x[i - m + 1];
            if (i - 1 >= 0)     s += b[3 * n + i] * x[i - 1];
            s += b[4 * n + i] * x[i];
            if (i + 1 < n)      s += b[5 * n + i] * x[i + 1];
            if (i + m - 1 < n)  s += b[6 * n + i] * x[i + m - 1];
            if (i + m < n)      s += b[7 * n + i] * x[i + m];
            if (i + m + 1 < n)  s += b[8 * n + i] * x[i + m + 1];
            return s;
        }
        float s = b[4 * n + i] * x[i];
        if (i - m - 1 >= 0) s += b[i] * x[i - m - 1];
        if (i - m >= 0)     s += b[n + i] * x[i - m];
        if (i - m + 1 >= 0) s += b[2 * n + i] * x[i - m + 1];
        if (i - 1 >= 0)     s += b[3 * n + i] * x[i - 1];
        if (i + 1 < n)      s += b[5 * n + i] * x[i + 1];
        if (i + m - 1 < n)  s += b[6 * n + i] * x[i + m - 1];
        if (i + m < n)      s += b[7 * n + i] * x[i + m];
        if (i + m + 1 < n)  s += b[8 * n + i] * x[i + m + 1];
        return s;
    }

    // A level held in LDS as the operator of the one-workgroup CG
    template <int ORD> struct LdsRowOp
    {
        const float * b;
        int n, m;
        __device__ __forceinline__ float row(const float * __restrict__ x, int64_t i) const
        {
            return lds_row<ORD>(b, x, (int)i, n, m);
        }
    };

    // Block of level L in LDS: bands (9n), dinv, rhs, x, then tmp (levels
    // above minl) or the CG's 4n of work (minl).
    inline int bottom_floats(int n, bool coarsest) { return (coarsest ? 16 : 13) * n; }

    template <int MK>
    __global__ __launch_bounds__(1024) void v_bottom_lds_kernel(BottomLdsArgs ba, const Slot * T)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        extern __shared__ float lds[];
        const int tid = threadIdx.x, nt = blockDim.x;
        // bands and dinv of every level: each lane issues the loads of two
        // rows of all ten arrays before it stores any, so a level costs one
        // or two memory round trips, not one per array and row
        for (int L = ba.minl; L <= ba.b.top; ++L)
        {
            const int n = (int)ba.b.lv[L].n;
            float * b = lds + ba.off[L];
            const float * src[10];
            for (int k = 0; k < 9; ++k)
                src[k] = (const float *)ba.b.lv[L].B.b[k];
            src[9] = ba.b.lv[L].dinv;
            for (int i0 = tid; i0 < n; i0 += 2 * nt)
            {
                float v[2][10];
#pragma unroll
                for (int h = 0; h < 2; ++h)
                {
                    const int i = min(i0 + h * nt, n - 1);
#pragma unroll
                    for (int k = 0; k < 10; ++k)
                        v[h][k] = src[k][i];
                }
#pragma unroll
                for (int h = 0; h < 2; ++h)
                {
                    const int i = i0 + h * nt;
                    if (i < n)
                    {
#pragma unroll
                        for (int k = 0; k < 10; ++k)
                            b[k * n + i] = v[h][k];
                    }
                }
            }
        }
        {
            const int n = (int)ba.b.lv[ba.b.top].n;
            const float * g = sl.v[ba.b.top][F_RHS];
            float * rhs = lds + ba.off[ba.b.top] + 10 * n;
            for (int i = tid; i < n; i += nt)
                rhs[i] = g[i];
        }
        __syncthreads();
        // down: x = c1 + dinv (rhs - A c1) with c1 = dinv rhs, d' = rhs - A x,
        // rhs of L - 1 = R d'
        for (int L = ba.b.top; L > ba.minl; --L)
        {
            const int n = (int)ba.b.lv[L].n, m = (int)ba.b.lv[L].m;
            const float * b = lds + ba.off[L];
            const float * dinv = b + 9 * n;
            const float * rhs = b + 10 * n;
            float * x = lds + ba.off[L] + 11 * n;
            float * tmp = lds + ba.off[L] + 12 * n;
            for (int i = tid; i < n; i += nt)
                tmp[i] = dinv[i] * rhs[i];
            __syncthreads();
            for (int i = tid; i < n; i += nt)
            {
                const float t = rhs[i] - lds_row<kOrd<MK>>(b, tmp, i, n, m);
                x[i] = tmp[i] + t * dinv[i];
            }
            __syncthreads();
            for (int i = tid; i < n; i += nt)
                tmp[i] = rhs[i] - lds_row<kOrd<MK>>(b, x, i, n, m);
            __syncthreads();
            const int Nc = (int)ba.b.lv[L - 1].m;
            float * crhs = lds + ba.off[L - 1] + 10 * Nc * Nc;
            for (int q = tid; q < Nc * Nc; q += nt)
            {
                const int r = q / Nc, sc = q - r * Nc;
                crhs[q] = k::restrict_node<float>(
                    [&](int dr, int ds) {
                        const int idx = (2 * r + dr) * m + 2 * sc + ds;
                        return tmp[min(max(idx, 0), n - 1)];
                    },
                    r, sc, Nc, ba.b.mk);
            }
            __syncthreads();
        }
        // the coarse solve, as v_coarse_lds_kernel, on the first wave
        {
            const int L = ba.minl;
            const int n = (int)ba.b.lv[L].n;
            float * b = lds + ba.off[L];
            const LdsRowOp<kOrd<MK>> A{b, n, (int)ba.b.lv[L].m};
            if (threadIdx.x < 64)
                k::cg_konv_body_op<float, LdsRowOp<kOrd<MK>>, 64>(A, b + 10 * n, b + 11 * n, b + 12 * n, (int64_t)n,
                                                                 ba.b.konv_rad, ba.b.max_iters, &sl.s->cg_iters);
            __syncthreads();
        }
        // up: x_in = x + alpha P (coarse iterate), then two sweeps into tmp
        for (int L = ba.minl + 1; L <= ba.b.top; ++L)
        {
            const int n = (int)ba.b.lv[L].n, m = (int)ba.b.lv[L].m;
            const int Nc = (int)ba.b.lv[L - 1].m;
            const float * cf = lds + ba.off[L - 1] + (L - 1 == ba.minl ? 11 : 12) * Nc * Nc;
            const float * b = lds + ba.off[L];
            const float * dinv = b + 9 * n;
            const float * rhs = b + 10 * n;
            float * x = lds + ba.off[L] + 11 * n;
            float * tmp = lds + ba.off[L] + 12 * n;
            for (int i = tid; i < n; i += nt)
            {
                const int R = i / m, S = i - R * m;
                tmp[i] = x[i] + ba.b.alpha * k::prolongation_node<float>(cf, m, ba.b.mk, R, S);
            }
            __syncthreads();
            for (int i = tid; i < n; i += nt)
            {
                const float t = rhs[i] - lds_row<kOrd<MK>>(b, tmp, i, n, m);
                x[i] = tmp[i] + t * dinv[i];
            }
            __syncthreads();
            for (int i = tid; i < n; i += nt)
            {
                const float t = rhs[i] - lds_row<kOrd<MK>>(b, x, i, n, m);
                tmp[i] = x[i] + t * dinv[i];
            }
            __syncthreads();
        }
        {
            const int n = (int)ba.b.lv[ba.b.top].n;
            const float * tmp = lds + ba.off[ba.b.top] + 12 * n;
            float * g = sl.v[ba.b.top][F_TMP];
            for (int i = tid; i < n; i += nt)
                g[i] = tmp[i];
        }
    }

    // level L's fout (+)= alpha * P (x of level L-1)
    template <bool AXPY>
    __global__ __launch_bounds__(256) void v_prolong_kernel(const Slot * T, int L, int Nf, float alpha, k::Mask mk,
                                                            int fout, int fcoarse)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        k::prolongation2_body<float, AXPY>(sl.v[L][fout], sl.v[L - 1][fcoarse], Nf, alpha, mk, vb.y,
                                           vb.x * blockDim.x + threadIdx.x);
    }

    // adapt_correction_factor == 0: alpha = (d.c) / ((A c).c)
    template <int MK>
    __global__ __launch_bounds__(256) void v_adapt_alpha_kernel(LevelArgs a, const Slot * T, int L)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        const float * d = sl.v[L][F_D];
        const float * c = sl.v[L][F_C];
        double a1 = 0.0, a2 = 0.0;
        const int64_t stride = (int64_t)gridDim.x * blockDim.x;
        for (int64_t i = (int64_t)vb.x * blockDim.x + threadIdx.x; i < a.n; i += stride)
        {
            const float t = level_row<MK>(a, c, i);
            a1 += (double)d[i] * (double)c[i];
            a2 += (double)t * (double)c[i];
        }
        k::put_partials2(a1, a2, sl.partials, vb.x);
    }

    // alpha from v_adapt_alpha_kernel's partials; one block per slot
    __global__ __launch_bounds__(256) void v_adapt_alpha_finish_kernel(const Slot * T, unsigned nb)
    {
        const Slot & sl = T[blockIdx.z];
        if (! live(sl) || sl.s->run == 0)
            return;
        double d1, d2;
        k::sum_partials2(sl.partials, nb, d1, d2);
        if (threadIdx.x == 0)
            sl.s->alpha = (float)d1 / (float)d2;
    }

    __global__ __launch_bounds__(256) void v_axpy_alpha_kernel(const Slot * T, int L, int64_t n)
    {
        const VB vb = vblock();
        HS_GATE_RUN
        const int64_t i = (int64_t)vb.x * blockDim.x + threadIdx.x;
        if (i >= n)
            return;
        const float alpha = sl.s->alpha;
        float * x = sl.v[L][F_X];
        const float * c = sl.v[L][F_C];
        x[i] = x[i] + alpha * c[i];
    }
#undef HS_GATE_RUN

    __global__ void report_kernel(const Slot * T, unsigned nslots, Report * out)
    {
        const unsigned z = blockIdx.x * blockDim.x + threadIdx.x;
        if (z >= nslots)
            return;
        const Scalars * s = T[z].s;
        Report r;
        if (s == nullptr)
        {
            r.phase = PH_IDLE;
            r.status = 0;
            r.outer_iters = r.inner_total = r.cg_iters = r.ticks = 0;
            r.initial_defect = r.def_norm = 0.0;
        }
        else
        {
            r.phase = s->phase;
            r.status = s->status;
            r.outer_iters = s->outer_iters;
            r.inner_total = s->inner_total;
            r.cg_iters = s->cg_iters;
            r.ticks = s->ticks;
            r.initial_defect = s->initial_defect;
            r.def_norm = s->def_norm;
        }
        out[z] = r;
    }

    // ----------------------------------------------------------------- setup
    // b_i = -1 + 2 u_i, u_i = (bits_i >> 11) 2^-53 with SplitMix64 counters;
    // 0 on the boundary nodes of the square grid
    __global__ __launch_bounds__(256) void rhs_uniform_kernel(double * b, int64_t n, int64_t sq, uint64_t key)
    {
        const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
        if (i >= n)
            return;
        const int64_t r = i / sq, c = i - r * sq;
        if (r == 0 || r == sq - 1 || c == 0 || c == sq - 1)
        {
            b[i] = 0.0;
            return;
        }
        const uint64_t bits = mix64(key + 0x9E3779B97F4A7C15ull * ((uint64_t)i + 1));
        const double u = (double)(bits >> 11) * 0x1.0p-53;
        b[i] = -1.0 + 2.0 * u;
    }

    // dinv = (float)((double)(1/dd) * 0.7): ElementInverse then Scale by a
    // double factor, as the reference tests build MGInfo::diags_inverted
    __global__ void dinv_kernel(const float * __restrict__ dd, float * __restrict__ dinv, int64_t n)
    {
        const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
        if (k >= n)
            return;
        float v = dd[k];
        if (v != 0.0f)
            v = 1.0f / v;
        dinv[k] = (float)((double)v * 0.7);
    }

    inline uint64_t align256(uint64_t b) { return (b + 255) & ~(uint64_t)255; }
    inline unsigned lanes4(uint64_t n) { return grid_for((n + 3) / 4, kBlock); }
}  // namespace

void * Hierarchy::alloc(size_t b)
{
    void * ptr = nullptr;
    hipError_t e = hipMalloc(&ptr, b ? b : 1);
    if (e != hipSuccess)
        throw Error(HSOLVE_ERR_ALLOC, "MG hierarchy allocation of " + std::to_string(b) + " bytes failed");
    allocations.push_back(ptr);
    bytes += b;
    return ptr;
}

Hierarchy::~Hierarchy()
{
    for (void * a : allocations)
        (void)hipFree(a);
}

Params make_params(const hsolve_mg_params & p)
{
    Params q;
    q.min_level = p.min_level;
    q.n_max_iter = p.n_max_iter;
    q.initial_zero = p.initial_zero;
    q.convergence_check = p.convergence_check;
    q.tolerance = (float)p.tolerance;
    q.n_pre_smooth = p.n_pre_smooth;
    q.adapt = (float)p.adapt_correction_factor;
    for (int i = 0; i < 8; ++i)
        q.mask.dir[i] = (p.macro_border_mask[i] == 2) ? 1 : 0;
    q.max_outer = p.max_outer;
    return q;
}

namespace
{
    // The occupancy of every one-pass kernel, looked up at set-up, never
    // under stream capture.
    // Dynamic LDS v_bottom_lds_kernel may take on the current device (cached per
    // device): the device's per-workgroup limit, once the kernels are allowed
    // more than 64 KiB, else 60 KiB (4 KiB of either left for its static LDS)
    inline unsigned bottom_lds_limit()
    {
        static std::mutex mu;
        static std::map<int, unsigned> cache;
        int dev = 0;
        HIP_CHECK(hipGetDevice(&dev));
        std::lock_guard<std::mutex> lock(mu);
        auto it = cache.find(dev);
        if (it != cache.end())
            return it->second;
        int v = 0;
        HIP_CHECK(hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        // (4 KiB left for the kernel's static LDS)
        const int want = v - 4096;
        unsigned r = (unsigned)std::min(std::max(want, 0), 65536 - 4096);
        if (want > 65536 &&
            hipFuncSetAttribute((const void *)v_bottom_lds_kernel<0>, hipFuncAttributeMaxDynamicSharedMemorySize, want) ==
                hipSuccess &&
            hipFuncSetAttribute((const void *)v_bottom_lds_kernel<2>, hipFuncAttributeMaxDynamicSharedMemorySize, want) ==
                hipSuccess)
            r = (unsigned)want;
        (void)hipGetLastError();
        cache.emplace(dev, r);
        return r;
    }

    void warm_post_kernels()
    {
#define HS_W(MK, KS, VS, CB)                                                                                   \
    (const void *)v_pre2r_kernel<MK, 0, KS, VS, CB>, (const void *)v_pre2r_kernel<MK, 1, KS, VS, CB>,          \
        (const void *)v_post2_kernel<MK, 0, 0, KS, VS, CB>, (const void *)v_post2_kernel<MK, 0, 1, KS, VS, CB>, \
        (const void *)v_post2_kernel<MK, 1, 0, KS, VS, CB>, (const void *)v_post2_kernel<MK, 1, 1, KS, VS, CB>
        const void * fns[] = {HS_W(0, 1, 1, 0), HS_W(0, 2, 1, 0), HS_W(0, 1, 2, 1), HS_W(0, 1, 1, 2),
                              HS_W(2, 1, 1, 0), HS_W(2, 2, 1, 0), HS_W(2, 1, 2, 1), HS_W(2, 1, 1, 2)};
#undef HS_W
        for (const void * f : fns)
            (void)post_resident(f);
        (void)bottom_lds_limit();
    }
}

void hierarchy_alloc(Hierarchy & h, const Params & p, uint64_t max_level)
{
    warm_post_kernels();
    require(p.min_level >= 1 && p.min_level <= max_level && max_level < (uint64_t)kMaxLevels, HSOLVE_ERR_INVALID,
            "mg: need 1 <= min_level <= max_level <= 14");
    require(p.n_pre_smooth >= 1, HSOLVE_ERR_INVALID, "mg: n_pre_smooth must be >= 1");
    require(p.n_max_iter >= 1, HSOLVE_ERR_INVALID, "mg: n_max_iter must be >= 1");
    require(size_of(p.min_level) <= 16641, HSOLVE_ERR_INVALID, "mg: coarsest level above 129^2");
    h.p = p;
    h.max_level = max_level;
    for (uint64_t L = p.min_level; L <= max_level; ++L)
    {
        HierLevel & l = h.lv[L];
        l.side = side_of(L);
        l.n = size_of(L);
        l.bs = band_stride(l.n);
        l.bands = (float *)h.alloc(sizeof(float) * 9 * l.bs);
        l.dinv = (float *)h.alloc(sizeof(float) * l.bs);
    }
}

void hierarchy_alloc64(Hierarchy & h, uint64_t L)
{
    require(L >= h.p.min_level && L <= h.max_level, HSOLVE_ERR_INVALID, "mg: FP64 level outside the hierarchy");
    if (h.bands64[L])
        return;
    h.bs64[L] = band_stride(size_of(L));
    h.bands64[L] = (double *)h.alloc(sizeof(double) * 9 * h.bs64[L]);
}

void hierarchy_dinv(Hierarchy & h, uint64_t L, hipStream_t st)
{
    HierLevel & l = h.lv[L];
    hipLaunchKernelGGL(dinv_kernel, dim3(grid_for(l.n, kBlock)), dim3(kBlock), 0, st,
                       (const float *)(l.bands + 4 * l.bs), l.dinv, (int64_t)l.n);
    HIP_CHECK(hipGetLastError());
}

void hierarchy_fill_poisson(Hierarchy & h, hipStream_t st)
{
    for (uint64_t L = h.p.min_level; L <= h.max_level; ++L)
    {
        HierLevel & l = h.lv[L];
        hipLaunchKernelGGL((k::fill_poisson_kernel<float>), dim3(grid_for(l.n, kBlock)), dim3(kBlock), 0, st, l.B(),
                           (int64_t)l.n, l.side);
        hierarchy_dinv(h, L, st);
        if (h.bands64[L])
            hipLaunchKernelGGL((k::fill_poisson_kernel<double>), dim3(grid_for(l.n, kBlock)), dim3(kBlock), 0, st,
                               h.B64(L), (int64_t)l.n, l.side);
    }
    HIP_CHECK(hipGetLastError());
    hierarchy_codes(h);
}

namespace
{
    // The distinct words of `code` (at most kRowCodes of them) and each
    // entry's index among them; false when there are more.
    bool row_codes(const std::vector<uint64_t> & code, std::vector<uint8_t> & rc, std::vector<uint64_t> & words)
    {
        std::unordered_map<uint64_t, uint8_t> at;
        rc.resize(code.size());
        uint64_t last = 0;
        uint8_t last_t = 0;
        for (size_t i = 0; i < code.size(); ++i)
        {
            if (i == 0 || code[i] != last)
            {
                auto it = at.find(code[i]);
                if (it == at.end())
                {
                    if (words.size() == (size_t)kRowCodes)
                        return false;
                    it = at.emplace(code[i], (uint8_t)words.size()).first;
                    words.push_back(code[i]);
                }
                last = code[i];
                last_t = it->second;
            }
            rc[i] = last_t;
        }
        return true;
    }
}

// Value-indexed storage of a level's bands (Q1, or a 9-point structured ELL
// matrix kept as bands) and dinv (the value-index
// compression of Kourtis, Goumas and Koziris, "Optimizing sparse
// matrix-vector multiplication using index and value compression", 2008):
// when each of the ten arrays holds at most 16 distinct values (as bit
// patterns) over the level's n nodes, node i's ten 4-bit indices go into one
// 64-bit word and the values into a 16-entry table per array.  The one-pass
// kernels then read 8 bytes per node instead of 40 and look the values up
// in LDS: the same floats, so the same bits.  Where at most kRowCodes of the
// words are distinct (Poisson rows: a handful) a node keeps one byte, the
// index of its row among them.  Levels whose arrays hold more values keep the
// plain bands only.  The FP64 bands of a finest level likewise.
void hierarchy_codes(Hierarchy & h)
{
    if (h.kind == 1)    // ELL matrices: no bands
        return;
    HIP_CHECK(hipDeviceSynchronize());
    for (uint64_t L = h.p.min_level; L <= h.max_level; ++L)
    {
        HierLevel & l = h.lv[L];
        l.codes = nullptr;
        l.ctab = nullptr;
        l.rcode = nullptr;
        if (l.n < 4225)     // the one-pass kernels run on levels of 65^2 and up
            continue;
        const uint64_t n = l.n;
        std::vector<uint32_t> v(n);
        std::vector<uint64_t> code(n, 0);
        uint32_t tab[160] = {};
        bool ok = true;
        for (int k = 0; k < 10 && ok; ++k)
        {
            const float * src = k < 9 ? l.bands + (uint64_t)k * l.bs : l.dinv;
            HIP_CHECK(hipMemcpy(v.data(), src, sizeof(float) * n, hipMemcpyDeviceToHost));
            int cnt = 0;
            uint32_t last = 0;
            uint64_t last_t = 0;
            for (uint64_t i = 0; i < n; ++i)
            {
                const uint32_t bits = v[i];
                uint64_t t = last_t;
                if (cnt == 0 || bits != last)
                {
                    int f = -1;
                    for (int q = 0; q < cnt; ++q)
                        if (tab[16 * k + q] == bits)
                        {
                            f = q;
                            break;
                        }
                    if (f < 0)
                    {
                        if (cnt == 16)
                        {
                            ok = false;
                            break;
                        }
                        f = cnt;
                        tab[16 * k + cnt++] = bits;
                    }
                    t = (uint64_t)f;
                    last = bits;
                    last_t = t;
                }
                code[i] |= t << (4 * k);
            }
        }
        if (! ok)
            continue;
        std::vector<uint8_t> rc;
        std::vector<uint64_t> words;
        if (row_codes(code, rc, words))
        {
            // (16 bytes of padding on either side: the kernels load pairs)
            std::vector<float> rows(12 * words.size(), 0.0f);
            for (size_t t = 0; t < words.size(); ++t)
                for (int k = 0; k < 10; ++k)
                    std::memcpy(&rows[12 * t + k], &tab[16 * k + ((words[t] >> (4 * k)) & 15u)], sizeof(float));
            l.rcode = (uint8_t *)h.alloc(n + 32) + 16;
            l.rtab = (float *)h.alloc(sizeof(float) * rows.size());
            l.rows = (int)words.size();
            HIP_CHECK(hipMemcpy(l.rcode, rc.data(), n, hipMemcpyHostToDevice));
            HIP_CHECK(hipMemcpy(l.rtab, rows.data(), sizeof(float) * rows.size(), hipMemcpyHostToDevice));
            continue;
        }
        l.codes = (uint64_t *)h.alloc(sizeof(uint64_t) * n);
        l.ctab = (float *)h.alloc(sizeof(tab));
        HIP_CHECK(hipMemcpy(l.codes, code.data(), sizeof(uint64_t) * n, hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(l.ctab, tab, sizeof(tab), hipMemcpyHostToDevice));
    }
    // the FP64 bands of the finest levels solved on (the outer defect, whose
    // coded path forms Product<Q1>'s order: Q1 hierarchies only)
    for (uint64_t L = h.p.min_level; h.kind == 0 && L <= h.max_level; ++L)
    {
        h.codes64[L] = nullptr;
        h.ctab64[L] = nullptr;
        h.rcode64[L] = nullptr;
        if (! h.bands64[L] || size_of(L) < 4225)
            continue;
        const uint64_t n = size_of(L);
        std::vector<uint64_t> v(n), code(n, 0);
        uint64_t tab[144] = {};
        bool ok = true;
        for (int k = 0; k < 9 && ok; ++k)
        {
            HIP_CHECK(hipMemcpy(v.data(), h.bands64[L] + (uint64_t)k * h.bs64[L], sizeof(double) * n,
                                hipMemcpyDeviceToHost));
            int cnt = 0;
            uint64_t last = 0, last_t = 0;
            for (uint64_t i = 0; i < n; ++i)
            {
                const uint64_t bits = v[i];
                uint64_t t = last_t;
                if (cnt == 0 || bits != last)
                {
                    int f = -1;
                    for (int q = 0; q < cnt; ++q)
                        if (tab[16 * k + q] == bits)
                        {
                            f = q;
                            break;
                        }
                    if (f < 0)
                    {
                        if (cnt == 16)
                        {
                            ok = false;
                            break;
                        }
                        f = cnt;
                        tab[16 * k + cnt++] = bits;
                    }
                    t = (uint64_t)f;
                    last = bits;
                    last_t = t;
                }
                code[i] |= t << (4 * k);
            }
        }
        if (! ok)
            continue;
        std::vector<uint8_t> rc;
        std::vector<uint64_t> words;
        if (row_codes(code, rc, words))
        {
            std::vector<uint64_t> rows(9 * words.size());
            for (size_t t = 0; t < words.size(); ++t)
                for (int k = 0; k < 9; ++k)
                    rows[9 * t + k] = tab[16 * k + ((words[t] >> (4 * k)) & 15u)];
            h.rcode64[L] = (uint8_t *)h.alloc(n);
            h.rtab64[L] = (double *)h.alloc(sizeof(double) * rows.size());
            h.rows64[L] = (int)words.size();
            HIP_CHECK(hipMemcpy(h.rcode64[L], rc.data(), n, hipMemcpyHostToDevice));
            HIP_CHECK(hipMemcpy(h.rtab64[L], rows.data(), sizeof(double) * rows.size(), hipMemcpyHostToDevice));
            continue;
        }
        h.codes64[L] = (uint64_t *)h.alloc(sizeof(uint64_t) * n);
        h.ctab64[L] = (double *)h.alloc(sizeof(tab));
        HIP_CHECK(hipMemcpy(h.codes64[L], code.data(), sizeof(uint64_t) * n, hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(h.ctab64[L], tab, sizeof(tab), hipMemcpyHostToDevice));
    }
}

namespace
{
    // HONEI-layout host ELL (threads == 1) -> engine ELL in device memory
    template <typename DT>
    EllMat<DT> upload_ell(Hierarchy & h, const EllHost & e)
    {
        require(e.Aj && e.Ax && e.Arl, HSOLVE_ERR_INVALID, "mg ELL level: null array");
        require(e.rows < (1ull << 32) && e.cols < (1ull << 32), HSOLVE_ERR_SIZE, "mg ELL level: too many rows");
        require(e.stride >= e.rows, HSOLVE_ERR_INVALID, "mg ELL level: stride below rows");
        const uint64_t size = e.stride * e.ncpr;
        std::vector<uint32_t> col(size), len(e.rows);
        for (uint64_t i = 0; i < size; ++i)
        {
            require(e.Aj[i] < (e.cols ? e.cols : 1), HSOLVE_ERR_INVALID, "mg ELL level: column out of range");
            col[i] = (uint32_t)e.Aj[i];
        }
        for (uint64_t r = 0; r < e.rows; ++r)
        {
            require(e.Arl[r] <= e.ncpr, HSOLVE_ERR_INVALID, "mg ELL level: row length above num_cols_per_row");
            len[r] = (uint32_t)e.Arl[r];
        }
        EllMat<DT> m;
        uint32_t * c = (uint32_t *)h.alloc(sizeof(uint32_t) * (size ? size : 1));
        DT * v = (DT *)h.alloc(sizeof(DT) * (size ? size : 1));
        uint32_t * l = (uint32_t *)h.alloc(sizeof(uint32_t) * (e.rows ? e.rows : 1));
        HIP_CHECK(hipMemcpy(c, col.data(), sizeof(uint32_t) * size, hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(v, e.Ax, sizeof(DT) * size, hipMemcpyHostToDevice));
        HIP_CHECK(hipMemcpy(l, len.data(), sizeof(uint32_t) * e.rows, hipMemcpyHostToDevice));
        m.col = c;
        m.val = v;
        m.len = l;
        m.stride = e.stride;
        m.rows = e.rows;
        m.cols = e.cols;
        m.ncpr = (uint32_t)e.ncpr;
        return m;
    }
}

namespace
{
    // neighbour position (dy + 1) * 3 + (dx + 1) of column c in row r of a
    // side-M grid, or -1 when c is not one of the 9 neighbours
    int q1_position(uint64_t r, uint64_t c, uint64_t M)
    {
        const int64_t dy = (int64_t)(c / M) - (int64_t)(r / M), dx = (int64_t)(c % M) - (int64_t)(r % M);
        if (dy < -1 || dy > 1 || dx < -1 || dx > 1)
            return -1;
        return (int)((dy + 1) * 3 + (dx + 1));
    }

    // 9-point structure of a host ELL on the (2^L+1)^2 grid: every stored
    // column of a row is one of its neighbours, in ascending order
    bool ell_is_q1(const EllHost & e, uint64_t L)
    {
        const uint64_t M = (uint64_t)side_of(L);
        if (e.rows != size_of(L) || e.cols != e.rows || e.ncpr > 9 || ! e.Aj || ! e.Ax || ! e.Arl)
            return false;
        for (uint64_t r = 0; r < e.rows; ++r)
        {
            if (e.Arl[r] > e.ncpr)
                return false;
            int prev = -1;
            for (uint64_t k = 0; k < e.Arl[r]; ++k)
            {
                const int q = q1_position(r, e.Aj[r + k * e.stride], M);
                if (q <= prev)
                    return false;
                prev = q;
            }
        }
        return true;
    }

    // the matrix as 9 bands LL .. UU (band b of row r at b * bs + r), zero
    // where the row has no entry
    template <typename DT>
    std::vector<DT> ell_bands(const EllHost & e, uint64_t L, uint64_t bs)
    {
        const uint64_t M = (uint64_t)side_of(L);
        std::vector<DT> out(9 * bs, DT(0));
        const DT * ax = (const DT *)e.Ax;
        for (uint64_t r = 0; r < e.rows; ++r)
            for (uint64_t k = 0; k < e.Arl[r]; ++k)
                out[(uint64_t)q1_position(r, e.Aj[r + k * e.stride], M) * bs + r] = ax[r + k * e.stride];
        return out;
    }
}

void hierarchy_alloc_ell(Hierarchy & h, const Params & p, uint64_t max_level, const EllHost * a32,
                         const EllHost & A64, const float * const * dinv32, const EllHost * prol32,
                         const EllHost * res32)
{
    require(p.min_level >= 1 && p.min_level <= max_level && max_level < (uint64_t)kMaxLevels, HSOLVE_ERR_INVALID,
            "mg: need 1 <= min_level <= max_level <= 14");
    require(p.n_pre_smooth >= 1, HSOLVE_ERR_INVALID, "mg: n_pre_smooth must be >= 1");
    require(p.n_max_iter >= 1, HSOLVE_ERR_INVALID, "mg: n_max_iter must be >= 1");
    require(a32 != nullptr, HSOLVE_ERR_INVALID, "mg: null level matrices");
    require((prol32 == nullptr) == (res32 == nullptr), HSOLVE_ERR_INVALID, "mg: give both prol and res or neither");
    // 9-point structured levels with structured transfers: kept as bands
    // (kind 2, summed in the ELL rows' order), read with 16-byte vectors
    bool banded = prol32 == nullptr && ell_is_q1(A64, max_level) && size_of(p.min_level) <= 16641;
    for (uint64_t L = p.min_level; banded && L <= max_level; ++L)
        banded = ell_is_q1(a32[L], L);
    if (banded)
    {
        hierarchy_alloc(h, p, max_level);
        hierarchy_alloc64(h, max_level);
        h.kind = 2;
        h.prolmat = 0;
        for (uint64_t L = p.min_level; L <= max_level; ++L)
        {
            HierLevel & l = h.lv[L];
            const std::vector<float> b = ell_bands<float>(a32[L], L, l.bs);
            HIP_CHECK(hipMemcpy(l.bands, b.data(), sizeof(float) * b.size(), hipMemcpyHostToDevice));
            std::vector<float> dv(l.n);
            if (dinv32 && dinv32[L])
                std::memcpy(dv.data(), dinv32[L], sizeof(float) * l.n);
            else
                for (uint64_t r = 0; r < l.n; ++r)
                {
                    // diags_inverted as the reference tests build it
                    const float dd = b[4 * l.bs + r];
                    const float inv = dd != 0.0f ? 1.0f / dd : 0.0f;
                    dv[r] = (float)((double)inv * 0.7);
                }
            HIP_CHECK(hipMemcpy(l.dinv, dv.data(), sizeof(float) * l.n, hipMemcpyHostToDevice));
        }
        const std::vector<double> b64 = ell_bands<double>(A64, max_level, h.bs64[max_level]);
        HIP_CHECK(hipMemcpy(h.bands64[max_level], b64.data(), sizeof(double) * b64.size(), hipMemcpyHostToDevice));
        hierarchy_codes(h);
        return;
    }
    h.p = p;
    h.kind = 1;
    h.prolmat = prol32 ? 1 : 0;
    h.max_level = max_level;
    for (uint64_t L = p.min_level; L <= max_level; ++L)
    {
        const EllHost & e = a32[L];
        require(e.rows == e.cols, HSOLVE_ERR_SIZE, "mg: level matrix is not square");
        HierLevel & l = h.lv[L];
        l.n = e.rows;
        l.side = (int64_t)std::sqrt((double)e.rows);
        if (! h.prolmat)
            require(e.rows == size_of(L), HSOLVE_ERR_SIZE,
                    "mg: structured transfers need level L of size (2^L+1)^2");
        l.ell = upload_ell<float>(h, e);
        l.dinv = (float *)h.alloc(sizeof(float) * (l.n ? l.n : 1));
        std::vector<float> dv(l.n);
        if (dinv32 && dinv32[L])
            std::memcpy(dv.data(), dinv32[L], sizeof(float) * l.n);
        else
        {
            // diags_inverted as the reference tests build it: ElementInverse, then
            // Scale by 0.7 in double
            const float * ax = (const float *)e.Ax;
            for (uint64_t r = 0; r < l.n; ++r)
            {
                float dd = 0.0f;
                for (uint64_t k = 0; k < e.Arl[r]; ++k)
                    if (e.Aj[r + k * e.stride] == r)
                    {
                        dd = ax[r + k * e.stride];
                        break;
                    }
                const float inv = dd != 0.0f ? 1.0f / dd : 0.0f;
                dv[r] = (float)((double)inv * 0.7);
            }
        }
        HIP_CHECK(hipMemcpy(l.dinv, dv.data(), sizeof(float) * l.n, hipMemcpyHostToDevice));
        if (h.prolmat && L > p.min_level)
        {
            require(prol32[L].rows == l.n && prol32[L].cols == a32[L - 1].rows, HSOLVE_ERR_SIZE,
                    "mg: prolongation matrix shape");
            require(res32[L].rows == a32[L - 1].rows && res32[L].cols == l.n, HSOLVE_ERR_SIZE,
                    "mg: restriction matrix shape");
            l.prol = upload_ell<float>(h, prol32[L]);
            l.res = upload_ell<float>(h, res32[L]);
        }
    }
    require(h.lv[p.min_level].n <= 1048576, HSOLVE_ERR_INVALID, "mg: coarsest level above 2^20 rows");
    require(A64.rows == h.lv[max_level].n && A64.cols == A64.rows, HSOLVE_ERR_SIZE,
            "mg: FP64 matrix size differs from the finest level");
    h.ell64[max_level] = upload_ell<double>(h, A64);
}

namespace
{
    // doubles of a slot's partial sums, finest level of side m: the regions
    // named in mg_engine.hh
    uint64_t slot_partials(int64_t m)
    {
        return kCyclePartials + std::min<uint64_t>(kMaxTiles, march_tiles<1>(m, 2));
    }
}

uint64_t slot_bytes(const Hierarchy & h, uint64_t L, bool own_b, bool own_result)
{
    const uint64_t n = h.lv[L].n;
    uint64_t b = align256(sizeof(Scalars)) + align256(sizeof(double) * slot_partials(h.lv[L].side));
    b += align256(sizeof(double) * n);                                  // od
    if (own_b)
        b += align256(sizeof(double) * n);
    if (own_result)
        b += align256(sizeof(double) * n);
    b += align256(sizeof(float) * 4 * h.lv[h.p.min_level].n);           // coarse CG
    for (uint64_t l = h.p.min_level; l <= L; ++l)
        b += 5 * align256(sizeof(float) * h.lv[l].n);
    return b;
}

Slot slot_carve(const Hierarchy & h, uint64_t L, char * base, bool own_b, bool own_result)
{
    Slot sl;
    std::memset(&sl, 0, sizeof(sl));
    const uint64_t n = h.lv[L].n;
    char * c = base;
    auto take = [&](uint64_t bytes) {
        char * r = c;
        c += align256(bytes);
        return r;
    };
    sl.s = (Scalars *)take(sizeof(Scalars));
    sl.partials = (double *)take(sizeof(double) * slot_partials(h.lv[L].side));
    sl.od = (double *)take(sizeof(double) * n);
    if (own_b)
        sl.b = (const double *)take(sizeof(double) * n);
    if (own_result)
        sl.result = (double *)take(sizeof(double) * n);
    sl.cg_work = (float *)take(sizeof(float) * 4 * h.lv[h.p.min_level].n);
    for (uint64_t l = h.p.min_level; l <= L; ++l)
        for (int f = 0; f < 5; ++f)
            sl.v[l][f] = (float *)take(sizeof(float) * h.lv[l].n);
    return sl;
}

Scalars start_scalars(bool zero_guess)
{
    Scalars s;
    std::memset(&s, 0, sizeof(s));
    s.phase = PH_START;
    s.outer_active = 1;
    s.zero_guess = zero_guess ? 1 : 0;
    return s;
}

void enqueue_rhs_uniform(double * b, uint64_t L, uint64_t seed, uint64_t stream, hipStream_t st)
{
    const uint64_t key = mix64(seed + 0x9E3779B97F4A7C15ull * (stream + 1));
    const uint64_t n = size_of(L);
    hipLaunchKernelGGL(rhs_uniform_kernel, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, st, b, (int64_t)n,
                       side_of(L), key);
    HIP_CHECK(hipGetLastError());
}

void enqueue_report(const Slot * table, unsigned nslots, Report * reports, hipStream_t st)
{
    hipLaunchKernelGGL(report_kernel, dim3(grid_for(nslots, 64)), dim3(64), 0, st, table, nslots, reports);
    HIP_CHECK(hipGetLastError());
}

namespace
{
template <int MK>
void tick_impl(const Hierarchy & h, uint64_t maxl, const Slot * T, unsigned S, unsigned part, hipStream_t st)
{
    const Params & p = h.p;
    const uint64_t minl = p.min_level;
    require(maxl >= minl && maxl <= h.max_level && (MK == 1 ? h.ell64[maxl].val != nullptr : h.bands64[maxl] != nullptr),
            HSOLVE_ERR_INVALID,
            "mg tick: level not prepared");
    const HierLevel & top = h.lv[maxl];
    const int64_t n = (int64_t)top.n;
    const dim3 blk(kBlock);
    auto largs = [&](uint64_t L) {
        const HierLevel & l = h.lv[L];
        LevelArgs a;
        a.B = l.B();
        a.E = l.ell;
        a.dinv = l.dinv;
        a.n = (int64_t)l.n;
        a.m = l.side;
        a.bs = (int64_t)l.bs;
        a.rcode = h.use_codes ? l.rcode : nullptr;
        a.rtab = l.rtab;
        a.rows = l.rows;
        a.codes = h.use_codes ? l.codes : nullptr;
        a.ctab = l.ctab;
        return a;
    };
    // The form of the one-pass kernels on a level: slots per workgroup, columns
    // per lane, matrix storage.  Row codes leave registers for two columns a
    // lane; with plain bands several slots share a tile's 40 bytes per node.
    auto march_form = [&](const LevelArgs & a, auto && f) {
        if (a.rcode)
            f(IntC<1>{}, IntC<2>{}, IntC<1>{});
        else if (a.codes)
            f(IntC<1>{}, IntC<1>{}, IntC<2>{});
        else if (S > 1)
            f(IntC<2>{}, IntC<1>{}, IntC<0>{});
        else
            f(IntC<1>{}, IntC<1>{}, IntC<0>{});
    };
    auto norm_grid = [&](uint64_t nn) { return dim3(std::min<unsigned>(lanes4(nn), kNormBlocks), 1, S); };
    // row kernels: 4 rows per lane on Q1 bands, one row per lane on ELL
    auto rgrid = [&](uint64_t nn) { return kBands<MK> ? lanes4(nn) : grid_for(nn, kBlock); };
    // Post-smoothing in one pass (v_post2_kernel) on Q1 bands with two
    // sweeps: a level's smoothed iterate then lands in F_TMP, so the
    // prolongation out of a level above the coarsest reads F_TMP, and the
    // finest level's iterate lives in F_TMP between V-cycles (the start
    // writes it there, the outer step and the next cycle's first sweeps
    // read it there).
    // (the one-pass kernels address a level's nine bands by 32-bit offsets
    // from the first: levels up to 8193^2)
    const bool post2 = kBands<MK> && p.n_pre_smooth == 2 && maxl > minl && 36 * h.lv[maxl].bs < (1ull << 32);
    const int fx_top = post2 ? F_TMP : F_X;
    // Pre-smoothing, defect and restriction in one pass (v_pre2r_kernel)
    // when the transfers are the structured ones and the correction factor
    // is fixed (the adaptive one reads the level's defect again).
    const bool pre2r = post2 && p.adapt != 0.0f && ! h.prolmat;
    // With the one-pass kernels, levels minl .. btop (btop <= 6, below the
    // finest) run in one launch, one workgroup per slot: v_bottom_kernel when
    // the coarsest level fits one wave (5^2 or less), v_bottom_lds_kernel with
    // as many levels as fit the LDS of a workgroup otherwise; btop = 0: none.
    int btop = 0;
    BottomLdsArgs ba{};
    size_t bbytes = 0;
    if (pre2r && maxl - 1 > minl)
    {
        const int most = (int)std::min<uint64_t>(kBottomMax, maxl - 1);
        if (minl <= 2)
            btop = most;
        else
            for (int top = most; top > (int)minl; --top)
            {
                size_t fl = 0;
                for (int L = (int)minl; L <= top; ++L)
                    fl += (size_t)bottom_floats((int)h.lv[L].n, L == (int)minl);
                if (fl * sizeof(float) <= bottom_lds_limit())
                {
                    btop = top;
                    bbytes = fl * sizeof(float);
                    break;
                }
            }
        if (btop)
        {
            int off = 0;
            for (int L = (int)minl; L <= btop; ++L)
            {
                ba.b.lv[L] = largs(L);
                ba.off[L] = off;
                off += bottom_floats((int)h.lv[L].n, L == (int)minl);
            }
            ba.minl = (int)minl;
            ba.b.top = btop;
            ba.b.alpha = p.adapt;
            ba.b.mk = p.mask;
            ba.b.konv_rad = (double)1.19209290e-07F;
            ba.b.max_iters = (uint64_t)(100 * h.lv[minl].n + 1000);
        }
    }

    // ---- start of new solves, FP64 outer step, opening of inner solves
    // the per-tick kernels that most ticks skip (start, outer step, opening
    // of an inner solve) loop over their rows on a capped grid, so a skipped
    // launch costs a few thousand empty workgroups, not one per 256 rows
    auto ggrid = [&](uint64_t blocks) {
        return dim3((unsigned)std::min<uint64_t>(blocks, std::max<unsigned>(64u, kGateBlocks / S)), 1, S);
    };
    // The opening of an inner solve folded into its neighbours: the cast to
    // FP32 forms the initial norm, the first cycle reads rhs as its defect
    // (initial_zero) and the first stopping test finishes the norm.
    const bool fold = pre2r && p.initial_zero && ! p.convergence_check;
    const unsigned open_blocks = fold ? std::min<unsigned>(ggrid(lanes4(top.n)).x, kNormBlocks) : 0;
    if (part & kTickOpen)
    {
        hipLaunchKernelGGL(tick_begin_kernel, ggrid(grid_for(top.n, kBlock)), blk, 0, st, T, (int)maxl, n, top.side, fx_top);
        if (maxl > minl && ! pre2r)
        {
            // (the one-pass kernels write every coarser iterate before it is read)
            LevelSizes sz;
            for (int l = 0; l < kMaxLevels; ++l)
                sz.n[l] = (int64_t)h.lv[l].n;
            hipLaunchKernelGGL(start_zero_kernel, ggrid(grid_for(h.lv[maxl - 1].n, kBlock)), blk, 0, st, T,
                               (int)minl, (int)maxl, sz);
        }
        const unsigned od_blocks = std::min<unsigned>(grid_for((top.n + 1) / 2, kBlock), kNormBlocks);
        bool od_coded = false;
        if constexpr (MK == 0)
        {
            auto go = [&](auto cb_tag, const void * codes, const double * tab) {
                hipLaunchKernelGGL((outer_defect_kernel<MK, decltype(cb_tag)::value>), dim3(od_blocks, 1, S), blk, 0, st,
                                   h.B64(maxl), h.ell64[maxl], T, n, top.side, codes, tab, h.rows64[maxl], (int)S);
                od_coded = true;
            };
            if (h.use_codes && h.rcode64[maxl])
                go(IntC<1>{}, h.rcode64[maxl], h.rtab64[maxl]);
            else if (h.use_codes && h.codes64[maxl])
                go(IntC<2>{}, h.codes64[maxl], h.ctab64[maxl]);
        }
        if (! od_coded)
        {
            auto go = [&](auto k_tag) {
                constexpr int KS = decltype(k_tag)::value;
                hipLaunchKernelGGL((outer_defect_kernel<MK, 0, KS>), dim3(od_blocks, 1, (S + KS - 1) / KS), blk, 0, st,
                                   kBands<MK> ? h.B64(maxl) : k::Bands{}, h.ell64[maxl], T, n, top.side,
                                   (const void *)nullptr, (const double *)nullptr, 0, (int)S);
            };
            if constexpr (kBands<MK>)
            {
                if (S > 2)
                    go(IntC<4>{});
                else if (S == 2)
                    go(IntC<2>{});
                else
                    go(IntC<1>{});
            }
            else
                go(IntC<1>{});
        }
        hipLaunchKernelGGL(outer_defect_finish_kernel, dim3(1, 1, S), blk, 0, st, T, od_blocks, (double)p.tolerance,
                           p.max_outer, fold ? 1 : 0);
        if (fold)
        {
            hipLaunchKernelGGL((to_inner_kernel<true>), dim3(open_blocks, 1, S), blk, 0, st, T, (int)maxl, n);
        }
        else
        {
            hipLaunchKernelGGL((to_inner_kernel<false>), ggrid(lanes4(top.n)), blk, 0, st, T, (int)maxl, n);
            if (p.initial_zero)
                hipLaunchKernelGGL((open_inner_kernel<1, MK>), ggrid(lanes4(top.n)), blk, 0, st, largs(maxl), T,
                                   (int)maxl, fx_top);
            else
                hipLaunchKernelGGL((open_inner_kernel<0, MK>), ggrid(rgrid(top.n)), blk, 0, st, largs(maxl), T,
                                   (int)maxl, fx_top);
            hipLaunchKernelGGL((inner_norm_kernel<0>), norm_grid(top.n), blk, 0, st, T, (int)maxl, n);
            hipLaunchKernelGGL((inner_norm_finish_kernel<0>), dim3(1, 1, S), blk, 0, st, T, norm_grid(top.n).x,
                               p.tolerance, p.convergence_check, p.n_max_iter);
        }
    }
    if (! (part & kTickCycle))
    {
        HIP_CHECK(hipGetLastError());
        return;
    }

    // ---- one V-cycle (multigrid.hh:1660-1905)
    const uint64_t npre = p.n_pre_smooth;
    auto sweeps = [&](uint64_t L, int & xc, int & xa, int frhs, uint64_t count) {
        const LevelArgs a = largs(L);
        for (uint64_t i = 0; i < count; ++i)
        {
            hipLaunchKernelGGL((v_sweep_kernel<MK>), dim3(rgrid(a.n), 1, S), blk, 0, st, a, T, (int)L, xc, xa, frhs);
            std::swap(xc, xa);
        }
    };
    auto move = [&](uint64_t L, int fsrc, int fdst, bool add) {
        const int64_t nn = (int64_t)h.lv[L].n;
        if (add)
            hipLaunchKernelGGL((v_move_kernel<1>), dim3(lanes4(nn), 1, S), blk, 0, st, T, (int)L, nn, fsrc, fdst);
        else
            hipLaunchKernelGGL((v_move_kernel<0>), dim3(lanes4(nn), 1, S), blk, 0, st, T, (int)L, nn, fsrc, fdst);
    };
    auto defect = [&](uint64_t L) {
        const LevelArgs a = largs(L);
        hipLaunchKernelGGL((v_defect_kernel<MK>), dim3(rgrid(a.n), 1, S), blk, 0, st, a, T, (int)L);
    };

    if (minl != maxl)
    {
        for (uint64_t L = maxl; L > minl; --L)
        {
            if (btop && L <= (uint64_t)btop)
                break;
            const LevelArgs a = largs(L);
            // the finest level's defect is d; coarser levels' defect is the
            // restricted one in rhs
            const int dsrc = (L == maxl) ? F_D : F_RHS;
            if constexpr (kBands<MK>)
            {
                if (pre2r)
                {
                    const int64_t Nc = h.lv[L - 1].side;
                    auto go = [&](auto acc_tag, auto k_tag, auto v_tag, auto cb_tag) {
                        constexpr int ACC = decltype(acc_tag)::value, KS = decltype(k_tag)::value;
                        constexpr int VS = decltype(v_tag)::value, CB = decltype(cb_tag)::value;
                        auto kern = v_pre2r_kernel<MK, ACC, KS, VS, CB>;
                        const unsigned groups = (S + KS - 1) / KS;
                        const int th = march_rows<VS>(a.m, groups, kMarchWaves * post_resident((const void *)kern));
                        const unsigned tiles = march_tiles<VS>(a.m, th);
                        hipLaunchKernelGGL(kern, dim3((tiles + kMarchWaves - 1) / kMarchWaves, 1, groups), blk, 0, st,
                                           a, T, (int)L, ACC ? fx_top : (int)F_X, Nc, p.mask, th, tiles, (int)S, fold ? 1 : 0);
                    };
                    if (L == maxl)
                        march_form(a, [&](auto k_tag, auto v_tag, auto cb_tag) { go(IntC<1>{}, k_tag, v_tag, cb_tag); });
                    else
                        march_form(a, [&](auto k_tag, auto v_tag, auto cb_tag) { go(IntC<0>{}, k_tag, v_tag, cb_tag); });
                    continue;
                }
            }
            if (L == maxl)
            {
                // c = dinv*d, (npre-1) sweeps on c with rhs d, x += c
                if (npre == 1)
                    hipLaunchKernelGGL((v_zero1_kernel<1>), dim3(grid_for(a.n, kBlock), 1, S), blk, 0, st, a, T,
                                       (int)L, dsrc, (int)F_X);
                else if (npre == 2)
                    hipLaunchKernelGGL((v_zero2_kernel<1, MK>), dim3(rgrid(a.n), 1, S), blk, 0, st, a, T, (int)L, dsrc,
                                       (int)F_X, fx_top);
                else
                {
                    hipLaunchKernelGGL((v_zero2_kernel<0, MK>), dim3(rgrid(a.n), 1, S), blk, 0, st, a, T, (int)L, dsrc,
                                       (int)F_C, (int)F_C);
                    int cc = F_C, ca = F_TMP;
                    sweeps(L, cc, ca, dsrc, npre - 2);
                    move(L, cc, F_X, true);
                }
            }
            else
            {
                // x = dinv*d, (npre-1) sweeps on x with rhs d
                if (npre == 1)
                    hipLaunchKernelGGL((v_zero1_kernel<0>), dim3(grid_for(a.n, kBlock), 1, S), blk, 0, st, a, T,
                                       (int)L, dsrc, (int)F_X);
                else
                {
                    hipLaunchKernelGGL((v_zero2_kernel<0, MK>), dim3(rgrid(a.n), 1, S), blk, 0, st, a, T, (int)L, dsrc,
                                       (int)F_X, (int)F_X);
                    int xc = F_X, xa = F_TMP;
                    sweeps(L, xc, xa, dsrc, npre - 2);
                    if (xc != F_X)
                        move(L, xc, F_X, false);
                }
            }
            defect(L);
            if (h.prolmat)
                hipLaunchKernelGGL(v_apply_ell_kernel, dim3(grid_for(h.lv[L].res.rows, kBlock), 1, S), blk, 0, st, h.lv[L].res,
                                   T, (int)L, (int)F_D, (int)(L - 1), (int)F_RHS);
            else
            {
                const int64_t Nc = h.lv[L - 1].side;
                hipLaunchKernelGGL(v_restrict_kernel, dim3(grid_for(Nc, kBlock), (unsigned)Nc, S), blk, 0, st, T,
                                   (int)L, Nc, p.mask);
            }
        }
    }
    {
        // coarse grid solve: ConjugateGradients<NONE>(A, d, x, FLT_EPSILON);
        // with one level it sees the finest defect d
        const LevelArgs a = largs(minl);
        const int crhs = (minl == maxl) ? F_D : F_RHS;
        auto bottom = [&](auto minl_tag, auto top6_tag) {
            hipLaunchKernelGGL((v_bottom_kernel<MK, decltype(minl_tag)::value, decltype(top6_tag)::value != 0>),
                               dim3(1, 1, S), dim3(kBottomLanes), 0, st, ba.b, T);
        };
        if (btop == 6 && minl == 1)
            bottom(IntC<1>{}, IntC<1>{});
        else if (btop == 6 && minl == 2)
            bottom(IntC<2>{}, IntC<1>{});
        else if (btop && minl == 1)
            bottom(IntC<1>{}, IntC<0>{});
        else if (btop && minl == 2)
            bottom(IntC<2>{}, IntC<0>{});
        else if (btop)
            hipLaunchKernelGGL((v_bottom_lds_kernel<MK>), dim3(1, 1, S), dim3(1024), bbytes, st, ba, T);
        else if (a.n <= kCoarseLdsMax)
            hipLaunchKernelGGL((v_coarse_lds_kernel<MK>), dim3(1, 1, S), dim3(64), 0, st, a, T, (int)minl, crhs,
                               (double)1.19209290e-07F, (uint64_t)(100 * a.n + 1000));
        else
            hipLaunchKernelGGL((v_coarse_kernel<MK>), dim3(1, 1, S), blk, 0, st, a, T, (int)minl, crhs,
                               (double)1.19209290e-07F, (uint64_t)(100 * a.n + 1000));
        if (minl == maxl)
        {
            defect(minl);
            hipLaunchKernelGGL(one_level_end_kernel, dim3(grid_for(S, 64)), dim3(64), 0, st, T, S);
            HIP_CHECK(hipGetLastError());
            return;
        }
    }
    // v_post2_kernel on level L (DEFECT on the finest)
    unsigned cycle_tiles = 0;
    auto post2_launch = [&](uint64_t L, const LevelArgs & a, int fcoarse, float alpha, auto prol_tag) {
        constexpr int PROL = decltype(prol_tag)::value;
        auto go = [&](auto def_tag, auto k_tag, auto v_tag, auto cb_tag) {
            constexpr int DEF = decltype(def_tag)::value, KS = decltype(k_tag)::value;
            constexpr int VS = decltype(v_tag)::value, CB = decltype(cb_tag)::value;
            auto kern = v_post2_kernel<MK, DEF, PROL, KS, VS, CB>;
            const unsigned groups = (S + KS - 1) / KS;
            const int th = march_rows<VS>(a.m, groups, kMarchWaves * post_resident((const void *)kern));
            const unsigned tiles = march_tiles<VS>(a.m, th);
            if (DEF)
                cycle_tiles = tiles;
            hipLaunchKernelGGL(kern, dim3((tiles + kMarchWaves - 1) / kMarchWaves, 1, groups), blk, 0, st, a, T, (int)L,
                               (int)F_X, (int)F_TMP, fcoarse, alpha, p.mask, th, tiles, (int)S);
        };
        if (L == maxl)
            march_form(a, [&](auto k_tag, auto v_tag, auto cb_tag) { go(IntC<1>{}, k_tag, v_tag, cb_tag); });
        else
            march_form(a, [&](auto k_tag, auto v_tag, auto cb_tag) { go(IntC<0>{}, k_tag, v_tag, cb_tag); });
    };
    for (uint64_t L = minl + 1; L <= maxl; ++L)
    {
        if (btop && L <= (uint64_t)btop)
            continue;
        const LevelArgs a = largs(L);
        const int Nf = (int)h.lv[L].side;
        const int Nc = (int)h.lv[L - 1].side;
        const dim3 pg(grid_for((uint64_t)Nc, kBlock), (unsigned)Nf, S);
        // the coarse level's iterate: the coarse solve's F_X, or F_TMP
        // after that level's one-pass post-smoothing
        const int fcoarse = (post2 && L - 1 > minl) ? F_TMP : F_X;
        if constexpr (kBands<MK>)
        {
            if (pre2r)
            {
                // prolongation, correction and post-smoothing in one pass
                post2_launch(L, a, fcoarse, p.adapt, IntC<1>{});
                continue;
            }
        }
        if (h.prolmat)
        {
            // c = P x_coarse, then x += alpha c
            hipLaunchKernelGGL(v_apply_ell_kernel, dim3(grid_for(h.lv[L].prol.rows, kBlock), 1, S), blk, 0, st, h.lv[L].prol, T,
                               (int)(L - 1), fcoarse, (int)L, (int)F_C);
            if (p.adapt != 0.0f)
                hipLaunchKernelGGL(v_axpy_const_kernel, dim3(grid_for(a.n, kBlock), 1, S), blk, 0, st, T, (int)L, a.n,
                                   p.adapt);
        }
        else if (p.adapt != 0.0f)
            hipLaunchKernelGGL((v_prolong_kernel<true>), pg, blk, 0, st, T, (int)L, Nf, p.adapt, p.mask, (int)F_X,
                               fcoarse);
        else
            hipLaunchKernelGGL((v_prolong_kernel<false>), pg, blk, 0, st, T, (int)L, Nf, 0.0f, p.mask, (int)F_C,
                               fcoarse);
        if (p.adapt == 0.0f)
        {
            const unsigned ab = std::min<unsigned>(grid_for(a.n, kBlock), kNormBlocks);
            hipLaunchKernelGGL((v_adapt_alpha_kernel<MK>), dim3(ab, 1, S), blk, 0, st, a, T, (int)L);
            hipLaunchKernelGGL(v_adapt_alpha_finish_kernel, dim3(1, 1, S), blk, 0, st, T, ab);
            hipLaunchKernelGGL(v_axpy_alpha_kernel, dim3(grid_for(a.n, kBlock), 1, S), blk, 0, st, T, (int)L, a.n);
        }
        // post-smoothing: n_pre_smooth sweeps (multigrid.hh:1851)
        if constexpr (kBands<MK>)
        {
            if (post2)
            {
                post2_launch(L, a, fcoarse, 0.0f, IntC<0>{});
                continue;
            }
        }
        int xc = F_X, xa = F_TMP;
        sweeps(L, xc, xa, F_RHS, npre);
        if (xc != F_X)
            move(L, xc, F_X, false);
        if (L == maxl)
            defect(L);
    }
    if (fold)
        hipLaunchKernelGGL((inner_end_kernel<true>), dim3(1, 1, S), dim3(1024), 0, st, T, (int)maxl, n, cycle_tiles,
                           open_blocks, p.tolerance, p.n_max_iter);
    else if (post2)
        hipLaunchKernelGGL((inner_end_kernel<false>), dim3(1, 1, S), dim3(1024), 0, st, T, (int)maxl, n, cycle_tiles, 0u,
                           p.tolerance, p.n_max_iter);
    else
    {
        hipLaunchKernelGGL((inner_norm_kernel<1>), norm_grid(top.n), blk, 0, st, T, (int)maxl, n);
        hipLaunchKernelGGL((inner_norm_finish_kernel<1>), dim3(1, 1, S), blk, 0, st, T, norm_grid(top.n).x,
                           p.tolerance, p.convergence_check, p.n_max_iter);
    }
    HIP_CHECK(hipGetLastError());
}
}  // namespace

void enqueue_tick(const Hierarchy & h, uint64_t maxl, const Slot * T, unsigned S, hipStream_t st)
{
    enqueue_tick_part(h, maxl, T, S, kTickOpen | kTickCycle, st);
}

void enqueue_tick_part(const Hierarchy & h, uint64_t maxl, const Slot * T, unsigned S, unsigned part, hipStream_t st)
{
    if (h.kind == 1)
        tick_impl<1>(h, maxl, T, S, part, st);
    else if (h.kind == 2)
        tick_impl<2>(h, maxl, T, S, part, st);
    else
        tick_impl<0>(h, maxl, T, S, part, st);
}

}  // namespace mg
}  // namespace hsolve
