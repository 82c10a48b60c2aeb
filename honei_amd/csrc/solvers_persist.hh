// solvers_persist.hh -- CG, CGSolver<VAR> and ConjugateGradients<JAC> on small
// systems in one launch.  Included by solvers.hip.
//
// Systems whose vectors stay in cache are bound by latency: three to five
// launches per iteration, each a few dependent memory round trips.  Measured
// per iteration by launches and here, FP64: CG 65^2 14.4 and 5.9 us, 257^2 13.4
// and 6.7, 513^2 23.1 and 8.8, 724^2 32.1 and 13.1; Jacobi-PCG on ELL 257^2 14.9
// and 7.1 us, 513^2 27.8 and 10.2, 700^2 36.7 and 17.3.  (Above 524,288 rows a
// thread's rows no longer fit its registers and LDS.)  One workgroup per CU
// keeps its rows' matrix entries, x, r and the direction (at the row and
// at its columns) in registers for the whole solve.  What crosses
// workgroups is the new residual (or preconditioned residual) z and two sets
// of block partials per iteration, written and read past the caches that the
// XCDs do not share (device-scope accesses).
//
// Every workgroup forms the next direction at its rows' columns itself, with
// the launch path's operations, so each iteration waits twice: for all
// partials of v.p, and for all partials of r.r (and r.z), behind which the z
// values are known to be in place.  A partial doubles as its own flag: its
// place holds kNoSum, a NaN that no sum is stored as, until it is written.
//
// The partials are those of the launch path (one per 256 rows, wave by wave)
// and each workgroup adds them in its order, so iterates, counts and defects
// are the same bits.
//
// Waits are bounded: a workgroup that has polled kSpins times gives up, and
// the host then solves by launches; results go to buffers of the solve's own
// until every workgroup has finished.  A poll takes about 0.12 us, so a wait ends
// after 10 ms: several times what other streams' kernels hold a CU for and of the
// order of one solve (a bound in polls, not by the clock: time in which the
// process is switched off the device does not count, and no register is spent; a
// bound of 16 bits shortens the loop's code by four bytes, which moved it within
// the fetch lines and made 513^2 Jacobi-PCG 5% slower).  After a solve that gave
// up, the device's next kPersistPause go by launches at once: where the CUs stay
// taken, giving up costs each a third of a millisecond.
//
// The launch is an ordinary one, of at most one workgroup per CU (checked to
// fit), on streams without a CU mask, so that all of them are resident as soon
// as other streams' kernels leave room.  Solves of several threads run side by
// side while there is a CU for each of their workgroups (PersistHold), with more
// rows a thread if need be; one that finds too few CUs goes by launches (measured,
// four threads solving 257^2 by CG: 2.05 ms a solve, one after another 3.5).  A
// cooperative launch promises the same, but the queue that the runtime opens for
// it stays: streams of the process that run side by side afterwards (the request
// server's) took 10.7 ms instead of 8.5 ms for 48 mixed requests.
#pragma once

    constexpr int kPersistThreads = 512;                      // two blocks of 256 rows side by side
    constexpr uint64_t kNoSum = 0x7ff8dead0000beefull;
    constexpr int kSpins = 80000;                             // polls after which a wait is given up
    constexpr int kPersistPause = 32;                         // solves by launches after one that gave up
    constexpr uint64_t kPersistIters = 1 << 14;               // iterations per launch at most

    // The launch of the calling thread's solves that is made to give up
    // (hsolve_krylov_give_up) and how its last solve ran (hsolve_krylov_path).
    inline uint64_t & persist_fail()
    {
        static thread_local uint64_t launch = ~(uint64_t)0;
        return launch;
    }
    enum PersistPath : int
    {
        PP_LAUNCHES = 0,
        PP_ONE = 1,
        PP_GAVE_UP = 2
    };
    inline int & persist_path()
    {
        static thread_local int path = PP_LAUNCHES;
        return path;
    }

    enum PersistKind : int
    {
        PK_NONE = 0,
        PK_VAR = 1,
        PK_JAC = 2
    };

    // The matrix as the kernel loads it once: Q1 bands, or an ELL handle with
    // one lane per row.
    struct PersistMatrix
    {
        k::Bands B;
        int64_t m;
        const void *Aj, *Ax, *Arl;
        int idx_kind, len_bytes;
        uint64_t stride;
    };

    template <typename DT> struct PersistArgs
    {
        PersistMatrix A;
        const DT * x;          // iterate at the launch's start
        DT * xo;               // and at its end
        DT *r, *p, *z;         // residual and direction (in and out), published z
        const DT * P;          // VAR / JAC: the diagonal
        int64_t n;
        unsigned nb;           // blocks of 256 rows
        uint64_t * sums;       // kPersistSums, then the give-up flag
        CgScalars<DT> * s;
        int resume;            // the launch continues a solve (z and talpha are the last update's)
    };

    __global__ __launch_bounds__(256) void persist_clear_kernel(uint64_t * sums)
    {
        const unsigned i = blockIdx.x * 256 + threadIdx.x;
        if (i < kPersistSums)
            sums[i] = kNoSum;
        else if (i < kPersistSums + kPersistFlags)
            sums[i] = 0;
    }

    // The iterate of a solve that has ended, and in which no workgroup gave up,
    // to the caller's array.
    template <typename DT>
    __global__ __launch_bounds__(256) void persist_copy_kernel(const DT * __restrict__ from, DT * __restrict__ to,
            int64_t n, const uint64_t * sums, const CgScalars<DT> * s)
    {
        if (s->run != 0 || sums[kPersistSums] != 0)
            return;
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
            to[i] = from[i];
    }

    template <typename T> __device__ __forceinline__ T load_device(const T * p)
    {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    template <typename T> __device__ __forceinline__ void store_device(T * p, T v)
    {
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // the entry at byte offset `at` of a vector: a wave-uniform base and a
    // 32-bit offset per lane (kept as such; 64-bit addresses of every column
    // would take twice the registers)
    template <typename T> __device__ __forceinline__ T load_at(const T * p, uint32_t at)
    {
        return *(gptr<const T>)((gptr<const char>)as_global(p) + at);
    }
    template <typename T> __device__ __forceinline__ T load_device_at(const T * p, uint32_t at)
    {
        return __hip_atomic_load((gptr<const T>)((gptr<const char>)as_global(p) + at), __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
    }
    template <typename T> __device__ __forceinline__ void store_device_at(T * p, uint32_t at, T v)
    {
        __hip_atomic_store((gptr<T>)((gptr<char>)as_global(p) + at), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // this wave's stores have reached the point where other XCDs read them
    __device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

    // Row i: its entries a[k] at byte offsets c[k] of their columns, in
    // summation order, `valid` those that count.  Q1: q1_row's order, the
    // diagonal first.
    template <typename DT, bool Q1, int K>
    __device__ __forceinline__ void persist_row(const PersistMatrix & A, int64_t n, int64_t i, DT (&a)[K],
                                                uint32_t (&c)[K], uint32_t & valid)
    {
        if constexpr (Q1)
        {
            static_assert(K == 9, "nine bands");
            const int band[9] = {4, 0, 1, 2, 3, 5, 6, 7, 8};
            const int64_t m = A.m;
            const int64_t off[9] = {0, -m - 1, -m, -m + 1, -1, 1, m - 1, m, m + 1};
            valid = 0;
#pragma unroll
            for (int k = 0; k < 9; ++k)
            {
                const int64_t j = i + off[k];
                const bool in = j >= 0 && j < n;
                valid |= (in ? 1u : 0u) << k;
                c[k] = (uint32_t)(in ? j : i) * (uint32_t)sizeof(DT);
                a[k] = ((const DT *)A.B.b[band[k]])[i];
            }
        }
        else
        {
            const uint32_t len = A.len_bytes == 1   ? ((const uint8_t *)A.Arl)[i]
                                 : A.len_bytes == 2 ? ((const uint16_t *)A.Arl)[i]
                                                    : ((const uint32_t *)A.Arl)[i];
            valid = (1u << len) - 1u;
#pragma unroll
            for (int k = 0; k < K; ++k)
            {
                c[k] = (uint32_t)i;
                a[k] = DT(0);
                if ((uint32_t)k < len)
                {
                    const uint64_t at = (uint64_t)k * A.stride + (uint64_t)i;
                    a[k] = ((const DT *)A.Ax)[at];
                    c[k] = A.idx_kind == 1 ? (uint32_t)(i + (int64_t)((const int16_t *)A.Aj)[at])
                                           : ((const uint32_t *)A.Aj)[at];
                }
                c[k] *= (uint32_t)sizeof(DT);
            }
        }
    }

    // The matrix entries of three or more FP64 rows a thread (two of sixteen
    // entries) go to LDS, lane by lane: with them the rest stays in registers
    // (513^2 Jacobi-PCG: 10.3 us an iteration, 12.8 with spills).
    template <typename DT, int K, int RPT> constexpr bool kEntriesInLds = sizeof(DT) * K * RPT >= 27 * sizeof(double);

    // RPT rows per thread: block (of 256 rows) w 2 RPT + 2 q + (thread / 256)
    // is row slot q of workgroup w.
    template <typename DT, int KIND, bool Q1, int K, int RPT>
    __global__ __launch_bounds__(kPersistThreads) void persist_cg_kernel(PersistArgs<DT> ar)
    {
        constexpr int NV = KIND == PK_NONE ? 1 : 2;     // partials after an update
        constexpr int W = kPersistThreads / 64;
        __shared__ double part[2][2][RPT][W];           // [phase][value][row slot][wave]
        __shared__ double tot[2][2][4];                 // [phase][value][wave]
        __shared__ int gave_up;
        const int tid = threadIdx.x, wave = tid >> 6, half = tid >> 8;
        const unsigned nb = ar.nb, blk0 = blockIdx.x * 2 * RPT;
        const int64_t n = ar.n;
        if (tid == 0)
            gave_up = 0;

        constexpr bool AL = kEntriesInLds<DT, K, RPT>;
        extern __shared__ __align__(16) unsigned char dyn[];
        DT * al = reinterpret_cast<DT *>(dyn) + tid;      // entry k of row slot q at (q K + k) kPersistThreads
        DT a[AL ? 1 : RPT][K], pn[RPT][K], x[RPT], r[RPT], po[RPT], P[RPT];
        uint32_t c[RPT][K], valid[RPT];
        uint32_t row[RPT];          // byte offset of the thread's rows
        bool on[RPT];
        const bool resume = ar.resume != 0;
#pragma unroll
        for (int q = 0; q < RPT; ++q)
        {
            const int64_t i = (int64_t)(blk0 + 2 * q + half) * 256 + (tid & 255);
            on[q] = i < n;
            const int64_t j = on[q] ? i : n - 1;
            row[q] = (uint32_t)j * (uint32_t)sizeof(DT);
            persist_row<DT, Q1, K>(ar.A, n, j, a[AL ? 0 : q], c[q], valid[q]);
            if (AL)
#pragma unroll
                for (int k = 0; k < K; ++k)
                    al[(q * K + k) * kPersistThreads] = a[0][k];
            x[q] = ar.x[j];
            r[q] = ar.r[j];
            po[q] = ar.p[j];
            P[q] = KIND == PK_NONE ? DT(0) : ar.P[j];
#pragma unroll
            for (int k = 0; k < K; ++k)
                pn[q][k] = load_at(ar.p, c[q][k]);
        }
        CgScalars<DT> s = *ar.s;
        uint64_t left = kPersistIters;
        unsigned turn = 0;
        __syncthreads();

        // Block partials of the lanes' values: wave sums to LDS, then one
        // thread per block adds its four waves in order and publishes them.
        // On return a, b are the totals over all blocks (sum_partials2's
        // order); false: a wait was given up.
        auto all_sum = [&](auto nv_tag, int phase, double (&va)[RPT], double (&vb)[RPT], double & ta, double & tb) {
            constexpr int N = decltype(nv_tag)::value;
            uint64_t * set = ar.sums + (turn % 3) * 2 * kSolverBlocks;
            uint64_t * old = ar.sums + ((turn + 2) % 3) * 2 * kSolverBlocks;
            ++turn;
#pragma unroll
            for (int q = 0; q < RPT; ++q)
            {
                const double wa = k::wave_sum(va[q]);
                const double wb = N > 1 ? k::wave_sum(vb[q]) : 0.0;
                if ((tid & 63) == 0)
                {
                    part[phase][0][q][wave] = wa;
                    if (N > 1)
                        part[phase][1][q][wave] = wb;
                }
            }
            stores_done();      // the wave's z, and a cleared place, before the partials
            __syncthreads();
            if (tid < 2 * RPT * N)
            {
                const int v = tid / (2 * RPT), l = tid % (2 * RPT), h = l & 1, q = l >> 1;
                const unsigned blk = blk0 + l;
                if (blk < nb)
                {
                    double t = 0.0;
#pragma unroll
                    for (int w = 0; w < 4; ++w)
                        t += part[phase][v][q][4 * h + w];
                    const uint64_t bits = t != t ? 0x7ff8000000000000ull : (uint64_t)__double_as_longlong(t);
                    store_device(set + v * kSolverBlocks + blk, bits);
                }
            }
            if (tid < 256)
            {
                // places tid, tid + 256, ...: every load of a round is in
                // flight before the first is looked at
                constexpr int S = 2 * RPT;     // (at most 256 workgroups' blocks)
                uint64_t got[N][S];
                int spin = 0;
                bool missing = true;
                while (missing && spin <= kSpins)
                {
#pragma unroll
                    for (int u = 0; u < S; ++u)
                    {
                        const unsigned i = (unsigned)tid + 256 * u;
#pragma unroll
                        for (int v = 0; v < N; ++v)
                            got[v][u] = load_device(set + v * kSolverBlocks + (i < nb ? i : 0));
                    }
                    missing = false;
#pragma unroll
                    for (int u = 0; u < S; ++u)
#pragma unroll
                        for (int v = 0; v < N; ++v)
                            missing = missing || got[v][u] == kNoSum;
                    ++spin;
                }
                const bool bad = missing;
                double sa = 0.0, sb = 0.0;
#pragma unroll
                for (int u = 0; u < S; ++u)
                    if ((unsigned)tid + 256 * u < nb)
                    {
                        sa += __longlong_as_double((long long)got[0][u]);
                        if (N > 1)
                            sb += __longlong_as_double((long long)got[N - 1][u]);
                    }
                if (bad)
                    gave_up = 1;
                sa = k::wave_sum(sa);
                if (N > 1)
                    sb = k::wave_sum(sb);
                if ((tid & 63) == 0)
                {
                    tot[phase][0][wave] = sa;
                    tot[phase][1][wave] = sb;
                }
            }
            __syncthreads();
            ta = tb = 0.0;
#pragma unroll
            for (int w = 0; w < 4; ++w)
            {
                ta += tot[phase][0][w];
                if (N > 1)
                    tb += tot[phase][1][w];
            }
            // every workgroup is past the set before this one
            if (tid < 2 * RPT && blk0 + tid < nb)
            {
                store_device(old + blk0 + tid, kNoSum);
                store_device(old + kSolverBlocks + blk0 + tid, kNoSum);
            }
            return gave_up == 0;
        };

        bool direction = resume;     // the next direction is still to be formed
        bool ok = true;
        while (s.run && left != 0)
        {
            --left;
            if (direction)
            {
#pragma unroll
                for (int q = 0; q < RPT; ++q)
                {
                    DT zn[K];
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        zn[k] = load_device_at(ar.z, c[q][k]);
                    const DT zo = KIND == PK_NONE ? r[q] : P[q] * r[q];
                    const DT t = po[q] * s.talpha;
                    po[q] = t + zo;
#pragma unroll
                    for (int k = 0; k < K; ++k)
                    {
                        const DT u = pn[q][k] * s.talpha;
                        pn[q][k] = u + zn[k];
                    }
                }
            }
            direction = true;
            DT v[RPT];
            double va[RPT], vb[RPT], ta, tb;
#pragma unroll
            for (int q = 0; q < RPT; ++q)
            {
                auto entry = [&](int k) { return AL ? al[(q * K + k) * kPersistThreads] : a[AL ? 0 : q][k]; };
                DT sum = Q1 ? entry(0) * pn[q][0] : DT(0);
#pragma unroll
                for (int k = Q1 ? 1 : 0; k < K; ++k)
                {
                    const DT t = sum + entry(k) * pn[q][k];
                    sum = ((valid[q] >> k) & 1u) ? t : sum;
                }
                v[q] = sum;
                va[q] = on[q] ? (double)sum * (double)po[q] : 0.0;
                vb[q] = 0.0;
            }
            if (! (ok = all_sum(std::integral_constant<int, 1>{}, 0, va, vb, ta, tb)))
                break;
            DT lambda;
            if (KIND == PK_JAC)
                lambda = div_guard<DT>(s.temp, (DT)ta);
            else
            {
                const DT temp = (DT)ta;
                if (KIND == PK_VAR)
                    lambda = s.alpha_new / guard_signed<DT>(temp);
                else
                    lambda = s.alpha / (s.plain ? temp : guard<DT>(temp));
                s.temp = temp;
                s.lambda = lambda;
            }
            const DT mlambda = -lambda;
#pragma unroll
            for (int q = 0; q < RPT; ++q)
            {
                x[q] = x[q] + lambda * po[q];
                const DT ri = r[q] + mlambda * v[q];
                r[q] = ri;
                const DT zi = KIND == PK_NONE ? ri : P[q] * ri;
                if (on[q])
                    store_device_at(ar.z, row[q], zi);
                const double rr = on[q] ? (double)ri * (double)ri : 0.0;
                const double rz = on[q] ? (double)ri * (double)zi : 0.0;
                va[q] = rr;
                vb[q] = rz;
            }
            if (! (ok = all_sum(std::integral_constant<int, NV>{}, 1, va, vb, ta, tb)))
                break;
            if (KIND == PK_JAC)
                jac_test<DT>(s, tb, ta);
            else
                cg_test<DT, KIND == PK_VAR>(s, ta, tb);
        }
        if (! ok)
        {
            if (tid == 0)
                store_device((unsigned long long *)(ar.sums + kPersistSums), 1ull);
            return;
        }
#pragma unroll
        for (int q = 0; q < RPT; ++q)
            if (on[q])
            {
                const uint32_t j = row[q] / (uint32_t)sizeof(DT);
                ar.xo[j] = x[q];
                ar.r[j] = r[q];
                ar.p[j] = po[q];
            }
        if (blockIdx.x == 0 && tid == 0)
            *ar.s = s;
    }

    // Rows per thread and workgroups for nb blocks: the fewest rows a thread
    // with which one workgroup per CU covers the system; 0: none does.
    inline int persist_rows_per_thread(unsigned nb, unsigned cus)
    {
        const unsigned w = std::min(cus, 256u);     // (a thread collects the places of at most 256 workgroups)
        for (int rpt = 1; rpt <= 4; ++rpt)
            if ((uint64_t)w * 2 * rpt >= nb)
                return rpt;
        return 0;
    }

    struct PersistKernel
    {
        const void * fn = nullptr;
        size_t lds = 0;            // dynamic LDS
    };
    template <typename DT, int KIND, bool Q1, int K, int RPT> PersistKernel persist_pick()
    {
        PersistKernel p;
        p.fn = (const void *)persist_cg_kernel<DT, KIND, Q1, K, RPT>;
        if (kEntriesInLds<DT, K, RPT>)
            p.lds = sizeof(DT) * K * RPT * kPersistThreads;
        return p;
    }

    // The kernel for a matrix (fn null: none).  Longer rows take more
    // registers: up to nine entries with four rows a thread, up to sixteen
    // with two.
    template <typename DT, int KIND> PersistKernel persist_kernel(bool q1, uint64_t width, int rpt)
    {
#define HS_P(Q, K, R) persist_pick<DT, KIND, Q, K, R>()
        if (q1)
        {
            if constexpr (KIND == PK_NONE)
                return rpt == 1 ? HS_P(true, 9, 1) : rpt == 2 ? HS_P(true, 9, 2) : rpt == 3 ? HS_P(true, 9, 3) : HS_P(true, 9, 4);
            return PersistKernel();
        }
        if (width <= 9)
            return rpt == 1 ? HS_P(false, 9, 1) : rpt == 2 ? HS_P(false, 9, 2) : rpt == 3 ? HS_P(false, 9, 3) : HS_P(false, 9, 4);
        if (width <= 16)
            return rpt == 1 ? HS_P(false, 16, 1) : (rpt == 2 ? HS_P(false, 16, 2) : PersistKernel());
#undef HS_P
        return PersistKernel();
    }

    // What one-launch solves keep per device.
    struct PersistDevice
    {
        unsigned cus = 0;              // compute units
        std::atomic<unsigned> held{0}; // workgroups per shader engine of the solves that run
        std::atomic<int> pause{0};     // solves still to go by launches after one that gave up
        std::mutex mu;
        std::map<const void *, bool> fits;
        // whether a workgroup of kernel k fits a CU (looked up once)
        bool fit(const PersistKernel & k)
        {
            std::lock_guard<std::mutex> lock(mu);
            auto it = fits.find(k.fn);
            if (it != fits.end())
                return it->second;
            int n = 0;
            const bool ok =
                (k.lds == 0 || hipFuncSetAttribute(k.fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)k.lds) ==
                                   hipSuccess) &&
                hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k.fn, kPersistThreads, k.lds) == hipSuccess && n > 0;
            if (! ok)
                (void)hipGetLastError();
            fits.emplace(k.fn, ok);
            return ok;
        }
        bool paused()
        {
            int p = pause.load();
            while (p > 0)
                if (pause.compare_exchange_weak(p, p - 1))
                    return true;
            return false;
        }
    };
    // of the current device (null: beyond kMaxDevices)
    inline PersistDevice * persist_device()
    {
        static std::mutex mu;
        static PersistDevice devices[kMaxDevices];
        int dev = 0;
        HIP_CHECK(hipGetDevice(&dev));
        if (dev < 0 || dev >= kMaxDevices)
            return nullptr;
        PersistDevice & d = devices[dev];
        std::lock_guard<std::mutex> lock(mu);
        if (d.cus == 0)
        {
            int cu = 0;
            HIP_CHECK(hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev));
            d.cus = (unsigned)cu;
        }
        return &d;
    }

    // A solve's workgroups among the device's CUs.  Consecutive workgroups go to
    // its 32 shader engines in turn (8 XCDs of 4), so the CUs are counted in each.
    constexpr unsigned kEngines = 32;
    struct PersistHold
    {
        PersistDevice & d;
        unsigned share = 0;
        explicit PersistHold(PersistDevice & dev) : d(dev) {}
        bool take(unsigned workgroups)
        {
            const unsigned want = (workgroups + kEngines - 1) / kEngines;
            unsigned h = d.held.load();
            while (h + want <= d.cus / kEngines)
                if (d.held.compare_exchange_weak(h, h + want))
                {
                    share = want;
                    return true;
                }
            return false;
        }
        ~PersistHold() { d.held -= share; }
        PersistHold(const PersistHold &) = delete;
    };

    // Whether stream st may use every compute unit of the current device (of
    // cus): a stream or a process with a CU mask cannot hold the grid at once.
    inline bool persist_whole_device(hipStream_t st, unsigned cus)
    {
        constexpr unsigned W = 64;
        uint32_t mask[W] = {};
        if (cus > 32 * W || hipExtStreamGetCUMask(st, W, mask) != hipSuccess)
        {
            (void)hipGetLastError();
            return false;
        }
        unsigned on = 0;
        for (unsigned w = 0; w < W; ++w)
            on += (unsigned)__builtin_popcount(mask[w]);
        return on >= cus;
    }

    enum PersistEnd : int
    {
        PE_NOT = 0,      // the system does not qualify: nothing was touched
        PE_DONE = 1,     // *h holds the final scalars, x the iterate
        PE_GAVE_UP = 2   // x is untouched, the workspace is not
    };

    // The iterations of a solve whose init kernel has run (w.r, w.p, *w.s).
    template <typename DT, int KIND, typename Work>
    PersistEnd run_persist(const PersistMatrix & A, bool q1, uint64_t width, const Work & w, DT * x, const DT * P, uint64_t n,
                     CgScalars<DT> * h, hipStream_t st)
    {
        // (one iteration by launches is over before the one launch has read its
        // rows: 129^2 Jacobi-PCG 44 us against 51, three iterations 82 against 64)
        if (n > kPersistRows || w.sums == nullptr || h->max_iters < 2)
            return PE_NOT;
        PersistDevice * const dev = persist_device();
        if (! dev)
            return PE_NOT;
        const unsigned nb = grid_for(n, 256);
        if (! persist_whole_device(st, dev->cus) || dev->paused())
            return PE_NOT;
        // the fewest rows a thread, or more of them where other solves have
        // left fewer CUs
        PersistHold hold(*dev);
        PersistKernel kern;
        dim3 grid(0);
        for (int rpt = persist_rows_per_thread(nb, dev->cus); rpt != 0 && rpt <= 4 && hold.share == 0; ++rpt)
        {
            kern = persist_kernel<DT, KIND>(q1, width, rpt);
            grid.x = grid_for(nb, 2 * rpt);
            if (! kern.fn || ! dev->fit(kern) || ! hold.take(grid.x))
                kern.fn = nullptr;
        }
        if (! kern.fn)
            return PE_NOT;
        hipLaunchKernelGGL(persist_clear_kernel, dim3(grid_for(kPersistSums + kPersistFlags, 256)), dim3(256), 0, st, w.sums);
        PersistArgs<DT> ar{A, x, w.p2, w.r, w.p, w.v, P, (int64_t)n, nb, w.sums, w.s, 0};
        for (uint64_t launch = 0;; ++launch)
        {
            // (the launch that is made to give up lacks a workgroup)
            const unsigned present = launch == persist_fail() && grid.x > 1 ? grid.x - 1 : grid.x;
            void * args[] = {&ar};
            if (hipLaunchKernel(kern.fn, dim3(present), dim3(kPersistThreads), args, kern.lds, st) != hipSuccess)
            {
                (void)hipGetLastError();
                return PE_GAVE_UP;
            }
            hipLaunchKernelGGL((persist_copy_kernel<DT>), dim3(std::min<unsigned>(grid_for(n, 1024), 256)), dim3(256), 0,
                               st, (const DT *)w.p2, x, (int64_t)n, (const uint64_t *)w.sums, (const CgScalars<DT> *)w.s);
            // the give-up flag and the scalars behind it (after a wait of its own:
            // a copy to host memory right behind the kernels took up to 4 ms for a
            // solve on arrays that were new)
            struct
            {
                uint64_t gave_up[kPersistFlags];
                CgScalars<DT> s;
            } end;
            static_assert(sizeof(end) == sizeof(end.gave_up) + sizeof(end.s), "laid out as CgWork lays them out");
            HIP_CHECK(hipStreamSynchronize(st));
            HIP_CHECK(hipMemcpyAsync(&end, w.sums + kPersistSums, sizeof(end), hipMemcpyDeviceToHost, st));
            HIP_CHECK(hipStreamSynchronize(st));
            if (end.gave_up[0])
            {
                dev->pause = kPersistPause;
                return PE_GAVE_UP;
            }
            *h = end.s;
            if (h->run == 0)
                return PE_DONE;
            hipLaunchKernelGGL(persist_clear_kernel, dim3(grid_for(kPersistSums + kPersistFlags, 256)), dim3(256), 0, st,
                               w.sums);
            ar.x = w.p2;
            ar.resume = 1;
        }
    }
