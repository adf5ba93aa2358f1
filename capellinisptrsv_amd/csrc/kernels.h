// Device kernels of the gfx950 sync-free lower-triangular solve.
//
// Execution model shared by every solve kernel:
//  * Work is handed out by an atomic ticket, one atomicAdd per workgroup
//    (CUDA/ourWrtFst/spts_syncfree_cuda_csr_wrt.h:24 takes one per thread; a
//    single counter serialises at ~11 ns per increment on MI355X, so per-thread
//    or per-wavefront tickets alone would cost 0.1-0.4 ms on 2M rows).  The
//    grid is persistent: a workgroup takes tickets until the rows run out.
//    Tickets are only taken by running workgroups, so every row a workgroup
//    waits for belongs to a workgroup that is running or finished; that is
//    what makes spinning safe without a grid barrier.
//  * Readiness of x[c] is observed either through the value itself (SYNC
//    VALUE: the readiness array -- x, or a staged copy in uncached memory --
//    starts as a signalling-NaN sentinel that arithmetic can never produce; a
//    relaxed agent-scope 32/64-bit atomic load both tests and fetches it) or
//    through an int flag per row holding the solve's epoch (SYNC FLAG: the
//    value is published with a returning agent-scope exchange and the flag
//    store depends on it; readers load the value with an agent-scope atomic
//    after seeing the flag -- no cache-wide release/acquire fences; the
//    epoch makes resets between solves unnecessary).
//  * Thread-per-row kernels use the write-first loop of
//    spts_syncfree_cuda_csr_wrt.h:37-55: a lane publishes x[i] from inside the
//    loop in which it polls, so lanes of one wavefront that depend on each
//    other always make progress.  Each lane polls a small window of its next
//    dependencies at once (two in the value protocol, kWin with flags) and
//    consumes the ready prefix in stored order, so the accumulation order is
//    the sequential one (bit-exact against the oracle's fused forward
//    substitution).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "device_base.h"

namespace cap {

constexpr int kBlockSmall = 128;  // the thread-per-row kernels' other workgroup size
// Thread-per-row workgroups of several right-hand sides (value protocol, no
// LDS window): a ticket covers BLOCK / lanes-per-row rows, and each ticket
// is one atomic on the one ticket counter, which serializes at about 12 ns
// an atomic; 16 right-hand sides give 16 rows a ticket at 256 threads.
constexpr int kBlockLarge = 1024;
constexpr int kWin = 4;      // dependencies polled concurrently per lane (flag protocol)


template <typename U>
__device__ __forceinline__ U ld_agent(const U *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ __forceinline__ void st_agent(U *p, U v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// hardware FP / int atomic add at agent scope (global_atomic_add_f64 / _f32)
template <typename V>
__device__ __forceinline__ void atomic_add_agent(V *p, V v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Readiness protocol state shared by the solve kernels.
//  flags/epoch: SYNC FLAG only.  spin_limit / wait_ticks: polls without
//  progress / wall time without progress after which a lane gives up,
//  publishes NaN (so every dependent row, and with it the whole grid, still
//  finishes) and sets bit 0 of *err; <= 0 = no bound of that kind.
//  ready: SYNC VALUE only -- the array that is polled and published (same
//  shape as x, sentinel-filled before the solve); results are also stored
//  into x with plain stores.  nullptr = x itself is polled.  The library
//  places it in uncached device memory, where a poll goes straight to the
//  memory side instead of through an L2 that agent-scope loads must miss.
//  unfused: accumulate s + v*x as a rounded product and a rounded sum (the
//  arithmetic of the reference's serial executor,
//  openCL/SynFree_csc/sptrsv_syncfree_serialref.h:67-68, compiled without
//  contraction) instead of one fused multiply-add.
struct SyncCtx {
    int *flags;
    int epoch;
    int spin_limit;
    int *err;
    void *ready;
    int unfused;
    int wait_ticks;  // wall-time bound of one wait, in 10 ns ticks (<= 0: none)
    // kPollCounters counters of the polls the value-protocol write-first
    // solve issued (its counting instantiation only; nullptr otherwise)
    unsigned long long *polls;
};
constexpr int kPollCounters = 64;

// One accumulation step of a row's sum, in the plan's arithmetic.  The
// operand order and the stored-order chain are the same in both forms; only
// the rounding of the product differs.
template <typename T>
__device__ __forceinline__ T acc(const SyncCtx &sc, T v, T x, T s)
{
    return sc.unfused ? s + v * x : fmac(v, x, s);
}

template <typename T>
__device__ __forceinline__ typename VBits<T>::U *ready_array(const SyncCtx &sc, T *x)
{
    typedef typename VBits<T>::U U;
    return sc.ready ? reinterpret_cast<U *>(sc.ready) : reinterpret_cast<U *>(x);
}
template <typename T>
__device__ __forceinline__ const typename VBits<T>::U *ready_array(const SyncCtx &sc, const T *x)
{
    typedef typename VBits<T>::U U;
    return sc.ready ? reinterpret_cast<const U *>(sc.ready) : reinterpret_cast<const U *>(x);
}

// Watchdog state of one wait: polls since the last progress and the
// real-time counter (100 MHz, s_memrealtime) read at the kWatchCheck-th of
// them.  A wait gives up after sc.spin_limit polls (when > 0) or once
// sc.wait_ticks of wall time have passed since that read (when > 0), so a
// kernel drains in bounded wall time however long each poll takes under
// memory contention.  The counter is read once every kWatchCheck polls.
constexpr unsigned kWatchCheck = 1024;
struct Idle {
    unsigned n = 0, t0 = 0;
    __device__ __forceinline__ void progress() { n = 0; }
};
__device__ __forceinline__ bool expired(const SyncCtx &sc, Idle &w)
{
    ++w.n;
    if (sc.spin_limit > 0 && w.n > (unsigned)sc.spin_limit) return true;
    if ((w.n & (kWatchCheck - 1)) != 0 || sc.wait_ticks <= 0) return false;
    const unsigned now = (unsigned)__builtin_amdgcn_s_memrealtime();
    if (w.n == kWatchCheck) {
        w.t0 = now;
        return false;
    }
    return now - w.t0 > (unsigned)sc.wait_ticks;
}
__device__ __forceinline__ bool give_up(const SyncCtx &sc, Idle &w)
{
    if (!expired(sc, w)) return false;
    atomicOr(sc.err, 1);
    return true;
}

// Persistent ticket loop: the workgroup takes `per_block` work items at a time
// (one atomicAdd, broadcast through LDS), runs init(base) on every thread
// between two barriers (all threads have left the previous body), then
// body(base), until `total` items are handed out.  body must not contain
// workgroup barriers.
template <typename FI, typename F>
__device__ __forceinline__ void ticket_loop(unsigned *ticket, int per_block, int total, FI init, F body)
{
    __shared__ int s_base;
    while (true) {
        if (threadIdx.x == 0) s_base = (int)atomicAdd(ticket, (unsigned)per_block);
        __syncthreads();
        const int base = s_base;
        init(base);
        __syncthreads();
        if (base >= total) return;
        body(base);
    }
}
template <typename F>
__device__ __forceinline__ void ticket_loop(unsigned *ticket, int per_block, int total, F body)
{
    ticket_loop(ticket, per_block, total, [](int) {}, body);
}

// Workgroup-local readiness window: values of the rows [lo, lo + len) the
// workgroup is solving, kept in LDS next to their global copies.  A
// dependency inside the window is polled in LDS (one CU, no memory traffic);
// older rows are polled in global memory.  len == 0 disables it.
template <typename U>
struct LdsWin {
    U *s;
    int lo, len, k;
    __device__ __forceinline__ bool has(int c) const { return (unsigned)(c - lo) < (unsigned)len; }
    __device__ __forceinline__ U load(int c, int q) const
    {
        return __hip_atomic_load(s + (c - lo) * k + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ void store(int c, int q, U v) const
    {
        __hip_atomic_store(s + (c - lo) * k + q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
};

// Publish x[i] in the value protocol: the sentinel can never be published
// (division results are never signalling NaNs; the guard keeps that true for
// any input bit pattern).
template <typename T>
__device__ __forceinline__ void publish_value(T *x, long long idx, T xi)
{
    typedef typename VBits<T>::U U;
    U o = as_bits(xi);
    if (o == VBits<T>::kSentinel) o = VBits<T>::kQNaN;
    st_agent(reinterpret_cast<U *>(x) + idx, o);
}

// ------------------------------------------------------------------ fills
template <typename U>
__global__ void __launch_bounds__(kBlock) k_fill(U *__restrict__ p, long long count, U value)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < count; i += stride) p[i] = value;
}

// Per-solve reset: tickets (and the value protocol's sentinel fill of x) in
// one launch, so no memset node is needed when a caller captures solves in a
// graph.
template <typename U>
__global__ void __launch_bounds__(kBlock)
    k_prepare(U *__restrict__ p, long long count, U value, unsigned *__restrict__ ticket, int n_ticket)
{
    if (blockIdx.x == 0 && (int)threadIdx.x < n_ticket) ticket[threadIdx.x] = 0u;
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < count; i += stride) p[i] = value;
}

// k_prepare plus zeroed convergence norms (two words): the fused refinement
// sweep's whole reset in one launch.
template <typename U>
__global__ void __launch_bounds__(kBlock)
    k_prepare_norms(U *__restrict__ p, long long count, U value, unsigned *__restrict__ ticket, int n_ticket,
                    unsigned long long *__restrict__ norms)
{
    if (blockIdx.x == 0 && (int)threadIdx.x < n_ticket) ticket[threadIdx.x] = 0u;
    if (blockIdx.x == 0 && threadIdx.x < 2) norms[threadIdx.x] = 0ULL;
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < count; i += stride) p[i] = value;
}

// ------------------------------------------------- write-first row solver
// Publishes x[o] (o = row*k + q) in the protocol SYNC (1 value, 2 flag).
template <typename T, int SYNC>
__device__ __forceinline__ void publish(T *x, const SyncCtx &sc, long long o, T xi)
{
    if (SYNC == 1) {
        if (sc.ready) {
            publish_value(reinterpret_cast<T *>(sc.ready), o, xi);
            x[o] = xi;
        } else {
            publish_value(x, o, xi);
        }
    } else {
        // flag protocol without cache-wide fences: the value goes out as a
        // returning agent-scope exchange, and the flag store depends on the
        // returned word, so the flag is issued only once the value is in place
        typedef typename VBits<T>::U U;
        const U old = __hip_atomic_exchange(reinterpret_cast<U *>(x) + o, as_bits(xi), __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
        int ep = sc.epoch;
        asm volatile("" : "+v"(ep) : "v"(old));
        __hip_atomic_store(sc.flags + o, ep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Blocking wait for x[o] (used where every dependency belongs to an earlier
// wavefront).  Returns the value; NaN if the watchdog fired.
template <typename T, int SYNC>
__device__ __forceinline__ T wait_value(const T *x, const SyncCtx &sc, long long o)
{
    typedef typename VBits<T>::U U;
    const U *xu = reinterpret_cast<const U *>(x);
    Idle idle;
    if (SYNC == 1) {
        const U *xr = ready_array(sc, x);
        U raw;
        while ((raw = ld_agent(xr + o)) == VBits<T>::kSentinel)
            if (give_up(sc, idle)) return as_val(VBits<T>::kQNaN);
        return as_val(raw);
    } else {
        while (ld_agent(sc.flags + o) != sc.epoch)
            if (give_up(sc, idle)) return as_val(VBits<T>::kQNaN);
        return as_val(ld_agent(xu + o));  // issued after the flag was seen
    }
}

// Non-blocking test of x[o]: true and the value when published.
template <typename T, int SYNC>
__device__ __forceinline__ bool try_value(const T *x, const SyncCtx &sc, long long o, T *out)
{
    typedef typename VBits<T>::U U;
    const U *xu = reinterpret_cast<const U *>(x);
    if (SYNC == 1) {
        const U raw = ld_agent(ready_array(sc, x) + o);
        *out = as_val(raw);
        return raw != VBits<T>::kSentinel;
    }
    if (ld_agent(sc.flags + o) != sc.epoch) return false;
    *out = as_val(ld_agent(xu + o));  // issued after the flag was seen
    return true;
}

__device__ __forceinline__ double bcast(double v, int lane)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float bcast(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// One row solved by a whole wavefront in the sequential order: lane l polls
// off-diagonal l of the current 64-entry window; the wavefront then adds the
// ready prefix term by term, s = fma(v_t, x_t, s) with broadcast operands, so
// the sum is the oracle's fused sequential one and only the last dependency
// to arrive sits on the critical path (one fma and the division after it).
// Every dependency is an earlier row, solved by an earlier wavefront.
template <typename T, int SYNC>
__device__ __forceinline__ void wave_row(const int *__restrict__ rp, const int *__restrict__ ci,
                                         const T *__restrict__ val, const T *__restrict__ b, T *__restrict__ x,
                                         const SyncCtx &sc, const LdsWin<typename VBits<T>::U> &win, int row)
{
    typedef typename VBits<T>::U U;
    const int lane = threadIdx.x & (kWave - 1);
    const int d = rp[row + 1] - 1;
    const T brow = b[row], vd = val[d];  // loaded now, off the critical path
    T s = (T)0;
    Idle idle;
    bool failed = false;
    for (int j0 = rp[row]; j0 < d; j0 += kWave) {
        const int cnt = min(kWave, d - j0);
        const int c = lane < cnt ? ci[j0 + lane] : 0;
        const T v = lane < cnt ? val[j0 + lane] : (T)0;
        T xv = (T)0;
        bool rdy = lane >= cnt;
        int used = 0;
        while (used < cnt) {
            if (!rdy) {
                if (win.has(c)) {
                    const U raw = win.load(c, 0);
                    rdy = raw != VBits<T>::kSentinel;
                    xv = as_val(raw);
                } else {
                    rdy = try_value<T, SYNC>(x, sc, c, &xv);
                }
            }
            const unsigned long long ready = __ballot(rdy);
            const int prefix = ~ready ? __builtin_ctzll(~ready) : kWave;
            const int upto = min(prefix, cnt);
            for (int t = used; t < upto; ++t) s = acc(sc, bcast(v, t), bcast(xv, t), s);
            if (upto > used) {
                idle.progress();
            } else if (give_up(sc, idle)) {  // uniform: idle is the same in every lane
                failed = true;
                break;
            }
            used = upto;
        }
        if (failed) break;
    }
    if (lane == 0) {
        const T xi = failed ? as_val(VBits<T>::kQNaN) : (brow - s) / vd;
        if (win.len) {
            U o = as_bits(xi);
            if (o == VBits<T>::kSentinel) o = VBits<T>::kQNaN;
            win.store(row, 0, o);
        }
        publish<T, SYNC>(x, sc, row, xi);
    }
}

// Value protocol form of wrtfst_row: a window of the next two dependencies
// (entries j and j+1) is polled at once and slides by the number consumed,
// so most rows (one or two off-diagonals) are covered by a single window and
// the loop body stays short.  Consumption is in stored order (fma chain).
// COUNT: add the number of poll loads issued to *np (the per-row spin
// counter of the counting instantiation).
template <typename T, bool COUNT = false>
__device__ __forceinline__ void wrtfst_row_value(const int *__restrict__ ci, const T *__restrict__ val,
                                                 const T *__restrict__ b, T *__restrict__ x, const SyncCtx &sc,
                                                 int i, int j, int d, int k, int q, T s, int n_rev,
                                                 const LdsWin<typename VBits<T>::U> &win, unsigned *np = nullptr)
{
    typedef typename VBits<T>::U U;
    constexpr U kS = VBits<T>::kSentinel;
    U *xr = ready_array(sc, x);
    // b and the diagonal are loaded before the polling loop: read after the
    // last dependency arrives, they would add a memory round trip per level
    const long long o = (long long)(n_rev ? n_rev - 1 - i : i) * k + q;
    const T bo = b[o], vd = val[d];
    int c0 = 0, c1 = 0;
    T v0 = (T)0, v1 = (T)0;
    U x0 = kS, x1 = kS;
    if (j < d) {
        c0 = n_rev ? n_rev - 1 - ci[j] : ci[j];
        v0 = val[j];
    }
    if (j + 1 < d) {
        c1 = n_rev ? n_rev - 1 - ci[j + 1] : ci[j + 1];
        v1 = val[j + 1];
    }
    Idle idle;
    bool done = false;
    do {  // wave-uniform exit: see wrtfst_row
        if (!done) {
            bool prog = false;
            if (COUNT) *np += (j < d && x0 == kS) + (j + 1 < d && x1 == kS);
            if (j < d && x0 == kS) x0 = win.has(c0) ? win.load(c0, q) : ld_agent(xr + (long long)c0 * k + q);
            if (j + 1 < d && x1 == kS) x1 = win.has(c1) ? win.load(c1, q) : ld_agent(xr + (long long)c1 * k + q);
            if (j < d && x0 != kS) {
                s = acc(sc, v0, as_val(x0), s);
                ++j;
                prog = true;
                if (j < d && x1 != kS) {  // both consumed: a fresh window
                    s = acc(sc, v1, as_val(x1), s);
                    ++j;
                    x0 = kS;
                    if (j < d) {
                        c0 = n_rev ? n_rev - 1 - ci[j] : ci[j];
                        v0 = val[j];
                    }
                } else {  // slide by one
                    c0 = c1;
                    v0 = v1;
                    x0 = x1;
                }
                x1 = kS;
                if (j + 1 < d) {
                    c1 = n_rev ? n_rev - 1 - ci[j + 1] : ci[j + 1];
                    v1 = val[j + 1];
                }
            }
            if (prog) {
                idle.progress();
            } else if (j < d && give_up(sc, idle)) {
                s = as_val(VBits<T>::kQNaN);  // poison this row; it still publishes below
                j = d;
            }
            if (j >= d) {  // write first: publish inside the polling loop
                const T xi = (bo - s) / vd;
                U u = as_bits(xi);
                if (u == kS) u = VBits<T>::kQNaN;
                if (win.len) win.store(i, q, u);
                st_agent(xr + o, u);
                if (sc.ready) x[o] = xi;
                asm volatile("" ::: "memory");
                done = true;
            }
        }
    } while (__any(!done));
}

// Solves row i (off-diagonal entries [j, d), diagonal at d) for right-hand
// side q of k (x and b interleaved: x[row*k + q]) and publishes it.  `s`
// carries a partial sum when the caller already consumed a prefix (two-part).
// n_rev > 0 stores row r at position n_rev-1-r of b and x (the adjoint solves
// L^T in reversed row order, which is lower triangular).
template <typename T, int SYNC, bool COUNT = false>
__device__ __forceinline__ void wrtfst_row(const int *__restrict__ ci, const T *__restrict__ val,
                                           const T *__restrict__ b, T *__restrict__ x, const SyncCtx &sc,
                                           int i, int j, int d, int k, int q, T s, int n_rev = 0,
                                           LdsWin<typename VBits<T>::U> win = {nullptr, 0, 0, 1},
                                           unsigned *np = nullptr)
{
    if constexpr (SYNC == 1) {
        wrtfst_row_value<T, COUNT>(ci, val, b, x, sc, i, j, d, k, q, s, n_rev, win, np);
        return;
    }
    // flag protocol: a fixed window of up to kWin entries, refilled when consumed
    typedef typename VBits<T>::U U;
    U *xu = reinterpret_cast<U *>(x);
    const long long o = (long long)(n_rev ? n_rev - 1 - i : i) * k + q;
    const T bo = b[o], vd = val[d];  // before the loop, off the critical path
    int cw[kWin];
    T vw[kWin];
    U xw[kWin];
    bool rdy[kWin];
    int cnt = min(kWin, d - j), used = 0;
    Idle idle;
#pragma unroll
    for (int t = 0; t < kWin; ++t) {
        rdy[t] = false;
        xw[t] = 0;
        cw[t] = t < cnt ? (n_rev ? n_rev - 1 - ci[j + t] : ci[j + t]) : 0;
        vw[t] = t < cnt ? val[j + t] : (T)0;
    }
    // The loop exits only when every lane of the wavefront has published
    // (wave-uniform exit).  With a per-lane exit the compiler may legally
    // move the publishing store to the loop exit, where a finished lane waits
    // for the rest of its wavefront -- which may be waiting for that store.
    bool done = false;
    do {
        if (!done) {
            if (used < cnt) {
                int fl[kWin];
                bool any = false;
#pragma unroll
                for (int t = 0; t < kWin; ++t)
                    fl[t] = (t >= used && t < cnt && !rdy[t]) ? ld_agent(sc.flags + (long long)cw[t] * k + q) : 0;
#pragma unroll
                for (int t = 0; t < kWin; ++t)
                    if (t >= used && t < cnt && !rdy[t] && fl[t] == sc.epoch) any = true;
                if (any) {  // values read after their flags were seen (agent-scope loads)
#pragma unroll
                    for (int t = 0; t < kWin; ++t)
                        if (t >= used && t < cnt && !rdy[t] && fl[t] == sc.epoch) {
                            xw[t] = ld_agent(xu + (long long)cw[t] * k + q);
                            rdy[t] = true;
                        }
                }
                // consume the ready prefix in stored order
                const int before = used;
#pragma unroll
                for (int t = 0; t < kWin; ++t)
                    if (t == used && t < cnt && rdy[t]) {
                        s = acc(sc, vw[t], as_val(xw[t]), s);
                        ++used;
                    }
                if (used != before) {
                    idle.progress();
                } else if (give_up(sc, idle)) {
                    s = as_val(VBits<T>::kQNaN);  // poison this row; it still publishes below
                    used = cnt;
                    j = d;
                }
                if (used == cnt && j < d) {
                    j += cnt;
                    if (j < d) {  // next window
                        cnt = min(kWin, d - j);
                        used = 0;
#pragma unroll
                        for (int t = 0; t < kWin; ++t) {
                            rdy[t] = false;
                            if (t < cnt) {
                                cw[t] = n_rev ? n_rev - 1 - ci[j + t] : ci[j + t];
                                vw[t] = val[j + t];
                            }
                        }
                    }
                }
            }
            if (used == cnt && j >= d) {  // write first: publish inside the polling loop
                publish<T, SYNC>(x, sc, o, (bo - s) / vd);
                asm volatile("" ::: "memory");
                done = true;
            }
        }
    } while (__any(!done));
}

// ourWrtFst (CUDA/ourWrtFst/spts_syncfree_cuda_csr_wrt.h:10-57): one lane
// per row and right-hand side; a workgroup of BLOCK threads (128 or 256)
// takes tickets of BLOCK >> lpr_log2 rows with 1 << lpr_log2 lanes per row,
// lane q of a row owning right-hand side q (lanes with q >= k idle).  The
// workgroup size sets how many rows poll at once on each compute unit.
// sched (optional, n_sched blocks): ticket t solves rows [sched[t].x,
// sched[t].x + sched[t].y) instead of the t-th run of consecutive rows.  The
// host orders the blocks so that every row comes after the rows it depends
// on (each matrix of a batch keeps its row order), which keeps the
// forward-progress argument of the ticket loop.
// COUNT (value protocol only): every lane counts the poll loads it issues;
// each wavefront adds its total to one of sc.polls' kPollCounters counters
// when the grid drains (one atomic per wavefront).
// TILE: a ticket's rows are consecutive, so their entries are one range
// [rp[lo], rp[lo + len]) of col_idx and val; the workgroup first copies it
// into LDS with coalesced loads (consecutive lanes, consecutive entries),
// and the rows read their entries there.  A range longer than kRowTile
// entries (uniform in the workgroup) is read from global memory as usual.
constexpr int kRowTile = 2048;
template <typename T, int SYNC, int LDS, int BLOCK, bool COUNT = false, bool TILE = false>
__global__ void __launch_bounds__(BLOCK)
    k_wrtfst(const int *__restrict__ rp, const int *__restrict__ ci, const T *__restrict__ val,
             const T *__restrict__ b, T *__restrict__ x, SyncCtx sc, int n, int k, int lpr_log2,
             unsigned *__restrict__ ticket, int n_rev, const int2 *__restrict__ sched, int n_sched)
{
    typedef typename VBits<T>::U U;
    static_assert(!COUNT || SYNC == 1, "the poll counter is for the value protocol");
    __shared__ U s_x[LDS ? BLOCK : 1];
    __shared__ int s_ci[TILE ? kRowTile : 1];
    __shared__ T s_v[TILE ? kRowTile : 1];
    const int q = threadIdx.x & ((1 << lpr_log2) - 1);
    const int r = threadIdx.x >> lpr_log2;
    const int rows = BLOCK >> lpr_log2;
    unsigned np = 0;
    ticket_loop(
        ticket, sched ? 1 : rows, sched ? n_sched : n,
        [&](int) {
            if (LDS) s_x[threadIdx.x] = VBits<T>::kSentinel;
        },
        [&](int base) {
            int lo = base, len = rows;
            if (sched) {
                const int2 blk = sched[base];
                lo = blk.x;
                len = blk.y;
            }
            const int i = lo + r;
            LdsWin<U> win{s_x, lo, (LDS && !n_rev) ? len : 0, k};
            const int *cix = ci;
            const T *vx = val;
            int e0 = 0;  // entry j of a row is cix[j - e0]
            if constexpr (TILE) {
                const int first = rp[lo], last = rp[min(lo + len, n)];
                if (last - first <= kRowTile) {  // uniform in the workgroup
                    for (int e = threadIdx.x; e < last - first; e += BLOCK) {
                        s_ci[e] = ci[first + e];
                        s_v[e] = val[first + e];
                    }
                    __syncthreads();
                    cix = s_ci;
                    vx = s_v;
                    e0 = first;
                }
            }
            if (r < len && i < n && q < k)
                wrtfst_row<T, SYNC, COUNT>(cix, vx, b, x, sc, i, rp[i] - e0, rp[i + 1] - 1 - e0, k, q, (T)0, n_rev,
                                           win, &np);
        });
    if constexpr (COUNT) {
        unsigned long long t = np;
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) t += (unsigned long long)__shfl_xor((long long)t, o, kWave);
        if ((threadIdx.x & (kWave - 1)) == 0)
            atomic_add_agent(sc.polls + (blockIdx.x * (BLOCK / kWave) + threadIdx.x / kWave) % kPollCounters, t);
    }
}

// ------------------------------------------------ look-through solve
// Solve of matrices whose rows hold at most kHopMax off-diagonals, with half
// the dependency hops.  A row that would wait for a value of the newest wave
// of results does not wait for it: it waits for the values THAT row needs
// and computes it again itself (the same operations on the same operands, so
// the same bits).  Each cross-CU hop then covers two levels.
//   hop(i) = 1 + max over i's entries c of min(hop(c), look(c)),
//   look(c) = max of hop over c's own entries;
// entry c of row i is looked through where hop(c) exceeds hop(i) - 1.
//
// Why: with readiness polled in device memory, a solve of wide levels costs
// one publish -> observe hop per level, and the hop's length is set by the
// polls themselves: each lane's poll is a 64-byte fabric request, 64 of them
// per wavefront, and 65,536 polling rows fill the fabric for about 1.3 us a
// round (with polls that share lines the same rows poll in a quarter of
// that).  So this kernel
//  * halves the hops (155 -> 78 on the wide-level 2M matrix) at 1.2 x the polls;
//  * hands out rows in hop order and indexes the readiness array by position
//    in that order, not by row: a wavefront publishes 64 adjacent values, and
//    where neighbouring rows depend on neighbouring rows (grids) their polls
//    share lines;
//  * reads a row's whole description with one coalesced round of loads
//    (tables laid out at plan creation; the values themselves stay in the
//    caller's array, which may change between solves), so a workgroup is
//    ready to poll two memory round trips after its ticket instead of five.
// Measured (kernel alone, FP64): wide-level 2M 213 -> 148 us; a 100 x 90 x 80
// grid's 7-point lower factor (268 levels) 2,050 -> 220 us.  In the same
// tests: hop order without looking through 196 / 311 us; looking through
// without the reordered readiness array 173 / 275 us; looking through two
// rows deep (52 hops) 235 us on the wide-level matrix (its longer load
// chains outweigh the saved hops).
//
// Table of slot s (position in hop order; field f at base[f * npad + s]):
// the row, its first entry, the counts word, then per entry the slot to poll
// (or, looked through, the row).  Counts word: bits 0-2 the row's entries,
// bit 3 + j entry j is looked through, bits 8 + 3j the polls of entry j
// (1, or the looked-through row's entries).  ex holds, per wavefront of
// slots, for each entry the looked-through row's first entry and its entries'
// slots, 64 of each.
constexpr int kHopMax = 4;
struct HopTab {
    const int *base, *ex;
    int npad;
};

// The tables of E entries per row, from the hop order (order[s] = row of slot
// s), its inverse and each row's look-through bits.  One thread per slot;
// slots past n describe row 0 with no entries (their lanes stay idle).
template <int E>
__global__ void __launch_bounds__(kBlock)
    k_hop_tables(const int *__restrict__ rp, const int *__restrict__ ci, const int *__restrict__ order,
                 const int *__restrict__ slot, const unsigned char *__restrict__ look, int n, int npad,
                 int *__restrict__ base, int *__restrict__ ex)
{
    const int s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= npad) return;
    const bool in = s < n;
    const int row = in ? order[s] : 0;
    const int e0 = rp[row], cnt = in ? rp[row + 1] - 1 - e0 : 0;
    const unsigned m = in ? look[row] : 0;
    int cw = cnt;
    int *x = ex + (size_t)(s >> 6) * (kWave * E * (E + 1)) + (s & (kWave - 1));
#pragma unroll
    for (int j = 0; j < E; ++j) {
        int c = 0, first = 0, nn = 0, to[E] = {};
        if (j < cnt) {
            c = ci[e0 + j];
            nn = 1;
            if ((m >> j) & 1) {
                cw |= 1 << (3 + j);
                first = rp[c];
                nn = rp[c + 1] - 1 - first;
#pragma unroll
                for (int t = 0; t < E; ++t)
                    if (t < nn) to[t] = slot[ci[first + t]];
            } else {
                c = slot[c];
            }
        }
        cw |= nn << (8 + 3 * j);
        base[(size_t)(3 + j) * npad + s] = c;
        x[(j * (E + 1)) * kWave] = first;
#pragma unroll
        for (int t = 0; t < E; ++t) x[(j * (E + 1) + 1 + t) * kWave] = to[t];
    }
    base[s] = row;
    base[(size_t)npad + s] = e0;
    base[(size_t)2 * npad + s] = cw;
}

__global__ void __launch_bounds__(kBlock)
    k_invert(const int *__restrict__ order, int n, int *__restrict__ slot)
{
    const int s = blockIdx.x * kBlock + threadIdx.x;
    if (s < n) slot[order[s]] = s;
}

// One lane per row, tickets of BLOCK slots; wavefront 0 takes the next ticket
// when its own rows are done, while the others may still poll.  n_rev > 0: row r is
// stored at n_rev - 1 - r of b and x (upper-triangular plans).
template <typename T, int E, int BLOCK>
__global__ void __launch_bounds__(BLOCK)
    k_hop(HopTab tab, const T *__restrict__ val, const T *__restrict__ b, T *__restrict__ x, SyncCtx sc, int n,
          unsigned *__restrict__ ticket, int n_rev)
{
    typedef typename VBits<T>::U U;
    constexpr U kS = VBits<T>::kSentinel;
    U *xr = reinterpret_cast<U *>(sc.ready);
    __shared__ int s_base[2];
    if (threadIdx.x == 0) s_base[0] = (int)atomicAdd(ticket, (unsigned)BLOCK);
    for (int turn = 0;; turn ^= 1) {
        lds_barrier();
        const int first = s_base[turn];
        if (first >= n) return;
        const int s = first + (int)threadIdx.x;
        const bool in = s < n;
        // one coalesced round: the row's description (slot 0's past the end)
        const int sl = in ? s : 0;
        const int row = tab.base[sl], e0 = tab.base[(size_t)tab.npad + sl];
        const int cw = in ? tab.base[(size_t)2 * tab.npad + sl] : 0;
        int c[E], f[E], to[E][E];
        const int *ex = tab.ex + (size_t)(sl >> 6) * (kWave * E * (E + 1)) + (sl & (kWave - 1));
#pragma unroll
        for (int j = 0; j < E; ++j) {
            c[j] = tab.base[(size_t)(3 + j) * tab.npad + sl];
            f[j] = ex[(j * (E + 1)) * kWave];
#pragma unroll
            for (int t = 0; t < E; ++t) to[j][t] = ex[(j * (E + 1) + 1 + t) * kWave];
        }
        const int cnt = cw & 7;
        U r[E][E];
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const bool lk = (cw >> (3 + j)) & 1;
            const int nn = (cw >> (8 + 3 * j)) & 7;
            if (!lk) to[j][0] = c[j];
#pragma unroll
            for (int t = 0; t < E; ++t) r[j][t] = t < nn ? kS : (U)0;
        }
        // second round: every value of the row and of the rows it looks
        // through.  Unused ones read an entry that exists (no branch, so the
        // loads are issued together) and are left out of the sums below.
        const int o = n_rev ? n_rev - 1 - row : row;
        const T bo = b[o], vd = val[e0 + cnt];
        T v[E], vv[E][E], bb[E], dd[E];
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const bool lk = (cw >> (3 + j)) & 1;
            const int nn = lk ? (cw >> (8 + 3 * j)) & 7 : 0, g = lk ? c[j] : 0, fj = lk ? f[j] : 0;
            v[j] = val[e0 + min(j, cnt)];
            bb[j] = b[n_rev ? n_rev - 1 - g : g];
            dd[j] = val[fj + nn];
#pragma unroll
            for (int t = 0; t < E; ++t) vv[j][t] = val[fj + min(t, nn)];
        }
        Idle idle;
        int missing = -1;
        bool done = !in;
        do {  // wave-uniform exit: see wrtfst_row
            if (!done) {
                int left = 0;  // values still missing
#pragma unroll
                for (int j = 0; j < E; ++j)
#pragma unroll
                    for (int t = 0; t < E; ++t)
                        if (r[j][t] == kS) r[j][t] = ld_agent(xr + to[j][t]);
#pragma unroll
                for (int j = 0; j < E; ++j)
#pragma unroll
                    for (int t = 0; t < E; ++t) left += r[j][t] == kS;
                if (left != missing) idle.progress();
                const bool failed = left != 0 && left == missing && give_up(sc, idle);
                missing = left;
                if (left == 0 || failed) {
                    T sum = (T)0;
#pragma unroll
                    for (int j = 0; j < E; ++j) {
                        T xj = as_val(r[j][0]);
                        if ((cw >> (3 + j)) & 1) {
                            const int nn = (cw >> (8 + 3 * j)) & 7;
                            T q = (T)0;
#pragma unroll
                            for (int t = 0; t < E; ++t)
                                if (t < nn) q = acc(sc, vv[j][t], as_val(r[j][t]), q);
                            xj = (bb[j] - q) / dd[j];
                        }
                        if (j < cnt) sum = acc(sc, v[j], xj, sum);
                    }
                    if (failed) sum = as_val(VBits<T>::kQNaN);  // poison this row; it still publishes
                    const T xi = (bo - sum) / vd;
                    U u = as_bits(xi);
                    if (u == kS) u = VBits<T>::kQNaN;
                    st_agent(xr + s, u);
                    x[o] = xi;
                    asm volatile("" ::: "memory");
                    done = true;
                }
            }
        } while (__any(!done));
        // read by the others after the next barrier; the slot they read for
        // this turn is not written again before the one after it
        if (threadIdx.x == 0) s_base[turn ^ 1] = (int)atomicAdd(ticket, (unsigned)BLOCK);
    }
}

// Value protocol row solver for R right-hand sides per lane: the lane owns
// right-hand sides q, q + L, ..., q + (R-1)L of row i (those below k), L
// lanes per row, so each poll instruction of the row's L lanes reads L
// contiguous values.  A dependency is consumed once all of the lane's R
// values of it are published; each right-hand side keeps its own sum in
// stored order, so the results are those of R single-RHS lanes.  The window
// (two dependencies, sliding) and the wave-uniform exit are those of
// wrtfst_row_value.
template <typename T, int R>
__device__ __forceinline__ void wrtfst_row_value_r(const int *__restrict__ ci, const T *__restrict__ val,
                                                   const T *__restrict__ b, T *__restrict__ x, const SyncCtx &sc,
                                                   int i, int j, int d, int k, int q, int L)
{
    typedef typename VBits<T>::U U;
    constexpr U kS = VBits<T>::kSentinel;
    U *xr = ready_array(sc, x);
    int nr = 0;  // right-hand sides of this lane
#pragma unroll
    for (int t = 0; t < R; ++t) nr += q + t * L < k;
    const long long o = (long long)i * k + q;
    T bo[R], s[R];
    const T vd = val[d];
#pragma unroll
    for (int t = 0; t < R; ++t) {
        bo[t] = t < nr ? b[o + t * L] : (T)0;  // before the polling loop, as in wrtfst_row_value
        s[t] = (T)0;
    }
    int c0 = 0, c1 = 0;
    T v0 = (T)0, v1 = (T)0;
    U x0[R], x1[R];
#pragma unroll
    for (int t = 0; t < R; ++t) x0[t] = x1[t] = kS;
    if (j < d) {
        c0 = ci[j];
        v0 = val[j];
    }
    if (j + 1 < d) {
        c1 = ci[j + 1];
        v1 = val[j + 1];
    }
    Idle idle;
    bool done = false;
    do {  // wave-uniform exit: see wrtfst_row
        if (!done) {
            bool prog = false, r0 = j < d, r1 = j + 1 < d;
#pragma unroll
            for (int t = 0; t < R; ++t) {
                if (t < nr && j < d && x0[t] == kS) x0[t] = ld_agent(xr + (long long)c0 * k + q + t * L);
                if (t < nr && j + 1 < d && x1[t] == kS) x1[t] = ld_agent(xr + (long long)c1 * k + q + t * L);
                r0 = r0 && (t >= nr || x0[t] != kS);
                r1 = r1 && (t >= nr || x1[t] != kS);
            }
            if (r0) {
#pragma unroll
                for (int t = 0; t < R; ++t) s[t] = acc(sc, v0, as_val(x0[t]), s[t]);
                ++j;
                prog = true;
                if (r1) {  // both consumed: a fresh window
#pragma unroll
                    for (int t = 0; t < R; ++t) {
                        s[t] = acc(sc, v1, as_val(x1[t]), s[t]);
                        x0[t] = kS;
                    }
                    ++j;
                    if (j < d) {
                        c0 = ci[j];
                        v0 = val[j];
                    }
                } else {  // slide by one
                    c0 = c1;
                    v0 = v1;
#pragma unroll
                    for (int t = 0; t < R; ++t) x0[t] = x1[t];
                }
#pragma unroll
                for (int t = 0; t < R; ++t) x1[t] = kS;
                if (j + 1 < d) {
                    c1 = ci[j + 1];
                    v1 = val[j + 1];
                }
            }
            if (prog) {
                idle.progress();
            } else if (j < d && give_up(sc, idle)) {
#pragma unroll
                for (int t = 0; t < R; ++t) s[t] = as_val(VBits<T>::kQNaN);  // poison; still published below
                j = d;
            }
            if (j >= d) {  // write first: publish inside the polling loop
#pragma unroll
                for (int t = 0; t < R; ++t) {
                    if (t < nr) {
                        const T xi = (bo[t] - s[t]) / vd;
                        U u = as_bits(xi);
                        if (u == kS) u = VBits<T>::kQNaN;
                        st_agent(xr + o + t * L, u);
                        if (sc.ready) x[o + t * L] = xi;
                    }
                }
                asm volatile("" ::: "memory");
                done = true;
            }
        }
    } while (__any(!done));
}

// Thread-per-row solve with R right-hand sides per lane (value protocol, no
// LDS window): L = 1 << lpr_log2 lanes per row, BLOCK >> lpr_log2 rows per
// ticket.  With k right-hand sides, R per lane makes a ticket R times as
// many rows as k_wrtfst's, every row still polled by its own lanes at once
// (a ticket's rows are all in flight together).  Tickets, batch schedule
// and forward progress as in k_wrtfst.
template <typename T, int BLOCK, int R>
__global__ void __launch_bounds__(BLOCK)
    k_wrtfst_r(const int *__restrict__ rp, const int *__restrict__ ci, const T *__restrict__ val,
               const T *__restrict__ b, T *__restrict__ x, SyncCtx sc, int n, int k, int lpr_log2,
               unsigned *__restrict__ ticket, const int2 *__restrict__ sched, int n_sched)
{
    const int L = 1 << lpr_log2;
    const int q = threadIdx.x & (L - 1);
    const int r = threadIdx.x >> lpr_log2;
    const int rows = BLOCK >> lpr_log2;
    ticket_loop(ticket, sched ? 1 : rows, sched ? n_sched : n, [&](int base) {
        int lo = base, len = rows;
        if (sched) {
            const int2 blk = sched[base];
            lo = blk.x;
            len = blk.y;
        }
        const int i = lo + r;
        if (r < len && i < n && q < k) wrtfst_row_value_r<T, R>(ci, val, b, x, sc, i, rp[i], rp[i + 1] - 1, k, q, L);
    });
}

// ------------------------------------------------------------ refinement
// Maxima of non-negative doubles are taken on their bit patterns (which
// order like the values): per thread over a grid-stride loop, then across
// the workgroup in LDS, then one atomicMax per workgroup -- an atomic per
// element on one address serialises in the memory side.
__device__ __forceinline__ void block_max_to(unsigned long long v, unsigned long long *__restrict__ out)
{
    __shared__ unsigned long long s_max[kBlock / kWave];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const unsigned long long w = (unsigned long long)__shfl_xor((long long)v, o, kWave);
        v = w > v ? w : v;
    }
    if ((threadIdx.x & (kWave - 1)) == 0) s_max[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x / kWave); ++w) v = s_max[w] > v ? s_max[w] : v;
        atomicMax(out, v);
    }
}

// The two norms into the host's memory, then the count they belong to.
__global__ void k_echo(const unsigned long long *__restrict__ norms, unsigned long long *echo, unsigned long long count)
{
    if (threadIdx.x != 0) return;
    __hip_atomic_store(echo, norms[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(echo + 1, norms[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(echo + 2, count, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ------------------------------------------------ fused refinement sweep
// The first two steps of mixed-precision refinement in one dependency sweep.
// Row i computes, from the pairs (x0_j, d_j) of its dependencies j:
//   x0_i = ((float)b_i - sum v32_j x0_j) * r32_i           FP32 solve of b
//   r_i  = b_i - (sum v_j x0_j + v_ii x0_i)                FP64 residual
//   d_i  = ((float)r_i - sum v32_j d_j) * r32_i            FP32 correction
//   x_i  = (double)x0_i + (double)d_i
// (v32 = (float)v, r32_i = 1.0f / v32_ii computed before the row's polling
// loop, so no division is left on the critical path; the correction absorbs
// the extra rounding of the product; every sum an fma chain in stored order),
// which is bit for bit what the two steps give when run one after the other:
// FP32 solve, residual, FP32 solve of the residual, accumulation.  Row i publishes
// (x0_i, d_i) as one 64-bit word (x0 in the low half) in the value protocol;
// a dependency's word is read once and feeds all three chains, so the sweep
// has the dependency depth of a single solve.  The polling window is the one
// of wrtfst_row_value (two entries, sliding by the number consumed).
constexpr unsigned long long kPairQNaN = 0x7FC000007FC00000ULL;

__device__ __forceinline__ void refine_pair_take(double v, unsigned long long p, float &s0, double &s, float &s1)
{
    const float xa = __uint_as_float((unsigned)p), da = __uint_as_float((unsigned)(p >> 32));
    const float v32 = (float)v;
    s0 = __builtin_fmaf(v32, xa, s0);
    s = __builtin_fma(v, (double)xa, s);
    s1 = __builtin_fmaf(v32, da, s1);
}

__device__ __forceinline__ void refine_pair_row(const int *__restrict__ ci, const double *__restrict__ val,
                                                const double *__restrict__ b, double *__restrict__ x,
                                                unsigned long long *__restrict__ pr, const SyncCtx &sc, int i,
                                                int j, int d, int k, int q,
                                                const LdsWin<unsigned long long> &win, unsigned long long &dmax,
                                                unsigned long long &xmax)
{
    typedef unsigned long long U;
    constexpr U kS = VBits<double>::kSentinel;
    int c0 = 0, c1 = 0;
    double v0 = 0.0, v1 = 0.0;
    U p0 = kS, p1 = kS;
    float s0 = 0.0f, s1 = 0.0f;
    double s = 0.0;
    const long long o = (long long)i * k + q;
    const double vd = val[d], bo = b[o];  // before the loop, off the critical path
    const float rd32 = 1.0f / (float)vd;
    if (j < d) {
        c0 = ci[j];
        v0 = val[j];
    }
    if (j + 1 < d) {
        c1 = ci[j + 1];
        v1 = val[j + 1];
    }
    Idle idle;
    bool done = false;
    do {  // wave-uniform exit: see wrtfst_row
        if (!done) {
            bool prog = false;
            if (j < d && p0 == kS) p0 = win.has(c0) ? win.load(c0, q) : ld_agent(pr + (long long)c0 * k + q);
            if (j + 1 < d && p1 == kS) p1 = win.has(c1) ? win.load(c1, q) : ld_agent(pr + (long long)c1 * k + q);
            if (j < d && p0 != kS) {
                refine_pair_take(v0, p0, s0, s, s1);
                ++j;
                prog = true;
                if (j < d && p1 != kS) {  // both consumed: a fresh window
                    refine_pair_take(v1, p1, s0, s, s1);
                    ++j;
                    p0 = kS;
                    if (j < d) {
                        c0 = ci[j];
                        v0 = val[j];
                    }
                } else {  // slide by one
                    c0 = c1;
                    v0 = v1;
                    p0 = p1;
                }
                p1 = kS;
                if (j + 1 < d) {
                    c1 = ci[j + 1];
                    v1 = val[j + 1];
                }
            }
            if (prog) {
                idle.progress();
            } else if (j < d && give_up(sc, idle)) {
                s0 = s1 = __builtin_nanf("");  // poison this row; it still publishes below
                s = __builtin_nan("");
                j = d;
            }
            if (j >= d) {  // write first: publish inside the polling loop
                const float x0 = ((float)bo - s0) * rd32;
                s = __builtin_fma(vd, (double)x0, s);
                const float dc = ((float)(bo - s) - s1) * rd32;
                U u = ((U)__float_as_uint(dc) << 32) | (U)__float_as_uint(x0);
                if (u == kS) u = kPairQNaN;
                if (win.len) win.store(i, q, u);
                st_agent(pr + o, u);
                const double xd = (double)x0, dd = (double)dc;
                x[o] = xd + dd;
                const U ad = (U)__double_as_longlong(fabs(dd)), ax = (U)__double_as_longlong(fabs(xd));
                dmax = ad > dmax ? ad : dmax;
                xmax = ax > xmax ? ax : xmax;
                asm volatile("" ::: "memory");
                done = true;
            }
        }
    } while (__any(!done));
}

// Thread-per-row launch of the fused sweep (workgroup size, lane layout,
// tickets, batch schedule and LDS window as in k_wrtfst); pr holds the pairs
// and starts filled with the sentinel.  norms[0] = max|d|, norms[1] =
// max|x0| (bits of non-negative doubles, atomicMax per workgroup).  (Row
// tiles, which speed up the batch's 1024-thread solve, gave this sweep
// nothing: 9.60 against 9.45-9.58 ms on 253 matrices x 16 right-hand sides.)
template <int LDS, int BLOCK>
__global__ void __launch_bounds__(BLOCK)
    k_refine2(const int *__restrict__ rp, const int *__restrict__ ci, const double *__restrict__ val,
              const double *__restrict__ b, double *__restrict__ x, unsigned long long *__restrict__ pr, SyncCtx sc,
              int n, int k, int lpr_log2, unsigned *__restrict__ ticket, const int2 *__restrict__ sched, int n_sched,
              unsigned long long *__restrict__ norms)
{
    typedef unsigned long long U;
    __shared__ U s_x[LDS ? BLOCK : 1];
    const int q = threadIdx.x & ((1 << lpr_log2) - 1);
    const int r = threadIdx.x >> lpr_log2;
    const int rows = BLOCK >> lpr_log2;
    U dmax = 0, xmax = 0;
    ticket_loop(
        ticket, sched ? 1 : rows, sched ? n_sched : n,
        [&](int) {
            if (LDS) s_x[threadIdx.x] = VBits<double>::kSentinel;
        },
        [&](int base) {
            int lo = base, len = rows;
            if (sched) {
                const int2 blk = sched[base];
                lo = blk.x;
                len = blk.y;
            }
            const int i = lo + r;
            LdsWin<U> win{s_x, lo, LDS ? len : 0, k};
            if (r < len && i < n && q < k)
                refine_pair_row(ci, val, b, x, pr, sc, i, rp[i], rp[i + 1] - 1, k, q, win, dmax, xmax);
        });
    block_max_to(dmax, norms);
    __syncthreads();  // block_max_to's LDS slots are reused by the second reduction
    block_max_to(xmax, norms + 1);
}

// The same sweep over look-through tables (k_hop's layout and order of rows;
// the pair array is indexed by slot): a row that would wait for a row of its
// own hop works that row's pair out again from its entries, with the
// operations of the row itself, and so the same bits.  One right-hand side.
// n = 1,000,000, 100 levels of up to 2 entries (80 hops, 50 looked through):
// 113 -> 80 us.
template <int E, int BLOCK>
__global__ void __launch_bounds__(BLOCK)
    k_refine_hop(HopTab tab, const double *__restrict__ val, const double *__restrict__ b, double *__restrict__ x,
                 unsigned long long *__restrict__ pr, SyncCtx sc, int n, unsigned *__restrict__ ticket,
                 unsigned long long *__restrict__ norms)
{
    typedef unsigned long long U;
    constexpr U kS = VBits<double>::kSentinel;
    __shared__ int s_base[2];
    U dmax = 0, xmax = 0;
    if (threadIdx.x == 0) s_base[0] = (int)atomicAdd(ticket, (unsigned)BLOCK);
    for (int turn = 0;; turn ^= 1) {
        lds_barrier();
        const int first = s_base[turn];
        if (first >= n) break;
        const int s = first + (int)threadIdx.x;
        const bool in = s < n;
        const int sl = in ? s : 0;  // slot 0's description past the end
        const int row = tab.base[sl], e0 = tab.base[(size_t)tab.npad + sl];
        const int cw = in ? tab.base[(size_t)2 * tab.npad + sl] : 0, cnt = cw & 7;
        int c[E], f[E], to[E][E];
        const int *ex = tab.ex + (size_t)(sl >> 6) * (kWave * E * (E + 1)) + (sl & (kWave - 1));
#pragma unroll
        for (int j = 0; j < E; ++j) {
            c[j] = tab.base[(size_t)(3 + j) * tab.npad + sl];
            f[j] = ex[(j * (E + 1)) * kWave];
#pragma unroll
            for (int t = 0; t < E; ++t) to[j][t] = ex[(j * (E + 1) + 1 + t) * kWave];
        }
        U r[E][E];
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const bool lk = (cw >> (3 + j)) & 1;
            const int nn = (cw >> (8 + 3 * j)) & 7;
            if (!lk) to[j][0] = c[j];
#pragma unroll
            for (int t = 0; t < E; ++t) r[j][t] = t < nn ? kS : (U)0;
        }
        const double bo = b[row], vd = val[e0 + cnt];
        double v[E], vv[E][E], bb[E], dd[E];
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const bool lk = (cw >> (3 + j)) & 1;
            const int nn = lk ? (cw >> (8 + 3 * j)) & 7 : 0, g = lk ? c[j] : 0, fj = lk ? f[j] : 0;
            v[j] = val[e0 + min(j, cnt)];
            bb[j] = b[g];
            dd[j] = val[fj + nn];
#pragma unroll
            for (int t = 0; t < E; ++t) vv[j][t] = val[fj + min(t, nn)];
        }
        // a row's pair (first step and correction) from its sums, as bits
        auto pair = [](double bo, double vd, float s0, double s, float s1) {
            const float rd32 = 1.0f / (float)vd;
            const float x0 = ((float)bo - s0) * rd32;
            s = __builtin_fma(vd, (double)x0, s);
            const float dc = ((float)(bo - s) - s1) * rd32;
            const U u = ((U)__float_as_uint(dc) << 32) | (U)__float_as_uint(x0);
            return u == kS ? (U)kPairQNaN : u;
        };
        Idle idle;
        int missing = -1;
        bool done = !in;
        do {  // wave-uniform exit: see wrtfst_row
            if (!done) {
                int left = 0;  // values still missing
#pragma unroll
                for (int j = 0; j < E; ++j)
#pragma unroll
                    for (int t = 0; t < E; ++t)
                        if (r[j][t] == kS) r[j][t] = ld_agent(pr + to[j][t]);
#pragma unroll
                for (int j = 0; j < E; ++j)
#pragma unroll
                    for (int t = 0; t < E; ++t) left += r[j][t] == kS;
                if (left != missing) idle.progress();
                const bool failed = left != 0 && left == missing && give_up(sc, idle);
                missing = left;
                if (left == 0 || failed) {
                    float s0 = 0.0f, s1 = 0.0f;
                    double sum = 0.0;
#pragma unroll
                    for (int j = 0; j < E; ++j) {
                        U pj = r[j][0];
                        if ((cw >> (3 + j)) & 1) {
                            const int nn = (cw >> (8 + 3 * j)) & 7;
                            float q0 = 0.0f, q1 = 0.0f;
                            double q = 0.0;
#pragma unroll
                            for (int t = 0; t < E; ++t)
                                if (t < nn) refine_pair_take(vv[j][t], r[j][t], q0, q, q1);
                            pj = pair(bb[j], dd[j], q0, q, q1);
                        }
                        if (j < cnt) refine_pair_take(v[j], pj, s0, sum, s1);
                    }
                    if (failed) {  // poison this row; it still publishes
                        s0 = s1 = __builtin_nanf("");
                        sum = __builtin_nan("");
                    }
                    const U u = pair(bo, vd, s0, sum, s1);
                    st_agent(pr + s, u);
                    const double xd = (double)__uint_as_float((unsigned)u);
                    const double ddx = (double)__uint_as_float((unsigned)(u >> 32));
                    x[row] = xd + ddx;
                    const U ad = (U)__double_as_longlong(fabs(ddx)), ax = (U)__double_as_longlong(fabs(xd));
                    dmax = ad > dmax ? ad : dmax;
                    xmax = ax > xmax ? ax : xmax;
                    asm volatile("" ::: "memory");
                    done = true;
                }
            }
        } while (__any(!done));
        if (threadIdx.x == 0) s_base[turn ^ 1] = (int)atomicAdd(ticket, (unsigned)BLOCK);
    }
    __syncthreads();
    block_max_to(dmax, norms);
    __syncthreads();  // block_max_to's LDS slots are reused by the second reduction
    block_max_to(xmax, norms + 1);
}

// our2Part (CUDA/our2Part/spts_syncfree_cuda_csr.h:10-124): dependencies on
// rows of earlier wavefronts (col < first row of this wave) are waited for
// one by one; the rest is the write-first loop.  Single right-hand side.
template <typename T, int SYNC>
__global__ void __launch_bounds__(kBlock)
    k_twopart(const int *__restrict__ rp, const int *__restrict__ ci, const T *__restrict__ val,
              const T *__restrict__ b, T *__restrict__ x, SyncCtx sc, int n, unsigned *__restrict__ ticket)
{
    ticket_loop(ticket, kBlock, n, [&](int base) {
        const int wave_begin = base + (threadIdx.x & ~(kWave - 1));
        const int i = base + threadIdx.x;
        if (i >= n) return;
        int j = rp[i];
        const int d = rp[i + 1] - 1;
        T s = (T)0;
        for (; j < d; ++j) {  // rows of earlier wavefronts: blocking waits
            const int c = ci[j];
            if (c >= wave_begin) break;
            s = acc(sc, val[j], wait_value<T, SYNC>(x, sc, c), s);
        }
        wrtfst_row<T, SYNC>(ci, val, b, x, sc, i, j, d, 1, 0, s);
    });
}

// mix (CUDA/mix/spts_syncfree_cuda_csr_wrt.h:15-137): unit u covers rows
// [unit[u], unit[u+1]).  A unit of one row is solved by the whole wavefront
// (wave_row: parallel polls, sequential fused sum); a longer unit is solved
// thread-per-row with the write-first loop.  The 16 units of a ticket share
// an LDS window.  Single right-hand side.
// TILE: the ticket's units are consecutive rows [s_lo, s_lo + s_len), whose
// entries are first copied into LDS with coalesced loads (up to kMixTile of
// them; a longer range, uniform in the workgroup, is read from global memory)
// for the thread-per-row units.  Single-row units read global memory.
constexpr int kMixTile = 4096;
template <typename T, int SYNC, int BS, bool TILE = false>
__global__ void __launch_bounds__(BS)
    k_mix(const int *__restrict__ rp, const int *__restrict__ ci, const T *__restrict__ val,
          const T *__restrict__ b, T *__restrict__ x, SyncCtx sc, const int *__restrict__ unit, int n_units,
          unsigned *__restrict__ ticket)
{
    typedef typename VBits<T>::U U;
    constexpr int kUnits = BS / kWave;     // one unit per wavefront per ticket
    __shared__ U s_x[BS / kWave * kWave];  // rows of the ticket: <= 64 per unit
    __shared__ int s_lo, s_len;
    __shared__ int s_ci[TILE ? kMixTile : 1];
    __shared__ T s_v[TILE ? kMixTile : 1];
    const int lane = threadIdx.x & (kWave - 1);
    ticket_loop(
        ticket, kUnits, n_units,
        [&](int base) {
            if (SYNC == 1) s_x[threadIdx.x] = VBits<T>::kSentinel;
            if (threadIdx.x == 0 && base < n_units) {
                s_lo = unit[base];
                s_len = unit[min(base + kUnits, n_units)] - s_lo;
            }
        },
        [&](int base) {
            const int *cix = ci;
            const T *vx = val;
            int e0 = 0;  // entry j of a thread-per-row unit's row is cix[j - e0]
            if constexpr (TILE) {
                const int first = rp[s_lo], last = rp[s_lo + s_len];
                if (last - first <= kMixTile) {  // uniform in the workgroup
                    for (int e = threadIdx.x; e < last - first; e += BS) {
                        s_ci[e] = ci[first + e];
                        s_v[e] = val[first + e];
                    }
                    __syncthreads();
                    cix = s_ci;
                    vx = s_v;
                    e0 = first;
                }
            }
            const int u = base + (int)(threadIdx.x / kWave);
            if (u >= n_units) return;
            const LdsWin<U> win{s_x, s_lo, SYNC == 1 ? s_len : 0, 1};
            const int r0 = unit[u], r1 = unit[u + 1];
            if (r1 - r0 > 1) {
                const int i = r0 + lane;
                if (i < r1)
                    wrtfst_row<T, SYNC>(cix, vx, b, x, sc, i, rp[i] - e0, rp[i + 1] - 1 - e0, 1, 0, (T)0, 0, win);
                return;
            }
            wave_row<T, SYNC>(rp, ci, val, b, x, sc, win, r0);
        });
}

// ---------------------------------------- local: one matrix per workgroup
// For deep matrices (few rows per level) the cross-CU publish -> observe
// round trip (~0.5-2 us) is paid once per level.  Here one workgroup of
// kLocalBlock threads solves a whole matrix -- a segment [lo, hi) of rows
// whose dependencies never leave it -- so every hop stays inside one
// compute unit.  Wavefront w solves the rows lo + w, lo + w + W, ... (W
// wavefronts) one at a time: a row's entries are loaded 64 at a time into
// the lanes (coalesced; the next row's first 64 are prefetched while the
// current row is solved) and broadcast one by one, lane q < k accumulating
// right-hand side q in stored order (fused, bit-exact against the oracle).
//
// Readiness, per segment:
//  * ring (bandwidth + 2 W <= R slots): results are published into an LDS
//    ring -- slot r mod R holds the k values of row r, then a tag r written
//    after them -- and polled there (tag read before the value).  A
//    wavefront publishes row p only once every row <= p - R + bandwidth is
//    done, so no reader of the slot's previous row p - R is left; the
//    frontier is the lowest row any wavefront is still solving.  The
//    lowest unfinished row can always publish (R > bandwidth), so the
//    workgroup always makes progress.
//  * global: x itself (sentinel-filled) is polled with workgroup-scope
//    atomics.
// Results always go to x.  Segments are taken by ticket, largest first.
constexpr int kLocalBlock = 1024;
constexpr int kLocalGroup = 8;  // dependencies polled together
constexpr int kLocalPre = 8;    // rows of prefetch per wavefront
constexpr int kLocalStaticLds = 20 * 1024;  // k_local's static LDS (staging, frontier, ticket), rounded up

// segment {lo, hi, bandwidth, longest row's off-diagonal count}: ring mode
// needs the bandwidth plus two rounds of rows in flight within the ring and
// rows whose entries and diagonal fit one 64-lane load
__device__ __forceinline__ bool local_ring_fits(int4 sg, int R)
{
    return sg.z + 2 * (kLocalBlock / kWave) <= R && sg.w < kWave;
}

// The rows of one segment for one wavefront of k_local, ring mode (rows of
// at most 64 off-diagonal entries).  The wavefront's rows m = 0, 1, ... (row
// lo + w + m W) go in batches of kLocalPre: at the start of a batch the
// registers prefetched during the previous batch (each row's first 64
// entries with the diagonal in lanes, its right-hand sides in lanes < k) are
// copied -- the only wait for global memory, on loads issued a whole batch
// earlier -- and only then are the next batch's loads issued, into other
// registers, so that solving the batch never waits on a fresh load.  Row
// bounds (lanes 0-7: rp[row], lanes 8-15: rp[row + 1]) run one batch ahead
// of the entries.  The watchdog only sets a flag, reported once at the end.
template <typename T, bool K1>
__device__ __forceinline__ void local_rows_ring(const int *__restrict__ rp, const int *__restrict__ ci,
                                                const T *__restrict__ val, const T *__restrict__ b,
                                                typename VBits<T>::U *__restrict__ xu, const SyncCtx &sc, int k,
                                                int4 sg, int R, typename VBits<T>::U *rv, int *rt, int *s_cur,
                                                typename VBits<T>::U *xs, T *vs)
{
    typedef typename VBits<T>::U U;
    constexpr U kS = VBits<T>::kSentinel;
    constexpr int kWaves = kLocalBlock / kWave;
    constexpr int B = kLocalPre;
    static_assert(2 * B <= kWave, "bounds of a batch fit one register");
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int qk = min(lane, k - 1);
    const int lo = sg.x, hi = sg.y, bw = sg.z;
    auto row_of = [&](int m) { return lo + w + m * kWaves; };
    auto poll = [&](int c) -> U {
        const int sl = c & (R - 1);
        const int tg = __hip_atomic_load(rt + sl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        asm volatile("" ::: "memory");  // tag before value (the writer stores the value first)
        const U v = __hip_atomic_load(rv + (size_t)sl * k + qk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return tg == c ? v : kS;
    };
    auto load_bounds = [&](int mb) {
        const int r = row_of(mb + (lane & (B - 1)));
        return (lane < 2 * B && r < hi) ? rp[r + (lane >= B)] : 0;
    };
    // loads of batch mb from its bounds register: entries into c/v, right-hand
    // sides into bq; row bounds kept as scalars in a/e (e = diagonal's index)
    int nc[B], na[B], ne[B];
    T nv[B], nbq[B];
    auto issue_batch = [&](int mb, int bnd) {
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int r = row_of(mb + u);
            na[u] = __builtin_amdgcn_readlane(bnd, u);
            ne[u] = __builtin_amdgcn_readlane(bnd, u + B) - 1;
            if (r < hi) {
                if (lane <= ne[u] - na[u]) {
                    nc[u] = ci[na[u] + lane];
                    nv[u] = val[na[u] + lane];
                }
                nbq[u] = b[(long long)r * k + qk];
            }
        }
    };
#pragma unroll
    for (int u = 0; u < B; ++u) {
        nc[u] = 0;
        nv[u] = (T)0;
        nbq[u] = (T)0;
    }
    int bnd_next = load_bounds(0);
    {
        const int bnd = bnd_next;  // waits once, at the start
        issue_batch(0, bnd);
        bnd_next = load_bounds(B);
    }
    int front = lo;
    bool failed = false;
    for (int mb = 0; row_of(mb) < hi; mb += B) {
        // the previous batch's loads (and this batch's bounds) are complete: copy
        int cc[B], ca[B], ce[B];
        T cv[B], cbq[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            cc[u] = nc[u];
            cv[u] = nv[u];
            cbq[u] = nbq[u];
            ca[u] = na[u];
            ce[u] = ne[u];
        }
        const int bnd = bnd_next;
        if (row_of(mb + B) < hi) {
            issue_batch(mb + B, bnd);
            bnd_next = load_bounds(mb + 2 * B);
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int row = row_of(mb + u);
            if (row < hi) {
                const int a = ca[u], d = ce[u];
                const int cnt = d - a;
                Idle idle;
                T s = (T)0;
                if constexpr (K1) {
                    // one right-hand side: lane t polls entry t; values that
                    // arrive go to this wavefront's staging array, and the
                    // ready prefix is added in stored order from there (LDS
                    // reads at a wave-uniform address: a broadcast)
                    if (lane < cnt) vs[lane] = cv[u];
                    U xt = kS;
                    bool rdy = lane >= cnt;
                    int used = 0;
                    while (used < cnt) {
                        if (!rdy) {
                            xt = poll(cc[u]);
                            rdy = xt != kS;
                            if (rdy) xs[lane] = xt;
                        }
                        const unsigned long long ready = __ballot(rdy);
                        const int upto = min(cnt, ~ready ? (int)__builtin_ctzll(~ready) : kWave);
                        // a row with at most two entries left is about to be on
                        // the critical path: raise its issue priority early
                        // (measured 110 -> 104 ms on the deep band)
                        if (cnt - upto <= 2) __builtin_amdgcn_s_setprio(1);
                        if (upto == used) {
                            if (expired(sc, idle)) {
                                failed = true;
                                s = as_val(VBits<T>::kQNaN);
                                break;
                            }
                            continue;
                        }
                        // the rest of this row (chain tail, division, publish)
                        // is the critical path: take issue priority over the
                        // wavefronts that are still polling (reset after the
                        // publish); measured 117 -> 109 ms on the deep band
                        if (upto == cnt) __builtin_amdgcn_s_setprio(2);
                        idle.progress();
                        int t = used;
                        for (; t + 4 <= upto; t += 4) {
                            const T x0 = as_val(xs[t]), x1 = as_val(xs[t + 1]), x2 = as_val(xs[t + 2]),
                                    x3 = as_val(xs[t + 3]);
                            const T v0 = vs[t], v1 = vs[t + 1], v2 = vs[t + 2], v3 = vs[t + 3];
                            s = acc(sc, v0, x0, s);
                            s = acc(sc, v1, x1, s);
                            s = acc(sc, v2, x2, s);
                            s = acc(sc, v3, x3, s);
                        }
                        for (; t < upto; ++t) s = acc(sc, vs[t], as_val(xs[t]), s);
                        used = upto;
                    }
                } else
                for (int u0 = 0; u0 < cnt; u0 += kLocalGroup) {
                    int cu[kLocalGroup];
                    U xr[kLocalGroup];
#pragma unroll
                    for (int g = 0; g < kLocalGroup; ++g) {
                        cu[g] = __builtin_amdgcn_readlane(cc[u], min(u0 + g, cnt - 1));
                        xr[g] = u0 + g < cnt ? poll(cu[g]) : (U)0;
                    }
#pragma unroll
                    for (int g = 0; g < kLocalGroup; ++g) {
                        if (u0 + g < cnt) {
                            while (xr[g] == kS) {
                                if (expired(sc, idle)) {
                                    failed = true;
                                    xr[g] = VBits<T>::kQNaN;
                                    break;
                                }
                                xr[g] = poll(cu[g]);
                            }
                            s = acc(sc, bcast(cv[u], u0 + g), as_val(xr[g]), s);
                        }
                    }
                }
                __builtin_amdgcn_s_setprio(2);  // division and publish: the critical path
                // the slot's previous row and all its readers must be done
                idle.progress();
                while (row - R + bw >= front) {
                    int f = hi;
#pragma unroll
                    for (int v = 0; v < kWaves; ++v)
                        f = min(f, __hip_atomic_load(s_cur + v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
                    front = f;
                    if (row - R + bw < front) break;
                    if (expired(sc, idle)) {
                        failed = true;
                        break;
                    }
                }
                if (lane < k) {
                    const long long o = (long long)row * k + lane;
                    U uo = as_bits((cbq[u] - s) / bcast(cv[u], cnt));
                    if (uo == kS) uo = VBits<T>::kQNaN;
                    const int sl = row & (R - 1);
                    __hip_atomic_store(rv + (size_t)sl * k + lane, uo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    asm volatile("" ::: "memory");  // value before tag
                    if (lane == 0) __hip_atomic_store(rt + sl, row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    xu[o] = uo;
                }
                asm volatile("" ::: "memory");
                if (lane == 0) __hip_atomic_store(s_cur + w, row + kWaves, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __builtin_amdgcn_s_setprio(0);
            }
        }
    }
    if (__any(failed) && lane == 0) atomicOr(sc.err, 1);
}

// The rows of one segment for one wavefront of k_local, global mode (any
// row length): x itself is polled; each row's entries are loaded when the
// row starts.
template <typename T>
__device__ __forceinline__ void local_rows_global(const int *__restrict__ rp, const int *__restrict__ ci,
                                                  const T *__restrict__ val, const T *__restrict__ b,
                                                  typename VBits<T>::U *__restrict__ xu, const SyncCtx &sc, int k,
                                                  int4 sg, int *s_cur)
{
    typedef typename VBits<T>::U U;
    constexpr U kS = VBits<T>::kSentinel;
    constexpr int kWaves = kLocalBlock / kWave;
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int qk = min(lane, k - 1);
    for (int row = sg.x + w; row < sg.y; row += kWaves) {
        const int a = rp[row], d = rp[row + 1] - 1;
        Idle idle;
        T s = (T)0;
        for (int j0 = a; j0 < d; j0 += kWave) {
            const int cnt = min(kWave, d - j0);
            const int cl = lane < cnt ? ci[j0 + lane] : 0;
            const T vl = lane < cnt ? val[j0 + lane] : (T)0;
            for (int u0 = 0; u0 < cnt; u0 += kLocalGroup) {
                int cu[kLocalGroup];
                U xr[kLocalGroup];
#pragma unroll
                for (int g = 0; g < kLocalGroup; ++g) {
                    cu[g] = __builtin_amdgcn_readlane(cl, min(u0 + g, cnt - 1));
                    xr[g] = u0 + g < cnt ? __hip_atomic_load(xu + (long long)cu[g] * k + qk, __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_WORKGROUP)
                                         : (U)0;
                }
#pragma unroll
                for (int g = 0; g < kLocalGroup; ++g) {
                    if (u0 + g < cnt) {
                        while (xr[g] == kS) {
                            if (give_up(sc, idle)) {
                                xr[g] = VBits<T>::kQNaN;
                                break;
                            }
                            xr[g] = __hip_atomic_load(xu + (long long)cu[g] * k + qk, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_WORKGROUP);
                        }
                        s = acc(sc, bcast(vl, u0 + g), as_val(xr[g]), s);
                    }
                }
            }
        }
        if (lane < k) {
            const long long o = (long long)row * k + lane;
            U uo = as_bits((b[o] - s) / val[d]);
            if (uo == kS) uo = VBits<T>::kQNaN;
            __hip_atomic_store(xu + o, uo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_store(s_cur + w, row + kWaves, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

template <typename T>
__global__ void __launch_bounds__(kLocalBlock)
    k_local(const int *__restrict__ rp, const int *__restrict__ ci, const T *__restrict__ val,
            const T *__restrict__ b, T *__restrict__ x, SyncCtx sc, int k, const int4 *__restrict__ seg, int n_seg,
            unsigned *__restrict__ ticket, int ring_log2)
{
    typedef typename VBits<T>::U U;
    constexpr int kWaves = kLocalBlock / kWave;
    extern __shared__ unsigned long long smem_local[];
    const int R = 1 << ring_log2;
    U *rv = reinterpret_cast<U *>(smem_local);              // R * k values
    int *rt = reinterpret_cast<int *>(rv + (size_t)R * k);  // R tags
    __shared__ int s_cur[kWaves];                            // row each wavefront is solving
    __shared__ U s_xs[kWaves][kWave];                        // k = 1: per-wavefront staging of x
    __shared__ T s_vs[kWaves][kWave];                        // and of the row's coefficients
    U *xu = reinterpret_cast<U *>(x);
    const int lane = threadIdx.x & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    ticket_loop(
        ticket, 1, n_seg,
        [&](int t) {
            if (t >= n_seg) return;
            const int4 sg = seg[t];
            if (local_ring_fits(sg, R))
                for (int i = threadIdx.x; i < R; i += blockDim.x) rt[i] = -1;
            if (lane == 0) s_cur[w] = sg.x + w;
        },
        [&](int t) {
            const int4 sg = seg[t];
            if (local_ring_fits(sg, R) && k == 1)
                local_rows_ring<T, true>(rp, ci, val, b, xu, sc, k, sg, R, rv, rt, s_cur, s_xs[w], s_vs[w]);
            else if (local_ring_fits(sg, R))
                local_rows_ring<T, false>(rp, ci, val, b, xu, sc, k, sg, R, rv, rt, s_cur, s_xs[w], s_vs[w]);
            else
                local_rows_global<T>(rp, ci, val, b, xu, sc, k, sg, s_cur);
            if (lane == 0) __hip_atomic_store(s_cur + w, sg.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        });
}

// ------------------------------------------------ SyncFree CSC (K4 / K5)
// sptrsv_syncfree_cuda_analyser (CUDA/SyncFree_csc/spts_syncfree_cuda2.h:10-21)
__global__ void __launch_bounds__(kBlock) k_indegree(const int *__restrict__ idx, int nnz, int *__restrict__ deg)
{
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < nnz) atomic_add_agent(deg + idx[g], 1);
}

// sptrsv_syncfree_cuda_executor_update (spts_syncfree_cuda2.h:24-86),
// redesigned for short columns: a group of G lanes per column (G chosen by
// the host from the mean column length; the reference uses one warp per
// column), kBlock / G columns per workgroup ticket.  A column waits until
// only its diagonal's own count remains, computes x_i = (b_i - left_sum_i) /
// diag, then its lanes scatter left_sum[r] += x_i * v and release one count
// of each row r.  Columns of one wavefront can depend on each other, so the
// loop is write-first with a wave-uniform exit (as in wrtfst_row).
// Ordering without cache-wide fences: the left-sum atomics return their old
// values and the in-degree decrements are issued only after those returned
// (a data dependency), so a reader that sees the count drop to 1 finds every
// contribution performed; it then reads left_sum with an agent-scope atomic
// load.  FORWARD takes the diagonal from the first entry of the column,
// BACKWARD from the last.
template <typename T, int G>
__global__ void __launch_bounds__(kBlock)
    k_csc(const int *__restrict__ cp, const int *__restrict__ ri, const T *__restrict__ cv,
          int *__restrict__ deg, T *__restrict__ left_sum, const T *__restrict__ b, T *__restrict__ x, int m,
          int backward, SyncCtx sc, unsigned *__restrict__ ticket)
{
    typedef typename VBits<T>::U U;
    constexpr int kCols = kBlock / G;
    const int g = threadIdx.x & (G - 1);
    ticket_loop(ticket, kCols, m, [&](int base) {
        int col = base + (int)(threadIdx.x / G);
        bool done = col >= m;
        if (!done && backward) col = m - 1 - col;
        int dpos = 0, start = 0, stop = 0;
        T bc = (T)0, dg = (T)1;  // loaded before the wait, off the critical path
        if (!done) {
            dpos = backward ? cp[col + 1] - 1 : cp[col];
            start = backward ? cp[col] : cp[col] + 1;
            stop = backward ? cp[col + 1] - 1 : cp[col + 1];
            bc = b[col];
            dg = cv[dpos];
        }
        Idle idle;
        do {  // wave-uniform exit
            if (!done) {
                const bool ready = ld_agent(deg + col) == 1;
                const bool failed = !ready && give_up(sc, idle);
                if (ready || failed) {
                    const T ls = as_val(ld_agent(reinterpret_cast<const U *>(left_sum) + col));
                    const T xi = failed ? as_val(VBits<T>::kQNaN) : (bc - ls) / dg;
                    T token = (T)0;
                    for (int j = start + g; j < stop; j += G)
                        token += __hip_atomic_fetch_add(left_sum + ri[j], xi * cv[j], __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
                    // the decrements depend on the returned sums: `one` passes
                    // through an asm that consumes token, so the compiler waits
                    // for the returning atomics before issuing the decrements
                    int one = 1;
                    asm volatile("" : "+v"(one) : "v"(token));
                    for (int j = start + g; j < stop; j += G) atomic_add_agent(deg + ri[j], -one);
                    if (g == 0) x[col] = xi;
                    asm volatile("" ::: "memory");
                    done = true;
                }
            }
        } while (__any(!done));
    });
}

// ---------------------------------------------------------------- adjoint
// grad_b = L^{-T} g: the CSC executor's BACKWARD mode
// (spts_syncfree_cuda2.h:50-55, :70-76) applied to the CSR of L read as the
// CSC of L^T, at thread granularity: one lane per node i (tickets taken in
// descending i), write-first so lanes of one wave never block each other.
// cnt[c] counts the off-diagonal entries of column c of L still unapplied.
// The same lane writes grad_val[j] = -grad_b[i] * x[col_j] for its row.
__global__ void __launch_bounds__(kBlock)
    k_adjoint(const int *__restrict__ rp, const int *__restrict__ ci, const double *__restrict__ val,
              const double *__restrict__ g, const double *__restrict__ xfwd, int *__restrict__ cnt,
              double *__restrict__ left_sum, double *__restrict__ grad_b, double *__restrict__ grad_val, int n,
              SyncCtx sc, unsigned *__restrict__ ticket)
{
    ticket_loop(ticket, kBlock, n, [&](int base) {
        const int t = base + threadIdx.x;
        if (t >= n) return;
        const int i = n - 1 - t;
        const int a = rp[i], d = rp[i + 1] - 1;
        const double gi = g[i], vd = val[d];  // before the wait, off the critical path
        Idle idle;
        bool done = false;
        do {  // wave-uniform exit, as in wrtfst_row
            if (!done) {
                const bool ready = ld_agent(cnt + i) == 0;
                const bool failed = !ready && give_up(sc, idle);
                if (ready || failed) {
                    // ordered as in k_csc: left_sum read with an agent-scope
                    // load after the count was seen; the count decrements
                    // depend on the returned left-sum atomics
                    const double ls = as_val(ld_agent(reinterpret_cast<const unsigned long long *>(left_sum) + i));
                    const double y = failed ? as_val(VBits<double>::kQNaN) : (gi - ls) / vd;
                    grad_b[i] = y;
                    double token = 0.0;
                    for (int j = a; j < d; ++j)
                        token += __hip_atomic_fetch_add(left_sum + ci[j], y * val[j], __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
                    int one = 1;
                    asm volatile("" : "+v"(one) : "v"(token));
                    for (int j = a; j < d; ++j) atomic_add_agent(cnt + ci[j], -one);
                    if (grad_val)
                        for (int j = a; j <= d; ++j) grad_val[j] = -y * xfwd[ci[j]];
                    asm volatile("" ::: "memory");
                    done = true;
                }
            }
        } while (__any(!done));
    });
}

// grad_val[j] = -grad_b[row_j] * x[col_j] over the stored pattern (gather
// adjoint; the scatter adjoint fuses this into k_adjoint).  A workgroup takes
// kBlock rows and goes over their entries one to a thread, so that columns
// are read and gradients written in one run; an entry's row is found among
// the rows' starts in LDS.  (A thread per row, its entries one after another:
// 24.8 us for 1,000,000 rows of 2.2 entries, now 18.6.)
__global__ void __launch_bounds__(kBlock)
    k_grad_val(const int *__restrict__ rp, const int *__restrict__ ci, const double *__restrict__ grad_b,
               const double *__restrict__ x, double *__restrict__ grad_val, int n)
{
    __shared__ int start[kBlock + 1];
    __shared__ double y[kBlock];
    const int lo = (int)blockIdx.x * kBlock, rows = min(kBlock, n - lo), t = (int)threadIdx.x;
    if (t < rows) {
        start[t] = rp[lo + t];
        y[t] = grad_b[lo + t];
    }
    if (t == 0) start[rows] = rp[lo + rows];
    __syncthreads();
    // unsigned: past the last entry of a matrix of nearly 2^31 the next e still is
    for (unsigned e = (unsigned)start[0] + t, end = (unsigned)start[rows]; e < end; e += kBlock) {
        int r = 0;  // the last row that starts at or before e
#pragma unroll
        for (int step = kBlock / 2; step > 0; step /= 2)
            if (r + step < rows && (unsigned)start[r + step] <= e) r += step;
        grad_val[e] = -y[r] * x[ci[e]];
    }
}

// off-diagonal column counts of L (the adjoint's in-degrees)
__global__ void __launch_bounds__(kBlock)
    k_offdiag_colcount(const int *__restrict__ rp, const int *__restrict__ ci, int n, int *__restrict__ cnt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int d = rp[i + 1] - 1;
    for (int j = rp[i]; j < d; ++j) atomic_add_agent(cnt + ci[j], 1);
}

// r = b - L x in FP64 (rows in CSR order, fused multiply-add chain), written
// as FP32 for the next correction solve; also max|x| for the convergence
// test.  Grid-stride over the n*k (row, right-hand side) pairs.
__global__ void __launch_bounds__(kBlock)
    k_residual32(const int *__restrict__ rp, const int *__restrict__ ci, const double *__restrict__ val,
                 const double *__restrict__ b, const double *__restrict__ x, float *__restrict__ r32, int n, int k,
                 unsigned long long *__restrict__ xmax_bits)
{
    const long long count = (long long)n * k;
    const long long stride = (long long)gridDim.x * blockDim.x;
    unsigned long long m = 0;
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < count; g += stride) {
        const int i = (int)(g / k), q = (int)(g - (long long)i * k);
        double s = 0.0;
        for (int j = rp[i]; j < rp[i + 1]; ++j) s = __builtin_fma(val[j], x[(long long)ci[j] * k + q], s);
        r32[g] = (float)(b[g] - s);
        const unsigned long long a = (unsigned long long)__double_as_longlong(fabs(x[g]));
        m = a > m ? a : m;
    }
    block_max_to(m, xmax_bits);
}

// r = b - L x in FP64 (one right-hand side, fma chain in CSR order) and
// max|x|: the residual of a refinement whose corrections are FP64 solves.
__global__ void __launch_bounds__(kBlock)
    k_residual64(const int *__restrict__ rp, const int *__restrict__ ci, const double *__restrict__ val,
                 const double *__restrict__ b, const double *__restrict__ x, double *__restrict__ r, int n, int k,
                 unsigned long long *__restrict__ xmax_bits)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    unsigned long long m = 0;
    // g = row * k + RHS: the k threads of a row read its entries together
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < (long long)n * k; g += stride) {
        const int i = (int)(g / k), q = (int)(g % k);
        double s = 0.0;
        for (int j = rp[i]; j < rp[i + 1]; ++j) s = __builtin_fma(val[j], x[(long long)ci[j] * k + q], s);
        r[g] = b[g] - s;
        const unsigned long long a = (unsigned long long)__double_as_longlong(fabs(x[g]));
        m = a > m ? a : m;
    }
    block_max_to(m, xmax_bits);
}

// x += d (FP64 correction) and max|d| (grid-stride)
__global__ void __launch_bounds__(kBlock)
    k_accumulate64(double *__restrict__ x, const double *__restrict__ d, long long count,
                   unsigned long long *__restrict__ dmax_bits)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    unsigned long long m = 0;
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < count; g += stride) {
        x[g] += d[g];
        const unsigned long long a = (unsigned long long)__double_as_longlong(fabs(d[g]));
        m = a > m ? a : m;
    }
    block_max_to(m, dmax_bits);
}

// x += d (FP32 correction) and max|d| for the convergence test (grid-stride)
__global__ void __launch_bounds__(kBlock)
    k_accumulate(double *__restrict__ x, const float *__restrict__ dcor, long long count,
                 unsigned long long *__restrict__ dmax_bits, int first)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    unsigned long long m = 0;
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < count; g += stride) {
        const double dv = (double)dcor[g];
        x[g] = first ? dv : x[g] + dv;
        const unsigned long long a = (unsigned long long)__double_as_longlong(fabs(dv));
        m = a > m ? a : m;
    }
    block_max_to(m, dmax_bits);
}

__global__ void k_cast_f32(const double *__restrict__ a, float *__restrict__ o, long long count)
{
    const long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g < count) o[g] = (float)a[g];
}

// dst row n-1-i = src row i (k interleaved values per row): an upper
// triangular plan solves the row- and column-reversed (lower) matrix
template <typename T>
__global__ void __launch_bounds__(kBlock) k_reverse_rows(const T *__restrict__ src, T *__restrict__ dst, int n, int k)
{
    const long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= (long long)n * k) return;
    const int i = (int)(g / k), q = (int)(g - (long long)i * k);
    dst[(long long)(n - 1 - i) * k + q] = src[g];
}

// Batch: local column indices -> columns of the block-diagonal matrix
// (matrix of each row found by binary search over row_off).
__global__ void __launch_bounds__(kBlock)
    k_globalize(const int *__restrict__ row_off, int n_mat, const int *__restrict__ rp,
                const int *__restrict__ ci_local, int n, int *__restrict__ ci)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int lo = 0, hi = n_mat - 1;
    while (lo < hi) {  // largest m with row_off[m] <= i
        const int mid = (lo + hi + 1) >> 1;
        if (row_off[mid] <= i) lo = mid;
        else hi = mid - 1;
    }
    const int off = row_off[lo];
    for (int j = rp[i]; j < rp[i + 1]; ++j) ci[j] = ci_local[j] + off;
}

// ------------------------------------------------ partitioned banded solve
// For deep matrices whose lower bandwidth w = max(i - col) is at most the
// tail width W (the dependency chain is ~n/levels rows long and no row order
// can shorten it).  Rows are cut into P blocks of m >= W rows; block p's
// rows only reach back into the last W rows of block p-1, its history.  A
// solve sweeps all blocks at once, twice: first with the history 0, for the
// block's last W values a_p, and then, with the blocks' true tails t_p at
// hand, from t_{p-1}, for x.  In between the tails are joined,
//   t_p = a_p + B_p t_{p-1},
// with column c of B_p the tail that block p has for b = 0 and the unit
// vector e_c as its history (W sweeps, once per plan).
// The second sweep reads the rows again instead of adding V_p t_{p-1} with a
// stored V_p (n x W): 4.2 KB per 8 rows at 38 entries against 8 KB, and V
// takes no memory (half a gigabyte at n = 500,000).
// The join is a walk (k_part_walk) where the plan finds that a block damps
// its history, else a scan of the recurrence over the Q = P - 1 tails in two
// levels: in groups of gs consecutive tails sequentially (u_p from the
// group's first tail on), then over the group carries T_g in ceil(log2 G)
// rounds, then every tail is fixed up with its in-group product W_p = B_p
// ... B_first: t_p = u_p + W_p T_{g-1}.  The matrix products are formed once
// per plan (k_part_gemm); a solve only touches vectors.  The sums are
// reassociated, so results match the sequential solve to rounding, not bit
// for bit.  The tail width W (128 or 256) is the smallest of those at least
// the matrix's lower bandwidth; blocks hold at least W rows.  Matrices are
// column-major W x W (element (c, k) at k * W + c).  The tables and the
// solve's work vectors are FP64 for FP32 plans too: b is widened when a sweep
// reads it and x rounded once when it is written.
constexpr int kPartW = 128;     // the narrower tail width
constexpr int kPartWMax = 256;  // the wider one

// A double moved between lanes by DPP (the GFX9 DPP set).  Lanes whose
// source lies outside their row read 0 (bound_ctrl); lanes in rows outside
// ROW_MASK are left undefined (no old value to set up: two moves fewer per
// step).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_d(double v)
{
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)u, CTRL, ROW_MASK, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), CTRL, ROW_MASK, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Each v[q] summed over groups of 8 lanes, in all 8 of them: butterflies by
// quad_perm [1,0,3,2], quad_perm [2,3,0,1] and row_half_mirror (lane i and
// 7 - i of each half row).  Each lane adds the same two halves, in either
// order, so all 8 hold the same bits.  (Step by step for all q: one after
// another their chains do not overlap.)
template <int K>
__device__ __forceinline__ void part_sum8(double (&v)[K])
{
#pragma unroll
    for (int q = 0; q < K; ++q) v[q] += dpp_d<0xB1, 0xf>(v[q]);
#pragma unroll
    for (int q = 0; q < K; ++q) v[q] += dpp_d<0x4E, 0xf>(v[q]);
#pragma unroll
    for (int q = 0; q < K; ++q) v[q] += dpp_d<0x141, 0xf>(v[q]);
}

// v plus the other of its pair of rows of 16 lanes (or of halves of 32)
template <bool HALVES>
__device__ __forceinline__ double part_swap_add(double v)
{
    const unsigned long long u = as_bits(v);
    const unsigned l = (unsigned)u, h = (unsigned)(u >> 32);
    const auto lo = HALVES ? __builtin_amdgcn_permlane32_swap(l, l, false, false)
                           : __builtin_amdgcn_permlane16_swap(l, l, false, false);
    const auto hi = HALVES ? __builtin_amdgcn_permlane32_swap(h, h, false, false)
                           : __builtin_amdgcn_permlane16_swap(h, h, false, false);
    return as_val((unsigned long long)hi[0] << 32 | lo[0]) + as_val((unsigned long long)hi[1] << 32 | lo[1]);
}

// Each v[q] summed over the 8 lanes with the same lane mod 8, in all of them:
// row_ror:8, then the rows of 16 lanes and the halves of 32 swapped.
template <int K>
__device__ __forceinline__ void part_sum_across(double (&v)[K])
{
#pragma unroll
    for (int q = 0; q < K; ++q) v[q] += dpp_d<0x128, 0xf>(v[q]);
#pragma unroll
    for (int q = 0; q < K; ++q) v[q] = part_swap_add<false>(v[q]);
#pragma unroll
    for (int q = 0; q < K; ++q) v[q] = part_swap_add<true>(v[q]);
}

// v of lane `src` (0..63, may differ per lane; every lane active), through
// the LDS crossbar (ds_bpermute): no LDS memory and no VALU work
__device__ __forceinline__ double lane_read(double v, int src)
{
    const long long u = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_ds_bpermute(src * 4, (int)u);
    const int hi = __builtin_amdgcn_ds_bpermute(src * 4, (int)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ float lane_read(float v, int src)
{
    return __int_as_float(__builtin_amdgcn_ds_bpermute(src * 4, __float_as_int(v)));
}

// A record holds up to 8 consecutive rows of one block for one step of a
// wavefront.  Its 64 lanes are 8 segments of 8; a segment takes up to 8 J
// entries of one row in columns before the record's first row r0 (entry e in
// lane e mod 8), so a longer row has several.  The entries inside the record
// are in M, the inverse of the rows' 8 x 8 triangle, a column per segment:
//   y_j = sum over segments u of M[j][u] (b_u - S_u),
// S_u the segment's sum of value * earlier value, b_u its row's b (0 in a
// row's further segments).  In lane 8 u + j: M[j][u], the lane's J values, r0
// - 1 - column per entry in a byte (columns reach back at most W <= 256 rows),
// and 16 bits: the segment's row in the record, flags for a further segment
// and for a segment without entries, the record's row count, and how many
// rows on the record kPartAhead records later starts (the sweep loads that
// far ahead).  Unused entries repeat a column of their row with the value 0:
// they read no value that the row does not depend on.
// NP = J / 2 + 1 pieces of 16 bytes per lane; piece i of record r at
// (r * NP + i) * 64 + lane.
constexpr int kPartSeg = 8;      // segments, and rows at most, of a record
constexpr int kPartAhead = 6;    // records loaded ahead
constexpr int kPartMaxJ = 6;     // J is 2, 4 or 6
constexpr int kPartWaves = 4;    // wavefronts of a sweep's workgroup, at most
constexpr unsigned kPartFurther = 8u, kPartEmpty = 16u;
constexpr int part_pieces(int J) { return J / 2 + 1; }

// The records of a plan, one wavefront each.  rows[r]: record r's first row
// (one entry more than records); at[p]: block p's first record.
template <int J, typename T>
__global__ void __launch_bounds__(kWave)
    k_part_records(const int *__restrict__ rp, const int *__restrict__ ci, const T *__restrict__ val,
                   const int *__restrict__ rows, const int *__restrict__ at, int m, uint4 *__restrict__ rec)
{
    constexpr int S = kPartSeg;
    __shared__ double tri[S][S], inv[S][S], vals[kWave][J];
    __shared__ unsigned dist[kWave][J];
    __shared__ int out[S], seg0[S + 1];
    const int r = (int)blockIdx.x, lane = (int)threadIdx.x, u = lane / S, j = lane % S;
    const int r0 = rows[r], count = rows[r + 1] - r0;
    tri[u][j] = inv[u][j] = 0.0;
#pragma unroll
    for (int s = 0; s < J; ++s) vals[lane][s] = 0.0;
    __syncthreads();
    if (lane < count) {
        int n_out = 0;
        for (int e = rp[r0 + lane]; e < rp[r0 + lane + 1]; ++e) {
            if (ci[e] < r0)
                ++n_out;
            else
                tri[lane][ci[e] - r0] += (double)val[e];  // duplicated entries add up
        }
        out[lane] = n_out;
    }
    __syncthreads();
    if (lane == 0) {
        int s = 0;
        for (int i = 0; i < count; ++i) {
            seg0[i] = s;
            s += max(1, (out[i] + S * J - 1) / (S * J));
        }
        seg0[count] = s;
    }
    if (lane < count) {  // column `lane` of the inverse
        for (int i = lane; i < count; ++i) {
            double s = i == lane ? 1.0 : 0.0;
            for (int l = lane; l < i; ++l) s = __builtin_fma(-tri[i][l], inv[l][lane], s);
            inv[i][lane] = s / tri[i][i];
        }
    }
    __syncthreads();
    int row = -1;
    for (int i = 0; i < count; ++i)
        if (u >= seg0[i] && u < seg0[i + 1]) row = i;
    unsigned flags = kPartFurther | kPartEmpty, pad = 0;
    if (row >= 0) {
        const int h = u - seg0[row];
        flags = (unsigned)row | (h > 0 ? kPartFurther : 0u) | (out[row] == 0 ? kPartEmpty : 0u);
        int idx = 0;
        for (int e = rp[r0 + row]; e < rp[r0 + row + 1]; ++e) {
            if (ci[e] >= r0) continue;
            if (idx == 0) pad = (unsigned)(r0 - 1 - ci[e]);
            if (idx / (S * J) == h && idx % S == j) {
                vals[lane][idx / S % J] = (double)val[e];
                dist[lane][idx / S % J] = (unsigned)(r0 - 1 - ci[e]) + 1u;
            }
            ++idx;
        }
        // the slots past the segment's last entry
        for (int s = 0; s < J; ++s)
            if ((h * J + s) * S + j >= idx) dist[lane][s] = pad + 1u;
    } else {
        for (int s = 0; s < J; ++s) dist[lane][s] = 1u;
    }
    const int last = at[r0 / m + 1];
    const unsigned ahead = r + kPartAhead < last ? (unsigned)(rows[r + kPartAhead] - r0) : 0u;
    flags |= (unsigned)count << 5 | ahead << 9;
    uint4 *o = rec + (long long)r * part_pieces(J) * kWave + lane;
#pragma unroll
    for (int s = 0; s < J; s += 2) {
        const unsigned long long a = as_bits(vals[lane][s]), b = as_bits(vals[lane][s + 1]);
        o[s / 2 * kWave] = make_uint4((unsigned)a, (unsigned)(a >> 32), (unsigned)b, (unsigned)(b >> 32));
    }
    unsigned w[2] = {0u, flags << 16};
#pragma unroll
    for (int s = 0; s < J; ++s) w[s / 4] |= (dist[lane][s] - 1u) << (8 * (s % 4));
    const unsigned long long mm = as_bits(row >= 0 ? inv[j][row] : 0.0);
    o[J / 2 * kWave] = make_uint4((unsigned)mm, (unsigned)(mm >> 32), w[0], w[1]);
}

// What a sweep is for: the tails a_p of history 0 (and of each the bits of the
// largest magnitude, a NaN's above all, and of the smallest: top[2i],
// top[2i + 1]), the B_p (right-hand side q's history is e_q and b is 0), or x
// from the tails t.
enum PartSweep { kPartTails, kPartUnit, kPartX };

// One wavefront per block and KR right-hand sides (b and x interleaved, k per
// row), a record per step; a workgroup's wavefronts have right-hand sides of
// one block, so that the others find in L1 the records that one has loaded.  The block's latest values are in an LDS ring of
// 2W slots, KR values each.  A step's chain is: the ring's values read (J per
// lane), their sum over the segment's 8 lanes, b - S times M, the sum over
// the 8 segments, the ring's slots written: 0.2 us for 8 rows (0.33 and 0.5
// with 2 and 4 right-hand sides per wavefront), where a row at a time took
// 0.2 us a row.  So the rows' bytes bound it, with records loaded kPartAhead
// steps early: 42 and 46 us for the 250 MB of n = 500,000 at 38 entries a row
// (97 us for a row at a time in 384 MB of padded rows, and 92 for V's 512 MB).
// Products with a zero of M are left out: a row's infinity or NaN reaches
// only the rows that depend on it.
// Every right-hand side gets the same bits whatever KR.
template <int W, int KR, int J, typename T, PartSweep MODE>
__global__ void __launch_bounds__(kPartWaves * kWave)
    k_part_sweep(const uint4 *__restrict__ rec, const int *__restrict__ at, const uint2 *__restrict__ first,
                 const T *b, const double *__restrict__ hist, double *__restrict__ tails,
                 unsigned long long *__restrict__ top, T *x, int n, int m, int k, int blocks)
{
    constexpr int D = kPartAhead, NP = part_pieces(J), kMask = 2 * W - 1, kRec = NP * kWave * 16;
    const int p = (int)blockIdx.x + (MODE == kPartUnit ? 1 : 0);
    if ((int)blockIdx.x >= blocks) return;
    __shared__ double rings[kPartWaves][2 * W + 1][KR];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
    double (&ring)[2 * W + 1][KR] = rings[wave];  // the last slot: 0
    const int lane = (int)threadIdx.x % kWave, j = lane & 7;
    const int q0 = ((int)blockIdx.y * ((int)blockDim.x / kWave) + wave) * KR;
    const int start = p * m, rows = min(n - start, m);
    const int r_at = at[p], n_rec = at[p + 1] - r_at;
#pragma unroll
    for (int c = lane; c < W; c += kWave) {
#pragma unroll
        for (int q = 0; q < KR; ++q) {
            double v = 0.0;
            if (MODE == kPartUnit) v = c == q0 + q ? 1.0 : 0.0;
            if (MODE == kPartX && p > 0) v = hist[((long long)(p - 1) * k + q0 + q) * W + c];
            ring[c][q] = 0.0;
            ring[W + c][q] = v;
        }
    }
    if (lane < KR) ring[2 * W][lane] = 0.0;
    const unsigned row_bytes = (unsigned)(k * sizeof(T)), lane16 = 16u * (unsigned)lane;
    const unsigned span = (unsigned)rows * row_bytes - (unsigned)(q0 * sizeof(T));
    const Rsrc rt = make_rsrc(rec + (long long)r_at * NP * kWave, (unsigned)n_rec * kRec);
    // records past the block's last read as 0: no rows, and nothing is stored
    const long long at_b = uniform((long long)start * k + q0);
    const Rsrc rb = make_rsrc(b + at_b, span), rx = make_rsrc(x + at_b, span);
    Words4 st[D][NP];
    T bs[D][KR];
    auto fetch = [&](int d, int at_rec, unsigned row) {
#pragma unroll
        for (int i = 0; i < NP; ++i)
            st[d][i] = __builtin_amdgcn_raw_buffer_load_b128(rt, (int)(lane16 + (unsigned)(at_rec * kRec + i * kWave * 16)),
                                                             0, 0);
        if (MODE != kPartUnit) {
#pragma unroll
            for (int q = 0; q < KR; ++q)
                load_value(rb, (row + (unsigned)j) * row_bytes, (unsigned)(q * sizeof(T)), &bs[d][q]);
        }
    };
    {
        const uint2 f = first[p];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            fetch(d, d, ((d < 4 ? f.x : f.y) >> (8 * (d % 4))) & 255u);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // What the chain needs of a record, worked out during the record before:
    // the ring slots its entries read (a segment without entries reads the
    // zero slot), the segment's b, M, whether M is 0, the slot it writes, its
    // place in x and its rows.
    struct Stage {
        int slot[J], own, count;
        unsigned ahead, at_x;
        double mm, bu[KR];
        bool none;
    };
    auto decode = [&](int d, int lr) {
        Stage w;
        const Words4 head = st[d][NP - 1];
        const unsigned flags = head.w >> 16;
        const unsigned uni = (unsigned)__builtin_amdgcn_readfirstlane((int)flags);
        w.count = (int)(uni >> 5 & 15u);
        w.ahead = uni >> 9;
#pragma unroll
        for (int s = 0; s < J; ++s) {
            const int back = (int)((s < 4 ? head.z : head.w) >> (8 * (s % 4)) & 255u);
            w.slot[s] = (flags & kPartEmpty) ? 2 * W : (lr - 1 - back) & kMask;
        }
        w.own = (lr + j) & kMask;
        w.at_x = lane < w.count ? (unsigned)(lr + j) * row_bytes : 0x80000000u;  // else dropped
        w.mm = as_val((unsigned long long)head.y << 32 | head.x);
        w.none = w.mm == 0.0;
#pragma unroll
        for (int q = 0; q < KR; ++q) {
            w.bu[q] = 0.0;
            if (MODE != kPartUnit) {
                const double t = (double)lane_read(bs[d][q], (int)(flags & 7u));
                w.bu[q] = (flags & kPartFurther) ? 0.0 : t;
            }
        }
        return w;
    };
    int lr = 0;  // the record's first row in the block
    Stage now = decode(0, 0);
    for (int r0 = 0; r0 < n_rec; r0 += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            double sum[KR][2];
#pragma unroll
            for (int q = 0; q < KR; ++q) sum[q][0] = sum[q][1] = 0.0;
#pragma unroll
            for (int s = 0; s < J; ++s) {
                const Words4 w = st[d][s / 2];
                const double v = s & 1 ? as_val((unsigned long long)w.w << 32 | w.z)
                                       : as_val((unsigned long long)w.y << 32 | w.x);
#pragma unroll
                for (int q = 0; q < KR; ++q) sum[q][s & 1] = __builtin_fma(v, ring[now.slot[s]][q], sum[q][s & 1]);
            }
            const unsigned ahead = (unsigned)lr + now.ahead;
            lr += now.count;
            const Stage next = decode((d + 1) % D, lr);
            double y[KR];
#pragma unroll
            for (int q = 0; q < KR; ++q) y[q] = sum[q][0] + sum[q][1];
            part_sum8(y);
#pragma unroll
            for (int q = 0; q < KR; ++q) y[q] = now.none ? 0.0 : now.mm * (now.bu[q] - y[q]);
            part_sum_across(y);
            // every lane writes (those of a row the same value): the slots of
            // the rows past the record's are the next record's
#pragma unroll
            for (int q = 0; q < KR; ++q) ring[now.own][q] = y[q];
            if (MODE == kPartX) {
#pragma unroll
                for (int q = 0; q < KR; ++q) store_value(rx, now.at_x, (unsigned)(q * sizeof(T)), (T)y[q]);
            }
            now = next;
            // the loads neither before M's last use (they take its registers)
            // nor later than here
            __builtin_amdgcn_sched_barrier(0);
            fetch(d, r0 + d + D, ahead);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (MODE != kPartX) {  // the block's last W values: blocks of m >= W rows
        const long long out = MODE == kPartUnit ? p - 1 : p;
        unsigned long long big[KR], low[KR];
#pragma unroll
        for (int q = 0; q < KR; ++q) {
            big[q] = 0;
            low[q] = ~0ull;
        }
#pragma unroll
        for (int c = lane; c < W; c += kWave) {
#pragma unroll
            for (int q = 0; q < KR; ++q) {
                const double v = ring[(m - W + c) & kMask][q];
                tails[(out * k + q0 + q) * W + c] = v;
                const unsigned long long u = as_bits(v) & ~(1ull << 63);
                big[q] = max(big[q], u);
                low[q] = min(low[q], u);
            }
        }
        if (MODE == kPartTails) {
#pragma unroll
            for (int q = 0; q < KR; ++q) {
#pragma unroll
                for (int s = 1; s < kWave; s *= 2) {
                    big[q] = max(big[q], (unsigned long long)__shfl_xor((long long)big[q], s));
                    low[q] = min(low[q], (unsigned long long)__shfl_xor((long long)low[q], s));
                }
                if (lane == 0) {
                    top[2 * (out * k + q0 + q)] = big[q];
                    top[2 * (out * k + q0 + q) + 1] = low[q];
                }
            }
        }
    }
}

// Plan-time matrix products C = A * B of the partition's W x W tables:
// ops[i] = {C, A, B} as matrix indices into bm (B < 0: C = A, a copy), one
// per blockIdx.x, each split into (W / 128)^2 quadrants of 128 x 128 by
// blockIdx.y.  Each of the 256 threads owns an 8 x 8 tile of its quadrant;
// the inner dimension is staged through LDS 16 at a time.
template <int W>
__global__ void __launch_bounds__(256) k_part_gemm(const int3 *__restrict__ ops, double *__restrict__ bm)
{
    constexpr long long kMat = (long long)W * W;
    constexpr int kQ = 128, kQn = W / kQ;
    const int3 op = ops[blockIdx.x];
    const double *A = bm + (long long)op.y * kMat;
    double *C = bm + (long long)op.x * kMat;
    const int t = threadIdx.x;
    const int qr = (int)blockIdx.y % kQn * kQ, qc = (int)blockIdx.y / kQn * kQ;  // quadrant: rows, columns
    if (op.z < 0) {  // copy (uniform) of the quadrant
        for (int e = t; e < kQ * kQ; e += 256) {
            const long long o = (long long)(qc + e / kQ) * W + qr + e % kQ;
            C[o] = A[o];
        }
        return;
    }
    const double *B = bm + (long long)op.z * kMat;
    __shared__ double sa[16][kQ];  // A(qr + c, j0 + jj)
    __shared__ double sb[16][kQ];  // B(j0 + jj, qc + k)
    const int c0 = (t & 15) * 8, k0 = (t >> 4) * 8;
    double acc[8][8];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 8; ++b) acc[a][b] = 0.0;
    for (int j0 = 0; j0 < W; j0 += 16) {
        __syncthreads();
        for (int e = t; e < 16 * kQ; e += 256) {
            sa[e / kQ][e % kQ] = A[(long long)(j0 + e / kQ) * W + qr + e % kQ];
            sb[e % 16][e / 16] = B[(long long)(qc + e / 16) * W + j0 + e % 16];
        }
        __syncthreads();
#pragma unroll 4
        for (int jj = 0; jj < 16; ++jj) {
            double av[8], bv[8];
#pragma unroll
            for (int a = 0; a < 8; ++a) av[a] = sa[jj][c0 + a];
#pragma unroll
            for (int b = 0; b < 8; ++b) bv[b] = sb[jj][k0 + b];
#pragma unroll
            for (int a = 0; a < 8; ++a)
#pragma unroll
                for (int b = 0; b < 8; ++b) acc[a][b] = __builtin_fma(av[a], bv[b], acc[a][b]);
        }
    }
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 8; ++b) C[(long long)(qc + k0 + b) * W + qr + c0 + a] = acc[a][b];
}

// y_j = M v_j for one W x W column-major M and KQ vectors v_j in LDS:
// thread c returns row c of each (four partial sums, by index mod 4, in the
// same order for every KQ, so a right-hand side gets the same bits whichever
// chunk it is solved in).  M is read once for all KQ vectors.
template <int W, int KQ, bool NT>
__device__ __forceinline__ void part_matvec(const double *__restrict__ M, const double (*sv)[W], int c,
                                            double (&out)[KQ])
{
    double d[KQ][4];
#pragma unroll
    for (int j = 0; j < KQ; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) d[j][u] = 0.0;
    constexpr int kUnroll = KQ >= 8 ? 2 : 8;
#pragma unroll kUnroll
    for (int kk = 0; kk < W; kk += 4) {
        double mv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            mv[u] = NT ? __builtin_nontemporal_load(M + (long long)(kk + u) * W + c) : M[(long long)(kk + u) * W + c];
#pragma unroll
        for (int j = 0; j < KQ; ++j)
#pragma unroll
            for (int u = 0; u < 4; ++u) d[j][u] = __builtin_fma(mv[u], sv[j][kk + u], d[j][u]);
    }
#pragma unroll
    for (int j = 0; j < KQ; ++j) out[j] = (d[j][0] + d[j][1]) + (d[j][2] + d[j][3]);
}

// The part of y_j = M v_j that columns k0 .. k0 + KLEN - 1 of M contribute,
// for row c (four partial sums by index mod 4, joined as in part_matvec).
template <int W, int KQ, int KLEN, bool NT>
__device__ __forceinline__ void part_matvec_cols(const double *__restrict__ M, const double (*sv)[W], int c, int k0,
                                                 double (&out)[KQ])
{
    double d[KQ][4];
#pragma unroll
    for (int j = 0; j < KQ; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) d[j][u] = 0.0;
#pragma unroll 4
    for (int kk = k0; kk < k0 + KLEN; kk += 4) {
        double mv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            mv[u] = NT ? __builtin_nontemporal_load(M + (long long)(kk + u) * W + c) : M[(long long)(kk + u) * W + c];
#pragma unroll
        for (int j = 0; j < KQ; ++j)
#pragma unroll
            for (int u = 0; u < 4; ++u) d[j][u] = __builtin_fma(mv[u], sv[j][kk + u], d[j][u]);
    }
#pragma unroll
    for (int j = 0; j < KQ; ++j) out[j] = (d[j][0] + d[j][1]) + (d[j][2] + d[j][3]);
}

// The scan kernels that split a product's columns into kPartSplit quarters
// (one thread per row and quarter) and join the partial sums in LDS.
constexpr int kPartSplit = 4;

// The scan's vectors hold k right-hand sides: tail p of RHS q at (p * k + q)
// * W.  A workgroup takes the KQ right-hand sides from blockIdx.y * KQ;
// part_vec gives the j-th of them.
template <int W, int KQ>
__device__ __forceinline__ long long part_vec(int p, int k, int j)
{
    return ((long long)p * k + (long long)blockIdx.y * KQ + j) * W;
}

// Level 1 of the tail scan, one workgroup of kPartSplit x W threads per
// group of `gs` consecutive tails and chunk of KQ right-hand sides: u_first
// = a_first, u_p = a_p + B_p u_{p-1} (B_p at index p - 1 of bm).  The group's
// last u also goes to carry[g].  A step is sequential, so each product is
// split over the columns (thread: row c, quarter kq) to have four times the
// loads in flight; the first W threads own the vectors.  At W = 256 with
// several right-hand sides the workgroup is 16 wavefronts; holding it to 72
// VGPRs (7 waves per SIMD; 36 bytes per lane spill at KQ = 4) lets it share
// a CU with a 1024-thread workgroup of the thread-per-row solve (42 VGPRs)
// or of the fused refinement sweep (52), so a batch's partitioned solve runs
// beside the rest's persistent kernel instead of waiting for it.  Alone it
// is 2 % slower for that (758 against 743 us at 16 right-hand sides,
// n = 160,000).
template <int W, int KQ, bool NT>
__global__ void __launch_bounds__(kPartSplit * W, W >= 256 && KQ >= 2 ? 7 : 1)
    k_part_group_scan(const double *__restrict__ a, double *__restrict__ u, double *__restrict__ carry,
                      const double *__restrict__ bm, int gs, int q_count, int k)
{
    constexpr int kLen = W / kPartSplit;
    const int g = (int)blockIdx.x, t = (int)threadIdx.x, c = t % W, kq = t / W;
    const int p0 = g * gs, p1 = min(q_count, p0 + gs);
    __shared__ double sv[KQ][W];
    __shared__ double red[kPartSplit][KQ][W];
    double v[KQ];
    if (t < W) {
#pragma unroll
        for (int j = 0; j < KQ; ++j) {
            v[j] = a[part_vec<W, KQ>(p0, k, j) + c];
            u[part_vec<W, KQ>(p0, k, j) + c] = v[j];
        }
    }
    for (int p = p0 + 1; p < p1; ++p) {
        __syncthreads();  // the previous product is done with sv and red
        if (t < W) {
#pragma unroll
            for (int j = 0; j < KQ; ++j) sv[j][c] = v[j];
        }
        __syncthreads();
        double mv[KQ];
        part_matvec_cols<W, KQ, kLen, NT>(bm + (long long)(p - 1) * W * W, sv, c, kq * kLen, mv);
#pragma unroll
        for (int j = 0; j < KQ; ++j) red[kq][j][c] = mv[j];
        __syncthreads();
        if (t < W) {
#pragma unroll
            for (int j = 0; j < KQ; ++j) {
                v[j] = a[part_vec<W, KQ>(p, k, j) + c] + ((red[0][j][c] + red[1][j][c]) + (red[2][j][c] + red[3][j][c]));
                u[part_vec<W, KQ>(p, k, j) + c] = v[j];
            }
        }
    }
    if (t < W) {
#pragma unroll
        for (int j = 0; j < KQ; ++j) carry[part_vec<W, KQ>(g, k, j) + c] = v[j];
    }
}

// Level 3: t_p = u_p + W_p T_{g-1} for tails of groups g >= 1 (W_p at index
// p - gs of wm, T the scanned group carries), t_p = u_p in group 0.
template <int W, int KQ, bool NT>
__global__ void __launch_bounds__(W)
    k_part_fixup(const double *__restrict__ u, const double *__restrict__ tg, const double *__restrict__ wm, int gs,
                 double *__restrict__ t, int k)
{
    const int p = (int)blockIdx.x, c = (int)threadIdx.x;
    const int g = p / gs;
    __shared__ double sv[KQ][W];
    double v[KQ];
#pragma unroll
    for (int j = 0; j < KQ; ++j) v[j] = u[part_vec<W, KQ>(p, k, j) + c];
    if (g > 0) {  // uniform in the workgroup
#pragma unroll
        for (int j = 0; j < KQ; ++j) sv[j][c] = tg[part_vec<W, KQ>(g - 1, k, j) + c];
        __syncthreads();
        double mv[KQ];
        part_matvec<W, KQ, NT>(wm + (long long)(p - gs) * W * W, sv, c, mv);
#pragma unroll
        for (int j = 0; j < KQ; ++j) v[j] += mv[j];
    }
#pragma unroll
    for (int j = 0; j < KQ; ++j) t[part_vec<W, KQ>(p, k, j) + c] = v[j];
}


// One round of the log-depth scan over the group carries (kPartSplit
// workgroups of W threads per entry and chunk of KQ right-hand sides,
// each for a quarter of the rows: the round has only G entries, so each
// product is spread over four workgroups; thread: row, quarter of the
// columns, partial sums joined in LDS): dst_g = src_g + M_g src_{g-s} for g >= s (M_g at
// index g - s of the round's matrices), dst_g = src_g below s.
template <int W, int KQ, bool NT>
__global__ void __launch_bounds__(W)
    k_part_scan(const double *__restrict__ src, double *__restrict__ dst, const double *__restrict__ bm, int s, int k)
{
    constexpr int kRows = W / kPartSplit, kLen = W / kPartSplit;
    const int p = (int)blockIdx.x / kPartSplit, part = (int)blockIdx.x % kPartSplit;
    const int t = (int)threadIdx.x, r = t % kRows, kq = t / kRows, c = part * kRows + r;
    __shared__ double sv[KQ][W];
    __shared__ double red[kPartSplit][KQ][kRows];
    if (p >= s) {  // uniform in the workgroup
#pragma unroll
        for (int j = 0; j < KQ; ++j) sv[j][t] = src[part_vec<W, KQ>(p - s, k, j) + t];
        __syncthreads();
        double mv[KQ];
        part_matvec_cols<W, KQ, kLen, NT>(bm + (long long)(p - s) * W * W, sv, c, kq * kLen, mv);
#pragma unroll
        for (int j = 0; j < KQ; ++j) red[kq][j][r] = mv[j];
        __syncthreads();
        if (t < kRows) {
#pragma unroll
            for (int j = 0; j < KQ; ++j)
                dst[part_vec<W, KQ>(p, k, j) + c] = src[part_vec<W, KQ>(p, k, j) + c] +
                                                    ((red[0][j][r] + red[1][j][r]) + (red[2][j][r] + red[3][j][r]));
        }
    } else if (t < kRows) {
#pragma unroll
        for (int j = 0; j < KQ; ++j) dst[part_vec<W, KQ>(p, k, j) + c] = src[part_vec<W, KQ>(p, k, j) + c];
    }
}

// The largest absolute row sum of each B_p (p = 1 + blockIdx.x), rounded up.
template <int W>
__global__ void __launch_bounds__(W) k_part_norm(const double *__restrict__ bm, double *__restrict__ norm)
{
    __shared__ double red[W];
    const int c = (int)threadIdx.x;
    const double *M = bm + (long long)blockIdx.x * W * W;
    double s = 0.0;
    for (int kk = 0; kk < W; ++kk) s += fabs(M[(long long)kk * W + c]);
    red[c] = s;
    __syncthreads();
    if (c == 0) {
        for (int i = 1; i < W; ++i) s = red[i] <= s ? s : red[i];  // a NaN stays or replaces the rest
        norm[blockIdx.x] = s * (1.0 + 1e-9);
    }
}

// The tails by walks, one workgroup of kPartSplit x W threads per run of
// consecutive tails and chunk of KQ right-hand sides.  Used where blocks damp
// their history (four in a row by kPartDamp or more) or are few.  What block p
// - s adds to t_p is at most norm(B_p ... B_{p-s+1}) max|a_{p-s}|; the walk to
// t_p starts at the farthest block for which a bound of that is above
// 2^-(57 + s/2) of the smallest magnitude in a_p and not below the smallest
// double (all the way to that where a_p holds a 0: such a row's value is its
// history alone).  All that is left out then stays below 2^-55.7 of each of
// a_p's values, a sixth of the rounding of t_p's own terms, also where the
// tail's rows belong to systems that do not touch each other: measured against
// the largest magnitude, one huge row of b took the digits of all the others
// in its block's tail (4e-10 of the largest, now 4e-16), and without the
// zeros a system whose right-hand side ended was 0 two blocks later.  The
// smallest is about 9 bits below the largest with a dense right-hand side:
// 18.8 -> 19.6 us at n = 500,000.  How far that is depends on the right-hand
// side alone, so it gets the same bits in every chunk.  Blocks are looked at kPartReach back: there
// the factor has passed 2^-2048, the whole range of a double.  After a block
// with an infinity or a NaN in its tail every tail is NaN (0 times an
// infinity is NaN, and each product has all W columns).
// The bound is taken in logarithms, whole numbers of 1 / 256 rounded up, of
// the norms of four matrices' products, and of single matrices for the rest:
// fade[i].x is the sum of those of B_1 ... B_i, fade[i].y of B_i ... B_{i-3},
// B_{i-4} ... (sums whose differences are right whether or not they wrap).
// Four matrices' product is smaller than their norms' product: 2^-58 against
// 2^-36 at 512 rows of bandwidth 96, which is 5 products to a tail, not 8.
// d[j] += sum over kk of m[kk] times s[j] of lane kk of the 16 lanes' row, in
// two chains by kk mod 2
template <int KK, int KQ>
__device__ __forceinline__ void part_rank(const double (&m)[16], const double (&s)[KQ], double (&d)[KQ][2])
{
    if constexpr (KK < 16) {
#pragma unroll
        for (int j = 0; j < KQ; ++j)
            d[j][KK % 2] = __builtin_fma(
                m[KK], __builtin_amdgcn_update_dpp(0.0, s[j], 0x150 + KK, 0xf, 0xf, true), d[j][KK % 2]);  // row_newbcast
        part_rank<KK + 1, KQ>(m, s, d);
    }
}

constexpr double kPartDamp = 0x1p-32;
constexpr int kPartReach = 4 * kWave;
template <int W, int KQ>
__global__ void __launch_bounds__(kPartSplit * W, W >= 256 && KQ >= 2 ? 7 : 1)
    k_part_walk(const double *__restrict__ a, const unsigned long long *__restrict__ top,
                const double *__restrict__ bm, const uint2 *__restrict__ fade, double *__restrict__ tail,
                int q_count, int run, int k)
{
    constexpr int kLen = W / kPartSplit, kThreads = kPartSplit * W;
    constexpr unsigned long long kInf = 0x7FF0000000000000ULL, kNormal = 0x0010000000000000ULL;
    // neighbours read the same matrices: each of the 8 XCDs, to which
    // workgroups go in turn, takes consecutive runs (gridDim.x is a multiple)
    const int p0 = ((int)blockIdx.x % 8 * ((int)gridDim.x / 8) + (int)blockIdx.x / 8) * run;
    const int p1 = min(q_count, p0 + run);
    if (p0 >= q_count) return;
    const int t = (int)threadIdx.x, c = t % W, kq = t / W, lane = t % kWave, wave = t / kWave;
    __shared__ double sv[KQ][W];
    __shared__ double red[kPartSplit][KQ][W];
    __shared__ int from[KQ], lost[KQ];  // per right-hand side: its walk's start, the first block past repair
    if (t < KQ) {
        from[t] = p0;
        lost[t] = q_count;
    }
    __syncthreads();
    const unsigned long long *tq = top + 2LL * blockIdx.y * KQ;
    for (int h = t; h < p1 - 1; h += kThreads) {
#pragma unroll
        for (int j = 0; j < KQ; ++j)
            if (tq[2 * ((long long)h * k + j)] >= kInf) atomicMin(&lost[j], h);
    }
    // (tail, right-hand side) pairs, one to a wavefront: lane l looks at the
    // blocks l, l + 64, ... back
    for (int e = wave; e < (p1 - p0) * KQ; e += kThreads / kWave) {
        const int p = p0 + e / KQ, j = e % KQ;
        const unsigned long long own = tq[2 * ((long long)p * k + j) + 1];
        int far = 0;
#pragma unroll
        for (int i = 0; i < kPartReach; i += kWave) {
            const int s = i + lane, h = p - s;
            if (s == 0 || h < 0) continue;
            const unsigned long long bits = tq[2 * ((long long)h * k + j)];
            // log2 in 256ths, the exponent biased: above the term's (an
            // exponent and a fraction fall short of it by 0.087 at most)
            const int mid = p - (s & ~3);
            const int term = (int)(bits >> 44) + 24 + (int)(fade[p].y - fade[mid].y) + (int)(fade[mid].x - fade[h].x);
            const int floor = own >= kNormal && own < kInf ? (int)(own >> 44) - 57 * 256 - 128 * s : -60 * 256;
            if (bits != 0 && term > max(floor, -60 * 256)) far = s;
        }
#pragma unroll
        for (int s = 1; s < kWave; s *= 2) far = max(far, __shfl_xor(far, s));
        if (lane == 0) atomicMin(&from[j], p - far);
    }
    __syncthreads();
    int h = p0;
#pragma unroll
    for (int j = 0; j < KQ; ++j) h = min(h, lost[j] < p0 ? p0 : from[j]);
    // A thread has one row and kLen columns of a product, the vectors' values
    // 16 columns at a time, one to a lane: a lane's value goes to its row of
    // 16 by DPP, one LDS read per lane for 16 columns.  At W = 128 the part of
    // the next product's matrix is loaded while the current one is joined.
    // The matrices' bytes bound it: at n = 500,000 (m = 1000, 97 MB) 20 us; at
    // n = 200,000 with 8 right-hand sides (m = 512) 35 us (31 as one chunk and
    // 50 as two of 4 while walks started later).  The scan's launches took 83
    // and 140 (1023 tails).
    constexpr bool kAhead = W == kPartW;
    constexpr int kCols = 16;
    double mat[kAhead ? kLen / kCols : 1][kCols];
    auto load = [&](int p, int g, double (&m)[kCols]) {
        const double *M = bm + ((long long)(p - 1) * W + kq * kLen + g * kCols) * W + c;
#pragma unroll
        for (int kk = 0; kk < kCols; ++kk) m[kk] = M[(long long)kk * W];
    };
    double v[KQ];
#pragma unroll
    for (int j = 0; j < KQ; ++j) v[j] = 0.0;
    for (bool head = true;; head = false) {
        double mv[KQ], ah[KQ];
        if (t < W) {
#pragma unroll
            for (int j = 0; j < KQ; ++j) ah[j] = a[part_vec<W, KQ>(h, k, j) + c];
        }
        if (!head) {
            __syncthreads();  // sv is written, red is read
            double d[KQ][2];
#pragma unroll
            for (int j = 0; j < KQ; ++j) d[j][0] = d[j][1] = 0.0;
#pragma unroll(kAhead ? kLen / kCols : 1)
            for (int g = 0; g < kLen / kCols; ++g) {
                double (&m)[kCols] = mat[kAhead ? g : 0];
                if (!kAhead) load(h, g, m);
                double s[KQ];
#pragma unroll
                for (int j = 0; j < KQ; ++j) s[j] = sv[j][kq * kLen + g * kCols + t % kCols];
                part_rank<0, KQ>(m, s, d);
            }
#pragma unroll
            for (int j = 0; j < KQ; ++j) mv[j] = d[j][0] + d[j][1];
#pragma unroll
            for (int j = 0; j < KQ; ++j) red[kq][j][c] = mv[j];
        }
        if (kAhead && h + 1 < p1) {
#pragma unroll
            for (int g = 0; g < kLen / kCols; ++g) load(h + 1, g, mat[kAhead ? g : 0]);
        }
        if (!head) __syncthreads();
        if (t < W) {
#pragma unroll
            for (int j = 0; j < KQ; ++j) {
                v[j] = ah[j];
                if (!head && h > from[j])
                    v[j] += (red[0][j][c] + red[1][j][c]) + (red[2][j][c] + red[3][j][c]);
                sv[j][c] = v[j];
                if (h >= p0)
                    tail[part_vec<W, KQ>(h, k, j) + c] = lost[j] < h ? as_val(VBits<double>::kQNaN) : v[j];
            }
        }
        if (++h == p1) break;
    }
}

}  // namespace cap
