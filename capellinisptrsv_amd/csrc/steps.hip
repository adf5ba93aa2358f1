// Step solves (see steps.h): schedule, tables and kernel.
#include "steps.h"

#include <algorithm>
#include <cstdint>
#include <new>

#include "../../include/capellini_sptrsv.h"
#include "cap_internal.h"
#include "device_base.h"

namespace cap {

// ---------------------------------------------------------------- layout
// Slot s * block + thread of a job describes the row that thread solves in
// step s, in 16-byte pieces; piece p of the step lies at
// (s * P + p) * block + thread, so a wavefront's loads of a piece are one
// contiguous run.  Pieces: the head {own ring slot | long << 16, start of the
// rest (long rows), and with E = 4 the four entries' ring slots, 16 bits
// each}; with E > 4 the E ring slots, 8 per piece; the E values; {diagonal,
// its reciprocal}.  Unused entries name slot `ring`, which holds +0, with the
// value -0: the sum of s and their product is s for every s, also for the -0
// that a negative product too small for a number leaves.
// Slots a step does not need repeat the step's first row: they compute the
// same value into the same places, so every thread runs the same
// straight-line step and none needs a place to put a result nobody reads.
// The arrays hold kStepTail more steps, copies of the last: the kernel runs
// whole rounds of 2D steps and reads up to 2D ahead.
template <typename T, int E>
struct StepLayout {
    static constexpr int kCols = E > 4 ? E / 8 : 0;
    static constexpr int kVals = E * (int)sizeof(T) / 16;
    static constexpr int P = 1 + kCols + kVals + 1;
};

// Steps of row data in flight.  Each step issues P + 1 + K loads and K stores
// per thread and the load counter holds 63 operations; with 4 entries and
// one right-hand side 10 steps cover the memory latency at 0.13 us a step.
template <int E, int K>
constexpr int step_depth()
{
    return E == 4 ? (K == 4 ? 6 : K == 2 ? 8 : 10) : E == 8 ? (K == 4 ? 4 : 6) : (K == 4 ? 3 : 4);
}

constexpr int kXcds = 8;
constexpr int kStepTail = 40;  // 4 x the largest depth
constexpr int kStepBlock = 256;

// ----------------------------------------------------------- division
// a / d with r = 1 / d at hand, correctly rounded: two corrections of a * r
// by the exactly representable residual (Markstein 1990: a faithful quotient
// corrected once with the correctly rounded reciprocal is the correctly
// rounded quotient; a * r may be two units off, so the first correction makes
// it faithful).  5 dependent operations instead of the 11 of the divide
// sequence, whose reciprocal part does not depend on a.  Valid while nothing
// overflows or loses bits to underflow: |a| within 2^+-500 (FP32: 2^+-60) or
// a = +0, and r is NaN unless |d| is within the same range.  Everything else
// takes the plain division.
template <typename T>
struct DivRange;
template <>
struct DivRange<double> {
    static constexpr unsigned lo = (1023u - 500u) << 20, span = 1000u << 20;
    static __device__ __forceinline__ bool fast(double a)
    {
        const unsigned long long u = as_bits(a);
        return ((unsigned)(u >> 32) & 0x7fffffffu) - lo < span || u == 0;
    }
};
template <>
struct DivRange<float> {
    static constexpr unsigned lo = (127u - 60u) << 23, span = 120u << 23;
    static __device__ __forceinline__ bool fast(float a)
    {
        const unsigned u = as_bits(a);
        return (u & 0x7fffffffu) - lo < span || u == 0;
    }
};
template <typename T>
__device__ __forceinline__ T step_divide(T a, T d, T r)
{
    T q = a * r;
    T e = fmac(-d, q, a);
    q = fmac(e, r, q);
    e = fmac(-d, q, a);
    q = fmac(e, r, q);
    const bool fast = DivRange<T>::fast(a) && q == q;
    if (__builtin_expect(__any(!fast), 0)) {  // a branch of the wavefront: a per-lane one is computed always
        if (!fast) q = a / d;
    }
    return q;
}
// The table's reciprocal of a diagonal.
__device__ __forceinline__ double step_reciprocal(double d)
{
    const unsigned h = (unsigned)(as_bits(d) >> 32) & 0x7fffffffu;
    return h - DivRange<double>::lo < DivRange<double>::span ? 1.0 / d : as_val(VBits<double>::kQNaN);
}
__device__ __forceinline__ float step_reciprocal(float d)
{
    const unsigned h = as_bits(d) & 0x7fffffffu;
    return h - DivRange<float>::lo < DivRange<float>::span ? 1.0f / d : as_val(VBits<float>::kQNaN);
}

// ------------------------------------------------------------- tables
// One thread per slot of one job (blockIdx.y): its pieces from the CSR.
// values_only: the pattern is in place, the caller's values changed.
// spread: one workgroup in so many works (a power of two; 8 keeps them on the
// chiplet of workgroup 0, whose L2 the solve then reads the pieces from).
template <typename T, int E>
__global__ void __launch_bounds__(kBlock)
    k_step_tables(const StepJob *__restrict__ jobs, const unsigned *__restrict__ rows, const int *__restrict__ rp,
                  const int *__restrict__ ci, const T *__restrict__ val, uint4 *__restrict__ tab,
                  const int *__restrict__ ov_at, int *__restrict__ ov_c, T *__restrict__ ov_v, bool values_only, int spread)
{
    typedef StepLayout<T, E> L;
    if (blockIdx.x % spread) return;
    const StepJob job = jobs[blockIdx.y];
    const int count = (job.steps + kStepTail) * job.block;
    for (int s = blockIdx.x / spread * kBlock + threadIdx.x; s < count; s += gridDim.x / spread * kBlock) {
        const int step = s / job.block, t = s % job.block;
        const int row = job.row0 + (int)rows[job.rows + s];
        const int e0 = rp[row], cnt = rp[row + 1] - 1 - e0;
        uint4 *out = tab + job.tab + (size_t)step * L::P * job.block + t;
        const int rest = ov_at ? ov_at[job.rows + s] : -1;
        if (!values_only) {
            unsigned c[E];
#pragma unroll
            for (int u = 0; u < E; ++u)
                c[u] = u < cnt ? (unsigned)(ci[e0 + u] - job.row0) % (unsigned)job.ring : (unsigned)job.ring;
            const unsigned own = (unsigned)(row - job.row0) % (unsigned)job.ring | (rest >= 0 ? 0x10000u : 0u);
            if constexpr (E == 4) {
                out[0] = make_uint4(own, (unsigned)rest, c[0] | c[1] << 16, c[2] | c[3] << 16);
            } else {
                out[0] = make_uint4(own, (unsigned)rest, 0u, 0u);
#pragma unroll
                for (int h = 0; h < L::kCols; ++h)
                    out[(1 + h) * job.block] =
                        make_uint4(c[8 * h] | c[8 * h + 1] << 16, c[8 * h + 2] | c[8 * h + 3] << 16,
                                   c[8 * h + 4] | c[8 * h + 5] << 16, c[8 * h + 6] | c[8 * h + 7] << 16);
            }
            if (rest >= 0) {
                ov_c[rest] = cnt - E;
                for (int u = E; u < cnt; ++u)
                    ov_c[rest + 1 + u - E] = (int)((unsigned)(ci[e0 + u] - job.row0) % (unsigned)job.ring);
            }
        }
        T v[E];
#pragma unroll
        for (int u = 0; u < E; ++u) v[u] = u < cnt ? val[e0 + u] : -(T)0;
#pragma unroll
        for (int h = 0; h < L::kVals; ++h) {
            uint4 w;
            __builtin_memcpy(&w, reinterpret_cast<const char *>(v) + 16 * h, 16);
            out[(1 + L::kCols + h) * job.block] = w;
        }
        T dr[16 / sizeof(T)] = {};
        dr[0] = val[e0 + cnt];
        dr[1] = step_reciprocal(dr[0]);
        uint4 w;
        __builtin_memcpy(&w, dr, 16);
        out[(1 + L::kCols + L::kVals) * job.block] = w;
        if (rest >= 0)
            for (int u = E; u < cnt; ++u) ov_v[rest + 1 + u - E] = val[e0 + u];
    }
}

// ------------------------------------------------------------- kernel
template <typename T, int E, int K>
struct StepStage {
    unsigned own, rest, xo;
    unsigned c[E / 2];
    T v[E], d, r, bo[K];
};

// off: the step's first piece (uniform), t16 = 16 * thread, pb = 16 * block
// bytes from piece to piece; row_bytes: the row's offset in b and x.
template <typename T, int E, int K>
__device__ __forceinline__ void step_load(StepStage<T, E, K> &w, Rsrc tab, unsigned off, unsigned t16, unsigned pb,
                                          Rsrc b, unsigned row_bytes)
{
    typedef StepLayout<T, E> L;
    w.xo = row_bytes;
    const Words4 h = __builtin_amdgcn_raw_buffer_load_b128(tab, (int)t16, (int)off, 0);
    w.own = h.x;
    w.rest = h.y;
    if constexpr (E == 4) {
        w.c[0] = h.z;
        w.c[1] = h.w;
    }
#pragma unroll
    for (int q = 0; q < L::kCols; ++q) {
        const Words4 u = __builtin_amdgcn_raw_buffer_load_b128(tab, (int)t16, (int)(off + (1 + q) * pb), 0);
        w.c[4 * q] = u.x;
        w.c[4 * q + 1] = u.y;
        w.c[4 * q + 2] = u.z;
        w.c[4 * q + 3] = u.w;
    }
#pragma unroll
    for (int q = 0; q < L::kVals; ++q) {
        const Words4 u = __builtin_amdgcn_raw_buffer_load_b128(tab, (int)t16, (int)(off + (1 + L::kCols + q) * pb), 0);
        __builtin_memcpy(reinterpret_cast<char *>(w.v) + 16 * q, &u, 16);
    }
    const Words4 u =
        __builtin_amdgcn_raw_buffer_load_b128(tab, (int)t16, (int)(off + (1 + L::kCols + L::kVals) * pb), 0);
    T dr[16 / sizeof(T)];
    __builtin_memcpy(dr, &u, 16);
    w.d = dr[0];
    w.r = dr[1];
#pragma unroll
    for (int q = 0; q < K; ++q) load_value(b, row_bytes, q * sizeof(T), &w.bo[q]);
}

// One workgroup per job and chunk of K right-hand sides; thread per row of
// the step.  No polling and
// no readiness state: a step costs its LDS reads, the row's chain and one
// barrier inside one compute unit, against the memory round trip of a publish
// -> observe hop between compute units.
//
// The row data is loaded D steps ahead into registers, the row number 2D
// steps ahead (b is gathered through it); the barriers order LDS alone, so
// they do not wait for those loads.  The next step's ring addresses are
// unpacked before the barrier that ends this one.  What bounds it: one
// wavefront's chain of dependent instructions per step (LDS reads, E fused
// multiply-adds, the division, the ring write, the barrier) and the issue of
// its own loads, with nothing else on its SIMD to hide their latency: 60,000
// rows of up to 15 entries, 523 steps of 128 rows: 0.37 us a step, 59 vector,
// 17 LDS and 14 load instructions per wavefront, a tenth of the cycles lost to
// LDS bank conflicts, and 24.6 KB of table a step, 28 bytes a cycle, well
// below what a compute unit loads.
template <typename T, int E, int D, bool UNFUSED, bool LONG, int K>
__global__ void __launch_bounds__(kStepBlock)
    k_step(const StepJob *__restrict__ jobs, int n_jobs, const uint4 *__restrict__ tab,
           const unsigned *__restrict__ rows, const int *__restrict__ ov_c, const T *__restrict__ ov_v,
           const T *__restrict__ b, T *__restrict__ x, int k)
{
    typedef StepLayout<T, E> L;
    typedef T Vals __attribute__((ext_vector_type(K)));  // the K values of a ring slot
    constexpr unsigned kSlot = K * sizeof(T);
    // grid: jobs of a group, chunks, groups.  Workgroup i runs on chiplet i
    // mod 8, so with 8 jobs to a group all chunks of a job share a chiplet,
    // and its L2 the lines of b and x they share
    const int which = blockIdx.z * gridDim.x + blockIdx.x;
    if (which >= n_jobs) return;
    const StepJob job = jobs[which];
    const int q0 = blockIdx.y * K;
    const int B = job.block;
    if ((int)threadIdx.x >= B) return;  // whole wavefronts; barriers count the others
    // the launch's dynamic LDS is all of the kernel's: it starts at address 0
    typedef __attribute__((address_space(3))) Vals LdsVals;
    auto ring = [](unsigned byte) -> LdsVals * { return (LdsVals *)byte; };
    const unsigned t = threadIdx.x, t16 = 16 * t, t4 = 4 * t, pb = 16u * B, kb = (unsigned)(k * sizeof(T));
    const unsigned span = (unsigned)job.rows_of * kb - q0 * (unsigned)sizeof(T);
    const Rsrc rb = make_rsrc(b + (size_t)job.row0 * k + q0, span), rx = make_rsrc(x + (size_t)job.row0 * k + q0, span);
    const unsigned step16 = 16u * L::P * B, step4 = 4u * B;
    // a window of the pieces, moved with the steps: they may be more bytes
    // than a descriptor holds
    auto window = [&](int step) {
        return make_rsrc(tab + uniform((long long)(job.tab + (unsigned long long)step * (L::P * B))), 3 * D * step16);
    };
    Rsrc rt = window(0);
    const Rsrc rr = make_rsrc(rows + job.rows, (unsigned)(job.steps + kStepTail) * step4);
    auto row_at = [&](unsigned off) { return __builtin_amdgcn_raw_buffer_load_b32(rr, (int)t4, (int)off, 0); };
    StepStage<T, E, K> st[D];
    unsigned ahead[D], first[D];
#pragma unroll
    for (int r = 0; r < D; ++r) first[r] = row_at(r * step4);
#pragma unroll
    for (int r = 0; r < D; ++r) ahead[r] = row_at((D + r) * step4);
#pragma unroll
    for (int r = 0; r < D; ++r) step_load<T, E, K>(st[r], rt, r * step16, t16, pb, rb, first[r] * kb);
    if (t == 0) *ring((unsigned)job.ring * kSlot) = Vals(0);
    unsigned at[E];
#pragma unroll
    for (int u = 0; u < E; ++u) at[u] = ((u & 1) ? st[0].c[u / 2] >> 16 : st[0].c[u / 2] & 0xffffu) * kSlot;
    lds_barrier();
    unsigned nrow = 2 * D * step4;  // rows of step s + 2D
    // two rounds of the D stages per iteration: the compiler's load-counter
    // waits are exact in the second round (the first round's, merged at the
    // loop head, assume about half the loads in flight)
    for (int s0 = 0; s0 < job.steps; s0 += 2 * D) {
        rt = window(s0);
        unsigned next = D * step16;  // pieces of step s + D
#pragma unroll
        for (int h = 0; h < 2 * D; ++h) {
            constexpr int kD = D;
            StepStage<T, E, K> &w = st[h % kD];
            T sum[K];
#pragma unroll
            for (int q = 0; q < K; ++q) sum[q] = (T)0;
            // K values per entry; at most 16 values read ahead of the chain
            constexpr int kGroup = K == 1 ? E : K == 2 ? (E < 8 ? E : 8) : 4;
#pragma unroll
            for (int g = 0; g < E; g += kGroup) {
                Vals xv[kGroup];
#pragma unroll
                for (int u = 0; u < kGroup; ++u) xv[u] = *ring(at[g + u]);
#pragma unroll
                for (int u = 0; u < kGroup; ++u)
#pragma unroll
                    for (int q = 0; q < K; ++q)
                        sum[q] = UNFUSED ? sum[q] + w.v[g + u] * xv[u][q] : fmac(w.v[g + u], xv[u][q], sum[q]);
            }
            if (LONG && (w.own & 0x10000u)) {
                const int cnt = ov_c[w.rest];
                for (int u = 0; u < cnt; ++u) {
                    const T a = ov_v[w.rest + 1 + u];
                    const Vals xv = *ring((unsigned)ov_c[w.rest + 1 + u] * kSlot);
#pragma unroll
                    for (int q = 0; q < K; ++q) sum[q] = UNFUSED ? sum[q] + a * xv[q] : fmac(a, xv[q], sum[q]);
                }
            }
            Vals xi;
#pragma unroll
            for (int q = 0; q < K; ++q) xi[q] = step_divide(w.bo[q] - sum[q], w.d, w.r);
            *ring((w.own & 0xffffu) * kSlot) = xi;
#pragma unroll
            for (int q = 0; q < K; ++q) store_value(rx, w.xo, q * sizeof(T), xi[q]);
            // refill this stage for step s + D and its row for step s + 2D,
            // after the step's own work: interleaved with it, the compiler
            // parks in-flight load results in accumulation registers, and
            // each such move waits for its load
            __builtin_amdgcn_sched_barrier(0);
            step_load<T, E, K>(w, rt, next, t16, pb, rb, ahead[h % kD] * kb);
            ahead[h % kD] = row_at(nrow);
            next += step16;
            nrow += step4;
            const StepStage<T, E, K> &n = st[(h + 1) % kD];
#pragma unroll
            for (int u = 0; u < E; ++u) at[u] = ((u & 1) ? n.c[u / 2] >> 16 : n.c[u / 2] & 0xffffu) * kSlot;
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
        }
    }
}

// The same steps, for rows of up to 4 entries and one right-hand side, with
// the loads in wavefronts of their own.  Issuing a step's loads is half of a
// step's time where a wavefront does both (194 ns a step, 99 without its
// loads), and a compute unit has room for more wavefronts.  Thread B + t loads
// what thread t solves: its row data D steps ahead into registers, and two
// steps ahead of the solve from there into one of two LDS buffers; thread t
// reads its next step's data while it solves this one.  A head's unused word
// carries the row's offset in b and x.  Both sides meet at the one barrier
// per step.
// What bounds it: with one solving wavefront its chain (107 ns a step, 159
// with k_step: 24.6 against 34.1 us for n = 2,000 in 193 steps, both without
// the values' copy before it), with more
// the LDS traffic of the steps' data too: 194 / 279 / 333 ns with two, three
// and four (k_step 221 / 303 / 355; n = 100,000 in 807 steps 156 against 178
// us).  With 8 or 16 entries a row the data through LDS costs more than its
// loads (n = 68,170, 7 entries: 163 against 140 us; n = 60,000, 15 entries:
// 231 against 212), and where there are more workgroups than compute units
// the loads of one overlap the chains of the others: those keep k_step.
constexpr int kSplitEntries = 4;
constexpr int kSplitDepth = 10;

template <typename T>
constexpr int split_bytes()  // of a step's data in LDS, per thread
{
    return 16 * StepLayout<T, kSplitEntries>::P + (int)sizeof(T);
}

template <typename T, bool UNFUSED>
__global__ void __launch_bounds__(2 * kStepBlock)
    k_step_split(const StepJob *__restrict__ jobs, int n_jobs, const uint4 *__restrict__ tab,
                 const unsigned *__restrict__ rows, const T *__restrict__ b, T *__restrict__ x, int k)
{
    constexpr int E = kSplitEntries, D = kSplitDepth;
    typedef StepLayout<T, E> L;
    const int which = blockIdx.z * gridDim.x + blockIdx.x;
    if (which >= n_jobs) return;
    const StepJob job = jobs[which];
    const int q0 = blockIdx.y, B = job.block;
    if ((int)threadIdx.x >= 2 * B) return;  // whole wavefronts; barriers count the others
    typedef __attribute__((address_space(3))) T LdsVal;
    typedef __attribute__((address_space(3))) Words4 LdsWords;
    auto value = [](unsigned byte) -> LdsVal * { return (LdsVal *)byte; };
    auto words = [](unsigned byte) -> LdsWords * { return (LdsWords *)byte; };
    const bool loads = __builtin_amdgcn_readfirstlane((int)threadIdx.x) >= B;
    const unsigned t = loads ? threadIdx.x - B : threadIdx.x, pb = 16u * B;
    // after the ring: two buffers of a step's pieces, then its values of b
    const unsigned buf0 = ((unsigned)(job.ring + 1) * sizeof(T) + 15u) & ~15u, size = (unsigned)split_bytes<T>() * B;
    const unsigned my_piece = buf0 + 16 * t, my_b = buf0 + L::P * pb + (unsigned)sizeof(T) * t;
    const unsigned kb = (unsigned)(k * sizeof(T));
    const unsigned span = (unsigned)job.rows_of * kb - q0 * (unsigned)sizeof(T);
    const int total = (job.steps + 1) & ~1;  // the solving side unrolls by two
    if (loads) {
        const unsigned t16 = 16 * t, t4 = 4 * t;
        const Rsrc rb = make_rsrc(b + (size_t)job.row0 * k + q0, span);
        const unsigned step16 = 16u * L::P * B, step4 = 4u * B;
        auto window = [&](int step) {  // see k_step
            return make_rsrc(tab + uniform((long long)(job.tab + (unsigned long long)step * (L::P * B))),
                             (2 * D + 2) * step16);
        };
        Rsrc rt = window(0);
        const Rsrc rr = make_rsrc(rows + job.rows, (unsigned)(job.steps + kStepTail) * step4);
        Words4 w[D][L::P];
        T bo[D];
        unsigned xo[D], ahead[D];
        unsigned next = 0, nrow = 0;
        auto fetch = [&](int d, unsigned row) {
            xo[d] = row * kb;
#pragma unroll
            for (int q = 0; q < L::P; ++q)
                w[d][q] = __builtin_amdgcn_raw_buffer_load_b128(rt, (int)t16, (int)(next + q * pb), 0);
            load_value(rb, xo[d], 0, &bo[d]);
            next += step16;
        };
        auto fetch_row = [&](int d) {
            ahead[d] = __builtin_amdgcn_raw_buffer_load_b32(rr, (int)t4, (int)nrow, 0);
            nrow += step4;
        };
        auto pass_on = [&](int d, unsigned at) {  // into the buffer `at` bytes on, then the next step but D - 1
            Words4 head = w[d][0];
            head.y = xo[d];
            *words(my_piece + at) = head;
#pragma unroll
            for (int q = 1; q < L::P; ++q) *words(my_piece + at + q * pb) = w[d][q];
            *value(my_b + at) = bo[d];
            __builtin_amdgcn_sched_barrier(0);
            fetch(d, ahead[d]);
            fetch_row(d);
            __builtin_amdgcn_sched_barrier(0);
        };
        unsigned first[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            first[d] = __builtin_amdgcn_raw_buffer_load_b32(rr, (int)t4, (int)nrow, 0);
            nrow += step4;
        }
#pragma unroll
        for (int d = 0; d < D; ++d) fetch_row(d);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            fetch(d, first[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
        pass_on(0, 0);
        pass_on(1, size);
        lds_barrier();
        lds_barrier();  // step 0 is read
        unsigned at = 0;
        for (int s0 = 0; s0 < total; s0 += D) {
            rt = window(s0);
            next = (D + 2) * step16;  // step s0 + D + 2
#pragma unroll
            for (int h = 0; h < D; ++h) {
                if (s0 + h >= total) return;
                pass_on((h + 2) % D, at);  // step s0 + h + 2
                at = size - at;
                lds_barrier();
            }
        }
        return;
    }
    const Rsrc rx = make_rsrc(x + (size_t)job.row0 * k + q0, span);
    if (t == 0) *value((unsigned)job.ring * sizeof(T)) = (T)0;
    struct Step {
        Words4 w[L::P];
        T bo;
    };
    auto read = [&](Step &n, unsigned at) {
#pragma unroll
        for (int q = 0; q < L::P; ++q) n.w[q] = *words(my_piece + at + q * pb);
        n.bo = *value(my_b + at);
    };
    auto slots = [&](const Step &n, unsigned (&at)[E]) {
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const unsigned pair = u < 2 ? n.w[0].z : n.w[0].w;
            at[u] = ((u & 1) ? pair >> 16 : pair & 0xffffu) * (unsigned)sizeof(T);
        }
    };
    Step st[2];
    unsigned at[E];
    lds_barrier();
    read(st[0], 0);
    slots(st[0], at);
    lds_barrier();
    for (int s0 = 0; s0 < total; s0 += 2) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const Step &w = st[h];
            T xv[E], v[E], dr[16 / sizeof(T)], sum = (T)0;
#pragma unroll
            for (int u = 0; u < E; ++u) xv[u] = *value(at[u]);
            __builtin_amdgcn_sched_barrier(0);
            read(st[1 - h], (1 - h) * size);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_memcpy(v, &w.w[1], sizeof(v));
            __builtin_memcpy(dr, &w.w[L::P - 1], 16);
#pragma unroll
            for (int u = 0; u < E; ++u) sum = UNFUSED ? sum + v[u] * xv[u] : fmac(v[u], xv[u], sum);
            const T xi = step_divide(w.bo - sum, dr[0], dr[1]);
            *value((w.w[0].x & 0xffffu) * (unsigned)sizeof(T)) = xi;
            store_value(rx, w.w[0].y, 0, xi);
            slots(st[1 - h], at);
            lds_barrier();
        }
    }
}

// ----------------------------------------------------------- schedule
namespace {

// Steps of at most B rows over the rows [lo, hi), in row order: each row goes
// to the first step with a free place after every row it reads, and after
// the last reader of the row whose ring slot it takes (row - R).  With R
// beyond the bandwidth that reader is always an earlier row, so one pass
// places everything, and lower rows go first -- which keeps the reach of the
// dependencies, and with it the ring, short: a level-by-level order would
// solve the first levels' rows all over the matrix before the second.
// step: each row's step; returns how many.
int place_rows(const std::vector<int> &rp, const std::vector<int> &ci, int lo, int hi, int B, int R,
               std::vector<int> *step_out, std::vector<int> *last_out)
{
    std::vector<int> &step = *step_out, &last = *last_out;
    const int n = hi - lo;
    step.resize((size_t)n);
    last.resize((size_t)n);
    std::vector<int> fill, free_at;  // rows per step; the first step >= s with a free place (path-halving links)
    auto link = [&](int s) -> int & {
        while ((int)free_at.size() <= s) {
            free_at.push_back((int)free_at.size());
            fill.push_back(0);
        }
        return free_at[(size_t)s];
    };
    auto room = [&](int s) {
        for (int f = link(s); f != s; f = link(s)) {
            const int g = link(f);
            s = link(s) = g;
        }
        return s;
    };
    int steps = 0;
    for (int i = 0; i < n; ++i) {
        int s = i >= R ? last[(size_t)(i - R)] + 1 : 0;
        const int e1 = rp[(size_t)(lo + i) + 1] - 1;
        for (int j = rp[(size_t)(lo + i)]; j < e1; ++j) s = std::max(s, step[(size_t)(ci[(size_t)j] - lo)] + 1);
        s = room(s);
        if (++fill[(size_t)s] == B) free_at[(size_t)s] = s + 1;
        step[(size_t)i] = last[(size_t)i] = s;
        for (int j = rp[(size_t)(lo + i)]; j < e1; ++j) {
            int &l = last[(size_t)(ci[(size_t)j] - lo)];
            l = std::max(l, s);
        }
        steps = std::max(steps, s + 1);
    }
    return steps;
}

// Time of a step in ns, fitted to measured ones (FP64): with one wavefront
// 194 / 222 / 324 (E = 4, 8, 16), with four 328 / 433 / 744; four right-hand
// sides per thread 397 and 700 (E = 4, 16).  Chooses the workgroup size and
// the right-hand sides per thread.
double step_ns(int E, int K, int waves)
{
    return (150.0 + 11.0 * E + (waves - 1) * (8.0 + 8.0 * E)) * (1.0 + 0.37 * (K - 1));
}

}  // namespace

bool steps_take(const StepTables *t, int k)
{
    // b and x are addressed by 32-bit offsets from a matrix's first row
    return t && k >= 1 && k <= kWave && (long long)t->tallest * k * (t->vt == CAP_F64 ? 8 : 4) < (1LL << 32);
}

void steps_free(StepTables *t)
{
    if (!t) return;
    for (void *p : {(void *)t->d_jobs, (void *)t->tab, (void *)t->rows, (void *)t->ov_at, (void *)t->ov_c, t->ov_v})
        if (p) (void)hipFree(p);
    delete t;
}

namespace {

template <typename T, int E>
int fill_tables(const StepTables *t, const int *d_rp, const int *d_ci, const void *d_val, bool values_only,
                hipStream_t st)
{
    long long most = 1;
    for (const StepJob &j : t->jobs) most = std::max(most, (long long)(j.steps + kStepTail) * j.block);
    // a small table is made again where one right-hand side's solve reads it
    // (n = 2,000: the solve after it 27.6 -> 25.1 us), as long as one chiplet
    // takes all of its workgroups at once
    const int spread = values_only && t->n_jobs == 1 && most <= 256 * kBlock ? kXcds : 1;
    const dim3 grid((unsigned)(spread * std::min(2048LL, (most + kBlock - 1) / kBlock)), (unsigned)t->n_jobs);
    k_step_tables<T, E><<<grid, kBlock, 0, st>>>(t->d_jobs, t->rows, d_rp, d_ci, (const T *)d_val, t->tab, t->ov_at,
                                                 t->ov_c, (T *)t->ov_v, values_only, spread);
    return hipGetLastError() == hipSuccess ? CAP_OK : CAP_ERR_HIP;
}

template <typename T>
int fill_tables_t(const StepTables *t, const int *d_rp, const int *d_ci, const void *d_val, bool values_only,
                  hipStream_t st)
{
    if (t->E == 4) return fill_tables<T, 4>(t, d_rp, d_ci, d_val, values_only, st);
    if (t->E == 8) return fill_tables<T, 8>(t, d_rp, d_ci, d_val, values_only, st);
    return fill_tables<T, 16>(t, d_rp, d_ci, d_val, values_only, st);
}

int fill_any(const StepTables *t, const int *d_rp, const int *d_ci, const void *d_val, bool values_only, hipStream_t st)
{
    return t->vt == CAP_F64 ? fill_tables_t<double>(t, d_rp, d_ci, d_val, values_only, st)
                            : fill_tables_t<float>(t, d_rp, d_ci, d_val, values_only, st);
}

int build(StepTables *t, const std::vector<int> &rp, const std::vector<int> &ci, const std::vector<int2> &mats,
          int want_rhs, int want_block, int lds_bytes, int pad_max, double max_bytes)
{
    const int vb = t->vt == CAP_F64 ? 8 : 4;
    int longest = 0, reach = 0, tallest = 0;
    long long total = 0;
    for (const int2 &m : mats) {
        tallest = std::max(tallest, m.y - m.x);
        total += m.y - m.x;
        for (int i = m.x; i < m.y; ++i) {
            longest = std::max(longest, rp[(size_t)i + 1] - 1 - rp[(size_t)i]);
            for (int j = rp[(size_t)i]; j < rp[(size_t)i + 1] - 1; ++j) reach = std::max(reach, i - ci[(size_t)j]);
        }
    }
    if (tallest < 1 || mats.size() > 65535) return CAP_ERR_UNSUPPORTED;
    t->tallest = tallest;
    t->E = longest <= 4 ? 4 : longest <= 8 ? 8 : 16;
    t->long_rows = longest > t->E;
    // the ring: room to run ahead of the slowest row (1,024 rows past the
    // reach give the schedule of an unbounded ring within 1 % on bands of 64
    // to 4,000), less where K values per slot do not fit; one more slot holds 0
    auto slots_for = [&](int K) { return std::min(lds_bytes / (K * vb) - 2, 60000); };
    int K = want_rhs;
    while (K > 1 && slots_for(K) < std::min(tallest, reach + kStepBlock)) K /= 2;
    const int R = std::min(std::min(slots_for(K), reach + 1024), tallest);
    if (R < tallest && R <= reach) return CAP_ERR_UNSUPPORTED;
    const int P = vb == 8 ? (t->E == 4 ? StepLayout<double, 4>::P : t->E == 8 ? StepLayout<double, 8>::P : StepLayout<double, 16>::P)
                          : (t->E == 4 ? StepLayout<float, 4>::P : t->E == 8 ? StepLayout<float, 8>::P : StepLayout<float, 16>::P);
    t->max_rhs = K;
    t->ring = R;
    std::vector<unsigned> rows;
    std::vector<int> ov_at, step, best, last, fill;
    long long pieces = 0, padded = 0;
    int ov_len = 0;
    for (const int2 &m : mats) {
        const int lo = m.x, hi = m.y, n = hi - lo;
        if (n == 0) continue;
        int B = 0, steps = 0;
        double cost = 0;
        for (int cand = kWave; cand <= kStepBlock; cand += kWave) {
            if (want_block && cand != want_block) continue;
            const int s = place_rows(rp, ci, lo, hi, cand, R, &step, &last);
            const double c = s * step_ns(t->E, K, cand / kWave);
            if (!B || c < cost) {
                B = cand;
                cost = c;
                steps = s;
                best.swap(step);
            }
            // fewer rows than threads in every step: wider ones cannot help
            if ((long long)s * cand >= 3LL * n) break;
        }
        padded += (long long)steps * B;
        const size_t first = rows.size(), count = (size_t)(steps + kStepTail) * B;
        rows.resize(first + count);
        if (t->long_rows) ov_at.resize(first + count, -1);
        fill.assign((size_t)steps, 0);
        std::vector<int> rest;  // where a long row's rest starts
        if (t->long_rows) {
            rest.assign((size_t)n, -1);
            for (int i = 0; i < n; ++i) {
                const int cnt = rp[(size_t)(lo + i) + 1] - 1 - rp[(size_t)(lo + i)];
                if (cnt <= t->E) continue;
                rest[(size_t)i] = ov_len;
                if ((long long)ov_len + cnt > INT32_MAX / 2) return CAP_ERR_UNSUPPORTED;
                ov_len += 1 + cnt - t->E;
            }
        }
        for (int i = 0; i < n; ++i) {
            const size_t s = (size_t)best[(size_t)i], at = first + s * B + (size_t)fill[s]++;
            rows[at] = (unsigned)i;
            if (t->long_rows) ov_at[at] = rest[(size_t)i];
        }
        for (size_t s = 0; s < (size_t)(steps + kStepTail); ++s) {
            const size_t from = std::min(s, (size_t)steps - 1);
            for (int q = from == s ? fill[s] : 0; q < B; ++q) {
                const size_t src = first + from * B + (size_t)(from == s ? 0 : q);
                rows[first + s * B + (size_t)q] = rows[src];
                if (t->long_rows) ov_at[first + s * B + (size_t)q] = ov_at[src];
            }
        }
        t->jobs.push_back(StepJob{(unsigned long long)pieces, (unsigned)first, steps, R, B, lo, n});
        pieces += (long long)count * P;
        t->block = std::max(t->block, B);
        // a job's row table is addressed by 32-bit byte offsets
        if (rows.size() >= (size_t)1 << 30 || (double)pieces * 16 > max_bytes) return CAP_ERR_UNSUPPORTED;
    }
    if (t->jobs.empty() || padded > std::max((long long)pad_max * total, 1LL << 16)) return CAP_ERR_UNSUPPORTED;
    // the longest chains start first
    std::stable_sort(t->jobs.begin(), t->jobs.end(), [&](const StepJob &a, const StepJob &c) {
        return a.steps * step_ns(t->E, K, a.block / kWave) > c.steps * step_ns(t->E, K, c.block / kWave);
    });
    t->n_jobs = (int)t->jobs.size();
    t->slots = (long long)rows.size();
    auto put = [](auto **d, const auto &h) {
        const size_t bytes = sizeof(h[0]) * h.size();
        return hipMalloc((void **)d, bytes + 16) == hipSuccess &&
               hipMemcpy(*d, h.data(), bytes, hipMemcpyHostToDevice) == hipSuccess;
    };
    if (!put(&t->d_jobs, t->jobs) || !put(&t->rows, rows)) return CAP_ERR_ALLOC;
    if (hipMalloc((void **)&t->tab, (size_t)pieces * 16) != hipSuccess) return CAP_ERR_ALLOC;
    if (t->long_rows &&
        (!put(&t->ov_at, ov_at) || hipMalloc((void **)&t->ov_c, sizeof(int) * (size_t)(ov_len + 1)) != hipSuccess ||
         hipMalloc(&t->ov_v, (size_t)vb * (size_t)(ov_len + 1)) != hipSuccess))
        return CAP_ERR_ALLOC;
    return CAP_OK;
}

template <typename T, int E, bool LONG, int K>
int launch_k(const StepTables *t, const T *b, T *x, int k, bool unfused, hipStream_t st, int allow_lds)
{
    constexpr int D = step_depth<E, K>();
    const size_t ring = (size_t)(t->ring + 1) * K * sizeof(T);
    const int group = std::min(t->n_jobs, kXcds);
    const dim3 grid((unsigned)group, (unsigned)(k / K), (unsigned)((t->n_jobs + group - 1) / group));
    auto allow = [&](auto kernel) {  // once, when the tables are built
        return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   allow_lds);
    };
    if constexpr (K == 1 && E == kSplitEntries) {
        auto kernel = unfused ? k_step_split<T, true> : k_step_split<T, false>;
        const size_t bytes = (ring + 15) / 16 * 16 + 2 * (size_t)split_bytes<T>() * t->block;
        if (allow_lds) {
            CAP_HIP_TRY(allow(kernel));
        } else if (bytes <= t->lds && (long long)t->n_jobs * k <= t->cus) {
            kernel<<<grid, 2 * t->block, bytes, st>>>(t->d_jobs, t->n_jobs, t->tab, t->rows, b, x, k);
            CAP_HIP_TRY(hipGetLastError());
            return CAP_OK;
        }
    }
    auto kernel = unfused ? k_step<T, E, D, true, LONG, K> : k_step<T, E, D, false, LONG, K>;
    if (allow_lds) {
        CAP_HIP_TRY(allow(kernel));
        return CAP_OK;
    }
    kernel<<<grid, t->block, ring, st>>>(t->d_jobs, t->n_jobs, t->tab, t->rows, t->ov_c, (const T *)t->ov_v, b, x, k);
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

// Right-hand sides per thread for k of them: fewer mean more workgroups, each
// with shorter steps; more mean less work in all.  The estimate is the longer
// of the longest job's chain and the whole work over the compute units: a
// plan's one matrix takes 1 (four right-hand sides on the 100k band: 183 us
// as four workgroups, 457 in one), a batch of thousands of chunks up to 4.
int rhs_per_thread(const StepTables *t, int k)
{
    int best = 1;
    double best_ns = 0;
    for (int K = 1; K <= t->max_rhs; K *= 2) {
        if (k % K) break;
        double chain = 0, all = 0;
        for (const StepJob &j : t->jobs) {
            const double ns = j.steps * step_ns(t->E, K, j.block / kWave);
            chain = std::max(chain, ns);
            all += ns * (k / K);
        }
        const double ns = std::max(chain, all / t->cus);
        if (K == 1 || ns < best_ns) {
            best = K;
            best_ns = ns;
        }
    }
    return best;
}

template <typename T, int E, bool LONG>
int launch_e(const StepTables *t, const T *b, T *x, int k, bool unfused, hipStream_t st, int allow_lds)
{
    const int K = allow_lds ? std::min(k, t->max_rhs) : rhs_per_thread(t, k);
    if (K == 4) return launch_k<T, E, LONG, 4>(t, b, x, k, unfused, st, allow_lds);
    if (K == 2) return launch_k<T, E, LONG, 2>(t, b, x, k, unfused, st, allow_lds);
    return launch_k<T, E, LONG, 1>(t, b, x, k, unfused, st, allow_lds);
}

template <typename T>
int launch_t(const StepTables *t, const T *b, T *x, int k, bool unfused, hipStream_t st, int allow_lds)
{
    if (t->E == 4) return launch_e<T, 4, false>(t, b, x, k, unfused, st, allow_lds);
    if (t->E == 8) return launch_e<T, 8, false>(t, b, x, k, unfused, st, allow_lds);
    return t->long_rows ? launch_e<T, 16, true>(t, b, x, k, unfused, st, allow_lds) : launch_e<T, 16, false>(t, b, x, k, unfused, st, allow_lds);
}

int launch_any(const StepTables *t, const void *b, void *x, int k, bool unfused, hipStream_t st, int allow_lds)
{
    return t->vt == CAP_F64 ? launch_t<double>(t, (const double *)b, (double *)x, k, unfused, st, allow_lds)
                            : launch_t<float>(t, (const float *)b, (float *)x, k, unfused, st, allow_lds);
}

}  // namespace

int steps_build(StepTables **out, const std::vector<int> &rp, const std::vector<int> &ci,
                const std::vector<int2> &mats, int vt, int want_rhs, int want_block, int lds_bytes, int pad_max,
                double max_bytes, const int *d_rp, const int *d_ci, const void *d_val, hipStream_t st)
{
    *out = nullptr;
    int dev = 0, cus = 0;
    CAP_HIP_TRY(hipGetDevice(&dev));
    CAP_HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    StepTables *t = new (std::nothrow) StepTables();
    if (!t) return CAP_ERR_ALLOC;
    t->vt = vt;
    t->cus = std::max(1, cus);
    t->lds = (size_t)std::max(0, lds_bytes);
    int rc;
    try {
        rc = build(t, rp, ci, mats, want_rhs, want_block, lds_bytes, pad_max, max_bytes);
    } catch (const std::bad_alloc &) {
        rc = CAP_ERR_ALLOC;
    }
    for (int k : {1, 2, 4})
        for (bool unfused : {false, true})
            if (rc == CAP_OK) rc = launch_any(t, nullptr, nullptr, k, unfused, st, lds_bytes);
    if (rc == CAP_OK) rc = fill_any(t, d_rp, d_ci, d_val, false, st);
    if (rc == CAP_OK && hipStreamSynchronize(st) != hipSuccess) rc = CAP_ERR_HIP;
    if (rc != CAP_OK) {
        (void)hipGetLastError();  // not for the next launch's check: callers go on without the tables
        steps_free(t);
        return rc;
    }
    *out = t;
    return CAP_OK;
}

int steps_refresh(const StepTables *t, const int *d_rp, const int *d_ci, const void *d_val, hipStream_t st)
{
    return fill_any(t, d_rp, d_ci, d_val, true, st);
}

int steps_launch(const StepTables *t, const void *b, void *x, int k, bool unfused, hipStream_t st)
{
    if (!steps_take(t, k)) return CAP_ERR_UNSUPPORTED;
    return launch_any(t, b, x, k, unfused, st, 0);
}

}  // namespace cap
