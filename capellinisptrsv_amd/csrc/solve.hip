// C ABI of the gfx950 SpTRSV: plans (device-resident solves, adjoint,
// FP32+FP64 refinement), batches, one-shot host solves and the
// benchmark-compatible wrappers that replace the reference's host wrappers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <tuple>
#include <vector>

#include "../../include/capellini_sptrsv.h"
#include "cap_internal.h"
#include "kernels.h"
#include "steps.h"

using namespace cap;

namespace {

// Threshold of the mix selector for 64-row chunks: a chunk whose mean
// nnz/row reaches it is solved wavefront-per-row.  The reference hard-codes
// 10 for 32-lane warps (CUDA/mix/spts_syncfree_cuda_csr_wrt.h:188).  Here it
// follows the matrix's rows per level.  Measured on MI355X (n = 200,000; mix
// time with every chunk wavefront-per-row over every chunk thread-per-row):
//   level matrices (dependencies in the previous two levels), 250 to 4,000
//   rows per level: 1.13 at 3 nnz/row (4,000 rows per level); 0.47-0.73 at
//   5; 0.28-0.52 at 9; 0.17-0.32 at 17; 0.15 at 64;
//   bands of 1,000 (dependencies among the previous 1,000 rows), 11 to 136
//   rows per level: 1.02, 1.05, 1.06, 1.01 at 4, 7, 13, 25 nnz/row; 0.91 at 49.
// So chunks of 4 or more nnz/row go wavefront-per-row where levels hold at
// least 200 rows; below that the chain sets the time either way, and rows
// gain from a wavefront from about 32 entries on (between the 1.01 at 25 and
// the 0.91 at 49).
constexpr int kMixWideLevel = 200;    // rows per level from which levels count as wide
constexpr int kMixBorderWide = 4;     // threshold where they are
constexpr int kMixBorderNarrow = 32;  // threshold where they are not
// Workgroups of mix per CU, whatever cap_opts.blocks_per_cu says.  Two of 1024
// threads fill all 32 wave slots of a CU, 524,288 polling lanes on the chip,
// and in FP32 without row tiles a 777,001-row wide-level matrix then made no
// progress for the whole wait limit (10 s), as a batch of thread-per-row
// workgroups once did at 8 per CU, the same number of lanes.  By tickets
// alone either must progress; why polls starve there is not known.  Where two
// did run they gave nothing: 268 us against 270 (row tiles).
constexpr int kMixBlocks = 1;
inline int mix_border_for(int n, int levels)
{
    return (long long)n >= (long long)kMixWideLevel * std::max(1, levels) ? kMixBorderWide : kMixBorderNarrow;
}
// A wait gives up after this much wall time without progress (10 ns ticks of
// the real-time counter): far above any legitimate wait -- a lane waits only
// for rows the persistent grid already holds, tens of milliseconds at most
// on the deepest matrices -- and small enough that a grid that cannot make
// progress drains in seconds.  No poll-count bound by default.
constexpr int kWaitMsDefault = 10000;
constexpr int kWaitMsMax = 40000;  // the 32-bit tick difference wraps at 42.9 s
// Persistent grids hold at most 4 workgroups per compute unit.  A batch
// solve with 8 (2048 resident workgroups, one right-hand side) stopped
// making progress, so larger values are refused.
constexpr int kMaxBlocksPerCu = 4;
constexpr int kTickets = 4;
// The autotuner times CAP_ALGO_LOCAL when rows per level (n / levels) are at
// most this: one compute unit then keeps up with the level-by-level pace.
constexpr double kLocalMaxWidth = 256.0;

inline hipStream_t S(void *s) { return reinterpret_cast<hipStream_t>(s); }
inline unsigned blocks_for(long long threads) { return (unsigned)((threads + kBlock - 1) / kBlock); }
inline int lpr_log2_for(int k)
{
    int l = 0;
    while ((1 << l) < k) ++l;
    return l;
}

}  // namespace

// State of a partitioned banded solve: blocks of m rows (P of them, Q = P - 1
// coupled tails of W values, W = 128 or 256); the blocks' rows as records
// (layout in kernels.h, k_part_records) of J entries per lane, block p's from
// at[p], and where its first few records start; the tail scan's W x W
// matrices in bm: B_p at p - 1 and, unless the tails are walked, the in-group
// products W_p at w_off + p - gs, and for each round r of the group-carry
// scan G - 2^r matrices from m_off[r]; the solve's work vectors.
struct PartState {
    int W = kPartW;                 // tail width: the coupling columns
    int m = 0, P = 0, Q = 0, J = 0;
    bool walk = false;              // the blocks damp their history, or are few: k_part_walk
    int gs = 0, G = 0, rounds = 0;  // tails per group, groups, carry-scan rounds
    uint4 *rec = nullptr;
    int *at = nullptr;
    uint2 *first = nullptr;
    double *bm = nullptr;
    uint2 *fade = nullptr;     // k_part_walk: how the blocks damp
    long long w_off = 0;
    std::vector<long long> m_off;
    // work vectors, sized for kcap right-hand sides (grown by a solve with more)
    int kcap = 0;
    double *a = nullptr, *u = nullptr, *t = nullptr, *c0 = nullptr, *c1 = nullptr;
    unsigned long long *top = nullptr;      // the largest and smallest magnitude of each a_p
    double *res = nullptr, *cor = nullptr;  // refinement: FP64 residual and correction (n * kcap)
};

// Look-through tables of the write-first solve (layout in kernels.h, k_hop):
// E entries per row, `hops` publish -> observe hops on the longest chain.
struct HopState {
    int *base = nullptr, *ex = nullptr;
    int E = 0, npad = 0, hops = 0;
};

// The RHS-block pick of an autotuned plan for one right-hand-side count:
// thread-per-row workgroups per CU, threads per workgroup and right-hand
// sides per lane, or the partitioned sweeps' right-hand sides per
// wavefront (0: the plan's).
struct RhsPick {
    int bpc = 0, block = 0, kr = 0, rpl = 0;
    int staged = -1;  // readiness: 1 staged, 0 in x itself, -1 the plan's
    int lds = -1;     // LDS window: 0 off (the 1024-thread shapes), -1 the plan's
    int tile = -1;    // row tiles: 1 on, 0 off, -1 the plan's
    bool rows = false;  // a level plan's: the write-first kernel, not the steps
};

// The fastest plain write-first shape (value protocol, the plan's readiness)
// of an autotuned plan whose pick solves one right-hand side otherwise, by
// look-through tables or steps: what its several right-hand sides and its
// fused sweeps start from.  bpc 0: none.
struct PlainShape {
    int bpc = 0, block = 0, lds = 0, tile = 0, staged = 0;
};

struct cap_plan_s {
    int n = 0, nnz = 0, vt = CAP_F64, vbytes = 8;
    int algo = CAP_ALGO_WRTFST, sync = CAP_SYNC_VALUE, border = kMixBorderWide;
    int device = 0;
    int *rp = nullptr, *ci = nullptr;
    void *val = nullptr;
    bool owns_matrix = false;
    // hybrid batch: rows {first, count} that partitioned plans solve; the
    // refinement's later steps leave them unchanged (their correction is 0)
    std::vector<int2> skip_rows;
    // synchronisation state
    int *flags = nullptr;
    long long flags_len = 0;
    int epoch = 0;
    // control block (one 4 KiB allocation): tickets at +0, watchdog word at
    // +256, refinement norms at +512, poll counters at +1024
    unsigned char *ctrl = nullptr;
    unsigned *ticket = nullptr;
    int *err = nullptr;
    int spin_limit = 0;                   // polls without progress (0: no count bound)
    int wait_ticks = kWaitMsDefault * 100000;  // wall time without progress, 10 ns ticks
    int ncu = 256, bpc = 1;  // persistent grid: bpc workgroups per compute unit
    int wblock = kBlock;     // threads per workgroup of k_wrtfst (128 or 256)
    int rblock = 0;          // of k_refine2; 0 = not chosen yet (autotuned plans time it)
    int lds = 0;             // thread-per-row: workgroup-local LDS readiness window
    int tile = 0;            // thread-per-row, value protocol: tickets' col_idx/val tiles staged in LDS
    int unfused = 0;         // CAP_ARITH_REFERENCE: rounded products, then rounded sums
    int count_polls = 0;     // the write-first solve counts its poll loads (ctrl + 1024)
    // multi-RHS solves of an autotuned plan: the RHS block is timed per
    // right-hand-side count on the first cap_plan_solve with that count
    bool tune_rhs = false;
    std::map<int, RhsPick> rhs_pick;
    PlainShape plain;
    float lvl_lead = 0;  // a level pick: the plain shape's time over the steps', one right-hand side
    int part_kr = 0;  // partition sweeps: right-hand sides per wavefront (0: the fixed rule)
    int rpl = 1;      // thread-per-row, several right-hand sides: right-hand sides per lane
    int fixed_rpl = 0;  // cap_opts.rhs_per_lane: the multi-RHS block the caller fixed (0: none)
    bool auto_algo = false;  // created with CAP_ALGO_AUTO
    // batch: block schedules (relative level order), by rows per block: the
    // thread-per-row solve's and the refinement sweep's (device array, count)
    std::map<int, std::pair<int2 *, int>> scheds;
    // CAP_ALGO_LOCAL: row segments [x, y) with bandwidth z, one per matrix,
    // largest first; LDS available to one workgroup
    int4 *seg = nullptr;
    int n_seg = 0;
    int lds_max = 65536;
    // upper-triangular plans solve the reversed matrix (b and x reversed
    // around the solve through rev_b / rev_x); unit_diag: the diagonal was implicit
    bool reversed = false, unit_diag = false;
    void *rev_b = nullptr, *rev_x = nullptr;
    size_t rev_bytes = 0;
    // value protocol: staged readiness array (uncached pool block) or x itself
    int staged = 1;
    void *ready = nullptr;
    size_t ready_bytes = 0;
    // mix
    int *unit = nullptr;
    int n_units = 0, mix_len = 0;
    double wocc = 0, eocc = 0;
    // CSC executor (forward)
    int *cp = nullptr, *cri = nullptr, *deg0 = nullptr, *deg = nullptr;
    void *cv = nullptr, *left_sum = nullptr;
    // adjoint: scatter (in-degree counters + atomic left sums) or gather
    // (reversed transpose of L, solved with the write-first kernel)
    int adjoint_mode = CAP_ADJOINT_GATHER;
    int *cnt0 = nullptr, *cnt = nullptr;
    double *adj_ls = nullptr;
    int *rpT = nullptr, *ciT = nullptr;
    double *vT = nullptr;
    // refinement
    float *val32 = nullptr, *r32 = nullptr, *d32 = nullptr;
    long long refine_len = 0;
    unsigned long long *pair = nullptr;  // fused refinement pairs when readiness is in place
    long long pair_len = 0;
    unsigned long long *norms = nullptr;  // inside ctrl
    // the norms for the host: pinned memory, two norms and the count of the
    // read they belong to
    unsigned long long *echo = nullptr, echoes = 0;
    hipGraphExec_t refine_graph = nullptr;
    const void *graph_b = nullptr;
    void *graph_x = nullptr;
    int graph_rhs = 0;
    // partitioned banded solve (CAP_ALGO_PARTITION)
    struct PartState *part = nullptr;
    // steps in one workgroup (CAP_ALGO_LEVEL).  lvl_rhs: right-hand sides per
    // solve an explicit plan takes (1, 2 or 4; 0: any).  lvl_live: the tables
    // take the caller's values again on every solve (autotuned plans)
    StepTables *lvl = nullptr;
    int lvl_rhs = 0;
    bool lvl_live = false;
    // batch: the matrices outside the partitioned ones solved by steps, one
    // workgroup per matrix and right-hand-side chunk (nullptr: by algo)
    StepTables *batch_steps = nullptr;
    // write-first solve of one right-hand side with look-through tables
    // (autotuned plans, value protocol, staged readiness)
    HopState *hop = nullptr;
    bool hop_reset = false;  // reversed plans: a solve or reset over the tables has run
};

// One right-hand side of a plan whose pick has look-through tables.  The
// kernel reverses rows itself, so upper-triangular plans need no copies.
inline bool hop_takes(const cap_plan_s *p, int rhs)
{
    return p->hop && rhs == 1 && p->algo == CAP_ALGO_WRTFST && p->sync == CAP_SYNC_VALUE && p->staged;
}

// Right-hand-side counts a plan's steps solve: an explicit level plan's 1,
// and 2 or 4 where its rule allows; any of an autotuned one's.
inline bool level_allows(const cap_plan_s *p, int rhs)
{
    return p->lvl_rhs == 0 || rhs == 1 || ((rhs == 2 || rhs == 4) && rhs <= p->lvl_rhs);
}
inline bool level_takes(const cap_plan_s *p, int rhs) { return steps_take(p->lvl, rhs) && level_allows(p, rhs); }

// Side streams of a hybrid batch: its partitioned matrices' solves run
// concurrently with each other (and with the rest's reset), forked from and
// joined back into the caller's stream by events, so a batch solve stays
// one stream-ordered operation (and can be captured into a graph).  Default
// priority, non-blocking.
struct Fork {
    std::vector<hipStream_t> s;
    std::vector<hipEvent_t> done;
    hipEvent_t start = nullptr;
    int make(int n)
    {
        if (hipEventCreateWithFlags(&start, hipEventDisableTiming) != hipSuccess) return CAP_ERR_HIP;
        for (int i = 0; i < n; ++i) {
            hipStream_t q = nullptr;
            hipEvent_t e = nullptr;
            if (hipStreamCreateWithFlags(&q, hipStreamNonBlocking) != hipSuccess) return CAP_ERR_HIP;
            s.push_back(q);
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return CAP_ERR_HIP;
            done.push_back(e);
        }
        return CAP_OK;
    }
    void release()
    {
        for (hipStream_t q : s) (void)hipStreamDestroy(q);
        for (hipEvent_t e : done) (void)hipEventDestroy(e);
        if (start) (void)hipEventDestroy(start);
        s.clear();
        done.clear();
        start = nullptr;
    }
};

struct cap_batch_s {
    cap_plan plan = nullptr;
    int k = 1;
    int n_mat = 0;
    // hybrid: the deepest matrices solved by partitioned plans of their own
    // (first rows part_lo), the rest by `plan` over a schedule without them
    std::vector<cap_plan> parts;
    std::vector<int> part_lo;
    Fork fork;  // the partitioned solves' side streams
};

namespace {

// The partitioned matrices' solves (each writes only its own rows), part h
// on side stream h mod ns, forked from st (they start after what st holds
// so far) and joined back into it (what st gets later waits for them);
// without side streams they run on st in turn.  Whatever st gets between
// the fork and the join runs alongside them.
template <typename Solve>
int fork_parts(size_t count, const Fork *fk, hipStream_t st, Solve solve)
{
    const size_t ns = fk ? fk->s.size() : 0;
    if (ns == 0) {
        for (size_t h = 0; h < count; ++h) CAP_TRY(solve(h, st));
        return CAP_OK;
    }
    CAP_HIP_TRY(hipEventRecord(fk->start, st));
    for (size_t i = 0; i < ns; ++i) CAP_HIP_TRY(hipStreamWaitEvent(fk->s[i], fk->start, 0));
    for (size_t h = 0; h < count; ++h) CAP_TRY(solve(h, fk->s[h % ns]));
    return CAP_OK;
}

int join_parts(const Fork *fk, hipStream_t st)
{
    const size_t ns = fk ? fk->s.size() : 0;
    for (size_t i = 0; i < ns; ++i) {
        CAP_HIP_TRY(hipEventRecord(fk->done[i], fk->s[i]));
        CAP_HIP_TRY(hipStreamWaitEvent(st, fk->done[i], 0));
    }
    return CAP_OK;
}


// ------------------------------------------------------------ device check
int check_device(int *dev)
{
    int count = 0;
    const hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count < 1) {
        std::fprintf(stderr, "capellini: hipGetDeviceCount -> %d (%s), count %d\n", (int)e, hipGetErrorString(e),
                     count);
        return CAP_ERR_NO_DEVICE;
    }
    CAP_HIP_TRY(hipGetDevice(dev));
    hipDeviceProp_t prop;
    CAP_HIP_TRY(hipGetDeviceProperties(&prop, *dev));
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        std::fprintf(stderr, "capellini: device %d is %s, this library is built for gfx950\n", *dev,
                     prop.gcnArchName);
        return CAP_ERR_NO_DEVICE;
    }
    return CAP_OK;
}

template <typename P>
int dev_alloc(P **p, size_t count)
{
    *p = nullptr;
    if (count == 0) count = 1;
    if (hipMalloc((void **)p, count * sizeof(P)) != hipSuccess) {
        (void)hipGetLastError();  // not for the next launch's check: callers may go on without
        *p = nullptr;
        return CAP_ERR_ALLOC;
    }
    return CAP_OK;
}

// ------------------------------------------------- uncached readiness pool
// Blocks of uncached device memory for staged readiness arrays.  Uncached
// memory that a kernel has read is never freed before the process ends
// (later allocations have been seen to read wrong values after such a free),
// so blocks return to this pool when a plan lets go of them and are handed to
// later plans on the same device (best fit).
struct ReadyBlock {
    int device;
    void *ptr;
    size_t bytes;
    bool used;
};
std::mutex g_ready_mu;
std::vector<ReadyBlock> g_ready_pool;

int ready_acquire(int device, size_t bytes, void **out, size_t *got)
{
    std::lock_guard<std::mutex> g(g_ready_mu);
    ReadyBlock *best = nullptr;
    for (ReadyBlock &r : g_ready_pool)
        if (!r.used && r.device == device && r.bytes >= bytes && (!best || r.bytes < best->bytes)) best = &r;
    if (!best) {
        const size_t grain = (size_t)2 << 20;
        const size_t sz = (bytes + grain - 1) / grain * grain;
        void *ptr = nullptr;
        if (hipExtMallocWithFlags(&ptr, sz, hipDeviceMallocUncached) != hipSuccess || !ptr) {
            (void)hipGetLastError();
            return CAP_ERR_ALLOC;
        }
        g_ready_pool.push_back({device, ptr, sz, false});
        best = &g_ready_pool.back();
    }
    best->used = true;
    *out = best->ptr;
    *got = best->bytes;
    return CAP_OK;
}

void ready_release(void *ptr)
{
    if (!ptr) return;
    std::lock_guard<std::mutex> g(g_ready_mu);
    for (ReadyBlock &r : g_ready_pool)
        if (r.ptr == ptr) r.used = false;
}

// ------------------------------------------------------------ pinned words
// What refined solves read their norms from, 64 bytes a plan.  A pinned
// allocation takes 25 us, inside a new plan's first refined solve, so up to
// kEchoKept of them stay for later plans.
constexpr size_t kEchoKept = 16;
std::mutex g_echo_mu;
std::vector<unsigned long long *> g_echo_free;

int echo_acquire(unsigned long long **out)
{
    {
        std::lock_guard<std::mutex> g(g_echo_mu);
        if (!g_echo_free.empty()) {
            *out = g_echo_free.back();
            g_echo_free.pop_back();
        }
    }
    if (!*out && hipHostMalloc(reinterpret_cast<void **>(out), 64, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        *out = nullptr;
        return CAP_ERR_ALLOC;
    }
    std::memset(*out, 0, 64);  // another plan's counts
    return CAP_OK;
}

// After the last kernel that writes the words.
void echo_release(unsigned long long *words)
{
    if (!words) return;
    {
        std::lock_guard<std::mutex> g(g_echo_mu);
        if (g_echo_free.size() < kEchoKept) {
            g_echo_free.push_back(words);
            return;
        }
    }
    (void)hipHostFree(words);
}

// The plan's staged readiness array holds at least `bytes`.  Growing it
// waits for the device (kernels in flight may still poll the old block) and
// drops the captured refinement graph, which has the old block's address.
int ensure_ready(cap_plan p, size_t bytes)
{
    if (p->ready_bytes >= bytes) return CAP_OK;
    if (p->ready) {
        CAP_HIP_TRY(hipDeviceSynchronize());
        if (p->refine_graph) CAP_HIP_TRY(hipGraphExecDestroy(p->refine_graph));
        p->refine_graph = nullptr;
        ready_release(p->ready);
        p->ready = nullptr;
        p->ready_bytes = 0;
    }
    return ready_acquire(p->device, bytes, &p->ready, &p->ready_bytes);
}

void free_partition(cap_plan p)
{
    PartState *ps = p->part;
    if (!ps) return;
    (void)hipDeviceSynchronize();
    for (void *b : {(void *)ps->rec, (void *)ps->at, (void *)ps->first, (void *)ps->bm, (void *)ps->fade,
                    (void *)ps->a, (void *)ps->u, (void *)ps->t, (void *)ps->c0, (void *)ps->c1, (void *)ps->top,
                    (void *)ps->res, (void *)ps->cor})
        if (b) (void)hipFree(b);
    delete ps;
    p->part = nullptr;
}

void free_level(cap_plan p)
{
    if (!p->lvl) return;
    (void)hipDeviceSynchronize();
    steps_free(p->lvl);
    p->lvl = nullptr;
}

void free_hop(cap_plan p)
{
    if (!p->hop) return;
    (void)hipDeviceSynchronize();
    for (int *b : {p->hop->base, p->hop->ex})
        if (b) (void)hipFree(b);
    delete p->hop;
    p->hop = nullptr;
}

void plan_free(cap_plan p)
{
    if (!p) return;
    free_partition(p);
    free_level(p);
    free_hop(p);
    steps_free(p->batch_steps);
    if (p->ready) {
        (void)hipDeviceSynchronize();  // no kernel of this plan may still poll the block
        ready_release(p->ready);
    }
    if (p->owns_matrix) {
        (void)hipFree(p->rp);
        (void)hipFree(p->ci);
        (void)hipFree(p->val);
    }
    for (auto &e : p->scheds) (void)hipFree(e.second.first);
    void *bufs[] = {p->rev_b, p->rev_x, p->seg, p->flags, p->ctrl, p->unit, p->cp, p->cri, p->deg0, p->deg, p->cv, p->left_sum,
                    p->cnt0, p->cnt, p->adj_ls, p->rpT, p->ciT, p->vT, p->val32, p->r32, p->d32, p->pair};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    if (p->refine_graph) (void)hipGraphExecDestroy(p->refine_graph);
    if (p->echo) {
        (void)hipDeviceSynchronize();
        echo_release(p->echo);
    }
    delete p;
}

// Control block and device shape (compute units for the persistent grid).
int init_ctrl(cap_plan p)
{
    CAP_TRY(dev_alloc(&p->ctrl, 4096));
    CAP_HIP_TRY(hipMemset(p->ctrl, 0, 4096));
    p->ticket = reinterpret_cast<unsigned *>(p->ctrl);
    p->err = reinterpret_cast<int *>(p->ctrl + 256);
    p->norms = reinterpret_cast<unsigned long long *>(p->ctrl + 512);
    int ncu = 0, lds = 0;
    CAP_HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, p->device));
    CAP_HIP_TRY(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, p->device));
    p->ncu = ncu > 0 ? ncu : 256;
    p->lds_max = lds > 0 ? lds : 65536;
    // k_local sizes its LDS ring to the device limit
    CAP_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_local<double>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, p->lds_max - kLocalStaticLds));
    CAP_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_local<float>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, p->lds_max - kLocalStaticLds));
    return CAP_OK;
}

// Persistent grid: never more workgroups than the work needs, never more
// than bpc per compute unit (more resident pollers only add memory traffic).
inline unsigned grid_for(const cap_plan p, long long work_blocks)
{
    const long long cap = (long long)p->ncu * p->bpc;
    return (unsigned)std::max(1LL, std::min(work_blocks, cap));
}

int ensure_flags(cap_plan p, long long len, hipStream_t st)
{
    if (p->flags_len >= len) return CAP_OK;
    if (p->flags) CAP_HIP_TRY(hipFree(p->flags));
    p->flags = nullptr;
    CAP_TRY(dev_alloc(&p->flags, (size_t)len));
    k_prepare<unsigned><<<blocks_for(len), kBlock, 0, st>>>((unsigned *)p->flags, len, 0u, p->ticket, 0);
    CAP_HIP_TRY(hipGetLastError());
    p->flags_len = len;
    p->epoch = 0;
    return CAP_OK;
}

// Per-solve reset (tickets; sentinel fill of the readiness array -- staged
// or x -- in the value protocol; CAP_ALGO_LOCAL always polls x itself).
template <typename T>
int launch_prepare(cap_plan p, int algo, int sync, void *x, long long count, hipStream_t st)
{
    typedef typename VBits<T>::U U;
    // the partitioned solve and the level steps keep no readiness state
    if (algo == CAP_ALGO_PARTITION || algo == CAP_ALGO_LEVEL) return CAP_OK;
    if (algo == CAP_ALGO_LOCAL) sync = CAP_SYNC_VALUE;
    if (sync == CAP_SYNC_VALUE) {
        void *target = x;
        if (p->staged && algo != CAP_ALGO_LOCAL) {
            CAP_TRY(ensure_ready(p, sizeof(U) * (size_t)count));
            target = p->ready;
        }
        const unsigned nb = std::max(1u, std::min(blocks_for(count), 2048u));
        k_prepare<U><<<nb, kBlock, 0, st>>>((U *)target, count, VBits<T>::kSentinel, p->ticket, kTickets);
    } else {
        CAP_TRY(ensure_flags(p, count, st));
        if (++p->epoch == 0x7fffffff) {  // wrap: clear the flags once
            k_prepare<unsigned><<<blocks_for(p->flags_len), kBlock, 0, st>>>((unsigned *)p->flags, p->flags_len,
                                                                             0u, p->ticket, 0);
            p->epoch = 1;
        }
        k_prepare<U><<<1, kBlock, 0, st>>>((U *)x, 0, (U)0, p->ticket, kTickets);
    }
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

// The solve kernel itself (after launch_prepare).
// Segment table of CAP_ALGO_LOCAL: {lo, hi, bandwidth, longest row's
// off-diagonal count} for the whole
// matrix, or (batches) for every matrix, ordered by decreasing nonzero count
// so that the largest matrices start first.  The bandwidth (largest row -
// column distance) decides whether a segment's dependencies fit the LDS ring.
// rp_host, ci_host: host copies of the rows where the caller has them.
int ensure_segments(cap_plan p, const std::vector<int> *row_off, const std::vector<int> *rp_host = nullptr,
                    const std::vector<int> *ci_host = nullptr)
{
    if (p->seg && !row_off) return CAP_OK;
    const int n = p->n;
    std::vector<int> rp_own, ci_own, bw((size_t)std::max(n, 1), 0);
    if (!rp_host) {
        rp_own.resize((size_t)n + 1);
        ci_own.resize((size_t)p->nnz);
        CAP_HIP_TRY(hipMemcpy(rp_own.data(), p->rp, sizeof(int) * rp_own.size(), hipMemcpyDeviceToHost));
        CAP_HIP_TRY(hipMemcpy(ci_own.data(), p->ci, sizeof(int) * ci_own.size(), hipMemcpyDeviceToHost));
    }
    const std::vector<int> &rp = rp_host ? *rp_host : rp_own, &ci = rp_host ? *ci_host : ci_own;
    for (int i = 0; i < n; ++i)
        for (int j = rp[i]; j < rp[i + 1]; ++j) bw[i] = std::max(bw[i], i - ci[j]);
    std::vector<int4> h;
    auto add = [&](int lo, int hi) {
        int w = 0, len = 0;
        for (int i = lo; i < hi; ++i) {
            w = std::max(w, bw[i]);
            len = std::max(len, rp[i + 1] - 1 - rp[i]);
        }
        h.push_back(make_int4(lo, hi, w, len));
    };
    if (!row_off) {
        add(0, n);
    } else {
        const std::vector<int> &ro = *row_off;
        for (size_t m = 0; m + 1 < ro.size(); ++m)
            if (ro[m + 1] > ro[m]) add(ro[m], ro[m + 1]);
        std::stable_sort(h.begin(), h.end(), [&](const int4 &a, const int4 &b) {
            return rp[a.y] - rp[a.x] > rp[b.y] - rp[b.x];
        });
        if (h.empty()) h.push_back(make_int4(0, 0, 0, 0));
    }
    if (p->seg) CAP_HIP_TRY(hipFree(p->seg));
    p->seg = nullptr;
    CAP_TRY(dev_alloc(&p->seg, h.size()));
    CAP_HIP_TRY(hipMemcpy(p->seg, h.data(), sizeof(int4) * h.size(), hipMemcpyHostToDevice));
    p->n_seg = (int)h.size();
    return CAP_OK;
}

// LDS ring of k_local: the largest power of two R of slots (k values and a
// tag each) that fits the workgroup's LDS; returns log2(R), bytes in *bytes.
template <typename T>
int local_ring_log2(const cap_plan p, int rhs, size_t *bytes)
{
    const size_t slot = (size_t)rhs * sizeof(typename VBits<T>::U) + sizeof(int);
    const size_t budget = (size_t)std::max(0, p->lds_max - kLocalStaticLds);
    int l = 0;
    while ((slot << (l + 1)) <= budget && l < 24) ++l;
    *bytes = slot << l;
    return l;
}

// Protocol state of a launch over `count` values; nullptr-ready unless the
// value protocol is staged.  A staged array smaller than count means the
// launch was not preceded by its reset.
template <typename T>
int sync_ctx(cap_plan p, int sync, long long count, SyncCtx *sc)
{
    *sc = SyncCtx{p->flags, p->epoch, p->spin_limit, p->err, nullptr, p->unfused, p->wait_ticks};
    if (sync == CAP_SYNC_VALUE && p->staged) {
        if (!p->ready || p->ready_bytes < sizeof(typename VBits<T>::U) * (size_t)count) return CAP_ERR_ARG;
        sc->ready = p->ready;
    }
    return CAP_OK;
}

// The partitioned solve's work vectors for k right-hand sides.  Growing them
// waits for the device (earlier solves may still use the old ones), so a
// caller that captures solves into a graph runs one uncaptured solve with its
// largest k first.
int ensure_part_rhs(cap_plan p, int k)
{
    PartState *ps = p->part;
    if (k <= ps->kcap) return CAP_OK;
    CAP_HIP_TRY(hipDeviceSynchronize());
    for (double **v : {&ps->a, &ps->u, &ps->t, &ps->c0, &ps->c1, &ps->res, &ps->cor}) {
        if (*v) (void)hipFree(*v);
        *v = nullptr;  // res / cor come back at the new size when a refined solve needs them
    }
    if (ps->top) (void)hipFree(ps->top);
    ps->top = nullptr;
    ps->kcap = 0;
    const size_t tails = (size_t)ps->Q * k * ps->W, carries = (size_t)ps->G * k * ps->W;
    CAP_TRY(dev_alloc(&ps->a, tails));
    CAP_TRY(dev_alloc(&ps->t, tails));
    CAP_TRY(dev_alloc(&ps->top, (size_t)ps->Q * k * 2));
    if (!ps->walk) {
        CAP_TRY(dev_alloc(&ps->u, tails));
        CAP_TRY(dev_alloc(&ps->c0, carries));
        CAP_TRY(dev_alloc(&ps->c1, carries));
    }
    ps->kcap = k;
    return CAP_OK;
}

// Right-hand sides per wavefront of a sweep, at most (they share the row
// data; each adds an independent chain and 2W LDS slots).
constexpr int kPartSweepRhs = 4;

// The largest power of two up to `cap` that divides k: the chunk of
// right-hand sides one workgroup takes.
inline int part_chunk(int k, int cap)
{
    int c = 1;
    while (c < cap && k % (2 * c) == 0) c *= 2;
    return c;
}

// One sweep over `blocks` blocks, k right-hand sides (KR | k) of them to a
// wavefront.  The grid's x is rounded up to the 8 XCDs, so that the
// wavefronts of a block's right-hand sides share an L2.
template <int W, int KR, typename T, PartSweep MODE>
void launch_part_sweep(const PartState *ps, int n, const T *b, const double *hist, double *tails, T *x, int k,
                       int blocks, hipStream_t st)
{
    const int waves = part_chunk(k / KR, kPartWaves);
    const dim3 grid((unsigned)((blocks + 7) / 8 * 8), (unsigned)(k / KR / waves));
    auto go = [&](auto j) {
        k_part_sweep<W, KR, decltype(j)::value, T, MODE>
            <<<grid, waves * kWave, 0, st>>>(ps->rec, ps->at, ps->first, b, hist, tails, ps->top, x, n, ps->m, k, blocks);
    };
    switch (ps->J) {
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    default: go(std::integral_constant<int, kPartMaxJ>{}); break;
    }
}

template <int W, typename T, PartSweep MODE>
void part_sweep(const PartState *ps, int n, int kr, const T *b, const double *hist, double *tails, T *x, int k,
                int blocks, hipStream_t st)
{
    switch (kr) {
    case 4: launch_part_sweep<W, 4, T, MODE>(ps, n, b, hist, tails, x, k, blocks, st); break;
    case 2: launch_part_sweep<W, 2, T, MODE>(ps, n, b, hist, tails, x, k, blocks, st); break;
    default: launch_part_sweep<W, 1, T, MODE>(ps, n, b, hist, tails, x, k, blocks, st); break;
    }
}

// Right-hand sides per wavefront without a tuned pick: n = 200,000, bandwidth
// 96, four of them: one 80 us, two 100; eight: 140, two 114, four 159.
inline int part_sweep_rhs(int k) { return part_chunk(k, std::min(kPartSweepRhs, std::max(1, k / kPartWaves))); }

// Right-hand sides per workgroup of the group scan and the carry rounds, at
// most: those grids have only G (= P / gs) workgroups per chunk, and each step
// of a workgroup is a chain, so they keep more, smaller chunks than the
// fix-up (Q workgroups), which takes 16 (8 at W = 256).  The walk's products
// are a chain too.
constexpr int kPartScanRhs = 4;

// The tail scan over the group carries, KQ right-hand sides per workgroup
// (KQ | k); returns the buffer that holds the scanned carries.  NT: the
// matrices are read with non-temporal loads, when one chunk covers every
// RHS and each matrix is read once (with several chunks, cached reads let
// later chunks reuse them).
template <int W, int KQ, bool NT>
double *part_carries(cap_plan p, int k, hipStream_t st)
{
    const PartState *ps = p->part;
    const int Q = ps->Q;
    const unsigned chunks = (unsigned)(k / KQ);
    const long long mat = (long long)W * W;
    k_part_group_scan<W, KQ, NT><<<dim3(ps->G, chunks), kPartSplit * W, 0, st>>>(ps->a, ps->u, ps->c0, ps->bm,
                                                                                 ps->gs, Q, k);
    double *cur = ps->c0, *nxt = ps->c1;
    for (int r = 0; r < ps->rounds; ++r) {
        k_part_scan<W, KQ, NT><<<dim3(ps->G * kPartSplit, chunks), W, 0, st>>>(
            cur, nxt, ps->bm + ps->m_off[(size_t)r] * mat, 1 << r, k);
        std::swap(cur, nxt);
    }
    return cur;
}

template <int W, int KQ>
double *launch_part_carries(cap_plan p, int k, hipStream_t st)
{
    return k == KQ ? part_carries<W, KQ, true>(p, k, st) : part_carries<W, KQ, false>(p, k, st);
}

// The fix-up of every tail, KQ right-hand sides per workgroup (KQ | k);
// `tg`: the scanned group carries.
template <int W, int KQ>
void launch_part_fix(cap_plan p, const double *tg, int k, hipStream_t st)
{
    const PartState *ps = p->part;
    const dim3 grid((unsigned)ps->Q, (unsigned)(k / KQ));
    const double *wm = ps->bm + ps->w_off * W * W;
    if (k == KQ)  // non-temporal matrix reads when each W_p is read once
        k_part_fixup<W, KQ, true><<<grid, W, 0, st>>>(ps->u, tg, wm, ps->gs, ps->t, k);
    else
        k_part_fixup<W, KQ, false><<<grid, W, 0, st>>>(ps->u, tg, wm, ps->gs, ps->t, k);
}

// One workgroup per CU, about.  A run of tails walks to its first one and
// takes one product for each further one, so fewer and longer runs read fewer
// matrices.  Whatever k: the runs set where walks start, and so a right-hand
// side's bits.
template <int W, int KQ>
void launch_part_walk(cap_plan p, int k, hipStream_t st)
{
    const PartState *ps = p->part;
    const int run = (ps->Q + p->ncu - 1) / p->ncu;
    k_part_walk<W, KQ><<<dim3((unsigned)(((ps->Q + run - 1) / run + 7) / 8 * 8), (unsigned)(k / KQ)), kPartSplit * W, 0, st>>>(
        ps->a, ps->top, ps->bm, ps->fade, ps->t, ps->Q, run, k);
}

// One solve of a partitioned plan (k FP64 right-hand sides, interleaved:
// b[row * k + q]): the sweep for the block tails, the tails joined (walked,
// or the scan in groups, over the group carries and the fix-up; grids over
// tails x chunks), and the sweep for x.  Every step is on `st`; none of them
// waits on another workgroup.  Each right-hand side gets the bits of its own
// one-RHS solve.  x may be b: a block's rows of b are read before they are
// written, by the same wavefront.
template <int W, typename T>
int launch_partition_w(cap_plan p, const T *b, T *x, int k, hipStream_t st)
{
    // right-hand sides per wavefront: the plan's tuned pick for k when it has
    // one, else as many as leave a workgroup's wavefronts work
    const PartState *ps = p->part;
    int kr = part_sweep_rhs(k);
    if (p->part_kr > 0 && p->part_kr <= kPartSweepRhs && k % p->part_kr == 0) kr = p->part_kr;
    part_sweep<W, T, kPartTails>(ps, p->n, kr, b, nullptr, ps->a, (T *)nullptr, k, ps->Q, st);
    if (ps->walk) {
        switch (part_chunk(k, W == kPartW ? 2 * kPartScanRhs : kPartScanRhs)) {
        case 8:
            if constexpr (W == kPartW) launch_part_walk<W, 8>(p, k, st);
            break;
        case 4: launch_part_walk<W, 4>(p, k, st); break;
        case 2: launch_part_walk<W, 2>(p, k, st); break;
        default: launch_part_walk<W, 1>(p, k, st); break;
        }
    } else {
        const double *tg = nullptr;
        switch (part_chunk(k, kPartScanRhs)) {
        case 4: tg = launch_part_carries<W, 4>(p, k, st); break;
        case 2: tg = launch_part_carries<W, 2>(p, k, st); break;
        default: tg = launch_part_carries<W, 1>(p, k, st); break;
        }
        switch (part_chunk(k, W == kPartW ? 16 : 8)) {
        case 16:
            if constexpr (W == kPartW) launch_part_fix<W, 16>(p, tg, k, st);
            break;
        case 8: launch_part_fix<W, 8>(p, tg, k, st); break;
        case 4: launch_part_fix<W, 4>(p, tg, k, st); break;
        case 2: launch_part_fix<W, 2>(p, tg, k, st); break;
        default: launch_part_fix<W, 1>(p, tg, k, st); break;
        }
    }
    part_sweep<W, T, kPartX>(ps, p->n, kr, b, ps->t, nullptr, x, k, ps->P, st);
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

template <typename T>
int launch_partition(cap_plan p, const T *b, T *x, int k, hipStream_t st)
{
    PartState *ps = p->part;
    if (!ps || k < 1 || k > kWave || ps->m < ps->W) return CAP_ERR_ARG;
    CAP_TRY(ensure_part_rhs(p, k));
    if (ps->W == kPartWMax) return launch_partition_w<kPartWMax, T>(p, b, x, k, st);
    return launch_partition_w<kPartW, T>(p, b, x, k, st);
}

// Threads per workgroup of the fused refinement sweep for rhs right-hand
// sides: the plan's sweep size (128 or 256), or 1024 when the plan's solve
// uses 1024-thread workgroups for several right-hand sides (a batch's pick;
// tickets then hold 4 x the rows).
inline int refine_block(cap_plan p, int rhs)
{
    if (rhs > 1 && p->rblock == kBlockLarge && !p->lds) return kBlockLarge;
    return (p->rblock ? p->rblock : p->wblock) == kBlockSmall ? kBlockSmall : kBlock;
}

// A batch's block schedule for blocks of `rows` rows (nullptr if none was
// built for that size: the solve then hands out rows in plain order, which
// is correct, only without the relative-level pacing).
inline const int2 *sched_for(cap_plan p, int rows, int *n_sched)
{
    const auto it = p->scheds.find(rows);
    *n_sched = it == p->scheds.end() ? 0 : it->second.second;
    return it == p->scheds.end() ? nullptr : it->second.first;
}

// Applies the plan's RHS-block pick for k right-hand sides for the length
// of one launch (and puts the plan's own settings back).
struct RhsScope {
    cap_plan p;
    int bpc, block, kr, rpl, lds, tile;
    bool staged;
    RhsScope(cap_plan q, int k)
        : p(q), bpc(q->bpc), block(q->wblock), kr(q->part_kr), rpl(q->rpl), lds(q->lds), tile(q->tile),
          staged(q->staged)
    {
        const auto it = k > 1 ? p->rhs_pick.find(k) : p->rhs_pick.end();
        if (it == p->rhs_pick.end()) {
            if (k > 1 && p->plain.bpc && (!p->tune_rhs || p->reversed)) take(p->plain);
            if (k > 1 && p->fixed_rpl > 0) {  // cap_opts.rhs_per_lane
                p->bpc = 1;
                p->wblock = kBlockLarge;
                p->rpl = p->fixed_rpl;
            }
            return;
        }
        if (it->second.bpc) p->bpc = it->second.bpc;
        if (it->second.block) p->wblock = it->second.block;
        if (it->second.kr) p->part_kr = it->second.kr;
        if (it->second.rpl) p->rpl = it->second.rpl;
        if (it->second.staged >= 0) p->staged = it->second.staged != 0;
        if (it->second.lds >= 0) p->lds = it->second.lds;
        if (it->second.tile >= 0) p->tile = it->second.tile;
    }
    void take(const PlainShape &s)
    {
        p->bpc = s.bpc;
        p->wblock = s.block;
        p->lds = s.lds;
        p->tile = s.tile;
        p->staged = s.staged;
    }
    ~RhsScope()
    {
        p->bpc = bpc;
        p->wblock = block;
        p->part_kr = kr;
        p->rpl = rpl;
        p->lds = lds;
        p->tile = tile;
        p->staged = staged;
    }
};

// fused: accumulate with fused multiply-adds whatever the plan's arithmetic
// (the refinement's FP32 corrections, which belong to this library's own
// method and follow the oracle's fused steps).
template <typename T>
int launch_kernel(cap_plan p, int algo, int sync, const T *val, const T *b, T *x, int rhs, hipStream_t st,
                  bool fused = false)
{
    const int n = p->n;
    if (n == 0) return CAP_OK;
    const RhsScope scope(p, rhs);
    if (algo == CAP_ALGO_PARTITION) return launch_partition<T>(p, b, x, rhs, st);
    SyncCtx sc{p->flags, p->epoch, p->spin_limit, p->err, nullptr, p->unfused, p->wait_ticks};
    if (algo != CAP_ALGO_CSC && algo != CAP_ALGO_LOCAL && algo != CAP_ALGO_LEVEL)
        CAP_TRY(sync_ctx<T>(p, sync, (long long)n * rhs, &sc));
    if (fused) sc.unfused = 0;
    if (algo == CAP_ALGO_WRTFST && sync == CAP_SYNC_VALUE && hop_takes(p, rhs)) {
        const HopState *h = p->hop;
        const HopTab tab{h->base, h->ex, h->npad};
        const unsigned nb = grid_for(p, ((long long)n + p->wblock - 1) / p->wblock);
        auto go = [&](auto kernel) {
            kernel<<<nb, p->wblock, 0, st>>>(tab, val, b, x, sc, n, p->ticket, p->reversed ? n : 0);
        };
        const bool small = p->wblock == kBlockSmall;
        if (h->E == 2)
            small ? go(k_hop<T, 2, kBlockSmall>) : go(k_hop<T, 2, kBlock>);
        else if (h->E == 3)
            small ? go(k_hop<T, 3, kBlockSmall>) : go(k_hop<T, 3, kBlock>);
        else
            small ? go(k_hop<T, 4, kBlockSmall>) : go(k_hop<T, 4, kBlock>);
    } else if (algo == CAP_ALGO_WRTFST && p->rpl > 1 && rhs > 1) {  // several right-hand sides per lane
        if (rhs > kWave || sync != CAP_SYNC_VALUE || p->lds || p->count_polls) return CAP_ERR_UNSUPPORTED;
        const int l = lpr_log2_for((rhs + p->rpl - 1) / p->rpl);
        const int rows_per_block = p->wblock >> l;
        int n_sched = 0;
        const int2 *sched = sched_for(p, rows_per_block, &n_sched);
        const bool use_sched = sched != nullptr;
        const unsigned nb =
            grid_for(p, use_sched ? n_sched : ((long long)n + rows_per_block - 1) / rows_per_block);
        auto go = [&](auto kernel) {
            kernel<<<nb, p->wblock, 0, st>>>(p->rp, p->ci, val, b, x, sc, n, rhs, l, p->ticket, sched, n_sched);
        };
        // 8 FP64 right-hand sides per lane would spill at 1024 threads
        const int key = p->wblock * 16 + p->rpl;
        if (key == kBlockLarge * 16 + 2) go(k_wrtfst_r<T, kBlockLarge, 2>);
        else if (key == kBlockLarge * 16 + 4) go(k_wrtfst_r<T, kBlockLarge, 4>);
        else if (key == kBlock * 16 + 4) go(k_wrtfst_r<T, kBlock, 4>);
        else if constexpr (sizeof(T) == 4) {
            if (key == kBlockLarge * 16 + 8) go(k_wrtfst_r<T, kBlockLarge, 8>);
            else return CAP_ERR_UNSUPPORTED;
        } else {
            return CAP_ERR_UNSUPPORTED;
        }
    } else if (algo == CAP_ALGO_WRTFST) {
        if (rhs < 1 || rhs > kWave) return CAP_ERR_UNSUPPORTED;
        const int l = lpr_log2_for(rhs);
        const int rows_per_block = p->wblock >> l;
        // a batch's block schedule, when built for this block size
        int n_sched = 0;
        const int2 *sched = sched_for(p, rows_per_block, &n_sched);
        const bool use_sched = sched != nullptr;
        const unsigned nb =
            grid_for(p, use_sched ? n_sched : ((long long)n + rows_per_block - 1) / rows_per_block);
        auto go = [&](auto kernel) {
            kernel<<<nb, p->wblock, 0, st>>>(p->rp, p->ci, val, b, x, sc, n, rhs, l, p->ticket, 0, sched, n_sched);
        };
        const bool small = p->wblock == kBlockSmall;
        if (p->wblock == kBlockLarge) {  // the multi-RHS pick only
            if (sync != CAP_SYNC_VALUE || p->lds || p->count_polls || rhs < 2) return CAP_ERR_UNSUPPORTED;
            p->tile ? go(k_wrtfst<T, 1, 0, kBlockLarge, false, true>) : go(k_wrtfst<T, 1, 0, kBlockLarge>);
        } else if (sync == CAP_SYNC_VALUE && p->count_polls) {  // the counting instantiations
            sc.polls = reinterpret_cast<unsigned long long *>(p->ctrl + 1024);
            if (p->lds)
                small ? go(k_wrtfst<T, 1, 1, kBlockSmall, true>) : go(k_wrtfst<T, 1, 1, kBlock, true>);
            else
                small ? go(k_wrtfst<T, 1, 0, kBlockSmall, true>) : go(k_wrtfst<T, 1, 0, kBlock, true>);
        } else if (sync == CAP_SYNC_VALUE && p->tile && p->lds)
            small ? go(k_wrtfst<T, 1, 1, kBlockSmall, false, true>) : go(k_wrtfst<T, 1, 1, kBlock, false, true>);
        else if (sync == CAP_SYNC_VALUE && p->tile)
            small ? go(k_wrtfst<T, 1, 0, kBlockSmall, false, true>) : go(k_wrtfst<T, 1, 0, kBlock, false, true>);
        else if (sync == CAP_SYNC_VALUE && p->lds)
            small ? go(k_wrtfst<T, 1, 1, kBlockSmall>) : go(k_wrtfst<T, 1, 1, kBlock>);
        else if (sync == CAP_SYNC_VALUE)
            small ? go(k_wrtfst<T, 1, 0, kBlockSmall>) : go(k_wrtfst<T, 1, 0, kBlock>);
        else
            small ? go(k_wrtfst<T, 2, 0, kBlockSmall>) : go(k_wrtfst<T, 2, 0, kBlock>);
    } else if (algo == CAP_ALGO_TWOPART) {
        if (rhs != 1) return CAP_ERR_UNSUPPORTED;
        const unsigned nb = grid_for(p, ((long long)n + kBlock - 1) / kBlock);
        if (sync == CAP_SYNC_VALUE)
            k_twopart<T, 1><<<nb, kBlock, 0, st>>>(p->rp, p->ci, val, b, x, sc, n, p->ticket);
        else
            k_twopart<T, 2><<<nb, kBlock, 0, st>>>(p->rp, p->ci, val, b, x, sc, n, p->ticket);
    } else if (algo == CAP_ALGO_MIX) {
        if (rhs != 1) return CAP_ERR_UNSUPPORTED;
        constexpr int kMixBlock = 1024;  // 16 units per ticket share an LDS window
        const unsigned nb = std::min(grid_for(p, ((long long)p->n_units * kWave + kMixBlock - 1) / kMixBlock),
                                     (unsigned)(p->ncu * kMixBlocks));
        if (sync == CAP_SYNC_VALUE && p->tile)
            k_mix<T, 1, kMixBlock, true><<<nb, kMixBlock, 0, st>>>(p->rp, p->ci, val, b, x, sc, p->unit,
                                                                   p->n_units, p->ticket);
        else if (sync == CAP_SYNC_VALUE)
            k_mix<T, 1, kMixBlock><<<nb, kMixBlock, 0, st>>>(p->rp, p->ci, val, b, x, sc, p->unit, p->n_units,
                                                             p->ticket);
        else
            k_mix<T, 2, kMixBlock><<<nb, kMixBlock, 0, st>>>(p->rp, p->ci, val, b, x, sc, p->unit, p->n_units,
                                                             p->ticket);
    } else if (algo == CAP_ALGO_LOCAL) {
        if (rhs < 1 || rhs > kWave) return CAP_ERR_UNSUPPORTED;
        CAP_TRY(ensure_segments(p, nullptr));
        const unsigned nb = (unsigned)std::max(1, std::min(p->n_seg, p->ncu * p->bpc));
        size_t bytes = 0;
        const int rl = local_ring_log2<T>(p, rhs, &bytes);
        k_local<T><<<nb, kLocalBlock, bytes, st>>>(p->rp, p->ci, val, b, x, sc, rhs, p->seg, p->n_seg, p->ticket,
                                                    rl);
    } else if (algo == CAP_ALGO_LEVEL) {
        // the plan's own values (the tables hold them)
        if (!level_takes(p, rhs) || (const void *)val != p->val) return CAP_ERR_UNSUPPORTED;
        if (p->lvl_live) CAP_TRY(steps_refresh(p->lvl, p->rp, p->ci, p->val, st));
        return steps_launch(p->lvl, b, x, rhs, sc.unfused != 0, st);
    } else if (algo == CAP_ALGO_CSC) {
        if (rhs != 1) return CAP_ERR_UNSUPPORTED;
        // lanes per column from the mean column length (diagonal included)
        const double avg = (double)p->nnz / std::max(1, n);
        const int G = avg <= 4.0 ? 4 : avg <= 16.0 ? 16 : kWave;
        const unsigned nb = grid_for(p, ((long long)n * G + kBlock - 1) / kBlock);
        const int *cp = p->cp, *cr = p->cri;
        const T *cv = (const T *)p->cv;
        if (G == 4)
            k_csc<T, 4><<<nb, kBlock, 0, st>>>(cp, cr, cv, p->deg, (T *)p->left_sum, b, x, n, 0, sc, p->ticket);
        else if (G == 16)
            k_csc<T, 16><<<nb, kBlock, 0, st>>>(cp, cr, cv, p->deg, (T *)p->left_sum, b, x, n, 0, sc, p->ticket);
        else
            k_csc<T, kWave><<<nb, kBlock, 0, st>>>(cp, cr, cv, p->deg, (T *)p->left_sum, b, x, n, 0, sc, p->ticket);
    } else {
        return CAP_ERR_UNSUPPORTED;
    }
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

// CSC executor reset: in-degrees restored, left sums cleared (kernels only).
template <typename T>
int launch_csc_reset(cap_plan p, hipStream_t st)
{
    typedef typename VBits<T>::U U;
    CAP_HIP_TRY(hipMemcpyAsync(p->deg, p->deg0, sizeof(int) * (size_t)p->n, hipMemcpyDeviceToDevice, st));
    k_prepare<U><<<blocks_for(p->n), kBlock, 0, st>>>((U *)p->left_sum, p->n, (U)0, p->ticket, kTickets);
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

template <typename T>
int solve_t(cap_plan p, int algo, int sync, const void *b, void *x, int rhs, hipStream_t st)
{
    const RhsScope scope(p, rhs);  // the reset and the launch see the same RHS-block pick
    if (algo == CAP_ALGO_CSC) {
        CAP_TRY(launch_csc_reset<T>(p, st));
    } else {
        CAP_TRY(launch_prepare<T>(p, algo, sync, x, (long long)p->n * rhs, st));
    }
    return launch_kernel<T>(p, algo, sync, (const T *)p->val, (const T *)b, (T *)x, rhs, st);
}

template <typename T>
int reset_t(cap_plan p, int algo, int sync, void *x, int rhs, hipStream_t st)
{
    const RhsScope scope(p, rhs);
    if (algo == CAP_ALGO_CSC) return launch_csc_reset<T>(p, st);
    return launch_prepare<T>(p, algo, sync, x, (long long)p->n * rhs, st);
}

// The algorithm and protocol that solve rhs right-hand sides: the plan's,
// except that an autotuned plan whose pick has no multi-RHS form (mix,
// two-part, CSC, level steps) solves several with the write-first kernel in the value
// protocol (its RHS block tuned like any other).  So do level plans whose b
// and x are more bytes than the steps address.
inline int algo_for(cap_plan p, int rhs)
{
    if (p->algo == CAP_ALGO_LEVEL && level_allows(p, rhs) && !steps_take(p->lvl, rhs) && rhs >= 1 && rhs <= kWave)
        return CAP_ALGO_WRTFST;
    if (p->algo == CAP_ALGO_LEVEL && rhs > 1) {
        const auto it = p->rhs_pick.find(rhs);
        if (it != p->rhs_pick.end() && it->second.rows) return CAP_ALGO_WRTFST;
    }
    if (rhs > 1 && p->auto_algo &&
        (p->algo == CAP_ALGO_MIX || p->algo == CAP_ALGO_TWOPART || p->algo == CAP_ALGO_CSC ||
         (p->algo == CAP_ALGO_LEVEL && !level_takes(p, rhs))))
        return CAP_ALGO_WRTFST;
    return p->algo;
}
inline int sync_for(cap_plan p, int rhs) { return algo_for(p, rhs) != p->algo ? CAP_SYNC_VALUE : p->sync; }

int plan_solve_with(cap_plan p, int algo, int sync, const void *b, void *x, int rhs, hipStream_t st)
{
    return p->vt == CAP_F64 ? solve_t<double>(p, algo, sync, b, x, rhs, st)
                            : solve_t<float>(p, algo, sync, b, x, rhs, st);
}

// ----------------------------------------------------------- plan analysis
int build_mix(cap_plan p, const std::vector<int> &rp_host, int border)
{
    std::vector<int> wn((size_t)p->n + 1);
    int len = 0;
    cap_matrix_warp4(p->n, p->nnz, rp_host.data(), border, kWave, &len, wn.data(), &p->wocc, &p->eocc);
    if (p->unit) CAP_HIP_TRY(hipFree(p->unit));
    p->unit = nullptr;
    CAP_TRY(dev_alloc(&p->unit, (size_t)len));
    CAP_HIP_TRY(hipMemcpy(p->unit, wn.data(), sizeof(int) * (size_t)len, hipMemcpyHostToDevice));
    p->mix_len = len;
    p->n_units = len - 1;
    p->border = border;
    return CAP_OK;
}

template <typename T>
int build_csc(cap_plan p, const std::vector<int> &rp_host, hipStream_t st)
{
    const int n = p->n, nnz = p->nnz;
    std::vector<int> ci((size_t)nnz), cp((size_t)n + 1), cr((size_t)nnz);
    std::vector<T> v((size_t)nnz), cv((size_t)nnz);
    CAP_HIP_TRY(hipMemcpy(ci.data(), p->ci, sizeof(int) * nnz, hipMemcpyDeviceToHost));
    CAP_HIP_TRY(hipMemcpy(v.data(), p->val, sizeof(T) * nnz, hipMemcpyDeviceToHost));
    if (sizeof(T) == 8)
        cap_transpose_d(n, n, nnz, rp_host.data(), ci.data(), (const double *)(const void *)v.data(), cr.data(),
                        cp.data(), (double *)(void *)cv.data());
    else
        cap_transpose_s(n, n, nnz, rp_host.data(), ci.data(), (const float *)(const void *)v.data(), cr.data(),
                        cp.data(), (float *)(void *)cv.data());
    CAP_TRY(dev_alloc(&p->cp, (size_t)n + 1));
    CAP_TRY(dev_alloc(&p->cri, (size_t)nnz));
    CAP_TRY(dev_alloc((T **)&p->cv, (size_t)nnz));
    CAP_TRY(dev_alloc(&p->deg0, (size_t)n));
    CAP_TRY(dev_alloc(&p->deg, (size_t)n));
    CAP_TRY(dev_alloc((T **)&p->left_sum, (size_t)n));
    CAP_HIP_TRY(hipMemcpy(p->cp, cp.data(), sizeof(int) * ((size_t)n + 1), hipMemcpyHostToDevice));
    CAP_HIP_TRY(hipMemcpy(p->cri, cr.data(), sizeof(int) * (size_t)nnz, hipMemcpyHostToDevice));
    CAP_HIP_TRY(hipMemcpy(p->cv, cv.data(), sizeof(T) * (size_t)nnz, hipMemcpyHostToDevice));
    k_prepare<unsigned><<<blocks_for(n), kBlock, 0, st>>>((unsigned *)p->deg0, n, 0u, p->ticket, 0);
    k_indegree<<<blocks_for(nnz), kBlock, 0, st>>>(p->cri, nnz, p->deg0);
    CAP_HIP_TRY(hipGetLastError());
    CAP_HIP_TRY(hipStreamSynchronize(st));
    return CAP_OK;
}

int ensure_csc(cap_plan p, hipStream_t st)
{
    if (p->cp) return CAP_OK;
    std::vector<int> rp((size_t)p->n + 1);
    CAP_HIP_TRY(hipMemcpy(rp.data(), p->rp, sizeof(int) * ((size_t)p->n + 1), hipMemcpyDeviceToHost));
    return p->vt == CAP_F64 ? build_csc<double>(p, rp, st) : build_csc<float>(p, rp, st);
}

// ----------------------------------------------------------- autotuner
// A pick is cached per matrix shape: size, value type, readiness, the
// dependency depth (level count), whether the plan owns the values (steps
// over the caller's copy them on every solve) and a hash of sampled row
// pointers and column indices.  Two matrices with one row-length profile but different
// dependencies (a chain and a wide-level matrix) never share a pick.
struct TuneKey {
    int n, nnz, vt, staged, unfused, count_polls, levels, owned;
    unsigned long long fp;
    bool operator<(const TuneKey &o) const
    {
        return std::tie(n, nnz, vt, staged, unfused, count_polls, levels, owned, fp) <
               std::tie(o.n, o.nnz, o.vt, o.staged, o.unfused, o.count_polls, o.levels, o.owned, o.fp);
    }
};
std::mutex g_tune_mu;
struct TuneChoice {
    int algo, sync, border, bpc, lds, staged, block, tile = 0, hop = 0;
    int width = 0;  // rows per step of the level steps
    PlainShape plain{};
    float lead = 0;
};
std::map<TuneKey, TuneChoice> g_tune_cache;

unsigned long long fingerprint(const std::vector<int> &rp, const std::vector<int> &ci)
{
    unsigned long long h = 1469598103934665603ULL;
    for (const std::vector<int> *a : {&rp, &ci}) {
        const size_t n = a->size();
        for (int s = 0; s < 257 && n; ++s) {
            h ^= (unsigned long long)(unsigned)(*a)[(n - 1) * (size_t)s / 256];
            h *= 1099511628211ULL;
        }
    }
    return h;
}

// The right-hand side candidates are timed on: all ones.  The dependency
// structure sets most kernels' time, but a partitioned solve of b = 0 has no
// tails to join: n = 2,000, bandwidth 250: under 36 us, and 67 with a dense b,
// against 36 by steps.
int tuning_rhs(cap_plan p, void *b, long long count, hipStream_t st)
{
    const unsigned nb = std::max(1u, std::min(blocks_for(count), 2048u));
    if (p->vt == CAP_F64)
        k_fill<unsigned long long><<<nb, kBlock, 0, st>>>((unsigned long long *)b, count, 0x3FF0000000000000ULL);
    else
        k_fill<unsigned><<<nb, kBlock, 0, st>>>((unsigned *)b, count, 0x3F800000u);
    return hipGetLastError() == hipSuccess ? CAP_OK : CAP_ERR_HIP;
}

// Best of three timed solves after one warm-up; stops early once a run is
// 1.5x slower than `bound` (the best candidate so far).
int time_candidate(cap_plan p, int algo, int sync, const void *b, void *x, int rhs, hipStream_t st, float bound,
                   float *ms)
{
    hipEvent_t e0, e1;
    CAP_HIP_TRY(hipEventCreate(&e0));
    CAP_HIP_TRY(hipEventCreate(&e1));
    float best = 1e30f;
    int rc = CAP_OK;
    for (int r = 0; r < 4 && rc == CAP_OK; ++r) {
        rc = plan_solve_with(p, algo, sync, b, x, rhs, st);
        if (rc != CAP_OK) break;
        (void)hipEventRecord(e0, st);
        rc = plan_solve_with(p, algo, sync, b, x, rhs, st);
        (void)hipEventRecord(e1, st);
        (void)hipEventSynchronize(e1);
        float t = 0;
        (void)hipEventElapsedTime(&t, e0, e1);
        if (r > 0) {
            best = std::min(best, t);
        } else if (t > 1.5f * bound) {  // the warm-up alone rules it out
            best = t;
            break;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = best;
    return rc;
}

// The RHS block of an autotuned plan for k > 1 right-hand sides, timed on
// the caller's b and x (x is overwritten by the solve that follows) the first
// time cap_plan_solve sees that k: thread-per-row plans time 1, 2 and 4
// workgroups per CU at 256 and 128 threads (how many rows, each with k
// lanes, poll at once), 1024-thread workgroups with 1, 2, 4 (8 in FP32)
// right-hand sides per lane, and the pick again with readiness in x;
// partitioned plans time 1, 2 and 4 right-hand sides per wavefront of the
// sweeps (the ones that divide k); level plans, where it may be close, the
// steps and then the thread-per-row shapes (not in a capture).  Every
// candidate gives the same bits.  The plan's own settings (PlainShape) are
// timed first and another must be 2 % faster to win.  Waits for the device
// (events).
int tune_rhs_block(cap_plan p, const void *b, void *x, int k, hipStream_t st)
{
    std::vector<RhsPick> cands;
    int algo = algo_for(p, k), sync = sync_for(p, k);
    const bool steps = algo == CAP_ALGO_LEVEL;
    float t_steps = 1e30f;
    if (steps) {
        // with k right-hand sides a step takes up to 1 + log2(k) / 5 as long
        // (100k band: 1.03, 1.2, 1.6, 1.9 and 2.2 with 2, 4, 8, 16 and 64),
        // the write-first kernel at least 3/4 of its time with one: only near
        // ties are timed
        if (p->plain.bpc == 0 || 0.75f * p->lvl_lead >= 1.0f + 0.2f * std::log2((float)k)) {
            p->rhs_pick[k] = RhsPick{};
            return CAP_OK;
        }
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(st, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) {
            (void)hipGetLastError();
            return CAP_OK;
        }
        CAP_TRY(time_candidate(p, algo, sync, b, x, k, st, t_steps, &t_steps));
        algo = CAP_ALGO_WRTFST;
        sync = CAP_SYNC_VALUE;
    }
    RhsScope own(p, 1);  // puts the plan's settings back
    if (p->plain.bpc) own.take(p->plain);
    if (algo == CAP_ALGO_WRTFST) {
        cands.push_back({p->bpc, p->wblock, 0});
        for (int blk : {kBlock, kBlockSmall})
            for (int bpc : {1, 2, 4})
                if (!(bpc == p->bpc && blk == p->wblock)) cands.push_back({bpc, blk, 0});
        // fewer tickets: 1024 threads (one workgroup per CU: 16 wavefronts,
        // as many as four of 256), and R right-hand sides per lane (R times
        // the rows per ticket); these run without the LDS window whatever the
        // plan's single-RHS pick
        if (sync == CAP_SYNC_VALUE && !p->count_polls) {
            cands.push_back({1, kBlockLarge, 0, 1, -1, 0, 0});
            cands.push_back({1, kBlockLarge, 0, 1, -1, 0, 1});  // the ticket's entries staged in LDS
            for (int r : {2, 4, 8})
                if (r <= k && (r < 8 || p->vt == CAP_F32)) cands.push_back({1, kBlockLarge, 0, r, -1, 0, 0});
            if (k >= 4) cands.push_back({1, kBlock, 0, 4, -1, 0, 0});
        }
    } else if (algo == CAP_ALGO_PARTITION) {
        const int dflt = part_sweep_rhs(k);
        cands.push_back({0, 0, dflt});
        for (int kr : {1, 2, 4})
            if (kr != dflt && k % kr == 0) cands.push_back({0, 0, kr});
    } else {
        p->rhs_pick[k] = RhsPick{};
        return CAP_OK;
    }
    const int bpc0 = p->bpc, blk0 = p->wblock, kr0 = p->part_kr, rpl0 = p->rpl, lds0 = p->lds, tile0 = p->tile;
    float best = 1e30f;
    RhsPick pick = cands[0];
    int rc = CAP_OK;
    for (size_t c = 0; c < cands.size() && rc == CAP_OK; ++c) {
        if (cands[c].bpc) p->bpc = cands[c].bpc;
        if (cands[c].block) p->wblock = cands[c].block;
        if (cands[c].rpl) p->rpl = cands[c].rpl;
        if (cands[c].lds >= 0) p->lds = cands[c].lds;
        if (cands[c].tile >= 0) p->tile = cands[c].tile;
        p->part_kr = cands[c].kr;
        float t = 0;
        rc = time_candidate(p, algo, sync, b, x, k, st, std::min(best, t_steps), &t);
        if (rc == CAP_OK && t < (c ? 0.98f : 1.0f) * best) {
            best = t;
            pick = cands[c];
        }
        p->bpc = bpc0;
        p->wblock = blk0;
        p->part_kr = kr0;
        p->rpl = rpl0;
        p->lds = lds0;
        p->tile = tile0;
    }
    // readiness in x itself for the pick: one store per value instead of
    // two (x and the staged copy), at k > 1 the larger share of the bytes
    if (rc == CAP_OK && algo == CAP_ALGO_WRTFST && sync == CAP_SYNC_VALUE && p->staged && !p->count_polls) {
        if (pick.bpc) p->bpc = pick.bpc;
        if (pick.block) p->wblock = pick.block;
        if (pick.rpl) p->rpl = pick.rpl;
        if (pick.lds >= 0) p->lds = pick.lds;
        if (pick.tile >= 0) p->tile = pick.tile;
        p->staged = false;
        float t = 0;
        rc = time_candidate(p, algo, sync, b, x, k, st, best, &t);
        p->staged = true;
        p->bpc = bpc0;
        p->wblock = blk0;
        p->rpl = rpl0;
        p->lds = lds0;
        p->tile = tile0;
        if (rc == CAP_OK && t < 0.98f * best) {
            best = t;
            pick.staged = 0;
        }
    }
    if (rc != CAP_OK) return rc;
    if (p->plain.bpc) {
        if (pick.staged < 0) pick.staged = p->plain.staged;
        if (pick.lds < 0) pick.lds = p->plain.lds;
        if (pick.tile < 0) pick.tile = p->plain.tile;
    }
    if (steps && best >= 0.98f * t_steps)
        pick = RhsPick{};
    else
        pick.rows = steps;
    p->rhs_pick[k] = pick;
    return CAP_OK;
}

void apply_choice(cap_plan p, const TuneChoice &c)
{
    p->algo = c.algo;
    p->sync = c.sync;
    p->bpc = c.bpc;
    p->lds = c.lds;
    p->staged = c.staged;
    p->wblock = c.block;
    p->tile = c.tile;
    p->plain = c.plain;
    p->lvl_lead = c.lead;
}

// Tables of the partitioned banded solve (CAP_ALGO_PARTITION), built once:
// plans whose lower bandwidth is at most kPartWMax and that split into at
// least two blocks; CAP_ERR_UNSUPPORTED otherwise.  The tail width W is 128
// when the bandwidth allows, else 256.  Blocks hold at least W and n /
// kPartBlocks rows, and more, kPartRows (twice that at W = 256, whose matrices
// are four times the bytes: n = 158,094, 16 right-hand sides 640 -> 277 us) or
// n / kPartSpread, where that leaves 16 blocks: a sweep takes about 0.2 us per 8 rows of a block, 14 us for 512
// rows, and its bytes take 0.1 us per 1000 rows of the matrix, so up to n /
// kPartSpread rows cost nothing, while fewer blocks are fewer matrices to
// read and more damping in each.  Blocks that damp too little to be walked
// are made longer, up to kPartLongest rows, when that is enough (n = 200,000,
// bandwidth 128, 13 entries a row: 640 rows and the scan 107 us, 720 rows and
// the walk 72, 1440 rows 96).  The blocks' number is brought down to a whole
// multiple of the compute units where that takes a quarter more rows at most,
// as the last round of workgroups is as long as a full one: n = 140,000, 274
// or 256 blocks: 63 and 59 us, with 8 right-hand sides 112 and 87; half as
// many rows again did not pay (n = 200,000, 391 or 256 blocks: 66 and 74).  A
// matrix whose blocks grow (refused at that size) is tried with the smallest.
// The host groups the rows into records; the records are filled, the B_p
// swept and the scan's matrices formed on the device.
constexpr int kPartBlocks = 1024;
constexpr int kPartRows = 512;
constexpr int kPartSpread = 500;
constexpr int kPartLongest = 1280;
// largest relative max-norm difference from the sequential solve accepted
// when the tables are checked at plan creation (the FP64 bar is 1e-12)
constexpr double kPartStableTol = 1e-13;
constexpr int kPartGroup = 8;  // tails per group of the scan's first level
// Largest table set a partitioned plan may hold: larger matrices are refused
// rather than risk exhausting memory behind the caller's back.
constexpr double kPartMaxBytes = 16.0 * (1ull << 30);

// The matrix a plan's records are made of: the plan's own, or, when a row has
// more entries than a record (duplicates), a copy with the duplicates added up.
struct PartRows {
    std::vector<int> rp, ci;
    std::vector<double> v;
};

int build_partition_tables(cap_plan p, const PartRows &mat, int w, int m, bool merged, int *longer, hipStream_t st);

int build_partition(cap_plan p, const std::vector<int> &rp_host, hipStream_t st)
{
    if (p->part) return CAP_OK;
    try {
        const int n = p->n, nnz = p->nnz;
        PartRows mat;
        mat.rp = rp_host;
        mat.ci.resize((size_t)nnz);
        CAP_HIP_TRY(hipMemcpy(mat.ci.data(), p->ci, sizeof(int) * (size_t)nnz, hipMemcpyDeviceToHost));
        int w = 0, longest = 0;
        for (int i = 0; i < n; ++i) {
            longest = std::max(longest, mat.rp[i + 1] - mat.rp[i]);
            for (int j = mat.rp[i]; j < mat.rp[i + 1]; ++j) w = std::max(w, i - mat.ci[j]);
        }
        if (w > kPartWMax) return CAP_ERR_UNSUPPORTED;
        mat.v.resize((size_t)nnz);  // FP32 values widen exactly
        if (p->vt == CAP_F64) {
            CAP_HIP_TRY(hipMemcpy(mat.v.data(), p->val, sizeof(double) * (size_t)nnz, hipMemcpyDeviceToHost));
        } else {
            std::vector<float> vf((size_t)nnz);
            CAP_HIP_TRY(hipMemcpy(vf.data(), p->val, sizeof(float) * (size_t)nnz, hipMemcpyDeviceToHost));
            for (size_t e = 0; e < vf.size(); ++e) mat.v[e] = (double)vf[e];
        }
        const bool merged = longest > kPartSeg * kPartSeg * kPartMaxJ;
        if (merged) {
            PartRows u;
            std::vector<double> sum((size_t)w + 1);
            std::vector<char> has((size_t)w + 1);
            u.rp.push_back(0);
            for (int i = 0; i < n; ++i) {
                std::fill(sum.begin(), sum.end(), 0.0);
                std::fill(has.begin(), has.end(), 0);
                for (int j = mat.rp[i]; j < mat.rp[i + 1]; ++j) {
                    sum[(size_t)(i - mat.ci[j])] += mat.v[(size_t)j];
                    has[(size_t)(i - mat.ci[j])] = 1;
                }
                for (int d = std::min(i, w); d >= 0; --d) {
                    if (!has[(size_t)d]) continue;
                    u.ci.push_back(i - d);
                    u.v.push_back(sum[(size_t)d]);
                }
                u.rp.push_back((int)u.ci.size());
            }
            mat = std::move(u);
        }
        const int W = w <= kPartW ? kPartW : kPartWMax;
        const int least = std::max(W, (n + kPartBlocks - 1) / kPartBlocks);
        int m = std::max(least, std::min(std::max(kPartRows * (W / kPartW), n / kPartSpread), (n + 15) / 16));
        // whole rounds of the compute units, where a quarter more rows give them
        const int rounds = n / m / p->ncu;
        if (rounds > 0 && n / m % p->ncu > 0) {
            const int even = (n + rounds * p->ncu - 1) / (rounds * p->ncu);
            if (even <= m + m / 4) m = std::max(m, even);
        }
        int longer = 0;
        int rc = build_partition_tables(p, mat, w, m, merged, &longer, st);
        if (longer > 0) rc = build_partition_tables(p, mat, w, longer, merged, nullptr, st);
        if (rc == CAP_ERR_UNSUPPORTED && m > least) rc = build_partition_tables(p, mat, w, least, merged, nullptr, st);
        return rc;
    } catch (const std::bad_alloc &) {
        free_partition(p);
        return CAP_ERR_ALLOC;
    }
}

template <int J, typename T>
void fill_records(const int *rp, const int *ci, const T *val, const int *rows, int count, PartState *ps, hipStream_t st)
{
    k_part_records<J, T><<<(unsigned)count, kWave, 0, st>>>(rp, ci, val, rows, ps->at, ps->m, ps->rec);
}
template <typename T>
void fill_records(const int *rp, const int *ci, const T *val, const int *rows, int count, PartState *ps, hipStream_t st)
{
    switch (ps->J) {
    case 2: fill_records<2, T>(rp, ci, val, rows, count, ps, st); break;
    case 4: fill_records<4, T>(rp, ci, val, rows, count, ps, st); break;
    default: fill_records<kPartMaxJ, T>(rp, ci, val, rows, count, ps, st); break;
    }
}

// The norms of B_q (one[q], q >= 1) and of B_q B_{q-1} B_{q-2} B_{q-3}
// (four[q], q >= 4); B_q at bm + (q - 1) W^2.  Waits for st.
template <int W>
int part_norms(const double *bm, int Q, double *one, double *four, hipStream_t st)
{
    double *prod = nullptr, *norm = nullptr;
    int3 *d_ops = nullptr;
    const long long mat = (long long)W * W;
    const int B = Q - 1;
    std::vector<int3> ops;  // pairs behind the copies of the B_q, then fours behind the pairs
    for (int q = 2; q < Q; ++q) ops.push_back(make_int3(B + q - 1, q - 1, q - 2));
    const int pairs = (int)ops.size();
    for (int q = 4; q < Q; ++q) ops.push_back(make_int3(2 * B + q - 1, B + q - 1, B + q - 3));
    const int fours = (int)ops.size() - pairs;
    int rc = CAP_OK;
    do {
        if ((rc = dev_alloc(&norm, (size_t)(2 * B))) || (rc = dev_alloc(&prod, (size_t)(3 * B * mat))) ||
            (rc = dev_alloc(&d_ops, std::max<size_t>(1, ops.size()))))
            break;
        rc = CAP_ERR_HIP;
        if (hipMemcpyAsync(prod, bm, sizeof(double) * (size_t)(B * mat), hipMemcpyDeviceToDevice, st) != hipSuccess ||
            hipMemcpy(d_ops, ops.data(), sizeof(int3) * ops.size(), hipMemcpyHostToDevice) != hipSuccess)
            break;
        const unsigned quads = (W / 128) * (W / 128);
        if (pairs > 0) k_part_gemm<W><<<dim3((unsigned)pairs, quads), 256, 0, st>>>(d_ops, prod);
        if (fours > 0) k_part_gemm<W><<<dim3((unsigned)fours, quads), 256, 0, st>>>(d_ops + pairs, prod);
        k_part_norm<W><<<(unsigned)B, W, 0, st>>>(prod, norm);
        if (fours > 0) k_part_norm<W><<<(unsigned)fours, W, 0, st>>>(prod + (2LL * B + 3) * mat, norm + B);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess ||
            hipMemcpy(one + 1, norm, sizeof(double) * (size_t)B, hipMemcpyDeviceToHost) != hipSuccess ||
            (fours > 0 &&
             hipMemcpy(four + 4, norm + B, sizeof(double) * (size_t)fours, hipMemcpyDeviceToHost) != hipSuccess))
            break;
        rc = CAP_OK;
    } while (0);
    (void)hipStreamSynchronize(st);
    for (void *t : {(void *)norm, (void *)prod, (void *)d_ops})
        if (t) (void)hipFree(t);
    return rc;
}
int part_norms(const double *bm, int W, int Q, double *one, double *four, hipStream_t st)
{
    if (Q < 2) return hipGetLastError() == hipSuccess && hipStreamSynchronize(st) == hipSuccess ? CAP_OK : CAP_ERR_HIP;
    return W == kPartWMax ? part_norms<kPartWMax>(bm, Q, one, four, st) : part_norms<kPartW>(bm, Q, one, four, st);
}

int build_partition_tables(cap_plan p, const PartRows &mat, int w, int m, bool merged, int *longer, hipStream_t st)
{
    const int n = p->n, nnz = (int)mat.ci.size();
    const std::vector<int> &rp_host = mat.rp, &ci = mat.ci;
    const std::vector<double> &v = mat.v;
    const int W = w <= kPartW ? kPartW : kPartWMax;
    const int P = n > 0 ? (n + m - 1) / m : 0;
    if (P < 2) return CAP_ERR_UNSUPPORTED;
    // entries per lane: the fewest bytes, as if all of a row's entries but
    // the last were outside its record; a row fits one record
    int J = 0;
    double best = 0.0;
    for (int j = 2; j <= kPartMaxJ; j += 2) {
        double segs = 0.0;
        int most = 0;
        for (int i = 0; i < n; ++i) {
            const int s = std::max(1, (rp_host[i + 1] - rp_host[i] - 2 + kPartSeg * j - 1) / (kPartSeg * j));
            segs += s;
            most = std::max(most, (rp_host[i + 1] - rp_host[i] - 1 + kPartSeg * j - 1) / (kPartSeg * j));
        }
        const double cost = segs * part_pieces(j);
        if (most <= kPartSeg && (J == 0 || cost < best)) {
            J = j;
            best = cost;
        }
    }
    if (J == 0) return CAP_ERR_UNSUPPORTED;
    // the records: as many of a block's next rows as their segments fit
    std::vector<int> rows, at{0};
    std::vector<uint2> first;
    for (int q = 0; q < P; ++q) {
        const int end = (int)std::min<long long>(n, (long long)(q + 1) * m);
        for (int i = q * m; i < end;) {
            const int r0 = i;
            rows.push_back(r0);
            for (int segs = 0; i < end && i < r0 + kPartSeg; ++i) {
                int out = 0;
                for (int j = rp_host[i]; j < rp_host[i + 1]; ++j) out += ci[j] < r0;
                segs += std::max(1, (out + kPartSeg * J - 1) / (kPartSeg * J));
                if (segs > kPartSeg) break;
            }
        }
        unsigned f[2] = {0, 0};
        for (int d = 0; d < kPartAhead && at.back() + d < (int)rows.size(); ++d)
            f[d / 4] |= (unsigned)(rows[(size_t)(at.back() + d)] - q * m) << (8 * (d % 4));
        first.push_back(make_uint2(f[0], f[1]));
        at.push_back((int)rows.size());
    }
    const int n_rec = (int)rows.size();
    rows.push_back(n);
    // the tail scan's matrix count: B (Q - 1), W (Q - gs), carry rounds
    const int Q = P - 1, gs = kPartGroup, G = (Q + gs - 1) / gs;
    int rounds = 0;
    while ((1 << rounds) < G) ++rounds;
    std::vector<long long> m_off((size_t)rounds + 1);
    const long long w_off = Q - 1;
    m_off[0] = w_off + std::max(0, Q - gs);
    for (int r = 0; r < rounds; ++r) m_off[(size_t)r + 1] = m_off[(size_t)r] + (G - (1 << r));
    const long long n_mat = m_off[(size_t)rounds], mat_len = (long long)W * W;
    const size_t rec_len = (size_t)n_rec * part_pieces(J) * kWave;
    if ((double)rec_len * 16.0 + (double)n_mat * mat_len * 8.0 + 12.0 * nnz > kPartMaxBytes)
        return CAP_ERR_UNSUPPORTED;
    PartState *ps = new PartState();
    p->part = ps;  // freed by free_partition on every failure from here on
    ps->W = W;
    ps->m = m;
    ps->J = J;
    ps->P = P;
    ps->Q = Q;
    ps->gs = gs;
    ps->G = G;
    ps->rounds = rounds;
    ps->w_off = w_off;
    ps->m_off = m_off;
    int *d_rows = nullptr, *d_rp = nullptr, *d_ci = nullptr;
    double *d_v = nullptr, *bm = nullptr;
    int3 *d_ops = nullptr;
    int rc = CAP_OK;
    do {
        if ((rc = dev_alloc(&ps->rec, rec_len)) || (rc = dev_alloc(&ps->at, at.size())) ||
            (rc = dev_alloc(&ps->first, first.size())) || (rc = dev_alloc(&d_rows, rows.size())) ||
            (rc = dev_alloc(&ps->fade, (size_t)Q)) ||
            (Q > 1 && (rc = dev_alloc(&bm, (size_t)((Q - 1) * mat_len)))))
            break;
        ps->bm = bm;
        rc = CAP_ERR_HIP;
        if (hipMemcpy(ps->at, at.data(), sizeof(int) * at.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(ps->first, first.data(), sizeof(uint2) * first.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(d_rows, rows.data(), sizeof(int) * rows.size(), hipMemcpyHostToDevice) != hipSuccess)
            break;
        if (merged) {
            if ((rc = dev_alloc(&d_rp, rp_host.size())) || (rc = dev_alloc(&d_ci, ci.size())) ||
                (rc = dev_alloc(&d_v, v.size())))
                break;
            rc = CAP_ERR_HIP;
            if (hipMemcpy(d_rp, rp_host.data(), sizeof(int) * rp_host.size(), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(d_ci, ci.data(), sizeof(int) * ci.size(), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(d_v, v.data(), sizeof(double) * v.size(), hipMemcpyHostToDevice) != hipSuccess)
                break;
            fill_records<double>(d_rp, d_ci, d_v, d_rows, n_rec, ps, st);
        } else if (p->vt == CAP_F64) {
            fill_records<double>(p->rp, p->ci, (const double *)p->val, d_rows, n_rec, ps, st);
        } else {
            fill_records<float>(p->rp, p->ci, (const float *)p->val, d_rows, n_rec, ps, st);
        }
        if (Q > 1) {
            if (W == kPartWMax)
                launch_part_sweep<kPartWMax, kPartSweepRhs, double, kPartUnit>(ps, n, nullptr, nullptr, bm, nullptr, W,
                                                                               Q - 1, st);
            else
                launch_part_sweep<kPartW, kPartSweepRhs, double, kPartUnit>(ps, n, nullptr, nullptr, bm, nullptr, W,
                                                                            Q - 1, st);
        }
        std::vector<double> one((size_t)Q), four((size_t)Q);
        if ((rc = part_norms(bm, W, Q, one.data(), four.data(), st)) != CAP_OK) break;
        double worst = 0.0;  // of four blocks in a row
        for (int q = 4; q < Q; ++q) worst = four[(size_t)q] <= worst ? worst : four[(size_t)q];
        bool finite = true;
        for (int q = 1; q < Q; ++q) finite = finite && one[(size_t)q] < 0x1p1000 && four[(size_t)q] < 0x1p1000;
        ps->walk = finite && (worst <= kPartDamp || Q <= kPartGroup);
        if (!ps->walk && longer && worst < 0.0625 && n >= 16 * kPartLongest) {
            const int rows_of = (int)std::ceil(m * 36.0 / -std::log2(worst));
            if (rows_of <= kPartLongest) {
                *longer = rows_of;
                rc = CAP_ERR_UNSUPPORTED;
                break;
            }
        }
        std::vector<uint2> fade((size_t)Q, make_uint2(0u, 0u));
        auto log256 = [](double v) { return (unsigned)(int)std::ceil(256.0 * std::log2(std::max(v, 0x1p-1022))); };
        for (int q = 1; q < Q && ps->walk; ++q) {
            fade[(size_t)q].x = fade[(size_t)q - 1].x + log256(one[(size_t)q]);
            if (q >= 4) fade[(size_t)q].y = fade[(size_t)q - 4].y + log256(four[(size_t)q]);
        }
        rc = CAP_ERR_HIP;
        if (hipMemcpy(ps->fade, fade.data(), sizeof(uint2) * (size_t)Q, hipMemcpyHostToDevice) != hipSuccess) break;
        rc = CAP_OK;
        if (ps->walk) break;
        // the scan's products, launch by launch (each list depends on the one
        // before): the in-group products W_p = B_p W_{p-1} (W_first = B_first)
        // for groups g >= 1, the carries' first-round matrices (the W of each
        // group's last tail), then each carry round's products
        std::vector<std::vector<int3>> launches;
        for (int j = 0; j < gs; ++j) {
            std::vector<int3> ops;
            for (int g = 1; g * gs + j < Q; ++g) {
                const int q = g * gs + j;
                ops.push_back(j == 0 ? make_int3((int)(w_off + q - gs), q - 1, -1)
                                     : make_int3((int)(w_off + q - gs), q - 1, (int)(w_off + q - 1 - gs)));
            }
            if (!ops.empty()) launches.push_back(ops);
        }
        {
            std::vector<int3> ops;
            for (int g = 1; g < G; ++g) {
                const int last = std::min(Q, (g + 1) * gs) - 1;
                ops.push_back(make_int3((int)(m_off[0] + g - 1), (int)(w_off + last - gs), -1));
            }
            if (!ops.empty()) launches.push_back(ops);
        }
        for (int r = 0; r + 1 < rounds; ++r) {
            std::vector<int3> ops;
            const int s = 1 << r;
            for (int g = 2 * s; g < G; ++g)
                ops.push_back(make_int3((int)(m_off[(size_t)r + 1] + g - 2 * s), (int)(m_off[(size_t)r] + g - s),
                                        (int)(m_off[(size_t)r] + g - 2 * s)));
            if (!ops.empty()) launches.push_back(ops);
        }
        std::vector<int3> all_ops;
        std::vector<size_t> op_start;
        for (const auto &l : launches) {
            op_start.push_back(all_ops.size());
            all_ops.insert(all_ops.end(), l.begin(), l.end());
        }
        if (all_ops.empty()) break;
        // the same B_p, at the head of a larger set
        if ((rc = dev_alloc(&ps->bm, (size_t)(n_mat * mat_len)))) break;
        if ((rc = dev_alloc(&d_ops, all_ops.size()))) break;
        rc = CAP_ERR_HIP;
        if (hipMemcpy(ps->bm, bm, sizeof(double) * (size_t)((Q - 1) * mat_len), hipMemcpyDeviceToDevice) != hipSuccess ||
            hipMemcpy(d_ops, all_ops.data(), sizeof(int3) * all_ops.size(), hipMemcpyHostToDevice) != hipSuccess)
            break;
        const unsigned quads = (unsigned)((W / 128) * (W / 128));
        for (size_t l = 0; l < launches.size(); ++l) {
            const dim3 grid((unsigned)launches[l].size(), quads);
            if (W == kPartWMax)
                k_part_gemm<kPartWMax><<<grid, 256, 0, st>>>(d_ops + op_start[l], ps->bm);
            else
                k_part_gemm<kPartW><<<grid, 256, 0, st>>>(d_ops + op_start[l], ps->bm);
        }
        if (hipGetLastError() == hipSuccess && hipStreamSynchronize(st) == hipSuccess) rc = CAP_OK;
    } while (0);
    (void)hipStreamSynchronize(st);
    for (void *t : {(void *)d_rows, (void *)d_rp, (void *)d_ci, (void *)d_v, (void *)d_ops})
        if (t) (void)hipFree(t);
    if (bm && bm != ps->bm) (void)hipFree(bm);
    // Accuracy check against the sequential solve.  The records and the B_p
    // multiply by inverses of diagonal blocks, which the sequential solve never
    // forms; when the blocks are not diagonally dominant their entries grow
    // along a block (unit values in a band, as the reference's .mtx reader
    // makes them, grow as 1.47^m) and the sums cancel.  The tables solve two
    // right-hand sides -- b = L 1 (row sums in FP64) and a seeded U[-1,1] b
    // -- and each must agree with a sequential FP64 forward substitution of
    // the same system on the host to kPartStableTol relative max-norm, ten
    // times inside the FP64 bar of 1e-12; otherwise the matrix is refused.
    if (rc == CAP_OK) {
        std::vector<double> bh((size_t)n * 2), xs((size_t)n * 2), xr((size_t)n * 2);
        cap_uniform_d(0x5eedULL, n, -1.0, 1.0, xr.data());  // reused below as the reference solution
        for (int i = 0; i < n; ++i) {
            double rs = 0.0;
            for (int j = rp_host[i]; j < rp_host[i + 1]; ++j) rs += v[(size_t)j];
            bh[(size_t)i * 2] = rs;
            bh[(size_t)i * 2 + 1] = xr[(size_t)i];
        }
        for (int i = 0; i < n; ++i) {
            const int d = rp_host[i + 1] - 1;
            for (int q = 0; q < 2; ++q) {
                double sum = 0.0;
                for (int j = rp_host[i]; j < d; ++j) sum = std::fma(v[(size_t)j], xr[(size_t)ci[j] * 2 + q], sum);
                xr[(size_t)i * 2 + q] = (bh[(size_t)i * 2 + q] - sum) / v[(size_t)d];
            }
        }
        double *db = nullptr, *dx = nullptr;
        if ((rc = ensure_part_rhs(p, 2)) == CAP_OK && (rc = dev_alloc(&db, (size_t)n * 2)) == CAP_OK &&
            (rc = dev_alloc(&dx, (size_t)n * 2)) == CAP_OK) {
            if (hipMemcpy(db, bh.data(), sizeof(double) * bh.size(), hipMemcpyHostToDevice) != hipSuccess)
                rc = CAP_ERR_HIP;
            if (rc == CAP_OK) rc = launch_partition<double>(p, db, dx, 2, st);
            if (rc == CAP_OK && (hipStreamSynchronize(st) != hipSuccess ||
                                 hipMemcpy(xs.data(), dx, sizeof(double) * xs.size(), hipMemcpyDeviceToHost) !=
                                     hipSuccess))
                rc = CAP_ERR_HIP;
        }
        (void)hipFree(db);
        (void)hipFree(dx);
        for (int q = 0; q < 2 && rc == CAP_OK; ++q) {
            double err = 0.0, ref = 0.0;
            for (int i = 0; i < n; ++i) {
                err = std::max(err, std::fabs(xs[(size_t)i * 2 + q] - xr[(size_t)i * 2 + q]));
                ref = std::max(ref, std::fabs(xr[(size_t)i * 2 + q]));
            }
            // NaN or inf anywhere (err or ref) fails the test too
            if (!(err <= kPartStableTol * ref) || !std::isfinite(ref)) rc = CAP_ERR_UNSUPPORTED;
        }
    }
    if (rc != CAP_OK) free_partition(p);
    return rc;
}

// What an explicit CAP_ALGO_LEVEL plan takes, from its levels.  Every
// off-diagonal entry c of a row in level L must satisfy c > M_L - R (M_L:
// the largest row index in levels <= L) with a ring R, a power of two >= 64,
// of at most kLevelRingBytes of values; and the levels padded to whole steps
// of B rows -- B the smallest of 64, 128, 192 and 256 that needs at most 1/8
// more steps than 256 -- must hold at most kLevelPadMax slots per row.  The
// solve schedules rows more freely (steps.hip) and needs less; an autotuned
// plan uses the steps wherever that schedule fits.  *max_rhs: 1, or 2 or 4
// where rows hold at most 4 off-diagonals and R values of each fit LDS.
constexpr size_t kLevelRingBytes = 65536;
constexpr double kLevelMaxWidth = 4096;  // the autotuner tries the steps up to these rows per level
constexpr int kLevelPadMax = 4;
// An autotuned plan's steps may be mostly idle threads: with 4 rows per
// level a step still costs a third of what the one-workgroup kernel spends
// on them one by one.
constexpr int kStepPadMax = 16;
// Largest step tables a plan or batch makes without being asked for them.
constexpr double kStepMaxBytes = 4.0 * (1ull << 30);

int level_accepts(cap_plan p, const std::vector<int> &rp, const std::vector<int> &ci, int *max_rhs)
{
    const int n = p->n, vb = p->vbytes;
    std::vector<int> lv((size_t)std::max(n, 1));
    const int L = n ? cap_matrix_layer(n, rp.data(), ci.data(), nullptr, nullptr, lv.data()) : 0;  // 1-based
    std::vector<long long> width((size_t)L + 1, 0);
    std::vector<int> top((size_t)L + 1, -1);  // largest row index in levels <= l
    int maxoff = 0;
    for (int i = 0; i < n; ++i) {
        ++width[(size_t)lv[i]];
        top[(size_t)lv[i]] = std::max(top[(size_t)lv[i]], i);
        maxoff = std::max(maxoff, rp[i + 1] - 1 - rp[i]);
    }
    for (int l = 1; l <= L; ++l) top[(size_t)l] = std::max(top[(size_t)l], top[(size_t)l - 1]);
    long long need = 1;
    for (int i = 0; i < n; ++i)
        for (int j = rp[i]; j < rp[i + 1] - 1; ++j) need = std::max(need, (long long)top[(size_t)lv[i]] - ci[j] + 1);
    long long R = 64;
    while (R < need) R *= 2;
    if ((size_t)(R * vb) > kLevelRingBytes) return CAP_ERR_UNSUPPORTED;
    auto steps_for = [&](int B) {
        long long c = 0;
        for (int l = 1; l <= L; ++l) c += (width[(size_t)l] + B - 1) / B;
        return c;
    };
    int B = 256;
    const long long full = steps_for(B);
    for (int cand = B - kWave; cand >= kWave; cand -= kWave)
        if (steps_for(cand) <= full + full / 8) B = cand;
    const long long slots = steps_for(B) * B;
    if (slots > std::max((long long)kLevelPadMax * n, 1LL << 16)) return CAP_ERR_UNSUPPORTED;
    if (slots * (maxoff <= 4 ? 4 : 8) > INT32_MAX) return CAP_ERR_UNSUPPORTED;
    *max_rhs = maxoff > 4                              ? 1
               : (R + 2) * 4 * vb <= (long long)p->lds_max ? 4
               : (R + 2) * 2 * vb <= (long long)p->lds_max ? 2
                                                           : 1;
    return CAP_OK;
}

// The plan's step tables.  An explicit plan is held to level_accepts and
// keeps the values of its creation.  An autotuned plan over the caller's own
// values copies them into the tables again on every solve (6 us at n = 2,000,
// 8 at n = 100,000): the kernels it would run otherwise read them there, and
// which of them wins is a matter of microseconds.  width: rows per step, when
// a cached pick knows them.
int build_level(cap_plan p, const std::vector<int> &rp, const std::vector<int> &ci, bool explicit_algo, hipStream_t st,
                int width = 0)
{
    int rhs = 0;
    if (explicit_algo) CAP_TRY(level_accepts(p, rp, ci, &rhs));
    free_level(p);
    CAP_TRY(steps_build(&p->lvl, rp, ci, {make_int2(0, p->n)}, p->vt, explicit_algo ? rhs : 4, width, p->lds_max,
                        kStepPadMax, explicit_algo ? HUGE_VAL : kStepMaxBytes, p->rp, p->ci, p->val, st));
    p->lvl_rhs = rhs;
    p->lvl_live = !explicit_algo && !p->owns_matrix;
    return CAP_OK;
}

// Look-through tables of the write-first solve (k_hop): each row's hop
// number and look-through bits on the host, one pass over the entries; the
// tables on the device.  CAP_ERR_UNSUPPORTED for rows of more than kHopMax
// off-diagonals: the kernel keeps E values of each of E entries in registers.
int build_hop(cap_plan p, const std::vector<int> &rp, const std::vector<int> &ci, hipStream_t st)
{
    const int n = p->n;
    int most = 0;
    for (int i = 0; i < n; ++i) most = std::max(most, rp[i + 1] - 1 - rp[i]);
    if (n < 1 || most > kHopMax) return CAP_ERR_UNSUPPORTED;
    const int E = std::max(2, most);
    struct Ready {
        int hop, look;  // look: the hop in which all the row's entries are there, were it looked through
    };
    std::vector<Ready> at_row;
    std::vector<int> order;
    std::vector<unsigned char> bits;
    int hops = 0;
    try {
        at_row.resize((size_t)n);
        order.resize((size_t)n);
        bits.resize((size_t)n);
        for (int i = 0; i < n; ++i) {
            const int lo = rp[i], cnt = rp[i + 1] - 1 - lo;
            int ready = 0, newest = 0, of[kHopMax];
            for (int j = 0; j < cnt; ++j) {
                const Ready e = at_row[(size_t)ci[(size_t)(lo + j)]];
                of[j] = e.hop;
                newest = std::max(newest, e.hop);
                ready = std::max(ready, std::min(e.hop, e.look));
            }
            unsigned m = 0;
            for (int j = 0; j < cnt; ++j) m |= (unsigned)(of[j] > ready) << j;
            at_row[(size_t)i] = Ready{ready + 1, newest};
            bits[(size_t)i] = (unsigned char)m;
            hops = std::max(hops, ready + 1);
        }
        // rows in hop order, by index within a hop
        std::vector<int> at((size_t)hops + 2, 0);
        for (int i = 0; i < n; ++i) ++at[(size_t)at_row[(size_t)i].hop + 1];
        for (int h = 0; h <= hops; ++h) at[(size_t)h + 1] += at[(size_t)h];
        for (int i = 0; i < n; ++i) order[(size_t)at[(size_t)at_row[(size_t)i].hop]++] = i;
    } catch (const std::bad_alloc &) {
        return CAP_ERR_ALLOC;
    }
    free_hop(p);
    HopState *hs = new HopState();
    p->hop = hs;
    hs->E = E;
    hs->hops = hops;
    hs->npad = (n + kWave - 1) / kWave * kWave;
    int *d_order = nullptr, *d_slot = nullptr;
    unsigned char *d_bits = nullptr;
    int rc = dev_alloc(&hs->base, (size_t)hs->npad * (3 + E));
    if (rc == CAP_OK) rc = dev_alloc(&hs->ex, (size_t)hs->npad * E * (E + 1));
    if (rc == CAP_OK) rc = dev_alloc(&d_order, (size_t)n);
    if (rc == CAP_OK) rc = dev_alloc(&d_slot, (size_t)n);
    if (rc == CAP_OK) rc = dev_alloc(&d_bits, (size_t)n);
    if (rc == CAP_OK && (hipMemcpy(d_order, order.data(), sizeof(int) * (size_t)n, hipMemcpyHostToDevice) != hipSuccess ||
                         hipMemcpy(d_bits, bits.data(), (size_t)n, hipMemcpyHostToDevice) != hipSuccess))
        rc = CAP_ERR_HIP;
    if (rc == CAP_OK) {
        k_invert<<<blocks_for(n), kBlock, 0, st>>>(d_order, n, d_slot);
        auto fill = [&](auto kernel) {
            kernel<<<blocks_for(hs->npad), kBlock, 0, st>>>(p->rp, p->ci, d_order, d_slot, d_bits, n, hs->npad, hs->base,
                                                            hs->ex);
        };
        E == 2 ? fill(k_hop_tables<2>) : E == 3 ? fill(k_hop_tables<3>) : fill(k_hop_tables<4>);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) rc = CAP_ERR_HIP;
    }
    for (void *b : {(void *)d_order, (void *)d_slot, (void *)d_bits})
        if (b) (void)hipFree(b);
    if (rc != CAP_OK) free_hop(p);
    return rc;
}

// The partition keeps the values of plan creation, the other candidates read
// the caller's on every solve.  Over the caller's own values it is the pick
// only where it takes less than half their time: matrices of short chains
// (n = 20,000, bandwidth 120, 89 levels: 45 us, 51 by look-through) stay with a
// kernel that follows the values.  Bands that explicit level plans take are
// compared as they are: long chains of narrow levels, where only the steps,
// which held the values too until they were made to follow them, come near.
constexpr float kPartLiveFactor = 2.0f;

// Candidates are timed on the plan's own matrix (b = 1, tuning_rhs) and the
// fastest is cached per matrix shape: thread-per-row with and without the LDS
// window, at 1 or 2 workgroups per CU, with the staged or the in-place
// readiness array, the flag protocol, and mix at three thresholds when the
// rows are long enough for wavefront mode to matter.  A plan created with
// readiness in place keeps it in every candidate.
int autotune(cap_plan p, const std::vector<int> &rp_host, const std::vector<int> &ci, hipStream_t st)
{
    const int levels = p->n ? cap_matrix_layer(p->n, rp_host.data(), ci.data(), nullptr, nullptr, nullptr) : 1;
    const TuneKey key{p->n,           p->nnz,         p->vt,  p->staged,
                      p->unfused,     p->count_polls, levels, p->owns_matrix,
                      fingerprint(rp_host, ci)};
    {
        std::lock_guard<std::mutex> g(g_tune_mu);
        auto it = g_tune_cache.find(key);
        if (it != g_tune_cache.end()) {
            const TuneChoice &c = it->second;
            apply_choice(p, c);
            int rc = CAP_OK;
            if (c.algo == CAP_ALGO_MIX) rc = build_mix(p, rp_host, c.border);
            else if (c.algo == CAP_ALGO_LOCAL) rc = ensure_segments(p, nullptr);
            else if (c.algo == CAP_ALGO_LEVEL) rc = build_level(p, rp_host, ci, false, st, c.width);
            else if (c.algo == CAP_ALGO_PARTITION) rc = build_partition(p, rp_host, st);
            else if (c.hop) rc = build_hop(p, rp_host, ci, st);
            // The key samples the pattern: this matrix may have a row too long
            // for the look-through tables or reach beyond the steps' ring, its
            // values may not keep the partition stable, its tables may not
            // fit.  Then it is tuned afresh.
            if (rc != CAP_ERR_UNSUPPORTED && rc != CAP_ERR_ALLOC) return rc;
            p->staged = key.staged;
        }
    }
    void *b = nullptr, *x = nullptr;
    CAP_HIP_TRY(hipMalloc(&b, (size_t)p->n * p->vbytes + 8));
    CAP_HIP_TRY(hipMalloc(&x, (size_t)p->n * p->vbytes + 8));
    CAP_TRY(tuning_rhs(p, b, p->n, st));
    const int stg = p->staged;
    constexpr int B = kBlock, S = kBlockSmall;
    std::vector<TuneChoice> cands = {{CAP_ALGO_WRTFST, CAP_SYNC_VALUE, 0, 1, 0, stg, B},
                                     {CAP_ALGO_WRTFST, CAP_SYNC_VALUE, 0, 2, 0, stg, B},
                                     {CAP_ALGO_WRTFST, CAP_SYNC_VALUE, 0, 1, 1, stg, B},
                                     {CAP_ALGO_WRTFST, CAP_SYNC_VALUE, 0, 2, 1, stg, B},
                                     {CAP_ALGO_WRTFST, CAP_SYNC_VALUE, 0, 1, 0, stg, S},
                                     {CAP_ALGO_WRTFST, CAP_SYNC_VALUE, 0, 1, 1, stg, S},
                                     {CAP_ALGO_WRTFST, CAP_SYNC_FLAG, 0, 1, 0, 0, B}};
    if (stg) cands.push_back({CAP_ALGO_WRTFST, CAP_SYNC_VALUE, 0, 1, 0, 0, B});
    // look-through tables, where rows are short: half the hops
    if (stg && !p->count_polls && build_hop(p, rp_host, ci, st) == CAP_OK)
        for (int blk : {B, S})
            cands.insert(cands.begin(), {CAP_ALGO_WRTFST, CAP_SYNC_VALUE, 0, 1, 0, stg, blk, 0, 1});
    HopState *const hop_tables = p->hop;
    // the same value-protocol shapes with each ticket's col_idx/val tile staged in LDS
    for (int lds : {0, 1})
        for (int blk : {B, S}) cands.push_back({CAP_ALGO_WRTFST, CAP_SYNC_VALUE, 0, 1, lds, stg, blk, 1});
    const double avg = (double)p->nnz / std::max(1, p->n);
    float part_factor = 1.0f;
    // one workgroup per matrix pays off only with few rows per level
    {
        // timed first: on such matrices it sets a low bound that lets the
        // slower candidates stop after their warm-up
        if ((double)p->n / std::max(1, levels) <= kLocalMaxWidth) {
            cands.insert(cands.begin(), {CAP_ALGO_LOCAL, CAP_SYNC_VALUE, 0, 1, 0, 0, B});
            // deep and narrow-banded: the partitioned solve, timed before all
            // (reassociated sums: not a candidate in the reference arithmetic)
            if (!p->unfused && build_partition(p, rp_host, st) == CAP_OK) {
                cands.insert(cands.begin(), {CAP_ALGO_PARTITION, CAP_SYNC_VALUE, 0, 1, 0, 0, B});
                int rhs = 0;
                if (!p->owns_matrix && level_accepts(p, rp_host, ci, &rhs) != CAP_OK) part_factor = kPartLiveFactor;
            }
        }
        // steps in one workgroup, where the ring and the padding allow: up to
        // a few thousand rows per level a step per 256 rows can still beat a
        // cross-CU hop per level
        if ((double)p->n / std::max(1, levels) <= kLevelMaxWidth && build_level(p, rp_host, ci, false, st) == CAP_OK)
            cands.insert(cands.begin(), {CAP_ALGO_LEVEL, CAP_SYNC_VALUE, 0, 1, 0, 0, B});
    }
    // thresholds 4 and 32 (see mix_border_for) always; 16 where the mean row
    // length is at least 4 (some chunks may then reach it)
    for (int bd : {kMixBorderWide, 16, kMixBorderNarrow})
        if (bd != 16 || avg * 4 >= bd) {
            cands.push_back({CAP_ALGO_MIX, CAP_SYNC_VALUE, bd, kMixBlocks, 0, stg, B});
            cands.push_back({CAP_ALGO_MIX, CAP_SYNC_VALUE, bd, kMixBlocks, 0, stg, B, 1});
        }
    float best = 1e30f;
    TuneChoice pick = cands[0];
    bool pick_set = false;
    PlainShape plain;
    float t_plain = 1e30f, t_steps = 0;
    int rc = CAP_OK;
    for (const TuneChoice &c : cands) {
        apply_choice(p, c);
        p->hop = c.hop ? hop_tables : nullptr;
        if (c.algo == CAP_ALGO_MIX && (rc = build_mix(p, rp_host, c.border)) != CAP_OK) break;
        if (c.algo == CAP_ALGO_LOCAL && (rc = ensure_segments(p, nullptr)) != CAP_OK) break;
        float t = 0;
        if ((rc = time_candidate(p, c.algo, c.sync, b, x, 1, st, best, &t)) != CAP_OK) break;
        if (c.algo == CAP_ALGO_PARTITION) t *= part_factor;
        if (c.algo == CAP_ALGO_LEVEL) t_steps = t;
        if (c.algo == CAP_ALGO_WRTFST && c.sync == CAP_SYNC_VALUE && c.staged == stg && !c.hop && t < t_plain) {
            t_plain = t;
            plain = PlainShape{c.bpc, c.block, c.lds, c.tile, c.staged};
        }
        // a later (less preferred) candidate must be 2% faster to win, so
        // near-ties resolve the same way from run to run
        if (t < (pick_set ? 0.98f : 1.0f) * best) {
            best = t;
            pick = c;
            pick_set = true;
        }
    }
    (void)hipFree(b);
    (void)hipFree(x);
    p->hop = hop_tables;
    if (rc != CAP_OK) return rc;
    if (pick.hop || pick.algo == CAP_ALGO_LEVEL) pick.plain = plain;
    if (pick.algo == CAP_ALGO_LEVEL && t_steps > 0) pick.lead = t_plain / t_steps;
    apply_choice(p, pick);
    if (!pick.hop) free_hop(p);
    if (pick.algo == CAP_ALGO_MIX) CAP_TRY(build_mix(p, rp_host, pick.border));
    if (pick.algo == CAP_ALGO_LOCAL) CAP_TRY(ensure_segments(p, nullptr));
    if (pick.algo != CAP_ALGO_PARTITION) free_partition(p);
    if (pick.algo == CAP_ALGO_LEVEL)
        pick.width = p->lvl->block;
    else
        free_level(p);
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tune_cache[key] = pick;
    return CAP_OK;
}

template <typename T>
int validate_device_matrix(cap_plan p, std::vector<int> *rp_host, std::vector<int> *ci_host)
{
    const int n = p->n, nnz = p->nnz;
    std::vector<int> &ci = *ci_host;  // kept for the autotuner's analysis
    ci.resize((size_t)nnz);
    std::vector<T> v((size_t)nnz);
    CAP_HIP_TRY(hipMemcpy(ci.data(), p->ci, sizeof(int) * (size_t)nnz, hipMemcpyDeviceToHost));
    CAP_HIP_TRY(hipMemcpy(v.data(), p->val, sizeof(T) * (size_t)nnz, hipMemcpyDeviceToHost));
    int bad = -1;
    if (sizeof(T) == 8)
        return cap_validate_csr_d(n, nnz, rp_host->data(), ci.data(), (const double *)(const void *)v.data(), &bad);
    return cap_validate_csr_s(n, nnz, rp_host->data(), ci.data(), (const float *)(const void *)v.data(), &bad);
}

// A host copy of the column indices, unless the layout check already took one.
int host_columns(cap_plan p, std::vector<int> *ci)
{
    if (ci->size() == (size_t)p->nnz) return CAP_OK;
    ci->resize((size_t)p->nnz);
    CAP_HIP_TRY(hipMemcpy(ci->data(), p->ci, sizeof(int) * (size_t)p->nnz, hipMemcpyDeviceToHost));
    return CAP_OK;
}

// Upper-triangular and implicit-unit-diagonal matrices become the lower,
// diagonal-last CSR every kernel solves: row t of the result is row
// i = n-1-t of an upper matrix (columns c -> n-1-c), or row t of a lower
// one; its off-diagonal entries keep their stored order (so the
// accumulation order is the caller's) and the diagonal -- stored, or 1 --
// comes last.  Rejects a stored diagonal that is not where the layout puts
// it and, with unit_diag, any diagonal entry.
template <typename T>
int convert_triangular(int n, int nnz, const int *rp, const int *ci, const T *val, bool upper, bool unit,
                       std::vector<int> *rp2, std::vector<int> *ci2, std::vector<T> *v2)
{
    rp2->assign((size_t)n + 1, 0);
    ci2->clear();
    v2->clear();
    ci2->reserve((size_t)nnz + (unit ? n : 0));
    v2->reserve((size_t)nnz + (unit ? n : 0));
    for (int t = 0; t < n; ++t) {
        const int i = upper ? n - 1 - t : t;
        int lo = rp[i], hi = rp[i + 1];
        if (hi < lo || lo < 0 || hi > nnz) return CAP_ERR_ROWPTR;
        T d = (T)1;
        if (!unit) {
            if (hi == lo) return CAP_ERR_NO_DIAG;
            const int dj = upper ? lo++ : --hi;
            if (ci[dj] != i) return CAP_ERR_NO_DIAG;
            d = val[dj];
        }
        for (int j = lo; j < hi; ++j) {
            const int c = ci[j];
            if (c < 0 || c >= n || (upper ? c <= i : c >= i)) return CAP_ERR_UPPER;
            ci2->push_back(upper ? n - 1 - c : c);
            v2->push_back(val[j]);
        }
        ci2->push_back(t);
        v2->push_back(d);
        (*rp2)[(size_t)t + 1] = (int)ci2->size();
    }
    return CAP_OK;
}

int plan_create_impl(cap_plan *out, int n, int nnz, const int *rp, const int *ci, const void *val, int vt,
                     const cap_opts *opts, hipStream_t st)
{
    cap_opts o;
    cap_opts_default(&o);
    if (opts) o = *opts;
    if (!out || n < 0 || nnz < 0 || (vt != CAP_F64 && vt != CAP_F32) || !rp || (nnz > 0 && (!ci || !val)))
        return CAP_ERR_ARG;
    if (!o.unit_diag && nnz < n) return CAP_ERR_ARG;
    if (o.blocks_per_cu < 0 || o.blocks_per_cu > kMaxBlocksPerCu) return CAP_ERR_ARG;
    if (o.row_threads != 0 && o.row_threads != kBlock && o.row_threads != kBlockSmall) return CAP_ERR_ARG;
    if (o.arith != CAP_ARITH_FUSED && o.arith != CAP_ARITH_REFERENCE) return CAP_ERR_ARG;
    if (o.wait_limit_ms > kWaitMsMax) return CAP_ERR_ARG;
    if (o.arith == CAP_ARITH_REFERENCE && (o.algo == CAP_ALGO_CSC || o.algo == CAP_ALGO_PARTITION))
        return CAP_ERR_UNSUPPORTED;
    if (o.rhs_per_lane != 0 && o.rhs_per_lane != 1 && o.rhs_per_lane != 2 && o.rhs_per_lane != 4 &&
        o.rhs_per_lane != 8)
        return CAP_ERR_ARG;
    if (o.row_tiles != 0 && o.row_tiles != 1) return CAP_ERR_ARG;
    if (o.algo == CAP_ALGO_HOP && ((o.sync != CAP_SYNC_AUTO && o.sync != CAP_SYNC_VALUE) ||
                                   o.readiness == CAP_READY_IN_PLACE || o.lds_window > 0 || o.count_polls))
        return CAP_ERR_UNSUPPORTED;
    if (o.row_tiles &&
        ((o.algo != CAP_ALGO_WRTFST && o.algo != CAP_ALGO_MIX) || (o.sync != CAP_SYNC_AUTO && o.sync != CAP_SYNC_VALUE) ||
         o.count_polls || o.rhs_per_lane > 1))
        return CAP_ERR_UNSUPPORTED;
    if (o.rhs_per_lane > 0 &&
        (o.algo != CAP_ALGO_WRTFST || (o.sync != CAP_SYNC_AUTO && o.sync != CAP_SYNC_VALUE) || o.lds_window ||
         o.count_polls || (o.rhs_per_lane == 8 && vt != CAP_F32)))
        return CAP_ERR_UNSUPPORTED;
    *out = nullptr;
    if (o.upper || o.unit_diag) {
        // convert on the host, then create a plan over the owned lower matrix
        std::vector<int> rph((size_t)n + 1), cih((size_t)nnz);
        std::vector<unsigned char> vh((size_t)nnz * (vt == CAP_F64 ? 8 : 4));
        const hipMemcpyKind kind = o.host_inputs ? hipMemcpyHostToHost : hipMemcpyDeviceToHost;
        CAP_HIP_TRY(hipMemcpy(rph.data(), rp, sizeof(int) * rph.size(), kind));
        if (nnz) {
            CAP_HIP_TRY(hipMemcpy(cih.data(), ci, sizeof(int) * cih.size(), kind));
            CAP_HIP_TRY(hipMemcpy(vh.data(), val, vh.size(), kind));
        }
        if (rph[0] != 0 || rph[n] != nnz) return CAP_ERR_ROWPTR;
        std::vector<int> rp2, ci2;
        std::vector<unsigned char> v2;
        int rc;
        if (vt == CAP_F64) {
            std::vector<double> t;
            rc = convert_triangular<double>(n, nnz, rph.data(), cih.data(), (const double *)(const void *)vh.data(),
                                            o.upper != 0, o.unit_diag != 0, &rp2, &ci2, &t);
            v2.assign((const unsigned char *)t.data(), (const unsigned char *)t.data() + t.size() * 8);
        } else {
            std::vector<float> t;
            rc = convert_triangular<float>(n, nnz, rph.data(), cih.data(), (const float *)(const void *)vh.data(),
                                           o.upper != 0, o.unit_diag != 0, &rp2, &ci2, &t);
            v2.assign((const unsigned char *)t.data(), (const unsigned char *)t.data() + t.size() * 4);
        }
        if (rc != CAP_OK) return rc;
        cap_opts o2 = o;
        o2.upper = 0;
        o2.unit_diag = 0;
        o2.host_inputs = 1;
        cap_plan p = nullptr;
        CAP_TRY(plan_create_impl(&p, n, (int)ci2.size(), rp2.data(), ci2.data(), v2.data(), vt, &o2, st));
        p->reversed = o.upper != 0;
        p->unit_diag = o.unit_diag != 0;
        *out = p;
        return CAP_OK;
    }
    int dev = 0;
    CAP_TRY(check_device(&dev));
    cap_plan p = new cap_plan_s();
    p->n = n;
    p->nnz = nnz;
    p->vt = vt;
    p->vbytes = vt == CAP_F64 ? 8 : 4;
    p->device = dev;
    int rc = CAP_OK;
    std::vector<int> rp_host((size_t)n + 1), ci_host;  // ci_host: filled where it is needed, once
    do {
        if (o.host_inputs) {
            if (o.validate) {
                int bad = -1;
                rc = vt == CAP_F64 ? cap_validate_csr_d(n, nnz, rp, ci, (const double *)val, &bad)
                                   : cap_validate_csr_s(n, nnz, rp, ci, (const float *)val, &bad);
                if (rc != CAP_OK) break;
            }
            p->owns_matrix = true;
            if ((rc = dev_alloc(&p->rp, (size_t)n + 1)) != CAP_OK) break;
            if ((rc = dev_alloc(&p->ci, (size_t)nnz)) != CAP_OK) break;
            if (hipMalloc(&p->val, (size_t)nnz * p->vbytes + 8) != hipSuccess) { rc = CAP_ERR_ALLOC; break; }
            if (hipMemcpy(p->rp, rp, sizeof(int) * ((size_t)n + 1), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(p->ci, ci, sizeof(int) * (size_t)nnz, hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(p->val, val, (size_t)nnz * p->vbytes, hipMemcpyHostToDevice) != hipSuccess) {
                rc = CAP_ERR_HIP;
                break;
            }
            std::memcpy(rp_host.data(), rp, sizeof(int) * ((size_t)n + 1));
        } else {
            p->rp = const_cast<int *>(rp);
            p->ci = const_cast<int *>(ci);
            p->val = const_cast<void *>(val);
            if (hipMemcpy(rp_host.data(), rp, sizeof(int) * ((size_t)n + 1), hipMemcpyDeviceToHost) != hipSuccess) {
                rc = CAP_ERR_HIP;
                break;
            }
            if (o.validate) {
                rc = vt == CAP_F64 ? validate_device_matrix<double>(p, &rp_host, &ci_host)
                                   : validate_device_matrix<float>(p, &rp_host, &ci_host);
                if (rc != CAP_OK) break;
            }
        }
        if ((rc = init_ctrl(p)) != CAP_OK) break;
        if (o.spin_limit > 0) p->spin_limit = o.spin_limit;
        if (o.wait_limit_ms != 0) p->wait_ticks = o.wait_limit_ms > 0 ? o.wait_limit_ms * 100000 : 0;
        if (o.blocks_per_cu > 0) p->bpc = o.blocks_per_cu;
        if (o.row_threads > 0) p->wblock = o.row_threads;
        p->fixed_rpl = o.rhs_per_lane;
        p->tile = o.row_tiles != 0;
        p->auto_algo = o.algo == CAP_ALGO_AUTO;
        p->lds = o.lds_window > 0;
        p->unfused = o.arith == CAP_ARITH_REFERENCE;
        p->count_polls = o.count_polls != 0;
        // the caller fixed neither the grid nor the workgroup size: multi-RHS
        // solves get their RHS block timed per right-hand-side count
        p->tune_rhs = o.algo == CAP_ALGO_AUTO && o.blocks_per_cu == 0 && o.row_threads == 0;
        p->staged = o.readiness != CAP_READY_IN_PLACE;
        if (o.adjoint == CAP_ADJOINT_SCATTER || o.adjoint == CAP_ADJOINT_GATHER) p->adjoint_mode = o.adjoint;
        p->algo = o.algo;
        p->sync = o.sync ? o.sync : CAP_SYNC_VALUE;
        if (p->algo == CAP_ALGO_MIX) {
            int border = o.border;
            if (border <= 0) {  // from the matrix's rows per level
                rc = host_columns(p, &ci_host);
                const int levels =
                    rc == CAP_OK && p->n
                        ? cap_matrix_layer(p->n, rp_host.data(), ci_host.data(), nullptr, nullptr, nullptr)
                        : 1;
                border = mix_border_for(p->n, levels);
            }
            if (rc == CAP_OK) rc = build_mix(p, rp_host, border);
        } else if (p->algo == CAP_ALGO_CSC) {
            rc = ensure_csc(p, st);
        } else if (p->algo == CAP_ALGO_AUTO) {
            if ((rc = host_columns(p, &ci_host)) == CAP_OK) rc = autotune(p, rp_host, ci_host, st);
        } else if (p->algo == CAP_ALGO_LOCAL) {
            rc = ensure_segments(p, nullptr);
        } else if (p->algo == CAP_ALGO_PARTITION) {
            rc = build_partition(p, rp_host, st);
        } else if (p->algo == CAP_ALGO_LEVEL) {
            if ((rc = host_columns(p, &ci_host)) == CAP_OK) rc = build_level(p, rp_host, ci_host, true, st);
        } else if (p->algo == CAP_ALGO_HOP) {
            p->algo = CAP_ALGO_WRTFST;
            if ((rc = host_columns(p, &ci_host)) == CAP_OK) rc = build_hop(p, rp_host, ci_host, st);
        } else if (p->algo != CAP_ALGO_WRTFST && p->algo != CAP_ALGO_TWOPART) {
            rc = CAP_ERR_ARG;
        }
    } while (0);
    if (rc != CAP_OK) {
        plan_free(p);
        return rc;
    }
    if (o.algo != CAP_ALGO_AUTO) p->rblock = p->wblock;
    *out = p;
    return CAP_OK;
}

// Reversed transpose of L for the gather adjoint: row i' = n-1-c lists the
// entries of column c of L, rows r mapped to n-1-r, in the order the
// executor's BACKWARD mode adds them into left_sum[c] (serialref.h:75-100):
// rows of L in descending order, entries of a row in stored order (which
// keeps duplicate columns of one row in their stored order).  The diagonal
// (row c) comes last.  Solving this lower triangular matrix with the
// write-first kernel makes the gather adjoint deterministic and bit-equal to
// that order.
int ensure_reversed_transpose(cap_plan p)
{
    if (p->rpT) return CAP_OK;
    const int n = p->n, nnz = p->nnz;
    std::vector<int> rp((size_t)n + 1), ci((size_t)nnz);
    std::vector<double> v((size_t)nnz);
    CAP_HIP_TRY(hipMemcpy(rp.data(), p->rp, sizeof(int) * ((size_t)n + 1), hipMemcpyDeviceToHost));
    CAP_HIP_TRY(hipMemcpy(ci.data(), p->ci, sizeof(int) * (size_t)nnz, hipMemcpyDeviceToHost));
    CAP_HIP_TRY(hipMemcpy(v.data(), p->val, sizeof(double) * (size_t)nnz, hipMemcpyDeviceToHost));
    std::vector<int> rT((size_t)n + 1, 0), cT((size_t)nnz);
    std::vector<double> vT((size_t)nnz);
    for (int j = 0; j < nnz; ++j) rT[(size_t)(n - 1 - ci[j]) + 1]++;
    for (int r = 0; r < n; ++r) rT[r + 1] += rT[r];
    std::vector<int> fill(rT.begin(), rT.end() - 1);
    for (int i = n - 1; i >= 0; --i)
        for (int j = rp[i]; j < rp[i + 1]; ++j) {
            const int o = fill[n - 1 - ci[j]]++;
            cT[o] = n - 1 - i;
            vT[o] = v[j];
        }
    CAP_TRY(dev_alloc(&p->rpT, (size_t)n + 1));
    CAP_TRY(dev_alloc(&p->ciT, (size_t)nnz));
    CAP_TRY(dev_alloc(&p->vT, (size_t)nnz));
    CAP_HIP_TRY(hipMemcpy(p->rpT, rT.data(), sizeof(int) * ((size_t)n + 1), hipMemcpyHostToDevice));
    CAP_HIP_TRY(hipMemcpy(p->ciT, cT.data(), sizeof(int) * (size_t)nnz, hipMemcpyHostToDevice));
    CAP_HIP_TRY(hipMemcpy(p->vT, vT.data(), sizeof(double) * (size_t)nnz, hipMemcpyHostToDevice));
    return CAP_OK;
}

}  // namespace

// =================================================================== C ABI
extern "C" {

void cap_opts_default(cap_opts *o)
{
    std::memset(o, 0, sizeof(*o));
    o->algo = CAP_ALGO_AUTO;
    o->sync = CAP_SYNC_AUTO;
    o->validate = 1;
}

int cap_device_count(void)
{
    int c = 0;
    if (hipGetDeviceCount(&c) != hipSuccess) return 0;
    return c;
}

int cap_plan_create(cap_plan *plan, int n, int nnz, const int *row_ptr, const int *col_idx, const void *val,
                    int value_type, const cap_opts *opts, void *stream)
{
    return plan_create_impl(plan, n, nnz, row_ptr, col_idx, val, value_type, opts, S(stream));
}

}  // extern "C"

namespace {

// Upper-triangular plans: reversed copies of b and x around the solve.
int ensure_reversal(cap_plan p, int rhs)
{
    const size_t bytes = (size_t)p->n * rhs * p->vbytes + 8;
    if (p->rev_bytes >= bytes) return CAP_OK;
    CAP_HIP_TRY(hipDeviceSynchronize());  // kernels in flight may use the old buffers
    if (p->rev_b) CAP_HIP_TRY(hipFree(p->rev_b));
    if (p->rev_x) CAP_HIP_TRY(hipFree(p->rev_x));
    p->rev_b = p->rev_x = nullptr;
    p->rev_bytes = 0;
    if (hipMalloc(&p->rev_b, bytes) != hipSuccess || hipMalloc(&p->rev_x, bytes) != hipSuccess) return CAP_ERR_ALLOC;
    p->rev_bytes = bytes;
    return CAP_OK;
}

int reverse_rows(cap_plan p, const void *src, void *dst, int rhs, hipStream_t st)
{
    const long long cnt = (long long)p->n * rhs;
    if (cnt == 0) return CAP_OK;
    if (p->vt == CAP_F64)
        k_reverse_rows<double><<<blocks_for(cnt), kBlock, 0, st>>>((const double *)src, (double *)dst, p->n, rhs);
    else
        k_reverse_rows<float><<<blocks_for(cnt), kBlock, 0, st>>>((const float *)src, (float *)dst, p->n, rhs);
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

int launch_plain(cap_plan p, const void *b, void *x, int rhs, hipStream_t st)
{
    const int algo = algo_for(p, rhs), sync = sync_for(p, rhs);
    if (p->vt == CAP_F64)
        return launch_kernel<double>(p, algo, sync, (const double *)p->val, (const double *)b, (double *)x, rhs, st);
    return launch_kernel<float>(p, algo, sync, (const float *)p->val, (const float *)b, (float *)x, rhs, st);
}

}  // namespace

extern "C" {

int cap_plan_solve(cap_plan p, const void *b, void *x, int rhs, void *stream)
{
    if (!p || !b || !x || rhs < 1) return CAP_ERR_ARG;
    if (p->tune_rhs && rhs > 1 && rhs <= kWave && !p->reversed && !p->rhs_pick.count(rhs))
        CAP_TRY(tune_rhs_block(p, b, x, rhs, S(stream)));
    const int algo = algo_for(p, rhs), sync = sync_for(p, rhs);
    if (hop_takes(p, rhs)) p->hop_reset = true;
    if (!p->reversed || hop_takes(p, rhs)) return plan_solve_with(p, algo, sync, b, x, rhs, S(stream));
    CAP_TRY(ensure_reversal(p, rhs));
    CAP_TRY(reverse_rows(p, b, p->rev_b, rhs, S(stream)));
    CAP_TRY(plan_solve_with(p, algo, sync, p->rev_b, p->rev_x, rhs, S(stream)));
    return reverse_rows(p, p->rev_x, x, rhs, S(stream));
}

int cap_plan_reset(cap_plan p, void *x, int rhs, void *stream)
{
    if (!p || !x || rhs < 1) return CAP_ERR_ARG;
    if (hop_takes(p, rhs)) {
        p->hop_reset = true;
    } else if (p->reversed) {
        CAP_TRY(ensure_reversal(p, rhs));
        x = p->rev_x;
    }
    const int algo = algo_for(p, rhs), sync = sync_for(p, rhs);
    return p->vt == CAP_F64 ? reset_t<double>(p, algo, sync, x, rhs, S(stream))
                            : reset_t<float>(p, algo, sync, x, rhs, S(stream));
}

int cap_plan_launch(cap_plan p, const void *b, void *x, int rhs, void *stream)
{
    if (!p || !b || !x || rhs < 1) return CAP_ERR_ARG;
    if (p->reversed && hop_takes(p, rhs) && !p->hop_reset) return CAP_ERR_ARG;  // launch without its reset
    if (!p->reversed || hop_takes(p, rhs)) return launch_plain(p, b, x, rhs, S(stream));
    if (p->rev_bytes < (size_t)p->n * rhs * p->vbytes) return CAP_ERR_ARG;  // launch without its reset
    CAP_TRY(reverse_rows(p, b, p->rev_b, rhs, S(stream)));
    CAP_TRY(launch_plain(p, p->rev_b, p->rev_x, rhs, S(stream)));
    return reverse_rows(p, p->rev_x, x, rhs, S(stream));
}

int cap_plan_info(cap_plan p, int *algo, int *sync, int *border, int *mix_len, double *wocc, double *eocc)
{
    if (!p) return CAP_ERR_ARG;
    if (algo) *algo = p->algo;
    if (sync) *sync = p->sync;
    if (border) *border = p->border;
    if (mix_len) *mix_len = p->mix_len;
    if (wocc) *wocc = p->wocc;
    if (eocc) *eocc = p->eocc;
    return CAP_OK;
}

// Reads and clears the watchdog word: CAP_OK, or CAP_ERR_NOT_CONVERGED when
// a wait gave up since the last call (the affected rows hold NaN).
int cap_plan_status(cap_plan p, void *stream)
{
    if (!p) return CAP_ERR_ARG;
    int e = 0;
    CAP_HIP_TRY(hipStreamSynchronize(S(stream)));
    CAP_HIP_TRY(hipMemcpy(&e, p->err, sizeof(int), hipMemcpyDeviceToHost));
    if (e) CAP_HIP_TRY(hipMemset(p->err, 0, sizeof(int)));
    return e ? CAP_ERR_WATCHDOG : CAP_OK;
}

int cap_plan_hops(cap_plan p, int *hops)
{
    if (!p || !hops) return CAP_ERR_ARG;
    if (!hop_takes(p, 1)) return CAP_ERR_UNSUPPORTED;
    *hops = p->hop->hops;
    return CAP_OK;
}

int cap_plan_poll_count(cap_plan p, unsigned long long *polls, void *stream)
{
    if (!p || !polls) return CAP_ERR_ARG;
    if (!p->count_polls) return CAP_ERR_UNSUPPORTED;
    hipStream_t st = S(stream);
    unsigned long long h[kPollCounters];
    unsigned long long *d = reinterpret_cast<unsigned long long *>(p->ctrl + 1024);
    CAP_HIP_TRY(hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, st));
    CAP_HIP_TRY(hipStreamSynchronize(st));
    k_prepare<unsigned long long><<<1, kBlock, 0, st>>>(d, kPollCounters, 0ULL, p->ticket, 0);
    CAP_HIP_TRY(hipGetLastError());
    unsigned long long sum = 0;
    for (unsigned long long v : h) sum += v;
    *polls = sum;
    return CAP_OK;
}

int cap_plan_rhs_block(cap_plan p, int k, int *blocks_per_cu, int *row_threads, int *rhs_per_wave,
                       int *rhs_per_lane, int *readiness, int *row_tiles)
{
    if (!p || k < 1) return CAP_ERR_ARG;
    const auto it = p->rhs_pick.find(k);
    if (it == p->rhs_pick.end()) return CAP_ERR_UNSUPPORTED;
    if (row_tiles) {
        const int blk = it->second.block ? it->second.block : p->wblock;
        const int rpl = it->second.rpl ? it->second.rpl : p->rpl;
        const bool tiled = it->second.tile >= 0 ? it->second.tile != 0 : p->tile != 0;
        // k_wrtfst_r (several right-hand sides per lane) has no tiled form
        *row_tiles = algo_for(p, k) == CAP_ALGO_WRTFST && tiled && !(blk == kBlockLarge && rpl > 1);
    }
    if (blocks_per_cu) *blocks_per_cu = it->second.bpc ? it->second.bpc : p->bpc;
    if (row_threads) *row_threads = it->second.block ? it->second.block : p->wblock;
    if (rhs_per_wave) *rhs_per_wave = it->second.kr;
    if (rhs_per_lane)
        *rhs_per_lane = algo_for(p, k) == CAP_ALGO_WRTFST ? (it->second.rpl ? it->second.rpl : p->rpl) : 0;
    if (readiness) {
        const bool staged = it->second.staged >= 0 ? it->second.staged != 0 : p->staged;
        *readiness = staged ? CAP_READY_STAGED : CAP_READY_IN_PLACE;
    }
    return CAP_OK;
}

int cap_plan_tuning(cap_plan p, int *blocks_per_cu, int *lds_window, int *adjoint, int *readiness,
                    int *row_threads, int *row_tiles)
{
    if (!p) return CAP_ERR_ARG;
    if (row_tiles) *row_tiles = p->tile;
    if (blocks_per_cu) *blocks_per_cu = p->algo == CAP_ALGO_MIX ? kMixBlocks : p->bpc;
    if (row_threads) *row_threads = p->algo == CAP_ALGO_LEVEL && p->lvl ? p->lvl->block : p->wblock;
    if (lds_window) *lds_window = p->lds;
    if (adjoint) *adjoint = p->adjoint_mode;
    if (readiness) *readiness = p->staged ? CAP_READY_STAGED : CAP_READY_IN_PLACE;
    return CAP_OK;
}

int cap_plan_destroy(cap_plan p)
{
    if (!p) return CAP_ERR_ARG;
    (void)hipDeviceSynchronize();
    plan_free(p);
    return CAP_OK;
}

int cap_plan_adjoint(cap_plan p, const void *g, const void *x, void *grad_b, void *grad_val, void *stream)
{
    if (!p || !g || !x || !grad_b) return CAP_ERR_ARG;
    if (p->vt != CAP_F64 || p->reversed || p->unit_diag) return CAP_ERR_UNSUPPORTED;
    hipStream_t st = S(stream);
    const int n = p->n;
    if (n == 0) return CAP_OK;
    if (p->adjoint_mode == CAP_ADJOINT_GATHER) {
        CAP_TRY(ensure_reversed_transpose(p));
        CAP_TRY(launch_prepare<double>(p, CAP_ALGO_WRTFST, CAP_SYNC_VALUE, grad_b, n, st));
        SyncCtx sc;
        CAP_TRY(sync_ctx<double>(p, CAP_SYNC_VALUE, n, &sc));
        k_wrtfst<double, 1, 0, kBlock><<<grid_for(p, ((long long)n + kBlock - 1) / kBlock), kBlock, 0, st>>>(
            p->rpT, p->ciT, p->vT, (const double *)g, (double *)grad_b, sc, n, 1, 0, p->ticket, n, nullptr, 0);
        if (grad_val)
            k_grad_val<<<blocks_for(n), kBlock, 0, st>>>(p->rp, p->ci, (const double *)grad_b, (const double *)x,
                                                          (double *)grad_val, n);
        CAP_HIP_TRY(hipGetLastError());
        return CAP_OK;
    }
    if (!p->cnt0) {
        CAP_TRY(dev_alloc(&p->cnt0, (size_t)n));
        CAP_TRY(dev_alloc(&p->cnt, (size_t)n));
        CAP_TRY(dev_alloc(&p->adj_ls, (size_t)n));
        k_prepare<unsigned><<<blocks_for(n), kBlock, 0, st>>>((unsigned *)p->cnt0, n, 0u, p->ticket, 0);
        k_offdiag_colcount<<<blocks_for(n), kBlock, 0, st>>>(p->rp, p->ci, n, p->cnt0);
        CAP_HIP_TRY(hipGetLastError());
    }
    CAP_HIP_TRY(hipMemcpyAsync(p->cnt, p->cnt0, sizeof(int) * (size_t)n, hipMemcpyDeviceToDevice, st));
    k_prepare<unsigned long long><<<blocks_for(n), kBlock, 0, st>>>((unsigned long long *)p->adj_ls, n, 0ULL,
                                                                    p->ticket, kTickets);
    SyncCtx sc{p->flags, p->epoch, p->spin_limit, p->err, nullptr, p->unfused, p->wait_ticks};
    k_adjoint<<<grid_for(p, ((long long)n + kBlock - 1) / kBlock), kBlock, 0, st>>>(
        p->rp, p->ci, (const double *)p->val, (const double *)g, (const double *)x, p->cnt, p->adj_ls,
        (double *)grad_b, (double *)grad_val, n, sc, p->ticket);
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

}  // extern "C"

// ------------------------------------------------------------- refinement
namespace {

// Grid of the grid-stride streaming kernels: 8 workgroups per compute unit,
// fewer when the work is small.
inline unsigned stream_blocks(const cap_plan p, long long count)
{
    return std::max(1u, std::min(blocks_for(count), (unsigned)p->ncu * 8u));
}

// Plans whose solve is thread-per-row run the first two refinement steps as
// one fused sweep; one-workgroup (LOCAL) and partitioned plans run them as
// separate one-workgroup solves.
inline bool refine_fuses(const cap_plan p) { return p->algo != CAP_ALGO_LOCAL && p->algo != CAP_ALGO_PARTITION; }

// What the steps after a fused sweep, or all of them, work on: the FP32
// values, residual and correction.
int ensure_refine(cap_plan p, int rhs, hipStream_t st)
{
    const long long len = (long long)p->n * rhs;
    if (!p->val32) {
        CAP_TRY(dev_alloc(&p->val32, (size_t)p->nnz));
        k_cast_f32<<<blocks_for(p->nnz), kBlock, 0, st>>>((const double *)p->val, p->val32, p->nnz);
        CAP_HIP_TRY(hipGetLastError());
    }
    if (p->refine_len < len) {
        if (p->r32) CAP_HIP_TRY(hipFree(p->r32));
        if (p->d32) CAP_HIP_TRY(hipFree(p->d32));
        p->r32 = p->d32 = nullptr;
        CAP_TRY(dev_alloc(&p->r32, (size_t)len));
        CAP_TRY(dev_alloc(&p->d32, (size_t)len));
        p->refine_len = len;
    }
    return CAP_OK;
}

// Where the fused sweep publishes its pairs, when readiness is in place.
int ensure_pairs(cap_plan p, int rhs)
{
    const long long len = (long long)p->n * rhs;
    if (p->staged || p->pair_len >= len) return CAP_OK;
    if (p->pair) CAP_HIP_TRY(hipFree(p->pair));
    p->pair = nullptr;
    p->pair_len = 0;
    CAP_TRY(dev_alloc(&p->pair, (size_t)len));
    p->pair_len = len;
    return CAP_OK;
}

// The first two refinement steps as one sweep (k_refine2): the norms and
// the pair array (staged: the readiness array; else the plan's own) reset
// with the tickets, then the thread-per-row launch with the plan's grid,
// LDS window and batch schedule.
// join (hybrid batches): side streams that end before the sweep starts.  Its
// persistent workgroups need a compute unit each: started while others still
// hold some, two of them shared one for all of the sweep (256 matrices, 16
// right-hand sides: sweep 9.55 ms instead of 9.25).
int refine_fused(cap_plan p, const double *b, double *x, int rhs, hipStream_t st, const Fork *join = nullptr)
{
    typedef unsigned long long U;
    const long long len = (long long)p->n * rhs;
    U *pr = p->staged ? reinterpret_cast<U *>(p->ready) : p->pair;
    if (!pr || (p->staged && p->ready_bytes < sizeof(U) * (size_t)len) || (!p->staged && p->pair_len < len))
        return CAP_ERR_ARG;
    const unsigned nbp = std::max(1u, std::min(blocks_for(len), 2048u));
    k_prepare_norms<U><<<nbp, kBlock, 0, st>>>(pr, len, VBits<double>::kSentinel, p->ticket, kTickets, p->norms);
    CAP_HIP_TRY(hipGetLastError());
    if (join) CAP_TRY(join_parts(join, st));
    if (p->n == 0) return CAP_OK;
    RhsScope own(p, 1);
    if (p->plain.bpc && !hop_takes(p, rhs)) {
        const int staged = p->staged;  // where pr is
        own.take(p->plain);
        p->staged = staged;
    }
    const int l = lpr_log2_for(rhs);
    // the sweep's own sizes: 128 or 256 threads, or 1024 for a batch that
    // picked it for several right-hand sides (no LDS window)
    const int block = refine_block(p, rhs);
    const int rows_per_block = block >> l;
    int n_sched = 0;
    const int2 *sched = sched_for(p, rows_per_block, &n_sched);
    const bool use_sched = sched != nullptr;
    const unsigned nb = grid_for(p, use_sched ? n_sched : ((long long)p->n + rows_per_block - 1) / rows_per_block);
    const SyncCtx sc{p->flags, p->epoch, p->spin_limit, p->err, nullptr, 0, p->wait_ticks};
    const double *val = (const double *)p->val;
    auto go = [&](auto kernel) {
        kernel<<<nb, block, 0, st>>>(p->rp, p->ci, val, b, x, pr, sc, p->n, rhs, l, p->ticket, sched, n_sched,
                                     p->norms);
    };
    const bool small = block == kBlockSmall;
    if (hop_takes(p, rhs)) {
        const HopTab tab{p->hop->base, p->hop->ex, p->hop->npad};
        auto look = [&](auto kernel) {
            kernel<<<nb, block, 0, st>>>(tab, val, b, x, pr, sc, p->n, p->ticket, p->norms);
        };
        if (p->hop->E == 2)
            small ? look(k_refine_hop<2, kBlockSmall>) : look(k_refine_hop<2, kBlock>);
        else if (p->hop->E == 3)
            small ? look(k_refine_hop<3, kBlockSmall>) : look(k_refine_hop<3, kBlock>);
        else
            small ? look(k_refine_hop<4, kBlockSmall>) : look(k_refine_hop<4, kBlock>);
    } else if (block == kBlockLarge)
        go(k_refine2<0, kBlockLarge>);
    else if (p->lds)
        small ? go(k_refine2<1, kBlockSmall>) : go(k_refine2<1, kBlock>);
    else
        small ? go(k_refine2<0, kBlockSmall>) : go(k_refine2<0, kBlock>);
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

// The refinement norms, once everything before on `st` is done.  A kernel
// writes them into pinned memory with a count, which the host watches for: a
// refined solve of n = 1,000,000 takes 102.5 us, and 118.7 with a copy to the
// stack and a stream synchronization.  After 2 ms the host waits for the
// stream.
int read_norms(cap_plan p, unsigned long long *nb, hipStream_t st)
{
    if (!p->echo) CAP_TRY(echo_acquire(&p->echo));
    const unsigned long long count = ++p->echoes;
    k_echo<<<1, kWave, 0, st>>>(p->norms, p->echo, count);
    CAP_HIP_TRY(hipGetLastError());
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
    while (__atomic_load_n(p->echo + 2, __ATOMIC_ACQUIRE) != count) {
        if (std::chrono::steady_clock::now() < until) continue;
        CAP_HIP_TRY(hipStreamSynchronize(st));
        break;
    }
    nb[0] = p->echo[0];
    nb[1] = p->echo[1];
    return CAP_OK;
}

// One refinement step on `st`: r32 = b - L x (or b when first), d = L32^{-1} r32
// in FP32 (value protocol), x += d; norms[0] = max|d| bits, norms[1] = max|x|.
int refine_step(cap_plan p, const double *b, double *x, int rhs, bool first, hipStream_t st)
{
    const long long len = (long long)p->n * rhs;
    k_prepare<unsigned long long><<<1, kBlock, 0, st>>>(p->norms, 2, 0ULL, p->ticket, 0);
    if (first)
        k_cast_f32<<<blocks_for(len), kBlock, 0, st>>>(b, p->r32, len);
    else
        k_residual32<<<stream_blocks(p, len), kBlock, 0, st>>>(p->rp, p->ci, (const double *)p->val, b, x, p->r32,
                                                                p->n, rhs, p->norms + 1);
    CAP_HIP_TRY(hipGetLastError());
    // the correction solves use the plan's multi-RHS path: LOCAL (deep plans,
    // partitioned ones included) or WRTFST
    const int algo = p->algo == CAP_ALGO_LOCAL || p->algo == CAP_ALGO_PARTITION ? CAP_ALGO_LOCAL : CAP_ALGO_WRTFST;
    CAP_TRY(launch_prepare<float>(p, algo, CAP_SYNC_VALUE, p->d32, len, st));
    CAP_TRY(launch_kernel<float>(p, algo, CAP_SYNC_VALUE, p->val32, p->r32, p->d32, rhs, st, true));
    for (const int2 &sk : p->skip_rows) {  // rows no schedule block covers: no correction
        const long long c = (long long)sk.y * rhs;
        k_fill<unsigned><<<blocks_for(c), kBlock, 0, st>>>((unsigned *)p->d32 + (long long)sk.x * rhs, c, 0u);
    }
    k_accumulate<<<stream_blocks(p, len), kBlock, 0, st>>>(x, p->d32, len, p->norms, first ? 1 : 0);
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

// Workgroup size of the fused sweep on an autotuned plan: its critical path
// (two FP32 divisions and an FP64 fma per row) is longer than the solve's, so
// its best size can differ.  The first refined solve times 128 and 256
// threads on the caller's b and x (x is overwritten by the solve that
// follows) and keeps the faster; 256 must be 2% faster to win.
int tune_refine_block(cap_plan p, const double *b, double *x, int rhs, hipStream_t st)
{
    hipEvent_t e0, e1;
    CAP_HIP_TRY(hipEventCreate(&e0));
    CAP_HIP_TRY(hipEventCreate(&e1));
    float best[2] = {1e30f, 1e30f};
    const int sizes[2] = {kBlockSmall, kBlock};
    int rc = CAP_OK;
    for (int c = 0; c < 2 && rc == CAP_OK; ++c) {
        p->rblock = sizes[c];
        for (int r = 0; r < 3 && rc == CAP_OK; ++r) {
            (void)hipEventRecord(e0, st);
            rc = refine_fused(p, b, x, rhs, st);
            (void)hipEventRecord(e1, st);
            if (hipEventSynchronize(e1) != hipSuccess) rc = CAP_ERR_HIP;
            float t = 0;
            (void)hipEventElapsedTime(&t, e0, e1);
            if (r > 0) best[c] = std::min(best[c], t);
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    p->rblock = best[1] < 0.98f * best[0] ? kBlock : kBlockSmall;
    return rc;
}

// Refined solve of a partitioned plan (k right-hand sides).  The partition
// keeps FP64 tables only, so the solves are FP64 partitioned solves: x = P b,
// then corrections d = P (b - L x), x += d, with the same convergence test as
// the FP32 refinement, over all right-hand sides (the first correction is
// normally the last).
int refined_partition(cap_plan p, const double *b, double *x, int k, double tol, int max_iter, int *iters,
                      double *last_rel, hipStream_t st)
{
    PartState *ps = p->part;
    const long long count = (long long)p->n * k;
    CAP_TRY(launch_partition(p, b, x, k, st));  // sizes the work vectors for k
    if (!ps->res) {
        CAP_TRY(dev_alloc(&ps->res, (size_t)p->n * ps->kcap));
        CAP_TRY(dev_alloc(&ps->cor, (size_t)p->n * ps->kcap));
    }
    const unsigned nb = stream_blocks(p, count);
    double prev_rel = 1.0, rel = 1.0;
    int it = 1, rc = CAP_OK;
    while (true) {
        k_prepare<unsigned long long><<<1, kBlock, 0, st>>>(p->norms, 2, 0ULL, p->ticket, 0);
        k_residual64<<<nb, kBlock, 0, st>>>(p->rp, p->ci, (const double *)p->val, b, x, ps->res, p->n, k,
                                            p->norms + 1);
        CAP_HIP_TRY(hipGetLastError());
        CAP_TRY(launch_partition(p, ps->res, ps->cor, k, st));
        k_accumulate64<<<nb, kBlock, 0, st>>>(x, ps->cor, count, p->norms);
        CAP_HIP_TRY(hipGetLastError());
        ++it;
        unsigned long long nbits[2];
        CAP_TRY(read_norms(p, nbits, st));
        double dmax, xmax;
        std::memcpy(&dmax, &nbits[0], 8);
        std::memcpy(&xmax, &nbits[1], 8);
        prev_rel = it == 2 ? 1.0 : rel;
        rel = xmax > 0 ? dmax / xmax : dmax;
        const double est = rel * std::min(1.0, rel / std::max(prev_rel, 1e-300));
        if (rel <= tol || est <= tol) break;
        if (it >= max_iter) {
            rc = CAP_ERR_NOT_CONVERGED;
            break;
        }
    }
    if (iters) *iters = it;
    if (last_rel) *last_rel = rel;
    return rc;
}

// join (hybrid batches): side streams whose partitioned solves run beside the
// fused sweep's reset (or the first two steps, which touch only the plan's
// scheduled rows); they are joined into st before the sweep, at the latest
// before the convergence readback, since the later steps read and update
// every row of x.
int refined_impl(cap_plan p, const double *b, double *x, int rhs, double tol, int max_iter, int *iters,
                 double *last_rel, hipStream_t st, const Fork *join = nullptr)
{
    if (!p || !b || !x || rhs < 1 || rhs > kWave || max_iter < 1) return CAP_ERR_ARG;
    if (p->vt != CAP_F64 || p->reversed || p->unit_diag) return CAP_ERR_UNSUPPORTED;
    // every refined solve of a partitioned plan (any max_iter) runs FP64
    // partitioned solves: the plan has no segment table for LOCAL FP32
    // corrections, and building one inside the graph capture below would
    // allocate there
    if (p->algo == CAP_ALGO_PARTITION && p->part)
        return refined_partition(p, b, x, rhs, tol, max_iter, iters, last_rel, st);
    // the staged readiness array must exist before capture (no allocation
    // inside the captured steps, whose kernels bake in its address); the
    // fused sweep publishes 8-byte pairs, the correction solves 4-byte values
    const bool fused = refine_fuses(p);
    CAP_TRY(fused ? ensure_pairs(p, rhs) : ensure_refine(p, rhs, st));
    if (p->staged) CAP_TRY(ensure_ready(p, (fused ? 8 : 4) * (size_t)p->n * rhs));
    if (fused && !p->rblock) CAP_TRY(tune_refine_block(p, b, x, rhs, st));
    // The fused sweep is two launches: a graph of them saves nothing (101 us a
    // call, 96 without, n = 1,000,000) and its stream, capture and
    // instantiation, up to 0.5 ms, fall on every new (b, x).  The first two
    // unfused steps (solve from b, one correction) are one, captured once per
    // (b, x, rhs), replayed on later calls.
    if (fused) {
        CAP_TRY(refine_fused(p, b, x, rhs, st, join));
    } else if (!p->refine_graph || p->graph_b != b || p->graph_x != x || p->graph_rhs != rhs) {
        if (p->refine_graph) CAP_HIP_TRY(hipGraphExecDestroy(p->refine_graph));
        p->refine_graph = nullptr;
        hipStream_t cs;
        CAP_HIP_TRY(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
        hipGraph_t graph;
        CAP_HIP_TRY(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
        int rc = refine_step(p, b, x, rhs, true, cs);
        if (rc == CAP_OK) rc = refine_step(p, b, x, rhs, false, cs);
        hipError_t ec = hipStreamEndCapture(cs, &graph);
        if (rc != CAP_OK || ec != hipSuccess) {
            (void)hipStreamDestroy(cs);
            return rc != CAP_OK ? rc : CAP_ERR_HIP;
        }
        CAP_HIP_TRY(hipGraphInstantiate(&p->refine_graph, graph, nullptr, nullptr, 0));
        CAP_HIP_TRY(hipGraphDestroy(graph));
        CAP_HIP_TRY(hipStreamDestroy(cs));
        p->graph_b = b;
        p->graph_x = x;
        p->graph_rhs = rhs;
    }
    double prev_rel = 1.0, rel = 1.0;
    int it = 0;
    unsigned long long nb[2];
    int rc = CAP_OK;
    if (!fused) CAP_HIP_TRY(hipGraphLaunch(p->refine_graph, st));
    if (join) CAP_TRY(join_parts(join, st));
    it = 2;
    while (true) {
        CAP_TRY(read_norms(p, nb, st));
        double dmax, xmax;
        std::memcpy(&dmax, &nb[0], 8);
        std::memcpy(&xmax, &nb[1], 8);
        prev_rel = it == 2 ? 1.0 : rel;
        rel = xmax > 0 ? dmax / xmax : dmax;
        // the error left after this correction is about rel times the
        // observed contraction rel/prev_rel
        const double est = rel * std::min(1.0, rel / std::max(prev_rel, 1e-300));
        if (rel <= tol || est <= tol) break;
        if (it >= max_iter) {
            rc = CAP_ERR_NOT_CONVERGED;
            break;
        }
        CAP_TRY(ensure_refine(p, rhs, st));
        CAP_TRY(refine_step(p, b, x, rhs, false, st));
        ++it;
    }
    if (iters) *iters = it;
    if (last_rel) *last_rel = rel;
    return rc;
}

}  // namespace

extern "C" int cap_plan_solve_refined(cap_plan p, const double *b, double *x, int rhs, double tol, int max_iter,
                                      int *iters, double *last_rel, void *stream)
{
    return refined_impl(p, b, x, rhs, tol, max_iter, iters, last_rel, S(stream));
}

// ---------------------------------------------------------------- batches
namespace {

// Row levels of a batch's block-diagonal matrix (host copy).
int batch_levels(cap_plan p, std::vector<int> *rp, std::vector<int> *ci, std::vector<int> *lv)
{
    const int n = p->n, nnz = p->nnz;
    rp->resize((size_t)n + 1);
    ci->resize((size_t)nnz);
    lv->assign((size_t)std::max(n, 1), 0);
    CAP_HIP_TRY(hipMemcpy(rp->data(), p->rp, sizeof(int) * ((size_t)n + 1), hipMemcpyDeviceToHost));
    CAP_HIP_TRY(hipMemcpy(ci->data(), p->ci, sizeof(int) * (size_t)nnz, hipMemcpyDeviceToHost));
    cap_matrix_layer(n, rp->data(), ci->data(), nullptr, nullptr, lv->data());
    return CAP_OK;
}

// Block schedule of a batch: every matrix is cut into blocks of `rows`
// consecutive rows, and a stable sort by key interleaves the matrices so
// that all of them advance in one launch instead of one after another.
// Built once per size into `into` (default: the plan's schedules); matrices
// with skip[m] set get no blocks (a hybrid batch solves them apart).
int build_batch_schedule(cap_plan p, const std::vector<int> &ro, const std::vector<int> &lv, int rows,
                         hipStream_t st, const std::vector<char> *skip = nullptr,
                         std::map<int, std::pair<int2 *, int>> *into = nullptr)
{
    if (!into) into = &p->scheds;
    if (into->count(rows)) return CAP_OK;
    const int n = p->n, n_mat = (int)ro.size() - 1;
    struct Blk {
        double key;
        int lo, len;
    };
    // Blocks are handed out by relative progress: a block's key is the
    // running maximum level of its rows divided by its matrix's depth, so
    // every matrix advances through its levels at the same pace and the
    // deepest one does not wait behind the early levels of all the others.
    // Keys never decrease along a matrix's rows and the sort is stable, so
    // each matrix keeps its row order.
    std::vector<Blk> blks;
    blks.reserve((size_t)n / rows + n_mat + 1);
    for (int m = 0; m < n_mat; ++m) {
        if (skip && (*skip)[(size_t)m]) continue;
        int depth = 1;
        for (int r = ro[m]; r < ro[m + 1]; ++r) depth = std::max(depth, lv[r] + 1);
        int run = 0;
        for (int lo = ro[m]; lo < ro[m + 1]; lo += rows) {
            const int hi = std::min(lo + rows, ro[m + 1]);
            run = std::max(run, lv[lo]);
            blks.push_back({(double)run / depth, lo, hi - lo});
            for (int r = lo; r < hi; ++r) run = std::max(run, lv[r]);
        }
    }
    std::stable_sort(blks.begin(), blks.end(), [](const Blk &a, const Blk &b) { return a.key < b.key; });
    std::vector<int2> h(blks.size());
    for (size_t t = 0; t < blks.size(); ++t) h[t] = make_int2(blks[t].lo, blks[t].len);
    int2 *d = nullptr;
    CAP_TRY(dev_alloc(&d, std::max<size_t>(h.size(), 1)));
    (*into)[rows] = {d, (int)h.size()};
    CAP_HIP_TRY(hipMemcpyAsync(d, h.data(), sizeof(int2) * h.size(), hipMemcpyHostToDevice, st));
    CAP_HIP_TRY(hipStreamSynchronize(st));
    return CAP_OK;
}

// Rows per block of the thread-per-row solve and of the fused refinement
// sweep of a batch plan with k right-hand sides (their schedules' sizes).
int batch_solve_rows(cap_plan p, int k)
{
    if (p->wblock == kBlockLarge && p->rpl > 1) return kBlockLarge >> lpr_log2_for((k + p->rpl - 1) / p->rpl);
    return p->wblock >> lpr_log2_for(k);
}
int batch_refine_rows(cap_plan p, int k) { return refine_block(p, k) >> lpr_log2_for(k); }

// A batch runs either the scheduled thread-per-row kernel over all matrices
// or one workgroup per matrix; unless the caller named one, both are timed
// on the batch itself (b = 1) and the faster is kept.  Unless the caller set
// blocks_per_cu, the thread-per-row grid is timed at 1, 2 and 4 workgroups
// per compute unit (the schedule's pace depends on how many blocks are in
// flight); a size must be 2% faster than a smaller one to win.
int choose_batch_algo(cap_plan p, int requested, int bpc_fixed, int k, const std::vector<int> &ro,
                      const std::vector<int> &lv, hipStream_t st)
{
    if (requested == CAP_ALGO_LOCAL || (requested == CAP_ALGO_WRTFST && bpc_fixed)) {
        p->algo = requested;
        return CAP_OK;
    }
    if (requested != CAP_ALGO_AUTO && requested != CAP_ALGO_WRTFST) return CAP_ERR_ARG;
    const size_t bytes = (size_t)p->n * k * p->vbytes + 8;
    void *b = nullptr, *x = nullptr;
    CAP_HIP_TRY(hipMalloc(&b, bytes));
    if (hipMalloc(&x, bytes) != hipSuccess) {
        (void)hipFree(b);
        return CAP_ERR_ALLOC;
    }
    int rc = tuning_rhs(p, b, (long long)p->n * k, st);
    float t_w = 1e30f, t_l = 1e30f;
    int best_bpc = p->bpc;
    std::vector<int> sizes = {1, 2, 4};
    if (bpc_fixed) sizes = {p->bpc};
    for (int bpc : sizes) {
        if (rc != CAP_OK) break;
        const int keep = p->bpc;
        p->bpc = bpc;
        float t = 1e30f;
        rc = time_candidate(p, CAP_ALGO_WRTFST, p->sync, b, x, k, st, t_w, &t);
        p->bpc = keep;
        if (t < (t_w < 1e30f ? 0.98f : 1.0f) * t_w) {
            t_w = t;
            best_bpc = bpc;
        }
    }
    p->bpc = best_bpc;
    // several right-hand sides: 1024-thread workgroups with R per lane put
    // more rows in each ticket (one atomic on one counter, ~12 ns each),
    // each with a schedule of its own block size
    if (rc == CAP_OK && k > 1 && !bpc_fixed && p->sync == CAP_SYNC_VALUE && !p->lds && !p->count_polls) {
        int best_r = 0, best_tile = 0;
        for (int rt : {1, -1, 2, 4}) {  // R per lane; -1: one per lane with row tiles
            const int r = rt < 0 ? 1 : rt, tile = rt < 0 ? 1 : 0;
            if (rc != CAP_OK || r > k) break;
            const int keep_bpc = p->bpc, keep_blk = p->wblock, keep_rpl = p->rpl, keep_tile = p->tile;
            p->bpc = 1;
            p->wblock = kBlockLarge;
            p->rpl = r;
            p->tile = tile;
            rc = build_batch_schedule(p, ro, lv, kBlockLarge >> lpr_log2_for((k + r - 1) / r), st);
            float t = 1e30f;
            if (rc == CAP_OK) rc = time_candidate(p, CAP_ALGO_WRTFST, p->sync, b, x, k, st, t_w, &t);
            p->bpc = keep_bpc;
            p->wblock = keep_blk;
            p->rpl = keep_rpl;
            p->tile = keep_tile;
            if (t < 0.98f * t_w) {
                t_w = t;
                best_r = r;
                best_tile = tile;
            }
        }
        if (best_r) {
            p->bpc = 1;
            p->wblock = kBlockLarge;
            p->rpl = best_r;
            p->tile = best_tile;
            p->rblock = kBlockLarge;  // the refinement sweep's tickets too
            rc = build_batch_schedule(p, ro, lv, batch_refine_rows(p, k), st);
        }
    }
    if (rc == CAP_OK && requested == CAP_ALGO_AUTO)
        rc = time_candidate(p, CAP_ALGO_LOCAL, CAP_SYNC_VALUE, b, x, k, st, t_w, &t_l);
    (void)hipStreamSynchronize(st);
    (void)hipFree(b);
    (void)hipFree(x);
    if (rc != CAP_OK) return rc;
    p->algo = t_l < t_w ? CAP_ALGO_LOCAL : CAP_ALGO_WRTFST;
    return CAP_OK;
}

// One solve of a batch, all on st: the partitioned matrices (each writes
// only its own rows) and the thread-per-row or one-workgroup solve of the
// rest.  With staged readiness the partitioned ones go first; with
// readiness in x the rest goes first, since its reset fills all of x with
// the sentinel.  (On a second stream, overlapping the rest's persistent
// kernel, the partitioned solves slowed its chain more than they saved:
// 256 x 16 batch 11.5 against 10.9 ms.)
int plan_reset_with(cap_plan p, int algo, int sync, void *x, int rhs, hipStream_t st)
{
    return p->vt == CAP_F64 ? reset_t<double>(p, algo, sync, x, rhs, st) : reset_t<float>(p, algo, sync, x, rhs, st);
}

int plan_launch_with(cap_plan p, int algo, int sync, const void *b, void *x, int rhs, hipStream_t st)
{
    return p->vt == CAP_F64
               ? launch_kernel<double>(p, algo, sync, (const double *)p->val, (const double *)b, (double *)x, rhs, st)
               : launch_kernel<float>(p, algo, sync, (const float *)p->val, (const float *)b, (float *)x, rhs, st);
}

// One solve of a batch on st: the partitioned matrices on the side streams
// alongside the rest's solve on st.  The rest's reset and kernel touch only
// the rest's rows of x and its own readiness state, except that a reset
// with readiness in x fills every row of x: then it runs before the fork.
int batch_solve_parts(cap_plan p, const std::vector<cap_plan> &parts, const std::vector<int> &lo, int k,
                      const void *b, void *x, hipStream_t st, const Fork *fk)
{
    // the rest by steps: no reset, only the rest's rows of x are touched
    const StepTables *steps = p->batch_steps;
    if (parts.empty())
        return steps ? steps_launch(steps, b, x, k, p->unfused != 0, st)
                     : plan_solve_with(p, p->algo, p->sync, b, x, k, st);
    const size_t row_bytes = (size_t)k * p->vbytes;
    const bool x_reset = !steps && !p->staged && p->algo != CAP_ALGO_LOCAL;
    if (x_reset) CAP_TRY(plan_reset_with(p, p->algo, p->sync, x, k, st));
    int rc = fork_parts(parts.size(), fk, st, [&](size_t h, hipStream_t s) {
        return plan_solve_with(parts[h], parts[h]->algo, parts[h]->sync, (const char *)b + lo[h] * row_bytes,
                               (char *)x + lo[h] * row_bytes, k, s);
    });
    if (rc == CAP_OK && steps) {
        rc = steps_launch(steps, b, x, k, p->unfused != 0, st);
    } else {
        if (rc == CAP_OK && !x_reset) rc = plan_reset_with(p, p->algo, p->sync, x, k, st);
        if (rc == CAP_OK) rc = plan_launch_with(p, p->algo, p->sync, b, x, k, st);
    }
    const int rj = join_parts(fk, st);  // joined whatever happened
    return rc != CAP_OK ? rc : rj;
}

float time_batch(cap_plan p, const std::vector<cap_plan> &parts, const std::vector<int> &lo, int k, const void *b,
                 void *x, hipStream_t st, int *rc, const Fork *fk = nullptr)
{
    hipEvent_t e0 = nullptr, e1 = nullptr;
    float best = 1e30f;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        *rc = CAP_ERR_HIP;
    } else {
        for (int r = 0; r < 3 && *rc == CAP_OK; ++r) {
            (void)hipEventRecord(e0, st);
            *rc = batch_solve_parts(p, parts, lo, k, b, x, st, fk);
            (void)hipEventRecord(e1, st);
            (void)hipEventSynchronize(e1);
            float t = 0;
            (void)hipEventElapsedTime(&t, e0, e1);
            if (r > 0) best = std::min(best, t);  // the first run is a warm-up
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return best;
}

// Steps for a batch's matrices (those outside `lo`, the partitioned ones):
// kept where the tables fit and the whole batch solve is 2 % faster with
// them.  The thread-per-row schedule pays a cross-CU hop per level of the
// deepest matrix (1.16 us on 40 matrices of up to 775 levels with 16
// right-hand sides, 898 us); a step inside one CU costs 0.33 us there.
int choose_batch_steps(cap_plan p, int k, const std::vector<int> &ro, const std::vector<int> &rp,
                       const std::vector<int> &ci, const std::vector<cap_plan> &parts, const std::vector<int> &lo,
                       const Fork *fk, hipStream_t st)
{
    std::vector<int2> mats;
    for (size_t m = 0; m + 1 < ro.size(); ++m)
        if (ro[m + 1] > ro[m] && std::find(lo.begin(), lo.end(), ro[m]) == lo.end())
            mats.push_back(make_int2(ro[m], ro[m + 1]));
    if (mats.empty()) return CAP_OK;
    StepTables *t = nullptr;
    int rc = steps_build(&t, rp, ci, mats, p->vt, 4, 0, p->lds_max, kStepPadMax, kStepMaxBytes, p->rp, p->ci, p->val, st);
    if (rc == CAP_ERR_UNSUPPORTED || rc == CAP_ERR_ALLOC) return CAP_OK;  // the plain batch stays
    if (rc != CAP_OK) return rc;
    if (!steps_take(t, k)) {
        steps_free(t);
        return CAP_OK;
    }
    const size_t bytes = (size_t)p->n * k * p->vbytes + 8;
    void *b = nullptr, *x = nullptr;
    if (hipMalloc(&b, bytes) != hipSuccess || hipMalloc(&x, bytes) != hipSuccess ||
        tuning_rhs(p, b, (long long)p->n * k, st) != CAP_OK)
        rc = CAP_ERR_ALLOC;
    float plain = 0, with = 0;
    if (rc == CAP_OK) plain = time_batch(p, parts, lo, k, b, x, st, &rc, fk);
    p->batch_steps = t;
    if (rc == CAP_OK) with = time_batch(p, parts, lo, k, b, x, st, &rc, fk);
    (void)hipStreamSynchronize(st);
    (void)hipFree(b);
    (void)hipFree(x);
    if (rc != CAP_OK || with >= 0.98f * plain) {
        p->batch_steps = nullptr;
        steps_free(t);
    }
    return rc;
}

// Hybrid batch: a deep matrix (few rows per level) sets the whole batch's
// time with its chain of levels, and a partitioned solve shortens exactly
// that.  Matrices are taken deepest first while each is deep and its
// partitioned plan builds (lower bandwidth <= 256, blocks stable); the first
// matrix that is not stops the list, since the rest's time is the deepest
// remaining chain.  Without its deep chains the rest is bound by how fast
// rows are handed out (one ticket atomic per block, ~12 ns each), so its
// thread-per-row shape is timed again: 1, 2 and 4 workgroups of 256 threads
// per CU, and 1024-thread workgroups with 1, 2 or 4 right-hand sides per
// lane, each over a schedule without the partitioned matrices.  The
// fastest hybrid is kept when 2 % faster than the plain batch as it
// resolved (thread-per-row or one workgroup per matrix).  The kept plans go
// to *parts.  With several right-hand sides the rest is also timed with
// readiness in x itself (one store per value instead of two).  Plans in the
// reference arithmetic or created with readiness in place are left as they
// are.
constexpr int kHybridMax = 8;           // partitioned matrices per batch, at most
constexpr int kHybridMinLevels = 1024;  // deep enough for a chain to matter

constexpr int kSideStreams = 3;  // the partitioned solves' streams (hardware queues are few)

int choose_batch_hybrid(cap_plan p, int k, bool bpc_fixed, const std::vector<int> &ro, const std::vector<int> &lv,
                        hipStream_t st, std::vector<cap_plan> *parts, std::vector<int> *lo, Fork *fk)
{
    if (p->unfused || !p->staged) return CAP_OK;
    const int n_mat = (int)ro.size() - 1;
    std::vector<int> depth((size_t)n_mat, 1), order((size_t)n_mat);
    for (int m = 0; m < n_mat; ++m) {
        for (int r = ro[m]; r < ro[m + 1]; ++r) depth[(size_t)m] = std::max(depth[(size_t)m], lv[r] + 1);
        order[(size_t)m] = m;
    }
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return depth[(size_t)a] > depth[(size_t)b]; });
    // the deep matrices' partitioned plans, from host copies of their rows
    std::vector<cap_plan> cand;
    std::vector<int> cand_lo;
    std::vector<char> skip((size_t)n_mat, 0);
    int rc = CAP_OK;
    for (int m : order) {
        const int nm = ro[m + 1] - ro[m];
        if ((int)cand.size() >= kHybridMax || depth[(size_t)m] < kHybridMinLevels ||
            (double)nm / depth[(size_t)m] > kLocalMaxWidth)
            break;
        std::vector<int> rp((size_t)nm + 1);
        CAP_HIP_TRY(hipMemcpy(rp.data(), p->rp + ro[m], sizeof(int) * rp.size(), hipMemcpyDeviceToHost));
        const int e0 = rp[0], nnz = rp[(size_t)nm] - e0;
        std::vector<int> ci((size_t)nnz);
        std::vector<char> val((size_t)nnz * p->vbytes);
        CAP_HIP_TRY(hipMemcpy(ci.data(), p->ci + e0, sizeof(int) * ci.size(), hipMemcpyDeviceToHost));
        CAP_HIP_TRY(hipMemcpy(val.data(), (const char *)p->val + (size_t)e0 * p->vbytes, val.size(),
                              hipMemcpyDeviceToHost));
        for (int &r : rp) r -= e0;
        for (int &c : ci) c -= ro[m];  // global columns to the matrix's own
        cap_opts o;
        cap_opts_default(&o);
        o.algo = CAP_ALGO_PARTITION;
        o.host_inputs = 1;
        o.validate = 0;  // checked with the batch
        o.spin_limit = p->spin_limit;
        o.wait_limit_ms = p->wait_ticks > 0 ? p->wait_ticks / 100000 : -1;
        cap_plan q = nullptr;
        rc = plan_create_impl(&q, nm, nnz, rp.data(), ci.data(), val.data(), p->vt, &o, st);
        if (rc == CAP_ERR_UNSUPPORTED) {  // band or stability: the list stops here
            rc = CAP_OK;
            break;
        }
        if (rc != CAP_OK) break;
        cand.push_back(q);
        cand_lo.push_back(ro[m]);
        skip[(size_t)m] = 1;
    }
    if (rc == CAP_OK && cand.size() > 1) rc = fk->make(std::min((int)cand.size(), kSideStreams));
    if (rc != CAP_OK || cand.empty()) {
        for (cap_plan q : cand) cap_plan_destroy(q);
        fk->release();
        return rc;
    }
    const size_t bytes = (size_t)p->n * k * p->vbytes + 8;
    void *b = nullptr, *x = nullptr;
    if (hipMalloc(&b, bytes) != hipSuccess || hipMalloc(&x, bytes) != hipSuccess ||
        tuning_rhs(p, b, (long long)p->n * k, st) != CAP_OK)
        rc = CAP_ERR_ALLOC;
    struct Shape {
        int bpc, block, rpl;
        bool staged;
        int tile;
    };
    std::vector<Shape> shapes = {{1, kBlock, 1, true, 0}, {2, kBlock, 1, true, 0}, {4, kBlock, 1, true, 0}};
    if (k > 1 && p->sync == CAP_SYNC_VALUE && !p->lds && !p->count_polls)  // the multi-RHS shapes
        for (int r : {1, 2, 4})
            if (r <= k)
                for (bool sg : {true, false}) {
                    shapes.push_back({1, kBlockLarge, r, sg, 0});
                    if (r == 1) shapes.push_back({1, kBlockLarge, r, sg, 1});  // with row tiles
                }
    if (bpc_fixed) shapes = {{p->bpc, p->wblock, p->rpl, true, p->tile}};  // the caller's grid stays
    const Shape plain{p->bpc, p->wblock, p->rpl, p->staged != 0, p->tile};
    const int plain_algo = p->algo;
    Shape pick{0, 0, 0, true, 0};
    float best = 1e30f;
    std::map<int, std::pair<int2 *, int>> trial;  // the rest's schedules, by rows per block
    if (rc == CAP_OK) best = time_batch(p, {}, {}, k, b, x, st, &rc);
    if (rc == CAP_OK) {
        float best_h = 1e30f;
        std::swap(p->scheds, trial);  // the hybrid's rest runs over the trial schedules
        p->algo = CAP_ALGO_WRTFST;
        for (const Shape &sh : shapes) {
            p->bpc = sh.bpc;
            p->wblock = sh.block;
            p->rpl = sh.rpl;
            p->staged = sh.staged;
            p->tile = sh.tile;
            if ((rc = build_batch_schedule(p, ro, lv, batch_solve_rows(p, k), st, &skip)) != CAP_OK) break;
            const float t = time_batch(p, cand, cand_lo, k, b, x, st, &rc, fk);
            if (rc != CAP_OK) break;
            if (t < best_h) {
                best_h = t;
                pick = sh;
            }
        }
        std::swap(p->scheds, trial);
        if (rc == CAP_OK && best_h < 0.98f * best) {
            p->algo = CAP_ALGO_WRTFST;
            p->bpc = pick.bpc;
            p->wblock = pick.block;
            p->rpl = pick.rpl;
            p->staged = pick.staged;
            p->tile = pick.tile;
            // the refinement sweep follows the solve's ticket size
            p->rblock = pick.block == kBlockLarge ? kBlockLarge : (p->rblock == kBlockLarge ? kBlock : p->rblock);
        } else {
            p->algo = plain_algo;
            p->bpc = plain.bpc;
            p->wblock = plain.block;
            p->rpl = plain.rpl;
            p->staged = plain.staged;
            p->tile = plain.tile;
            pick.block = 0;
        }
    }
    (void)hipStreamSynchronize(st);
    (void)hipFree(b);
    (void)hipFree(x);
    for (auto &e : trial) (void)hipFree(e.second.first);
    if (rc == CAP_OK && pick.block) {
        // the kept matrices leave every schedule the plan solves with
        for (auto &e : p->scheds) (void)hipFree(e.second.first);
        p->scheds.clear();
        if ((rc = build_batch_schedule(p, ro, lv, batch_solve_rows(p, k), st, &skip)) == CAP_OK)
            rc = build_batch_schedule(p, ro, lv, batch_refine_rows(p, k), st, &skip);
    }
    if (rc == CAP_OK && pick.block) {
        *parts = cand;
        *lo = cand_lo;
    } else {
        for (cap_plan q : cand) cap_plan_destroy(q);
        fk->release();
    }
    return rc;
}

}  // namespace

extern "C" {

int cap_batch_create(cap_batch *out, int n_mat, const int *row_off, const int *row_ptr, const int *col_idx,
                     const void *val, int vt, int k, const cap_opts *opts, void *stream)
{
    if (!out || n_mat < 1 || !row_off || !row_ptr || !col_idx || !val || k < 1 || k > kWave ||
        (vt != CAP_F64 && vt != CAP_F32))
        return CAP_ERR_ARG;
    *out = nullptr;
    cap_opts o;
    cap_opts_default(&o);
    if (opts) o = *opts;
    if (o.upper || o.unit_diag || o.rhs_per_lane || o.row_tiles) return CAP_ERR_UNSUPPORTED;
    hipStream_t st = S(stream);
    int dev = 0;
    CAP_TRY(check_device(&dev));
    const size_t vb = vt == CAP_F64 ? 8 : 4;
    std::vector<int> ro((size_t)n_mat + 1);
    if (o.host_inputs)
        std::memcpy(ro.data(), row_off, sizeof(int) * ro.size());
    else
        CAP_HIP_TRY(hipMemcpy(ro.data(), row_off, sizeof(int) * ro.size(), hipMemcpyDeviceToHost));
    const int n = ro[n_mat];
    if (ro[0] != 0 || n < 0) return CAP_ERR_ARG;
    for (int m = 0; m < n_mat; ++m)
        if (ro[m + 1] < ro[m]) return CAP_ERR_ARG;
    int nnz = 0;
    if (o.host_inputs)
        nnz = row_ptr[n];
    else
        CAP_HIP_TRY(hipMemcpy(&nnz, row_ptr + n, sizeof(int), hipMemcpyDeviceToHost));
    if (nnz < n) return CAP_ERR_ARG;
    int *d_ro = nullptr, *d_cil = nullptr, *g_rp = nullptr, *g_ci = nullptr;
    void *g_val = nullptr;
    int rc = CAP_OK;
    const hipMemcpyKind kind = o.host_inputs ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice;
    do {
        if ((rc = dev_alloc(&d_ro, ro.size())) || (rc = dev_alloc(&g_rp, (size_t)n + 1)) ||
            (rc = dev_alloc(&g_ci, (size_t)nnz)) || (rc = dev_alloc(&d_cil, (size_t)nnz)))
            break;
        if (hipMalloc(&g_val, (size_t)nnz * vb + 8) != hipSuccess) { rc = CAP_ERR_ALLOC; break; }
        if (hipMemcpy(d_ro, ro.data(), sizeof(int) * ro.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(g_rp, row_ptr, sizeof(int) * ((size_t)n + 1), kind) != hipSuccess ||
            hipMemcpy(d_cil, col_idx, sizeof(int) * (size_t)nnz, kind) != hipSuccess ||
            hipMemcpy(g_val, val, (size_t)nnz * vb, kind) != hipSuccess) {
            rc = CAP_ERR_HIP;
            break;
        }
        k_globalize<<<blocks_for(n), kBlock, 0, st>>>(d_ro, n_mat, g_rp, d_cil, n, g_ci);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess) {
            rc = CAP_ERR_HIP;
            break;
        }
    } while (0);
    (void)hipFree(d_ro);
    (void)hipFree(d_cil);
    cap_plan p = nullptr;
    if (rc == CAP_OK) {
        cap_opts po = o;
        po.host_inputs = 0;
        po.algo = CAP_ALGO_WRTFST;
        if (!po.sync) po.sync = CAP_SYNC_VALUE;
        rc = plan_create_impl(&p, n, nnz, g_rp, g_ci, g_val, vt, &po, st);
    }
    if (rc != CAP_OK) {
        (void)hipFree(g_rp);
        (void)hipFree(g_ci);
        (void)hipFree(g_val);
        return rc;
    }
    p->owns_matrix = true;
    std::vector<int> lv, rp_host, ci_host;
    if ((rc = batch_levels(p, &rp_host, &ci_host, &lv)) != CAP_OK ||
        (rc = build_batch_schedule(p, ro, lv, p->wblock >> lpr_log2_for(k), st)) != CAP_OK ||
        (rc = ensure_segments(p, &ro, &rp_host, &ci_host)) != CAP_OK ||
        (rc = choose_batch_algo(p, o.algo, o.blocks_per_cu > 0, k, ro, lv, st)) != CAP_OK) {
        cap_plan_destroy(p);
        return rc;
    }
    std::vector<cap_plan> parts;
    std::vector<int> part_lo;
    Fork fork;
    if (o.algo == CAP_ALGO_AUTO &&
        (rc = choose_batch_hybrid(p, k, o.blocks_per_cu > 0, ro, lv, st, &parts, &part_lo, &fork)) != CAP_OK) {
        cap_plan_destroy(p);
        return rc;
    }
    if (o.algo == CAP_ALGO_AUTO && o.blocks_per_cu == 0 && p->sync == CAP_SYNC_VALUE && !p->count_polls &&
        (rc = choose_batch_steps(p, k, ro, rp_host, ci_host, parts, part_lo, &fork, st)) != CAP_OK) {
        for (cap_plan q : parts) cap_plan_destroy(q);
        fork.release();
        cap_plan_destroy(p);
        return rc;
    }
    cap_batch bt = new cap_batch_s();
    bt->plan = p;
    bt->k = k;
    bt->n_mat = n_mat;
    bt->parts = parts;
    bt->part_lo = part_lo;
    bt->fork = fork;
    for (size_t h = 0; h < parts.size(); ++h) p->skip_rows.push_back(make_int2(part_lo[h], parts[h]->n));
    *out = bt;
    return CAP_OK;
}

int cap_batch_info(cap_batch bt, int *algo, int *blocks_per_cu)
{
    if (!bt) return CAP_ERR_ARG;
    if (algo) *algo = bt->plan->algo;
    if (blocks_per_cu) *blocks_per_cu = bt->plan->bpc;
    return CAP_OK;
}

int cap_batch_tuning(cap_batch bt, int *row_threads, int *rhs_per_lane, int *partitioned, int *row_tiles)
{
    if (!bt) return CAP_ERR_ARG;
    if (row_tiles) *row_tiles = bt->plan->algo == CAP_ALGO_WRTFST ? bt->plan->tile : 0;
    if (row_threads) *row_threads = bt->plan->wblock;
    if (rhs_per_lane) *rhs_per_lane = bt->plan->wblock == kBlockLarge ? bt->plan->rpl : 1;
    if (partitioned) *partitioned = (int)bt->parts.size();
    return CAP_OK;
}

int cap_batch_partitioned(cap_batch bt, int *first_rows, int capacity)
{
    if (!bt || capacity < 0 || (capacity > 0 && !first_rows)) return CAP_ERR_ARG;
    const int cnt = (int)bt->part_lo.size();
    for (int h = 0; h < std::min(cnt, capacity); ++h) first_rows[h] = bt->part_lo[(size_t)h];
    return cnt;
}

int cap_batch_steps(cap_batch bt, int *matrices)
{
    if (!bt || !matrices) return CAP_ERR_ARG;
    *matrices = bt->plan->batch_steps ? bt->plan->batch_steps->n_jobs : 0;
    return CAP_OK;
}

int cap_batch_solve(cap_batch bt, const void *b, void *x, void *stream)
{
    if (!bt || !b || !x) return CAP_ERR_ARG;
    return batch_solve_parts(bt->plan, bt->parts, bt->part_lo, bt->k, b, x, S(stream), &bt->fork);
}

int cap_batch_solve_refined(cap_batch bt, const double *b, double *x, double tol, int max_iter, int *iters,
                            double *last_rel, void *stream)
{
    if (!bt || !b || !x) return CAP_ERR_ARG;
    // Iterations and correction are the largest over the parts.  A
    // partitioned plan's tables are FP64 and its creation checked its solves
    // against a sequential FP64 solve to kPartStableTol, so at tol >=
    // kPartStableTol its one FP64 solve is the answer (no FP32 step to
    // refine; a correction would only re-solve the rounding noise).  A
    // tighter tol refines each of them in FP64, one after another, before the
    // rest.
    int it_max = 0;
    double rel_max = 0.0;
    int rc = CAP_OK;
    const size_t row = (size_t)bt->k;
    // tol >= kPartStableTol: the partitioned solves on the side streams,
    // enqueued first, alongside the rest's first two steps (joined inside
    // refined_impl).  Enqueued after the sweep's launch instead, so that
    // they start with it rather than ahead of it, the batch took 10.31 ms
    // against 9.95 (256 matrices x 16 right-hand sides): the sweep loses
    // less beside their late, lighter kernels.
    const bool overlap = tol >= kPartStableTol && !bt->parts.empty();
    if (overlap) {
        rc = fork_parts(bt->parts.size(), &bt->fork, S(stream), [&](size_t h, hipStream_t s) {
            return cap_plan_solve(bt->parts[h], b + bt->part_lo[h] * row, x + bt->part_lo[h] * row, bt->k, s);
        });
        it_max = 1;
    }
    // a part that does not converge still leaves its best x: the others run
    for (size_t h = 0; h < bt->parts.size() && tol < kPartStableTol &&
                       (rc == CAP_OK || rc == CAP_ERR_NOT_CONVERGED);
         ++h) {
        const double *bh = b + bt->part_lo[h] * row;
        double *xh = x + bt->part_lo[h] * row;
        int it = 0;
        double rel = 0.0;
        const int rh = refined_impl(bt->parts[h], bh, xh, bt->k, tol, max_iter, &it, &rel, S(stream));
        if (rh != CAP_OK) rc = rh;
        it_max = std::max(it_max, it);
        rel_max = std::max(rel_max, rel);
    }
    if (rc == CAP_OK || rc == CAP_ERR_NOT_CONVERGED) {
        int it = 0;
        double rel = 0.0;
        const int rc2 = refined_impl(bt->plan, b, x, bt->k, tol, max_iter, &it, &rel, S(stream),
                                     overlap ? &bt->fork : nullptr);
        it_max = std::max(it_max, it);
        rel_max = std::max(rel_max, rel);
        if (rc == CAP_OK || (rc2 != CAP_OK && rc2 != CAP_ERR_NOT_CONVERGED)) rc = rc2;
    }
    if (overlap) {  // joined already unless an error came first; joining twice is harmless
        const int rj = join_parts(&bt->fork, S(stream));
        if (rc == CAP_OK) rc = rj;
    }
    if (iters) *iters = it_max;
    if (last_rel) *last_rel = rel_max;
    return rc;
}

int cap_batch_destroy(cap_batch bt)
{
    if (!bt) return CAP_ERR_ARG;
    for (cap_plan q : bt->parts) cap_plan_destroy(q);
    cap_plan_destroy(bt->plan);
    bt->fork.release();
    delete bt;
    return CAP_OK;
}

// -------------------------------------------------------- one-shot solves
}  // extern "C"

namespace {

template <typename T>
int oneshot(int n, int nnz, const int *rp, const int *ci, const T *val, const T *b, T *x, const cap_opts *opts)
{
    if (!rp || !b || !x || n < 0) return CAP_ERR_ARG;
    cap_opts o;
    cap_opts_default(&o);
    if (opts) o = *opts;
    o.host_inputs = 1;
    if (o.algo == CAP_ALGO_AUTO) o.algo = CAP_ALGO_WRTFST;
    cap_plan p = nullptr;
    CAP_TRY(plan_create_impl(&p, n, nnz, rp, ci, val, sizeof(T) == 8 ? CAP_F64 : CAP_F32, &o, nullptr));
    T *db = nullptr, *dx = nullptr;
    int rc = CAP_OK;
    do {
        if ((rc = dev_alloc(&db, (size_t)n)) || (rc = dev_alloc(&dx, (size_t)n))) break;
        if (hipMemcpy(db, b, sizeof(T) * (size_t)n, hipMemcpyHostToDevice) != hipSuccess) { rc = CAP_ERR_HIP; break; }
        if ((rc = cap_plan_solve(p, db, dx, 1, nullptr)) != CAP_OK) break;
        if (hipMemcpy(x, dx, sizeof(T) * (size_t)n, hipMemcpyDeviceToHost) != hipSuccess) { rc = CAP_ERR_HIP; break; }
        rc = cap_plan_status(p, nullptr);
    } while (0);
    (void)hipFree(db);
    (void)hipFree(dx);
    plan_free(p);
    return rc;
}

// ------------------------------------------------ benchmark-compatible
// Shared body of the CSR wrappers (spts_syncfree_cuda_csr_wrt.h:66-242).
template <typename T>
int bench_csr(int algo, const int *rp, const int *ci, const T *val, int m, int n, int nnzL, double *solve_time,
              double *gflops, double *bw, double *pre_time, double *wocc, double *eocc)
{
    if (m != n) {
        std::printf("This is not a square matrix, return.\n");
        return -1;
    }
    if (!solve_time || !gflops || !bw) return CAP_ERR_ARG;
    std::vector<T> x_ref((size_t)n), b((size_t)m), x((size_t)n);
    // get_x_b (read_mtx.h:260-278)
    if (sizeof(T) == 8)
        cap_get_x_b_d(m, n, rp, ci, (const double *)(const void *)val, (double *)(void *)x_ref.data(),
                      (double *)(void *)b.data());
    else
        cap_get_x_b_s(m, n, rp, ci, (const float *)(const void *)val, (float *)(void *)x_ref.data(),
                      (float *)(void *)b.data());
    double pre_ms = 0.0;
    cap_opts o;
    cap_opts_default(&o);
    o.algo = algo;
    o.sync = CAP_SYNC_VALUE;
    o.host_inputs = 1;
    if (algo == CAP_ALGO_MIX) {
        // pre_time: mean host time of the chunk table over the repeats
        // (CUDA/mix/spts_syncfree_cuda_csr_wrt.h:185-194)
        std::vector<int> wn((size_t)m + 1);
        int len = 0;
        double wo = 0, eo = 0;
        auto t0 = std::chrono::steady_clock::now();
        const int levels = m ? cap_matrix_layer(m, rp, ci, nullptr, nullptr, nullptr) : 1;
        o.border = mix_border_for(m, levels);
        for (int r = 0; r < CAP_BENCH_REPEAT; ++r)
            cap_matrix_warp4(m, nnzL, rp, o.border, kWave, &len, wn.data(), &wo, &eo);
        auto t1 = std::chrono::steady_clock::now();
        pre_ms = std::chrono::duration<double, std::milli>(t1 - t0).count() / CAP_BENCH_REPEAT;
    }
    cap_plan p = nullptr;
    CAP_TRY(plan_create_impl(&p, n, nnzL, rp, ci, val, sizeof(T) == 8 ? CAP_F64 : CAP_F32, &o, nullptr));
    T *db = nullptr, *dx = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = CAP_OK, passed = 0;
    double total_ms = 0.0;
    do {
        if ((rc = dev_alloc(&db, (size_t)m)) || (rc = dev_alloc(&dx, (size_t)n))) break;
        if (hipMemcpy(db, b.data(), sizeof(T) * (size_t)m, hipMemcpyHostToDevice) != hipSuccess ||
            hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
            rc = CAP_ERR_HIP;
            break;
        }
        // warm-up (the reference's driver calls the wrapper twice)
        if ((rc = plan_solve_with(p, p->algo, p->sync, db, dx, 1, nullptr)) != CAP_OK) break;
        for (int r = 0; r < CAP_BENCH_REPEAT && rc == CAP_OK; ++r) {
            // reset outside the timed region, as the reference does (:154-156)
            if ((rc = launch_prepare<T>(p, p->algo, p->sync, dx, n, nullptr)) != CAP_OK) break;
            (void)hipEventRecord(e0, nullptr);
            if ((rc = launch_kernel<T>(p, p->algo, p->sync, (const T *)p->val, db, dx, 1, nullptr)) != CAP_OK) break;
            (void)hipEventRecord(e1, nullptr);
            if (hipEventSynchronize(e1) != hipSuccess) { rc = CAP_ERR_HIP; break; }
            float ms = 0;
            (void)hipEventElapsedTime(&ms, e0, e1);
            total_ms += ms;
            if (hipMemcpy(x.data(), dx, sizeof(T) * (size_t)n, hipMemcpyDeviceToHost) != hipSuccess) {
                rc = CAP_ERR_HIP;
                break;
            }
            // validation of spts_syncfree_cuda_csr_wrt.h:190-201
            int errs = 0;
            for (int i = 0; i < n; ++i)
                if (!(std::fabs((double)x_ref[i] - (double)x[i]) <= 0.01 * std::fabs((double)x_ref[i]))) ++errs;
            if (!errs) ++passed;
        }
        if (rc == CAP_OK && cap_plan_status(p, nullptr) != CAP_OK) passed = 0;
    } while (0);
    int len = p->mix_len;
    if (wocc) *wocc = p->wocc;
    if (eocc) *eocc = p->eocc;
    if (pre_time) *pre_time = pre_ms;
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(db);
    (void)hipFree(dx);
    plan_free(p);
    if (rc != CAP_OK) return rc;
    const double ms = total_ms / CAP_BENCH_REPEAT;
    *solve_time = ms;
    *gflops = 2.0 * nnzL / (1e6 * ms);
    *bw = cap_datasize(m, n, nnzL, (int)sizeof(T), algo == CAP_ALGO_MIX ? len : 0) / (1e6 * ms);
    if (passed != CAP_BENCH_REPEAT) {
        std::printf("hip syncfree SpTS on L failed!\n");
        *solve_time = -1;
        *gflops = 0;
        *bw = 0;
    }
    return 0;
}

// sptrsv_syncfree_cuda (CUDA/SyncFree_csc/spts_syncfree_cuda2.h:89-292)
template <typename T>
int bench_csc(const int *cp, const int *ri, const T *cv, int m, int n, int nnz, T *x, const T *b, const T *x_ref,
              double *pre_time, double *solve_time, double *gflops, double *bw)
{
    if (m != n) {
        std::printf("This is not a square matrix, return.\n");
        return -1;
    }
    if (!cp || !ri || !cv || !x || !b || !x_ref || !pre_time || !solve_time || !gflops || !bw) return CAP_ERR_ARG;
    int dev = 0;
    CAP_TRY(check_device(&dev));
    cap_plan p = new cap_plan_s();
    p->device = dev;
    p->n = n;
    p->nnz = nnz;
    p->vt = sizeof(T) == 8 ? CAP_F64 : CAP_F32;
    p->vbytes = sizeof(T);
    p->algo = CAP_ALGO_CSC;
    int rc = CAP_OK;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    T *db = nullptr, *dx = nullptr;
    double analyse_ms = 0.0, total_ms = 0.0;
    do {
        if ((rc = init_ctrl(p)) || (rc = dev_alloc(&p->cp, (size_t)n + 1)) || (rc = dev_alloc(&p->cri, (size_t)nnz)) ||
            (rc = dev_alloc((T **)&p->cv, (size_t)nnz)) || (rc = dev_alloc(&p->deg0, (size_t)n)) ||
            (rc = dev_alloc(&p->deg, (size_t)n)) || (rc = dev_alloc((T **)&p->left_sum, (size_t)n)) ||
            (rc = dev_alloc(&db, (size_t)n)) || (rc = dev_alloc(&dx, (size_t)n)))
            break;
        if (hipMemcpy(p->cp, cp, sizeof(int) * ((size_t)n + 1), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(p->cri, ri, sizeof(int) * (size_t)nnz, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(p->cv, cv, sizeof(T) * (size_t)nnz, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(db, b, sizeof(T) * (size_t)n, hipMemcpyHostToDevice) != hipSuccess ||
            hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
            rc = CAP_ERR_HIP;
            break;
        }
        // analysis (K4), timed over the repeats (:151-166)
        for (int r = 0; r < CAP_BENCH_REPEAT; ++r) {
            k_prepare<unsigned><<<blocks_for(n), kBlock, 0, nullptr>>>((unsigned *)p->deg0, n, 0u, p->ticket, 0);
            (void)hipEventRecord(e0, nullptr);
            k_indegree<<<blocks_for(nnz), kBlock, 0, nullptr>>>(p->cri, nnz, p->deg0);
            (void)hipEventRecord(e1, nullptr);
            (void)hipEventSynchronize(e1);
            float ms = 0;
            (void)hipEventElapsedTime(&ms, e0, e1);
            analyse_ms += ms;
        }
        if (hipGetLastError() != hipSuccess) { rc = CAP_ERR_HIP; break; }
        for (int r = 0; r <= CAP_BENCH_REPEAT && rc == CAP_OK; ++r) {  // r == 0: warm-up
            if ((rc = launch_csc_reset<T>(p, nullptr)) != CAP_OK) break;
            (void)hipEventRecord(e0, nullptr);
            if ((rc = launch_kernel<T>(p, CAP_ALGO_CSC, CAP_SYNC_VALUE, nullptr, db, dx, 1, nullptr)) != CAP_OK) break;
            (void)hipEventRecord(e1, nullptr);
            if (hipEventSynchronize(e1) != hipSuccess) { rc = CAP_ERR_HIP; break; }
            float ms = 0;
            (void)hipEventElapsedTime(&ms, e0, e1);
            if (r > 0) total_ms += ms;
        }
        if (rc == CAP_OK && hipMemcpy(x, dx, sizeof(T) * (size_t)n, hipMemcpyDeviceToHost) != hipSuccess)
            rc = CAP_ERR_HIP;
        if (rc == CAP_OK && cap_plan_status(p, nullptr) != CAP_OK) std::printf("hip syncfree SpTRSV watchdog fired\n");
    } while (0);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(db);
    (void)hipFree(dx);
    plan_free(p);
    if (rc != CAP_OK) return rc;
    *pre_time = analyse_ms / CAP_BENCH_REPEAT;
    const double ms = total_ms / CAP_BENCH_REPEAT;
    *solve_time = ms;
    *gflops = 2.0 * nnz / (1e6 * ms);
    *bw = cap_datasize(m, n, nnz, (int)sizeof(T), 0) / (1e6 * ms);
    // relative L1 validation (:245-264)
    double ref = 0, res = 0;
    for (int i = 0; i < n; ++i) {
        ref += std::fabs((double)x_ref[i]);
        res += std::fabs((double)x[i] - (double)x_ref[i]);
    }
    res = ref == 0 ? res : res / ref;
    if (!(res < 1e-4)) {
        std::printf("hip syncfree SpTRSV executor _NOT_ passed! |x-xref|/|xref| = %8.2e\n", res);
        *solve_time = -1;
    }
    return 0;
}

}  // namespace

extern "C" {

int sptrsv_csr_solve_d(int n, int nnz, const int *rp, const int *ci, const double *v, const double *b, double *x,
                       const cap_opts *o)
{
    return oneshot<double>(n, nnz, rp, ci, v, b, x, o);
}
int sptrsv_csr_solve_s(int n, int nnz, const int *rp, const int *ci, const float *v, const float *b, float *x,
                       const cap_opts *o)
{
    return oneshot<float>(n, nnz, rp, ci, v, b, x, o);
}
}  // extern "C"

// ------------------------------------------------- allocation-free solve
// The one-shot solve above allocates: a plan (control block with the
// tickets and the watchdog word, a staged readiness array) and device copies
// of the inputs.  sptrsv_csr_solve_noalloc_d runs the same write-first
// kernel on the caller's device arrays with nothing allocated: x itself is
// the readiness array (sentinel-filled by the reset launch), and the tickets
// and the watchdog word live in `scratch`, one static array per device that
// every call on that device shares (calls that overlap on one device race).
// Its layout: kTickets ticket words, then the watchdog word.
constexpr size_t kScratchBytes = 256;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
static_assert((kTickets + 1) * sizeof(unsigned) <= kScratchBytes, "tickets and the watchdog word fit scratch");

namespace {

struct ScratchDev {
    unsigned char *ptr = nullptr;  // device address of this device's copy of scratch
    int ncu = 0;
};
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
ScratchDev g_scratch[kMaxDevices];

// Set-up on a device's first call, with that device current: checks that it
// is a gfx950, takes the device address of its copy of `scratch` (the host
// name is only a stand-in for it) and its compute-unit count.
int scratch_of(int dev, ScratchDev *out)
{
    if (dev < 0 || dev >= kMaxDevices) return CAP_ERR_NO_DEVICE;
    std::lock_guard<std::mutex> g(g_scratch_mu);
    ScratchDev &sd = g_scratch[dev];
    if (!sd.ptr) {
        int cur = -1;
        CAP_TRY(check_device(&cur));
        if (cur != dev) return CAP_ERR_NO_DEVICE;
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            std::fprintf(stderr, "capellini: hipGetSymbolAddress(scratch) failed: %s\n", hipGetErrorString(e));
            return CAP_ERR_HIP;
        }
        int ncu = 0;
        CAP_HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
        sd.ncu = ncu > 0 ? ncu : 256;
        sd.ptr = static_cast<unsigned char *>(p);
    }
    *out = sd;
    return CAP_OK;
}

}  // namespace

extern "C" {

int sptrsv_csr_solve_noalloc_d(int n, int nnz, const int *row_ptr, const int *col_idx, const double *val,
                               const double *b, double *x, void *stream)
{
    typedef unsigned long long U;
    if (n < 0 || nnz < n || !row_ptr || (n > 0 && (!col_idx || !val || !b || !x))) return CAP_ERR_ARG;
    int dev = 0;
    CAP_HIP_TRY(hipGetDevice(&dev));
    ScratchDev sd;
    CAP_TRY(scratch_of(dev, &sd));
    if (n == 0) return CAP_OK;
    hipStream_t st = S(stream);
    unsigned *ticket = reinterpret_cast<unsigned *>(sd.ptr);
    int *err = reinterpret_cast<int *>(sd.ptr + kTickets * sizeof(unsigned));
    // one reset launch: x <- sentinel, tickets and the watchdog word <- 0
    const unsigned nbp = std::max(1u, std::min(blocks_for(n), 2048u));
    k_prepare<U><<<nbp, kBlock, 0, st>>>(reinterpret_cast<U *>(x), n, VBits<double>::kSentinel, ticket, kTickets + 1);
    const SyncCtx sc{nullptr, 0, 0, err, nullptr, 0, kWaitMsDefault * 100000};
    const unsigned nb = (unsigned)std::max(1LL, std::min<long long>(sd.ncu, ((long long)n + kBlock - 1) / kBlock));
    k_wrtfst<double, 1, 0, kBlock><<<nb, kBlock, 0, st>>>(row_ptr, col_idx, val, b, x, sc, n, 1, 0, ticket, 0,
                                                            nullptr, 0);
    CAP_HIP_TRY(hipGetLastError());
    return CAP_OK;
}

int spts_syncfree_hip_csr_wrt_d(const int *rp, const int *ci, const double *v, int m, int n, int nnzL, double *t,
                                double *gf, double *bw)
{
    return bench_csr<double>(CAP_ALGO_WRTFST, rp, ci, v, m, n, nnzL, t, gf, bw, nullptr, nullptr, nullptr);
}
int spts_syncfree_hip_csr_wrt_s(const int *rp, const int *ci, const float *v, int m, int n, int nnzL, double *t,
                                double *gf, double *bw)
{
    return bench_csr<float>(CAP_ALGO_WRTFST, rp, ci, v, m, n, nnzL, t, gf, bw, nullptr, nullptr, nullptr);
}
int spts_syncfree_hip_csr_algo_d(const int *rp, const int *ci, const double *v, int m, int n, int nnzL, int algo,
                                 double *t, double *gf, double *bw)
{
    if (algo == CAP_ALGO_MIX || algo < CAP_ALGO_AUTO || algo > CAP_ALGO_LEVEL) return CAP_ERR_ARG;
    return bench_csr<double>(algo, rp, ci, v, m, n, nnzL, t, gf, bw, nullptr, nullptr, nullptr);
}
int spts_syncfree_hip_csr_algo_s(const int *rp, const int *ci, const float *v, int m, int n, int nnzL, int algo,
                                 double *t, double *gf, double *bw)
{
    if (algo == CAP_ALGO_MIX || algo < CAP_ALGO_AUTO || algo > CAP_ALGO_LEVEL) return CAP_ERR_ARG;
    return bench_csr<float>(algo, rp, ci, v, m, n, nnzL, t, gf, bw, nullptr, nullptr, nullptr);
}
int spts_syncfree_hip_csr_d(const int *rp, const int *ci, const double *v, int m, int n, int nnzL, double *t,
                            double *gf, double *bw)
{
    return bench_csr<double>(CAP_ALGO_TWOPART, rp, ci, v, m, n, nnzL, t, gf, bw, nullptr, nullptr, nullptr);
}
int spts_syncfree_hip_csr_s(const int *rp, const int *ci, const float *v, int m, int n, int nnzL, double *t,
                            double *gf, double *bw)
{
    return bench_csr<float>(CAP_ALGO_TWOPART, rp, ci, v, m, n, nnzL, t, gf, bw, nullptr, nullptr, nullptr);
}
int spts_syncfree_hip_mix_d(const int *rp, const int *ci, const double *v, int m, int n, int nnzL, double *t,
                            double *gf, double *bw, double *pre, double *wo, double *eo)
{
    return bench_csr<double>(CAP_ALGO_MIX, rp, ci, v, m, n, nnzL, t, gf, bw, pre, wo, eo);
}
int spts_syncfree_hip_mix_s(const int *rp, const int *ci, const float *v, int m, int n, int nnzL, double *t,
                            double *gf, double *bw, double *pre, double *wo, double *eo)
{
    return bench_csr<float>(CAP_ALGO_MIX, rp, ci, v, m, n, nnzL, t, gf, bw, pre, wo, eo);
}
int sptrsv_syncfree_hip_csc_d(const int *cp, const int *ri, const double *cv, int m, int n, int nnz, double *x,
                              const double *b, const double *xr, double *pre, double *t, double *gf, double *bw)
{
    return bench_csc<double>(cp, ri, cv, m, n, nnz, x, b, xr, pre, t, gf, bw);
}
int sptrsv_syncfree_hip_csc_s(const int *cp, const int *ri, const float *cv, int m, int n, int nnz, float *x,
                              const float *b, const float *xr, double *pre, double *t, double *gf, double *bw)
{
    return bench_csc<float>(cp, ri, cv, m, n, nnz, x, b, xr, pre, t, gf, bw);
}

}  // extern "C"
