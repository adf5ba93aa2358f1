// Step solves: one workgroup per matrix walks a schedule of steps, a step's
// rows in parallel, one per thread, a workgroup barrier between steps, values
// in an LDS ring (kernel and tables in steps.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

namespace cap {

// One matrix of a launch: its pieces from tab (16-byte units), its row table
// from rows, `steps` steps of `block` slots,
// a ring of `ring` slots; its rows_of rows start at row0 of b and x.
struct StepJob {
    unsigned long long tab;
    unsigned rows;
    int steps, ring, block, row0, rows_of;
};

struct StepTables {
    int vt = 0, E = 4, n_jobs = 0, block = 64, ring = 0, max_rhs = 1;
    int tallest = 0;  // rows of the largest matrix
    int cus = 256;    // compute units of the device
    size_t lds = 0;   // bytes of LDS a workgroup may have
    bool long_rows = false;
    long long slots = 0;
    std::vector<StepJob> jobs;
    StepJob *d_jobs = nullptr;
    uint4 *tab = nullptr;
    unsigned *rows = nullptr;
    // rows longer than E: where a slot's rest starts in ov_c / ov_v (a count,
    // then that many ring slots; values at the same index + 1), -1 for none
    int *ov_at = nullptr, *ov_c = nullptr;
    void *ov_v = nullptr;
};

// Schedules the rows of each matrix [first, last) of a block-diagonal CSR (host copies rp, ci with global columns; the same arrays
// and the values on the device) and lays out the tables.  want_rhs: right-hand
// sides a thread should solve (4, 2 or 1); fewer where the ring does not
// fit lds_bytes (max_rhs says how many).  want_block: rows per step (64, 128,
// 192 or 256; 0: each matrix's best, by scheduling it for all of them).  CAP_ERR_UNSUPPORTED when a matrix's
// dependencies reach further back than any ring, or its steps would be mostly
// padding (more than pad_max slots per row), or the tables more than
// max_bytes.
int steps_build(StepTables **out, const std::vector<int> &rp, const std::vector<int> &ci,
                const std::vector<int2> &mats, int vt, int want_rhs, int want_block, int lds_bytes, int pad_max,
                double max_bytes, const int *d_rp, const int *d_ci, const void *d_val, hipStream_t st);
// Copies the values into the tables again (they changed in place).
int steps_refresh(const StepTables *t, const int *d_rp, const int *d_ci, const void *d_val, hipStream_t st);
// Solves k right-hand sides (interleaved, row * k + q), 1, 2 or 4 of them per
// workgroup.
int steps_launch(const StepTables *t, const void *b, void *x, int k, bool unfused, hipStream_t st);
bool steps_take(const StepTables *t, int k);
void steps_free(StepTables *t);

}  // namespace cap
