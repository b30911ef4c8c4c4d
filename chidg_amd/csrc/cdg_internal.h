// Internal types of the gfx950 linear-solve library (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <map>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/chidg_hip.h"

#define CDG_HIP_TRY(expr)                                                              \
    do {                                                                               \
        hipError_t e_ = (expr);                                                        \
        if (e_ != hipSuccess) return cdg_fail(ctx, CDG_ERR_HIP, "%s: %s (%s:%d)", #expr, \
                                              hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)

int cdg_fail(const cdg_ctx *ctx, int code, const char *fmt, ...);

// 16-bit brain float storage
typedef uint16_t cdg_bf16;

// Device memory owned by a context (freed in the owner's destructor path).
struct DevMem {
    void *p = nullptr;
    size_t bytes = 0;
};

struct cdg_ctx {
    int device = 0;
    int num_cus = 0;
    hipStream_t stream = nullptr;
    mutable std::string err;
    int64_t mem_used = 0;              // bytes held by live objects
    int64_t mem_cached = 0;            // bytes freed by objects, kept for reuse
    std::unordered_map<void *, size_t> alloc_size;
    std::multimap<size_t, void *> cache;
    // reduction scratch (device) and pinned host mirror
    double *d_part = nullptr;     // partial sums
    size_t part_cap = 0;          // doubles
    double *d_small = nullptr;    // small results (dots, norms)
    double *h_small = nullptr;    // pinned host copy
    size_t small_cap = 0;
    // staging for host pointers passed to the ABI
    double *d_stage[3] = {nullptr, nullptr, nullptr};
    size_t stage_cap[3] = {0, 0, 0};
    // completion event of ctx_wait (the solver's per-step waits poll it)
    hipEvent_t done_ev = nullptr;
    hipEvent_t order_ev = nullptr;     // cdg_ctx_wait_stream / cdg_ctx_signal_stream
    bool spin = true;
    // one FGMRES step on the device (k_arnoldi.hip): the launches' number, results in pinned memory,
    // and where the step's kernels put their start times / find whether any lane still runs
    uint32_t arn_seq = 0;
    struct ArnRes *h_arn = nullptr;
    int arn_cap = 0;
    uint64_t *hook_stamp = nullptr;
    const int *hook_nact = nullptr;
    // pinned words, one per preconditioner, that a sweep which gave up waiting raises: the pages, and
    // those of their words that no preconditioner holds
    std::vector<uint32_t *> word_pages, word_free;
};

// Waits until the context's stream has finished its work: polls a completion
// event (a few microseconds of latency instead of a blocking wait's tens), and
// falls back to a blocking wait after 5 ms.  CDG_SPIN=0 always blocks.
int ctx_wait(cdg_ctx *ctx);

// Block-row streaming launch shape for one block size / element width.
struct StreamShape {
    int T = 0;     // threads per workgroup (V*T is a multiple of n)
    int dc = 0;    // column advance per iteration = V*T/n
};
// Launch shape of the fixed-row walk; T <= tmax is a multiple of n/gcd(n,V)
// chosen for lane utilization, preferring sizes near `target`.
StreamShape stream_shape(int n, int V, int target, int tmax = 1024);

// Task shape of the ILU(0) sweep (k_sweep.hip) for one block size and storage
// type: C column chunks of cw columns, gq row groups by dc columns per walk step
// (T threads, TP padded to whole wavefronts), R steps, 2^ls lanes per row sum.
struct SweepShape {
    int C = 1, cw = 1, gq = 1, dc = 1, T = 1, TP = 64, R = 1, ls = 0;
};
// A sweep over rows [lo, hi) for up to KT right-hand sides: its units in ticket
// order, exchange words and ticket counter (device memory of the preconditioner).
struct SweepPlan {
    SweepShape sh;
    int KT = 1, lo = 0, hi = 0, G = 1, nunits = 0, grid = 0, spin = 0, dep = 1;
    bool fold = false;            // over W = Dinv U
    size_t lds = 0;
    const void *fn = nullptr;
    int32_t *recs = nullptr;
    void *P = nullptr;
    unsigned long long *ctl = nullptr;
};

struct cdg_mat {
    int32_t nrows = 0, n = 0, nnzb = 0;
    int64_t ld = 0;                    // elements per block slot (padded, multiple of 64)
    double *blocks = nullptr;          // nnzb * ld, device
    int32_t *d_row_ptr = nullptr, *d_col = nullptr;
    std::vector<int32_t> row_ptr, col, kind;
    std::vector<int32_t> part;         // rank of each row (empty: one rank), see cdg_mat_set_partition
    int32_t max_row_blocks = 0;
    uint64_t stamp = 0;
    // kind-0 structure (type_domain_matrix.f90:295-302, 592-627)
    std::vector<int32_t> diag, lo_ptr, lo_blk, lo_col, lo_tr, up_ptr, up_blk, up_col, up_tr;
    int32_t struct_err = CDG_OK;       // CDG_ERR_NO_TRANSPOSE if the kind-0 pattern is not symmetric
    std::vector<int32_t> flevel, blevel;
    int32_t nflev = 0, nblev = 0;
    StreamShape shape64;
    int32_t mv_unroll = 8;             // 16-byte loads in flight per thread (matvec)
};

struct cdg_prec {
    int32_t type = CDG_PREC_IDENTITY;
    int32_t jacobi = 0;                // created as CDG_PREC_JACOBI (ILU(0) with no off-diagonal blocks)
    int32_t precision = CDG_FP64;
    int32_t nrows = 0, n = 0, nlo = 0, nup = 0;
    int64_t ld = 0;                    // elements per factor slot
    // factor storage (element type by precision)
    void *L = nullptr;                 // nlo slots
    void *U = nullptr;                 // nup slots (FP32/BF16 copies of A's upper blocks)
    // nup slots, FP64/FP32: W_u = A_{up_blk[u]} Dinv_{up_col[u]}, the upper
    // blocks with the Dinv of their column folded in (the level schedule's
    // backward sweep is then one stage per level).  BF16: W_u = Dinv_{row(u)} A_{up_blk[u]}, of the
    // sweep's folded form (fold_ok)
    void *W = nullptr;
    int32_t w_ready = 0;               // W holds the current factor's products
    int32_t *d_up_all = nullptr;       // 0..nup-1 (the W jobs)
    int32_t *d_up_row = nullptr;       // row of each upper entry (fold_ok)
    void *Dinv = nullptr;              // nrows slots
    float *L32 = nullptr, *D32 = nullptr;   // FP32 work for the BF16 variant
    void *inv_w = nullptr;             // working slots of the global-memory block inverse
    int32_t *d_redo = nullptr;         // per row: block inverse must be redone with partial pivoting
    // device index arrays
    int32_t *d_lo_ptr = nullptr, *d_lo_blk = nullptr, *d_lo_col = nullptr, *d_lo_tr = nullptr;
    int32_t *d_lo_tru = nullptr;       // U slot of lo_tr[q] (FP32/BF16: the upper blocks' copies)
    int32_t *d_up_ptr = nullptr, *d_up_idx = nullptr, *d_up_col = nullptr, *d_up_blk = nullptr;
    int32_t *d_diag = nullptr;
    int32_t *d_err = nullptr;          // first singular row (factor)
    double *d_part = nullptr;          // partial sums of the column-slice schedules: 3 arrays of part_len doubles (null: none chosen)
    int64_t part_len = 0;              // nrows * slices * n
    int64_t part_cap = 0;              // doubles allocated at d_part
    // forward levels: rows grouped by level (factor and forward sweep); lower
    // blocks of those rows grouped the same way (factor phase 1)
    std::vector<int32_t> lev_lo_ptr, lev_row_ptr;
    int32_t *d_lev_lo = nullptr, *d_lev_rows = nullptr;
    int32_t nlev = 0;
    // backward levels (backward sweep)
    std::vector<int32_t> blev_row_ptr;
    int32_t *d_blev_rows = nullptr;
    int32_t nblev = 0;
    std::vector<int32_t> h_lev_rows, h_blev_rows;   // host copies of the level orders
    std::vector<int32_t> h_lo_ptr, h_lo_col, h_up_ptr, h_up_col, h_up_idx;   // host copies of the kind-0 lists (h_up_idx: U slots)
    int32_t maxdep = 1;               // max lower/upper blocks of a row
    // apply launch shape: each block's columns are cut into `slices` ranges of
    // `slice_w` columns; shape[precision] is the fixed-row walk for that element
    int32_t slices = 1, slice_w = 1, unroll = 4;
    StreamShape shape[3];
    // apply schedule: CDG_APPLY_DATAFLOW (one persistent launch, k_dfapply.hip),
    // CDG_APPLY_FOLDED (levels, backward over W = U Dinv); every other one is the sweep
    // (k_sweep.hip), or one launch per level and stage where rows have too many blocks for it
    int32_t apply_mode = 0;
    int32_t df_T = 0, df_dc = 0, df_rounds = 0, df_w = 0, df_S = 0, df_grid = 0, df_ntasks = 0;
    size_t df_lds = 0;
    int32_t *d_tasks = nullptr;        // task codes in ticket order
    int32_t *d_cnt = nullptr;          // [3][nrows] finished slices (cumulative)
    unsigned long long *d_ticket = nullptr;
    int32_t *d_dferr = nullptr;        // raised by a sweep that gave up waiting
    int32_t df_epoch = 0;              // calls since the counters were zeroed
    int32_t df_spin = 1 << 21;         // polls before a dependency wait gives up
    // the sweep (k_sweep.hip): plans made so far (row range, right-hand sides)
    std::vector<SweepPlan *> sweeps;
    SweepShape sweep_sh[2];            // plain, and over W
    int32_t sweep_shaped[2] = {0, 0};
    int32_t sweep_ok = 1;              // 0: the pattern does not fit the sweep (level launches instead)
    // BF16, where a row's upper blocks and its Dinv fit a task: the sweep over W = Dinv U.  CDG_APPLY_AUTO
    // takes it once the factor has served fold_after applies (0: never), from the first apply when the
    // previous factor served more, or when another call has formed W for this factor.
    int32_t fold_ok = 0, fold_after = 12, napply = 0, prev_napply = 0;
    int32_t w_asked = 0;               // W of this factor was asked for by name or for several vectors
    int32_t w_keep = 0;                // a captured launch reads W: every update forms it anew
    uint32_t *h_err = nullptr;         // pinned: raised by one of its sweeps that gave up waiting
    int32_t noalloc_ok = 0;            // CDG_SCHEDULE_ROWSLICE or _STREAM was set (cdg_prec_apply_noalloc)
    uint64_t stamp = 0;
    int32_t factored = 0;
    std::vector<DevMem> owned;
};

// ---- the vector part of FGMRES steps (k_arnoldi.hip) --------------------------
enum { ARN_CGS = 0, ARN_MGS = 1, ARN_START = 2, ARN_NORM = 3 };
enum { ARN_ACTIVE, ARN_DONE, ARN_NVECS, ARN_NITER, ARN_CONV, ARN_NREORTH, ARN_SECOND, ARN_RUN, ARN_NREALL, ARN_NST = 32 };   // int state of a lane (a line); NREALL: second passes of all solves on this workspace
enum { ARN_R0INIT, ARN_RES, ARN_TP, ARN_TM, ARN_TO, ARN_TN, ARN_NSC = 16 };                 // doubles of a lane
// What launches report per lane, in pinned memory: after each step one word, the
// launch's number, the lane's steps in this cycle and ARN_W_* bits; the rest with the word of an
// ARN_NORM launch.
enum { ARN_W_ACTIVE = 1, ARN_W_DONE = 2, ARN_W_ERR = 4, ARN_W_BITS = 3 };
struct ArnRes {
    uint64_t word;
    double res, t[4];             // ||b - A x||; ticks: preconditioner, product, vectors, norms
    int niter, nreorth;
};
struct ArnArgs {
    int mode, nl, G, jj, m, nx, first;
    int64_t len, slice, hlen, rlen;
    const double *V, *b, *ax;     // basis (step stride nl len, lane stride len); START/NORM: r = b - ax
    double *w;                    // the vector orthogonalized: V_jj (START: V_0)
    int *st;
    double *sc, *y, *cs, *sn, *p, *R;
    double *part, *sums;          // [lane][value][slice], [lane][value]
    uint64_t *stamp;
    int *nact;                    // lanes still running
    const int *inner_st;          // NORM: null, or the state of the nested solver's lane
    ArnRes *hres;
    uint32_t seq;
    double tol, rtol;
    int nmax;
};
struct Arnoldi {
    ArnArgs a{};
    int nl = 0, m = 0, NI = 1, G = 1;
    bool mgs = false;
    int64_t len = 0;
    void *base = nullptr;
    size_t bytes = 0;
};
int arn_alloc(cdg_ctx *ctx, Arnoldi &A, int nl, int m, int64_t len, bool mgs);
void arn_free(cdg_ctx *ctx, Arnoldi &A);
int arn_launch(cdg_ctx *ctx, Arnoldi &A, int mode, int jj);
int arn_cycle_end(cdg_ctx *ctx, Arnoldi &A, const double *Z, double *x, double *x0, bool first);
int arn_stamp(cdg_ctx *ctx, Arnoldi &A, int i);

// ---- kernel launchers (defined in the .hip files) ----------------------------
int launch_mv(cdg_ctx *ctx, const cdg_mat *A, const double *x, double *y);
bool mv_flat(const cdg_ctx *ctx, const cdg_mat *A, const StreamShape &s);
int launch_ilu_apply(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const double *v, double *z);
int launch_ilu_apply_df(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const double *v, double *z);
int df_configure(cdg_ctx *ctx, cdg_prec *M);
int df_reset(cdg_ctx *ctx, cdg_prec *M);
enum { CDG_APPLY_LEVELS = 0, CDG_APPLY_DATAFLOW = 1, CDG_APPLY_FOLDED = 2, CDG_APPLY_AUTO = 3, CDG_APPLY_STREAM = 4,
       CDG_APPLY_ROWSLICE = 5 };
// the sweep (k_sweep.hip)
bool sweep_shape(int n, int precision, int maxdep, int width, int mean, int cus, SweepShape *out);
int sweep_plan(cdg_ctx *ctx, cdg_prec *M, int K, int lo, int hi, bool fold, SweepPlan **out);
int sweep_fold(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A);
int sweep_check(cdg_ctx *ctx, cdg_prec *M);   // an error if a sweep of M has given up since the last look
void sweep_free(cdg_prec *M);
int launch_ilu_sweep(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const double *v, double *z, int64_t stride, int k,
                     bool fold, const int32_t *row_k = nullptr, int lo = 0, int hi = -1);
int launch_diag(cdg_ctx *ctx, const cdg_prec *M, const double *v, double *z, int64_t stride, int k, const int32_t *row_k,
                int lo, int hi);
int launch_fold_left(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A);
int launch_mv_multi(cdg_ctx *ctx, const cdg_mat *A, const double *X, double *Y, int64_t stride, int k,
                    const int32_t *row_k = nullptr, int row_lo = 0, int row_hi = -1);
bool is_device_ptr(const void *p);
// W_u = A_{up_blk[u]} Dinv_{up_col[u]} for all upper blocks (after a factor)
int launch_fold_all(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A);
// Uniform hex-box pattern in ChiDG row order (cdg_serve.hip); periodic: bit d
// for direction d; face (optional) 1..6 face id per entry, 7 the diagonal
void cdg_hex_box(int nx, int ny, int nz, int periodic, std::vector<int32_t> &row_ptr, std::vector<int32_t> &col,
                 std::vector<int32_t> &kind, std::vector<int32_t> *face = nullptr);
int launch_ilu_factor(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, int32_t *bad_row);
int launch_fill_synthetic(cdg_ctx *ctx, cdg_mat *A, uint64_t seed, double s_diag, double s_off);
int launch_vec_synthetic(cdg_ctx *ctx, int64_t len, uint64_t seed, double scale, double *v);
int launch_widen(cdg_ctx *ctx, const void *src, int precision, double *dst, int64_t count);

// Krylov vector kernels (k_krylov.hip); all on ctx->stream, device pointers
int kv_multidot(cdg_ctx *ctx, int64_t len, const double *w, const double *V, int64_t vstride, int j,
                double *d_out /* j doubles */);
int kv_sumsq(cdg_ctx *ctx, int64_t len, const double *w, double *d_out);
int kv_sub(cdg_ctx *ctx, int64_t len, const double *b, const double *Ax, double *r);   // r = b - Ax
int kv_add(cdg_ctx *ctx, int64_t len, double *z, const double *dz);                   // z += dz
int kv_zero(cdg_ctx *ctx, int64_t len, double *x);
int kv_axpby(cdg_ctx *ctx, int64_t len, double a, const double *x, double b, double *y);   // y = a x + b y
int launch_euler_residual(cdg_ctx *ctx, int nx, int ny, int nz, int order, const double *q, double *R);
int kv_copy(cdg_ctx *ctx, int64_t len, const double *src, double *dst);

int ctx_ensure_small(cdg_ctx *ctx, size_t n);
int ctx_norm2(cdg_ctx *ctx, int64_t len, const double *v, double *out);   // ||v|| (synchronizes)
int64_t slot_elems(int n);   // elements per block slot: n*n rounded up to 64
int ctx_ensure_part(cdg_ctx *ctx, size_t n);
int dev_alloc(cdg_ctx *ctx, void **p, size_t bytes);
void dev_free(cdg_ctx *ctx, void *p, size_t bytes);
