// Allocation-free ILU(0) apply (no counterpart in the reference): for callers
// that cannot allocate device memory -- code under HIP graph capture, tight
// serving loops, harnesses that forbid hipMalloc.
//
// cdg_prec_apply_noalloc is the sweep of k_sweep.hip, the kernel and the bits of
// CDG_SCHEDULE_ROWSLICE, on the preconditioner's own plan: its exchange words were
// allocated with the preconditioner and which set of them a call uses follows from a
// device counter, so a captured call replays.  The entry keeps its conditions:
// the row-slice or stream schedule has been chosen, and the forward vector
// fits CDG_NOALLOC_SCRATCH_BYTES.
#include "cdg_internal.h"

extern "C" int cdg_prec_apply_noalloc(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const double *v, double *z) {
    if (!ctx || !M || !A || !v || !z) return CDG_ERR_ARG;
    if (!is_device_ptr(v) || !is_device_ptr(z))
        return cdg_fail(ctx, CDG_ERR_ARG, "cdg_prec_apply_noalloc needs device pointers");
    if (M->type != CDG_PREC_ILU0) return cdg_fail(ctx, CDG_ERR_UNSUPPORTED, "cdg_prec_apply_noalloc: ILU(0) only");
    if (A->nrows != M->nrows || A->n != M->n) return cdg_fail(ctx, CDG_ERR_ARG, "matrix does not match preconditioner");
    const size_t need = (size_t)M->nrows * M->n * (M->precision == CDG_FP64 ? 8 : 4);
    if (need > (size_t)CDG_NOALLOC_SCRATCH_BYTES)
        return cdg_fail(ctx, CDG_ERR_ARG,
                        "cdg_prec_apply_noalloc: the forward vector needs %zu bytes, the scratch array holds %d",
                        need, CDG_NOALLOC_SCRATCH_BYTES);
    if (!M->factored) return cdg_fail(ctx, CDG_ERR_STATE, "ILU0 apply before update");
    if (!M->noalloc_ok)
        return cdg_fail(ctx, CDG_ERR_STATE, "cdg_prec_apply_noalloc: set CDG_SCHEDULE_ROWSLICE or CDG_SCHEDULE_STREAM first");
    if (M->fold_ok) {   // W is there; the first call after an update forms its values
        M->w_asked = 1;
        int e = sweep_fold(ctx, M, A);
        if (e) return e;
    }
    return launch_ilu_sweep(ctx, M, A, v, z, (int64_t)M->nrows * M->n, 1, M->fold_ok != 0);
}
