// C ABI of the gfx950 linear-solve library: contexts, block-sparse matrices,
// ILU(0)/identity preconditioners and restarted FGMRES.
#include "cdg_internal.h"

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <mutex>

// ---------------------------------------------------------------------------
// errors and memory
// ---------------------------------------------------------------------------
int cdg_fail(const cdg_ctx *ctx, int code, const char *fmt, ...) {
    if (ctx) {
        char buf[512];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(buf, sizeof(buf), fmt, ap);
        va_end(ap);
        ctx->err = buf;
    }
    return code;
}

// Device memory of a context.  Freed blocks stay cached in the context and
// are handed out again to later requests of up to their size (at most twice
// the request): every use of a context's memory is ordered on its one
// stream, and hipFree would synchronize the whole device, stalling the other
// contexts' work.  The cache is released when the context is destroyed, or
// when an allocation fails.
static void ctx_flush_cache(cdg_ctx *ctx) {
    if (ctx->cache.empty()) return;
    (void)hipStreamSynchronize(ctx->stream);
    for (auto &kv : ctx->cache) (void)hipFree(kv.second);
    ctx->cache.clear();
    ctx->mem_cached = 0;
}

int dev_alloc(cdg_ctx *ctx, void **p, size_t bytes) {
    *p = nullptr;
    if (bytes == 0) return CDG_OK;
    bytes = (bytes + 255) / 256 * 256;
    auto it = ctx->cache.lower_bound(bytes);
    if (it != ctx->cache.end() && it->first <= 2 * bytes) {
        *p = it->second;
        ctx->alloc_size[*p] = it->first;
        ctx->mem_cached -= (int64_t)it->first;
        ctx->mem_used += (int64_t)it->first;
        ctx->cache.erase(it);
        return CDG_OK;
    }
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        ctx_flush_cache(ctx);
        e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        return cdg_fail(ctx, CDG_ERR_OOM, "hipMalloc(%zu bytes): %s", bytes, hipGetErrorString(e));
    }
    ctx->alloc_size[*p] = bytes;
    ctx->mem_used += (int64_t)bytes;
    return CDG_OK;
}

void dev_free(cdg_ctx *ctx, void *p, size_t) {
    if (!p) return;
    auto it = ctx->alloc_size.find(p);
    if (it == ctx->alloc_size.end()) return;
    const size_t bytes = it->second;
    ctx->alloc_size.erase(it);
    ctx->mem_used -= (int64_t)bytes;
    ctx->mem_cached += (int64_t)bytes;
    ctx->cache.emplace(bytes, p);
}

int ctx_norm2(cdg_ctx *ctx, int64_t len, const double *v, double *out) {
    int e = kv_sumsq(ctx, len, v, ctx->d_small);
    if (!e) {
        CDG_HIP_TRY(hipMemcpyAsync(ctx->h_small, ctx->d_small, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
        *out = std::sqrt(ctx->h_small[0]);
    }
    return e;
}

int ctx_ensure_part(cdg_ctx *ctx, size_t n) {
    if (n <= ctx->part_cap) return CDG_OK;
    CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    dev_free(ctx, ctx->d_part, ctx->part_cap * sizeof(double));
    ctx->d_part = nullptr;
    ctx->part_cap = 0;
    size_t cap = std::max<size_t>(n, 4096);
    int e = dev_alloc(ctx, (void **)&ctx->d_part, cap * sizeof(double));
    if (e) return e;
    ctx->part_cap = cap;
    return CDG_OK;
}

int ctx_ensure_small(cdg_ctx *ctx, size_t n) {
    if (n <= ctx->small_cap) return CDG_OK;
    CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    dev_free(ctx, ctx->d_small, ctx->small_cap * sizeof(double));
    if (ctx->h_small) (void)hipHostFree(ctx->h_small);
    ctx->d_small = nullptr;
    ctx->h_small = nullptr;
    ctx->small_cap = 0;
    size_t cap = std::max<size_t>(n, 256);
    int e = dev_alloc(ctx, (void **)&ctx->d_small, cap * sizeof(double));
    if (e) return e;
    if (hipHostMalloc((void **)&ctx->h_small, cap * sizeof(double), hipHostMallocDefault) != hipSuccess)
        return cdg_fail(ctx, CDG_ERR_OOM, "hipHostMalloc failed");
    ctx->small_cap = cap;
    return CDG_OK;
}

bool is_device_ptr(const void *p) {
    if (!p) return false;
    hipPointerAttribute_t attr;
    hipError_t e = hipPointerGetAttributes(&attr, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return attr.type == hipMemoryTypeDevice;
}

namespace {

std::atomic<uint64_t> g_stamp{0};

// Device view of a vector argument: device pointers pass through, host
// pointers go through a per-slot staging buffer.
struct VecArg {
    double *dev = nullptr;
    double *host = nullptr;
    int64_t len = 0;
};

int stage_in(cdg_ctx *ctx, int slot, const double *p, int64_t len, VecArg &a) {
    a.len = len;
    if (is_device_ptr(p)) { a.dev = const_cast<double *>(p); return CDG_OK; }
    a.host = const_cast<double *>(p);
    size_t need = (size_t)std::max<int64_t>(len, 1);
    if (ctx->stage_cap[slot] < need) {
        CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
        dev_free(ctx, ctx->d_stage[slot], ctx->stage_cap[slot] * sizeof(double));
        ctx->d_stage[slot] = nullptr;
        ctx->stage_cap[slot] = 0;
        int e = dev_alloc(ctx, (void **)&ctx->d_stage[slot], need * sizeof(double));
        if (e) return e;
        ctx->stage_cap[slot] = need;
    }
    a.dev = ctx->d_stage[slot];
    return CDG_OK;
}

int upload_in(cdg_ctx *ctx, const VecArg &a) {
    if (a.host && a.len) CDG_HIP_TRY(hipMemcpyAsync(a.dev, a.host, sizeof(double) * a.len, hipMemcpyHostToDevice, ctx->stream));
    return CDG_OK;
}

int finish_out(cdg_ctx *ctx, const VecArg &a) {
    if (a.host && a.len) CDG_HIP_TRY(hipMemcpyAsync(a.host, a.dev, sizeof(double) * a.len, hipMemcpyDeviceToHost, ctx->stream));
    CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    return CDG_OK;
}

}  // namespace

int64_t slot_elems(int n) { return ((int64_t)n * n + 63) / 64 * 64; }

// ---- launch shapes and their autotuner ----------------------------------------
// The apply's shape: column-slice width, threads per workgroup (target of
// stream_shape) and 16-byte loads in flight; the matvec's: threads and loads
// in flight.  Defaults are the measured best at n = 135; cdg_prec_tune /
// cdg_mat_tune time candidates on a live factor / matrix and keep the fastest,
// and remember it per (block size, precision) for objects created afterwards.
namespace {
struct ApplyShape {
    int sw, target, unroll;
};
struct MvShape {
    int target, unroll;
};
std::mutex g_tune_mu;
std::map<std::pair<int, int>, ApplyShape> g_apply_tuned;   // (n, precision)
std::map<int, MvShape> g_mv_tuned;                          // n

// measured at n = 135: 32-column slices; 8 loads in flight for FP64, 4 for FP32/BF16
ApplyShape apply_default(int n, int precision) {
    const bool p2 = n > 64 && n <= 192;
    return {p2 ? 32 : 40, 256, p2 && precision == CDG_FP64 ? 8 : 4};
}
MvShape mv_default() { return {540, 8}; }

bool apply_tuned(int n, int precision, ApplyShape *out) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_apply_tuned.find({n, precision});
    if (it == g_apply_tuned.end()) return false;
    *out = it->second;
    return true;
}

bool mv_tuned(int n, MvShape *out) {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_mv_tuned.find(n);
    if (it == g_mv_tuned.end()) return false;
    *out = it->second;
    return true;
}

// Column slices are multiples of 8 columns, so every slice starts 16-byte
// aligned for all element widths.  False if the shape does not fit (LDS,
// threads); M is then unchanged.
bool apply_shape_set(cdg_prec *M, int precision, const ApplyShape &a) {
    const int n = M->n;
    int slices = std::max(1, (n + a.sw - 1) / a.sw);
    const int slice_w = ((n + slices - 1) / slices + 7) / 8 * 8;
    slices = (n + slice_w - 1) / slice_w;
    const StreamShape sh[3] = {stream_shape(n, 2, a.target), stream_shape(n, 4, a.target), stream_shape(n, 8, a.target)};
    const int V = precision == CDG_FP64 ? 2 : (precision == CDG_FP32 ? 4 : 8);
    const size_t accsz = precision == CDG_FP64 ? 8 : 4;
    const size_t lds = accsz * ((size_t)M->maxdep * slice_w + (size_t)V * sh[precision].T);
    if (sh[precision].T == 0 || lds > 64 * 1024) return false;
    M->slices = slices;
    M->slice_w = slice_w;
    M->unroll = a.unroll == 8 ? 8 : 4;
    for (int i = 0; i < 3; ++i) M->shape[i] = sh[i];
    M->part_len = (int64_t)M->nrows * slices * n;
    return true;
}
}  // namespace

namespace {

// Allocates and fills a device array.  Waits for the copy: callers pass
// temporaries, and an asynchronous copy from pageable memory may read its
// source after the call returns.
template <typename T>
int upload_array(cdg_ctx *ctx, T **d, const std::vector<T> &h, std::vector<DevMem> *owned) {
    size_t bytes = std::max<size_t>(1, h.size()) * sizeof(T);
    int e = dev_alloc(ctx, (void **)d, bytes);
    if (e) return e;
    if (owned) owned->push_back({*d, bytes});
    if (!h.empty()) {
        CDG_HIP_TRY(hipMemcpyAsync(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, ctx->stream));
        CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    return CDG_OK;
}

// kind-0 structure, transposes and wavefront levels of a pattern
void analyze(cdg_mat *A) {
    const int nr = A->nrows;
    A->diag.assign(nr, -1);
    A->lo_ptr.assign(nr + 1, 0);
    A->up_ptr.assign(nr + 1, 0);
    A->lo_blk.clear(); A->lo_col.clear(); A->up_blk.clear(); A->up_col.clear();
    A->struct_err = CDG_OK;
    for (int i = 0; i < nr; ++i) {
        for (int b = A->row_ptr[i]; b < A->row_ptr[i + 1]; ++b) {
            if (A->kind[b] != CDG_KIND_LOCAL) continue;
            const int j = A->col[b];
            if (j == i) { if (A->diag[i] < 0) A->diag[i] = b; }
            else if (!A->part.empty() && A->part[j] != A->part[i]) continue;   // parent on another rank
            else if (j < i) { A->lo_blk.push_back(b); A->lo_col.push_back(j); }
            else { A->up_blk.push_back(b); A->up_col.push_back(j); }
        }
        A->lo_ptr[i + 1] = (int32_t)A->lo_blk.size();
        A->up_ptr[i + 1] = (int32_t)A->up_blk.size();
        if (A->diag[i] < 0) A->struct_err = CDG_ERR_ARG;
    }
    auto find_t = [&](int row, int parent) {
        for (int b = A->row_ptr[row]; b < A->row_ptr[row + 1]; ++b)
            if (A->kind[b] == CDG_KIND_LOCAL && A->col[b] == parent) return b;
        return -1;
    };
    A->lo_tr.resize(A->lo_blk.size());
    A->up_tr.resize(A->up_blk.size());
    for (int i = 0; i < nr; ++i) {
        for (int q = A->lo_ptr[i]; q < A->lo_ptr[i + 1]; ++q) {
            A->lo_tr[q] = find_t(A->lo_col[q], i);
            if (A->lo_tr[q] < 0 && A->struct_err == CDG_OK) A->struct_err = CDG_ERR_NO_TRANSPOSE;
        }
        for (int u = A->up_ptr[i]; u < A->up_ptr[i + 1]; ++u) {
            A->up_tr[u] = find_t(A->up_col[u], i);
            if (A->up_tr[u] < 0 && A->struct_err == CDG_OK) A->struct_err = CDG_ERR_NO_TRANSPOSE;
        }
    }
    A->flevel.assign(nr, 0);
    A->blevel.assign(nr, 0);
    A->nflev = nr ? 1 : 0;
    A->nblev = nr ? 1 : 0;
    for (int i = 0; i < nr; ++i) {
        int l = 0;
        for (int q = A->lo_ptr[i]; q < A->lo_ptr[i + 1]; ++q) l = std::max(l, A->flevel[A->lo_col[q]] + 1);
        A->flevel[i] = l;
        A->nflev = std::max(A->nflev, l + 1);
    }
    for (int i = nr - 1; i >= 0; --i) {
        int l = 0;
        for (int u = A->up_ptr[i]; u < A->up_ptr[i + 1]; ++u) l = std::max(l, A->blevel[A->up_col[u]] + 1);
        A->blevel[i] = l;
        A->nblev = std::max(A->nblev, l + 1);
    }
    A->max_row_blocks = 0;
    for (int i = 0; i < nr; ++i) A->max_row_blocks = std::max(A->max_row_blocks, A->row_ptr[i + 1] - A->row_ptr[i]);
}

std::vector<int32_t> order_by_level(const std::vector<int32_t> &lev, int nlev, std::vector<int32_t> *ptr_out) {
    std::vector<int32_t> ptr(nlev + 1, 0), rows(lev.size());
    for (int32_t l : lev) ptr[l + 1]++;
    for (int l = 0; l < nlev; ++l) ptr[l + 1] += ptr[l];
    std::vector<int32_t> fill(ptr.begin(), ptr.end() - 1);
    for (size_t i = 0; i < lev.size(); ++i) rows[fill[lev[i]]++] = (int32_t)i;
    if (ptr_out) *ptr_out = ptr;
    return rows;
}

}  // namespace

// ---------------------------------------------------------------------------
// context
// ---------------------------------------------------------------------------
int ctx_wait(cdg_ctx *ctx) {
    if (!ctx->spin || !ctx->done_ev) {
        CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
        return CDG_OK;
    }
    CDG_HIP_TRY(hipEventRecord(ctx->done_ev, ctx->stream));
    const auto t0 = std::chrono::steady_clock::now();
    hipError_t q;
    while ((q = hipEventQuery(ctx->done_ev)) == hipErrorNotReady) {
        if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(5)) {
            q = hipEventSynchronize(ctx->done_ev);
            break;
        }
    }
    if (q != hipSuccess) return cdg_fail(ctx, CDG_ERR_HIP, "%s", hipGetErrorString(q));
    return CDG_OK;
}

extern "C" int cdg_ctx_create(int32_t device, cdg_ctx **out) {
    if (!out) return CDG_ERR_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) { (void)hipGetLastError(); return CDG_ERR_HIP; }
    if (device < 0 || device >= ndev) return CDG_ERR_ARG;
    if (hipSetDevice(device) != hipSuccess) return CDG_ERR_HIP;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return CDG_ERR_HIP;
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return CDG_ERR_UNSUPPORTED;
    cdg_ctx *ctx = new cdg_ctx();
    ctx->device = device;
    ctx->num_cus = prop.multiProcessorCount;
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) { delete ctx; return CDG_ERR_HIP; }
    if (hipEventCreateWithFlags(&ctx->done_ev, hipEventDisableTiming) != hipSuccess) {
        ctx->done_ev = nullptr;
        cdg_ctx_destroy(ctx);
        return CDG_ERR_HIP;
    }
    if (const char *sp = std::getenv("CDG_SPIN")) ctx->spin = std::atoi(sp) != 0;
    if (ctx_ensure_small(ctx, 4096) || ctx_ensure_part(ctx, 1 << 16)) { cdg_ctx_destroy(ctx); return CDG_ERR_OOM; }
    *out = ctx;
    return CDG_OK;
}

extern "C" int cdg_ctx_destroy(cdg_ctx *ctx) {
    if (!ctx) return CDG_OK;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    dev_free(ctx, ctx->d_part, ctx->part_cap * sizeof(double));
    dev_free(ctx, ctx->d_small, ctx->small_cap * sizeof(double));
    if (ctx->h_small) (void)hipHostFree(ctx->h_small);
    for (int s = 0; s < 3; ++s) dev_free(ctx, ctx->d_stage[s], ctx->stage_cap[s] * sizeof(double));
    for (auto &kv : ctx->alloc_size) (void)hipFree(kv.first);   // blocks of objects never destroyed
    ctx->alloc_size.clear();
    ctx_flush_cache(ctx);
    if (ctx->done_ev) (void)hipEventDestroy(ctx->done_ev);
    if (ctx->order_ev) (void)hipEventDestroy(ctx->order_ev);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    for (uint32_t *p : ctx->word_pages) (void)hipHostFree(p);
    if (ctx->h_arn) (void)hipHostFree(ctx->h_arn);
    delete ctx;
    return CDG_OK;
}

extern "C" const char *cdg_last_error(const cdg_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

extern "C" int cdg_ctx_mem_used(const cdg_ctx *ctx, int64_t *bytes) {
    if (!ctx || !bytes) return CDG_ERR_ARG;
    *bytes = ctx->mem_used;
    return CDG_OK;
}

extern "C" int cdg_ctx_stream(const cdg_ctx *ctx, void **stream) {
    if (!ctx || !stream) return CDG_ERR_ARG;
    *stream = static_cast<void *>(ctx->stream);
    return CDG_OK;
}

// Cross-stream ordering without a host wait: an event recorded on one stream,
// waited on by the other.
static int stream_order(cdg_ctx *ctx, hipStream_t before, hipStream_t after) {
    CDG_HIP_TRY(hipSetDevice(ctx->device));
    if (!ctx->order_ev) CDG_HIP_TRY(hipEventCreateWithFlags(&ctx->order_ev, hipEventDisableTiming));
    CDG_HIP_TRY(hipEventRecord(ctx->order_ev, before));
    CDG_HIP_TRY(hipStreamWaitEvent(after, ctx->order_ev, 0));
    return CDG_OK;
}

extern "C" int cdg_ctx_wait_stream(cdg_ctx *ctx, void *stream) {
    if (!ctx) return CDG_ERR_ARG;
    return stream_order(ctx, static_cast<hipStream_t>(stream), ctx->stream);
}

extern "C" int cdg_ctx_signal_stream(cdg_ctx *ctx, void *stream) {
    if (!ctx) return CDG_ERR_ARG;
    return stream_order(ctx, ctx->stream, static_cast<hipStream_t>(stream));
}

// ---------------------------------------------------------------------------
// matrix
// ---------------------------------------------------------------------------
extern "C" int cdg_mat_create(cdg_ctx *ctx, int32_t nrows, int32_t block_n, const int32_t *row_ptr,
                              const int32_t *col, const int32_t *kind, cdg_mat **out) {
    if (!ctx || !out) return CDG_ERR_ARG;
    *out = nullptr;
    if (nrows < 0 || block_n <= 0 || block_n > 1024 || !row_ptr || (nrows > 0 && (!col || !kind)))
        return cdg_fail(ctx, CDG_ERR_ARG, "cdg_mat_create: bad sizes or null arrays");
    if (row_ptr[0] != 0) return cdg_fail(ctx, CDG_ERR_ARG, "row_ptr[0] must be 0");
    for (int i = 0; i < nrows; ++i)
        if (row_ptr[i + 1] < row_ptr[i]) return cdg_fail(ctx, CDG_ERR_ARG, "row_ptr not monotone at %d", i);
    const int nnzb = row_ptr[nrows];
    for (int b = 0; b < nnzb; ++b) {
        if (col[b] < 0 || col[b] >= nrows) return cdg_fail(ctx, CDG_ERR_ARG, "col[%d]=%d out of range", b, col[b]);
        if (kind[b] != CDG_KIND_LOCAL && kind[b] != CDG_KIND_COUPLING)
            return cdg_fail(ctx, CDG_ERR_ARG, "kind[%d]=%d invalid", b, kind[b]);
    }
    CDG_HIP_TRY(hipSetDevice(ctx->device));
    cdg_mat *A = new cdg_mat();
    A->nrows = nrows;
    A->n = block_n;
    A->nnzb = nnzb;
    A->ld = slot_elems(block_n);
    A->row_ptr.assign(row_ptr, row_ptr + nrows + 1);
    A->col.assign(col, col + nnzb);
    A->kind.assign(kind, kind + nnzb);
    analyze(A);
    {   // matvec launch shape: tuned for this block size if cdg_mat_tune has run,
        // else ~540 threads with 8 loads in flight each, the measured best at
        // n = 135 (0.611 ms = 6.85 TB/s, against 0.652 ms with ~1024 threads and
        // 4); CDG_MV_THREADS / CDG_MV_UNROLL override either
        MvShape ms = mv_default();
        (void)mv_tuned(block_n, &ms);
        if (const char *t = std::getenv("CDG_MV_THREADS")) ms.target = std::max(64, std::atoi(t));
        if (const char *u = std::getenv("CDG_MV_UNROLL")) ms.unroll = std::atoi(u);
        A->shape64 = stream_shape(block_n, 2, ms.target);
        A->mv_unroll = ms.unroll == 16 ? 16 : ms.unroll == 8 ? 8 : 4;
    }
    int e = dev_alloc(ctx, (void **)&A->blocks, sizeof(double) * (size_t)std::max(1, nnzb) * A->ld);
    if (!e) e = upload_array(ctx, &A->d_row_ptr, A->row_ptr, nullptr);
    if (!e) e = upload_array(ctx, &A->d_col, A->col, nullptr);
    if (e) { cdg_mat_destroy(ctx, A); return e; }
    hipError_t he = hipMemsetAsync(A->blocks, 0, sizeof(double) * (size_t)std::max(1, nnzb) * A->ld, ctx->stream);
    if (he == hipSuccess) he = hipStreamSynchronize(ctx->stream);
    if (he != hipSuccess) { cdg_mat_destroy(ctx, A); return cdg_fail(ctx, CDG_ERR_HIP, "%s", hipGetErrorString(he)); }
    *out = A;
    return CDG_OK;
}

extern "C" int cdg_mat_destroy(cdg_ctx *ctx, cdg_mat *A) {
    if (!A) return CDG_OK;
    if (ctx) {
        (void)hipStreamSynchronize(ctx->stream);
        dev_free(ctx, A->blocks, sizeof(double) * (size_t)std::max(1, A->nnzb) * A->ld);
        dev_free(ctx, A->d_row_ptr, sizeof(int32_t) * (A->row_ptr.size()));
        dev_free(ctx, A->d_col, sizeof(int32_t) * std::max<size_t>(1, A->col.size()));
    }
    delete A;
    return CDG_OK;
}

extern "C" int cdg_mat_upload(cdg_ctx *ctx, cdg_mat *A, const double *blocks) {
    if (!ctx || !A || (!blocks && A->nnzb)) return CDG_ERR_ARG;
    if (A->nnzb == 0) { A->stamp = ++g_stamp; return CDG_OK; }
    const size_t nn = (size_t)A->n * A->n;
    const hipMemcpyKind kind = is_device_ptr(blocks) ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    CDG_HIP_TRY(hipMemcpy2DAsync(A->blocks, sizeof(double) * A->ld, blocks, sizeof(double) * nn, sizeof(double) * nn,
                                 A->nnzb, kind, ctx->stream));
    CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    A->stamp = ++g_stamp;
    return CDG_OK;
}

extern "C" int cdg_mat_download(cdg_ctx *ctx, const cdg_mat *A, double *blocks) {
    if (!ctx || !A || (!blocks && A->nnzb)) return CDG_ERR_ARG;
    if (A->nnzb == 0) return CDG_OK;
    const size_t nn = (size_t)A->n * A->n;
    const hipMemcpyKind kind = is_device_ptr(blocks) ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
    CDG_HIP_TRY(hipMemcpy2DAsync(blocks, sizeof(double) * nn, A->blocks, sizeof(double) * A->ld, sizeof(double) * nn,
                                 A->nnzb, kind, ctx->stream));
    CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    return CDG_OK;
}

extern "C" int cdg_mat_fill_synthetic(cdg_ctx *ctx, cdg_mat *A, uint64_t seed, double s_diag, double s_off) {
    if (!ctx || !A) return CDG_ERR_ARG;
    int e = launch_fill_synthetic(ctx, A, seed, s_diag, s_off);
    if (e) return e;
    A->stamp = ++g_stamp;
    return CDG_OK;
}

extern "C" int cdg_vec_fill_synthetic(cdg_ctx *ctx, const cdg_mat *A, uint64_t seed, double scale, double *v) {
    if (!ctx || !A || !v) return CDG_ERR_ARG;
    VecArg o;
    const int64_t len = (int64_t)A->nrows * A->n;
    int e = stage_in(ctx, 2, v, len, o);
    if (!e) e = launch_vec_synthetic(ctx, len, seed, scale, o.dev);
    if (!e) e = finish_out(ctx, o);
    return e;
}

extern "C" int cdg_mat_set_partition(cdg_ctx *ctx, cdg_mat *A, const int32_t *part) {
    if (!ctx || !A) return CDG_ERR_ARG;
    if (part) {
        for (int i = 0; i < A->nrows; ++i)
            if (part[i] < 0) return cdg_fail(ctx, CDG_ERR_ARG, "part[%d] = %d is negative", i, part[i]);
        A->part.assign(part, part + A->nrows);
    } else {
        A->part.clear();
    }
    analyze(A);
    return CDG_OK;
}

extern "C" int cdg_mat_stamp(const cdg_mat *A, uint64_t *stamp) {
    if (!A || !stamp) return CDG_ERR_ARG;
    *stamp = A->stamp;
    return CDG_OK;
}

extern "C" int cdg_mat_info(const cdg_mat *A, int32_t *nrows, int32_t *block_n, int32_t *nnzb) {
    if (!A) return CDG_ERR_ARG;
    if (nrows) *nrows = A->nrows;
    if (block_n) *block_n = A->n;
    if (nnzb) *nnzb = A->nnzb;
    return CDG_OK;
}

extern "C" int cdg_mv(cdg_ctx *ctx, const cdg_mat *A, const double *x, double *y) {
    if (!ctx || !A || !x || !y) return CDG_ERR_ARG;
    const int64_t len = (int64_t)A->nrows * A->n;
    VecArg xi, yo;
    int e = stage_in(ctx, 0, x, len, xi);
    if (!e) e = stage_in(ctx, 1, y, len, yo);
    if (!e) e = upload_in(ctx, xi);
    if (!e) e = launch_mv(ctx, A, xi.dev, yo.dev);
    if (!e) e = finish_out(ctx, yo);
    return e;
}

extern "C" int cdg_mv_async(cdg_ctx *ctx, const cdg_mat *A, const double *x, double *y) {
    if (!ctx || !A || !x || !y) return CDG_ERR_ARG;
    if (!is_device_ptr(x) || !is_device_ptr(y)) return cdg_fail(ctx, CDG_ERR_ARG, "cdg_mv_async needs device pointers");
    return launch_mv(ctx, A, x, y);
}

// ---------------------------------------------------------------------------
// preconditioner
// ---------------------------------------------------------------------------
// The partial sums' storage of the column-slice schedules (FOLDED, DATAFLOW and the level
// launches), at least 3 part_len doubles; the sweep has none.  (+2: a launch whose
// rows have no entries issues its 16-byte block prefetch from the start of a partial
// array, unused.)
static int prec_part_fit(cdg_ctx *ctx, cdg_prec *M) {
    const int64_t need = 3 * M->part_len + 2;
    if (need <= M->part_cap) return CDG_OK;
    double *np = nullptr;
    const size_t bytes = sizeof(double) * (size_t)need;
    int e = dev_alloc(ctx, (void **)&np, bytes);
    if (e) return e;
    if (!M->d_part) M->owned.push_back({np, bytes});
    for (DevMem &m : M->owned)
        if (M->d_part && m.p == M->d_part) { dev_free(ctx, m.p, m.bytes); m.p = np; m.bytes = bytes; }
    M->d_part = np;
    M->part_cap = need;
    return CDG_OK;
}

// Task list, counters and partial storage of the dataflow sweep (once per
// preconditioner).  Tickets: forward levels ascending; per backward level its
// BA tasks then its BB tasks, so every input of a task has a smaller ticket.
static int df_setup(cdg_ctx *ctx, cdg_prec *M) {
    if (M->d_tasks) return prec_part_fit(ctx, M);
    int e = df_configure(ctx, M);
    if (e) return e;
    const int S = M->df_S;
    std::vector<int32_t> tasks;
    tasks.reserve((size_t)3 * M->nrows * S);
    for (int l = 0; l < M->nlev; ++l)
        for (int k = M->lev_row_ptr[l]; k < M->lev_row_ptr[l + 1]; ++k)
            for (int sl = 0; sl < S; ++sl) tasks.push_back(((M->h_lev_rows[k] * S + sl) << 2) | 0);
    for (int l = 0; l < M->nblev; ++l)
        for (int stg = 1; stg <= 2; ++stg)
            for (int k = M->blev_row_ptr[l]; k < M->blev_row_ptr[l + 1]; ++k)
                for (int sl = 0; sl < S; ++sl) tasks.push_back(((M->h_blev_rows[k] * S + sl) << 2) | stg);
    M->df_ntasks = (int32_t)tasks.size();
    const int64_t need = 3 * (int64_t)M->nrows * S * M->n;
    M->part_len = std::max(M->part_len, need / 3);   // partial storage shared with the level schedule
    e = prec_part_fit(ctx, M);
    if (e) return e;
    e = upload_array(ctx, &M->d_tasks, tasks, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_cnt, std::vector<int32_t>((size_t)3 * M->nrows, 0), &M->owned);
    if (!e) e = upload_array(ctx, &M->d_dferr, std::vector<int32_t>(1, 0), &M->owned);
    if (!e) {
        e = dev_alloc(ctx, (void **)&M->d_ticket, sizeof(unsigned long long));
        if (!e) M->owned.push_back({M->d_ticket, sizeof(unsigned long long)});
    }
    if (!e) e = df_reset(ctx, M);
    return e;
}

extern "C" int cdg_prec_destroy(cdg_ctx *ctx, cdg_prec *M) {
    if (!M) return CDG_OK;
    if (ctx) {
        (void)hipStreamSynchronize(ctx->stream);
        for (DevMem &m : M->owned) dev_free(ctx, m.p, m.bytes);
        if (M->h_err) ctx->word_free.push_back(M->h_err);
    }
    sweep_free(M);
    delete M;
    return CDG_OK;
}

extern "C" int cdg_prec_create(cdg_ctx *ctx, const cdg_mat *A, int32_t type, int32_t precision, cdg_prec **out) {
    if (!ctx || !A || !out) return CDG_ERR_ARG;
    *out = nullptr;
    if (type != CDG_PREC_IDENTITY && type != CDG_PREC_ILU0 && type != CDG_PREC_JACOBI)
        return cdg_fail(ctx, CDG_ERR_ARG, "unknown preconditioner %d", type);
    if (precision < CDG_FP64 || precision > CDG_BF16) return cdg_fail(ctx, CDG_ERR_ARG, "unknown precision %d", precision);
    cdg_prec *M = new cdg_prec();
    M->type = type;
    M->precision = precision;
    M->nrows = A->nrows;
    M->n = A->n;
    if (type == CDG_PREC_IDENTITY) { *out = M; return CDG_OK; }
    // The kind-0 structure the factor follows: A's, or for block Jacobi
    // (precon_jacobi.f90:95-215) the diagonal alone -- ILU(0) of a matrix
    // whose every row is its own rank: L = 0, U = 0, Dinv_i = inv(A_ii), and
    // the apply is z_i = Dinv_i v_i.
    cdg_mat jview;
    const cdg_mat *S = A;
    if (type == CDG_PREC_JACOBI) {
        jview.nrows = A->nrows;
        jview.n = A->n;
        jview.nnzb = A->nnzb;
        jview.row_ptr = A->row_ptr;
        jview.col = A->col;
        jview.kind = A->kind;
        jview.part.resize(A->nrows);
        for (int i = 0; i < A->nrows; ++i) jview.part[i] = i;
        analyze(&jview);
        S = &jview;
        M->type = CDG_PREC_ILU0;   // the ILU(0) machinery with no off-diagonal blocks
        M->jacobi = 1;
    }
    if (S->struct_err != CDG_OK) {
        delete M;
        return cdg_fail(ctx, S->struct_err, S->struct_err == CDG_ERR_NO_TRANSPOSE
                                                ? "lblks entry without a transposed partner"
                                                : "block row without a diagonal block");
    }
    M->nlo = (int32_t)S->lo_blk.size();
    M->nup = (int32_t)S->up_blk.size();
    M->ld = slot_elems(A->n);
    const size_t es = precision == CDG_FP64 ? 8 : (precision == CDG_FP32 ? 4 : 2);
    auto alloc = [&](void **p, size_t bytes) -> int {
        bytes = std::max<size_t>(bytes, 16);
        int e = dev_alloc(ctx, p, bytes);
        if (!e) M->owned.push_back({*p, bytes});
        return e;
    };
    int e = alloc(&M->L, es * (size_t)M->nlo * M->ld);
    if (!e) e = alloc(&M->Dinv, es * (size_t)M->nrows * M->ld);
    if (!e && precision != CDG_FP64) e = alloc(&M->U, es * (size_t)M->nup * M->ld);
    if (!e && precision == CDG_BF16) {
        e = alloc((void **)&M->L32, 4 * (size_t)M->nlo * M->ld);
        if (!e) e = alloc((void **)&M->D32, 4 * (size_t)M->nrows * M->ld);
    }
    // structure arrays
    std::vector<int32_t> up_idx(M->nup);
    for (int u = 0; u < M->nup; ++u) up_idx[u] = precision == CDG_FP64 ? S->up_blk[u] : u;
    if (!e) e = upload_array(ctx, &M->d_lo_ptr, S->lo_ptr, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_lo_blk, S->lo_blk, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_lo_col, S->lo_col, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_lo_tr, S->lo_tr, &M->owned);
    if (!e && precision != CDG_FP64) {
        // A_ji (j < i) is an upper block of row j, so every lo_tr[q] has a U slot
        std::vector<int32_t> slot_of(std::max(A->nnzb, 1), -1), lo_tru(S->lo_tr.size());
        for (int u = 0; u < M->nup; ++u) slot_of[S->up_blk[u]] = u;
        for (size_t q = 0; q < lo_tru.size(); ++q) lo_tru[q] = slot_of[S->lo_tr[q]];
        e = upload_array(ctx, &M->d_lo_tru, lo_tru, &M->owned);
    }
    if (!e) e = upload_array(ctx, &M->d_up_ptr, S->up_ptr, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_up_blk, S->up_blk, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_up_idx, up_idx, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_up_col, S->up_col, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_diag, S->diag, &M->owned);
    // forward levels (factor schedule and forward sweep), backward levels
    std::vector<int32_t> fptr, bptr;
    std::vector<int32_t> forder = order_by_level(S->flevel, S->nflev, &fptr);
    std::vector<int32_t> border = order_by_level(S->blevel, S->nblev, &bptr);
    M->nlev = S->nflev;
    M->lev_row_ptr = fptr;
    M->nblev = S->nblev;
    M->blev_row_ptr = bptr;
    std::vector<int32_t> lev_lo;
    M->lev_lo_ptr.assign(M->nlev + 1, 0);
    for (int l = 0; l < M->nlev; ++l) {
        for (int k = fptr[l]; k < fptr[l + 1]; ++k) {
            const int i = forder[k];
            for (int q = S->lo_ptr[i]; q < S->lo_ptr[i + 1]; ++q) lev_lo.push_back(q);
        }
        M->lev_lo_ptr[l + 1] = (int32_t)lev_lo.size();
    }
    if (!e) e = upload_array(ctx, &M->d_lev_lo, lev_lo, &M->owned);
    {   // the W jobs: every upper slot
        std::vector<int32_t> all(std::max(M->nup, 1));
        for (int u = 0; u < M->nup; ++u) all[u] = u;
        if (!e) e = upload_array(ctx, &M->d_up_all, all, &M->owned);
    }
    if (!e) e = upload_array(ctx, &M->d_lev_rows, forder, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_blev_rows, border, &M->owned);
    if (!e) e = upload_array(ctx, &M->d_err, std::vector<int32_t>(1, 0), &M->owned);
    if (!e) {
        hipError_t he = hipStreamSynchronize(ctx->stream);
        if (he != hipSuccess) e = cdg_fail(ctx, CDG_ERR_HIP, "%s", hipGetErrorString(he));
    }
    if (e) { cdg_prec_destroy(ctx, M); return e; }
    M->maxdep = 1;
    for (int i = 0; i < A->nrows; ++i) {
        M->maxdep = std::max(M->maxdep, S->lo_ptr[i + 1] - S->lo_ptr[i]);
        M->maxdep = std::max(M->maxdep, S->up_ptr[i + 1] - S->up_ptr[i]);
    }
    // Apply launch shape: the tuned one for this block size and precision if
    // cdg_prec_tune has run, else the default; CDG_APPLY_SLICE_W /
    // CDG_APPLY_THREADS / CDG_APPLY_UNROLL override either.
    ApplyShape ash = apply_default(A->n, precision);
    (void)apply_tuned(A->n, precision, &ash);
    if (const char *ev = std::getenv("CDG_APPLY_SLICE_W")) ash.sw = std::max(8, std::atoi(ev));
    if (const char *ev = std::getenv("CDG_APPLY_THREADS")) ash.target = std::max(64, std::atoi(ev));
    if (const char *ev = std::getenv("CDG_APPLY_UNROLL")) ash.unroll = std::atoi(ev) == 8 ? 8 : 4;
    if (e || !apply_shape_set(M, precision, ash)) {
        cdg_prec_destroy(ctx, M);
        return e ? e : cdg_fail(ctx, CDG_ERR_UNSUPPORTED, "ILU apply launch shape does not fit (block size %d)", A->n);
    }
    // apply schedule (CDG_APPLY_MODE=levels|dataflow|folded|auto overrides the default)
    M->apply_mode = CDG_APPLY_AUTO;
    if (const char *m = std::getenv("CDG_APPLY_MODE")) {
        if (!std::strcmp(m, "dataflow")) M->apply_mode = CDG_APPLY_DATAFLOW;
        else if (!std::strcmp(m, "auto")) M->apply_mode = CDG_APPLY_AUTO;
        else if (!std::strcmp(m, "levels")) M->apply_mode = CDG_APPLY_LEVELS;
        else if (!std::strcmp(m, "folded") && precision != CDG_BF16) M->apply_mode = CDG_APPLY_FOLDED;
        else if (!std::strcmp(m, "stream")) M->apply_mode = CDG_APPLY_STREAM;
    }
    M->h_lev_rows = forder;
    M->h_lo_ptr = S->lo_ptr;
    M->h_lo_col = S->lo_col;
    M->h_up_ptr = S->up_ptr;
    M->h_up_col = S->up_col;
    M->h_up_idx = up_idx;
    M->h_blev_rows = border;
    if (!e && M->apply_mode == CDG_APPLY_DATAFLOW) e = df_setup(ctx, M);
    if (!e && M->apply_mode == CDG_APPLY_FOLDED) e = alloc(&M->W, es * (size_t)M->nup * M->ld);
    if (!e && ctx->word_free.empty()) {
        uint32_t *page = nullptr;
        constexpr size_t kWords = 64, kPitch = 16;   // a word per cache line
        if (hipHostMalloc((void **)&page, sizeof(uint32_t) * kWords * kPitch) == hipSuccess) {
            ctx->word_pages.push_back(page);
            for (size_t i = 0; i < kWords; ++i) ctx->word_free.push_back(page + kPitch * i);
        } else {
            e = cdg_fail(ctx, CDG_ERR_OOM, "pinned error words");
        }
    }
    if (!e) {
        M->h_err = ctx->word_free.back();
        ctx->word_free.pop_back();
        *M->h_err = 0;
    }
    if (const char *f = std::getenv("CDG_FOLD_AFTER")) M->fold_after = std::max(0, std::atoi(f));
    if (!e) {   // the single-vector sweep's plans and W, so that an apply never allocates
        SweepPlan *p = nullptr;
        int ep = sweep_plan(ctx, M, 1, 0, M->nrows, false, &p);
        if (ep == CDG_ERR_UNSUPPORTED) M->sweep_ok = 0;
        else e = ep;
        if (!e && (!M->sweep_ok || M->apply_mode == CDG_APPLY_FOLDED)) e = prec_part_fit(ctx, M);
        if (!e && M->sweep_ok && precision == CDG_BF16 && M->nup > 0 && M->maxdep <= 6) {
            ep = sweep_plan(ctx, M, 1, 0, M->nrows, true, &p);
            if (!ep) {
                std::vector<int32_t> up_row(M->nup);
                for (int i = 0; i < M->nrows; ++i)
                    for (int u = S->up_ptr[i]; u < S->up_ptr[i + 1]; ++u) up_row[u] = i;
                M->fold_ok = 1;
                e = alloc(&M->W, es * (size_t)M->nup * M->ld);
                if (!e) e = upload_array(ctx, &M->d_up_row, up_row, &M->owned);
                if (!e && hipStreamSynchronize(ctx->stream) != hipSuccess)   // up_row is host memory
                    e = cdg_fail(ctx, CDG_ERR_HIP, "upload of the upper entries' rows");
            } else if (ep != CDG_ERR_UNSUPPORTED) {
                e = ep;
            }
        }
    }
    if (!e) {
        hipError_t he = hipStreamSynchronize(ctx->stream);
        if (he != hipSuccess) e = cdg_fail(ctx, CDG_ERR_HIP, "%s", hipGetErrorString(he));
    }
    if (e) { cdg_prec_destroy(ctx, M); return e; }
    *out = M;
    return CDG_OK;
}

extern "C" int cdg_prec_set_schedule(cdg_ctx *ctx, cdg_prec *M, int32_t schedule) {
    if (!ctx || !M) return CDG_ERR_ARG;
    if (schedule != CDG_SCHEDULE_LEVELS && schedule != CDG_SCHEDULE_DATAFLOW && schedule != CDG_SCHEDULE_FOLDED &&
        schedule != CDG_SCHEDULE_AUTO && schedule != CDG_SCHEDULE_STREAM && schedule != CDG_SCHEDULE_ROWSLICE)
        return cdg_fail(ctx, CDG_ERR_ARG, "unknown apply schedule %d", schedule);
    if (M->type != CDG_PREC_ILU0) return CDG_OK;
    if (schedule == CDG_SCHEDULE_DATAFLOW) {
        int e = df_setup(ctx, M);
        if (e) return e;
        CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    }
    if (schedule == CDG_SCHEDULE_STREAM || schedule == CDG_SCHEDULE_ROWSLICE) {
        if (!M->sweep_ok || M->maxdep > 6)
            return cdg_fail(ctx, CDG_ERR_UNSUPPORTED, "stream schedule: a row has more than 6 lower or upper blocks");
        M->noalloc_ok = 1;
    }
    if (schedule == CDG_SCHEDULE_FOLDED) {
        if (M->precision == CDG_BF16)
            return cdg_fail(ctx, CDG_ERR_UNSUPPORTED, "folded schedule: FP64 and FP32 factors only");
        if (!M->W) {
            const size_t bytes = std::max<size_t>(16, (M->precision == CDG_FP64 ? 8 : 4) * (size_t)M->nup * M->ld);
            int e = dev_alloc(ctx, &M->W, bytes);
            if (e) return e;
            M->owned.push_back({M->W, bytes});
        }
        int e = prec_part_fit(ctx, M);
        if (e) return e;
    }
    M->apply_mode = schedule == CDG_SCHEDULE_DATAFLOW ? CDG_APPLY_DATAFLOW
                    : schedule == CDG_SCHEDULE_FOLDED ? CDG_APPLY_FOLDED
                    : schedule == CDG_SCHEDULE_STREAM ? CDG_APPLY_STREAM
                    : schedule == CDG_SCHEDULE_ROWSLICE ? CDG_APPLY_ROWSLICE
                    : schedule == CDG_SCHEDULE_AUTO ? CDG_APPLY_AUTO : CDG_APPLY_LEVELS;
    return CDG_OK;
}

// Whether the next apply of k vectors takes the sweep over W (BF16).
static bool takes_w(const cdg_prec *M, int k) {
    if (!M->fold_ok || M->apply_mode == CDG_APPLY_DATAFLOW) return false;
    if (k > 1 || M->apply_mode == CDG_APPLY_STREAM || M->apply_mode == CDG_APPLY_ROWSLICE) return true;
    if (M->apply_mode != CDG_APPLY_AUTO) return false;
    return M->w_asked || (M->fold_after > 0 && (M->napply + k > M->fold_after || M->prev_napply > M->fold_after));
}

// ---- launch-shape autotuner (no reference counterpart) ---------------------------
namespace {
// Times fn() `reps` times on the context's stream (one untimed call first).
template <typename F>
int time_on_stream(cdg_ctx *ctx, hipEvent_t e0, hipEvent_t e1, int reps, F fn, double *ms_out) {
    int e = fn();
    if (e) return e;
    CDG_HIP_TRY(hipEventRecord(e0, ctx->stream));
    for (int r = 0; r < reps && !e; ++r) e = fn();
    if (e) return e;
    CDG_HIP_TRY(hipEventRecord(e1, ctx->stream));
    CDG_HIP_TRY(hipEventSynchronize(e1));
    float ms = 0.f;
    CDG_HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
    *ms_out = (double)ms / reps;
    return CDG_OK;
}

struct Scratch {   // tuning vectors and events, released on every path out
    cdg_ctx *ctx;
    double *v = nullptr, *z = nullptr;
    size_t bytes = 0;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    explicit Scratch(cdg_ctx *c) : ctx(c) {}
    int init(int64_t len) {
        bytes = sizeof(double) * (size_t)std::max<int64_t>(len, 1);
        int e = dev_alloc(ctx, (void **)&v, bytes);
        if (!e) e = dev_alloc(ctx, (void **)&z, bytes);
        if (!e) e = kv_zero(ctx, std::max<int64_t>(len, 1), v);
        if (!e && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess))
            e = cdg_fail(ctx, CDG_ERR_HIP, "hipEventCreate failed");
        return e;
    }
    ~Scratch() {
        (void)hipStreamSynchronize(ctx->stream);
        if (v) dev_free(ctx, v, bytes);
        if (z) dev_free(ctx, z, bytes);
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
    }
};
}  // namespace

extern "C" int cdg_prec_tune(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, int32_t reps, double *best_ms) {
    if (!ctx || !M || !A) return CDG_ERR_ARG;
    if (best_ms) *best_ms = 0.0;
    if (M->type != CDG_PREC_ILU0 || M->nrows == 0) return CDG_OK;
    if (A->nrows != M->nrows || A->n != M->n) return cdg_fail(ctx, CDG_ERR_ARG, "matrix does not match preconditioner");
    if (!M->factored) return cdg_fail(ctx, CDG_ERR_STATE, "cdg_prec_tune before cdg_prec_update");
    if (M->apply_mode == CDG_APPLY_DATAFLOW)
        return cdg_fail(ctx, CDG_ERR_UNSUPPORTED, "cdg_prec_tune: the level schedules only");
    reps = std::max(1, std::min<int32_t>(reps, 1000));
    const int n = M->n, prec = M->precision;
    Scratch sc(ctx);
    int e = sc.init((int64_t)M->nrows * n);
    if (e) return e;
    if (M->apply_mode != CDG_APPLY_FOLDED && M->sweep_ok) {   // the sweep has its shape by a rule: its time only
        const bool fold = takes_w(M, 1);
        double ms = 0.0;
        if (fold) e = sweep_fold(ctx, M, A);
        if (!e) e = time_on_stream(ctx, sc.e0, sc.e1, reps,
                                   [&] { return launch_ilu_sweep(ctx, M, A, sc.v, sc.z, (int64_t)M->nrows * n, 1, fold); }, &ms);
        if (!e && best_ms) *best_ms = ms;
        return e;
    }
    // the default first; another shape must beat the best so far by 2 % (the
    // run-to-run spread of one candidate's timing) to replace it
    const ApplyShape def = apply_default(n, prec);
    std::vector<ApplyShape> cands{def};
    for (int sw : {16, 24, 32, 40, 48, 64, 96, 128, n})
        for (int tg : {128, 256, 512})
            for (int un : {4, 8}) cands.push_back({sw, tg, un});
    std::vector<std::array<int, 4>> seen;
    double best = std::numeric_limits<double>::max();
    ApplyShape bestc = def;
    for (const ApplyShape &c : cands) {
        if (!apply_shape_set(M, prec, c)) continue;
        const std::array<int, 4> key{M->slices, M->slice_w, M->shape[prec].T, M->unroll};
        if (std::find(seen.begin(), seen.end(), key) != seen.end()) continue;
        seen.push_back(key);
        e = prec_part_fit(ctx, M);
        double ms = 0.0;
        if (!e) e = time_on_stream(ctx, sc.e0, sc.e1, reps,
                                   [&] { return launch_ilu_apply(ctx, M, A, sc.v, sc.z); }, &ms);
        if (e) {
            (void)apply_shape_set(M, prec, bestc);
            return e;
        }
        if (ms < 0.98 * best || best == std::numeric_limits<double>::max()) { best = ms; bestc = c; }
    }
    if (!apply_shape_set(M, prec, bestc)) return cdg_fail(ctx, CDG_ERR_STATE, "tuned shape no longer fits");
    e = prec_part_fit(ctx, M);
    if (e) return e;
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_apply_tuned[{n, prec}] = bestc;
    }
    if (best_ms) *best_ms = best;
    return CDG_OK;
}

extern "C" int cdg_mat_tune(cdg_ctx *ctx, cdg_mat *A, int32_t reps, double *best_ms) {
    if (!ctx || !A) return CDG_ERR_ARG;
    if (best_ms) *best_ms = 0.0;
    if (A->nrows == 0) return CDG_OK;
    reps = std::max(1, std::min<int32_t>(reps, 1000));
    Scratch sc(ctx);
    int e = sc.init((int64_t)A->nrows * A->n);
    if (e) return e;
    // the default first; another shape must beat the best so far by 2 %
    const MvShape def = mv_default();
    std::vector<MvShape> cands{def};
    for (int tg : {128, 256, 384, 540, 768, 1024})
        for (int un : {4, 8, 16}) cands.push_back({tg, un});
    // (where the flat kernel runs, the loads in flight are its own: the default's number stays)
    std::vector<std::array<int, 2>> seen;
    double best = std::numeric_limits<double>::max();
    const StreamShape keep = A->shape64;
    const int32_t keep_u = A->mv_unroll;
    MvShape bestc{0, keep_u};
    StreamShape bests = keep;
    for (const MvShape &cand : cands) {
        const int tg = cand.target, un = cand.unroll;
        const StreamShape sh = stream_shape(A->n, 2, tg);
        if (sh.T == 0 || (un != def.unroll && mv_flat(ctx, A, sh))) continue;
        const std::array<int, 2> key{sh.T, un};
        if (std::find(seen.begin(), seen.end(), key) != seen.end()) continue;
        seen.push_back(key);
        A->shape64 = sh;
        A->mv_unroll = un;
        double ms = 0.0;
        e = time_on_stream(ctx, sc.e0, sc.e1, reps, [&] { return launch_mv(ctx, A, sc.v, sc.z); }, &ms);
        if (e) {
            A->shape64 = keep;
            A->mv_unroll = keep_u;
            return e;
        }
        if (ms < 0.98 * best || best == std::numeric_limits<double>::max()) { best = ms; bestc = {tg, un}; bests = sh; }
    }
    A->shape64 = bests;
    A->mv_unroll = bestc.unroll;
    if (bestc.target > 0) {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_mv_tuned[A->n] = bestc;
    }
    if (best_ms) *best_ms = best;
    return CDG_OK;
}

extern "C" int cdg_prec_launch_shape(const cdg_prec *M, int32_t *out) {
    if (!M || !out) return CDG_ERR_ARG;
    out[0] = M->slices;
    out[1] = M->slice_w;
    out[2] = M->shape[M->precision].T;
    out[3] = M->unroll;
    return CDG_OK;
}

extern "C" int cdg_mat_launch_shape(const cdg_mat *A, int32_t *out) {
    if (!A || !out) return CDG_ERR_ARG;
    out[0] = A->shape64.T;
    out[1] = A->mv_unroll;
    return CDG_OK;
}

// An abandoned wait left NaN in z and raised its preconditioner's word (call when the stream is idle).
int sweep_check(cdg_ctx *ctx, cdg_prec *M) {
    if (M->h_err && __atomic_exchange_n(M->h_err, 0u, __ATOMIC_ACQ_REL) != 0)
        return cdg_fail(ctx, CDG_ERR_HIP, "ILU(0) sweep gave up waiting for a dependency");
    return CDG_OK;
}

// A dataflow sweep that gave up waiting leaves its counters unusable: report
// it and reset them (called from the synchronizing entry points).
static int df_check(cdg_ctx *ctx, cdg_prec *M) {
    if (int e = sweep_check(ctx, M)) return e;
    if (M->apply_mode != CDG_APPLY_DATAFLOW || !M->d_dferr) return CDG_OK;
    int32_t err = 0;
    CDG_HIP_TRY(hipMemcpyAsync(&err, M->d_dferr, sizeof(err), hipMemcpyDeviceToHost, ctx->stream));
    CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (!err) return CDG_OK;
    int e = df_reset(ctx, M);
    if (e) return e;
    return cdg_fail(ctx, CDG_ERR_HIP, "ILU(0) dataflow sweep gave up waiting for a dependency; counters reset");
}

extern "C" int cdg_prec_update(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, int32_t *bad_row) {
    if (!ctx || !M || !A) return CDG_ERR_ARG;
    if (bad_row) *bad_row = -1;
    if (A->nrows != M->nrows || A->n != M->n) return cdg_fail(ctx, CDG_ERR_ARG, "matrix does not match preconditioner");
    if (M->type == CDG_PREC_IDENTITY) { M->stamp = A->stamp; M->factored = 1; return CDG_OK; }
    M->factored = 0;
    M->w_ready = 0;
    M->w_asked = 0;
    M->prev_napply = M->napply;
    M->napply = 0;
    int e = launch_ilu_factor(ctx, M, A, bad_row);
    if (e) return e;
    M->stamp = A->stamp;
    M->factored = 1;
    return M->w_keep ? sweep_fold(ctx, M, A) : CDG_OK;
}

// W of the current factor, formed once per factor (kernels only).  Under capture the launch that
// forms it belongs to the graph: it has not run yet, so the next eager apply forms W itself; and
// as a captured apply may also read a W that is there already, updates form it from then on.
int sweep_fold(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    CDG_HIP_TRY(hipStreamIsCapturing(ctx->stream, &cap));
    const bool captured = cap != hipStreamCaptureStatusNone;
    if (captured) M->w_keep = 1;
    if (M->w_ready) return CDG_OK;
    int e = launch_fold_left(ctx, M, A);
    if (!e && !captured) M->w_ready = 1;
    return e;
}

// The sweep for k vectors, in the form that M's schedule and history ask for.  Several vectors and
// the schedules STREAM and ROWSLICE take W where there is one.
static int prec_sweep(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const double *v, double *z, int64_t len, int k) {
    const bool fold = takes_w(M, k);
    if (M->fold_ok) {
        M->napply += k;
        if (k > 1 || M->apply_mode == CDG_APPLY_STREAM || M->apply_mode == CDG_APPLY_ROWSLICE) M->w_asked = 1;
    }
    if (fold) {
        int e = sweep_fold(ctx, M, A);
        if (e) return e;
    }
    return launch_ilu_sweep(ctx, M, A, v, z, len, k, fold);
}

static int prec_apply_dev(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const double *v, double *z) {
    const int64_t len = (int64_t)M->nrows * M->n;
    if (M->type == CDG_PREC_IDENTITY) return kv_copy(ctx, len, v, z);
    if (!M->factored) return cdg_fail(ctx, CDG_ERR_STATE, "ILU0 apply before update");
    if (M->apply_mode == CDG_APPLY_DATAFLOW) return launch_ilu_apply_df(ctx, M, A, v, z);
    // one persistent sweep for every schedule but FOLDED; patterns it does not
    // take (more blocks in a row than a task record holds) use level launches
    if (M->apply_mode != CDG_APPLY_FOLDED && M->sweep_ok) return prec_sweep(ctx, M, A, v, z, len, 1);
    const bool fold_now = !M->w_ready && M->apply_mode == CDG_APPLY_FOLDED;   // schedule chosen after the factor
    if (fold_now) {
        if (!M->W) {
            const size_t bytes = std::max<size_t>(16, (M->precision == CDG_FP64 ? 8 : 4) * (size_t)M->nup * M->ld);
            int e = dev_alloc(ctx, &M->W, bytes);
            if (e) return e;
            M->owned.push_back({M->W, bytes});
        }
        int e = launch_fold_all(ctx, M, A);
        if (e) return e;
        M->w_ready = 1;
    }
    int e = prec_part_fit(ctx, M);   // (there, unless the tuned shape has grown)
    if (e) return e;
    return launch_ilu_apply(ctx, M, A, v, z);
}

extern "C" int cdg_prec_apply(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const double *v, double *z) {
    if (!ctx || !M || !A || !v || !z) return CDG_ERR_ARG;
    const int64_t len = (int64_t)M->nrows * M->n;
    VecArg vi, zo;
    int e = stage_in(ctx, 0, v, len, vi);
    if (!e) e = stage_in(ctx, 1, z, len, zo);
    if (!e) e = upload_in(ctx, vi);
    if (!e) e = prec_apply_dev(ctx, M, A, vi.dev, zo.dev);
    if (!e) e = finish_out(ctx, zo);
    if (!e) e = df_check(ctx, M);
    return e;
}

extern "C" int cdg_prec_apply_async(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const double *v, double *z) {
    if (!ctx || !M || !A || !v || !z) return CDG_ERR_ARG;
    if (!is_device_ptr(v) || !is_device_ptr(z)) return cdg_fail(ctx, CDG_ERR_ARG, "cdg_prec_apply_async needs device pointers");
    return prec_apply_dev(ctx, M, A, v, z);
}

extern "C" int cdg_prec_download(cdg_ctx *ctx, const cdg_prec *M, double *L, double *Dinv) {
    if (!ctx || !M) return CDG_ERR_ARG;
    if (M->type != CDG_PREC_ILU0 || !M->factored) return cdg_fail(ctx, CDG_ERR_STATE, "no ILU0 factor to download");
    const size_t nn = (size_t)M->n * M->n;
    double *tmp = nullptr;
    const int64_t cnt = (int64_t)std::max(M->nlo, M->nrows) * M->ld;
    int e = dev_alloc(ctx, (void **)&tmp, sizeof(double) * std::max<int64_t>(cnt, 1));
    if (e) return e;
    std::vector<double> h((size_t)std::max<int64_t>(cnt, 1));
    const size_t es = M->precision == CDG_FP64 ? 8 : (M->precision == CDG_FP32 ? 4 : 2);
    auto fetch = [&](const void *src, int nslots, auto put) -> int {
        if (nslots == 0) return CDG_OK;
        int ee = launch_widen(ctx, src, M->precision, tmp, (int64_t)nslots * M->ld);
        if (ee) return ee;
        CDG_HIP_TRY(hipMemcpyAsync(h.data(), tmp, sizeof(double) * (size_t)nslots * M->ld, hipMemcpyDeviceToHost, ctx->stream));
        CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
        for (int s = 0; s < nslots; ++s) put(s, h.data() + (size_t)s * M->ld);
        return CDG_OK;
    };
    (void)es;
    // slot q of L belongs to the q-th lower block in pattern order
    std::vector<int32_t> lo_blk_host;
    // The prec does not keep the pattern; recover block indices from the device copy.
    if (M->nlo) {
        lo_blk_host.resize(M->nlo);
        hipError_t he = hipMemcpy(lo_blk_host.data(), M->d_lo_blk, sizeof(int32_t) * M->nlo, hipMemcpyDeviceToHost);
        if (he != hipSuccess) { dev_free(ctx, tmp, sizeof(double) * cnt); return cdg_fail(ctx, CDG_ERR_HIP, "%s", hipGetErrorString(he)); }
    }
    if (L) {
        e = fetch(M->L, M->nlo, [&](int q, const double *src) {
            std::memcpy(L + (size_t)lo_blk_host[q] * nn, src, sizeof(double) * nn);
        });
    }
    if (!e && Dinv) {
        e = fetch(M->Dinv, M->nrows, [&](int i, const double *src) {
            std::memcpy(Dinv + (size_t)i * nn, src, sizeof(double) * nn);
        });
    }
    dev_free(ctx, tmp, sizeof(double) * std::max<int64_t>(cnt, 1));
    return e;
}

// ---------------------------------------------------------------------------
// FGMRES (type_fgmres.f90:81-310)
// ---------------------------------------------------------------------------
extern "C" void cdg_fgmres_default_params(cdg_fgmres_params *p) {
    if (!p) return;
    p->nkrylov = 2000;
    p->tol = 1.e-8;
    p->rtol = 1.e-10;
    p->nmax = -1;
    p->orthogonalization = CDG_CGS;
    p->inner_fgmres = 1;
    p->inner_nkrylov = 100;
    p->inner_tol = 1.e-1;
    p->inner_rtol = 1.e-1;
    p->inner_nmax = 100;
    p->inner_orthogonalization = CDG_CGS;
    p->update_preconditioner = 1;
}

namespace {

using clk = std::chrono::steady_clock;
double secs(clk::time_point a, clk::time_point b) { return std::chrono::duration<double>(b - a).count(); }

// One FGMRES level (outer, or the nested inner one): basis, search directions and
// the step kernel's state for k right-hand sides in lockstep.  Vectors are laid
// out V[(j k + r) len], Z likewise.
struct Level {
    int m = 0, k = 0;
    int64_t len = 0;
    bool inner_bufs = false;
    double *V = nullptr, *Z = nullptr, *r0 = nullptr, *x0 = nullptr, *zr = nullptr, *dz = nullptr;
    size_t bytes = 0;
    void *base = nullptr;
    Arnoldi arn;
};

void level_free(cdg_ctx *ctx, Level &lv) {
    if (lv.base) dev_free(ctx, lv.base, lv.bytes);
    arn_free(ctx, lv.arn);
    lv = Level();
}

int level_alloc(cdg_ctx *ctx, Level &lv, int m, int k, int64_t len, bool inner_bufs, bool mgs) {
    lv.m = m;
    lv.k = k;
    lv.len = len;
    lv.inner_bufs = inner_bufs;
    const size_t kl = (size_t)std::max<int64_t>(len, 1) * k;
    lv.bytes = (2 * (size_t)(m + 1) + 2 + (inner_bufs ? 2 : 0)) * kl * sizeof(double);
    int e = dev_alloc(ctx, &lv.base, lv.bytes);
    if (e) return e;
    double *p = static_cast<double *>(lv.base);
    lv.V = p; p += (size_t)(m + 1) * kl;
    lv.Z = p; p += (size_t)(m + 1) * kl;
    lv.r0 = p; p += kl;
    lv.x0 = p; p += kl;
    if (inner_bufs) { lv.zr = p; p += kl; lv.dz = p; p += kl; }
    return arn_alloc(ctx, lv.arn, k, m, len, mgs);
}

// Pinned results of the step launches: two levels of up to k lanes.
int arn_results(cdg_ctx *ctx, int k) {
    if (ctx->arn_cap >= 2 * k) return CDG_OK;
    CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (ctx->h_arn) (void)hipHostFree(ctx->h_arn);
    ctx->h_arn = nullptr;
    ctx->arn_cap = 0;
    if (hipHostMalloc((void **)&ctx->h_arn, sizeof(ArnRes) * 2 * k) != hipSuccess)
        return cdg_fail(ctx, CDG_ERR_OOM, "pinned results of %d right-hand sides", k);
    std::memset(ctx->h_arn, 0, sizeof(ArnRes) * 2 * k);
    ctx->arn_cap = 2 * k;
    return CDG_OK;
}

// Waits until launch `seq` has reported every lane: polls pinned memory (no
// HIP call on the way), and after 5 ms waits for the stream.
int arn_wait(cdg_ctx *ctx, const ArnRes *res, int k, uint32_t seq) {
    const auto t0 = clk::now();
    auto all = [&] {
        for (int r = 0; r < k; ++r)
            if ((int32_t)((uint32_t)(__atomic_load_n(&res[r].word, __ATOMIC_ACQUIRE) >> 32) - seq) < 0) return false;
        return true;
    };
    for (int spins = 0; ctx->spin; ++spins) {
        if (all()) return CDG_OK;
        if ((spins & 255) == 255 && clk::now() - t0 > std::chrono::milliseconds(5)) break;
    }
    CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    return all() ? CDG_OK : cdg_fail(ctx, CDG_ERR_HIP, "an FGMRES step ended without its result");
}

struct Solver {
    cdg_ctx *ctx;
    const cdg_mat *A;
    cdg_prec *M;
    int64_t len;
};

// fetch n device scalars from ctx->d_small into ctx->h_small
int fetch_small(cdg_ctx *ctx, size_t n) {
    CDG_HIP_TRY(hipMemcpyAsync(ctx->h_small, ctx->d_small, sizeof(double) * n, hipMemcpyDeviceToHost, ctx->stream));
    return ctx_wait(ctx);
}

// z_r = M^-1 v_r for r < k (vectors `len` apart): the k-vector sweep for
// ILU(0), else one apply per vector.
int prec_apply_multi(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const double *v, double *z, int64_t len, int k) {
    if (M->type == CDG_PREC_IDENTITY) return kv_copy(ctx, len * k, v, z);
    if (!M->factored) return cdg_fail(ctx, CDG_ERR_STATE, "ILU0 apply before update");
    if (k > 1 && M->sweep_ok) return prec_sweep(ctx, M, A, v, z, len, k);
    for (int r = 0; r < k; ++r) {
        int e = prec_apply_dev(ctx, M, A, v + (size_t)r * len, z + (size_t)r * len);
        if (e) return e;
    }
    return CDG_OK;
}

// The outer FGMRES of fgmres_t%solve (type_fgmres.f90:81-310) for k right-hand
// sides in lockstep: independent Arnoldi processes, rotations, residual
// estimates and stopping tests (on the device, k_arnoldi.hip) whose steps share one
// k-vector apply and one k-vector matvec; a right-hand side that stops waits
// for the others' cycle to end.  B and X: k vectors `len` apart.  With `inner`
// (k = 1) every search direction gets the nested FGMRES correction (:179-183).
//
// The host queues one step ahead of the last one it has seen end: the kernels of a
// step queued after every lane stopped return at once (the sweep and the matvec
// look at the count of running lanes).
int fgmres_lanes(Solver &S, std::vector<Level> &lvs, int depth, int k, const double *B, double *X, int m, double tol,
                 double rtol, int nmax, int orth, const cdg_fgmres_params *inner, std::vector<int> &nrestart) {
    cdg_ctx *ctx = S.ctx;
    const int64_t len = S.len, kl = (int64_t)k * len;
    if (m < 1) return cdg_fail(ctx, CDG_ERR_ARG, "nkrylov must be >= 1");
    if (depth >= (int)lvs.size()) return cdg_fail(ctx, CDG_ERR_ARG, "FGMRES nesting deeper than one inner level");
    Level &lv = lvs[depth];   // lvs is never resized during a solve
    const bool mgs = orth == CDG_MGS;
    if (lv.m != m || lv.len != len || lv.k != k || (inner && !lv.inner_bufs) || lv.arn.mgs != mgs) {
        level_free(ctx, lv);
        int e = level_alloc(ctx, lv, m, k, len, inner != nullptr, mgs);
        if (e) return e;
    }
    ArnArgs &a = lv.arn.a;
    ArnRes *const res = ctx->h_arn + (size_t)depth * (ctx->arn_cap / 2);
    a.hres = res;
    a.tol = tol;
    a.rtol = rtol;
    a.nmax = nmax;
    a.V = lv.V;
    // steps queued past the last one seen: with the sweep, which stops early
    const int ahead = !inner && S.M->type == CDG_PREC_ILU0 && S.M->sweep_ok &&
                      S.M->apply_mode != CDG_APPLY_FOLDED && S.M->apply_mode != CDG_APPLY_DATAFLOW ? 1 : 0;
    std::vector<char> done(k, 0), ended(k, 0);   // ended: by the stopping test
    std::vector<uint32_t> seqs;
    int e = CDG_OK;
    for (bool first = true;; first = false) {
        // r0 = b - A x0, v1 = r0 / ||r0||, p1 = ||r0||   (:160-163); x0 = 0 in the first cycle
        a.first = first;
        a.b = B;
        a.ax = first ? nullptr : lv.r0;
        a.w = lv.V;
        if (!first) e = k == 1 ? launch_mv(ctx, S.A, lv.x0, lv.r0) : launch_mv_multi(ctx, S.A, lv.x0, lv.r0, len, k);
        if (!e) e = arn_launch(ctx, lv.arn, ARN_START, 0);
        if (e) return e;
        seqs.assign(1, a.seq);
        std::fill(ended.begin(), ended.end(), 0);
        bool stopped = false;
        size_t seen = 0;
        auto see = [&](size_t upto) -> int {   // results of launches [seen, upto)
            for (; seen < upto && !stopped; ++seen) {
                int e2 = arn_wait(ctx, res, k, seqs[seen]);
                if (e2) return e2;
                bool any = false;
                for (int r = 0; r < k; ++r) {
                    if (done[r]) continue;
                    if (res[r].word & ARN_W_ERR)
                        return cdg_fail(ctx, CDG_ERR_NAN, "non-finite FGMRES residual (vector %d)", r);
                    // (a launch after a lane's last step reports again how it ended)
                    ended[r] = (res[r].word & ARN_W_DONE) != 0;
                    any |= (res[r].word & ARN_W_ACTIVE) != 0;
                }
                stopped = !any;
            }
            return CDG_OK;
        };
        if (!ahead) e = see(1);
        if (e) return e;
        for (int j = 0; j < m && !stopped; ++j) {
            double *vj = lv.V + (size_t)j * kl, *zj = lv.Z + (size_t)j * kl, *wj = lv.V + (size_t)(j + 1) * kl;
            ctx->hook_nact = ahead ? a.nact : nullptr;
            ctx->hook_stamp = a.stamp;
            if (!ahead) e = arn_stamp(ctx, lv.arn, 0);
            if (!e) e = k == 1 ? prec_apply_dev(ctx, S.M, S.A, vj, zj) : prec_apply_multi(ctx, S.M, S.A, vj, zj, len, k);
            if (inner && !e) {
                // zr = v_j - A z_j ; inner solve ; z_j += dz   (:179-183)
                ctx->hook_nact = nullptr;
                ctx->hook_stamp = nullptr;
                std::vector<int> nr(1, 0);                 // (its restarts are not reported)
                e = launch_mv(ctx, S.A, zj, lv.zr);
                if (!e) e = kv_sub(ctx, len, vj, lv.zr, lv.zr);
                if (!e) e = fgmres_lanes(S, lvs, depth + 1, 1, lv.zr, lv.dz, inner->inner_nkrylov, inner->inner_tol,
                                         inner->inner_rtol, inner->inner_nmax, inner->inner_orthogonalization, nullptr, nr);
                if (!e) e = kv_add(ctx, len, zj, lv.dz);
                ctx->hook_stamp = a.stamp;
            }
            // w = A z_j, written into the slot of v_{j+1}   (:189)
            if (!e) e = k == 1 ? launch_mv(ctx, S.A, zj, wj) : launch_mv_multi(ctx, S.A, zj, wj, len, k);
            ctx->hook_nact = nullptr;
            ctx->hook_stamp = nullptr;
            a.w = wj;
            if (!e) e = arn_launch(ctx, lv.arn, mgs ? ARN_MGS : ARN_CGS, j + 1);
            if (e) return e;
            seqs.push_back(a.seq);
            e = see(seqs.size() - ahead);
            if (e) return e;
        }
        e = see(seqs.size());
        if (!e && S.M->fold_ok) {   // applies that were queued after every lane had stopped did not happen
            int steps = 0;
            for (int r = 0; r < k; ++r)
                if (!done[r]) steps = std::max(steps, (int)((uint32_t)res[r].word >> ARN_W_BITS));
            S.M->napply -= k * ((int)seqs.size() - 1 - steps);
        }
        // x = x0 + Z y   (:287-295); stopped lanes are done, the others restart
        if (!e) e = arn_cycle_end(ctx, lv.arn, lv.Z, X, lv.x0, first);
        if (e) return e;
        bool all = true;
        for (int r = 0; r < k; ++r) {
            if (done[r]) continue;
            done[r] = ended[r];
            if (!done[r]) { nrestart[r]++; all = false; }
        }
        if (all) return CDG_OK;
    }
}

// k right-hand sides of one system: the solves, the true residuals, the statistics.
int solve_lanes(cdg_ctx *ctx, const cdg_mat *A, cdg_prec *M, int k, const double *b, double *x,
                const cdg_fgmres_params *prm, cdg_fgmres_stats *st) {
    auto t_start = clk::now();
    int e = CDG_OK;
    double t_factor = 0.0;
    int factored = 0;
    // M%update(A,b) when the controller asks (type_fgmres.f90:118-122)
    if (prm->update_preconditioner || !M->factored || M->stamp != A->stamp) {
        auto tf = clk::now();
        e = cdg_prec_update(ctx, M, A, nullptr);
        if (e) return e;
        factored = 1;
        t_factor = secs(tf, clk::now());
    }
    const int64_t len = (int64_t)A->nrows * A->n;
    if (len == 0) {   // no rows: x = (), nothing to launch (the step's kernels need a value)
        if (prm->nkrylov < 1) return cdg_fail(ctx, CDG_ERR_ARG, "nkrylov must be >= 1");
        for (int r = 0; r < k; ++r) {
            std::memset(&st[r], 0, sizeof(st[r]));
            st[r].factored = factored;
            st[r].t_factor = t_factor;
            st[r].t_total = secs(t_start, clk::now());
        }
        return CDG_OK;
    }
    VecArg bi, xo;
    e = stage_in(ctx, 0, b, len * k, bi);
    if (!e) e = stage_in(ctx, 1, x, len * k, xo);
    if (!e) e = upload_in(ctx, bi);
    if (!e) e = arn_results(ctx, k);
    if (e) return e;
    Solver S{ctx, A, M, len};
    std::vector<Level> lvs(2);   // outer and inner level
    std::vector<int> nrestart(k, 0);
    e = fgmres_lanes(S, lvs, 0, k, bi.dev, xo.dev, prm->nkrylov, prm->tol, prm->rtol, prm->nmax, prm->orthogonalization,
                     prm->inner_fgmres ? prm : nullptr, nrestart);
    ctx->hook_nact = nullptr;
    ctx->hook_stamp = nullptr;
    // residual_norm = ||b - A x||   (type_fgmres.f90:305,515)
    Level &lv = lvs[0];
    if (!e) e = k == 1 ? launch_mv(ctx, A, xo.dev, lv.r0) : launch_mv_multi(ctx, A, xo.dev, lv.r0, len, k);
    if (!e) {
        lv.arn.a.b = bi.dev;
        lv.arn.a.ax = lv.r0;
        lv.arn.a.inner_st = lvs[1].arn.a.st;
        e = arn_launch(ctx, lv.arn, ARN_NORM, 0);
    }
    if (!e) e = arn_wait(ctx, ctx->h_arn, k, lv.arn.a.seq);
    // the last launch has reported, so every earlier one has ended: x is complete
    if (!e && xo.host) e = finish_out(ctx, xo);
    const double t_total = secs(t_start, clk::now());
    int khz = 100000;
    (void)hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, ctx->device);
    const double tick = 1e-3 / std::max(1, khz);
    for (int r = 0; r < k && !e; ++r) {
        const ArnRes &o = ctx->h_arn[r];
        cdg_fgmres_stats &q = st[r];
        std::memset(&q, 0, sizeof(q));
        q.niter = o.niter;
        q.residual_norm = o.res;
        q.nrestart = nrestart[r];
        q.nreorth = o.nreorth;
        q.factored = factored;
        q.t_total = t_total;
        q.t_factor = t_factor;
        q.t_precon = o.t[0] * tick;
        q.t_mv = o.t[1] * tick;
        q.t_dot = o.t[2] * tick;
        q.t_norm = o.t[3] * tick;
    }
    for (int r = 0; r < k && !e; ++r)
        if (!std::isfinite(st[r].residual_norm)) e = cdg_fail(ctx, CDG_ERR_NAN, "non-finite final residual");
    for (Level &l : lvs) level_free(ctx, l);
    if (e == CDG_ERR_NAN) {   // a sweep that gave up left NaN behind
        const int e2 = df_check(ctx, M);
        if (e2) return e2;
    }
    return e;
}

}  // namespace

extern "C" int cdg_fgmres_solve(cdg_ctx *ctx, const cdg_mat *A, cdg_prec *M, const double *b, double *x,
                                const cdg_fgmres_params *prm, cdg_fgmres_stats *st) {
    if (!ctx || !A || !M || !b || !x || !prm) return CDG_ERR_ARG;
    if (A->nrows != M->nrows || A->n != M->n) return cdg_fail(ctx, CDG_ERR_ARG, "matrix does not match preconditioner");
    cdg_fgmres_stats local;
    std::memset(st ? st : &local, 0, sizeof(local));
    return solve_lanes(ctx, A, M, 1, b, x, prm, st ? st : &local);
}

extern "C" int cdg_fgmres_solve_multi(cdg_ctx *ctx, const cdg_mat *A, cdg_prec *M, int32_t k, const double *b, double *x,
                                      const cdg_fgmres_params *prm, cdg_fgmres_stats *st) {
    if (!ctx || !A || !M || !b || !x || !prm || k < 1) return CDG_ERR_ARG;
    if (A->nrows != M->nrows || A->n != M->n) return cdg_fail(ctx, CDG_ERR_ARG, "matrix does not match preconditioner");
    const int64_t len = (int64_t)A->nrows * A->n;
    if (k == 1 || prm->inner_fgmres) {   // one vector, or nested FGMRES: one solve per vector
        for (int r = 0; r < k; ++r) {
            cdg_fgmres_params p1 = *prm;
            if (r > 0) p1.update_preconditioner = 0;   // the first solve's factor serves the others
            int e = cdg_fgmres_solve(ctx, A, M, b + (size_t)r * len, x + (size_t)r * len, &p1, st ? st + r : nullptr);
            if (e) return e;
        }
        return CDG_OK;
    }
    std::vector<cdg_fgmres_stats> local(k);
    // the step's kernels have a grid row per vector: 65535 at most
    constexpr int32_t kMost = 32768;
    int e = CDG_OK;
    for (int32_t r = 0; r < k && !e; r += kMost) {
        cdg_fgmres_params p1 = *prm;
        if (r > 0) p1.update_preconditioner = 0;
        e = solve_lanes(ctx, A, M, std::min(kMost, k - r), b + (size_t)r * len, x + (size_t)r * len, &p1, local.data() + r);
    }
    if (st) std::memcpy(st, local.data(), sizeof(cdg_fgmres_stats) * k);
    return e;
}

extern "C" int cdg_mv_multi(cdg_ctx *ctx, const cdg_mat *A, int32_t k, const double *X, double *Y) {
    if (!ctx || !A || !X || !Y || k < 1) return CDG_ERR_ARG;
    const int64_t len = (int64_t)A->nrows * A->n;
    VecArg xi, yo;
    int e = stage_in(ctx, 0, X, len * k, xi);
    if (!e) e = stage_in(ctx, 1, Y, len * k, yo);
    if (!e) e = upload_in(ctx, xi);
    if (!e) e = launch_mv_multi(ctx, A, xi.dev, yo.dev, len, k);
    if (!e) e = finish_out(ctx, yo);
    return e;
}

extern "C" int cdg_prec_apply_multi(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, int32_t k, const double *V, double *Z) {
    if (!ctx || !M || !A || !V || !Z || k < 1) return CDG_ERR_ARG;
    if (A->nrows != M->nrows || A->n != M->n) return cdg_fail(ctx, CDG_ERR_ARG, "matrix does not match preconditioner");
    const int64_t len = (int64_t)A->nrows * A->n;
    VecArg vi, zo;
    int e = stage_in(ctx, 0, V, len * k, vi);
    if (!e) e = stage_in(ctx, 1, Z, len * k, zo);
    if (!e) e = upload_in(ctx, vi);
    if (!e) e = prec_apply_multi(ctx, M, A, vi.dev, zo.dev, len, k);
    if (!e) e = finish_out(ctx, zo);
    if (!e) e = df_check(ctx, M);
    return e;
}

// ---- device-resident vectors (chidg_vector_t operations, type_chidg_vector.f90) ----
extern "C" int cdg_vec_create(cdg_ctx *ctx, int64_t len, double **out) {
    if (!ctx || !out || len < 0) return CDG_ERR_ARG;
    *out = nullptr;
    CDG_HIP_TRY(hipSetDevice(ctx->device));
    void *p = nullptr;
    int e = dev_alloc(ctx, &p, sizeof(double) * (size_t)std::max<int64_t>(len, 1));
    if (!e) e = kv_zero(ctx, len, static_cast<double *>(p));
    if (!e) e = ctx_wait(ctx);
    if (e) { if (p) dev_free(ctx, p, 0); return e; }
    *out = static_cast<double *>(p);
    return CDG_OK;
}

extern "C" int cdg_vec_destroy(cdg_ctx *ctx, double *v) {
    if (!ctx) return CDG_ERR_ARG;
    if (v) {
        CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
        dev_free(ctx, v, 0);
    }
    return CDG_OK;
}

extern "C" int cdg_vec_copy(cdg_ctx *ctx, int64_t len, const double *src, double *dst) {
    if (!ctx || !src || !dst || len < 0) return CDG_ERR_ARG;
    CDG_HIP_TRY(hipMemcpyAsync(dst, src, sizeof(double) * (size_t)len, hipMemcpyDefault, ctx->stream));
    return ctx_wait(ctx);
}

extern "C" int cdg_vec_axpby(cdg_ctx *ctx, int64_t len, double a, const double *x, double b, double *y) {
    if (!ctx || !x || !y || len < 0) return CDG_ERR_ARG;
    if (!is_device_ptr(x) || !is_device_ptr(y)) return cdg_fail(ctx, CDG_ERR_ARG, "cdg_vec_axpby needs device pointers");
    int e = kv_axpby(ctx, len, a, x, b, y);
    if (!e) e = ctx_wait(ctx);
    return e;
}

extern "C" int cdg_vec_dot(cdg_ctx *ctx, int64_t len, const double *x, const double *y, double *out) {
    if (!ctx || !x || !y || !out || len < 0) return CDG_ERR_ARG;
    VecArg xi, yi;
    int e = stage_in(ctx, 0, x, len, xi);
    if (!e) e = stage_in(ctx, 1, y, len, yi);
    if (!e) e = upload_in(ctx, xi);
    if (!e) e = upload_in(ctx, yi);
    if (!e) e = kv_multidot(ctx, len, xi.dev, yi.dev, len, 1, ctx->d_small);
    if (!e) e = fetch_small(ctx, 1);
    if (!e) *out = ctx->h_small[0];
    return e;
}

extern "C" int cdg_vec_norm(cdg_ctx *ctx, int64_t len, const double *x, double *out) {
    if (!ctx || !x || !out || len < 0) return CDG_ERR_ARG;
    VecArg xi;
    int e = stage_in(ctx, 0, x, len, xi);
    if (!e) e = upload_in(ctx, xi);
    if (!e) e = kv_sumsq(ctx, len, xi.dev, ctx->d_small);
    if (!e) e = fetch_small(ctx, 1);
    if (!e) *out = std::sqrt(ctx->h_small[0]);
    return e;
}

// ---- DG Euler residual on the device (mod_spatial.f90:40-197) ----------------
extern "C" int cdg_euler_residual_gpu(cdg_ctx *ctx, int32_t nx, int32_t ny, int32_t nz, int32_t order, const double *q,
                                      double *R) {
    if (!ctx || !q || !R) return CDG_ERR_ARG;
    if (nx < 2 || nx > 256 || ny != nx || nz != nx || order < 0 || order > 3) return CDG_ERR_ARG;
    const int64_t len = (int64_t)nx * ny * nz * 5 * (order + 1) * (order + 1) * (order + 1);
    VecArg qi, ro;
    int e = stage_in(ctx, 0, q, len, qi);
    if (!e) e = stage_in(ctx, 1, R, len, ro);
    if (!e) e = upload_in(ctx, qi);
    if (!e) e = launch_euler_residual(ctx, nx, ny, nz, order, qi.dev, ro.dev);
    if (!e) e = finish_out(ctx, ro);
    if (!e) {   // a state with negative pressure gives a non-finite residual, as on the host
        e = kv_sumsq(ctx, len, ro.dev, ctx->d_small);
        if (!e) e = fetch_small(ctx, 1);
        if (!e && !std::isfinite(ctx->h_small[0])) e = cdg_fail(ctx, CDG_ERR_NAN, "non-finite Euler residual");
    }
    return e;
}
