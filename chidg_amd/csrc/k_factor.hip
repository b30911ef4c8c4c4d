// ILU(0) factorization kernels for gfx950 (precon_ILU0.f90:111-265).
//
// Rows are processed in wavefront levels (rows of one level are independent).
// Per level:
//   phase 1  L_ij = A_ij * Dinv_j            batched GEMM on MFMA (one job per lower block)
//   phase 2  D_i  = A_ii - sum_j L_ij A_ji   batched GEMM on MFMA (one job per row)
//   phase 3  Dinv_i = inv(D_i)               one workgroup per block, register-resident
//                                            Gauss-Jordan with partial (row) pivoting
// FP64 uses v_mfma_f64_16x16x4f64, FP32 v_mfma_f32_16x16x4f32.  A 48x48 output
// tile per workgroup (3 waves, each 16x48 = three 16x16 MFMA tiles) covers the
// block sizes 40/135/320 with little padding.
#include "cdg_internal.h"

#include <type_traits>

#include <algorithm>
#include <cstdlib>
#include <mutex>

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// 16x16x4 MFMA.  Operands: lane l supplies A[l%16][l/16] and B[l/16][l%16].
// Result row held by lane l in accumulator register r (column is l%16): the
// f64 instruction strides rows by 4 across registers, the f32 one keeps four
// consecutive rows per lane group (measured on gfx950).
template <typename T> struct Mfma;
template <> struct Mfma<double> {
    typedef f64x4 acc_t;
    __device__ static __forceinline__ acc_t run(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <> struct Mfma<float> {
    typedef f32x4 acc_t;
    __device__ static __forceinline__ acc_t run(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

constexpr int KC = 16;       // K chunk staged in LDS

// Batched block GEMM.  A workgroup of TM / 16 waves computes a TM x TM tile
// (TM = 48 or 64) of one output block, acc = sum_p A_p B_p over the
// concatenated K of its operand pairs (A_p, B_p column-major n x n); wave w
// holds rows 16w..16w+15 (TM / 16 MFMA tiles of 16 x 16).  K advances in
// chunks of KC through two LDS buffers; the global fetch of chunk c + 2 goes
// out before chunk c's products, so a fetch has two chunks of products to
// arrive.  What bounds it: in wide levels the matrix units (64 to 70 % busy in FP32 at n = 320,
// about 50 % in FP64 at n = 135, a ninth of it padding), in narrow ones one tile's chain of
// chunks.  16-byte loads kept whole in LDS, without masks inside the tile: factor of 16^3 P3
// FP32, p1 + p2, 19.8 -> 16.9 ms; 16^3 P2 FP64 5.5 -> 5.0, FP32 3.6 -> 3.25.  Chunks of 32 gain in
// narrow levels and lose more in wide ones (p1 8.6 -> 9.4 ms at P3, 2.3 -> 2.9 at P2 FP64).  The 64-edge tile serves n > 192 (320 = 5 x 64: no padding, and 16
// products per wave between barriers instead of 12).
template <int TM> struct Geo {
    static constexpr int GW = TM / 16;   // waves per workgroup
    static constexpr int GT = 64 * GW;   // threads per workgroup
};
constexpr int LE = KC / 4;    // elements per thread, chunk and operand (KC * TM / GT)
// LDS tiles as their readers take them.  As[k][r] = A(r0 + r, kc + k): a fetched vector
// of A (rows of one column) is stored whole.  Bs[c][k] = B(kc + k, c0 + c), likewise.  An
// MFMA sums over k, so lane l takes the contiguous k range (KC/4)(l/16) .. +KC/4 for both
// operands: B's in one read.
template <typename T> struct KPitch { static constexpr int P = KC + 16 / (int)sizeof(T); };
template <typename T, int TM> using ATile = T[KC][TM + 16 / (int)sizeof(T)];
template <typename T, int TM> using BTile = T[TM][KPitch<T>::P];

// 16 bytes of S from any element on
template <typename S> struct __attribute__((packed, aligned(sizeof(S)))) Vec16 { S v[16 / sizeof(S)]; };
template <typename S> constexpr int VecN = 16 / (int)sizeof(S);

// The fetch loads raw source values (SA, SB), 16 bytes at a time and with no
// conditions, so nothing waits for them here.  (A conversion at fetch time makes every
// fetch wait for its own loads.)  A vector starts at a row below n or holds no value that
// is used, and slots are padded to 64 elements, so a start clamped to the slot's last
// vector shifts none that is; rows and columns from n on only reach results that are
// not stored, and k from n on is zeroed in LDS.
template <typename S, int TM> struct Fetched { Vec16<S> v[LE / VecN<S>]; };
template <typename S, int TM>
__device__ __forceinline__ void fetch_a(const S *__restrict__ A, int n, int top, int r0, int kc, Fetched<S, TM> &f) {
    constexpr int V = VecN<S>, PC = TM / V;
#pragma unroll
    for (int i = 0; i < LE / V; ++i) {
        const int idx = threadIdx.x + Geo<TM>::GT * i, kk = idx / PC, rr = (idx - kk * PC) * V;
        f.v[i] = *reinterpret_cast<const Vec16<S> *>(reinterpret_cast<const char *>(A) +
                                                     (uint32_t)(min((kc + kk) * n + r0 + rr, top - V) * (int)sizeof(S)));
    }
}
template <typename S, int TM>
__device__ __forceinline__ void fetch_b(const S *__restrict__ B, int n, int top, int c0, int kc, Fetched<S, TM> &f) {
    constexpr int V = VecN<S>, PC = KC / V;
#pragma unroll
    for (int i = 0; i < LE / V; ++i) {
        const int idx = threadIdx.x + Geo<TM>::GT * i, cc = idx / PC, kb = (idx - cc * PC) * V;
        f.v[i] = *reinterpret_cast<const Vec16<S> *>(reinterpret_cast<const char *>(B) +
                                                     (uint32_t)(min((c0 + cc) * n + kc + kb, top - V) * (int)sizeof(S)));
    }
}
// nk: values of k in the chunk (less than KC in an operand's last one)
template <typename T, typename S, int TM>
__device__ __forceinline__ void store_a(ATile<T, TM> &As, const Fetched<S, TM> &f, int nk) {
    constexpr int V = VecN<S>, PC = TM / V;
    typedef T out_t __attribute__((ext_vector_type(V)));
#pragma unroll
    for (int i = 0; i < LE / V; ++i) {
        const int idx = threadIdx.x + Geo<TM>::GT * i, kk = idx / PC, rr = (idx - kk * PC) * V;
        out_t o;
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = kk < nk ? static_cast<T>(f.v[i].v[e]) : T(0);
        *reinterpret_cast<out_t *>(&As[kk][rr]) = o;
    }
}
template <typename T, typename S, int TM>
__device__ __forceinline__ void store_b(BTile<T, TM> &Bs, const Fetched<S, TM> &f, int nk) {
    constexpr int V = VecN<S>, PC = KC / V;
    typedef T out_t __attribute__((ext_vector_type(V)));
#pragma unroll
    for (int i = 0; i < LE / V; ++i) {
        const int idx = threadIdx.x + Geo<TM>::GT * i, cc = idx / PC, kb = (idx - cc * PC) * V;
        out_t o;
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = kb + e < nk ? static_cast<T>(f.v[i].v[e]) : T(0);
        *reinterpret_cast<out_t *>(&Bs[cc][kb]) = o;
    }
}

template <typename T, int TM>
__device__ __forceinline__ void gemm_chunk(const ATile<T, TM> &As, const BTile<T, TM> &Bs,
                                           typename Mfma<T>::acc_t (&acc)[TM / 16]) {
    constexpr int NJ = TM / 16;
    constexpr int KS = KC / 4;                   // k values per lane and chunk
    typedef T vec_t __attribute__((ext_vector_type(KS)));
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int k0 = KS * (lane >> 4);
    T a[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) a[s] = As[k0 + s][16 * wv + (lane & 15)];
    vec_t b[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) b[j] = *reinterpret_cast<const vec_t *>(&Bs[16 * j + (lane & 15)][k0]);
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[j] = Mfma<T>::run(a[s], b[j][s], acc[j]);
}

// acc = sum over the npairs operand pairs, pair(p, A, B) naming pair p.
template <typename T, typename SA, typename SB, int TM, typename Pair>
__device__ __forceinline__ void gemm_pairs(Pair pair, int npairs, int n, int r0, int c0, ATile<T, TM> (&As)[2],
                                           BTile<T, TM> (&Bs)[2], typename Mfma<T>::acc_t (&acc)[TM / 16]) {
    // Branch-free pipeline over an even number of chunks: fetches past the
    // last chunk reload it (in bounds) and their stores write zeros, so the
    // compiler's wait counts see loads in issue order (a conditional fetch
    // makes it wait for every outstanding load at each store).
    const int cpb = (n + KC - 1) / KC, nch = npairs * cpb, nch2 = (nch + 1) & ~1;
    Fetched<SA, TM> ra0, ra1;
    Fetched<SB, TM> rb0, rb1;
    const int top = (n * n + 63) & ~63;          // a slot's elements
    auto fetch = [&](int c, Fetched<SA, TM> &ra, Fetched<SB, TM> &rb) {
        c = min(c, nch - 1);
        const int p = c / cpb;
        const SA *A;
        const SB *B;
        pair(p, A, B);
        fetch_a<SA, TM>(A, n, top, r0, (c - p * cpb) * KC, ra);
        fetch_b<SB, TM>(B, n, top, c0, (c - p * cpb) * KC, rb);
    };
    auto store = [&](int c, int buf, const Fetched<SA, TM> &ra, const Fetched<SB, TM> &rb) {
        const int nk = c < nch ? n - (c - (c / cpb) * cpb) * KC : 0;   // chunk c >= nch: zeros
        store_a<T, SA, TM>(As[buf], ra, nk);
        store_b<T, SB, TM>(Bs[buf], rb, nk);
    };
    fetch(0, ra0, rb0);
    fetch(1, ra1, rb1);
    store(0, 0, ra0, rb0);
    __syncthreads();
    for (int c = 0; c < nch2; c += 2) {
        fetch(c + 2, ra0, rb0);
        gemm_chunk<T, TM>(As[0], Bs[0], acc);
        store(c + 1, 1, ra1, rb1);
        __syncthreads();
        fetch(c + 3, ra1, rb1);
        gemm_chunk<T, TM>(As[1], Bs[1], acc);
        store(c + 2, 0, ra0, rb0);
        __syncthreads();
    }
}

// XCD-aware job/tile numbering.  Workgroups go to the 8 XCDs (each with its
// own L2) round-robin by linear id; id L runs tile (L / 8) % tiles2 of job
// 8 * ((L / 8) / tiles2) + L % 8, so all tiles of a job share one XCD's L2
// (they read the same operand strips).  Returns false for the ids past the
// last job.
__device__ __forceinline__ bool xcd_job(int njobs, int tiles2, int &job, int &tile) {
    const int L = blockIdx.x, k = L >> 3;
    job = 8 * (k / tiles2) + (L & 7);
    tile = k - (k / tiles2) * tiles2;
    return job < njobs;
}
inline int xcd_grid(int njobs, int tiles2) { return 8 * tiles2 * ((njobs + 7) / 8); }

template <typename T, int TM, typename F>
__device__ __forceinline__ void gemm_out(int tm, int tn, int n, typename Mfma<T>::acc_t (&acc)[TM / 16], F put) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < TM / 16; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = tm * TM + 16 * wv + Mfma<T>::row(lane, r);
            const int col = tn * TM + 16 * j + (lane & 15);
            if (row < n && col < n) put(row, col, acc[j][r]);
        }
}

// phase 1: L_q = A_{lo_blk[q]} * Dinv_{lo_col[q]} (with the upper lists in
// place of the lower ones: W_u = A_{up_blk[u]} * Dinv_{up_col[u]}); the A
// operand is A's own FP64 blocks or, for the FP32 fold, their FP32 copies
template <typename T, typename SA, int TM>
__global__ void __launch_bounds__(Geo<TM>::GT)
k_fac_p1(const SA *__restrict__ Ab, int64_t lda, T *__restrict__ L, const T *__restrict__ D, int64_t ld,
         const int32_t *__restrict__ jobs, int njobs, const int32_t *__restrict__ lo_blk,
         const int32_t *__restrict__ lo_col, int n, int tiles) {
    __shared__ __attribute__((aligned(16))) ATile<T, TM> As[2];
    __shared__ __attribute__((aligned(16))) BTile<T, TM> Bs[2];
    int job, tile;
    if (!xcd_job(njobs, tiles * tiles, job, tile)) return;
    const int q = jobs[job];
    const int tm = tile % tiles, tn = tile / tiles;
    typename Mfma<T>::acc_t acc[TM / 16];
#pragma unroll
    for (int j = 0; j < TM / 16; ++j) acc[j] = typename Mfma<T>::acc_t{0, 0, 0, 0};
    const SA *A = Ab + (size_t)lo_blk[q] * lda;
    const T *B = D + (size_t)lo_col[q] * ld;
    gemm_pairs<T, SA, T, TM>([&](int, const SA *&a, const T *&b) { a = A; b = B; }, 1, n, tm * TM, tn * TM, As, Bs,
                             acc);
    T *out = L + (size_t)q * ld;
    gemm_out<T, TM>(tm, tn, n, acc, [&](int row, int col, T v) { out[(size_t)col * n + row] = v; });
}

// phase 2: D_i = A_{diag[i]} - sum_q L_q * U_q, U_q = A_{lo_tr[q]} read from
// Ub (stride ldu): A's own blocks (FP64), or their FP32 copies.
template <typename T, typename SB, int TM>
__global__ void __launch_bounds__(Geo<TM>::GT)
k_fac_p2(const double *__restrict__ Ab, int64_t lda, const SB *__restrict__ Ub, int64_t ldu, const T *__restrict__ L,
         T *__restrict__ D, int64_t ld, const int32_t *__restrict__ rows, int njobs, const int32_t *__restrict__ lo_ptr,
         const int32_t *__restrict__ lo_tr, const int32_t *__restrict__ diag, int n, int tiles) {
    __shared__ __attribute__((aligned(16))) ATile<T, TM> As[2];
    __shared__ __attribute__((aligned(16))) BTile<T, TM> Bs[2];
    int job, tile;
    if (!xcd_job(njobs, tiles * tiles, job, tile)) return;
    const int i = rows[job];
    const int tm = tile % tiles, tn = tile / tiles;
    typename Mfma<T>::acc_t acc[TM / 16];
#pragma unroll
    for (int j = 0; j < TM / 16; ++j) acc[j] = typename Mfma<T>::acc_t{0, 0, 0, 0};
    const int q0 = lo_ptr[i], nq = lo_ptr[i + 1] - q0;
    if (nq > 0)
        gemm_pairs<T, T, SB, TM>(
            [&](int p, const T *&a, const SB *&b) {
                a = L + (size_t)(q0 + p) * ld;
                b = Ub + (size_t)lo_tr[q0 + p] * ldu;
            },
            nq, n, tm * TM, tn * TM, As, Bs, acc);
    const double *a = Ab + (size_t)diag[i] * lda;
    T *out = D + (size_t)i * ld;
    gemm_out<T, TM>(tm, tn, n, acc, [&](int row, int col, T v) {
        out[(size_t)col * n + row] = static_cast<T>(a[(size_t)col * n + row]) - v;
    });
}

// BF16 storage: W_u = bf16(Dinv_{row(u)} U_u) (round to nearest even) for every upper entry u, from the
// FP32 Dinv and A's own blocks: one rounding to BF16 in the operator of the sweep's folded form.
// Per factor at 16^3 P2 1.4 ms, 16^3 P3 8.7 ms.
template <int TM>
__global__ void __launch_bounds__(Geo<TM>::GT)
k_fold_left(const float *__restrict__ D, int64_t ld, const double *__restrict__ Ab, int64_t lda,
            const int32_t *__restrict__ up_row, const int32_t *__restrict__ up_blk, int nup, cdg_bf16 *__restrict__ W,
            int n, int tiles) {
    __shared__ __attribute__((aligned(16))) ATile<float, TM> As[2];
    __shared__ __attribute__((aligned(16))) BTile<float, TM> Bs[2];
    int u, tile;
    if (!xcd_job(nup, tiles * tiles, u, tile)) return;
    const int tm = tile % tiles, tn = tile / tiles;
    Mfma<float>::acc_t acc[TM / 16];
#pragma unroll
    for (int j = 0; j < TM / 16; ++j) acc[j] = Mfma<float>::acc_t{0, 0, 0, 0};
    const float *A = D + (size_t)up_row[u] * ld;
    const double *B = Ab + (size_t)up_blk[u] * lda;
    gemm_pairs<float, float, double, TM>([&](int, const float *&a, const double *&b) { a = A; b = B; }, 1, n, tm * TM,
                                         tn * TM, As, Bs, acc);
    cdg_bf16 *out = W + (size_t)u * ld;
    gemm_out<float, TM>(tm, tn, n, acc, [&](int row, int col, float v) {
        uint32_t b = __float_as_uint(v);
        b += 0x7fffu + ((b >> 16) & 1u);
        out[(size_t)col * n + row] = static_cast<cdg_bf16>(b >> 16);
    });
}

// DPP moves inside a 16-lane row: xor 1, xor 2 (quad permutes), rotate 4, 8.
template <int CTRL> __device__ __forceinline__ int dpp_i32(int x) {
    return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xF, 0xF, false);
}
template <int CTRL> __device__ __forceinline__ double dpp(double x) {
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, int2{dpp_i32<CTRL>(v.x), dpp_i32<CTRL>(v.y)});
}
template <int CTRL> __device__ __forceinline__ float dpp(float x) {
    return __builtin_bit_cast(float, dpp_i32<CTRL>(__builtin_bit_cast(int, x)));
}

// (value, index) max with the lower index on ties, and a min of `fu`, over the
// 16 lanes of a DPP row; every lane of the row ends with the result.
template <typename T, int CTRL>
__device__ __forceinline__ void argmax_step(T &best, int &bi, int &fu) {
    const T ob = dpp<CTRL>(best);
    const int oi = dpp_i32<CTRL>(bi);
    fu = min(fu, dpp_i32<CTRL>(fu));
    if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
}

// phase 3: in-place inverse of D_i, one workgroup of 4 waves (one per SIMD)
// per block.  Thread (tr, tc) of the 16 x 16 thread grid keeps rows
// tr + 16a and columns tc + 16b (a, b < R) in registers; the 16 owners of a
// column are one 16-lane DPP row.  Gauss-Jordan with partial pivoting and two
// barriers per pivot step:
//   1. the owners of column k publish it and reduce it among themselves
//      (largest |a(r,k)| over unused rows, lower row index on ties);
//   2. everyone reads the pivot row p; its owners publish it;
//   3. everyone applies  S -= c_r * prow  (c_p = 0) and rewrites column k.
// Rows are never swapped; the final scatter inv(rowstep[r], pivrow[m]) undoes
// the implicit permutation.  The pivot row is not scaled in place: row r keeps
// its unscaled values and sigma_r = 1/pivot is applied when the result is
// written (later eliminations are linear in the row, so they act on the
// unscaled values consistently).  Register indices are compile-time: the
// pivot loop runs k = 16*kb + kt with kb unrolled, and the pivot row is
// published through one LDS buffer per register row.
template <typename T, int R>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
k_fac_inv(T *__restrict__ D, int64_t ld, const int32_t *__restrict__ rows, int n, int32_t *__restrict__ err) {
    constexpr int TR = 16;
    constexpr int NMAX = TR * R;
    __shared__ T colv[2][NMAX];
    __shared__ T rowv[2][R][NMAX];
    __shared__ T sig[NMAX];
    __shared__ int32_t pivrow[NMAX], rowstep[NMAX];
    __shared__ int32_t piv_sh[2], bad_sh;
    const int blk = rows[blockIdx.x];
    T *M = D + (size_t)blk * ld;
    const int tid = threadIdx.x, tr = tid % TR, tc = tid / TR;
    T S[R][R];
#pragma unroll
    for (int a = 0; a < R; ++a)
#pragma unroll
        for (int b = 0; b < R; ++b) {
            const int r = tr + TR * a, m = tc + TR * b;
            S[a][b] = (r < n && m < n) ? M[(size_t)m * n + r] : T(0);
        }
    for (int i = tid; i < 2 * R * NMAX; i += 256) (&rowv[0][0][0])[i] = T(0);
    if (tid == 0) bad_sh = 0;
    bool used[R];
#pragma unroll
    for (int a = 0; a < R; ++a) used[a] = (tr + TR * a >= n);   // padding rows never pivot
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < R; ++kb) {
        const int kt_end = min(TR, n - kb * TR);
        for (int kt = 0; kt < kt_end; ++kt) {
            const int k = kb * TR + kt;
            const int buf = k & 1;
            if (tc == kt) {
                T best = T(-1);
                int bi = 0x7fffffff, fu = 0x7fffffff;
#pragma unroll
                for (int a = 0; a < R; ++a) {
                    const int r = tr + TR * a;
                    const T v = S[a][kb];
                    colv[buf][r] = v;   // padding rows hold zeros
                    if (!used[a]) {
                        const T av = fabs(v);
                        if (av > best) { best = av; bi = r; }
                        fu = min(fu, r);
                    }
                }
                argmax_step<T, 0xB1>(best, bi, fu);    // quad_perm [1,0,3,2]
                argmax_step<T, 0x4E>(best, bi, fu);    // quad_perm [2,3,0,1]
                argmax_step<T, 0x124>(best, bi, fu);   // row_ror:4
                argmax_step<T, 0x128>(best, bi, fu);   // row_ror:8
                if (tr == 0) {
                    if (!(best > T(0)) || bi >= n) { bad_sh = 1; bi = fu; }   // zero or non-finite column
                    piv_sh[buf] = bi;
                }
            }
            __syncthreads();
            const int p = __builtin_amdgcn_readfirstlane(piv_sh[buf]);
#pragma unroll
            for (int a = 0; a < R; ++a) used[a] = used[a] || (tr + TR * a == p);
            const int pa = p / TR, pt = p - pa * TR;
            const T rinv = T(1) / colv[buf][p];
            if (tid == 0) { pivrow[k] = p; rowstep[p] = k; sig[p] = rinv; }
            if (tr == pt) {
#pragma unroll
                for (int a = 0; a < R; ++a)
                    if (a == pa) {
#pragma unroll
                        for (int b = 0; b < R; ++b) rowv[buf][a][tc + TR * b] = S[a][b];
                    }
            }
            __syncthreads();
            T prow[R], cr[R];
#pragma unroll
            for (int b = 0; b < R; ++b) prow[b] = rowv[buf][pa][tc + TR * b] * rinv;
#pragma unroll
            for (int a = 0; a < R; ++a) cr[a] = (tr + TR * a == p) ? T(0) : colv[buf][tr + TR * a];
#pragma unroll
            for (int a = 0; a < R; ++a)
#pragma unroll
                for (int b = 0; b < R; ++b) S[a][b] -= cr[a] * prow[b];
            // column k: -c_r/pivot, and 1 (times sigma_p = 1/pivot) in row p
#pragma unroll
            for (int a = 0; a < R; ++a) {
                const T v = (tr + TR * a == p) ? T(1) : -cr[a] * rinv;
                S[a][kb] = (tc == kt) ? v : S[a][kb];
            }
        }
    }
    __syncthreads();
    if (tid == 0 && bad_sh) atomicMin(err, blk);
#pragma unroll
    for (int a = 0; a < R; ++a)
#pragma unroll
        for (int b = 0; b < R; ++b) {
            const int r = tr + TR * a, m = tc + TR * b;
            if (r < n && m < n) M[(size_t)pivrow[m] * n + rowstep[r]] = sig[r] * S[a][b];
        }
}

// ---- blocked Gauss-Jordan inverse -------------------------------------------
// DPP with a row mask (lanes outside the mask keep their own value).
template <int CTRL, int RM> __device__ __forceinline__ int dpp_rm_i32(int x) {
    return __builtin_amdgcn_update_dpp(x, x, CTRL, RM, 0xF, false);
}
template <int CTRL, int RM> __device__ __forceinline__ double dpp_rm(double x) {
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, int2{dpp_rm_i32<CTRL, RM>(v.x), dpp_rm_i32<CTRL, RM>(v.y)});
}
template <int CTRL, int RM> __device__ __forceinline__ float dpp_rm(float x) {
    return __builtin_bit_cast(float, dpp_rm_i32<CTRL, RM>(__builtin_bit_cast(int, x)));
}
template <typename T, int CTRL, int RM>
__device__ __forceinline__ void wargmax_step(T &best, int &bi, int &fu) {
    const T ob = dpp_rm<CTRL, RM>(best);
    const int oi = dpp_rm_i32<CTRL, RM>(bi);
    fu = min(fu, dpp_rm_i32<CTRL, RM>(fu));
    if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
}
// (value, index) maximum over the wave, lower index on ties, and the minimum
// of fu; the result is complete in lane 63.
template <typename T>
__device__ __forceinline__ void wave_argmax(T &best, int &bi, int &fu) {
    wargmax_step<T, 0xB1, 0xF>(best, bi, fu);    // quad_perm [1,0,3,2]
    wargmax_step<T, 0x4E, 0xF>(best, bi, fu);    // quad_perm [2,3,0,1]
    wargmax_step<T, 0x124, 0xF>(best, bi, fu);   // row_ror:4
    wargmax_step<T, 0x128, 0xF>(best, bi, fu);   // row_ror:8  (every lane: its row's result)
    wargmax_step<T, 0x142, 0xA>(best, bi, fu);   // row_bcast:15 into rows 1, 3
    wargmax_step<T, 0x143, 0xC>(best, bi, fu);   // row_bcast:31 into rows 2, 3
}
// Lanes of one wave exchanging data through LDS: without this the compiler
// may order another lane's load before the writing lane's store (each lane's
// program alone allows it).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ double readlane(double x, int l) {
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, int2{__builtin_amdgcn_readlane(v.x, l), __builtin_amdgcn_readlane(v.y, l)});
}
__device__ __forceinline__ float readlane(float x, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
}

// Diagonal-pivot threshold of the checked inverses: the diagonal a_kk is
// taken as the pivot of column k when |a_kk| >= kPivTau * |a_rk| for every
// unused row r (threshold partial pivoting with u = 0.1, the usual choice of
// sparse direct solvers: Duff, Erisman & Reid, Direct Methods for Sparse
// Matrices, ch. 5), which bounds the growth of a step by 1 + 1/kPivTau.  A
// block where some step fails the test is inverted with full partial
// pivoting instead.  Both give the inverse up to rounding; DG Jacobian
// blocks (dR/dq + mass/dtau) pass with |a_kk| / max_r |a_rk| >= 0.33 where
// strict partial pivoting would swap a third of the rows.
constexpr double kPivTau = 0.1;

// Gauss-Jordan with partial pivoting on one 16-column panel, run by one
// wave.  On entry G[r*gp + c] holds the panel (rows r < NP, zero beyond n and
// beyond the panel width w) and rowtag[r] != 0 marks rows pivoted in earlier
// panels.  On exit G holds C - E_P (C = [W on the pivot rows, -A(r,P) W
// elsewhere], W the inverse of the pivot block), rowtag[p] = 1 + step and
// pivrow[step] = p for this panel's pivots.  The pivot is the largest |a(r,k)|
// over unused rows, lower row on ties (DPP argmax); rows are never swapped.
// The panel's columns rotate left by one per step, so the column being
// eliminated always sits at register position 0 and the loop body is not
// unrolled; after 16 rotations the columns are back in place.
template <typename T, int NR>
__device__ __forceinline__ bool panel_gj(T *G, int gp, int NP, int n, int k0, int w, int32_t *rowtag,
                                         int32_t *pivrow, T *prow_sh) {
    const int lane = threadIdx.x & 63;
    T pr[NR][16];
    bool used[NR];
#pragma unroll
    for (int a = 0; a < NR; ++a) {
        const int r = lane + 64 * a;
        used[a] = r >= n || (r < NP && rowtag[r] != 0);
#pragma unroll
        for (int c = 0; c < 16; ++c) pr[a][c] = r < NP ? G[r * gp + c] : T(0);
    }
    bool bad = false;
#pragma unroll 1
    for (int j = 0; j < 16; ++j) {
        if (j < w) {
            T best = T(-1);
            int bi = 0x7fffffff, fu = 0x7fffffff;
#pragma unroll
            for (int a = 0; a < NR; ++a) {
                const int r = lane + 64 * a;
                if (!used[a]) {
                    const T av = fabs(pr[a][0]);
                    if (av > best) { best = av; bi = r; }
                    fu = min(fu, r);
                }
            }
            wave_argmax<T>(best, bi, fu);
            const T bbest = readlane(best, 63);
            int p = __builtin_amdgcn_readlane(bi, 63);
            if (!(bbest > T(0)) || p >= n) { bad = true; p = __builtin_amdgcn_readlane(fu, 63); }
            const int pa = p >> 6, pl = p & 63;
            // the pivot row through LDS
            if (lane == pl) {
#pragma unroll
                for (int a = 0; a < NR; ++a)
                    if (a == pa) {
#pragma unroll
                        for (int c = 0; c < 16; ++c) prow_sh[c] = pr[a][c];
                    }
            }
            wave_sync();
            T prow[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) prow[c] = prow_sh[c];
            const T rinv = T(1) / prow[0];
#pragma unroll
            for (int c = 0; c < 16; ++c) prow[c] *= rinv;
#pragma unroll
            for (int a = 0; a < NR; ++a) {
                const bool isp = (a == pa) && (lane == pl);
                const T cr = isp ? T(0) : pr[a][0];
#pragma unroll
                for (int c = 1; c < 16; ++c) pr[a][c] -= cr * prow[c];
                pr[a][0] = -cr * rinv;
                used[a] = used[a] || isp;
            }
            if (lane == pl) {
#pragma unroll
                for (int a = 0; a < NR; ++a)
                    if (a == pa) {
#pragma unroll
                        for (int c = 1; c < 16; ++c) pr[a][c] = prow[c];
                        pr[a][0] = rinv;
                    }
            }
            if (lane == 0) { rowtag[p] = k0 + j + 1; pivrow[k0 + j] = p; }
            wave_sync();   // prow_sh is rewritten by the next step; rowtag is read below
        }
#pragma unroll
        for (int a = 0; a < NR; ++a) {
            const T first = pr[a][0];
#pragma unroll
            for (int c = 0; c < 15; ++c) pr[a][c] = pr[a][c + 1];
            pr[a][15] = first;
        }
    }
    // C - E_P back to LDS (the ones of E_P sit at (p_j, j))
#pragma unroll
    for (int a = 0; a < NR; ++a) {
        const int r = lane + 64 * a;
        if (r < NP) {
            const int tg = rowtag[r] - 1 - k0;     // panel step of this row, if any
#pragma unroll
            for (int c = 0; c < 16; ++c) G[r * gp + c] = pr[a][c] - ((tg == c) ? T(1) : T(0));
        }
    }
    return bad;
}

// 1/x for the pivot chain: v_rcp and Newton steps, 3 dependent operations in FP32 and 7 in FP64 instead
// of the division's 11, which sit on the chain of every pivot step.  In FP64 the last step rounds
// like the division (a start off by up to 2^-22, 2e8 random x in host FMAs: no difference); in FP32 within an ulp.
__device__ __forceinline__ float recip(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(r, fmaf(-x, r, 1.0f), r);
}
__device__ __forceinline__ double recip(double x) {
    double r = __builtin_amdgcn_rcp(x);
#pragma unroll
    for (int i = 0; i < 3; ++i) r = fma(r, fma(-x, r, 1.0), r);
    return r;
}

// Lanes 16 Q .. 16 Q + 15 copied to all four such rows (v_permlane32_swap puts a half of the
// wave in both halves, v_permlane16_swap a row in its neighbour).
template <int Q> __device__ __forceinline__ int row_all(int x) {
    const auto h = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    const int y = h[Q >> 1];
    const auto r = __builtin_amdgcn_permlane16_swap(y, y, false, false);
    return r[Q & 1];
}
template <int Q> __device__ __forceinline__ float row_all(float x) {
    return __builtin_bit_cast(float, row_all<Q>(__builtin_bit_cast(int, x)));
}
template <int Q> __device__ __forceinline__ double row_all(double x) {
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, int2{row_all<Q>(v.x), row_all<Q>(v.y)});
}

// lane J of each row of 16, to the row
template <int J> __device__ __forceinline__ float newbcast(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + J, 0xF, 0xF, true));
}
template <int J> __device__ __forceinline__ double newbcast(double x) {
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, int2{__builtin_amdgcn_update_dpp(0, v.x, 0x150 + J, 0xF, 0xF, true),
                                           __builtin_amdgcn_update_dpp(0, v.y, 0x150 + J, 0xF, 0xF, true)});
}

template <int J, int N, typename F> __device__ __forceinline__ void unrolled(const F &f) {
    if constexpr (J < N) {
        f(std::integral_constant<int, J>{});
        unrolled<J + 1, N>(f);
    }
}

// Gauss-Jordan with checked diagonal pivots on the 16-column panel G (NP rows, pitch
// gp, zero beyond n and beyond the panel width w) whose pivot rows are k0 ..
// k0 + w - 1, by a workgroup of NW wavefronts.  On exit G holds C - E_P: W - I on the
// pivot rows, W the inverse of the pivot block, and -A(r,P) W on the others.
//   Stage A (wavefront 0): the 16 steps on the 16 x 16 pivot block.  Lane 16 q + i holds row i,
//   columns 4q .. 4q+3: the pivot row comes to the other rows by DPP (row_newbcast), each row's
//   multiplier from the four columns that hold it by two lane swaps, so no step touches LDS.
//   The multipliers below the diagonal are L of the pivot block's factors L U.
//   Stage B (a tile of 16 rows per wavefront and turn): X = A(r,P) W on MFMA, and for the
//   rows not used yet X L, which are the multipliers A(r,P) U^-1 that the steps would have
//   met there.  (Transposed tiles: X^T comes out as the second product takes it.)
// Both stages check the diagonal pivot of each step against the threshold: no unused row
// (row > k0 + j, row < n) with kPivTau * |a(r,j)| > |a(j,j)|, and a nonzero finite pivot.
// Returns whether some step needed another pivot.
//
// What bounds it: stage A, whose one wavefront issues some 25 (FP32) or 50 (FP64)
// instructions a step.  Panel at n = 135, cycles of stage A + B: FP64 9350 + 6100 before (the
// pivot row by ds_bpermute through LDS, the other rows replaying each step from LDS), now
// 5200 + 3200; FP32 10000 (the two stages at once), now 3150 + 2050.  Blocks of 89 rows at
// once: n = 135 FP64 112 -> 84 us, FP32 78 -> 60; n = 40 28 -> 18 and 22 -> 15.
template <typename T, int NW>
__device__ __forceinline__ bool panel_steps(T *G, int gp, int NP, int n, int k0, int w, T (*Ws)[17], T (*Ls)[17],
                                            int32_t *miss_sh) {
    typedef typename Mfma<T>::acc_t acc_t;
    const int tid = threadIdx.x, lane = tid & 63;
    if (tid < 64) {
        const int i = lane & 15, q = lane >> 4;
        T a[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = i == 4 * q + e && i >= w ? T(1) : G[(k0 + i) * gp + 4 * q + e];   // (steps past w change nothing)
        T ri = T(1);                                       // 1 / pivot of step i
        unrolled<0, 16>([&](auto jc) {
            constexpr int j = decltype(jc)::value, jq = j >> 2, je = j & 3;
            const T rinv = recip(readlane(a[je], 16 * jq + j));
            const T cc = row_all<jq>(a[je]);               // column j
            const bool isp = i == j, mine = q == jq;
            if (jq == 0) lo[je] = cc * rinv;               // (kept by the lanes of column j)
            else lo[je] = mine ? cc * rinv : lo[je];
            ri = isp ? rinv : ri;
            // the pivot row stays unscaled until the end (its updates are linear)
            const T cr = isp ? T(0) : cc;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                T sv = newbcast<j>(a[e]) * rinv;
                if (e == je) {                             // column j itself
                    sv = mine ? rinv : sv;
                    a[e] = mine ? (isp ? T(1) : T(0)) : a[e];
                }
                a[e] = fma(-cr, sv, a[e]);
            }
        });
        const T ar = fabs(ri);
        bool viol = !(ar > T(0)) || !(ar < T(INFINITY));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = 4 * q + e;
            const T v = a[e] * ri;
            Ws[i][c] = -v;
            Ls[i][c] = i > c ? lo[e] : i == c ? T(1) : T(0);
            viol = viol || (i > c && T(kPivTau) * fabs(lo[e]) > T(1));
            G[(k0 + i) * gp + c] = v - (i == c ? T(1) : T(0));
        }
        if (viol) *miss_sh = 1;
    }
    __syncthreads();
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), kt = k0 >> 4;
    T bw[4], bl[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        bw[kk] = Ws[4 * kk + (lane >> 4)][lane & 15];
        bl[kk] = Ls[Mfma<T>::row(lane, kk)][lane & 15];
    }
    bool viol = false;
    for (int ti = wv; ti < NP / 16; ti += NW) {
        if (ti == kt) continue;
        T *const Gr = G + (16 * ti + (lane & 15)) * gp;
        T av[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) av[kk] = Gr[4 * kk + (lane >> 4)];
        acc_t x = {};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) x = Mfma<T>::run(bw[kk], av[kk], x);
        if (ti > kt) {
            acc_t m = {};
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) m = Mfma<T>::run(bl[kk], x[kk], m);
#pragma unroll
            for (int r = 0; r < 4; ++r) viol = viol || T(kPivTau) * fabs(m[r]) > T(1);   // (rows beyond n are zero)
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) Gr[Mfma<T>::row(lane, r)] = x[r];
    }
    if (viol) *miss_sh = 1;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*miss_sh) != 0;
}

// The panel of BF16-stored factors (FP32): the same Gauss-Jordan, rounded step by step as an unblocked
// one rounds.  A factor in BF16 is read through its 8 bits: where FP32 rounds the other way, one
// entry in 20000 lands on the next BF16 value, which moves the apply by 4e-5 and a solve's residual
// norm by 1e-4 of itself.  So this storage keeps one order of operations: each step's pivot row is scaled by
// 1 / pivot and subtracted, by every row, before the next step.
//   Stage A (wavefront 0): the pivot block as in panel_steps; each step's scaled pivot row (1 / pivot
//   in its own column) and the pivot itself go to H[j] (zeros for steps from w on), then *step_sh rises to
//   k0 + j + 1.
//   Stage B (wavefronts 1..NW-1, a row per lane) replays step j once *step_sh shows it.  Wavefront 0
//   never waits, so every wait ends; k0 only grows during a kernel, *step_sh starts at 0.
// G, the checks and the result as in panel_steps.  Whole BF16 factors with it and with panel_steps:
// 16^3 P2 7.4 and 6.9 ms, 16^3 P3 37.2 and 34.4, 31x17x13 P1 1.84 and 1.53.
constexpr int kHP = 20;   // pitch of H: 16 values and the pivot, 16-byte rows
template <int NW>
__device__ __forceinline__ bool panel_replay(float *G, int gp, int NP, int n, int k0, int w, float (*H)[kHP],
                                             int32_t *step_sh, int32_t *miss_sh) {
    const int tid = threadIdx.x, lane = tid & 63;
    bool viol = false;
    if (tid < 64) {
        const int i = lane & 15, q = lane >> 4;
        float a[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = G[(k0 + i) * gp + 4 * q + e];
        unrolled<0, 16>([&](auto jc) {
            constexpr int j = decltype(jc)::value, jq = j >> 2, je = j & 3;
            const bool isp = i == j, mine = q == jq;
            float sv[4] = {0.f, 0.f, 0.f, 0.f}, piv = 0.f;
            if (j < w) {
                piv = readlane(a[je], 16 * jq + j);
                const float rinv = recip(piv), ap = fabsf(piv), cc = row_all<jq>(a[je]);
                viol = viol || !(ap > 0.f) || !(ap < INFINITY) || (i > j && k0 + i < n && (float)kPivTau * fabsf(cc) > ap);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sv[e] = newbcast<j>(a[e]) * rinv;
                    if (e == je) sv[e] = mine ? rinv : sv[e];
                    const float t = isp ? sv[e] : fmaf(-cc, sv[e], a[e]);
                    a[e] = e == je && mine ? (isp ? rinv : -cc * rinv) : t;
                }
            }
            if (i == 0) {
#pragma unroll
                for (int e = 0; e < 4; ++e) H[j][4 * q + e] = sv[e];
                if (q == 0) H[j][16] = piv;
            }
            if (tid == 0) __hip_atomic_store(step_sh, k0 + j + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        });
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = 4 * q + e;
            G[(k0 + i) * gp + c] = a[e] - (i == c && c < w ? 1.f : 0.f);
        }
    } else {
        const int row = lane * (NW - 1) + (tid >> 6) - 1;
        const bool live = row < NP && (row < k0 || row >= k0 + 16), unused = row >= k0 + 16 && row < n;
        float pr[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) pr[c] = live ? G[row * gp + c] : 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            while (__hip_atomic_load(step_sh, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) <= k0 + j)
                __builtin_amdgcn_s_sleep(1);
            float sv[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) sv[c] = H[j][c];
            const float cc = pr[j];
            viol = viol || (j < w && unused && (float)kPivTau * fabsf(cc) > fabsf(H[j][16]));
#pragma unroll
            for (int c = 0; c < 16; ++c)
                if (c != j) pr[c] = fmaf(-cc, sv[c], pr[c]);
            pr[j] = -cc * sv[j];
        }
        if (live)
#pragma unroll
            for (int c = 0; c < 16; ++c) G[row * gp + c] = pr[c];
    }
    if (viol) *miss_sh = 1;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*miss_sh) != 0;
}

// The same steps spread over a workgroup of 16 wavefronts (128 VGPRs a lane leave no room for stage
// A beside stage B): row r in lane r, one barrier a step.  The owner of the pivot row publishes it, scaled,
// and the pivot's size in H[j % 2].
template <int NW>
__device__ __forceinline__ bool panel_rows(float *G, int gp, int NP, int n, int k0, int w, float (*H)[kHP],
                                           int32_t *miss_sh) {
    const int row = threadIdx.x;
    const bool live = row < NP, wave_live = __builtin_amdgcn_readfirstlane(row & ~63) < NP;
    float pr[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) pr[c] = live ? G[row * gp + c] : 0.f;
    bool used = row >= n || row < k0, viol = false;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        if (j < w) {
            float *const h = H[j & 1];
            const bool isp = row == k0 + j;
            if (isp) {
                const float ap = fabsf(pr[j]), rinv = 1.f / pr[j];
                viol = viol || !(ap > 0.f) || !(ap < INFINITY);
#pragma unroll
                for (int c = 0; c < 16; ++c) h[c] = pr[c] = c == j ? rinv : pr[c] * rinv;
                h[16] = ap;
            }
            __syncthreads();   // (the next step writes the other half of H)
            if (wave_live && !isp) {
                float sv[17];
#pragma unroll
                for (int c = 0; c < 17; ++c) sv[c] = h[c];
                const float cc = pr[j];
                viol = viol || (!used && (float)kPivTau * fabsf(cc) > sv[16]);
#pragma unroll
                for (int c = 0; c < 16; ++c) pr[c] = c == j ? -cc * sv[j] : fmaf(-cc, sv[c], pr[c]);
            }
            used = used || isp;
        }
    }
    if (live)
#pragma unroll
        for (int c = 0; c < 16; ++c) G[row * gp + c] = pr[c] - (row - k0 == c && c < w ? 1.f : 0.f);
    if (viol) *miss_sh = 1;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*miss_sh) != 0;
}

// LDS of a panel's steps, and the steps: REPLAY for BF16-stored factors.
template <typename T, bool REPLAY> struct PanelLds {
    T Ws[16][17], Ls[16][17];
    __device__ __forceinline__ void start() {}
    template <int NW>
    __device__ __forceinline__ bool run(T *G, int gp, int NP, int n, int k0, int w, int32_t *miss_sh) {
        return panel_steps<T, NW>(G, gp, NP, n, k0, w, Ws, Ls, miss_sh);
    }
};
template <> struct PanelLds<float, true> {
    float H[16][kHP];
    int32_t step;
    __device__ __forceinline__ void start() { if (threadIdx.x == 0) step = 0; }   // (a barrier follows)
    template <int NW>
    __device__ __forceinline__ bool run(float *G, int gp, int NP, int n, int k0, int w, int32_t *miss_sh) {
        if constexpr (NW > 4) return panel_rows<NW>(G, gp, NP, n, k0, w, H, miss_sh);
        else return panel_replay<NW>(G, gp, NP, n, k0, w, H, &step, miss_sh);
    }
};

// Raw buffer access to one block's slot: a byte offset at or beyond the
// descriptor's size (kOob) reads 0 and drops the store, so masked lanes need
// no branch (descriptor word 3: raw, untyped access on CDNA).
typedef unsigned int bu32x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kOob = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t slot_rsrc(void *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(p, (short)0, bytes, 0x00020000);
}
template <typename T> __device__ __forceinline__ T bload(__amdgpu_buffer_rsrc_t r, uint32_t off);
template <> __device__ __forceinline__ float bload<float>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
template <> __device__ __forceinline__ double bload<double>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
template <typename T> __device__ __forceinline__ void bstore(T v, __amdgpu_buffer_rsrc_t r, uint32_t off);
template <> __device__ __forceinline__ void bstore<float>(float v, __amdgpu_buffer_rsrc_t r, uint32_t off) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, off, 0, 0);
}
template <> __device__ __forceinline__ void bstore<double>(double v, __amdgpu_buffer_rsrc_t r, uint32_t off) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(bu32x2, v), r, off, 0, 0);
}

// Blocked Gauss-Jordan inverse with partial pivoting of the n x n block M
// (n <= 64*NR) by one workgroup, working in the global slot S (L2-resident):
// the rare blocks that the diagonal-pivot inverse hands over.  The rank-16
// update runs on the transposed tiles, D'(c, r) = S(r, c): an MFMA tile row
// is then a matrix column, so its 16 lanes touch 16 consecutive elements of
// the column-major block.  LDS: the panel G (NP x 17), the pivot rows XP
// (16 x (NP + 1)), prow_sh, rowtag, pivrow (NP = 16 * ceil(n/16)).  M
// receives the inverse and *bad reports a zero or non-finite pivot column.
template <typename T, int NR, int NTH>
__device__ void ginv_pivot_body(T *__restrict__ M, T *__restrict__ S, int n, T *G, T *XP, T *prow_sh,
                                int32_t *rowtag, int32_t *pivrow, int32_t *flag_sh, bool *bad) {
    constexpr int GP = 17, NWV = NTH / 64, UBP = 4;
    typedef typename Mfma<T>::acc_t acc_t;
    const int NT = (n + 15) / 16, NP = 16 * NT, XPP = NP + 1;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nn = n * n;
    for (int e = tid; e < nn; e += NTH) S[e] = M[e];
    for (int i = tid; i < NP; i += NTH) { rowtag[i] = 0; pivrow[i] = 0; }
    for (int i = tid; i < 16 * XPP; i += NTH) XP[i] = T(0);
    if (tid == 0) *flag_sh = 0;
    __syncthreads();
    for (int kb = 0; kb < NT; ++kb) {
        const int k0 = 16 * kb;
        const int w = min(16, n - k0);
        // 1. panel to LDS (zero beyond n and beyond the panel width)
        for (int e = tid; e < NP * 16; e += NTH) {
            const int c = e / NP, r = e - c * NP;
            G[r * GP + c] = (r < n && c < w) ? S[(size_t)(k0 + c) * n + r] : T(0);
        }
        __syncthreads();
        // 2. panel Gauss-Jordan with partial pivoting (wave 0); flag: zero pivot
        if (wv == 0) {
            const bool b = panel_gj<T, NR>(G, GP, NP, n, k0, w, rowtag, pivrow, prow_sh);
            if (lane == 0 && b) *flag_sh = 1;
        }
        __syncthreads();
        // 3. pivot rows X(P, :) of the other columns
        for (int e = tid; e < w * n; e += NTH) {
            const int c = e / w, j = e - c * w;
            if (c < k0 || c >= k0 + w) XP[j * XPP + c] = S[(size_t)c * n + pivrow[k0 + j]];
        }
        __syncthreads();
        // 4. X += (C - E_P) X(P,:) on MFMA (transposed tiles) for the tiles outside
        //    the panel's tile column, then the panel's tiles take C
        for (int t0 = wv; t0 < NT * NT; t0 += NWV * UBP) {
            acc_t acc[UBP];
#pragma unroll
            for (int u = 0; u < UBP; ++u) {
                const int t = t0 + NWV * u;
                const int ti = t % NT, tj = t / NT;
                const int r = 16 * ti + (lane & 15);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int c = 16 * tj + Mfma<T>::row(lane, q);
                    acc[u][q] = (t < NT * NT && tj != kb && r < n && c < n) ? S[(size_t)c * n + r] : T(0);
                }
            }
#pragma unroll
            for (int u = 0; u < UBP; ++u) {
                const int t = t0 + NWV * u;
                if (t >= NT * NT) continue;
                const int ti = t % NT, tj = t / NT;
                const int r = 16 * ti + (lane & 15);
                if (tj != kb) {
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk) {
                        const T a = XP[(4 * kk + (lane >> 4)) * XPP + 16 * tj + (lane & 15)];
                        const T bb = G[(16 * ti + (lane & 15)) * GP + 4 * kk + (lane >> 4)];
                        acc[u] = Mfma<T>::run(a, bb, acc[u]);
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int c = 16 * tj + Mfma<T>::row(lane, q);
                        if (r < n && c < n) S[(size_t)c * n + r] = acc[u][q];
                    }
                } else if (r < n) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int cc = Mfma<T>::row(lane, q);
                        const int c = k0 + cc;
                        if (cc < w) S[(size_t)c * n + r] = G[r * GP + cc] + ((rowtag[r] - 1 - k0 == cc) ? T(1) : T(0));
                    }
                }
            }
        }
        __syncthreads();
    }
    *bad = __builtin_amdgcn_readfirstlane(*flag_sh) != 0;
    // inv(rowstep(r), pivrow(c)) = S(r, c)
    for (int e = tid; e < nn; e += NTH) {
        const int c = e / n, r = e - c * n;
        M[(size_t)pivrow[c] * n + (rowtag[r] - 1)] = S[e];
    }
}

// Wide-panel inverse with the pivot rows in registers: panels of H 16-column
// halves in LDS (each half's Gauss-Jordan steps, PanelLds::run, then their
// transform on the other halves on MFMA), then every tile outside the panel
// takes the rank-16H update.
// Each wave owns whole tile columns; before updating any tile of a column it
// loads that column's pivot-row operands (16H rows, 4H values per lane) into
// registers, so no other wave can have changed them (the column's tiles, its
// pivot-row tiles among them, are only this wave's).  Fewer, wider panels
// mean fewer passes over the slot (each reads and writes the whole block);
// with the pivot rows out of LDS, the halves alone take it.  The first panel
// reads M and the last writes M (the slot S holds the passes between), so
// neither a copy of M nor a copy back is needed; the result is inv(M) with
// no permutation, as every pivot is diagonal.  LDS (ginv_lds): H halves of
// NP x 17.  n = 320, 89 blocks, FP32: 410 us -> 276 (steps 384 -> 183 kcycles with panel_steps;
// update 347 -> 256, 205 of them products, with offsets that take one addition per
// access); FP64, 40 blocks: 700 -> 501.
template <typename T> struct GinvHalves { static constexpr int H = sizeof(T) == 4 ? 4 : 3; };
template <typename T, int NR, int NTH, int UB, int H, bool REPLAY>
__device__ bool ginv_body_wide_rx(T *__restrict__ M, T *__restrict__ S, int n, T *G, PanelLds<T, REPLAY> &pl,
                                  int32_t *flag_sh) {
    typedef typename Mfma<T>::acc_t acc_t;
    constexpr int GP = 17, NWV = NTH / 64, PW = 16 * H;
    const int NT = (n + 15) / 16, NP = 16 * NT;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nn = n * n;
    auto half = [&](int h) -> T * { return G + (size_t)h * NP * GP; };
    if (tid == 0) *flag_sh = 0;
    pl.start();
    __syncthreads();
    // the first panel reads the block, the last one writes it, the others work in the
    // slot (M stays as it was until the last panel's pivots have passed their check)
    const __amdgpu_buffer_rsrc_t rsM = slot_rsrc(M, nn * (int)sizeof(T)), rsS = slot_rsrc(S, nn * (int)sizeof(T));
    constexpr int PC = PW / NWV;         // panel columns per wave
    static_assert(PW % NWV == 0, "every wave loads the same number of columns");
    for (int kb = 0; kb < NT; kb += H) {
        const int k0 = 16 * kb;
        const int np = min(H, NT - kb);                         // halves (tile columns) of this panel
        auto width = [&](int h) { return h < np ? min(16, n - k0 - 16 * h) : 0; };
        const __amdgpu_buffer_rsrc_t src = kb == 0 ? rsM : rsS, dst = kb + H >= NT ? rsM : rsS;
        // 1. the halves to LDS (zero beyond n and beyond each half's width)
        for (int i = 0; i < PC; ++i) {
            const int c = wv * PC + i, h = c >> 4;
            const uint32_t co = (c & 15) < width(h) ? (uint32_t)((k0 + c) * n * (int)sizeof(T)) : kOob;
            T v[NR];
#pragma unroll
            for (int u = 0; u < NR; ++u) {
                const int r = lane + 64 * u;
                v[u] = bload<T>(src, r < n ? co + (uint32_t)(r * (int)sizeof(T)) : kOob);
            }
#pragma unroll
            for (int u = 0; u < NR; ++u)
                if (lane + 64 * u < NP) half(h)[(lane + 64 * u) * GP + (c & 15)] = v[u];
        }
        __syncthreads();
        // 2. each half's steps, then their transform on the panel's other halves t:
        //    G_t += G_h G_t(P_h, :) on MFMA tiles (P_h: half h's pivot rows), whose
        //    pivot-row operands every wave reads before any tile changes
        for (int h = 0; h < np; ++h) {
            const int kh = k0 + 16 * h, wh = width(h);
            if (pl.template run<NWV>(half(h), GP, NP, n, kh, wh, flag_sh)) return false;
            if (np == 1) break;
            T b[H][4];
#pragma unroll
            for (int t = 0; t < H; ++t)
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    const int j = 4 * kk + (lane >> 4);
                    b[t][kk] = (t < np && t != h && j < wh) ? half(t)[(kh + j) * GP + (lane & 15)] : T(0);
                }
            __syncthreads();
            const T *Gs = half(h);
            for (int idx = wv; idx < NT * (np - 1); idx += NWV) {
                const int s = idx / NT, ti = idx - s * NT, t = s + (s >= h);
                T bs[4];
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    bs[kk] = b[0][kk];
#pragma unroll
                    for (int u = 1; u < H; ++u) bs[kk] = t == u ? b[u][kk] : bs[kk];
                }
                T *Gt = half(t);
                acc_t acc;
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[q] = Gt[(16 * ti + Mfma<T>::row(lane, q)) * GP + (lane & 15)];
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
                    acc = Mfma<T>::run(Gs[(16 * ti + (lane & 15)) * GP + 4 * kk + (lane >> 4)], bs[kk], acc);
#pragma unroll
                for (int q = 0; q < 4; ++q) Gt[(16 * ti + Mfma<T>::row(lane, q)) * GP + (lane & 15)] = acc[q];
            }
            __syncthreads();
        }
        // 3. X += (C - E_P) X(P, :) on the tiles outside the panel (transposed tiles,
        //    branch-free, the next round's loads before this round's stores), then the
        //    panel's tiles take C.  A wave's work item is a tile column, or half of one
        //    when the columns do not divide evenly among the waves (17 columns on 16
        //    waves: three rounds of halves instead of two of columns).  Both waves of a
        //    split column read its pivot rows before either changes them (one barrier per
        //    round; a column's two halves are items 2j, 2j + 1 of one round).
        const int ncol = NT - np;
        const int split = ncol % NWV != 0 ? 2 : 1;
        const int nh = split == 2 ? (NT + 1) / 2 : NT;     // tiles in a column's first half
        for (int it0 = 0; it0 < split * ncol; it0 += NWV) {
            const int item = it0 + wv;
            const bool act = item < split * ncol;           // uniform per wave
            const int tjp = min(item, split * ncol - 1) / split, part = item - tjp * split;
            const int tj = tjp + (tjp >= kb ? np : 0);
            const int lo = part == 1 ? nh : 0, hi = part == 1 || split == 1 ? NT : nh;
            const int c = 16 * tj + (lane & 15);
            T a[4 * H];   // X(P, c): pivot row 4 kk + lane / 16 of the panel, this lane's column
#pragma unroll
            for (int kk = 0; kk < 4 * H; ++kk) {
                const int h = kk >> 2, j = 4 * (kk & 3) + (lane >> 4);
                const bool ok = act && h < np && j < width(h) && c < n;
                a[kk] = bload<T>(src, ok ? (uint32_t)((c * n + k0 + 16 * h + j) * (int)sizeof(T)) : kOob);
            }
            if (split == 2) __syncthreads();
            if (!act) continue;
            // byte offset of (row, column): beyond the slot when either is (the sum of both marks does
            // not wrap around)
            uint32_t oc[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int cq = 16 * tj + Mfma<T>::row(lane, q);
                oc[q] = cq < n ? (uint32_t)((cq * n + (lane & 15)) * (int)sizeof(T)) : kOob;
            }
            const int rl = n - (lane & 15);
            auto offs = [&](int ti, int q) -> uint32_t {
                return oc[q] + (ti < hi && 16 * ti < rl ? (uint32_t)(16 * ti * (int)sizeof(T)) : kOob >> 1);
            };
            auto load_round = [&](T (&v)[UB][4], int i0) {
#pragma unroll
                for (int u = 0; u < UB; ++u)
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[u][q] = bload<T>(src, offs(i0 + u, q));
            };
            auto update_round = [&](const T (&v)[UB][4], int i0) {
#pragma unroll
                for (int u = 0; u < UB; ++u) {
                    const int ti = min(i0 + u, NT - 1);
                    const T *grow = G + (16 * ti + (lane & 15)) * GP + (lane >> 4);
                    acc_t acc;
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[q] = v[u][q];
#pragma unroll
                    for (int kk = 0; kk < 4 * H; ++kk) {
                        if (kk < 4 * np) {
                            const T bb = grow[(kk >> 2) * NP * GP + 4 * (kk & 3)];
                            acc = Mfma<T>::run(a[kk], bb, acc);
                        }
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) bstore<T>(acc[q], dst, offs(i0 + u, q));
                }
            };
            T va[UB][4], vb[UB][4];
            load_round(va, lo);
            for (int i0 = lo; i0 < hi; i0 += 2 * UB) {
                load_round(vb, i0 + UB);
                update_round(va, i0);
                load_round(va, i0 + 2 * UB);
                if (i0 + UB < hi) update_round(vb, i0 + UB);
            }
        }
        for (int h = 0; h < np; ++h) {
            const T *Gh = half(h);
            const int kh = k0 + 16 * h, wh = width(h);
            for (int ti = wv; ti < NT; ti += NWV) {
                const int r = 16 * ti + (lane & 15);
                if (r < n) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int cc = Mfma<T>::row(lane, q);
                        if (cc < wh)
                            bstore<T>(Gh[r * GP + cc] + ((r - kh == cc) ? T(1) : T(0)), dst,
                                      (uint32_t)(((kh + cc) * n + r) * (int)sizeof(T)));
                    }
                }
            }
        }
        __syncthreads();
    }
    return true;   // every pivot was diagonal: the last panel left inv(M) in place
}

// Dinv_i = inv(D_i) for any n <= 64*NR: ginv_body_wide_rx with diagonal
// pivots; a block whose check fails is flagged for k_fac_pivot.  LDS is dynamic.
constexpr int kInvThreads = 512;    // partial-pivoting inverse (k_fac_pivot): 8 waves per block
constexpr int kWideThreads = 1024;   // wide-panel inverse: 16 waves per block

template <typename T, int NR, int UB, bool REPLAY>
__global__ void __launch_bounds__(kWideThreads) k_fac_ginv(T *__restrict__ D, int64_t ld, T *__restrict__ Wk, int64_t ldw,
                                                   const int32_t *__restrict__ rows, int n,
                                                   int32_t *__restrict__ redo) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    __shared__ int32_t flag_sh;
    __shared__ __attribute__((aligned(16))) unsigned char pl_raw[sizeof(PanelLds<T, REPLAY>)];
    PanelLds<T, REPLAY> &pl = *reinterpret_cast<PanelLds<T, REPLAY> *>(pl_raw);
    const int blk = rows[blockIdx.x];
    T *M = D + (size_t)blk * ld;
    T *S = Wk + (size_t)blockIdx.x * ldw;
    // panels of GinvHalves<T>::H 16-column halves, pivot rows in registers (LDS: ginv_lds)
    constexpr int H = GinvHalves<T>::H;
    T *G = reinterpret_cast<T *>(smem_raw);                 // H * NP * 17
    const bool ok = ginv_body_wide_rx<T, NR, kWideThreads, UB, H, REPLAY>(M, S, n, G, pl, &flag_sh);
    if (!ok && threadIdx.x == 0) redo[blk] = 1;    // left to k_fac_pivot; M untouched
}

// Dinv_i = inv(D_i) for blocks of n <= 16*NT, one workgroup of 4 waves per
// block, pivoting on the diagonal.  The block lives in MFMA accumulator tiles.
// Wave v holds the whole tile columns tj = v + 4c (c < NT / 4), so that those
// tiles' operands sit at compile-time offsets from a per-lane base; the tiles
// of the last NT % 4 columns are dealt round-robin (tile e to wave e % 4), so
// that no wave holds more than ceil(NT^2 / 4) tiles.  Columns are processed in
// panels of 16:
//   1. the panel's tiles go to LDS (G), and so do the other tiles of the
//      panel's pivot rows k0..k0+15 (XP);
//   2. PanelLds::run takes the checked-diagonal Gauss-Jordan steps on the n x 16 panel,
//      which then holds C = [W on the pivot rows P, -A(r,P) W elsewhere], W
//      the inverse of the panel's pivot block;
//   3. every other column is updated at once, X += (C - E_P) X(P,:), one
//      rank-16 product on MFMA (E_P: ones at (k0 + j, j)), and the panel's
//      tiles take C, formed on MFMA as (C - E_P + E_P) I from a zero
//      accumulator (an accumulator written by VALU makes the compiler hold
//      every tile in arch VGPRs and copy them all in each panel).
// This is the unblocked in-place Gauss-Jordan reorganized, on diagonal pivots
// that pass the kPivTau threshold; a block where one fails is inverted with
// partial pivoting instead (ginv_pivot_body here, or left to k_fac_pivot).
//
// SB not void (n <= 48): the block is not read but made here, D_i = A_ii - sum_q L_q U_q
// with L_q = A_q Dinv_k, so that a level is one launch and not three.  Small blocks leave a
// level of few workgroups to three chains of launch, load and product (n = 40 FP32:
// p1 10 us, p2 13, inverse 11, with the gaps between them).  The row's workgroup takes its lower
// blocks in turn, the next one's operands on their way meanwhile; each product
// sums in the order of k_fac_p1 and k_fac_p2, so both ways give the same bits.  Whole
// factors, with the partial pivoting in the same launch: 31x17x13 n = 40 FP32 1.96 -> 1.43 ms
// (a level of up to 221 rows 36 us -> 22), FP64 2.38 -> 1.77; 4^3 FP64 0.37 -> 0.29; wide
// levels (40^3, up to 1200 rows) FP32 8.05 -> 7.49, FP64 9.69 -> 8.91; n = 5 at 30^3 2.75 ->
// 2.05.  Larger blocks have tiles enough to fill the chip and too many operands for one workgroup's LDS.
template <typename T, typename SB> struct RowIn {
    const double *Ab;             // A's blocks
    const SB *Ub;                 // the upper blocks (A's own, or their FP32 copies)
    T *L, *Wk;                    // Wk: a working slot per workgroup (as D's), for the partial pivoting
    const int32_t *lo_ptr, *lo_blk, *lo_col, *lo_tr, *diag;
    int64_t lda, ldu;
};
template <typename T> struct RowIn<T, void> {
    T *Wk;
    int32_t *redo;
};
// Whether a block that needs other pivots is inverted by k_fac_binv itself (a launch for
// that, which nearly always finds nothing to do, is 4.6 us a level).  In FP64 with 9 tile columns
// the code for it makes the compiler spill: 89 us instead of 78 at n = 135.
template <typename T, int NT> constexpr bool kPivotsHere = sizeof(T) == 4 || NT < 9;
constexpr int kRowN = 48;         // largest block of the fused form

// 48 x 48 values of a block from its slot, 16 bytes at a time: column (vector / (48 / V)), rows from V (vector % ..)
template <typename S> struct Fetched48 { Vec16<S> v[(kRowN * kRowN / VecN<S> + 255) / 256]; };
template <typename S>
__device__ __forceinline__ void fetch48(const S *__restrict__ B, int n, int top, Fetched48<S> &f) {
    constexpr int V = VecN<S>, PC = kRowN / V;
#pragma unroll
    for (int i = 0; i < (kRowN * PC + 255) / 256; ++i) {
        const int idx = threadIdx.x + 256 * i, cc = idx / PC, rr = (idx - cc * PC) * V;
        f.v[i] = *reinterpret_cast<const Vec16<S> *>(reinterpret_cast<const char *>(B) +
                                                     (uint32_t)(min(cc * n + rr, top - V) * (int)sizeof(S)));
    }
}
// into LDS column by column; zero where the index that the product sums over is n or more: the column
// (A operand) or the row (B operand)
template <bool AOP, typename T, typename S, int P>
__device__ __forceinline__ void store48(T (&X)[kRowN][P], const Fetched48<S> &f, int n) {
    constexpr int V = VecN<S>, PC = kRowN / V;
    typedef T out_t __attribute__((ext_vector_type(V)));
#pragma unroll
    for (int i = 0; i < (kRowN * PC + 255) / 256; ++i) {
        const int idx = threadIdx.x + 256 * i, cc = idx / PC, rr = (idx - cc * PC) * V;
        if (idx >= kRowN * PC) break;
        out_t o;
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = (AOP ? cc : rr + e) < n ? static_cast<T>(f.v[i].v[e]) : T(0);
        *reinterpret_cast<out_t *>(&X[cc][rr]) = o;
    }
}

template <typename T, int NT, typename SB = void, bool REPLAY = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
k_fac_binv(T *__restrict__ D, int64_t ld, const int32_t *__restrict__ rows, int n, int32_t *__restrict__ err,
           RowIn<T, SB> in) {
    constexpr bool ROW = !std::is_void<SB>::value;
    static_assert(!ROW || NT == kRowN / 16, "the fused form is for blocks of up to 48");
    constexpr int NP = 16 * NT;                  // padded size
    constexpr int NFC = NT / 4;                  // whole tile columns per wave
    constexpr int NFA = NFC > 0 ? NFC : 1;
    constexpr int NXT = (NT - 4 * NFC) * NT;     // tiles of the remaining columns
    constexpr int NX = (NXT + 3) / 4;            // of which one wave holds at most NX
    constexpr int NXA = NX > 0 ? NX : 1;
    constexpr int GP = 17;                       // LDS pitch of the panel (bank spread)
    constexpr int XPP = NP + 1;                  // LDS pitch of the pivot rows
    __shared__ T G[NP * GP];                     // panel in, C - E_P out
    __shared__ T XP[16 * XPP];                   // pivot rows of the other columns
    __shared__ __attribute__((aligned(16))) unsigned char pl_raw[sizeof(PanelLds<T, REPLAY>)];   // of the panel's steps
    PanelLds<T, REPLAY> &pl = *reinterpret_cast<PanelLds<T, REPLAY> *>(pl_raw);
    __shared__ int32_t miss_sh;
    typedef typename Mfma<T>::acc_t acc_t;
    const int blk = rows[blockIdx.x];
    T *M = D + (size_t)blk * ld;
    const int tid = threadIdx.x, lane0 = tid & 63;
    const int wv0 = __builtin_amdgcn_readfirstlane(tid >> 6);
    acc_t acc[NFA][NT];     // tile (ti, wave + 4c)
    acc_t accx[NXA];        // remaining tile e = wave + 4x: (e % NT, 4 NFC + e / NT)
    if constexpr (ROW) {
        constexpr int P = kRowN + 16 / (int)sizeof(T);
        typedef T vec_t __attribute__((ext_vector_type(4)));
        __shared__ __attribute__((aligned(16))) T X[kRowN][P], Y[kRowN][P];   // A operand [k][row], B operand [column][k]
        const int top = (n * n + 63) & ~63, q0 = in.lo_ptr[blk], q1 = in.lo_ptr[blk + 1];
        const int fr = lane0 & 15, fk = 4 * (lane0 >> 4), nt = (n + 15) / 16;   // nt: tiles that are not all padding
        auto used = [&](int e) { return e < NXT && e % NT < nt && e / NT < nt; };
        auto product = [&](int ti, int tj, acc_t &c) {
#pragma unroll
            for (int h = 0; h < kRowN / 16; ++h) {
                T a[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) a[e] = X[16 * h + fk + e][16 * ti + fr];
                const vec_t b = *reinterpret_cast<const vec_t *>(&Y[16 * tj + fr][16 * h + fk]);
#pragma unroll
                for (int e = 0; e < 4; ++e) c = Mfma<T>::run(a[e], b[e], c);
            }
        };
        double dv[NXA][4];
        const double *const Ad = in.Ab + (size_t)in.diag[blk] * in.lda;
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            const int e = min(wv0 + 4 * x, NXT - 1), ei = e % NT, ej = e / NT;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                dv[x][r] = Ad[min((16 * ej + fr) * n + 16 * ei + Mfma<T>::row(lane0, r), n * n - 1)];
            accx[x] = acc_t{0, 0, 0, 0};
        }
        if (q1 > q0) {
            Fetched48<double> fa;
            Fetched48<T> fd;
            Fetched48<SB> fu;
            auto fetch_ad = [&](int q) {
                fetch48<double>(in.Ab + (size_t)in.lo_blk[q] * in.lda, n, top, fa);
                fetch48<T>(D + (size_t)in.lo_col[q] * ld, n, top, fd);
            };
            auto fetch_u = [&](int q) { fetch48<SB>(in.Ub + (size_t)in.lo_tr[q] * in.ldu, n, top, fu); };
            fetch_ad(q0);
            fetch_u(q0);
            for (int q = q0; q < q1; ++q) {
                const int qn = min(q + 1, q1 - 1);          // (the last round reloads: no load under a branch)
                store48<true>(X, fa, n);
                store48<false>(Y, fd, n);
                __syncthreads();
                fetch_ad(qn);
                acc_t lt[NXA];
#pragma unroll
                for (int x = 0; x < NX; ++x) {
                    const int e = wv0 + 4 * x;
                    lt[x] = acc_t{0, 0, 0, 0};
                    if (used(e)) product(e % NT, e / NT, lt[x]);
                }
                __syncthreads();
                T *const Lq = in.L + (size_t)q * ld;
#pragma unroll
                for (int x = 0; x < NX; ++x) {
                    const int e = wv0 + 4 * x, col = 16 * (e / NT) + fr;
                    if (e < NXT)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int row = 16 * (e % NT) + Mfma<T>::row(lane0, r);
                            X[col][row] = col < n ? lt[x][r] : T(0);
                            if (row < n && col < n) Lq[col * n + row] = lt[x][r];
                        }
                }
                store48<false>(Y, fu, n);
                __syncthreads();
                fetch_u(qn);
#pragma unroll
                for (int x = 0; x < NX; ++x) {
                    const int e = wv0 + 4 * x;
                    if (used(e)) product(e % NT, e / NT, accx[x]);
                }
                __syncthreads();
            }
        }
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            const int e = wv0 + 4 * x, col = 16 * (e / NT) + fr;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * (e % NT) + Mfma<T>::row(lane0, r);
                const bool ok = e < NXT && row < n && col < n;
                accx[x][r] = ok ? static_cast<T>(dv[x][r]) - accx[x][r] : T(0);
                if (ok) M[col * n + row] = accx[x][r];      // for the partial pivoting
            }
        }
    }
    // a 32-bit byte offset from the block's (uniform) base keeps one VGPR per address
    auto ldM = [&](int row, int col, bool ok) -> T {
        return (ok && row < n && col < n) ? *reinterpret_cast<const T *>(
                   reinterpret_cast<const char *>(M) + (uint32_t)((col * n + row) * (int)sizeof(T))) : T(0);
    };
#pragma unroll
    for (int c = 0; c < NFC; ++c)
#pragma unroll
        for (int ti = 0; ti < NT; ++ti)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[c][ti][r] = ldM(16 * ti + Mfma<T>::row(lane0, r), 16 * (wv0 + 4 * c) + (lane0 & 15), true);
#pragma unroll
    for (int x = 0; x < NX; ++x) {
        const int e = wv0 + 4 * x, eti = e % NT, etj = 4 * NFC + e / NT;
#pragma unroll
        for (int r = 0; r < 4 && !ROW; ++r) accx[x][r] = ldM(16 * eti + Mfma<T>::row(lane0, r), 16 * etj + (lane0 & 15), e < NXT);
    }
    for (int e = tid; e < 16 * XPP; e += 256) XP[e] = T(0);
    if (tid == 0) miss_sh = 0;
    pl.start();
    // B operand of the identity: I[4kk + lane/16][lane%16]
    T ident[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) ident[kk] = (lane0 & 15) == 4 * kk + (lane0 >> 4) ? T(1) : T(0);
    __syncthreads();
    for (int kb = 0; kb < NT && 16 * kb < n; ++kb) {
        const int k0 = 16 * kb;
        const int w = min(16, n - k0);
        // wave and lane indices made opaque per panel: the LDS addresses below
        // are recomputed in each panel rather than hoisted out of the loop
        // (kept live across it they exceed the register file)
        int wv, lane;
        asm volatile("s_mov_b32 %0, %1" : "=s"(wv) : "s"(wv0));
        asm volatile("v_mov_b32 %0, %1" : "=v"(lane) : "v"(lane0));
        auto storeG = [&](const acc_t &v, int ti) {
#pragma unroll
            for (int r = 0; r < 4; ++r) G[(16 * ti + Mfma<T>::row(lane, r)) * GP + (lane & 15)] = v[r];
        };
        auto storeXP = [&](const acc_t &v, int tj) {
#pragma unroll
            for (int r = 0; r < 4; ++r) XP[Mfma<T>::row(lane, r) * XPP + 16 * tj + (lane & 15)] = v[r];
        };
        // 1. the panel's tile column to G, the pivot rows' other tiles to XP
#pragma unroll
        for (int c = 0; c < NFC; ++c) {
            const int tj = wv + 4 * c;
            if (tj == kb) {
#pragma unroll
                for (int ti = 0; ti < NT; ++ti) storeG(acc[c][ti], ti);
            } else {
#pragma unroll
                for (int ti = 0; ti < NT; ++ti)
                    if (ti == kb) storeXP(acc[c][ti], tj);
            }
        }
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            const int e = wv + 4 * x, eti = e % NT, etj = 4 * NFC + e / NT;
            if (e < NXT) {
                if (etj == kb) storeG(accx[x], eti);
                else if (eti == kb) storeXP(accx[x], etj);
            }
        }
        __syncthreads();
        // the pivot rows (B operands of step 3) are final now
        T b[NFA][4], bx[NXA][4];
#pragma unroll
        for (int c = 0; c < NFC; ++c)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) b[c][kk] = XP[(4 * kk + (lane >> 4)) * XPP + 16 * (wv + 4 * c) + (lane & 15)];
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            const int e = min(wv + 4 * x, NXT - 1), etj = 4 * NFC + e / NT;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) bx[x][kk] = XP[(4 * kk + (lane >> 4)) * XPP + 16 * etj + (lane & 15)];
        }
        // 2. panel Gauss-Jordan (checked diagonal pivots)
        if (pl.template run<4>(G, GP, NP, n, k0, w, &miss_sh)) break;
        // 3. X += (C - E_P) X(P,:) on MFMA; the panel's tiles take C
        auto ldA = [&](int ti, int kk) -> T { return G[(16 * ti + (lane & 15)) * GP + 4 * kk + (lane >> 4)]; };
        auto panel_tile = [&](const T (&av)[4], int ti) -> acc_t {
            acc_t r = {};
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int cc = 4 * kk + (lane >> 4);
                const T ae = av[kk] + ((ti == kb && (lane & 15) == cc && cc < w) ? T(1) : T(0));
                r = Mfma<T>::run(ae, ident[kk], r);
            }
            return r;
        };
        if (NFC > 0) {
            T a[NT][4];
#pragma unroll
            for (int ti = 0; ti < NT; ++ti)
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) a[ti][kk] = ldA(ti, kk);
#pragma unroll
            for (int c = 0; c < NFC; ++c) {
                if (wv + 4 * c == kb) {
#pragma unroll
                    for (int ti = 0; ti < NT; ++ti) acc[c][ti] = panel_tile(a[ti], ti);
                } else {
#pragma unroll
                    for (int ti = 0; ti < NT; ++ti)
#pragma unroll
                        for (int kk = 0; kk < 4; ++kk) acc[c][ti] = Mfma<T>::run(a[ti][kk], b[c][kk], acc[c][ti]);
                }
            }
        }
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            const int e = wv + 4 * x, eti = e % NT, etj = 4 * NFC + e / NT;
            if (e < NXT) {
                T ax[4];
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) ax[kk] = ldA(eti, kk);
                if (etj == kb) {
                    accx[x] = panel_tile(ax, eti);
                } else {
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk) accx[x] = Mfma<T>::run(ax[kk], bx[x][kk], accx[x]);
                }
            }
        }
        __syncthreads();
    }
    if (__builtin_amdgcn_readfirstlane(miss_sh)) {
        // another pivot than the diagonal was needed: M is untouched, and the block is
        // inverted with partial pivoting instead
        if constexpr (kPivotsHere<T, NT>) {
            __shared__ T prow_sh[16];
            __shared__ int32_t rowtag[NP], pivrow[NP], flag_sh;
            bool bad = false;
            ginv_pivot_body<T, (NP + 63) / 64, 256>(M, in.Wk + (size_t)blockIdx.x * ld, n, G, XP, prow_sh, rowtag, pivrow,
                                                    &flag_sh, &bad);
            if (tid == 0 && bad) atomicMin(err, blk);
        } else if (tid == 0) {
            in.redo[blk] = 1;
        }
        return;
    }
    // the lane index again, opaque to the compiler: the store offsets are then
    // recomputed here instead of being kept live (spilled) since the loads
    int lane2;
    asm volatile("v_mov_b32 %0, %1" : "=v"(lane2) : "v"(lane0));
    auto stM = [&](int row, int col, T v) {
        if (row < n && col < n)
            *reinterpret_cast<T *>(reinterpret_cast<char *>(M) + (uint32_t)((col * n + row) * (int)sizeof(T))) = v;
    };
#pragma unroll
    for (int c = 0; c < NFC; ++c)
#pragma unroll
        for (int ti = 0; ti < NT; ++ti)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                stM(16 * ti + Mfma<T>::row(lane2, r), 16 * (wv0 + 4 * c) + (lane2 & 15), acc[c][ti][r]);
#pragma unroll
    for (int x = 0; x < NX; ++x) {
        const int e = wv0 + 4 * x, eti = e % NT, etj = 4 * NFC + e / NT;
        if (e < NXT) {
#pragma unroll
            for (int r = 0; r < 4; ++r) stM(16 * eti + Mfma<T>::row(lane2, r), 16 * etj + (lane2 & 15), accx[x][r]);
        }
    }
}

// Partial-pivoting inverse of the blocks that k_fac_ginv or k_fac_binv flagged in
// redo[]; the other workgroups leave at once.
template <typename T, int NR>
__global__ void __launch_bounds__(kInvThreads) k_fac_pivot(T *__restrict__ D, int64_t ld, T *__restrict__ Wk, int64_t ldw,
                                                    const int32_t *__restrict__ rows, int n,
                                                    int32_t *__restrict__ err, int32_t *__restrict__ redo) {
    const int blk = rows[blockIdx.x];
    if (__builtin_amdgcn_readfirstlane(redo[blk]) == 0) return;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    const int NP = 16 * ((n + 15) / 16), XPP = NP + 1;
    T *G = reinterpret_cast<T *>(smem_raw);
    T *XP = G + (size_t)NP * 17;
    T *prow_sh = XP + (size_t)16 * XPP;
    int32_t *rowtag = reinterpret_cast<int32_t *>(prow_sh + 16);
    int32_t *pivrow = rowtag + NP;
    __shared__ int32_t flag_sh;
    bool bad = false;
    ginv_pivot_body<T, NR, kInvThreads>(D + (size_t)blk * ld, Wk + (size_t)blockIdx.x * ldw, n, G, XP, prow_sh,
                                        rowtag, pivrow, &flag_sh, &bad);
    if (threadIdx.x == 0) {
        redo[blk] = 0;
        if (bad) atomicMin(err, blk);
    }
}

// Dynamic LDS of k_fac_ginv (the wide panel's halves) and k_fac_pivot (one
// 16-column panel and its pivot rows); both kernels get the larger.
template <typename T, int NR>
size_t ginv_lds(int n) {
    const int NP = 16 * ((n + 15) / 16);
    const size_t pivot_form = sizeof(T) * ((size_t)NP * 17 + (size_t)16 * (NP + 1) + 16) + sizeof(int32_t) * 2 * (size_t)NP;
    const size_t wide = sizeof(T) * (size_t)GinvHalves<T>::H * NP * 17;
    return std::max(wide, pivot_form);
}

__device__ __forceinline__ cdg_bf16 to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);   // round to nearest even
    return static_cast<cdg_bf16>(u >> 16);
}

template <typename S> __device__ __forceinline__ S narrow(double v);
template <> __device__ __forceinline__ float narrow<float>(double v) { return static_cast<float>(v); }
template <> __device__ __forceinline__ cdg_bf16 narrow<cdg_bf16>(double v) { return to_bf16(static_cast<float>(v)); }

// Four narrowed values to dst[0..3] in one store (dst 8- or 16-byte aligned).
__device__ __forceinline__ void store4(float *dst, double a, double b, double c, double d) {
    *reinterpret_cast<float4 *>(dst) = make_float4((float)a, (float)b, (float)c, (float)d);
}
__device__ __forceinline__ void store4(cdg_bf16 *dst, double a, double b, double c, double d) {
    const uint32_t lo = (uint32_t)narrow<cdg_bf16>(a) | ((uint32_t)narrow<cdg_bf16>(b) << 16);
    const uint32_t hi = (uint32_t)narrow<cdg_bf16>(c) | ((uint32_t)narrow<cdg_bf16>(d) << 16);
    *reinterpret_cast<uint2 *>(dst) = make_uint2(lo, hi);
}

// U_u = (S) A_{up_blk[u]}   (the apply's copy of A's upper blocks).  One
// workgroup per block: 16-byte loads of two doubles, four values per thread and
// step, four steps' loads before their stores (slots start 512-byte aligned in
// A and 128-byte aligned in U).
template <typename S>
__global__ void __launch_bounds__(256) k_copy_upper(const double *__restrict__ Ab, int64_t lda, S *__restrict__ U,
                                                    int64_t ld, const int32_t *__restrict__ up_blk, int nup, int nn) {
    const int B = blockDim.x;
    for (int u = blockIdx.x; u < nup; u += gridDim.x) {
        const double2 *src = reinterpret_cast<const double2 *>(Ab + (size_t)up_blk[u] * lda);
        S *dst = U + (size_t)u * ld;
        const int n4 = nn / 4;
        int q = threadIdx.x;
        for (; q + 3 * B < n4; q += 4 * B) {
            double2 a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a[i] = src[2 * (q + i * B)];
                b[i] = src[2 * (q + i * B) + 1];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) store4(dst + 4 * (q + i * B), a[i].x, a[i].y, b[i].x, b[i].y);
        }
        for (; q < n4; q += B) {
            const double2 a = src[2 * q], b = src[2 * q + 1];
            store4(dst + 4 * q, a.x, a.y, b.x, b.y);
        }
        const double *srcd = reinterpret_cast<const double *>(src);
        for (int e = 4 * n4 + threadIdx.x; e < nn; e += B) dst[e] = narrow<S>(srcd[e]);
    }
}

__global__ void k_f32_to_bf16(const float *__restrict__ src, cdg_bf16 *__restrict__ dst, int64_t count) {
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < count; k += (int64_t)gridDim.x * blockDim.x)
        dst[k] = to_bf16(src[k]);
}

// BF16-stored factors are computed in FP32 and take the REPLAY panels.
template <typename T> constexpr bool kReplays = sizeof(T) == 4;

template <typename T, int NR>
int launch_ginv(cdg_ctx *ctx, cdg_prec *M, T *D, int64_t ld, const int32_t *rows, int nrows_lvl, int n,
                int32_t *err) {
    const size_t lds = ginv_lds<T, NR>(n);
    // Both kernels may take the LDS of the largest block this template serves
    // (n <= 64 NR, at most 320): set once per process, thread-safe (request-loop
    // workers launch concurrently), whatever block size comes first.
    // tiles each wave loads per round of the rank-16H update (two rounds' tiles
    // are in registers at once); CDG_GINV_TILES = 2, 4 or 8 overrides 2
    static const int ub = [] {
        const char *e = std::getenv("CDG_GINV_TILES");
        const int v = e ? std::atoi(e) : 2;
        return v <= 2 ? 2 : v <= 4 ? 4 : 8;
    }();
    static const void *const fns[2][3] = {
        {reinterpret_cast<const void *>(&k_fac_ginv<T, NR, 2, false>), reinterpret_cast<const void *>(&k_fac_ginv<T, NR, 4, false>),
         reinterpret_cast<const void *>(&k_fac_ginv<T, NR, 8, false>)},
        {reinterpret_cast<const void *>(&k_fac_ginv<T, NR, 2, kReplays<T>>), reinterpret_cast<const void *>(&k_fac_ginv<T, NR, 4, kReplays<T>>),
         reinterpret_cast<const void *>(&k_fac_ginv<T, NR, 8, kReplays<T>>)}};
    const void *fn = fns[M->precision == CDG_BF16][ub == 2 ? 0 : ub == 4 ? 1 : 2];
    static std::once_flag once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(once, [] {
        const int most = (int)ginv_lds<T, NR>(std::min(64 * NR, 320));
        auto set = [&](const void *f) {
            if (attr_err == hipSuccess)
                attr_err = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, most);
        };
        for (auto &r : fns)
            for (const void *f : r) set(f);
        set(reinterpret_cast<const void *>(&k_fac_pivot<T, NR>));
    });
    if (attr_err != hipSuccess)
        return cdg_fail(ctx, CDG_ERR_HIP, "hipFuncSetAttribute (block inverse LDS): %s", hipGetErrorString(attr_err));
    {
        T *Dp = D, *Wp = static_cast<T *>(M->inv_w);
        int64_t ldp = ld, ldw = M->ld;
        const int32_t *rp = rows;
        int np = n;
        int32_t *redo = M->d_redo;
        void *args[] = {&Dp, &ldp, &Wp, &ldw, &rp, &np, &redo};
        CDG_HIP_TRY(hipLaunchKernel(fn, dim3(nrows_lvl), dim3(kWideThreads), args, lds, ctx->stream));
    }
    CDG_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL((k_fac_pivot<T, NR>), dim3(nrows_lvl), dim3(kInvThreads), lds, ctx->stream, D, ld,
                       static_cast<T *>(M->inv_w), M->ld, rows, n, err, M->d_redo);
    CDG_HIP_TRY(hipGetLastError());
    return CDG_OK;
}

// Block-inverse kernel: 0 register-resident Gauss-Jordan (n <= 192), 1 blocked
// in registers with checked diagonal pivots (n <= 144), 2 blocked in global
// memory (any n <= 320; larger blocks always take it).  CDG_INV overrides
// the default, the fastest measured at 16^3: 1 up to n = 144, 0 above.
int inv_mode_env() {
    static const int mode = [] { const char *e = std::getenv("CDG_INV"); return e ? std::atoi(e) : -1; }();
    return mode;
}
template <typename T> int inv_mode(int n) {
    const int m = inv_mode_env();
    if (m >= 0) return m;
    return n <= 144 ? 1 : 0;
}

template <typename T>
int launch_inv(cdg_ctx *ctx, cdg_prec *M, T *D, int64_t ld, const int32_t *rows, int nrows_lvl, int n, int32_t *err) {
    if (!M->inv_w) return cdg_fail(ctx, CDG_ERR_STATE, "inverse scratch missing");
    const int mode = inv_mode<T>(n);
    if (n > 192 || mode == 2) {
        if (n <= 64) return launch_ginv<T, 1>(ctx, M, D, ld, rows, nrows_lvl, n, err);
        if (n <= 192) return launch_ginv<T, 3>(ctx, M, D, ld, rows, nrows_lvl, n, err);
        if (n <= 256) return launch_ginv<T, 4>(ctx, M, D, ld, rows, nrows_lvl, n, err);
        return launch_ginv<T, 5>(ctx, M, D, ld, rows, nrows_lvl, n, err);
    }
    dim3 grid(nrows_lvl), block(256);
    if (mode == 1 && n <= 144) {
        const RowIn<T, void> in{static_cast<T *>(M->inv_w), M->d_redo};
        auto go = [&](auto rp) {
            constexpr bool RP = decltype(rp)::value;
            if (n <= 96) hipLaunchKernelGGL((k_fac_binv<T, 6, void, RP>), grid, block, 0, ctx->stream, D, ld, rows, n, err, in);
            else hipLaunchKernelGGL((k_fac_binv<T, 9, void, RP>), grid, block, 0, ctx->stream, D, ld, rows, n, err, in);
        };
        if (M->precision == CDG_BF16) go(std::integral_constant<bool, kReplays<T>>{});
        else go(std::false_type{});
        CDG_HIP_TRY(hipGetLastError());
        if (n <= 96 || kPivotsHere<T, 9>) return CDG_OK;
        const size_t lds = ginv_lds<T, 3>(n);
        hipLaunchKernelGGL((k_fac_pivot<T, 3>), grid, dim3(kInvThreads), lds, ctx->stream, D, ld,
                           static_cast<T *>(M->inv_w), M->ld, rows, n, err, M->d_redo);
        CDG_HIP_TRY(hipGetLastError());
        return CDG_OK;
    }
    if (n <= 48) hipLaunchKernelGGL((k_fac_inv<T, 3>), grid, block, 0, ctx->stream, D, ld, rows, n, err);
    else if (n <= 96) hipLaunchKernelGGL((k_fac_inv<T, 6>), grid, block, 0, ctx->stream, D, ld, rows, n, err);
    else if (n <= 144) hipLaunchKernelGGL((k_fac_inv<T, 9>), grid, block, 0, ctx->stream, D, ld, rows, n, err);
    else if (n <= 192) hipLaunchKernelGGL((k_fac_inv<T, 12>), grid, block, 0, ctx->stream, D, ld, rows, n, err);
    else return cdg_fail(ctx, CDG_ERR_UNSUPPORTED, "block inverse for n=%d not built", n);
    CDG_HIP_TRY(hipGetLastError());
    return CDG_OK;
}

// Tile edge of the factor GEMMs: 64 above n = 192 (320 = 5 x 64), else 48
// (n = 135: 3 x 48 = 144, where 64-edge tiles would pad to 192).
inline bool gemm_wide(int n) { return n > 192; }

template <typename T, int TM>
int fold_all_tm(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const T *D) {
    const int n = M->n, tiles = (n + TM - 1) / TM;
    const int u1 = M->nup;
    const dim3 blk(Geo<TM>::GT);
    if (std::is_same<T, float>::value && M->precision == CDG_FP32 && M->U)
        // the upper blocks' FP32 copies (slot u; the values the FP64 reads convert to): half the bytes
        hipLaunchKernelGGL((k_fac_p1<T, float, TM>), dim3(xcd_grid(u1, tiles * tiles)), blk, 0, ctx->stream,
                           static_cast<const float *>(M->U), M->ld, static_cast<T *>(M->W), D, M->ld, M->d_up_all, u1,
                           M->d_up_all, M->d_up_col, n, tiles);
    else
        hipLaunchKernelGGL((k_fac_p1<T, double, TM>), dim3(xcd_grid(u1, tiles * tiles)), blk, 0, ctx->stream,
                           A->blocks, A->ld, static_cast<T *>(M->W), D, M->ld, M->d_up_all, u1, M->d_up_blk,
                           M->d_up_col, n, tiles);
    CDG_HIP_TRY(hipGetLastError());
    return CDG_OK;
}

template <typename T>
int fold_all(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, const T *D) {
    if (M->nup == 0) return CDG_OK;
    return gemm_wide(M->n) ? fold_all_tm<T, 64>(ctx, M, A, D) : fold_all_tm<T, 48>(ctx, M, A, D);
}

// One level's GEMMs: L for the level's lower entries, then the rows' D.
template <typename T, int TM>
int gemm_level(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, T *L, T *D, const float *Ub32, int q0, int q1, int r0,
               int r1) {
    const int n = M->n, tiles = (n + TM - 1) / TM;
    const dim3 blk(Geo<TM>::GT);
    if (q1 > q0) {
        hipLaunchKernelGGL((k_fac_p1<T, double, TM>), dim3(xcd_grid(q1 - q0, tiles * tiles)), blk, 0, ctx->stream,
                           A->blocks, A->ld, L, D, M->ld, M->d_lev_lo + q0, q1 - q0, M->d_lo_blk, M->d_lo_col, n,
                           tiles);
        CDG_HIP_TRY(hipGetLastError());
    }
    if (r1 > r0) {
        if (Ub32)   // FP32 factor: the upper blocks' FP32 copies (the same values the FP64 reads convert to)
            hipLaunchKernelGGL((k_fac_p2<T, float, TM>), dim3(xcd_grid(r1 - r0, tiles * tiles)), blk, 0,
                               ctx->stream, A->blocks, A->ld, Ub32, M->ld, L, D, M->ld, M->d_lev_rows + r0, r1 - r0,
                               M->d_lo_ptr, M->d_lo_tru, M->d_diag, n, tiles);
        else
            hipLaunchKernelGGL((k_fac_p2<T, double, TM>), dim3(xcd_grid(r1 - r0, tiles * tiles)), blk, 0,
                               ctx->stream, A->blocks, A->ld, A->blocks, A->ld, L, D, M->ld, M->d_lev_rows + r0,
                               r1 - r0, M->d_lo_ptr, M->d_lo_tr, M->d_diag, n, tiles);
        CDG_HIP_TRY(hipGetLastError());
    }
    return CDG_OK;
}

// One level of blocks of up to 48 as one launch (k_fac_binv's fused form).
template <typename T>
int row_level(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, T *L, T *D, const float *Ub32, int r0, int r1) {
    const int32_t *rows = M->d_lev_rows + r0;
    auto go = [&](auto in) {
        typedef typename std::remove_const<typename std::remove_pointer<decltype(in.Ub)>::type>::type SB;
        in.Ab = A->blocks;
        in.lda = A->ld;
        in.L = L;
        in.Wk = static_cast<T *>(M->inv_w);
        in.lo_ptr = M->d_lo_ptr;
        in.lo_blk = M->d_lo_blk;
        in.lo_col = M->d_lo_col;
        in.diag = M->d_diag;
        // (FP32 from A's FP64 blocks: BF16 storage)
        constexpr bool RP = sizeof(T) == 4 && std::is_same<SB, double>::value;
        hipLaunchKernelGGL((k_fac_binv<T, kRowN / 16, SB, RP>), dim3(r1 - r0), dim3(256), 0, ctx->stream, D, M->ld, rows, M->n,
                           M->d_err, in);
    };
    bool done = false;
    if constexpr (sizeof(T) == 4)
        if (Ub32) {
            RowIn<T, float> in{};
            in.Ub = Ub32;
            in.ldu = M->ld;
            in.lo_tr = M->d_lo_tru;
            go(in);
            done = true;
        }
    if (!done) {
        RowIn<T, double> in{};
        in.Ub = A->blocks;
        in.ldu = A->ld;
        in.lo_tr = M->d_lo_tr;
        go(in);
    }
    CDG_HIP_TRY(hipGetLastError());
    return CDG_OK;
}

template <typename T>
int factor_levels(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, T *L, T *D, const float *Ub32) {
    const int n = M->n;
    const bool fold = M->apply_mode == CDG_APPLY_FOLDED && M->W && M->precision != CDG_BF16;
    for (int l = 0; l < M->nlev; ++l) {
        const int q0 = M->lev_lo_ptr[l], q1 = M->lev_lo_ptr[l + 1];
        const int r0 = M->lev_row_ptr[l], r1 = M->lev_row_ptr[l + 1];
        if (n <= kRowN && inv_mode<T>(n) == 1) {
            int e = r1 > r0 ? row_level<T>(ctx, M, A, L, D, Ub32, r0, r1) : CDG_OK;
            if (e) return e;
            continue;
        }
        int e = gemm_wide(n) ? gemm_level<T, 64>(ctx, M, A, L, D, Ub32, q0, q1, r0, r1)
                             : gemm_level<T, 48>(ctx, M, A, L, D, Ub32, q0, q1, r0, r1);
        if (e) return e;
        if (r1 > r0) {
            e = launch_inv<T>(ctx, M, D, M->ld, M->d_lev_rows + r0, r1 - r0, n, M->d_err);
            if (e) return e;
        }
    }
    if (fold) {   // W = U Dinv for all upper blocks, one batched launch
        int e = fold_all<T>(ctx, M, A, D);
        if (e) return e;
        M->w_ready = 1;
    }
    return CDG_OK;
}


}  // namespace

int launch_ilu_factor(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A, int32_t *bad_row) {
    const int n = M->n;
    if (n > 320) return cdg_fail(ctx, CDG_ERR_UNSUPPORTED, "ILU factor for block size %d not built (n <= 320)", n);
    if (!M->d_redo) {
        int e = dev_alloc(ctx, (void **)&M->d_redo, sizeof(int32_t) * std::max(1, M->nrows));
        if (e) return e;
        M->owned.push_back({M->d_redo, sizeof(int32_t) * std::max(1, M->nrows)});
        CDG_HIP_TRY(hipMemsetAsync(M->d_redo, 0, sizeof(int32_t) * std::max(1, M->nrows), ctx->stream));
    }
    if (!M->inv_w) {   // global working slots of the block inverse, one per row of a level
        int maxrows = 1;
        for (int l = 0; l < M->nlev; ++l) maxrows = std::max(maxrows, M->lev_row_ptr[l + 1] - M->lev_row_ptr[l]);
        const size_t bytes = (M->precision == CDG_FP64 ? 8 : 4) * (size_t)maxrows * M->ld;
        int e = dev_alloc(ctx, &M->inv_w, bytes);
        if (e) return e;
        M->owned.push_back({M->inv_w, bytes});
    }
    const int32_t big = 0x7fffffff;
    CDG_HIP_TRY(hipMemcpyAsync(M->d_err, &big, sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream));
    const int nn = n * n;
    // the FP32/BF16 copies of A's upper blocks (read by the backward sweep; the
    // FP32 factor's phase 2 reads its U_q from them too)
    if (M->precision != CDG_FP64 && M->nup > 0) {
        const dim3 grid(std::min(M->nup, 16384));
        if (M->precision == CDG_FP32)
            hipLaunchKernelGGL(k_copy_upper<float>, grid, dim3(256), 0, ctx->stream, A->blocks, A->ld,
                               static_cast<float *>(M->U), M->ld, M->d_up_blk, M->nup, nn);
        else
            hipLaunchKernelGGL(k_copy_upper<cdg_bf16>, grid, dim3(256), 0, ctx->stream, A->blocks, A->ld,
                               static_cast<cdg_bf16 *>(M->U), M->ld, M->d_up_blk, M->nup, nn);
        CDG_HIP_TRY(hipGetLastError());
    }
    int e = CDG_OK;
    if (M->precision == CDG_FP64) {
        e = factor_levels<double>(ctx, M, A, static_cast<double *>(M->L), static_cast<double *>(M->Dinv), nullptr);
    } else if (M->precision == CDG_FP32) {
        e = factor_levels<float>(ctx, M, A, static_cast<float *>(M->L), static_cast<float *>(M->Dinv),
                                 static_cast<const float *>(M->U));
    } else {
        e = factor_levels<float>(ctx, M, A, M->L32, M->D32, nullptr);
    }
    if (e) return e;
    if (M->precision == CDG_BF16) {
        const int64_t cl = (int64_t)M->nlo * M->ld, cd = (int64_t)M->nrows * M->ld;
        if (cl) hipLaunchKernelGGL(k_f32_to_bf16, dim3(2048), dim3(256), 0, ctx->stream, M->L32,
                                   static_cast<cdg_bf16 *>(M->L), cl);
        if (cd) hipLaunchKernelGGL(k_f32_to_bf16, dim3(2048), dim3(256), 0, ctx->stream, M->D32,
                                   static_cast<cdg_bf16 *>(M->Dinv), cd);
        CDG_HIP_TRY(hipGetLastError());
    }
    int32_t err = big;
    CDG_HIP_TRY(hipMemcpyAsync(&err, M->d_err, sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
    CDG_HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (err != big) {
        if (bad_row) *bad_row = err;
        return cdg_fail(ctx, CDG_ERR_SINGULAR, "singular diagonal block in row %d", err);
    }
    return CDG_OK;
}

template <int TM>
int fold_left_tm(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A) {
    const int tiles = (M->n + TM - 1) / TM;
    hipLaunchKernelGGL(k_fold_left<TM>, dim3(xcd_grid(M->nup, tiles * tiles)), dim3(Geo<TM>::GT), 0, ctx->stream, M->D32,
                       M->ld, A->blocks, A->ld, M->d_up_row, M->d_up_blk, M->nup, static_cast<cdg_bf16 *>(M->W), M->n,
                       tiles);
    CDG_HIP_TRY(hipGetLastError());
    return CDG_OK;
}

int launch_fold_left(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A) {
    if (M->nup == 0) return CDG_OK;
    return gemm_wide(M->n) ? fold_left_tm<64>(ctx, M, A) : fold_left_tm<48>(ctx, M, A);
}

int launch_fold_all(cdg_ctx *ctx, cdg_prec *M, const cdg_mat *A) {
    if (!M->W) return cdg_fail(ctx, CDG_ERR_STATE, "folded schedule without W storage");
    if (M->precision == CDG_FP64) return fold_all<double>(ctx, M, A, static_cast<const double *>(M->Dinv));
    if (M->precision == CDG_FP32) return fold_all<float>(ctx, M, A, static_cast<const float *>(M->Dinv));
    return cdg_fail(ctx, CDG_ERR_UNSUPPORTED, "folded schedule: FP64 and FP32 factors only");
}
