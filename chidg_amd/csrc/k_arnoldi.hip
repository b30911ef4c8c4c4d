// The vector part of one FGMRES step (type_fgmres.f90:191-264), for one right-hand
// side or several ("lanes") in lockstep:
//
//   CGS    h_i = v_i . w, w -= sum h_i v_i, ||w||; the second pass when the
//          selective re-orthogonalization test asks for it; v_{j+1} = w / ||w||
//   MGS    the same with one product and one update per basis vector
//   start  r0 = b - A x0, ||r0||, v_1 = r0 / ||r0||                  (:160-163)
//   norm   ||b - A x|| (the residual reported at the end)
//
// then the lane's rotations, residual estimate and stopping test, all on the device: the
// host queues the next step and watches a word in pinned memory one step behind.
//
// What bounds it.  The basis is read from cache or HBM three times (16^3 P2: 4.4 MB a
// vector); below about that size launches are the cost.  So each phase is one launch
// that adds up the previous one's partial products (every workgroup by itself, in the
// same order: 270 x 31 numbers at 16^3 P2, against 12 ns per workgroup for a counter that would find
// the last one), does what they ask for (w -= sum h_i v_i) and multiplies what it then
// holds in registers (v_i . w, w . w).  CGS takes three launches and the scaling one
// more, not two products, two updates, four reductions, a scaling and a host round trip.
// Measured: with 28 vectors, two passes, 8.5 + 13 + 9.4 + 4.9 us at 4^3 P1 (2560
// values) and 35 + 55 + 36 + 8 us at 16^3 P2 (124 MB of basis a phase: 3.5 to 4.5 TB/s);
// whole solves against the separate launches: 4^3 P1 FP64 3.39 -> 2.90 ms, 8^3 P2 Newton
// step 16.1 -> 14.9, nested default solve 11.7 -> 9.7, eight right-hand sides at
// 10x9x8 P2 10.6 -> 8.9, 16^3 P2 unchanged (56.4 and 73.9).
#include "cdg_internal.h"

#include <algorithm>
#include <cstring>

namespace {

constexpr int AT = 512;            // threads per workgroup
constexpr int AW = AT / 64;
constexpr int kChunk = 64;         // basis vectors per LDS round
constexpr int kMaxG = 512;         // slices of a lane at most

struct __attribute__((packed, aligned(8))) D2 { double x, y; };

__device__ __forceinline__ double wsum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
// Sums of eight values over the 64 lanes: each exchange halves the values a lane still
// carries (10 exchanges, not 48).  Returns value (lane >> 3)'s total, the same in
// the eight lanes of that group.
__device__ __forceinline__ double wsum8(double (&v)[8], int lane) {
#pragma unroll
    for (int s = 4, o = 32; s > 0; s >>= 1, o >>= 1) {
        const bool up = (lane & o) != 0;
#pragma unroll
        for (int i = 0; i < s; ++i) {
            const double give = up ? v[i] : v[i + s], keep = up ? v[i + s] : v[i];
            v[i] = keep + __shfl_xor(give, o, 64);
        }
    }
    double t = v[0];
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    return t;
}

__device__ __forceinline__ double rdlane(double v, int l) {
    const int2 i = __builtin_bit_cast(int2, v);
    return __builtin_bit_cast(double, int2{__builtin_amdgcn_readlane(i.x, l), __builtin_amdgcn_readlane(i.y, l)});
}

// Numbers of a step's sums.  CGS: phase 0 holds the jj products and w.w before,
// phase 1 the second products and w.w, phase 2 the last w.w.  MGS: two values per
// phase, the product and w.w.  start, norm: w.w is number 0.
__device__ __forceinline__ int xid_h1(bool mgs, int m, int i) { return mgs ? 2 * i : i; }
__device__ __forceinline__ int xid_h2(bool mgs, int m, int jj, int i) { return mgs ? 2 * (jj + i) : m + 2 + i; }
__device__ __forceinline__ int xid_nb2(bool mgs, int jj) { return mgs ? 1 : jj; }
__device__ __forceinline__ int xid_norm(bool mgs, int m, int jj, bool second) {
    return mgs ? 2 * (second ? 2 * jj : jj) + 1 : second ? 2 * (m + 2) : m + 2 + jj;
}

// Phase ph of a step on slice blockIdx.x of lane blockIdx.y.  NI element pairs per thread
// and pass over the slice.  Phases of the second pass do nothing for lanes whose
// test did not ask for it (ARN_SECOND, set by workgroup 0 in the phase before).
template <int NI>
__global__ void __launch_bounds__(AT) k_arn_pass(ArnArgs a, int ph) {
    __shared__ double sh[AW][kChunk + 1];
    __shared__ double hsh[kChunk + 2];
    constexpr int U = 8 / NI;                               // basis vectors per load
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int jj = a.jj, G = a.G, m = a.m, s = blockIdx.x, l = blockIdx.y;
    const bool mgs = a.mode == ARN_MGS, steps = a.mode <= ARN_MGS, lone = a.len < 2;
    int *const st = a.st + l * ARN_NST;
    // lanes that take no part: stopped ones, and those done before this cycle
    if (steps ? !st[ARN_ACTIVE] : a.mode == ARN_START && !a.first && st[ARN_DONE]) return;
    if (ph == 0 && s == 0 && tid == 0) a.stamp[2] = wall_clock64();
    const bool extra = mgs ? ph > jj : ph == 2;             // part of the second pass
    if (extra && !st[ARN_SECOND]) return;
    double *const sums = a.sums + (int64_t)l * a.nx, *const part = a.part + (int64_t)l * a.nx * G;
    double x[NI][2];
    // ranges of this phase's updates and products, the numbers of their values, w.w's (or -1)
    int u0 = 0, u1 = 0, uid = 0, d0 = 0, nd = 0, did = 0, nid = -1;
    if (!steps) {
        nid = 0;
    } else if (!mgs) {
        if (ph == 0) { nd = jj; nid = jj; }
        else if (ph == 1) { u1 = jj; nid = m + 2 + jj; nd = jj; did = m + 2; }
        else { u1 = jj; uid = m + 2; nid = 2 * (m + 2); }
    } else {
        const int q = ph <= jj ? ph : ph - jj;      // vector of this phase's product
        if (ph > 0) { u0 = q - 1; u1 = q; uid = 2 * (ph - 1); }
        if (ph == 0) { nd = 1; nid = 1; }
        else if (ph == jj) { nid = 2 * jj + 1; nd = 1; did = 2 * jj; }
        else if (ph == 2 * jj) nid = 4 * jj + 1;
        else { d0 = q; nd = 1; did = 2 * ph; }
    }
    // the slice: n1 values from w on; 32-bit offsets in it (a slice of one value past the first
    // loads the pair before it)
    const int64_t e0 = (int64_t)s * a.slice;
    const int n1 = (int)min((int64_t)a.slice, a.len - e0), low = n1 == 1 && s > 0 ? 1 : 0;
    const char *const Vb = reinterpret_cast<const char *>(a.V + (size_t)l * a.len + e0 - low);
    double *const w = a.w + (size_t)l * a.len + e0;
    const size_t vstep = (size_t)a.nl * a.len * sizeof(double);
    // Sums of the previous launch's partials, numbers id .. id + nv - 1, into hsh (every
    // workgroup adds them up itself; workgroup 0 keeps them).  A wavefront adds four numbers at
    // a time.
    auto sum4 = [&](int id, int cnt, double (&v)[4]) {
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = 0.0;
        const double *const p = part + (int64_t)id * G;
        for (int g = lane; g < G; g += 64)
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] += p[(int64_t)min(c, cnt - 1) * G + g];
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = wsum(v[c]);
    };
    auto total = [&](int id, int nv) {
        __syncthreads();
        for (int i = 4 * wave; i < kChunk; i += 4 * AW) {
            double v[4] = {0.0, 0.0, 0.0, 0.0};
            if (i < nv) sum4(id + i, nv - i, v);
            if (lane < 4 && i + lane < kChunk) {
                const double o = lane == 0 ? v[0] : lane == 1 ? v[1] : lane == 2 ? v[2] : v[3];
                hsh[i + lane] = i + lane < nv ? o : 0.0;
                if (s == 0 && i + lane < nv) sums[id + i + lane] = o;
            }
        }
        __syncthreads();
    };
    bool ready = false;                                     // hsh holds the coefficients of the updates
    if (steps && ph == (mgs ? jj : 1)) {
        // whether the second orthogonalization pass runs: sum |h_i| / ||w before|| >= 1
        // (type_fgmres.f90:212-223)
        double crit = 0.0, nb2 = 0.0;
        for (int v0 = 0; !mgs && v0 <= jj; v0 += kChunk) {  // the products, then w.w
            total(v0, min(kChunk, jj + 1 - v0));
            crit += wsum(v0 + lane < jj ? fabs(hsh[lane]) : 0.0);
            nb2 = hsh[min(jj - v0, kChunk - 1)];
        }
        if (mgs) {
            double v[4];
            sum4(xid_nb2(mgs, jj), 1, v);
            nb2 = v[0];
            total(uid, 1);
            for (int i0 = 0; i0 < jj - 1; i0 += 64) crit += wsum(i0 + lane < jj - 1 ? fabs(sums[xid_h1(mgs, m, i0 + lane)]) : 0.0);
            crit += fabs(hsh[0]);
        }
        ready = mgs || jj < kChunk;
        const bool second = crit / sqrt(nb2) >= 1.0;
        if (!second) nd = 0;
        if (s == 0 && tid == 0) {
            st[ARN_SECOND] = second;
            st[ARN_RUN] = (int)a.seq;                       // this step's last launch takes the lane
        }
    }
    const int np = nd + (nid >= 0 ? 1 : 0);
    const bool whole = n1 <= 2 * AT * NI;           // one pass covers the slice
    bool keep = false;                              // x holds the slice
    for (int c0 = 0; c0 < max(np, 1); c0 += kChunk) {
        const int nc = min(kChunk, np - c0);
        for (int b0 = 0; b0 < n1; b0 += 2 * AT * NI) {
            uint32_t el[NI];
            bool hi[NI];                            // odd end: the pair's address is one element low
#pragma unroll
            for (int q = 0; q < NI; ++q) {
                const int e = b0 + 2 * (q * AT + tid) + low, top = max(n1 + low - 2, 0);
                el[q] = (uint32_t)min(e, top) * (uint32_t)sizeof(double);
                hi[q] = e > top;
            }
            // U vectors from v0 on, those past `last` read as the last
            auto load = [&](D2 (&d)[U][NI], int v0, int last) {
#pragma unroll
                for (int c = 0; c < U; ++c) {
                    const char *vp = Vb + (size_t)min(v0 + c, last) * vstep;
#pragma unroll
                    for (int q = 0; q < NI; ++q) {
                        d[c][q] = *reinterpret_cast<const D2 *>(vp + el[q]);
                        if (lone) d[c][q].y = d[c][q].x;
                        if (hi[q]) d[c][q].x = d[c][q].y;
                    }
                }
            };
            // (vectors are loaded as soon as the registers of the last ones are free)
            const bool ups = c0 == 0 && u1 > u0;
            D2 d[U][NI];
            const int dlast = max(d0 + nd - 1, 0);
            load(d, ups ? u0 : d0 + c0, ups ? u1 - 1 : dlast);
            if (!keep) {
                const double *const b = a.b + (size_t)l * a.len + e0;
                const double *const ax = a.ax ? a.ax + (size_t)l * a.len + e0 : nullptr;
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    const int e = b0 + 2 * (q * AT + tid);
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        x[q][i] = 0.0;
                        if (e + i < n1) {
                            x[q][i] = steps ? w[e + i] : b[e + i] - (ax ? ax[e + i] : 0.0);   // r = b - A x0
                            if (a.mode == ARN_START) w[e + i] = x[q][i];
                        }
                    }
                }
            }
            if (ups) {
                for (int v0 = u0; v0 < u1; v0 += kChunk) {
                    const int nv = min(kChunk, u1 - v0);
                    if (!ready) total(uid + (v0 - u0), nv);
                    ready = u1 - u0 <= kChunk;
#pragma unroll 1
                    for (int i = 0; i < nv; i += U) {
#pragma unroll
                        for (int c = 0; c < U; ++c) {
                            const double hv = i + c < nv ? hsh[i + c] : 0.0;
#pragma unroll
                            for (int q = 0; q < NI; ++q) {
                                x[q][0] -= hv * d[c][q].x;
                                x[q][1] -= hv * d[c][q].y;
                            }
                        }
                        load(d, v0 + i + U, u1 - 1);
                    }
                }
                load(d, d0, dlast);
#pragma unroll
                for (int q = 0; q < NI; ++q) {
                    const int e = b0 + 2 * (q * AT + tid);
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        if (e + i < n1) w[e + i] = x[q][i];
                        else x[q][i] = 0.0;         // past the end: out of every product
                    }
                }
            }
#pragma unroll 1
            for (int g = 0; g < nc; g += 8) {
                double acc[8];
#pragma unroll
                for (int v0 = 0; v0 < 8; v0 += U) {
#pragma unroll
                    for (int c = 0; c < U; ++c) {
                        // the product of w with itself reads w's registers
                        const bool vec = c0 + g + v0 + c < nd;
                        double t = 0.0;
#pragma unroll
                        for (int q = 0; q < NI; ++q) {
                            t += x[q][0] * (vec ? d[c][q].x : x[q][0]);
                            t += x[q][1] * (vec ? d[c][q].y : x[q][1]);
                        }
                        acc[v0 + c] = t;
                    }
                    load(d, d0 + c0 + g + v0 + U, dlast);
                }
                const double t = wsum8(acc, lane);
                if ((lane & 7) == 0) {              // (each wavefront its own row)
                    double *const o = &sh[wave][g + (lane >> 3)];
                    *o = b0 == 0 ? t : *o + t;
                }
            }
        }
        __syncthreads();
        if (tid < nc) {
            double v = sh[0][tid];
#pragma unroll
            for (int q = 1; q < AW; ++q) v += sh[q][tid];
            const int i = c0 + tid, id = i < nd ? did + i : nid;
            part[(int64_t)id * G + s] = v;
        }
        __syncthreads();
        keep = keep || whole;                       // (x is up to date for the next round)
    }
}

// The step's last launch: v = w / ||w||, and (workgroup 0 of a lane) the rotations and
// the stopping test.
__global__ void __launch_bounds__(256) k_arn_finish(ArnArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, jj = a.jj, m = a.m, l = blockIdx.y;
    const bool mgs = a.mode == ARN_MGS, steps = a.mode <= ARN_MGS;
    int *const st = a.st + l * ARN_NST;
    double *const sc = a.sc + l * ARN_NSC;
    auto put = [](auto *pp, auto v) { __hip_atomic_store(pp, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
    // (a step's passes marked their lanes: the state itself changes here)
    const bool runs = steps ? st[ARN_RUN] == (int)a.seq : !(a.mode == ARN_START && !a.first && st[ARN_DONE]);
    if (!runs) {
        if (blockIdx.x == 0 && tid == 0) {                  // say again how the lane ended
            const double res = sc[ARN_RES];
            uint64_t word = (uint64_t)a.seq << 32 | (uint64_t)(uint32_t)st[ARN_NVECS] << ARN_W_BITS | (isfinite(res) ? 0 : ARN_W_ERR);
            if (st[ARN_CONV] || !(res > a.tol)) word |= ARN_W_DONE;
            put(&a.hres[l].word, word);
        }
        return;
    }
    const double *const h = a.sums + (int64_t)l * a.nx;
    const bool second = steps && st[ARN_SECOND];
    double ww = 0.0;
    const double *const pn = a.part + ((int64_t)l * a.nx + (steps ? xid_norm(mgs, m, jj, second) : 0)) * a.G;
    for (int g = lane; g < a.G; g += 64) ww += pn[g];
    const double hn = sqrt(wsum(ww));
    if (blockIdx.x > 0) {
        double *const w = a.w + (size_t)l * a.len;
        for (int64_t e = (int64_t)(blockIdx.x - 1) * 256 + tid; e < a.len; e += (int64_t)(gridDim.x - 1) * 256) w[e] = w[e] / hn;
        return;
    }
    if (tid >= 64) return;
    // one wavefront: column j of H rotated, the next rotation, the stopping test
    double *const cs = a.cs + (size_t)l * a.hlen, *const sn = a.sn + (size_t)l * a.hlen;
    double *const p = a.p + (size_t)l * a.hlen;
    double *const R = a.R + (size_t)l * a.rlen + (size_t)(jj - 1) * jj / 2;   // packed columns
    auto col = [&](int i) { return h[xid_h1(mgs, m, i)] + (second ? h[xid_h2(mgs, m, jj, i)] : 0.0); };
    double res = hn;
    int conv = 0, err = 0, active = 1;
    if (steps) {
#pragma clang fp contract(off)
        const int j = jj - 1;
        double run = col(0);                            // H(i,j), rotated as far as i
        for (int i0 = 0; i0 < j; i0 += 64) {
            const int i = i0 + lane, nq = min(64, j - i0);
            double c = 0.0, s1 = 0.0, hx = 0.0, out = 0.0;
            if (i < j) {
                c = cs[i];
                s1 = sn[i];
                hx = col(i + 1);
            }
            for (int q = 0; q < nq; ++q) {
                const double cq = rdlane(c, q), sq = rdlane(s1, q), hq = rdlane(hx, q);
                const double hij = cq * run + sq * hq;
                run = -sq * run + cq * hq;
                if (lane == q) out = hij;
            }
            if (i < j) R[i] = out;
        }
        if (lane == 0) {
            const double gam = hypot(run, hn);
            const double c = run / gam, s1 = hn / gam;
            cs[j] = c;
            sn[j] = s1;
            R[j] = gam;
            const double pj = p[j];
            p[j] = c * pj;
            p[j + 1] = -s1 * pj;
            res = fabs(-s1 * pj);
            const int it = ++st[ARN_NITER];
            st[ARN_NVECS] = jj;
            if (second) {
                ++st[ARN_NREORTH];
                ++st[ARN_NREALL];
            }
            const bool ca = res < a.tol, cr = (res / sc[ARN_R0INIT]) < a.rtol, cn = it >= a.nmax && a.nmax > 0;
            if (!isfinite(res)) err = 1;
            else if (ca || cr || cn) conv = 1;
            active = !err && !conv;
        }
    } else if (lane == 0 && a.mode == ARN_START) {
        if (a.first) {
            st[ARN_NITER] = st[ARN_NREORTH] = st[ARN_DONE] = 0;
            sc[ARN_TP] = sc[ARN_TM] = sc[ARN_TO] = sc[ARN_TN] = 0.0;
            sc[ARN_R0INIT] = hn;
        }
        st[ARN_NVECS] = 0;
        p[0] = hn;
        if (!isfinite(hn)) err = 1;
        active = !err && hn != 0.0;
        if (hn == 0.0) { conv = 1; res = 0.0; }         // exact x0: x = x0
    }
    if (lane == 0) {
        const uint64_t now = wall_clock64();
        // ticks of the preconditioner, the product and the vector part of this step
        if (steps) {
            sc[ARN_TP] += (double)(a.stamp[1] - a.stamp[0]);
            sc[ARN_TM] += (double)(a.stamp[2] - a.stamp[1]);
            sc[ARN_TO] += (double)(now - a.stamp[2]);
        } else {
            sc[ARN_TN] += (double)(now - a.stamp[2]);
        }
        ArnRes *const o = a.hres + l;
        uint64_t word = (uint64_t)a.seq << 32 | (uint64_t)(steps ? jj : 0) << ARN_W_BITS | (active ? ARN_W_ACTIVE : 0) |
                        (err ? ARN_W_ERR : 0);
        if (conv || !(res > a.tol)) word |= ARN_W_DONE;
        if (a.mode == ARN_NORM) {                       // the report of the whole solve
            put(&o->res, res);
            put(&o->t[0], sc[ARN_TP]);
            put(&o->t[1], sc[ARN_TM]);
            put(&o->t[2], sc[ARN_TO]);
            put(&o->t[3], sc[ARN_TN]);
            put(&o->niter, st[ARN_NITER]);
            put(&o->nreorth, st[ARN_NREORTH] + (a.inner_st ? a.inner_st[ARN_NREALL] : 0));
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_s_waitcnt(0);              // before the word that announces it
        } else {
            st[ARN_CONV] = conv;
            st[ARN_ACTIVE] = active;
            sc[ARN_RES] = res;
            if (!steps && active) __hip_atomic_fetch_add(a.nact, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (steps && !active) __hip_atomic_fetch_sub(a.nact, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        put(&o->word, word);
    }
}

// y = R^-1 p of every lane that took steps this cycle (:287-288); one wavefront per lane.
__global__ void __launch_bounds__(64) k_arn_solve(ArnArgs a) {
    const int l = blockIdx.x, lane = threadIdx.x;
    const int *st = a.st + l * ARN_NST;
    if (st[ARN_DONE]) return;
    const int nv = st[ARN_NVECS];
    const double *R = a.R + (size_t)l * a.rlen;
    double *y = a.y + (size_t)l * a.hlen;
    const double *p = a.p + (size_t)l * a.hlen;
    if (nv <= 64) {
        double pi = lane < nv ? p[lane] : 0.0;
        for (int k = nv - 1; k >= 0; --k) {
            const double *Rk = R + (size_t)k * (k + 1) / 2;
            const double rik = lane <= k ? Rk[lane] : 1.0;
            const double yk = rdlane(pi, k) / rdlane(rik, k);
            if (lane == k) pi = yk;
            else if (lane < k) pi -= rik * yk;
        }
        if (lane < nv) y[lane] = pi;
        return;
    }
    for (int i = lane; i < nv; i += 64) y[i] = p[i];
    __syncthreads();
    for (int k = nv - 1; k >= 0; --k) {
        const double *Rk = R + (size_t)k * (k + 1) / 2;
        const double yk = y[k] / Rk[k];
        __syncthreads();
        if (lane == 0) y[k] = yk;
        for (int i = lane; i < k; i += 64) y[i] -= Rk[i] * yk;
        __syncthreads();
    }
}

// x = x0 + sum y_i z_i of every lane still running (:292-295), kept in x0 for a restart;
// the lane is done when its cycle ended by the stopping test (:296-302).
__global__ void __launch_bounds__(256) k_arn_combine(ArnArgs a, const double *Z, double *x, double *x0, int first) {
    const int l = blockIdx.y;
    const int *st = a.st + l * ARN_NST;
    if (st[ARN_DONE]) return;
    const int nv = st[ARN_NVECS];
    const double *y = a.y + (size_t)l * a.hlen;
    const int64_t vstep = (int64_t)a.nl * a.len, o = (int64_t)l * a.len;
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < a.len; k += (int64_t)gridDim.x * blockDim.x) {
        double v = first ? 0.0 : x0[o + k];
        int i = 0;
        for (; i + 4 <= nv; i += 4) {
            double z[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) z[u] = Z[(size_t)(i + u) * vstep + o + k];
#pragma unroll
            for (int u = 0; u < 4; ++u) v = v + y[i + u] * z[u];
        }
        for (; i < nv; ++i) v = v + y[i] * Z[(size_t)i * vstep + o + k];
        x[o + k] = v;
        x0[o + k] = v;
    }
}

__global__ void k_arn_cycle_end(ArnArgs a) {
    for (int l = threadIdx.x; l < a.nl; l += blockDim.x) {
        int *st = a.st + l * ARN_NST;
        if (st[ARN_CONV] || !(a.sc[l * ARN_NSC + ARN_RES] > a.tol)) st[ARN_DONE] = 1;
        st[ARN_ACTIVE] = 0;
    }
    if (threadIdx.x == 0) *a.nact = 0;
}

__global__ void k_stamp(uint64_t *p) { *p = wall_clock64(); }

}  // namespace

// Workspace of one FGMRES level: nl lanes, up to m steps, vectors of len >= 1 values.
int arn_alloc(cdg_ctx *ctx, Arnoldi &A, int nl, int m, int64_t len, bool mgs) {
    A.nl = nl;
    A.m = m;
    A.len = len;
    A.mgs = mgs;
    // One pair of elements per thread while that makes at most 512 slices (two workgroups per
    // CU), then two, then several passes per slice; whatever the lanes, so that
    // each lane's sums are the same alone and among others.
    const int64_t unit = 2 * AT;
    A.NI = (len + unit - 1) / unit > kMaxG ? 2 : 1;
    const int64_t blocks = std::max<int64_t>(1, (len + unit * A.NI - 1) / (unit * A.NI));
    const int64_t passes = (blocks + kMaxG - 1) / kMaxG;
    A.G = (int)((blocks + passes - 1) / passes);
    const int64_t slice = passes * unit * A.NI;
    const int nx = mgs ? 4 * m + 4 : 3 * (m + 2);
    const int64_t hlen = m + 2, rlen = (int64_t)m * (m + 1) / 2;
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += (bytes + 255) & ~(size_t)255; return o; };
    const size_t o_st = take(sizeof(int) * ARN_NST * nl), o_sc = take(sizeof(double) * ARN_NSC * nl), o_nact = take(4),
                 o_stamp = take(8 * 4);
    const size_t zeroed = off;
    const size_t o_h = take(sizeof(double) * 4 * (size_t)nl * hlen), o_R = take(sizeof(double) * (size_t)nl * rlen);
    const size_t o_s = take(sizeof(double) * (size_t)nl * nx), o_p = take(sizeof(double) * (size_t)nl * nx * A.G);
    int e = dev_alloc(ctx, &A.base, off);
    if (e) return e;
    A.bytes = off;
    char *b = static_cast<char *>(A.base);
    CDG_HIP_TRY(hipMemsetAsync(A.base, 0, zeroed, ctx->stream));
    ArnArgs &a = A.a;
    a = ArnArgs{};
    a.nl = nl;
    a.G = A.G;
    a.m = m;
    a.nx = nx;
    a.slice = slice;
    a.len = len;
    a.hlen = hlen;
    a.rlen = rlen;
    a.st = reinterpret_cast<int *>(b + o_st);
    a.sc = reinterpret_cast<double *>(b + o_sc);
    a.nact = reinterpret_cast<int *>(b + o_nact);
    a.stamp = reinterpret_cast<uint64_t *>(b + o_stamp);
    double *h = reinterpret_cast<double *>(b + o_h);
    a.y = h;
    a.cs = a.y + (size_t)nl * hlen;
    a.sn = a.cs + (size_t)nl * hlen;
    a.p = a.sn + (size_t)nl * hlen;
    a.R = reinterpret_cast<double *>(b + o_R);
    a.sums = reinterpret_cast<double *>(b + o_s);
    a.part = reinterpret_cast<double *>(b + o_p);
    return CDG_OK;
}

void arn_free(cdg_ctx *ctx, Arnoldi &A) {
    if (A.base) dev_free(ctx, A.base, A.bytes);
    A.base = nullptr;
}

int arn_launch(cdg_ctx *ctx, Arnoldi &A, int mode, int jj) {
    ArnArgs &a = A.a;
    a.mode = mode;
    a.jj = jj;
    a.seq = ++ctx->arn_seq;
    const dim3 grid((unsigned)a.G, (unsigned)a.nl);
    const int nph = mode == ARN_CGS ? 3 : mode == ARN_MGS ? 2 * jj + 1 : 1;
    for (int ph = 0; ph < nph; ++ph) {
        if (A.NI == 1) hipLaunchKernelGGL(k_arn_pass<1>, grid, dim3(AT), 0, ctx->stream, a, ph);
        else hipLaunchKernelGGL(k_arn_pass<2>, grid, dim3(AT), 0, ctx->stream, a, ph);
    }
    // workgroup 0: the scalar part; a few elements per thread for the others
    const int64_t scale = mode == ARN_NORM ? 0 : std::min<int64_t>(2048, (a.len + 511) / 512);
    hipLaunchKernelGGL(k_arn_finish, dim3((unsigned)scale + 1, (unsigned)a.nl), dim3(256), 0, ctx->stream, a);
    CDG_HIP_TRY(hipGetLastError());
    return CDG_OK;
}

int arn_cycle_end(cdg_ctx *ctx, Arnoldi &A, const double *Z, double *x, double *x0, bool first) {
    const dim3 grid((unsigned)std::min<int64_t>(std::max<int64_t>(1, (A.len + 255) / 256), 2048), A.nl);
    hipLaunchKernelGGL(k_arn_solve, dim3(A.nl), dim3(64), 0, ctx->stream, A.a);
    hipLaunchKernelGGL(k_arn_combine, grid, dim3(256), 0, ctx->stream, A.a, Z, x, x0, first ? 1 : 0);
    hipLaunchKernelGGL(k_arn_cycle_end, dim3(1), dim3(64), 0, ctx->stream, A.a);
    CDG_HIP_TRY(hipGetLastError());
    return CDG_OK;
}

int arn_stamp(cdg_ctx *ctx, Arnoldi &A, int i) {
    hipLaunchKernelGGL(k_stamp, dim3(1), dim3(1), 0, ctx->stream, A.a.stamp + i);
    CDG_HIP_TRY(hipGetLastError());
    return CDG_OK;
}
