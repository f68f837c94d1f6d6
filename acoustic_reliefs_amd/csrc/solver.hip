// Batched BiCGSTAB on the H-matrix, one independent iteration per right-hand side.
//
// Per rhs it follows Eigen 3.4's BiCGSTAB (the solver the reference instantiates as
// Eigen::BiCGSTAB<HMatrix, Eigen::IdentityPreconditioner>, adjoint.cpp:92-95):
//   x = 0, r = b, r0 = r, rho = alpha = w = 1, v = p = 0
//   while ||r||^2 > tol^2 ||b||^2 and i < maxit:
//     rho_old = rho; rho = r0^H r
//     if |rho| < eps^2 ||r0||^2: r = b - A x; r0 = r; rho = ||r0||^2 (first restart resets i)
//     beta = (rho / rho_old)(alpha / w); p = r + beta (p - w v); v = A p
//     alpha = rho / (r0^H v); s = r - alpha v; t = A s
//     w = t^H s / ||t||^2 (0 if ||t|| = 0); x += alpha p + w s; r = s - w t; i++
// The reductions are two-stage with a fixed split, so every rhs gets the same bits whatever
// the batch. The loop control (convergence, maxit, breakdown restarts) runs on the device at
// the end of an iteration (finish_rhs), so the host launches K iterations between synchronisations, K chosen from the
// observed convergence rate; a right-hand side that meets a restart pauses until the host
// restarts it at the next synchronisation, which leaves its arithmetic unchanged.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <chrono>
#include <cmath>
#include <cstring>

#include "arh_internal.h"
#include "device_common.h"

namespace arh {

// ARH_TRACE=1 in the environment: one line per solver sweep on stderr (precision, right-hand sides
// in the sweep, iterations, true residuals) for diagnosing refinement on hard problems.
static bool trace_on() {
    static const bool on = [] {
        const char *e = std::getenv("ARH_TRACE");
        return e && e[0] == '1';
    }();
    return on;
}

static void trace_sweep(const char *what, int sweep, const std::vector<int> &in, const std::vector<int> &iters,
                        const std::vector<double> &tres) {
    if (!trace_on()) return;
    int n = 0, imax = 0;
    double rmax = 0.0, rmin = 1e300;
    for (size_t j = 0; j < in.size(); j++) {
        if (!in[j]) continue;
        n++;
        imax = std::max(imax, j < iters.size() ? iters[j] : 0);
    }
    for (double r : tres) rmax = std::max(rmax, r), rmin = std::min(rmin, r);
    std::fprintf(stderr, "[arh solve] %s sweep %d: %d rhs, max iters %d, true residual %.3e .. %.3e\n", what, sweep, n,
                 imax, tres.empty() ? 0.0 : rmin, rmax);
}

struct RhsState {
    double2 rho;      // rho of the previous iteration (Eigen's rho_old at the next step)
    double2 rho_new;  // r0^H r for the coming iteration
    double2 alpha, w;
    double r0sq, rhs_sq, rn, tol2;  // tol2 = tol^2 ||b||^2 (tol until the start)
    int active;    // iterating
    int restart;   // restart pending (set at init, or by finish_rhs on breakdown: then paused)
    int it;        // iterations counted toward maxit (reset at the first restart)
    int iters;     // iterations done
    int nrestart;  // restarts done
    int maxit;
    int pad;
    double rn0;  // |b|^2 at the start, when x = 0
};

constexpr int kVT = 256;      // threads per block of vector kernels
constexpr double kInnerFloor = 1e-7;  // mixed refinement: tightest inner (FP32-operator) tolerance
#ifndef ARH_INNER_FRAC
#define ARH_INNER_FRAC 0.5
#endif
constexpr double kInnerFrac = ARH_INNER_FRAC;  // mixed refinement: inner target as a fraction of the remaining one
constexpr int kInnerBudget = 256;      // mixed refinement: iterations an inner solve may take
#ifndef ARH_SOLVER_MAXK
#define ARH_SOLVER_MAXK 8
#endif
constexpr int kMaxK = ARH_SOLVER_MAXK;  // iterations per host synchronisation, at most
constexpr int kMaxNB = 128;   // blocks per rhs of a reduction
constexpr int kLoads = 8, kXrLoads = 4;  // elements of a thread loaded together by the reductions

// v summed over the block, in thread 0
__device__ __forceinline__ void block_reduce4(double v[4], double *sh) {
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE;
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = wave_sum(v[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < 4; k++) sh[w * 4 + k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int k = 0; k < 4; k++) {
            double s = sh[k];
            for (int q = 1; q < kVT / ARH_WAVE; q++) s += sh[q * 4 + k];
            v[k] = s;
        }
}

// Sums of the first K components of NB (<= 128) partial quadruples in order, by a wavefront: lane b loads partials b
// and b + 64 (one load latency instead of NB), then they are added up one by one.
template <int K>
__device__ __forceinline__ void sum_parts(const double *part, int NB, double out[K]) {
    const int lane = threadIdx.x % ARH_WAVE;
    double v[K], u[K];
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = part[min(lane, NB - 1) * 4 + k];
    if (NB > ARH_WAVE)
#pragma unroll
        for (int k = 0; k < K; k++) u[k] = part[min(lane + ARH_WAVE, NB - 1) * 4 + k];
#pragma unroll
    for (int k = 0; k < K; k++) out[k] = 0.0;
    for (int b = 0; b < min(NB, ARH_WAVE); b++)
#pragma unroll
        for (int k = 0; k < K; k++) out[k] += lane_f64(v[k], b);
    for (int b = ARH_WAVE; b < NB; b++)
#pragma unroll
        for (int k = 0; k < K; k++) out[k] += lane_f64(u[k], b - ARH_WAVE);
}

// Complex products of the vector updates with their rounding written out. BiCGSTAB amplifies a last-bit change to
// the size of its tolerance within a hundred iterations, so the fused forms are part of the solver's results: the
// imaginary part rounds a.x b.y (cmul_xy) or a.y b.x (cmul_yx) before the fused multiply-add of the other.
__device__ __forceinline__ double2 cmul_xy(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.y, b.x, a.x * b.y));
}
__device__ __forceinline__ double2 cmul_yx(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}

struct Chunk {
    int lo, hi;
};
__device__ __forceinline__ Chunk chunk_of(int N, int NB) {
    int len = (N + NB - 1) / NB;
    int lo = blockIdx.x * len;
    return Chunk{lo, min(N, lo + len)};
}

// partial sums of conj(a) b (complex) and |c|^2 over the block's chunk
__global__ __launch_bounds__(kVT) void k_dot(const RhsState *__restrict__ S, int N, int NB,
                                             const double2 *__restrict__ a, const double2 *__restrict__ b,
                                             const double2 *__restrict__ c, double *__restrict__ part) {
    __shared__ double sh[4 * kVT / ARH_WAVE];
    const int j = blockIdx.y;
    if (!S[j].active) return;
    const Chunk ch = chunk_of(N, NB);
    const int64_t o = (int64_t)j * N;
    double v[4] = {0, 0, 0, 0};
    // the elements of a thread in order, kLoads of them in flight (surplus loads repeat the chunk's last)
    for (int i0 = ch.lo + threadIdx.x; i0 < ch.hi; i0 += kLoads * kVT) {
        double2 av[kLoads], bv[kLoads], cv[kLoads];
#pragma unroll
        for (int q = 0; q < kLoads; q++) {
            const int64_t e = o + min(i0 + q * kVT, ch.hi - 1);
            av[q] = a[e], bv[q] = b[e];
            if (c) cv[q] = c[e];
        }
#pragma unroll
        for (int q = 0; q < kLoads; q++) {
            if (i0 + q * kVT >= ch.hi) break;
            const double2 ai = av[q], bi = bv[q];
            v[0] += ai.x * bi.x + ai.y * bi.y;
            v[1] += ai.x * bi.y - ai.y * bi.x;
            if (c) {
                const double2 ci = cv[q];
                v[2] += ci.x * ci.x + ci.y * ci.y;
            }
        }
    }
    block_reduce4(v, sh);
    if (threadIdx.x == 0)
        for (int k = 0; k < 4; k++) part[((int64_t)j * NB + blockIdx.x) * 4 + k] = v[k];
}

// The end of an iteration for one rhs, by a wavefront: alpha, w, rho committed; rho_new = r0^H r, rn = |r|^2; then
// Eigen's loop control: stop when ||r||^2 <= tol2 or it == maxit, pause for a restart when |r0^H r| < eps^2 ||r0||^2.
__device__ __forceinline__ void finish_rhs(RhsState &st, int j, int NB, const double *__restrict__ part_r0v,
                                           const double *__restrict__ part_ts, const double *__restrict__ part_rr) {
    const double eps2 = 4.930380657631324e-32;  // (2^-52)^2, Eigen's NumTraits<double>::epsilon() squared
    double d[2], e[3], f[3];
    const int64_t o = (int64_t)j * NB * 4;
    sum_parts<2>(part_r0v + o, NB, d);
    sum_parts<3>(part_ts + o, NB, e);
    sum_parts<3>(part_rr + o, NB, f);
    st.alpha = cdiv(st.rho_new, make_double2(d[0], d[1]));
    st.w = e[2] > 0.0 ? make_double2(e[0] / e[2], e[1] / e[2]) : make_double2(0.0, 0.0);
    st.rho = st.rho_new;
    st.rho_new = make_double2(f[0], f[1]);
    st.rn = f[2];
    st.it++;
    st.iters++;
    if (!(st.rn > st.tol2 && st.it < st.maxit)) {
        st.active = 0;
    } else if (hypot(st.rho_new.x, st.rho_new.y) < eps2 * st.r0sq) {
        st.active = 0;
        st.restart = 1;
    }
}

// States of all rhs after finish_rhs (their new values to out; history of ||r|| / ||b|| on request), a wavefront per rhs:
// wavefront q of nq. gate[0] (zero before) receives the number of right-hand sides still active.
__device__ __forceinline__ void finish_all(const RhsState *__restrict__ S, RhsState *__restrict__ out, int R, int NB,
                                           const double *__restrict__ part_r0v, const double *__restrict__ part_ts,
                                           const double *__restrict__ part_rr, double *__restrict__ hist, int hist_cap,
                                           int *__restrict__ gate, int q, int nq, RhsState *__restrict__ host) {
    const int lane = threadIdx.x % ARH_WAVE;
    for (int j = q; j < R; j += nq) {
        RhsState st = S[j];
        if (st.active) {
            finish_rhs(st, j, NB, part_r0v, part_ts, part_rr);
            if (lane == 0) {
                if (hist && st.iters < hist_cap) hist[(int64_t)j * hist_cap + st.iters] = sqrt(st.rn / st.rhs_sq);
                if (st.active) atomicAdd(gate, 1);
            }
        }
        if (lane == 0) {
            out[j] = st;
            if (host) host[j] = st;
        }
    }
}

// The end of a batch's last iteration (one wavefront per workgroup); host: the host's copy of the states, in pinned
// memory.
__global__ __launch_bounds__(ARH_WAVE) void k_finish(const RhsState *__restrict__ S, RhsState *__restrict__ out, int R,
                                                     int NB, const double *__restrict__ part_r0v,
                                                     const double *__restrict__ part_ts,
                                                     const double *__restrict__ part_rr, double *__restrict__ hist,
                                                     int hist_cap, int *__restrict__ gate,
                                                     RhsState *__restrict__ host) {
    finish_all(S, out, R, NB, part_r0v, part_ts, part_rr, hist, hist_cap, gate, blockIdx.x, gridDim.x, host);
}

// The vector updates before a product also write the product's packed rows (row i: rw complex values, listed column c
// at c, zero from nc on), through LDS: a workgroup takes up_rows of the rows and kUpCols of the columns, a wavefront each
// (every wavefront forms its rhs's scalars, some 400 operations; N = 9,828, p update: 37 right-hand sides FP32 11.3,
// 9.7, 9.4 us at 64, 128, 192 rows, one FP64 4.8, 5.1, 5.4 us. The end of the previous iteration and the packing
// were launches of their own: 16.4 us for 37, 15 us for one). T2: complex type of the operator's precision; xf == nullptr
// leaves the packing to the product. Four columns per workgroup: beside other streams' products a workgroup of sixteen
// wavefronts waits for as many free slots on one compute unit (13 bands served, p and s updates 104 and 63 us instead of
// the 9.7 and 6.3 they take alone, now 39 and 28); alone the two are equal, served bands 223.5 -> 221 ms, the sphere's band
// 1.13 -> 1.11 ms.
constexpr int kUpCols = 4;
template <class T2>
constexpr int up_rows() {
    return sizeof(T2) == 8 ? 128 : 64;
}
__device__ __forceinline__ float2 to_packed(double2 v, float2) { return make_float2((float)v.x, (float)v.y); }
__device__ __forceinline__ double2 to_packed(double2 v, double2) { return v; }
template <class T2>
__device__ __forceinline__ void write_packed(const T2 (*tile)[kUpCols + 1], int bx, int N, int nc, int rw,
                                             T2 *__restrict__ xf) {
    __syncthreads();
    const int r0 = bx * up_rows<T2>(), rows = min(up_rows<T2>(), N - r0);
    const int c0 = (int)blockIdx.y * kUpCols;
    const int c = threadIdx.x % kUpCols;
    if (c0 + c >= rw) return;
    for (int r = threadIdx.x / kUpCols; r < rows; r += blockDim.x / kUpCols) {
        T2 v{};
        if (c0 + c < nc) v = tile[r][c];
        xf[(int64_t)(r0 + r) * rw + c0 + c] = v;
    }
}

// p = r + beta (p - w v), beta = (rho_new / rho)(alpha / w), for the listed right-hand sides. finish: the states are
// those before the end of the previous iteration; every workgroup derives the new ones from the partials, and the
// workgroups with x = 0 do nothing but write them to out (the others read S, which nothing writes).
template <class T2>
__global__ __launch_bounds__(ARH_WAVE * kUpCols) void k_p_update(const RhsState *__restrict__ S, RhsState *__restrict__ out, int R,
                                                   int finish, int N, int NB, const int *__restrict__ cols, int nc,
                                                   const double *__restrict__ part_r0v,
                                                   const double *__restrict__ part_ts,
                                                   const double *__restrict__ part_rr, const double2 *__restrict__ r,
                                                   double2 *__restrict__ p, const double2 *__restrict__ v,
                                                   double *__restrict__ hist, int hist_cap, int *__restrict__ gate,
                                                   T2 *__restrict__ xf, int rw) {
    constexpr int Q = up_rows<T2>() / ARH_WAVE;  // rows per lane
    __shared__ T2 tile[up_rows<T2>()][kUpCols + 1];
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE, nw = blockDim.x / ARH_WAVE;
    if (finish && blockIdx.x == 0) {
        finish_all(S, out, R, NB, part_r0v, part_ts, part_rr, hist, hist_cap, gate, (int)blockIdx.y * nw + w,
                   (int)gridDim.y * nw, nullptr);
        return;
    }
    const int bx = (int)blockIdx.x - (finish ? 1 : 0);
    const int i0 = bx * up_rows<T2>() + lane;
    const int c0 = (int)blockIdx.y * kUpCols;
    for (int c = w; c < kUpCols && c0 + c < nc; c += nw) {
        const int j = cols[c0 + c];
        RhsState st = S[j];
        const int64_t o = (int64_t)j * N;
        double2 q[Q], vi[Q], ri[Q];
#pragma unroll
        for (int t = 0; t < Q; t++) {
            const int64_t e = o + min(i0 + t * ARH_WAVE, N - 1);
            q[t] = p[e], vi[t] = v[e], ri[t] = r[e];
        }
        if (st.active) {
            if (finish) finish_rhs(st, j, NB, part_r0v, part_ts, part_rr);
            if (st.active) {
                const double2 beta = cmul_xy(cdiv(st.rho_new, st.rho), cdiv(st.alpha, st.w));
#pragma unroll
                for (int t = 0; t < Q; t++) {
                    q[t] = cadd(ri[t], cmul_yx(beta, csub(q[t], cmul_xy(st.w, vi[t]))));
                    if (i0 + t * ARH_WAVE < N) p[o + i0 + t * ARH_WAVE] = q[t];
                }
            }
        }
        if (xf)
#pragma unroll
            for (int t = 0; t < Q; t++) tile[t * ARH_WAVE + lane][c] = to_packed(q[t], T2{});
    }
    if (xf) write_packed<T2>(tile, bx, N, nc, rw, xf);
}

// s = r - alpha v, alpha = rho_new / (r0^H v) from the partials, for the listed right-hand sides
template <class T2>
__global__ __launch_bounds__(ARH_WAVE * kUpCols) void k_s_update(const RhsState *__restrict__ S, int N, int NB,
                                                   const int *__restrict__ cols, int nc,
                                                   const double *__restrict__ part_r0v, const double2 *__restrict__ r,
                                                   const double2 *__restrict__ v, double2 *__restrict__ s,
                                                   T2 *__restrict__ xf, int rw) {
    constexpr int Q = up_rows<T2>() / ARH_WAVE;  // rows per lane
    __shared__ T2 tile[up_rows<T2>()][kUpCols + 1];
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE, nw = blockDim.x / ARH_WAVE;
    const int i0 = (int)blockIdx.x * up_rows<T2>() + lane;
    const int c0 = (int)blockIdx.y * kUpCols;
    for (int c = w; c < kUpCols && c0 + c < nc; c += nw) {
        const int j = cols[c0 + c];
        const int64_t o = (int64_t)j * N;
        double2 q[Q];
        if (S[j].active) {
            double2 vi[Q];
#pragma unroll
            for (int t = 0; t < Q; t++) {
                const int64_t e = o + min(i0 + t * ARH_WAVE, N - 1);
                q[t] = r[e], vi[t] = v[e];
            }
            double d[2];
            sum_parts<2>(part_r0v + (int64_t)j * NB * 4, NB, d);
            const double2 alpha = cdiv(S[j].rho_new, make_double2(d[0], d[1]));
#pragma unroll
            for (int t = 0; t < Q; t++) {
                q[t] = csub(q[t], cmul_xy(alpha, vi[t]));
                if (i0 + t * ARH_WAVE < N) s[o + i0 + t * ARH_WAVE] = q[t];
            }
        } else {  // a paused rhs keeps its vectors: the product recomputes the same t
#pragma unroll
            for (int t = 0; t < Q; t++) q[t] = s[o + min(i0 + t * ARH_WAVE, N - 1)];
        }
        if (xf)
#pragma unroll
            for (int t = 0; t < Q; t++) tile[t * ARH_WAVE + lane][c] = to_packed(q[t], T2{});
    }
    if (xf) write_packed<T2>(tile, (int)blockIdx.x, N, nc, rw, xf);
}

// x += alpha p + w s; r = s - w t; partials of r0^H r and |r|^2
__global__ __launch_bounds__(kVT) void k_xr_update(const RhsState *__restrict__ S, int N, int NB,
                                                   const double *__restrict__ part_r0v,
                                                   const double *__restrict__ part_ts, const double2 *__restrict__ p,
                                                   const double2 *__restrict__ s, const double2 *__restrict__ t,
                                                   const double2 *__restrict__ r0, double2 *__restrict__ x,
                                                   double2 *__restrict__ r, double *__restrict__ part_rr) {
    __shared__ double sh[4 * kVT / ARH_WAVE];
    const int j = blockIdx.y;
    const RhsState st = S[j];
    if (!st.active) return;
    double d[2], e[3];
    sum_parts<2>(part_r0v + (int64_t)j * NB * 4, NB, d);
    sum_parts<3>(part_ts + (int64_t)j * NB * 4, NB, e);
    const double2 alpha = cdiv(st.rho_new, make_double2(d[0], d[1]));
    const double tt = e[2];
    const double2 w = tt > 0.0 ? make_double2(e[0] / tt, e[1] / tt) : make_double2(0.0, 0.0);
    const Chunk ch = chunk_of(N, NB);
    const int64_t o = (int64_t)j * N;
    double v[4] = {0, 0, 0, 0};
    for (int i0 = ch.lo + threadIdx.x; i0 < ch.hi; i0 += kXrLoads * kVT) {
        double2 sv[kXrLoads], tv[kXrLoads], xv[kXrLoads], pv[kXrLoads], qv[kXrLoads];
#pragma unroll
        for (int q = 0; q < kXrLoads; q++) {
            const int64_t e = o + min(i0 + q * kVT, ch.hi - 1);
            sv[q] = s[e], tv[q] = t[e], xv[q] = x[e], pv[q] = p[e], qv[q] = r0[e];
        }
#pragma unroll
        for (int q = 0; q < kXrLoads; q++) {
            const int i = i0 + q * kVT;
            if (i >= ch.hi) break;
            const double2 si = sv[q], ti = tv[q];
            double2 xi = xv[q];
            xi = cadd(xi, cadd(cmul_xy(alpha, pv[q]), cmul_xy(w, si)));
            x[o + i] = xi;
            double2 ri = csub(si, cmul_xy(w, ti));
            r[o + i] = ri;
            double2 qi = qv[q];
            v[0] += qi.x * ri.x + qi.y * ri.y;
            v[1] += qi.x * ri.y - qi.y * ri.x;
            v[2] += ri.x * ri.x + ri.y * ri.y;
        }
    }
    block_reduce4(v, sh);
    if (threadIdx.x == 0)
        for (int k = 0; k < 4; k++) part_rr[((int64_t)j * NB + blockIdx.x) * 4 + k] = v[k];
}

// Host lists to the device: two arrays of ints from pinned memory, which the host rewrites only after a
// synchronisation. (A small hipMemcpyAsync each way cost 25 to 45 us of an idle GPU at every synchronisation.)
__global__ __launch_bounds__(256) void k_load(int *__restrict__ d0, const int *__restrict__ s0, int n0,
                                              int *__restrict__ d1, const int *__restrict__ s1, int n1) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e < n0)
        d0[e] = s0[e];
    else if (e - n0 < n1)
        d1[e - n0] = s1[e - n0];
}

// (re)start of rhs j: r = b - Ax, r0 = r, partials of |r|^2 and b^2. A fresh start (Ax null) is from x = 0: it zeroes
// x, p and v too (launches of their own otherwise).
__global__ __launch_bounds__(kVT) void k_restart(const RhsState *__restrict__ S, int N, int NB,
                                                 const double2 *__restrict__ b, const double2 *__restrict__ Ax,
                                                 double2 *__restrict__ r, double2 *__restrict__ r0,
                                                 double2 *__restrict__ x, double2 *__restrict__ p,
                                                 double2 *__restrict__ v_, double *__restrict__ part) {
    __shared__ double sh[4 * kVT / ARH_WAVE];
    const int j = blockIdx.y;
    if (!S[j].restart) return;
    const Chunk ch = chunk_of(N, NB);
    const int64_t o = (int64_t)j * N;
    double v[4] = {0, 0, 0, 0};
    for (int i = ch.lo + threadIdx.x; i < ch.hi; i += kVT) {
        double2 bi = b[o + i];
        double2 ri = Ax ? csub(bi, Ax[o + i]) : bi;
        r[o + i] = ri;
        r0[o + i] = ri;
        if (!Ax) x[o + i] = p[o + i] = v_[o + i] = make_double2(0.0, 0.0);
        v[0] += ri.x * ri.x + ri.y * ri.y;
        v[1] += bi.x * bi.x + bi.y * bi.y;
    }
    block_reduce4(v, sh);
    if (threadIdx.x == 0)
        for (int k = 0; k < 4; k++) part[((int64_t)j * NB + blockIdx.x) * 4 + k] = v[k];
}

// full restart: rho = r0sq = |r|^2; fresh: also alpha = w = rho_old = 1, rhs_sq, the stopping bound, and
// whether the rhs iterates at all (a zero right-hand side does not, nor one that meets its tolerance already), counted in
// count; a breakdown restart resumes the iteration (active again) and resets the iteration count on the
// first restart (Eigen)
// (a wavefront per rhs)
__global__ __launch_bounds__(ARH_WAVE) void k_restart_finish(RhsState *__restrict__ S, int NB,
                                                             const double *__restrict__ part, int fresh,
                                                             int *__restrict__ count) {
    const int j = blockIdx.x;
    if (!S[j].restart) return;
    RhsState st = S[j];
    double f[2];
    sum_parts<2>(part + (int64_t)j * NB * 4, NB, f);
    st.r0sq = f[0];
    st.rho_new = make_double2(f[0], 0.0);
    st.rn = f[0];
    if (fresh) {
        st.rhs_sq = f[1];
        st.rho = make_double2(1.0, 0.0);
        st.alpha = make_double2(1.0, 0.0);
        st.w = make_double2(1.0, 0.0);
        st.rn0 = f[0];
        st.tol2 = st.tol2 * st.tol2 * st.rhs_sq;
        st.active = st.rhs_sq != 0.0 && st.rn > st.tol2 && st.maxit > 0 ? 1 : 0;
        if (threadIdx.x == 0 && st.active) atomicAdd(count, 1);
    } else {
        if (st.nrestart++ == 0) st.it = 0;
        st.active = 1;
    }
    st.restart = 0;
    if (threadIdx.x == 0) S[j] = st;
}

// x += f d (refinement; f = -1 reverts a correction), masked per column
__global__ void k_axpy_cols(const int *__restrict__ mask, int N, double2 *__restrict__ x,
                            const double2 *__restrict__ d, double f) {
    const int j = blockIdx.y;
    if (!mask[j]) return;
    const int64_t o = (int64_t)j * N;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        const double2 di = d[o + i];
        x[o + i] = cadd(x[o + i], make_double2(f * di.x, f * di.y));
    }
}

// r = b - Ax, per rhs partials of |r|^2 and |b|^2 (true residual)
__global__ __launch_bounds__(kVT) void k_resid(int N, int NB, const double2 *__restrict__ b,
                                               const double2 *__restrict__ Ax, double2 *__restrict__ r,
                                               double *__restrict__ part) {
    __shared__ double sh[4 * kVT / ARH_WAVE];
    const int j = blockIdx.y;
    const Chunk ch = chunk_of(N, NB);
    const int64_t o = (int64_t)j * N;
    double v[4] = {0, 0, 0, 0};
    for (int i = ch.lo + threadIdx.x; i < ch.hi; i += kVT) {
        double2 bi = b[o + i];
        double2 ri = csub(bi, Ax[o + i]);
        if (r) r[o + i] = ri;
        v[0] += ri.x * ri.x + ri.y * ri.y;
        v[1] += bi.x * bi.x + bi.y * bi.y;
    }
    block_reduce4(v, sh);
    if (threadIdx.x == 0)
        for (int k = 0; k < 4; k++) part[((int64_t)j * NB + blockIdx.x) * 4 + k] = v[k];
}

// ------------------------------------------------------------------ host driver
namespace {

struct Work {
    DBuf buf, hbuf;
    double2 *r, *r0, *p, *v, *s, *t, *Ax;
    double *part;
    RhsState *S, *S2;  // states, and the other copy an iteration writes
    int *mask;
    int *ctl;  // [0]: active count at a batch's start, [1..R]: column list
    int *ghist;  // after the list: active count after each iteration of a batch (the gate of the next one)
    // pinned host block: states as the device last wrote them, states and lists on their way to the device, the
    // partials of the true residual
    HostBuf host;
    RhsState *hs, *hs_up;
    int *h_ctl, *h_rs, *h_mask;
    double *h_part;
    static size_t host_bytes(int R, int NB) {
        return 2 * sizeof(RhsState) * R + sizeof(double) * 4 * (size_t)R * NB + sizeof(int) * (3 * (size_t)R + 2 + kMaxK);
    }
    Work(int64_t N, int R, int NB, hipStream_t stream) : host(host_bytes(R, NB), stream) {
        hs = host.as<RhsState>(), hs_up = hs + R;
        h_part = (double *)(hs_up + R);
        h_ctl = (int *)(h_part + 4 * (size_t)R * NB), h_rs = h_ctl + R + 1 + kMaxK, h_mask = h_rs + R + 1;
        const int64_t vec = N * R;
        const size_t vb = sizeof(double2) * vec;
        const size_t pb = sizeof(double) * 4 * (size_t)R * NB;
        // every piece starts on a 256-byte boundary: the total is the sum of the rounded sizes
        auto rnd = [](size_t n) { return (n + 255) / 256 * 256; };
        const size_t total = 7 * rnd(vb) + rnd(3 * pb) + 2 * rnd(sizeof(RhsState) * R) + rnd(sizeof(int) * R) +
                             rnd(sizeof(int) * (R + 1 + kMaxK));
        buf.alloc(total);
        char *c = buf.as<char>();
        char *const end = c + total;
        auto take = [&](size_t n) {
            char *q = c;
            c += rnd(n);
            ARH_CHECK(c <= end, ARH_EINVAL, "internal: solver workspace overflow");
            return q;
        };
        r = (double2 *)take(vb), r0 = (double2 *)take(vb), p = (double2 *)take(vb), v = (double2 *)take(vb);
        s = (double2 *)take(vb), t = (double2 *)take(vb), Ax = (double2 *)take(vb);
        part = (double *)take(3 * pb);
        S = (RhsState *)take(sizeof(RhsState) * R);
        S2 = (RhsState *)take(sizeof(RhsState) * R);
        mask = (int *)take(sizeof(int) * R);
        ctl = (int *)take(sizeof(int) * (R + 1 + kMaxK));
        ghist = ctl + R + 1;
    }
    // int arrays from the pinned block to the device
    void load(void *d0, const void *s0, size_t b0, void *d1 = nullptr, const void *s1 = nullptr, size_t b1 = 0) const {
        const int n0 = (int)(b0 / sizeof(int)), n1 = (int)(b1 / sizeof(int));
        hipLaunchKernelGGL(k_load, dim3((n0 + n1 + 255) / 256), dim3(256), 0, host.s, (int *)d0, (const int *)s0, n0,
                           (int *)d1, (const int *)s1, n1);
        ARH_HIP(hipGetLastError());
    }
    // x += f d for the masked right-hand sides (a true residual, which synchronises, follows every call: the mask of
    // the previous one has been read)
    void axpy(const std::vector<int> &m, int N, double2 *x, const double2 *d, double f) {
        std::copy(m.begin(), m.end(), h_mask);
        load(mask, h_mask, sizeof(int) * m.size());
        hipLaunchKernelGGL(k_axpy_cols, dim3(std::max(1, std::min(1024, (N + 255) / 256)), (unsigned)m.size()), dim3(256),
                           0, host.s, mask, N, x, d, f);
        ARH_HIP(hipGetLastError());
    }
};

#ifndef ARH_SOLVER_ROWS
#define ARH_SOLVER_ROWS 2048
#endif
// blocks per right-hand side of the vector kernels: about ARH_SOLVER_ROWS rows each
int pick_nb(int N) { return std::max(1, std::min(kMaxNB, (N + ARH_SOLVER_ROWS - 1) / ARH_SOLVER_ROWS)); }

}  // namespace

// BiCGSTAB on operator `prec` (ARH_FP64 / ARH_MIXED) for the rhs with want[j] != 0, from x = 0.
// Returns per-rhs iterations; fills recursive residual history.
// stall_window > 0 (inner solves of the refinement only): a right-hand side whose recursive
// residual has not halved within stall_window iterations is stopped, and so is one that has run
// budget iterations (budget > 0) without converging (both checked at synchronisations); 0 keeps
// Eigen's loop control exactly.
static void bicgstab(arh_hmat *h, int transpose, int prec, int R, const double2 *b, double2 *x,
                     const std::vector<int> &want, const std::vector<double> &tolj, int maxit, const arh_solve_opts &o,
                     arh_solve_stats *st, std::vector<int> &iters, std::vector<double> &err, Work &W, int NB,
                     bool record_hist, int stall_window = 0, int budget = 0) {
    arh_ctx *ctx = h->g->ctx;
    hipStream_t s = ctx->stream;
    const int N = h->g->N;
    const dim3 gv(NB, R), bv(kVT);
    double *P1 = W.part, *P2 = W.part + 4 * (size_t)R * NB, *P3 = W.part + 8 * (size_t)R * NB;
    const bool hist_on = record_hist && st && st->hist && st->hist_len && o.hist_cap > 0;
    const int cap = hist_on ? o.hist_cap : 0;
    double *hist_dev = nullptr;
    if (hist_on) {
        W.hbuf.alloc(sizeof(double) * (size_t)R * cap);
        hist_dev = W.hbuf.as<double>();
    }
    RhsState *hs = W.hs;
    int *ctl = W.h_ctl, *ctl_rs = W.h_rs;
    int nlist = 0;
    for (int j = 0; j < R; j++) {
        RhsState st;
        std::memset(&st, 0, sizeof(RhsState));
        st.restart = want[j] ? 1 : 0;
        st.tol2 = tolj[j];
        st.maxit = maxit;
        W.hs_up[j] = st;
        if (want[j]) ctl[1 + nlist++] = j;
    }
    iters.assign(R, 0);
    err.assign(R, 0.0);
    if (nlist == 0) return;
    // the first batch follows the start at once: its list is every wanted rhs, and the device says which of them
    // iterate (in ctl[0], the batch's gate)
    ctl[0] = 0;
    std::fill(ctl + R + 1, ctl + R + 1 + kMaxK, 0);
    W.load(W.S, W.hs_up, sizeof(RhsState) * R, W.ctl, ctl, sizeof(int) * (R + 1 + kMaxK));
    hipLaunchKernelGGL(k_restart, gv, bv, 0, s, W.S, N, NB, b, (const double2 *)nullptr, W.r, W.r0, x, W.p, W.v, P1);
    hipLaunchKernelGGL(k_restart_finish, dim3(R), dim3(ARH_WAVE), 0, s, W.S, NB, P1, 1, W.ctl);
    ARH_HIP(hipGetLastError());
    std::vector<double> hist0(R, 0.0);
    // K from the observed convergence: iterations until the fastest active rhs is predicted to
    // reach its tolerance (so that few iterations run past convergence), 1..kMaxK
    std::vector<double> e_prev(R, 0.0);
    std::vector<int> i_prev(R, 0);
    int K = 2;
    std::vector<double> best;
    std::vector<int> best_it(R, 0);
    RhsState *S = W.S, *So = W.S2;  // current states, and where the next iteration's go
    const bool fp64 = prec != ARH_MIXED, fused = h->g->max_leaf <= mfma_max_leaf();
    bool first = true;
    for (int nact = nlist; nact > 0;) {
        int nc = nlist;
        if (!first) {
            nc = 0;
            for (int j = 0; j < R; j++)
                if (hs[j].active) ctl[1 + nc++] = j;
            ctl[0] = nc;
            W.load(W.ctl, ctl, sizeof(int) * (R + 1 + kMaxK));
        }
        const int *cols = W.ctl + 1;
        // the updates write the product's packed rows where one pass takes every active rhs
        int rw = 0;
        void *xf = fused ? mfma_packed_rows(h, transpose, fp64 ? 1 : 0, nc, &rw) : nullptr;
        // a wavefront per listed rhs, and enough of them for the workgroups that write all states
        const dim3 bu(ARH_WAVE * std::min(kUpCols, std::max(nc, (R + 3) / 4)));
        const unsigned guy = (unsigned)((std::max(nc, rw) + kUpCols - 1) / kUpCols);
        const int ur = xf && !fp64 ? up_rows<float2>() : up_rows<double2>();
        const unsigned gu = (unsigned)((N + ur - 1) / ur);
        auto apply = [&](const double2 *in, double2 *out, const int *gate) {
            if (xf)
                hmat_apply_mfma(h, transpose, fp64 ? 1 : 0, R, in, out, s, cols, nc, gate, true);
            else
                hmat_apply(h, transpose, prec, R, in, out, s, cols, nc, gate);
        };
        for (int k = 0; k < K; k++) {
            ctx->prof.cur_slot = k;
            const int fin = k > 0 ? 1 : 0;  // the end of the previous iteration
            int *gate = fin ? W.ghist + k - 1 : W.ctl;  // active right-hand sides
            if (xf && !fp64)
                hipLaunchKernelGGL(k_p_update<float2>, dim3(gu + fin, guy), bu, 0, s, S, So, R, fin, N, NB, cols, nc, P1, P2,
                                   P3, W.r, W.p, W.v, hist_dev, cap, gate, (float2 *)xf, rw);
            else
                hipLaunchKernelGGL(k_p_update<double2>, dim3(gu + fin, guy), bu, 0, s, S, So, R, fin, N, NB, cols, nc, P1,
                                   P2, P3, W.r, W.p, W.v, hist_dev, cap, gate, (double2 *)xf, rw);
            if (fin) std::swap(S, So);
            apply(W.p, W.v, gate);
            hipLaunchKernelGGL(k_dot, gv, bv, 0, s, S, N, NB, W.r0, W.v, (const double2 *)nullptr, P1);
            if (xf && !fp64)
                hipLaunchKernelGGL(k_s_update<float2>, dim3(gu, guy), bu, 0, s, S, N, NB, cols, nc, P1, W.r, W.v, W.s,
                                   (float2 *)xf, rw);
            else
                hipLaunchKernelGGL(k_s_update<double2>, dim3(gu, guy), bu, 0, s, S, N, NB, cols, nc, P1, W.r, W.v, W.s,
                                   (double2 *)xf, rw);
            apply(W.s, W.t, gate);
            hipLaunchKernelGGL(k_dot, gv, bv, 0, s, S, N, NB, W.t, W.s, W.t, P2);
            hipLaunchKernelGGL(k_xr_update, gv, bv, 0, s, S, N, NB, P1, P2, W.p, W.s, W.t, W.r0, x, W.r, P3);
        }
        hipLaunchKernelGGL(k_finish, dim3(R), dim3(ARH_WAVE), 0, s, S, So, R, NB, P1, P2, P3, hist_dev, cap,
                           W.ghist + K - 1, hs);
        std::swap(S, So);
        ARH_HIP(hipGetLastError());
        ctx->prof.cur_slot = -1;
        int gh[kMaxK];
        if (ctx->prof.on) ARH_HIP(hipMemcpyAsync(gh, W.ghist, sizeof(int) * K, hipMemcpyDeviceToHost, s));
        ARH_HIP(hipStreamSynchronize(s));
        bool none = false;  // the device found no rhs to iterate at the start
        if (first) {
            none = true;
            for (int j = 0; j < R; j++) {
                if (!want[j] || hs[j].rhs_sq == 0.0) continue;  // Eigen: x = 0, done
                hist0[j] = err[j] = e_prev[j] = std::sqrt(hs[j].rn0 / hs[j].rhs_sq);
                if (hs[j].iters > 0) none = false;
            }
            best = err;
            first = false;
        }
        if (ctx->prof.on) {
            // iteration k's products ran iff some rhs was active after iteration k - 1
            ctx->prof.slot_ok.assign(K, none ? 0 : 1);
            for (int k = 1; k < K; k++) ctx->prof.slot_ok[k] = gh[k - 1] > 0;
            ctx->prof.flush(false);
            ctx->prof.slot_ok.clear();
        }
        if (none) break;
        // stalled inner solves stop here (nothing has run on the device since the state was read)
        if (stall_window > 0 || budget > 0) {
            bool changed = false;
            for (int j = 0; j < R; j++) {
                if (!(hs[j].active || hs[j].restart) || hs[j].rhs_sq == 0.0) continue;
                const double e = std::sqrt(hs[j].rn / hs[j].rhs_sq);
                if (budget > 0 && hs[j].iters >= budget) {
                    hs[j].active = 0;
                    hs[j].restart = 0;
                    changed = true;
                } else if (e < 0.5 * best[j]) {
                    best[j] = e;
                    best_it[j] = hs[j].iters;
                } else if (stall_window > 0 && hs[j].iters - best_it[j] >= stall_window) {
                    hs[j].active = 0;
                    hs[j].restart = 0;
                    changed = true;
                }
            }
            if (changed) {  // from a copy: hs changes below before the device reads it
                std::copy(hs, hs + R, W.hs_up);
                W.load(S, W.hs_up, sizeof(RhsState) * R);
            }
        }
        // breakdown restarts: r = b - A x, r0 = r for the paused right-hand sides
        int nrs = 0;
        for (int j = 0; j < R; j++)
            if (hs[j].restart) ctl_rs[1 + nrs++] = j;
        if (nrs) {
            ctl_rs[0] = nrs;
            W.load(W.ctl, ctl_rs, sizeof(int) * (nrs + 1));
            hmat_apply(h, transpose, prec, R, x, W.Ax, s, W.ctl + 1, nrs, W.ctl);
            if (st) st->matvecs++;
            hipLaunchKernelGGL(k_restart, gv, bv, 0, s, S, N, NB, b, W.Ax, W.r, W.r0, x, W.p, W.v, P1);
            hipLaunchKernelGGL(k_restart_finish, dim3(R), dim3(ARH_WAVE), 0, s, S, NB, P1, 0, (int *)nullptr);
            ARH_HIP(hipGetLastError());
            for (int j = 0; j < R; j++)
                if (hs[j].restart) {
                    hs[j].restart = 0;
                    hs[j].active = 1;
                    if (st) st->restarts++;
                }
        }
        if (st) st->matvecs += 2 * K;
        nact = 0;
        double kpred = kMaxK;
        for (int j = 0; j < R; j++) {
            if (!want[j] || hs[j].rhs_sq == 0.0) continue;
            err[j] = std::sqrt(hs[j].rn / hs[j].rhs_sq);
            if (!hs[j].active) continue;
            nact++;
            // geometric extrapolation of the residual since the previous synchronisation
            const int di = hs[j].iters - i_prev[j];
            if (di > 0 && err[j] > 0.0 && e_prev[j] > err[j]) {
                const double rate = std::log(e_prev[j] / err[j]) / di;
                kpred = std::min(kpred, std::log(err[j] / tolj[j]) / rate);
            }
            e_prev[j] = err[j];
            i_prev[j] = hs[j].iters;
        }
        K = std::max(1, std::min(kMaxK, (int)std::floor(kpred)));
    }
    for (int j = 0; j < R; j++) iters[j] = hs[j].iters;
    if (hist_on) {
        std::vector<double> hh((size_t)R * cap);
        ARH_HIP(hipMemcpyAsync(hh.data(), hist_dev, sizeof(double) * hh.size(), hipMemcpyDeviceToHost, s));
        ARH_HIP(hipStreamSynchronize(s));
        for (int j = 0; j < R; j++) {
            if (!want[j] || hs[j].rhs_sq == 0.0) continue;
            const int n = std::min(cap, 1 + hs[j].iters);
            double *dst = st->hist + (size_t)j * cap;
            dst[0] = hist0[j];
            for (int k = 1; k < n; k++) dst[k] = hh[(size_t)j * cap + k];
            st->hist_len[j] = n;
        }
    }
}

// true residual ||b - A x|| / ||b|| per rhs (FP64 operator); r receives b - A x if non-null
static void true_residual(arh_hmat *h, int transpose, int R, const double2 *b, const double2 *x, double2 *r, Work &W,
                          int NB, std::vector<double> &res, arh_solve_stats *st) {
    hipStream_t s = h->g->ctx->stream;
    const int N = h->g->N;
    hmat_apply(h, transpose, ARH_FP64, R, x, W.Ax, s);
    if (st) st->matvecs++;
    hipLaunchKernelGGL(k_resid, dim3(NB, R), dim3(kVT), 0, s, N, NB, b, W.Ax, r, W.h_part);
    ARH_HIP(hipGetLastError());
    ARH_HIP(hipStreamSynchronize(s));
    const double *part = W.h_part;
    res.assign(R, 0.0);
    for (int j = 0; j < R; j++) {
        double rr = 0, bb = 0;
        for (int q = 0; q < NB; q++) rr += part[((size_t)j * NB + q) * 4], bb += part[((size_t)j * NB + q) * 4 + 1];
        res[j] = bb > 0 ? std::sqrt(rr / bb) : 0.0;
    }
}

void solve(arh_hmat *h, int transpose, int R, const double2 *b, double2 *x, const arh_solve_opts &o,
           arh_solve_stats *st) {
    arh_geom *g = h->g;
    hipStream_t s = g->ctx->stream;
    const int N = g->N;
    const int NB = pick_nb(N);
    const int maxit = o.maxit > 0 ? o.maxit : 2 * N;
    const double tol = o.tol;
    ARH_CHECK(R >= 1, ARH_EINVAL, "nrhs must be >= 1");
    ARH_CHECK(tol >= 0.0, ARH_EINVAL, "tol must be >= 0");
    const auto t0 = std::chrono::steady_clock::now();
    Work W(N, R, NB, s);
    if (st) {
        st->iters = st->matvecs = st->refinements = st->restarts = 0;
        st->max_err = st->max_true_res = 0.0;
        if (st->hist_len)
            for (int j = 0; j < R; j++) st->hist_len[j] = 0;
    }
    std::vector<int> want(R, 1), iters, iters_tot(R, 0);
    std::vector<double> err, tres;
    if (h->storage != ARH_MIXED) {
        bicgstab(h, transpose, ARH_FP64, R, b, x, want, std::vector<double>(R, tol), maxit, o, st, iters, err, W, NB, true);
        for (int j = 0; j < R; j++) iters_tot[j] = iters[j];
        // optional: continue from x until the FP64 true residual meets tol; the correction solves
        // share what is left of maxit and stop when one no longer halves the worst residual
        int sweeps = 0;
        int left = maxit - *std::max_element(iters.begin(), iters.end());
        std::vector<double> last_err = err;
        if (o.true_residual || st) true_residual(h, transpose, R, b, x, nullptr, W, NB, tres, st);
        trace_sweep("fp64", 0, want, iters, tres);
        while (o.true_residual && sweeps < 8 && left > 0) {
            std::vector<int> redo(R, 0);
            int nre = 0;
            for (int j = 0; j < R; j++)
                if (tres[j] > tol) redo[j] = 1, nre++;
            if (!nre) break;
            const double worst = *std::max_element(tres.begin(), tres.end());
            // correction solve A d = b - A x for the unconverged rhs, then x += d
            DBuf rb, dx;
            rb.alloc(sizeof(double2) * (size_t)N * R);
            dx.alloc(sizeof(double2) * (size_t)N * R);
            true_residual(h, transpose, R, b, x, rb.as<double2>(), W, NB, tres, nullptr);
            // per-rhs tolerance relative to the current residual (no coupling between right-hand sides)
            std::vector<double> ctol(R);
            for (int j = 0; j < R; j++) ctol[j] = std::min(0.5, 0.5 * tol / std::max(tres[j], 1e-300));
            bicgstab(h, transpose, ARH_FP64, R, rb.as<double2>(), dx.as<double2>(), redo, ctol, left, o, st, iters,
                     err, W, NB, false);
            left -= *std::max_element(iters.begin(), iters.end());
            W.axpy(redo, N, x, dx.as<double2>(), 1.0);
            for (int j = 0; j < R; j++) iters_tot[j] += redo[j] ? iters[j] : 0;
            true_residual(h, transpose, R, b, x, nullptr, W, NB, tres, st);
            sweeps++;
            if (st) st->refinements++;
            if (*std::max_element(tres.begin(), tres.end()) > 0.5 * worst) break;
        }
        err = last_err;
    } else {
        // mixed: FP32-operator BiCGSTAB inside FP64 true-residual refinement. A sweep's correction is
        // kept for a right-hand side only if it cuts the FP64 true residual; an inner solve that
        // stalls, or a correction that does not pay, sends the right-hand side to FP64 correction
        // solves (the FP64 operator, Eigen's loop control), which converge whenever the FP64 path does.
        DBuf rb, dx;
        rb.alloc(sizeof(double2) * (size_t)N * R);
        dx.alloc(sizeof(double2) * (size_t)N * R);
        ARH_HIP(hipMemsetAsync(x, 0, sizeof(double2) * (size_t)N * R, s));
        std::vector<double> bnorm_rel(R, 1.0);  // ||r|| / ||b|| of the current residual
        std::vector<int> redo(R, 1), fp64(R, 0);
        const int stall = std::max(200, std::min(maxit, 400));
        for (int sweep = 0; sweep < 10; sweep++) {
            // per-rhs inner tolerance relative to its current residual, aiming at half the target (not
            // below kInnerFloor); no coupling between right-hand sides. An inner solve gets at most
            // kInnerBudget iterations: on a hard (ill-conditioned) problem the FP32 operator's
            // rounding slows BiCGSTAB to two or three times the FP64 iteration count, so such a
            // right-hand side goes to FP64 after a bounded FP32 attempt
            std::vector<double> itol(R);
            for (int j = 0; j < R; j++)
                itol[j] = std::min(0.5, std::max(kInnerFloor, kInnerFrac * tol / std::max(bnorm_rel[j], 1e-300)));
            bicgstab(h, transpose, ARH_MIXED, R, sweep == 0 ? b : rb.as<double2>(), dx.as<double2>(), redo, itol, maxit, o, st, iters,
                     err, W, NB, sweep == 0, stall, kInnerBudget);
            for (int j = 0; j < R; j++) iters_tot[j] += redo[j] ? iters[j] : 0;
            W.axpy(redo, N, x, dx.as<double2>(), 1.0);
            true_residual(h, transpose, R, b, x, rb.as<double2>(), W, NB, tres, st);
            if (st) st->refinements++;
            trace_sweep("fp32", sweep, redo, iters, tres);
            std::vector<int> undo(R, 0);
            int nundo = 0, nre = 0;
            for (int j = 0; j < R; j++) {
                // an inner solve that stopped short of its tolerance (stalled or hit maxit) marks a
                // problem the FP32 operator cannot resolve: finish in FP64 from here
                if (redo[j] && tres[j] > tol && err[j] > itol[j]) fp64[j] = 1;
                if (redo[j] && tres[j] > tol && tres[j] > 0.5 * bnorm_rel[j]) {
                    fp64[j] = 1;  // the FP32 correction did not pay: finish in FP64
                    if (tres[j] > bnorm_rel[j]) undo[j] = 1, nundo++;
                }
                if (!undo[j]) bnorm_rel[j] = tres[j];
                redo[j] = (bnorm_rel[j] > tol && !fp64[j]) ? 1 : 0;
                nre += redo[j];
            }
            if (nundo) {  // revert corrections that made the residual worse
                W.axpy(undo, N, x, dx.as<double2>(), -1.0);
                true_residual(h, transpose, R, b, x, rb.as<double2>(), W, NB, tres, st);
                for (int j = 0; j < R; j++) bnorm_rel[j] = tres[j];
            }
            if (!nre) break;
        }
        // FP64 correction solves for the right-hand sides still above tol; together they get maxit
        // iterations and stop when one no longer halves the worst residual
        int left = maxit;
        for (int sweep = 0; sweep < 8 && left > 0; sweep++) {
            std::vector<int> f64(R, 0);
            int nf = 0;
            double worst = 0.0;
            for (int j = 0; j < R; j++)
                if (tres[j] > tol) f64[j] = 1, nf++, worst = std::max(worst, tres[j]);
            if (!nf) break;
            std::vector<double> ctol(R);
            for (int j = 0; j < R; j++) ctol[j] = std::min(0.5, 0.5 * tol / std::max(tres[j], 1e-300));
            bicgstab(h, transpose, ARH_FP64, R, rb.as<double2>(), dx.as<double2>(), f64, ctol, left, o, st, iters,
                     err, W, NB, false);
            for (int j = 0; j < R; j++) iters_tot[j] += f64[j] ? iters[j] : 0;
            left -= *std::max_element(iters.begin(), iters.end());
            W.axpy(f64, N, x, dx.as<double2>(), 1.0);
            true_residual(h, transpose, R, b, x, rb.as<double2>(), W, NB, tres, st);
            if (st) st->refinements++;
            trace_sweep("fp64 correction", sweep, f64, iters, tres);
            double now = 0.0;
            for (int j = 0; j < R; j++)
                if (f64[j]) now = std::max(now, tres[j]);
            if (now > 0.5 * worst) break;
        }
        err = tres;
    }
    if (tres.empty()) true_residual(h, transpose, R, b, x, nullptr, W, NB, tres, st);
    if (st) {
        for (int j = 0; j < R; j++) {
            st->iters = std::max(st->iters, iters_tot[j]);
            st->max_err = std::max(st->max_err, err[j]);
            st->max_true_res = std::max(st->max_true_res, tres[j]);
            if (st->iters_per_rhs) st->iters_per_rhs[j] = iters_tot[j];
            if (st->true_res) st->true_res[j] = tres[j];
        }
        st->solve_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    }
    if (o.fail_on_noconv) {
        // true-residual modes are judged on the FP64 true residual, Eigen semantics on the recursive one
        const bool use_true = o.true_residual || h->storage == ARH_MIXED;
        for (int j = 0; j < R; j++) {
            const double e = use_true ? tres[j] : err[j];
            ARH_CHECK(e <= tol, ARH_ECONV,
                      "BiCGSTAB did not reach the tolerance (rhs " + std::to_string(j) + ", residual " +
                          std::to_string(e) + " > " + std::to_string(tol) + ")");
        }
    }
}

}  // namespace arh
