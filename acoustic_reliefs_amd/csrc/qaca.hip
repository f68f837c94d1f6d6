// Listener ACA on gfx950: one partially pivoted ACA over the whole LL x N receiver matrix
// Q_lj = entry(listener l, element j) (compute_ACA_listener, aca.cpp:84-134), then y = U (V x) and
// its transpose V^T (U^T x) (adjoint.cpp:101-102, 177-178).
//
// Unlike the block ACA (one workgroup per block), this is a single large block, so every stage of a
// cross is a grid-wide kernel, two launches per cross c:
//   k_qa_row: the next row from the column maxima of cross c - 1; residual row c (N entries) with block-partial
//     first-max; in further workgroups the non-conjugated dot products of cross c - 1 with the stored crosses (chunk
//     partials);
//   k_qa_normcol: pivot, row normalisation and residual column c (LL entries, masked first-max); in one further
//     workgroup the stopping rule for cross c - 1.
// So cross c is begun before the rule has seen cross c - 1; if that one stops, c is left behind unused. A launch takes
// 4 to 7 us whatever it holds (serial chains: maxima, entry, stored crosses, sums) and the gap to the next
// one 5, so the count of launches is what the time goes with: with the dots and the rule as launches of their own
// a cross of the 1297 x 9828 matrix (rank 195) took 28 us, now 17.6.
// A residual row or column block takes 64 entries (one per lane), the sum over the stored crosses split between kQS
// wavefronts and the entry formed by another one, so the grid grows with the rank as well as with
// N or LL. All reductions are two-stage with a fixed order. The loop control lives on the device (a `done` flag every
// kernel checks); the host launches a few crosses at a time and reads the state of one such batch while the next one runs.
//
// Semantics kept from aca.cpp:84-134: start at row 0 (used = {0}); V row = v / v_j with no zero-pivot
// guard (aca.cpp:104); error estimate with |u|^2 |v|^2 + 2 sum |u_p^T u| |v v_p^T|; stop when
// sqrt(|u|^2 |v|^2 / err) <= eps discarding the current cross; crosses are kept even when zero;
// iteration limit min(max_rank, LL - 1, N - 1).
#include <algorithm>

#include "arh_internal.h"
#include "device_common.h"

namespace arh {

constexpr int kQT = 256;  // threads per block of the products, per half block of the dots
constexpr int kQS = 8;    // slices of the stored crosses in a residual row / column block, a wavefront each
constexpr int kQB = (kQS + 1) * ARH_WAVE;  // its threads: one more wavefront for the entries
constexpr int kQBatch = 8;  // crosses launched together

// State after the stopping rule has seen crosses < it (it crosses kept), in two copies: k_qa_normcol of cross c
// reads copy (c + 1) & 1 and writes copy c & 1.
struct QAcaState {
    double err;
    int it, done, lim, pad;
};

// sum over the block's first kQT threads; every thread of the block calls it
__device__ __forceinline__ double block_sum_q(double v, double *sv) {
    v = wave_sum(v);
    const int w = threadIdx.x / ARH_WAVE, lane = threadIdx.x % ARH_WAVE;
    __syncthreads();
    if (lane == 0 && w < kQT / ARH_WAVE) sv[w] = v;
    __syncthreads();
    double s = sv[0];
    for (int q = 1; q < kQT / ARH_WAVE; q++) s += sv[q];
    return s;
}

// Slice w of the stored-cross sum of a residual entry: sum over p in wave w's share of [0, it) of
// a(p) b(p), where the lane's own operand is own[p * ostride] and the shared one is shared[p * sstride].
__device__ __forceinline__ double2 cross_slice(int it, int w, const double2 *__restrict__ own, int64_t ostride,
                                               const double2 *__restrict__ shared, int64_t sstride) {
    const int chunk = (it + kQS - 1) / kQS, p0 = w * chunk, p1 = min(it, p0 + chunk);
    double2 acc = make_double2(0.0, 0.0);
#pragma unroll 8
    for (int p = p0; p < p1; p++) {
        const double2 a = shared[p * sstride], b = own[p * ostride];
        acc.x += a.x * b.x - a.y * b.y;
        acc.y += a.x * b.y + a.y * b.x;
    }
    return acc;
}

// entry - (slice 0 + ... ): the last wave subtracts the kQS slice sums in order (the others leave theirs in red and
// return false)
__device__ __forceinline__ bool combine_slices(double2 &v, double2 (*red)[ARH_WAVE], int w, int lane) {
    if (w < kQS) red[w][lane] = v;
    __syncthreads();
    if (w < kQS) return false;
#pragma unroll
    for (int q = 0; q < kQS; q++) v.x -= red[q][lane].x, v.y -= red[q][lane].y;
    return true;
}

constexpr int kQC = 8 * kQT;  // entries of a dot product chunk

// Workgroups [0, nbr): residual row i of cross c into V row c (unnormalised) + block partial first-max of |v|^2 (64
// columns a block). The row is 0 for c = 0, else the first maximum over the column blocks' partials of cross c - 1 (ties to
// the lower index; 0 if every row is used), which the first workgroup marks as used.
// The others: chunk partials of the non-conjugated products u^T u_p and v v_p^T of cross c - 1 with the stored
// crosses p < c - 1 (aca.cpp:64-69 / :114-116), two (p, chunk) pairs per workgroup: chunks [0, ncu) over U's LL rows
// and [ncu, ncu + ncv) over V's N columns; pu[p * ncu + chunk], pv[p * ncv + chunk].
__global__ __launch_bounds__(kQB) void k_qa_row(const QAcaState *__restrict__ S, int c, const double *__restrict__ L,
                                                const Tri *__restrict__ tri, double k, int LL, int N,
                                                const double2 *__restrict__ U, double2 *__restrict__ V,
                                                unsigned char *__restrict__ used, const double *__restrict__ pcol,
                                                int nbc, int nbr, double *__restrict__ pmax, int ncu, int ncv,
                                                double2 *__restrict__ pu, double2 *__restrict__ pv) {
    __shared__ double2 red[kQS][ARH_WAVE];
    __shared__ double sv[kQB / ARH_WAVE];
    __shared__ int si;
    if (S->done) return;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / ARH_WAVE)), lane = threadIdx.x % ARH_WAVE;
    if ((int)blockIdx.x >= nbr) {
        const int half = w / (kQT / ARH_WAVE);  // the last wave takes no part
        const int e = 2 * ((int)blockIdx.x - nbr) + half, p = e / (ncu + ncv), h = e - p * (ncu + ncv);
        const bool on = half < 2 && p < c - 1, isu = h < ncu;
        double2 acc = make_double2(0.0, 0.0);
        if (on) {
            const int n = isu ? LL : N, c0 = (isu ? h : h - ncu) * kQC, c1 = min(n, c0 + kQC);
            const double2 *a = isu ? U + (int64_t)(c - 1) * LL : V + (int64_t)(c - 1) * N;
            const double2 *b = isu ? U + (int64_t)p * LL : V + (int64_t)p * N;
            for (int q = c0 + (int)threadIdx.x % kQT; q < c1; q += kQT) cfma(acc, a[q], b[q]);
        }
        acc.x = wave_sum(acc.x);
        acc.y = wave_sum(acc.y);
        if (lane == 0) red[0][w] = acc;
        __syncthreads();
        if (on && threadIdx.x % kQT == 0) {
            const int w0 = half * (kQT / ARH_WAVE);
            double2 s = red[0][w0];
            for (int q = 1; q < kQT / ARH_WAVE; q++) s.x += red[0][w0 + q].x, s.y += red[0][w0 + q].y;
            if (isu)
                pu[(int64_t)p * ncu + h] = s;
            else
                pv[(int64_t)p * ncv + (h - ncu)] = s;
        }
        return;
    }
    int i = 0;
    if (c > 0) {
        if (w == 0) {
            double bv = -1.0;
            int bi = 0x7fffffff;
            for (int b = lane; b < nbc; b += ARH_WAVE) {
                const double v = pcol[3 * b + 1];
                const int l = (int)pcol[3 * b + 2];
                if (v > bv || (v == bv && l < bi)) bv = v, bi = l;
            }
            wave_argmax(bv, bi);
            if (lane == 0) si = bv < 0.0 ? 0 : bi;
        }
        __syncthreads();
        i = __builtin_amdgcn_readfirstlane(si);
        if (blockIdx.x == 0 && threadIdx.x == 0) used[i] = 1;
    }
    const int col = blockIdx.x * ARH_WAVE + lane, cc = min(col, N - 1);  // loads clamped, stores guarded
    double2 v;
    if (w == kQS)
        v = bem_entry(k, L[3 * i], L[3 * i + 1], L[3 * i + 2], tri[cc]);
    else
        v = cross_slice(c, w, V + cc, N, U + i, LL);
    if (!combine_slices(v, red, w, lane)) return;
    double best = -1.0;
    int bi = 0x7fffffff;
    if (col < N) {
        V[(int64_t)c * N + col] = v;
        const double a = cnorm2(v);
        best = a == a ? a : -1.0, bi = col;  // NaN never wins
    }
    wave_argmax(best, bi);
    // the partial carries v at the block's first maximum, so the pivot value is known without reading the
    // row while it is being normalised
    const int src = bi - (int)blockIdx.x * ARH_WAVE;
    const int sl = src >= 0 && src < ARH_WAVE ? src : 0;
    const double vr = __shfl(v.x, sl, ARH_WAVE), vi = __shfl(v.y, sl, ARH_WAVE);
    if (lane == 0) {
        double *o = pmax + 4 * blockIdx.x;
        o[0] = best, o[1] = (double)bi, o[2] = vr, o[3] = vi;
    }
}

// Stopping rule for cross c - 1 (a whole workgroup; fixed-order reductions): error estimate with its norms and dot
// products, the new state to out and, for the last launch of a batch, to the host's pinned copy.
__device__ __forceinline__ void qa_finish(const QAcaState &st0, QAcaState *__restrict__ out, QAcaState *host, int c,
                                          double eps, const double *__restrict__ pvn, int nbn,
                                          const double *__restrict__ pcol, int nbc, const double2 *__restrict__ pu, int ncu,
                                          const double2 *__restrict__ pv, int ncv, double *sv) {
    QAcaState st = st0;
    if (c > 0 && !st0.done) {
        const int t = threadIdx.x;
        double vn = 0.0, un = 0.0, d = 0.0;
        if (t < kQT) {
            for (int b = t; b < nbn; b += kQT) vn += pvn[b];
            for (int b = t; b < nbc; b += kQT) un += pcol[3 * b];
            for (int p = t; p < c - 1; p += kQT) {
                double2 su = make_double2(0.0, 0.0), sq = make_double2(0.0, 0.0);
                for (int q = 0; q < ncu; q++) su.x += pu[(int64_t)p * ncu + q].x, su.y += pu[(int64_t)p * ncu + q].y;
                for (int q = 0; q < ncv; q++) sq.x += pv[(int64_t)p * ncv + q].x, sq.y += pv[(int64_t)p * ncv + q].y;
                d += cabs_(su) * cabs_(sq);
            }
        }
        vn = block_sum_q(vn, sv);
        un = block_sum_q(un, sv);
        d = block_sum_q(d, sv);
        st.err += un * vn + 2.0 * d;
        if (sqrt(un * vn / st.err) <= eps) {
            st.done = 1;  // cross c - 1 discarded: rank = c - 1
        } else {
            st.it = c;
            if (st.it >= st.lim) st.done = 1;
        }
    }
    if (threadIdx.x == 0) {
        *out = st;
        if (host) *host = st;
    }
}

// One launch after the residual row of cross c, workgroups [0, nbn) normalising V row c (512 columns each, block
// partials of |v|^2), [nbn, nbn + nbc) forming the residual column j (64 rows each), and a last one applying the stopping
// rule to cross c - 1. Every workgroup of the first two kinds
// first finds the pivot column j = the first maximum over the row blocks' partials (ties to the lower
// index, so it is the sequential first maximum) and takes v_j from the winning partial.
__global__ __launch_bounds__(kQB) void k_qa_normcol(const QAcaState *__restrict__ S, QAcaState *__restrict__ So,
                                                    QAcaState *__restrict__ host, int c, double eps,
                                                    const double *__restrict__ L, const Tri *__restrict__ tri, double k,
                                                    int LL, int N, double2 *__restrict__ U, double2 *__restrict__ V,
                                                    const unsigned char *__restrict__ used,
                                                    const double *__restrict__ pmax, int nbr, int nbn, int nbc,
                                                    double *__restrict__ pvn, double *__restrict__ pcol,
                                                    const double *__restrict__ pvn1, const double *__restrict__ pcol1,
                                                    const double2 *__restrict__ pu, int ncu,
                                                    const double2 *__restrict__ pv, int ncv) {
    __shared__ double2 red[kQS][ARH_WAVE];
    __shared__ double sv[kQB / ARH_WAVE];
    __shared__ int sj;
    __shared__ double2 spiv;
    const QAcaState st = *S;
    if (blockIdx.x == gridDim.x - 1) {
        // (nbn and nbc are 0 in a launch of this workgroup alone: the partials' counts come from the sizes)
        qa_finish(st, So, host, c, eps, pvn1, (N + kQS * ARH_WAVE - 1) / (kQS * ARH_WAVE), pcol1,
                  (LL + ARH_WAVE - 1) / ARH_WAVE, pu, ncu, pv, ncv, sv);
        return;
    }
    if (st.done) return;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / ARH_WAVE)), lane = threadIdx.x % ARH_WAVE;
    if (w == 0) {
        double bv = -1.0;
        int bj = 0x7fffffff;
        for (int b = lane; b < nbr; b += ARH_WAVE) {
            const double v = pmax[4 * b];
            const int j = (int)pmax[4 * b + 1];
            if (v > bv || (v == bv && j < bj)) bv = v, bj = j;
        }
        wave_argmax(bv, bj);
        if (lane == 0) {
            const double *o = pmax + 4 * (bj / ARH_WAVE);  // the row block holding column bj
            sj = bj, spiv = make_double2(o[2], o[3]);
        }
    }
    __syncthreads();
    const int j = __builtin_amdgcn_readfirstlane(sj);
    if ((int)blockIdx.x < nbn) {
        // V row c /= v_j (no zero-pivot guard, aca.cpp:104) + block partial of |v|^2 (the last wave has no columns)
        const int col = blockIdx.x * (kQS * ARH_WAVE) + threadIdx.x;
        double a = 0.0;
        if (w < kQS && col < N) {
            const double2 v = cdiv(V[(int64_t)c * N + col], spiv);
            V[(int64_t)c * N + col] = v;
            a = cnorm2(v);
        }
        a = wave_sum(a);
        if (lane == 0) sv[w] = a;
        __syncthreads();
        if (threadIdx.x == 0) {
            double t = sv[0];
            for (int q = 1; q < kQS; q++) t += sv[q];
            pvn[blockIdx.x] = t;
        }
        return;
    }
    // residual column j into U column c + block partials of |u|^2 and of the masked first-max
    const int bc = (int)blockIdx.x - nbn;
    const int l = bc * ARH_WAVE + lane, ll = min(l, LL - 1);
    double2 u;
    if (w == kQS)
        u = bem_entry(k, L[3 * ll], L[3 * ll + 1], L[3 * ll + 2], tri[j]);
    else
        u = cross_slice(c, w, U + ll, LL, V + j, N);
    if (!combine_slices(u, red, w, lane)) return;
    double a = 0.0, best = -1.0;
    int bi = 0x7fffffff;
    if (l < LL) {
        U[(int64_t)c * LL + l] = u;
        a = cnorm2(u);
        if (!used[l]) best = a == a ? a : -1.0, bi = l;
    }
    a = wave_sum(a);
    wave_argmax(best, bi);
    if (lane == 0) pcol[3 * bc] = a, pcol[3 * bc + 1] = best, pcol[3 * bc + 2] = (double)bi;
}

// products: t = V x (rank x nrhs, one block per (p, j)); y = U t (a thread per row: eight loads in flight keep its
// serial sum from waiting for each: 43 -> 26 us at 1297 x 9828, rank 182)
__global__ __launch_bounds__(kQT) void k_qa_vx(int N, int r, const double2 *__restrict__ V, const double2 *__restrict__ x,
                                              double2 *__restrict__ t) {
    __shared__ double sv[kQT / ARH_WAVE];
    const int p = blockIdx.x, j = blockIdx.y;
    double2 s = make_double2(0.0, 0.0);
    for (int c = threadIdx.x; c < N; c += kQT) {
        const double2 a = V[(int64_t)p * N + c], b = x[(int64_t)j * N + c];
        s.x += a.x * b.x - a.y * b.y;
        s.y += a.x * b.y + a.y * b.x;
    }
    s.x = block_sum_q(s.x, sv);
    s.y = block_sum_q(s.y, sv);
    if (threadIdx.x == 0) t[(int64_t)j * r + p] = s;
}

__global__ void k_qa_ut(int LL, int r, int nrhs, const double2 *__restrict__ U, const double2 *__restrict__ t,
                        double2 *__restrict__ y) {
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (e >= (int64_t)LL * nrhs) return;
    const int j = (int)(e / LL), l = (int)(e % LL);
    double2 s = make_double2(0.0, 0.0);
#pragma unroll 8
    for (int p = 0; p < r; p++) {
        const double2 a = U[(int64_t)p * LL + l], b = t[(int64_t)j * r + p];
        s.x += a.x * b.x - a.y * b.y;
        s.y += a.x * b.y + a.y * b.x;
    }
    y[e] = s;
}

// transposed: s = U^T x (rank x nrhs, one block per (p, j)); y = V^T s
__global__ __launch_bounds__(kQT) void k_qa_utx(int LL, int r, const double2 *__restrict__ U,
                                               const double2 *__restrict__ x, double2 *__restrict__ t) {
    __shared__ double sv[kQT / ARH_WAVE];
    const int p = blockIdx.x, j = blockIdx.y;
    double2 s = make_double2(0.0, 0.0);
    for (int l = threadIdx.x; l < LL; l += kQT) {
        const double2 a = U[(int64_t)p * LL + l], b = x[(int64_t)j * LL + l];
        s.x += a.x * b.x - a.y * b.y;
        s.y += a.x * b.y + a.y * b.x;
    }
    s.x = block_sum_q(s.x, sv);
    s.y = block_sum_q(s.y, sv);
    if (threadIdx.x == 0) t[(int64_t)j * r + p] = s;
}

__global__ void k_qa_vts(int N, int r, int nrhs, const double2 *__restrict__ V, const double2 *__restrict__ t,
                         double2 *__restrict__ y) {
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (e >= (int64_t)N * nrhs) return;
    const int j = (int)(e / N), c = (int)(e % N);
    double2 s = make_double2(0.0, 0.0);
#pragma unroll 8
    for (int p = 0; p < r; p++) {
        const double2 a = V[(int64_t)p * N + c], b = t[(int64_t)j * r + p];
        s.x += a.x * b.x - a.y * b.y;
        s.y += a.x * b.y + a.y * b.x;
    }
    y[e] = s;
}

// build the factors (host loop over batches of crosses)
void qaca_build(arh_qaca *q, const double *L_host) {
    arh_geom *g = q->g;
    hipStream_t s = g->ctx->stream;
    const int LL = q->LL, N = q->N, lim = q->lim;
    const std::vector<double> hL(L_host, L_host + 3 * (size_t)LL);  // alive until the stream is synchronised
    upload(q->L, hL, s);
    q->U.alloc(sizeof(double2) * std::max<int64_t>(1, (int64_t)LL * lim));
    q->V.alloc(sizeof(double2) * std::max<int64_t>(1, (int64_t)lim * N));
    q->nbr = (N + ARH_WAVE - 1) / ARH_WAVE;               // residual row blocks
    q->nbn = (N + kQS * ARH_WAVE - 1) / (kQS * ARH_WAVE);  // row normalisation blocks
    q->nbc = (LL + ARH_WAVE - 1) / ARH_WAVE;               // residual column blocks
    // first maxima of the row blocks, then norms and first maxima of two crosses
    const size_t np = q->nbn + 3 * (size_t)q->nbc;
    q->part.alloc(sizeof(double) * (4 * (size_t)q->nbr + 2 * np + 16));
    const int ncu = (LL + kQC - 1) / kQC, ncv = (N + kQC - 1) / kQC;
    q->dots.alloc(sizeof(double2) * (size_t)std::max(1, lim) * (ncu + ncv));
    q->rank = 0;
    if (lim <= 0) {
        ARH_HIP(hipStreamSynchronize(s));
        return;
    }
    std::vector<unsigned char> used(LL, 0);
    used[0] = 1;
    upload(q->used, used, s);
    HostBuf hb(4 * sizeof(QAcaState), s);
    QAcaState *hst = hb.as<QAcaState>();  // state after batch b at b & 1; then the initial copies
    hst[2].err = 0.0, hst[2].it = 0, hst[2].done = 0, hst[2].lim = lim, hst[2].pad = 0;
    hst[3] = hst[2];
    q->st.alloc(2 * sizeof(QAcaState));
    ARH_HIP(hipMemcpyAsync(q->st.p, hst + 2, 2 * sizeof(QAcaState), hipMemcpyHostToDevice, s));
    double *pmax = q->part.as<double>(), *par = pmax + 4 * q->nbr;
    QAcaState *S = q->st.as<QAcaState>();
    const Tri *tri = g->tri.as<Tri>();
    double2 *U = q->U.as<double2>(), *V = q->V.as<double2>();
    double2 *pu = q->dots.as<double2>(), *pv = pu + (size_t)lim * ncu;
    // cross c (c == lim: the stopping rule for the last cross alone)
    auto cross = [&](int c, QAcaState *host) {
        double *cur = par + (c & 1) * np, *prev = par + ((c + 1) & 1) * np;
        const QAcaState *Si = S + ((c + 1) & 1);
        const int nbr = c < lim ? q->nbr : 0, nbn = c < lim ? q->nbn : 0, nbc = c < lim ? q->nbc : 0;
        const int nd = c > 1 ? ((c - 1) * (ncu + ncv) + 1) / 2 : 0;
        if (nbr + nd > 0)
            hipLaunchKernelGGL(k_qa_row, dim3(nbr + nd), dim3(kQB), 0, s, Si, c, q->L.as<double>(), tri, q->k, LL, N, U,
                               V, q->used.as<unsigned char>(), prev + q->nbn, q->nbc, nbr, pmax, ncu, ncv, pu, pv);
        hipLaunchKernelGGL(k_qa_normcol, dim3(nbn + nbc + 1), dim3(kQB), 0, s, Si, S + (c & 1), host, c, q->tol,
                           q->L.as<double>(), tri, q->k, LL, N, U, V, q->used.as<unsigned char>(), pmax, nbr, nbn, nbc,
                           cur, cur + q->nbn, prev, prev + q->nbn, pu, ncu, pv, ncv);
    };
    struct Events {
        hipEvent_t e[2] = {};
        ~Events() {
            for (hipEvent_t v : e)
                if (v) (void)hipEventDestroy(v);
        }
    } ev;
    for (hipEvent_t &e : ev.e) ARH_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    // batch b is launched before the state after batch b - 1 is read (launches after the stop return at once)
    int launched = 0;  // crosses 0 .. launched - 1
    for (int b = 0;; b++) {
        if (launched < lim) {
            const int end = std::min(lim, launched + kQBatch);
            for (; launched < end; launched++)
                cross(launched, launched + 1 == end && end < lim ? hst + (b & 1) : nullptr);
            if (end == lim) cross(lim, hst + (b & 1));
            ARH_HIP(hipGetLastError());
            ARH_HIP(hipEventRecord(ev.e[b & 1], s));
        }
        if (b == 0) continue;
        ARH_HIP(hipEventSynchronize(ev.e[(b - 1) & 1]));
        const QAcaState hs = hst[(b - 1) & 1];
        if (hs.done) {
            q->rank = hs.it;
            break;
        }
        ARH_CHECK(b <= lim, ARH_EINVAL, "internal: listener ACA ran past its limit");
    }
}

void qaca_apply(arh_qaca *q, int transpose, int nrhs, const double2 *x, double2 *y) {
    hipStream_t s = q->g->ctx->stream;
    const int r = q->rank;
    const int64_t ny = (int64_t)(transpose ? q->N : q->LL) * nrhs;
    if (r == 0) {
        ARH_HIP(hipMemsetAsync(y, 0, sizeof(double2) * ny, s));
        return;
    }
    q->t.alloc(sizeof(double2) * (size_t)r * nrhs);
    if (!transpose) {
        hipLaunchKernelGGL(k_qa_vx, dim3(r, nrhs), dim3(kQT), 0, s, q->N, r, q->V.as<double2>(), x, q->t.as<double2>());
        hipLaunchKernelGGL(k_qa_ut, dim3((unsigned)((ny + 255) / 256)), dim3(256), 0, s, q->LL, r, nrhs,
                           q->U.as<double2>(), q->t.as<double2>(), y);
    } else {
        hipLaunchKernelGGL(k_qa_utx, dim3(r, nrhs), dim3(kQT), 0, s, q->LL, r, q->U.as<double2>(), x,
                           q->t.as<double2>());
        hipLaunchKernelGGL(k_qa_vts, dim3((unsigned)((ny + 255) / 256)), dim3(256), 0, s, q->N, r, nrhs,
                           q->V.as<double2>(), q->t.as<double2>(), y);
    }
    ARH_HIP(hipGetLastError());
}

}  // namespace arh
