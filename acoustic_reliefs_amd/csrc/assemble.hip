// H-matrix assembly on gfx950: dense near-field panels and batched partially pivoted ACA.
#include <algorithm>
#include <numeric>
#include <type_traits>

#include "arh_internal.h"
#include "device_common.h"

namespace arh {

// Up to so many big blocks, one per compute unit, take 8 wavefronts each, more of them 4. Norms and dot products are
// summed per wavefront, so the stopping rule's left side rounds differently in the two: a cross within a few 1e-16 of the
// tolerance may be kept in one and not in the other, and a big block's rank then depends on how many the partition has.
// (One grouping for both would have 4 wavefronts form 8 partial sums: twice the dot products' reductions, for the meshes
// that are bound by VALU issue.) A geometry's own factors are the same in every assembly.
constexpr int kAcaFew = 256;
constexpr int kAcaWaves = 8;  // wavefronts of a big block's workgroup, at most
constexpr int kMaxRankLds = 128;  // max ACA rank kept in LDS coefficient arrays
#ifndef ARH_ACA_BIGDIM
#define ARH_ACA_BIGDIM 512
#endif
constexpr int kAcaBigDim = ARH_ACA_BIGDIM;  // blocks with m + n at least this get a workgroup, smaller ones a wavefront

// ------------------------------------------------------------------ dense panels
// One thread per entry of a (row leaf, column chunk) task; entries of a column are contiguous,
// so the store of a task is one coalesced run of nc * m complex values (compute_block,
// integrate.cpp:87-100, column by column).
__global__ __launch_bounds__(256) void k_dense(const DenseTask *__restrict__ tasks, const int *__restrict__ leaf_start,
                                               const int *__restrict__ pcol_ptr, const int64_t *__restrict__ panel_off,
                                               const int *__restrict__ pcol_idx, const Tri *__restrict__ tri, double k,
                                               double2 *__restrict__ out, int *__restrict__ nanflag) {
    const DenseTask t = tasks[blockIdx.x];
    const int rs = leaf_start[t.leaf];
    const int m = leaf_start[t.leaf + 1] - rs;
    const int tid = threadIdx.x;
    if (tid >= t.nc * m) return;
    const int cc = tid / m, i = tid - cc * m;
    const int c = t.c0 + cc;
    const int j = pcol_idx[pcol_ptr[t.leaf] + c];
    const Tri p = tri[rs + i];
    const Tri q = tri[j];
    double2 v = bem_entry(k, p.gx, p.gy, p.gz, q);
    if (isnan(v.x) || isnan(v.y)) atomicOr(nanflag, 1);
    out[panel_off[t.leaf] + (int64_t)c * m + i] = v;
}

// ------------------------------------------------------------------ wavefront maxima
__device__ __forceinline__ double wmax(double v) {
    v = fmax(v, dpp_f64<0x111>(v, v));
    v = fmax(v, dpp_f64<0x112>(v, v));
    v = fmax(v, dpp_f64<0x114>(v, v));
    v = fmax(v, dpp_f64<0x118>(v, v));
    v = fmax(v, dpp_f64<0x142>(v, v));
    v = fmax(v, dpp_f64<0x143>(v, v));
    return lane_f64(v, 63);
}
__device__ __forceinline__ int wmin_i(int v) {
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x118, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xF, 0xF, false));
    return __builtin_amdgcn_readlane(v, 63);
}

// Sums over the wavefront of eight complex values per lane, halving what each lane carries: after exchanging
// halves (permlane32_swap) and rows (permlane16_swap) row r (lanes 16 r ..) holds values 2 r and 2 r + 1 and sums
// them over its 16 lanes. Returns |value 2 r| in x and |value 2 r + 1| in y, the same in every lane of the row.
__device__ __forceinline__ void wsum8(const double2 *s, double2 &a, double2 &b) {
    double y[8];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        double p = s[t].x, q = s[t + 4].x;
        swap32(p, q);
        y[2 * t] = p + q;
        p = s[t].y, q = s[t + 4].y;
        swap32(p, q);
        y[2 * t + 1] = p + q;
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
        swap16(y[t], y[t + 4]);
        y[t] += y[t + 4];
    }
    a = make_double2(row_sum(y[0]), row_sum(y[1]));
    b = make_double2(row_sum(y[2]), row_sum(y[3]));
}

// ------------------------------------------------------------------ ACA
// compute_ACA_block (aca.cpp:38-82): start at row 0; residual row, first-max pivot column,
// normalised row (unnormalised if the pivot is 0), residual column, non-conjugated norm
// estimate, stop when sqrt(|u|^2|v|^2 / err) <= eps discarding the current cross, next row =
// first max of |u| over unused rows; rank limit min(max_rank, m-1, n-1).
// Crosses whose u or v is exactly zero add nothing to any later quantity, so they are counted
// (rank_ref) but not stored (rank).
//
// Crosses follow one another, so a block is a serial chain of entry evaluations (about 590 VALU operations for
// 64 entries), updates by the stored crosses, reductions and dot products. Blocks of up to 64 x 64 (four in five)
// are one wavefront each with a row and a column per lane in registers; larger ones loop over their rows and
// columns, as one wavefront or, from m + n >= kAcaBigDim, a workgroup. Loads of the stored crosses go out in batches
// ahead of their use (the first before the entry is evaluated), and reductions run on DPP: through ds_bpermute the
// dot products alone, 24 steps per stored cross, were half of a cross's time.
// 0.6 m relief, 16,058 blocks: 1.95 ms at 4000 Hz and 1.2 ms at 1000 Hz (3.95 and 1.9 ms with the bpermute
// reductions and unbatched loads), the factors bit for bit the same. Of that, at 4000 Hz, VALU instructions took 60 %
// and a third of the wavefront slots stood empty: the four blocks of a workgroup held their registers until the
// longest was done, and the largest block's chain alone took 1.94 ms, all others 1.65. So a block that a wavefront
// takes is a workgroup of its own, and up to kAcaFew big blocks get eight wavefronts instead of four, on a stream beside
// the others: whole FP64 assembly 2.30 -> 2.10 ms at 4000 Hz, 2.25 -> 1.99 with leaves of 64, 1.48 -> 1.44 with leaves of
// 128 at 1000 Hz, where leaves of 32 (1.53 -> 1.51) are bound by VALU issue throughout. Eight wavefronts for every big
// block of a larger mesh (0.9 m, 1000 Hz) take 18.2 ms instead of 16.2: there the chip is full anyway and the blocks' idle
// wavefronts cost. A queue that persistent wavefronts pull from keeps the slots full too, but the loop around the
// chains spills (2.42 ms at 4000 Hz). 2 or 4 wavefronts per SIMD (4: spills) measured the same or slower.

// |v|^2 of the pivot searches. On symmetric meshes two entries can tie exactly, and this rounding decides between
// them: it is part of the result, so the fused form is written out.
__device__ __forceinline__ double pivot_norm(double2 v) { return fma(v.x, v.x, v.y * v.y); }

// Factors of the rule's point (w, xi, eta) in bem_entry: its contribution is f (tr, ti).
struct EntryPoint {
    double f, tr, ti;
};
__device__ __forceinline__ EntryPoint entry_point(double k, double px, double py, double pz, const Tri &t, double w,
                                                  double xi, double eta) {
    const double qx = t.ax + xi * t.bx + eta * t.cx;
    const double qy = t.ay + xi * t.by + eta * t.cy;
    const double qz = t.az + xi * t.bz + eta * t.cz;
    const double dx = px - qx, dy = py - qy, dz = pz - qz;
    const double r2 = dx * dx + dy * dy + dz * dz;
    const double r = sqrt(r2);
    const double s = -(dx * t.nx + dy * t.ny + dz * t.nz);
    const double kr = k * r;
    double sn, cs;
    trig_sincos(kr, &sn, &cs);
    return EntryPoint{w * s / (r2 * r), -cs - kr * sn, sn - kr * cs};
}

// bem_entry of up to 64 rows or columns, one per lane, bit for bit, with the six points in three pairs shared out
// when lanes are left over: `share` lanes per entry (3 for up to 21 entries, 2 for up to 32, else 1), lane e + s
// 64 / share (s < share) works on entry e, lane e < 64 / share adds the pairs up in order.
__device__ __forceinline__ double2 entry_shared(double k, double px, double py, double pz, const Tri &t, int share,
                                                int lane) {
    const int width = share == 3 ? 21 : share == 2 ? 32 : 64;
    const int s = share == 1 ? 0 : lane / width;
    double re = 0.0, im = 0.0;
    const int rounds = 4 - share;
#pragma unroll 1
    for (int z = 0; z < rounds; z++) {
        const int b = z == 0 ? s : share == 1 ? z : 2;  // (lane 63 of three shares repeats a pair, unused)
        const bool b1 = b == 1, b2 = b >= 2;
        const EntryPoint A = entry_point(k, px, py, pz, t, b2 ? ARH_QW_B : ARH_QW_A,
                                         b1 ? ARH_Q_2 : b2 ? ARH_Q_3 : ARH_Q_1, b1 ? ARH_Q_1 : b2 ? ARH_Q_3 : ARH_Q_2);
        const EntryPoint C = entry_point(k, px, py, pz, t, b1 || b2 ? ARH_QW_B : ARH_QW_A,
                                         b1 ? ARH_Q_3 : b2 ? ARH_Q_4 : ARH_Q_1, b1 ? ARH_Q_4 : b2 ? ARH_Q_3 : ARH_Q_1);
        re = fma(A.f, A.tr, re), im = fma(A.f, A.ti, im);
        re = fma(C.f, C.tr, re), im = fma(C.f, C.ti, im);
        for (int o = 1; z == 0 && o < share; o++) {
            const int src = lane + o * width;
            double f = __shfl(A.f, src, ARH_WAVE);
            re = fma(f, __shfl(A.tr, src, ARH_WAVE), re), im = fma(f, __shfl(A.ti, src, ARH_WAVE), im);
            f = __shfl(C.f, src, ARH_WAVE);
            re = fma(f, __shfl(C.tr, src, ARH_WAVE), re), im = fma(f, __shfl(C.ti, src, ARH_WAVE), im);
        }
    }
    return make_double2(re * kInv8Pi, im * kInv8Pi);
}

// v - sum_p a_p b_p over the stored crosses p < sr in order: b_p = own[p * stride], a_p = coef(p) (uniform).
// Batches of kAcaBatch loads, two in flight; `first` was loaded by load_batch(.., 0) before.
constexpr int kAcaBatch = 8;
struct AcaBatch {
    double2 b[kAcaBatch];
};
__device__ __forceinline__ void load_batch(AcaBatch &B, const double2 *__restrict__ own, int64_t stride, int p0,
                                           int sr) {
    const int last = max(sr - 1, 0);  // row 0 always exists; surplus loads repeat the last cross, unused
#pragma unroll
    for (int t = 0; t < kAcaBatch; t++) B.b[t] = own[min(p0 + t, last) * stride];
}
template <class Coef>
__device__ __forceinline__ void use_batch(double2 &v, const AcaBatch &B, int p0, int sr, Coef &&coef) {
#pragma unroll
    for (int t = 0; t < kAcaBatch; t++)
        if (p0 + t < sr) {
            const double2 up = coef(p0 + t), vp = B.b[t];
            v.x -= up.x * vp.x - up.y * vp.y;
            v.y -= up.x * vp.y + up.y * vp.x;
        }
}
template <class Coef>
__device__ __forceinline__ void residual(double2 &v, AcaBatch &first, const double2 *__restrict__ own, int64_t stride,
                                         int sr, Coef &&coef) {
    AcaBatch next;
    for (int p0 = 0; p0 < sr; p0 += 2 * kAcaBatch) {
        load_batch(next, own, stride, p0 + kAcaBatch, sr);
        use_batch(v, first, p0, sr, coef);
        if (p0 + kAcaBatch >= sr) break;
        load_batch(first, own, stride, p0 + 2 * kAcaBatch, sr);
        use_batch(v, next, p0 + kAcaBatch, sr, coef);
    }
}

// A block of at most 64 x 64, one wavefront: lane q holds row q and column q of the current cross.
__device__ __forceinline__ void aca_small(int2 *__restrict__ ranks, int bid, const LRBlock &B, int lane,
                                          const Tri *__restrict__ tri, double k, double eps, double2 *__restrict__ U,
                                          double2 *__restrict__ V) {
    const int m = B.re - B.rs, n = B.ce - B.cs, lim = B.lim;
    const int q = min(lane, m - 1), c = min(lane, n - 1);
    const bool rowon = lane < m, colon = lane < n;
    // lanes that share an entry hold its row or column too
    auto share_of = [](int e) { return e <= 21 ? 3 : e <= 32 ? 2 : 1; };
    auto entry_of = [&](int e) { return min(e <= 21 ? lane % 21 : e <= 32 ? lane % 32 : lane, e - 1); };
    const int mshare = share_of(m), nshare = share_of(n);
    const Tri tc = tri[B.cs + entry_of(n)];
    const Tri &tq = tri[B.rs + entry_of(m)];
    const double gx = tq.gx, gy = tq.gy, gz = tq.gz;
    bool used = lane == 0;
    int i = 0, it = 0, sr = 0;
    double err = 0.0;
    // coefficient p of the current cross is in lane p (lim <= 63 here)
    auto coef_in = [&](const double2 &cf) {
        return [&cf](int p) { return make_double2(lane_f64(cf.x, p), lane_f64(cf.y, p)); };
    };
    while (it < lim) {
        AcaBatch b;
        load_batch(b, V + c, n, 0, sr);
        double2 cf = U[(int64_t)min(lane, max(sr - 1, 0)) * m + i];
        double2 v = entry_shared(k, lane_f64(gx, i), lane_f64(gy, i), lane_f64(gz, i), tc, nshare, lane);
        residual(v, b, V + c, n, sr, coef_in(cf));
        // first maximum of |v|^2 (NaN never wins; column 0 if nothing does)
        double a = pivot_norm(v);
        a = colon && a == a ? a : -1.0;
        double best = wmax(a);
        const int j = best < 0.0 ? 0 : __builtin_ctzll(__ballot(a == best));
        load_batch(b, U + q, m, 0, sr);
        cf = V[(int64_t)min(lane, max(sr - 1, 0)) * n + j];
        const double2 piv = make_double2(lane_f64(v.x, j), lane_f64(v.y, j));
        if (piv.x != 0.0 || piv.y != 0.0) v = cdiv(v, piv);
        if (colon) V[(int64_t)sr * n + lane] = v;
        double2 u = entry_shared(k, gx, gy, gz, tri[B.cs + j], mshare, lane);
        residual(u, b, U + q, m, sr, coef_in(cf));
        if (rowon) U[(int64_t)sr * m + lane] = u;
        a = pivot_norm(u);
        const double un = wsum(rowon ? a : 0.0), vn = wsum(colon ? cnorm2(v) : 0.0);
        a = rowon && !used && a == a ? a : -1.0;
        best = wmax(a);
        const int ni = best < 0.0 ? 0 : __builtin_ctzll(__ballot(a == best));
        // |u_p^T u| and |v v_p^T| for the stored crosses p < sr (aca.cpp:64-69), eight at a time
        double dots = 0.0;
        const double2 uz = rowon ? u : make_double2(0.0, 0.0), vz = colon ? v : make_double2(0.0, 0.0);
        for (int p0 = 0; p0 < sr; p0 += kAcaBatch) {
            AcaBatch bu, bv;
            load_batch(bu, U + q, m, p0, sr);
            load_batch(bv, V + c, n, p0, sr);
#pragma unroll
            for (int t = 0; t < kAcaBatch; t++) bu.b[t] = cmul(uz, bu.b[t]), bv.b[t] = cmul(vz, bv.b[t]);
            double2 su, su1, sv, sv1;
            wsum8(bu.b, su, su1);
            wsum8(bv.b, sv, sv1);
            const int p = p0 + 2 * (lane >> 4);  // surplus crosses (repeats) and lanes are not added
            if ((lane & 15) == 0 && p < sr) dots += sqrt(cnorm2(su)) * sqrt(cnorm2(sv));
            if ((lane & 15) == 1 && p + 1 < sr) dots += sqrt(cnorm2(su1)) * sqrt(cnorm2(sv1));
        }
        dots = wsum(dots);
        err += un * vn + 2.0 * dots;
        if (sqrt(un * vn / err) <= eps) break;
        if (un * vn > 0.0) sr++;
        i = ni;
        used = used || lane == i;
        it++;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the new cross is read by other lanes
        __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0) ranks[bid] = make_int2(sr, it);
}

struct AcaShared {
    double2 coef[kMaxRankLds];
    double2 piv;
    double rv[4][kAcaWaves];
    int ri[kAcaWaves];
};
template <int W>
struct AcaSharedGroup : AcaShared {
    double2 dd[W][kMaxRankLds][2];  // kMaxRankLds is a multiple of the batch
};

// The threads working on one larger block: a workgroup of W wavefronts or a single wavefront (W = 1, no
// workgroup barrier: a wavefront's memory operations complete in order, so a fence at wavefront scope, which
// also stops compiler reordering, is its barrier).
template <int W>
struct AcaGroup {
    static constexpr bool WAVE = W == 1;
    int tid, w, lane;
    std::conditional_t<WAVE, AcaShared, AcaSharedGroup<W>> &sh;
    static constexpr int nthr = W * ARH_WAVE;
    __device__ __forceinline__ void sync() const {
        if (WAVE) {
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
    }
    // fixed-order sum, the same bits in every thread; slot: one of the shared arrays (a later sum with the same
    // slot needs a sync in between)
    __device__ __forceinline__ double sum(double v, int slot) const {
        v = wsum(v);
        if (WAVE) return v;
        if (lane == 0) sh.rv[slot][w] = v;
        __syncthreads();
        double s = sh.rv[slot][0];
#pragma unroll
        for (int q = 1; q < W; q++) s += sh.rv[slot][q];
        return s;
    }
    // (value, index) max with ties to the lower index
    __device__ __forceinline__ void argmax(double &v, int &i, int slot) const {
        const double b = wmax(v);
        i = wmin_i(v == b ? i : 0x7fffffff);
        v = b;
        if (WAVE) return;
        if (lane == 0) sh.rv[slot][w] = v, sh.ri[w] = i;
        __syncthreads();
        v = sh.rv[slot][0];
        i = sh.ri[0];
#pragma unroll
        for (int q = 1; q < W; q++)
            if (sh.rv[slot][q] > v || (sh.rv[slot][q] == v && sh.ri[q] < i)) v = sh.rv[slot][q], i = sh.ri[q];
    }
};

template <int W>
__device__ __forceinline__ void aca_block(const AcaGroup<W> &G, int2 *__restrict__ ranks, int bid,
                                          const LRBlock &B, const Tri *__restrict__ tri, double k, double eps,
                                          double2 *__restrict__ U, double2 *__restrict__ V,
                                          unsigned char *__restrict__ used) {
    auto &sh = G.sh;
    const int rs = B.rs, cs = B.cs, m = B.re - B.rs, n = B.ce - B.cs, lim = B.lim;
    const int tid = G.tid, lane = G.lane;
    constexpr bool WAVE = W == 1;
    constexpr int nthr = AcaGroup<W>::nthr;
    for (int q = tid; q < m; q += nthr) used[q] = (q == 0) ? 1 : 0;
    int i = 0, it = 0, sr = 0;
    double err = 0.0;
    const auto coef = [&](int p) { return sh.coef[p]; };
    G.sync();
    while (it < lim) {
        // coefficients U(i, p), p < sr
        for (int p = tid; p < sr; p += nthr) sh.coef[p] = U[(int64_t)p * m + i];
        G.sync();
        // residual row into V row `sr`, with the first-max pivot search
        const Tri ti = tri[rs + i];
        double2 *vrow = V + (int64_t)sr * n;
        double best = -1.0;
        double2 bv = make_double2(0.0, 0.0);
        int bi = 0x7fffffff;
        for (int c = tid; c < n; c += nthr) {
            AcaBatch b;
            load_batch(b, V + c, n, 0, sr);
            double2 v = bem_entry(k, ti.gx, ti.gy, ti.gz, tri[cs + c]);
            residual(v, b, V + c, n, sr, coef);
            vrow[c] = v;
            const double a = pivot_norm(v);
            if (a > best) best = a, bi = c, bv = v;
            if (c == 0 && best < 0.0) bv = v;  // the pivot when no entry wins (all NaN)
        }
        const int mine = bi;
        G.argmax(best, bi, 0);
        const int j = (best < 0.0) ? 0 : bi;
        if (best < 0.0 ? tid == 0 : mine == j) sh.piv = bv;
        // the coefficients of the column: every use of the row's is over (argmax has synchronised, or in order)
        for (int p = tid; p < sr; p += nthr) sh.coef[p] = V[(int64_t)p * n + j];
        G.sync();
        const double2 piv = sh.piv;
        const bool nz = (piv.x != 0.0 || piv.y != 0.0);
        double vn = 0.0;
        for (int c = tid; c < n; c += nthr) {
            double2 v = vrow[c];
            if (nz) v = cdiv(v, piv), vrow[c] = v;
            vn += cnorm2(v);
        }
        // residual column into U column `sr`, with the masked first-max search for the next row
        const Tri tj = tri[cs + j];
        double2 *ucol = U + (int64_t)sr * m;
        double un = 0.0, bu = -1.0;
        int bq = 0x7fffffff;
        for (int q = tid; q < m; q += nthr) {
            AcaBatch b;
            load_batch(b, U + q, m, 0, sr);
            const Tri &tq = tri[rs + q];
            double2 u = bem_entry(k, tq.gx, tq.gy, tq.gz, tj);
            residual(u, b, U + q, m, sr, coef);
            ucol[q] = u;
            const double a = pivot_norm(u);
            un += a;
            if (!used[q] && a > bu) bu = a, bq = q;
        }
        vn = G.sum(vn, 1);
        un = G.sum(un, 2);
        G.argmax(bu, bq, 3);
        G.sync();  // the new cross is written (a wavefront alone has passed no barrier since)
        // |u_p^T u| and |v v_p^T| for stored crosses p < sr (aca.cpp:64-69), eight at a time: every thread takes its
        // own rows and columns, wavefront sums through wsum8, wavefronts added in order
        double dots = 0.0;
        for (int p0 = 0; p0 < sr; p0 += kAcaBatch) {
            double2 su[kAcaBatch], sv[kAcaBatch];
#pragma unroll
            for (int t = 0; t < kAcaBatch; t++) su[t] = sv[t] = make_double2(0.0, 0.0);
            for (int q = tid; q < m; q += nthr) {
                AcaBatch b;
                load_batch(b, U + q, m, p0, sr);
                const double2 uq = ucol[q];
#pragma unroll
                for (int t = 0; t < kAcaBatch; t++) cfma(su[t], uq, b.b[t]);
            }
            for (int c = tid; c < n; c += nthr) {
                AcaBatch b;
                load_batch(b, V + c, n, p0, sr);
                const double2 vc = vrow[c];
#pragma unroll
                for (int t = 0; t < kAcaBatch; t++) cfma(sv[t], vc, b.b[t]);
            }
            double2 a[4];
            wsum8(su, a[0], a[1]);
            wsum8(sv, a[2], a[3]);
            const int p = p0 + 2 * (lane >> 4);  // surplus crosses (repeats) are not added
            if constexpr (WAVE) {
                if ((lane & 15) == 0 && p < sr) dots += sqrt(cnorm2(a[0])) * sqrt(cnorm2(a[2]));
                if ((lane & 15) == 1 && p + 1 < sr) dots += sqrt(cnorm2(a[1])) * sqrt(cnorm2(a[3]));
            } else if ((lane & 15) == 0) {
                sh.dd[G.w][p][0] = a[0], sh.dd[G.w][p][1] = a[2];
                sh.dd[G.w][p + 1][0] = a[1], sh.dd[G.w][p + 1][1] = a[3];
            }
        }
        if constexpr (!WAVE) {
            __syncthreads();
            for (int p = lane; p < sr; p += ARH_WAVE) {
                double2 su = sh.dd[0][p][0], sv = sh.dd[0][p][1];
#pragma unroll
                for (int q = 1; q < W; q++) su = cadd(su, sh.dd[q][p][0]), sv = cadd(sv, sh.dd[q][p][1]);
                dots += sqrt(cnorm2(su)) * sqrt(cnorm2(sv));
            }
        }
        dots = wsum(dots);
        err += un * vn + 2.0 * dots;
        if (sqrt(un * vn / err) <= eps) break;
        if (un * vn > 0.0) sr++;
        i = (bu < 0.0) ? 0 : bq;
        if (tid == 0) used[i] = 1;
        it++;
        G.sync();
    }
    if (tid == 0) ranks[bid] = make_int2(sr, it);
}

// A workgroup of W wavefronts per big block (order[0..nbig)). nan: raised by the dense blocks.
template <int W>
__global__ __launch_bounds__(W * ARH_WAVE, 2) void k_aca_big(const LRBlock *__restrict__ blocks,
                                                          const int *__restrict__ order, const Tri *__restrict__ tri,
                                                          double k, double eps, double2 *__restrict__ Us,
                                                          double2 *__restrict__ Vs, unsigned char *__restrict__ flags,
                                                          const int *__restrict__ nan, int2 *__restrict__ ranks) {
    __shared__ AcaSharedGroup<W> sh;
    if (*nan) return;  // the assembly fails
    const int bid = order[blockIdx.x];
    const LRBlock B = blocks[bid];
    if (B.lim <= 0) {  // a single row or column, or max_rank 0
        if (threadIdx.x == 0) ranks[bid] = make_int2(0, 0);
        return;
    }
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / ARH_WAVE));
    const AcaGroup<W> G{(int)threadIdx.x, w, (int)(threadIdx.x % ARH_WAVE), sh};
    aca_block<W>(G, ranks, bid, B, tri, k, eps, Us + B.us_off, Vs + B.vs_off, flags + B.flag_off);
}

// A wavefront per other block, each a workgroup of its own (so that a finished block's slot is free at once).
__global__ __launch_bounds__(ARH_WAVE, 3) void k_aca(const LRBlock *__restrict__ blocks, const int *__restrict__ order,
                                                  const Tri *__restrict__ tri, double k, double eps,
                                                  double2 *__restrict__ Us, double2 *__restrict__ Vs,
                                                  unsigned char *__restrict__ flags, const int *__restrict__ nan,
                                                  int2 *__restrict__ ranks) {
    __shared__ AcaShared sh;
    if (*nan) return;
    const int lane = threadIdx.x;
    const int bid = order[blockIdx.x];
    const LRBlock B = blocks[bid];
    double2 *U = Us + B.us_off, *V = Vs + B.vs_off;
    if (B.lim <= 0) {
        if (lane == 0) ranks[bid] = make_int2(0, 0);
    } else if (B.re - B.rs <= ARH_WAVE && B.ce - B.cs <= ARH_WAVE) {
        aca_small(ranks, bid, B, lane, tri, k, eps, U, V);
    } else {
        const AcaGroup<1> G{lane, 0, lane, sh};
        aca_block<1>(G, ranks, bid, B, tri, k, eps, U, V, flags + B.flag_off);
    }
}

// ------------------------------------------------------------------ offsets
// The blocks' descriptors with their ranks and the offsets of their factors (running sums over the blocks in order), the
// blocks of rank > 0, and for the host, in pinned memory, ranks and totals. Workgroup b takes blocks [1024 b, 1024 b +
// 1024) and sums up all before them by itself, so one launch does. (The host ran the sums between two 1.3 MB copies of
// the descriptors, 0.7 ms of an idle GPU at 17,500 blocks.)
struct LrTotals {
    int64_t u, v, t;
    int nact, nan;
};
__device__ __forceinline__ void lr_sizes(const LRBlock &B, int r, int64_t q[4]) {
    q[0] = (int64_t)r * (B.re - B.rs), q[1] = (int64_t)r * (B.ce - B.cs), q[2] = r, q[3] = r > 0 ? 1 : 0;
}
__global__ __launch_bounds__(1024) void k_lr_offsets(int na, const LRBlock *__restrict__ lr0,
                                                     const int2 *__restrict__ ranks, const int *__restrict__ nan,
                                                     LRBlock *__restrict__ blocks, int *__restrict__ active,
                                                     int2 *__restrict__ hranks, LrTotals *__restrict__ tot) {
    __shared__ int64_t sh[2][1024 / ARH_WAVE][4];
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE;
    const int a0 = (int)blockIdx.x * 1024, a = a0 + (int)threadIdx.x;
    if (*nan) {
        if (a == na - 1) tot->nan = 1;
        return;
    }
    int64_t pre[4] = {0, 0, 0, 0}, own[4] = {0, 0, 0, 0}, q[4];
#pragma unroll 8
    for (int b = threadIdx.x; b < a0; b += 1024) {
        lr_sizes(lr0[b], ranks[b].x, q);
#pragma unroll
        for (int k = 0; k < 4; k++) pre[k] += q[k];
    }
    LRBlock B{};
    int2 r = make_int2(0, 0);
    if (a < na) {
        B = lr0[a], r = ranks[a];
        lr_sizes(B, r.x, own);
    }
    int64_t inc[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        inc[k] = own[k];
        for (int d = 1; d < ARH_WAVE; d <<= 1) {
            const int64_t up = __shfl_up(inc[k], d, ARH_WAVE);
            if (lane >= d) inc[k] += up;
            pre[k] += __shfl_xor(pre[k], d, ARH_WAVE);
        }
        if (lane == ARH_WAVE - 1) sh[0][w][k] = inc[k], sh[1][w][k] = pre[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; k++)
        for (int v = 0; v < 1024 / ARH_WAVE; v++) inc[k] += sh[1][v][k] + (v < w ? sh[0][v][k] : 0);
    if (a >= na) return;
    B.rank = r.x, B.u_off = inc[0] - own[0], B.v_off = inc[1] - own[1], B.t_off = inc[2] - own[2];
    blocks[a] = B;
    if (r.x > 0) active[inc[3] - 1] = a;
    hranks[a] = r;
    if (a == na - 1) {
        tot->u = inc[0], tot->v = inc[1], tot->t = inc[2], tot->nact = (int)inc[3];
        tot->nan = 0;
    }
}

// ------------------------------------------------------------------ compaction
// U scratch (m x lim) -> leaf-segmented packed U: for each row leaf [ls, le) of the block, an
// (le-ls) x rank column-major chunk at u_off + (ls - rs) * rank. V scratch -> rank x n row-major.
// A block's crosses are shared out over gridDim.y workgroups, a wavefront per cross: with one workgroup per
// block the largest blocks' copies were a tail: 255 us at 4000 Hz (790 MB), 224 with two, 202 with four or eight.
constexpr int kPackSplit = 4;
__global__ __launch_bounds__(256) void k_pack(const LRBlock *__restrict__ blocks, const int *__restrict__ active,
                                              const int *__restrict__ leaf_start, const int *__restrict__ leaf_of,
                                              const double2 *__restrict__ Us, const double2 *__restrict__ Vs,
                                              double2 *__restrict__ U, double2 *__restrict__ V) {
    const LRBlock B = blocks[active[blockIdx.x]];
    const int m = B.re - B.rs, n = B.ce - B.cs, r = B.rank;
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE, nw = 256 / ARH_WAVE;
    for (int p = (int)blockIdx.y * nw + w; p < r; p += (int)gridDim.y * nw) {
        const double2 *us = Us + B.us_off + (int64_t)p * m, *vs = Vs + B.vs_off + (int64_t)p * n;
        double2 *v = V + B.v_off + (int64_t)p * n;
#pragma unroll 4
        for (int c = lane; c < n; c += ARH_WAVE) v[c] = vs[c];
        for (int i = lane; i < m; i += ARH_WAVE) {
            const int l = leaf_of[B.rs + i];
            const int ls = leaf_start[l] - B.rs, ms = leaf_start[l + 1] - leaf_start[l];
            U[B.u_off + (int64_t)ls * r + (int64_t)p * ms + (i - ls)] = us[i];
        }
    }
}

// FP32 copy of V, transposed per block to column-major (n x r, V32[v_off + c r + p]): the MFMA
// product reads 16 consecutive rank rows of one column.
__global__ __launch_bounds__(256) void k_v_to_c64_cm(const LRBlock *__restrict__ blocks, const int *__restrict__ active,
                                                     const double2 *__restrict__ V, float2 *__restrict__ V32) {
    const LRBlock B = blocks[active[blockIdx.x]];
    const int n = B.ce - B.cs, r = B.rank;
    const int64_t tot = (int64_t)r * n;
    for (int64_t e = threadIdx.x; e < tot; e += blockDim.x) {
        const int c = (int)(e / r), p = (int)(e - (int64_t)c * r);
        const double2 v = V[B.v_off + (int64_t)p * n + c];
        V32[B.v_off + e] = make_float2((float)v.x, (float)v.y);
    }
}

__global__ void k_to_c64(const double2 *__restrict__ a, float2 *__restrict__ b, int64_t n) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        double2 v = a[e];
        b[e] = make_float2((float)v.x, (float)v.y);
    }
}

// ------------------------------------------------------------------ host drivers
static void check_nan(int nan) {
    ARH_CHECK(!nan, ARH_ENAN, "NaN in a dense near-field block (a collocation point coincides with a quadrature point)");
}

// Low-rank blocks as the partition and max_rank fix them.
static void lr_plan(arh_geom *g, int max_rank) {
    if (g->lr_plan_rank == max_rank) return;
    g->lr_plan_rank = -1;
    hipStream_t s = g->ctx->stream;
    const int na = g->na;
    std::vector<LRBlock> lr(na, LRBlock{});
    int64_t uo = 0, vo = 0, fo = 0;
    for (int a = 0; a < na; a++) {
        LRBlock &B = lr[a];
        B.rs = g->lowrank[4 * a], B.re = g->lowrank[4 * a + 1], B.cs = g->lowrank[4 * a + 2];
        B.ce = g->lowrank[4 * a + 3];
        const int m = B.re - B.rs, n = B.ce - B.cs;
        B.lim = std::max(0, std::min(max_rank, std::min(m - 1, n - 1)));
        B.l0 = g->leaf_of[B.rs];
        B.us_off = uo, B.vs_off = vo, B.flag_off = fo;
        uo += (int64_t)m * B.lim, vo += (int64_t)B.lim * n, fo += m;
    }
    g->aca_u_total = uo, g->aca_v_total = vo, g->aca_f_total = fo;
    // largest work first: the ACA cost grows like lim^2 (m + n)
    std::vector<int> order(na);
    std::vector<double> work(na);
    for (int a = 0; a < na; a++) {
        const LRBlock &B = lr[a];
        const double mn = B.re - B.rs + B.ce - B.cs;
        order[a] = a, work[a] = (double)B.lim * B.lim * mn + mn;
    }
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return work[x] > work[y]; });
    // blocks with m + n >= kAcaBigDim get a workgroup each (they lead the order, largest first);
    // the rest one wavefront each
    const auto big = [&](int x) { return lr[x].re - lr[x].rs + lr[x].ce - lr[x].cs >= kAcaBigDim; };
    const auto mid = std::stable_partition(order.begin(), order.end(), big);
    g->aca_nbig = (int)(mid - order.begin());
    upload(g->d_lr0, lr, s);
    upload(g->d_aca_order, order, s);
    ARH_HIP(hipStreamSynchronize(s));  // the host vectors are freed on return
    g->lr_plan_rank = max_rank;
}

// Work on a second stream beside a stream's own, between everything before and everything after on that one. Left
// without join (an error on the way), it waits for the second stream, whose kernels use the first one's buffers.
struct Fork {
    hipStream_t main, side;
    bool joined = false;
    Fork(hipStream_t m, hipStream_t s) : main(m), side(s) {
        if (side != main) order(main, side);
    }
    void join() {
        if (side != main) order(side, main);
        joined = true;
    }
    ~Fork() {
        if (!joined && side != main) (void)hipStreamSynchronize(side);
    }
    static void order(hipStream_t from, hipStream_t to) {
        hipEvent_t e;
        ARH_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        hipError_t r = hipEventRecord(e, from);
        if (r == hipSuccess) r = hipStreamWaitEvent(to, e, 0);
        (void)hipEventDestroy(e);
        ARH_HIP(r);
    }
};

// Dense panels, then the ACA: one wait for the device, with the ranks (and whether a dense entry was a NaN) in pinned
// memory, before the factors' storage can be allocated.
void assemble(arh_hmat *h) {
    arh_geom *g = h->g;
    hipStream_t s = g->ctx->stream;
    const int na = g->na;
    h->dense.alloc(sizeof(double2) * std::max<int64_t>(1, g->dense_entries));
    DBuf flag;
    flag.alloc(sizeof(int));
    ARH_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), s));
    if (!g->dtasks.empty()) {
        hipLaunchKernelGGL(k_dense, dim3((unsigned)g->dtasks.size()), dim3(256), 0, s, g->d_dtasks.as<DenseTask>(),
                           g->d_leaf_start.as<int>(), g->d_pcol_ptr.as<int>(), g->d_panel_off.as<int64_t>(),
                           g->d_pcol_idx.as<int>(), g->tri.as<Tri>(), h->k, h->dense.as<double2>(), flag.as<int>());
        ARH_HIP(hipGetLastError());
    }
    h->ranks.clear();
    h->n_active = 0;
    h->u_total = h->v_total = h->t_total = 0;
    if (na == 0 || h->max_rank > kMaxRankLds) {
        int nan = 0;
        ARH_HIP(hipMemcpyAsync(&nan, flag.p, sizeof(int), hipMemcpyDeviceToHost, s));
        ARH_HIP(hipStreamSynchronize(s));
        check_nan(nan);
        ARH_CHECK(na == 0, ARH_EINVAL, "max_rank above the supported 128");
        if (h->storage == ARH_MIXED) make_fp32_copy(h);
        return;
    }
    lr_plan(g, h->max_rank);
    // scratch from the device memory cache; it goes back there once the factors are packed, so an idle geometry holds none
    DBuf us, vs, used, ranks, active;
    us.alloc(sizeof(double2) * std::max<int64_t>(1, g->aca_u_total));
    vs.alloc(sizeof(double2) * std::max<int64_t>(1, g->aca_v_total));
    used.alloc(std::max<int64_t>(16, g->aca_f_total));
    ranks.alloc(sizeof(int2) * (size_t)na);
    active.alloc(sizeof(int) * (size_t)na);
    h->blocks.alloc(sizeof(LRBlock) * (size_t)na);
    HostBuf hb(sizeof(LrTotals) + sizeof(int2) * (size_t)na, s);
    LrTotals *tot = hb.as<LrTotals>();
    int2 *hranks = (int2 *)(tot + 1);
    const int nbig = g->aca_nbig;
    {
        // the big blocks go first, on the context's stream; the others beside them on the auxiliary one
        Fork fork(s, nbig && na > nbig ? g->ctx->aux() : s);
        auto big = [&](auto kern, int waves) {
            hipLaunchKernelGGL(kern, dim3(nbig), dim3(waves * ARH_WAVE), 0, s, g->d_lr0.as<LRBlock>(),
                               g->d_aca_order.as<int>(), g->tri.as<Tri>(), h->k, h->aca_tol, us.as<double2>(),
                               vs.as<double2>(), used.as<unsigned char>(), flag.as<int>(), ranks.as<int2>());
        };
        if (nbig > kAcaFew)
            big(k_aca_big<4>, 4);
        else if (nbig)
            big(k_aca_big<8>, 8);
        if (na > nbig)
            hipLaunchKernelGGL(k_aca, dim3(na - nbig), dim3(ARH_WAVE), 0, fork.side, g->d_lr0.as<LRBlock>(),
                               g->d_aca_order.as<int>() + nbig, g->tri.as<Tri>(), h->k, h->aca_tol, us.as<double2>(),
                               vs.as<double2>(), used.as<unsigned char>(), flag.as<int>(), ranks.as<int2>());
        ARH_HIP(hipGetLastError());
        fork.join();
    }
    hipLaunchKernelGGL(k_lr_offsets, dim3((na + 1023) / 1024), dim3(1024), 0, s, na, g->d_lr0.as<LRBlock>(),
                       ranks.as<int2>(), flag.as<int>(), h->blocks.as<LRBlock>(), active.as<int>(), hranks, tot);
    ARH_HIP(hipGetLastError());
    ARH_HIP(hipStreamSynchronize(s));
    check_nan(tot->nan);
    h->u_total = tot->u, h->v_total = tot->v, h->t_total = tot->t;
    h->n_active = tot->nact;
    h->U.alloc(sizeof(double2) * std::max<int64_t>(1, h->u_total));
    h->V.alloc(sizeof(double2) * std::max<int64_t>(1, h->v_total));
    h->d_active_lr.alloc(sizeof(int) * (size_t)h->n_active);
    if (h->n_active) {
        hipLaunchKernelGGL(k_pack, dim3((unsigned)h->n_active, kPackSplit), dim3(256), 0, s, h->blocks.as<LRBlock>(),
                           active.as<int>(), g->d_leaf_start.as<int>(), g->d_leaf_of.as<int>(), us.as<double2>(),
                           vs.as<double2>(), h->U.as<double2>(), h->V.as<double2>());
        ARH_HIP(hipGetLastError());
        ARH_HIP(hipMemcpyAsync(h->d_active_lr.p, active.p, sizeof(int) * (size_t)h->n_active, hipMemcpyDeviceToDevice, s));
    }
    // The scratch goes back before the FP32 layout takes its room (the packing above precedes it on the stream), so the
    // two do not add up: 0.9 m relief, N = 58,724, peak of a mixed assembly 24.8 GB at 1000 Hz (27.0 with the scratch
    // held until the return), 25.6 at 3150 Hz (28.2).
    us.reset();
    vs.reset();
    used.reset();
    // while the factors are packed
    h->ranks.assign(hranks, hranks + na);
    if (h->storage == ARH_MIXED) make_fp32_copy(h);
}

// FP32 copy for the generic (non-MFMA) product: dense panels and U elementwise, V column-major
// per block. Built on first use.
void make_generic_fp32(arh_hmat *h) {
    if (h->generic32) return;
    arh_geom *g = h->g;
    hipStream_t s = g->ctx->stream;
    auto conv = [&](DBuf &src, DBuf &dst, int64_t n) {
        dst.alloc(sizeof(float2) * std::max<int64_t>(1, n));
        if (n > 0) {
            int blocks = (int)std::min<int64_t>(4096, (n + 255) / 256);
            hipLaunchKernelGGL(k_to_c64, dim3(blocks), dim3(256), 0, s, src.as<double2>(), dst.as<float2>(), n);
            ARH_HIP(hipGetLastError());
        }
    };
    conv(h->dense, h->dense32, g->dense_entries);
    conv(h->U, h->U32, h->u_total);
    h->V32.alloc(sizeof(float2) * std::max<int64_t>(1, h->v_total));
    if (h->n_active) {
        hipLaunchKernelGGL(k_v_to_c64_cm, dim3((unsigned)h->n_active), dim3(256), 0, s, h->blocks.as<LRBlock>(),
                           h->d_active_lr.as<int>(), h->V.as<double2>(), h->V32.as<float2>());
        ARH_HIP(hipGetLastError());
    }
    ARH_HIP(hipStreamSynchronize(s));
    h->generic32 = true;
}

// FP32 copy at assembly: the MFMA layout when the leaves fit it, else the generic one.
void make_fp32_copy(arh_hmat *h) {
    if (h->g->max_leaf <= mfma_max_leaf())
        mfma_prepare(h, 0, 0);
    else
        make_generic_fp32(h);
}

}  // namespace arh
