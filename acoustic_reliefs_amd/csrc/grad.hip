// Shape gradient of the diffusion coefficient w.r.t. vertex heights (y coordinates).
//
// Restates compute_der_A/B/C (adjoint.cpp:244-386) restructured per "touched" element i (an
// element with at least one differentiable vertex) so each derivative is evaluated once and
// shared by the three corners and by every rhs of a batch:
//   A_(i,c) = sum_rhs Re( x_i  sum_l  vf_l  dQ_li / dq_(i,c) )                 (adjoint.cpp:268-277)
//   B_(i,c) = sum_rhs Re( lam_i sum_e x_e dM_ie / dp_i ) + Re( x_i sum_e lam_e dM_ei / dq_(i,c) )   (:314-339)
//   C_(i,c) = -sum_rhs Re( lam_i db_i / dp_i )                                  (:373)
// and gradient_h = sum_{(i,c) : E[i][c] = h} A - B + C (element order, then corner order, as the
// reference's elements[h] lists, acoustics3d.cpp:83-98).
// Derivatives (derived from the kernel, not transcribed from derivatives.cpp): with d = p - q,
// r = |d|, s = -(d . n), F = e^{-ikr}(-ikr-1)/(4 pi r^3), F' = e^{-ikr}(-k^2/r^2 + 3(1+ikr)/r^4)/(4 pi):
//   collocation centroid moves (dp/dh = e_y/3):   dK = (F' d_y s / r - F n_y) / 3
//   corner c of the integration triangle moves (dq/dh = beta_c e_y, beta = (1-xi-eta, xi, eta)):
//                                                 dK = -F' beta_c d_y s / r + F (beta_c n_y - d . dn_c)
//   dn_a = e_y x (b - c), dn_b = e_y x (c - a), dn_c = (b - a) x e_y.
#include <algorithm>
#include <vector>

#include "arh_internal.h"
#include "device_common.h"

namespace arh {

// Restructured over the right-hand sides too: the sums over rhs and over elements commute, so
//   B_(i,c) = Re sum_e ( dM_ie/dp_i G(i,e) + dM_ei/dq_(i,c) G(e,i) ),  G(i,e) = sum_rhs lam_i x_e,
//   A_(i,c) = Re sum_l dQ_li/dq_(i,c) W(i,l),                          W(i,l) = sum_rhs x_i vf_l,
// and a derivative is evaluated once per pair whatever the number of right-hand sides. G and W are GEMMs: a
// wavefront forms a 16 x 16 tile of pairs with v_mfma_f64_16x16x4_f64 and consumes it from the accumulators,
// so they are never stored.
//
// Per pair, with ir = 1 / r and the quadrature sums over a triangle's six points (weights w, beta the corner's
// barycentric coordinate): s = -(d . n) does not depend on the point (q stays in the triangle's plane, so
// d . n = (p - a) . n), and neither does beta_c n_y - d . dn_c, the y derivative of d . n for a moving corner
// (it is linear in q). With D_c = (p - a) . dn_c it equals n_y - D_a for corner a and -D_b, -D_c for the others:
//   dM_ie/dp_i     = (s sum w F' d_y ir - n_y sum w F) / 6
//   dM_ei/dq_(i,c) = (-s sum w beta_c F' d_y ir + (n_y [c = a] - D_c) sum w F) / 2.
//
// Bound by FP64 VALU issue: about 68 FP64 operations per quadrature point, 12 points per pair, against 4 MFMAs per
// two right-hand sides for 256 pairs. Reciprocal distances come from one v_rsq_f64 and one cubic correction step
// (below 1 ulp) instead of a square root and five divisions. The loop over a lane's four pairs stays rolled: unrolled
// it needs 249 registers, 2 wavefronts per SIMD instead of 3, and 3-5 % more time; 4 wavefronts spill (+14 %).
// N = 9,828 with 8,442 touched elements, 8e7 pairs: 3.1 ms for one right-hand side and 4.6 ms for 37, where
// accumulating every right-hand side's sums per lane took 10.3 ms and 24.6 ms (two passes, each with its own
// derivatives); 1297 listeners, one right-hand side: 0.24 ms from 2.6 ms. With the pairs of touched elements taken
// both ways at once (k_grad_both) the whole call goes from 3.27 to 2.15 ms and from 4.47 to 2.90 ms.
constexpr int kGW = 4;           // wavefronts per workgroup; they take every kGW-th 16-column tile of the split
constexpr int kGT = 64 * kGW;
constexpr int kGSlots = 2048;    // workgroups aimed for (8 per compute unit): the column range is split to reach it

// Blocks of touched elements from which their pairs are taken both ways at once: fewer leave the chip half empty. The
// two are equal at 26 (N = 2,618) to 40 (N = 58,724) blocks, and little apart around there. Whole call, one way and
// both ways:
//   N = 2,618:  24 blocks, one rhs 424 and 432 us, 37 rhs 523 and 536 us; 28 blocks 442 and 425, 564 and 530
//   N = 9,828:  28 blocks 866 and 881 us, 1174 and 1180 us; 36 blocks 1008 and 997, 1396 and 1349
//   N = 58,724: 28 blocks 3.93 and 4.00 ms, 5.78 and 5.82 ms; 48 blocks 6.62 and 6.50, 9.77 and 9.62
constexpr int kGMinBlocks = 28;
// Room for their partial sums at a time, 48 bytes per touched element and offset (k_grad_both): all of them up to
// 13,000 touched elements, else strips of offsets one after the other. 0.9 m relief (51,834 touched, 406 offsets, whole
// call): one rhs 56.2 ms, 37 82.1 ms in 16 strips; 55.9 and 81.2 ms at once, which takes 1.0 GB. Strips of 128 and 256
// MB measured the same.
constexpr int64_t kGPartBytes = int64_t(64) << 20;

typedef double V4d __attribute__((ext_vector_type(4)));

// 1 / sqrt(x): with e = 1 - x y^2 of the hardware's y (about 2^-24), y (1 + e / 2 + 3 e^2 / 8) leaves O(e^3).
__device__ __forceinline__ double rsqrt_f64(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// Kernel factors at distance vector d without the 1 / (4 pi): F = e^{-ikr} (-1 - ikr) / r^3 and
// H = d_y / r e^{-ikr} (-k^2 / r^2 + 3 (1 + ikr) / r^4). FAR: r2 ir is off by up to 1.5 units in the last place, which
// the phase k r of a far point takes over (k r reaches some thousands at listeners), so one correction step makes r as
// good as a rounded root. The listener term against 80 bits, 50 m and 3150 Hz, 5 m and 4000 Hz: 1.28e-13 and 2.25e-14
// without the step, 1.11e-13 and 1.82e-14 with it; plain double precision 1.11e-13 and 1.92e-14; no time measurable
// (1297 listeners, whole call 2.08 ms). Element pairs are a metre apart at most: their error comes from the near pairs
// and is below a rounded root's formula by division either way (7.5e-15 against 9.2e-15 at 4000 Hz), and the step would
// cost 2.5 % of the call there.
template <bool FAR = false>
__device__ __forceinline__ void FdF(double k, double dx, double dy, double dz, double2 &F, double2 &H) {
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const double ir = rsqrt_f64(r2);
    double r = r2 * ir;
    if (FAR) r = fma(0.5 * ir, fma(-r, r, r2), r);
    const double kr = k * r;
    double sn, cs;
    trig_sincos(kr, &sn, &cs);
    const double ir2 = ir * ir, ir3 = ir2 * ir;
    F = make_double2(fma(-kr, sn, -cs) * ir3, fma(-kr, cs, sn) * ir3);
    const double g = dy * ir * ir2;
    const double A = fma(3.0, ir2, -k * k) * g, B = 3.0 * k * ir * g;
    H = make_double2(fma(cs, A, sn * B), fma(cs, B, -sn * A));
}

// Rows of a pair tile: the touched elements' derived geometry, in LDS (wavefront lanes of one row read the same
// address, rows are an odd number of doubles apart).
struct GradRow {
    double q[6][3];         // quadrature points
    double ax, ay, az, nx, ny, nz, gx, gy, gz;
    double cx, cz, bx, bz;  // c - a and b - a (dn of the corners)
    double pad[2];
};
static_assert(sizeof(GradRow) % 16 == 8, "odd number of doubles");

__device__ __forceinline__ void fill_row(GradRow &r, const Tri &t) {
#pragma unroll
    for (int g = 0; g < 6; g++) {
        double wt, xi, eta;
        quad_point(g, wt, xi, eta);
        r.q[g][0] = t.ax + xi * t.bx + eta * t.cx;
        r.q[g][1] = t.ay + xi * t.by + eta * t.cy;
        r.q[g][2] = t.az + xi * t.bz + eta * t.cz;
    }
    r.ax = t.ax, r.ay = t.ay, r.az = t.az, r.nx = t.nx, r.ny = t.ny, r.nz = t.nz;
    r.gx = t.gx, r.gy = t.gy, r.gz = t.gz;
    r.bx = t.bx, r.bz = t.bz, r.cx = t.cx, r.cz = t.cz;
}

// Right-hand-side values element by element for the pair GEMMs: row e holds (re, im) of the R values of one vector
// set, zero-padded to K = 4 ceil(R / 2) reals.
__global__ void k_grad_pack(int N, int R, int K, const double2 *__restrict__ x, double *__restrict__ out) {
    const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int h = K / 2;
    if (q >= (int64_t)N * h) return;
    const int e = (int)(q / h), j = (int)(q % h);
    reinterpret_cast<double2 *>(out)[q] = j < R ? x[(int64_t)j * N + e] : make_double2(0.0, 0.0);
}

// Tile of sum_k of the complex products a_i b_e over the packed rows: re and im parts, v_mfma_f64_16x16x4 (A[i][k]
// in lane i + 16 k, B[k][e] in lane e + 16 k, D[i][e] in lane e + 16 (i % 4), element i / 4). Reals alternate
// (re, im): re = sum +-a[k] b[k], im = sum a[k ^ 1] b[k].
__device__ __forceinline__ void pair_gemm(const double *__restrict__ a, const double *__restrict__ b, int K, int kk,
                                          V4d &re, V4d &im) {
    const double sg = (kk & 1) ? -1.0 : 1.0;
#pragma unroll 2
    for (int k = 0; k < K; k += 4) {
        const double a0 = a[k + kk] * sg, a1 = a[k + (kk ^ 1)], bk = b[k + kk];
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, bk, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, bk, im, 0, 0, 0);
    }
}

// Partial sums over a range of columns for 16 touched elements. Columns are elements (LISTEN false: B; cols: a list of
// them, or null for all) or listeners (LISTEN true: A); grid (row tiles, column splits); out[(split * T + t) * 3 + c].
// xi, li: packed x and lambda by element; pc: the columns' packed values that multiply x_i (lambda by element, or vf by
// listener).
template <bool LISTEN>
__global__ __launch_bounds__(kGT, 3) void k_grad_pairs(
    const Tri *__restrict__ tri, const double *__restrict__ L, const int *__restrict__ cols, int ncol, int T,
    const int *__restrict__ touched, double k, int K, const double *__restrict__ xp, const double *__restrict__ lp,
    const double *__restrict__ pc, int nsplit, double *__restrict__ out) {
    __shared__ GradRow rows[16];
    __shared__ double red[kGW][16][3];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i16 = lane & 15, kk = lane >> 4;
    const int t0 = (int)blockIdx.x * 16, sp = blockIdx.y;
    if (threadIdx.x < 16)  // surplus rows repeat the last, unused
        fill_row(rows[threadIdx.x], tri[touched[min(t0 + (int)threadIdx.x, T - 1)]]);
    const int64_t ei = touched[min(t0 + i16, T - 1)];  // the row whose packed values this lane feeds
    const double *xa = xp + ei * K, *la = LISTEN ? nullptr : lp + ei * K;
    __syncthreads();
    double acc[3] = {0.0, 0.0, 0.0};  // lane i16 = v holds row 4 v + kk
    const int ntile = (ncol + 15) >> 4;
    const int c0 = (int)((int64_t)ntile * sp / nsplit), c1 = (int)((int64_t)ntile * (sp + 1) / nsplit);
    for (int ct = c0 + w; ct < c1; ct += kGW) {
        const int ec = min(ct * 16 + i16, ncol - 1), e = !LISTEN && cols ? cols[ec] : ec;
        const bool on = ct * 16 + i16 < ncol;  // surplus columns repeat the last, not added
        V4d gr = {0, 0, 0, 0}, gi = {0, 0, 0, 0}, hr = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
        pair_gemm(xa, pc + (int64_t)e * K, K, kk, hr, hi);
        Tri te{};
        double px, py, pz;  // the column's collocation point
        if constexpr (LISTEN) {
            px = L[3 * e], py = L[3 * e + 1], pz = L[3 * e + 2];
        } else {
            pair_gemm(la, xp + (int64_t)e * K, K, kk, gr, gi);
            te = tri[e];
            px = te.gx, py = te.gy, pz = te.gz;
        }
#pragma unroll 1
        for (int v = 0; v < 4; v++) {
            const GradRow &r = rows[v * 4 + kk];
            double d = 0.0;
            if constexpr (!LISTEN) {
                // dM_ie/dp_i: rule points on the column's triangle, collocation at the row's centroid
                double2 SF[2], SH[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    SF[h] = SH[h] = make_double2(0.0, 0.0);
#pragma unroll
                    for (int g = 3 * h; g < 3 * h + 3; g++) {
                        double wt, xi, eta;
                        quad_point(g, wt, xi, eta);
                        const double dx = r.gx - (te.ax + xi * te.bx + eta * te.cx);
                        const double dy = r.gy - (te.ay + xi * te.by + eta * te.cy);
                        const double dz = r.gz - (te.az + xi * te.bz + eta * te.cz);
                        double2 F, H;
                        FdF(k, dx, dy, dz, F, H);
                        SF[h] = cadd(SF[h], F);
                        SH[h] = cadd(SH[h], H);
                    }
                }
                const double s = -((r.gx - te.ax) * te.nx + (r.gy - te.ay) * te.ny + (r.gz - te.az) * te.nz);
                const double fa = ARH_QW_A * (kInv8Pi / 3.0), fb = ARH_QW_B * (kInv8Pi / 3.0);
                const double dpx = s * (fa * SH[0].x + fb * SH[1].x) - te.ny * (fa * SF[0].x + fb * SF[1].x);
                const double dpy = s * (fa * SH[0].y + fb * SH[1].y) - te.ny * (fa * SF[0].y + fb * SF[1].y);
                d = dpx * gr[v] - dpy * gi[v];
            }
            // dM_ei/dq_(i,c): rule points on the row's triangle, collocation at the column's point
            double2 S0 = make_double2(0.0, 0.0), T0 = S0, T1 = S0, T2 = S0;
#pragma unroll
            for (int g = 0; g < 6; g++) {
                double wt, xi, eta;
                quad_point(g, wt, xi, eta);
                double2 F, H;
                FdF<LISTEN>(k, px - r.q[g][0], py - r.q[g][1], pz - r.q[g][2], F, H);
                const double w0 = wt * kInv8Pi;
                S0.x = fma(w0, F.x, S0.x), S0.y = fma(w0, F.y, S0.y);
                T0.x = fma(w0 * (1.0 - xi - eta), H.x, T0.x), T0.y = fma(w0 * (1.0 - xi - eta), H.y, T0.y);
                T1.x = fma(w0 * xi, H.x, T1.x), T1.y = fma(w0 * xi, H.y, T1.y);
                T2.x = fma(w0 * eta, H.x, T2.x), T2.y = fma(w0 * eta, H.y, T2.y);
            }
            const double ux = px - r.ax, uy = py - r.ay, uz = pz - r.az;
            const double s = ux * r.nx + uy * r.ny + uz * r.nz;  // -s of the formulas above
            // D_c = (p - a) . dn_c with dn_a = e_y x (b - c), dn_b = e_y x (c - a), dn_c = (b - a) x e_y
            const double E0 = r.ny - (ux * (r.bz - r.cz) - uz * (r.bx - r.cx));
            const double E1 = uz * r.cx - ux * r.cz, E2 = ux * r.bz - uz * r.bx;
            const double h_r = hr[v], h_i = hi[v];
            double o0 = (s * T0.x + E0 * S0.x) * h_r - (s * T0.y + E0 * S0.y) * h_i;
            double o1 = (s * T1.x + E1 * S0.x) * h_r - (s * T1.y + E1 * S0.y) * h_i;
            double o2 = (s * T2.x + E2 * S0.x) * h_r - (s * T2.y + E2 * S0.y) * h_i;
            o0 += d, o1 += d, o2 += d;
            o0 = row_sum(on ? o0 : 0.0), o1 = row_sum(on ? o1 : 0.0), o2 = row_sum(on ? o2 : 0.0);
            if (i16 == v) acc[0] += o0, acc[1] += o1, acc[2] += o2;
        }
    }
    if (i16 < 4)
#pragma unroll
        for (int c = 0; c < 3; c++) red[w][i16 * 4 + kk][c] = acc[c];
    __syncthreads();
    if (threadIdx.x < 48) {
        const int r = (int)threadIdx.x / 3, c = (int)threadIdx.x % 3;
        if (t0 + r < T) {
            double a = red[0][r][c];
            for (int q = 1; q < kGW; q++) a += red[q][r][c];
            out[((int64_t)sp * T + t0 + r) * 3 + c] = a;
        }
    }
}

// Pairs of touched elements, both ways at once. The distances between the collocation point of i and the rule points of
// e serve dM_ie/dp_i (i's centroid moves, times G(i, e)) and dM_ie/dq_(e,c) (e's corners move, times the same G(i, e)),
// so a pair {i, e} takes the twelve distances and the two products once where k_grad_pairs, for i and for e, takes them
// twice. A workgroup takes a pair of blocks of kGB touched elements (grid: block b with block b + d in circular order,
// the offsets d up to half of the blocks, so each pair of blocks once), a wavefront 16 of the second block's elements
// as columns; both blocks' geometry is in LDS. The two directions of a pair come one after the other, each with its own
// product tile: with both tiles in registers at once the kernel spills at 3 wavefronts per SIMD (one rhs 2.4 ms, 37
// 3.4; now 2.15 and 2.9, 159 registers; at 4 wavefronts 2.6 and 3.6). The offsets are those from d0 on, gridDim.y of
// them; out[((2 (d - d0) + s) * T + t) * 3 + c]: the sum of element t, in block b, with the elements of block b + d (s
// = 0) or b - d (s = 1).
constexpr int kGB = 64;
static_assert(kGB == 16 * kGW, "a column tile per wavefront");

// Pair of a collocation point p and a triangle, times g: the y derivative for p's centroid (o[3]) and for the
// triangle's corners (o[0..2]).
__device__ __forceinline__ void pair_side(double k, const GradRow &r, double px, double py, double pz, double g_r,
                                          double g_i, double o[4]) {
    double2 S0 = make_double2(0.0, 0.0), T0 = S0, T1 = S0, T2 = S0;
#pragma unroll
    for (int g = 0; g < 6; g++) {
        double wt, xi, eta;
        quad_point(g, wt, xi, eta);
        double2 F, H;
        FdF(k, px - r.q[g][0], py - r.q[g][1], pz - r.q[g][2], F, H);
        const double w0 = wt * kInv8Pi;
        S0.x = fma(w0, F.x, S0.x), S0.y = fma(w0, F.y, S0.y);
        T0.x = fma(w0 * (1.0 - xi - eta), H.x, T0.x), T0.y = fma(w0 * (1.0 - xi - eta), H.y, T0.y);
        T1.x = fma(w0 * xi, H.x, T1.x), T1.y = fma(w0 * xi, H.y, T1.y);
        T2.x = fma(w0 * eta, H.x, T2.x), T2.y = fma(w0 * eta, H.y, T2.y);
    }
    const double ux = px - r.ax, uy = py - r.ay, uz = pz - r.az;
    const double s = ux * r.nx + uy * r.ny + uz * r.nz;  // -s of the formulas above
    const double E0 = r.ny - (ux * (r.bz - r.cz) - uz * (r.bx - r.cx));
    const double E1 = uz * r.cx - ux * r.cz, E2 = ux * r.bz - uz * r.bx;
    o[0] = (s * T0.x + E0 * S0.x) * g_r - (s * T0.y + E0 * S0.y) * g_i;
    o[1] = (s * T1.x + E1 * S0.x) * g_r - (s * T1.y + E1 * S0.y) * g_i;
    o[2] = (s * T2.x + E2 * S0.x) * g_r - (s * T2.y + E2 * S0.y) * g_i;
    const double cr = s * (T0.x + T1.x + T2.x) + r.ny * S0.x, ci = s * (T0.y + T1.y + T2.y) + r.ny * S0.y;
    o[3] = (ci * g_i - cr * g_r) * (1.0 / 3.0);
}

__global__ __launch_bounds__(kGT, 3) void k_grad_both(const Tri *__restrict__ tri, int T,
                                                      const int *__restrict__ touched, double k, int K,
                                                      const double *__restrict__ xp, const double *__restrict__ lp,
                                                      int d0, double *__restrict__ out) {
    __shared__ GradRow rows[2][kGB];
    __shared__ double red[kGW][kGB][3];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i16 = lane & 15, kk = lane >> 4;
    const int nb = gridDim.x, d = d0 + (int)blockIdx.y, rb = blockIdx.x, cb = (rb + d) % nb;
    if (2 * d == nb && 2 * rb >= nb) return;  // its partner has the pair
    out += (int64_t)blockIdx.y * 6 * T;
    if (threadIdx.x < 2 * kGB) {  // surplus elements repeat the last, not added
        const int b = threadIdx.x / kGB, i = threadIdx.x % kGB;
        fill_row(rows[b][i], tri[touched[min((b ? cb : rb) * kGB + i, T - 1)]]);
    }
    __syncthreads();
    const int u = cb * kGB + w * 16 + i16;
    const bool on = u < T;
    const int64_t e = touched[min(u, T - 1)];
    const GradRow &ce = rows[1][w * 16 + i16];
    double col[3] = {0.0, 0.0, 0.0};
#pragma unroll 1
    for (int rt = 0; rt < kGB / 16; rt++) {
        const int t0 = rb * kGB + rt * 16;
        const int64_t ei = touched[min(t0 + i16, T - 1)];
        double acc[3] = {0.0, 0.0, 0.0};  // lane i16 = v holds row 4 v + kk
#pragma unroll 1
        for (int side = 0; side < 2; side++) {  // the column's triangle with G(i, e), then the row's with G(e, i)
            V4d gr = {0, 0, 0, 0}, gi = {0, 0, 0, 0};
            pair_gemm((side ? xp : lp) + ei * K, (side ? lp : xp) + e * K, K, kk, gr, gi);
#pragma unroll 1
            for (int v = 0; v < 4; v++) {
                const GradRow &r = rows[0][rt * 16 + v * 4 + kk], &t = side ? r : ce, &p = side ? ce : r;
                const bool both = on && t0 + v * 4 + kk < T;
                double a[4];
                pair_side(k, t, p.gx, p.gy, p.gz, gr[v], gi[v], a);
#pragma unroll
                for (int c = 0; c < 4; c++) a[c] = both ? a[c] : 0.0;
                if (side) {
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        const double o = row_sum(a[c]);
                        col[c] += a[3];
                        if (i16 == v) acc[c] += o;
                    }
                } else {
                    const double o = row_sum(a[3]);
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        col[c] += a[c];
                        if (i16 == v) acc[c] += o;
                    }
                }
            }
        }
        if (i16 < 4)
#pragma unroll
            for (int c = 0; c < 3; c++) red[w][rt * 16 + i16 * 4 + kk][c] = acc[c];
    }
    if (cb != rb) {  // a block with itself: every ordered pair has come by as row and column
#pragma unroll
        for (int c = 0; c < 3; c++) {
            col[c] += __shfl_xor(col[c], 16, ARH_WAVE);
            col[c] += __shfl_xor(col[c], 32, ARH_WAVE);
        }
        if (kk == 0 && on)
#pragma unroll
            for (int c = 0; c < 3; c++) out[((int64_t)T + u) * 3 + c] = col[c];
    }
    __syncthreads();
    if (threadIdx.x < 3 * kGB) {
        const int r = (int)threadIdx.x / 3, c = (int)threadIdx.x % 3;
        if (rb * kGB + r < T) {
            double a = red[0][r][c];
            for (int q = 1; q < kGW; q++) a += red[q][r][c];
            out[(rb * kGB + r) * 3 + c] = a;
        }
    }
}

// Sums over the other blocks of a strip of offsets, in order of the offset; added to out from the second strip on. At
// offset 0 a block's sum with itself is in s = 0 alone, at offset nb / 2 a block's sum is in s = 0 for the first half
// of the blocks and in s = 1 for the others; both lie outside the loop, whose loads go out together that way (10 us
// instead of 25 at 8,442 touched elements).
__global__ __launch_bounds__(256) void k_grad_blocks(int n3, int nb, int d0, int nd, const double *__restrict__ part,
                                                     double *__restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n3) return;
    const bool half = 2 * (d0 + nd - 1) == nb;
    double a = d0 > 0 ? out[i] : part[i];
#pragma unroll 4
    for (int q = d0 > 0 ? 0 : 1; q < nd - (half ? 1 : 0); q++) {
        a += part[(int64_t)(2 * q) * n3 + i];
        a += part[(int64_t)(2 * q + 1) * n3 + i];
    }
    if (half) a += part[(int64_t)(2 * (nd - 1) + (2 * (i / (3 * kGB)) < nb ? 0 : 1)) * n3 + i];
    out[i] = a;
}

// C per touched element (one thread each): -sum_rhs Re( lam_i db_i / dp_i ).
__global__ __launch_bounds__(64) void k_grad_C(const Tri *__restrict__ tri, int N, int T,
                                               const int *__restrict__ touched, double k, int R,
                                               const double2 *__restrict__ lam, int src_kind,
                                               const double *__restrict__ src, double *__restrict__ cC) {
    const int t = blockIdx.x * 64 + threadIdx.x;
    if (t >= T) return;
    const int i = touched[t];
    const Tri ti = tri[i];
    double cc = 0.0;
    for (int j = 0; j < R; j++) {
        double2 db;
        const double sx = src[3 * j], sy = src[3 * j + 1], sz = src[3 * j + 2];
        double sn, cs;
        if (src_kind == ARH_RHS_POINT) {
            const double dx = ti.gx - sx, dy = ti.gy - sy, dz = ti.gz - sz;
            const double r = sqrt(dx * dx + dy * dy + dz * dz);
            trig_sincos(k * r, &sn, &cs);
            // e^{-ikr}(-1 - ikr) / (4 pi r^2) * d_y / (3 r)
            const double f = dy / (3.0 * r) / (4.0 * kPi * r * r);
            db = make_double2((-cs - k * r * sn) * f, (sn - k * r * cs) * f);
        } else {
            trig_sincos(k * (sx * ti.gx + sy * ti.gy + sz * ti.gz), &sn, &cs);
            // (i f) e^{-i k d.c} with f = -k d_y / 3
            const double f = -k * sy / 3.0;
            db = make_double2(f * sn, f * cs);
        }
        cc -= cmul(db, lam[(int64_t)j * N + i]).x;
    }
    cC[t] = cc;
}

// gradient_h: sum over (touched element, corner) in list order; A and B summed over their splits first. With G,
// the terms are not stored but added: G_h = G_h + ((A_h - B_h) + C_h), the order of the host sum A - B + C.
__global__ void k_grad_scatter(int HH, int T, int asplit, int bsplit, const int *__restrict__ hptr,
                               const int *__restrict__ hlist, const double *__restrict__ partA,
                               const double *__restrict__ partB, const double *__restrict__ cC,
                               double *__restrict__ A, double *__restrict__ B, double *__restrict__ C,
                               double *__restrict__ G) {
    const int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= HH) return;
    double a = 0.0, b = 0.0, c = 0.0;
    for (int e = hptr[h]; e < hptr[h + 1]; e++) {
        const int tc = hlist[e];  // t * 3 + corner
        double aa = 0.0, bb = 0.0;
        for (int sp = 0; sp < asplit; sp++) aa += partA[(int64_t)sp * T * 3 + tc];
        for (int sp = 0; sp < bsplit; sp++) bb += partB[(int64_t)sp * T * 3 + tc];
        a += aa;
        b += bb;
        c += cC[tc / 3];
    }
    if (G)
        G[h] = G[h] + ((a - b) + c);
    else
        A[h] = a, B[h] = b, C[h] = c;
}

void launch_shape_grad(arh_geom *g, double k, const double *L_dev, int LL, const int *diff, int HH, int nrhs,
                       const double2 *x, const double2 *lam, const double2 *vf, int src_kind, const double *src_dev,
                       double *A, double *B, double *C, double *G) {
    hipStream_t s = g->ctx->stream;
    const int N = g->N, V = g->V;
    // slots of differentiable vertices; touched elements; per-h (element, corner) lists
    std::vector<int> slot(V, -1);
    for (int h = 0; h < HH; h++) {
        ARH_CHECK(diff[h] >= 0 && diff[h] < V, ARH_EINVAL, "diff vertex id out of range");
        slot[diff[h]] = h;  // a repeated id keeps its last slot, as the reference's map assignment does
    }
    const std::vector<int> &Eh = g->hE;
    std::vector<int> touched, others, tpos(N, -1), hptr(HH + 1, 0);
    for (int e = 0; e < N; e++) {
        bool any = false;
        for (int c = 0; c < 3; c++) {
            const int h = slot[Eh[3 * e + c]];
            if (h >= 0) any = true, hptr[h + 1]++;
        }
        if (any)
            tpos[e] = (int)touched.size(), touched.push_back(e);
        else
            others.push_back(e);
    }
    const int T = (int)touched.size();
    for (int h = 0; h < HH; h++) hptr[h + 1] += hptr[h];
    std::vector<int> hlist(hptr[HH]), fill(hptr.begin(), hptr.end() - 1);
    for (int e : touched)
        for (int c = 0; c < 3; c++) {
            const int h = slot[Eh[3 * e + c]];
            if (h >= 0) hlist[fill[h]++] = tpos[e] * 3 + c;
        }
    if (T == 0 && G) return;  // nothing to add
    if (T == 0) {
        ARH_HIP(hipMemsetAsync(A, 0, sizeof(double) * HH, s));
        ARH_HIP(hipMemsetAsync(B, 0, sizeof(double) * HH, s));
        ARH_HIP(hipMemsetAsync(C, 0, sizeof(double) * HH, s));
        ARH_HIP(hipStreamSynchronize(s));
        return;
    }
    const int gx = (T + 15) / 16;
    // column splits: enough workgroups to fill the chip, at least one 16-column tile per wavefront of each
    auto splits = [&](int ncol) {
        const int most = std::max(1, (ncol + 16 * kGW - 1) / (16 * kGW));
        return std::max(1, std::min(most, (kGSlots + gx - 1) / gx));
    };
    // enough blocks of touched elements to fill the chip: their pairs both ways at once, then the other columns
    const int nb = (T + kGB - 1) / kGB;
    const bool both = nb >= kGMinBlocks;
    const int ncol = both ? (int)others.size() : N;
    const int bsplit = ncol ? splits(ncol) : 0, asplit = splits(LL), first = both ? 1 : 0;  // first: the blocks' sum
    const int K = 4 * ((nrhs + 1) / 2);
    DBuf d_touched, d_others, d_hptr, d_hlist, pA, pB, pS, cC, xp, lp, vp;
    upload(d_touched, touched, s);
    upload(d_hptr, hptr, s);
    upload(d_hlist, hlist, s);
    pA.alloc(sizeof(double) * 3 * (size_t)T * asplit);
    pB.alloc(sizeof(double) * 3 * (size_t)T * (first + bsplit));
    cC.alloc(sizeof(double) * T);
    auto pack = [&](DBuf &out, int n, const double2 *v) {
        out.alloc(sizeof(double) * (size_t)n * K);
        hipLaunchKernelGGL(k_grad_pack, dim3((unsigned)(((int64_t)n * (K / 2) + 255) / 256)), dim3(256), 0, s, n, nrhs,
                           K, v, out.as<double>());
    };
    pack(xp, N, x);
    pack(lp, N, lam);
    pack(vp, LL, vf);
    if (both) {
        upload(d_others, others, s);
        const int no = nb / 2 + 1;  // offsets, in equal strips
        const int64_t per = 2 * 3 * (int64_t)sizeof(double) * T, most = std::max<int64_t>(1, kGPartBytes / per);
        const int strips = (int)((no + most - 1) / most), len = (no + strips - 1) / strips;
        pS.alloc((size_t)per * len);
        for (int d0 = 0; d0 < no; d0 += len) {
            const int nd = std::min(len, no - d0);
            hipLaunchKernelGGL(k_grad_both, dim3(nb, nd), dim3(kGT), 0, s, g->tri.as<Tri>(), T, d_touched.as<int>(), k,
                               K, xp.as<double>(), lp.as<double>(), d0, pS.as<double>());
            hipLaunchKernelGGL(k_grad_blocks, dim3((3 * T + 255) / 256), dim3(256), 0, s, 3 * T, nb, d0, nd,
                               pS.as<double>(), pB.as<double>());
        }
    }
    if (bsplit)
        hipLaunchKernelGGL(k_grad_pairs<false>, dim3(gx, bsplit), dim3(kGT), 0, s, g->tri.as<Tri>(),
                           (const double *)nullptr, both ? d_others.as<int>() : nullptr, ncol, T, d_touched.as<int>(),
                           k, K, xp.as<double>(), lp.as<double>(), lp.as<double>(), bsplit,
                           pB.as<double>() + first * 3 * (size_t)T);
    hipLaunchKernelGGL(k_grad_pairs<true>, dim3(gx, asplit), dim3(kGT), 0, s, g->tri.as<Tri>(), L_dev,
                       (const int *)nullptr, LL, T, d_touched.as<int>(), k, K, xp.as<double>(),
                       (const double *)nullptr, vp.as<double>(), asplit, pA.as<double>());
    hipLaunchKernelGGL(k_grad_C, dim3((T + 63) / 64), dim3(64), 0, s, g->tri.as<Tri>(), N, T, d_touched.as<int>(), k,
                       nrhs, lam, src_kind, src_dev, cC.as<double>());
    hipLaunchKernelGGL(k_grad_scatter, dim3((HH + 255) / 256), dim3(256), 0, s, HH, T, asplit, first + bsplit,
                       d_hptr.as<int>(), d_hlist.as<int>(), pA.as<double>(), pB.as<double>(), cC.as<double>(), A, B, C,
                       G);
    ARH_HIP(hipGetLastError());
    ARH_HIP(hipStreamSynchronize(s));
}

}  // namespace arh
