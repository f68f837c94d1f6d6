// Right-hand sides, the receiver (listener) matrix product and the diffusion coefficient.
#include <algorithm>
#include <mutex>
#include <string>
#include <type_traits>

#include "arh_internal.h"
#include "device_common.h"

namespace arh {

// b_j,i: point source e^{-ikr}/(4 pi r), r = |c_i - s_j| (helpers.cpp:46-50), or plane wave
// e^{-ik d_j . c_i} (sphere.h:22-26).
__global__ void k_rhs(const Tri *__restrict__ tri, int N, double k, int kind, const double *__restrict__ vecs,
                      double2 *__restrict__ b) {
    const int j = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const Tri t = tri[i];
    const double vx = vecs[3 * j], vy = vecs[3 * j + 1], vz = vecs[3 * j + 2];
    double2 out;
    if (kind == ARH_RHS_POINT) {
        double dx = t.gx - vx, dy = t.gy - vy, dz = t.gz - vz;
        double r = sqrt(dx * dx + dy * dy + dz * dz);
        double sn, cs;
        trig_sincos(k * r, &sn, &cs);
        double f = 1.0 / (4.0 * kPi * r);
        out = make_double2(cs * f, -sn * f);
    } else {
        double ph = k * (vx * t.gx + vy * t.gy + vz * t.gz);
        double sn, cs;
        trig_sincos(ph, &sn, &cs);
        out = make_double2(cs, -sn);
    }
    b[(int64_t)j * N + i] = out;
}

void launch_rhs(arh_geom *g, double k, int kind, int nrhs, const double *vecs_dev, double2 *b) {
    hipLaunchKernelGGL(k_rhs, dim3((g->N + 255) / 256, nrhs), dim3(256), 0, g->ctx->stream, g->tri.as<Tri>(), g->N, k,
                       kind, vecs_dev, b);
    ARH_HIP(hipGetLastError());
}

// ---------------------------------------------------------------- receiver products
// Q_l,i = M(L_l, element i) (integrate.cpp:46-57) times a batch of vectors, without storing Q: a wavefront evaluates
// a 16 x 4 tile of entries, one per lane in the A layout of v_mfma_f64_16x16x4, and multiplies it at once by up to
// 40 right-hand sides. A complex product is a real one with the rhs as interleaved (re, im) columns: output column
// n = 2 j + s is part s of rhs j, the lane holds that part of x and takes the other from its neighbour. A right-hand
// side's result does not depend on the batch (columns are independent, the split of the sum is fixed by LL and N).
//
// Bound by the entries' FP64 VALU work, about 590 operations for 64 entries against 2 MFMAs per 8 right-hand sides.
// 181 receivers, N = 9,828, 37 right-hand sides: 55 us and 57 us transposed (41 and 44 us for one); storing Q
// (40 us) and multiplying by it with vector FMAs took 355 and 57 us more.
constexpr int kRW = 4;            // wavefronts per workgroup
constexpr int kRT = kRW * ARH_WAVE;
constexpr int kRMax = 40;         // right-hand sides per pass
constexpr int kRSlots = 768;      // workgroups aimed for in the forward product (384: 111, 768: 100, 1536: 104 us a call)

typedef double V4d __attribute__((ext_vector_type(4)));

// The value of lane l ^ 1 (DPP quad permutation [1, 0, 3, 2]; every lane of the wavefront is active).
__device__ __forceinline__ double neighbour(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// acc += (entries q, one per lane) times rows `at` of the R vectors x (length len each): column n of tile nt. A lane
// that is not `on` takes a zero: its entry is one too, and its row may hold an infinity.
template <int NT>
__device__ __forceinline__ void recv_mma(V4d (&acc)[NT], double2 q, const double2 *__restrict__ x, int64_t len, int at,
                                         bool on, int R, int n16) {
    const double *xd = reinterpret_cast<const double *>(x);
    const int s = n16 & 1;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int j = min(nt * 8 + (n16 >> 1), R - 1);  // surplus columns repeat the last, not written
        const double xv = xd[(j * len + at) * 2 + s], v = on ? xv : 0.0;
        const double w = neighbour(v);
        acc[nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(q.x, v, acc[nt], 0, 0, 0);
        acc[nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(q.y, s ? w : -w, acc[nt], 0, 0, 0);
    }
}

// The wavefronts' 16 x 16 NT tiles summed in order into red[0] (D[i][n]: lane n + 16 (i % 4), element i / 4).
template <int NT>
__device__ __forceinline__ void recv_reduce(const V4d (&acc)[NT], double (*red)[16][16 * NT], int w, int lane) {
    const int n16 = lane & 15, kk = lane >> 4;
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int v = 0; v < 4; v++) red[w][v * 4 + kk][nt * 16 + n16] = acc[nt][v];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * 16 * NT; e += kRT) {
        double *p = &red[0][0][0] + e;
        double t = p[0];
#pragma unroll
        for (int q = 1; q < kRW; q++) t += p[q * 16 * 16 * NT];
        p[0] = t;
    }
    __syncthreads();
}

// part[(split * tiles + tile) * 16 + l][n]: sums over a split of the elements; grid (16-receiver tiles, splits).
template <int NT>
__global__ __launch_bounds__(kRT) void k_recv(const Tri *__restrict__ tri, int N, double k, const double *__restrict__ L,
                                              int LL, int R, const double2 *__restrict__ x, int nsplit,
                                              double *__restrict__ part) {
    __shared__ double red[kRW][16][16 * NT];
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE;
    const int n16 = lane & 15, kk = lane >> 4;
    const int l = min((int)blockIdx.x * 16 + n16, LL - 1);
    const double px = L[3 * l], py = L[3 * l + 1], pz = L[3 * l + 2];
    V4d acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[nt] = V4d{0, 0, 0, 0};
    const int ng = (N + 3) >> 2, sp = blockIdx.y;
    const int g0 = (int)((int64_t)ng * sp / nsplit), g1 = (int)((int64_t)ng * (sp + 1) / nsplit);
    auto step = [&](int g, auto whole) {
        const int e = 4 * g + kk, ec = min(e, N - 1);
        const bool on = whole() || e < N;
        double2 q = bem_entry(k, px, py, pz, tri[ec]);
        if (!on) q = make_double2(0.0, 0.0);
        recv_mma<NT>(acc, q, x, N, ec, on, R, n16);
    };
    int g = g0 + w;
    for (; g < min(g1, N >> 2); g += kRW) step(g, std::true_type{});
    if (g < g1) step(g, std::false_type{});
    recv_reduce<NT>(acc, red, w, lane);
    double *o = part + ((int64_t)sp * gridDim.x + blockIdx.x) * 16 * 16 * NT;
    for (int e = threadIdx.x; e < 16 * 16 * NT; e += kRT) o[e] = (&red[0][0][0])[e];
}

// y[j, l] = the splits' sums in order
__global__ __launch_bounds__(256) void k_recv_sum(int LL, int R, int tiles, int W, int nsplit,
                                                  const double *__restrict__ part, double2 *__restrict__ y) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    const int l = e / (2 * R), n = e - l * 2 * R;
    if (l >= LL) return;
    const double *p = part + (int64_t)l * W + n;
    double s = 0.0;
#pragma unroll 8
    for (int q = 0; q < nsplit; q++) s += p[(int64_t)q * tiles * 16 * W];
    reinterpret_cast<double *>(y)[((int64_t)(n >> 1) * LL + l) * 2 + (n & 1)] = s;
}

// y[j, i] = sum_l Q[l, i] x[j, l] (the adjoint right-hand side Q^T vf, adjoint.cpp:198): 16 elements per workgroup, its
// wavefronts take every kRW-th group of four receivers.
template <int NT>
__global__ __launch_bounds__(kRT) void k_recv_t(const Tri *__restrict__ tri, int N, double k,
                                                const double *__restrict__ L, int LL, int R,
                                                const double2 *__restrict__ x, double2 *__restrict__ y) {
    __shared__ double red[kRW][16][16 * NT];
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE;
    const int n16 = lane & 15, kk = lane >> 4;
    const int i0 = (int)blockIdx.x * 16;
    const Tri t = tri[min(i0 + n16, N - 1)];
    V4d acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[nt] = V4d{0, 0, 0, 0};
    const int ng = (LL + 3) >> 2;
    auto step = [&](int g, auto whole) {
        const int l = 4 * g + kk, lc = min(l, LL - 1);
        const bool on = whole() || l < LL;
        double2 q = bem_entry(k, L[3 * lc], L[3 * lc + 1], L[3 * lc + 2], t);
        if (!on) q = make_double2(0.0, 0.0);
        recv_mma<NT>(acc, q, x, LL, lc, on, R, n16);
    };
    int g = w;
    for (; g < LL >> 2; g += kRW) step(g, std::true_type{});
    if (g < ng) step(g, std::false_type{});
    recv_reduce<NT>(acc, red, w, lane);
    const int m = min(16, N - i0);
    for (int e = threadIdx.x; e < R * 2 * m; e += kRT) {
        const int j = e / (2 * m), r = e - j * 2 * m;
        reinterpret_cast<double *>(y)[((int64_t)j * N + i0) * 2 + r] = red[0][r >> 1][2 * j + (r & 1)];
    }
}

// The kernels' width for a pass of R right-hand sides.
template <class F>
static void with_nt(int R, F &&f) {
    switch ((R + 7) / 8) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    default: f(std::integral_constant<int, 5>{}); break;
    }
}

static void launch_recv_t(arh_geom *g, double k, const double *L_dev, int LL, int nrhs, const double2 *x, double2 *y) {
    hipStream_t s = g->ctx->stream;
    const int N = g->N;
    for (int j0 = 0; j0 < nrhs; j0 += kRMax) {
        const int R = std::min(kRMax, nrhs - j0);
        with_nt(R, [&](auto nt) {
            hipLaunchKernelGGL(k_recv_t<nt()>, dim3((N + 15) / 16), dim3(kRT), 0, s, g->tri.as<Tri>(), N, k, L_dev, LL,
                               R, x + (int64_t)j0 * LL, y + (int64_t)j0 * N);
        });
    }
    ARH_HIP(hipGetLastError());
}

void launch_receivers(arh_geom *g, double k, const double *L_dev, int LL, int transpose, int nrhs, const double2 *x,
                      double2 *y) {
    hipStream_t s = g->ctx->stream;
    const int N = g->N;
    if (transpose) {
        launch_recv_t(g, k, L_dev, LL, nrhs, x, y);
    } else {
        const int tiles = (LL + 15) / 16;
        // splits of the element sum: at least two groups of four per wavefront
        const int nsplit = std::max(1, std::min((kRSlots + tiles - 1) / tiles, (N + 8 * kRW - 1) / (8 * kRW)));
        DBuf part;
        for (int j0 = 0; j0 < nrhs; j0 += kRMax) {
            const int R = std::min(kRMax, nrhs - j0), W = 16 * ((R + 7) / 8);
            part.alloc(sizeof(double) * (size_t)nsplit * tiles * 16 * W);
            with_nt(R, [&](auto nt) {
                hipLaunchKernelGGL(k_recv<nt()>, dim3(tiles, nsplit), dim3(kRT), 0, s, g->tri.as<Tri>(), N, k, L_dev,
                                   LL, R, x + (int64_t)j0 * N, nsplit, part.as<double>());
            });
            hipLaunchKernelGGL(k_recv_sum, dim3((unsigned)(((int64_t)LL * 2 * R + 255) / 256)), dim3(256), 0, s, LL, R,
                               tiles, W, nsplit, part.as<double>(), y + (int64_t)j0 * LL);
        }
    }
    ARH_HIP(hipGetLastError());
    ARH_HIP(hipStreamSynchronize(s));
}

// ---------------------------------------------------------------- receivers without allocation
// arh_receivers_noalloc keeps the receiver coordinates in this file-scope device array (one copy
// per GPU, held until the process ends) and evaluates the receiver-matrix entries on the fly, so it
// needs no device memory beyond its inputs and outputs. Every call on a GPU shares that GPU's
// array: calls that overlap on one GPU (other streams, other threads) race.
static __device__ __align__(256) double scratch[3 * kNoAllocMaxReceivers];

namespace {
std::mutex scratch_mu;
double *scratch_ptr[kNoAllocMaxDevices] = {};
}  // namespace

// The device address of this GPU's copy of scratch (the array's name is only a host-side stand-in);
// looked up once per device, with that device current.
static double *scratch_on(int device) {
    ARH_CHECK(device >= 0 && device < kNoAllocMaxDevices, ARH_EINVAL, "device ordinal out of range");
    std::lock_guard<std::mutex> lk(scratch_mu);
    if (!scratch_ptr[device]) {
        void *p = nullptr;
        ARH_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        ARH_CHECK(p != nullptr, ARH_EHIP, "hipGetSymbolAddress returned no address for the receiver scratch");
        scratch_ptr[device] = static_cast<double *>(p);
    }
    return scratch_ptr[device];
}

// y[j, l] = sum_i Q[l, i] x[j, i]; one workgroup per receiver, entries evaluated on the fly, rhs in chunks of kRC.
// (k_recv needs room for its splits' sums; without them it would be 12 workgroups for 181 receivers.)
constexpr int kRC = 8;
__global__ __launch_bounds__(kRT) void k_qx(const Tri *__restrict__ tri, double k, const double *__restrict__ L, int N,
                                            int LL, int R, const double2 *__restrict__ x, double2 *__restrict__ y) {
    __shared__ double2 sh[kRT / ARH_WAVE][kRC];
    const int l = blockIdx.x;
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE;
    for (int j0 = 0; j0 < R; j0 += kRC) {
        double2 acc[kRC];
#pragma unroll
        for (int c = 0; c < kRC; c++) acc[c] = make_double2(0.0, 0.0);
        for (int i = threadIdx.x; i < N; i += kRT) {
            double2 a = bem_entry(k, L[3 * l], L[3 * l + 1], L[3 * l + 2], tri[i]);
#pragma unroll
            for (int c = 0; c < kRC; c++)
                if (j0 + c < R) cfma(acc[c], a, x[(int64_t)(j0 + c) * N + i]);
        }
#pragma unroll
        for (int c = 0; c < kRC; c++) acc[c] = wave_sum2(acc[c]);
        __syncthreads();
        if (lane == 0)
#pragma unroll
            for (int c = 0; c < kRC; c++) sh[w][c] = acc[c];
        __syncthreads();
        if (threadIdx.x < kRC && j0 + threadIdx.x < R) {
            double2 s = sh[0][threadIdx.x];
            for (int ww = 1; ww < kRT / ARH_WAVE; ww++) s = cadd(s, sh[ww][threadIdx.x]);
            y[(int64_t)(j0 + threadIdx.x) * LL + l] = s;
        }
    }
}

void launch_receivers_noalloc(arh_geom *g, double k, const double *L_host, int LL, int transpose, int nrhs,
                              const double2 *x, double2 *y) {
    ARH_CHECK(LL <= kNoAllocMaxReceivers, ARH_EINVAL,
              "arh_receivers_noalloc takes at most " + std::to_string(kNoAllocMaxReceivers) + " receivers, got " +
                  std::to_string(LL));
    arh_ctx *ctx = g->ctx;
    hipStream_t s = ctx->stream;
    double *Ld = scratch_on(ctx->device);
    // stream-ordered after earlier work on this stream that may still read the previous coordinates
    ARH_HIP(hipMemcpyAsync(Ld, L_host, sizeof(double) * 3 * (size_t)LL, hipMemcpyHostToDevice, s));
    if (transpose) {
        launch_recv_t(g, k, Ld, LL, nrhs, x, y);
        return;
    }
    hipLaunchKernelGGL(k_qx, dim3(LL), dim3(kRT), 0, s, g->tri.as<Tri>(), k, Ld, g->N, LL, nrhs, x, y);
    ARH_HIP(hipGetLastError());
}

// Diffusion coefficient per rhs with n_freqs = 1 (adjoint.cpp:112-127, 145, 388-397).
__global__ __launch_bounds__(256) void k_diffusion(int LL, const double2 *__restrict__ y, double *__restrict__ d,
                                                   double *__restrict__ u, double2 *__restrict__ vf) {
    __shared__ double sh[2][4];
    const int j = blockIdx.x;
    const double2 *yj = y + (int64_t)j * LL;
    double s = 0.0, q = 0.0;
    for (int l = threadIdx.x; l < LL; l += 256) {
        double a = cabs_(yj[l]);
        double L = a * a;
        s += L;
        q += L * L;
    }
    s = wave_sum(s);
    q = wave_sum(q);
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE;
    __shared__ double part[2][4];
    if (lane == 0) part[0][w] = s, part[1][w] = q;
    __syncthreads();
    const double S = part[0][0] + part[0][1] + part[0][2] + part[0][3];
    const double Qs = part[1][0] + part[1][1] + part[1][2] + part[1][3];
    (void)sh;
    if (threadIdx.x == 0) d[j] = (S * S - Qs) / ((LL - 1) * Qs);
    for (int l = threadIdx.x; l < LL; l += 256) {
        double2 yl = yj[l];
        double a = cabs_(yl);
        double L = a * a;
        double ul = 4.0 * (S * Qs - L * S * S) / ((LL - 1) * Qs * Qs) * a;
        if (u) u[(int64_t)j * LL + l] = ul;
        if (vf) vf[(int64_t)j * LL + l] = make_double2(ul * yl.x / a, -ul * yl.y / a);
    }
}

__global__ void k_scale(double2 *__restrict__ a, int64_t n, double f) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        a[i] = make_double2(f * a[i].x, f * a[i].y);
}

__global__ void k_add(const double *__restrict__ x, double *__restrict__ y, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = y[i] + x[i];
}

void launch_add(hipStream_t s, const double *x, double *y, int64_t n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_add, dim3((unsigned)std::min<int64_t>(1024, (n + 255) / 256)), dim3(256), 0, s, x, y, n);
    ARH_HIP(hipGetLastError());
}

void launch_scale(hipStream_t s, double2 *a, int64_t n, double f) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_scale, dim3((unsigned)std::min<int64_t>(1024, (n + 255) / 256)), dim3(256), 0, s, a, n, f);
    ARH_HIP(hipGetLastError());
}

void launch_diffusion(hipStream_t s, int LL, int nrhs, const double2 *y, double *d, double *u, double2 *vf) {
    hipLaunchKernelGGL(k_diffusion, dim3(nrhs), dim3(256), 0, s, LL, y, d, u, vf);
    ARH_HIP(hipGetLastError());
}

}  // namespace arh
