// Multi-rhs complex H-matrix product on gfx950 MFMA: v_mfma_f32_16x16x4_f32 on the FP32 copy of
// the operator (mixed precision) and v_mfma_f64_16x16x4_f64 on an FP64 copy (FP64 true residuals
// and FP64 multi-rhs solves), one templated engine.
//
// A complex product Y = A X is one real product with A read as interleaved (re, im) columns:
//   Y' = A' X',  A'[:, 2c] = Re A[:, c], A'[:, 2c+1] = Im A[:, c],
//   X'[2c, 2j] = Re X[c, j], X'[2c, 2j+1] = Im X[c, j], X'[2c+1, 2j] = -Im X[c, j], X'[2c+1, 2j+1] = Re X[c, j],
// so Y'[:, 2j] = Re Y[:, j] and Y'[:, 2j+1] = Im Y[:, j]. Each lane loads one complex A entry for
// 4 consecutive complex columns (the K = 4 of the instruction) and feeds the real part to one MFMA
// (with the Re rows of X') and the imaginary part to a second (with the Im rows). The output
// columns 0..2R-1 are the interleaved re/im parts of the R right-hand sides, padded to NT tiles of 16.
//
// The operator copy has its own layout, built once per assembly (per precision):
//  * V stacks: the V factors of all low-rank blocks sharing a column cluster, stacked row-wise and
//    stored column-major, so phase 1 (t = V x) runs on full 16-row tiles even when ranks are small
//    and reads each x row once per stack instead of once per block;
//  * fused row-leaf panels: per row leaf, its dense columns followed by the U columns of every
//    low-rank block covering it (zero-padded to a multiple of 4 columns), with one source row per
//    column into the packed [x; t] buffer, so phase 2 (y = D x + U t) is one uniform column sweep.
// The rhs block and the intermediates share one row-major buffer xt (row i: row_width(R) complex
// values).
//
// Work is cut into "groups" of 4 consecutive columns. Each wavefront loads the next stage of groups
// (A entries + xt rows) before multiplying the current one, which hides the memory latency
// behind the MFMAs. Accumulation in the operator's precision; y = -x/2 + A x is formed in FP64.
//
// Lane layouts (64 lanes, 16x16x4): A[i][k] in lane i + 16 k, B[k][j] in lane j + 16 k; D[i][j] in
// lane j + 16 (i / 4), element i % 4 for f32, lane j + 16 (i % 4), element i / 4 for f64.
#include <algorithm>
#include <memory>
#include <type_traits>
#include <unordered_map>

#include "arh_internal.h"
#include "device_common.h"
#include "lr_units.h"

namespace arh {

template <class T>
struct Mfma;
template <>
struct Mfma<float> {
    typedef float2 T2;
    typedef float V4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V4 mma(float a, float b, V4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __host__ __device__ __forceinline__ T2 make(double x, double y) { return make_float2((float)x, (float)y); }
    // row (within the 16-row tile) of accumulator element v of lane group kk = lane / 16
    static __device__ __forceinline__ int row(int kk, int v) { return kk * 4 + v; }
};
template <>
struct Mfma<double> {
    typedef double2 T2;
    typedef double V4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V4 mma(double a, double b, V4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __host__ __device__ __forceinline__ T2 make(double x, double y) { return make_double2(x, y); }
    static __device__ __forceinline__ int row(int kk, int v) { return v * 4 + kk; }
};

#ifndef ARH_MV_DEPTH32
#define ARH_MV_DEPTH32 2
#endif
#ifndef ARH_MV_DEPTH64
#define ARH_MV_DEPTH64 2
#endif
#ifndef ARH_MV_RDEPTH32
#define ARH_MV_RDEPTH32 3
#endif
#ifndef ARH_MV_RDEPTH64
#define ARH_MV_RDEPTH64 2
#endif
#ifndef ARH_MV_WAVES
#define ARH_MV_WAVES 8
#endif
#ifndef ARH_MV_RWAVES
#define ARH_MV_RWAVES 4
#endif
#ifndef ARH_MV_CHUNKED
#define ARH_MV_CHUNKED 1
#endif
#ifndef ARH_MV_XCD
#define ARH_MV_XCD 1
#endif
#ifndef ARH_MV_SLOTS
#define ARH_MV_SLOTS 2048
#endif
// Groups per pipeline stage of a wavefront, for the V-stack (lr) and the row-task kernels (FP64 groups hold
// twice the registers).
template <class T>
constexpr int lr_depth() {
    return sizeof(T) == 4 ? ARH_MV_DEPTH32 : ARH_MV_DEPTH64;
}
template <class T>
constexpr int row_depth() {
    return sizeof(T) == 4 ? ARH_MV_RDEPTH32 : ARH_MV_RDEPTH64;
}
// Wavefronts per workgroup (powers of 2). Row tasks take 4: a workgroup then holds one wavefront per SIMD,
// so the register budget, not the workgroup size, sets how many fit a compute unit.
constexpr int kLrWaves = ARH_MV_WAVES;    // V-stack units (big stacks: the whole workgroup)
constexpr int kRowWaves = ARH_MV_RWAVES;  // row tasks
constexpr bool kChunked = ARH_MV_CHUNKED;  // a workgroup's waves take contiguous group ranges (else strided)
constexpr bool kXcdOrder = ARH_MV_XCD;     // row tasks ordered for the per-die L2s
constexpr int kXcds = 8;                   // dies (XCDs) of an MI355X, each with its own L2
#ifndef ARH_MV_BIGCOLS
#define ARH_MV_BIGCOLS 256
#endif
constexpr int kBigCols = ARH_MV_BIGCOLS;  // stacks with at least this many columns get a whole workgroup per unit
constexpr int kPartRows = 64;     // rows of a partial tile for leaves of up to 64 elements
constexpr int kMaxLeaf = 128;     // the largest leaf the engine takes (8 row tiles; partial tiles of 128 rows)
constexpr int kTaskSlots = ARH_MV_SLOTS;  // row tasks aimed for: a few per compute unit
constexpr int kMaxRC = 40;        // right-hand sides per pass (RP <= 40)

// Right-hand side j of a pass is column cols[j0 + j] of x / y (j0 + j without a list).
__device__ __forceinline__ int64_t col_of(const int *cols, int j0, int j) { return cols ? cols[j0 + j] : j0 + j; }

// A pass is skipped when the gate (the solver's count of active right-hand sides) is 0.
__device__ __forceinline__ bool gated(const int *gate) { return gate && *gate == 0; }

// xt[i * RW + j] = x[col j][i] for j < R, 0 for R <= j < RW (rows i < N)
template <class T>
__global__ void k_pack_xf(const double2 *__restrict__ x, int N, int R, int RW, typename Mfma<T>::T2 *__restrict__ xf,
                          const int *__restrict__ cols, int j0, const int *__restrict__ gate) {
    if (gated(gate)) return;
    const int64_t total = (int64_t)N * RW;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e / RW), j = (int)(e % RW);
        double2 d = make_double2(0.0, 0.0);
        if (j < R) d = x[col_of(cols, j0, j) * N + i];
        xf[e] = Mfma<T>::make(d.x, d.y);
    }
}

// The value of lane l ^ 1 (DPP quad permutation [1, 0, 3, 2]; every lane of the wavefront is active).
__device__ __forceinline__ float pair_swap(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false));
}
__device__ __forceinline__ double pair_swap(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// The B operands of output column n = 16 nt + i16 (rhs n / 2, part s = n % 2) from the one real
// value the lane holds, xb = component s of that rhs's xt entry (the lane pair n, n ^ 1 holds its
// real and imaginary parts): br = xb, bi = the partner's value, negated on the real-part lane.
template <class T>
__device__ __forceinline__ void b_pair(T xb, int s, T &br, T &bi) {
    const T nb = pair_swap(xb);
    br = xb;
    bi = s ? nb : -nb;
}

// A group in registers: A entries of NRT 16-row tiles, one real rhs value per output tile.
template <class T, int NT, int NRT>
struct Grp {
    typename Mfma<T>::T2 a[NRT];
    T xb[NT];
    T okf;  // 0 for a padding column (masked groups only)
};

template <class T, int NT, int NRT>
using Acc = typename Mfma<T>::V4[NRT][NT];

// acc += group: all real-part products first, then all imaginary-part products, so consecutive
// MFMAs never write the same accumulator.
template <class T, int NT, int NRT, bool MASK>
__device__ __forceinline__ void grp_mma(Acc<T, NT, NRT> &acc, const Grp<T, NT, NRT> &g, int s) {
    T br[NT], bi[NT], ar[NRT], ai[NRT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) b_pair(g.xb[nt], s, br[nt], bi[nt]);
#pragma unroll
    for (int rt = 0; rt < NRT; rt++) {
        ar[rt] = MASK ? g.a[rt].x * g.okf : g.a[rt].x;
        ai[rt] = MASK ? g.a[rt].y * g.okf : g.a[rt].y;
    }
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int rt = 0; rt < NRT; rt++) acc[rt][nt] = Mfma<T>::mma(ar[rt], br[nt], acc[rt][nt]);
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int rt = 0; rt < NRT; rt++) acc[rt][nt] = Mfma<T>::mma(ai[rt], bi[nt], acc[rt][nt]);
}

// Load one column of a group: A column at acol (rows past amax clamped: their outputs are dropped), xt row
// at brow (real values: the lane's output column is brow[16 nt]). No load is conditional, and nothing waits
// on a load before the group is consumed (a padding mask is applied then).
template <class T, int NT, int NRT>
__device__ __forceinline__ void grp_load(Grp<T, NT, NRT> &g, T okf, const typename Mfma<T>::T2 *acol, int amax,
                                         int i16, const T *brow) {
    g.okf = okf;
#pragma unroll
    for (int rt = 0; rt < NRT; rt++) g.a[rt] = acol[min(rt * 16 + i16, amax)];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) g.xb[nt] = brow[nt * 16];
}

// Packed rows hold row_width(R) complex values: R up to kNarrow, so that one right-hand side does not move eight values a
// row through the caches (FP64, one rhs, 2000 Hz: V stacks 42 -> 37 us, rows 60 -> 55 us), else R rounded up to whole
// tiles (rows of 37 values are not aligned: stacks 60 -> 62.5 us, 0.9 m relief 444 -> 477 us).
constexpr int kNarrow = 4;
__host__ __device__ constexpr int row_width(int R) { return R <= kNarrow ? R : (R + 7) / 8 * 8; }

// Column of a packed row that a lane reads for its tiles: lanes past the last rhs of a narrow row read that one again
// (their outputs are dropped).
template <bool NARROW>
__device__ __forceinline__ int lane_col(int i16, int R) {
    return NARROW ? 2 * min(i16 >> 1, R - 1) + (i16 & 1) : i16;
}

// Component kk (0..3) of v as bit selects (lane-dependent kk: no branches, no exec-mask changes).
__device__ __forceinline__ int pick4(const int4 &v, int kk) {
    const int m1 = -(kk & 1), m2 = -((kk >> 1) & 1);
    const int lo = (v.y & m1) | (v.x & ~m1), hi = (v.w & m1) | (v.z & ~m1);
    return (hi & m2) | (lo & ~m2);
}

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

template <class T, int NT, int NRT>
__device__ __forceinline__ void zero_acc(Acc<T, NT, NRT> &acc) {
#pragma unroll
    for (int rt = 0; rt < NRT; rt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[rt][nt][v] = T(0);
}

// An empty use of a group's registers. Placed on the loop's exit path it makes the loaded values live
// there too, so the compiler cannot sink a stage's loads past the loop's branches to just before the
// products that read them (which would leave no load in flight while a wavefront multiplies).
template <class T, int NT, int NRT>
__device__ __forceinline__ void keep(const Grp<T, NT, NRT> &g) {
#pragma unroll
    for (int rt = 0; rt < NRT; rt++) asm volatile("" ::"v"(g.a[rt].x), "v"(g.a[rt].y));
#pragma unroll
    for (int nt = 0; nt < NT; nt++) asm volatile("" ::"v"(g.xb[nt]));
}

// Groups q0, q0 + qstride, ... < qend, kDepth at a time, double-buffered as two register sets that
// swap roles every stage (stage A multiplies set a while set b loads, stage B the other way round), so
// no register copy has to wait for a load: the only wait is for the set about to be multiplied, one
// stage after its loads were issued. A group's uniform metadata (pre: scalar loads) is fetched two
// stages before its data. Every load is issued unconditionally (indices past the end re-read the last
// group, whose values are then not used), which keeps the count of loads in flight fixed.
template <class T, int NT, int NRT, bool MASK, int kDepth, class Meta, class Pre, class Load>
__device__ __forceinline__ void ring_run(Acc<T, NT, NRT> &acc, int q0, int qstride, int qend, int s, Pre &&pre,
                                         Load &&ld) {
    if (q0 >= qend) return;
    const int qlast = qend - 1;
    const int step = kDepth * qstride;
    Grp<T, NT, NRT> ga[kDepth], gb[kDepth];
    Meta ma[kDepth], mb[kDepth];
#pragma unroll
    for (int j = 0; j < kDepth; j++) ma[j] = pre(min(q0 + j * qstride, qlast));
#pragma unroll
    for (int j = 0; j < kDepth; j++) ld(min(q0 + j * qstride, qlast), ma[j], ga[j]);
#pragma unroll
    for (int j = 0; j < kDepth; j++) mb[j] = pre(min(q0 + step + j * qstride, qlast));
    for (int qb = q0; qb < qend; qb += 2 * step) {
        // stage A: groups qb.. from set a; set b loads groups qb + step..
#pragma unroll
        for (int j = 0; j < kDepth; j++) ld(min(qb + step + j * qstride, qlast), mb[j], gb[j]);
#pragma unroll
        for (int j = 0; j < kDepth; j++) ma[j] = pre(min(qb + 2 * step + j * qstride, qlast));
        __builtin_amdgcn_sched_barrier(0);  // the loads go out before the products that wait for the other set
#pragma unroll
        for (int j = 0; j < kDepth; j++)
            if (qb + j * qstride < qend)
                grp_mma<T, NT, NRT, MASK>(acc, ga[j], s);
            else
                keep(ga[j]);  // a skipped group's loads are waited for here, not at the next loop head
        __builtin_amdgcn_sched_barrier(0);
        if (qb + step >= qend) break;
        // stage B: groups qb + step.. from set b; set a loads groups qb + 2 step..
#pragma unroll
        for (int j = 0; j < kDepth; j++) ld(min(qb + 2 * step + j * qstride, qlast), ma[j], ga[j]);
#pragma unroll
        for (int j = 0; j < kDepth; j++) mb[j] = pre(min(qb + 3 * step + j * qstride, qlast));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kDepth; j++)
            if (qb + step + j * qstride < qend)
                grp_mma<T, NT, NRT, MASK>(acc, gb[j], s);
            else
                keep(gb[j]);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < kDepth; j++) keep(ga[j]), keep(gb[j]);
}

// The groups of [0, n) that wave w of a W-wave workgroup takes: (first, stride, end).
template <int W>
__device__ __forceinline__ int3 wave_share(int n, int w) {
    if (kChunked) {
        const int chunk = (n + W - 1) / W;
        return make_int3(w * chunk, 1, min(n, (w + 1) * chunk));
    }
    return make_int3(w, W, n);
}

// LDS of a reduction / output staging: W / 2 slots of NT * 256 values (one row tile each), and room for
// PR x 16 NT values of an output tile.
template <class T, int NT, int W, int PR = kPartRows>
struct alignas(16) Lds {
    T v[std::max((W / 2) * NT * 256, PR * 16 * NT)];
};

// Fixed-order tree reduction of the W wave partials into wave 0, one row tile at a time:
// (w, w + W/2), ..., (0, 1).
template <int W, class T, int NT, int NRT>
__device__ __forceinline__ void reduce_waves(Acc<T, NT, NRT> &acc, T *red, int w, int lane) {
#pragma unroll
    for (int rt = 0; rt < NRT; rt++) {
#pragma unroll
        for (int half = W / 2; half >= 1; half >>= 1) {
            __syncthreads();
            if (w >= half && w < 2 * half) {
                T *r = red + (w - half) * NT * 256;
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int v = 0; v < 4; v++) r[nt * 256 + v * 64 + lane] = acc[rt][nt][v];
            }
            __syncthreads();
            if (w < half) {
                const T *r = red + w * NT * 256;
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int v = 0; v < 4; v++) acc[rt][nt][v] += r[nt * 256 + v * 64 + lane];
            }
        }
    }
}

// Write a wave's result tile as rows of W <= 16 NT values: tile[row * W + n] (row < rows, n < W).
template <class T, int NT, int NRT>
__device__ __forceinline__ void store_tile(const Acc<T, NT, NRT> &acc, T *tile, int rows, int W, int lane) {
    const int i16 = lane & 15, kk = lane >> 4;
#pragma unroll
    for (int rt = 0; rt < NRT; rt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = rt * 16 + Mfma<T>::row(kk, v);
                if (row < rows && nt * 16 + i16 < W) tile[row * W + nt * 16 + i16] = acc[rt][nt][v];
            }
}

// ---------------------------------------------------------------- phase 1: t_s = V_s x[cs:ce]
// A unit is (stack, 32 stacked rows). Units [0, nbig) belong to stacks with at least kBigCols
// columns: the whole workgroup takes the unit and reduces in LDS. The rest are taken one per
// wavefront. The results go to xt rows t_row + p.
template <class T, int NT, bool NARROW, int NRT>
__device__ __forceinline__ void lr_run(const VStack &S, int base, const typename Mfma<T>::T2 *__restrict__ V,
                                       typename Mfma<T>::T2 *__restrict__ xt, int R, T *red, bool big, int w,
                                       int lane) {
    typedef typename Mfma<T>::T2 T2;
    const int r = S.rtot, n = S.n;
    const int i16 = lane & 15, kk = lane >> 4, s = i16 & 1;
    const int amax = min(32, r - base) - 1;
    const T2 *A0 = V + S.v_off + base;
    const int RW = NARROW ? R : 8 * NT;
    const T *B0 = reinterpret_cast<const T *>(xt) + (int64_t)S.cs * 2 * RW + lane_col<NARROW>(i16, R);
    Acc<T, NT, NRT> acc;
    zero_acc<T, NT, NRT>(acc);
    const int ngr = (n + 3) >> 2;
    const int3 sh = big ? wave_share<kLrWaves>(ngr, w) : make_int3(0, 1, ngr);
    ring_run<T, NT, NRT, true, lr_depth<T>(), int>(
        acc, sh.x, sh.y, sh.z, s, [](int) { return 0; },
        [&](int q, int, Grp<T, NT, NRT> &g) {
            const int c = q * 4 + kk;
            const bool ok = c < n;
            const int cc = ok ? c : q * 4;
            grp_load<T, NT, NRT>(g, ok ? T(1) : T(0), A0 + (int64_t)cc * r, amax, i16, B0 + (int64_t)cc * 2 * RW);
        });
    if (big) {
        reduce_waves<kLrWaves, T, NT, NRT>(acc, red, w, lane);
        if (w != 0) return;
    }
    T *out = reinterpret_cast<T *>(xt + (S.t_row + base) * RW);
    store_tile<T, NT, NRT>(acc, out, r - base, 2 * RW, lane);
}

template <class T, int NT, bool NARROW = false>
__global__ __launch_bounds__(64 * kLrWaves) void k_lr_mfma(const VStack *__restrict__ stacks,
                                                         const int2 *__restrict__ units, int nbig, int nunits,
                                                         const typename Mfma<T>::T2 *__restrict__ V,
                                                         typename Mfma<T>::T2 *__restrict__ xt, int R,
                                                         const int *__restrict__ gate) {
    __shared__ Lds<T, NT, kLrWaves> red;
    if (gated(gate)) return;
    const int w = wave_id(), lane = threadIdx.x & 63;
    const bool big = (int)blockIdx.x < nbig;
    const int u = big ? (int)blockIdx.x : nbig + ((int)blockIdx.x - nbig) * kLrWaves + w;
    if (u >= nunits) return;  // small units only: big workgroups always have a unit
    const int2 un = units[u];
    if (un.x < 0) return;  // padding
    const VStack S = stacks[un.x];
    const int base = un.y * 32;
    if (S.rtot - base > 16)
        lr_run<T, NT, NARROW, 2>(S, base, V, xt, R, red.v, big, w, lane);
    else
        lr_run<T, NT, NARROW, 1>(S, base, V, xt, R, red.v, big, w, lane);
}

// ---------------------------------------------------------------- phase 2: row-leaf tasks
// A task is a range of one row leaf's panel groups, taken by one workgroup: each wave takes a share
// of the groups (wave_share) and the partial tiles are summed in a fixed order in LDS. A leaf with
// a single task writes y = -x/2 + acc itself; the tasks of a split leaf write partial tiles that
// k_rows_sum adds in task order. Output goes through LDS so that y rows are written contiguously.
//
// With narrow rows the last of a split leaf's tasks to finish adds the tiles up itself, in task order whichever task that
// is, which saves a launch. The tiles pass between workgroups on dies with caches of their own: they are written and read
// with agent-scope (write-through, cache-bypassing) accesses, and the arrival is counted after every wavefront's
// stores are acknowledged, so neither side flushes or invalidates a cache. Whole product, one right-hand side: FP64 2000 Hz
// 105.3 -> 101.6 us, FP64 leaves of 128 transposed 144.6 -> 135.2, FP32 4000 Hz 69.6 -> 67.0; four: 111.1 -> 109.6, 147.9
// -> 148.1, 70.9 -> 68.2. From five on the tiles' round trip at the end of each task costs what the launch
// did, and more as they grow (FP32 4000 Hz, 37: 158.6 -> 165.0), so the other kernels leave the sum to k_rows_sum.
__device__ __forceinline__ void store_agent(uint64_t *p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t load_agent(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A split leaf's tile (in red) to its slot; true in every thread of the task that arrives last, with the leaf's sum in
// red instead. Only the 2 R values of a row that are used pass through memory, as 64-bit words.
constexpr int kSumBatch = 8;
template <class T, int RP>
__device__ __forceinline__ bool sum_tasks(const RowTask &T_, int m, int R, T *__restrict__ part, int prow,
                                          int *__restrict__ count, T *red, int *arrived) {
    constexpr int kVals = 8 / (int)sizeof(T), kStride = 2 * RP / kVals;  // values per word, words per row of red
    const int rw = 2 * R / kVals, n = m * rw;                            // words per row, words
    const int64_t slot_words = (int64_t)prow * kStride;
    uint64_t *words = reinterpret_cast<uint64_t *>(red), *p0 = reinterpret_cast<uint64_t *>(part) + T_.slot0 * slot_words;
    uint64_t *dst = p0 + (T_.slot - T_.slot0) * slot_words;
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        const int row = e / rw;
        store_agent(dst + e, words[row * kStride + (e - row * rw)]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's stores are at the point of coherence
    __syncthreads();
    if (threadIdx.x == 0) {
        const int a = __hip_atomic_fetch_add(count + T_.count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a == T_.ntask - 1) __hip_atomic_store(count + T_.count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *arrived = a;
    }
    __syncthreads();
    if (*arrived != T_.ntask - 1) return false;
    union Word {
        uint64_t w;
        T v[kVals];
    };
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        Word a;
#pragma unroll
        for (int i = 0; i < kVals; i++) a.v[i] = T(0);
        for (int k0 = 0; k0 < T_.ntask; k0 += kSumBatch) {
            Word v[kSumBatch];
#pragma unroll
            for (int b = 0; b < kSumBatch; b++) v[b].w = load_agent(p0 + min(k0 + b, T_.ntask - 1) * slot_words + e);
#pragma unroll
            for (int b = 0; b < kSumBatch; b++)
#pragma unroll
                for (int i = 0; i < kVals; i++) a.v[i] = k0 + b < T_.ntask ? a.v[i] + v[b].v[i] : a.v[i];
        }
        const int row = e / rw;
        words[row * kStride + (e - row * rw)] = a.w;
    }
    __syncthreads();
    return true;
}

template <class T, int NT, bool NARROW, int NRT>
__device__ __forceinline__ void rows_run(const RowTask &T_, int rs, int m, const LeafPanel &L,
                                         const int *__restrict__ psrc,
                                         const typename Mfma<T>::T2 *__restrict__ panel,
                                         const typename Mfma<T>::T2 *__restrict__ xt, const double *__restrict__ x,
                                         int N, int R, double *__restrict__ y, const int *__restrict__ cols, int j0,
                                         T *__restrict__ part, int prow, int *__restrict__ count, T *red, int *arrived,
                                         int w, int lane) {
    typedef typename Mfma<T>::T2 T2;
    constexpr int RP = 8 * NT;
    const int i16 = lane & 15, kk = lane >> 4, s = i16 & 1;
    Acc<T, NT, NRT> acc;
    zero_acc<T, NT, NRT>(acc);
    const T2 *A0 = panel + L.off + (int64_t)kk * m;
    const int RW = NARROW ? R : RP;
    const int bcol = lane_col<NARROW>(i16, R);
    const int4 *src4 = reinterpret_cast<const int4 *>(psrc + L.col0) + T_.g0;
    const int3 sh = wave_share<kRowWaves>(T_.g1 - T_.g0, w);
    ring_run<T, NT, NRT, false, row_depth<T>(), int4>(
        acc, sh.x, sh.y, sh.z, s, [&](int q) { return src4[q]; },  // the group's 4 source rows (scalar load)
        [&](int q, const int4 &sr, Grp<T, NT, NRT> &g) {
            const int row = pick4(sr, kk);
            grp_load<T, NT, NRT>(g, T(1), A0 + (int64_t)(T_.g0 + q) * 4 * m, m - 1, i16,
                                 reinterpret_cast<const T *>(xt) + (int64_t)row * 2 * RW + bcol);
        });
    reduce_waves<kRowWaves, T, NT, NRT>(acc, red, w, lane);
    __syncthreads();  // every wave has read the reduction buffer before it is reused for staging
    if (w == 0) store_tile<T, NT, NRT>(acc, red, m, 2 * RP, lane);
    __syncthreads();
    if (T_.slot >= 0) {
        if constexpr (NARROW) {
            if (!sum_tasks<T, RP>(T_, m, R, part, prow, count, red, arrived)) return;
        } else {
            T *dst = part + (int64_t)T_.slot * prow * (2 * RP);
            for (int e = threadIdx.x; e < m * 2 * RP; e += blockDim.x) dst[e] = red[e];
            return;
        }
    }
    for (int e = threadIdx.x; e < 2 * m * R; e += blockDim.x) {
        const int j = e / (2 * m), q = e - j * 2 * m, row = q >> 1, p = q & 1;
        const int64_t idx = (col_of(cols, j0, j) * N + rs + row) * 2 + p;
        y[idx] = -0.5 * x[idx] + (double)red[row * 2 * RP + 2 * j + p];
    }
}

template <class T, int NT, int MAXRT, bool NARROW = false>
__global__ __launch_bounds__(64 * kRowWaves) void k_rows_mfma(
    const RowTask *__restrict__ tasks, const int *__restrict__ leaf_start, const LeafPanel *__restrict__ lpanel,
    const int *__restrict__ psrc, const typename Mfma<T>::T2 *__restrict__ panel,
    const typename Mfma<T>::T2 *__restrict__ xt, const double *__restrict__ x, int N, int R, double *__restrict__ y,
    const int *__restrict__ cols, int j0, const int *__restrict__ gate, T *__restrict__ part, int prow,
    int *__restrict__ count) {
    constexpr int PR = MAXRT > 4 ? kMaxLeaf : kPartRows;  // output staging rows
    __shared__ Lds<T, NT, kRowWaves, PR> red;
    __shared__ int arrived;
    if (gated(gate)) return;
    const int w = wave_id(), lane = threadIdx.x & 63;
    const RowTask T_ = tasks[blockIdx.x];
    if (T_.leaf < 0) return;  // padding task
    const int rs = leaf_start[T_.leaf], m = leaf_start[T_.leaf + 1] - rs;
    const LeafPanel L = lpanel[T_.leaf];
    const int nrt = (m + 15) >> 4;
    if (nrt <= 1)
        rows_run<T, NT, NARROW, 1>(T_, rs, m, L, psrc, panel, xt, x, N, R, y, cols, j0, part, prow, count, red.v, &arrived, w,
                                     lane);
    else if (nrt == 2 || MAXRT == 2)
        rows_run<T, NT, NARROW, 2>(T_, rs, m, L, psrc, panel, xt, x, N, R, y, cols, j0, part, prow, count, red.v, &arrived, w,
                                     lane);
    else if constexpr (MAXRT == 4) {
        if (nrt == 3)
            rows_run<T, NT, NARROW, 3>(T_, rs, m, L, psrc, panel, xt, x, N, R, y, cols, j0, part, prow, count, red.v, &arrived, w,
                                     lane);
        else
            rows_run<T, NT, NARROW, 4>(T_, rs, m, L, psrc, panel, xt, x, N, R, y, cols, j0, part, prow, count, red.v, &arrived, w,
                                     lane);
    } else if constexpr (MAXRT == 8) {
        if (nrt <= 4)
            rows_run<T, NT, NARROW, 4>(T_, rs, m, L, psrc, panel, xt, x, N, R, y, cols, j0, part, prow, count, red.v, &arrived, w,
                                     lane);
        else if (nrt <= 6)
            rows_run<T, NT, NARROW, 6>(T_, rs, m, L, psrc, panel, xt, x, N, R, y, cols, j0, part, prow, count, red.v, &arrived, w,
                                     lane);
        else
            rows_run<T, NT, NARROW, 8>(T_, rs, m, L, psrc, panel, xt, x, N, R, y, cols, j0, part, prow, count, red.v, &arrived, w,
                                     lane);
    }
}

// y = -x/2 + the task partials of each split leaf, summed in task order. Workgroup (leaf, chunk) takes
// kSumRows rows of one split leaf: every thread holds its few elements in registers and issues the loads
// of up to kSumBatch partials together (indices clamped, surplus values not added), so a workgroup waits
// about once per batch rather than once per partial; the summed rows go through LDS so that y rows are
// written contiguously.
constexpr int kSumRows = 8;
template <class T, int NT>
__global__ __launch_bounds__(256) void k_rows_sum(const int4 *__restrict__ split, const int *__restrict__ leaf_start,
                                                  const T *__restrict__ part, const double *__restrict__ x, int N,
                                                  int R, double *__restrict__ y, const int *__restrict__ cols, int j0,
                                                  const int *__restrict__ gate, int prow) {
    constexpr int W = 16 * NT, E = kSumRows * W, EPT = (E + 255) / 256;
    __shared__ T tile[E];
    if (gated(gate)) return;
    const int4 S = split[blockIdx.x];
    const int rs = leaf_start[S.x], m = leaf_start[S.x + 1] - rs;
    const int r0 = (int)blockIdx.y * kSumRows;
    if (r0 >= m) return;
    const int mr = min(kSumRows, m - r0), ne = mr * W;
    const T *src = part + (int64_t)S.y * prow * W + (int64_t)r0 * W;
    T acc[EPT];
#pragma unroll
    for (int i = 0; i < EPT; i++) acc[i] = T(0);
    for (int k0 = 0; k0 < S.z; k0 += kSumBatch) {
        T v[kSumBatch][EPT];
#pragma unroll
        for (int b = 0; b < kSumBatch; b++) {
            const T *sk = src + (int64_t)min(k0 + b, S.z - 1) * prow * W;
#pragma unroll
            for (int i = 0; i < EPT; i++) v[b][i] = sk[min((int)threadIdx.x + i * 256, ne - 1)];
        }
#pragma unroll
        for (int b = 0; b < kSumBatch; b++)
#pragma unroll
            for (int i = 0; i < EPT; i++) acc[i] = k0 + b < S.z ? acc[i] + v[b][i] : acc[i];
    }
#pragma unroll
    for (int i = 0; i < EPT; i++) {
        const int e = (int)threadIdx.x + i * 256;
        if (e < ne) tile[e] = acc[i];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 2 * mr * R; e += blockDim.x) {
        const int j = e / (2 * mr), q = e - j * 2 * mr, row = q >> 1, p = q & 1;
        const int64_t idx = (col_of(cols, j0, j) * N + rs + r0 + row) * 2 + p;
        y[idx] = -0.5 * x[idx] + (double)tile[row * W + 2 * j + p];
    }
}

// ---------------------------------------------------------------- layout (once per assembly)
// Stacked factors, column-major per stack: entry (c, p) of stack row o_b + p <- V_b[p][c] (forward,
// FP64 V row-major) or U_b[c][p] (transposed, FP64 U leaf-segmented: the row's leaf chunk). Workgroup (block, y)
// takes every gridDim.y-th tile of kStackCols entries by kStackRanks crosses through LDS: read along the entries,
// written along the crosses, contiguous on both sides (FP32, 4000 Hz: 103 us; 157 us reading F with the stride of
// the crosses, one workgroup per block).
constexpr int kStackCols = 64, kStackRanks = 16, kStackSplit = 8;
template <class T, bool UT>
__global__ __launch_bounds__(256) void k_stack(const LRBlock *__restrict__ blocks, const StackMap *__restrict__ maps,
                                               const double2 *__restrict__ F, const int *__restrict__ leaf_start,
                                               const int *__restrict__ leaf_of,
                                               typename Mfma<T>::T2 *__restrict__ Vs) {
    typedef typename Mfma<T>::T2 T2;
    __shared__ T2 tile[kStackRanks][kStackCols + 1];
    const StackMap M = maps[blockIdx.x];
    const LRBlock B = blocks[M.blk];
    const int r = B.rank, n = UT ? B.re - B.rs : B.ce - B.cs;
    const int lane = threadIdx.x % ARH_WAVE, w = threadIdx.x / ARH_WAVE;
    for (int c0 = (int)blockIdx.y * kStackCols; c0 < n; c0 += (int)gridDim.y * kStackCols) {
        const int c = c0 + lane, cn = min(kStackCols, n - c0);
        // the lane's entry: cross p at F[base + p * step]
        int64_t base = 0, step = 0;
        if (c < n) {
            if (UT) {
                const int l = leaf_of[B.rs + c];
                const int ls = leaf_start[l] - B.rs;
                step = leaf_start[l + 1] - leaf_start[l];
                base = B.u_off + (int64_t)ls * r + (c - ls);
            } else {
                step = n, base = B.v_off + c;
            }
        }
        for (int p0 = 0; p0 < r; p0 += kStackRanks) {
            const int pn = min(kStackRanks, r - p0);
            __syncthreads();
            if (c < n)
#pragma unroll
                for (int q = w; q < kStackRanks; q += 256 / ARH_WAVE)
                    if (q < pn) {
                        const double2 v = F[base + (p0 + q) * step];
                        tile[q][lane] = Mfma<T>::make(v.x, v.y);
                    }
            __syncthreads();
            const int q = threadIdx.x % kStackRanks;
            if (q < pn)
                for (int i = threadIdx.x / kStackRanks; i < cn; i += 256 / kStackRanks)
                    Vs[M.dst + (int64_t)(c0 + i) * M.rtot + p0 + q] = tile[q][i];
        }
    }
}

// Fused panels: entry i of panel column c of leaf l <- the FP64 value at csrc[col0 + c]. Workgroup (leaf, y): its
// wavefronts take the leaf's panel columns in groups of as many as fit 64 lanes (one if m > 32), lane q of a group
// row q % m of column q / m: leaves of about 20 rows used a third of a wavefront's lanes at one column each (FP32, 4000
// Hz: 163 us, now 109 us).
constexpr int kFuseSplit = 64;
template <class T>
__global__ __launch_bounds__(256) void k_fuse_panel(const int *__restrict__ leaf_start,
                                                    const LeafPanel *__restrict__ lpanel,
                                                    const ColSrc *__restrict__ csrc, const double2 *__restrict__ dense,
                                                    const double2 *__restrict__ U, const double2 *__restrict__ V,
                                                    typename Mfma<T>::T2 *__restrict__ panel,
                                                    const int *__restrict__ bad) {
    if (*bad) return;  // the lists are refused
    const int l = blockIdx.x;
    const int m = leaf_start[l + 1] - leaf_start[l];
    const LeafPanel L = lpanel[l];
    const int ncol = L.ngroups * 4;
    const int w = threadIdx.x / ARH_WAVE, lane = threadIdx.x % ARH_WAVE;
    const int per = max(1, ARH_WAVE / m);
    const int cc = per > 1 ? lane / m : 0, i0 = lane - cc * m;
    if (cc >= per) return;
    const int step = (int)gridDim.y * 4 * per;
#pragma unroll 4
    for (int c = ((int)blockIdx.y * 4 + w) * per + cc; c < ncol; c += step) {
        const ColSrc cs = csrc[L.col0 + c];
        const double2 *src = cs.kind == 1 ? dense : cs.kind == 2 ? U : V;
        typename Mfma<T>::T2 *dst = panel + L.off + (int64_t)c * m;
        for (int i = i0; i < m; i += ARH_WAVE) {
            double2 v = make_double2(0.0, 0.0);
            if (cs.kind) v = src[cs.off + (int64_t)i * cs.stride];
            dst[i] = Mfma<T>::make(v.x, v.y);
        }
    }
}

// Panel column lists of one leaf, written by one wavefront: the source row (psrc: x row, or N + the
// intermediates row) and the FP64 gather source (csrc) of every column of the leaf's fused panel.
//  forward:    the row leaf's dense columns (panel column c of the dense panel), then for each low-rank
//              block covering the leaf (lr list order) its rank U columns restricted to the leaf;
//  transposed: for each dense block in the column leaf's list, its mr rows as columns (a row of the
//              column-major block in its row leaf's panel, stride mr), then the V columns restricted to
//              the leaf of each low-rank block whose column range covers it;
// zero columns (source row 0, kind 0) up to the leaf's ncol. A list's column offsets are a wavefront
// prefix sum of the entries' widths. bad[0], and hbad[0] in pinned memory, are raised when a column count disagrees
// with the host's ncol, a source row falls outside [0, nsrc), or a low-rank block does not cover the leaf.
__device__ __forceinline__ int wave_incl_scan(int v, int lane) {
#pragma unroll
    for (int d = 1; d < ARH_WAVE; d <<= 1) {
        const int t = __shfl_up(v, d, ARH_WAVE);
        if (lane >= d) v += t;
    }
    return v;
}

__global__ __launch_bounds__(ARH_WAVE) void k_panel_cols(
    int tr, const LeafPanel *__restrict__ lpanel, const int *__restrict__ leaf_start,
    const int *__restrict__ pcol_ptr, const int64_t *__restrict__ panel_off, const int *__restrict__ pcol_idx,
    const int *__restrict__ dT_ptr, const int *__restrict__ dT_blk, const int *__restrict__ dblk_info,
    const int *__restrict__ lr_ptr, const int *__restrict__ lr_blk,
    const LRBlock *__restrict__ blocks, const int *__restrict__ t_row, int nsrc, int *__restrict__ psrc,
    ColSrc *__restrict__ csrc, int *__restrict__ bad, int *__restrict__ hbad) {
    const int l = blockIdx.x, lane = threadIdx.x;
    const int ls = leaf_start[l], m = leaf_start[l + 1] - ls;
    const LeafPanel L = lpanel[l];
    const int ncol = L.ngroups * 4;
    int *ps = psrc + L.col0;
    ColSrc *cs = csrc + L.col0;
    int base = 0;
    bool ok = true;
    if (!tr) {
        const int p0 = pcol_ptr[l], nd = pcol_ptr[l + 1] - p0;
        for (int c = lane; c < nd && c < ncol; c += ARH_WAVE) {
            ps[c] = pcol_idx[p0 + c];
            cs[c] = ColSrc{panel_off[l] + (int64_t)c * m, 1, 1};
        }
        base = nd;
    } else {
        const int e0 = dT_ptr[l], e1 = dT_ptr[l + 1];
        for (int c0 = e0; c0 < e1; c0 += ARH_WAVE) {
            const int e = c0 + lane;
            int b = 0, rl = 0, pc = 0, mr = 0;
            if (e < e1) {
                b = dT_blk[e];
                rl = dblk_info[2 * b], pc = dblk_info[2 * b + 1];
                mr = leaf_start[rl + 1] - leaf_start[rl];
            }
            const int inc = wave_incl_scan(mr, lane);
            const int start = base + inc - mr;
            const int rs = e < e1 ? leaf_start[rl] : 0;
            for (int j = 0; j < mr && start + j < ncol; j++) {
                ps[start + j] = rs + j;
                cs[start + j] = ColSrc{panel_off[rl] + (int64_t)pc * mr + j, mr, 1};
            }
            base += __shfl(inc, ARH_WAVE - 1, ARH_WAVE);
        }
    }
    const int e0 = lr_ptr[l], e1 = lr_ptr[l + 1];
    for (int c0 = e0; c0 < e1; c0 += ARH_WAVE) {
        const int e = c0 + lane;
        int r = 0, b = 0;
        LRBlock B{};
        if (e < e1) {
            b = lr_blk[e];
            B = blocks[b];
            r = B.rank;
            if (tr ? (ls < B.cs || ls + m > B.ce) : (ls < B.rs || ls + m > B.re)) ok = false;
        }
        const int inc = wave_incl_scan(r, lane);
        const int start = base + inc - r;
        for (int p = 0; p < r && start + p < ncol; p++) {
            const int src = t_row[b] + p;
            ps[start + p] = src;
            if (src < 0 || src >= nsrc) ok = false;
            cs[start + p] = tr ? ColSrc{B.v_off + (int64_t)p * (B.ce - B.cs) + (ls - B.cs), 1, 3}
                               : ColSrc{B.u_off + (int64_t)(ls - B.rs) * B.rank + (int64_t)p * m, 1, 2};
        }
        base += __shfl(inc, ARH_WAVE - 1, ARH_WAVE);
    }
    // the host rounded the leaf's column count up to a multiple of 4
    if (base > ncol || base + 4 <= ncol) ok = false;
    for (int c = base + lane; c < ncol; c += ARH_WAVE) {
        ps[c] = 0;
        cs[c] = ColSrc{0, 0, 0};
    }
    if (!ok) *bad = 1, *hbad = 1;  // every writer writes the same
}

// Where the stacks' members go, a wavefront per stack: the rows of a stack are its members' crosses in order, so a
// member's first row is the sum of the ranks before it.
__global__ __launch_bounds__(256) void k_stack_maps(int ns, const VStack *__restrict__ stacks, const int *__restrict__ ptr,
                                                    const int *__restrict__ mem, const LRBlock *__restrict__ blocks,
                                                    StackMap *__restrict__ maps, int *__restrict__ t_row) {
    const int k = (int)blockIdx.x * 4 + threadIdx.x / ARH_WAVE, lane = threadIdx.x % ARH_WAVE;
    if (k >= ns) return;
    const VStack S = stacks[k];
    int base = 0;
    for (int q0 = ptr[k], q1 = ptr[k + 1]; q0 < q1; q0 += ARH_WAVE) {
        const int q = q0 + lane, b = q < q1 ? mem[q] : 0, r = q < q1 ? blocks[b].rank : 0;
        const int inc = wave_incl_scan(r, lane);
        if (q < q1) {
            const int o = base + inc - r;
            maps[q] = StackMap{b, S.rtot, S.v_off + o};
            t_row[b] = (int)(S.t_row + o);
        }
        base += __shfl(inc, ARH_WAVE - 1, ARH_WAVE);
    }
}

// Low-rank blocks by the cluster that their stacked factor belongs to, fixed by the partition.
static arh_geom_s::Clusters &clusters_of(arh_geom *g, int tr) {
    arh_geom_s::Clusters &C = g->clusters[tr];
    if (C.made) return C;
    hipStream_t s = g->ctx->stream;
    const int na = g->na, *lr = g->lowrank.data() + (tr ? 0 : 2);  // row or column range of block a: lr[4 a], lr[4 a + 1]
    std::unordered_map<int64_t, int> id;
    std::vector<int> of(na);
    C.start.clear(), C.n.clear();
    for (int a = 0; a < na; a++) {
        const auto it = id.emplace(((int64_t)lr[4 * a] << 32) | (uint32_t)lr[4 * a + 1], (int)C.start.size());
        if (it.second) C.start.push_back(lr[4 * a]), C.n.push_back(lr[4 * a + 1] - lr[4 * a]);
        of[a] = it.first->second;
    }
    const int ns = (int)C.start.size();
    C.ptr.assign(ns + 1, 0);
    C.mem.resize(na);
    for (int a = 0; a < na; a++) C.ptr[of[a] + 1]++;
    for (int k = 0; k < ns; k++) C.ptr[k + 1] += C.ptr[k];
    std::vector<int> fill(C.ptr.begin(), C.ptr.end() - 1);
    for (int a = 0; a < na; a++) C.mem[fill[of[a]]++] = a;
    C.by_size.resize(ns);
    for (int k = 0; k < ns; k++) C.by_size[k] = k;
    std::stable_sort(C.by_size.begin(), C.by_size.end(), [&](int p, int q) { return C.n[p] > C.n[q]; });
    upload(C.d_ptr, C.ptr, s);
    upload(C.d_mem, C.mem, s);
    C.made = true;
    return C;
}

// Work lists of one orientation, shared by both precisions (host + device copies).
//  forward:    stacks of V by column cluster; panels of row leaves: dense columns, then the U
//              columns (leaf segment) of the low-rank blocks covering the leaf.
//  transposed: stacks of U^T by row cluster; panels of column leaves: the transposed dense blocks
//              of the leaf, then the V columns (restricted to the leaf) of the low-rank blocks
//              whose column range covers it.
// Returns the pinned block that the lists are uploaded from; its first int is raised by the device if the lists are not
// to be used, which the caller asks after a synchronisation.
static std::unique_ptr<HostBuf> build_lists(arh_hmat *h, int tr) {
    arh_geom *g = h->g;
    MfmaLayout &M = h->mf[tr];
    hipStream_t s = g->ctx->stream;
    const int N = g->N;
    const int2 *rank = h->ranks.data();
    ARH_CHECK(g->max_leaf <= kMaxLeaf, ARH_EINVAL, "MFMA product supports leaves of at most 128 elements");
    // stacks: the low-rank blocks grouped by their column (forward) / row (transposed) cluster
    const arh_geom_s::Clusters &C = clusters_of(g, tr);
    const int ns = (int)C.start.size();
    std::vector<VStack> stacks(ns);
    int64_t voff = 0, trow = N;
    size_t nsmall = 0, nbig = 0;
    for (int k = 0; k < ns; k++) {
        VStack S{C.start[k], C.n[k], 0, 0, voff, trow};
        for (int q = C.ptr[k]; q < C.ptr[k + 1]; q++) S.rtot += rank[C.mem[q]].x;
        ARH_CHECK(trow + S.rtot < INT32_MAX, ARH_EINVAL, "stacked intermediates exceed the 32-bit row range");
        stacks[k] = S;
        voff += (int64_t)S.n * S.rtot;
        trow += S.rtot;
        (S.n >= kBigCols ? nbig : nsmall) += (S.rtot + 31) / 32;
    }
    M.vs_total = voff;
    ARH_CHECK(trow - N == h->t_total, ARH_EINVAL, "stacked intermediates do not match the ranks");
    // phase-1 units: big stacks first, each list by decreasing column count
    std::vector<int2> units(nbig + lr_slots(nsmall, kLrWaves), int2{-1, 0});
    size_t ub = 0, us = 0;
    for (int k : C.by_size)
        for (int rt = 0; rt * 32 < stacks[k].rtot; rt++) {
            if (stacks[k].n >= kBigCols)
                units[ub++] = int2{k, rt};
            else
                units[nbig + lr_slot(us++, kLrWaves)] = int2{k, rt};
        }
    M.p1big = (int)nbig;
    M.nunits = (int)units.size();
    // fused panels: column counts here, the column lists on the device (k_panel_cols)
    std::vector<LeafPanel> lpanel(g->nleaf);
    int64_t poff = 0, ncols = 0;
    for (int l = 0; l < g->nleaf; l++) {
        const int ls = g->leaf_start[l], m = g->leaf_start[l + 1] - ls;
        int64_t nc = 0;
        if (!tr) {
            nc = g->pcol_ptr[l + 1] - g->pcol_ptr[l];
            for (int e = g->lrR_ptr[l]; e < g->lrR_ptr[l + 1]; e++) nc += rank[g->lrR_blk[e]].x;
        } else {
            for (int e = g->dT_ptr[l]; e < g->dT_ptr[l + 1]; e++) {
                const int b = g->dT_blk[e], rl = g->dblk_leafr[b];
                ARH_CHECK(g->dense[4 * b + 2] == ls && g->dense[4 * b + 3] == ls + m, ARH_EINVAL,
                          "dense block is not a leaf column");
                nc += g->leaf_start[rl + 1] - g->leaf_start[rl];
            }
            for (int e = g->lrC_ptr[l]; e < g->lrC_ptr[l + 1]; e++) nc += rank[g->lrC_blk[e]].x;
        }
        nc = (nc + 3) / 4 * 4;
        ARH_CHECK(ncols + nc < INT32_MAX, ARH_EINVAL, "panel columns exceed the 32-bit range");
        lpanel[l] = LeafPanel{poff, (int)ncols, (int)(nc / 4)};
        ncols += nc;
        poff += nc * m;
    }
    M.panel_total = poff;
    // row tasks: leaves with more than tg groups are split evenly
    int64_t gt = 0;
    for (const LeafPanel &L : lpanel) gt += L.ngroups;
    int tg = (int)std::max<int64_t>(8 * kRowWaves, (gt + kTaskSlots - 1) / kTaskSlots);
    tg = (tg + kRowWaves - 1) / kRowWaves * kRowWaves;
    std::vector<RowTask> rtasks;
    std::vector<int4> rsplit;
    M.nslots = 0;
    for (int l = 0; l < g->nleaf; l++) {
        const int n = lpanel[l].ngroups;
        const int nt = std::max(1, (n + tg - 1) / tg);
        for (int t = 0; t < nt; t++)
            rtasks.push_back(RowTask{l, (int)((int64_t)n * t / nt), (int)((int64_t)n * (t + 1) / nt),
                                     nt > 1 ? M.nslots + t : -1, M.nslots, nt, (int)rsplit.size(), 0});
        if (nt > 1) {
            rsplit.push_back(int4{l, M.nslots, nt, 0});
            M.nslots += nt;
        }
    }
    // XCD-aware order: workgroups are dispatched round-robin over the kXcds dies, each with its own
    // L2, so die x gets a contiguous run of leaves (in tree order, which neighbouring leaves share
    // most of their low-rank blocks and hence their intermediates rows) with about 1/kXcds of the
    // groups; padding tasks (leaf -1) even out the runs. Otherwise: largest tasks first.
    if (kXcdOrder) {
        std::vector<std::vector<RowTask>> run(kXcds);
        int64_t acc = 0;
        for (const RowTask &T : rtasks) {
            const int x = (int)std::min<int64_t>(kXcds - 1, acc * kXcds / std::max<int64_t>(1, gt));
            run[x].push_back(T);
            acc += T.g1 - T.g0;
        }
        size_t len = 0;
        for (auto &r : run) len = std::max(len, r.size());
        rtasks.assign(len * kXcds, RowTask{-1, 0, 0, -1, 0, 0, 0, 0});
        for (int x = 0; x < kXcds; x++)
            for (size_t i = 0; i < run[x].size(); i++) rtasks[i * kXcds + x] = run[x][i];
    } else {
        std::stable_sort(rtasks.begin(), rtasks.end(),
                         [](const RowTask &p, const RowTask &q) { return p.g1 - p.g0 > q.g1 - q.g0; });
    }
    M.ntasks = (int)rtasks.size();
    // all lists in one block, one upload; in front of them the flag of the device's check
    size_t total = 0;
    auto room = [&](size_t bytes) {
        const size_t o = total;
        total += (bytes + 255) / 256 * 256;
        return o;
    };
    auto bytes_of = [](const auto &v) { return v.size() * sizeof(v[0]); };
    const size_t o_bad = room(sizeof(int)), o_st = room(bytes_of(stacks)), o_un = room(bytes_of(units)),
                 o_lp = room(bytes_of(lpanel)), o_rt = room(bytes_of(rtasks)), o_rs = room(bytes_of(rsplit)),
                 o_ct = room(sizeof(int) * rsplit.size());
    auto hb = std::make_unique<HostBuf>(total, s);
    M.d_lists.alloc(total);
    char *hp = hb->as<char>(), *dp = M.d_lists.as<char>();
    auto put = [&](size_t o, const auto &v) { std::copy(v.begin(), v.end(), (std::decay_t<decltype(v[0])> *)(hp + o)); };
    *(int *)(hp + o_bad) = 0;
    put(o_st, stacks), put(o_un, units), put(o_lp, lpanel), put(o_rt, rtasks), put(o_rs, rsplit);
    std::fill((int *)(hp + o_ct), (int *)(hp + o_ct) + rsplit.size(), 0);
    M.bad = (const int *)(dp + o_bad);
    M.stacks = (const VStack *)(dp + o_st), M.p1units = (const int2 *)(dp + o_un);
    M.lpanel = (const LeafPanel *)(dp + o_lp), M.rtasks = (const RowTask *)(dp + o_rt);
    M.rsplit = (const int4 *)(dp + o_rs), M.count = (int *)(dp + o_ct);
    M.nsplit = (int)rsplit.size();
    ARH_HIP(hipMemcpyAsync(dp, hp, total, hipMemcpyHostToDevice, s));
    // the lists that follow from these on the device
    M.nmaps = g->na;
    M.d_maps.alloc(sizeof(StackMap) * std::max(1, M.nmaps));
    M.d_trow.alloc(sizeof(int) * std::max(1, M.nmaps));
    M.d_psrc.alloc(sizeof(int) * std::max<int64_t>(1, ncols));
    M.d_csrc.alloc(sizeof(ColSrc) * std::max<int64_t>(1, ncols));
    if (ns)
        hipLaunchKernelGGL(k_stack_maps, dim3((ns + 3) / 4), dim3(256), 0, s, ns, M.stacks, C.d_ptr.as<int>(),
                           C.d_mem.as<int>(), h->blocks.as<LRBlock>(), M.d_maps.as<StackMap>(), M.d_trow.as<int>());
    hipLaunchKernelGGL(k_panel_cols, dim3(g->nleaf), dim3(ARH_WAVE), 0, s, tr, M.lpanel, g->d_leaf_start.as<int>(),
                       g->d_pcol_ptr.as<int>(), g->d_panel_off.as<int64_t>(), g->d_pcol_idx.as<int>(),
                       g->d_dT_ptr.as<int>(), g->d_dT_blk.as<int>(), g->d_dblk_info.as<int>(),
                       tr ? g->d_lrC_ptr.as<int>() : g->d_lrR_ptr.as<int>(),
                       tr ? g->d_lrC_blk.as<int>() : g->d_lrR_blk.as<int>(), h->blocks.as<LRBlock>(), M.d_trow.as<int>(),
                       (int)(N + h->t_total), M.d_psrc.as<int>(), M.d_csrc.as<ColSrc>(), (int *)(dp + o_bad),
                       (int *)(hp + o_bad));
    ARH_HIP(hipGetLastError());
    return hb;
}

// The operator copy of one orientation and precision (0: FP32, 1: FP64) in the MFMA layout.
template <class T>
static void build_copy(arh_hmat *h, int tr, int pi) {
    typedef typename Mfma<T>::T2 T2;
    arh_geom *g = h->g;
    MfmaLayout &M = h->mf[tr];
    hipStream_t s = g->ctx->stream;
    M.vs[pi].alloc(sizeof(T2) * std::max<int64_t>(1, M.vs_total));
    M.panel[pi].alloc(sizeof(T2) * std::max<int64_t>(1, M.panel_total));
    if (M.nmaps) {
        if (tr)
            hipLaunchKernelGGL((k_stack<T, true>), dim3((unsigned)M.nmaps, kStackSplit), dim3(256), 0, s, h->blocks.as<LRBlock>(),
                               M.d_maps.as<StackMap>(), h->U.as<double2>(), g->d_leaf_start.as<int>(),
                               g->d_leaf_of.as<int>(), M.vs[pi].as<T2>());
        else
            hipLaunchKernelGGL((k_stack<T, false>), dim3((unsigned)M.nmaps, kStackSplit), dim3(256), 0, s, h->blocks.as<LRBlock>(),
                               M.d_maps.as<StackMap>(), h->V.as<double2>(), g->d_leaf_start.as<int>(),
                               g->d_leaf_of.as<int>(), M.vs[pi].as<T2>());
    }
    hipLaunchKernelGGL(k_fuse_panel<T>, dim3(g->nleaf, kFuseSplit), dim3(256), 0, s, g->d_leaf_start.as<int>(),
                       M.lpanel, M.d_csrc.as<ColSrc>(), h->dense.as<double2>(), h->U.as<double2>(),
                       h->V.as<double2>(), M.panel[pi].as<T2>(), M.bad);
    ARH_HIP(hipGetLastError());
}

void mfma_prepare(arh_hmat *h, int tr, int fp64) {
    MfmaLayout &M = h->mf[tr];
    if (M.built[fp64]) return;
    std::unique_ptr<HostBuf> up;
    if (!M.lists) up = build_lists(h, tr);
    if (fp64)
        build_copy<double>(h, tr, 1);
    else
        build_copy<float>(h, tr, 0);
    if (up) {
        ARH_HIP(hipStreamSynchronize(h->g->ctx->stream));
        ARH_CHECK(!*up->as<int>(), ARH_EINVAL, "panel column lists disagree with the partition or the ranks");
    }
    M.lists = M.built[fp64] = true;
}

// Widest pass (NT output tiles) that fits the registers with 4 row tiles (leaves over 32 elements) and with
// 8 row tiles (leaves over 64 elements).
template <class T>
constexpr int max_nt_tall() {
    return sizeof(T) == 8 ? 3 : 5;
}
template <class T>
constexpr int max_nt_xtall() {
    return sizeof(T) == 8 ? 1 : 2;
}

// Rows of a partial tile: the largest leaf's row tiles (64 rows up to 4 tiles, else 128).
inline int part_rows(int maxrt) { return maxrt > 4 ? kMaxLeaf : kPartRows; }

template <class T, int NT>
static void launch_nt(arh_hmat *h, MfmaLayout &M, int R, const double2 *x, double2 *y, const int *cols, int j0,
                      const int *gate, hipStream_t s, int maxrt, bool packed) {
    typedef typename Mfma<T>::T2 T2;
    constexpr int pi = sizeof(T) == 8 ? 1 : 0;
    arh_geom *g = h->g;
    Profiler &pf = g->ctx->prof;
    const int N = g->N;
    constexpr int RP = 8 * NT;
    const int RW = row_width(R);
    M.xt[pi].alloc(sizeof(T2) * (size_t)(N + h->t_total) * RW);
    const int prow = part_rows(maxrt);
    if (M.nslots) M.part[pi].alloc(sizeof(T) * (size_t)M.nslots * prow * 2 * RP);
    T2 *xt = M.xt[pi].as<T2>();
    if (!packed)
        hipLaunchKernelGGL(k_pack_xf<T>, dim3((unsigned)std::min<int64_t>(2048, ((int64_t)N * RW + 255) / 256)),
                           dim3(256), 0, s, x, N, R, RW, xt, cols, j0, gate);
    auto timed = [&](int kind, double bytes, double flops, auto &&launch) {
        if (!pf.on) {
            launch();
            return;
        }
        Profiler::Entry e{pf.get(), pf.get(), kind, bytes, flops, gate ? pf.cur_slot : -1};
        ARH_HIP(hipEventRecord(e.a, s));
        launch();
        ARH_HIP(hipEventRecord(e.b, s));
        pf.pending.push_back(e);
    };
    // Algorithmic bytes: every operator entry once (eb = one complex entry of T) and every packed rhs
    // / intermediates value once per rhs (also eb: xt holds T2 values), plus the FP64 x read for the
    // -x/2 term and the FP64 y write (16 B per rhs per element) in phase 2. Partial tiles of split
    // leaves and re-reads are not algorithmic.
    const double eb = 2.0 * sizeof(T);
    const int nu = M.nunits, nb = M.p1big;
    const bool narrow = R <= kNarrow;
    // phase-1 entries: V (forward) or U (transposed); both total sum_b r_b (m_b or n_b)
    const int64_t e1 = M.vs_total;
    if (nu)
        timed(pi ? PROF_LR64 : PROF_LR32, eb * e1 + eb * R * (N + h->t_total), 8.0 * R * e1, [&] {
            auto launch_lr = [&](auto kern) {
                hipLaunchKernelGGL(kern, dim3(nb + (nu - nb + kLrWaves - 1) / kLrWaves), dim3(64 * kLrWaves), 0, s,
                                   M.stacks, M.p1units, nb, nu, M.vs[pi].as<T2>(), xt, R,
                                   gate);
            };
            if constexpr (NT == 1)
                if (narrow) return launch_lr(k_lr_mfma<T, 1, true>);
            launch_lr(k_lr_mfma<T, NT>);
        });
    const int64_t ent = g->dense_entries + (h->u_total + h->v_total - e1);
    T *part = M.nslots ? M.part[pi].as<T>() : nullptr;
    const int ntask = M.ntasks;

    const double *xd = (const double *)x;
    double *yd = (double *)y;
    timed(pi ? PROF_ROWS64 : PROF_ROWS32, eb * ent + eb * R * (N + h->t_total) + 32.0 * R * N, 8.0 * R * ent, [&] {
        auto launch_rows = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(ntask), dim3(64 * kRowWaves), 0, s, M.rtasks,
                               g->d_leaf_start.as<int>(), M.lpanel, M.d_psrc.as<int>(),
                               M.panel[pi].as<T2>(), (const T2 *)xt, xd, N, R, yd, cols, j0, gate, part, prow,
                               M.count);
        };
        if constexpr (NT == 1)
            if (narrow)
                return launch_rows(maxrt <= 2   ? k_rows_mfma<T, 1, 2, true>
                                   : maxrt <= 4 ? k_rows_mfma<T, 1, 4, true>
                                                : k_rows_mfma<T, 1, 8, true>);
        if (maxrt <= 2) {
            launch_rows(k_rows_mfma<T, NT, 2>);
        } else if (maxrt <= 4) {
            if constexpr (NT <= max_nt_tall<T>())
                launch_rows(k_rows_mfma<T, NT, 4>);
            else
                ARH_CHECK(false, ARH_EINVAL, "internal: pass too wide for leaves of more than 32 elements");
        } else {
            if constexpr (NT <= max_nt_xtall<T>())
                launch_rows(k_rows_mfma<T, NT, 8>);
            else
                ARH_CHECK(false, ARH_EINVAL, "internal: pass too wide for leaves of more than 64 elements");
        }
    });
    if (M.nsplit && !narrow)
        hipLaunchKernelGGL((k_rows_sum<T, NT>), dim3(M.nsplit, (g->max_leaf + kSumRows - 1) / kSumRows), dim3(256), 0, s,
                           M.rsplit, g->d_leaf_start.as<int>(), part, xd, N, R, yd, cols, j0, gate, prow);
    ARH_HIP(hipGetLastError());
}

int mfma_max_leaf() { return kMaxLeaf; }

// Right-hand sides per pass of a geometry's leaves.
template <class T>
static int pass_width(const arh_geom *g) {
    const int maxrt = (g->max_leaf + 15) / 16;
    return maxrt > 4 ? 8 * max_nt_xtall<T>() : maxrt > 2 ? 8 * max_nt_tall<T>() : kMaxRC;
}

// y = (M - I/2) x, or its transpose, on the MFMA layout of one precision, right-hand sides in passes
// of up to kMaxRC. With a column list (device array of ncols indices into the nrhs columns of x
// and y), only those columns are computed; the others of y are left untouched. A non-null gate
// skips every pass when *gate is 0. packed: the caller has filled the packed rows (mfma_packed_rows).
template <class T>
static void apply_t(arh_hmat *h, MfmaLayout &M, int R, const double2 *x, double2 *y, hipStream_t s, const int *cols,
                    int ncols, const int *gate, bool packed) {
    arh_geom *g = h->g;
    const int maxrt = (g->max_leaf + 15) / 16;
    const int nc = cols ? ncols : R;
    ARH_CHECK(nc >= 0 && nc <= R, ARH_EINVAL, "column list longer than the number of right-hand sides");
    const int maxrc = pass_width<T>(g);
    for (int j0 = 0; j0 < nc; j0 += maxrc) {
        const int Rc = std::min(maxrc, nc - j0);
        switch ((Rc + 7) / 8) {
        case 1: launch_nt<T, 1>(h, M, Rc, x, y, cols, j0, gate, s, maxrt, packed); break;
        case 2: launch_nt<T, 2>(h, M, Rc, x, y, cols, j0, gate, s, maxrt, packed); break;
        case 3: launch_nt<T, 3>(h, M, Rc, x, y, cols, j0, gate, s, maxrt, packed); break;
        case 4: launch_nt<T, 4>(h, M, Rc, x, y, cols, j0, gate, s, maxrt, packed); break;
        default: launch_nt<T, 5>(h, M, Rc, x, y, cols, j0, gate, s, maxrt, packed); break;
        }
    }
}

// Where the packed rows of a product with nc right-hand sides go (N rows of *rw complex values of the operator's
// precision, columns nc .. *rw - 1 zero), for a caller that fills them itself; nullptr if the product takes more
// than one pass, each of which packs its own rows.
template <class T>
static void *packed_rows_t(arh_hmat *h, MfmaLayout &M, int nc, int *rw) {
    typedef typename Mfma<T>::T2 T2;
    if (nc < 1 || nc > pass_width<T>(h->g)) return nullptr;
    *rw = row_width(nc);
    DBuf &xt = M.xt[sizeof(T) == 8 ? 1 : 0];
    xt.alloc(sizeof(T2) * (size_t)(h->g->N + h->t_total) * *rw);
    return xt.p;
}

void *mfma_packed_rows(arh_hmat *h, int transpose, int fp64, int nc, int *rw) {
    const int tr = transpose ? 1 : 0;
    mfma_prepare(h, tr, fp64 ? 1 : 0);
    return fp64 ? packed_rows_t<double>(h, h->mf[tr], nc, rw) : packed_rows_t<float>(h, h->mf[tr], nc, rw);
}

void hmat_apply_mfma(arh_hmat *h, int transpose, int fp64, int R, const double2 *x, double2 *y, hipStream_t s,
                     const int *cols, int ncols, const int *gate, bool packed) {
    ARH_CHECK(h->g->max_leaf <= mfma_max_leaf(), ARH_EINVAL, "MFMA product supports leaves of at most 128 elements");
    const int tr = transpose ? 1 : 0;
    mfma_prepare(h, tr, fp64 ? 1 : 0);
    if (fp64)
        apply_t<double>(h, h->mf[tr], R, x, y, s, cols, ncols, gate, packed);
    else
        apply_t<float>(h, h->mf[tr], R, x, y, s, cols, ncols, gate, packed);
}

}  // namespace arh
