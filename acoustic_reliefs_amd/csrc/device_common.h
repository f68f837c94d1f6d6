// Device helpers shared by the gfx950 kernels: complex arithmetic on double2/float2, the
// 6-point Green's-function quadrature entry, wavefront reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "trig.h"

#define ARH_WAVE 64

namespace arh {

// Degree-4, 6-point triangle rule: weight, barycentric coordinates of b and c
// (constants.h:39-46; the table must equal the reference's value for value).
#define ARH_QW_A 0.223381589678011
#define ARH_QW_B 0.109951743655322
#define ARH_Q_1 0.445948490915965
#define ARH_Q_2 0.108103018168070
#define ARH_Q_3 0.091576213509771
#define ARH_Q_4 0.816847572980459

__device__ __forceinline__ void quad_point(int g, double &w, double &xi, double &eta) {
    switch (g) {
    case 0: w = ARH_QW_A; xi = ARH_Q_1; eta = ARH_Q_2; break;
    case 1: w = ARH_QW_A; xi = ARH_Q_1; eta = ARH_Q_1; break;
    case 2: w = ARH_QW_A; xi = ARH_Q_2; eta = ARH_Q_1; break;
    case 3: w = ARH_QW_B; xi = ARH_Q_3; eta = ARH_Q_4; break;
    case 4: w = ARH_QW_B; xi = ARH_Q_3; eta = ARH_Q_3; break;
    default: w = ARH_QW_B; xi = ARH_Q_4; eta = ARH_Q_3; break;
    }
}

constexpr double kPi = 3.14159265358979323846;
constexpr double kInv8Pi = 1.0 / (8.0 * kPi);  // (1/2 rule factor) * 1/(4 pi)

// Per-element geometry record (16 doubles = 128 B): a, b - a, c - a, n = (b-a)x(c-a), centroid.
struct Tri {
    double ax, ay, az, bx, by, bz, cx, cy, cz, nx, ny, nz, gx, gy, gz, pad;
};
static_assert(sizeof(Tri) == 128, "Tri layout");

// M(p, triangle) = 1/2 sum_g w_g K(p, q_g, n),  K = e^{-ikr}(-ikr-1)/(4 pi r^2) * (-(p-q).n / r)
// (integrate.h:11-19, integrate.cpp:5-14). With d = p - q, s = -(d.n):
// e^{-ikr}(-1-ikr) = (-cos - kr sin) + i(sin - kr cos).
__device__ __forceinline__ double2 bem_entry(double k, double px, double py, double pz, const Tri &t) {
    double re = 0.0, im = 0.0;
#pragma unroll
    for (int g = 0; g < 6; g++) {
        double w, xi, eta;
        quad_point(g, w, xi, eta);
        double qx = t.ax + xi * t.bx + eta * t.cx;
        double qy = t.ay + xi * t.by + eta * t.cy;
        double qz = t.az + xi * t.bz + eta * t.cz;
        double dx = px - qx, dy = py - qy, dz = pz - qz;
        double r2 = dx * dx + dy * dy + dz * dz;
        double r = sqrt(r2);
        double s = -(dx * t.nx + dy * t.ny + dz * t.nz);
        double kr = k * r;
        double sn, cs;
        trig_sincos(kr, &sn, &cs);
        double f = w * s / (r2 * r);
        re += f * (-cs - kr * sn);
        im += f * (sn - kr * cs);
    }
    return make_double2(re * kInv8Pi, im * kInv8Pi);
}

__device__ __forceinline__ Tri load_tri(const Tri *__restrict__ tri, int e) { return tri[e]; }

// ---------------------------------------------------------------- complex helpers
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// acc += a * b
__device__ __forceinline__ void cfma(double2 &acc, double2 a, double2 b) {
    acc.x = fma(a.x, b.x, acc.x);
    acc.x = fma(-a.y, b.y, acc.x);
    acc.y = fma(a.x, b.y, acc.y);
    acc.y = fma(a.y, b.x, acc.y);
}
// conj(a) * b
__device__ __forceinline__ double2 cconjmul(double2 a, double2 b) {
    return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ double2 cdiv(double2 a, double2 b) {
    // Smith's algorithm
    if (fabs(b.x) >= fabs(b.y)) {
        double r = b.y / b.x, den = b.x + b.y * r;
        return make_double2((a.x + a.y * r) / den, (a.y - a.x * r) / den);
    } else {
        double r = b.x / b.y, den = b.y + b.x * r;
        return make_double2((a.x * r + a.y) / den, (a.y * r - a.x) / den);
    }
}
__device__ __forceinline__ double cnorm2(double2 a) { return a.x * a.x + a.y * a.y; }
__device__ __forceinline__ double cabs_(double2 a) { return hypot(a.x, a.y); }

// ---------------------------------------------------------------- wavefront reductions (64 lanes, all active)
// Exchange of wavefront halves and of 16-lane rows: a takes b's lower half (even rows) into its upper half (odd rows),
// b the other way round.
__device__ __forceinline__ void swap32(double &a, double &b) {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]), b = __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ void swap16(double &a, double &b) {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    a = __hiloint2double((int)hi[0], (int)lo[0]), b = __hiloint2double((int)hi[1], (int)lo[1]);
}
template <int CTRL>
__device__ __forceinline__ double row_step(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double row_sum(double v) {  // over a row of 16 lanes: row_ror 8, 4, 2, 1
    return row_step<0x121>(row_step<0x122>(row_step<0x124>(row_step<0x128>(v))));
}
// The sum of v over the wavefront, in every lane: lanes 32 apart first, then 16, 8, 4, 2, 1 apart. (Rotating a row by 4
// after the step by 8 meets the same value as exchanging lanes 4 apart, and so on.)
__device__ __forceinline__ double wave_sum(double v) {
    double a = v, b = v;
    swap32(a, b);
    a = b = a + b;
    swap16(a, b);
    return row_sum(a + b);
}
__device__ __forceinline__ double2 wave_sum2(double2 v) { return make_double2(wave_sum(v.x), wave_sum(v.y)); }
// ---------------------------------------------------------------- wavefront reductions on DPP (no LDS)
// Steps towards lane 63 (row_shr 1, 2, 4, 8, then row_bcast 15 and 31); lanes without a source keep `old`.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double old, double x) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(x), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(x), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
// A lane's value as a wavefront-uniform one (lane uniform).
__device__ __forceinline__ double lane_f64(double x, int lane) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(x), lane);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wsum63(double v) {  // the sum, in lane 63
    v += dpp_f64<0x111>(0.0, v);
    v += dpp_f64<0x112>(0.0, v);
    v += dpp_f64<0x114>(0.0, v);
    v += dpp_f64<0x118>(0.0, v);
    v += dpp_f64<0x142>(0.0, v);
    v += dpp_f64<0x143>(0.0, v);
    return v;
}
__device__ __forceinline__ double wsum(double v) { return lane_f64(wsum63(v), 63); }
// (value, index) max with ties to the lower index; value -1 = empty.
__device__ __forceinline__ void wave_argmax(double &v, int &i) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        double ov = __shfl_xor(v, o, 64);
        int oi = __shfl_xor(i, o, 64);
        if (ov > v || (ov == v && oi < i)) {
            v = ov;
            i = oi;
        }
    }
}

}  // namespace arh
