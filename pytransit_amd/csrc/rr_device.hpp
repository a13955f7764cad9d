// Device-side building blocks of the RoadRunner model for gfx950 (CDNA4).
//
// Geometry, limb-darkening interpolation, Kepler/Taylor orbit and the epoch
// reduction, written once and instantiated for FP64 and FP32 where the flux
// stage needs both.  Reference citations are to PyTransit 2.8.1.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/rr_hip.h"

namespace rr {

constexpr double kPi = 3.14159265358979323846;
constexpr double kTwoPi = 2.0 * kPi;
constexpr double kHalfPi = 0.5 * kPi;
constexpr float kPiF = 3.14159265358979323846f;

// ---- overloads so templates read the same for float and double -----------------------
__device__ __forceinline__ double d_sqrt(double x) { return sqrt(x); }
// FP32: the hardware square root (1 ulp) without sqrtf's denormal rescaling; the
// arguments here are squared distances and kite products, never denormal.
__device__ __forceinline__ float d_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

// FP64 reciprocal, quotient and square root of ordinary magnitudes (no denormal or
// overflow rescaling): the hardware's seed refined by Newton steps, for the root in
// Goldschmidt's coupled form of sqrt(x) and 1 / (2 sqrt(x)), to an ulp or so.
// The compiler's forms add the scaling and fix-up steps that only extreme exponents
// need, twice the instructions.
__device__ __forceinline__ double f64_rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}
__device__ __forceinline__ double f64_div(double a, double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}
__device__ __forceinline__ double f64_sqrt(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    g = fma(fma(-g, g, x), h, g);
    return __builtin_amdgcn_class(x, 0x260) ? x : g;   // +-0 and +inf are their own roots
}

// Coefficient tables in constant memory, read inside loops through a pointer the
// compiler cannot follow.  Written as literals, a loop's 64-bit constants are hoisted
// out of it, two registers each, and a kernel with three such polynomials held 185
// vector registers (2 waves per SIMD) for them; scalar loads from a hot cache line
// leave it at half of that.
typedef const double __attribute__((address_space(4)))* ConstTable;
__device__ __forceinline__ ConstTable const_table(const double* t) {
    ConstTable p = (ConstTable)t;
    asm volatile("" : "+s"(p));
    return p;
}
__constant__ const double kLogTable[8] = {
    0.66666666666667606655, 0.39999999999325053235, 0.285714287554372115, 0.22222197590380998733,
    0.18183604510887957373, 0.15313202419441696023, 0.14803194289933532812, 0.69314718055994530942};
__constant__ const double kAtanTable[12] = {
    -0.33333333333333120541, 0.19999999999940004658, -0.14285714279170125263, 0.11111110741399687907,
    -0.090908967204580554133, 0.076920439540218640828, -0.066629381856421199259, 0.058467923393252907438,
    -0.050347684883633600506, 0.037957984254848413375, -0.017798614429732888959, 0.0};
// sum_j t[j] x^j over N coefficients
template <int N>
__device__ __forceinline__ double table_poly(ConstTable t, double x) {
    double q = t[N - 1];
#pragma unroll
    for (int j = N - 2; j >= 0; --j) q = fma(q, x, t[j]);
    return q;
}

// sqrt(x) and 1 / sqrt(x) together, x > 0.
__device__ __forceinline__ void f64_sqrt_rsqrt(double x, double& s, double& r) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    s = fma(fma(-g, g, x), h, g);
    r = h + h;
    r = fma(fma(-s, r, 1.0), r, r);
}

// log(x) in FP64: x = m 2^e with m in [sqrt(1/2), sqrt 2), log m = 2 atanh(s) with
// s = (m - 1) / (m + 1), atanh(s) / s an interpolating polynomial in s^2 at Chebyshev
// nodes (relative error 2.1e-18 with the coefficients as stored).
__device__ __forceinline__ double f64_log(double x) {
    double m = __builtin_amdgcn_frexp_mant(x);
    int e = __builtin_amdgcn_frexp_exp(x);
    const bool low = m < 0.70710678118654752;
    m = low ? m + m : m;
    e -= low ? 1 : 0;
    const double s = f64_div(m - 1.0, m + 1.0), u = s * s;
    const ConstTable c = const_table(kLogTable);
    const double q = table_poly<7>(c, u);
    const double r = fma((double)e, c[7], fma(s * u, q, s + s));
    return x > 0.0 ? r : (x == 0.0 ? -INFINITY : (double)NAN);
}

// atan2(y, x) in FP64 for y >= 0, not both 0: the quotient of the smaller by the larger
// side, taken about tan(pi/4) above tan(pi/8), then atan(t) / t on |t| <= tan(pi/8) as
// an interpolating polynomial in t^2 at Chebyshev nodes (relative error 4.6e-18 with
// the coefficients as stored).  One division; libm's form handles signs, zeros and
// infinities that the kite never gives.
__device__ __forceinline__ double f64_atan2_ypos(double y, double x) {
    const double ax = fabs(x);
    const bool steep = y > ax;
    const double mx = steep ? y : ax, mn = steep ? ax : y;
    const bool big = mn > 0.41421356237309504880 * mx;
    const double t = f64_div(big ? mn - mx : mn, big ? mn + mx : mx), s = t * t;
    const double q = table_poly<11>(const_table(kAtanTable), s);
    double r = fma(t * s, q, t);
    r = big ? r + 0.25 * kPi : r;
    r = steep ? kHalfPi - r : r;
    return x < 0.0 ? kPi - r : r;
}

// atan2(y, x) for y >= 0 in FP32: octant reduction with one hardware reciprocal
// and atan(t) = t P(t^2) on [0, 1], P of degree 7 fitted by Lawson's minimax
// iteration (pytransit_amd/csrc/atan_poly.py).  Max error 1.4e-7 rad.
__device__ __forceinline__ float atan2_ypos_f(float y, float x) {
    const float ax = fabsf(x);
    const float mx = fmaxf(ax, y), mn = fminf(ax, y);
    const float t = mx > 0.0f ? mn * __builtin_amdgcn_rcpf(mx) : 0.0f;
    const float s = t * t;
    float p = -0.00405456312f;
    p = fmaf(p, s, 0.0218629446f);
    p = fmaf(p, s, -0.0559123158f);
    p = fmaf(p, s, 0.0964219719f);
    p = fmaf(p, s, -0.139086291f);
    p = fmaf(p, s, 0.199465662f);
    p = fmaf(p, s, -0.333298594f);
    p = fmaf(p, s, 0.999999344f);
    float r = t * p;
    r = (y > ax) ? 1.57079633f - r : r;
    return (x < 0.0f) ? 3.14159265f - r : r;
}

// atan2 with y >= 0 (the kite angles): libm in FP64, the polynomial in FP32.
__device__ __forceinline__ double d_atan2_ypos(double y, double x) { return atan2(y, x); }
__device__ __forceinline__ float d_atan2_ypos(float y, float x) { return atan2_ypos_f(y, x); }
__device__ __forceinline__ double d_fma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float d_fma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double d_abs(double x) { return fabs(x); }
__device__ __forceinline__ float d_abs(float x) { return fabsf(x); }
__device__ __forceinline__ double d_max(double a, double b) { return fmax(a, b); }
// FP32 min/max as selects: no NaN canonicalisation (the FP32 geometry never sees NaN).
__device__ __forceinline__ float d_max(float a, float b) { return a > b ? a : b; }
__device__ __forceinline__ double d_min(double a, double b) { return fmin(a, b); }
__device__ __forceinline__ float d_min(float a, float b) { return a < b ? a : b; }
template <typename T> __device__ __forceinline__ T pi_of();
template <> __device__ __forceinline__ double pi_of<double>() { return kPi; }
template <> __device__ __forceinline__ float pi_of<float>() { return kPiF; }

// numpy.linspace element i of n: i*step + start with the last element exactly b.
__device__ __forceinline__ double linspace_at(double a, double b, int n, int i) {
#pragma clang fp contract(off)
    if (i == n - 1) return b;
    double step = (b - a) / (double)(n - 1);
    return (double)i * step + a;
}

// Area of the intersection of two circles; common.py:36-49 (FP64, init-time tables).
__device__ __forceinline__ double cci_area(double r1, double r2, double b) {
    if (r1 < b - r2) return 0.0;
    if (r1 >= b + r2) return kPi * (r2 * r2);
    if (b - r2 <= -r1) return kPi * (r1 * r1);
    return r2 * r2 * acos((b * b + r2 * r2 - r1 * r1) / (2.0 * b * r2)) +
           r1 * r1 * acos((b * b + r1 * r1 - r2 * r2) / (2.0 * b * r1)) -
           0.5 * sqrt((-b + r2 + r1) * (b + r2 - r1) * (b - r2 + r1) * (b + r2 + r1));
}

// Lens area and kappa_0 of circles r1, r2 at separation b by the kite formula
// (Agol et al. 2020); common.py:52-73 with tsort common.py:5-33.  akite is the
// area of the kite spanned by the centres and the intersection points (0 outside
// the lens case).
template <typename T>
__device__ __forceinline__ void ccia_kite3(T r1, T r2, T b, T& area, T& kap0, T& akite_out) {
    akite_out = T(0);
    if (r1 + r2 <= b) { area = T(0); kap0 = T(0); return; }
    if (d_abs(r1 - r2) < b && b <= r1 + r2) {
        // descending sort of (r1, r2, b): x >= y >= z
        const T hi12 = d_max(r1, r2), lo12 = d_min(r1, r2);
        const T x = d_max(hi12, b);
        const T z = d_min(lo12, b);
        const T y = d_max(lo12, d_min(hi12, b));
        const T akite = T(0.5) * d_sqrt((x + (y + z)) * (z - (x - y)) * (z + (x - y)) * (x + (y - z)));
        const T k0 = d_atan2_ypos(T(2) * akite, (r2 - r1) * (r2 + r1) + b * b);
        const T k1 = d_atan2_ypos(T(2) * akite, (r1 - r2) * (r1 + r2) + b * b);
        area = r1 * r1 * k1 + r2 * r2 * k0 - akite;
        kap0 = k0;
        akite_out = akite;
        return;
    }
    if (b <= r1 - r2) { area = pi_of<T>() * (r2 * r2); kap0 = pi_of<T>(); return; }
    if (b <= r2 - r1) { area = pi_of<T>() * (r1 * r1); kap0 = T(0); return; }
    area = T(NAN); kap0 = T(NAN);
}

// Lens area of the unit disk and a disk of radius k at separation z, |1 - k| < z < 1 + k:
// the kite form above, in FP64 with the arctangent and square root of f64_*.  Products
// and sums are fused where written, so every kernel that calls it rounds alike.
__device__ __forceinline__ double lens_f64(double k, double z, double& kap0, double& akite) {
#pragma clang fp contract(off)
    const double hi = fmax(1.0, k), lo = fmin(1.0, k);
    const double x = fmax(hi, z), c = fmin(lo, z), y = fmax(lo, fmin(hi, z));
    const double sq = f64_sqrt((x + (y + c)) * (c - (x - y)) * (c + (x - y)) * (x + (y - c)));
    const double kk = (k - 1.0) * (k + 1.0);
    const double k1 = f64_atan2_ypos(sq, fma(z, z, -kk));
    kap0 = f64_atan2_ypos(sq, fma(z, z, kk));
    akite = 0.5 * sq;
    return fma(-0.5, sq, fma(k * k, kap0, k1));
}
__device__ __forceinline__ double lens_area_f64(double k, double z) {
    double kap0, akite;
    return lens_f64(k, z, kap0, akite);
}
__device__ __forceinline__ float lens_area_f32(float k, float z) {
#pragma clang fp contract(off)
    const float hi = d_max(1.0f, k), lo = d_min(1.0f, k);
    const float x = d_max(hi, z), c = d_min(lo, z), y = d_max(lo, d_min(hi, z));
    const float sq = d_sqrt((x + (y + c)) * (c - (x - y)) * (c + (x - y)) * (x + (y - c)));
    const float kk = (k - 1.0f) * (k + 1.0f);
    const float k1 = atan2_ypos_f(sq, fmaf(z, z, -kk)), k0 = atan2_ypos_f(sq, fmaf(z, z, kk));
    return fmaf(-0.5f, sq, fmaf(k * k, k0, k1));
}

// ---- One exposure sample, rounded alike in every kernel that evaluates it -------------

// Time of sample `is` (0-based) of an exposure centred at tc.
__device__ __forceinline__ double sample_time(double tc, double ext, double inv_ns, int is) {
#pragma clang fp contract(off)
    return fma(ext, fma(is + 0.5, inv_ns, -0.5), tc);
}

// Separation from the Taylor coefficients, Horner's rule in fused steps.
__device__ __forceinline__ double sample_z(double t, const double* c) {
#pragma clang fp contract(off)
    const double x = fma(fma(fma(fma(c[4], t, c[3]), t, c[2]), t, c[1]), t, c[0]);
    const double y = fma(fma(fma(fma(c[9], t, c[8]), t, c[7]), t, c[6]), t, c[5]);
    return f64_sqrt(fma(x, x, y * y));
}
__device__ __forceinline__ float sample_z(float t, const float* c) {
#pragma clang fp contract(off)
    const float x = fmaf(fmaf(fmaf(fmaf(c[4], t, c[3]), t, c[2]), t, c[1]), t, c[0]);
    const float y = fmaf(fmaf(fmaf(fmaf(c[9], t, c[8]), t, c[7]), t, c[6]), t, c[5]);
    return d_sqrt(fmaf(x, x, y * y));
}

// Mean limb darkening at g = z / (1 + k) <= 1, from the reciprocals of 1 + k and dg.
template <typename T>
__device__ __forceinline__ T sample_mean(T z, T inv_1pk, T inv_dg, const T* __restrict__ row, int ng) {
#pragma clang fp contract(off)
    const T x = z * inv_1pk * inv_dg;
    int i = (int)x;
    i = i > ng - 2 ? ng - 2 : (i < 0 ? 0 : i);
    const T a = x - (T)i, l0 = row[i], l1 = row[i + 1];
    return a * l1 + (T(1) - a) * l0;
}

template <typename T>
__device__ __forceinline__ void ccia_kite(T r1, T r2, T b, T& area, T& kap0) {
    T akite;
    ccia_kite3<T>(r1, r2, b, area, kap0, akite);
}

// Mean limb darkening for grazing parameter g; common.py:225-233.  The interval
// index is clamped to ng-2 (the reference reads lda[ng] for g in (1-1e-7, 1]).
__device__ __forceinline__ double interp_ld(double g, double dg, const double* __restrict__ row, int ng) {
    if (g < 0.0) return NAN;
    if (g > 1.0) return 0.0;
    int i = (int)floor(g / dg);
    i = i > ng - 2 ? ng - 2 : (i < 0 ? 0 : i);
    const double a = (g - i * dg) / dg;
    return (1.0 - a) * row[i] + a * row[i + 1];
}

// interp_ld with g / dg as g * (1 / dg)
__device__ __forceinline__ double interp_ld_r(double g, double dg, double inv_dg, const double* __restrict__ row, int ng) {
    if (g < 0.0) return NAN;
    if (g > 1.0) return 0.0;
    int i = (int)floor(g * inv_dg);
    i = i > ng - 2 ? ng - 2 : (i < 0 ? 0 : i);
    const double a = (g - i * dg) * inv_dg;
    return (1.0 - a) * row[i] + a * row[i + 1];
}

// FP32 form: g / dg by a multiply with 1/dg.  The lerp is continuous across
// knots, so a knot assigned to the neighbouring interval changes the value by
// rounding only.
__device__ __forceinline__ float interp_ld_f(float g, float inv_dg, const float* __restrict__ row, int ng) {
    if (g > 1.0f) return 0.0f;
    const float x = g * inv_dg;
    int i = (int)x;  // g >= 0
    i = i > ng - 2 ? ng - 2 : (i < 0 ? 0 : i);
    const float a = x - (float)i;
    const float l0 = row[i], l1 = row[i + 1];
    return fmaf(a, l1 - l0, l0);
}

// ---- Orbit: Kepler solve (orbits_py.py) and Taylor coefficients (taylor_z.py) ---------

// numpy.mod: the result has the sign of the divisor.
__device__ __forceinline__ double py_mod(double x, double y) {
    double r = fmod(x, y);
    if (r != 0.0) {
        if ((r < 0.0) != (y < 0.0)) r += y;
    } else {
        r = copysign(0.0, y);
    }
    return r;
}

// orbits_py.py:82-86
__device__ __forceinline__ double mean_anomaly_offset(double e, double w) {
    double m = atan2(sqrt(1.0 - e * e) * sin(kHalfPi - w), e + cos(kHalfPi - w));
    return m - e * sin(m);
}

// True anomaly at time t for t0 = 0: mean anomaly (orbits_py.py:115-119), Newton
// eccentric anomaly with tol 1e-8 and at most 1000 steps (:144-154), true anomaly
// (:191-196).  The Newton loop is bounded, so every lane exits.
__device__ __forceinline__ double ta_newton(double t, double p, double e, double w) {
    const double off = mean_anomaly_offset(e, w);
    const double ma = py_mod(kTwoPi * (t - (0.0 - off * p / kTwoPi)) / p, kTwoPi);
    double ea = ma, err = 0.05;
    int k = 0;
    while (fabs(err) > 1e-8 && k < 1000) {
        err = ea - e * sin(ea) - ma;
        ea = ea - err / (1.0 - e * cos(ea));
        ++k;
    }
    const double ce = cos(ea), se = sin(ea);
    const double sta = sqrt(1.0 - e * e) * se / (1.0 - e * ce);
    const double cta = (ce - e) / (1.0 - e * ce);
    return atan2(sta, cta);
}

// Sky-plane position at time t (t0 = 0) for the finite-difference stencil;
// taylor_z.py:54-76 with the orbits_py.py steps of ta_newton.  The setup kernels are
// bound by this serial chain, so the angles stay sines and cosines: the true anomaly's
// come from the eccentric anomaly's, the position's from the addition formulas, and
// sin m of the offset from its atan2's arguments, (e + sin w)^2 + (1 - e^2) cos^2 w =
// (1 + e sin w)^2.  That leaves one atan2 and, for each Newton step, one sincos of
// what were two atan2, a fmod and eleven sines and cosines (orbits
// and contacts of 1,000 pvs 9 -> 6.3 us transiting, 13 -> 8.2 us eclipsing).
__device__ __forceinline__ void kepler_xy(double t, double p, double a, double ci, double e, double w,
                                          double& x, double& y) {
    double sw, cw;
    sincos(w, &sw, &cw);
    const double q = 1.0 - e * e, sq = sqrt(q);
    const double off = atan2(sq * cw, e + sw) - e * (sq * cw / (1.0 + e * sw));
    double ma = kTwoPi * (t - (0.0 - off * p / kTwoPi)) / p;
    // py_mod; less than a turn from transit its fmod is the identity
    if (fabs(ma) < kTwoPi) ma = ma < 0.0 ? ma + kTwoPi : ma;
    else ma = py_mod(ma, kTwoPi);
    double ea = ma, err = 0.05, se, ce;
    sincos(ea, &se, &ce);
    int k = 0;
    while (fabs(err) > 1e-8 && k < 1000) {
        err = ea - e * se - ma;
        const double step = err / (1.0 - e * ce);
        ea = ea - step;
        ++k;
        if (step != 0.0) sincos(ea, &se, &ce);
    }
    const double den = 1.0 / (1.0 - e * ce);
    const double sta = sq * se * den, cta = (ce - e) * den;
    const double r = a * q / (1.0 + e * cta);
    x = -r * (cw * cta - sw * sta);
    y = -r * (sw * cta + cw * sta) * ci;
}

// Taylor coefficients from the seven stencil positions x[0..6], y[0..6] at
// t = (j-3)*dt, dt = 0.02 d; taylor_z.py:78-102.  c[0..4] is x, c[5..9] is y, each
// divided by n!; the x constant term is 0 (taylor_z.py:224).
__device__ __forceinline__ void taylor_from_stencil(const double* x, const double* y, double* c) {
    const double dt = 2e-2;
    const double a1 = 1.0 / 60, b1 = 9.0 / 60, c1 = 45.0 / 60;
    const double a2 = 1.0 / 90, b2 = 3.0 / 20, c2 = 3.0 / 2, d2 = 49.0 / 18;
    const double a3 = 1.0 / 8, b3 = 1.0, c3 = 13.0 / 8;
    const double a4 = 1.0 / 6, b4 = 2.0, c4 = 13.0 / 2, d4 = 28.0 / 3;
    const double dt2 = dt * dt, dt3 = dt2 * dt, dt4 = dt3 * dt;
    const double vx = (a1 * (x[6] - x[0]) + b1 * (x[1] - x[5]) + c1 * (x[4] - x[2])) / dt;
    const double vy = (a1 * (y[6] - y[0]) + b1 * (y[1] - y[5]) + c1 * (y[4] - y[2])) / dt;
    const double ax = (a2 * (x[0] + x[6]) - b2 * (x[1] + x[5]) + c2 * (x[2] + x[4]) - d2 * x[3]) / dt2;
    const double ay = (a2 * (y[0] + y[6]) - b2 * (y[1] + y[5]) + c2 * (y[2] + y[4]) - d2 * y[3]) / dt2;
    const double jx = (a3 * (x[0] - x[6]) + b3 * (x[5] - x[1]) + c3 * (x[2] - x[4])) / dt3;
    const double jy = (a3 * (y[0] - y[6]) + b3 * (y[5] - y[1]) + c3 * (y[2] - y[4])) / dt3;
    const double sx = (-a4 * (x[0] + x[6]) + b4 * (x[1] + x[5]) - c4 * (x[2] + x[4]) + d4 * x[3]) / dt4;
    const double sy = (-a4 * (y[0] + y[6]) + b4 * (y[1] + y[5]) - c4 * (y[2] + y[4]) + d4 * y[3]) / dt4;
    c[0] = 0.0; c[1] = vx; c[2] = 0.5 * ax; c[3] = jx / 6.0; c[4] = sx / 24.0;
    c[5] = y[3]; c[6] = vy; c[7] = 0.5 * ay; c[8] = jy / 6.0; c[9] = sy / 24.0;
}

// Separation z(t) from the Taylor coefficients by Horner's rule (sep_c).
template <typename T>
__device__ __forceinline__ T taylor_z(T t, const T* c) {
    const T px = (((c[4] * t + c[3]) * t + c[2]) * t + c[1]) * t + c[0];
    const T py = (((c[9] * t + c[8]) * t + c[7]) * t + c[6]) * t + c[5];
    return d_sqrt(px * px + py * py);
}

// `v` of lane q of the caller's quad (four neighbouring lanes, all active).
template <int q>
__device__ __forceinline__ double quad_lane(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x55 * q, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x55 * q, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// Contact time by bisection, tol 1e-6 d and at most 100 steps; taylor_z.py:298-328.
// point 1 or 4 (first/fourth contact, z = 1+k).  The first bracket is [0, s 2/v]
// with s = -1 before mid-transit and +1 after; the reference takes v = vx, the
// sky-plane x velocity (positive at a transit).  The eclipse path passes |vx|:
// behind the star the planet moves in -x, and v = vx would put first contact after
// mid-eclipse.
// Called by the four lanes of a quad with the same arguments.  A step is a chain of
// some 25 dependent FP64 operations, so two steps share one: the lanes evaluate the
// next midpoint and both that can follow it, and the brackets taken are the
// bisection's own.  The sign of z - zt is taken from z^2 - zt^2, without the root.
__device__ __forceinline__ double contact_bisect(double k, int point, const double* c, double v) {
    const double s = point == 1 ? -1.0 : 1.0;
    const double zt = 1.0 + k, zt2 = zt * fabs(zt);
    const int lane = threadIdx.x & 3;
    auto above = [&](double t) {
        const double tt = t - floor(t + 0.5);   // z_taylor_s with p = 1; taylor_z.py:198-226
        const double x = (((c[4] * tt + c[3]) * tt + c[2]) * tt + c[1]) * tt + c[0];
        const double y = (((c[9] * tt + c[8]) * tt + c[7]) * tt + c[6]) * tt + c[5];
        return x * x + y * y - zt2;
    };
    double t0 = 0.0;
    double t2 = s * 2.0 / v;
    double t1 = 0.5 * t2;
    double d0 = above(lane == 0 ? t0 : t1);
    double d1 = quad_lane<1>(d0);
    d0 = quad_lane<0>(d0);
    int i = 0;
    while (fabs(t2 - t0) > 1e-6 && i < 100) {
        if (d0 * d1 < 0.0) {
            t2 = t1;
        } else {
            t0 = t1;
            d0 = d1;
        }
        t1 = 0.5 * (t0 + t2);
        ++i;
        const double tl = 0.5 * (t0 + t1), tr = 0.5 * (t1 + t2);
        const double d = above(lane == 1 ? tl : (lane == 2 ? tr : t1));
        d1 = quad_lane<0>(d);
        if (!(fabs(t2 - t0) > 1e-6 && i < 100)) break;
        if (d0 * d1 < 0.0) {
            t2 = t1;
            t1 = tl;
            d1 = quad_lane<1>(d);
        } else {
            t0 = t1;
            t1 = tr;
            d0 = d1;
            d1 = quad_lane<2>(d);
        }
        ++i;
    }
    return t1;
}

__device__ __forceinline__ double find_contact_point(double k, int point, const double* c) {
    return contact_bisect(k, point, c, c[1]);
}

// ---- Epoch reduction (model_full.py:88-89) -------------------------------------------

// Division-free form of epoch = floor((t - t0 + p/2) / p), tc = t - (t0 + epoch*p): the
// epoch from a multiply by 1/p, then one correction step so that
// r = (t - t0 + p/2) - epoch*p lies in [0, p), or in (p, 0] for a negative period, with no
// contraction so each step rounds as in numpy.  It can differ from the division only
// where the quotient is within rounding of an integer, i.e. at tc = +-p/2, far outside
// any transit window.
__device__ __forceinline__ double epoch_phase(double t, double t0, double p, double inv_p, double& epoch) {
#pragma clang fp contract(off)
    const double u = t - t0 + 0.5 * p;
    double ep = floor(u * inv_p);
    const double r = u - ep * p;
    // r / p has the sign of r with p's sign taken off
    const double rs = __hiloint2double(__double2hiint(r) ^ (__double2hiint(p) & (int)0x80000000), __double2loint(r));
    ep += (rs < 0.0) ? -1.0 : ((rs >= fabs(p)) ? 1.0 : 0.0);
    epoch = ep;
    return t - (t0 + ep * p);
}

// ---- Limb-darkening laws; models/numba/ldmodels.py:22-139 -----------------------------

__device__ __forceinline__ double ld_law(int law, double mu, const double* c, int nc) {
    switch (law) {
        case RR_LD_UNIFORM: return 1.0;
        case RR_LD_LINEAR: return 1.0 - c[0] * (1.0 - mu);
        case RR_LD_QUADRATIC: return 1.0 - c[0] * (1.0 - mu) - c[1] * ((1.0 - mu) * (1.0 - mu));
        case RR_LD_QUADRATIC_TRI: {
            const double a = sqrt(c[0]), b = 2.0 * c[1];
            const double u = a * b, v = a * (1.0 - b);
            return 1.0 - u * (1.0 - mu) - v * ((1.0 - mu) * (1.0 - mu));
        }
        case RR_LD_NONLINEAR: {
            // mu^1.5 as mu * sqrt(mu): within 2 ulp of pow
            const double sm = sqrt(mu);
            return 1.0 - c[0] * (1.0 - sm) - c[1] * (1.0 - mu) - c[2] * (1.0 - mu * sm) - c[3] * (1.0 - mu * mu);
        }
        case RR_LD_GENERAL: {
            double s = 0.0, mp = mu;  // mp = mu^(i+1) by repeated products
            for (int i = 0; i < nc; ++i, mp *= mu) s += c[i] * (1.0 - mp);
            return s;
        }
        case RR_LD_SQUARE_ROOT: return 1.0 - c[0] * (1.0 - mu) - c[1] * (1.0 - sqrt(mu));
        case RR_LD_LOGARITHMIC: return 1.0 - c[0] * (1.0 - mu) - c[1] * mu * log(mu);
        case RR_LD_EXPONENTIAL: return 1.0 - c[0] * (1.0 - mu) - c[1] / (1.0 - exp(mu));
        case RR_LD_POWER_2: return 1.0 - c[0] * (1.0 - pow(mu, c[1]));
        case RR_LD_POWER_2_PM: {
            const double cc = 1.0 - c[0] + c[1];
            const double a = log2(cc / c[1]);
            return 1.0 - cc * (1.0 - pow(mu, a));
        }
        default: return NAN;
    }
}

// ---- Laws that are linear in their coefficients -------------------------------------
//
// I(mu) = sum_i coef_i(c) B_i(mu) for every named law but power-2, power-2-pm and
// tabulated profiles: the constant and the coefficient terms of ldmodels.py:22-113.
// Then every linear functional of the profile (its limb-darkening means, its disk
// integral) of any passband is the same combination of the functional of the
// basis, which a pv computes once for all its passbands.
constexpr int kMaxBasis = 6;

// Number of basis functions of the law, 0 when it is not linear in its coefficients.
__host__ __device__ inline int ld_basis_count(int law, int nc) {
    switch (law) {
        case RR_LD_UNIFORM: return 1;
        case RR_LD_LINEAR: return 2;
        case RR_LD_QUADRATIC:
        case RR_LD_QUADRATIC_TRI:
        case RR_LD_SQUARE_ROOT:
        case RR_LD_LOGARITHMIC:
        case RR_LD_EXPONENTIAL: return 3;
        case RR_LD_NONLINEAR: return 5;
        case RR_LD_GENERAL: return nc >= 1 && nc <= kMaxBasis ? nc : 0;
        default: return 0;
    }
}

// B_i(mu), in the form of the matching term of ld_law.
__device__ __forceinline__ double ld_basis(int law, int i, double mu) {
    if (law == RR_LD_GENERAL) {
        double mp = mu;  // mu^(i+1) by repeated products
        for (int j = 0; j < i; ++j) mp *= mu;
        return 1.0 - mp;
    }
    if (i == 0) return 1.0;
    switch (law) {
        case RR_LD_LINEAR: return 1.0 - mu;
        case RR_LD_QUADRATIC:
        case RR_LD_QUADRATIC_TRI: return i == 1 ? 1.0 - mu : (1.0 - mu) * (1.0 - mu);
        case RR_LD_NONLINEAR: {
            const double sm = sqrt(mu);
            return i == 1 ? 1.0 - sm : (i == 2 ? 1.0 - mu : (i == 3 ? 1.0 - mu * sm : 1.0 - mu * mu));
        }
        case RR_LD_SQUARE_ROOT: return i == 1 ? 1.0 - mu : 1.0 - sqrt(mu);
        case RR_LD_LOGARITHMIC: return i == 1 ? 1.0 - mu : mu * log(mu);
        case RR_LD_EXPONENTIAL: return i == 1 ? 1.0 - mu : 1.0 / (1.0 - exp(mu));
        default: return NAN;
    }
}

// coef_i of the coefficients c[0..nc).
__device__ __forceinline__ double ld_basis_coef(int law, int i, const double* c) {
    switch (law) {
        case RR_LD_GENERAL: return c[i];
        case RR_LD_QUADRATIC_TRI: {
            if (i == 0) return 1.0;
            const double a = sqrt(c[0]), b = 2.0 * c[1];
            return i == 1 ? -(a * b) : -(a * (1.0 - b));
        }
        default: return i == 0 ? 1.0 : -c[i - 1];
    }
}

// Analytic disk integral where the reference has one (ldmodels.py:27-123); false
// for the laws that use the 200-node trapezoid (rrmodel.py:220-227, Q8).
__device__ __forceinline__ bool ld_integral(int law, const double* c, double& out) {
    switch (law) {
        case RR_LD_UNIFORM: out = kPi; return true;
        case RR_LD_LINEAR: out = 2.0 * kPi * 1.0 / 6.0 * (3.0 - 2.0 * c[0]); return true;  // Q7, as the reference
        case RR_LD_QUADRATIC: out = 2.0 * kPi * 1.0 / 12.0 * (-2.0 * c[0] - c[1] + 6.0); return true;
        case RR_LD_QUADRATIC_TRI: {
            const double a = sqrt(c[0]), b = 2.0 * c[1];
            const double u = a * b, v = a * (1.0 - b);
            out = 2.0 * kPi * 1.0 / 12.0 * (-2.0 * u - v + 6.0);
            return true;
        }
        case RR_LD_POWER_2: out = 2.0 * kPi * (-c[0] * c[1] + c[1] + 2.0) / (2.0 * c[1] + 4.0); return true;
        default: return false;
    }
}

// One trapezoid segment m (1..199) of 2*pi*trapz(z*I(mu), z) on mu = linspace(1, 0, 200).
__device__ __forceinline__ double ld_trapz_segment(int law, const double* c, int nc, int m) {
    const double mu1 = linspace_at(1.0, 0.0, 200, m), mu0 = linspace_at(1.0, 0.0, 200, m - 1);
    const double z1 = sqrt(1.0 - mu1 * mu1), z0 = sqrt(1.0 - mu0 * mu0);
    return (z1 - z0) * (z1 * ld_law(law, mu1, c, nc) + z0 * ld_law(law, mu0, c, nc)) / 2.0;
}

// ---- Orbit for 8 parameter vectors per 64-lane block: lane j (0..6) of a group of 8
// solves Kepler at t = (j-3)*dt, lane 0 forms the stencils, lanes 0-3 and 4-7 find
// the first and fourth contacts.  Writes coefficients[10] and the window.
constexpr int kOrbitGroup = 8;

constexpr int kOrbitLds = kOrbitGroup * (8 + 8 + 10 + 2);  // doubles of LDS per block

// `sm` is block-shared storage of kOrbitLds doubles.
__device__ __forceinline__ void orbit_group(int pv, bool valid, double p, double a, double inc, double e, double w,
                                            double kw, double* out_c, double* out_win, double* sm) {
    const int sub = threadIdx.x / kOrbitGroup, j = threadIdx.x % kOrbitGroup;
    double* s_x = sm + sub * 8;
    double* s_y = sm + kOrbitGroup * 8 + sub * 8;
    double* s_c = sm + kOrbitGroup * 16 + sub * 10;
    double* s_w = sm + kOrbitGroup * 26 + sub * 2;
    if (valid && j < 7) {
        double x, y;
        kepler_xy((j - 3) * 2e-2, p, a, cos(inc), e, w, x, y);
        s_x[j] = x;
        s_y[j] = y;
    }
    __syncthreads();
    if (valid && j == 0) taylor_from_stencil(s_x, s_y, s_c);
    __syncthreads();
    if (valid) {
        const double tc = find_contact_point(kw, j < 4 ? 1 : 4, s_c);
        if ((j & 3) == 0) s_w[j >> 2] = tc;
    }
    __syncthreads();
    if (valid) {
        out_c[j] = s_c[j];
        if (j < 2) out_c[8 + j] = s_c[8 + j];
        if (j < 2) out_win[j] = s_w[j];
    }
}

// Workgroups are dealt to the 8 XCDs of the chip round-robin (XCD = blockIdx % 8).
// Block b is given work item xcd_remap(b, n) instead, so that each XCD works through
// one contiguous eighth of the n items: a pattern in the item order (a transit in the
// first tile of every pv, say) is spread over all XCDs rather than landing on the few
// that the round-robin assigns it to, and an XCD's L2 keeps the pvs it works on.
// A bijection of [0, n).
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_remap(int b, int n) {
    const int x = b % kXcds, j = b / kXcds;
    const int per = n / kXcds, r = n % kXcds;
    return x * per + min(x, r) + j;
}

// Sum over a wavefront (64 lanes) by butterfly shuffles; every lane gets the total.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// 2*pi*trapz(z*I(mu), z) on mu = linspace(1, 0, 200) (rrmodel.py:151-152,220-227) by a
// whole wavefront, for the profile I = f(mu).  Each node's value z*I(mu) is computed
// once into `s_y` (kTrapzNodes doubles of LDS), then segment m pairs node m with node
// m-1, each lane summing its segments in node order before the wave sum.  Staging
// the values in LDS keeps the law's evaluation (an FP64 pow for the power laws) out
// of the summation loop, whose registers would otherwise spill.  Every lane of the
// block must call it (it holds two barriers).
constexpr int kTrapzNodes = 200;
template <class F>
__device__ __forceinline__ double trapz_disk_wave(F f, double* s_y) {
    const int lane = threadIdx.x & 63;
    for (int m = lane; m < kTrapzNodes; m += 64) {
        const double mu = linspace_at(1.0, 0.0, kTrapzNodes, m);
        s_y[m] = sqrt(1.0 - mu * mu) * f(mu);
    }
    __syncthreads();
    double part = 0.0;
    for (int m = lane; m < kTrapzNodes; m += 64) {
        if (m >= 1) {
            const double mu = linspace_at(1.0, 0.0, kTrapzNodes, m);
            const double ml = linspace_at(1.0, 0.0, kTrapzNodes, m - 1);
            const double z = sqrt(1.0 - mu * mu), zl = sqrt(1.0 - ml * ml);
            part += (z - zl) * (s_y[m] + s_y[m - 1]) / 2.0;
        }
    }
    __syncthreads();
    return 2.0 * kPi * wave_sum(part);
}

// The disk integral of a law's profile, and of its basis function i.
__device__ __forceinline__ double ld_trapz_wave(int law, const double* c, int nc, double* s_y) {
    return trapz_disk_wave([&](double mu) { return ld_law(law, mu, c, nc); }, s_y);
}
__device__ __forceinline__ double ld_basis_trapz_wave(int law, int i, double* s_y) {
    return trapz_disk_wave([&](double mu) { return ld_basis(law, i, mu); }, s_y);
}

}  // namespace rr
