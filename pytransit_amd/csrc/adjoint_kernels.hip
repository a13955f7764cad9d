// Gaussian log-likelihood of the RoadRunner model and its gradient (hand-written
// adjoint) for one light curve, fused so the flux is never written.
//
//   lnL(pv) = sum_t [ -ln sigma - 1/2 ln 2pi - 1/2 ((o_t - m_t)/sigma)^2 ]
// (the form of lnlike_normal, pytransit/lpf/loglikelihood/wnloglikelihood.py:22-35)
// and d lnL / d(k, t0, p, a, i, c0, c1) with c the two limb-darkening coefficients
// of the quadratic or power-2 law.  The model m_t is rr_full's (model_full.py:
// 75-99); its derivatives follow the chain
//   m <- (I(g), A(k, z)) <- z(Taylor series of the orbit) <- coefficients(p, a, i)
//   and phase tc(t0, p),  I <- table lerp in k and g, ldp(c), istar(c).
// Coefficient derivatives are exact derivatives of the finite-difference stencil
// (taylor_z.py:23-102): d/da = c/a, d/di scales the y row by -tan(i), and d/dp
// propagates dM/dp = -2 pi t / p^2 through Kepler's equation at the converged
// solution, df/dM = (1 + e cos f)^2 / (1 - e^2)^(3/2).  Lens area: dA/dz = -2 a_kite / z (minus the
// chord), dA/dk = 2 k kappa0.  Points outside the window have m = 1 and zero
// gradient.  FP64 epoch reduction and accumulation; per-sample arithmetic in
// Real (float for RR_MIXED, double for RR_FP64).
//
// Kernels (rr_lnlike_vec):
//   rr_lnlike_setup_kernel   orbits of 8 pvs a block, a pv's limb-darkening rows a block,
//                            and each tile's sum of (o - 1)^2
//   rr_lnlike_kernel         (pv, range of times) a block: window test of tiles, queue of
//                            the points in the window, samples, block sums
//   rr_lnlike_reduce_kernel  the blocks' sums of a pv, where a light curve is split
// One block per pv did all of it before: the setup idled three of its four waves for
// 10-15 us, every pv read every time, a population of 250 left the chip two thirds
// empty and the gradient was computed whether asked for or not.  250 pv x 18,000 t over
// 24 d, nss 5, FP64, value only: 50 -> 8 + 13 + 4 us; 2048 pv x 10,000 t, 22 % in the
// window, nss 5, mixed, with the gradient: 125 -> 14 + 72 us, VALU-bound (about 150
// instructions a sample at 128 registers).
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "rr_device.hpp"
#include "rr_internal.hpp"

namespace rr {

// A per-pv input: element i at p[i * stride] (stride 0: one value for every pv), or the
// value v where there is no array.  The callers' strided columns and plain numbers are
// read as they are, without a copy or an upload for each.
struct LnlVec {
    const double* p;
    long long stride;
    double v;
    __device__ __forceinline__ double at(int i, int off = 0) const { return p ? p[i * stride + off] : v; }
};

// Per-pv state between the setup and the main kernel.
struct alignas(16) LnlRec {
    double c[20];                  // orbit coefficients, then their period derivatives
    double lo, hi;                 // the window
    double k, t0, p, inv_p, inv_a, tan_i;
    double ist, dist0, dist1;      // disk integral and its coefficient derivatives
    int32_t orbit_ok, ld_ok;
};
static_assert(sizeof(LnlRec) == 256, "LnlRec must be 256 bytes");

struct LnlArgs {
    const double* times; const double* obs;
    const int32_t* nsamples; const double* exptimes; const int32_t* epids;
    LnlVec k, t0, p, a, inc, e, w, sigma, c0, c1;
    const double* W; const double* mu;
    double* lnl; double* grad;
    LnlRec* rec; void* rows; double* tsum; double* part;
    int law, npv, npt, t0cols, nk, ng, nz;
    int sorted;        // times non-decreasing: tiles outside the window are skipped
    int ntile, per, nsplit;   // tiles of the light curve, tiles per block, blocks per pv
    double kmin, kmax, dk, dg;
};

constexpr int kLnlThreads = 256;
constexpr int kLnlTile = 256;     // times of a tile
constexpr int kLnlMaxNg = 512;
constexpr int kLnlMaxNz = 1024;
constexpr int kLnlQueue = 5 * kLnlTile;

// A pv's limb-darkening rows: L and, for the gradient, dL/dk, dL/dc0 and dL/dc1.
// FP64: per interval of g each row's value at the left knot and its rise to the right
// one.  FP32: per knot the rows' values (one 16-byte read), then, for the gradient, the
// g slope of each interval from the FP64 means: the difference of two rounded values
// would lose ~1e-5 of the slope, which the t0, p, a and i gradients carry through the
// chain rule.
template <typename Real, bool kGrad>
__host__ __device__ inline int lnl_rows_count(int ng) {
    if (sizeof(Real) == 4) return kGrad ? 5 * ng : ng;
    return (ng - 1) * (kGrad ? 8 : 2);
}
template <typename Real, bool kGrad>
__host__ __device__ inline size_t lnl_rows_bytes(int ng) {
    return ((size_t)lnl_rows_count<Real, kGrad>(ng) * sizeof(Real) + 15) / 16 * 16;
}

// Position at stencil time t and its derivative with respect to the period:
// dM/dp = -2 pi t / p^2 (t0 = 0) and df/dM = (1 + e cos f)^2 / (1 - e^2)^(3/2).
__device__ void kepler_xy_dp(double t, double p, double a, double ci, double e, double w, double& x, double& y,
                             double& dxdp, double& dydp) {
    const double f = ta_newton(t, p, e, w);
    const double ecf = 1.0 + e * cos(f);
    const double om = 1.0 - e * e;
    const double df_dp = (ecf * ecf / (om * sqrt(om))) * (-kTwoPi * t / (p * p));
    const double r = a * om / ecf;
    const double dr_df = r * e * sin(f) / ecf;
    const double cw = cos(w + f), sw = sin(w + f);
    x = -r * cw;
    y = -r * sw * ci;
    dxdp = (-dr_df * cw + r * sw) * df_dp;
    dydp = (-dr_df * sw - r * cw) * ci * df_dp;
}

__device__ __forceinline__ double dld_dc(int law, double mu, const double* c, int j) {
    if (law == RR_LD_QUADRATIC) return j == 0 ? -(1.0 - mu) : -((1.0 - mu) * (1.0 - mu));
    if (law == RR_LD_POWER_2) {
        const double ma = pow(mu, c[1]);
        return j == 0 ? -(1.0 - ma) : c[0] * ma * log(mu);
    }
    return 0.0;
}

__device__ __forceinline__ double distar_dc(int law, const double* c, int j) {
    if (law == RR_LD_QUADRATIC) return j == 0 ? -kPi / 3.0 : -kPi / 6.0;
    if (law == RR_LD_POWER_2) {
        const double d = 2.0 * c[1] + 4.0;
        return j == 0 ? 2.0 * kPi * (-c[1]) / d : -8.0 * kPi * c[0] / (d * d);
    }
    return 0.0;
}

template <typename Real>
__device__ __forceinline__ Real horner5(const Real* c, Real t) {
    return (((c[4] * t + c[3]) * t + c[2]) * t + c[1]) * t + c[0];
}
template <typename Real>
__device__ __forceinline__ Real dhorner5(const Real* c, Real t) {
    return ((Real(4) * c[4] * t + Real(3) * c[3]) * t + Real(2) * c[2]) * t + c[1];
}

// a times the hardware's reciprocal of a divisor: the bits of the FP32 quotient without
// its exponent scaling, and never fused into a following sum.
__device__ __forceinline__ float f32_quotient(float a, float rcp) {
#pragma clang fp contract(off)
    return a * rcp;
}

// Lens area of the unit disk and a disk of radius k < 1 at separation z, in the
// lens case |z - 1| < k, from u = z - 1 given to full FP32 precision.  With the
// kite area written as akite = z sin kappa1 (Heron), the kite form
// A = kappa1 + k^2 kappa0 - akite becomes
//   A = k^2 kappa0 + S(kappa1) - u akite / z,   S(x) = x - sin x,
// so a small planet's nearly equal kappa1 and akite are not subtracted (in FP32
// that cancellation leaves ~1e-7 of the area's scale, 0.1 k); S is its Taylor
// series up to x^11 for kappa1 <= 0.6 (truncation < 1e-13), the kite form above
// it.  The kite's square root is ((1 + z)^2 - k^2)(k^2 - u^2), the sorted-sides
// product of common.py:5-33,52-73 regrouped, and z^2 - 1 = u (2 + u).  Returns A,
// kappa0 and akite.
__device__ __forceinline__ void lens_seg_f32(float k, float z, float inv_z, float u, float& area, float& kap0,
                                             float& akite) {
    const float zp1 = 1.0f + z;
    const float sq = __builtin_amdgcn_sqrtf((zp1 * zp1 - k * k) * ((k - u) * (k + u)));  // 2 akite
    const float zm = u * (2.0f + u);                                                     // z^2 - 1
    kap0 = atan2_ypos_f(sq, zm + k * k);
    const float kap1 = atan2_ypos_f(sq, 2.0f + zm - k * k);
    akite = 0.5f * sq;
    if (kap1 <= 0.6f) {
        const float x2 = kap1 * kap1;
        float sr = 1.0f / 39916800.0f;
        sr = fmaf(sr, x2, -1.0f / 362880.0f);
        sr = fmaf(sr, x2, 1.0f / 5040.0f);
        sr = fmaf(sr, x2, -1.0f / 120.0f);
        sr = fmaf(sr, x2, 1.0f / 6.0f);
        area = d_fma(k * k, kap0, kap1 * x2 * sr) - f32_quotient(u * akite, inv_z);
    } else {
        area = kap1 + k * k * kap0 - akite;
    }
}

// ---- per-pv setup ---------------------------------------------------------------------

constexpr int kLnlOrbitLds = kOrbitGroup * (4 * 8 + 20 + 2);   // doubles

// Orbit, its period derivative and the window of a pv by a group of 8 lanes (sub: the
// group, j: its lane); every thread of the block calls it (barriers).
template <bool kGrad>
__device__ __forceinline__ void lnl_orbit(const LnlArgs& s, int pv, bool active, int sub, int j, LnlRec* rec, double* sm) {
    double* s_x = sm + sub * 32;       // x, y, dx, dy at the seven stencil times
    double* s_c = sm + kOrbitGroup * 32 + sub * 20;
    double* s_w = sm + kOrbitGroup * 52 + sub * 2;
    const int q = active ? pv : 0;
    const double p = s.p.at(q), a = s.a.at(q), inc = s.inc.at(q), e = s.e.at(q), w = s.w.at(q), k = s.k.at(q);
    const bool valid = active && !(isnan(a) || a <= 1.0 || e < 0.0);
    if (valid && j < 7) {
        if (kGrad) kepler_xy_dp((j - 3) * 2e-2, p, a, cos(inc), e, w, s_x[j], s_x[8 + j], s_x[16 + j], s_x[24 + j]);
        else kepler_xy((j - 3) * 2e-2, p, a, cos(inc), e, w, s_x[j], s_x[8 + j]);
    }
    __syncthreads();
    if (valid && j < (kGrad ? 2 : 1)) taylor_from_stencil(s_x + 16 * j, s_x + 16 * j + 8, s_c + 10 * j);
    __syncthreads();
    if (valid) {
        const double tc = find_contact_point(k, j < 4 ? 1 : 4, s_c);
        if ((j & 3) == 0) s_w[j >> 2] = tc;
    }
    __syncthreads();
    if (!active) return;
    if (valid)
        for (int m = j; m < (kGrad ? 20 : 10); m += 8) rec->c[m] = s_c[m];
    if (j == 0) {
        const double ext = s.exptimes[0];
        // the light curve's epoch column, clamped as the evaluate path does
        const int ep = min(max(s.epids[0], 0), s.t0cols - 1);
        rec->lo = valid ? s_w[0] - (0.003 + ext) : 0.0;
        rec->hi = valid ? s_w[1] + (0.003 + ext) : 0.0;
        rec->k = k;
        rec->t0 = s.t0.at(q, ep);
        rec->p = p;
        rec->inv_p = 1.0 / p;
        rec->inv_a = 1.0 / a;
        rec->tan_i = tan(inc);
        rec->orbit_ok = valid ? 1 : 0;
    }
}

// The limb-darkening intervals of a pv by NT threads: the profile and its coefficient
// derivatives at the mu nodes in LDS, the table's two rows of k contracted with them
// (lanes over g), then the intervals.  `sm`: lnl_ld_lds doubles.
template <bool kGrad> __host__ __device__ inline int lnl_ld_lds(int nz, int ng) { return (kGrad ? 3 : 1) * nz + (kGrad ? 4 : 1) * ng; }

// The rows' means at every g: V neighbouring g a lane, eight mu nodes' loads together.
template <bool kGrad, int V, int NT>
__device__ __forceinline__ void lnl_contract(const LnlArgs& s, int ik, double ak, const double* s_l, double* s_m) {
    typedef double vec __attribute__((ext_vector_type(V)));
    constexpr int kP = kGrad ? 3 : 1;
    constexpr int kB = 8;
    const int nz = s.nz, ng = s.ng;
    for (int iv = threadIdx.x; iv < ng / V; iv += NT) {
        const double* w0 = s.W + (size_t)ik * nz * ng + V * iv;
        const double* w1 = w0 + (size_t)nz * ng;
        double a0[kP][V], a1[kP][V];
#pragma unroll
        for (int m = 0; m < kP; ++m)
#pragma unroll
            for (int e = 0; e < V; ++e) a0[m][e] = a1[m][e] = 0.0;
        for (int iz0 = 0; iz0 < nz; iz0 += kB) {
            vec u0[kB], u1[kB];
#pragma unroll
            for (int u = 0; u < kB; ++u) {
                const size_t o = (size_t)min(iz0 + u, nz - 1) * ng;
                u0[u] = *(const vec*)(w0 + o);
                u1[u] = *(const vec*)(w1 + o);
            }
#pragma unroll
            for (int u = 0; u < kB; ++u) {
                if (iz0 + u < nz) {
#pragma unroll
                    for (int m = 0; m < kP; ++m)
#pragma unroll
                        for (int e = 0; e < V; ++e) {
                            a0[m][e] += u0[u][e] * s_l[m * nz + iz0 + u];
                            a1[m][e] += u1[u][e] * s_l[m * nz + iz0 + u];
                        }
                }
            }
        }
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const int ig = V * iv + e;
            s_m[ig] = (1.0 - ak) * a0[0][e] + ak * a1[0][e];
            if constexpr (kGrad) {
                s_m[ng + ig] = (a1[0][e] - a0[0][e]) / s.dk;
                s_m[2 * ng + ig] = (1.0 - ak) * a0[1][e] + ak * a1[1][e];
                s_m[3 * ng + ig] = (1.0 - ak) * a0[2][e] + ak * a1[2][e];
            }
        }
    }
}

template <typename Real, bool kGrad, int NT>
__device__ __forceinline__ void lnl_rows(const LnlArgs& s, int pv, LnlRec* rec, Real* rows, double* sm) {
    constexpr int kP = kGrad ? 3 : 1;
    const int tid = threadIdx.x, nz = s.nz, ng = s.ng;
    double* s_l = sm;                  // [kP][nz]
    double* s_m = sm + kP * nz;        // [kGrad ? 4 : 1][ng]
    const double c[2] = {s.c0.at(pv), s.c1.at(pv)};
    const double kk = s.k.at(pv);
    for (int iz = tid; iz < nz; iz += NT) {
        const double mu = s.mu[iz];
        s_l[iz] = ld_law(s.law, mu, c, 2);
        if (kGrad) {
            s_l[nz + iz] = dld_dc(s.law, mu, c, 0);
            s_l[2 * nz + iz] = dld_dc(s.law, mu, c, 1);
        }
    }
    const bool in_table = s.kmin <= kk && kk <= s.kmax;
    int ik = 0;
    double ak = 0.0;
    if (in_table) {
        ik = (int)floor((kk - s.kmin) / s.dk);
        ik = ik > s.nk - 2 ? s.nk - 2 : ik;
        ak = (kk - s.kmin - ik * s.dk) / s.dk;
    }
    __syncthreads();
    if (tid == 0) {
        double ist = NAN;
        ld_integral(s.law, c, ist);    // analytic for both laws
        rec->ist = ist;
        rec->dist0 = distar_dc(s.law, c, 0);
        rec->dist1 = distar_dc(s.law, c, 1);
        rec->ld_ok = (in_table && !isnan(s_l[0])) ? 1 : 0;
    }
    // two neighbouring g a lane (16-byte loads) where the table's rows allow it
    if (ng % 2 == 0 && ((uintptr_t)s.W & 15) == 0) lnl_contract<kGrad, 2, NT>(s, ik, ak, s_l, s_m);
    else lnl_contract<kGrad, 1, NT>(s, ik, ak, s_l, s_m);
    __syncthreads();
    constexpr int kR = kGrad ? 4 : 1;
    if constexpr (std::is_same<Real, float>::value) {
        for (int i = tid; i < kR * ng; i += NT) rows[i] = (float)s_m[(i % kR) * ng + i / kR];
        if (kGrad)
            for (int ig = tid; ig < ng - 1; ig += NT) rows[kR * ng + ig] = (float)((s_m[ig + 1] - s_m[ig]) / s.dg);
    } else {
        for (int i = tid; i < (ng - 1) * 2 * kR; i += NT) {
            const int ig = i / (2 * kR), m = i - ig * 2 * kR, r = (m >> 1) * ng + ig;
            rows[i] = (m & 1) ? s_m[r + 1] - s_m[r] : s_m[r];
        }
    }
}

// Blocks of 64: the orbits of 8 pvs, then one per pv for its limb-darkening intervals,
// then one per tile of times for its sum of (o - 1)^2 (a tile outside a pv's window
// adds that to the pv's chi^2 without being read again).
template <typename Real, bool kGrad>
__global__ void __launch_bounds__(64) rr_lnlike_setup_kernel(LnlArgs s) {
    extern __shared__ __align__(16) unsigned char lds[];
    double* sm = (double*)lds;
    const int nob = (s.npv + kOrbitGroup - 1) / kOrbitGroup;
    const int b = blockIdx.x;
    if (b < nob) {
        const int sub = threadIdx.x / kOrbitGroup, pv = b * kOrbitGroup + sub;
        lnl_orbit<kGrad>(s, pv, pv < s.npv, sub, threadIdx.x % kOrbitGroup, s.rec + pv, sm);
    } else if (b < nob + s.npv) {
        const int pv = b - nob;
        lnl_rows<Real, kGrad, 64>(s, pv, s.rec + pv, (Real*)((char*)s.rows + pv * lnl_rows_bytes<Real, kGrad>(s.ng)), sm);
    } else {
        const int t = b - nob - s.npv;
        double v = 0.0;
#pragma unroll
        for (int j = 0; j < kLnlTile / 64; ++j) {
            const int it = t * kLnlTile + j * 64 + threadIdx.x;
            const double om1 = it < s.npt ? s.obs[it] - 1.0 : 0.0;
            v += om1 * om1;
        }
        v = wave_sum(v);
        if (threadIdx.x == 0) s.tsum[t] = v;
    }
}

// ---- samples --------------------------------------------------------------------------

typedef float f32x4 __attribute__((ext_vector_type(4)));

// A pv's constants of the sample loop in the working precision.
template <typename Real>
struct LnlPv {
    Real cx[5], cy[5], dcx[5], dcy[5];
    double c0, c1, c5, c6;         // constant and linear terms of the position in FP64
    double g_scale, dg;            // g / dg = z g_scale
    Real k, zlim, inv1pk, inv_dg, tan_i, inv_a, pik2, dpik2;
};

// Sums over a point's samples: I A and its derivatives by k, t0, p, a, i, c0, c1.
template <typename Real, bool kGrad>
struct LnlSums {
    Real v[kGrad ? 8 : 1];
};

// A sample's terms of these sums as the factors of their products, so that a sum takes
// the same fused steps whichever lane evaluated the sample: I, A, then the k derivative,
// G = dI/dz A + I dA/dz, dz by t0, p, a and i, and dI by c0 and c1.
template <typename Real, bool kGrad>
struct LnlTerm {
    static constexpr int kN = kGrad ? 10 : 2;
    Real f[kN];
};

template <typename Real, bool kGrad>
__device__ __forceinline__ void lnl_add(LnlSums<Real, kGrad>& d, const LnlTerm<Real, kGrad>& t) {
    d.v[0] = d_fma(t.f[0], t.f[1], d.v[0]);
    if constexpr (kGrad) {
        d.v[1] += t.f[2];
#pragma unroll
        for (int m = 0; m < 4; ++m) d.v[2 + m] = d_fma(t.f[3], t.f[4 + m], d.v[2 + m]);
        d.v[6] = d_fma(t.f[8], t.f[1], d.v[6]);
        d.v[7] = d_fma(t.f[9], t.f[1], d.v[7]);
    }
}

// One sample; `d` keeps its zeros where the planet is off the disk.
template <typename Real, bool kGrad>
__device__ __forceinline__ void lnl_sample(const LnlPv<Real>& v, const Real* rows, int ng, double taud, Real ep,
                                           LnlTerm<Real, kGrad>& d) {
    constexpr bool kMixed = std::is_same<Real, float>::value;
    const Real tau = (Real)taud;
    Real x, y, z, u, inv_z;
    if constexpr (kMixed) {
        // the constant and linear terms of the position in FP64: the phase resolves
        // ~1e-9 d that an FP32 time would drop, ~1e-7 of the position at sky speeds of
        // ~40 stellar radii per day.  z - 1 is formed from the FP64 squared distance,
        // so the lens area below does not see the rounding of z.
        const Real t2 = tau * tau;
        const double xd = v.c0 + v.c1 * taud + (double)(((v.cx[4] * tau + v.cx[3]) * tau + v.cx[2]) * t2);
        const double yd = v.c5 + v.c6 * taud + (double)(((v.cy[4] * tau + v.cy[3]) * tau + v.cy[2]) * t2);
        const double s2 = xd * xd + yd * yd;
        x = (Real)xd;
        y = (Real)yd;
        z = d_sqrt((Real)s2);
        if (!(z < v.zlim)) return;
        u = f32_quotient((Real)(s2 - 1.0), __builtin_amdgcn_rcpf(Real(1) + z));
        inv_z = __builtin_amdgcn_rcpf(z);
    } else {
        x = horner5(v.cx, tau);
        y = horner5(v.cy, tau);
        f64_sqrt_rsqrt(x * x + y * y, z, inv_z);
        if (!(z < v.zlim)) return;
        u = z - Real(1);
    }
    // limb darkening and its slopes at g = z/(1+k), in units of the g step: in the mixed
    // form from 1 + u in FP64, so the lerp position keeps the precision of u
    Real gx;
    if constexpr (kMixed) {
        const double gxd = (1.0 + (double)u) * v.g_scale;
        gx = (Real)gxd;
        if (!((Real)(gxd * v.dg) <= Real(1))) return;   // g > 1: the mean and its slopes are 0
    } else {
        gx = z * v.inv1pk * v.inv_dg;
    }
    int i = (int)gx;
    i = i > ng - 2 ? ng - 2 : (i < 0 ? 0 : i);
    const Real al = gx - (Real)i;
    Real Ii, dIdg = 0, Ik = 0, Ic0 = 0, Ic1 = 0;
    if constexpr (kMixed && kGrad) {
        const f32x4 l = *(const f32x4*)(rows + 4 * i), r = *(const f32x4*)(rows + 4 * i + 4);
        Ii = l[0] + al * (r[0] - l[0]);
        dIdg = rows[4 * ng + i];
        Ik = l[1] + al * (r[1] - l[1]);
        Ic0 = l[2] + al * (r[2] - l[2]);
        Ic1 = l[3] + al * (r[3] - l[3]);
    } else if constexpr (kMixed) {
        Ii = rows[i] + al * (rows[i + 1] - rows[i]);
    } else {
        const Real* r = rows + i * (kGrad ? 8 : 2);
        Ii = r[0] + al * r[1];
        if constexpr (kGrad) {
            dIdg = r[1] * v.inv_dg;
            Ik = r[2] + al * r[3];
            Ic0 = r[4] + al * r[5];
            Ic1 = r[6] + al * r[7];
        }
    }
    // area and its slopes
    Real A, dAdz = 0, dAdk;
    if (z <= Real(1) - v.k) {
        A = v.pik2;
        dAdk = v.dpik2;
    } else {
        Real kap, akite;
        if constexpr (kMixed) {
            if (v.k < Real(1)) lens_seg_f32(v.k, z, inv_z, u, A, kap, akite);
            else ccia_kite3<Real>(Real(1), v.k, z, A, kap, akite);
        } else if (fabs(1.0 - v.k) < z) {
            A = lens_f64(v.k, z, kap, akite);
        } else {
            A = kPi;
            kap = akite = 0.0;
        }
        dAdz = Real(-2) * akite * inv_z;   // minus the chord of the lens
        dAdk = Real(2) * v.k * kap;
    }
    d.f[0] = Ii;
    d.f[1] = A;
    if constexpr (kGrad) {
        const Real vx = dhorner5(v.cx, tau), vy = dhorner5(v.cy, tau);
        const Real px = horner5(v.dcx, tau), py = horner5(v.dcy, tau);
        d.f[2] = d_fma(Ik - dIdg * z * v.inv1pk * v.inv1pk, A, Ii * dAdk);
        d.f[3] = d_fma(dIdg * v.inv1pk, A, Ii * dAdz);
        d.f[4] = -(x * vx + y * vy) * inv_z;
        d.f[5] = (x * (px - ep * vx) + y * (py - ep * vy)) * inv_z;
        d.f[6] = z * v.inv_a;
        d.f[7] = -(y * y) * v.tan_i * inv_z;
        d.f[8] = Ic0;
        d.f[9] = Ic1;
    }
}

// lnL (value 0) and its gradient (1-7) of a pv from the sums over its times.
__device__ __forceinline__ void lnl_store(const LnlArgs& s, int pv, int j, double tot, bool ok) {
    const double sig = s.sigma.at(pv);
    const double is2 = 1.0 / (sig * sig);
    if (j == 0) s.lnl[pv] = s.npt * (-log(sig) - 0.5 * log(2.0 * kPi)) - 0.5 * tot * is2;
    else s.grad[(size_t)pv * 7 + j - 1] = ok ? tot * is2 : (double)NAN;
}

// ---- main kernel ----------------------------------------------------------------------
//
// One block per (pv, range of tiles).  A lane of each wave tests one of 64 tiles
// against the window; tiles outside add their sum of (o - 1)^2, the others are
// classified point by point and the points in the window queued, so that the samples
// run on full waves.  The last points, fewer than the block, take several lanes each.
// kFused computes the pv's setup in the block itself (no workspace, one block per pv).
template <typename Real, bool kGrad, bool kFused>
__global__ void __launch_bounds__(kLnlThreads) rr_lnlike_kernel(LnlArgs s) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ LnlRec s_rec;
    __shared__ double s_red[kLnlThreads / 64][8];
    __shared__ int s_cnt[4][kLnlThreads / 64];
    Real* s_rows = (Real*)lds;
    int* s_q = (int*)(lds + lnl_rows_bytes<Real, kGrad>(s.ng));
    const int tid = threadIdx.x, lane = tid & 63;
    const int pv = blockIdx.x / s.nsplit, part = blockIdx.x - pv * s.nsplit;
    if (kFused) {
        double* sm = (double*)(s_q + kLnlQueue);
        lnl_orbit<kGrad>(s, pv, tid < kOrbitGroup, 0, tid % kOrbitGroup, &s_rec, sm);
        lnl_rows<Real, kGrad, kLnlThreads>(s, pv, &s_rec, s_rows, sm + kLnlOrbitLds);
    } else {
        const int4* rows = (const int4*)((const char*)s.rows + pv * lnl_rows_bytes<Real, kGrad>(s.ng));
        for (int i = tid; i < (int)(lnl_rows_bytes<Real, kGrad>(s.ng) / 16); i += kLnlThreads) ((int4*)s_rows)[i] = rows[i];
    }
    __syncthreads();
    const LnlRec& r = kFused ? s_rec : s.rec[pv];
    const bool ok = r.orbit_ok && r.ld_ok;
    double chi = 0.0, g[7] = {0, 0, 0, 0, 0, 0, 0};
    if (ok) {
        const int ns = s.nsamples[0];
        const double ext = s.exptimes[0], inv_ns = 1.0 / ns;
        const double t0 = r.t0, p = r.p, inv_p = r.inv_p, lo = r.lo, hi = r.hi;
        const double scale = 1.0 / (ns * r.ist), scale_ist = scale / r.ist;
        LnlPv<Real> v;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            v.cx[i] = (Real)r.c[i];
            v.cy[i] = (Real)r.c[5 + i];
            v.dcx[i] = kGrad ? (Real)r.c[10 + i] : Real(0);
            v.dcy[i] = kGrad ? (Real)r.c[15 + i] : Real(0);
        }
        v.c0 = r.c[0]; v.c1 = r.c[1]; v.c5 = r.c[5]; v.c6 = r.c[6];
        v.k = (Real)r.k;
        v.zlim = Real(1) + v.k;
        v.inv1pk = Real(1) / v.zlim;
        v.inv_dg = (Real)(1.0 / s.dg);
        v.g_scale = 1.0 / ((1.0 + r.k) * s.dg);
        v.dg = s.dg;
        v.tan_i = (Real)r.tan_i;
        v.inv_a = (Real)r.inv_a;
        v.pik2 = (Real)(kPi * r.k * r.k);
        v.dpik2 = (Real)(2.0 * kPi * r.k);
        // point `it` by G lanes of a wave, this one the sub-th
        auto point = [&](int it, int G, int sub) {
            const double om1 = s.obs[it] - 1.0;
            double epoch;
            const double tc = epoch_phase(s.times[it], t0, p, inv_p, epoch);
            LnlSums<Real, kGrad> d = {};
            const Real ep = (Real)epoch;
            if (G == 1) {
#pragma unroll 1
                for (int is = 0; is < ns; ++is) {
                    LnlTerm<Real, kGrad> one = {};
                    lnl_sample<Real, kGrad>(v, s_rows, s.ng, tc + ext * ((is + 0.5) * inv_ns - 0.5), ep, one);
                    lnl_add(d, one);
                }
            } else {
                // a sample a lane, summed in sample order as by one lane
#pragma unroll 1
                for (int i0 = 0; i0 < ns; i0 += G) {
                    LnlTerm<Real, kGrad> one = {};
                    if (i0 + sub < ns)
                        lnl_sample<Real, kGrad>(v, s_rows, s.ng, tc + ext * ((i0 + sub + 0.5) * inv_ns - 0.5), ep, one);
                    for (int q = 0; q < G; ++q) {
                        LnlTerm<Real, kGrad> of;
#pragma unroll
                        for (int m = 0; m < LnlTerm<Real, kGrad>::kN; ++m)
                            of.f[m] = __shfl(one.f[m], (lane & ~(G - 1)) + q, 64);
                        lnl_add(d, of);
                    }
                }
            }
            if (sub != 0) return;
            const double D = (double)d.v[0];
            const double res = om1 + (double)(d.v[0] * (Real)scale);  // o - m, with m = 1 - D/(ns istar)
            chi += res * res;
            if constexpr (kGrad) {
                const double rs = -res * scale;                       // r * dm/dD
#pragma unroll
                for (int m = 0; m < 7; ++m) g[m] += rs * (double)d.v[m + 1];
                g[5] += res * D * scale_ist * r.dist0;
                g[6] += res * D * scale_ist * r.dist1;
            }
        };
        const int tb = part * s.per, te = min(tb + s.per, s.ntile);
        int n = 0;
        for (int g0 = tb; g0 < te; g0 += 64) {
            // tiles outside the window, one a lane (every wave alike)
            const int tile = g0 + lane;
            bool inside = tile < te;
            if (inside && s.sorted) {
                double ea, eb;
                const double ta = epoch_phase(s.times[tile * kLnlTile], t0, p, inv_p, ea);
                const double tl = epoch_phase(s.times[tile * kLnlTile + min(kLnlTile, s.npt - tile * kLnlTile) - 1], t0, p, inv_p, eb);
                if (ea == eb ? (tl < lo || ta > hi) : (eb == ea + 1.0 && ta > hi && tl < lo)) {
                    inside = false;
                    if (tid < 64) chi += s.tsum[tile];
                }
            }
            unsigned long long mask = __ballot(inside);
            while (mask) {
                // four tiles at a time, their loads in flight together
                int tl[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    tl[j] = mask ? g0 + __ffsll((long long)mask) - 1 : -1;
                    mask &= mask - 1;
                }
                double tv[4], ov[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int it = tl[j] * kLnlTile + tid;
                    const bool in = tl[j] >= 0 && tid < s.npt - tl[j] * kLnlTile;
                    tv[j] = in ? s.times[it] : 0.0;
                    ov[j] = in ? s.obs[it] : 1.0;
                }
                unsigned long long mk[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    bool inw = false;
                    if (tl[j] >= 0 && tid < s.npt - tl[j] * kLnlTile) {
                        double epoch;
                        const double tc = epoch_phase(tv[j], t0, p, inv_p, epoch);
                        inw = lo <= tc && tc <= hi;
                        if (!inw) chi += (ov[j] - 1.0) * (ov[j] - 1.0);
                    }
                    mk[j] = __ballot(inw);
                    if (lane == 0) s_cnt[j][tid >> 6] = __popcll(mk[j]);
                }
                __syncthreads();
                // queue slots in time order: the sums do not depend on the schedule
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    int at = n;
                    for (int wv = 0; wv < kLnlThreads / 64; ++wv) {
                        at += wv < (tid >> 6) ? s_cnt[j][wv] : 0;
                        n += s_cnt[j][wv];
                    }
                    if ((mk[j] >> lane) & 1ull) s_q[at + __popcll(mk[j] & ((1ull << lane) - 1ull))] = tl[j] * kLnlTile + tid;
                }
                __syncthreads();
                for (; n >= kLnlThreads; n -= kLnlThreads) point(s_q[n - kLnlThreads + tid], 1, 0);
            }
        }
        if (n > 0) {
            int G = 1;
            while (G < 16 && 2 * G * n <= kLnlThreads && 2 * G <= ns) G *= 2;
            if (tid / G < n) point(s_q[tid / G], G, tid % G);
        }
    } else {
        chi = NAN;
    }
    // ---- block reduction ----------------------------------------------------------
    double t[8] = {chi, g[0], g[1], g[2], g[3], g[4], g[5], g[6]};
#pragma unroll
    for (int j = 0; j < (kGrad ? 8 : 1); ++j) {
        t[j] = wave_sum(t[j]);
        if (lane == 0) s_red[tid >> 6][j] = t[j];
    }
    __syncthreads();
    if (tid < (kGrad ? 8 : 1)) {
        double tot = 0.0;
        for (int wv = 0; wv < kLnlThreads / 64; ++wv) tot += s_red[wv][tid];
        if (s.nsplit > 1) s.part[((size_t)pv * s.nsplit + part) * 8 + tid] = tot;
        else lnl_store(s, pv, tid, tot, ok);
    }
}

// Sums the blocks' parts of a pv in order; one lane per (pv, value).
__global__ void __launch_bounds__(256) rr_lnlike_reduce_kernel(LnlArgs s) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int pv = i >> 3, j = i & 7;
    if (pv >= s.npv || (j > 0 && !s.grad)) return;
    double tot = 0.0;
    for (int q = 0; q < s.nsplit; ++q) tot += s.part[((size_t)pv * s.nsplit + q) * 8 + j];
    lnl_store(s, pv, j, tot, s.rec[pv].orbit_ok && s.rec[pv].ld_ok);
}

template <typename Real, bool kGrad>
static int lnl_launch(LnlArgs& s, bool fused, hipStream_t st) {
    const size_t rows = lnl_rows_bytes<Real, kGrad>(s.ng) + kLnlQueue * sizeof(int);
    const size_t ld = sizeof(double) * (size_t)lnl_ld_lds<kGrad>(s.nz, s.ng), orb = sizeof(double) * kLnlOrbitLds;
    if (fused) {
        hipLaunchKernelGGL((rr_lnlike_kernel<Real, kGrad, true>), dim3(s.npv), dim3(kLnlThreads), rows + orb + ld, st, s);
        return check_launch("rr_lnlike_kernel");
    }
    const int nob = (s.npv + kOrbitGroup - 1) / kOrbitGroup;
    const long long nb = (long long)nob + s.npv + (s.sorted ? s.ntile : 0);
    if (nb > 0x7fffffffLL || (long long)s.npv * s.nsplit > 0x7fffffffLL)
        return set_error(RR_ERANGE, "rr_lnlike: grid too large");
    hipLaunchKernelGGL((rr_lnlike_setup_kernel<Real, kGrad>), dim3((unsigned)nb), dim3(64), ld > orb ? ld : orb, st, s);
    int rc = check_launch("rr_lnlike_setup_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL((rr_lnlike_kernel<Real, kGrad, false>), dim3((unsigned)(s.npv * s.nsplit)), dim3(kLnlThreads),
                       rows, st, s);
    rc = check_launch("rr_lnlike_kernel");
    if (rc || s.nsplit == 1) return rc;
    hipLaunchKernelGGL(rr_lnlike_reduce_kernel, dim3((s.npv * 8 + 255) / 256), dim3(256), 0, st, s);
    return check_launch("rr_lnlike_reduce_kernel");
}

static int lnl_dispatch(int precision, LnlArgs& s, bool fused, hipStream_t st) {
    if (precision == RR_MIXED) return s.grad ? lnl_launch<float, true>(s, fused, st) : lnl_launch<float, false>(s, fused, st);
    return s.grad ? lnl_launch<double, true>(s, fused, st) : lnl_launch<double, false>(s, fused, st);
}

// Checks shared by the two entries; fills the light curve's and table's arguments.
static int lnl_prepare(const char* who, int precision, const rr_table* tab, const rr_lcdata* lc, int npv, int t0cols,
                       int law, const double* obs, double* lnl, double* grad, LnlArgs& s) {
    if (precision != RR_FP64 && precision != RR_MIXED) return set_error(RR_EINVAL, "%s: bad precision", who);
    if (lc->nlc != 1) return set_error(RR_EINVAL, "%s: one light curve only (nlc = %d)", who, lc->nlc);
    if (law != RR_LD_QUADRATIC && law != RR_LD_POWER_2)
        return set_error(RR_EINVAL, "%s: the quadratic and power-2 laws are supported", who);
    if (tab->ng < 2 || tab->ng > kLnlMaxNg || tab->nz < 1 || tab->nz > kLnlMaxNz || !tab->weights || !tab->mu)
        return set_error(RR_EINVAL, "%s: bad weight table (ng <= %d, nz <= %d)", who, kLnlMaxNg, kLnlMaxNz);
    if (npv < 0 || lc->npt < 0 || t0cols < 1) return set_error(RR_EINVAL, "%s: bad sizes", who);
    if (npv == 0) return RR_OK;
    if (!lc->times || !lc->nsamples || !lc->exptimes || !lc->epids || !obs || !lnl)
        return set_error(RR_EINVAL, "%s: null array", who);
    s.times = lc->times; s.obs = obs; s.nsamples = lc->nsamples; s.exptimes = lc->exptimes; s.epids = lc->epids;
    s.W = tab->weights; s.mu = tab->mu; s.lnl = lnl; s.grad = grad;
    s.rec = nullptr; s.rows = nullptr; s.tsum = nullptr; s.part = nullptr;
    s.law = law; s.npv = npv; s.npt = lc->npt; s.t0cols = t0cols; s.nk = tab->nk; s.ng = tab->ng; s.nz = tab->nz;
    s.sorted = 0;
    s.ntile = (int)(((long long)lc->npt + kLnlTile - 1) / kLnlTile);
    s.per = s.ntile;
    s.nsplit = 1;
    s.kmin = tab->kmin; s.kmax = tab->kmax; s.dk = tab->dk; s.dg = tab->dg;
    return RR_OK;
}

// Blocks per pv: enough for four on each of 256 CUs, of at least four tiles each.
static int lnl_split(int npv, int npt) {
    const int ntile = (int)(((long long)npt + kLnlTile - 1) / kLnlTile);
    int n = (1024 + npv - 1) / (npv > 0 ? npv : 1);
    n = n < ntile / 4 ? n : ntile / 4;
    return n < 1 ? 1 : n;
}

// Parameter vectors of a launch: the state between its kernels, up to 6.7 KB a vector
// at 100 g (FP64 with the gradient; 0.4 KB as FP32 values only), stays below a quarter
// of a GB however many vectors a call has.  Equal parts, the last one shorter.
constexpr int kLnlMaxPvs = 32768;
static int lnl_chunk(int npv) {
    const int n = (int)(((long long)npv + kLnlMaxPvs - 1) / kLnlMaxPvs);
    return n < 2 ? npv : (int)(((long long)npv + n - 1) / n);
}
static size_t lnl_rows_bytes(int precision, bool grad, int ng) {
    if (precision == RR_MIXED) return grad ? lnl_rows_bytes<float, true>(ng) : lnl_rows_bytes<float, false>(ng);
    return grad ? lnl_rows_bytes<double, true>(ng) : lnl_rows_bytes<double, false>(ng);
}

}  // namespace rr

using namespace rr;

extern "C" {

int rr_lnlike(int precision, const rr_table* tab, const rr_lcdata* lc, const rr_params* pv, const rr_ld* ld,
              const double* obs, const double* sigma, double* lnl, double* grad, void* stream) {
    if (!tab || !lc || !pv || !ld) return set_error(RR_EINVAL, "rr_lnlike: null descriptor");
    if (precision != RR_FP64 && precision != RR_MIXED) return set_error(RR_EINVAL, "rr_lnlike: bad precision");
    if (lc->nlc != 1) return set_error(RR_EINVAL, "rr_lnlike: one light curve only (nlc = %d)", lc->nlc);
    if (pv->kcols != 1) return set_error(RR_EINVAL, "rr_lnlike: k must be [npv, 1]");
    if (ld->law != RR_LD_QUADRATIC && ld->law != RR_LD_POWER_2)
        return set_error(RR_EINVAL, "rr_lnlike: the quadratic and power-2 laws are supported");
    if (ld->nldc < 2 || !ld->ldc) return set_error(RR_EINVAL, "rr_lnlike: two limb-darkening coefficients needed");
    LnlArgs s;
    int rc = lnl_prepare("rr_lnlike", precision, tab, lc, pv->npv, pv->t0cols, ld->law, obs, lnl, grad, s);
    if (rc || pv->npv == 0) return rc;
    if (!sigma) return set_error(RR_EINVAL, "rr_lnlike: null array");
    if (!pv->k || !pv->t0 || !pv->p || !pv->a || !pv->inc || !pv->e || !pv->w)
        return set_error(RR_EINVAL, "rr_lnlike: null parameter array");
    auto vec = [](const double* p, long long stride) { return LnlVec{p, stride, 0.0}; };
    s.k = vec(pv->k, 1); s.t0 = vec(pv->t0, pv->t0cols); s.p = vec(pv->p, 1); s.a = vec(pv->a, 1);
    s.inc = vec(pv->inc, 1); s.e = vec(pv->e, 1); s.w = vec(pv->w, 1); s.sigma = vec(sigma, 1);
    s.c0 = vec(ld->ldc, ld->nldc); s.c1 = vec(ld->ldc + 1, ld->nldc);
    return lnl_dispatch(precision, s, true, (hipStream_t)stream);
}

size_t rr_lnlike_vec_workspace_bytes(int precision, int grad, int npv, int npt, int ng) {
    if (npv < 0 || npt < 0 || ng < 2) return 0;
    const size_t n = lnl_chunk(npv), ntile = ((size_t)npt + kLnlTile - 1) / kLnlTile;
    size_t b = align_up(n * sizeof(LnlRec), 256);
    b += align_up(n * lnl_rows_bytes(precision, grad != 0, ng), 256);
    b += align_up(ntile * sizeof(double), 256);
    return b + align_up(n * lnl_split((int)n, npt) * 8 * sizeof(double), 256);
}

size_t rr_lnlike_workspace_bytes(int npv, int npt, int ng) {
    return rr_lnlike_vec_workspace_bytes(RR_FP64, 1, npv, npt, ng);
}

int rr_lnlike_vec(int precision, const rr_table* tab, const rr_lcdata* lc, int npv, int t0cols, const rr_vec* par,
                  int law, const rr_vec* ldc, const double* obs, const rr_vec* sigma, void* workspace,
                  size_t workspace_bytes, double* lnl, double* grad, void* stream) {
    if (!tab || !lc || !par || !ldc || !sigma) return set_error(RR_EINVAL, "rr_lnlike_vec: null descriptor");
    LnlArgs s;
    int rc = lnl_prepare("rr_lnlike_vec", precision, tab, lc, npv, t0cols, law, obs, lnl, grad, s);
    if (rc || npv == 0) return rc;
    const size_t need = rr_lnlike_vec_workspace_bytes(precision, grad != nullptr, npv, lc->npt, tab->ng);
    if (!workspace || workspace_bytes < need)
        return set_error(RR_EINVAL, "rr_lnlike_vec: workspace of %zu bytes needed, got %zu", need, workspace_bytes);
    const int chunk = lnl_chunk(npv);
    s.sorted = (lc->sorted & RR_SORTED_RUNS) != 0;
    s.nsplit = lnl_split(chunk, lc->npt);
    s.per = (s.ntile + s.nsplit - 1) / s.nsplit;
    char* ws = (char*)workspace;
    s.rec = (LnlRec*)ws;
    ws += align_up((size_t)chunk * sizeof(LnlRec), 256);
    s.rows = ws;
    ws += align_up((size_t)chunk * lnl_rows_bytes(precision, grad != nullptr, tab->ng), 256);
    s.tsum = (double*)ws;
    ws += align_up((size_t)s.ntile * sizeof(double), 256);
    s.part = (double*)ws;
    for (long long pv0 = 0; pv0 < npv && rc == RR_OK; pv0 += chunk) {
        auto vec = [pv0](const rr_vec& v) {
            return LnlVec{v.ptr ? v.ptr + v.stride * pv0 : nullptr, (long long)v.stride, v.value};
        };
        s.k = vec(par[0]); s.t0 = vec(par[1]); s.p = vec(par[2]); s.a = vec(par[3]); s.inc = vec(par[4]);
        s.e = vec(par[5]); s.w = vec(par[6]); s.c0 = vec(ldc[0]); s.c1 = vec(ldc[1]); s.sigma = vec(*sigma);
        s.npv = (int)(npv - pv0 < chunk ? npv - pv0 : chunk);
        s.lnl = lnl + pv0;
        s.grad = grad ? grad + 7 * pv0 : nullptr;
        rc = lnl_dispatch(precision, s, false, (hipStream_t)stream);
    }
    return rc;
}

}  // extern "C"
