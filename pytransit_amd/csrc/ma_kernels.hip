// Mandel & Agol (2002) quadratic limb-darkening transit model on MI355X (gfx950).
//
// Replaces quadratic_model_v (pytransit/models/numba/ma_quadratic_nb.py:532-595) as
// called by QuadraticModel.evaluate (pytransit/models/ma_quadratic.py:74-140), with
// the analytic flux eval_quad_z_s (ma_quadratic_nb.py:277-389) and its complete
// elliptic integrals (ma_quadratic_nb.py:55-126).  FP64 throughout.
//
// Kernels:
//   ma_orbit_kernel   8 pv per 64-lane block: the Taylor orbit and contact window of
//                     the RoadRunner path (taylor_z.py:23-102,298-328)
//   ma_flux_kernel    epoch, window (contact times +- 0.025 d),
//                     supersampling and analytic flux of a tile of times of one pv;
//                     flux [npv, npt] (window_flux.hpp)
//
// 1000 pv x 10,007 t with 5 samples (80 MB written, 2 % of the points in transit): the
// flux kernel takes 62 us (65-72 between other work) against 430 us with one lane per
// (pv, time), the orbits 6 us.
// The write alone is 12 us and the samples' FP64 arithmetic about as much again; the
// rest is the latency of the workgroups that hold a window (about 10 us each, four
// resident per CU).
#include <hip/hip_runtime.h>

#include <cmath>

#include "rr_device.hpp"
#include "rr_internal.hpp"
#include "window_flux.hpp"

namespace rr {

// Hastings' coefficients of K (both polynomials in m1, the second with the logarithm)
// and of E
__constant__ const double kEllipticTable[19] = {
    1.38629436112, 0.09666344259, 0.03590092383, 0.03742563713, 0.01451196212,
    0.5, 0.12498593597, 0.06880248576, 0.03328355346, 0.00441787012,
    1.0, 0.44325141463, 0.06260601220, 0.04757383546, 0.01736506451,
    0.24998368310, 0.09200180037, 0.04069697526, 0.00526449639};

// Flux of a star with quadratic limb darkening (u1, u2) occulted by a disk of
// radius k at separation z <= 1 + k; the case analysis of Mandel & Agol (2002) as in
// ma_quadratic_nb.py:277-389 (uniform part le, linear part ld, quadratic part ed).
// `inside` says z < 1 - k.
//
// The cases are written with the quantities they share, since a wave pays for every
// case it holds.  With x1 = (k-z)^2, x2 = (k+z)^2 and D = 1 - x1 (inside) or 4 k z
// (limb), the squared complementary modulus is |1 - x2| / D in both, the prefactor
// 2 / (9 pi sqrt D), and the start value sqrt(n + 1) of Bulirsch's algorithm
// (k+z) / |k-z| inside and 1 / |k-z| on the limb: neither the modulus nor n is formed.
// K and E are Hastings' polynomials (Hastings 1955; Abramowitz & Stegun 17.3.34 and
// 17.3.36, the forms of ma_quadratic_nb.py:93-126) on one logarithm; Pi is Bulirsch's
// iteration (Bulirsch 1965, Numer. Math. 7, 78-90; ma_quadratic_nb.py:55-91, relative
// tolerance 1e-8, at most 1000 steps), a reciprocal and a square root a step.
__device__ __forceinline__ double ma_quad_z(double z, double k, double u1, double u2, bool inside) {
    const double inv_pi = 1.0 / kPi;
    if (fabs(k - 0.5) < 1.0e-4) {
        k = 0.5;
        inside = z < 0.5;
    }
    if (fabs(z - k) < 1e-6) {
        z += 1e-6;
        inside = inside && z < 1.0 - k;
    }
    if (z > 1.0 + k) return 1.0;
    if (k >= 1.0 && z <= k - 1.0) return 0.0;
    if (k < 0.0) return NAN;                                 // the modulus' square is negative
    const double k2 = k * k, z2 = z * z;
    const double dm = k - z, sp = k + z;
    const double x1 = dm * dm, x2 = sp * sp, x3 = dm * sp;
    const bool edge = fabs(dm) < 1.e-4 * sp;                 // the planet's edge at the disk's centre
    const double D = inside ? 1.0 - x1 : 4.0 * k * z;
    const double rD = f64_rcp(D);
    const double qe = z > 0.5 ? 0.5 / k : 2.0 * k;           // the modulus of the edge case
    const double m1 = edge ? 1.0 - qe * qe : fabs(1.0 - x2) * rD;
    const double lm = f64_log(m1);
    const ConstTable ct = const_table(kEllipticTable);
    const double kk = table_poly<5>(ct, m1) - table_poly<5>(ct + 5, m1) * lm;
    const double ek = table_poly<5>(ct + 10, m1) - m1 * table_poly<4>(ct + 15, m1) * lm;
    double ld;
    if (!edge) {
        const double ratio = f64_div(sp, dm);
        double kc = f64_sqrt(m1), p = inside ? fabs(ratio) : f64_rcp(fabs(dm));
        double e = kc, m0 = 1.0, c = 1.0, d = inside ? f64_rcp(p) : fabs(dm), rp = d, pk = 0.0;
        for (int it = 0; it < 1000; ++it) {
            const double f = c;
            c = fma(d, rp, c);
            const double g = e * rp;
            d = 2.0 * fma(f, g, d);
            p = g + p;
            const double mo = m0;
            m0 = kc + m0;
            if (!(fabs(mo - kc) > 1e-8 * mo)) {
                pk = kHalfPi * f64_div(fma(c, m0, d), m0 * (m0 + p));
                break;
            }
            kc = 2.0 * f64_sqrt(e);
            e = kc * m0;
            rp = f64_rcp(p);
        }
        const double A = inside ? 1.0 - 5.0 * z2 + k2 + x3 * x3 : (1.0 - x2) * (2.0 * x2 + x1 - 3.0) - 3.0 * x3 * (x2 - 2.0);
        ld = 2.0 / 9.0 * inv_pi * f64_sqrt(rD) * (A * kk + (inside ? 1.0 - x1 : D) * (z2 + 7.0 * k2 - 4.0) * ek - 3.0 * ratio * pk);
        if (z < k) ld += 2.0 / 3.0;
        if (inside && fabs(k + z - 1.0) < 1.e-4)
            ld = 2.0 / 3.0 * inv_pi * acos(1.0 - 2.0 * k) -
                 4.0 / 9.0 * inv_pi * sqrt(k * (1.0 - k)) * (3.0 + 2.0 * k - 8.0 * k2);
    } else if (k == 0.5) {
        ld = 1.0 / 3.0 - 4.0 * inv_pi / 9.0;
    } else if (z > 0.5) {
        ld = 1.0 / 3.0 + 16.0 * k / 9.0 * inv_pi * (2.0 * k2 - 1.0) * ek -
             (32.0 * k2 * k2 - 20.0 * k2 + 3.0) / 9.0 * inv_pi / k * kk;
    } else {
        ld = 1.0 / 3.0 + 2.0 / 9.0 * inv_pi * (4.0 * (2.0 * k2 - 1.0) * ek + (1.0 - 4.0 * k2) * kk);
    }
    double le, ed = 0.5 * k2 * (k2 + 2.0 * z2);
    if (z <= 1.0 - k) {
        le = k2;
        // first or last contact of the inner limb itself: the limb case's ed with no lune
        if (!inside && !(edge && !(z > 0.5))) ed = 0.0 - 0.125 * inv_pi * (1.0 + 5.0 * k2 + z2) * sqrt((1.0 - x1) * (x2 - 1.0));
    } else {
        // cos kappa1 = (1 - k^2 + z^2) / 2z and cos kappa0 = (k^2 + z^2 - 1) / 2kz, whose
        // sines are the lune term over 2z and 2kz: angles without the quotients
        const double lune = f64_sqrt(fmax((1.0 - x1) * (x2 - 1.0), 0.0));
        const double kap1 = f64_atan2_ypos(lune, 1.0 - k2 + z2);
        const double kap0 = f64_atan2_ypos(lune, k2 + z2 - 1.0);
        le = (k2 * kap0 + kap1 - 0.5 * lune) * inv_pi;
        if (!(edge && !(z > 0.5)))
            ed = 0.5 * inv_pi * (kap1 + k2 * (k2 + 2.0 * z2) * kap0 - 0.25 * (1.0 + 5.0 * k2 + z2) * lune);
    }
    if (edge && k == 0.5) ed = 3.0 / 32.0;
    // (an IEEE quotient: coefficients whose disk integral is 0 give an infinity)
    return 1.0 - ((1.0 - u1 - 2.0 * u2) * le + (u1 + 2.0 * u2) * ld + u2 * ed) / (1.0 - u1 / 3.0 - u2 / 6.0);
}

struct MaArgs {
    WfData d;
    const int32_t* pbids; const int32_t* epids; const double* exptimes;
    const double* k; const double* t0; const double* ldc;
    const PvRec* rec;
    double* flux;
    int npv, npb, kcols, t0cols;
};

// Orbit and contact window of each pv (the reference computes them for every pv).
__global__ void __launch_bounds__(64) ma_orbit_kernel(int npv, const double* P, const double* A, const double* I,
                                                      const double* E, const double* W, const double* K, int kcols,
                                                      PvRec* rec) {
    const int pv = blockIdx.x * kOrbitGroup + threadIdx.x / kOrbitGroup;
    const int j = threadIdx.x % kOrbitGroup;
    const bool inrange = pv < npv;
    const int q = inrange ? pv : 0;
    const double k0 = K[(size_t)q * kcols];
    PvRec* r = rec + q;
    __shared__ double sm[kOrbitLds];
    orbit_group(pv, inrange, P[q], A[q], I[q], E[q], W[q], k0, r->c, &r->bt1, sm);
    if (inrange && j == 0) {
        r->p = P[q];
        r->inv_p = 1.0 / P[q];
        r->k0 = k0;
        // ma_quadratic_nb.py:549-555: a NaN radius ratio or semi-major axis gives inf
        bool good = !isnan(A[q]);
        for (int c = 0; c < kcols; ++c) good = good && !isnan(K[(size_t)q * kcols + c]);
        r->good = good ? 1 : 0;
        r->ldok = 1;
    }
}

// ma_quadratic_nb.py:557-594 on the window kernel.
struct MaModel {
    using Real = double;
    using Args = MaArgs;
    static constexpr int kKinds = 2;    // 1 inside the disk, 2 on the limb
    static constexpr int kDense = 4096, kDenseNs = 16;
    static constexpr int kBlocks = 4;   // workgroups per CU: 128 registers (3: 87, 4: 80, 5 with spills: 84 us)
    struct Pv {
        double c[10], lo, hi, p, inv_p;
        bool good;
    };
    struct Item {
        double ext, inv_ns, k, u1, u2;
    };
    static __device__ __forceinline__ Pv load(const MaArgs& f, int pv) {
        const PvRec& r = f.rec[pv];
        Pv o;
#pragma unroll
        for (int j = 0; j < 10; ++j) o.c[j] = r.c[j];
        o.lo = r.bt1 - 0.025;
        o.hi = r.bt4 + 0.025;
        o.p = r.p;
        o.inv_p = r.inv_p;
        o.good = r.good != 0;
        return o;
    }
    static __device__ __forceinline__ double fill(const Pv&) { return 1.0; }
    static __device__ __forceinline__ double bad() { return INFINITY; }
    static __device__ __forceinline__ WfWindow window(const MaArgs& f, const Pv& c, int pv, int ilc) {
        return {f.t0[(size_t)pv * f.t0cols + min(max(f.epids[ilc], 0), f.t0cols - 1)], c.lo, c.hi};
    }
    static __device__ __forceinline__ Item item(const MaArgs& f, const Pv&, int pv, int ilc) {
        const int ipb = min(max(f.pbids[ilc], 0), f.npb - 1);
        const double* u = f.ldc + (size_t)pv * 2 * f.npb + 2 * ipb;
        return {f.exptimes[ilc], 1.0 / f.d.nsamples[ilc], f.k[(size_t)pv * f.kcols + (f.kcols == 1 ? 0 : ipb)], u[0], u[1]};
    }
    static __device__ __forceinline__ int classify(const MaArgs&, const Pv& c, const Item& I, double t, double& v) {
        if (isnan(I.u1) || isnan(I.u2)) {
            v = INFINITY;
            return 0;
        }
        const double z = taylor_z<double>(t, c.c);
        v = z > 1.0 + I.k ? 1.0 : z;
        if (z > 1.0 + I.k) return 0;
        return z < 1.0 - I.k ? 1 : 2;
    }
    static __device__ __forceinline__ double heavy(const MaArgs&, const Pv&, const Item& I, double, double z, int kind,
                                                   int, int, unsigned char*) {
        return ma_quad_z(z, I.k, I.u1, I.u2, kind == 1);
    }
    static __device__ __forceinline__ int group(const MaArgs&) { return 1; }
    static __device__ __forceinline__ double finish(const Pv&, double acc, int ns, const Item&) { return acc / ns; }
    static __device__ __forceinline__ void stage(const MaArgs&, const Pv&, int, unsigned char*) {}
};

template <int P, bool kMulti>
__global__ void __launch_bounds__(kWfThreads, MaModel::kBlocks) ma_flux_kernel(MaArgs f) {
    window_flux_body<MaModel, P, kMulti>(f);
}

}  // namespace rr

using namespace rr;

extern "C" {

size_t ma_workspace_bytes(int npv) { return npv < 0 ? 0 : align_up((size_t)npv * sizeof(PvRec), 256); }

int ma_evaluate(const rr_lcdata* lc, const rr_params* pv, const double* ldc, void* workspace, size_t workspace_bytes,
                double* flux, void* stream) {
    if (!lc || !pv) return set_error(RR_EINVAL, "ma_evaluate: null descriptor");
    const int npv = pv->npv, npt = lc->npt, npb = lc->npb, nlc = lc->nlc;
    if (npv < 0 || npt < 0 || npb < 1 || nlc < 1) return set_error(RR_EINVAL, "ma_evaluate: bad sizes");
    if (pv->kcols != 1 && pv->kcols != npb)
        return set_error(RR_EINVAL, "Radius ratios should be given either as an [npv, 1] or [npv, npb] array.");
    if (pv->t0cols < 1) return set_error(RR_EINVAL, "ma_evaluate: t0 needs at least one column");
    if (npv == 0 || npt == 0) return RR_OK;
    if ((long long)npv * npt > (1LL << 40)) return set_error(RR_ERANGE, "ma_evaluate: problem too large");
    if (!lc->times || !lc->pbids || !lc->epids || !lc->nsamples || !lc->exptimes || (nlc > 1 && !lc->lcids))
        return set_error(RR_EINVAL, "ma_evaluate: null light-curve array");
    if (!pv->k || !pv->t0 || !pv->p || !pv->a || !pv->inc || !pv->e || !pv->w || !ldc || !flux)
        return set_error(RR_EINVAL, "ma_evaluate: null parameter array");
    if (!workspace || workspace_bytes < ma_workspace_bytes(npv))
        return set_error(RR_EINVAL, "ma_evaluate: workspace of %zu bytes needed, got %zu", ma_workspace_bytes(npv),
                         workspace_bytes);
    hipStream_t s = (hipStream_t)stream;
    PvRec* rec = (PvRec*)workspace;
    hipLaunchKernelGGL(ma_orbit_kernel, dim3((npv + kOrbitGroup - 1) / kOrbitGroup), dim3(64), 0, s, npv, pv->p,
                       pv->a, pv->inc, pv->e, pv->w, pv->k, pv->kcols, rec);
    int rc = check_launch("ma_orbit_kernel");
    if (rc) return rc;
    MaArgs f;
    f.d = wf_data(lc, true);
    f.pbids = lc->pbids; f.epids = lc->epids; f.exptimes = lc->exptimes;
    f.k = pv->k; f.t0 = pv->t0; f.ldc = ldc; f.rec = rec; f.flux = flux;
    f.npv = npv; f.npb = npb; f.kcols = pv->kcols; f.t0cols = pv->t0cols;
    return wf_launch<MaModel>("ma_evaluate",
                              {ma_flux_kernel<4, false>, ma_flux_kernel<1, false>, ma_flux_kernel<4, true>, ma_flux_kernel<1, true>},
                              f, npv, 0, s);
}

}  // extern "C"
