// Secondary-eclipse, eclipse-spectroscopy and oblate-planet variants of the
// RoadRunner model on MI355X (gfx950).  FP64 throughout, as the reference.
//
// Replaces
//   eclipse_model   pytransit/models/roadrunner/model_eclipse.py:11-81
//                   (EclipseModel.evaluate, models/new_eclipse_model.py:34-70)
//   esmodel         models/roadrunner/model_ecspec.py:13-65
//                   (EclipseSpectroscopyModel.evaluate, models/roadrunner/esmodel.py:46-90)
//   op_full_serial  models/roadrunner/opmodel_full.py:40-134 with the ellipse
//                   scanlines of models/roadrunner/ecintersection.py:93-207
//                   (OblatePlanetModel.evaluate, models/roadrunner/opmodel.py:50-111)
//
// Kernels:
//   ec_orbit_kernel   8 pv per 64-lane block: the mid-eclipse time from the
//                     conjunction phase (orbits/orbits_py.py:544-555), the 7 Kepler
//                     solves of the Taylor stencil about it (orbits/taylor_z.py:
//                     106-185), the light travel time and the contact window
//   ec_flux_kernel    the planet disk area left visible by the star
//                     over a tile of times of one pv (window_flux.hpp).  1000 pv x
//                     20,001 t with 5 samples (160 MB written, 23 us): 55 us against
//                     147 us with one lane per (pv, time), whose samples ran in series
//                     with two libm arctangents each
//   es_flux_kernel    one lane per (pv, time): the mean lens area, fanned out over the
//                     passbands of the spectroscopy model
//   op_flux_kernel    the oblate planet's flux: the pv's ellipse
//                     scanlines in LDS, shared by the lanes that evaluate a sample; the
//                     per-pv state comes from rr_setup
#include <hip/hip_runtime.h>

#include <cmath>

#include "rr_device.hpp"
#include "rr_internal.hpp"
#include "window_flux.hpp"

namespace rr {

// Per-pv state of the eclipse models.
struct alignas(16) EcRec {
    double c[10];      // Taylor coefficients about mid-eclipse (x then y, divided by n!)
    double bt1, bt4;   // first and fourth contact about mid-eclipse, before the margin
    double p;
    double shift;      // mid-eclipse time after mid-transit, light travel time included
    double k;
    int32_t good, pad_;
};
static_assert(sizeof(EcRec) == 128, "EcRec must be 128 bytes");

constexpr double kRsunM = 6.957e8;          // IAU 2015 nominal solar radius [m]
constexpr double kCLight = 299792458.0;     // [m/s]
constexpr double kDaySec = 86400.0;

// Time from mid-transit to mid-eclipse: the mean-anomaly difference between the
// two conjunctions (true anomalies pi/2 - w and 3pi/2 - w); orbits_py.py:544-555.
__device__ __forceinline__ double eclipse_phase(double p, double e, double w) {
    // eccentric anomalies from sin(pi/2 - w) = cos w and so on; their sines from the
    // atan2's arguments, whose squares sum to (1 +- e sin w)^2
    double sw, cw;
    sincos(w, &sw, &cw);
    const double q = sqrt(1.0 - e * e) * cw;
    const double mtr = atan2(q, e + sw) - e * (q / (1.0 + e * sw));
    const double mec = atan2(-q, e - sw) - e * (-q / (1.0 - e * sw));
    const double ph = (mec - mtr) * p / kTwoPi;
    return ph > 0.0 ? ph : p + ph;
}

// Extra light path of the eclipse over the transit, (r_tr + r_ec) sin i, in days
// for a star of rstar solar radii (r: star-planet distance at each conjunction).
__device__ __forceinline__ double light_travel_time(double a, double inc, double e, double w, double rstar) {
    const double om = a * (1.0 - e * e);
    const double r_tr = om / (1.0 + e * sin(w));
    const double r_ec = om / (1.0 - e * sin(w));
    return (r_tr + r_ec) * sin(inc) * rstar * kRsunM / kCLight / kDaySec;
}

__global__ void __launch_bounds__(64) ec_orbit_kernel(int npv, const double* P, const double* A, const double* I,
                                                      const double* E, const double* W, const double* K,
                                                      const double* rstar, EcRec* rec) {
    const int sub = threadIdx.x / kOrbitGroup, j = threadIdx.x % kOrbitGroup;
    const int pv = blockIdx.x * kOrbitGroup + sub;
    const bool inrange = pv < npv;
    const int q = inrange ? pv : 0;
    __shared__ double s_x[kOrbitGroup][8], s_y[kOrbitGroup][8], s_c[kOrbitGroup][10], s_w[kOrbitGroup][2];
    const double p = P[q], a = A[q], inc = I[q], e = E[q], w = W[q], k = K[q];
    const bool valid = inrange && !(isnan(a) || a <= 1.0 || e < 0.0);
    const double te = valid ? eclipse_phase(p, e, w) : 0.0;
    if (valid && j < 7) {
        double x, y;
        kepler_xy(te + (j - 3) * 2e-2, p, a, cos(inc), e, w, x, y);
        s_x[sub][j] = x;
        s_y[sub][j] = y;
    }
    __syncthreads();
    if (valid && j == 0) taylor_from_stencil(s_x[sub], s_y[sub], s_c[sub]);
    __syncthreads();
    if (valid) {
        const double tc = contact_bisect(k, j < 4 ? 1 : 4, s_c[sub], fabs(s_c[sub][1]));
        if ((j & 3) == 0) s_w[sub][j >> 2] = tc;
    }
    __syncthreads();
    if (!inrange) return;
    EcRec* r = rec + pv;
    if (valid) {
        r->c[j] = s_c[sub][j];
        if (j < 2) r->c[8 + j] = s_c[sub][8 + j];
    }
    if (j == 0) {
        r->bt1 = valid ? s_w[sub][0] : 0.0;
        r->bt4 = valid ? s_w[sub][1] : 0.0;
        r->p = p;
        r->shift = valid ? te + light_travel_time(a, inc, e, w, rstar[q]) : 0.0;
        r->k = k;
        r->good = valid ? 1 : 0;
    }
}

struct EcArgs {
    const double* times; const int32_t* nsamples; const double* exptimes;
    const double* t0; const EcRec* rec; const double* fratio;
    double* flux;
    int npv, npt, npb, t0cols, ntiles;
};

constexpr int kEcThreads = 256;

// model_ecspec.py:51-64; the model reads the first light curve's sampling and a 1-D t0.
__global__ void __launch_bounds__(kEcThreads) es_flux_kernel(EcArgs f) {
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int pv = bid / f.ntiles;
    const int it = (bid - pv * f.ntiles) * kEcThreads + threadIdx.x;
    if (it >= f.npt) return;
    const EcRec& r = f.rec[pv];
    const size_t row = (size_t)f.npt;
    double* out = f.flux + (size_t)pv * f.npb * row + it;
    if (!r.good) {
        for (int b = 0; b < f.npb; ++b) out[b * row] = NAN;
        return;
    }
    const double te = f.t0[(size_t)pv * f.t0cols] + r.shift;
    const double p = r.p;
    double tc;
    {
#pragma clang fp contract(off)
        const double t = f.times[it];
        const double epoch = floor((t - te + 0.5 * p) / p);
        tc = t - (te + epoch * p);
    }
    const int ns = f.nsamples[0];
    const double ext = f.exptimes[0];
    const double margin = 0.0015 + ext;
    const double k = r.k;
    const bool inw = r.bt1 - margin <= tc && tc <= r.bt4 + margin;
    // the mean area over the exposure, then per passband 1 - (f A / pi) / (1 + f k^2)
    // (the per-sample terms of the reference, averaged)
    double amean = 0.0;
    if (inw) {
        double s = 0.0;
        for (int is = 1; is <= ns; ++is) {
            const double z = taylor_z<double>(tc + ext * ((is - 0.5) / ns - 0.5), r.c);
            double area, kap;
            ccia_kite<double>(1.0, k, z, area, kap);
            s += area;
        }
        amean = s / ns;
    }
    const double* fr = f.fratio + (size_t)pv * f.npb;
    for (int b = 0; b < f.npb; ++b) {
        const double fb = fr[b];
        out[b * row] = inw ? 1.0 - (fb * amean / kPi) / (1.0 + fb * (k * k)) : 1.0;
    }
}

// model_eclipse.py:56-80 on the window kernel: pi k^2 minus the mean lens area.
struct EclArgs {
    WfData d;
    const int32_t* epids; const double* exptimes; const double* t0;
    const EcRec* rec;
    double* flux;
    int t0cols;
};

struct EclipseFlux {
    using Real = double;
    using Args = EclArgs;
    static constexpr int kKinds = 1;    // the planet's limb crosses the star's
    static constexpr int kDense = 4096, kDenseNs = 16;
    static constexpr int kBlocks = 6;
    struct Pv {
        double c[10], bt1, bt4, p, inv_p, shift, k, k2;
        bool good;
    };
    struct Item {
        double ext, inv_ns;
    };
    static __device__ __forceinline__ Pv load(const EclArgs& f, int pv) {
        const EcRec& r = f.rec[pv];
        Pv o;
#pragma unroll
        for (int j = 0; j < 10; ++j) o.c[j] = r.c[j];
        o.bt1 = r.bt1;
        o.bt4 = r.bt4;
        o.p = r.p;
        o.inv_p = 1.0 / r.p;
        o.shift = r.shift;
        o.k = r.k;
        o.k2 = kPi * (r.k * r.k);
        o.good = r.good != 0;
        return o;
    }
    static __device__ __forceinline__ double fill(const Pv& c) { return c.k2; }
    static __device__ __forceinline__ double bad() { return NAN; }
    static __device__ __forceinline__ WfWindow window(const EclArgs& f, const Pv& c, int pv, int ilc) {
        const double margin = 0.003 + f.exptimes[ilc];
        return {f.t0[(size_t)pv * f.t0cols + min(max(f.epids[ilc], 0), f.t0cols - 1)] + c.shift, c.bt1 - margin,
                c.bt4 + margin};
    }
    static __device__ __forceinline__ Item item(const EclArgs& f, const Pv&, int, int ilc) {
        return {f.exptimes[ilc], 1.0 / f.d.nsamples[ilc]};
    }
    static __device__ __forceinline__ int classify(const EclArgs&, const Pv& c, const Item&, double t, double& v) {
        const double z = taylor_z<double>(t, c.c);
        v = z;
        if (fabs(1.0 - c.k) < z && z < 1.0 + c.k) return 1;
        // off the disk pi k^2 is left, behind it nothing (a planet larger than the star
        // keeps the excess); NaN stays NaN
        if (1.0 + c.k <= z) v = c.k2;
        else if (z <= 1.0 - c.k) v = 0.0;
        else if (z <= c.k - 1.0) v = c.k2 - kPi;
        else v = NAN;
        return 0;
    }
    static __device__ __forceinline__ double heavy(const EclArgs&, const Pv& c, const Item&, double, double z, int, int, int,
                                                   unsigned char*) {
        return c.k2 - lens_area_f64(c.k, z);
    }
    static __device__ __forceinline__ int group(const EclArgs&) { return 1; }
    static __device__ __forceinline__ double finish(const Pv&, double acc, int ns, const Item&) { return acc / ns; }
    static __device__ __forceinline__ void stage(const EclArgs&, const Pv&, int, unsigned char*) {}
};

template <int P, bool kMulti>
__global__ void __launch_bounds__(kWfThreads, EclipseFlux::kBlocks) ec_flux_kernel(EclArgs f) {
    window_flux_body<EclipseFlux, P, kMulti>(f);
}

// ---- Oblate planet ---------------------------------------------------------------

constexpr int kOpMaxLines = 2048;

struct OpArgs {
    WfData d;
    const int32_t* pbids; const int32_t* epids; const double* exptimes;
    const double* k; const double* t0; const double* fl; const double* alpha;
    const PvRec* rec; const double* istar; const double* ldm;
    double* flux;
    int npb, kcols, t0cols, ng, nlines;
    double dg, inv_dg;
};

// opmodel_full.py:95-131 on the window kernel.  The planet's ellipse is a table of
// scanlines (create_ellipse, ecintersection.py:93-134, at k[:, 0]) in LDS; a sample
// whose planet crosses the limb sums the part of every scanline on the stellar disk
// (ecintersection.py:137-207, the three branches by the centre's x).  Several lanes
// share a sample's scanlines (group): with one lane a sample the 100 square roots in a
// row ran on the few lanes of a wave that held one (400 pv x 10,000 t, 5 samples, 100
// lines: 744 us a call, now 81; floor 5 us of writes and 2 us of FP64).
struct OblateFlux {
    using Real = double;
    using Args = OpArgs;
    static constexpr int kKinds = 1;
    static constexpr int kDense = 1024, kDenseNs = 4;
    static constexpr int kBlocks = 4;
    struct Pv {
        double c[10], bt1, bt4, p, inv_p, fl;
        bool good;
    };
    struct Item {
        double ext, inv_ns, k, inv_1pk, ist;
        const double* row;
    };
    static __device__ __forceinline__ Pv load(const OpArgs& f, int pv) {
        const PvRec& r = f.rec[pv];
        Pv o;
#pragma unroll
        for (int j = 0; j < 10; ++j) o.c[j] = r.c[j];
        o.bt1 = r.bt1;
        o.bt4 = r.bt4;
        o.p = r.p;
        o.inv_p = r.inv_p;
        o.fl = f.fl[pv];
        o.good = r.good && r.ldok;
        return o;
    }
    static __device__ __forceinline__ double fill(const Pv&) { return 1.0; }
    static __device__ __forceinline__ double bad() { return NAN; }
    static __device__ __forceinline__ WfWindow window(const OpArgs& f, const Pv& c, int pv, int ilc) {
        const double margin = 0.0015 + f.exptimes[ilc];
        return {f.t0[(size_t)pv * f.t0cols + min(max(f.epids[ilc], 0), f.t0cols - 1)], c.bt1 - margin, c.bt4 + margin};
    }
    static __device__ __forceinline__ Item item(const OpArgs& f, const Pv&, int pv, int ilc) {
        const int ipb = min(max(f.pbids[ilc], 0), f.npb - 1);
        const double k = f.k[(size_t)pv * f.kcols + (f.kcols == 1 ? 0 : ipb)];
        const size_t j = (size_t)pv * f.npb + ipb;
        return {f.exptimes[ilc], 1.0 / f.d.nsamples[ilc], k, 1.0 / (1.0 + k), f.istar[j], f.ldm + j * f.ng};
    }
    static __device__ __forceinline__ double centre(const double* c, double t) {
        return (((c[4] * t + c[3]) * t + c[2]) * t + c[1]) * t + c[0];
    }
    static __device__ __forceinline__ double flux_of(const OpArgs& f, const Item& I, double z, double area) {
        return (I.ist - interp_ld_r(z * I.inv_1pk, f.dg, f.inv_dg, I.row, f.ng) * area) / I.ist;
    }
    static __device__ __forceinline__ int classify(const OpArgs& f, const Pv& c, const Item& I, double t, double& v) {
        const double z = taylor_z<double>(t, c.c);
        v = z;
        const bool in = z <= 1.0 - I.k;
        if (!in && !(z >= 1.0 + I.k)) return 1;
        v = flux_of(f, I, z, in ? kPi * I.k * (1.0 - c.fl) * I.k : 0.0);
        return 0;
    }
    static __device__ __forceinline__ double heavy(const OpArgs& f, const Pv& c, const Item& I, double t, double z, int,
                                                   int sub, int G, unsigned char* sh) {
        const double* ys = (const double*)sh;
        const double* xl = ys + f.nlines;
        const double* xr = xl + f.nlines;
        const double cx = centre(c.c, t), cy = centre(c.c + 5, t), k = I.k;
        const bool west = cx < -k, east = cx > k, swapped = c.fl > 1.0;
        double acc = 0.0;
        for (int j = sub; j < f.nlines; j += G) {
            const double x0 = xl[j], x1 = xr[j], v = ys[j] + cy;
            const double h2 = 1.0 - v * v;
            // a row without a chord or off the disk adds nothing
            if (isfinite(x0) && h2 >= 0.0) {
                const double half = f64_sqrt(h2);
                const double left = east ? x0 : fmax(x0, -half - cx);
                const double right = west ? x1 : fmin(x1, half - cx);
                const double w = right - left;
                // a chord that the disk's edge cuts on its side may leave nothing; with its
                // ends swapped (f > 1) an uncut one counts as it is, less than nothing
                if (!swapped) acc += west || east ? fmax(w, 0.0) : w;
                else acc += (west ? left > x0 : east && right < x1) ? 0.0 : w;
            }
        }
        for (int o = G / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
        return flux_of(f, I, z, acc * (ys[1] - ys[0]));
    }
    static __device__ __forceinline__ double finish(const Pv&, double acc, int ns, const Item&) { return acc / ns; }
    // Lanes of a listed sample.  Its own work is some 25 lines', so few lines take few lanes;
    // with fewer samples a point, lists are short and the sample's latency counts
    // (400 pv x 20,000 t over 36 d / 1.3 d, us with 8, 4 and 1 lanes: nss 5, 10 lines
    // 73, 64, 61 / 165, 126, 107, 100 lines 142, 137, 153 / 360, 328, 323; nss 1, 10 lines
    // 48, 49, 51 / 68, 55, 49, 100 lines 64, 70, 114 / 147, 132, 137; at 200 lines 8 and 4
    // are equal, and 8 answer a small call sooner).
    static __device__ __forceinline__ int group(const OpArgs& f) {
        const bool few = f.d.uniform_ns > 0 && f.d.uniform_ns < 4;
        return f.nlines >= 128 || (few && f.nlines >= 48) ? 8 : (f.nlines >= 16 || few ? 4 : 1);
    }
    static size_t shared_bytes(int nlines) { return 3 * (size_t)nlines * sizeof(double); }
    static __device__ __forceinline__ void stage(const OpArgs& f, const Pv& c, int pv, unsigned char* sh) {
        double* ys = (double*)sh;
        double* s_xl = ys + f.nlines;
        double* s_xr = s_xl + f.nlines;
        const double k0 = f.k[(size_t)pv * f.kcols];
        const double al = f.alpha[pv];
        const double ca = cos(al), sa = sin(al);
        const double b = 1.0 - c.fl, b2 = b * b, ca2 = ca * ca, sa2 = sa * sa;
        const double dy = 2.0 / (f.nlines + 1);
        for (int j = threadIdx.x; j < f.nlines; j += kWfThreads) {
            const double y = (double)(j + 1) * dy - 1.0;
            const double y2 = y * y;
            double d = b2 * ca2 + ca2 * ca2 * (-y2) - 2.0 * ca2 * sa2 * y2 - sa2 * sa2 * y2 + sa2;
            double xl = NAN, xr = NAN;
            if (d >= 0.0) {
                d = sqrt(d) / b;
                const double u = (ca * sa * y) / b2 - ca * sa * y;
                const double v = sa2 / b2 + ca2;
                xl = (-d + u) / v;
                xr = (d + u) / v;
            }
            ys[j] = k0 * y;
            s_xl[j] = k0 * xl;
            s_xr[j] = k0 * xr;
        }
    }
};

template <int P, bool kMulti>
__global__ void __launch_bounds__(kWfThreads, OblateFlux::kBlocks) op_flux_kernel(OpArgs f) {
    window_flux_body<OblateFlux, P, kMulti>(f);
}

}  // namespace rr

using namespace rr;

extern "C" {

size_t ec_workspace_bytes(int npv) { return npv < 0 ? 0 : align_up((size_t)npv * sizeof(EcRec), 256); }

static int ec_common(const char* who, const rr_lcdata* lc, const rr_params* pv, const double* rstar, void* workspace,
                     size_t workspace_bytes, double* flux, int spectro, const double* fratio, int npb,
                     void* stream) {
    if (!lc || !pv) return set_error(RR_EINVAL, "%s: null descriptor", who);
    const int npv = pv->npv, npt = lc->npt, nlc = lc->nlc;
    if (npv < 0 || npt < 0 || nlc < 1 || pv->t0cols < 1 || (spectro && npb < 1))
        return set_error(RR_EINVAL, "%s: bad sizes (npv=%d npt=%d nlc=%d npb=%d)", who, npv, npt, nlc, npb);
    if (pv->kcols != 1) return set_error(RR_EINVAL, "%s: the radius ratio must be one value per pv", who);
    if (npv == 0 || npt == 0) return RR_OK;
    if ((long long)npv * npt * (spectro ? npb : 1) > (1LL << 40))
        return set_error(RR_ERANGE, "%s: problem too large", who);
    if (!lc->times || !lc->nsamples || !lc->exptimes || (!spectro && (!lc->epids || (nlc > 1 && !lc->lcids))))
        return set_error(RR_EINVAL, "%s: null light-curve array", who);
    if (!pv->k || !pv->t0 || !pv->p || !pv->a || !pv->inc || !pv->e || !pv->w || !rstar || !flux ||
        (spectro && !fratio))
        return set_error(RR_EINVAL, "%s: null parameter array", who);
    if (!workspace || workspace_bytes < ec_workspace_bytes(npv))
        return set_error(RR_EINVAL, "%s: workspace of %zu bytes needed, got %zu", who, ec_workspace_bytes(npv),
                         workspace_bytes);
    hipStream_t s = (hipStream_t)stream;
    EcRec* rec = (EcRec*)workspace;
    hipLaunchKernelGGL(ec_orbit_kernel, dim3((npv + kOrbitGroup - 1) / kOrbitGroup), dim3(64), 0, s, npv, pv->p,
                       pv->a, pv->inc, pv->e, pv->w, pv->k, rstar, rec);
    int rc = check_launch("ec_orbit_kernel");
    if (rc) return rc;
    if (!spectro) {
        EclArgs f;
        // the epoch indices may be the caller's passband indices (EclipseModel), of which
        // the one-window bit says nothing: it holds when t0 has one column
        f.d = wf_data(lc, pv->t0cols == 1);
        f.epids = lc->epids; f.exptimes = lc->exptimes; f.t0 = pv->t0; f.rec = rec; f.flux = flux;
        f.t0cols = pv->t0cols;
        return wf_launch<EclipseFlux>(who,
                                      {ec_flux_kernel<4, false>, ec_flux_kernel<1, false>, ec_flux_kernel<4, true>, ec_flux_kernel<1, true>},
                                      f, npv, 0, s);
    }
    EcArgs f;
    f.times = lc->times; f.nsamples = lc->nsamples;
    f.exptimes = lc->exptimes; f.t0 = pv->t0; f.rec = rec; f.fratio = fratio; f.flux = flux;
    f.npv = npv; f.npt = npt; f.npb = npb; f.t0cols = pv->t0cols;
    f.ntiles = (npt + kEcThreads - 1) / kEcThreads;
    const long long nb = (long long)f.ntiles * npv;
    if (nb > 0x7fffffffLL) return set_error(RR_ERANGE, "%s: grid too large", who);
    hipLaunchKernelGGL(es_flux_kernel, dim3((unsigned)nb), dim3(kEcThreads), 0, s, f);
    return check_launch("es_flux_kernel");
}

int eclipse_evaluate(const rr_lcdata* lc, const rr_params* pv, const double* rstar, void* workspace,
                     size_t workspace_bytes, double* flux, void* stream) {
    return ec_common("eclipse_evaluate", lc, pv, rstar, workspace, workspace_bytes, flux, 0, nullptr, 0, stream);
}

int es_evaluate(const rr_lcdata* lc, const rr_params* pv, const double* rstar, const double* fratio, int npb,
                void* workspace, size_t workspace_bytes, double* flux, void* stream) {
    if (pv && pv->t0cols != 1) return set_error(RR_EINVAL, "es_evaluate: t0 must be one value per pv");
    return ec_common("es_evaluate", lc, pv, rstar, workspace, workspace_bytes, flux, 1, fratio, npb, stream);
}

int op_evaluate(const rr_table* tab, const rr_lcdata* lc, const rr_params* pv, const rr_ld* ld, const double* fl,
                const double* alpha, int nlines, void* workspace, size_t workspace_bytes, double* flux,
                void* stream) {
    if (nlines < 2 || nlines > kOpMaxLines)
        return set_error(RR_ERANGE, "op_evaluate: nlines must be in [2, %d], got %d", kOpMaxLines, nlines);
    if (!pv || !lc || !tab) return set_error(RR_EINVAL, "op_evaluate: null descriptor");
    if (pv->npv > 0 && lc->npt > 0 && (!fl || !alpha)) return set_error(RR_EINVAL, "op_evaluate: null f or alpha");
    // the per-pv state (orbit, window, limb-darkening means, disk integrals) is rr_full's
    int rc = rr_setup(RR_FP64, tab, lc, pv, ld, workspace, workspace_bytes, stream);
    if (rc) return rc;
    const int npv = pv->npv, npt = lc->npt, npb = lc->npb;
    if (npv == 0 || npt == 0) return RR_OK;
    if (!flux) return set_error(RR_EINVAL, "op_evaluate: null flux");
    // the workspace layout of rr_workspace_bytes: PvRec[npv] | istar[npv, npb] | ldm64[npv, npb, ng]
    char* ws = (char*)workspace;
    if (!lc->times || !lc->nsamples || !lc->exptimes || (lc->nlc > 1 && !lc->lcids))
        return set_error(RR_EINVAL, "op_evaluate: null light-curve array");
    OpArgs f;
    f.rec = (const PvRec*)ws;
    ws += align_up((size_t)npv * sizeof(PvRec), 256);
    f.istar = (const double*)ws;
    ws += align_up((size_t)npv * npb * sizeof(double), 256);
    f.ldm = (const double*)ws;
    f.d = wf_data(lc, true);
    f.pbids = lc->pbids; f.epids = lc->epids; f.exptimes = lc->exptimes;
    f.k = pv->k; f.t0 = pv->t0; f.fl = fl; f.alpha = alpha; f.flux = flux;
    f.npb = npb; f.kcols = pv->kcols; f.t0cols = pv->t0cols;
    f.ng = tab->ng; f.nlines = nlines; f.dg = tab->dg; f.inv_dg = 1.0 / tab->dg;
    return wf_launch<OblateFlux>("op_evaluate",
                                 {op_flux_kernel<4, false>, op_flux_kernel<1, false>, op_flux_kernel<4, true>, op_flux_kernel<1, true>},
                                 f, npv, OblateFlux::shared_bytes(nlines), (hipStream_t)stream);
}

}  // extern "C"
