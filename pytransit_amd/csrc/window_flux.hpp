// Light-curve kernel shared by the models whose flux is a constant outside a window
// around the conjunction and an average over exposure samples inside it.
//
// One workgroup of 256 lanes takes a tile of 256 * P consecutive times of one pv.
//   1. A tile of one sorted light curve whose first and last times lie on the same
//      side of the window is filled with the constant (16-byte stores).
//   2. Otherwise every lane classifies P times; the points in the window go to an
//      LDS queue with their phase, the others are stored as the constant.
//   3. The queue is worked through in chunks of up to 256 points and kWfCap (point,
//      sample) items, one item a lane: a first pass settles the cheap samples (planet
//      off the disk, wholly inside it) and lists the others, which a second pass
//      evaluates on full waves, M::kGroup lanes to a sample.
//   4. A lane sums the samples of a point in order and stores the point.
// One lane per (pv, time), the form this replaces, ran the samples of a point in
// series, paid every branch of the sample in any wave that held a window point, and
// left the rest of the chip waiting for those waves: only 2-10 % of the times of a
// survey light curve are in a window.
//
// A model M gives
//   Args                      kernel arguments, with a WfData member `d`
//   Pv, Item                  the pv's constants; a light curve's constants, with
//                             members ext (exposure time) and inv_ns (1 / nsamples)
//   load(f, pv)               -> Pv, with members p, inv_p, good
//   fill(P), bad()            the values outside the window and of an invalid pv
//   window(f, P, pv, ilc)     -> WfWindow
//   item(f, P, pv, ilc)       -> Item
//   classify(f, P, I, t, v)   the sample at time t from conjunction: 0 when v is its
//                             value, 1 or 2 when a heavy evaluation has to follow,
//                             with v the separation
//   heavy<G>(f, P, I, t, z, kind, sub, sh)   that evaluation by G lanes, this one the
//                             sub-th; every lane of the group returns the value
//   stage(f, P, pv, sh), shared_bytes(f)     block-wide tables in LDS
#pragma once

#include "rr_device.hpp"
#include "rr_internal.hpp"

namespace rr {

struct WfData {
    const double* times;
    const int32_t* lcids;
    const int32_t* nsamples;
    int npt, nlc, ntiles;
    int sorted;       // contiguous light curves, each sorted in time
    int one_window;   // with `sorted`: times sorted throughout, one window for all
    int uniform_ns;   // the common nsamples, or 0
};

struct WfWindow {
    double t0, lo, hi;
};

constexpr int kWfThreads = 256;
constexpr int kWfCap = 1024;    // (point, sample) items of a chunk

// Time from the nearest conjunction after the division-free epoch reduction.
__device__ __forceinline__ double wf_phase(double t, double t0, double p, double inv_p, double& epoch) {
#pragma clang fp contract(off)
    const double u = t - t0 + 0.5 * p;
    double ep = floor(u * inv_p);
    const double r = u - ep * p;
    ep += (r < 0.0) ? -1.0 : ((r >= p) ? 1.0 : 0.0);
    epoch = ep;
    return t - (t0 + ep * p);
}

// base[0 .. n) = v by the block: 16-byte vectors from the first aligned element on.
template <typename T>
__device__ __forceinline__ void block_fill(T* base, int n, T v) {
    typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
    constexpr int kVec = 16 / sizeof(T);
    int head = (int)(((16 - ((uintptr_t)base & 15)) & 15) / sizeof(T));
    if (((uintptr_t)base % sizeof(T)) != 0 || head > n) head = n;
    const int tid = threadIdx.x;
    for (int i = tid; i < head; i += kWfThreads) base[i] = v;
    vec vv;
#pragma unroll
    for (int j = 0; j < kVec; ++j) vv[j] = v;
    const int nv = (n - head) / kVec;
    for (int i = tid; i < nv; i += kWfThreads) __builtin_nontemporal_store(vv, (vec*)(base + head) + i);
    for (int i = head + nv * kVec + tid; i < n; i += kWfThreads) base[i] = v;
}

// Dynamic LDS of a launch: the queue, the chunk's item values, lists and contexts.
template <class M>
static inline size_t wf_lds_bytes(int P, int nlc, int uniform_ns, size_t shared) {
    size_t b = (size_t)kWfThreads * P * (sizeof(double) + sizeof(uint16_t));
    b += (size_t)kWfCap * (sizeof(typename M::Real) + sizeof(uint16_t));
    if (nlc > 1) b += (size_t)kWfThreads * sizeof(typename M::Item);
    if (uniform_ns == 0) b += (size_t)(kWfCap + kWfThreads) * sizeof(uint16_t);
    return (b + 15) / 16 * 16 + shared;
}

template <class M, int P>
__global__ void __launch_bounds__(kWfThreads) window_flux_kernel(typename M::Args f) {
    using Real = typename M::Real;
    using Item = typename M::Item;
    constexpr int kTileN = kWfThreads * P;
    constexpr int kWaves = kWfThreads / 64;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ int s_n, s_na, s_nb, s_sum[kWaves];
    const WfData& d = f.d;
    const bool multi = d.nlc > 1;
    double* s_tc = (double*)lds;                                   // [kTileN] phases of the queue
    Item* s_ctx = (Item*)(s_tc + kTileN);                          // [kWfThreads] of several light curves
    Real* s_val = (Real*)(s_ctx + (multi ? kWfThreads : 0));       // [kWfCap] item values
    uint16_t* s_it = (uint16_t*)(s_val + kWfCap);                  // [kTileN] time index in the tile
    uint16_t* s_list = s_it + kTileN;                              // [kWfCap] heavy items, kind 1 from the front, 2 from the back
    uint16_t* s_map = s_list + kWfCap;                             // [kWfCap] item -> point (uneven nsamples)
    uint16_t* s_beg = s_map + kWfCap;                              // [kWfThreads] point -> first item
    const uintptr_t end = (uintptr_t)(d.uniform_ns > 0 ? s_map : s_beg + kWfThreads);
    unsigned char* shared = (unsigned char*)((end + 15) & ~(uintptr_t)15);

    const int tid = threadIdx.x, lane = tid & 63;
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int pv = bid / d.ntiles;
    const int base = (bid - pv * d.ntiles) * kTileN;
    const int cnt = min(kTileN, d.npt - base);
    const typename M::Pv c = M::load(f, pv);
    Real* out = (Real*)f.flux + (size_t)pv * d.npt + base;
    if (!c.good) {
        block_fill<Real>(out, cnt, M::bad());
        return;
    }
    const Real fill = M::fill(c);
    auto lc_of = [&](int it) { return multi ? min(max(d.lcids[base + it], 0), d.nlc - 1) : 0; };
    if (d.sorted) {
        const int la = lc_of(0), lb = lc_of(cnt - 1);
        if (la == lb || d.one_window) {
            const WfWindow w = M::window(f, c, pv, la);
            double ea, eb;
            const double ta = wf_phase(d.times[base], w.t0, c.p, c.inv_p, ea);
            const double tb = wf_phase(d.times[base + cnt - 1], w.t0, c.p, c.inv_p, eb);
            const bool outside = ea == eb ? (tb < w.lo || ta > w.hi) : (eb == ea + 1.0 && ta > w.hi && tb < w.lo);
            if (outside) {
                block_fill<Real>(out, cnt, fill);
                return;
            }
        }
    }
    if (tid == 0) s_n = 0;
    M::stage(f, c, pv, shared);
    __syncthreads();
    // ---- the points in the window into the queue --------------------------------------
    WfWindow w = M::window(f, c, pv, 0);
    double tv[P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int it = j * kWfThreads + tid;
        tv[j] = it < cnt ? d.times[base + it] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int it = j * kWfThreads + tid;
        bool inw = false;
        double tc = 0.0;
        if (it < cnt) {
            if (multi) w = M::window(f, c, pv, lc_of(it));
            double ep;
            tc = wf_phase(tv[j], w.t0, c.p, c.inv_p, ep);
            inw = w.lo <= tc && tc <= w.hi;
            if (!inw) out[it] = fill;
        }
        const unsigned long long mk = __ballot(inw);
        if (mk) {
            int at = 0;
            if (lane == 0) at = atomicAdd(&s_n, __popcll(mk));
            at = __shfl(at, 0, 64) + __popcll(mk & ((1ull << lane) - 1ull));
            if (inw) {
                s_tc[at] = tc;
                s_it[at] = (uint16_t)it;
            }
        }
    }
    __syncthreads();
    const int n = s_n;
    const int uns = d.uniform_ns;
    const float inv_uns = uns > 0 ? 1.0f / (float)uns : 0.0f;
    Item ctx0;
    if (!multi) ctx0 = M::item(f, c, pv, 0);
    // ---- chunks of points -------------------------------------------------------------
    int c0 = 0;
    while (c0 < n) {
        int cn, tot;
        if (uns > 0) {
            cn = min(min(kWfThreads, kWfCap / uns), n - c0);
            tot = cn * uns;
        } else {
            // points whose samples fit the item arrays, by a block-wide prefix sum
            const int mine = c0 + tid < n ? max(0, min(d.nsamples[lc_of(s_it[c0 + tid])], kWfCap + 1)) : 0;
            int run = mine;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(run, o, 64);
                run += lane >= o ? v : 0;
            }
            if (lane == 63) s_sum[tid >> 6] = run;
            __syncthreads();
            for (int q = 0; q < (tid >> 6); ++q) run += s_sum[q];
            const bool fits = c0 + tid < n && run <= kWfCap;
            cn = __syncthreads_count(fits);     // the prefix sums are non-decreasing
            if (fits) {
                s_beg[tid] = (uint16_t)(run - mine);
                for (int i = run - mine; i < run; ++i) s_map[i] = (uint16_t)tid;
            }
            if (tid == cn - 1) s_sum[0] = run;
            __syncthreads();
            tot = cn > 0 ? s_sum[0] : 0;
        }
        if (cn == 0) break;                     // more samples a point than the arrays hold: below
        if (tid == 0) s_na = s_nb = 0;
        if (multi && tid < cn) s_ctx[tid] = M::item(f, c, pv, lc_of(s_it[c0 + tid]));
        __syncthreads();
        auto point_of = [&](int i) { return uns > 0 ? (int)(((float)i + 0.5f) * inv_uns) : (int)s_map[i]; };
        auto first_of = [&](int q) { return uns > 0 ? q * uns : (int)s_beg[q]; };
        for (int b = 0; b < tot; b += kWfThreads) {
            const int i = b + tid;
            int kind = 0;
            if (i < tot) {
                const int q = point_of(i);
                const Item I = multi ? s_ctx[q] : ctx0;
                const double t = s_tc[c0 + q] + I.ext * ((i - first_of(q) + 0.5) * I.inv_ns - 0.5);
                kind = M::classify(f, c, I, t, s_val[i]);
            }
#pragma unroll
            for (int kd = 1; kd <= M::kKinds; ++kd) {
                const unsigned long long mk = __ballot(kind == kd);
                if (mk) {
                    int at = 0;
                    if (lane == 0) at = atomicAdd(kd == 1 ? &s_na : &s_nb, __popcll(mk));
                    at = __shfl(at, 0, 64) + __popcll(mk & ((1ull << lane) - 1ull));
                    if (kind == kd) s_list[kd == 1 ? at : kWfCap - 1 - at] = (uint16_t)i;
                }
            }
        }
        __syncthreads();
        constexpr int G = M::kGroup;
        const int na = s_na, nh = na + s_nb;
        for (int j = tid / G; j < nh; j += kWfThreads / G) {
            const int kind = j < na ? 1 : 2;
            const int i = s_list[j < na ? j : kWfCap - 1 - (j - na)];
            const int q = point_of(i);
            const Item I = multi ? s_ctx[q] : ctx0;
            const double t = s_tc[c0 + q] + I.ext * ((i - first_of(q) + 0.5) * I.inv_ns - 0.5);
            const Real v = M::template heavy<G>(f, c, I, t, s_val[i], kind, tid % G, shared);
            if (tid % G == 0) s_val[i] = v;
        }
        __syncthreads();
        if (tid < cn) {
            const int it = s_it[c0 + tid];
            const int i0 = first_of(tid), ns = uns > 0 ? uns : d.nsamples[lc_of(it)];
            Real acc = Real(0);
            for (int k = 0; k < ns; ++k) acc += s_val[i0 + k];
            out[it] = M::finish(c, acc, ns, multi ? s_ctx[tid] : ctx0);
        }
        __syncthreads();
        c0 += cn;
    }
    // points with more samples than kWfCap: one lane a point
    for (int j = c0 + tid; j < n; j += kWfThreads) {
        const int ilc = lc_of(s_it[j]);
        const Item I = M::item(f, c, pv, ilc);
        const int ns = d.nsamples[ilc];
        Real acc = Real(0);
        for (int k = 0; k < ns; ++k) {
            const double t = s_tc[j] + I.ext * ((k + 0.5) * I.inv_ns - 0.5);
            Real v;
            const int kind = M::classify(f, c, I, t, v);
            acc += kind == 0 ? v : M::template heavy<1>(f, c, I, t, v, kind, 0, shared);
        }
        out[s_it[j]] = M::finish(c, acc, ns, I);
    }
}

// Launch over npv x npt.  Four times a lane; one time a lane (tiles of 256) when that
// would leave CUs without a workgroup.
template <class M>
static inline int wf_launch(const char* who, typename M::Args& f, int npv, size_t shared, hipStream_t s) {
    const int npt = f.d.npt;
    const long long tiles4 = (npt + 4 * kWfThreads - 1) / (4 * kWfThreads);
    const int P = tiles4 * npv < 2048 ? 1 : 4;
    const long long ntiles = P == 4 ? tiles4 : (npt + kWfThreads - 1) / kWfThreads;
    if (ntiles * npv > 0x7fffffffLL) return set_error(RR_ERANGE, "%s: grid too large", who);
    f.d.ntiles = (int)ntiles;
    const size_t lds = wf_lds_bytes<M>(P, f.d.nlc, f.d.uniform_ns, shared);
    const dim3 grid((unsigned)(ntiles * npv)), block(kWfThreads);
    if (P == 4) hipLaunchKernelGGL((window_flux_kernel<M, 4>), grid, block, lds, s, f);
    else hipLaunchKernelGGL((window_flux_kernel<M, 1>), grid, block, lds, s, f);
    return check_launch(who);
}

// The light-curve part of a model's arguments.  `shared_epochs` is false where the
// caller's epoch indices are not those the RR_ONE_WINDOW bit speaks of.
static inline WfData wf_data(const rr_lcdata* lc, bool shared_epochs) {
    WfData d;
    d.times = lc->times;
    d.lcids = lc->lcids;
    d.nsamples = lc->nsamples;
    d.npt = lc->npt;
    d.nlc = lc->nlc;
    d.ntiles = 0;
    d.sorted = (lc->sorted & RR_SORTED_RUNS) != 0;
    const int one = RR_SORTED_RUNS | RR_SORTED_TIMES | RR_ONE_WINDOW;
    d.one_window = shared_epochs && (lc->sorted & one) == one;
    d.uniform_ns = lc->uniform_nsamples > 0 ? lc->uniform_nsamples : 0;
    return d;
}

}  // namespace rr
