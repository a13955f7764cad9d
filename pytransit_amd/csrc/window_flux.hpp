// Light-curve kernel body shared by the models whose flux is a constant outside a window
// around the conjunction and an average over exposure samples inside it.
//
// One workgroup of 256 lanes takes up to kWfMaxSub sub-tiles of 256 * P consecutive
// times of one pv.
//   1. A sub-tile of one sorted light curve whose first and last times lie on the same
//      side of the window is outside it.  In the others every lane classifies P times;
//      the points in the window go to an LDS queue, the rest is stored as the constant.
//   2. The queue is worked through in chunks of up to 256 points and kWfCap (point,
//      sample) items, one item a lane: a first pass settles the cheap samples (planet
//      off the disk, wholly inside it) and lists the others, which a second pass
//      evaluates on full waves, M::group lanes to a sample.
//   3. A lane sums the samples of a point in order and stores the point.
//   4. The sub-tiles outside are filled with the constant (16-byte stores), last: loads
//      after them would wait for them.
// One lane per (pv, time), the form this replaces, ran the samples of a point in
// series, paid every branch of the sample in any wave that held a window point, and
// left the rest of the chip waiting for those waves: only 2-10 % of the times of a
// survey light curve are in a window.  A workgroup's entry (arguments, record, epoch,
// boundary times: four dependent loads) is 2-3 us however few points it has, so it
// takes several sub-tiles when that leaves enough workgroups, and few where a transit
// fills them.
//
// A model M gives
//   Args                      kernel arguments, with a WfData member `d`
//   Pv, Item                  the pv's constants; a light curve's constants, with
//                             members ext (exposure time) and inv_ns (1 / nsamples)
//   load(f, pv)               -> Pv, with members p, inv_p, good
//   fill(P), bad()            the values outside the window and of an invalid pv
//   window(f, P, pv, ilc)     -> WfWindow
//   item(f, P, pv, ilc)       -> Item
//   kDense, kDenseNs          when a launch takes small workgroups (wf_launch)
//   classify(f, P, I, t, v)   the sample at time t from conjunction: 0 when v is its
//                             value, 1 or 2 when a heavy evaluation has to follow,
//                             with v the separation
//   heavy(f, P, I, t, z, kind, sub, G, sh)   that evaluation by G = group(f) lanes, a power
//                             of two up to 64, this one the sub-th; lane 0 of the group
//                             returns the value
//   stage(f, P, pv, sh), shared_bytes(f)     block-wide tables in LDS
#pragma once

#include "rr_device.hpp"
#include "rr_internal.hpp"

namespace rr {

struct WfData {
    const double* times;
    const int32_t* lcids;
    const int32_t* nsamples;
    int npt, nlc;
    int ntiles, nsub;  // workgroups per pv, sub-tiles of each
    int sorted;       // contiguous light curves, each sorted in time
    int one_window;   // with `sorted`: times sorted throughout, one window for all
    int uniform_ns;   // the common nsamples, or 0
    int density;      // times in a tenth of a day, a power of two at most that, or 0: unknown
    int samples;      // with it: samples a point
};

struct WfWindow {
    double t0, lo, hi;
};

constexpr int kWfThreads = 256;
constexpr int kWfCap = 1024;    // (point, sample) items of a chunk

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

// Dynamic LDS of a launch: the queue, the chunk's phases, item values, lists and contexts.
constexpr int kWfMaxSub = 8;
template <class M>
static inline size_t wf_lds_bytes(int queue, bool multi, size_t shared) {
    size_t b = (size_t)kWfThreads * sizeof(double) + (size_t)queue * sizeof(uint16_t);
    b += (size_t)kWfCap * (sizeof(typename M::Real) + sizeof(uint16_t));
    if (multi) b += (size_t)kWfThreads * sizeof(typename M::Item) + (size_t)(kWfCap + kWfThreads) * sizeof(uint16_t);
    return (b + 15) / 16 * 16 + shared;
}

template <class M, int P, bool kMulti>
__device__ __forceinline__ void window_flux_body(const typename M::Args& f) {
    using Real = typename M::Real;
    using Item = typename M::Item;
    constexpr int kSub = kWfThreads * P;
    constexpr int kWaves = kWfThreads / 64;
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ int s_n, s_na, s_nb, s_sum[kWaves];
    const WfData& d = f.d;
    double* s_tc = (double*)lds;                                   // [kWfThreads] phases of the chunk's points
    Item* s_ctx = (Item*)(s_tc + kWfThreads);                      // [kWfThreads] of several light curves
    Real* s_val = (Real*)(s_ctx + (kMulti ? kWfThreads : 0));      // [kWfCap] item values
    uint16_t* s_it = (uint16_t*)(s_val + kWfCap);                  // [kSub * d.nsub] time index of the queued points
    uint16_t* s_list = s_it + kSub * d.nsub;                       // [kWfCap] heavy items, kind 1 from the front, 2 from the back
    uint16_t* s_map = s_list + kWfCap;                             // [kWfCap] item -> point (several light curves)
    uint16_t* s_beg = s_map + kWfCap;                              // [kWfThreads] point -> first item
    // (an offset from lds, not a rounded address: the compiler loses sight of LDS through a
    // cast to an integer and reads it with flat loads)
    const int end = (int)((kMulti ? (unsigned char*)(s_beg + kWfThreads) : (unsigned char*)s_map) - lds);
    unsigned char* shared = lds + (end + 15) / 16 * 16;

    const int tid = threadIdx.x, lane = tid & 63;
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int pv = bid / d.ntiles;
    const int base = (bid - pv * d.ntiles) * kSub * d.nsub;
    const int cnt = min(kSub * d.nsub, d.npt - base);
    const typename M::Pv c = M::load(f, pv);
    Real* out = (Real*)f.flux + (size_t)pv * d.npt + base;
    if (!c.good) {
        block_fill<Real>(out, cnt, M::bad());
        return;
    }
    const Real fill = M::fill(c);
    auto lc_of = [&](int it) { return kMulti ? min(max(d.lcids[base + it], 0), d.nlc - 1) : 0; };
    // ---- sub-tiles outside the window, one a lane (every wave alike) ------------------
    unsigned out_mask = 0u;
    const WfWindow w0 = M::window(f, c, pv, 0);
    if (d.sorted) {
        const int i0 = lane * kSub, i1 = min(i0 + kSub, cnt) - 1;
        bool outside = false;
        if (lane < d.nsub && i0 < cnt) {
            const double tf = d.times[base + i0], tl = d.times[base + i1];
            const int la = lc_of(i0);
            if (!kMulti || d.one_window || la == lc_of(i1)) {
                const WfWindow w = kMulti ? M::window(f, c, pv, la) : w0;
                double ea, eb;
                const double ta = epoch_phase(tf, w.t0, c.p, c.inv_p, ea);
                const double tb = epoch_phase(tl, w.t0, c.p, c.inv_p, eb);
                outside = ea == eb ? (tb < w.lo || ta > w.hi) : (eb == ea + 1.0 && ta > w.hi && tb < w.lo);
            }
        }
        out_mask = (unsigned)__ballot(outside);
    }
    const int nsub = (cnt + kSub - 1) / kSub;
    if (out_mask == (1u << nsub) - 1u) {
        block_fill<Real>(out, cnt, fill);
        return;
    }
    if (tid == 0) s_n = 0;
    __syncthreads();
    // ---- the points in the window into the queue --------------------------------------
    for (int j0 = 0; j0 < nsub; ++j0) {
        if ((out_mask >> j0) & 1u) continue;
        double tv[P];
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int it = j0 * kSub + j * kWfThreads + tid;
            tv[j] = it < cnt ? d.times[base + it] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int it = j0 * kSub + j * kWfThreads + tid;
            bool inw = false;
            if (it < cnt) {
                const WfWindow w = kMulti ? M::window(f, c, pv, lc_of(it)) : w0;
                double ep;
                const double tc = epoch_phase(tv[j], w.t0, c.p, c.inv_p, ep);
                inw = w.lo <= tc && tc <= w.hi;
                if (!inw) out[it] = fill;
            }
            const unsigned long long mk = __ballot(inw);
            if (mk) {
                int at = 0;
                if (lane == 0) at = atomicAdd(&s_n, __popcll(mk));
                at = __shfl(at, 0, 64) + __popcll(mk & ((1ull << lane) - 1ull));
                if (inw) s_it[at] = (uint16_t)it;
            }
        }
    }
    __syncthreads();
    const int n = s_n;
    // the common nsamples, or 0
    const int uns = d.uniform_ns > 0 ? d.uniform_ns : (kMulti ? 0 : max(d.nsamples[0], 1));
    const float inv_uns = uns > 0 ? 1.0f / (float)uns : 0.0f;
    Item ctx0;
    if (!kMulti) ctx0 = M::item(f, c, pv, 0);
    if (n > 0) M::stage(f, c, pv, shared);   // read after the chunk's first barrier
    // ---- chunks of points -------------------------------------------------------------
    // c0: first point of the chunk; s0: its first sample, above 0 only for a point with
    // more samples than the item arrays hold, which is a chunk of its own in several passes
    int c0 = 0, s0 = 0;
    Real carry = Real(0);
    while (c0 < n) {
        int cn, tot, ns1 = uns;
        if (uns > 0) {
            cn = min(max(1, min(kWfThreads, kWfCap / uns)), n - c0);
            tot = min(kWfCap, cn * (uns - s0));
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
            tot = s_sum[0];
            if (cn == 0) {
                ns1 = d.nsamples[lc_of(s_it[c0])];
                cn = 1;
                tot = min(kWfCap, ns1 - s0);
                for (int i = tid; i < tot; i += kWfThreads) s_map[i] = 0;
                if (tid == 0) s_beg[0] = 0;
            }
        }
        if (tid == 0) s_na = s_nb = 0;
        if (tid < cn) {
            const int it = s_it[c0 + tid];
            WfWindow w = w0;
            if (kMulti) {
                const int ilc = lc_of(it);
                w = M::window(f, c, pv, ilc);
                s_ctx[tid] = M::item(f, c, pv, ilc);
            }
            double ep;
            s_tc[tid] = epoch_phase(d.times[base + it], w.t0, c.p, c.inv_p, ep);
        }
        __syncthreads();
        auto point_of = [&](int i) {
            return uns > 0 ? (uns > kWfCap ? 0 : (int)(((float)i + 0.5f) * inv_uns)) : (int)s_map[i];
        };
        auto first_of = [&](int q) { return uns > 0 ? q * uns : (int)s_beg[q]; };
        for (int b = 0; b < tot; b += kWfThreads) {
            const int i = b + tid;
            int kind = 0;
            if (i < tot) {
                const int q = point_of(i);
                const Item I = kMulti ? s_ctx[q] : ctx0;
                const double t = sample_time(s_tc[q], I.ext, I.inv_ns, s0 + i - first_of(q));
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
        const int na = s_na, nh = na + s_nb, G = M::group(f);
#pragma unroll 1
        for (int j = tid / G; j < nh; j += kWfThreads / G) {
            const int kind = j < na ? 1 : 2;
            const int i = s_list[j < na ? j : kWfCap - 1 - (j - na)];
            const int q = point_of(i);
            const Item I = kMulti ? s_ctx[q] : ctx0;
            const double t = sample_time(s_tc[q], I.ext, I.inv_ns, s0 + i - first_of(q));
            const Real v = M::heavy(f, c, I, t, s_val[i], kind, tid % G, G, shared);
            if (tid % G == 0) s_val[i] = v;
        }
        __syncthreads();
        const bool partial = cn == 1 && tot < ns1 - s0;
        if (tid < cn) {
            const int it = s_it[c0 + tid];
            const int ns = uns > 0 ? uns : d.nsamples[lc_of(it)];
            const int i0 = first_of(tid), i1 = min(i0 + ns - s0, tot);
            Real acc = carry;
            for (int k = i0; k < i1; ++k) acc += s_val[k];
            carry = partial ? acc : Real(0);
            if (!partial) out[it] = M::finish(c, acc, ns, kMulti ? s_ctx[tid] : ctx0);
        }
        __syncthreads();
        s0 = partial ? s0 + tot : 0;
        c0 += partial ? 0 : cn;
    }
    for (int j0 = 0; j0 < nsub; ++j0)
        if ((out_mask >> j0) & 1u) block_fill<Real>(out + j0 * kSub, min(kSub, cnt - j0 * kSub), fill);
}

// Launch over npv x npt: four times a lane and as many sub-tiles a workgroup as leave
// kWfBlocks workgroups (the Mandel-Agol model at 1000 pv x 10,007 t, nss 5: 115, 80, 76
// and 92 us with 2000, 3000, 5000 and 10,000 workgroups; at 2000 x 20,000, nss 1: 119
// and 160 us with 6000 and 20,000); one time a lane where single sub-tiles of four
// leave CUs short of work.
//
// That suits long light curves, whose windows are a few points of each workgroup.  Where
// the times lie so close that a transit fills whole workgroups, these are the launch's
// length, and small ones even it out: from M::kDense samples in a tenth of a day single
// sub-tiles, and from M::kDenseNs samples a point one time a lane (1000 pv x 20,000 t with
// 1500 times in a tenth of a day, us by the first rule, with single sub-tiles of four, with
// one time a lane: MA nss 5 428, 381, 416, nss 20 1593, 1314, 1161, oblate 100 lines nss 5
// 1478, 914, 703, nss 20 5766, 3469, 2420; with 50 times, nss 5: MA 139, 201, 258, EC 62,
// 85, 128).  With the density known a pv also keeps four tiles (3000 x 3000, 225 times, nss
// 1, without and with: MA 129, 92, EC 60, 49, oblate 170, 122).
constexpr int kWfBlocks = 4096;
static inline long long wf_density(const rr_lcdata* lc) {
    const int c = (lc->sorted >> RR_DENSITY_SHIFT) & 31;
    return c ? 1ll << c : 0;
}
// Samples a point, known with the density
static inline long long wf_samples(const rr_lcdata* lc) { return 1ll << ((lc->sorted >> RR_SAMPLES_SHIFT) & 31); }
template <class M>
struct WfKernels {
    typedef void (*Fn)(typename M::Args);
    Fn one4, one1;     // one light curve: four times a lane, one time a lane
    Fn multi4, multi1; // several
};
template <class M>
static inline int wf_launch(const char* who, const WfKernels<M>& kn, typename M::Args& f, int npv, size_t shared,
                            hipStream_t s) {
    const int npt = f.d.npt;
    const long long sub4 = ((long long)npt + 4 * kWfThreads - 1) / (4 * kWfThreads);
    const int ns = f.d.samples;
    const bool known = f.d.density >= 64, dense = known && (long long)f.d.density * ns >= M::kDense;
    const int P = sub4 * npv < 2048 || (dense && ns >= M::kDenseNs) ? 1 : 4;
    const long long nsubs = P == 4 ? sub4 : ((long long)npt + kWfThreads - 1) / kWfThreads;
    int per = 1;
    const int least = known ? 4 : 1;      // tiles of a pv
    while (!dense && per < kWfMaxSub && (nsubs + 2 * per - 1) / (2 * per) >= least &&
           (nsubs + 2 * per - 1) / (2 * per) * npv >= kWfBlocks)
        per *= 2;
    const long long ntiles = (nsubs + per - 1) / per;
    if (ntiles * npv > 0x7fffffffLL) return set_error(RR_ERANGE, "%s: grid too large", who);
    f.d.ntiles = (int)ntiles;
    f.d.nsub = per;
    const bool multi = f.d.nlc > 1;
    const size_t lds = wf_lds_bytes<M>(kWfThreads * P * per, multi, shared);
    const dim3 grid((unsigned)(ntiles * npv)), block(kWfThreads);
    const auto fn = multi ? (P == 4 ? kn.multi4 : kn.multi1) : (P == 4 ? kn.one4 : kn.one1);
    hipLaunchKernelGGL(fn, grid, block, lds, s, f);
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
    d.ntiles = d.nsub = 1;
    d.sorted = (lc->sorted & RR_SORTED_RUNS) != 0;
    const int one = RR_SORTED_RUNS | RR_SORTED_TIMES | RR_ONE_WINDOW;
    d.one_window = shared_epochs && (lc->sorted & one) == one;
    d.uniform_ns = lc->uniform_nsamples > 0 ? lc->uniform_nsamples : 0;
    d.density = (int)(wf_density(lc) < 0x40000000 ? wf_density(lc) : 0x40000000);
    d.samples = d.uniform_ns > 0 ? d.uniform_ns : (int)(wf_samples(lc) < 0x40000000 ? wf_samples(lc) : 0x40000000);
    return d;
}

}  // namespace rr
