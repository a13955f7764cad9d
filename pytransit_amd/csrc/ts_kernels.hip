// Transmission-spectroscopy RoadRunner model (TSModel) on MI355X (gfx950).
//
// Replaces tsmodel_serial (pytransit/models/roadrunner/model_trspec.py:11-93):
//   per pv: k_mean = mean(k), k_max = max(k), Taylor orbit, contact window at
//   k_mean widened by 0.0015 + exptimes[0]; limb-darkening means
//   ldm[pb, g] = W(k_mean)[g, :] . ldp[pb, :] with exact 2-D weights at k_mean
//   (precompute_weights=False) or a k-lerp of the 3-D table; per (t, sample) one
//   lens geometry at k_mean, fanned out over passbands with the area scaled by
//   k^2/k_mean^2 (z <= 1 - k_max) or extrapolated linearly in k otherwise.
//
// Kernels:
//   ts_setup_kernel    8 pvs a 64-lane workgroup (orbit, mean and maximum k, window)
//   ts_weights_kernel  up to 16 (pv, g) rows per workgroup: the 2-D weight rows at
//                      k_mean, the lens areas that need arccos evaluated from a
//                      list on full waves, written transposed W2T[pv][z][g] (FP64
//                      and FP32, g padded to 16); the launch's last workgroups take
//                      the disk integrals
//   ts_ldm_tab_mfma_kernel  FP32 MFMA contraction ldm = ldp . W2T for tabulated FP64
//                      profiles: one 8-wave workgroup per pv, W2T in LDS, each row
//                      read as 128-byte pieces (16-byte loads, a permuted z order)
//   ts_ldm_mfma_kernel the same for named laws (profiles evaluated per element) and
//                      the shapes the first does not take
//   ts_ldm_mfma64_kernel the FP64 contraction on v_mfma_f64_16x16x4f64 (W2T in LDS
//                      when it fits in 128 KB), else ts_ldm_f64_kernel on the VALU
//   ts_flux_rows_aligned_kernel, ts_flux_rows_kernel  one sample, whole rows of a pv a
//                      workgroup
//   ts_flux_table_kernel  up to 32 samples, any row length: a tile of times of a pv a
//                      workgroup, its geometry in LDS
//   ts_flux_kernel     the rest (more samples, very fine g grids)
//
// Flux layout [npv, npb, npt].
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <type_traits>

#include "rr_device.hpp"
#include "rr_internal.hpp"

namespace rr {

struct TsRec {
    double c[10];
    double bt1, bt4;     // window incl. the 0.0015 + exptimes[0] margin
    double p, inv_p;
    double kmean, kmax;
    double ak;           // table mode: k-lerp weight
    int32_t ik;          // table mode: row index, -1 for exact 2-D weights
    int32_t good;
    int32_t pad[2];
};

struct TsArgs {
    const double* times; const double* k; const double* t0;
    const double* exptimes; const int32_t* nsamples;   // element 0 applies to every point (Q16)
    const double* p; const double* a; const double* inc; const double* e; const double* w;
    int law, nldc; const double* ldc; const double* ldp_in; const double* istar_in;
    const double* W; const double* ze; const double* mu;
    TsRec* rec; double* istar; double* w2_64; float* w2_32; double* ldm64; float* ldm32;
    int npv, npb, npt, nk, ng, ngp, nz, nzp, use_table;
    int row_split;       // workgroups of a pv in the row forms, each a range of passbands
    int ldm_split;       // workgroups of a pv in the contraction, each every ldm_split-th group of row tiles
    double kmin, kmax_tab, dk, dg;
};

constexpr int kTsGroup = 8;

// ---- per-pv setup; model_trspec.py:36-68 ----------------------------------------------
__global__ void __launch_bounds__(64) ts_setup_kernel(TsArgs s) {
    __shared__ double s_x[8][8], s_y[8][8], s_c[8][10], s_w[8][2], s_km[8];
    const int sub = threadIdx.x / kTsGroup, j = threadIdx.x % kTsGroup;
    const int pv = blockIdx.x * kTsGroup + sub;
    const bool inrange = pv < s.npv;
    const int q = inrange ? pv : 0;
    const double a = s.a[q], e = s.e[q];
    const bool valid = inrange && !(isnan(a) || a <= 1.0 || e < 0.0);
    // the mean and the maximum of the pv's row of radius ratios: each of its 8 lanes
    // takes every eighth value, eight loads in flight, and the lanes' sums meet by
    // shuffles (one lane summing 512 values in order took 8 us; the sums agree to
    // rounding)
    double sum = 0.0, kmx = -INFINITY;
    const double* kr = s.k + (size_t)q * s.npb;
    for (int c0 = j; c0 < s.npb; c0 += 8 * kTsGroup) {
        double v[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) v[m] = kr[min(c0 + m * kTsGroup, s.npb - 1)];
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const bool in = c0 + m * kTsGroup < s.npb;
            sum += in ? v[m] : 0.0;
            kmx = in ? fmax(kmx, v[m]) : kmx;
        }
    }
#pragma unroll
    for (int o = kTsGroup / 2; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o, 64);
        kmx = fmax(kmx, __shfl_xor(kmx, o, 64));
    }
    if (inrange && j == 0) {
        s_km[sub] = sum / s.npb;
        TsRec* r = s.rec + q;
        r->kmean = sum / s.npb;
        r->kmax = kmx;
        r->p = s.p[q];
        r->inv_p = 1.0 / s.p[q];
        r->good = valid ? 1 : 0;
        // The reference tests kmin <= kmean <= max(k) (its kmax is shadowed by max(k)),
        // which passes for every kmean >= kmin and reads past the table above kmax.
        // Defined here: the table serves kmean in [kmin, kmax] (the table's bounds);
        // elsewhere the exact 2-D weights at kmean are used, as the RR setup does.
        const double km = sum / s.npb;
        if (s.use_table && s.kmin <= km && km <= s.kmax_tab) {
            int ik = (int)floor((km - s.kmin) / s.dk);
            ik = ik > s.nk - 2 ? s.nk - 2 : ik;
            r->ik = ik;
            r->ak = (km - s.kmin - ik * s.dk) / s.dk;
        } else {
            r->ik = -1;
            r->ak = 0.0;
        }
    }
    __syncthreads();
    if (valid && j < 7) {
        double x, y;
        kepler_xy((j - 3) * 2e-2, s.p[q], a, cos(s.inc[q]), e, s.w[q], x, y);
        s_x[sub][j] = x;
        s_y[sub][j] = y;
    }
    __syncthreads();
    if (valid && j == 0) taylor_from_stencil(s_x[sub], s_y[sub], s_c[sub]);
    __syncthreads();
    if (valid) {
        const double tc = find_contact_point(s_km[sub], j < 4 ? 1 : 4, s_c[sub]);
        if ((j & 3) == 0) s_w[sub][j >> 2] = tc;
    }
    __syncthreads();
    if (valid) {
        TsRec* r = s.rec + q;
        r->c[j] = s_c[sub][j];
        if (j < 2) r->c[8 + j] = s_c[sub][8 + j];
        if (j == 0) r->bt1 = s_w[sub][0] - (0.0015 + s.exptimes[0]);
        if (j == 1) r->bt4 = s_w[sub][1] + (0.0015 + s.exptimes[0]);
    }
}

// Disk integral of (pv, passband) j: given, analytic, or the 200-node trapezoid.
__device__ __forceinline__ void ts_istar(const TsArgs& s, int j) {
    if (j >= s.npv * s.npb) return;
    double is;
    if (s.law == RR_LD_TABULATED) {
        is = s.istar_in[j];
    } else {
        const double* c = s.ldc + (size_t)j * s.nldc;
        if (!ld_integral(s.law, c, is)) {
            double sum = 0.0;
            for (int m = 1; m < 200; ++m) sum += ld_trapz_segment(s.law, c, s.nldc, m);
            is = 2.0 * kPi * sum;
        }
    }
    s.istar[j] = is;
}

// ---- weights at k_mean, transposed: W2T[pv][z][g] --------------------------------------
// A workgroup takes R rows (g values) of one pv.  The exact row
// (calculate_weights_2d, common.py:152-185) is the differences of the lens areas
// at consecutive z edges over their sum.  The areas go to LDS: the cheap cases of
// the lens area (no overlap, one disk inside the other) at once, the (r, z) pairs
// that need the arccos form to a list that all lanes then work through, so no lane
// idles in a wave that evaluates it.  The sum runs over the differences in z order
// as in the reference; the rows' values for one z are written next to each other.
constexpr int kTwMaxRows = 16;
__host__ __device__ inline int ts_weight_rows(int nz) {
    const int r = 2048 / (nz > 0 ? nz : 1);
    return r < 1 ? 1 : (r > kTwMaxRows ? kTwMaxRows : r);
}
// LDS of the exact-weight kernel: areas [R][nz], the list [R][nz] (16-bit, padded
// to 8 bytes), differences [R][nz]
__host__ __device__ inline size_t ts_list_bytes(int nz) {
    return ((size_t)ts_weight_rows(nz) * nz * sizeof(uint16_t) + 7) / 8 * 8;
}
__host__ __device__ inline size_t ts_weights_lds(int nz) {
    return (size_t)ts_weight_rows(nz) * nz * 2 * sizeof(double) + ts_list_bytes(nz);
}

__global__ void __launch_bounds__(256) ts_weights_kernel(TsArgs s) {
    extern __shared__ __align__(16) double s_a[];   // [R][nz] lens areas, the list, the differences
    __shared__ int s_n;
    __shared__ double s_sum[kTwMaxRows];
    const int R = ts_weight_rows(s.nz), nz = s.nz;
    const int nchunk = (s.ngp + R - 1) / R;
    // the launch's first blocks take the disk integrals, a long chain for the laws without
    // an analytic one: first, so that they spread over the CUs (340 x 82 of the power-2-pm
    // law: 343 us so, 343-517 us behind the weights, several to a CU)
    const int nint = (int)(gridDim.x - (unsigned)(s.npv * nchunk)), wb = (int)blockIdx.x - nint;
    if (wb < 0) {
        ts_istar(s, blockIdx.x * blockDim.x + threadIdx.x);
        return;
    }
    const int pv = wb / nchunk;
    const int g0 = (wb - pv * nchunk) * R;
    const int nr = min(R, s.ngp - g0);
    const int tid = threadIdx.x;
    const size_t base = (size_t)pv * s.nzp * s.ngp + g0;
    auto put = [&](int iz, int row, double v) {
        if (s.w2_64) s.w2_64[base + (size_t)iz * s.ngp + row] = v;
        if (s.w2_32) s.w2_32[base + (size_t)iz * s.ngp + row] = (float)v;
    };
    const TsRec& r = s.rec[pv];
    if (r.ik >= 0) {
        // (1-ak) W[ik] + ak W[ik+1] (device table layout [nk][nz][ng])
        const double* w0 = s.W + (size_t)r.ik * nz * s.ng;
        const double* w1 = w0 + (size_t)nz * s.ng;
        for (int i = tid; i < s.nzp * nr; i += blockDim.x) {
            const int iz = i / nr, row = i - iz * nr, ig = g0 + row;
            double v = 0.0;
            if (iz < nz && ig < s.ng) v = (1.0 - r.ak) * w0[(size_t)iz * s.ng + ig] + r.ak * w1[(size_t)iz * s.ng + ig];
            put(iz, row, v);
        }
        return;
    }
    uint16_t* s_list = (uint16_t*)(s_a + (size_t)R * nz);
    __shared__ double s_b[kTwMaxRows];
    const double km = r.kmean;
    if (tid == 0) s_n = 0;
    if (tid < nr) s_b[tid] = linspace_at(0.0, 1.0 - 1e-7, s.ng, g0 + tid) * (1.0 + km);
    __syncthreads();
    auto b_of = [&](int ig) { return s_b[ig - g0]; };
    const int lane = tid % 64;
    for (int i0 = tid - lane; i0 < nr * nz; i0 += blockDim.x) {   // wave-uniform trip count
        const int i = i0 + lane;
        const int row = i / nz, iz = i - row * nz;
        bool listed = false;
        if (i < nr * nz && g0 + row < s.ng) {
            const double b = b_of(g0 + row), r1 = s.ze[iz];
            if (r1 < b - km || r1 >= b + km || b - km <= -r1) s_a[i] = cci_area(r1, km, b);   // cci_area's cheap cases
            else listed = true;
        }
        // one LDS atomic per wave for its listed pairs
        const unsigned long long m = __ballot(listed);
        if (m) {
            const int first = __ffsll((long long)m) - 1;
            int at = 0;
            if (lane == first) at = atomicAdd(&s_n, __popcll(m));
            at = __shfl(at, first, 64);
            if (listed) s_list[at + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)i;
        }
    }
    __syncthreads();
    const int nl = s_n;
    for (int j = tid; j < nl; j += blockDim.x) {
        const int i = s_list[j], row = i / nz, iz = i - row * nz;
        s_a[i] = cci_area(s.ze[iz], km, b_of(g0 + row));
    }
    __syncthreads();
    // the differences, all at once, then each row's sum over them in z order
    double* s_d = (double*)((unsigned char*)s_list + ts_list_bytes(nz));
    for (int i = tid; i < nr * nz; i += blockDim.x) {
        const int iz = i % nz;
        s_d[i] = iz == 0 ? s_a[i] : s_a[i] - s_a[i - 1];
    }
    __syncthreads();
    if (tid < nr) {
        double sum = 0.0;
        if (g0 + tid < s.ng) {
            const double* d = s_d + (size_t)tid * nz;
#pragma unroll 8
            for (int iz = 0; iz < nz; ++iz) sum += d[iz];
        }
        s_sum[tid] = sum;
    }
    __syncthreads();
    for (int i = tid; i < s.nzp * nr; i += blockDim.x) {
        const int iz = i / nr, row = i - iz * nr;
        double v = 0.0;
        if (iz < nz && g0 + row < s.ng) v = s_d[(size_t)row * nz + iz] / s_sum[row];
        put(iz, row, v);
    }
}

// Profile value of (pv, pb) at mu node iz: a table read, or the named law (the
// template keeps the law code out of the table-read kernels' registers).
template <bool kTab>
__device__ __forceinline__ double ts_profile(const TsArgs& s, int pv, int pb, int iz) {
    const size_t j = (size_t)pv * s.npb + pb;
    if (kTab) return s.ldp_in[j * s.nz + iz];
    return ld_law(s.law, s.mu[iz], s.ldc + j * s.nldc, s.nldc);
}

// ---- FP32 MFMA contraction: ldm[pv][pb][g] = sum_z ldp[pv][pb][z] * W2T[pv][z][g] ----
// D(16x16) += A(16x4) B(4x16) per v_mfma_f32_16x16x4f32.  Lane l supplies
// A[l%16][l/16] and B[l/16][l%16] and holds D[4*(l/16)+r][l%16], r = 0..3.
// A rows are passbands, B columns are g.  W2T of the pv sits in LDS with a padded
// row stride so the 16 lanes reading one k hit distinct banks.
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// LDS row stride of W2T: a 16-byte multiple, 4 mod 8 floats, so that the four z rows of
// an MFMA step are in distinct banks.
__host__ __device__ inline int ts_tab_ldb(int ngp) { return ngp + ((4 - ngp % 8) + 8) % 8; }

template <bool kTab>
__global__ void __launch_bounds__(256) ts_ldm_mfma_kernel(TsArgs s) {
    extern __shared__ float lds_b[];  // [nzp][ldb]
    const int pv = blockIdx.x / s.ldm_split, part = blockIdx.x - pv * s.ldm_split;
    const int ldb = ts_tab_ldb(s.ngp);
    const f32x4_t* w2 = (const f32x4_t*)(s.w2_32 + (size_t)pv * s.nzp * s.ngp);
#pragma unroll 4
    for (int i = threadIdx.x; i < s.nzp * s.ngp / 4; i += 256) {
        const int iz = 4 * i / s.ngp;
        *(f32x4_t*)(lds_b + iz * ldb + 4 * i - iz * s.ngp) = w2[i];
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int nrt = (s.npb + 15) / 16, nct = s.ngp / 16;
    for (int rt = part * 4 + wave; rt < nrt; rt += 4 * s.ldm_split) {
        const int pb = rt * 16 + li;
        const bool row_ok = pb < s.npb;
        for (int ct0 = 0; ct0 < nct; ct0 += 8) {
            f32x4_t acc[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) acc[c] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
            // four steps' profile values at a time, their loads in flight together
            constexpr int kU = 4;
            for (int k0 = 0; k0 < s.nzp; k0 += 4 * kU) {
                float a[kU];
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    const int iz = k0 + 4 * u + lk;
                    a[u] = (row_ok && iz < s.nz) ? (float)ts_profile<kTab>(s, pv, pb, iz) : 0.0f;
                }
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    if (k0 + 4 * u >= s.nzp) break;
                    const int iz = k0 + 4 * u + lk;
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const int ct = ct0 + c;
                        if (ct < nct) {
                            const float b = lds_b[iz * ldb + ct * 16 + li];
                            acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b, acc[c], 0, 0, 0);
                        }
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int ct = ct0 + c;
                if (ct >= nct) break;
                const int g = ct * 16 + li;
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) {
                    const int pbo = rt * 16 + lk * 4 + rr;
                    if (pbo < s.npb && g < s.ng) s.ldm32[((size_t)pv * s.npb + pbo) * s.ng + g] = acc[c][rr];
                }
            }
        }
    }
}

// ---- FP32 MFMA contraction of tabulated FP64 profiles, row-contiguous loads ---------
// ldm[pv][pb][g] = sum_z ldp[pv][pb][z] W2T[pv][z][g] for profiles given as an
// FP64 table (the TSModel's LDModel input).  One workgroup of 8 waves per pv with
// W2T in LDS; a wave takes one 16-passband row tile at a time.  The sum over z is
// taken in a permuted order: lane (li, lk) holds row li at z = 16 j + 4 lk + q for
// MFMA step 4 j + q, so each lane loads 4 consecutive FP64 values (two 16-byte
// loads) and the four lanes of a row read 128 contiguous bytes; the B fragment
// reads of LDS follow the same permutation.  The LDS row stride (4 mod 8 floats)
// puts the four z rows of an MFMA step in distinct banks.
typedef double f64x2_t __attribute__((ext_vector_type(2)));
constexpr int kTabMfmaThreads = 512;
constexpr int kTabMfmaMaxJ = 8;    // z groups of 16: nz <= 128
constexpr int kTabMfmaMaxCt = 8;   // g tiles of 16: ngp <= 128

template <int NCT>
__global__ void __launch_bounds__(kTabMfmaThreads) ts_ldm_tab_mfma_kernel(TsArgs s) {
    extern __shared__ float lds_t[];  // [nz16][ldb]
    const int pv = blockIdx.x / s.ldm_split, part = blockIdx.x - pv * s.ldm_split;
    const int ldb = ts_tab_ldb(s.ngp);
    const int nj = (s.nz + 15) / 16, nz16 = nj * 16;
    // (ngp a multiple of 16 and ldb of 4: 16-byte pieces of one row)
    const f32x4_t* w2 = (const f32x4_t*)(s.w2_32 + (size_t)pv * s.nzp * s.ngp);
#pragma unroll 4
    for (int i = threadIdx.x; i < nz16 * s.ngp / 4; i += kTabMfmaThreads) {
        const int iz = 4 * i / s.ngp;
        const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
        const f32x4_t v = iz < s.nzp ? w2[i] : zero;
        *(f32x4_t*)(lds_t + iz * ldb + 4 * i - iz * s.ngp) = v;
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int nrt = (s.npb + 15) / 16;
    constexpr int kWaves = kTabMfmaThreads / 64;
    for (int rt = part * kWaves + wave; rt < nrt; rt += kWaves * s.ldm_split) {
        const int pb = rt * 16 + li;
        const bool row_ok = pb < s.npb;
        const double* arow = s.ldp_in + ((size_t)pv * s.npb + (row_ok ? pb : 0)) * s.nz;
        f32x4_t acc[NCT];
#pragma unroll
        for (int c = 0; c < NCT; ++c) acc[c] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
        // the row in two halves of 64 z values: 16 FP64 values in flight per lane
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            constexpr int kJh = kTabMfmaMaxJ / 2;
            float af[4 * kJh];
#pragma unroll
            for (int jj = 0; jj < kJh; ++jj) {
                const int j = h * kJh + jj, z0 = 16 * j + 4 * lk;
                f64x2_t v0 = {0.0, 0.0}, v1 = {0.0, 0.0};
                if (j < nj && row_ok && z0 < s.nz) {
                    v0 = *(const f64x2_t*)(arow + z0);
                    v1 = *(const f64x2_t*)(arow + z0 + 2);
                }
                af[4 * jj + 0] = (float)v0.x;
                af[4 * jj + 1] = (float)v0.y;
                af[4 * jj + 2] = (float)v1.x;
                af[4 * jj + 3] = (float)v1.y;
            }
#pragma unroll
            for (int jj = 0; jj < kJh; ++jj) {
                const int j = h * kJh + jj;
                if (j < nj) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float* brow = lds_t + (16 * j + 4 * lk + q) * ldb + li;
#pragma unroll
                        for (int c = 0; c < NCT; ++c)
                            acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[4 * jj + q], brow[c * 16], acc[c], 0, 0,
                                                                          0);
                    }
                }
            }
        }
#pragma unroll
        for (int c = 0; c < NCT; ++c) {
            const int g = c * 16 + li;
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) {
                const int pbo = rt * 16 + lk * 4 + rr;
                if (pbo < s.npb && g < s.ng) s.ldm32[((size_t)pv * s.npb + pbo) * s.ng + g] = acc[c][rr];
            }
        }
    }
}

// ---- FP64 MFMA contraction (v_mfma_f64_16x16x4f64), same tiling as the FP32 one ---------
// Lane l supplies A[l%16][l/16] and B[l/16][l%16] and holds D[(l/16)+4r][l%16]:
// unlike the FP32 16x16x4 form, the four result rows of a lane are interleaved.
// One workgroup of 8 waves per pv; W2T (FP64) sits in LDS with a padded row stride.
typedef double f64x4_t __attribute__((ext_vector_type(4)));
constexpr int kMfma64Threads = 512;
constexpr size_t kMfma64MaxLds = 128 * 1024;

template <bool kTab>
__global__ void __launch_bounds__(kMfma64Threads) ts_ldm_mfma64_kernel(TsArgs s) {
    extern __shared__ double lds_b64[];  // [nzp][ngp + 1]
    const int pv = blockIdx.x / s.ldm_split, part = blockIdx.x - pv * s.ldm_split;
    const int ldb = s.ngp + 1;
    // (ngp a multiple of 16: pairs of one row, several loads in flight)
    const f64x2_t* w2 = (const f64x2_t*)(s.w2_64 + (size_t)pv * s.nzp * s.ngp);
#pragma unroll 4
    for (int i = threadIdx.x; i < s.nzp * s.ngp / 2; i += kMfma64Threads) {
        const f64x2_t v = w2[i];
        const int iz = 2 * i / s.ngp, o = iz * ldb + 2 * i - iz * s.ngp;
        lds_b64[o] = v.x;
        lds_b64[o + 1] = v.y;
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int nrt = (s.npb + 15) / 16, nct = s.ngp / 16;
    constexpr int kWaves = kMfma64Threads / 64;
    for (int rt = part * kWaves + wave; rt < nrt; rt += kWaves * s.ldm_split) {
        const int pb = rt * 16 + li;
        const bool row_ok = pb < s.npb;
        for (int ct0 = 0; ct0 < nct; ct0 += 8) {
            f64x4_t acc[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) acc[c] = (f64x4_t){0.0, 0.0, 0.0, 0.0};
            // four steps' profile values at a time, their loads in flight together
            constexpr int kU = 4;
            for (int k0 = 0; k0 < s.nzp; k0 += 4 * kU) {
                double a[kU];
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    const int iz = k0 + 4 * u + lk;
                    a[u] = (row_ok && iz < s.nz) ? ts_profile<kTab>(s, pv, pb, iz) : 0.0;
                }
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    if (k0 + 4 * u >= s.nzp) break;
                    const int iz = k0 + 4 * u + lk;
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const int ct = ct0 + c;
                        if (ct < nct) {
                            const double b = lds_b64[iz * ldb + ct * 16 + li];
                            acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b, acc[c], 0, 0, 0);
                        }
                    }
                }
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int ct = ct0 + c;
                if (ct >= nct) break;
                const int g = ct * 16 + li;
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) {
                    const int pbo = rt * 16 + lk + 4 * rr;
                    if (pbo < s.npb && g < s.ng) s.ldm64[((size_t)pv * s.npb + pbo) * s.ng + g] = acc[c][rr];
                }
            }
        }
    }
}

// ---- FP64 contraction on the vector ALUs: one lane per (pv, pb, g) --------------------
template <bool kTab>
__global__ void __launch_bounds__(256) ts_ldm_f64_kernel(TsArgs s) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)s.npv * s.npb * s.ng) return;
    const int ig = (int)(idx % s.ng);
    const long long j = idx / s.ng;
    const int pv = (int)(j / s.npb), pb = (int)(j - (long long)pv * s.npb);
    const double* w = s.w2_64 + (size_t)pv * s.nzp * s.ngp + ig;
    double d = 0.0;
    for (int iz = 0; iz < s.nz; ++iz) d += w[(size_t)iz * s.ngp] * ts_profile<kTab>(s, pv, pb, iz);
    s.ldm64[idx] = d;
}

// The FP32 weights (W2T of the mixed path) when W2T does not fit the MFMA kernel's
// LDS: one lane per (pv, passband, g), the sum in FP64, the mean stored in FP32.
template <bool kTab>
__global__ void __launch_bounds__(256) ts_ldm_f32_kernel(TsArgs s) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)s.npv * s.npb * s.ng) return;
    const int ig = (int)(idx % s.ng);
    const long long j = idx / s.ng;
    const int pv = (int)(j / s.npb), pb = (int)(j - (long long)pv * s.npb);
    const float* w = s.w2_32 + (size_t)pv * s.nzp * s.ngp + ig;
    double d = 0.0;
    for (int iz = 0; iz < s.nz; ++iz) d += w[(size_t)iz * s.ngp] * ts_profile<kTab>(s, pv, pb, iz);
    s.ldm32[idx] = (float)d;
}

// ---- a law linear in its coefficients ----------------------------------------------
//
// Its basis functions are the same for every passband: a workgroup contracts the nb of
// them with the pv's weights into M_b(g) in LDS and writes ldm = sum_b coef_b M_b(g) of
// its passbands in order, in place of npb contractions of nz nodes.  FP64 sums, FP32
// means.  Quadratic law, mixed, whole call against the MFMA contraction: 300 x 512 x
// 1,000 230 -> 186 us, 1,024 x 512 x 1,000 645 -> 584, 8 x 200 x 1,237 39.7 -> 37.6.  FP64
// stays on MFMA: 100 x 203 x 1,237 x 3 96.6 us, 100.6 in this form.
// The nodes are split over the parts of a workgroup that its lanes over g leave.
__host__ __device__ inline int ts_basis_parts(int ng) {
    const int gw = (ng + 63) / 64 * 64;
    return gw >= 256 ? 1 : 256 / gw;
}
__host__ __device__ inline size_t ts_basis_lds(int nb, int nz, int ng, int pbs) {
    return (size_t)nb * (nz + ts_basis_parts(ng) * ng + pbs) * sizeof(double);
}

__global__ void __launch_bounds__(256) ts_ldm_basis_kernel(TsArgs s, int nb) {
    extern __shared__ double lds_basis[];
    const int pv = blockIdx.x / s.ldm_split, part = blockIdx.x - pv * s.ldm_split, tid = threadIdx.x;
    const int per = (s.npb + s.ldm_split - 1) / s.ldm_split, pa = min(part * per, s.npb), np = min(per, s.npb - pa);
    const int nz = s.nz, ng = s.ng, parts = ts_basis_parts(ng);
    double* s_B = lds_basis;                     // [nb][nz]
    double* s_M = s_B + nb * nz;                 // [parts][nb][ng]
    double* s_c = s_M + parts * nb * ng;         // [np][nb]
    const size_t j0 = (size_t)pv * s.npb + pa;
    for (int i = tid; i < nb * nz; i += 256) s_B[i] = ld_basis(s.law, i / nz, s.mu[i % nz]);
    for (int i = tid; i < np * nb; i += 256) s_c[i] = ld_basis_coef(s.law, i % nb, s.ldc + (j0 + i / nb) * s.nldc);
    __syncthreads();
    const float* w = s.w2_32 + (size_t)pv * s.nzp * s.ngp;
    const int gw = 256 / parts, zp = tid / gw, zn = (nz + parts - 1) / parts, za = zp * zn, ze = min(za + zn, nz);
    for (int g = tid - zp * gw; g < ng; g += gw) {
        double m[kMaxBasis];
#pragma unroll
        for (int b = 0; b < kMaxBasis; ++b) m[b] = 0.0;
        constexpr int kB = 20;                   // loads in flight
        for (int z0 = za; z0 < ze; z0 += kB) {
            float v[kB];
#pragma unroll
            for (int u = 0; u < kB; ++u) v[u] = w[(size_t)min(z0 + u, ze - 1) * s.ngp + g];
#pragma unroll
            for (int u = 0; u < kB; ++u) {
                if (z0 + u < ze) {
#pragma unroll
                    for (int b = 0; b < kMaxBasis; ++b)
                        if (b < nb) m[b] += (double)v[u] * s_B[b * nz + z0 + u];
                }
            }
        }
#pragma unroll
        for (int b = 0; b < kMaxBasis; ++b)
            if (b < nb) s_M[(zp * nb + b) * ng + g] = m[b];
    }
    __syncthreads();
    for (int i = tid; i < nb * ng; i += 256)
        for (int p = 1; p < parts; ++p) s_M[i] += s_M[p * nb * ng + i];
    __syncthreads();
    for (int i = tid; i < np * ng; i += 256) {
        const int q = i / ng, g = i - q * ng;
        double v = 0.0;
        for (int b = 0; b < nb; ++b) v += s_c[q * nb + b] * s_M[b * ng + g];
        s.ldm32[j0 * ng + i] = (float)v;
    }
}

// ---- flux --------------------------------------------------------------------------
constexpr int kTsThreads = 256;

// Passbands per LDS chunk where a lane keeps one accumulator per passband.
constexpr int ts_pb_chunk(bool mixed) { return mixed ? 32 : 16; }

// Geometry of one (time, sample): the lens at k_mean in FP64 (model_trspec.py:79-84)
// and the lerp position in g; shared by every passband.
template <typename Real>
struct TsGeo {
    Real ra, rb;      // lerp weights of l[ig + 1] and l[ig]
    Real ap0, dadk;   // area at k_mean and its k-derivative 2 k_mean kappa_0
    int ig;
    bool inside;      // z <= 1 - k_max: area scales as k^2 / k_mean^2
    bool gz;          // g > 1: the limb-darkening mean is 0
};

// inv_1pk, inv_dg and inv_ns: the reciprocals of 1 + k_mean, dg and nsamples.
template <typename Real>
__device__ __forceinline__ TsGeo<Real> ts_geometry(const TsRec& r, double tc, double ext, double inv_ns, int is,
                                                   double inv_1pk, double inv_dg, int ng) {
    TsGeo<Real> o;
    const double km = r.kmean;
    const double z = sample_z(sample_time(tc, ext, inv_ns, is), r.c);
    double ap0, kap;
    if (fabs(1.0 - km) < z && z < 1.0 + km) {
        double akite;
        ap0 = lens_f64(km, z, kap, akite);
    } else {
        ccia_kite<double>(1.0, km, z, ap0, kap);     // off the disk, inside it, NaN
    }
    o.inside = z <= 1.0 - r.kmax;
    const double g = z * inv_1pk;
    // lerp position (common.py:225-233, index clamped to ng-2)
    o.gz = g > 1.0;
    o.ig = 0;
    double al = 0.0;
    if (!o.gz) {
        const double x = g * inv_dg;
        const int ig = (int)x;
        o.ig = ig > ng - 2 ? ng - 2 : (ig < 0 ? 0 : ig);
        al = x - o.ig;
    }
    o.ra = (Real)al;
    o.rb = (Real)(1.0 - al);
    o.ap0 = (Real)ap0;
    o.dadk = (Real)(2.0 * km * kap);
    return o;
}

// times per lane of the row forms: one 16-byte store per passband row
template <typename Real> constexpr int ts_tpl() { return 16 / (int)sizeof(Real); }

template <typename Real>
__device__ __forceinline__ void ts_store(Real* o, const Real* v) {
    if constexpr (std::is_same<Real, float>::value) {
        const f32x4_t w = {v[0], v[1], v[2], v[3]};
        __builtin_nontemporal_store(w, (f32x4_t*)o);
    } else {
        const f64x2_t w = {v[0], v[1]};
        __builtin_nontemporal_store(w, (f64x2_t*)o);
    }
}

// ---- one sample, 32 whole rows a workgroup, written in order ----------------------------
//
// The tile form below has each workgroup write a piece of every passband row (rows npt
// apart), and HBM takes such strided pieces at ~4.3 TB/s where it takes the same bytes
// written in address order at ~5.3 TB/s.  With one sample and npt <= 8192 (FP64 6144;
// the usual transmission-spectroscopy shape: a few thousand times, hundreds of
// passbands) a workgroup of 1024 threads writes up to 32 rows of a pv front to back:
// thread i owns the 16-byte time vectors i, i + 1024 and so on of every row, and each
// step writes one whole row.
//
// A row costs few operations per value: the geometry of each time is reduced once
// to the LDS offset of its limb-darkening interval and five coefficients, with
//   I = rb l[ig] + ra l[ig+1],  area = c1 afac + (c2 + c3 (k - k_mean)),
//   F = 1 - (I area) / I*
// (c1 = A0 inside z <= 1 - k_max, else c2 = A0 and c3 = 2 k_mean kappa0, the
// serial model's two branches); outside the window, and for g > 1 where both the
// mean and the area vanish, F = 1 is selected, so a NaN row of limb-darkening
// means reaches only the in-window values, as in the reference.  The passbands' LD
// rows sit in LDS transposed, passband fastest, so the rows of a 16-passband group
// are read with immediate offsets from one address; the row stride is 33 values, so
// lanes reading different g hit different banks (a stride of 32 would put every lane
// of a row read in one bank).  A wave none of whose times is in the window stores
// ones without arithmetic.
constexpr int kTsRowThreads = 1024;
constexpr int kTsRowPc = 32;      // passbands of a workgroup
constexpr int kTsRowLd = kTsRowPc + 1;   // LDS stride of one g
constexpr int kTsRowQ = 16;       // passbands per unrolled group
// time vectors (16 bytes: 4 FP32 or 2 FP64 times) per thread; npt <= 8192 (FP32), 6144 (FP64)
template <typename Real> constexpr int ts_row_vec() { return sizeof(Real) == 4 ? 2 : 3; }
template <typename Real> constexpr int ts_row_max_npt() { return kTsRowThreads * ts_row_vec<Real>() * ts_tpl<Real>(); }
// finer g grids go to the tiles: the line of a workgroup that held 64 passbands' rows in
// 64 KB, not moved since
template <typename Real> constexpr int ts_row_max_ng() { return sizeof(Real) == 4 ? 249 : 123; }

__host__ __device__ inline size_t ts_rows_lds(int ng, size_t real) { return ((size_t)kTsRowLd * ng + 3 * kTsRowPc) * real; }

// A workgroup's pv and passband range, row_split to a pv.
__device__ __forceinline__ void ts_row_range(const TsArgs& s, int bid, int& pv, int& qa, int& qb) {
    pv = bid / s.row_split;
    const int part = bid - pv * s.row_split, per = (s.npb + s.row_split - 1) / s.row_split;
    qa = min(part * per, s.npb);
    qb = min(qa + per, s.npb);
}

template <typename Real>
__global__ void __launch_bounds__(kTsRowThreads) ts_flux_rows_kernel(TsArgs s, Real* flux) {
    constexpr int TPL = ts_tpl<Real>();
    constexpr int NV = ts_row_vec<Real>();
    extern __shared__ __align__(16) unsigned char lds[];
    Real* s_ldm = (Real*)lds;                        // [ng][kTsRowLd]
    Real* s_afac = s_ldm + (size_t)kTsRowLd * s.ng;
    Real* s_kd = s_afac + kTsRowPc;
    Real* s_iist = s_kd + kTsRowPc;

    int pv, qa, qb;      // this workgroup's pv and passbands
    ts_row_range(s, xcd_remap(blockIdx.x, gridDim.x), pv, qa, qb);
    const int npt = s.npt, nv = npt / TPL;
    const TsRec& r = s.rec[pv];
    Real* out = flux + (size_t)pv * s.npb * npt;
    Real vnan[TPL], vone[TPL];
#pragma unroll
    for (int j = 0; j < TPL; ++j) {
        vnan[j] = Real(NAN);
        vone[j] = Real(1);
    }
    if (!r.good) {
        for (size_t i = (size_t)qa * nv + threadIdx.x; i < (size_t)qb * nv; i += kTsRowThreads)
            ts_store(out + i * TPL, vnan);
        return;
    }
    // the geometry of the thread's times, once, as row coefficients
    const double ext = s.exptimes[0];
    const double inv_1pk = 1.0 / (1.0 + r.kmean), inv_dg = 1.0 / s.dg;
    int off[NV][TPL];
    Real rb[NV][TPL], ra[NV][TPL], c1[NV][TPL], c2[NV][TPL], c3[NV][TPL];
    bool use[NV][TPL];   // in the window with g <= 1
    bool act[NV];        // the wave has a time of vector u in the window
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int v = threadIdx.x + u * kTsRowThreads;
        bool any = false;
#pragma unroll
        for (int j = 0; j < TPL; ++j) {
            off[u][j] = 0;
            rb[u][j] = ra[u][j] = c1[u][j] = c2[u][j] = c3[u][j] = Real(0);
            use[u][j] = false;
            if (v < nv) {
                double ep;
                const double tc = epoch_phase(s.times[TPL * v + j], s.t0[pv], r.p, r.inv_p, ep);
                if ((r.bt1 <= tc) && (tc <= r.bt4)) {
                    const TsGeo<Real> g = ts_geometry<Real>(r, tc, ext, 1.0, 0, inv_1pk, inv_dg, s.ng);
                    any = true;
                    if (!g.gz) {
                        use[u][j] = true;
                        off[u][j] = g.ig * kTsRowLd;
                        rb[u][j] = g.rb;
                        ra[u][j] = g.ra;
                        c1[u][j] = g.inside ? g.ap0 : Real(0);
                        c2[u][j] = g.inside ? Real(0) : g.ap0;
                        c3[u][j] = g.inside ? Real(0) : g.dadk;
                    }
                }
            }
        }
        act[u] = __ballot(any) != 0ull;
    }
    const int npc = qb - qa;     // at most kTsRowPc
    for (int i = threadIdx.x; i < npc * s.ng; i += kTsRowThreads) {
        const int q = i / s.ng, g = i - q * s.ng;   // coalesced global reads along g
        const size_t src = ((size_t)pv * s.npb + qa + q) * s.ng + g;
        s_ldm[g * kTsRowLd + q] = sizeof(Real) == 4 ? (Real)s.ldm32[src] : (Real)s.ldm64[src];
    }
    for (int q = threadIdx.x; q < npc; q += kTsRowThreads) {
        const double kq = s.k[(size_t)pv * s.npb + qa + q];
        s_afac[q] = (Real)(kq * kq / (r.kmean * r.kmean));
        s_kd[q] = (Real)(kq - r.kmean);
        s_iist[q] = (Real)(1.0 / s.istar[(size_t)pv * s.npb + qa + q]);
    }
    __syncthreads();
#pragma unroll 1
    for (int q0 = 0; q0 < npc; q0 += kTsRowQ) {
        const Real* lq = s_ldm + q0;
#pragma unroll
        for (int qq = 0; qq < kTsRowQ; ++qq) {
            const int q = q0 + qq;
            if (q < npc) {
                const Real f = s_iist[q], afac = s_afac[q], kd = s_kd[q];
                Real* o = out + (size_t)(qa + q) * npt;
#pragma unroll
                for (int u = 0; u < NV; ++u) {
                    const int v = threadIdx.x + u * kTsRowThreads;
                    if (v < nv) {
                        if (act[u]) {
                            Real w[TPL];
#pragma unroll
                            for (int j = 0; j < TPL; ++j) {
                                const Real* l = lq + off[u][j] + qq;
                                const Real ip = rb[u][j] * l[0] + ra[u][j] * l[kTsRowLd];
                                const Real area = c1[u][j] * afac + (c2[u][j] + c3[u][j] * kd);
                                w[j] = use[u][j] ? Real(1) - (ip * area) * f : Real(1);
                            }
                            ts_store(o + (size_t)v * TPL, w);
                        } else {
                            ts_store(o + (size_t)v * TPL, vone);
                        }
                    }
                }
            }
        }
    }
}

// ---- FP32 rows in whole cache lines ----------------------------------------------------
//
// A row of npt FP32 values starts 4 (R npt mod 32) bytes past a 128-byte boundary
// (R the row's index in the flux array).  In the row form above, thread i owns the
// same time vectors in every row, so in a row that starts off a boundary every
// wave's 1 KB store straddles cache lines, and HBM takes those pieces at ~4.0
// TB/s against ~4.9 TB/s for whole lines (the same kernel at npt = 5000 and 4992).
// Here the geometry of every time is reduced once to its row coefficients in an
// LDS table, one array per coefficient, and in each row slot s takes time vector
// (s + head) mod nv, head being the number of 16-byte vectors before the row's
// first 128-byte boundary: the 64 slots of a wave then cover one aligned
// kilobyte.  Rows P = 32 / gcd(npt, 32) apart have the same head and share one
// load of the coefficients from the table into registers; the per-value
// arithmetic is the row form's.
//
// Bound by HBM's writes, whose rate falls with the span that is being written: a
// workgroup takes 32 rows of one segment of at most 512 slots, and neighbouring
// workgroups the segments of the same rows.  1024 pv x 512 x 5,000 (10.5 GB), whole
// call, against one workgroup of 1024 lanes per pv (2410 us): 64 rows 2357, 32 rows
// 2286, 16 rows 3363 (too few rows to a load of the coefficients); 300 x 512 x 5,000
// 746 -> 697 us, 500 x 200 x 1,236 262 -> 225.  Its table is computed by each workgroup
// (the cores are idle three quarters of the time): one made once per pv and read from
// memory was slower, 2405 us.
constexpr int kTsLine = 32;   // FP32 values per 128-byte cache line
constexpr int kTsAlThreads = 512;
constexpr int kTsAlPc = 32;        // passbands of a workgroup
constexpr int kTsAlLd = kTsAlPc + 1;   // LDS stride of one g
constexpr int kTsStageRegs = 8;    // LD values per thread: kTsAlPc x ng <= 8 x 512
constexpr size_t kTsRowsAlignedMaxLds = 160 * 1024;

__host__ __device__ inline size_t ts_rows_table_offset(int ng) {
    return (((size_t)kTsAlLd * ng + 3 * kTsAlPc) * 4 + 15) / 16 * 16;
}
// Vector slots of a segment of a row of nv, a multiple of a wave, and the segments of the row.
__host__ __device__ inline int ts_segments(int nv) { return (nv + kTsAlThreads - 1) / kTsAlThreads; }
__host__ __device__ inline int ts_segment_slots(int nv) {
    const int n = ts_segments(nv);
    return ((nv + n - 1) / n + 63) / 64 * 64;
}
// Values of a segment's table: its slots' vectors under every rotation (0 to 7 vectors).
__host__ __device__ inline int ts_segment_values(int nv) { return 4 * (ts_segment_slots(nv) + 8); }
__host__ __device__ inline size_t ts_rows_aligned_lds(int ng, int npt) {
    return ts_rows_table_offset(ng) + (size_t)ts_segment_values(npt / 4) * 5 * 4;
}

// The row coefficients of time `it` of a pv: LDS offset << 2 | inside << 1 | use, the lerp
// weights, the area at k_mean and its k-derivative.
__device__ __forceinline__ void ts_row_coefficients(const TsArgs& s, const TsRec& r, double t0v, double ext, double inv_1pk,
                                                    double inv_dg, int it, int& pk, float& ra, float& rb, float& a0,
                                                    float& dk) {
    double ep;
    const double tc = epoch_phase(s.times[it], t0v, r.p, r.inv_p, ep);
    pk = 0;
    ra = rb = a0 = dk = 0.0f;
    if ((r.bt1 <= tc) && (tc <= r.bt4)) {
        const TsGeo<float> g = ts_geometry<float>(r, tc, ext, 1.0, 0, inv_1pk, inv_dg, s.ng);
        if (!g.gz) {
            pk = ((g.ig * kTsAlLd) << 2) | (g.inside ? 2 : 0) | 1;
            ra = g.ra;
            rb = g.rb;
            a0 = g.ap0;
            dk = g.dadk;
        }
    }
}

// Four waves a SIMD: two workgroups a CU, though the registers would let three or four
// in, which widens the span being written (1024 pv x 512 x 1,000: 553 us, 561 with 7).
__global__ void __launch_bounds__(kTsAlThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
ts_flux_rows_aligned_kernel(TsArgs s, float* flux) {
    using Real = float;
    constexpr int TPL = ts_tpl<float>();
    extern __shared__ __align__(16) unsigned char lds[];
    Real* s_ldm = (Real*)lds;                        // [ng][kTsAlLd]
    Real* s_afac = s_ldm + (size_t)kTsAlLd * s.ng;
    Real* s_kd = s_afac + kTsAlPc;
    Real* s_iist = s_kd + kTsAlPc;
    const int npt = s.npt, nv = npt / TPL, ntab = ts_segment_values(nv);
    // the row coefficients of every time: LDS offset << 2 | inside << 1 | use, and
    // the lerp weights, the area at k_mean and its k-derivative
    int* t_pk = (int*)(lds + ts_rows_table_offset(s.ng));
    Real* t_ra = (Real*)(t_pk + ntab);
    Real* t_rb = t_ra + ntab;
    Real* t_a0 = t_rb + ntab;
    Real* t_dk = t_a0 + ntab;

    // this workgroup's pv, passbands and segment of the rows: slots v0 .. v0 + nslots
    int pv, qa, qb;
    const int bid = xcd_remap(blockIdx.x, gridDim.x), nseg = ts_segments(nv), seg = bid % nseg;
    ts_row_range(s, bid / nseg, pv, qa, qb);
    const int v0 = seg * ts_segment_slots(nv), nslots = min(ts_segment_slots(nv), nv - v0);
    const int tid = threadIdx.x;
    const TsRec& r = s.rec[pv];
    float* out = flux + (size_t)pv * s.npb * npt;
    if (!r.good) {
        const f32x4_t vnan = {NAN, NAN, NAN, NAN};
        for (int q = qa; q < qb; ++q)
            if (tid < nslots) __builtin_nontemporal_store(vnan, (f32x4_t*)(out + ((size_t)q * nv + v0 + tid) * TPL));
        return;
    }
    const int npc = qb - qa;         // at most kTsAlPc
    const double ext = s.exptimes[0];
    const double inv_1pk = 1.0 / (1.0 + r.kmean), inv_dg = 1.0 / s.dg;
    const double t0v = s.t0[pv];
    for (int t = tid; t < 4 * (nslots + 8); t += kTsAlThreads) {
        const int tv = 4 * v0 + t;      // the row's values go round
        int pk;
        Real ra, rb, a0, dk;
        ts_row_coefficients(s, r, t0v, ext, inv_1pk, inv_dg, tv < npt ? tv : tv - npt, pk, ra, rb, a0, dk);
        t_pk[t] = pk;
        t_ra[t] = ra;
        t_rb[t] = rb;
        t_a0[t] = a0;
        t_dk[t] = dk;
    }
    // the LD rows and the passbands' k and disk integrals: all loads in flight together
    float st[kTsStageRegs];
#pragma unroll
    for (int m = 0; m < kTsStageRegs; ++m) {
        const int i = tid + m * kTsAlThreads;
        st[m] = i < npc * s.ng ? s.ldm32[((size_t)pv * s.npb + qa) * s.ng + i] : 0.0f;
    }
    double kq = 0.0, isq = 1.0;
    if (tid < npc) {
        kq = s.k[(size_t)pv * s.npb + qa + tid];
        isq = s.istar[(size_t)pv * s.npb + qa + tid];
    }
#pragma unroll
    for (int m = 0; m < kTsStageRegs; ++m) {
        const int i = tid + m * kTsAlThreads;
        const int q = i / s.ng, g = i - q * s.ng;
        if (i < npc * s.ng) s_ldm[g * kTsAlLd + q] = st[m];
    }
    if (tid < npc) {
        s_afac[tid] = (Real)(kq * kq / (r.kmean * r.kmean));
        s_kd[tid] = (Real)(kq - r.kmean);
        s_iist[tid] = (Real)(1.0 / isq);
    }
    __syncthreads();
    // rows P apart start equally far past a 128-byte boundary
    const int gl = npt & -npt;   // lowest set bit of npt
    const int P = kTsLine / (gl < kTsLine ? gl : kTsLine);
    for (int q0 = 0; q0 < min(P, npc); ++q0) {
        // this class's head, and each slot's coefficients from the table
        const int mis = (int)(((uintptr_t)(out + (size_t)(qa + q0) * npt) >> 2) & (kTsLine - 1));
        const int head = ((kTsLine - mis) & (kTsLine - 1)) / TPL;
        // per value: LDS offset, lerp weights, the area at k_mean (negated when
        // the planet is inside the disk, where it scales by afac) and its
        // k-derivative (0 inside); bit j of `use` marks a value in the
        // window with g <= 1
        const int lv = tid + head, vi = v0 + lv < nv ? v0 + lv : v0 + lv - nv;
        int off[TPL];
        Real rb[TPL], ra[TPL], as[TPL], dk[TPL];
        unsigned use = 0u;
#pragma unroll
        for (int j = 0; j < TPL; ++j) {
            off[j] = 0;
            ra[j] = rb[j] = as[j] = dk[j] = Real(0);
        }
        if (tid < nslots) {
            const int4 pk4 = *(const int4*)(t_pk + TPL * lv);
            const f32x4_t ra4 = *(const f32x4_t*)(t_ra + TPL * lv);
            const f32x4_t rb4 = *(const f32x4_t*)(t_rb + TPL * lv);
            const f32x4_t a04 = *(const f32x4_t*)(t_a0 + TPL * lv);
            const f32x4_t dk4 = *(const f32x4_t*)(t_dk + TPL * lv);
            const int pk[TPL] = {pk4.x, pk4.y, pk4.z, pk4.w};
#pragma unroll
            for (int j = 0; j < TPL; ++j) {
                const bool inside = (pk[j] & 2) != 0;
                if (pk[j] & 1) use |= 1u << j;
                off[j] = pk[j] >> 2;
                ra[j] = ra4[j];
                rb[j] = rb4[j];
                as[j] = inside ? -a04[j] : a04[j];
                dk[j] = inside ? Real(0) : dk4[j];
            }
        }
        const bool act = __ballot(use != 0u) != 0ull;
#pragma unroll 1
        for (int q = q0; q < npc; q += P) {
            const Real f = s_iist[q], afac = s_afac[q], kd = s_kd[q];
            const Real* lq = s_ldm + q;
            float* o = out + (size_t)(qa + q) * npt;
            if (tid < nslots) {
                f32x4_t w = {1.0f, 1.0f, 1.0f, 1.0f};
                if (act) {
#pragma unroll
                    for (int j = 0; j < TPL; ++j) {
                        const Real* l = lq + off[j];
                        const Real ip = rb[j] * l[0] + ra[j] * l[kTsAlLd];
                        // the row form's c1 afac + (c2 + c3 (k - k_mean)), with c1 = A0
                        // inside and c2 = A0, c3 = 2 k_mean kappa_0 otherwise
                        const Real area = as[j] < Real(0) ? (-as[j]) * afac : dk[j] * kd + as[j];
                        w[j] = ((use >> j) & 1u) ? Real(1) - (ip * area) * f : Real(1);
                    }
                }
                __builtin_nontemporal_store(w, (f32x4_t*)(o + (size_t)vi * TPL));
            }
        }
    }
}

// ---- any number of samples up to kTsTabSamples: geometry in LDS --------------------------
//
// A workgroup of 4 waves takes a tile of T = 64, 128 or 256 times of one pv and a range
// of passbands.  The geometry of every (time, sample) of the tile goes to LDS once, and
// the passbands' LD rows pass through LDS in chunks; a wave takes every fourth group of
// four passbands of a chunk and all T times of the tile, 64 at a time, one a lane (so its
// stores are contiguous).  The form that recomputed the geometry for each chunk of 16
// passbands spent most of its time on FP64 arctangents: 100 pv x 203 passbands x 1,237 t, 3
// samples, FP64: 172 -> 60 us (201 MB written: 29 us at the rate of a fill, 45 as rows of odd length).
constexpr int kTsTabSamples = 32;
// passbands of a chunk (FP64: 32 takes 105, 16 takes 100 us at the size above)
template <typename Real> constexpr int ts_tab_pc() { return sizeof(Real) == 4 ? 32 : 16; }
constexpr int kTsTabQ = 4;        // passbands a lane takes together
// LDS stride of one g, a 16-byte multiple off a multiple of all banks
template <typename Real> constexpr int ts_tab_ld() { return ts_tab_pc<Real>() + 16 / (int)sizeof(Real); }

template <typename Real> struct TsTab { static constexpr int kBytes = 3 * (int)sizeof(Real) + 4; };

// Times of a tile: as many as keep the geometry within 40 KB.
template <typename Real>
__host__ __device__ inline int ts_tab_times(int ns) {
    int t = 256;
    while (t > 64 && t * ns * TsTab<Real>::kBytes > 40 * 1024) t /= 2;
    return t;
}
template <typename Real>
__host__ inline size_t ts_tab_lds(int ns, int ng) {
    const size_t geo = (size_t)ts_tab_times<Real>(ns) * ns * TsTab<Real>::kBytes;
    return (geo + 15) / 16 * 16 + ((size_t)ts_tab_ld<Real>() * ng + 3 * ts_tab_pc<Real>()) * sizeof(Real);
}

template <typename Real>
__global__ void __launch_bounds__(kTsThreads) ts_flux_table_kernel(TsArgs s, Real* flux, int ntiles, int nsplit, int ns) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ unsigned s_act;
    const int T = ts_tab_times<Real>(ns), n = T * ns;
    Real* t_ra = (Real*)lds;                    // [ns][T]
    Real* t_a0 = t_ra + n;
    Real* t_dk = t_a0 + n;
    int* t_pk = (int*)(t_dk + n);               // interval << 3 | in the window << 2 | inside << 1 | g <= 1
    constexpr int kLd = ts_tab_ld<Real>(), kPc = ts_tab_pc<Real>();
    // [ng][kLd], by its offset: through a rounded address its reads become flat loads
    Real* s_l = (Real*)(lds + (n * TsTab<Real>::kBytes + 15) / 16 * 16);
    Real* s_afac = s_l + (size_t)kLd * s.ng;
    Real* s_kd = s_afac + kPc;
    Real* s_f = s_kd + kPc;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int split = bid % nsplit, tile = (bid / nsplit) % ntiles, pv = bid / nsplit / ntiles;
    const int per = (s.npb + nsplit - 1) / nsplit;
    const int q0 = split * per, q1 = min(q0 + per, s.npb);
    const TsRec& r = s.rec[pv];
    const int nt = min(T, s.npt - tile * T);    // the tile's times
    Real* out = flux + (size_t)pv * s.npb * s.npt + (size_t)tile * T;
    auto fill = [&](Real v) {
        for (int q = q0 + wave; q < q1; q += 4)
            for (int t = lane; t < nt; t += 64) out[(size_t)q * s.npt + t] = v;
    };
    if (!r.good) {
        fill(Real(NAN));
        return;
    }
    if (tid == 0) s_act = 0u;
    __syncthreads();
    // geometry: item i is sample i / T of the tile's time i % T (T is a power of two)
    const double ext = s.exptimes[0], t0v = s.t0[pv], p = r.p, inv_p = r.inv_p, inv_ns = 1.0 / ns;
    const double inv_1pk = 1.0 / (1.0 + r.kmean), inv_dg = 1.0 / s.dg;
    for (int i = tid; i < n; i += kTsThreads) {
        const int t = i & (T - 1), is = i / T, jt = tile * T + t;
        int pk = 0;
        Real ra = Real(0), a0 = Real(0), dk = Real(0);
        if (jt < s.npt) {
            double ep;
            const double tc = epoch_phase(s.times[jt], t0v, p, inv_p, ep);
            if (r.bt1 <= tc && tc <= r.bt4) {
                const TsGeo<Real> g = ts_geometry<Real>(r, tc, ext, inv_ns, is, inv_1pk, inv_dg, s.ng);
                pk = (g.ig << 3) | 4 | (g.inside ? 2 : 0) | (g.gz ? 0 : 1);
                ra = g.ra;
                a0 = g.ap0;
                dk = g.dadk;
                if (is == 0) atomicOr(&s_act, 1u << (t >> 6));
            }
        }
        t_pk[i] = pk;
        t_ra[i] = ra;
        t_a0[i] = a0;
        t_dk[i] = dk;
    }
    __syncthreads();
    const unsigned act = s_act;                 // bit j: times 64 j .. 64 j + 63 hold a point in the window
    if (!act) {
        fill(Real(1));
        return;
    }
    const double km = r.kmean;
    // a wave stages every fourth row of a chunk, loaded (the first 128 g of each) one
    // chunk ahead
    constexpr int kRows = kPc / 4;
    const Real* ldm = sizeof(Real) == 4 ? (const Real*)s.ldm32 : (const Real*)s.ldm64;
    Real st[kRows][2];
    auto stage_load = [&](int pb0) {
#pragma unroll
        for (int m = 0; m < kRows; ++m) {
            const int q = pb0 + wave + 4 * m;
            const Real* src = ldm + ((size_t)pv * s.npb + q) * s.ng;
            st[m][0] = q < q1 && lane < s.ng ? src[lane] : Real(0);
            st[m][1] = q < q1 && lane + 64 < s.ng ? src[lane + 64] : Real(0);
        }
    };
    stage_load(q0);
    for (int pb0 = q0; pb0 < q1; pb0 += kPc) {
        const int npc = min(kPc, q1 - pb0);
        __syncthreads();  // the previous chunk's rows are no longer read
#pragma unroll
        for (int m = 0; m < kRows; ++m) {
            const int q = wave + 4 * m;
            if (lane < s.ng) s_l[lane * kLd + q] = st[m][0];
            if (lane + 64 < s.ng) s_l[(lane + 64) * kLd + q] = st[m][1];
            for (int g = lane + 128; g < s.ng; g += 64)
                s_l[g * kLd + q] = q < npc ? ldm[((size_t)pv * s.npb + pb0 + q) * s.ng + g] : Real(0);
        }
        if (pb0 + kPc < q1) stage_load(pb0 + kPc);
        if (tid < kPc) {
            const size_t j = (size_t)pv * s.npb + pb0 + min(tid, npc - 1);
            const double kq = s.k[j];
            s_afac[tid] = (Real)(kq * kq / (km * km));
            s_kd[tid] = (Real)(kq - km);
            s_f[tid] = (Real)(inv_ns / s.istar[j]);
        }
        __syncthreads();
        for (int q = wave * kTsTabQ; q < npc; q += 4 * kTsTabQ) {
            Real afac[kTsTabQ], kd[kTsTabQ], f[kTsTabQ];
#pragma unroll
            for (int j = 0; j < kTsTabQ; ++j) {
                afac[j] = s_afac[q + j];
                kd[j] = s_kd[q + j];
                f[j] = s_f[q + j];
            }
            Real* o = out + (size_t)(pb0 + q) * s.npt;
            for (int t0 = 0; t0 < nt; t0 += 64) {
                const int t = t0 + lane;
                Real v[kTsTabQ];
#pragma unroll
                for (int j = 0; j < kTsTabQ; ++j) v[j] = Real(1);
                if ((act >> (t0 >> 6)) & 1u) {
                    Real acc[kTsTabQ];
#pragma unroll
                    for (int j = 0; j < kTsTabQ; ++j) acc[j] = Real(0);
                    for (int is = 0; is < ns; ++is) {
                        const int i = is * T + t, pk = t_pk[i];
                        const Real ra = t_ra[i], rb = Real(1) - ra, a0 = t_a0[i], dk = t_dk[i];
                        const Real* l = s_l + (pk >> 3) * kLd + q;
#pragma unroll
                        for (int j = 0; j < kTsTabQ; ++j) {
                            const Real ip = rb * l[j] + ra * l[kLd + j];
                            const Real area = (pk & 2) ? a0 * afac[j] : a0 + kd[j] * dk;
                            acc[j] += (pk & 1) ? ip * area : Real(0);
                        }
                    }
                    const bool inw = (t_pk[t] & 4) != 0;
#pragma unroll
                    for (int j = 0; j < kTsTabQ; ++j) v[j] = inw ? Real(1) - acc[j] * f[j] : Real(1);
                }
#pragma unroll
                for (int j = 0; j < kTsTabQ; ++j)
                    if (t < nt && q + j < npc) o[(size_t)j * s.npt + t] = v[j];
            }
        }
    }
}

// ---- any number of samples, any g grid: the geometry recomputed for each chunk of
// passbands, one accumulator a passband and lane ------------------------------------------
template <bool kMixed>
__global__ void __launch_bounds__(kTsThreads) ts_flux_kernel(TsArgs s, void* flux, int ntiles) {
    using Real = typename std::conditional<kMixed, float, double>::type;
    constexpr int PC = ts_pb_chunk(kMixed);
    extern __shared__ __align__(16) unsigned char lds[];
    Real* s_ldm = (Real*)lds;                       // [PC][ng]
    Real* s_afac = s_ldm + (size_t)PC * s.ng;       // k^2 / k_mean^2
    Real* s_kd = s_afac + PC;                       // k - k_mean
    Real* s_f = s_kd + PC;                          // 1 / (ns istar)
    __shared__ int s_any;

    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int tile = bid % ntiles;
    const int pv = bid / ntiles;
    const int it = tile * kTsThreads + (int)threadIdx.x;
    const bool in = it < s.npt;
    const TsRec& r = s.rec[pv];
    Real* out = (Real*)flux + (size_t)pv * s.npb * s.npt + it;
    if (!r.good) {
        if (in)
            for (int q = 0; q < s.npb; ++q) out[(size_t)q * s.npt] = Real(NAN);
        return;
    }
    double tc = 0.0;
    bool inw = false;
    if (in) {
        double ep;
        tc = epoch_phase(s.times[it], s.t0[pv], r.p, r.inv_p, ep);
        inw = (r.bt1 <= tc) && (tc <= r.bt4);
    }
    if (threadIdx.x == 0) s_any = 0;
    __syncthreads();
    if (inw) s_any = 1;
    __syncthreads();
    if (!s_any) {
        if (in)
            for (int q = 0; q < s.npb; ++q) out[(size_t)q * s.npt] = Real(1);
        return;
    }
    const int ns = s.nsamples[0];
    const double ext = s.exptimes[0];
    const double km = r.kmean, inv_1pk = 1.0 / (1.0 + km), inv_dg = 1.0 / s.dg, inv_ns = 1.0 / ns;
    for (int pb0 = 0; pb0 < s.npb; pb0 += PC) {
        const int npc = min(PC, s.npb - pb0);
        __syncthreads();  // the previous chunk's rows are no longer read
        // stage the chunk's limb-darkening means and per-passband factors
        for (int i = threadIdx.x; i < npc * s.ng; i += kTsThreads) {
            const size_t src = ((size_t)pv * s.npb + pb0) * s.ng + i;
            s_ldm[i] = kMixed ? (Real)s.ldm32[src] : (Real)s.ldm64[src];
        }
        for (int q = threadIdx.x; q < npc; q += kTsThreads) {
            const double kq = s.k[(size_t)pv * s.npb + pb0 + q];
            s_afac[q] = (Real)(kq * kq / (km * km));
            s_kd[q] = (Real)(kq - km);
            s_f[q] = (Real)(inv_ns / s.istar[(size_t)pv * s.npb + pb0 + q]);
        }
        __syncthreads();
        if (!in) continue;
        Real acc[PC];
#pragma unroll
        for (int q = 0; q < PC; ++q) acc[q] = Real(0);
        if (inw) {
            for (int is = 0; is < ns; ++is) {
                const TsGeo<Real> g = ts_geometry<Real>(r, tc, ext, inv_ns, is, inv_1pk, inv_dg, s.ng);
#pragma unroll
                for (int q = 0; q < PC; ++q)
                    if (q < npc) {
                        const Real* l = s_ldm + (size_t)q * s.ng;
                        const Real ip = g.rb * l[g.ig] + g.ra * l[g.ig + 1];
                        const Real area = g.inside ? g.ap0 * s_afac[q] : g.ap0 + s_kd[q] * g.dadk;
                        acc[q] += g.gz ? Real(0) : ip * area;
                    }
            }
        }
#pragma unroll
        for (int q = 0; q < PC; ++q)
            if (q < npc) out[(size_t)(pb0 + q) * s.npt] = inw ? Real(1) - acc[q] * s_f[q] : Real(1);
    }
}

}  // namespace rr

using namespace rr;

extern "C" {

static size_t ts_sizes(int npv, int npb, int ng, int nz, int precision, size_t* off) {
    const int ngp = (ng + 15) / 16 * 16, nzp = (nz + 3) / 4 * 4;
    size_t b = 0;
    off[0] = b; b += align_up((size_t)npv * sizeof(TsRec), 256);
    off[1] = b; b += align_up((size_t)npv * npb * sizeof(double), 256);
    const size_t w2e = (size_t)npv * nzp * ngp;
    off[2] = b; b += align_up(w2e * (precision == RR_MIXED ? sizeof(float) : sizeof(double)), 256);
    off[3] = b; b += align_up((size_t)npv * npb * ng * (precision == RR_MIXED ? sizeof(float) : sizeof(double)), 256);
    return b;
}

size_t ts_workspace_bytes(int npv, int npb, int ng, int nz, int precision) {
    if (npv < 0 || npb < 0 || ng < 0 || nz < 0) return 0;
    size_t off[4];
    return ts_sizes(npv, npb, ng, nz, precision, off);
}

int ts_evaluate(int precision, const rr_table* tab, const rr_lcdata* lc, const rr_params* pv, const rr_ld* ld,
                void* workspace, size_t workspace_bytes, void* flux, void* stream) {
    if (!tab || !lc || !pv || !ld) return set_error(RR_EINVAL, "ts_evaluate: null descriptor");
    if (precision != RR_FP64 && precision != RR_MIXED) return set_error(RR_EINVAL, "ts_evaluate: bad precision");
    const int npv = pv->npv, npt = lc->npt, npb = lc->npb;
    if (npv < 0 || npt < 0 || npb < 1) return set_error(RR_EINVAL, "ts_evaluate: bad sizes");
    if (pv->kcols != npb)
        return set_error(RR_EINVAL, "The transmission spectrum transit model requires that the number or radius "
                                    "ratios and the number of passbands match.");
    if (tab->ng < 2 || tab->nz < 1 || tab->nz > 1024 || tab->ng > 2048 || !tab->ze || !tab->mu)
        return set_error(RR_EINVAL, "ts_evaluate: bad z grid / ng");
    if (npv == 0 || npt == 0) return RR_OK;
    if (!lc->times || !lc->nsamples || !lc->exptimes) return set_error(RR_EINVAL, "ts_evaluate: null time arrays");
    if (!pv->k || !pv->t0 || !pv->p || !pv->a || !pv->inc || !pv->e || !pv->w || !flux)
        return set_error(RR_EINVAL, "ts_evaluate: null parameter array");
    if (ld->law == RR_LD_TABULATED) {
        if (!ld->ldp || !ld->istar) return set_error(RR_EINVAL, "ts_evaluate: tabulated LD needs ldp and istar");
    } else if (ld->law < RR_LD_UNIFORM || ld->law > RR_LD_POWER_2_PM || (ld->nldc > 0 && !ld->ldc)) {
        return set_error(RR_EINVAL, "ts_evaluate: bad limb-darkening descriptor");
    }
    size_t off[4];
    const size_t need = ts_sizes(npv, npb, tab->ng, tab->nz, precision, off);
    if (!workspace || workspace_bytes < need)
        return set_error(RR_EINVAL, "ts_evaluate: workspace of %zu bytes needed, got %zu", need, workspace_bytes);
    if ((long long)npv * npb * npt > (1LL << 40)) return set_error(RR_ERANGE, "ts_evaluate: problem too large");

    char* ws = (char*)workspace;
    const bool mixed = precision == RR_MIXED;
    TsArgs a;
    a.times = lc->times; a.k = pv->k; a.t0 = pv->t0;
    a.exptimes = lc->exptimes; a.nsamples = lc->nsamples;
    a.p = pv->p; a.a = pv->a; a.inc = pv->inc; a.e = pv->e; a.w = pv->w;
    a.law = ld->law; a.nldc = ld->nldc; a.ldc = ld->ldc; a.ldp_in = ld->ldp; a.istar_in = ld->istar;
    a.W = tab->weights; a.ze = tab->ze; a.mu = tab->mu;
    a.rec = (TsRec*)(ws + off[0]);
    a.istar = (double*)(ws + off[1]);
    a.w2_64 = mixed ? nullptr : (double*)(ws + off[2]);
    a.w2_32 = mixed ? (float*)(ws + off[2]) : nullptr;
    a.ldm64 = mixed ? nullptr : (double*)(ws + off[3]);
    a.ldm32 = mixed ? (float*)(ws + off[3]) : nullptr;
    a.npv = npv; a.npb = npb; a.npt = npt; a.nk = tab->nk; a.ng = tab->ng; a.nz = tab->nz;
    a.ngp = (tab->ng + 15) / 16 * 16; a.nzp = (tab->nz + 3) / 4 * 4;
    a.use_table = tab->weights != nullptr && tab->nk >= 2;
    a.kmin = tab->kmin; a.kmax_tab = tab->kmax; a.dk = tab->dk; a.dg = tab->dg;
    a.ldm_split = a.row_split = 1;
    hipStream_t st = (hipStream_t)stream;
    const bool tab_ld = ld->law == RR_LD_TABULATED;
    // the weight kernel lists (g, z) pairs of a workgroup as 16-bit indices
    if ((size_t)ts_weight_rows(a.nz) * a.nz > 65535u) return set_error(RR_ERANGE, "ts_evaluate: nz must be <= 65535");

    hipLaunchKernelGGL(ts_setup_kernel, dim3((npv + kTsGroup - 1) / kTsGroup), dim3(64), 0, st, a);
    int rc = check_launch("ts_setup_kernel");
    if (rc) return rc;
    const int wrows = ts_weight_rows(a.nz);
    const long long nw = (long long)npv * ((a.ngp + wrows - 1) / wrows) + ((long long)npv * npb + 255) / 256;
    if (nw > 0x7fffffffLL) return set_error(RR_ERANGE, "ts_evaluate: grid too large");
    hipLaunchKernelGGL(ts_weights_kernel, dim3((unsigned)nw), dim3(256), ts_weights_lds(a.nz), st, a);
    if ((rc = check_launch("ts_weights_kernel"))) return rc;
    // tabulated FP64 profiles with nz a multiple of 4 (16-byte aligned rows), nz <= 128
    // and ngp <= 128: the row-contiguous kernel
    const int nct = a.ngp / 16;
    // few pvs: the row tiles of a pv over several workgroups (of 8 waves, the generic
    // FP32 form 4), one round of row tiles a wave at the least
    const int nrt = (npb + 15) / 16;
    auto ldm_split = [&](int waves) {
        const int most = (nrt + waves - 1) / waves, want = (512 + npv - 1) / npv;
        return want < 1 ? 1 : (want < most ? want : most);
    };
    const bool tab_rows = mixed && tab_ld && a.nz % 4 == 0 && a.nz <= 16 * kTabMfmaMaxJ && nct <= kTabMfmaMaxCt &&
                          ((uintptr_t)ld->ldp & 15) == 0;
    const int nbasis = !mixed || tab_ld ? 0 : ld_basis_count(ld->law, ld->nldc);
    if (nbasis > 0) {
        // workgroups for every CU four times, of at least 8 passbands each and at most 128
        const int want = (1024 + npv - 1) / npv, most = (npb + 7) / 8, least = (npb + 127) / 128;
        a.ldm_split = want < least ? least : (want < most ? want : most);
        const size_t lds = ts_basis_lds(nbasis, a.nz, a.ng, (npb + a.ldm_split - 1) / a.ldm_split);
        if ((long long)npv * a.ldm_split > 0x7fffffffLL) return set_error(RR_ERANGE, "ts_evaluate: grid too large");
        const dim3 g((unsigned)npv * a.ldm_split);
        hipLaunchKernelGGL(ts_ldm_basis_kernel, g, dim3(256), lds, st, a, nbasis);
        if ((rc = check_launch("ts_ldm_basis_kernel"))) return rc;
    } else if (tab_rows) {
        const size_t lds = (size_t)((a.nz + 15) / 16 * 16) * ts_tab_ldb(a.ngp) * sizeof(float);
        a.ldm_split = ldm_split(kTabMfmaThreads / 64);
        const dim3 g((unsigned)npv * a.ldm_split), b(kTabMfmaThreads);
        switch (nct) {
            case 1: hipLaunchKernelGGL(ts_ldm_tab_mfma_kernel<1>, g, b, lds, st, a); break;
            case 2: hipLaunchKernelGGL(ts_ldm_tab_mfma_kernel<2>, g, b, lds, st, a); break;
            case 3: hipLaunchKernelGGL(ts_ldm_tab_mfma_kernel<3>, g, b, lds, st, a); break;
            case 4: hipLaunchKernelGGL(ts_ldm_tab_mfma_kernel<4>, g, b, lds, st, a); break;
            case 5: hipLaunchKernelGGL(ts_ldm_tab_mfma_kernel<5>, g, b, lds, st, a); break;
            case 6: hipLaunchKernelGGL(ts_ldm_tab_mfma_kernel<6>, g, b, lds, st, a); break;
            case 7: hipLaunchKernelGGL(ts_ldm_tab_mfma_kernel<7>, g, b, lds, st, a); break;
            default: hipLaunchKernelGGL(ts_ldm_tab_mfma_kernel<8>, g, b, lds, st, a); break;
        }
        if ((rc = check_launch("ts_ldm_tab_mfma_kernel"))) return rc;
    } else if (mixed) {
        const size_t lds = (size_t)a.nzp * ts_tab_ldb(a.ngp) * sizeof(float);
        if (lds <= 160 * 1024) {
            a.ldm_split = ldm_split(4);
            const dim3 g((unsigned)npv * a.ldm_split);
            if (tab_ld) hipLaunchKernelGGL(ts_ldm_mfma_kernel<true>, g, dim3(256), lds, st, a);
            else hipLaunchKernelGGL(ts_ldm_mfma_kernel<false>, g, dim3(256), lds, st, a);
            if ((rc = check_launch("ts_ldm_mfma_kernel"))) return rc;
        } else {
            const long long n = (long long)npv * npb * a.ng;
            const dim3 g((unsigned)((n + 255) / 256));
            if (tab_ld) hipLaunchKernelGGL(ts_ldm_f32_kernel<true>, g, dim3(256), 0, st, a);
            else hipLaunchKernelGGL(ts_ldm_f32_kernel<false>, g, dim3(256), 0, st, a);
            if ((rc = check_launch("ts_ldm_f32_kernel"))) return rc;
        }
    } else {
        const size_t lds = (size_t)a.nzp * (a.ngp + 1) * sizeof(double);
        if (lds <= kMfma64MaxLds) {
            a.ldm_split = ldm_split(kMfma64Threads / 64);
            const dim3 g((unsigned)npv * a.ldm_split);
            if (tab_ld) hipLaunchKernelGGL(ts_ldm_mfma64_kernel<true>, g, dim3(kMfma64Threads), lds, st, a);
            else hipLaunchKernelGGL(ts_ldm_mfma64_kernel<false>, g, dim3(kMfma64Threads), lds, st, a);
            if ((rc = check_launch("ts_ldm_mfma64_kernel"))) return rc;
        } else {
            const long long n = (long long)npv * npb * a.ng;
            const dim3 g((unsigned)((n + 255) / 256));
            if (tab_ld) hipLaunchKernelGGL(ts_ldm_f64_kernel<true>, g, dim3(256), 0, st, a);
            else hipLaunchKernelGGL(ts_ldm_f64_kernel<false>, g, dim3(256), 0, st, a);
            if ((rc = check_launch("ts_ldm_f64_kernel"))) return rc;
        }
    }
    const dim3 block(kTsThreads);
    // nsamples[0] as given by the host (0: unknown)
    const int uns = lc->uniform_nsamples;
    // FP32 rows in whole cache lines (of at least one: the rotated slots wrap once), where
    // that gives every CU a workgroup (aligned against the forms below, us: 8 x 200 x 1,236
    // 47.7 / 45.5, 64 x 200 x 1,236 59.5 / 61.8, 32 x 512 x 5,000 111 / 139)
    if (mixed && uns == 1 && ((uintptr_t)flux % 16) == 0 && npt % 4 == 0 && npt >= kTsLine && npt <= ts_row_max_npt<float>() &&
        kTsAlPc * a.ng <= kTsStageRegs * kTsAlThreads && ts_rows_aligned_lds(a.ng, npt) <= kTsRowsAlignedMaxLds) {
        a.row_split = (npb + kTsAlPc - 1) / kTsAlPc;
        const long long nwg = (long long)npv * a.row_split * ts_segments(npt / 4);
        if (nwg >= 256 && nwg <= 0x7fffffffLL) {
            hipLaunchKernelGGL(ts_flux_rows_aligned_kernel, dim3((unsigned)nwg), dim3(kTsAlThreads),
                               ts_rows_aligned_lds(a.ng, npt), st, a, (float*)flux);
            return check_launch("ts_flux_rows_aligned_kernel");
        }
    }
    // one sample, rows of whole 16-byte vectors: 32 rows a workgroup, which computes its
    // geometry in registers (FP64 against one workgroup or few per pv: 1,024 x 256 x 5,000
    // 2187 -> 2135 us, 300 x 200 x 2,000 283 -> 245, 260 x 512 x 3,000 757 -> 717), where that
    // is a workgroup for every CU and 24 million values (rows against the tiles below, FP64,
    // us: 64 x 200 x 1,236 67.9 / 63.0, 128 x 200 x 1,236 101 / 109, 20 x 512 x 5,000 127 / 146,
    // 8 x 512 x 5,000 71.7 / 64.3)
    a.row_split = (npb + kTsRowPc - 1) / kTsRowPc;
    const long long nrow = (long long)npv * a.row_split;
    if (uns == 1 && ((uintptr_t)flux % 16) == 0 && nrow >= 256 && nrow <= 0x7fffffffLL &&
        (long long)npv * npb * npt >= 24000000LL) {
        if (mixed && npt % 4 == 0 && npt <= ts_row_max_npt<float>() && a.ng <= ts_row_max_ng<float>()) {
            hipLaunchKernelGGL(ts_flux_rows_kernel<float>, dim3((unsigned)nrow), dim3(kTsRowThreads),
                               ts_rows_lds(a.ng, 4), st, a, (float*)flux);
            return check_launch("ts_flux_rows_kernel");
        }
        if (!mixed && npt % 2 == 0 && npt <= ts_row_max_npt<double>() && a.ng <= ts_row_max_ng<double>()) {
            hipLaunchKernelGGL(ts_flux_rows_kernel<double>, dim3((unsigned)nrow), dim3(kTsRowThreads),
                               ts_rows_lds(a.ng, 8), st, a, (double*)flux);
            return check_launch("ts_flux_rows_kernel");
        }
    }
    // Few passbands of many times leave the table kernel's waves without a group of four:
    // they go to the kernel below, a lane a time with all passbands in its registers (us,
    // table / a lane a time: 60 pv x 20,000 t, 10 samples, in 2, 8 and 16 passbands FP64
    // 92 / 56, 96 / 67, 100 / 86, mixed 100 / 58, 106 / 66, 106 / 81; 1000 x 3000 mixed, 3
    // samples, 16 passbands 195 / 241; 300 x 1237 mixed, 30 samples, 8 passbands 164 / 227).
    const long long nlane = (long long)npv * ((npt + kTsThreads - 1) / kTsThreads);
    const bool big = nlane >= 3072;
    const bool few = nlane >= 1024 &&
                     npb <= (mixed ? (uns > 16 && !big ? 0 : 8) : (uns >= 8 && big ? 16 : 12));
    if (uns >= 1 && uns <= kTsTabSamples && !few) {
        const size_t lds = mixed ? ts_tab_lds<float>(uns, a.ng) : ts_tab_lds<double>(uns, a.ng);
        const int T = mixed ? ts_tab_times<float>(uns) : ts_tab_times<double>(uns);
        if (lds <= 160 * 1024) {
            // passbands split over workgroups where the tiles alone leave CUs without one
            const int nt = (npt + T - 1) / T;
            const long long tiles = (long long)npv * nt;
            const int pc = mixed ? ts_tab_pc<float>() : ts_tab_pc<double>(), most = (npb + pc - 1) / pc;
            const int nsplit = (int)(tiles >= 1024 ? 1 : (1024 + tiles - 1) / tiles < most ? (1024 + tiles - 1) / tiles : most);
            if (tiles * nsplit > 0x7fffffffLL) return set_error(RR_ERANGE, "ts_evaluate: grid too large");
            const dim3 g((unsigned)(tiles * nsplit));
            if (mixed) hipLaunchKernelGGL(ts_flux_table_kernel<float>, g, block, lds, st, a, (float*)flux, nt, nsplit, uns);
            else hipLaunchKernelGGL(ts_flux_table_kernel<double>, g, block, lds, st, a, (double*)flux, nt, nsplit, uns);
            return check_launch("ts_flux_table_kernel");
        }
    }
    const int ntiles = (npt + kTsThreads - 1) / kTsThreads;
    const long long nb = (long long)npv * ntiles;
    if (nb > 0x7fffffffLL) return set_error(RR_ERANGE, "ts_evaluate: grid too large");
    const int PC = ts_pb_chunk(mixed);
    const size_t lds = ((size_t)PC * a.ng + 3 * PC) * (mixed ? sizeof(float) : sizeof(double));
    const dim3 grid((unsigned)nb);
    if (mixed) hipLaunchKernelGGL(ts_flux_kernel<true>, grid, block, lds, st, a, flux, ntiles);
    else hipLaunchKernelGGL(ts_flux_kernel<false>, grid, block, lds, st, a, flux, ntiles);
    return check_launch("ts_flux_kernel");
}

}  // extern "C"
