// srf_sss.hip -- single-scatter simulation (SSS) on a coarse virtual-detector
// sinogram, and its C-ABI entry points (include/srf_hip.h, srf_sss_*).
//
// Physics of srfnef/corrections/scattering/scatter_fraction/scatter_fraction.py:
// 70-131 and kn_formula.py:6-46 (per LOR (A,B), a Klein-Nishina weighted sum
// over scatter points S of the emission and attenuation line integrals from S
// to both detectors).  The line integrals come from srf_sss_integrals (srf_project.hip)
// or the projector over the (detector, scatter point) LOR set; this file holds
//   k_sss_pairs   per (detector, scatter point): unit vector S->D, the
//                 obliquity / distance factor g = ((D-S).n_D)/|D-S|^3, and the
//                 emission and attenuation integrals, in the order the bin sum
//                 reads them (RowLayout);
//   k_sss_bins    per sinogram bin: the sum over scatter points, one bin per
//                 lane, the points split over workgroups;
//   k_sss_bins_any  the same with 16 or 64 lanes per bin (bins of unrelated
//                 detectors, or few of them).
// Energy-dependent factors depend only on the integer scattering angle
// (the reference quantises it to whole degrees, kn_formula.py:41), so E', the
// window efficiency and the KN factor are 181-entry tables.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "srf_hip.h"
#include "srf_internal.hpp"

namespace srf {

// The rows of the (detector, point) table: 24 bytes each, as 16 (unit vector, g) and
// 8 (emission integral, attenuation integral times log2 e), point groups of GS
// outermost, then the detector, then the point within its group.
//   GS = 4 (1 below 16 points), sinogram order: a lane's 4 points of one detector are
// 64 + 32 consecutive bytes, and neighbouring lanes' detectors are neighbours.  131072
// bins of a ring scanner, 2e4 points, 4096 detectors: 4.5 ms, VALU bound (about 61 issue
// cycles a pair); one point per group 6.0 ms (rows 64 KiB apart) and 1.8 instead of 0.7 ms
// to write them, 16 per group 7.8 ms.  Detector-major rows with acosf per pair and one bin
// per lane over all points, as before: 11.9 ms.
//   GS = 16, any order: 16 lanes read whole cache lines of one detector, which is what bins
// of unrelated detectors and sinograms with few bins need: 4000 pairs of 2048 detectors,
// 2000 points 52 us (4 per group: 127 one bin per wavefront, 166 one bin per lane;
// detector-major rows of 32 bytes: 58).
template <int GS>
struct RowLayout {
    int64_t nd;
    int ns;
    // GS = 4 is padded to whole groups, the others are not (their last group is narrower)
    static constexpr bool PAD = GS == 4;
    __host__ __device__ int64_t padded() const { return nd * (PAD ? (ns + GS - 1) / GS * GS : ns); }
    __device__ __forceinline__ int64_t at(int64_t d, int s) const
    {
        const int g = s / GS, w = PAD ? GS : min(GS, ns - g * GS);
        return (int64_t)g * GS * nd + d * w + s % GS;
    }
};

// Points per group in sinogram order: 4, or 1 where rounding ns up to 4 would outgrow the
// workspace (32 bytes per pair); in any order.
constexpr int SSS_GROUP = 4, SSS_GROUP_ANY = 16;
static bool grouped_rows(int n_points) { return n_points >= 16; }

// det: (nd, 4) x, y, z, normal angle; sp: (ns, 4) x, y, z, mu(S);
// em, mu: (nd, ns) line integrals (row-major by detector).  A workgroup takes 64
// points of 4 detectors; points past ns fill their group with zero rows.
template <int GS>
__global__ __launch_bounds__(256) void k_sss_pairs(const float *__restrict__ det, const float *__restrict__ sp,
                                                   const float *__restrict__ em, const float *__restrict__ mu,
                                                   int nd, int ns, float4 *__restrict__ dir, float2 *__restrict__ val)
{
    const int nsb = (ns + 63) / 64;
    const int s = blockIdx.x % nsb * 64 + (threadIdx.x & 63), d = blockIdx.x / nsb * 4 + (threadIdx.x >> 6);
    const RowLayout<GS> R{nd, ns};
    if (d >= nd || s >= (R.PAD ? (ns + GS - 1) / GS * GS : ns)) return;
    float4 u = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float2 v = make_float2(0.0f, 0.0f);
    if (s < ns) {
        const float vx = det[4 * d] - sp[4 * s], vy = det[4 * d + 1] - sp[4 * s + 1], vz = det[4 * d + 2] - sp[4 * s + 2];
        const float r2 = vx * vx + vy * vy + vz * vz;
        const float inv = 1.0f / sqrtf(r2);
        const float a = det[4 * d + 3];
        const int64_t i = (int64_t)d * ns + s;
        // the unit vector's length corrected to 1 (the rounding of r2 and inv scales all
        // three components, and with them the cosine whose whole degree is taken)
        const double l2 = fma((double)(vx * inv), (double)(vx * inv),
                              fma((double)(vy * inv), (double)(vy * inv), (double)(vz * inv) * (double)(vz * inv)));
        const float h = (float)(0.5 * (1.0 - l2));
        u = make_float4(fmaf(vx * inv, h, vx * inv), fmaf(vy * inv, h, vy * inv), fmaf(vz * inv, h, vz * inv),
                        (vx * cosf(a) + vy * sinf(a)) * inv / r2);
        v = make_float2(em[i], mu[i] * 1.44269504f);
    }
    dir[R.at(d, s)] = u;
    val[R.at(d, s)] = v;
}

// The whole-degree scattering angle k = (int)(acos(x) 180 / pi) of a pair
// (kn_formula.py:41) from two small tables instead of acosf: t = sqrt(1 - |x|) is
// nearly linear in the angle (0.0087 to 0.0123 per degree), so a cell of 1/256 in t
// holds at most one whole degree.  A cell stores the value of x below which the angle
// has passed that degree (cos in double, so a float x is put on the right side of
// it; acosf and the product by 180 / pi misplace x within about 2e-7), and the
// smaller angle.
constexpr int DEG_CELLS = 257;

constexpr int BINS_WG = 1024;

struct DegTable {
    float2 cell[2 * DEG_CELLS];   // x >= 0, then x < 0: threshold in x, angle index (as bits)
    float2 fac[181 + 1];          // 511 / E', window efficiency times KN / sigma_KN
};

__device__ __forceinline__ int degrees_of(float x) { return min((int)(acos((double)x) * 57.29577951308232), 180); }

// thr[k]: the angle is at least k where x < thr[k], the float above cos k; the degrees'
// factors.  tables: [0,181) 511/E', [181,362) window efficiency, [362,543) KN / sigma_KN
__device__ __forceinline__ void build_thresholds(float *thr, float2 *fac, const float *__restrict__ tables, int threads)
{
    for (int k = threadIdx.x; k <= 180; k += threads) {
        const double c = cos((double)k * 0.017453292519943295);
        const float f = (float)c;
        thr[k] = (double)f <= c ? nextafterf(f, 2.0f) : f;
        fac[k] = make_float2(tables[k], tables[181 + k] * tables[362 + k]);
    }
    __syncthreads();
}

__device__ __forceinline__ void build_degrees(DegTable &T, float *thr, const float *__restrict__ tables)
{
    build_thresholds(thr, T.fac, tables, BINS_WG);
    for (int i = threadIdx.x; i < 2 * DEG_CELLS; i += BINS_WG) {
        const bool neg = i >= DEG_CELLS;
        const float t0 = (float)(i - (neg ? DEG_CELLS : 0)) / 256.0f, t1 = t0 + 1.0f / 256.0f;
        const float m0 = 1.0f - t0 * t0, m1 = fmaxf(0.0f, 1.0f - t1 * t1);
        // the smaller angle of the cell, and the degree it passes (if any)
        const int k0 = degrees_of(neg ? -m1 : m0), k1 = degrees_of(neg ? -m0 : m1);
        T.cell[i] = make_float2(k1 > k0 ? thr[k0 + 1] : -2.0f, __int_as_float(k0));
    }
    __syncthreads();
}

// One pair of rows at the cosine x of its scattering angle: g g' eff KN (I_a + I_b), f the
// factors of the angle's whole degree.
__device__ __forceinline__ float pair_cos(const float4 ua, const float4 ub)
{
    // scattering angle = pi - angle(A S B) (law of cosines, kn_formula.py:36-41)
    return -fmaf(ua.x, ub.x, fmaf(ua.y, ub.y, ua.z * ub.z));
}
__device__ __forceinline__ float pair_value(const float2 f, const float4 ua, const float4 ub, const float2 va,
                                            const float2 vb)
{
    const float Ia = __builtin_amdgcn_exp2f(-fmaf(vb.y, f.x, va.y)) * va.x;
    const float Ib = __builtin_amdgcn_exp2f(-fmaf(va.y, f.x, vb.y)) * vb.x;
    return ua.w * ub.w * f.y * (Ia + Ib);
}
__device__ __forceinline__ float pair_term(const DegTable &T, const float4 ua, const float4 ub, const float2 va,
                                           const float2 vb)
{
    const float x = pair_cos(ua, ub);
    const float t = __builtin_amdgcn_sqrtf(fminf(fmaxf(1.0f - fabsf(x), 0.0f), 1.0f));
    const int ci = (int)(t * 256.0f) + (x < 0.0f ? DEG_CELLS : 0);
    const float2 c = T.cell[ci];
    return pair_value(T.fac[__float_as_int(c.y) + (x < c.x ? 1 : 0)], ua, ub, va, vb);
}

// One bin per lane, BINS_WG consecutive bins per workgroup, part p of the points per
// workgroup (., p).  The wavefronts of a workgroup walk the same points side by
// side: the bins of neighbouring angles use mostly the same detectors, whose rows
// then come from L1 (64 bins per workgroup and a quarter of the points per wavefront
// instead: 5.9 ms, each row read from L2 26 times).  The parts are summed by
// k_sss_sum in order; parts == 1 writes the sinogram itself.
template <int GS>
__global__ __launch_bounds__(BINS_WG) void k_sss_bins(const float4 *__restrict__ dir, const float2 *__restrict__ val,
                                                  const float *__restrict__ sp, int nd, int ns,
                                                  const int *__restrict__ bins, int nb,
                                                  const float *__restrict__ tables, float scale, int parts,
                                                  float *__restrict__ out)
{
    __shared__ DegTable T;
    __shared__ float thr[181];
    build_degrees(T, thr, tables);
    const int b = blockIdx.x * BINS_WG + threadIdx.x;
    const bool in = b < nb;
    const int da = in ? bins[2 * b] : 0, db = in ? bins[2 * b + 1] : 0;
    const bool ok = da >= 0 && da < nd && db >= 0 && db < nd;
    // byte offsets of the detectors' rows in a point group
    const unsigned oa = ok ? (unsigned)da * (16u * GS) : 0u, ob = ok ? (unsigned)db * (16u * GS) : 0u;
    // four points per trip: their 16 loads are in flight together
    constexpr int U = 4;
    const int ng = (ns + U - 1) / U, per = (ng + parts - 1) / parts;
    const int g0 = (int)blockIdx.y * per, g1 = min(ng, g0 + per);
    float acc = 0.0f;
    for (int g = g0; g < g1; ++g) {
        float m[U];
        bool any = false;
#pragma unroll
        for (int j = 0; j < U; ++j) {
            m[j] = U * g + j < ns ? sp[4 * (U * g + j) + 3] : 0.0f;
            any |= m[j] != 0.0f;
        }
        if (!any) continue;   // the kn term is proportional to mu(S) (kn_formula.py:16)
        float4 ua[U], ub[U];
        float2 va[U], vb[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            // (GS == 1 has no padding rows)
            const int64_t row = (int64_t)(GS == 1 ? min(U * g + j, ns - 1) : U * g) * nd;
            const char *D = reinterpret_cast<const char *>(dir + row), *V = reinterpret_cast<const char *>(val + row);
            const int k = GS == 1 ? 0 : j;
            ua[j] = *reinterpret_cast<const float4 *>(D + oa + 16 * k);
            ub[j] = *reinterpret_cast<const float4 *>(D + ob + 16 * k);
            va[j] = *reinterpret_cast<const float2 *>(V + (oa >> 1) + 8 * k);
            vb[j] = *reinterpret_cast<const float2 *>(V + (ob >> 1) + 8 * k);
        }
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const float t = fmaf(m[j], pair_term(T, ua[j], ub[j], va[j], vb[j]), sum);
            sum = m[j] == 0.0f ? sum : t;
        }
        acc += sum;
    }
    if (!in) return;
    // a detector index outside the table gives NaN
    if (!ok) acc = __builtin_nanf("");
    if (parts == 1) out[b] = acc * scale;
    else out[(int64_t)blockIdx.y * nb + b] = acc;
}

// The same sum for bins in any order, LP lanes per bin: lane j takes the points j, j + LP,
// ..., the lanes' sums are combined by a fixed butterfly.  The whole degree comes from acosf,
// put right by the thresholds on either side (the table's 514 cells cost a workgroup more
// than its few pairs).  Bound by the rows' traffic from L2.
template <int LP>
__global__ __launch_bounds__(256) void k_sss_bins_any(const float4 *__restrict__ dir, const float2 *__restrict__ val,
                                                      const float *__restrict__ sp, int nd, int ns,
                                                      const int *__restrict__ bins, int nb,
                                                      const float *__restrict__ tables, float scale,
                                                      float *__restrict__ out)
{
    __shared__ float thr[181];
    __shared__ float2 fac[181];
    build_thresholds(thr, fac, tables, 256);
    const int64_t b = (int64_t)blockIdx.x * (256 / LP) + (int)threadIdx.x / LP;
    const int lane = (int)threadIdx.x % LP;
    if (b >= nb) return;   // all lanes of a bin leave together
    const int da = bins[2 * b], db = bins[2 * b + 1];
    if (da < 0 || da >= nd || db < 0 || db >= nd) {   // a detector index outside the table
        if (lane == 0) out[b] = __builtin_nanf("");
        return;
    }
    const RowLayout<SSS_GROUP_ANY> R{nd, ns};
    constexpr int U = 2;   // points of a lane in flight
    float acc = 0.0f;
    for (int s0 = lane; s0 < ns; s0 += LP * U) {
        float m[U];
        float4 ua[U], ub[U];
        float2 va[U], vb[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int s = min(s0 + LP * j, ns - 1);
            m[j] = s0 + LP * j < ns ? sp[4 * s + 3] : 0.0f;
            const int64_t a = R.at(da, s), c = R.at(db, s);
            ua[j] = dir[a];
            ub[j] = dir[c];
            va[j] = val[a];
            vb[j] = val[c];
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const float x = pair_cos(ua[j], ub[j]);
            int k = min((int)(acosf(fminf(1.0f, fmaxf(-1.0f, x))) * 57.295779513082323f), 180);
            if (k < 180 && x < thr[k + 1]) ++k;
            else if (k > 0 && x >= thr[k]) --k;
            const float t = fmaf(m[j], pair_value(fac[k], ua[j], ub[j], va[j], vb[j]), acc);
            acc = m[j] == 0.0f ? acc : t;   // the kn term is proportional to mu(S) (kn_formula.py:16)
        }
    }
    for (int k = LP / 2; k > 0; k >>= 1) acc += __shfl_xor(acc, k);
    if (lane == 0) out[b] = acc * scale;
}

__global__ __launch_bounds__(256) void k_sss_sum(const float *__restrict__ part, int parts, int nb, float scale,
                                                 float *__restrict__ out)
{
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= nb) return;
    float acc = 0.0f;
    for (int p = 0; p < parts; ++p) acc += part[(int64_t)p * nb + b];
    out[b] = acc * scale;
}

// work[0] += sum_e sino[bins[e]], work[1] += sum_e y[e] (double, one atomic per block)
__device__ __forceinline__ float bin_value(const float *__restrict__ sino, const int32_t *__restrict__ bins,
                                           int64_t e, int64_t nbins)
{
    const int32_t b = bins[e];
    return (b >= 0 && b < nbins) ? sino[b] : 0.0f;
}

__global__ __launch_bounds__(256) void k_scatter_sums(const float *__restrict__ y, const int32_t *__restrict__ bins,
                                                      const float *__restrict__ sino, int64_t nbins, int64_t n,
                                                      double *__restrict__ work)
{
    __shared__ double rs[256], ry[256];
    double a = 0.0, b = 0.0;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        a += (double)bin_value(sino, bins, e, nbins);
        b += (double)(y ? y[e] : 1.0f);
    }
    rs[threadIdx.x] = a;
    ry[threadIdx.x] = b;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) {
            rs[threadIdx.x] += rs[threadIdx.x + k];
            ry[threadIdx.x] += ry[threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        atomicAdd(work, rs[0]);
        atomicAdd(work + 1, ry[0]);
    }
}

__global__ void k_zero2(double *__restrict__ work)
{
    if (threadIdx.x < 2) work[threadIdx.x] = 0.0;
}

// out[e] = (y[e] - sino[bins[e]] / S * Y * fraction) * w[e]   (S = 0: no subtraction)
__global__ __launch_bounds__(256) void k_scatter_apply(const float *__restrict__ y, const float *__restrict__ w,
                                                       const int32_t *__restrict__ bins,
                                                       const float *__restrict__ sino, int64_t nbins, int64_t n,
                                                       float fraction,
                                                       const double *__restrict__ work, float *__restrict__ out)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const double S = work[0];
    const float c = S > 0.0 ? (float)(work[1] * (double)fraction / S) : 0.0f;
    const float ye = y ? y[e] : 1.0f;
    float v = ye - bin_value(sino, bins, e, nbins) * c;
    if (w) v *= w[e];
    out[e] = v;
}

}  // namespace srf

using namespace srf;

// Rows in the layout of sinogram order or of any order (RowLayout).
static int prepare_rows(const float *det, int32_t n_det, const float *points, int32_t n_points, const float *em_int,
                        const float *mu_int, void *rows, size_t rows_bytes, bool ordered, hipStream_t s)
{
    if (n_det <= 0 || n_points <= 0) return SRF_ERR_INVALID_ARG;
    if (!det || !points || !em_int || !mu_int || !rows) return SRF_ERR_INVALID_ARG;
    if (rows_bytes < srf_sss_rows_bytes(n_det, n_points)) return SRF_ERR_WORKSPACE;
    if ((reinterpret_cast<uintptr_t>(rows) & 15) != 0) return SRF_ERR_INVALID_ARG;
    const int64_t nblk = (int64_t)((n_points + 63) / 64) * ((n_det + 3) / 4);
    if (nblk >= (int64_t)1 << 31) return SRF_ERR_UNSUPPORTED;   // 16 TiB of rows
    const dim3 grid((unsigned)nblk);
    float4 *dir = (float4 *)rows;
#define SRF_PAIRS(GS)                                                                                                  \
    hipLaunchKernelGGL(k_sss_pairs<GS>, grid, dim3(256), 0, s, det, points, em_int, mu_int, n_det, n_points, dir,     \
                       (float2 *)(dir + RowLayout<GS>{n_det, n_points}.padded()))
    if (!ordered) SRF_PAIRS(SSS_GROUP_ANY);
    else if (grouped_rows(n_points)) SRF_PAIRS(SSS_GROUP);
    else SRF_PAIRS(1);
#undef SRF_PAIRS
    return launch_status();
}

// Lanes per bin in any order: 16 for few points, whose lanes 64 would leave idle, and for
// enough bins to fill the chip with.  us, 16 / 64 lanes, random pairs: 131072 bins of 63
// points 31 / 60, 20000 of 250 21 / 21, 8192 of 300 17 / 19, 8192 of 5000 209 / 263, 4000 of
// 2000 62 / 52, 256 of 2000 56 / 17.  Detector-major rows, a wavefront per bin below 32768
// bins and a lane per bin from there on, as before: 88, 28, 24, 350, 58 and 26.
constexpr int SSS_FEW_POINTS = 256, SSS_MANY_BINS = 8192;

static int sum_bins(const void *rows, int32_t n_det, const float *points, int32_t n_points, const int32_t *bins,
                    int32_t n_bins, const float *tables, float scale, float *out, bool ordered, hipStream_t s)
{
    if (n_bins < 0 || n_det <= 0 || n_points <= 0) return SRF_ERR_INVALID_ARG;
    if (n_bins == 0) return SRF_OK;
    if (!rows || !points || !bins || !tables || !out) return SRF_ERR_INVALID_ARG;
    const float4 *dir = (const float4 *)rows;
    if (!ordered) {
        const float2 *val = (const float2 *)(dir + RowLayout<SSS_GROUP_ANY>{n_det, n_points}.padded());
        const int lp = n_points < SSS_FEW_POINTS || n_bins >= SSS_MANY_BINS ? 16 : 64;
        const dim3 grid((unsigned)(((int64_t)n_bins * lp + 255) / 256));
        if (lp == 16)
            hipLaunchKernelGGL(k_sss_bins_any<16>, grid, dim3(256), 0, s, dir, val, points, n_det, n_points, bins, n_bins,
                               tables, scale, out);
        else
            hipLaunchKernelGGL(k_sss_bins_any<64>, grid, dim3(256), 0, s, dir, val, points, n_det, n_points, bins, n_bins,
                               tables, scale, out);
        return launch_status();
    }
    const int nblk = (n_bins + BINS_WG - 1) / BINS_WG;
    // parts of the points: two rounds of workgroups on the chip, each part with at least 64
    // points (16 in up to 4 parts: 16384 ring bins of 300 points 41 -> 23 us)
    const int most = n_points / 64 > 4 ? n_points / 64 : n_points / 16 < 4 ? n_points / 16 : 4;
    int parts = (1024 + nblk - 1) / nblk;
    if (parts > most) parts = most;
    if (parts > 256) parts = 256;
    if (parts < 1) parts = 1;
    float *part = nullptr;
    if (parts > 1) {
        part = capturing(s) ? nullptr : static_cast<float *>(pool_get((size_t)parts * n_bins * sizeof(float), s));
        if (!part) parts = 1;
    }
    const dim3 grid((unsigned)nblk, (unsigned)parts);
    float *dst = part ? part : out;
#define SRF_BINS(GS)                                                                                                   \
    hipLaunchKernelGGL(k_sss_bins<GS>, grid, dim3(BINS_WG), 0, s, dir,                                                 \
                       (const float2 *)(dir + RowLayout<GS>{n_det, n_points}.padded()), points, n_det, n_points, bins, \
                       n_bins, tables, scale, parts, dst)
    if (grouped_rows(n_points)) SRF_BINS(SSS_GROUP);
    else SRF_BINS(1);
#undef SRF_BINS
    int rc = launch_status();
    if (part) {
        if (rc == SRF_OK) {
            hipLaunchKernelGGL(k_sss_sum, dim3((unsigned)((n_bins + 255) / 256)), dim3(256), 0, s, part, parts, n_bins,
                               scale, out);
            rc = launch_status();
        }
        pool_put(part, s, false, true);
    }
    return rc;
}

extern "C" {

size_t srf_sss_rows_bytes(int32_t n_det, int32_t n_points)
{
    if (n_det <= 0 || n_points <= 0) return 0;
    return (size_t)n_det * (size_t)n_points * 32;
}

int srf_sss_prepare(const float *det, int32_t n_det, const float *points, int32_t n_points, const float *em_int,
                    const float *mu_int, void *rows, size_t rows_bytes, void *stream)
{
    return prepare_rows(det, n_det, points, n_points, em_int, mu_int, rows, rows_bytes, false, (hipStream_t)stream);
}

int srf_sss_sinogram(const void *rows, int32_t n_det, const float *points, int32_t n_points, const int32_t *bins,
                     int32_t n_bins, const float *tables, float scale, float *out, void *stream)
{
    return sum_bins(rows, n_det, points, n_points, bins, n_bins, tables, scale, out, false, (hipStream_t)stream);
}

int srf_sss_prepare_ordered(const float *det, int32_t n_det, const float *points, int32_t n_points, const float *em_int,
                            const float *mu_int, void *rows, size_t rows_bytes, void *stream)
{
    return prepare_rows(det, n_det, points, n_points, em_int, mu_int, rows, rows_bytes, true, (hipStream_t)stream);
}

int srf_sss_sinogram_ordered(const void *rows, int32_t n_det, const float *points, int32_t n_points,
                             const int32_t *bins, int32_t n_bins, const float *tables, float scale, float *out,
                             void *stream)
{
    return sum_bins(rows, n_det, points, n_points, bins, n_bins, tables, scale, out, true, (hipStream_t)stream);
}

int srf_scatter_correct(const float *y, const float *weight, const int32_t *bins, const float *sino, int64_t n_bins,
                        int64_t n, float fraction, double *work, float *out, void *stream)
{
    if (n < 0 || n_bins < 1 || !bins || !sino || !work || !out) return SRF_ERR_INVALID_ARG;
    if (n == 0) return SRF_OK;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(k_zero2, dim3(1), dim3(64), 0, s, work);
    const unsigned nb = (unsigned)((n + 255) / 256);
    hipLaunchKernelGGL(k_scatter_sums, dim3(nb < 1024 ? nb : 1024), dim3(256), 0, s, y, bins, sino, n_bins, n, work);
    hipLaunchKernelGGL(k_scatter_apply, dim3(nb), dim3(256), 0, s, y, weight, bins, sino, n_bins, n, fraction,
                       (const double *)work, out);
    return launch_status();
}

}  // extern "C"
