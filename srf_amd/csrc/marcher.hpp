// marcher.hpp -- the device ray marcher shared by every projector/backprojector
// kernel of libsrf_hip.so (gfx950).
//
// Semantics: the Siddon-type slab marcher of srfnef/cc/siddon/siddon.cu.cc:12-656
// and srfnef/cc/siddon_tof/siddon_tof.cu.cc:14-707.  Every expression that
// decides WHICH voxel a term lands in is evaluated with the reference's own
// float operations in the reference's order (this translation unit is built
// with -ffp-contract=off; HIP's default float division and sqrt are correctly
// rounded), so voxel indices and branch choices are bit-identical to an
// un-contracted IEEE build of the reference.  Weights are re-associated
// (per-event constants hoisted, TOF Gaussian evaluated in fp32 through
// v_exp_f32) and agree to a few ulp.
//
// Pieces:
//   ray_setup     endpoints -> voxel units, early-out tests, L, dominance tests
//   make_branch   the primary/secondary description of one reference branch
//                 (x branch siddon.cu.cc:46-191, y branch :192-335)
//   clip_range    slabs whose secondary/axial coordinates can lie in the image
//                 (conservative; the exact per-slab tests still decide)
//   fp_cut_range  the projector's segment cuts (siddon.cu.cc:56-57,203-204;
//                 siddon_tof.cu.cc:67-74,228-235) as an exact slab interval
//   slab_cells, slab_fractions   one slab: cells, crossings, term fractions (the
//                 flattened branch tree); slab_eval: both
//   march_slabs   the slab loop: carried boundary values, every slab handed to a sink
//   march_event   all of the above for one event (one-event-per-lane kernels)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace srf {

enum : int { V_FP = 0, V_BP = 1 };

// Per-launch constants.  Computed on the host with the same float expressions
// as siddon.cu.cc:19-22,39-41 and siddon_tof.cu.cc:46-47,57 (bit-identical).
struct LaunchGeom {
    int nx, ny, nz;
    float cx, cy, cz;
    float dx_;            // sx / nx
    float dy, dz;         // sy / ny / dx_, sz / nz / dx_
    float nx2, ny2, nz2;  // n / 2.0f
    float tof_bin_;       // tof_bin / dx_
    float tof_sigma2_;    // tof_sigma2 / dx_ / dx_
    float tse;            // tof_sigma2_ + tof_bin_^2 / 12
    float tof_c0;         // (float)(tof_bin_ / sqrt(2*PI*tse))   (double, as the reference)
    float tof_c1;         // -0.5 * log2(e) / tse                 (exp(-t2/2) == exp2(c1 * d^2))
};

__device__ __forceinline__ int floor_to_int(float v)
{
    // v_floor_f32 + v_cvt_i32_f32: NaN -> 0, saturating (the oracle mirrors it)
    return (int)floorf(v);
}

__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// v_cvt_flr_i32_f32: floor and convert in one VALU op (NaN -> 0, saturating,
// as v_floor_f32 + v_cvt_i32_f32).
__device__ __forceinline__ int cvt_flr(float v)
{
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// med3(x, lo, hi) = min(max(x, lo), hi) for lo <= hi, one v_med3_i32 (the
// compiler emits it only for constant bounds), and a * b + c with a and b taken
// as signed 24-bit integers (v_mad_i32_i24: the clamped cell index is -1 on
// the low-edge halo of a tile at the image origin, which the unsigned form
// would read as 2^24 - 1).  Plain ALU instructions, no memory access.
__device__ __forceinline__ int med3_i32(int x, int lo, int hi)
{
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(lo), "v"(hi));
    return r;
}
__device__ __forceinline__ int mad_i24(int a, int b, int c)
{
    int r;
    asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Minimum / maximum of two non-negative finite floats as integer operations on
// their bit patterns (which order the same way): no NaN canonicalisation.
__device__ __forceinline__ float min_nonneg(float a, float b)
{
    return __uint_as_float(min(__float_as_uint(a), __float_as_uint(b)));
}
__device__ __forceinline__ float max_nonneg(float a, float b)
{
    return __uint_as_float(max(__float_as_uint(a), __float_as_uint(b)));
}

// Branch-independent part of one event.
struct RaySetup {
    float x1, y1, z1, x2, y2, z2;
    float xd, yd, zd, L;
    float ratio1;     // TOF position of the emission point along p1->p2 (siddon_tof.cu.cc:44)
    bool nan;         // non-finite endpoint: projection NaN, backprojection skips
    bool live;        // passes the 10-voxel transaxial cut (siddon.cu.cc:34)
    bool q2;          // non-TOF projector's axial cut fires (siddon.cu.cc:38)
    bool xdom_ge;     // |xd| >= |yd|  (non-TOF projector, siddon.cu.cc:46)
    bool xdom_gt;     // |xd| >  |yd|  (everything else)
};

template <bool TOF>
__device__ __forceinline__ void ray_setup(const float *__restrict__ lor, float tof_value, const LaunchGeom &G,
                                          RaySetup &r)
{
    r.x1 = (lor[0] - G.cx) / G.dx_;
    r.y1 = (lor[1] - G.cy) / G.dx_;
    r.z1 = (lor[2] - G.cz) / G.dx_;
    r.x2 = (lor[3] - G.cx) / G.dx_;
    r.y2 = (lor[4] - G.cy) / G.dx_;
    r.z2 = (lor[5] - G.cz) / G.dx_;
    r.nan = !(isfinite(r.x1) && isfinite(r.y1) && isfinite(r.z1) && isfinite(r.x2) && isfinite(r.y2) &&
              isfinite(r.z2));
    r.xd = r.x2 - r.x1;
    r.yd = r.y2 - r.y1;
    r.zd = r.z2 - r.z1;
    const float t2d = r.xd * r.xd + r.yd * r.yd;
    const float tlen = sqrtf(t2d);
    r.live = !r.nan && !(tlen < 10.0f);
    r.q2 = tlen < fabsf(r.zd);
    r.L = sqrtf(t2d + r.zd * r.zd);
    const float axd = fabsf(r.xd), ayd = fabsf(r.yd);
    r.xdom_ge = axd >= ayd;
    r.xdom_gt = axd > ayd;
    r.ratio1 = 0.0f;
    if (TOF) r.ratio1 = (float)((1.0 - (double)(tof_value / G.dx_ / r.L)) / 2);
}

// One primary-axis branch.
struct Branch {
    bool xdom;
    float p1, p2, sec1, ks, kz;
    float ds;              // secondary divisor: dy (x branch) or 1 (y branch; x / 1.0f == x)
    float ns2, np2;
    float pd_tof;          // dx (=1) on the x branch, dy on the y branch (siddon_tof.cu.cc:55,215)
    int np, ns, stride_p, stride_s;
    float sq;              // sqrt(1 + ks^2 + kz^2)
};

__device__ __forceinline__ void make_branch(const RaySetup &r, bool xdom, const LaunchGeom &G, Branch &B)
{
    B.xdom = xdom;
    if (xdom) {
        B.p1 = r.x1; B.p2 = r.x2; B.sec1 = r.y1;
        B.ks = r.yd / r.xd; B.kz = r.zd / r.xd;
        B.np = G.nx; B.ns = G.ny; B.np2 = G.nx2; B.ns2 = G.ny2;
        B.stride_p = 1; B.stride_s = G.nx;
        B.pd_tof = 1.0f;
        B.ds = G.dy;
    } else {
        B.p1 = r.y1; B.p2 = r.y2; B.sec1 = r.x1;
        B.ks = r.xd / r.yd; B.kz = r.zd / r.yd;
        B.np = G.ny; B.ns = G.nx; B.np2 = G.ny2; B.ns2 = G.nx2;
        B.stride_p = G.nx; B.stride_s = 1;
        B.pd_tof = G.dy;
        B.ds = 1.0f;
    }
    B.sq = sqrtf(1.0f + B.ks * B.ks + B.kz * B.kz);
}

// Term weight constant of a branch: sqrt(1+k^2+kz^2)*dx_ [/L/L] [* tof norm]
// (siddon.cu.cc:94 projector, :418 backprojector).
template <bool TOF>
__device__ __forceinline__ float branch_weight(const Branch &B, const RaySetup &r, const LaunchGeom &G, bool fp)
{
    float W = B.sq * G.dx_;
    if (fp) W = W / r.L / r.L;
    if (TOF) W = W * G.tof_c0;
    return W;
}

// Margin in cells for a coordinate (c + k (x - p1)) / d + n2 over |x| <= np2: a
// hundredth of a cell and 8 float ulps of its largest intermediate value, above the
// rounding of both the float estimates below and the marcher's own coordinates.
__device__ __forceinline__ float cell_margin(float c, float k, float p1, float np2, float d, float n2)
{
    return 1e-2f + 1e-6f * ((fabsf(c) + fabsf(k) * (np2 + fabsf(p1))) / d + n2);
}

// Interval of primary coordinate x on which value(x) = (c + k*(x - p1))/d + n2
// lies in [lo_v, hi_v] (a margin wider than exact, see cell_margin); empty => a > b.
__device__ __forceinline__ void axis_window(float c, float k, float p1, float d, float n2, float lo_v, float hi_v,
                                            float &a, float &b)
{
    if (k == 0.0f) {
        const float v = c / d + n2;
        if (v >= lo_v && v <= hi_v) { a = -1e30f; b = 1e30f; }
        else { a = 1e30f; b = -1e30f; }
    } else {
        const float xa = p1 + ((lo_v - n2) * d - c) / k;
        const float xb = p1 + ((hi_v - n2) * d - c) / k;
        a = fminf(xa, xb);
        b = fmaxf(xa, xb);
    }
}

// Slabs [lo, hi) that can hold a term: the secondary and axial coordinates of
// a slab must reach [-1, n] (widened by the margin, and by one slab on each side).
__device__ __forceinline__ void clip_range(const Branch &B, const RaySetup &r, const LaunchGeom &G, int &lo, int &hi)
{
    const float ms = cell_margin(B.sec1, B.ks, B.p1, B.np2, B.ds, B.ns2);
    const float mz = cell_margin(r.z1, B.kz, B.p1, B.np2, G.dz, G.nz2);
    float sa, sb, za, zb;
    axis_window(B.sec1, B.ks, B.p1, B.ds, B.ns2, -1.0f - ms, (float)B.ns + ms, sa, sb);
    axis_window(r.z1, B.kz, B.p1, G.dz, G.nz2, -1.0f - mz, (float)G.nz + mz, za, zb);
    const float xl = fmaxf(fmaxf(-B.np2, sa - 1.0f), za - 1.0f);
    const float xh = fminf(fminf(B.np2, sb + 1.0f), zb + 1.0f);
    if (!(xl <= xh)) {
        lo = 0; hi = 0;
    } else {
        lo = max(0, (int)floorf(xl + B.np2) - 1);
        hi = min(B.np, (int)ceilf(xh + B.np2) + 1);
    }
}

// (int) of a float clamped far inside the int range.
__device__ __forceinline__ int flt_to_int(float v)
{
    return (int)fminf(fmaxf(v, -1.0e9f), 1.0e9f);
}

// (int) of a double clamped far inside the int range.
__device__ __forceinline__ int dbl_to_int(double v)
{
    return (int)fmin(fmax(v, -1.0e9), 1.0e9);
}

// First ip in [lo, hi] with keep(ip) true for a predicate that is false then
// true along ip; `guess` only sets where the exact search starts.
template <class P>
__device__ __forceinline__ int first_true(P keep, int lo, int hi, int guess)
{
    int ip = min(max(guess, lo), hi);
    while (ip > lo && keep(ip - 1)) --ip;
    while (ip < hi && !keep(ip)) ++ip;
    return ip;
}

// The projector's segment cut as the exact slab interval [a, b) within [lo, hi).
// Each reference predicate is monotone in the slab index; the interval ends are
// located with the reference's own float comparisons (slab boundaries
// pp1 = ip - np2 and pp2 = pp1 + 1 are exact in float).
template <bool TOF>
__device__ __forceinline__ void fp_cut_range(const Branch &B, int lo, int hi, int &a, int &b)
{
    const float p1 = B.p1, p2 = B.p2, np2 = B.np2;
    a = lo;
    b = hi;
    if (!TOF) {
        // siddon.cu.cc:56-57 / 203-204: skip (p1<p2 && pp2>p2) || (p1>=p2 && pp1<p2)
        if (p1 < p2) {
            auto cut = [&](int ip) { return ((float)ip - np2) + 1.0f > p2; };
            b = first_true(cut, lo, hi, flt_to_int(floorf(p2 + np2)));
        } else {
            auto keep = [&](int ip) { return (float)ip - np2 >= p2; };
            a = first_true(keep, lo, hi, flt_to_int(ceilf(p2 + np2)));
        }
    } else if (B.xdom) {
        // siddon_tof.cu.cc:67-74: skip (p2>p1 && pp1<=p1) || (p2<p1 && pp2>=p1)
        if (p2 > p1) {
            auto keep = [&](int ip) { return (float)ip - np2 > p1; };
            a = first_true(keep, lo, hi, flt_to_int(floorf(p1 + np2)) + 1);
        } else if (p2 < p1) {
            auto cut = [&](int ip) { return ((float)ip - np2) + 1.0f >= p1; };
            b = first_true(cut, lo, hi, flt_to_int(ceilf(p1 + np2)) - 1);
        }
    } else {
        // siddon_tof.cu.cc:228-235: skip (p2>p1 && pp1<p1) || (p2<p1 && pp2>p1)
        if (p2 > p1) {
            auto keep = [&](int ip) { return (float)ip - np2 >= p1; };
            a = first_true(keep, lo, hi, flt_to_int(ceilf(p1 + np2)));
        } else if (p2 < p1) {
            auto cut = [&](int ip) { return ((float)ip - np2) + 1.0f > p1; };
            b = first_true(cut, lo, hi, flt_to_int(floorf(p1 + np2)));
        }
    }
    if (b < a) b = a;
}

// TOF Gaussian of siddon_tof.cu.cc:55-59 as a linear function of the slab's
// lower boundary pp1 = ip - np2 (exact in float):
//   pc = ((ip - np/2) + 0.5) * pd_tof = (pp1 + off) * pd_tof, off = np2 - np/2 + 0.5
//   d  = ((pc - p1) / (p2 - p1) - ratio1) * L
//   exp(-d^2 / (2 tse)) = exp2(-(d * sqrt(log2(e) / (2 tse)))^2)
// Coefficients in double, rounded once.
template <bool TOF>
__device__ __forceinline__ void tof_coeffs_d(const Branch &B, const RaySetup &r, const LaunchGeom &G, double &tA,
                                             double &tB)
{
    tA = tB = 0.0;
    if (!TOF) return;
    const double off = (double)B.np2 - (double)(B.np / 2) + 0.5;
    const double s = sqrt(0.5 * 1.4426950408889634 / (double)G.tse);
    const double k = (double)r.L / ((double)B.p2 - (double)B.p1);
    tA = (double)B.pd_tof * k * s;
    tB = ((off * (double)B.pd_tof - (double)B.p1) * k - (double)r.ratio1 * (double)r.L) * s;
}

template <bool TOF>
__device__ __forceinline__ void tof_coeffs(const Branch &B, const RaySetup &r, const LaunchGeom &G, float &tA,
                                           float &tB)
{
    double a, b;
    tof_coeffs_d<TOF>(B, r, G, a, b);
    tA = (float)a;
    tB = (float)b;
}

// One slab of a ray: its cells, crossings and term fractions.  With cs1 <= cs2
// the two secondary cells the slab spans and cz1 <= cz2 the axial ones, the
// reference's branch tree (siddon.cu.cc:86-189 x-dominant, 231-333 y-dominant;
// siddon_tof.cu.cc:102-210, 244-366) is, flattened:
//   term 1, fraction r1, cell (cs1, cz1);
//   term 2, fraction r2, cell (cs1, cz2) if rs > rz, else (cs2, cz1): where both
//           axes cross;
//   term 3, fraction r3, cell (cs2, cz2): where an axis crosses;
// each where its cell lies in the image, and term 2 only with cz1 >= -1 (resp.
// cs1 >= -1), term 3 with both (the top-level tests cs1 >= (crossing ? -1 : 0)
// && cs1 < ns, and the same along z, are implied by these).
struct Slab {
    int cs1, cs2, cz1, cz2;
    bool bs, bz;       // the slab crosses a secondary / axial cell boundary
    bool sgt;          // rs > rz
    float r1, r2, r3;
    float sl, sh, zl, zh;
};

// S0, Z0 (S1, Z1): secondary and axial coordinate at the slab's lower (upper)
// boundary.
__device__ __forceinline__ void slab_cells(Slab &c, float S0, float S1, float Z0, float Z1, bool ks_pos, bool kz_pos)
{
    c.sl = ks_pos ? S0 : S1;
    c.sh = ks_pos ? S1 : S0;
    c.zl = kz_pos ? Z0 : Z1;
    c.zh = kz_pos ? Z1 : Z0;
    c.cs1 = cvt_flr(c.sl);
    c.cs2 = cvt_flr(c.sh);
    c.cz1 = cvt_flr(c.zl);
    c.cz2 = cvt_flr(c.zh);
    c.bs = c.cs1 != c.cs2;
    c.bz = c.cz1 != c.cz2;
}

// Fractions from reciprocal estimates; exact quotients only where those cannot
// decide rs > rz, which picks term 2's cell (they lie in (0, 1]: the absolute
// margin is far above the estimates' few-ulp error).
__device__ __forceinline__ void slab_fractions(Slab &c)
{
    const float dsv = c.sh - c.sl, dzv = c.zh - c.zl;
    const float ns_ = (float)c.cs2 - c.sl, nz_ = (float)c.cz2 - c.zl;
    const float es_ = ns_ * __builtin_amdgcn_rcpf(dsv), ez_ = nz_ * __builtin_amdgcn_rcpf(dzv);
    float rs = c.bs ? es_ : 1.0f, rz = c.bz ? ez_ : 1.0f;
    float dr = rs - rz;
    if (c.bs && c.bz && !(fabsf(dr) > 4e-6f)) {
        rs = ns_ / dsv;
        rz = nz_ / dzv;
        dr = rs - rz;
    }
    asm("" : "+v"(dr));   // keeps |dr| a source modifier of its uses
    c.sgt = dr > 0.0f;
    c.r1 = min_nonneg(rs, rz);
    c.r2 = fabsf(dr);
    c.r3 = 1.0f - ((c.bs && c.bz) ? max_nonneg(rs, rz) : c.r1);
}

__device__ __forceinline__ Slab slab_eval(float S0, float S1, float Z0, float Z1, bool ks_pos, bool kz_pos)
{
    Slab c;
    slab_cells(c, S0, S1, Z0, Z1, ks_pos, kz_pos);
    slab_fractions(c);
    return c;
}

// Which of a slab's terms apply, and term 2's cell.
struct SlabTerms {
    bool v1, v2, v3;
    int csm, czm;
};
__device__ __forceinline__ SlabTerms slab_terms(const Slab &c, int ns, int nz)
{
    const bool s1 = (unsigned)c.cs1 < (unsigned)ns, s2 = (unsigned)c.cs2 < (unsigned)ns;
    const bool z1 = (unsigned)c.cz1 < (unsigned)nz, z2 = (unsigned)c.cz2 < (unsigned)nz;
    const bool los = c.cs1 >= -1, loz = c.cz1 >= -1, both = c.bs && c.bz;
    SlabTerms t;
    t.v1 = s1 && z1;
    t.v2 = both && (c.sgt ? (s1 && z2 && loz) : (s2 && z1 && los));
    t.v3 = (c.bs || c.bz) && s2 && z2 && los && loz;
    t.csm = c.sgt ? c.cs1 : c.cs2;
    t.czm = c.sgt ? c.cz2 : c.cz1;
    return t;
}

// Branch labels of a slab's terms (the digest's): siddon.cu.cc's cases in order.
__device__ __forceinline__ int slab_label1(const Slab &c) { return c.bs ? (c.bz ? (c.sgt ? 5 : 8) : 3) : (c.bz ? 1 : 0); }
__device__ __forceinline__ int slab_label2(const Slab &c) { return c.sgt ? 6 : 9; }
__device__ __forceinline__ int slab_label3(const Slab &c) { return c.bs ? (c.bz ? (c.sgt ? 7 : 10) : 4) : 2; }

// Secondary / axial coordinate of a ray at primary coordinate pp, in the
// reference's operations.
template <bool DIV_S>
__device__ __forceinline__ float coord_s(const Branch &B, float pp)
{
    const float s = B.sec1 + B.ks * (pp - B.p1);
    return (DIV_S ? s / B.ds : s) + B.ns2;
}
template <bool DIV_Z>
__device__ __forceinline__ float coord_z(const Branch &B, float z1, const LaunchGeom &G, float pp)
{
    const float z = z1 + B.kz * (pp - B.p1);
    return (DIV_Z ? z / G.dz : z) + G.nz2;
}

// The slab loop over [a, b).  Act provides
//   void slab(int ip, const Slab &c, float e)
// with ip the primary slab and e the TOF Gaussian at it (1 without TOF).
template <bool TOF, bool DIV_S, bool DIV_Z, class Act>
__device__ __forceinline__ void march_slabs(const Branch &B, float z1, const LaunchGeom &G, int a, int b, float tA,
                                            float tB, Act &act)
{
    const bool ks_pos = B.ks >= 0.0f, kz_pos = B.kz >= 0.0f;
    float pp1 = (float)a - B.np2;
    float S0 = coord_s<DIV_S>(B, pp1), Z0 = coord_z<DIV_Z>(B, z1, G, pp1);
    for (int ip = a; ip < b; ++ip) {
        const float pp2 = pp1 + 1.0f;
        const float S1 = coord_s<DIV_S>(B, pp2), Z1 = coord_z<DIV_Z>(B, z1, G, pp2);
        const Slab c = slab_eval(S0, S1, Z0, Z1, ks_pos, kz_pos);
        float e = 1.0f;
        if (TOF) {
            const float d = fmaf(pp1, tA, tB);
            e = __builtin_amdgcn_exp2f(-(d * d));
        }
        act.slab(ip, c, e);
        pp1 = pp2;
        S0 = S1;
        Z0 = Z1;
    }
}

// The slab interval and branch of one event, as one reference device function:
// [a, b) is empty where the event has no terms.  Not for r.nan events.
template <bool TOF, int VAR>
__device__ __forceinline__ void event_slabs(const RaySetup &r, const LaunchGeom &G, Branch &B, int &a, int &b)
{
    const bool xdom = (!TOF && VAR == V_FP) ? r.xdom_ge : r.xdom_gt;
    make_branch(r, xdom, G, B);
    a = b = 0;
    if (!r.live || (!TOF && VAR == V_FP && r.q2)) return;
    int lo, hi;
    clip_range(B, r, G, lo, hi);
    a = lo;
    b = hi;
    if (VAR == V_FP) fp_cut_range<TOF>(B, lo, hi, a, b);
}

// One event: Act provides
//   void begin(const Branch &B, float W)          its branch and weight constant
//   void slab(int ip, const Slab &c, float e)
//   void nan_event()                              (non-finite endpoints)
// lane `part` of `parts` takes its share of the event's slabs.
template <bool TOF, int VAR, bool DIV_S, bool DIV_Z, class Act>
__device__ __forceinline__ void march_event(const float *__restrict__ lor, float tof_value, const LaunchGeom &G,
                                            int part, int parts, Act &act)
{
    RaySetup r;
    ray_setup<TOF>(lor, tof_value, G, r);
    if (r.nan) {
        act.nan_event();
        return;
    }
    Branch B;
    int a, b;
    event_slabs<TOF, VAR>(r, G, B, a, b);
    if (parts > 1) {
        const int share = (b - a + parts - 1) / parts;
        a = min(b, a + part * share);
        b = min(b, a + share);
    }
    if (a >= b) return;
    float tA, tB;
    tof_coeffs<TOF>(B, r, G, tA, tB);
    act.begin(B, branch_weight<TOF>(B, r, G, VAR == V_FP));
    march_slabs<TOF, DIV_S, DIV_Z>(B, r.z1, G, a, b, tA, tB, act);
}

}  // namespace srf
