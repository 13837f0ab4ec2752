// srf_project.hip -- one-shot projector / backprojector kernels (no plan) and their
// C-ABI entry points (declared in include/srf_hip.h).
//
//   k_gather   forward projection, 1 to 16 lanes per event   (Projection[Tof] op)
//   k_bundle   forward projection of a long list, its events sorted into bundles
//              of neighbouring lines over transposed copies of the image
//   k_scatter  backprojection, one event per lane   (Backprojection[Tof] op / adjoint)
//   k_digest   per-event term digest        (verification of voxel indexing)
// All of them evaluate a slab through srf::slab_eval, so the digest proves the
// indexing of the projector and backprojector themselves.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <limits.h>
#include <math.h>
#include <stdint.h>

#include "marcher.hpp"
#include "srf_hip.h"
#include "srf_internal.hpp"

namespace srf {

// Kernel-layout voxel of a cell, for one branch.
struct VoxelIndex {
    int sp, ss, sz, ns, nz;
    __device__ __forceinline__ void set(const Branch &B, const LaunchGeom &G)
    {
        sp = B.stride_p;
        ss = B.stride_s;
        sz = G.nx * G.ny;
        ns = B.ns;
        nz = G.nz;
    }
    __device__ __forceinline__ unsigned at(int ip, int cs, int cz) const
    {
        return (unsigned)ip * (unsigned)sp + (unsigned)cs * (unsigned)ss + (unsigned)cz * (unsigned)sz;
    }
};

// Projections are summed in runs of SUM_RUN slabs, and the runs' sums then: along a
// uniform image the slabs' sums are one constant, which added up one by one in
// float32 rounds the same way over whole binades (4 times the error at 200 slabs).
constexpr int SUM_RUN = 16;

// The weight goes into every slab's sum, so that an image of values near float32's largest
// overflows only where its projection does.  The three loads of a slab are issued together: terms that do not apply read
// voxel 0 and are replaced by zero.
struct GatherAct {
    const float *__restrict__ img;
    float sum, part;
    float W;
    VoxelIndex V;
    __device__ __forceinline__ void begin(const Branch &B, float w)
    {
        V.set(B, *G);
        W = w;
    }
    __device__ __forceinline__ void slab(int ip, const Slab &c, float e)
    {
        const SlabTerms t = slab_terms(c, V.ns, V.nz);
        const unsigned i1 = t.v1 ? V.at(ip, c.cs1, c.cz1) : 0u;
        const unsigned i2 = t.v2 ? V.at(ip, t.csm, t.czm) : 0u;
        const unsigned i3 = t.v3 ? V.at(ip, c.cs2, c.cz2) : 0u;
        float g1 = img[i1], g2 = img[i2], g3 = img[i3];
        g1 = t.v1 ? g1 : 0.0f;
        g2 = t.v2 ? g2 : 0.0f;
        g3 = t.v3 ? g3 : 0.0f;
        part = fmaf(fmaf(g1, c.r1, fmaf(g2, c.r2, g3 * c.r3)), e * W, part);
        if ((ip & (SUM_RUN - 1)) == SUM_RUN - 1) {
            sum += part;
            part = 0.0f;
        }
    }
    __device__ __forceinline__ void nan_event() { sum = __builtin_nanf(""); }
    const LaunchGeom *G;
};

struct ScatterAct {
    float *__restrict__ img;
    float value;
    float vw;
    VoxelIndex V;
    const LaunchGeom *G;
    __device__ __forceinline__ void begin(const Branch &B, float w)
    {
        V.set(B, *G);
        vw = value * w;
    }
    __device__ __forceinline__ void slab(int ip, const Slab &c, float e)
    {
        const SlabTerms t = slab_terms(c, V.ns, V.nz);
        const float v = vw * e;
        if (t.v1) unsafeAtomicAdd(img + V.at(ip, c.cs1, c.cz1), v * c.r1);
        if (t.v2) unsafeAtomicAdd(img + V.at(ip, t.csm, t.czm), v * c.r2);
        if (t.v3) unsafeAtomicAdd(img + V.at(ip, c.cs2, c.cz2), v * c.r3);
    }
    __device__ __forceinline__ void nan_event() {}
};

struct DigestAct {
    uint64_t h;
    int cnt;
    VoxelIndex V;
    const LaunchGeom *G;
    __device__ __forceinline__ void begin(const Branch &B, float) { V.set(B, *G); }
    __device__ __forceinline__ void add(unsigned v, int br)
    {
        h += mix64(((uint64_t)v << 4) | (uint64_t)br);
        cnt += 1;
    }
    __device__ __forceinline__ void slab(int ip, const Slab &c, float)
    {
        const SlabTerms t = slab_terms(c, V.ns, V.nz);
        if (t.v1) add(V.at(ip, c.cs1, c.cz1), slab_label1(c));
        if (t.v2) add(V.at(ip, t.csm, t.czm), slab_label2(c));
        if (t.v3) add(V.at(ip, c.cs2, c.cz2), slab_label3(c));
    }
    __device__ __forceinline__ void nan_event() {}
};

__device__ __forceinline__ float event_ratio(const float *__restrict__ y, const float *__restrict__ p,
                                             int64_t e, int kind, float eps)
{
    const float yy = y[e];
    const float d = p[e] + eps;
    if (kind == SRF_RATIO_DIV_NO_NAN) return d == 0.0f ? 0.0f : yy / d;
    return yy / d;
}

// 2^lg lanes per event (lg <= 4), each on a run of its slabs: a short list then
// still fills the chip and its serial chain of dependent loads is shorter.  The
// lanes' sums are combined by a fixed butterfly.
template <bool TOF, int VAR, bool DS, bool DZ>
__global__ __launch_bounds__(256) void k_gather(const float *__restrict__ lors, int64_t n, int stride,
                                                const float *__restrict__ tofv, int tof_stride,
                                                const float *__restrict__ img, LaunchGeom G, int lg,
                                                float *__restrict__ out)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t e = t >> lg;
    const int parts = 1 << lg, part = (int)threadIdx.x & (parts - 1);
    const bool on = e < n;   // whole groups of lanes: the grid is rounded up to blocks of 256
    GatherAct act;
    act.img = img;
    act.sum = act.part = act.W = 0.0f;
    act.G = &G;
    if (on) march_event<TOF, VAR, DS, DZ>(lors + e * stride, TOF ? tofv[e * tof_stride] : 0.0f, G, part, parts, act);
    float s = act.sum + act.part;
    for (int k = parts >> 1; k > 0; k >>= 1) s += __shfl_xor(s, k);
    if (on && part == 0) out[e] = s;
}

// -------------------------------------------------------- bundled projector --
// A long list in arbitrary order: with one event per lane every term is a load
// of its own cache line that misses L2 (a 256 x 256 x 128 image is 32 MiB, an
// XCD's L2 4 MiB; 5e6 TOF events took 21.2 ms, 2e9 terms at one line each).
// Instead
//   - the events are sorted by the line they lie on: a bit-interleaved key of the
//     dominant axis, the secondary and axial position at the image centre and the
//     two slopes (k_line_keys, a radix sort of 24 key bits), so that a wavefront
//     holds a bundle of neighbouring lines;
//   - the image is copied once per dominant axis with the axial index fastest,
//     [primary][secondary][axial], inside a one-cell zero border along the last
//     two (k_border_image), and a wavefront steps through the planes of its
//     dominant axis together: its 64 lanes read a patch of one plane, a few
//     rows of a few lines each, from a scalar plane address.  Cells are clamped
//     into the border instead of being tested (they read zero there).
// Every XCD takes a contiguous run of bundles, whose lines its L2 keeps.

// The key of a line.
__device__ __forceinline__ unsigned line_key(const Branch &B, float z1, const LaunchGeom &G)
{
    auto cell = [](float v, float hi) { return (unsigned)fminf(fmaxf(v, 0.0f), hi); };
    const float is = 64.0f / (float)B.ns, iz = 32.0f / (float)G.nz;
    const float s = (B.sec1 - B.ks * B.p1) / B.ds + B.ns2, z = (z1 - B.kz * B.p1) / G.dz + G.nz2;
    const float t = B.ks * B.np2 / B.ds + B.ns2, w = B.kz * B.np2 / G.dz + G.nz2;
    const unsigned qs = cell(s * is, 63.0f), qt = cell(t * is, 63.0f), qz = cell(z * iz, 31.0f), qw = cell(w * iz, 31.0f);
    unsigned k = B.xdom ? 0u : 1u;
    auto put = [&](unsigned v, int bit) { k = (k << 1) | ((v >> bit) & 1u); };
    // positions and slopes of the secondary axis first: a line of 32 axial cells
    // is one 128-byte cache line, so a bundle may be wider along it
    put(qs, 5); put(qt, 5); put(qs, 4); put(qt, 4); put(qs, 3); put(qt, 3); put(qz, 4); put(qw, 4);
    put(qs, 2); put(qt, 2); put(qz, 3); put(qw, 3); put(qs, 1); put(qt, 1); put(qz, 2); put(qw, 2);
    put(qs, 0); put(qt, 0); put(qz, 1); put(qw, 1); put(qz, 0); put(qw, 0);
    return k;
}
constexpr int LINE_KEY_BITS = 24;

// Key and index of every event; events without terms (and non-finite ones) last.
template <bool TOF>
__global__ __launch_bounds__(256) void k_line_keys(const float *__restrict__ lors, int64_t n, int stride, LaunchGeom G,
                                                   unsigned *__restrict__ key, int *__restrict__ idx)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    RaySetup r;
    ray_setup<false>(lors + e * stride, 0.0f, G, r);
    unsigned k = (1u << LINE_KEY_BITS) - 1u;
    if (r.live && (TOF || !r.q2)) {
        Branch B;
        make_branch(r, TOF ? r.xdom_gt : r.xdom_ge, G, B);
        k = line_key(B, r.z1, G);
    }
    key[e] = k;
    idx[e] = (int)e;
}

// The two bordered copies: zx[x][y + 1][z + 1] and zy[y][x + 1][z + 1], rows of
// pz = nz + 2.  One workgroup per 32 x 32 (x, z) tile of a y row of the border
// box, transposed through LDS.
__global__ __launch_bounds__(256) void k_border_image(const float *__restrict__ img, int nx, int ny, int nz,
                                                      float *__restrict__ zx, float *__restrict__ zy)
{
    __shared__ float tile[32][33];
    const int x0 = blockIdx.x * 32 - 1, z0 = blockIdx.y * 32 - 1, y = (int)blockIdx.z - 1;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int pz = nz + 2;
    const bool iny = y >= 0 && y < ny;
    for (int k = ty; k < 32; k += 8) {
        const int x = x0 + tx, z = z0 + k;
        tile[k][tx] = (iny && x >= 0 && x < nx && z >= 0 && z < nz) ? img[x + (int64_t)nx * (y + (int64_t)ny * z)] : 0.0f;
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
        const int x = x0 + k, z = z0 + tx;
        if (x > nx || z > nz) continue;
        const float v = tile[tx][k];
        if (x >= 0 && x < nx) zx[((int64_t)x * (ny + 2) + y + 1) * pz + z + 1] = v;
        if (iny) zy[((int64_t)y * (nx + 2) + x + 1) * pz + z + 1] = v;
    }
}

__device__ __forceinline__ int wave_min(int v)
{
    for (int k = 32; k > 0; k >>= 1) v = min(v, __shfl_xor(v, k));
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ int wave_max(int v)
{
    for (int k = 32; k > 0; k >>= 1) v = max(v, __shfl_xor(v, k));
    return __builtin_amdgcn_readfirstlane(v);
}

// Weighted sum over the slabs [a, b) of every lane's ray (a >= b: none), the wavefront in
// step through the planes of a bordered copy of pl floats per plane; of `parts`
// wavefronts with the same rays, number `part` takes its share of the planes.
template <bool TOF, bool DS, bool DZ>
__device__ __forceinline__ float bundle_sum(const Branch &B, float W, float z1, const LaunchGeom &G, int a, int b, float tA,
                                            float tB, const float *__restrict__ copy, int64_t pl, int pz, int part, int parts)
{
    const bool on = a < b;
    int ia = wave_min(on ? a : INT_MAX), ib = wave_max(on ? b : INT_MIN);
    const int share = (ib - ia + parts - 1) / parts;
    ia = __builtin_amdgcn_readfirstlane(ia + part * share);
    ib = min(ib, ia + share);
    if (ia >= ib) return 0.0f;
    const bool ks_pos = B.ks >= 0.0f, kz_pos = B.kz >= 0.0f;
    // border clamps, row pitch and origin held in vector registers (v_med3 and
    // v_mad read at most one scalar register)
    int lo = -1, ns = B.ns, nz = G.nz, row = 4 * pz, org = 4 * (pz + 1);
    asm volatile("" : "+v"(lo), "+v"(ns), "+v"(nz), "+v"(row), "+v"(org));
    const float *plane = copy + ia * pl;
    float pp1 = (float)ia - B.np2;
    float S0 = coord_s<DS>(B, pp1), Z0 = coord_z<DZ>(B, z1, G, pp1);
    float acc = 0.0f, sum = 0.0f;
    const unsigned len = on ? (unsigned)(b - a) : 0u;
    int ip = ia;
    auto slab = [&]() {
        const float pp2 = pp1 + 1.0f;
        const float S1 = coord_s<DS>(B, pp2), Z1 = coord_z<DZ>(B, z1, G, pp2);
        if ((unsigned)(ip - a) < len) {
            Slab c;
            slab_cells(c, S0, S1, Z0, Z1, ks_pos, kz_pos);
            const bool los = c.cs1 >= -1, loz = c.cz1 >= -1;
            // byte offsets in the plane; offset 0 is a border cell
            const int c1 = med3_i32(c.cs1, lo, ns), c2 = med3_i32(c.cs2, lo, ns);
            const int d1 = med3_i32(c.cz1, lo, nz), d2 = med3_i32(c.cz2, lo, nz);
            const int A = mad_i24(c1, row, org), C = mad_i24(c2, row, org);
            const int j2a = A + 4 * d2, j2b = C + 4 * d1, j3 = C + 4 * d2;
            unsigned i1 = (unsigned)(A + 4 * d1);
            unsigned i2a = (c.bs && c.bz && loz) ? (unsigned)j2a : 0u, i2b = (c.bs && c.bz && los) ? (unsigned)j2b : 0u;
            unsigned i3 = ((c.bs || c.bz) && los && loz) ? (unsigned)j3 : 0u;
            // here: sunk past the branch in slab_fractions, their lane masks would
            // be carried across it as 0/1 vectors
            asm volatile("" : "+v"(i1), "+v"(i2a), "+v"(i2b), "+v"(i3));
            slab_fractions(c);
            const unsigned i2 = c.sgt ? i2a : i2b;
            const char *p = reinterpret_cast<const char *>(plane);
            const float g1 = *reinterpret_cast<const float *>(p + i1);
            const float g2 = *reinterpret_cast<const float *>(p + i2);
            const float g3 = *reinterpret_cast<const float *>(p + i3);
            float e = 1.0f;
            if (TOF) {
                const float dd = fmaf(pp1, tA, tB);
                e = __builtin_amdgcn_exp2f(-(dd * dd));
            }
            const float s = fmaf(g1, c.r1, fmaf(g2, c.r2, g3 * c.r3));
            acc = fmaf(s, TOF ? e * W : W, acc);
        }
        if ((ip & (SUM_RUN - 1)) == SUM_RUN - 1) {   // a scalar test: the wavefront is in step
            sum += acc;
            acc = 0.0f;
        }
        pp1 = pp2;
        S0 = S1;
        Z0 = Z1;
        plane += pl;
        ++ip;
    };
    // twice per trip, so that the values carried from slab to slab alternate
    // registers instead of moving
    while (ip < ib) {
        slab();
        if (!(ip < ib)) break;
        slab();
    }
    return sum + acc;
}

template <bool TOF, bool DS, bool DZ>
__global__ __launch_bounds__(256) void k_bundle(const float *__restrict__ lors, int64_t n, int stride,
                                                const float *__restrict__ tofv, int tof_stride,
                                                const int *__restrict__ order, const float *__restrict__ zx,
                                                const float *__restrict__ zy, LaunchGeom G, int lgp, int nblk,
                                                float *__restrict__ out)
{
    __shared__ float part_sum[256];
    // workgroup i runs on XCD i % 8: a contiguous run of bundles per XCD
    const int per = gridDim.x >> 3;
    const int blk = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (blk >= nblk) return;
    // 2^lgp wavefronts of the workgroup share a bundle
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int parts = 1 << lgp, part = wave & (parts - 1);
    const int64_t i = (int64_t)blk * (256 >> lgp) + (wave >> lgp) * 64 + (threadIdx.x & 63);
    const bool in = i < n;
    const int64_t e = in ? order[i] : 0;
    RaySetup r;
    ray_setup<TOF>(lors + e * stride, TOF ? tofv[e * tof_stride] : 0.0f, G, r);
    Branch B;
    int a, b;
    event_slabs<TOF, V_FP>(r, G, B, a, b);
    if (!in || r.nan) a = b = 0;
    float tA, tB;
    tof_coeffs<TOF>(B, r, G, tA, tB);
    const float W = branch_weight<TOF>(B, r, G, true);
    const int pz = G.nz + 2;
    float s = 0.0f;
    // a wavefront holds one branch, but for the one where the sorted list changes over
    if (__any(a < b && B.xdom))
        s = bundle_sum<TOF, DS, DZ>(B, W, r.z1, G, a, B.xdom ? b : a, tA, tB, zx, (int64_t)(G.ny + 2) * pz, pz,
                                    part, parts);
    if (__any(a < b && !B.xdom)) {
        const float t = bundle_sum<TOF, DS, DZ>(B, W, r.z1, G, a, B.xdom ? a : b, tA, tB, zy, (int64_t)(G.nx + 2) * pz, pz,
                                                  part, parts);
        s = B.xdom ? s : t;
    }
    if (lgp > 0) {
        part_sum[threadIdx.x] = s;
        __syncthreads();
        if (part != 0) return;
        for (int k = 1; k < parts; ++k) s += part_sum[threadIdx.x + 64 * k];
    }
    if (in) out[e] = r.nan ? __builtin_nanf("") : (a < b ? s : 0.0f);
}

// values == nullptr: all ones.  y/p != nullptr: value = ratio(y, p).
template <bool TOF, int VAR, bool DS, bool DZ>
__global__ __launch_bounds__(256) void k_scatter(const float *__restrict__ lors, int64_t n, int stride,
                                                 const float *__restrict__ tofv, int tof_stride,
                                                 const float *__restrict__ values,
                                                 const float *__restrict__ y, const float *__restrict__ p,
                                                 int kind, float eps, LaunchGeom G, float *__restrict__ img)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    float v = 1.0f;
    if (y) v = event_ratio(y, p, e, kind, eps);
    else if (values) v = values[e];
    ScatterAct act;
    act.img = img;
    act.value = v;
    act.G = &G;
    march_event<TOF, VAR, DS, DZ>(lors + e * stride, TOF ? tofv[e * tof_stride] : 0.0f, G, 0, 1, act);
}

template <bool TOF, int VAR, bool DS, bool DZ>
__global__ __launch_bounds__(256) void k_digest(const float *__restrict__ lors, int64_t n, int stride,
                                                const float *__restrict__ tofv, int tof_stride, LaunchGeom G,
                                                uint64_t *__restrict__ hash, int32_t *__restrict__ count)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    DigestAct act;
    act.h = 0ull;
    act.cnt = 0;
    act.G = &G;
    march_event<TOF, VAR, DS, DZ>(lors + e * stride, TOF ? tofv[e * tof_stride] : 0.0f, G, 0, 1, act);
    hash[e] = act.h;
    count[e] = act.cnt;
}

// --------------------------------------------------- point line integrals --
// Integral of an image from every detector to every scatter point: the projector
// along the LOR detector -> point, without the 1 / L^2 of its weight, so without
// an LOR array, its lengths and a product with them (4 of 48 ms of an estimate of
// 4096 detectors x 2e4 points) and without a sort: a wavefront takes 64 points in
// a row of one detector, a bundle by itself (its points lie on a few columns of the
// grid).  BORDER: over the axial-fastest copies of k_border_image, in step through
// their planes; else one ray per lane on the image as it is.
template <bool BORDER, bool DS, bool DZ>
__global__ __launch_bounds__(256) void k_point_integrals(const float *__restrict__ det, int nd,
                                                         const float *__restrict__ pts, int ns, int pstride,
                                                         const float *__restrict__ img, const float *__restrict__ zx,
                                                         const float *__restrict__ zy, LaunchGeom G, int64_t nblk,
                                                         float *__restrict__ out)
{
    const int64_t per = (int64_t)gridDim.x >> 3;   // a contiguous run of detectors per XCD
    const int64_t blk = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (blk >= nblk) return;
    const int nsb = (ns + 255) / 256;
    const int d = __builtin_amdgcn_readfirstlane((int)(blk / nsb));
    const int s = (int)(blk % nsb) * 256 + (int)threadIdx.x;
    const bool in = s < ns;
    const float *P = pts + (int64_t)(in ? s : 0) * pstride;
    const float lor[6] = {det[4 * d], det[4 * d + 1], det[4 * d + 2], P[0], P[1], P[2]};
    RaySetup r;
    ray_setup<false>(lor, 0.0f, G, r);
    Branch B;
    int a, b;
    event_slabs<false, V_FP>(r, G, B, a, b);
    if (!in || r.nan) a = b = 0;
    const float W = B.sq * G.dx_;
    float sum = 0.0f;
    if (BORDER) {
        const int pz = G.nz + 2;
        if (__any(a < b && B.xdom))
            sum = bundle_sum<false, DS, DZ>(B, W, r.z1, G, a, B.xdom ? b : a, 0.0f, 0.0f, zx, (int64_t)(G.ny + 2) * pz, pz, 0, 1);
        if (__any(a < b && !B.xdom)) {
            const float t = bundle_sum<false, DS, DZ>(B, W, r.z1, G, a, B.xdom ? a : b, 0.0f, 0.0f, zy,
                                                      (int64_t)(G.nx + 2) * pz, pz, 0, 1);
            sum = B.xdom ? sum : t;
        }
    } else if (a < b) {
        GatherAct act;
        act.img = img;
        act.sum = act.part = 0.0f;
        act.G = &G;
        act.begin(B, W);
        march_slabs<false, DS, DZ>(B, r.z1, G, a, b, 0.0f, 0.0f, act);
        sum = act.sum + act.part;
    }
    if (in) out[(int64_t)d * ns + s] = r.nan ? __builtin_nanf("") : (a < b ? sum : 0.0f);
}

// ----------------------------------------------------------------- host side --

int make_geom(const srf_grid_t &g, const srf_tof_t *tof, LaunchGeom &G)
{
    if (g.nx <= 0 || g.ny <= 0 || g.nz <= 0) return SRF_ERR_INVALID_ARG;
    if ((int64_t)g.nx * g.ny * g.nz >= ((int64_t)1 << 31)) return SRF_ERR_UNSUPPORTED;
    if (!(g.sx > 0.0f && g.sy > 0.0f && g.sz > 0.0f)) return SRF_ERR_INVALID_ARG;
    if (!(isfinite(g.cx) && isfinite(g.cy) && isfinite(g.cz))) return SRF_ERR_INVALID_ARG;
    G.nx = g.nx; G.ny = g.ny; G.nz = g.nz;
    G.cx = g.cx; G.cy = g.cy; G.cz = g.cz;
    // siddon.cu.cc:19-22, 39-41 -- same float expressions, host IEEE
    G.dx_ = g.sx / (float)g.nx;
    G.dy = g.sy / (float)g.ny / G.dx_;
    G.dz = g.sz / (float)g.nz / G.dx_;
    G.nx2 = g.nx / 2.0f;
    G.ny2 = g.ny / 2.0f;
    G.nz2 = g.nz / 2.0f;
    G.tof_bin_ = G.tof_sigma2_ = G.tse = G.tof_c0 = G.tof_c1 = 0.0f;
    if (tof) {
        if (!(tof->tof_sigma2 > 0.0f) || !(tof->tof_bin >= 0.0f)) return SRF_ERR_INVALID_ARG;
        // siddon_tof.cu.cc:46-47, 57, 59
        G.tof_bin_ = tof->tof_bin / G.dx_;
        G.tof_sigma2_ = tof->tof_sigma2 / G.dx_ / G.dx_;
        G.tse = G.tof_sigma2_ + (G.tof_bin_ * G.tof_bin_) / 12;
        const float PI_REF = 3.1415926f;  // siddon_tof.cu.cc:10
        G.tof_c0 = (float)((double)G.tof_bin_ / sqrt(2.0 * (double)PI_REF * (double)G.tse));
        G.tof_c1 = (float)(-0.5 * 1.4426950408889634 / (double)G.tse);
    }
    return SRF_OK;
}

static int check_events(const float *lors, int64_t n, int64_t stride, const float *tofv, int64_t tof_stride,
                        const srf_tof_t *tof)
{
    if (n < 0) return SRF_ERR_INVALID_ARG;
    if (n == 0) return SRF_OK;
    if (!lors || stride < 6 || stride > (1 << 20)) return SRF_ERR_INVALID_ARG;
    if (tof && (!tofv || tof_stride < 1 || tof_stride > (1 << 20))) return SRF_ERR_INVALID_ARG;
    if (n > ((int64_t)1 << 40)) return SRF_ERR_UNSUPPORTED;
    return SRF_OK;
}

#define SRF_DISPATCH(KERNEL, TOFV, VARV, DSV, DZV, ...)                                                     \
    do {                                                                                                   \
        if (TOFV) {                                                                                        \
            if (VARV == V_FP) {                                                                            \
                if (DSV) { if (DZV) KERNEL<true, V_FP, true, true> __VA_ARGS__; else KERNEL<true, V_FP, true, false> __VA_ARGS__; } \
                else { if (DZV) KERNEL<true, V_FP, false, true> __VA_ARGS__; else KERNEL<true, V_FP, false, false> __VA_ARGS__; } \
            } else {                                                                                       \
                if (DSV) { if (DZV) KERNEL<true, V_BP, true, true> __VA_ARGS__; else KERNEL<true, V_BP, true, false> __VA_ARGS__; } \
                else { if (DZV) KERNEL<true, V_BP, false, true> __VA_ARGS__; else KERNEL<true, V_BP, false, false> __VA_ARGS__; } \
            }                                                                                              \
        } else {                                                                                           \
            if (VARV == V_FP) {                                                                            \
                if (DSV) { if (DZV) KERNEL<false, V_FP, true, true> __VA_ARGS__; else KERNEL<false, V_FP, true, false> __VA_ARGS__; } \
                else { if (DZV) KERNEL<false, V_FP, false, true> __VA_ARGS__; else KERNEL<false, V_FP, false, false> __VA_ARGS__; } \
            } else {                                                                                       \
                if (DSV) { if (DZV) KERNEL<false, V_BP, true, true> __VA_ARGS__; else KERNEL<false, V_BP, true, false> __VA_ARGS__; } \
                else { if (DZV) KERNEL<false, V_BP, false, true> __VA_ARGS__; else KERNEL<false, V_BP, false, false> __VA_ARGS__; } \
            }                                                                                              \
        }                                                                                                  \
    } while (0)

static inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

// Lists of at least BUNDLE_SLABS slabs (events times the longer transaxial side of
// the image; three times that where the image fits an XCD's 4 MiB L2) are bundled,
// BUNDLE_CHUNK events at a time (the scratch of a chunk is about 20 bytes per event
// plus the two copies).  Images that fit L2 several times over never are.  Measured,
// us, bundled / one event per lane:
//   256 x 256 x 128   65536 events 148 / 126, 98304 188 / 230, 2^18 317 / 548, 2^20 780 / 2838
//   181 x 217 x 91    65536 109 / 97, 98304 141 / 167, 2^18 245 / 346, 2^20 630 / 1567
//   128 x 128 x 64    2^17 110 / 90, 2^18 183 / 174, 2^19 272 / 340, 2^20 442 / 672;
//                     random pairs of ends, many of which miss the image: 4e5 235 / 144,
//                     9e5 328 / 246, 1.4e6 345 / 367
//   48 x 48 x 24      2^20 275 / 189
// 5e6 TOF events on 256 x 256 x 128: 2.49 ms against 21.3 ms (each term a line of its
// own from beyond L2).  Now VALU bound: about 75 instructions per slab.
constexpr int64_t BUNDLE_SLABS = 20000000;
constexpr int64_t BUNDLE_IMAGE_MIN = 1 << 20;
constexpr int64_t BUNDLE_IMAGE_L2 = 4 << 20;
constexpr int64_t BUNDLE_CHUNK = 1 << 23;
constexpr int64_t BUNDLE_SPLIT = 1 << 17;
constexpr int64_t BUNDLE_IMAGE_BYTES = 1 << 30;   // of both copies

// The bordered copies: floats of one (np planes), whether they and their 24-bit
// cell addresses fit (and the grid of k_border_image), and the copying.
static int64_t border_floats(int np, int ns, int nz) { return (int64_t)np * (ns + 2) * ((int64_t)nz + 2); }

static bool border_fits(const LaunchGeom &G)
{
    return 4 * (border_floats(G.nx, G.ny, G.nz) + border_floats(G.ny, G.nx, G.nz)) <= BUNDLE_IMAGE_BYTES &&
           4 * ((int64_t)G.nz + 2) < (1 << 23) && G.nx < (1 << 22) && G.ny <= 65533 && (G.nz + 33) / 32 <= 65535;
}

static int border_image(const float *image, const LaunchGeom &G, float *zx, float *zy, hipStream_t s)
{
    hipLaunchKernelGGL(k_border_image, dim3((unsigned)((G.nx + 33) / 32), (unsigned)((G.nz + 33) / 32), (unsigned)(G.ny + 2)),
                       dim3(256), 0, s, image, G.nx, G.ny, G.nz, zx, zy);
    return launch_status();
}

// The bundled projection; false where it does not apply (nothing is queued then).
static bool project_bundled(const float *lors, int64_t n, int stride, const float *tofv, int tof_stride,
                            const float *image, const LaunchGeom &G, bool tof, bool ds, bool dz, float *out,
                            hipStream_t s, int &rc)
{
    const int64_t bytes = (int64_t)G.nx * G.ny * G.nz * 4, slabs = n * (G.nx > G.ny ? G.nx : G.ny);
    if (bytes < BUNDLE_IMAGE_MIN || slabs < (bytes > BUNDLE_IMAGE_L2 + (BUNDLE_IMAGE_L2 >> 2) ? 1 : 3) * BUNDLE_SLABS) return false;
    if (!border_fits(G) || capturing(s)) return false;
    const int64_t chunk = n < BUNDLE_CHUNK ? n : BUNDLE_CHUNK;
    size_t sort_bytes = 0;
    unsigned *k0 = nullptr, *k1 = nullptr;
    int *i0 = nullptr, *i1 = nullptr;
    if (hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, k0, k1, i0, i1, (int)chunk, 0, LINE_KEY_BITS, s) !=
        hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t b_list = up((size_t)chunk * 4), b_x = up((size_t)border_floats(G.nx, G.ny, G.nz) * 4),
                 b_y = up((size_t)border_floats(G.ny, G.nx, G.nz) * 4);
    char *w = static_cast<char *>(pool_get(4 * b_list + b_x + b_y + sort_bytes, s));
    if (!w) return false;
    k0 = reinterpret_cast<unsigned *>(w);
    k1 = reinterpret_cast<unsigned *>(w + b_list);
    i0 = reinterpret_cast<int *>(w + 2 * b_list);
    i1 = reinterpret_cast<int *>(w + 3 * b_list);
    float *zx = reinterpret_cast<float *>(w + 4 * b_list), *zy = reinterpret_cast<float *>(w + 4 * b_list + b_x);
    void *tmp = w + 4 * b_list + b_x + b_y;
    rc = border_image(image, G, zx, zy, s);
    for (int64_t c = 0; c < n && rc == SRF_OK; c += chunk) {
        const int64_t m = n - c < chunk ? n - c : chunk;
        const float *L = lors + c * stride, *T = tof ? tofv + c * tof_stride : nullptr;
        if (tof)
            hipLaunchKernelGGL(k_line_keys<true>, dim3(blocks_for(m)), dim3(256), 0, s, L, m, stride, G, k0, i0);
        else
            hipLaunchKernelGGL(k_line_keys<false>, dim3(blocks_for(m)), dim3(256), 0, s, L, m, stride, G, k0, i0);
        if (hipcub::DeviceRadixSort::SortPairs(tmp, sort_bytes, k0, k1, i0, i1, (int)m, 0, LINE_KEY_BITS, s) != hipSuccess) {
            (void)hipGetLastError();
            rc = SRF_ERR_LAUNCH;
            break;
        }
        // up to four wavefronts per bundle while there are few bundles (2^16 events on
        // 256 x 256 x 128: 148 us with four, 267 with one; 2^18: 345, 317)
        const int lgp = m <= BUNDLE_SPLIT ? 2 : m <= 2 * BUNDLE_SPLIT ? 1 : 0;
        const int nb = (int)blocks_for(m << lgp);
        const dim3 grid((unsigned)((nb + 7) / 8 * 8));
#define SRF_BUNDLE(T_, S_, Z_) \
    hipLaunchKernelGGL((k_bundle<T_, S_, Z_>), grid, dim3(256), 0, s, L, m, stride, T, tof_stride, i1, zx, zy, G, lgp, nb,  \
                       out + c)
        if (tof) {
            if (ds) { if (dz) SRF_BUNDLE(true, true, true); else SRF_BUNDLE(true, true, false); }
            else { if (dz) SRF_BUNDLE(true, false, true); else SRF_BUNDLE(true, false, false); }
        } else {
            if (ds) { if (dz) SRF_BUNDLE(false, true, true); else SRF_BUNDLE(false, true, false); }
            else { if (dz) SRF_BUNDLE(false, false, true); else SRF_BUNDLE(false, false, false); }
        }
#undef SRF_BUNDLE
        rc = launch_status();
    }
    pool_put(w, s, false, true);
    return true;
}

// Lanes per event of k_gather (log2): enough for about 2^17 lanes, at most 16.
static int gather_lanes(int64_t n)
{
    int lg = 0;
    while (lg < 4 && (n << (lg + 1)) <= (1 << 17)) ++lg;
    return lg;
}

}  // namespace srf

using namespace srf;

extern "C" {

int srf_project(const float *lors, int64_t n, int64_t lor_stride, const float *tof_values, int64_t tof_stride,
                const float *image, srf_grid_t grid, const srf_tof_t *tof, float *out, void *stream)
{
    int rc = check_events(lors, n, lor_stride, tof_values, tof_stride, tof);
    if (rc) return rc;
    if (n > 0 && (!out || !image)) return SRF_ERR_INVALID_ARG;
    LaunchGeom G;
    if ((rc = make_geom(grid, tof, G))) return rc;
    if (n == 0) return SRF_OK;
    hipStream_t s = (hipStream_t)stream;
    const bool ds = G.dy != 1.0f, dz = G.dz != 1.0f;
    if (project_bundled(lors, n, (int)lor_stride, tof_values, (int)tof_stride, image, G, tof != nullptr, ds, dz, out, s,
                        rc))
        return rc;
    const int lg = gather_lanes(n);
    SRF_DISPATCH(k_gather, tof != nullptr, V_FP, ds, dz,
                 <<<blocks_for(n << lg), 256, 0, s>>>(lors, n, (int)lor_stride, tof_values, (int)tof_stride, image, G,
                                                      lg, out));
    return launch_status();
}

int srf_sss_integrals(const float *det, int32_t n_det, const float *points, int32_t n_points, int32_t point_stride,
                      const float *image, srf_grid_t grid, float *out, void *stream)
{
    if (n_det <= 0 || n_points <= 0 || point_stride < 3) return SRF_ERR_INVALID_ARG;
    if (!det || !points || !image || !out) return SRF_ERR_INVALID_ARG;
    LaunchGeom G;
    int rc = make_geom(grid, nullptr, G);
    if (rc) return rc;
    const int64_t nblk = (int64_t)n_det * ((n_points + 255) / 256);
    if (nblk >= ((int64_t)1 << 31) - 8) return SRF_ERR_UNSUPPORTED;
    hipStream_t s = (hipStream_t)stream;
    const bool ds = G.dy != 1.0f, dz = G.dz != 1.0f;
    const dim3 blocks((unsigned)((nblk + 7) / 8 * 8));
    float *zx = nullptr, *zy = nullptr;
    // the copies pay for themselves from a few thousand rays on
    if (nblk >= 64 && border_fits(G) && !capturing(s)) {
        const size_t nx = (size_t)border_floats(G.nx, G.ny, G.nz), ny = (size_t)border_floats(G.ny, G.nx, G.nz);
        zx = static_cast<float *>(pool_get((nx + ny) * sizeof(float), s));
        if (zx) {
            zy = zx + nx;
            if ((rc = border_image(image, G, zx, zy, s))) {
                pool_put(zx, s, false, true);
                return rc;
            }
        }
    }
#define SRF_POINTS(B_, S_, Z_)                                                                                        \
    hipLaunchKernelGGL((k_point_integrals<B_, S_, Z_>), blocks, dim3(256), 0, s, det, n_det, points, n_points,       \
                       point_stride, image, zx, zy, G, nblk, out)
    if (zx) {
        if (ds) { if (dz) SRF_POINTS(true, true, true); else SRF_POINTS(true, true, false); }
        else { if (dz) SRF_POINTS(true, false, true); else SRF_POINTS(true, false, false); }
    } else {
        if (ds) { if (dz) SRF_POINTS(false, true, true); else SRF_POINTS(false, true, false); }
        else { if (dz) SRF_POINTS(false, false, true); else SRF_POINTS(false, false, false); }
    }
#undef SRF_POINTS
    rc = launch_status();
    pool_put(zx, s, false, true);
    return rc;
}

// One event per lane; zero > 0: the image's voxels are cleared first.
static int scatter_events(const float *lors, int64_t n, int64_t lor_stride, const float *tof_values, int64_t tof_stride,
                          const float *values, const float *y, const float *p, int kind, float eps,
                          const LaunchGeom &G, bool tof, srf_bp_mode_t mode, int64_t zero, float *image, hipStream_t s)
{
    int rc;
    if (zero > 0 && (rc = fill_f32(image, 0.0f, zero, s))) return rc;
    if (n == 0) return SRF_OK;
    const int var = mode == SRF_BP_ADJOINT ? V_FP : V_BP;
    const bool ds = G.dy != 1.0f, dz = G.dz != 1.0f;
    SRF_DISPATCH(k_scatter, tof, var, ds, dz,
                 <<<blocks_for(n), 256, 0, s>>>(lors, n, (int)lor_stride, tof_values, (int)tof_stride, values, y,
                                                p, kind, eps, G, image));
    return launch_status();
}

// Lists of at least BINNED_SLABS slabs (events times the longer transaxial side) and
// BINNED_TILE_SLABS for every 32 x 32 x 8 tile of the image are binned: binning has a
// fixed cost of about 0.2 ms and 0.45 us per tile, the atomics 0.075 ns per slab
// (2e10 device-scope float atomics a second, each a line beyond L2).  Measured, us,
// binned / one event per lane with atomics:
//   256 x 256 x 128   32768 events 732 / 641, 65536 737 / 1244, 2^20 2560 / 19600
//   181 x 217 x 91    16384 417 / 281, 32768 442 / 525, 2^20 1980 / 15200
//   128 x 128 x 64    16384 238 / 197, 32768 295 / 358, 2^20 1300 / 10100
//   48 x 48 x 24      65536 368 / 301, 2^17 421 / 541, 2^20 742 / 3730
// A part of BINNED_CHUNK events takes about 3.5 GB of scratch on 256 x 256 x 128 (4 times as
// many: 3% faster at 5e6 events); grids whose events have more segments take smaller parts
// (ONCE_SEGMENTS, srf_tiled.hip), at most about 4 GB.
constexpr int64_t BINNED_SLABS = 3500000;
constexpr int64_t BINNED_TILE_SLABS = 6000;
constexpr int64_t BINNED_CHUNK = 1 << 21;
static bool binned_pays(int64_t n, const LaunchGeom &G)
{
    const int64_t tiles = (int64_t)((G.nx + 31) / 32) * ((G.ny + 31) / 32) * ((G.nz + 7) / 8);
    return n * (G.nx > G.ny ? G.nx : G.ny) >= BINNED_SLABS + BINNED_TILE_SLABS * tiles;
}

static int backproject_impl(const float *lors, int64_t n, int64_t lor_stride, const float *tof_values,
                            int64_t tof_stride, const float *values, const float *y, const float *p, int kind,
                            float eps, srf_grid_t grid, const srf_tof_t *tof, srf_bp_mode_t mode, int accumulate,
                            float *image, void *stream)
{
    int rc = check_events(lors, n, lor_stride, tof_values, tof_stride, tof);
    if (rc) return rc;
    if (!image) return SRF_ERR_INVALID_ARG;
    if (mode != SRF_BP_REFERENCE && mode != SRF_BP_ADJOINT) return SRF_ERR_INVALID_ARG;
    LaunchGeom G;
    if ((rc = make_geom(grid, tof, G))) return rc;
    hipStream_t s = (hipStream_t)stream;
    const int64_t nvox = (int64_t)grid.nx * grid.ny * grid.nz;
    // a long list is binned into image tiles, in parts of equal size; a part that
    // cannot be (no memory, a grid beyond the plans') is scattered
    if (binned_pays(n, G) && !capturing(s)) {
        const int64_t parts = (n + BINNED_CHUNK - 1) / BINNED_CHUNK;
        int64_t chunk = (n + parts - 1) / parts;
        for (int64_t c = 0; c < n;) {
            const int64_t m = n - c < chunk ? n - c : chunk;
            const float *L = lors + c * lor_stride, *T = tof ? tof_values + c * tof_stride : nullptr;
            const float *V = values ? values + c : nullptr, *Y = y ? y + c : nullptr, *Q = p ? p + c : nullptr;
            int64_t fit = m;
            rc = backproject_binned(L, m, lor_stride, T, tof_stride, V, Y, Q, kind, eps, grid, tof, mode,
                                    accumulate || c > 0, image, s, fit);
            if (rc == SRF_ERR_WORKSPACE && fit < m) {   // too many segments for the scratch of a part
                chunk = fit;
                continue;
            }
            if (rc) rc = scatter_events(L, m, lor_stride, T, tof_stride, V, Y, Q, kind, eps, G, tof != nullptr, mode,
                                        accumulate || c > 0 ? 0 : nvox, image, s);
            if (rc) return rc;
            c += m;
        }
        return SRF_OK;
    }
    return scatter_events(lors, n, lor_stride, tof_values, tof_stride, values, y, p, kind, eps, G, tof != nullptr, mode,
                          accumulate ? 0 : nvox, image, s);
}

int srf_backproject(const float *lors, int64_t n, int64_t lor_stride, const float *tof_values, int64_t tof_stride,
                    const float *values, srf_grid_t grid, const srf_tof_t *tof, srf_bp_mode_t mode, int accumulate,
                    float *image, void *stream)
{
    return backproject_impl(lors, n, lor_stride, tof_values, tof_stride, values, nullptr, nullptr, 0, 0.0f, grid,
                            tof, mode, accumulate, image, stream);
}

int srf_backproject_ratio(const float *lors, int64_t n, int64_t lor_stride, const float *tof_values,
                          int64_t tof_stride, const float *y, const float *p, srf_ratio_kind_t kind, float eps,
                          srf_grid_t grid, const srf_tof_t *tof, srf_bp_mode_t mode, int accumulate, float *image,
                          void *stream)
{
    if (n > 0 && (!y || !p)) return SRF_ERR_INVALID_ARG;
    if (kind != SRF_RATIO_PLAIN && kind != SRF_RATIO_DIV_NO_NAN) return SRF_ERR_INVALID_ARG;
    return backproject_impl(lors, n, lor_stride, tof_values, tof_stride, nullptr, y, p, (int)kind, eps, grid, tof,
                            mode, accumulate, image, stream);
}

int srf_lor_digest(const float *lors, int64_t n, int64_t lor_stride, const float *tof_values, int64_t tof_stride,
                   srf_grid_t grid, const srf_tof_t *tof, srf_bp_mode_t mode, uint64_t *hash, int32_t *count,
                   void *stream)
{
    int rc = check_events(lors, n, lor_stride, tof_values, tof_stride, tof);
    if (rc) return rc;
    if (n > 0 && (!hash || !count)) return SRF_ERR_INVALID_ARG;
    if (mode != SRF_BP_REFERENCE && mode != SRF_BP_ADJOINT) return SRF_ERR_INVALID_ARG;
    LaunchGeom G;
    if ((rc = make_geom(grid, tof, G))) return rc;
    if (n == 0) return SRF_OK;
    hipStream_t s = (hipStream_t)stream;
    const int var = mode == SRF_BP_ADJOINT ? V_FP : V_BP;
    const bool ds = G.dy != 1.0f, dz = G.dz != 1.0f;
    SRF_DISPATCH(k_digest, tof != nullptr, var, ds, dz,
                 <<<blocks_for(n), 256, 0, s>>>(lors, n, (int)lor_stride, tof_values, (int)tof_stride, G, hash,
                                                count));
    return launch_status();
}

}  // extern "C"
