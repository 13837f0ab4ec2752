// srf_cnn.hip -- BF16 MFMA kernels of the scatter surrogate CNN (training and
// inference), and their C-ABI entry points (include/srf_hip.h, srf_cnn_*).
//
// Tensors are channels-last: act[v][c], v = (z*H + y)*W + x, with the channel
// count padded to a multiple of 8 (one MFMA k-step covers 8 channels) and
// BF16 storage; weights are [tap][cout][cin] (cin fastest, padded like the
// activations) in BF16 with FP32 master copies kept by the optimiser.
//
// Convolutions (3x3x3 or 1x1x1, stride 1, zero padding) are implicit GEMMs on
// v_mfma_f32_16x16x32_bf16 (FP32 accumulation) from tiles staged in LDS.
//   k_conv, k_conv_rows, k_conv_res  forward (bias + optional leaky ReLU epilogue), and the
//                 input gradient as a forward pass of flipped, transposed weights
//   k_conv_wgrad_tr  weight gradient: per tap, dW[co][ci] += sum_v dY[v][co] X[v+o][ci]
//                 (split over runs of tiles, partial sums added by k_wgrad_sum);
//                 k_conv_wgrad the same for rows that are not 16-byte aligned
// plus the elementwise kernels of the network (pooling, upsampling, channel
// copies, activation backward, bias gradient, MSE, Adam, casts).
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <math.h>
#include <stdint.h>

#include "srf_hip.h"
#include "srf_internal.hpp"

namespace srf {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

// float -> bf16 bits, round to nearest even (gfx950's v_cvt_pk_bf16_f32)
__device__ __forceinline__ unsigned short f2bf(float f) { return __builtin_bit_cast(unsigned short, (__bf16)f); }

struct ConvDims {
    int D, H, W;      // spatial size (same in and out)
    int cin_p;        // padded input channels (multiple of 8), also the input row stride
    int cout;         // real output channels
    int cout_p;       // output channels padded to a multiple of 32 (weight rows)
    int out_stride;   // output row stride (channels)
    int out_off;      // first output channel
    int taps;         // 27 or 1
    float slope;      // leaky ReLU slope; < 0: no activation
};

__device__ __forceinline__ void tap_offset(int t, int taps, int &dz, int &dy, int &dx)
{
    if (taps == 1) { dz = dy = dx = 0; return; }
    dz = t / 9 - 1;
    dy = (t / 3) % 3 - 1;
    dx = t % 3 - 1;
}

// Convolution as an implicit GEMM on gfx950's v_mfma_f32_16x16x32_bf16 (A: 16 output
// channels x 32 K values, B: 32 K values x 16 voxels, FP32 accumulation).  K runs over
// (tap, group of 8 input channels).
//
// A workgroup owns a tile of voxels and NBW blocks of 16 output channels.  Per chunk of 8,
// 16 or 32 input channels the tile's input halo is staged in LDS with coalesced 16-byte
// loads: zero outside the volume and outside the tile's own sample (a batch stacks samples
// along z, Ds slices each; a tile never straddles two), so taps never read a neighbouring
// sample.  A lane then reads its 8 K values of a voxel as one 16-byte LDS access; in
// k_conv a halo voxel's channel groups are padded to an odd count of 16-byte words so that
// eight voxels of a row start in different banks.  Weights (a few KiB to 440 KiB per layer)
// are read from global memory through the caches, some steps ahead (k_conv_res: once).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

struct ConvTile {
    int ntx, nty, ntz;   // tiles of a sample
    int Ds;              // slices per sample
    int nblk;            // tiles of the launch
};

// The input of a convolution: channels [0, cc) are the nearest-neighbour 2x
// upsampling of `coarse` (rows of cc channels on the half-size grid) and
// channels [cc, cin_p) come from `fine` (rows of cin_p - cc channels): the
// decoder's concatenation read in place.  cc = 0: every channel from fine.
struct ConvIn {
    const unsigned short *fine;
    const unsigned short *coarse;
    int cc;
};

// A 1x1 convolution to one channel applied to a layer's output in its
// epilogue: out[v] = b + sum_c bf16(y[v][c]) w[c] (the bf16 values the layer
// stores), so that the network's last layer needs no pass of its own.
struct ConvHead {
    const unsigned short *w;   // cout bf16 weights
    const float *b;            // the bias (one value)
    float *out;                // one value per voxel
};

constexpr int CX = 8;         // k_conv's tile along x and y
constexpr int64_t CONV_WANTED = 512;   // workgroups of a launch, where the volume has them

// Halo voxels of k_conv's tile of cz slices.
constexpr int halo_voxels(int R, int cz) { return (CX + 2 * R) * (CX + 2 * R) * (cz + 2 * R); }

// k_conv_rows' tile and its halo.
constexpr int RWX = 16, RWY = 8, RWZ = 4;
constexpr int RHX = RWX + 2, RHY = RWY + 2, RHV = RHX * RHY * (RWZ + 2);
constexpr int64_t ROWS_WANTED = 256;   // workgroups that pay for the larger tile

// Where channel group g of a voxel in halo column x lies among its groups.
template <int NG>
__device__ __forceinline__ int row_slot(int g, int x) { return NG == 4 ? g ^ ((x >> 2) & 3) : g; }

// The offset of tap t in a halo of rows of ex and planes of exy voxels.
template <int TAPS>
__device__ __forceinline__ int tap_delta(int t, int ex, int exy)
{
    if (TAPS == 1) return 0;
    return (t / 9) * exy + ((t / 3) % 3) * ex + t % 3;
}

// One chunk's products for RB blocks of 16 voxels: two rows of 8 (TX = 8) or a row of 16.
// v0: this lane's voxel of block 0 in the halo, x0 its column there; w: the weights of the
// chunk's first channel and output, read PF steps ahead.  The sums run over the taps in
// order, the channels of a chunk together: every kernel keeps this order, so that a
// layer's bf16 outputs do not depend on which one computes them.
template <int TAPS, int NG, int NBW, int RB, int TX>
__device__ __forceinline__ void conv_chunk(const u16x8 *halo, int v0, int x0, const unsigned short *__restrict__ w,
                                           int64_t tap_stride, int cin_p, int col, int q, f32x4 (&acc)[RB][NBW])
{
    constexpr int G = TAPS * NG;          // K groups of 8 in this chunk
    constexpr int S = (G + 3) / 4;        // MFMA steps (4 groups each)
    constexpr int K = 4 / NG;             // taps per step
    constexpr int R2 = TAPS == 27 ? 2 : 0, EX = TX + R2, EXY = EX * (8 + R2);
    constexpr int GP = TX == 8 ? NG | 1 : NG, STEP = TX == 8 ? 2 * EX : EX;   // words of a voxel; voxels between blocks
    constexpr int PF = RB * NBW >= 8 ? 2 : RB * NBW >= 4 ? 3 : RB * NBW >= 2 ? 5 : 10;   // steps ahead: weights,
    constexpr int AH = RB == 1 ? 4 : RB == 2 ? 2 : RB * NBW == 4 ? 1 : 0;               // and voxels
    // lane l's K group q is (tap K s + q / NG, channel group q % NG)
    int g = q & (NG - 1), tq = q / NG;
    asm volatile("" : "+v"(g), "+v"(tq));   // what depends on them is not kept across the chunks
    const unsigned mine = (unsigned)(col * cin_p + 8 * g) + (unsigned)tq * (unsigned)tap_stride;
    u16x8 wr[PF + 1][NBW];
    // in order of s: the place advances by a step's taps and is kept from the optimiser,
    // which would hold every step's address in registers across the chunks (the place and
    // not the pointer: that would lose its address space and be read by flat loads)
    int64_t at = 0;
    auto fetch = [&](int s, u16x8 (&to)[NBW]) {
        const bool valid = 4 * s + 3 < G || 4 * s + q < G;
#pragma unroll
        for (int j = 0; j < NBW; ++j) {
            to[j] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (valid) to[j] = *reinterpret_cast<const u16x8 *>(w + at + 16 * j * cin_p + mine);
        }
        at += K * tap_stride;
        asm volatile("" : "+s"(at));
    };
#pragma unroll
    for (int s = 0; s < PF; ++s)
        if (s < S) fetch(s, wr[s]);
    __syncthreads();   // the halo is there
    u16x8 a[AH + 1][RB];
    auto read = [&](int s, u16x8 (&to)[RB]) {
        // the taps of this step: uniform candidates, one picked per lane
        const int t = K * s;
        int delta = tap_delta<TAPS>(t, EX, EXY), dx = t % 3;
#pragma unroll
        for (int k = 1; k < K; ++k) {
            const int tk = t + k < TAPS ? t + k : TAPS - 1;
            delta = tq == k ? tap_delta<TAPS>(tk, EX, EXY) : delta;
            dx = tq == k ? tk % 3 : dx;
        }
        const u16x8 *p = halo + (v0 + delta) * GP + (TX == 8 ? g : row_slot<NG>(g, x0 + (TAPS == 27 ? dx : 0)));
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            to[r] = p[r * STEP * GP];
            // zeros on both sides past the last tap
            if (4 * s + 3 >= G && 4 * s + q >= G) to[r] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
        }
    };
#pragma unroll
    for (int s = 0; s < AH; ++s)
        if (s < S) read(s, a[s]);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (s + PF < S) fetch(s + PF, wr[(s + PF) % (PF + 1)]);
        if (s + AH < S) read(s + AH, a[(s + AH) % (AH + 1)]);
        if (AH > 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int j = 0; j < NBW; ++j)
                acc[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wr[s % (PF + 1)][j]),
                                                                    __builtin_bit_cast(bf16x8, a[s % (AH + 1)][r]),
                                                                    acc[r][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);   // a few steps' loads ahead, not all of them
    }
}

// A chunk's input and the sample's slices.  Both inputs are read through buffer resources:
// places outside the volume or the sample load zeros (an offset past the buffer's end).
struct HaloSrc {
    __amdgpu_buffer_rsrc_t p;   // the chunk's first channel
    int stride, up;             // bytes of a voxel's row; 1: the half-size grid
    int W, H;
    int x0, y0, z0, zs0, zs1;   // the tile and its sample
};

__device__ __forceinline__ HaloSrc halo_source(const ConvIn &in, const ConvDims &d, int c0)
{
    HaloSrc h;
    h.up = c0 < in.cc ? 1 : 0;   // a chunk lies wholly in one of the two inputs
    const int ch = h.up ? in.cc : d.cin_p - in.cc, skip = h.up ? c0 : c0 - in.cc;
    const unsigned vox = (unsigned)(d.D >> h.up) * (unsigned)(d.H >> h.up) * (unsigned)(d.W >> h.up);
    h.stride = 2 * ch;
    // (scalar registers, which a resource must be in)
    const uint64_t at = reinterpret_cast<uint64_t>((h.up ? in.coarse : in.fine) + skip);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)at), hi = __builtin_amdgcn_readfirstlane((unsigned)(at >> 32));
    h.p = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>((uint64_t)hi << 32 | lo), 0,
                                            __builtin_amdgcn_readfirstlane((vox * (unsigned)ch - (unsigned)skip) * 2),
                                            0x00020000);
    h.W = d.W;
    h.H = d.H;
    return h;
}

// Channel group g of voxel (gx, gy, gz).
__device__ __forceinline__ u16x8 halo_fetch(const HaloSrc &s, int gx, int gy, int gz, int g, bool ok)
{
    const int sh = s.up;
    const unsigned at = (unsigned)(((gz >> sh) * (s.H >> sh) + (gy >> sh)) * (s.W >> sh) + (gx >> sh)) *
                            (unsigned)s.stride + 16 * g;
    ok = ok && (unsigned)gx < (unsigned)s.W && (unsigned)gy < (unsigned)s.H && gz >= s.zs0 && gz < s.zs1;
    // 2^32 - 16: past any buffer (rows are of 16 bytes and more), and the 16 bytes do not wrap
    return __builtin_bit_cast(u16x8, __builtin_amdgcn_raw_buffer_load_b128(s.p, ok ? (int)at : -16, 0, 0));
}

// A layer's epilogue: bias, activation, stores and the head.
struct ConvOut {
    const float *bias;
    unsigned short *Ybf;
    float *Yf;
    ConvHead hd;
};

// Stores 16 voxels x 16 NBW channels from n0 on: lane l holds voxel l % 16 (number vox, if
// in_vol) and channels 4 (l / 16) + e of each block of 16, 8 (bf16) or 16 bytes (float)
// of a row where its layout allows.
template <int NBW>
__device__ __forceinline__ void conv_store(const f32x4 (&acc)[NBW], const float (&bn)[NBW][4],
                                           const float (&hw)[NBW][4], const ConvDims &d, const ConvOut &o, int n0, int q, unsigned vox, bool in_vol)
{
    const bool even = (d.out_stride | d.out_off) % 4 == 0;
    const bool vec_bf = even && !(reinterpret_cast<uintptr_t>(o.Ybf) & 7);
    const bool vec_f = even && !(reinterpret_cast<uintptr_t>(o.Yf) & 15);
    float sum = 0.0f;   // of the head, in channel order: passed on from lane group to lane group
    const int from = (threadIdx.x + 48) & 63;
#pragma unroll
    for (int j = 0; j < NBW; ++j) {
        const int n = n0 + 16 * j + 4 * q, left = d.cout - n;   // channels to store
        const unsigned at = vox * (unsigned)d.out_stride + (unsigned)(d.out_off + n);
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            y[e] = acc[j][e] + bn[j][e];
            if (d.slope >= 0.0f && y[e] < 0.0f) y[e] *= d.slope;
        }
        const u16x4 w = {f2bf(y[0]), f2bf(y[1]), f2bf(y[2]), f2bf(y[3])};
        if (o.hd.out)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (j + k > 0) sum = __shfl(sum, from);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (e < left) sum += bf2f(w[e]) * hw[j][e];   // products of bf16 values are exact
            }
        if (!in_vol || left <= 0) continue;
        if (o.Ybf) {
            if (vec_bf && left >= 4) *reinterpret_cast<u16x4 *>(o.Ybf + at) = w;
            else
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (e < left) o.Ybf[at + e] = w[e];
        }
        if (o.Yf) {
            if (vec_f && left >= 4) *reinterpret_cast<float4 *>(o.Yf + at) = float4{y[0], y[1], y[2], y[3]};
            else
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (e < left) o.Yf[at + e] = y[e];
        }
    }
    if (o.hd.out && q == 3 && in_vol) o.hd.out[vox] = sum + o.hd.b[0];
}

// This lane's biases and head weights.
template <int NBW>
__device__ __forceinline__ void conv_bias(float (&bn)[NBW][4], float (&hw)[NBW][4], const ConvDims &d, const ConvOut &o,
                                          int n0, int q)
{
#pragma unroll
    for (int j = 0; j < NBW; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = n0 + 16 * j + 4 * q + e;
            bn[j][e] = (o.bias && n < d.cout) ? o.bias[n] : 0.0f;
            hw[j][e] = (o.hd.out && n < d.cout) ? bf2f(o.hd.w[n]) : 0.0f;
        }
}

// Tiles of 8 x 8 x 4 / KW voxels: a slice per wavefront (KW = 1), or KW wavefronts share
// one, each with 4 / KW of its four blocks of 16 voxels.
// Bound by the latency of a workgroup's chain (halo, K steps in order, epilogue), so a layer
// is cut into CONV_WANTED workgroups where it has them: 128 -> 128 channels on four samples
// of 4 x 8 x 8 voxels 67 us with 16 workgroups of 128 x 64 outputs, 19 with 128 of 64 x 16;
// 192 -> 64 on four of 8 x 16 x 16 103 -> 45.  (Splitting K over the wavefronts gave 13 and
// 20, but the sums' order would change the bf16 outputs.)  1024 workgroups: 48 -> 64 us on
// the layers of 32 x 32 channels.
template <int TAPS, int NBW, int KW>
__global__ __launch_bounds__(256, NBW == 1 ? (KW == 2 ? 3 : 4) : NBW == 2 ? 3 : 2) void k_conv(ConvIn in, const unsigned short *__restrict__ Wt, ConvDims d,
                                              ConvTile T, ConvOut o)
{
    constexpr int R = TAPS == 27 ? 1 : 0, CZ = 4 / KW, RB = 4 / KW;
    constexpr int EX = CX + 2 * R, HV = halo_voxels(R, CZ);
    constexpr int U = (HV * 4 + 255) / 256;   // 16-byte halo loads of a thread
    extern __shared__ u16x8 halo[];
    // the hardware deals workgroup i to XCD i % 8: give every XCD a contiguous
    // run of tiles, so that the halos neighbouring tiles share hit its L2
    const int per = gridDim.x >> 3;
    const int b = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (b >= T.nblk) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kw = wave % KW, zw = wave / KW;
    const int col = lane & 15, q = lane >> 4;
    const int bx = b % T.ntx, by = (b / T.ntx) % T.nty, bz = b / (T.ntx * T.nty);
    const int zs0 = (bz / T.ntz) * T.Ds, zs1 = zs0 + T.Ds;   // the tile's sample
    const int x0 = bx * CX, y0 = by * CX, z0 = zs0 + (bz % T.ntz) * CZ;
    const int n0 = blockIdx.y * 16 * NBW;
    f32x4 acc[RB][NBW];
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int j = 0; j < NBW; ++j) acc[r][j] = f32x4{0, 0, 0, 0};
    const int64_t tap_stride = (int64_t)d.cout_p * d.cin_p;
    // log2 of the 8-channel groups of the chunk at c (a chunk lies in one input)
    auto groups = [&](int c) {
        const int left = ((c < in.cc ? in.cc : d.cin_p) - c) >> 3;
        return left >= 4 ? 2 : left >= 2 ? 1 : 0;
    };
    // thread i stages items i, i + 256, ...: 8-channel group g of halo voxel hv
    u16x8 v[U];
    auto load = [&](int c0, int lg) {
        HaloSrc h = halo_source(in, d, c0);
        h.zs0 = zs0;
        h.zs1 = zs1;
        const int g = threadIdx.x & ((1 << lg) - 1);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int hv = ((int)threadIdx.x + 256 * u) >> lg;
            v[u] = halo_fetch(h, x0 + hv % EX - R, y0 + (hv / EX) % EX - R, z0 + hv / (EX * EX) - R, g, hv < HV);
        }
    };
    constexpr bool AHEAD = KW > 1;
    int lg = groups(0);
    if (AHEAD) load(0, lg);
    for (int c0 = 0; c0 < d.cin_p;) {
        const int ng = 1 << lg, gp = ng | 1;
        if (!AHEAD) load(c0, lg);
        if (c0 > 0) __syncthreads();   // the previous chunk's reads are done
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int hv = ((int)threadIdx.x + 256 * u) >> lg;
            if (hv < HV) halo[hv * gp + (threadIdx.x & (ng - 1))] = v[u];
        }
        // the next chunk is loaded while this one is multiplied
        const int next = c0 + 8 * ng, lnext = next < d.cin_p ? groups(next) : 0;
        if (AHEAD && next < d.cin_p) load(next, lnext);
        const int v0 = (zw * EX + 2 * RB * kw + (col >> 3)) * EX + (col & 7);
        const unsigned short *wl = Wt + (int64_t)n0 * d.cin_p + c0;
        if (lg == 2)
            conv_chunk<TAPS, 4, NBW, RB, 8>(halo, v0, 0, wl, tap_stride, d.cin_p, col, q, acc);
        else if (lg == 1)
            conv_chunk<TAPS, 2, NBW, RB, 8>(halo, v0, 0, wl, tap_stride, d.cin_p, col, q, acc);
        else
            conv_chunk<TAPS, 1, NBW, RB, 8>(halo, v0, 0, wl, tap_stride, d.cin_p, col, q, acc);
        c0 = next;
        lg = lnext;
    }
    const int gz = z0 + zw, gx = x0 + (col & 7);
    float bn[NBW][4], hw[NBW][4];
    conv_bias(bn, hw, d, o, n0, q);
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        const int gy = y0 + 2 * (RB * kw + r) + (col >> 3);
        conv_store(acc[r], bn, hw, d, o, n0, q, (unsigned)((gz * d.H + gy) * d.W + gx), gx < d.W && gy < d.H && gz < zs1);
    }
}

// k_conv for larger volumes: tiles of 16 x 8 x 4 voxels, a slice per wavefront and a row of
// 16 voxels per MFMA, so that a weight read serves eight products and the halo is 2.1
// times the tile (2.3).  A voxel's channel groups lie side by side, with 32 channels
// exchanged by x so that eight voxels in a row are in different banks.
// Bound by latency and LDS reads.  96 -> 32 channels on 32 samples of 16 x 32 x 32: 99 us
// (176 with k_conv's tiles), 192 -> 64 on 32 of 8 x 16 x 16: 74 (98).
template <int NBW>
__global__ __launch_bounds__(256, NBW == 1 ? 3 : 2) void k_conv_rows(ConvIn in, const unsigned short *__restrict__ Wt,
                                                                     ConvDims d, ConvTile T, ConvOut o)
{
    constexpr int U = (RHV * 4 + 255) / 256, UB = 9;   // halo loads of a thread; in flight
    extern __shared__ u16x8 halo[];
    const int per = gridDim.x >> 3;   // XCD-contiguous tiles, as in k_conv
    const int b = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (b >= T.nblk) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, q = lane >> 4;
    const int bx = b % T.ntx, by = (b / T.ntx) % T.nty, bz = b / (T.ntx * T.nty);
    const int zs0 = (bz / T.ntz) * T.Ds, zs1 = zs0 + T.Ds;   // the tile's sample
    const int x0 = bx * RWX, y0 = by * RWY, z0 = zs0 + (bz % T.ntz) * RWZ;
    const int n0 = blockIdx.y * 16 * NBW;
    f32x4 acc[RWY][NBW];
#pragma unroll
    for (int r = 0; r < RWY; ++r)
#pragma unroll
        for (int j = 0; j < NBW; ++j) acc[r][j] = f32x4{0, 0, 0, 0};
    const int64_t tap_stride = (int64_t)d.cout_p * d.cin_p;
    const int v0 = wave * RHX * RHY + col;
    for (int c0 = 0; c0 < d.cin_p;) {
        const int left = ((c0 < in.cc ? in.cc : d.cin_p) - c0) >> 3;
        const int lg = left >= 4 ? 2 : left >= 2 ? 1 : 0, ng = 1 << lg;
        HaloSrc h = halo_source(in, d, c0);
        h.zs0 = zs0;
        h.zs1 = zs1;
        const int g = threadIdx.x & (ng - 1);
        if (c0 > 0) __syncthreads();   // the previous chunk's reads are done
#pragma unroll
        for (int u0 = 0; u0 < U; u0 += UB) {
            if (((256 * u0) >> lg) >= RHV) break;
            u16x8 v[UB];
#pragma unroll
            for (int u = 0; u < UB; ++u) {
                const int hv = ((int)threadIdx.x + 256 * (u0 + u)) >> lg;
                v[u] = halo_fetch(h, x0 + hv % RHX - 1, y0 + (hv / RHX) % RHY - 1, z0 + hv / (RHX * RHY) - 1, g, hv < RHV);
            }
#pragma unroll
            for (int u = 0; u < UB; ++u) {
                const int hv = ((int)threadIdx.x + 256 * (u0 + u)) >> lg;
                if (hv < RHV) halo[hv * ng + (lg == 2 ? row_slot<4>(g, hv % RHX) : g)] = v[u];
            }
        }
        const unsigned short *wl = Wt + (int64_t)n0 * d.cin_p + c0;
        if (lg == 2) conv_chunk<27, 4, NBW, RWY, 16>(halo, v0, col, wl, tap_stride, d.cin_p, col, q, acc);
        else if (lg == 1) conv_chunk<27, 2, NBW, RWY, 16>(halo, v0, col, wl, tap_stride, d.cin_p, col, q, acc);
        else conv_chunk<27, 1, NBW, RWY, 16>(halo, v0, col, wl, tap_stride, d.cin_p, col, q, acc);
        c0 += 8 * ng;
    }
    const int gx = x0 + col, gz = z0 + wave;
    float bn[NBW][4], hw[NBW][4];
    conv_bias(bn, hw, d, o, n0, q);
#pragma unroll
    for (int r = 0; r < RWY; ++r) {
        const int gy = y0 + r;
        conv_store(acc[r], bn, hw, d, o, n0, q, (unsigned)((gz * d.H + gy) * d.W + gx), gx < d.W && gy < d.H && gz < zs1);
    }
}

// k_conv_rows for 16 output channels whose weights fit in LDS beside the halo (the layers
// at full resolution): chunks of NG0 and NG1 groups of 8 input channels (NG1 = 0: one
// chunk).  The weights are laid there once, as the fragments the lanes read; the
// workgroups stay and walk runs of tiles of 16 x 8 x 8 voxels (eight wavefronts, a slice
// each), and the next chunk's halo is loaded into registers while this one is multiplied:
// no load is waited for inside a chunk.  LDS: 115 KB of halo with 32 channels (one
// workgroup on a CU), 58 KB with 16 (two).
// Bound by MFMA and vector issue together (48 -> 16 channels: 72 us of products and 50 of
// other instructions in 223).  32 samples of 32 x 64 x 64: 8 -> 16 channels 70 us, 16 -> 16
// 90 (floor by bytes 42 and 56), 48 -> 16 223, 16 -> 16 with the head 118; with tiles of
// 128 voxels, weights from global memory and every load waited for these were 193, 226,
// 560 and 255.
constexpr int RSZ = 8, RSV = RHX * RHY * (RSZ + 2);
constexpr int RES_CUS = 256;   // workgroups at a time, one a CU
constexpr int res_frags(int ng) { return (27 * ng + 3) / 4; }   // of a chunk
constexpr size_t res_lds(int ng0, int ng1) { return (size_t)RSV * ng0 * 16 + 1024 * (res_frags(ng0) + res_frags(ng1)); }
static_assert(res_lds(4, 2) + 128 <= 160 * 1024 && 2 * (res_lds(2, 0) + 128) <= 160 * 1024, "workgroups of a CU");

// The halo of one chunk between memory and LDS, by the eight wavefronts.  Rows of the
// tile's 16 columns are whole loads (4 / NG rows of 16 columns a wavefront), so that most
// of a place and its test are scalar; the two outer columns follow as items of their own.
template <int NG>
struct HaloStage {
    static constexpr int UM = NG == 4 ? 13 : NG == 2 ? 7 : 4;           // row loads of a wavefront
    static constexpr int EDGE = 2 * NG * RHY * (RSZ + 2), UE = (EDGE + 511) / 512;
    static constexpr int U = UM + UE;

    // Halo row y, slice z of load u (z past the tile: none); rs: the lane's row of the load.
    static __device__ __forceinline__ void row(int u, int wave, int rs, int &y, int &z)
    {
        if (NG == 4) {          // rows 0-7 one per wavefront, rows 8 and 9 of all slices after them
            const int r = wave + 8 * (u - 10);
            y = u < 10 ? wave : 8 + (r & 1);
            z = u < 10 ? u : r >> 1;
        } else if (NG == 2) {   // row pairs 0-3 of two slices, then pair 4 of eight
            y = (u < 5 ? 2 * (wave & 3) : 8) + rs;
            z = u < 5 ? 2 * u + (wave >> 2) : wave + 8 * (u - 5);
        } else {                // rows 0-3 and 4-7 of four slices, then rows 8 and 9 of two a wavefront
            y = u < 3 ? 4 * (wave & 1) + rs : 8 + (rs & 1);
            z = u < 3 ? (wave >> 1) + 4 * u : 2 * wave + (rs >> 1);
        }
    }

    static __device__ __forceinline__ void load(const HaloSrc &s, int lane, int wave, u16x8 (&v)[U])
    {
        const int g = lane & (NG - 1), gx = s.x0 + ((lane / NG) & 15), rs = lane / (16 * NG);
#pragma unroll
        for (int u = 0; u < UM; ++u) {
            int y, z;
            row(u, wave, rs, y, z);
            v[u] = halo_fetch(s, gx, s.y0 + y - 1, s.z0 + z - 1, g, z < RSZ + 2);
        }
#pragma unroll
        for (int u = 0; u < UE; ++u) {
            const int e = (int)threadIdx.x + 512 * u, r = e / (2 * NG), x = s.x0 + ((e / NG) & 1 ? RWX : -1);
            v[UM + u] = halo_fetch(s, x, s.y0 + r % RHY - 1, s.z0 + r / RHY - 1, e & (NG - 1), e < EDGE);
        }
    }

    static __device__ __forceinline__ void store(u16x8 *halo, int lane, int wave, const u16x8 (&v)[U])
    {
        const int g = lane & (NG - 1), x = ((lane / NG) & 15) + 1, rs = lane / (16 * NG);
        u16x8 *mine = halo + x * NG + row_slot<NG>(g, x);
#pragma unroll
        for (int u = 0; u < UM; ++u) {
            int y, z;
            row(u, wave, rs, y, z);
            if (z < RSZ + 2) mine[(z * RHY + y) * RHX * NG] = v[u];
        }
#pragma unroll
        for (int u = 0; u < UE; ++u) {
            const int e = (int)threadIdx.x + 512 * u, hx = (e / NG) & 1 ? RHX - 1 : 0;
            if (e < EDGE) halo[(e / (2 * NG) * RHX + hx) * NG + row_slot<NG>(e & (NG - 1), hx)] = v[UM + u];
        }
    }
};

// The weights of the NG groups from channel c0 on, as the fragments of conv_chunk's steps.
template <int NG>
__device__ __forceinline__ void res_weights(u16x8 *wf, const unsigned short *__restrict__ W, const ConvDims &d, int n0, int c0)
{
    constexpr int K = 4 / NG;
    for (int i = threadIdx.x; i < res_frags(NG) * 64; i += 512) {
        const int col = i & 15, q = (i >> 4) & 3, t = K * (i >> 6) + q / NG;
        u16x8 w = {0, 0, 0, 0, 0, 0, 0, 0};
        if (t < 27)
            w = *reinterpret_cast<const u16x8 *>(W + t * d.cout_p * d.cin_p + (n0 + col) * d.cin_p + c0 +
                                                 8 * (q & (NG - 1)));
        wf[i] = w;
    }
}

// conv_chunk's sums in its order.  Reads are issued AHEAD places before their use (the
// order is fixed: left to itself the compiler reads and waits).
template <int NG>
__device__ __forceinline__ void conv_res_chunk(const u16x8 *halo, const u16x8 *wf, int lane, int wave,
                                               f32x4 (&acc)[RWY])
{
    constexpr int EXY = RHX * RHY;
    const int col = lane & 15, q = lane >> 4;
    int g = q & (NG - 1), tq = q / NG;
    asm volatile("" : "+v"(g), "+v"(tq));   // addresses are not kept across the chunks
    const u16x8 *h = halo + (wave * EXY + col) * NG;
    auto product = [&](const u16x8 &w, const u16x8 &a, int r) {
        acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a),
                                                         acc[r], 0, 0, 0);
    };
    if constexpr (NG == 4) {
        // Per dz the nine weights, then the ten rows of the halo, each at the three dx: what
        // is read for (y, dx) serves the outputs y, y - 1 and y - 2 (with dy = 0, 1 and 2),
        // and an output meets its taps in order.  39 reads for 72 products.
        constexpr int AHEAD = 4;
        u16x8 w[9], a[2 * AHEAD];
        const u16x8 *p[3];
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) p[dx] = h + dx * NG + row_slot<NG>(g, col + dx);
        auto rows = [&](int dz, int k) { a[k % (2 * AHEAD)] = p[k % 3][(dz * EXY + k / 3 * RHX) * NG]; };
#pragma unroll
        for (int dz = 0; dz < 3; ++dz) {
#pragma unroll
            for (int k = 0; k < 3; ++k) w[k] = wf[(9 * dz + k) * 64 + lane];
#pragma unroll
            for (int k = 0; k < AHEAD; ++k) rows(dz, k);
#pragma unroll
            for (int k = 0; k < 3 * RHY; ++k) {
                const int y = k / 3, dx = k % 3;
                if (k < 6) w[3 + k] = wf[(9 * dz + 3 + k) * 64 + lane];   // dy = 1 and 2: first used at y = 1 and 2
                if (k + AHEAD < 3 * RHY) rows(dz, k + AHEAD);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int dy = 0; dy < 3; ++dy)
                    if (y - dy >= 0 && y - dy < RWY) product(w[3 * dy + dx], a[k % (2 * AHEAD)], y - dy);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    } else {
        // A step's two or four taps are picked per lane: a weight and eight rows a step.
        constexpr int K = 4 / NG, S = (27 + K - 1) / K, AHEAD = 3, PER = 1 + RWY;
        u16x8 w[2], a[2][RWY];
        const u16x8 *p = nullptr;
        auto read = [&](int i) {
            const int s = i / PER, k = i % PER;
            if (k == 0) {
                w[s & 1] = wf[s * 64 + lane];
                int delta = tap_delta<27>(K * s, RHX, EXY);
#pragma unroll
                for (int m = 1; m < K; ++m)
                    delta = tq == m ? tap_delta<27>(K * s + m < 27 ? K * s + m : 26, RHX, EXY) : delta;
                p = h + delta * NG + g;
                return;
            }
            a[s & 1][k - 1] = p[(k - 1) * RHX * NG];
            // the weights are zero there too
            if (K * s + K > 27 && K * s + tq >= 27) a[s & 1][k - 1] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
        };
#pragma unroll
        for (int i = 0; i < 1 + AHEAD; ++i) read(i);
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int r = 0; r < RWY; ++r) {
                const int i = PER * s + 1 + r + AHEAD;
                if (r == RWY - AHEAD && i < PER * S) read(i);   // the next step's weight
                if (r >= RWY - AHEAD ? i + 1 < PER * S : true) read(r >= RWY - AHEAD ? i + 1 : i);
                __builtin_amdgcn_sched_barrier(0);
                product(w[s & 1], a[s & 1][r], r);
                __builtin_amdgcn_sched_barrier(0);
            }
    }
}

template <int NG0, int NG1>
__global__ __launch_bounds__(512, NG0 == 4 ? 2 : 4) void k_conv_res(ConvIn in, const unsigned short *__restrict__ Wt,
                                                                    ConvDims d, ConvTile T, int run, ConvOut o)
{
    constexpr int NGB = NG1 ? NG1 : NG0;
    __shared__ u16x8 lds[res_lds(NG0, NG1) / 16];
    __shared__ float4 ends[2][4];
    u16x8 *halo = lds, *wf0 = lds + RSV * NG0, *wf1 = wf0 + 64 * res_frags(NG0);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, q = lane >> 4;
    // contiguous runs of tiles on every XCD
    const int b = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int t1 = min(T.nblk, (b + 1) * run);
    int tile = b * run;
    if (tile >= t1) return;
    const int n0 = 16 * blockIdx.y;
    res_weights<NG0>(wf0, Wt, d, n0, 0);
    if constexpr (NG1 > 0) res_weights<NG1>(wf1, Wt, d, n0, 8 * NG0);
    if (wave == 0) {   // biases and head weights of the lanes: not held in registers
        float bn[1][4], hw[1][4];
        conv_bias(bn, hw, d, o, n0, q);
        if (col == 0) {
            ends[0][q] = float4{bn[0][0], bn[0][1], bn[0][2], bn[0][3]};
            ends[1][q] = float4{hw[0][0], hw[0][1], hw[0][2], hw[0][3]};
        }
    }
    auto place = [&](int t, HaloSrc &h) {
        const int bx = t % T.ntx, by = (t / T.ntx) % T.nty, bz = t / (T.ntx * T.nty);
        h.zs0 = (bz / T.ntz) * T.Ds;   // the tile's sample
        h.zs1 = h.zs0 + T.Ds;
        h.x0 = bx * RWX;
        h.y0 = by * RWY;
        h.z0 = h.zs0 + (bz % T.ntz) * RSZ;
    };
    HaloSrc h0 = halo_source(in, d, 0), h1 = halo_source(in, d, NG1 ? 8 * NG0 : 0);
    u16x8 v0[HaloStage<NG0>::U], v1[HaloStage<NGB>::U];
    place(tile, h0);
    HaloStage<NG0>::load(h0, lane, wave, v0);
    for (; tile < t1; ++tile) {
        f32x4 acc[RWY];
#pragma unroll
        for (int r = 0; r < RWY; ++r) acc[r] = f32x4{0, 0, 0, 0};
        const int gx = h0.x0 + col, gy0 = h0.y0, gz = h0.z0 + wave;
        const bool inside = gx < d.W && gz < h0.zs1;
        __syncthreads();   // the previous chunk's reads are done
        HaloStage<NG0>::store(halo, lane, wave, v0);
        if constexpr (NG1 > 0) {
            place(tile, h1);
            HaloStage<NGB>::load(h1, lane, wave, v1);
        } else {
            place(min(tile + 1, t1 - 1), h0);
            HaloStage<NG0>::load(h0, lane, wave, v0);
        }
        __syncthreads();   // the halo (and, at first, the weights) are there
        conv_res_chunk<NG0>(halo, wf0, lane, wave, acc);
        if constexpr (NG1 > 0) {
            __syncthreads();
            HaloStage<NGB>::store(halo, lane, wave, v1);
            place(min(tile + 1, t1 - 1), h0);
            HaloStage<NG0>::load(h0, lane, wave, v0);
            __syncthreads();
            conv_res_chunk<NGB>(halo, wf1, lane, wave, acc);
        }
        const float4 bq = ends[0][q], hq = ends[1][q];
        const float bn[1][4] = {{bq.x, bq.y, bq.z, bq.w}}, hw[1][4] = {{hq.x, hq.y, hq.z, hq.w}};
#pragma unroll
        for (int r = 0; r < RWY; ++r) {
            const f32x4 a[1] = {acc[r]};
            conv_store(a, bn, hw, d, o, n0, q, (unsigned)((gz * d.H + gy0 + r) * d.W + gx), inside && gy0 + r < d.H);
        }
    }
}

// Weight gradient of one tap: dW[t][co][ci] += sum_v dY[v][co] * X[v + o_t][ci]
// (dY rows of stride dy_stride, channels [0, cout); X rows of stride cin_p;
// samples of Ds slices stacked along z).  The general-shape path: element
// loads from global memory.  Grid: (voxel chunks, taps, cout blocks of 32 *
// cin blocks of 32).
__global__ __launch_bounds__(256) void k_conv_wgrad(const unsigned short *__restrict__ X,
                                                    const unsigned short *__restrict__ dY, int dy_stride,
                                                    ConvDims d, int Ds, int chunk, float *__restrict__ dW)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int V = d.D * d.H * d.W;
    const int t = blockIdx.y;
    const int ncb = (d.cin_p + 31) / 32;
    const int co0 = (blockIdx.z / ncb) * 32, ci0 = (blockIdx.z % ncb) * 32;
    int dz, dy, dx;
    tap_offset(t, d.taps, dz, dy, dx);
    const int m = lane & 31, kq = (lane >> 5) * 4;
    const int co = co0 + m, ci = ci0 + m;
    const int vbeg = blockIdx.x * chunk, vend = min(V, vbeg + chunk);
    f32x16 acc = {0};
    // each wavefront walks every fourth group of 8 voxels of the chunk
    for (int vb = vbeg + wave * 8; vb < vend; vb += 32) {
        bf16x4 a, b;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int v = vb + kq + j;
            unsigned short av = 0, bv = 0;
            if (v < vend) {
                if (co < d.cout) av = dY[(int64_t)v * dy_stride + co];
                const int x = v % d.W, y = (v / d.W) % d.H, z = v / (d.W * d.H);
                const int zz = z + dz, yy = y + dy, xx = x + dx, zs = z - z % Ds;
                if (ci < d.cin_p && zz >= zs && zz < zs + Ds && yy >= 0 && yy < d.H && xx >= 0 && xx < d.W)
                    bv = X[((int64_t)(zz * d.H + yy) * d.W + xx) * d.cin_p + ci];
            }
            a[j] = (short)av;
            b[j] = (short)bv;
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int r = co0 + 8 * (i / 4) + kq + (i % 4);   // row = output channel
        const int c = ci;                                   // column = input channel
        if (r < d.cout && c < d.cin_p && acc[i] != 0.0f)
            atomicAdd(dW + ((int64_t)t * d.cout_p + r) * d.cin_p + c, acc[i]);
    }
}

// Weight gradient on gfx950's v_mfma_f32_16x16x32_bf16: dW[t][co][ci] +=
// sum_v dY[v][co] X[v + o_t][ci], per tap a GEMM with K = voxels.  A workgroup owns
// 16 FB x 16 SB channels of all taps and a run of 8 x 8 x 4 voxel tiles.  The operand
// with fewer channels is the shifted one: S holds its tile with a halo (X at v + o_t, or
// dY at u - o_t), F the other's without, so that a fragment read at a tap's shift serves
// FB products.  Both lie in LDS as they lie in memory, a plane of 16 channels per block,
// 32 bytes a voxel, and are turned into K-major fragments by the transposing LDS read:
// four lanes name a voxel, 16 lanes four voxels, and lane i receives channel i of them.
// Any voxel shift is then an address (a constant beside the lane's own), and staging is
// 16-byte loads and stores.  Wavefront w keeps taps w, w + 4, ... in registers (27 taps;
// the 28th place sums the bias gradient, against ones) or takes every fourth K step
// (1 tap).  Bound by the LDS reads (2 per SB x tap x K step, 8 cycles of the CU's LDS).
// A workgroup writes its sums to `part`, which k_wgrad_sum adds up in order; without
// scratch (part null: small layers, capture) it adds them to dW with atomics.
// The 15 layers of the 16-32-64-128 network on four 32 x 64 x 64 samples: 241 us and 123
// for the sums (1507 with a transposed copy of the tile in LDS, 32 x 32 channel blocks
// and atomics; 1150 with this kernel and atomics).
constexpr int WGX = 8, WGY = 8, WGZ = 4, WGV = WGX * WGY * WGZ;
constexpr int WG_KS = WGV / 32;   // K steps of a tile
// words of 2 bytes between planes; the 64 bytes over keep two planes in different banks
constexpr int wg_plane(int R) { return (WGX + 2 * R) * (WGY + 2 * R) * (WGZ + 2 * R) * 16 + 32; }
static_assert(2 * (2 * wg_plane(1) + 2 * wg_plane(0)) <= 65536, "static LDS");
// Workgroups of a launch.  The same layers, kernel and sums: 256 432 us, 512 364 us,
// 1024 397 us (more parts to add up).
constexpr int64_t WG_WANTED = 512;
// One tap (four parts a workgroup): two tiles a workgroup or more, beyond this many workgroups
// (16 -> 1 channels on 32 x 64 x 64, 512 workgroups or 256: 23, 17 us).
constexpr int64_t WG_ONE_TAP = 128;
constexpr size_t WG_SCRATCH = 64u << 20;   // bytes of partial sums at most
// Small layers add to dW by atomics: up to 64 additions per element, 2^23 in all, or 2^18 in
// all, cost less than the second launch and its pass over the parts.  us, atomics / parts:
// 128 -> 128 channels on 8 x 16 x 16 voxels 14 / 32 (the copied tiles of before: 17), 96 -> 32
// on 16 x 32 x 32 14 / 28, 16 -> 1, one tap, on 16 x 32 x 32 7 / 12; 16 -> 16 on 32 x 64 x 64
// (512 additions per element) 33 / 22.
constexpr int WG_ATOMIC_PARTS = 64;
constexpr int64_t WG_ATOMIC_ADDS = 1 << 23, WG_ATOMIC_FEW = 1 << 18;

struct WgCfg {
    int ntx, nty, ntz;   // tiles of a sample
    int ntiles, run;     // all tiles; tiles per workgroup
    int Ds;              // slices of a sample
    int swap;            // the shifted operand is dY
    int sstride, fstride;
    int NF, NS;          // channels of the grid's blocks, F and S
};

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 *lds_i16x4;

// The fragment (8 K values of this lane's channel) of 32 voxels: lane group q holds voxels
// 4 q .. 4 q + 3 of p's 16 and of those `next` words on.
__device__ __forceinline__ bf16x8 wg_frag(const unsigned short *p, int next)
{
    const i16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4)p);
    const i16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4)(p + next));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// NB planes of the tile at (x0, y0, z0), with a halo of R voxels: zero outside the sample's
// slices [zs0, zs1), outside the plane and past the row's channels.
template <int NB, int R>
__device__ __forceinline__ void wg_stage(unsigned short *lds, const unsigned short *__restrict__ src, int stride, int c0,
                                         int x0, int y0, int z0, int zs0, int zs1, const ConvDims &d)
{
    constexpr int EX = WGX + 2 * R, EY = WGY + 2 * R, EZ = WGZ + 2 * R, G = 2 * NB, N = EX * EY * EZ * G;
    constexpr int U = 6, PASSES = (N + 255) / 256;   // loads in flight per thread
#pragma unroll
    for (int b = 0; b < PASSES; b += U) {
        u16x8 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (b + u >= PASSES) continue;
            const int i = threadIdx.x + 256 * (b + u);
            const int g = i % G, hv = i / G;
            const int gx = x0 + hv % EX - R, gy = y0 + (hv / EX) % EY - R, gz = z0 + hv / (EX * EY) - R;
            const int c = c0 + 8 * g;
            v[u] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (i < N && (unsigned)gx < (unsigned)d.W && (unsigned)gy < (unsigned)d.H && gz >= zs0 && gz < zs1 && c < stride)
                v[u] = *reinterpret_cast<const u16x8 *>(src + (unsigned)((gz * d.H + gy) * d.W + gx) * (unsigned)stride + c);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = threadIdx.x + 256 * (b + u);
            const int g = i % G, hv = i / G;
            if (b + u < PASSES && i < N)
                *reinterpret_cast<u16x8 *>(lds + (g >> 1) * wg_plane(R) + 16 * hv + 8 * (g & 1)) = v[u];
        }
    }
}

template <int TAPS, int FB, int SB>
__global__ __launch_bounds__(256, 2) void k_conv_wgrad_tr(const unsigned short *__restrict__ S,
                                                          const unsigned short *__restrict__ F, ConvDims d, WgCfg c,
                                                          float *__restrict__ part, float *__restrict__ dW,
                                                          float *__restrict__ db)
{
    constexpr int R = TAPS == 27 ? 1 : 0;
    constexpr int EX = WGX + 2 * R, EXY = EX * (WGY + 2 * R);
    constexpr int NT = TAPS == 27 ? 7 : 2;   // places per wavefront (the last one of wavefront 3: bias)
    constexpr int SP = wg_plane(R), FP = wg_plane(0);
    __shared__ __align__(16) unsigned short lds[SB * SP + FB * FP];
    unsigned short *Sl = lds, *Fl = lds + SB * SP;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, q = lane >> 4;
    const int f0 = blockIdx.y * 16 * FB, s0 = blockIdx.z * 16 * SB;
    // this lane's voxel (of the first 16 of a K step) and 4-channel group in the reads
    const int lv = 4 * q + (col >> 2), lc = 4 * (col & 3);
    const unsigned short *sb = Sl + 16 * ((lv >> 3) * EX + (lv & 7)) + lc, *fb = Fl + 16 * lv + lc;
    // with dY fixed the bias sums its rows, else the columns of the shifted one
    const bool bias = db && (c.swap ? blockIdx.y == 0 : blockIdx.z == 0);
    const i16x8 ones16 = {0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80};
    const bf16x8 ones = __builtin_bit_cast(bf16x8, ones16);
    f32x4 acc[NT][FB][SB];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int r = 0; r < FB; ++r)
#pragma unroll
            for (int j = 0; j < SB; ++j) acc[i][r][j] = f32x4{0, 0, 0, 0};
    const int t_end = min(c.ntiles, (int)(blockIdx.x + 1) * c.run);
    for (int tile = blockIdx.x * c.run; tile < t_end; ++tile) {
        const int bx = tile % c.ntx, by = (tile / c.ntx) % c.nty, bz = tile / (c.ntx * c.nty);
        const int zs0 = (bz / c.ntz) * c.Ds;
        const int x0 = bx * WGX, y0 = by * WGY, z0 = zs0 + (bz % c.ntz) * WGZ;
        __syncthreads();   // the previous tile's reads are done
        wg_stage<SB, R>(Sl, S, c.sstride, s0, x0, y0, z0, zs0, zs0 + c.Ds, d);
        wg_stage<FB, 0>(Fl, F, c.fstride, f0, x0, y0, z0, zs0, zs0 + c.Ds, d);
        __syncthreads();
        if constexpr (TAPS == 27) {
#pragma unroll 1
            for (int k = 0; k < WG_KS; ++k) {   // half a slice of the tile each
                const unsigned short *pk = sb + 16 * ((k >> 1) * EXY + (k & 1) * 4 * EX);
                bf16x8 f[FB];
#pragma unroll
                for (int r = 0; r < FB; ++r) f[r] = wg_frag(fb + r * FP + 16 * 32 * k, 16 * 16);
#pragma unroll
                for (int i = 0; i < NT; ++i) {
                    // wavefront 3's last place: the bias, of the unshifted tap
                    const int t = i < NT - 1 || wave < 3 ? wave + 4 * i : 13;
                    const unsigned short *p = pk + 16 * ((t / 9) * EXY + ((t / 3) % 3) * EX + t % 3);
                    const bool sums = i == NT - 1 && wave == 3;
                    if (sums && !bias) continue;
#pragma unroll
                    for (int j = 0; j < SB; ++j) {
                        const bf16x8 s = sums && !c.swap ? ones : wg_frag(p + j * SP, 16 * 2 * EX);
#pragma unroll
                        for (int r = 0; r < FB; ++r)
                            acc[i][r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sums && c.swap ? ones : f[r], s,
                                                                                   acc[i][r][j], 0, 0, 0);
                    }
                }
            }
        } else {
#pragma unroll
            for (int h = 0; h < WG_KS / 4; ++h) {
                const int k = wave + 4 * h;
                bf16x8 f[FB], s[SB];
#pragma unroll
                for (int r = 0; r < FB; ++r) f[r] = wg_frag(fb + r * FP + 16 * 32 * k, 16 * 16);
#pragma unroll
                for (int j = 0; j < SB; ++j) s[j] = wg_frag(sb + j * SP + 16 * 32 * k, 16 * 16);
#pragma unroll
                for (int r = 0; r < FB; ++r)
#pragma unroll
                    for (int j = 0; j < SB; ++j)
                        acc[0][r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[r], s[j], acc[0][r][j], 0, 0, 0);
                if (bias && !c.swap) {
#pragma unroll
                    for (int r = 0; r < FB; ++r)
                        acc[1][r][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[r], ones, acc[1][r][0], 0, 0, 0);
                } else if (bias) {
#pragma unroll
                    for (int j = 0; j < SB; ++j)
                        acc[1][0][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, s[j], acc[1][0][j], 0, 0, 0);
                }
            }
        }
    }
    // C layout: lane l holds column (S) l % 16, rows (F) 4 (l / 16) + e
    if (part) {
        const int p = TAPS == 27 ? blockIdx.x : blockIdx.x * 4 + wave;
        const int mine = 4 * q * c.NS + col;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const int slot = TAPS == 27 ? wave + 4 * i : i;   // TAPS: the bias
            float *o = part + (((int64_t)p * (TAPS + 1) + slot) * c.NF + f0) * c.NS + s0;
#pragma unroll
            for (int r = 0; r < FB; ++r)
#pragma unroll
                for (int j = 0; j < SB; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[mine + ((16 * r + e) * c.NS + 16 * j)] = acc[i][r][j][e];
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int slot = TAPS == 27 ? wave + 4 * i : i;
#pragma unroll
        for (int r = 0; r < FB; ++r)
#pragma unroll
            for (int j = 0; j < SB; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int f = f0 + 16 * r + 4 * q + e, s = s0 + 16 * j + col;
                    const int co = c.swap ? s : f, ci = c.swap ? f : s;
                    const float v = acc[i][r][j][e];
                    if (co >= d.cout || ci >= d.cin_p || v == 0.0f) continue;
                    if (slot < TAPS)
                        atomicAdd(dW + ((int64_t)(c.swap ? TAPS - 1 - slot : slot) * d.cout_p + co) * d.cin_p + ci, v);
                    else if (bias && ci == 0)
                        atomicAdd(db + co, v);
                }
    }
}

// dW += the parts of k_conv_wgrad_tr, each element by eight groups of threads (parts g,
// g + 8, ...) whose sums are added in order.
__global__ __launch_bounds__(256) void k_wgrad_sum(const float *__restrict__ part, int nparts, int taps, ConvDims d,
                                                   WgCfg c, float *__restrict__ dW, float *__restrict__ db)
{
    __shared__ float red[8][32];
    const int64_t n = (int64_t)(taps + 1) * c.NF * c.NS;
    const int64_t i = (int64_t)blockIdx.x * 32 + (threadIdx.x & 31);
    const int g = threadIdx.x >> 5;
    const int s = (int)(i % c.NS), f = (int)(i / c.NS % c.NF), slot = (int)(i / ((int64_t)c.NS * c.NF));
    const int co = c.swap ? s : f, ci = c.swap ? f : s;
    const bool live = i < n && co < d.cout && (slot == taps ? db && ci == 0 : ci < d.cin_p);
    float sum = 0.0f;
    if (live) {
#pragma unroll 8
        for (int p = g; p < nparts; p += 8) sum += part[p * n + i];
    }
    red[g][threadIdx.x & 31] = sum;
    __syncthreads();
    if (g == 0 && live) {
        for (int k = 1; k < 8; ++k) sum += red[k][threadIdx.x];
        const int t = c.swap ? taps - 1 - slot : slot;
        float *out = slot == taps ? db + co : dW + ((int64_t)t * d.cout_p + co) * d.cin_p + ci;
        *out += sum;
    }
}

// W'[t'][ci][co] = W[26 - t'][co][ci]: the input gradient of a stride-1,
// zero-padded convolution is a convolution of dY with this kernel.
__global__ void k_flip_weights(const unsigned short *__restrict__ W, int taps, int cout, int cout_p, int cin_p,
                               int cin_real, unsigned short *__restrict__ Wf, int fcout_p, int fcin_p)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t n = (int64_t)taps * fcout_p * fcin_p;
    if (i >= n) return;
    const int cc = (int)(i % fcin_p);            // new input channel = old output channel
    const int rr = (int)((i / fcin_p) % fcout_p);// new output channel = old input channel
    const int t = (int)(i / ((int64_t)fcin_p * fcout_p));
    unsigned short val = 0;
    if (cc < cout && rr < cin_real) val = W[((int64_t)(taps - 1 - t) * cout_p + cc) * cin_p + rr];
    Wf[i] = val;
}

// ------------------------------------------------------------ elementwise --

// The elementwise kernels: a thread takes N neighbouring channels of a voxel (16 bytes of
// the wider type where rows and addresses allow, else one value), so that the index
// arithmetic (32-bit where the tensor has fewer than 2^31 elements) is paid once for them.
// Bound by memory, below about 4 MB by the launch.  32 samples' pooling (134 MB read) 62 ->
// 29 us, a batch of 4's upsampling to 524288 x 48 channels 55 -> 17 us, its activation
// gradient of 16 channels 20 -> 11 us; all of a training batch's 530 -> 300 us.
template <class T, int N>
struct Run {
    typedef T V __attribute__((ext_vector_type(N)));
    static __device__ __forceinline__ void load(const T *p, T (&x)[N])
    {
        const V v = *reinterpret_cast<const V *>(p);
#pragma unroll
        for (int k = 0; k < N; ++k) x[k] = v[k];
    }
    static __device__ __forceinline__ void store(T *p, const T (&x)[N])
    {
        V v;
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = x[k];
        *reinterpret_cast<V *>(p) = v;
    }
};
template <class T>
struct Run<T, 1> {
    static __device__ __forceinline__ void load(const T *p, T (&x)[1]) { x[0] = *p; }
    static __device__ __forceinline__ void store(T *p, const T (&x)[1]) { *p = x[0]; }
};

// The item's voxel and first channel (I: the index type), and the voxel's place.
template <class I, int N>
__device__ __forceinline__ bool item_of(I voxels, int C, I &v, int &c)
{
    const I i = (I)blockIdx.x * 256 + threadIdx.x, g = (I)(C / N);
    if (i >= voxels * g) return false;
    v = i / g;
    c = (int)(i - v * g) * N;
    return true;
}

template <class I>
__device__ __forceinline__ void place_of(I v, int H, int W, int &x, int &y, int &z)
{
    const I r = v / (I)W;
    x = (int)(v - r * (I)W);
    z = (int)(r / (I)H);
    y = (int)(r - (I)z * (I)H);
}

// 2x2x2 average pooling (D, H, W: the input's)
template <class I, int N>
__global__ void k_pool(const unsigned short *__restrict__ X, int D, int H, int W, int C, int xs,
                       unsigned short *__restrict__ Y, int ys)
{
    I v;
    int c, x, y, z;
    if (!item_of<I, N>((I)(D / 2) * (I)(H / 2) * (I)(W / 2), C, v, c)) return;
    place_of(v, H / 2, W / 2, x, y, z);
    float s[N] = {};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int zz = 2 * z + (k >> 2), yy = 2 * y + ((k >> 1) & 1), xx = 2 * x + (k & 1);
        unsigned short h[N];
        Run<unsigned short, N>::load(X + ((I)(zz * H + yy) * (I)W + (I)xx) * (I)xs + (I)c, h);
#pragma unroll
        for (int e = 0; e < N; ++e) s[e] += bf2f(h[e]);
    }
    unsigned short h[N];
#pragma unroll
    for (int e = 0; e < N; ++e) h[e] = f2bf(0.125f * s[e]);
    Run<unsigned short, N>::store(Y + v * (I)ys + (I)c, h);
}

// gradient of the pooling: dX[child] = dY[parent] / 8 (written, not added)
template <class I, int N>
__global__ void k_pool_bwd(const float *__restrict__ dY, int D, int H, int W, int C, int dys,
                           float *__restrict__ dX, int dxs)
{
    I v;
    int c, x, y, z;
    if (!item_of<I, N>((I)D * (I)H * (I)W, C, v, c)) return;
    place_of(v, H, W, x, y, z);
    float g[N];
    Run<float, N>::load(dY + ((I)((z / 2) * (H / 2) + y / 2) * (I)(W / 2) + (I)(x / 2)) * (I)dys + (I)c, g);
#pragma unroll
    for (int e = 0; e < N; ++e) g[e] *= 0.125f;
    Run<float, N>::store(dX + v * (I)dxs + (I)c, g);
}

// nearest 2x upsampling into channels [off, off + C) of a wider tensor
template <class I, int N>
__global__ void k_upsample(const unsigned short *__restrict__ X, int D, int H, int W, int C, int xs,
                           unsigned short *__restrict__ Y, int ys, int off)
{
    I v;
    int c, x, y, z;
    if (!item_of<I, N>((I)8 * (I)D * (I)H * (I)W, C, v, c)) return;
    place_of(v, 2 * H, 2 * W, x, y, z);
    unsigned short h[N];
    Run<unsigned short, N>::load(X + ((I)((z / 2) * H + y / 2) * (I)W + (I)(x / 2)) * (I)xs + (I)c, h);
    Run<unsigned short, N>::store(Y + v * (I)ys + (I)(off + c), h);
}

// gradient of the upsampling: dX[parent] = sum of the 8 children's dY (f32)
template <class I, int N>
__global__ void k_upsample_bwd(const float *__restrict__ dY, int D, int H, int W, int C, int dys, int off,
                               float *__restrict__ dX, int dxs)
{
    I v;
    int c, x, y, z;
    if (!item_of<I, N>((I)D * (I)H * (I)W, C, v, c)) return;
    place_of(v, H, W, x, y, z);
    float s[N] = {};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int zz = 2 * z + (k >> 2), yy = 2 * y + ((k >> 1) & 1), xx = 2 * x + (k & 1);
        float g[N];
        Run<float, N>::load(dY + ((I)(zz * 2 * H + yy) * (I)(2 * W) + (I)xx) * (I)dys + (I)(off + c), g);
#pragma unroll
        for (int e = 0; e < N; ++e) s[e] += g[e];
    }
    Run<float, N>::store(dX + v * (I)dxs + (I)c, s);
}

// copy channels [0,C) of X (stride xs) into channels [off, off+C) of Y (stride ys); bf16 or f32
template <class T, class I, int N>
__global__ void k_copy_channels(const T *__restrict__ X, I V, int C, int xs, int xoff, T *__restrict__ Y,
                                int ys, int yoff, int accumulate)
{
    I v;
    int c;
    if (!item_of<I, N>(V, C, v, c)) return;
    T a[N];
    Run<T, N>::load(X + v * (I)xs + (I)(xoff + c), a);
    T *y = Y + v * (I)ys + (I)(yoff + c);
    if (accumulate) {
        T b[N];
        Run<T, N>::load(y, b);
#pragma unroll
        for (int e = 0; e < N; ++e) a[e] = b[e] + a[e];
    }
    Run<T, N>::store(y, a);
}

// dPre = dAct * (act > 0 ? 1 : slope) -> bf16 (stride ps, zero-filled pad channels);
// act > 0 exactly when the pre-activation is > 0 (slope > 0).  WIDE: the rows of dA and A
// allow 16-byte reads (else one channel at a time).
template <class I, bool WIDE>
__global__ void k_act_bwd(const float *__restrict__ dA, int das, const unsigned short *__restrict__ A, int as,
                          I V, int C, int Cp, float slope, unsigned short *__restrict__ dP)
{
    I v;
    int c;
    if (!item_of<I, 8>(V, Cp, v, c)) return;
    float g[8] = {};
    unsigned short a[8] = {}, h[8];
    if (WIDE && c + 8 <= C) {
        float lo[4], hi[4];
        Run<float, 4>::load(dA + v * (I)das + (I)c, lo);
        Run<float, 4>::load(dA + v * (I)das + (I)(c + 4), hi);
        if (slope >= 0.0f) Run<unsigned short, 8>::load(A + v * (I)as + (I)c, a);
#pragma unroll
        for (int e = 0; e < 8; ++e) g[e] = e < 4 ? lo[e & 3] : hi[e & 3];
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (c + e < C) {
                g[e] = dA[v * (I)das + (I)(c + e)];
                if (slope >= 0.0f) a[e] = A[v * (I)as + (I)(c + e)];
            }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        if (slope >= 0.0f && c + e < C && !(bf2f(a[e]) > 0.0f)) g[e] *= slope;
        h[e] = f2bf(g[e]);
    }
    Run<unsigned short, 8>::store(dP + v * (I)Cp + (I)c, h);
}

// k_act_bwd into rows that are not 16-byte aligned
__global__ void k_act_bwd_one(const float *__restrict__ dA, int das, const unsigned short *__restrict__ A, int as,
                              int64_t V, int C, int Cp, float slope, unsigned short *__restrict__ dP)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= V * Cp) return;
    const int c = (int)(i % Cp);
    const int64_t v = i / Cp;
    float g = 0.0f;
    if (c < C) {
        g = dA[v * das + c];
        if (slope >= 0.0f && !(bf2f(A[v * as + c]) > 0.0f)) g *= slope;
    }
    dP[v * Cp + c] = f2bf(g);
}

// db[c] = sum_v dP[v][c] (bf16 rows of stride Cp), one block per channel
__global__ __launch_bounds__(256) void k_bias_grad(const unsigned short *__restrict__ dP, int64_t V, int Cp,
                                                   float *__restrict__ db)
{
    __shared__ float red[256];
    const int c = blockIdx.x;
    float s = 0.0f;
    for (int64_t v = threadIdx.x; v < V; v += 256) s += bf2f(dP[v * Cp + c]);
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) db[c] += red[0];
}

// loss = w mean((p - t)^2) accumulated into loss[0]; grad = 2 w (p - t) / n
__global__ __launch_bounds__(256) void k_mse(const float *__restrict__ p, const float *__restrict__ t, int64_t n,
                                             float w, float *__restrict__ grad, float *__restrict__ loss)
{
    __shared__ float red[256];
    float s = 0.0f;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const float e = p[i] - t[i];
        grad[i] = 2.0f * w * e / (float)n;
        s += e * e;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, w * red[0] / (float)n);
}

// Adam (Kingma & Ba 2015) on FP32 master weights; writes the bf16 copy.
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, int64_t n, float lr, float b1, float b2, float eps, float bc1,
                       float bc2, float gscale, unsigned short *__restrict__ wbf)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i] * gscale;
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
    w[i] = wi;
    if (wbf) wbf[i] = f2bf(wi);
}

__global__ void k_f32_to_bf16(const float *__restrict__ x, int64_t n, unsigned short *__restrict__ y)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

__global__ void k_bf16_to_f32(const unsigned short *__restrict__ x, int64_t n, float *__restrict__ y)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = bf2f(x[i]);
}

// Surrogate input features per sinogram bin from the emission and attenuation
// line integrals along the bin's LOR (scale[0] = 1 / mean emission integral)
// and an optional extra sinogram (scale[1]):
//   [e, exp(-mu), e * exp(-mu), mu / 4, extra * scale[1], 0, 0, 0], e = em * scale[0]
__global__ void k_features(const float *__restrict__ em, const float *__restrict__ mu,
                           const float *__restrict__ extra, int64_t n, const float *__restrict__ scale,
                           unsigned short *__restrict__ x)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float e = em[i] * scale[0];
    const float a = expf(-mu[i]);
    ushort4 lo, hi;
    lo.x = f2bf(e);
    lo.y = f2bf(a);
    lo.z = f2bf(e * a);
    lo.w = f2bf(0.25f * mu[i]);
    hi.x = extra ? f2bf(extra[i] * scale[1]) : (unsigned short)0;
    hi.y = hi.z = hi.w = 0;
    reinterpret_cast<ushort4 *>(x)[2 * i] = lo;
    reinterpret_cast<ushort4 *>(x)[2 * i + 1] = hi;
}

static inline unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

// Voxels x row fits a 32-bit index; rows and offsets are runs of n; both addresses 16-byte.
static inline bool index32(int64_t voxels, int64_t row) { return row > 0 && voxels * row < ((int64_t)1 << 31); }
static inline bool runs(int n, int a, int b, int c, int d = 0) { return a % n == 0 && b % n == 0 && c % n == 0 && d % n == 0; }
static inline bool aligned16(const void *a, const void *b)
{
    return !((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15);
}

}  // namespace srf

using namespace srf;

static int conv_launch(ConvIn in, const void *w, const float *bias, int32_t N, int32_t D, int32_t H, int32_t W,
                       int32_t cin_p, int32_t cout, int32_t cout_p, int32_t taps, int32_t out_stride, int32_t out_off,
                       float slope, void *y_bf16, float *y_f32, void *stream, ConvHead hd = ConvHead{nullptr, nullptr,
                                                                                                     nullptr})
{
    if (!in.fine || !w || N <= 0 || D <= 0 || H <= 0 || W <= 0) return SRF_ERR_INVALID_ARG;
    if (cin_p <= 0 || cin_p % 8 || cout <= 0 || cout_p % 32 || cout > cout_p) return SRF_ERR_INVALID_ARG;
    if (taps != 1 && taps != 27) return SRF_ERR_INVALID_ARG;
    if (out_off < 0 || out_off + cout > out_stride || (!y_bf16 && !y_f32)) return SRF_ERR_INVALID_ARG;
    if ((reinterpret_cast<uintptr_t>(in.fine) | reinterpret_cast<uintptr_t>(in.coarse) |
         reinterpret_cast<uintptr_t>(w)) & 15)
        return SRF_ERR_INVALID_ARG;
    if ((int64_t)N * D * H * W * (cin_p > out_stride ? cin_p : out_stride) >= ((int64_t)1 << 31))
        return SRF_ERR_UNSUPPORTED;
    ConvDims d{N * D, H, W, cin_p, cout, cout_p, out_stride, out_off, taps, slope};
    const int R = taps == 27 ? 1 : 0;
    const int nb = (cout + 15) / 16;
    const int widest = (nb >= 4 && cout_p % 64 == 0) ? 4 : nb >= 2 ? 2 : 1;
    if (hd.out && (nb > widest || !hd.w || !hd.b)) return SRF_ERR_UNSUPPORTED;   // the head needs every channel
    auto *ws = (const unsigned short *)w;
    auto st = (hipStream_t)stream;
    const ConvOut o{bias, (unsigned short *)y_bf16, y_f32, hd};
    // k_conv_res: up to three blocks of outputs (each reads the halo again: 16 -> 48 channels
    // 47 us, 76 in k_conv), chunks that it has, at most a quarter more voxels by padding to
    // its tiles (beyond that k_conv's 8 x 8 ones do less work) and two tiles for every CU.
    int ng[3] = {0, 0, 0}, nch = 0;
    for (int c = 0; c < cin_p && nch < 3; ++nch) {
        const int left = ((c < in.cc ? in.cc : cin_p) - c) >> 3;
        ng[nch] = left >= 4 ? 4 : left >= 2 ? 2 : 1;
        c += 8 * ng[nch];
    }
    const int64_t stx = (W + RWX - 1) / RWX, stz = (D + RSZ - 1) / RSZ, sblk = stx * ((H + RWY - 1) / RWY) * stz * N;
    const int kind = ng[2] ? 0 : 10 * ng[0] + ng[1];
    if (taps == 27 && nb <= 3 && (!hd.out || nb == 1) && (kind == 10 || kind == 20 || kind == 40 || kind == 42) && 4 * stx * RWX <= 5 * W &&
        4 * stz * RSZ <= 5 * D && sblk >= 2 * RES_CUS) {
        ConvTile T;
        T.ntx = (int)stx;
        T.nty = (H + RWY - 1) / RWY;
        T.ntz = (int)stz;
        T.Ds = D;
        T.nblk = (int)sblk;
        const int wgs = (ng[0] == 4 ? RES_CUS : 2 * RES_CUS) / nb / 8 * 8, run = (int)((sblk + wgs - 1) / wgs);
        const dim3 grid((unsigned)wgs, (unsigned)nb);
        if (kind == 42) hipLaunchKernelGGL((k_conv_res<4, 2>), grid, dim3(512), 0, st, in, ws, d, T, run, o);
        else if (kind == 40) hipLaunchKernelGGL((k_conv_res<4, 0>), grid, dim3(512), 0, st, in, ws, d, T, run, o);
        else if (kind == 20) hipLaunchKernelGGL((k_conv_res<2, 0>), grid, dim3(512), 0, st, in, ws, d, T, run, o);
        else hipLaunchKernelGGL((k_conv_res<1, 0>), grid, dim3(512), 0, st, in, ws, d, T, run, o);
        return launch_status();
    }
    // k_conv_rows from a workgroup for every CU on (half as many: 31 us for 26 in k_conv)
    const int rbw = nb % 2 == 0 ? 2 : 1;
    const int64_t rtx = (W + RWX - 1) / RWX, rblk = rtx * ((H + RWY - 1) / RWY) * ((D + RWZ - 1) / RWZ) * N;
    if (taps == 27 && 4 * rtx * RWX <= 5 * W && rblk * (nb / rbw) >= ROWS_WANTED && (!hd.out || nb <= rbw)) {
        ConvTile T;
        T.ntx = (int)rtx;
        T.nty = (H + RWY - 1) / RWY;
        T.ntz = (D + RWZ - 1) / RWZ;
        T.Ds = D;
        T.nblk = (int)rblk;
        const int ng = cin_p >= 32 ? 4 : cin_p >= 16 ? 2 : 1;
        const size_t lds = (size_t)RHV * ng * 16;
        dim3 grid((unsigned)((rblk + 7) / 8 * 8), (unsigned)(nb / rbw));
        if (rbw == 2) hipLaunchKernelGGL(k_conv_rows<2>, grid, dim3(256), lds, st, in, ws, d, T, o);
        else hipLaunchKernelGGL(k_conv_rows<1>, grid, dim3(256), lds, st, in, ws, d, T, o);
        return launch_status();
    }
    int nbw = widest, kw = 1;
    auto blocks = [&] {
        const int cz = 4 / kw;
        return (int64_t)((W + CX - 1) / CX) * ((H + CX - 1) / CX) * ((D + cz - 1) / cz) * N * ((nb + nbw - 1) / nbw);
    };
    if (!hd.out)
        while (nbw > 1 && blocks() < CONV_WANTED) nbw >>= 1;
    if (taps == 27)
        while (kw < 4 && blocks() < CONV_WANTED) kw <<= 1;
    ConvTile T;
    T.ntx = (W + CX - 1) / CX;
    T.nty = (H + CX - 1) / CX;
    T.ntz = (D + 4 / kw - 1) / (4 / kw);
    T.Ds = D;
    T.nblk = T.ntx * T.nty * T.ntz * N;
    const int lg = cin_p >= 32 ? 2 : cin_p >= 16 ? 1 : 0;
    const size_t lds = (size_t)halo_voxels(R, 4 / kw) * ((1 << lg) | 1) * 16;
    // a multiple of 8 workgroups (the XCD-contiguous tile order; extra ones exit)
    dim3 grid((unsigned)((T.nblk + 7) / 8 * 8), (unsigned)((nb + nbw - 1) / nbw));
#define SRF_CONV(TP, NBW, KW) \
    hipLaunchKernelGGL((k_conv<TP, NBW, KW>), grid, dim3(256), lds, st, in, ws, d, T, o)
    if (taps == 27) {
        if (kw == 1) {
            if (nbw == 4) SRF_CONV(27, 4, 1);
            else if (nbw == 2) SRF_CONV(27, 2, 1);
            else SRF_CONV(27, 1, 1);
        } else if (kw == 2) {
            if (nbw == 4) SRF_CONV(27, 4, 2);
            else if (nbw == 2) SRF_CONV(27, 2, 2);
            else SRF_CONV(27, 1, 2);
        } else {
            if (nbw == 4) SRF_CONV(27, 4, 4);
            else if (nbw == 2) SRF_CONV(27, 2, 4);
            else SRF_CONV(27, 1, 4);
        }
    } else {
        if (nbw == 4) SRF_CONV(1, 4, 1);
        else if (nbw == 2) SRF_CONV(1, 2, 1);
        else SRF_CONV(1, 1, 1);
    }
#undef SRF_CONV
    return launch_status();
}

extern "C" {

int srf_cnn_conv_batch(const void *x, const void *w, const float *bias, int32_t N, int32_t D, int32_t H, int32_t W,
                       int32_t cin_p, int32_t cout, int32_t cout_p, int32_t taps, int32_t out_stride, int32_t out_off,
                       float slope, void *y_bf16, float *y_f32, void *stream)
{
    return conv_launch(ConvIn{(const unsigned short *)x, nullptr, 0}, w, bias, N, D, H, W, cin_p, cout, cout_p, taps,
                       out_stride, out_off, slope, y_bf16, y_f32, stream);
}

int srf_cnn_conv_head_batch(const void *x, const void *w, const float *bias, int32_t N, int32_t D, int32_t H,
                            int32_t W, int32_t cin_p, int32_t cout, int32_t cout_p, int32_t taps, float slope,
                            void *y_bf16, const void *head_w, const float *head_b, float *head_out, void *stream)
{
    if (!y_bf16 || !head_out || !head_w || !head_b) return SRF_ERR_INVALID_ARG;
    return conv_launch(ConvIn{(const unsigned short *)x, nullptr, 0}, w, bias, N, D, H, W, cin_p, cout, cout_p, taps,
                       cout, 0, slope, y_bf16, nullptr, stream,
                       ConvHead{(const unsigned short *)head_w, head_b, head_out});
}

int srf_cnn_conv_up_batch(const void *fine, const void *coarse, int32_t cc, const void *w, const float *bias,
                          int32_t N, int32_t D, int32_t H, int32_t W, int32_t cin_p, int32_t cout, int32_t cout_p,
                          int32_t taps, int32_t out_stride, int32_t out_off, float slope, void *y_bf16, float *y_f32,
                          void *stream)
{
    if (!coarse || cc <= 0 || cc % 8 || cc >= cin_p || D % 2 || H % 2 || W % 2) return SRF_ERR_INVALID_ARG;
    return conv_launch(ConvIn{(const unsigned short *)fine, (const unsigned short *)coarse, cc}, w, bias, N, D, H, W,
                       cin_p, cout, cout_p, taps, out_stride, out_off, slope, y_bf16, y_f32, stream);
}

int srf_cnn_conv(const void *x, const void *w, const float *bias, int32_t D, int32_t H, int32_t W, int32_t cin_p,
                 int32_t cout, int32_t cout_p, int32_t taps, int32_t out_stride, int32_t out_off, float slope,
                 void *y_bf16, float *y_f32, void *stream)
{
    return srf_cnn_conv_batch(x, w, bias, 1, D, H, W, cin_p, cout, cout_p, taps, out_stride, out_off, slope, y_bf16,
                              y_f32, stream);
}

int srf_cnn_conv_wgrad_batch(const void *x, const void *dy, int32_t dy_stride, int32_t N, int32_t D, int32_t H,
                             int32_t W, int32_t cin_p, int32_t cout, int32_t cout_p, int32_t taps, float *dw,
                             float *db, void *stream)
{
    if (!x || !dy || !dw || N <= 0 || D <= 0 || H <= 0 || W <= 0) return SRF_ERR_INVALID_ARG;
    if (cin_p <= 0 || cin_p % 8 || cout <= 0 || cout_p % 32 || cout > cout_p || dy_stride < cout)
        return SRF_ERR_INVALID_ARG;
    if (taps != 1 && taps != 27) return SRF_ERR_INVALID_ARG;
    if ((int64_t)N * D * H * W * (cin_p > dy_stride ? cin_p : dy_stride) >= ((int64_t)1 << 31))
        return SRF_ERR_UNSUPPORTED;
    ConvDims d{N * D, H, W, cin_p, cout, cout_p, 0, 0, taps, -1.0f};
    auto st = (hipStream_t)stream;
    // the LDS path: 16-byte aligned rows of both operands
    if (dy_stride % 8 == 0 && !((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(dy)) & 15)) {
        const int nx = (cin_p + 15) / 16, ny = (cout + 15) / 16;
        WgCfg c;
        c.swap = ny < nx ? 1 : 0;
        const int nf = c.swap ? nx : ny, ns = c.swap ? ny : nx;
        // one tap: two blocks of each or one of each (32 -> 64 channels on 64 x 128 x 128 59 us,
        // one of each 107: both operands are read once per block of the other)
        const int SB = ns < 2 ? 1 : 2;
        const int FB = nf < 2 || (taps == 1 && SB == 1) ? 1 : nf % 3 == 0 && SB == 1 ? 3 : 2;   // (3, 2) would spill
        const int gf = (nf + FB - 1) / FB, gs = (ns + SB - 1) / SB;
        c.NF = gf * FB * 16;
        c.NS = gs * SB * 16;
        c.sstride = c.swap ? dy_stride : cin_p;
        c.fstride = c.swap ? cin_p : dy_stride;
        c.ntx = (W + WGX - 1) / WGX;
        c.nty = (H + WGY - 1) / WGY;
        c.ntz = (D + WGZ - 1) / WGZ;
        c.Ds = D;
        c.ntiles = c.ntx * c.nty * c.ntz * N;
        const size_t per = (size_t)(taps + 1) * c.NF * c.NS * sizeof(float) * (taps == 1 ? 4 : 1);
        // WG_WANTED workgroups, and at most WG_SCRATCH of partial sums
        int64_t parts = WG_WANTED / ((int64_t)gf * gs);
        const int64_t one = c.ntiles / 2 > WG_ONE_TAP ? c.ntiles / 2 : WG_ONE_TAP;
        if (taps == 1 && parts > one) parts = one;
        parts = parts < (int64_t)(WG_SCRATCH / per) ? parts : (int64_t)(WG_SCRATCH / per);
        parts = parts < 1 ? 1 : parts;
        c.run = (int)((c.ntiles + parts - 1) / parts);
        dim3 grid((unsigned)((c.ntiles + c.run - 1) / c.run), (unsigned)gf, (unsigned)gs);
        const int nparts = (int)grid.x * (taps == 1 ? 4 : 1);
        // no scratch under capture, where every element has one writer, nor for few additions
        // (WG_ATOMIC_*)
        const int64_t adds = (int64_t)(per / sizeof(float)) * grid.x;
        const bool few = (nparts <= WG_ATOMIC_PARTS && adds <= WG_ATOMIC_ADDS) || adds <= WG_ATOMIC_FEW;
        float *part = nullptr;
        if (!few && !capturing(st) && nparts > 1 && per * grid.x <= WG_SCRATCH)
            part = static_cast<float *>(pool_get(per * grid.x, st));
        auto *S = (const unsigned short *)(c.swap ? dy : x), *F = (const unsigned short *)(c.swap ? x : dy);
#define SRF_WGRAD(TP, FBK, SBK) \
    hipLaunchKernelGGL((k_conv_wgrad_tr<TP, FBK, SBK>), grid, dim3(256), 0, st, S, F, d, c, part, dw, db)
        if (taps == 1 && SB == 2) SRF_WGRAD(1, 2, 2);
        else if (taps == 1) SRF_WGRAD(1, 1, 1);
        else if (SB == 2) SRF_WGRAD(27, 2, 2);
        else if (FB == 3) SRF_WGRAD(27, 3, 1);
        else if (FB == 2) SRF_WGRAD(27, 2, 1);
        else SRF_WGRAD(27, 1, 1);
#undef SRF_WGRAD
        int rc = launch_status();
        if (part) {
            const int64_t n = (int64_t)(taps + 1) * c.NF * c.NS;
            if (rc == SRF_OK) {
                hipLaunchKernelGGL(k_wgrad_sum, dim3((unsigned)((n + 31) / 32)), dim3(256), 0, st, part, nparts, taps, d,
                                   c, dw, db);
                rc = launch_status();
            }
            pool_put(part, st, false, true);
        }
        return rc;
    }
    const int64_t V = (int64_t)N * D * H * W;
    const int chunk = 4096;
    dim3 grid((unsigned)((V + chunk - 1) / chunk), (unsigned)taps, (unsigned)((cout_p / 32) * ((cin_p + 31) / 32)));
    hipLaunchKernelGGL(k_conv_wgrad, grid, dim3(256), 0, st, (const unsigned short *)x, (const unsigned short *)dy,
                       dy_stride, d, D, chunk, dw);
    int rc = launch_status();
    if (rc == SRF_OK && db)
        hipLaunchKernelGGL(k_bias_grad, dim3((unsigned)cout), dim3(256), 0, st, (const unsigned short *)dy, V,
                           dy_stride, db);
    return rc == SRF_OK ? launch_status() : rc;
}

int srf_cnn_conv_wgrad(const void *x, const void *dy, int32_t dy_stride, int32_t D, int32_t H, int32_t W,
                       int32_t cin_p, int32_t cout, int32_t cout_p, int32_t taps, float *dw, void *stream)
{
    return srf_cnn_conv_wgrad_batch(x, dy, dy_stride, 1, D, H, W, cin_p, cout, cout_p, taps, dw, nullptr, stream);
}

int srf_cnn_flip_weights(const void *w, int32_t taps, int32_t cout, int32_t cout_p, int32_t cin_p, int32_t cin,
                         void *wf, int32_t fcout_p, int32_t fcin_p, void *stream)
{
    if (!w || !wf || (taps != 1 && taps != 27) || fcin_p % 8 || fcout_p % 32 || fcin_p < cout || fcout_p < cin)
        return SRF_ERR_INVALID_ARG;
    const int64_t n = (int64_t)taps * fcout_p * fcin_p;
    hipLaunchKernelGGL(k_flip_weights, dim3(nblk(n)), dim3(256), 0, (hipStream_t)stream,
                       (const unsigned short *)w, taps, cout, cout_p, cin_p, cin, (unsigned short *)wf, fcout_p,
                       fcin_p);
    return launch_status();
}

int srf_cnn_pool(const void *x, int32_t D, int32_t H, int32_t W, int32_t C, int32_t xs, void *y, int32_t ys,
                 void *stream)
{
    if (!x || !y || D % 2 || H % 2 || W % 2 || C <= 0) return SRF_ERR_INVALID_ARG;
    const int64_t V = (int64_t)D * H * W / 8;
    auto *in = (const unsigned short *)x;
    auto *out = (unsigned short *)y;
    const bool small = index32(8 * V, xs) && index32(V, ys);
#define GO(I, N) \
    hipLaunchKernelGGL((k_pool<I, N>), dim3(nblk(V * (C / N))), dim3(256), 0, (hipStream_t)stream, in, D, H, W, C, xs, out, ys)
    if (small && runs(8, C, xs, ys) && aligned16(x, y)) GO(unsigned, 8);
    else if (small) GO(unsigned, 1);
    else GO(int64_t, 1);
#undef GO
    return launch_status();
}

int srf_cnn_pool_bwd(const float *dy, int32_t D, int32_t H, int32_t W, int32_t C, int32_t dys, float *dx,
                     int32_t dxs, void *stream)
{
    if (!dy || !dx || D % 2 || H % 2 || W % 2 || C <= 0) return SRF_ERR_INVALID_ARG;
    const int64_t V = (int64_t)D * H * W;
    const bool small = index32(V, dxs) && index32(V, dys);
#define GO(I, N) \
    hipLaunchKernelGGL((k_pool_bwd<I, N>), dim3(nblk(V * (C / N))), dim3(256), 0, (hipStream_t)stream, dy, D, H, W, C, dys, dx, dxs)
    if (small && runs(4, C, dys, dxs) && aligned16(dy, dx)) GO(unsigned, 4);
    else if (small) GO(unsigned, 1);
    else GO(int64_t, 1);
#undef GO
    return launch_status();
}

int srf_cnn_upsample(const void *x, int32_t D, int32_t H, int32_t W, int32_t C, int32_t xs, void *y, int32_t ys,
                     int32_t off, void *stream)
{
    if (!x || !y || C <= 0 || off + C > ys) return SRF_ERR_INVALID_ARG;
    const int64_t V = (int64_t)8 * D * H * W;
    auto *in = (const unsigned short *)x;
    auto *out = (unsigned short *)y;
    const bool small = index32(V, xs) && index32(V, ys) && off >= 0;
#define GO(I, N) \
    hipLaunchKernelGGL((k_upsample<I, N>), dim3(nblk(V * (C / N))), dim3(256), 0, (hipStream_t)stream, in, D, H, W, C, xs, out, ys, off)
    if (small && runs(8, C, xs, ys, off) && aligned16(x, y)) GO(unsigned, 8);
    else if (small) GO(unsigned, 1);
    else GO(int64_t, 1);
#undef GO
    return launch_status();
}

int srf_cnn_upsample_bwd(const float *dy, int32_t D, int32_t H, int32_t W, int32_t C, int32_t dys, int32_t off,
                         float *dx, int32_t dxs, void *stream)
{
    if (!dy || !dx || C <= 0) return SRF_ERR_INVALID_ARG;
    const int64_t V = (int64_t)D * H * W;
    const bool small = index32(8 * V, dys) && index32(V, dxs) && off >= 0;
#define GO(I, N) \
    hipLaunchKernelGGL((k_upsample_bwd<I, N>), dim3(nblk(V * (C / N))), dim3(256), 0, (hipStream_t)stream, dy, D, H, W, C, dys, off, dx, dxs)
    if (small && runs(4, C, dys, dxs, off) && aligned16(dy, dx)) GO(unsigned, 4);
    else if (small) GO(unsigned, 1);
    else GO(int64_t, 1);
#undef GO
    return launch_status();
}

int srf_cnn_copy_channels(const void *x, int64_t V, int32_t C, int32_t xs, int32_t xoff, void *y, int32_t ys,
                          int32_t yoff, int32_t f32, int32_t accumulate, void *stream)
{
    if (!x || !y || C <= 0 || V < 0) return SRF_ERR_INVALID_ARG;
    if (!f32 && accumulate) return SRF_ERR_UNSUPPORTED;
    const bool small = index32(V, xs) && index32(V, ys) && index32(V, C) && xoff >= 0 && yoff >= 0;
    const bool wide = small && runs(f32 ? 4 : 8, C, xs, ys, xoff | yoff) && aligned16(x, y);
#define GO(T, I, N)                                                                                                  \
    hipLaunchKernelGGL((k_copy_channels<T, I, N>), dim3(nblk(V * (C / N))), dim3(256), 0, (hipStream_t)stream,       \
                       (const T *)x, (I)V, C, xs, xoff, (T *)y, ys, yoff, accumulate)
    if (f32) {
        if (wide) GO(float, unsigned, 4);
        else if (small) GO(float, unsigned, 1);
        else GO(float, int64_t, 1);
    } else {
        if (wide) GO(unsigned short, unsigned, 8);
        else if (small) GO(unsigned short, unsigned, 1);
        else GO(unsigned short, int64_t, 1);
    }
#undef GO
    return launch_status();
}

int srf_cnn_act_bwd(const float *da, int32_t das, const void *a, int32_t as, int64_t V, int32_t C, int32_t Cp,
                    float slope, void *dp, void *stream)
{
    if (!da || !a || !dp || C <= 0 || Cp < C || Cp % 8) return SRF_ERR_INVALID_ARG;
    auto *act = (const unsigned short *)a;
    auto *out = (unsigned short *)dp;
    const bool small = index32(V, das) && index32(V, as) && index32(V, Cp);
#define GO(I, WIDE) \
    hipLaunchKernelGGL((k_act_bwd<I, WIDE>), dim3(nblk(V * (Cp / 8))), dim3(256), 0, (hipStream_t)stream, da, das, act, as, (I)V, C, Cp, slope, out)
    if (!aligned16(dp, dp) || !small)
        hipLaunchKernelGGL(k_act_bwd_one, dim3(nblk(V * Cp)), dim3(256), 0, (hipStream_t)stream, da, das, act, as, V, C,
                           Cp, slope, out);
    else if (as % 8 == 0 && das % 4 == 0 && aligned16(da, a)) GO(unsigned, true);
    else GO(unsigned, false);
#undef GO
    return launch_status();
}

int srf_cnn_bias_grad(const void *dp, int64_t V, int32_t C, int32_t Cp, float *db, void *stream)
{
    if (!dp || !db || C <= 0) return SRF_ERR_INVALID_ARG;
    hipLaunchKernelGGL(k_bias_grad, dim3((unsigned)C), dim3(256), 0, (hipStream_t)stream, (const unsigned short *)dp,
                       V, Cp, db);
    return launch_status();
}

int srf_cnn_mse(const float *p, const float *t, int64_t n, float weight, float *grad, float *loss, void *stream)
{
    if (!p || !t || !grad || !loss || n <= 0 || !(weight >= 0.0f)) return SRF_ERR_INVALID_ARG;
    hipLaunchKernelGGL(k_mse, dim3((unsigned)((n + 255) / 256 < 128 ? (n + 255) / 256 : 128)), dim3(256), 0,
                       (hipStream_t)stream, p, t, n, weight, grad, loss);
    return launch_status();
}

int srf_cnn_adam(float *w, const float *g, float *m, float *v, int64_t n, float lr, float b1, float b2, float eps,
                 int32_t step, float gscale, void *wbf, void *stream)
{
    if (!w || !g || !m || !v || n <= 0 || step <= 0) return SRF_ERR_INVALID_ARG;
    const float bc1 = 1.0f - powf(b1, (float)step), bc2 = 1.0f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(nblk(n)), dim3(256), 0, (hipStream_t)stream, w, g, m, v, n, lr, b1, b2, eps, bc1,
                       bc2, gscale, (unsigned short *)wbf);
    return launch_status();
}

int srf_cnn_features(const float *em_int, const float *mu_int, const float *extra, int64_t n, const float *scale,
                     void *x, void *stream)
{
    if (!em_int || !mu_int || !scale || !x || n < 0) return SRF_ERR_INVALID_ARG;
    if (reinterpret_cast<uintptr_t>(x) & 7) return SRF_ERR_INVALID_ARG;
    if (n == 0) return SRF_OK;
    hipLaunchKernelGGL(k_features, dim3(nblk(n)), dim3(256), 0, (hipStream_t)stream, em_int, mu_int, extra, n,
                       scale, (unsigned short *)x);
    return launch_status();
}

int srf_cnn_cast(const void *x, int64_t n, int32_t to_bf16, void *y, void *stream)
{
    if (!x || !y || n < 0) return SRF_ERR_INVALID_ARG;
    if (to_bf16)
        hipLaunchKernelGGL(k_f32_to_bf16, dim3(nblk(n)), dim3(256), 0, (hipStream_t)stream, (const float *)x, n,
                           (unsigned short *)y);
    else
        hipLaunchKernelGGL(k_bf16_to_f32, dim3(nblk(n)), dim3(256), 0, (hipStream_t)stream,
                           (const unsigned short *)x, n, (float *)y);
    return launch_status();
}

}  // extern "C"
