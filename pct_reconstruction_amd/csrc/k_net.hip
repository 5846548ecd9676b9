// k_net.hip — learned warm start: a 4-level 3D U-Net mapping (FBP image, hull mask) to the DROP
// initial iterate x0, with its training (forward, backward, Adam) in hand-written gfx950 kernels.
//
// The reference has no learned component; its x0 is FBP, the hull, or their product
// (define_initial_iterate, DS.cu:8612-8646).  The net predicts a correction y to the FBP image and
// x0 = hull * (FBP + y), so a zero head reproduces the reference's hybrid x0.  DROP still defines the
// final image, and pct_net_apply keeps the FBP start when the net's x0 has the larger data residual.
//
// Network (channels 16-32-64-128, 3x3x3 convolutions, "same" zero padding):
//   enc1  conv(in8 -> 16)                       r0      in8 = (FBP, hull, 6 zero channels)
//   enc2  conv(avgpool(enc1) -> 32)             r0/2
//   enc3  conv(avgpool(enc2) -> 64)             r0/4
//   enc4  conv(avgpool(enc3) -> 128)            r0/8
//   dec3  conv(concat(up(enc4), enc3) -> 64)    r0/4    up = nearest x2, fused into the conv loader
//   dec2  conv(concat(up(dec3), enc2) -> 32)    r0/2
//   dec1  conv(concat(up(dec2), enc1) -> 16)    r0
//   head  1x1x1 conv(dec1 -> 1), linear
// ReLU after every 3x3x3 convolution.  Loss: mean over hull voxels of (x0 - target)^2.
//
// Numerics: BF16 weights and activations (round to nearest even), FP32 accumulation on MFMA
// (v_mfma_f32_16x16x32_bf16), FP32 master weights, gradients of weights in FP32, Adam in FP32.
// Layout: NDHWC (channels innermost) so a lane's 8 consecutive input channels are one 16-byte load.
// Convolution as implicit GEMM: M = voxels, N = output channels, K = 27 * input channels
// (k = tap * Cin + c, tap = (dz+1)*9 + (dy+1)*3 + (dx+1)), padded to a multiple of 64.
// Backward data = the same forward kernel over the masked output gradient with the taps flipped and
// the channel roles swapped.  Weight gradients: LDS-staged MFMA over 32-voxel slices, split over
// voxel chunks into FP32 partials that a second kernel sums in chunk order (deterministic).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

#include "internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kBlock = 256;
constexpr int kLayers = 7;  // 3x3x3 convolutions; the head is separate

__device__ __forceinline__ uint16_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)0x7fc0;  // NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ uint4 ld16(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// Input of a 3x3x3 convolution: channels [0, ca) from tensor a (at half resolution when a_coarse:
// nearest-neighbour upsampling), channels [ca, ca + cb) from tensor b at full resolution.
struct ConvIn {
    const uint16_t* a;
    const uint16_t* b;
    int ca, cb, a_coarse;
};

// 8 consecutive input channels [c, c+8) of voxel (z, y, x) of a D x H x W grid (zeros outside)
__device__ __forceinline__ uint4 load_in8(const ConvIn& in, int D, int H, int W, int z, int y, int x, int c)
{
    uint4 r = make_uint4(0, 0, 0, 0);
    if (z < 0 || y < 0 || x < 0 || z >= D || y >= H || x >= W) return r;
    if (c < in.ca) {
        if (in.a_coarse) {
            const int h2 = H >> 1, w2 = W >> 1;
            r = ld16(in.a + ((((int64_t)(z >> 1) * h2 + (y >> 1)) * w2 + (x >> 1)) * in.ca + c));
        } else {
            r = ld16(in.a + (((int64_t)z * H + y) * W + x) * in.ca + c);
        }
    } else {
        r = ld16(in.b + (((int64_t)z * H + y) * W + x) * in.cb + (c - in.ca));
    }
    return r;
}

// 3x3x3 convolution (forward, and backward data with flipped weights).  A workgroup takes an output tile of
// 16 (x) x ty x tz voxels: it loads the tile's input halo (all Cin channels, zeros outside the grid) into LDS once.
// Its four waves are 4 / wn groups of rows by wn groups of output channels; a wave computes RW rows of 16 voxels x
// 16 NT channels, so that an input fragment from LDS serves NT matrix products and a weight fragment from the caches
// RW.  Each output's products are accumulated in the order of k = tap * Cin + c, 32 to an instruction, whatever the
// tile: the values do not depend on the shape.
// The weights are the first operand: a lane then holds four consecutive output channels of one voxel.
// A voxel's channels are padded in LDS to an odd number of 16-byte units, so that the 16 voxels of a fragment lie in
// different banks.  The LDS offsets of the k groups come from a table (no division in the loop), and the fragments of
// kSteps k steps are read ahead of their products.
// Bound by the LDS reads of the input fragments where there are 16 or 32 output channels, by the matrix cores at 48
// and more.  The seven layers on 128 x 128 x 32: 732 us before (weights fetched row by row for every step, divisions
// in the loop, 128 workgroups without a halo at 192 channels), 140 now; 48 -> 16 channels on 256 x 256 x 96 1.6 ms,
// now 0.70 (0.24 at the card's matrix rate), 16 -> 48 0.48.
constexpr int kTileX = 16, kHaloX = kTileX + 2, kSteps = 4;

struct ConvShape {
    int ty, tz, wn;
    int stride;                    // 16-byte units per voxel in LDS
    int row_units, row_q, row_r;   // 16-byte loads of a halo row, and kBlock split by them
    uint32_t by_groups, by_hy;     // reciprocals, 16 bits of fraction
};

// Wt: bf16 [k step of 32][16 output channels][lane][8] (k_pack_weights); bias may be null
template <int RW, int NT>
__global__ void __launch_bounds__(kBlock) k_conv(ConvIn in, int D, int H, int W, ConvShape sh,
                                                 const uint16_t* __restrict__ Wt, const float* __restrict__ bias, int relu,
                                                 uint16_t* __restrict__ out)
{
    extern __shared__ uint4 lds[];
    const int Cin = in.ca + in.cb, groups = Cin / 8, ngroups = 27 * groups, steps = (ngroups + 3) / 4;
    const int tab_units = (steps * 4 + 4 * kSteps + 3) / 4;  // 16-byte units
    uint32_t* tab = reinterpret_cast<uint32_t*>(lds);
    uint4* halo = lds + tab_units;
    const int HY = sh.ty + 2, HZ = sh.tz + 2;
    const int tx = blockIdx.x * kTileX, ty = blockIdx.y * sh.ty, tz = blockIdx.z * sh.tz;
    for (int q = threadIdx.x; q < 4 * tab_units; q += kBlock) {
        const int tap = q / groups, c = q - tap * groups;
        tab[q] = q < ngroups ? (uint32_t)(((tap / 9 * HY + tap / 3 % 3) * kHaloX + tap % 3) * sh.stride + c) : 0u;
    }
    {
        // thread -> 16-byte units t, t + kBlock, ... of the halo, in (row, x, channel group) order
        const int rows = HY * HZ;
        int row = (int)threadIdx.x / sh.row_units, rem = (int)threadIdx.x - row * sh.row_units;
        constexpr int kAhead = 4;
        while (row < rows) {
            uint4 v[kAhead];
            int at[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                at[u] = -1;
                if (row < rows) {
                    const int hx = (int)(((uint32_t)rem * sh.by_groups) >> 16), cg = rem - hx * groups;
                    const int hz = (int)(((uint32_t)row * sh.by_hy) >> 16), hy = row - hz * HY;
                    at[u] = (row * kHaloX + hx) * sh.stride + cg;
                    v[u] = load_in8(in, D, H, W, tz + hz - 1, ty + hy - 1, tx + hx - 1, cg * 8);
                }
                row += sh.row_q;
                rem += sh.row_r;
                if (rem >= sh.row_units) {
                    rem -= sh.row_units;
                    row++;
                }
            }
#pragma unroll
            for (int u = 0; u < kAhead; u++)
                if (at[u] >= 0) halo[at[u]] = v[u];
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, i = lane & 15;
    const int wn = wave % sh.wn, wm = wave / sh.wn;
    const int ntiles = NT * sh.wn, Cout = 16 * ntiles;
    const uint4* rows[RW];
    f32x4 acc[RW][NT];
#pragma unroll
    for (int rr = 0; rr < RW; rr++) {
        const int r = RW * wm + rr, rz = r / sh.ty, ry = r - rz * sh.ty;
        rows[rr] = halo + ((rz * HY + ry) * kHaloX + i) * sh.stride;
#pragma unroll
        for (int t = 0; t < NT; t++) acc[rr][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const uint4* wp = reinterpret_cast<const uint4*>(Wt) + (int64_t)(NT * wn) * 64 + lane;
    const int wstep = ntiles * 64;  // 16-byte units of the weights of one step
    uint32_t off[kSteps];
    uint4 w[kSteps][NT];
#pragma unroll
    for (int u = 0; u < kSteps; u++) {
        off[u] = tab[4 * u + g];
        const int s = u < steps ? u : steps - 1;
#pragma unroll
        for (int t = 0; t < NT; t++) w[u][t] = wp[(int64_t)s * wstep + t * 64];
    }
    const int full = ngroups / 4;  // steps without padding
    int s0 = 0;
    for (; s0 + kSteps <= full; s0 += kSteps) {
        uint4 a[kSteps][RW], wnext[kSteps][NT];
#pragma unroll
        for (int u = 0; u < kSteps; u++)
#pragma unroll
            for (int rr = 0; rr < RW; rr++) a[u][rr] = rows[rr][off[u]];
#pragma unroll
        for (int u = 0; u < kSteps; u++) {
            off[u] = tab[4 * (s0 + kSteps + u) + g];
            const int s = s0 + kSteps + u < steps ? s0 + kSteps + u : steps - 1;
#pragma unroll
            for (int t = 0; t < NT; t++) wnext[u][t] = wp[(int64_t)s * wstep + t * 64];
        }
#pragma unroll
        for (int u = 0; u < kSteps; u++)
#pragma unroll
            for (int rr = 0; rr < RW; rr++)
#pragma unroll
                for (int t = 0; t < NT; t++)
                    acc[rr][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(w[u][t]), as_bf16x8(a[u][rr]), acc[rr][t], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < kSteps; u++)
#pragma unroll
            for (int t = 0; t < NT; t++) w[u][t] = wnext[u][t];
    }
#pragma unroll
    for (int u = 0; u < kSteps; u++) {
        if (s0 + u >= steps) break;
        const bool in_k = 4 * (s0 + u) + g < ngroups;
#pragma unroll
        for (int rr = 0; rr < RW; rr++) {
            uint4 a = rows[rr][off[u]];
            a.x = in_k ? a.x : 0u;
            a.y = in_k ? a.y : 0u;
            a.z = in_k ? a.z : 0u;
            a.w = in_k ? a.w : 0u;
#pragma unroll
            for (int t = 0; t < NT; t++)
                acc[rr][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(w[u][t]), as_bf16x8(a), acc[rr][t], 0, 0, 0);
        }
    }
    // D[row][col]: lane holds channels 4g..4g+3 of voxel i
    const int x = tx + i;
    if (x >= W) return;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int co = 16 * (NT * wn + t) + 4 * g;
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (bias) {
#pragma unroll
            for (int r = 0; r < 4; r++) bv[r] = bias[co + r];
        }
#pragma unroll
        for (int rr = 0; rr < RW; rr++) {
            const int r = RW * wm + rr, rz = r / sh.ty, y = ty + (r - rz * sh.ty), z = tz + rz;
            if (y >= H || z >= D) continue;
            uint32_t e[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float v = acc[rr][t][q] + bv[q];
                if (relu) v = v > 0.0f ? v : 0.0f;
                e[q] = f2bf(v);
            }
            *reinterpret_cast<uint2*>(out + (((int64_t)z * H + y) * W + x) * Cout + co) =
                make_uint2(e[0] | e[1] << 16, e[2] | e[3] << 16);
        }
    }
}

// Weight gradient partials: partial[chunk][co][k] = sum over the chunk's voxels v of A[v][k] * G[v][co], A the
// convolution input gathered as in the forward pass, G = dL/d(pre-ReLU); entry k = K is the sum of G[v][co], the bias
// gradient.  The contraction runs over voxels, so a lane's eight elements are eight voxels of one channel: a tile of
// 16 x kGY x kGZ voxels is transposed into LDS, channel by channel, rows along x.  A workgroup takes 16 input channels
// (blockIdx.y) and 16 NT output channels (blockIdx.z) over a chunk of tiles (blockIdx.x); its three waves take the taps'
// three dz.  An input row read once serves its three dx: dx = 0 and 2 are whole registers of it, dx = 1 a shift by 16
// bits.  Channels lie an odd number of 16-byte units apart, so that the fragment reads are free of bank conflicts.
// Bound by the staging (two 16-byte loads and eight 4-byte LDS writes for each 16 elements) at 16 and 32 output
// channels.  On 128 x 128 x 32 the seven layers take 275 us; one 64-wide slice of k per workgroup, staged element by
// element for one product per wave and barrier, took 1680, and the bias gradients apart another 1730.
constexpr int kGY = 8, kGZ = 2, kGRows = kGY * kGZ, kGBlock = 192;
constexpr int kGHalo = (kGY + 2) * (kGZ + 2);
constexpr int kGInStride = kGHalo * 12 + 4, kGOutStride = kGRows * 8 + 4;  // 4-byte words per channel
static_assert((kGInStride / 4) % 2 == 1 && (kGOutStride / 4) % 2 == 1, "channels in different banks");

// 8 channels of two voxels into rows of 8 channels, 4 bytes each
__device__ __forceinline__ void put_pair(uint32_t* at, int stride, uint4 a, uint4 b)
{
    const uint32_t va[4] = {a.x, a.y, a.z, a.w}, vb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        at[(2 * j) * stride] = (va[j] & 0xffffu) | vb[j] << 16;
        at[(2 * j + 1) * stride] = va[j] >> 16 | (vb[j] & 0xffff0000u);
    }
}

template <int NT>
__global__ void __launch_bounds__(kGBlock) k_conv_wgrad(ConvIn in, int D, int H, int W, const uint16_t* __restrict__ G,
                                                        int Cout, int tiles_x, int tiles_y, int tiles, int per_chunk,
                                                        float* __restrict__ partial)
{
    __shared__ __align__(16) uint32_t As[16 * kGInStride];
    __shared__ __align__(16) uint32_t Gs[16 * NT * kGOutStride];
    const int Cin = in.ca + in.cb, K = 27 * Cin, Kq = K + 4;
    const int c0 = 16 * blockIdx.y, co0 = 16 * NT * blockIdx.z, cgs = min(Cin - c0, 16) / 8;
    const int lane = threadIdx.x & 63, dz = threadIdx.x >> 6, g = lane >> 4, i = lane & 15;
    const int ic = cgs == 1 ? i & 7 : i;  // the rows of 8 missing channels are not written
    const bool bias = dz == 0 && blockIdx.y == 0;
    const bf16x8 ones = as_bf16x8(make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
    f32x4 acc[3][3][NT], accb[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        accb[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < 9; q++) acc[q / 3][q % 3][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int t0 = blockIdx.x * per_chunk, t1 = min(t0 + per_chunk, tiles);
    for (int tile = t0; tile < t1; tile++) {
        const int tx = tile % tiles_x * 16, ty = tile / tiles_x % tiles_y * kGY, tz = tile / (tiles_x * tiles_y) * kGZ;
        __syncthreads();
        for (int q = threadIdx.x; q < cgs * kGHalo * 9; q += kGBlock) {
            const int cg = q / (kGHalo * 9), r = q - cg * (kGHalo * 9), row = r / 9, p = r - row * 9;
            const int z = tz + row / (kGY + 2) - 1, y = ty + row % (kGY + 2) - 1, x = tx + 2 * p - 1, c = c0 + 8 * cg;
            const uint4 a = load_in8(in, D, H, W, z, y, x, c), b = load_in8(in, D, H, W, z, y, x + 1, c);
            put_pair(As + 8 * cg * kGInStride + row * 12 + p, kGInStride, a, b);
        }
        for (int q = threadIdx.x; q < 2 * NT * kGRows * 8; q += kGBlock) {
            const int cg = q / (kGRows * 8), row = q / 8 % kGRows, p = q & 7;
            const int z = tz + row / kGY, y = ty + row % kGY, x = tx + 2 * p;
            uint4 a = make_uint4(0, 0, 0, 0), b = a;
            if (z < D && y < H) {
                const uint16_t* src = G + (((int64_t)z * H + y) * W + x) * Cout + co0 + 8 * cg;
                if (x < W) a = ld16(src);
                if (x + 1 < W) b = ld16(src + Cout);
            }
            put_pair(Gs + 8 * cg * kGOutStride + row * 8 + p, kGOutStride, a, b);
        }
        __syncthreads();
#pragma unroll 2
        for (int s = 0; s < kGRows / 2; s++) {
            // the contraction's 32 voxels: two rows of 16, a lane's eight in row r from x = 8 (g & 1) on
            const int r = 2 * s + (g >> 1), ry = r % kGY, rz = r / kGY;
            bf16x8 b[NT];
#pragma unroll
            for (int t = 0; t < NT; t++)
                b[t] = as_bf16x8(*reinterpret_cast<const uint4*>(Gs + (16 * t + i) * kGOutStride + r * 8 + 4 * (g & 1)));
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
                const uint32_t* src = As + ic * kGInStride + ((rz + dz) * (kGY + 2) + ry + dy) * 12 + 4 * (g & 1);
                const uint4 d = *reinterpret_cast<const uint4*>(src);
                const uint32_t e = src[4];
                const uint4 a1 = make_uint4(__builtin_amdgcn_alignbit(d.y, d.x, 16), __builtin_amdgcn_alignbit(d.z, d.y, 16),
                                            __builtin_amdgcn_alignbit(d.w, d.z, 16), __builtin_amdgcn_alignbit(e, d.w, 16));
                const uint4 a2 = make_uint4(d.y, d.z, d.w, e);
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    acc[dy][0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(d), b[t], acc[dy][0][t], 0, 0, 0);
                    acc[dy][1][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a1), b[t], acc[dy][1][t], 0, 0, 0);
                    acc[dy][2][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a2), b[t], acc[dy][2][t], 0, 0, 0);
                }
            }
            if (bias) {
#pragma unroll
                for (int t = 0; t < NT; t++)
                    accb[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, b[t], accb[t], 0, 0, 0);
            }
        }
    }
    // D[c][co]: lane holds channels 4g..4g+3 of column co
    float* P = partial + (int64_t)blockIdx.x * Cout * Kq;
#pragma unroll
    for (int t = 0; t < NT; t++) {
        float* row = P + (int64_t)(co0 + 16 * t + i) * Kq;
        if (8 * cgs > 4 * g) {
#pragma unroll
            for (int q = 0; q < 9; q++)
                *reinterpret_cast<f32x4*>(row + (9 * dz + q) * Cin + c0 + 4 * g) = acc[q / 3][q % 3][t];
        }
        if (bias && g == 0) row[K] = accb[t][0];
    }
}

// grad[co][k] (k < K), then the bias gradients: sums over chunks of partial[chunk][co][k], in chunk order
__global__ void k_reduce_partials(int nchunks, int Cout, int K, const float* __restrict__ partial,
                                  float* __restrict__ grad)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)Cout * (K + 1)) return;
    const int co = (int)(idx / (K + 1)), k = (int)(idx % (K + 1)), Kq = K + 4;
    const float* p = partial + (int64_t)co * Kq + k;
    const int64_t step = (int64_t)Cout * Kq;
    float s = 0.0f;
    int c = 0;
    for (; c + 8 <= nchunks; c += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = p[(c + u) * step];
#pragma unroll
        for (int u = 0; u < 8; u++) s += v[u];
    }
    for (; c < nchunks; c++) s += p[c * step];
    grad[k < K ? (int64_t)co * K + k : (int64_t)Cout * K + co] = s;
}

// k index and output channel of element idx of a weight array in fragment order: [k step][ntiles][lane][8]
__device__ __forceinline__ void frag_index(int64_t idx, int ntiles, int* co, int* k)
{
    const int j = (int)(idx & 7), lane = (int)(idx >> 3) & 63;
    const int64_t f = idx >> 9;
    *co = 16 * (int)(f % ntiles) + (lane & 15);
    *k = 32 * (int)(f / ntiles) + 8 * (lane >> 4) + j;
}

// master [Cout][27][Cin] fp32 -> bf16 fragments of the forward weights (k = tap * Cin + c) and of the flipped ones
// (k' = tap' * Cout + co, tap' = 26 - tap, output channels Cin), zeros beyond K.  An input of 8 channels has no
// flipped weights: its gradient is not formed.
__global__ void k_pack_weights(const float* __restrict__ w, int Cin, int Cout, int Kp, int Kpf,
                               uint16_t* __restrict__ wt, uint16_t* __restrict__ wf)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n1 = (int64_t)Cout * Kp, n2 = Cin % 16 ? 0 : (int64_t)Cin * Kpf;
    int co, k;
    if (idx < n1) {
        frag_index(idx, Cout / 16, &co, &k);
        wt[idx] = k < 27 * Cin ? f2bf(w[(int64_t)co * 27 * Cin + k]) : (uint16_t)0;
    } else if (idx < n1 + n2) {
        int c;
        frag_index(idx - n1, Cin / 16, &c, &k);
        uint16_t v = 0;
        if (k < 27 * Cout) {
            const int tapf = k / Cout, o = k % Cout;
            v = f2bf(w[((int64_t)o * 27 + (26 - tapf)) * Cin + c]);
        }
        wf[idx - n1] = v;
    }
}

// in8 = (FBP, hull, 0...) as bf16
__global__ void k_pack_input(int64_t nvox, const float* __restrict__ fbp, const uint8_t* __restrict__ hull,
                             uint16_t* __restrict__ in8)
{
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nvox) return;
    uint16_t e[8] = {f2bf(fbp[v]), f2bf(hull[v] ? 1.0f : 0.0f), 0, 0, 0, 0, 0, 0};
    *reinterpret_cast<uint4*>(in8 + v * 8) = *reinterpret_cast<const uint4*>(e);
}

// 2x2x2 average pooling; out dims D/2 x H/2 x W/2
__global__ void k_avgpool(int D, int H, int W, int C, const uint16_t* __restrict__ in, uint16_t* __restrict__ out)
{
    const int64_t n = (int64_t)(D / 2) * (H / 2) * (W / 2) * C;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const int c = (int)(idx % C);
    const int64_t p = idx / C;
    const int w2 = W / 2, h2 = H / 2;
    const int x = (int)(p % w2), y = (int)((p / w2) % h2), z = (int)(p / ((int64_t)w2 * h2));
    float s = 0.0f;
    for (int dz = 0; dz < 2; dz++)
        for (int dy = 0; dy < 2; dy++)
            for (int dx = 0; dx < 2; dx++)
                s += bf2f(in[(((int64_t)(2 * z + dz) * H + (2 * y + dy)) * W + (2 * x + dx)) * C + c]);
    out[idx] = f2bf(s * 0.125f);
}

// dPre[v][c] = act[v][c] > 0 ? skip_grad[v][c_off + c] + (pool_grad ? pool_grad[parent][c] / 8 : 0) : 0
// skip_grad is the concat gradient at full resolution with cs channels (this tensor at offset c_off).
__global__ void k_merge_grad(int D, int H, int W, int C, const uint16_t* __restrict__ act,
                             const uint16_t* __restrict__ skip_grad, int cs, int c_off,
                             const uint16_t* __restrict__ pool_grad, uint16_t* __restrict__ dpre)
{
    const int64_t n = (int64_t)D * H * W * C;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const int c = (int)(idx % C);
    const int64_t v = idx / C;
    float gsum = bf2f(skip_grad[v * cs + c_off + c]);
    if (pool_grad) {
        const int x = (int)(v % W), y = (int)((v / W) % H), z = (int)(v / ((int64_t)W * H));
        const int64_t p = ((int64_t)(z >> 1) * (H >> 1) + (y >> 1)) * (W >> 1) + (x >> 1);
        gsum += bf2f(pool_grad[p * C + c]) * 0.125f;
    }
    dpre[idx] = bf2f(act[idx]) > 0.0f ? f2bf(gsum) : (uint16_t)0;
}

// Gradient of a coarse tensor that was upsampled into channels [0, C) of a concat at full resolution
// (cs channels): dPre[p][c] = act[p][c] > 0 ? sum over the 8 children of cat_grad[child][c] : 0
__global__ void k_up_grad(int D, int H, int W, int C, int cs, const uint16_t* __restrict__ cat_grad,
                          const uint16_t* __restrict__ act, uint16_t* __restrict__ dpre)
{
    const int64_t n = (int64_t)(D / 2) * (H / 2) * (W / 2) * C;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const int c = (int)(idx % C);
    const int64_t p = idx / C;
    const int w2 = W / 2, h2 = H / 2;
    const int x = (int)(p % w2), y = (int)((p / w2) % h2), z = (int)(p / ((int64_t)w2 * h2));
    float s = 0.0f;
    for (int dz = 0; dz < 2; dz++)
        for (int dy = 0; dy < 2; dy++)
            for (int dx = 0; dx < 2; dx++)
                s += bf2f(cat_grad[(((int64_t)(2 * z + dz) * H + (2 * y + dy)) * W + (2 * x + dx)) * cs + c]);
    dpre[idx] = bf2f(act[idx]) > 0.0f ? f2bf(s) : (uint16_t)0;
}

// head: y = w . d1 + b; x0 = hull ? FBP + y : 0; per-block partial sums of the masked squared error
// and of the hull count
__global__ void k_head_fwd(int64_t nvox, const uint16_t* __restrict__ d1, const float* __restrict__ wh,
                           const float* __restrict__ fbp, const uint8_t* __restrict__ hull,
                           const float* __restrict__ target, float* __restrict__ x0, double* __restrict__ part)
{
    __shared__ double s_err[kBlock], s_cnt[kBlock];
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    double e = 0.0, c = 0.0;
    if (v < nvox) {
        const uint4 q0 = ld16(d1 + v * 16), q1 = ld16(d1 + v * 16 + 8);
        const uint16_t* a = reinterpret_cast<const uint16_t*>(&q0);
        const uint16_t* b = reinterpret_cast<const uint16_t*>(&q1);
        float y = wh[16];
#pragma unroll
        for (int j = 0; j < 8; j++) y += wh[j] * bf2f(a[j]);
#pragma unroll
        for (int j = 0; j < 8; j++) y += wh[8 + j] * bf2f(b[j]);
        const float xv = hull[v] ? fbp[v] + y : 0.0f;
        x0[v] = xv;
        if (target && hull[v]) {
            const double d = (double)xv - (double)target[v];
            e = d * d;
            c = 1.0;
        }
    }
    s_err[threadIdx.x] = e;
    s_cnt[threadIdx.x] = c;
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            s_err[threadIdx.x] += s_err[threadIdx.x + o];
            s_cnt[threadIdx.x] += s_cnt[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = s_err[0];
        part[2 * blockIdx.x + 1] = s_cnt[0];
    }
}

// head backward: dy = 2 (x0 - t) / n_hull on hull voxels; dPre_dec1[v][c] = d1 > 0 ? dy * w[c] : 0;
// per-block partials of dw[c] = sum dy * d1[v][c] and db = sum dy
__global__ void k_head_bwd(int64_t nvox, double inv_n, const uint16_t* __restrict__ d1, const float* __restrict__ wh,
                           const uint8_t* __restrict__ hull, const float* __restrict__ x0,
                           const float* __restrict__ target, uint16_t* __restrict__ dpre, float* __restrict__ part)
{
    __shared__ float s[17][kBlock];
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float dy = 0.0f;
    float a[16];
#pragma unroll
    for (int j = 0; j < 16; j++) a[j] = 0.0f;
    if (v < nvox) {
        const uint4 q0 = ld16(d1 + v * 16), q1 = ld16(d1 + v * 16 + 8);
        const uint16_t* p0 = reinterpret_cast<const uint16_t*>(&q0);
        const uint16_t* p1 = reinterpret_cast<const uint16_t*>(&q1);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            a[j] = bf2f(p0[j]);
            a[8 + j] = bf2f(p1[j]);
        }
        if (hull[v]) dy = (float)(2.0 * ((double)x0[v] - (double)target[v]) * inv_n);
        uint16_t o[16];
#pragma unroll
        for (int j = 0; j < 16; j++) o[j] = a[j] > 0.0f ? f2bf(dy * wh[j]) : (uint16_t)0;
        *reinterpret_cast<uint4*>(dpre + v * 16) = *reinterpret_cast<const uint4*>(o);
        *reinterpret_cast<uint4*>(dpre + v * 16 + 8) = *reinterpret_cast<const uint4*>(o + 8);
    }
#pragma unroll
    for (int j = 0; j < 16; j++) s[j][threadIdx.x] = dy * a[j];
    s[16][threadIdx.x] = dy;
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o)
            for (int j = 0; j < 17; j++) s[j][threadIdx.x] += s[j][threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x < 17) part[(int64_t)blockIdx.x * 17 + threadIdx.x] = s[threadIdx.x][0];
}
// out[c] = sum over rows of part[row][c]; one workgroup per column (one lane per column took 577 us for 2048 rows)
__global__ void __launch_bounds__(kBlock) k_reduce_cols(int nrows, int ncols, const float* __restrict__ part,
                                                        float* __restrict__ out)
{
    __shared__ float s[kBlock];
    float v = 0.0f;
    for (int r = threadIdx.x; r < nrows; r += kBlock) v += part[(int64_t)r * ncols + blockIdx.x];
    s[threadIdx.x] = v;
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = s[0];
}

__global__ void k_adam(int64_t n, float lr, float b1, float b2, float eps, float c1, float c2,
                       float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

inline unsigned blocks_for(int64_t n, int b = kBlock) { return pct_grid_for(n, b); }

}  // namespace

// ------------------------------------------------------------------------------------ host side
struct pct_net {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    int D = 0, H = 0, W = 0;  // slices, rows, columns at full resolution
    int64_t nv[4] = {};       // voxels per level
    struct Layer {
        int cin, cout, level, Kp, Kpf;
        int64_t w_off, b_off;
        uint16_t* wt = nullptr;
        uint16_t* wf = nullptr;
    } L[kLayers];
    int64_t head_off = 0, n_params = 0;
    float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
    int64_t adam_t = 0;
    // activations (bf16)
    uint16_t *in8 = nullptr, *e[4] = {}, *pool[3] = {}, *dd[3] = {};  // dd[0] = dec1, dd[1] = dec2, dd[2] = dec3
    float* x0 = nullptr;
    // gradients (bf16)
    uint16_t *g_dd[3] = {}, *g_cat[3] = {}, *g_e[4] = {}, *g_pool[3] = {};
    float* partial = nullptr;
    int64_t partial_n = 0;
    double* loss_part = nullptr;
    float* head_part = nullptr;
    // scratch input / target (device)
    float *fbp = nullptr, *target = nullptr;
    uint8_t* hull = nullptr;
    struct Sample {
        float* fbp;
        uint8_t* hull;
        float* target;
    };
    std::vector<Sample> samples;
};

namespace {

#define NET_HIP(net, expr)                                                        \
    do {                                                                          \
        hipError_t e_ = (expr);                                                   \
        if (e_ != hipSuccess) {                                                   \
            (net)->err = std::string(#expr) + ": " + hipGetErrorString(e_);       \
            return PCT_E_HIP;                                                     \
        }                                                                         \
    } while (0)

template <class T>
int net_alloc(pct_net* net, T** ptr, int64_t n)
{
    if (hipMalloc((void**)ptr, (size_t)(n > 0 ? n : 1) * sizeof(T)) != hipSuccess) {
        net->err = "hipMalloc failed (" + std::to_string(n * sizeof(T)) + " B)";
        *ptr = nullptr;
        return PCT_E_NOMEM;
    }
    return PCT_OK;
}
template <class T>
void net_free(T** ptr)
{
    if (*ptr) (void)hipFree(*ptr);
    *ptr = nullptr;
}

// deterministic normal numbers (splitmix64 + Box-Muller)
struct Rng {
    uint64_t s;
    uint64_t next()
    {
        uint64_t z = (s += 0x9e3779b97f4a7c15ull);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        return z ^ (z >> 31);
    }
    double uniform() { return ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0); }
    double normal() { return std::sqrt(-2.0 * std::log(uniform())) * std::cos(6.283185307179586 * uniform()); }
};

int pack_weights(pct_net* net)
{
    for (int l = 0; l < kLayers; l++) {
        auto& Ly = net->L[l];
        const int64_t n = (int64_t)Ly.cout * Ly.Kp + (int64_t)Ly.cin * Ly.Kpf;
        hipLaunchKernelGGL(k_pack_weights, dim3(blocks_for(n)), dim3(kBlock), 0, net->stream, net->p + Ly.w_off, Ly.cin,
                           Ly.cout, Ly.Kp, Ly.Kpf, Ly.wt, Ly.wf);
    }
    NET_HIP(net, hipGetLastError());
    return PCT_OK;
}

// The tile of a convolution and what its kernel derives from it.
ConvShape conv_shape(int cin, int wn, int rw, int ty, size_t* lds)
{
    ConvShape sh{};
    sh.ty = ty;
    sh.tz = rw * (4 / wn) / ty;
    sh.wn = wn;
    const int groups = cin / 8;
    sh.stride = groups | 1;
    sh.row_units = kHaloX * groups;
    sh.row_q = kBlock / sh.row_units;
    sh.row_r = kBlock % sh.row_units;
    sh.by_groups = 65536u / groups + 1;  // exact for x < row_units (at most 432) and rows of a halo
    sh.by_hy = 65536u / (ty + 2) + 1;
    const int steps = (27 * groups + 3) / 4;
    *lds = 16 * ((size_t)(steps * 4 + 4 * kSteps + 3) / 4 + (size_t)kHaloX * (ty + 2) * (sh.tz + 2) * sh.stride);
    return sh;
}

template <int RW, int NT>
int launch_conv_as(pct_net* net, const ConvIn& in, int level, const ConvShape& sh, size_t lds, const uint16_t* w,
                   const float* bias, int relu, uint16_t* out)
{
    const int D = net->D >> level, H = net->H >> level, W = net->W >> level;
    const dim3 grid((W + kTileX - 1) / kTileX, (H + sh.ty - 1) / sh.ty, (D + sh.tz - 1) / sh.tz);
    if (lds > 64 * 1024)
        NET_HIP(net, hipFuncSetAttribute((const void*)k_conv<RW, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_conv<RW, NT>), grid, dim3(kBlock), lds, net->stream, in, D, H, W, sh, w, bias, relu, out);
    NET_HIP(net, hipGetLastError());
    return PCT_OK;
}

// The tile's rule.  More rows per wave use a weight fragment more often, and fewer waves along the channels an input
// fragment; both need rows, so fewer workgroups and a larger halo.  In order of rows per wave, and with the channels
// of 32 and 64 first on fewer waves, the first shape is taken that needs at most 64 KB of LDS, so that two or three
// workgroups share a compute unit, and has 384 workgroups; a halo of 192 channels needs more than that at any useful
// size and may take 160 KB.  Measured (us, taken | next): on 256 x 256 x 96, 48 -> 16 channels 8 rows in
// 47 KB 698 | 16 rows in 71 KB 738; 96 -> 32 at half size 4 rows in 59 KB 293 | 8 in 89 KB 380; 192 -> 64 at a quarter
// 4 rows in 115 KB 160 | 1 in 65 KB 205; 32 -> 64 there 8 rows, 768 workgroups 18.0 | 4 rows 19.9; on 128 x 128 x 32,
// 16 -> 32 at half size 8 rows, 512 workgroups 7.7 | 16 rows, 256 workgroups 9.5.
int launch_conv(pct_net* net, const ConvIn& in, int level, const uint16_t* w, const float* bias, int relu, int cout,
                uint16_t* out)
{
    const int tiles = cout / 16, cin = in.ca + in.cb;
    const int64_t D = net->D >> level, H = net->H >> level, W = net->W >> level;
    struct Split {
        int nt, wn;
    } split[2];
    int n_split = 0;
    for (int wn = 1; wn <= 4; wn *= 2)
        if (tiles % wn == 0 && tiles / wn <= 3 && n_split < 2) split[n_split++] = Split{tiles / wn, wn};
    if (cout % 16 || n_split == 0) {
        net->err = "unsupported channel count";
        return PCT_E_ARG;
    }
    int rw = 1, nt = split[n_split - 1].nt, wn = split[n_split - 1].wn;  // the most workgroups, if none is taken
    int ty = wn == 4 ? 1 : 2;
    bool found = false;
    for (const size_t room : {(size_t)64 << 10, (size_t)160 << 10})
        for (int r = 4; r >= 1 && !found; r /= 2)
            for (int k = 0; k < n_split && !found; k++) {
                const int rows = r * 4 / split[k].wn, t = rows >= 8 ? 4 : rows >= 2 ? 2 : 1;
                size_t lds = 0;
                const ConvShape sh = conv_shape(cin, split[k].wn, r, t, &lds);
                const int64_t groups = (W + kTileX - 1) / kTileX * ((H + t - 1) / t) * ((D + sh.tz - 1) / sh.tz);
                if (lds > room || groups < 384) continue;
                rw = r;
                ty = t;
                nt = split[k].nt;
                wn = split[k].wn;
                found = true;
            }
    size_t lds = 0;
    const ConvShape sh = conv_shape(cin, wn, rw, ty, &lds);
#define PCT_CONV(RW, NT) \
    if (rw == RW && nt == NT) return launch_conv_as<RW, NT>(net, in, level, sh, lds, w, bias, relu, out);
    PCT_CONV(4, 1) PCT_CONV(4, 2) PCT_CONV(4, 3)
    PCT_CONV(2, 1) PCT_CONV(2, 2) PCT_CONV(2, 3)
    PCT_CONV(1, 1) PCT_CONV(1, 2) PCT_CONV(1, 3)
#undef PCT_CONV
    net->err = "unsupported channel count";
    return PCT_E_ARG;
}

// Split of a weight-gradient launch: about 768 workgroups (three of them fill a compute unit's matrix cores and hide
// each other's staging), with at most 32 MB of partial sums.
struct WgradShape {
    int nt, ctiles, groups, tiles_x, tiles_y, tiles, per_chunk, chunks;
    int64_t chunk_floats;
};
WgradShape wgrad_shape(const pct_net* net, int l)
{
    const auto& Ly = net->L[l];
    const int D = net->D >> Ly.level, H = net->H >> Ly.level, W = net->W >> Ly.level;
    WgradShape w{};
    w.nt = Ly.cout % 64 == 0 ? 4 : Ly.cout % 32 == 0 ? 2 : 1;
    w.ctiles = (Ly.cin + 15) / 16;
    w.groups = Ly.cout / (16 * w.nt);
    w.tiles_x = (W + 15) / 16;
    w.tiles_y = (H + kGY - 1) / kGY;
    w.tiles = w.tiles_x * w.tiles_y * ((D + kGZ - 1) / kGZ);
    w.chunk_floats = (int64_t)Ly.cout * (27 * Ly.cin + 4);
    const int64_t most = std::max<int64_t>(1, std::min<int64_t>(768 / (w.ctiles * w.groups), (8 << 20) / w.chunk_floats));
    w.per_chunk = (int)((w.tiles + most - 1) / most);
    w.chunks = (w.tiles + w.per_chunk - 1) / w.per_chunk;
    return w;
}

int launch_wgrad(pct_net* net, const ConvIn& in, int level, int l, const uint16_t* G)
{
    auto& Ly = net->L[l];
    const int D = net->D >> level, H = net->H >> level, W = net->W >> level;
    const WgradShape w = wgrad_shape(net, l);
    if (w.chunks * w.chunk_floats > net->partial_n) {
        net->err = "gradient scratch too small";
        return PCT_E_LIMIT;
    }
    hipStream_t s = net->stream;
    const dim3 grid((unsigned)w.chunks, (unsigned)w.ctiles, (unsigned)w.groups);
    auto kern = w.nt == 4 ? k_conv_wgrad<4> : w.nt == 2 ? k_conv_wgrad<2> : k_conv_wgrad<1>;
    hipLaunchKernelGGL(kern, grid, dim3(kGBlock), 0, s, in, D, H, W, G, Ly.cout, w.tiles_x, w.tiles_y, w.tiles, w.per_chunk,
                       net->partial);
    const int K = 27 * Ly.cin;
    // the bias gradients follow the weights' (b_off = w_off + cout * K)
    hipLaunchKernelGGL(k_reduce_partials, dim3(blocks_for((int64_t)Ly.cout * (K + 1))), dim3(kBlock), 0, s, w.chunks,
                       Ly.cout, K, net->partial, net->g + Ly.w_off);
    NET_HIP(net, hipGetLastError());
    return PCT_OK;
}

ConvIn conv_input(pct_net* net, int l)
{
    ConvIn in{};
    switch (l) {
    case 0: in = ConvIn{net->in8, nullptr, 8, 0, 0}; break;
    case 1: in = ConvIn{net->pool[0], nullptr, 16, 0, 0}; break;
    case 2: in = ConvIn{net->pool[1], nullptr, 32, 0, 0}; break;
    case 3: in = ConvIn{net->pool[2], nullptr, 64, 0, 0}; break;
    case 4: in = ConvIn{net->e[3], net->e[2], 128, 64, 1}; break;   // dec3
    case 5: in = ConvIn{net->dd[2], net->e[1], 64, 32, 1}; break;   // dec2
    default: in = ConvIn{net->dd[1], net->e[0], 32, 16, 1}; break;  // dec1
    }
    return in;
}

// forward pass from the device arrays fbp/hull; x0 (and the loss when target != null)
int net_forward(pct_net* net, const float* fbp, const uint8_t* hull, const float* target, double* loss)
{
    hipStream_t s = net->stream;
    const int64_t n0 = net->nv[0];
    hipLaunchKernelGGL(k_pack_input, dim3(blocks_for(n0)), dim3(kBlock), 0, s, n0, fbp, hull, net->in8);
    uint16_t* outs[kLayers] = {net->e[0], net->e[1], net->e[2], net->e[3], net->dd[2], net->dd[1], net->dd[0]};
    const int level[kLayers] = {0, 1, 2, 3, 2, 1, 0};
    for (int l = 0; l < kLayers; l++) {
        auto& Ly = net->L[l];
        PCT_TRY(launch_conv(net, conv_input(net, l), level[l], Ly.wt, net->p + Ly.b_off, 1, Ly.cout, outs[l]));
        if (l < 3) {
            const int D = net->D >> l, H = net->H >> l, W = net->W >> l;
            const int64_t n = (int64_t)(D / 2) * (H / 2) * (W / 2) * Ly.cout;
            hipLaunchKernelGGL(k_avgpool, dim3(blocks_for(n)), dim3(kBlock), 0, s, D, H, W, Ly.cout, outs[l], net->pool[l]);
        }
    }
    const unsigned nb = blocks_for(n0);
    hipLaunchKernelGGL(k_head_fwd, dim3(nb), dim3(kBlock), 0, s, n0, net->dd[0], net->p + net->head_off, fbp, hull, target,
                       net->x0, net->loss_part);
    NET_HIP(net, hipGetLastError());
    if (loss) {
        std::vector<double> part(2 * (size_t)nb);
        NET_HIP(net, hipMemcpyAsync(part.data(), net->loss_part, part.size() * sizeof(double), hipMemcpyDeviceToHost, s));
        NET_HIP(net, hipStreamSynchronize(s));
        double e = 0, c = 0;
        for (unsigned b = 0; b < nb; b++) {
            e += part[2 * b];
            c += part[2 * b + 1];
        }
        *loss = c > 0 ? e / c : 0.0;
    }
    return PCT_OK;
}

int hull_count(pct_net* net, double* cnt)
{
    const unsigned nb = blocks_for(net->nv[0]);
    std::vector<double> part(2 * (size_t)nb);
    NET_HIP(net, hipMemcpyAsync(part.data(), net->loss_part, part.size() * sizeof(double), hipMemcpyDeviceToHost,
                                net->stream));
    NET_HIP(net, hipStreamSynchronize(net->stream));
    double c = 0;
    for (unsigned b = 0; b < nb; b++) c += part[2 * b + 1];
    *cnt = c;
    return PCT_OK;
}

// backward pass after net_forward with a target: fills net->g
int net_backward(pct_net* net, const uint8_t* hull, const float* target)
{
    hipStream_t s = net->stream;
    const int64_t n0 = net->nv[0];
    double cnt = 0;
    PCT_TRY(hull_count(net, &cnt));
    const double inv_n = cnt > 0 ? 1.0 / cnt : 0.0;
    const unsigned nb = blocks_for(n0);
    hipLaunchKernelGGL(k_head_bwd, dim3(nb), dim3(kBlock), 0, s, n0, inv_n, net->dd[0], net->p + net->head_off, hull,
                       net->x0, target, net->g_dd[0], net->head_part);
    hipLaunchKernelGGL(k_reduce_cols, dim3(17), dim3(kBlock), 0, s, (int)nb, 17, net->head_part, net->g + net->head_off);
    // decoder: l = 6 (dec1, level 0), 5 (dec2, level 1), 4 (dec3, level 2)
    for (int d = 0; d < 3; d++) {
        const int l = 6 - d, level = d;
        auto& Ly = net->L[l];
        const ConvIn in = conv_input(net, l);
        PCT_TRY(launch_wgrad(net, in, level, l, net->g_dd[d]));
        // concat gradient: conv of dPre with flipped weights (Cin' = Cout, Cout' = Cin)
        ConvIn gin{net->g_dd[d], nullptr, Ly.cout, 0, 0};
        PCT_TRY(launch_conv(net, gin, level, Ly.wf, nullptr, 0, Ly.cin, net->g_cat[d]));
        const int D = net->D >> level, H = net->H >> level, W = net->W >> level;
        const int ca = in.ca;
        // coarse part -> dPre of the tensor one level down (dec2, dec3 or enc4)
        uint16_t* coarse_act = d < 2 ? net->dd[d + 1] : net->e[3];
        uint16_t* coarse_g = d < 2 ? net->g_dd[d + 1] : net->g_e[3];
        const int64_t nc = (int64_t)(D / 2) * (H / 2) * (W / 2) * ca;
        hipLaunchKernelGGL(k_up_grad, dim3(blocks_for(nc)), dim3(kBlock), 0, s, D, H, W, ca, Ly.cin, net->g_cat[d],
                           coarse_act, coarse_g);
    }
    // encoder: enc4 (l = 3) .. enc1 (l = 0); g_e[l] holds dPre of enc l+1
    for (int l = 3; l >= 0; l--) {
        auto& Ly = net->L[l];
        const int level = l;
        if (l < 3) {
            // dPre(enc l) = mask * (skip part of the decoder concat at this level + pool gradient)
            const int D = net->D >> level, H = net->H >> level, W = net->W >> level;
            const int d = level;  // decoder index consuming enc l as skip
            const int cs = net->L[6 - d].cin, c_off = net->L[6 - d].cin - Ly.cout;
            const int64_t n = (int64_t)D * H * W * Ly.cout;
            hipLaunchKernelGGL(k_merge_grad, dim3(blocks_for(n)), dim3(kBlock), 0, s, D, H, W, Ly.cout, net->e[l],
                               net->g_cat[d], cs, c_off, net->g_pool[l], net->g_e[l]);
        }
        const ConvIn in = conv_input(net, l);
        PCT_TRY(launch_wgrad(net, in, level, l, net->g_e[l]));
        if (l > 0) {
            // gradient of the pooled input of this layer
            ConvIn gin{net->g_e[l], nullptr, Ly.cout, 0, 0};
            PCT_TRY(launch_conv(net, gin, level, Ly.wf, nullptr, 0, Ly.cin, net->g_pool[l - 1]));
        }
    }
    NET_HIP(net, hipGetLastError());
    return PCT_OK;
}

int upload_sample(pct_net* net, const float* fbp, const uint8_t* hull, const float* target)
{
    const int64_t n0 = net->nv[0];
    hipStream_t s = net->stream;
    NET_HIP(net, hipMemcpyAsync(net->fbp, fbp, n0 * sizeof(float), hipMemcpyHostToDevice, s));
    NET_HIP(net, hipMemcpyAsync(net->hull, hull, n0, hipMemcpyHostToDevice, s));
    if (target) NET_HIP(net, hipMemcpyAsync(net->target, target, n0 * sizeof(float), hipMemcpyHostToDevice, s));
    return PCT_OK;
}

}  // namespace

extern "C" {

int pct_net_create(int columns, int rows, int slices, uint64_t seed, int device, pct_net** out)
{
    if (!out || columns <= 0 || rows <= 0 || slices <= 0 || columns % 8 || rows % 8 || slices % 8) return PCT_E_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return PCT_E_ARG;
    if (hipSetDevice(device) != hipSuccess) return PCT_E_HIP;
    pct_net* net = new pct_net();
    net->device = device;
    net->D = slices;
    net->H = rows;
    net->W = columns;
    for (int lv = 0; lv < 4; lv++) net->nv[lv] = (int64_t)(slices >> lv) * (rows >> lv) * (columns >> lv);
    const int cin[kLayers] = {8, 16, 32, 64, 192, 96, 48};
    const int cout[kLayers] = {16, 32, 64, 128, 64, 32, 16};
    const int level[kLayers] = {0, 1, 2, 3, 2, 1, 0};
    int64_t off = 0;
    for (int l = 0; l < kLayers; l++) {
        auto& Ly = net->L[l];
        Ly.cin = cin[l];
        Ly.cout = cout[l];
        Ly.level = level[l];
        Ly.Kp = (27 * cin[l] + 63) / 64 * 64;
        Ly.Kpf = (27 * cout[l] + 63) / 64 * 64;
        Ly.w_off = off;
        off += (int64_t)cout[l] * 27 * cin[l];
        Ly.b_off = off;
        off += cout[l];
    }
    net->head_off = off;
    off += 17;
    net->n_params = off;
    auto fail = [&](int rc) {
        pct_net_destroy(net);
        return rc;
    };
    if (hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking) != hipSuccess) return fail(PCT_E_HIP);
    int rc = PCT_OK;
    if ((rc = net_alloc(net, &net->p, off)) || (rc = net_alloc(net, &net->g, off)) || (rc = net_alloc(net, &net->m, off)) ||
        (rc = net_alloc(net, &net->v, off)))
        return fail(rc);
    for (int l = 0; l < kLayers; l++) {
        auto& Ly = net->L[l];
        if ((rc = net_alloc(net, &Ly.wt, (int64_t)Ly.cout * Ly.Kp)) || (rc = net_alloc(net, &Ly.wf, (int64_t)Ly.cin * Ly.Kpf)))
            return fail(rc);
    }
    const int64_t* nv = net->nv;
    if ((rc = net_alloc(net, &net->in8, nv[0] * 8))) return fail(rc);
    for (int l = 0; l < 4; l++) {
        if ((rc = net_alloc(net, &net->e[l], nv[l] * cout[l]))) return fail(rc);
        if ((rc = net_alloc(net, &net->g_e[l], nv[l] * cout[l]))) return fail(rc);
    }
    for (int l = 0; l < 3; l++) {
        if ((rc = net_alloc(net, &net->pool[l], nv[l + 1] * cout[l]))) return fail(rc);
        if ((rc = net_alloc(net, &net->g_pool[l], nv[l + 1] * cout[l]))) return fail(rc);
        // decoder d at level d: dd[d] has cout[6 - d] channels, its concat cin[6 - d]
        if ((rc = net_alloc(net, &net->dd[l], nv[l] * cout[6 - l]))) return fail(rc);
        if ((rc = net_alloc(net, &net->g_dd[l], nv[l] * cout[6 - l]))) return fail(rc);
        if ((rc = net_alloc(net, &net->g_cat[l], nv[l] * cin[6 - l]))) return fail(rc);
    }
    if ((rc = net_alloc(net, &net->x0, nv[0])) || (rc = net_alloc(net, &net->fbp, nv[0])) ||
        (rc = net_alloc(net, &net->target, nv[0])) || (rc = net_alloc(net, &net->hull, nv[0])) ||
        (rc = net_alloc(net, &net->loss_part, 2 * (int64_t)blocks_for(nv[0]))) ||
        (rc = net_alloc(net, &net->head_part, 17 * (int64_t)blocks_for(nv[0]))))
        return fail(rc);
    for (int l = 0; l < kLayers; l++) {
        const WgradShape w = wgrad_shape(net, l);
        const int64_t need = w.chunks * w.chunk_floats;
        net->partial_n = need > net->partial_n ? need : net->partial_n;
    }
    if ((rc = net_alloc(net, &net->partial, net->partial_n))) return fail(rc);
    // He-normal weights, zero biases, zero head (x0 starts as hull * FBP)
    std::vector<float> h(off, 0.0f);
    Rng rng{seed * 0x2545f4914f6cdd1dull + 1};
    for (int l = 0; l < kLayers; l++) {
        auto& Ly = net->L[l];
        const double sd = std::sqrt(2.0 / (27.0 * Ly.cin));
        for (int64_t j = 0; j < (int64_t)Ly.cout * 27 * Ly.cin; j++) h[Ly.w_off + j] = (float)(sd * rng.normal());
    }
    if (hipMemcpy(net->p, h.data(), off * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) return fail(PCT_E_HIP);
    (void)hipMemset(net->m, 0, off * sizeof(float));
    (void)hipMemset(net->v, 0, off * sizeof(float));
    if (pack_weights(net) != PCT_OK) return fail(PCT_E_HIP);
    if (hipStreamSynchronize(net->stream) != hipSuccess) return fail(PCT_E_HIP);
    *out = net;
    return PCT_OK;
}

int pct_net_destroy(pct_net* net)
{
    if (!net) return PCT_E_ARG;
    if (net->stream) (void)hipStreamSynchronize(net->stream);
    net_free(&net->p);
    net_free(&net->g);
    net_free(&net->m);
    net_free(&net->v);
    for (auto& Ly : net->L) {
        net_free(&Ly.wt);
        net_free(&Ly.wf);
    }
    net_free(&net->in8);
    for (int l = 0; l < 4; l++) {
        net_free(&net->e[l]);
        net_free(&net->g_e[l]);
    }
    for (int l = 0; l < 3; l++) {
        net_free(&net->pool[l]);
        net_free(&net->g_pool[l]);
        net_free(&net->dd[l]);
        net_free(&net->g_dd[l]);
        net_free(&net->g_cat[l]);
    }
    net_free(&net->x0);
    net_free(&net->fbp);
    net_free(&net->target);
    net_free(&net->hull);
    net_free(&net->loss_part);
    net_free(&net->head_part);
    net_free(&net->partial);
    for (auto& sm : net->samples) {
        net_free(&sm.fbp);
        net_free(&sm.hull);
        net_free(&sm.target);
    }
    if (net->stream) (void)hipStreamDestroy(net->stream);
    delete net;
    return PCT_OK;
}

const char* pct_net_last_error(pct_net* net) { return net ? net->err.c_str() : "null net"; }

int64_t pct_net_num_params(pct_net* net) { return net ? net->n_params : -1; }

int pct_net_get_params(pct_net* net, float* out, int64_t n)
{
    if (!net || !out || n != net->n_params) return PCT_E_ARG;
    NET_HIP(net, hipMemcpy(out, net->p, n * sizeof(float), hipMemcpyDeviceToHost));
    return PCT_OK;
}

int pct_net_set_params(pct_net* net, const float* in, int64_t n)
{
    if (!net || !in || n != net->n_params) return PCT_E_ARG;
    NET_HIP(net, hipMemcpy(net->p, in, n * sizeof(float), hipMemcpyHostToDevice));
    PCT_TRY(pack_weights(net));
    NET_HIP(net, hipStreamSynchronize(net->stream));
    return PCT_OK;
}

int pct_net_loss_grad(pct_net* net, const float* fbp, const uint8_t* hull, const float* target, double* loss,
                      float* grad)
{
    if (!net || !fbp || !hull || !target || !loss) return PCT_E_ARG;
    PCT_TRY(upload_sample(net, fbp, hull, target));
    PCT_TRY(net_forward(net, net->fbp, net->hull, net->target, loss));
    if (grad) {
        PCT_TRY(net_backward(net, net->hull, net->target));
        NET_HIP(net, hipMemcpyAsync(grad, net->g, net->n_params * sizeof(float), hipMemcpyDeviceToHost, net->stream));
        NET_HIP(net, hipStreamSynchronize(net->stream));
    }
    return PCT_OK;
}

int pct_net_predict(pct_net* net, const float* fbp, const uint8_t* hull, float* x0)
{
    if (!net || !fbp || !hull || !x0) return PCT_E_ARG;
    PCT_TRY(upload_sample(net, fbp, hull, nullptr));
    PCT_TRY(net_forward(net, net->fbp, net->hull, nullptr, nullptr));
    NET_HIP(net, hipMemcpyAsync(x0, net->x0, net->nv[0] * sizeof(float), hipMemcpyDeviceToHost, net->stream));
    NET_HIP(net, hipStreamSynchronize(net->stream));
    return PCT_OK;
}

int pct_net_add_sample(pct_net* net, const float* fbp, const uint8_t* hull, const float* target)
{
    if (!net || !fbp || !hull || !target) return PCT_E_ARG;
    const int64_t n0 = net->nv[0];
    pct_net::Sample sm{nullptr, nullptr, nullptr};
    int rc;
    if ((rc = net_alloc(net, &sm.fbp, n0)) || (rc = net_alloc(net, &sm.hull, n0)) || (rc = net_alloc(net, &sm.target, n0))) {
        net_free(&sm.fbp);
        net_free(&sm.hull);
        net_free(&sm.target);
        return rc;
    }
    net->samples.push_back(sm);
    NET_HIP(net, hipMemcpy(sm.fbp, fbp, n0 * sizeof(float), hipMemcpyHostToDevice));
    NET_HIP(net, hipMemcpy(sm.hull, hull, n0, hipMemcpyHostToDevice));
    NET_HIP(net, hipMemcpy(sm.target, target, n0 * sizeof(float), hipMemcpyHostToDevice));
    return PCT_OK;
}

int pct_net_num_samples(pct_net* net) { return net ? (int)net->samples.size() : -1; }

int pct_net_train(pct_net* net, int steps, double lr, uint64_t seed, double* mean_loss)
{
    if (!net || steps < 0 || net->samples.empty()) return PCT_E_ARG;
    hipStream_t s = net->stream;
    const int ns = (int)net->samples.size();
    std::vector<int> order(ns);
    Rng rng{seed + 0x51ed27ull};
    double lsum = 0.0;
    int pos = ns;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int it = 0; it < steps; it++) {
        if (pos == ns) {  // reshuffle each epoch (Fisher-Yates)
            for (int k = 0; k < ns; k++) order[k] = k;
            for (int k = ns - 1; k > 0; k--) {
                int j = (int)(rng.next() % (uint64_t)(k + 1));
                std::swap(order[k], order[j]);
            }
            pos = 0;
        }
        const auto& sm = net->samples[order[pos++]];
        double loss = 0;
        PCT_TRY(net_forward(net, sm.fbp, sm.hull, sm.target, &loss));
        PCT_TRY(net_backward(net, sm.hull, sm.target));
        net->adam_t++;
        const float c1 = 1.0f - std::pow(b1, (float)net->adam_t), c2 = 1.0f - std::pow(b2, (float)net->adam_t);
        hipLaunchKernelGGL(k_adam, dim3(blocks_for(net->n_params)), dim3(kBlock), 0, s, net->n_params, (float)lr, b1, b2,
                           eps, c1, c2, net->p, net->g, net->m, net->v);
        PCT_TRY(pack_weights(net));
        lsum += loss;
    }
    NET_HIP(net, hipStreamSynchronize(s));
    if (mean_loss) *mean_loss = steps > 0 ? lsum / steps : 0.0;
    return PCT_OK;
}

int pct_net_save(pct_net* net, const char* path)
{
    if (!net || !path) return PCT_E_ARG;
    std::vector<float> h(net->n_params);
    NET_HIP(net, hipMemcpy(h.data(), net->p, h.size() * sizeof(float), hipMemcpyDeviceToHost));
    FILE* f = std::fopen(path, "wb");
    if (!f) return PCT_E_IO;
    const char magic[8] = {'P', 'C', 'T', 'N', 'E', 'T', '0', '1'};
    int64_t n = net->n_params;
    bool ok = std::fwrite(magic, 1, 8, f) == 8 && std::fwrite(&n, sizeof(n), 1, f) == 1 &&
              std::fwrite(h.data(), sizeof(float), h.size(), f) == h.size();
    ok = (std::fclose(f) == 0) && ok;
    return ok ? PCT_OK : PCT_E_IO;
}

int pct_net_load(pct_net* net, const char* path)
{
    if (!net || !path) return PCT_E_ARG;
    FILE* f = std::fopen(path, "rb");
    if (!f) return PCT_E_IO;
    char magic[8];
    int64_t n = 0;
    std::vector<float> h(net->n_params);
    bool ok = std::fread(magic, 1, 8, f) == 8 && std::memcmp(magic, "PCTNET01", 8) == 0 &&
              std::fread(&n, sizeof(n), 1, f) == 1 && n == net->n_params &&
              std::fread(h.data(), sizeof(float), h.size(), f) == h.size();
    std::fclose(f);
    if (!ok) {
        net->err = "not a weight file of this network";
        return PCT_E_IO;
    }
    return pct_net_set_params(net, h.data(), n);
}

// x0 := net(FBP, hull) on the device of ctx; the FBP-based x0 is kept instead when the net's x0 has
// the larger DROP data residual ||Ax - b|| (needs the MLP lists).
int pct_net_apply(pct_net* net, pct_ctx* ctx, int* used_net, double* residual_fbp, double* residual_net)
{
    if (!net || !ctx) return PCT_E_ARG;
    const pct_params& P = ctx->P;
    if (P.columns != net->W || P.rows != net->H || P.slices != net->D) {
        net->err = "network grid differs from the reconstruction grid";
        return PCT_E_ARG;
    }
    if (ctx->stage < ST_LISTS || !ctx->fbp || !ctx->hull || !ctx->x0 || !ctx->x) {
        net->err = "pct_net_apply needs FBP, hull, x0 and the MLP lists";
        return PCT_E_STATE;
    }
    const int64_t n0 = net->nv[0];
    // the context's stream finishes its work before the net reads FBP and hull
    NET_HIP(net, hipStreamSynchronize(ctx->stream));
    PCT_TRY(net_forward(net, ctx->fbp, ctx->hull, nullptr, nullptr));
    NET_HIP(net, hipStreamSynchronize(net->stream));
    // copies into the context run on its stream, ordered with its residual kernels
    hipStream_t cs = ctx->stream;
    double r_fbp = 0, r_net = 0;
    NET_HIP(net, hipMemcpyAsync(ctx->x, ctx->x0, n0 * sizeof(float), hipMemcpyDeviceToDevice, cs));
    if (pct_stage_residual(ctx, &r_fbp) != PCT_OK) {
        net->err = ctx->err;
        return PCT_E_HIP;
    }
    NET_HIP(net, hipMemcpyAsync(ctx->x, net->x0, n0 * sizeof(float), hipMemcpyDeviceToDevice, cs));
    if (pct_stage_residual(ctx, &r_net) != PCT_OK) {
        net->err = ctx->err;
        return PCT_E_HIP;
    }
    const int use = r_net < r_fbp;
    if (use) {
        NET_HIP(net, hipMemcpyAsync(ctx->x0, net->x0, n0 * sizeof(float), hipMemcpyDeviceToDevice, cs));
    } else {
        NET_HIP(net, hipMemcpyAsync(ctx->x, ctx->x0, n0 * sizeof(float), hipMemcpyDeviceToDevice, cs));
    }
    NET_HIP(net, hipStreamSynchronize(cs));
    if (used_net) *used_net = use;
    if (residual_fbp) *residual_fbp = r_fbp;
    if (residual_net) *residual_net = r_net;
    return PCT_OK;
}

int pct_net_apply_iterate(pct_net* net, pct_ctx* ctx, int* used_net, double* residual_x, double* residual_net)
{
    if (!net || !ctx) return PCT_E_ARG;
    const pct_params& P = ctx->P;
    if (P.columns != net->W || P.rows != net->H || P.slices != net->D) {
        net->err = "network grid differs from the reconstruction grid";
        return PCT_E_ARG;
    }
    if (ctx->stage < ST_LISTS || !ctx->hull || !ctx->x) {
        net->err = "pct_net_apply_iterate needs the hull, an iterate and the MLP lists";
        return PCT_E_STATE;
    }
    const int64_t n0 = net->nv[0];
    NET_HIP(net, hipStreamSynchronize(ctx->stream));
    PCT_TRY(net_forward(net, ctx->x, ctx->hull, nullptr, nullptr));
    NET_HIP(net, hipStreamSynchronize(net->stream));
    hipStream_t cs = ctx->stream;
    double r_x = 0, r_net = 0;
    if (pct_stage_residual(ctx, &r_x) != PCT_OK) {
        net->err = ctx->err;
        return PCT_E_HIP;
    }
    NET_HIP(net, hipMemcpyAsync(net->fbp, ctx->x, n0 * sizeof(float), hipMemcpyDeviceToDevice, cs));  // keep x
    NET_HIP(net, hipMemcpyAsync(ctx->x, net->x0, n0 * sizeof(float), hipMemcpyDeviceToDevice, cs));
    if (pct_stage_residual(ctx, &r_net) != PCT_OK) {
        net->err = ctx->err;
        return PCT_E_HIP;
    }
    const int use = r_net < r_x;
    if (!use) NET_HIP(net, hipMemcpyAsync(ctx->x, net->fbp, n0 * sizeof(float), hipMemcpyDeviceToDevice, cs));
    NET_HIP(net, hipStreamSynchronize(cs));
    if (used_net) *used_net = use;
    if (residual_x) *residual_x = r_x;
    if (residual_net) *residual_net = r_net;
    return PCT_OK;
}

}  // extern "C"
