// k_drop_tiles.hip — stage (e): DROP over image tiles held in LDS.
//
// The row and column kernels of k_drop2.hip gather every list entry from memory, and the rate of those
// gathers bounds them.  Here a DROP block's lists are cut, when they are built, into segments: runs of
// consecutive entries inside one tile of 16 x 16 x 2 voxels (512 floats, 2 KB).  A segment holds about 11
// entries, and 220 segments of a block pass through a tile (head, blocks of 60000), so a workgroup that owns a
// tile reads its 512 voxels once and each segment's update once, and every gather per entry is an LDS read.  Per
// block b two kernels run:
//   k_tile_rows  8 lanes per history: adds the partial row sums of its segments and forms u_i
//                (DS.cu:9321-9380), in visiting order;
//   k_tile_pass  a workgroup per tile: the column sums of block b (u of the tile's segments in LDS, one
//                lane per voxel, in history order), x += sum / S, and then, from the updated tile still in
//                LDS, the partial row sums of block b + 1.  A tile is written by its own workgroup only.
// The sums are those of k_drop2.hip to the bit: column sums add the same updates in the same order, and a
// row's partial sums are used only where no sum of its terms can round in any order (order_free, with the
// bounds of the whole tile, or of the segment's own values where the tile's span many powers of two: kWide);
// every other row is summed in list order from memory.
//
// Layout of one (block, tile), built by k_tile_fill:
//   segments in visiting order (neighbouring paths next to each other, so the loads of u and the reads of
//   the partial sums coalesce); the tile's touched voxels by descending entry count, 64 to a slice, their
//   segment numbers column-major, padded to the slice's largest count; and the segments by descending
//   length, 64 to a slice, the steps between their slots laid out the same way.
// 10 bits per entry of a column and 8 bits per entry of a row replace the 4-byte lists, and the sort of all
// list entries by (block, voxel) becomes one of the segments by (block, tile), an eleventh of the items.
//
// Head, 20M histories (148 blocks of 60000, 6.5M entries and 587K segments a block), against the sorted lists of
// k_drop2.hip: a block 19.1 + 6.4 us instead of 17.4 + 19.1, list build 39 instead of 61 ms, device memory 24 instead of 74 GB.
#include <hip/hip_ext.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "drop_sums.h"
#include "internal.h"

namespace {

constexpr int kBlock = 256;
constexpr int kTileVox = 512;       // 16 x 16 x 2 voxels
constexpr uint32_t kMaxSeg = 1022;  // segments of a block in one tile
constexpr uint32_t kMaxEnt = 16384; // entries of a block in one tile
constexpr uint32_t kMaxCnt = 127;   // entries of a block in one voxel
constexpr int kRound = 128;         // list entries cut at a time; a segment never crosses a multiple of this
// List slots (u-steps, 1.8 to an entry) of a block per tile at which the tiles take over from the sorted lists,
// DROP block and list build, tiles against sorted lists: cylinder-2M (1600 tiles) at 490 slots 13.2 against 12.7 us
// and 11.3 against 10.5 ms, at 980 slots 13.7 against 14.8 us and 8.1 against 10.2 ms; the head on 256 x 256 x 96
// with 3M histories (10.8K tiles) at 970 slots 58.9 against 54.2 us and 32.5 against 41.5 ms, at 2300 slots 69.0
// against 83.8 us and 25.6 against 40.8 ms.  Below, a tile's own costs (its voxels read and written, its
// descriptor) outweigh the gathers that it saves.
constexpr double kMinSlots = 1000.0;
// and in blocks of few slots, whose kernels are as short by sorted lists: 128 x 128 with 0.77M slots and 1000 to 2000 in a
// tile, lists built and 20 iterations, 1.04 to 1.08 of the sorted lists' time, 183 x 124 with 0.47M and 1440 1.02, but
// 201 x 112 with 0.80M and 2900 0.98, 110 x 215 with 0.61M and 2400 0.96.
constexpr double kMinSlotsSmall = 1500.0, kSmallBlock = 0.8e6;
// Paths through the busiest tile (a block's mean): its workgroup holds up the pass where few tiles take all the paths.
// With so many in it, a block must have kMinSpread slots for each of them.  The whole of a reconstruction, or of list
// build and iterations, or of iterations alone, tiles to sorted lists, by that ratio: 2860 (535 paths) 1.30, 4100 (541)
// 1.04, 4260 (340) 1.14, 5050 (387) 1.09, 5820 to 6540 (410 to 506) 1.07 to 1.15, 6930 to 8430 (280 to 410) 0.91 to
// 0.98, 8600 to 9800 0.89 to 0.96, above 12000 at most 0.96.  With fewer paths in it: 3190 to 6410 (147 to 304) 0.96 to
// 1.03.
constexpr double kManyPaths = 310.0, kMinSpread = 6800.0;
// Such paths from which another block will have more segments there than kMaxSeg.  Plans with 600 and more either did not
// fit (614 to 2060 of them), at 2.6 ms and more for the build until that was known, or gained nothing (600: 1.00, 639:
// 0.98, 674: 1.10, 740: 1.05, 813: 1.08); with 542, 981 segments: 0.77, with 574: 0.85.
constexpr double kMaxPaths = 600.0;
// and of the whole plan: below, the build's fixed launches and waits cost more than the sort of so few entries
// (head, 7M slots: list build 1.8 against 1.3 ms; cylinder-2M, 255M slots in blocks of 12800: 6.7 against 9.7 ms).
constexpr int64_t kMinTotalSlots = 1ll << 25;
constexpr int32_t kMaxBlock = 1 << 22;  // histories of a block (22 bits of the fill's history order)
constexpr int64_t kSample = 1 << 14;    // paths that the rule looks at
constexpr int64_t kSlack = 2048;       // readable elements past the lists (see k_tile_pass)
constexpr int kMaxDup = 64;         // repeated visits of a voxel by one segment, per tile

inline unsigned grid_for(int64_t n, int block = kBlock) { return pct_grid_for(n, block); }

// Tile and slot of a row-major voxel.  Divisions by the row length and row count as a product and a shift,
// exact for dividends below 2^31 (M = ceil(2^(31 + l) / d), l = ceil(log2 d)).
struct TileGeom {
    uint32_t C, R, ntx, nty, nt;
    uint64_t mC, mR;
    int sC, sR;
};
__device__ __forceinline__ void tile_xyz(uint32_t v, const TileGeom& g, uint32_t& tile, uint32_t& x, uint32_t& y,
                                         uint32_t& z)
{
    const uint32_t t = (uint32_t)(((uint64_t)v * g.mC) >> g.sC);
    x = v - t * g.C;
    z = (uint32_t)(((uint64_t)t * g.mR) >> g.sR);
    y = t - z * g.R;
    tile = ((z >> 1) * g.nty + (y >> 4)) * g.ntx + (x >> 4);
}
// Tile << 9 | slot.  Slots run z, x, y, so that the next voxel of a path is a few slots away (a signed byte).
__device__ __forceinline__ uint32_t tile_slot(uint32_t v, const TileGeom& g)
{
    uint32_t tile, x, y, z;
    tile_xyz(v, g, tile, x, y, z);
    return tile << 9 | (y & 15u) << 5 | (x & 15u) << 1 | (z & 1u);
}
// Index of a listed voxel in the tiled image: within a tile, 4 x 4 x 2 voxels to a 128-byte line.
struct TileIndex {
    TileGeom g;
    __device__ __forceinline__ uint32_t operator()(uint32_t v) const
    {
        uint32_t tile, x, y, z;
        tile_xyz(v, g, tile, x, y, z);
        return tile << 9 | ((y >> 2) & 3u) << 7 | ((x >> 2) & 3u) << 5 | (z & 1u) << 4 | (y & 3u) << 2 | (x & 3u);
    }
};
// The slot of the first of the four voxels 4 k .. 4 k + 3 of a tile in memory; the others are 2, 4 and 6 on.
__device__ __forceinline__ uint32_t slot_of_quad(uint32_t k)
{
    const uint32_t y = (k >> 5) * 4 + (k & 3u), x = ((k >> 3) & 3u) * 4, z = (k >> 2) & 1u;
    return y << 5 | x << 1 | z;
}

// image into (to_tiles) or out of the tiled layout
__global__ void k_x_tiles(int64_t nv, float* __restrict__ x, float* __restrict__ xt, TileIndex at, int to_tiles)
{
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    const uint32_t b = at((uint32_t)v);
    if (to_tiles) xt[b] = x[v];
    else x[v] = xt[b];
}

// ---------------------------------------------------------------- plan ----
// list slots of every raw block, and the first of them
__global__ void k_tile_block_caps(int64_t n_raw, int64_t BS, int64_t n,
                                  const int64_t* __restrict__ off, int64_t* __restrict__ out,
                                  int64_t* __restrict__ first)
{
    const int64_t rb = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (rb >= n_raw) return;
    const int64_t end = rb * BS + BS < n ? rb * BS + BS : n;
    out[rb] = off[end] - off[rb * BS];
    first[rb] = off[rb * BS];
}

// Counts a sample of the paths through every tile, by every 8th entry of their lists, or, before the lists exist, by
// points 8 voxels apart on their chords (the u-step is half a voxel).  Few tiles are counted in LDS first (300 tiles on
// 219 x 153 x 8: 98 us with every count in memory, now 12).
struct SampleArgs {
    int64_t n, every;
    TileGeom g;
    const float *x0, *y0, *z0, *x1, *y1, *z1;  // entry and exit; null: the lists
    DevGeom geom;
    const int64_t* off;
    const uint32_t *cnt, *vox;
};
constexpr uint32_t kSampleTiles = 8192;  // counted in LDS
template <class Through>
__device__ __forceinline__ void sample_path(const SampleArgs& a, int64_t i, Through through)
{
    if (!a.x0) {
        for (uint32_t j = 0; j < a.cnt[i]; j += 8) through(tile_slot(a.vox[a.off[i] + j], a.g) >> 9);
        return;
    }
    const DevGeom& g = a.geom;
    const double dx = (double)a.x1[i] - a.x0[i], dy = (double)a.y1[i] - a.y0[i], dz = (double)a.z1[i] - a.z0[i];
    const int steps = (int)fmin(sqrt(dx * dx + dy * dy) / (8 * g.VW), 4096.0) + 1;
    for (int k = 0; k <= steps; k++) {
        const double f = (double)k / steps;
        const int x = pct_calc_voxel(g.X0, a.x0[i] + f * dx, g.VW), y = pct_calc_voxel(g.Y0, a.y0[i] + f * dy, g.VH),
                  z = pct_calc_voxel(g.Z0, a.z0[i] + f * dz, g.VT);
        if (x < g.C && y < g.R && z < g.S)
            through((((uint32_t)z >> 1) * a.g.nty + ((uint32_t)y >> 4)) * a.g.ntx + ((uint32_t)x >> 4));
    }
}
template <bool LDS>
__global__ void __launch_bounds__(kBlock) k_tile_sample(SampleArgs a, uint32_t* __restrict__ count)
{
    extern __shared__ uint32_t local[];  // LDS: a.g.nt counts
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * a.every;
    if (LDS) {
        for (uint32_t t = threadIdx.x; t < a.g.nt; t += kBlock) local[t] = 0u;
        __syncthreads();
    }
    uint32_t last = ~0u;
    if (i < a.n)
        sample_path(a, i, [&](uint32_t tile) {
            if (tile != last) {
                if (LDS) atomicAdd(&local[tile], 1u);
                else atomicAdd(&count[tile], 1u);
            }
            last = tile;
        });
    if (LDS) {
        __syncthreads();
        for (uint32_t t = threadIdx.x; t < a.g.nt; t += kBlock)
            if (local[t]) atomicAdd(&count[t], local[t]);
    }
}

// out[0]: the tiles with a path, out[1]: the most paths through one
__global__ void __launch_bounds__(kBlock) k_tile_reach(uint32_t nt, const uint32_t* __restrict__ count,
                                                       uint32_t* __restrict__ out)
{
    uint32_t most = 0, reached = 0;
    for (uint32_t t = blockIdx.x * kBlock + threadIdx.x; t < nt; t += gridDim.x * kBlock) {
        const uint32_t c = count[t];
        reached += c > 0;
        most = c > most ? c : most;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const uint32_t m = __shfl_xor(most, o, 64);
        reached += __shfl_xor(reached, o, 64);
        most = m > most ? m : most;
    }
    if ((threadIdx.x & 63) == 0 && reached) {
        atomicAdd(out, reached);
        atomicMax(out + 1, most);
    }
}

// visiting order of a group: (block in group, sinogram bin) with unprocessed histories last in their block
__global__ void k_tile_hist_keys(int64_t h0, int64_t n, int64_t BS, int64_t rb0, const int32_t* __restrict__ proc_raw,
                                 const int32_t* __restrict__ bin_num, int bin_bits, uint32_t* __restrict__ keys,
                                 uint32_t* __restrict__ idx)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int64_t i = h0 + t, rb = i / BS;
    const uint32_t marker = (1u << bin_bits) - 1u;
    uint32_t b = marker;
    if (i - rb * BS < proc_raw[rb]) {
        const uint32_t bn = (uint32_t)bin_num[i];
        b = bn < marker ? bn : marker - 1u;
    }
    keys[t] = ((uint32_t)(rb - rb0) << bin_bits) | b;
    idx[t] = (uint32_t)t;
}

// Cuts every history's list into segments (consecutive entries of one tile, steps of at most 127 slots), 16 lanes per history, kRound entries at a time, the histories in
// visiting order.  EMIT false: the number of segments (0 when it is not processed or shorter than
// MIN_MLP_LENGTH).  EMIT true: its row descriptor, and per segment the key (block in group, tile) and its record;
// without any segment only the descriptors, and the arrays of the segments may be null.
struct CutArgs {
    int64_t h0, n, BS, rb0, slot0;  // slot0: the group's first list slot
    TileGeom g;
    int tile_bits, min_len;
    const int32_t* proc_raw;
    const uint32_t* order;  // sorted position -> history of the group
    const int64_t* off;
    const uint32_t* cnt;
    const uint32_t* vox;
    const double* chord;
    const float* wepl;
};
struct SegRec {  // visiting rank << 38 | first entry (slot of the group) << 8 | length; index in the block
    uint64_t v;
    uint32_t hist, pad;
};
constexpr uint64_t pack_seg(uint32_t rank, uint32_t pos, uint32_t len)
{
    return (uint64_t)rank << 38 | (uint64_t)pos << 8 | (uint64_t)len;
}
__device__ __forceinline__ uint32_t seg_rank_of(uint64_t v) { return (uint32_t)(v >> 38); }
__device__ __forceinline__ uint32_t seg_pos_of(uint64_t v) { return (uint32_t)(v >> 8) & 0x3fffffffu; }
__device__ __forceinline__ uint32_t seg_len_of(uint64_t v) { return (uint32_t)v & 255u; }

template <bool EMIT>
__global__ void __launch_bounds__(kBlock) k_tile_cut(CutArgs a, uint32_t* __restrict__ nseg,
                                                     const uint32_t* __restrict__ q0, TileRow* __restrict__ rows,
                                                     uint32_t* __restrict__ keys, uint32_t* __restrict__ idx,
                                                     SegRec* __restrict__ recs)
{
    constexpr int L = 16, K = kRound / L;
    const int lane = threadIdx.x & (L - 1), sh = threadIdx.x & 48;  // the group's place in its wavefront
    const int64_t n_groups = ((int64_t)gridDim.x * blockDim.x) / L;
    for (int64_t s = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / L; s < a.n; s += n_groups) {
        const int64_t i = a.h0 + a.order[s], rb = i / a.BS;
        const uint32_t c = a.cnt[i];
        const bool take = i - rb * a.BS < a.proc_raw[rb] && (int)c >= a.min_len;
        const int64_t o = a.off[i];
        const uint32_t rank = (uint32_t)(a.h0 + s - rb * a.BS), first = EMIT ? q0[s] : 0u;
        uint32_t total = 0;
        if (take) {
            for (uint32_t j0 = 0; j0 < c; j0 += kRound) {
                uint32_t tl[K];
#pragma unroll
                for (int q = 0; q < K; q++) {
                    const uint32_t j = j0 + q * L + lane;
                    tl[q] = j < c ? a.vox[o + j] : 0u;
                }
                uint64_t lo = 0, hi = 0;  // entries that start a segment
#pragma unroll
                for (int q = 0; q < K; q++) {
                    tl[q] = tile_slot(tl[q], a.g);
                    const uint32_t up = __shfl_up(tl[q], 1, L);
                    const uint32_t before = q > 0 ? __shfl(tl[q > 0 ? q - 1 : 0], L - 1, L) : ~0u;
                    const uint32_t prev = lane == 0 ? before : up;
                    // another tile, or a step beyond a signed byte
                    const bool head = j0 + q * L + lane < c && ((tl[q] ^ prev) >> 9 || tl[q] - prev + 128u > 255u);
                    const uint64_t m = (__ballot(head) >> sh) & 0xffffull;
                    if (q < 4) lo |= m << (16 * (q & 3));
                    else hi |= m << (16 * (q & 3));
                }
                if (EMIT) {
                    const uint32_t end = c - j0 < (uint32_t)kRound ? c - j0 : (uint32_t)kRound;
#pragma unroll
                    for (int q = 0; q < K; q++) {
                        const uint32_t e = q * L + lane;
                        const uint64_t own = q < 4 ? lo : hi;
                        if (!((own >> (e & 63u)) & 1ull)) continue;
                        const uint64_t above = (e & 63u) == 63u ? 0ull : own >> ((e & 63u) + 1u);
                        uint32_t next = end;
                        if (above) next = e + (uint32_t)__ffsll((unsigned long long)above);
                        else if (q < 4 && hi) next = 64u + (uint32_t)__ffsll((unsigned long long)hi) - 1u;
                        uint32_t ord = total + (uint32_t)__popcll(own & ((1ull << (e & 63u)) - 1ull));
                        if (q >= 4) ord += (uint32_t)__popcll(lo);
                        keys[first + ord] = (uint32_t)(rb - a.rb0) << a.tile_bits | tl[q] >> 9;
                        idx[first + ord] = first + ord;
                        SegRec rec;
                        rec.v = pack_seg(rank, (uint32_t)(o - a.slot0) + j0 + e, next - e);
                        rec.hist = (uint32_t)(i - rb * a.BS);
                        rec.pad = 0;
                        recs[first + ord] = rec;
                    }
                }
                total += (uint32_t)(__popcll(lo) + __popcll(hi));
            }
        }
        if (lane == 0) {
            if (EMIT) {
                TileRow d;
                d.off = o;
                d.chord = a.chord[i];
                d.cnt = c;
                d.wepl = a.wepl[i];
                d.seg = first;
                d.n_seg = total;
                rows[a.h0 + s] = d;  // a block's histories keep their positions
            } else {
                nseg[s] = total;
            }
        }
    }
}

// Per sorted segment: its record, its visiting rank, and where a history finds it.
__global__ void k_tile_gather(uint32_t n, const uint32_t* __restrict__ idx, const SegRec* __restrict__ recs,
                              SegRec* __restrict__ segs, uint32_t* __restrict__ seg_rank, uint32_t* __restrict__ place)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const uint32_t q = idx[j];
    const SegRec r = recs[q];
    segs[j] = r;
    seg_rank[j] = seg_rank_of(r.v);
    place[q] = j;  // segments are emitted history by history
}

// LDS of the fill of a tile (see k_tile_fill), and the launches it is dealt to by that size: 6, 5, 4, 3, 2 or 1
// workgroups on a CU.
constexpr uint32_t kLdsUnit = 512;
constexpr int kClasses = 6;
constexpr uint32_t kClassLds[kClasses] = {22528, 27648, 35840, 49152, 75776, 116736};
__host__ __device__ constexpr uint32_t fill_lds(uint32_t segs, uint32_t entries)
{
    return ((segs + 31) & ~31u) * (kTileVox / 8 + 16) + ((entries * 2 + 15) & ~15u);
}

constexpr int kLimits = 3 + kClasses;  // scratch words: [0] a list beyond the packed fields, [1] segments, [2] entries

// bounds[k]: how many tiles (by ascending need) fit class k
__global__ void k_tile_classes(uint32_t n, const uint32_t* __restrict__ need, uint32_t* __restrict__ bounds)
{
    if (threadIdx.x >= (unsigned)kClasses) return;
    const uint32_t limit = kClassLds[threadIdx.x] / kLdsUnit;
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) / 2;
        if (need[mid] <= limit) lo = mid + 1;
        else hi = mid;
    }
    bounds[threadIdx.x] = lo;
}

// Per (block, tile), one wavefront: its first segment, segments and entries, and the LDS its fill needs.
__global__ void __launch_bounds__(kBlock) k_tile_runs(uint32_t n_runs, int tile_bits, const uint32_t* __restrict__ ukeys,
                                                      const uint32_t* __restrict__ seg_start,
                                                      const uint32_t* __restrict__ seg_count,
                                                      const SegRec* __restrict__ segs, TileRun* __restrict__ runs,
                                                      uint32_t* __restrict__ entries, uint32_t* __restrict__ need,
                                                      uint32_t* __restrict__ idx, uint8_t* __restrict__ used)
{
    const uint32_t t = (uint32_t)(((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6), lane = threadIdx.x & 63u;
    if (t >= n_runs) return;
    const uint32_t s0 = seg_start[t], S = seg_count[t];
    uint32_t e = 0;
    for (uint32_t j = lane; j < S; j += 64) e += seg_len_of(segs[s0 + j].v);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
    if (lane == 0) {
        const uint32_t key = ukeys[t];
        TileRun r{};
        r.key = key;
        r.seg = s0;
        r.n = S;
        r.entries = e;
        runs[t] = r;
        entries[t] = e;
        const uint32_t k = (fill_lds(S, e) + kLdsUnit - 1) / kLdsUnit;
        need[t] = k < 255u ? k : 255u;
        idx[t] = t;
        used[key & ((1u << tile_bits) - 1u)] = 1;
    }
}

// Inclusive sum of `v` over the 256 lanes of a workgroup.
__device__ __forceinline__ uint32_t scan256(uint32_t v, uint32_t* part)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(v, o, 64);
        if (lane >= o) v += y;
    }
    __syncthreads();
    if (lane == 63) part[w] = v;
    __syncthreads();
    for (int q = 0; q < w; q++) v += part[q];
    return v;
}

// A unit is one 32-bit word: three 10-bit numbers of a voxel's segments, plus one (0: none), or four signed byte
// steps of a segment's slots.  Word of unit u of lane l in a slice of U units per lane:
// units 2k and 2k + 1 of a lane are one 8-byte load, an odd last unit a 4-byte one.
__device__ __forceinline__ uint32_t unit_word(uint32_t u, uint32_t U, uint32_t lane)
{
    return (u ^ 1u) < U ? (u >> 1) * 128 + lane * 2 + (u & 1u) : (u >> 1) * 128 + lane;
}

// One (block, tile) per workgroup: its column lists (the segments of every voxel in history order), its row
// lists (the slots of every segment in path order) and the orders they are stored in, written where the
// group's cursor has room (cursor[0]; past `capacity` words nothing is written and the host asks again).
// A voxel's list in history order is the set bits of its bitmap over the tile's segments in history order, so
// no placement is serial: every entry sets its bit with an LDS atomic.  A segment that visits a
// voxel twice finds its bit set; those few visits are kept in a list and repeated in the voxel's list.
struct FillArgs {
    TileGeom g;
    int tile_bits;
    int64_t slot0;
    const uint32_t* vox;
    const SegRec* segs;
    const uint32_t* order;  // the tiles this launch takes
    uint64_t capacity;
};
__global__ void __launch_bounds__(kBlock) k_tile_fill(FillArgs a, TileRun* __restrict__ runs,
                                                      uint16_t* __restrict__ tv, uint32_t* __restrict__ seg_ord,
                                                      uint32_t* __restrict__ words,
                                                      unsigned long long* __restrict__ cursor,
                                                      uint32_t* __restrict__ limits, BlockTotals* __restrict__ totals)
{
    extern __shared__ __align__(16) uint32_t bits[];  // [segment / 32][voxel]; `hist` is read 16 bytes at a time
    __shared__ uint32_t bins[128], len_bins[kRound + 1], part[4], heads[8], row_heads[16], n_dup;
    __shared__ uint32_t dup[kMaxDup];
    __shared__ uint16_t slot_at[kTileVox], cnt_at[kTileVox];
    __shared__ uint64_t base;
    __shared__ uint8_t len[kMaxSeg];
    const uint32_t t = a.order[blockIdx.x], tid = threadIdx.x;
    TileRun r = runs[t];
    const uint32_t S = r.n & 0xffffu, s0 = r.seg, nw = (S + 31) / 32, cap = nw * 32;
    uint32_t* pos = bits + nw * kTileVox;       // first list slot of every segment
    uint32_t* hist = pos + cap;                 // its history << 10 | its number
    uint16_t* eo = (uint16_t*)(hist + cap);     // its first entry in `ent`
    uint16_t* ord = eo + cap;                   // segments by descending length
    uint16_t* turn = ord + cap;                 // its turn in history order
    uint16_t* at_turn = turn + cap;             // the segment of every turn
    uint16_t* ent = at_turn + cap;              // slots of the tile's entries
    for (uint32_t k = tid; k < nw * kTileVox; k += kBlock) bits[k] = 0u;
    if (tid < 128) bins[tid] = 0u;
    if (tid <= kRound) len_bins[tid] = 0u;
    if (tid < 8) heads[tid] = 0u;
    if (tid < 16) row_heads[tid] = 0u;
    if (tid == 0) n_dup = 0u;
    __syncthreads();
    {   // each lane takes 4 consecutive segments
        uint32_t l4[4], sum = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t j = 4 * tid + q;
            const SegRec g = j < S ? a.segs[s0 + j] : SegRec{0ull, 0u, 0u};
            const uint64_t v = g.v;
            l4[q] = seg_len_of(v);
            if (j < cap) hist[j] = j < S ? g.hist << 10 | j : ~0u;
            if (j < S) {
                pos[j] = seg_pos_of(v);
                len[j] = (uint8_t)l4[q];
                atomicAdd(&len_bins[l4[q]], 1u);
            }
            sum += l4[q];
        }
        uint32_t ex = scan256(sum, part) - sum;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t j = 4 * tid + q;
            if (j < S) eo[j] = (uint16_t)ex;
            ex += l4[q];
        }
    }
    __syncthreads();
    for (uint32_t j = tid; j < S; j += kBlock) {  // (a history's own segments in path order)
        const uint32_t h = hist[j];
        uint32_t p = 0;
        for (uint32_t k = 0; k < S; k += 4) {  // the array is a multiple of 32 long, its rest ~0
            const uint4 o = *reinterpret_cast<const uint4*>(hist + k);
            p += (o.x < h) + (o.y < h) + (o.z < h) + (o.w < h);
        }
        turn[j] = (uint16_t)p;
        at_turn[p] = (uint16_t)j;
    }
    __syncthreads();
    // entries: 16 lanes per segment, 4 segments in flight
    {
        const uint32_t lane = tid & 15u;
        auto put = [&](uint32_t j, uint32_t e, uint32_t v) {
            const uint32_t s = tile_slot(v, a.g) & 511u, p = turn[j], bit = 1u << (p & 31u);
            ent[eo[j] + e] = (uint16_t)s;
            if (atomicOr(&bits[(p >> 5) * kTileVox + s], bit) & bit) {
                const uint32_t k = atomicAdd(&n_dup, 1u);
                if (k < (uint32_t)kMaxDup) dup[k] = s << 16 | p;
            }
        };
        const uint32_t* __restrict__ vox = a.vox + a.slot0;
        for (uint32_t j = tid >> 4; j < S; j += 64) {
            uint32_t v[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t jj = j + 16 * q;
                v[q] = jj < S && lane < len[jj] ? vox[pos[jj] + lane] : ~0u;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t jj = j + 16 * q;
                if (v[q] != ~0u) put(jj, lane, v[q]);
                if (jj < S)
                    for (uint32_t e = 16 + lane; e < len[jj]; e += 16) put(jj, e, vox[pos[jj] + e]);
            }
        }
    }
    __syncthreads();
    // voxels by descending entry count: places from a histogram of the counts (largest first)
    const uint32_t nd = n_dup < (uint32_t)kMaxDup ? n_dup : (uint32_t)kMaxDup;
    bool over = n_dup > (uint32_t)kMaxDup;
    uint32_t c[2], b[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t v = tid + 256 * h;
        c[h] = 0;
        for (uint32_t w = 0; w < nw; w++) c[h] += (uint32_t)__popc(bits[w * kTileVox + v]);
        for (uint32_t k = 0; k < nd; k++) c[h] += (dup[k] >> 16) == v ? 1u : 0u;
        over = over || c[h] > kMaxCnt;
        b[h] = c[h] > kMaxCnt ? 0u : kMaxCnt - c[h];
        if (c[h]) atomicAdd(&bins[b[h]], 1u);
    }
    __syncthreads();
    const uint32_t n0 = tid < 128 ? bins[tid] : 0u;
    const uint32_t ex = scan256(n0, part) - n0;
    const uint32_t nt = part[0] + part[1] + part[2] + part[3];
    __syncthreads();
    if (tid < 128) bins[tid] = ex;
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; h++)
        if (c[h]) {
            const uint32_t p = atomicAdd(&bins[b[h]], 1u);
            slot_at[p] = (uint16_t)(tid + 256 * h);
            cnt_at[p] = (uint16_t)c[h];
            tv[(size_t)t * kTileVox + p] = (uint16_t)(c[h] << 9 | (tid + 256 * h));
            if ((p & 63u) == 0) heads[p >> 6] = (c[h] + 2) / 3;
        }
    // segments by descending length
    const uint32_t lc = tid <= kRound ? len_bins[kRound - tid] : 0u;
    const uint32_t lincl = scan256(lc, part);
    __syncthreads();
    if (tid <= kRound) len_bins[kRound - tid] = lincl - lc;
    __syncthreads();
    for (uint32_t j = tid; j < S; j += kBlock) {
        const uint32_t l = len[j], p = atomicAdd(&len_bins[l], 1u);
        seg_ord[s0 + p] = j | l << 10 | (uint32_t)ent[eo[j]] << 18;
        ord[p] = (uint16_t)j;
        if ((p & 63u) == 0) row_heads[p >> 6] = (l + 2) >> 2;
    }
    if (over) limits[0] = 1u;
    __syncthreads();
    uint32_t col = 0, row = 0;
    for (int q = 0; q < 8; q++) col += heads[q];
    for (uint32_t q = 0; q < 16; q++) row += row_heads[q];
    if (tid == 0) {
        base = atomicAdd(cursor, (unsigned long long)(col + row));
        r.n = S | nt << 16;
        r.col = (uint32_t)base;
        r.row = (uint32_t)base + col;
        r.cw = r.rw[0] = r.rw[1] = 0;
        for (int q = 0; q < 8; q++) r.cw |= (uint64_t)heads[q] << (8 * q);
        for (uint32_t q = 0; q < 16; q++) r.rw[q >> 3] |= (uint64_t)row_heads[q] << (8 * (q & 7u));
        runs[t] = r;
        BlockTotals* bt = totals + (r.key >> a.tile_bits);
        atomicAdd(&bt->touched, nt);
        atomicAdd(&bt->entries, r.entries);
    }
    __syncthreads();
    if (over || base + col + row > a.capacity) return;  // uniform but for `over`, which ends the build
    const uint32_t wl = tid & 63u, wave = tid >> 6;
    uint32_t* out = words + base * 64;
    for (uint32_t j = 0; j * 64 < nt; j++) {  // a wavefront per slice
        const uint32_t U = heads[j];
        if ((j & 3u) == wave) {
            const uint32_t p = j * 64 + wl;
            const uint32_t n = p < nt ? cnt_at[p] : 0u, v = p < nt ? slot_at[p] : 0u;
            uint32_t w = 0, cur = n ? bits[v] : 0u, rep = 0, last = 0;
            auto next = [&]() -> uint32_t {  // the next segment of the voxel
                if (rep) {
                    rep--;
                    return last;
                }
                while (!cur) cur = bits[++w * kTileVox + v];
                last = w * 32 + (uint32_t)__ffs((int)cur) - 1u;
                cur &= cur - 1u;
                for (uint32_t k = 0; k < nd; k++) rep += dup[k] == (v << 16 | last) ? 1u : 0u;
                return last;
            };
            for (uint32_t u = 0; u < U; u++) {
                uint32_t e = 0;
#pragma unroll
                for (uint32_t i = 0; i < 3; i++)
                    if (3 * u + i < n) e |= (at_turn[next()] + 1u) << (10 * i);
                out[unit_word(u, U, wl)] = e;
            }
        }
        out += U * 64;
    }
    for (uint32_t j = 0; j * 64 < S; j++) {
        const uint32_t U = row_heads[j];
        if ((j & 3u) == wave) {
            const uint32_t p = j * 64 + wl;
            const uint32_t k = p < S ? ord[p] : 0u, n = p < S ? len[k] : 0u, o = eo[k];
            for (uint32_t u = 0; u < U; u++) {
                uint32_t e = 0;
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) {
                    const uint32_t m = 4 * u + i + 1;
                    if (m < n) e |= ((uint32_t)(ent[o + m] - ent[o + m - 1]) & 255u) << (8 * i);
                }
                out[unit_word(u, U, wl)] = e;
            }
        }
        out += U * 64;
    }
}

// the first segment of every plan block
__global__ void k_tile_block_seg(int64_t n_raw, int64_t BS, const int32_t* __restrict__ block_of,
                                 const TileRow* __restrict__ rows, BlockTotals* __restrict__ totals)
{
    const int64_t rb = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (rb < n_raw && block_of[rb] >= 0) totals[rb].seg = rows[rb * BS].seg;
}

// the group's tiles into the table of (block, used tile) descriptors
__global__ void k_tile_table(uint32_t n, int tile_bits, const TileRun* __restrict__ runs,
                             const int32_t* __restrict__ block_of, const uint32_t* __restrict__ index_of,
                             uint32_t n_used, TileDesc* __restrict__ table)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const TileRun r = runs[t];
    TileDesc d{};
    d.seg = r.seg;
    d.n = r.n;
    d.run = t;
    d.tile = r.key & ((1u << tile_bits) - 1u);
    d.col = r.col;
    d.row = r.row;
    d.cw = r.cw;
    d.rw[0] = r.rw[0];
    d.rw[1] = r.rw[1];
    table[(size_t)block_of[r.key >> tile_bits] * n_used + index_of[d.tile]] = d;
}

// ---------------------------------------------------------------- iterations ----
// Both descriptor rows are always there (a row of zeros where there are no columns or no rows), and the arrays
// have kSlack readable elements past the last one, so every first load is issued without a test.
struct PassCols {
    const TileDesc* table;
    const uint32_t* seg_rank;
    const uint16_t* tv;
    const uint32_t* words;
};
struct PassRows {
    const TileDesc* table;
    const uint32_t* seg_ord;
    const uint32_t* words;
    RowPart* part;  // of the block's segments
    uint32_t seg0;  // its first segment
};

// sum of the bytes of w
__device__ __forceinline__ uint32_t byte_sum(uint64_t w)
{
    w = (w & 0x00ff00ff00ff00ffull) + ((w >> 8) & 0x00ff00ff00ff00ffull);
    return (uint32_t)((w * 0x0001000100010001ull) >> 48);
}

// A lane's part of slice j: K pairs of units and an odd last one are loaded at once, needed or not (a slice is
// followed by the next one), so that nothing waits between the loads.
template <int K>
struct Slice {
    const uint32_t* p;
    uint32_t U, tail;
    uint2 u[K];
    __device__ __forceinline__ uint2 pair(uint32_t q) const { return *reinterpret_cast<const uint2*>(p + q * 128); }
    __device__ __forceinline__ void load(const uint32_t* words, uint32_t first, uint64_t w, uint32_t j, uint32_t lane)
    {
        U = (uint32_t)(w >> (8 * j)) & 255u;
        const uint32_t* slice = words + ((size_t)first + byte_sum(w & ((1ull << (8 * j)) - 1ull))) * 64;
        p = slice + 2 * lane;
#pragma unroll
        for (int q = 0; q < K; q++) u[q] = pair(q);
        tail = slice[(U >> 1) * 128 + lane];
    }
    // f(unit number, unit) over the lane's units
    template <class F>
    __device__ __forceinline__ void each(F f) const
    {
        const uint32_t pairs = U >> 1;
#pragma unroll
        for (int q = 0; q < K; q++)
            if ((uint32_t)q < pairs) {
                f(2u * q, u[q].x);
                f(2u * q + 1, u[q].y);
            }
        for (uint32_t q = K; q < pairs; q += 2) {
            const uint2 g0 = pair(q), g1 = pair(q + 1);
            f(2 * q, g0.x);
            f(2 * q + 1, g0.y);
            if (q + 1 < pairs) {
                f(2 * q + 2, g1.x);
                f(2 * q + 3, g1.y);
            }
        }
        if (U & 1u) f(U - 1, tail);
    }
};

constexpr int kPass = 128;  // lanes per tile
// A row of up to 512 entries cannot round while its largest value lies at most 44 powers of two above the lowest bit
// of its values.  The bounds of a whole tile stand for its segments where they keep that (with 2 for the largest
// value at least: the other tiles of a row hold values around 1); elsewhere a segment takes the bounds of its own
// values, so that one tiny voxel holds up the rows through it and not those through its tile.  Rows kernel and pass
// on 256 x 256 x 96, 3.4M histories: 23.6 + 24.3 us without, 9.7 + 24.5 with; a net's image 20.7 + 20.2, 11.6 + 21.7;
// at a limit of 42 the pass of the 8.8M-history plan, which has few such rows, takes 19.7 us instead of 19.0.
constexpr int kWide = 44;

template <int ACC>
__global__ void __launch_bounds__(kPass) k_tile_pass(PassCols c, PassRows w, const double* __restrict__ r,
                                                     float* __restrict__ x)
{
    extern __shared__ double seg0[];  // 0.0, then the updates of block b's segments and the sums of block b + 1's
    __shared__ float xs[kTileVox];
    __shared__ int s_top[2], s_lsb[2];
    double* seg = seg0 + 1;
    const uint32_t ui = blockIdx.x, tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const TileDesc dc = c.table[ui], dr = w.table[ui];
    const uint32_t n_col = dc.n >> 16, n_cseg = dc.n & 0xffffu, n_rseg = dr.n & 0xffffu;
    if (n_cseg == 0 && n_rseg == 0) return;
    float4* xt = (float4*)(x + (size_t)(n_cseg ? dc.tile : dr.tile) * kTileVox);
    // every load that only needs the descriptors: the wavefront's four slices of voxels (sorted by count: a
    // mix of long and short ones) and first two slices of segments
    uint32_t k0 = c.seg_rank[dc.seg + tid], k1 = c.seg_rank[dc.seg + kPass + tid];
    const float4 x_in = xt[tid];
    const uint16_t* tv = c.tv + (size_t)dc.run * kTileVox + lane;
    const uint32_t j0 = wave, j1 = 3 - wave, j2 = 4 + wave, j3 = 7 - wave;
    uint32_t v0 = tv[j0 * 64], v1 = tv[j1 * 64], v2 = tv[j2 * 64], v3 = tv[j3 * 64];
    Slice<2> c0, c1;
    Slice<1> c2, c3;
    c0.load(c.words, dc.col, dc.cw, j0, lane);
    c1.load(c.words, dc.col, dc.cw, j1, lane);
    c2.load(c.words, dc.col, dc.cw, j2, lane);
    c3.load(c.words, dc.col, dc.cw, j3, lane);
    const uint32_t* so = w.seg_ord + dr.seg + lane;
    uint32_t q0 = so[wave * 64], q1 = so[wave * 64 + 128];
    Slice<2> r0, r1;
    r0.load(w.words, dr.row, dr.rw[0], wave, lane);
    r1.load(w.words, dr.row, dr.rw[0], wave + 2, lane);
    k0 = tid < n_cseg ? k0 : 0u;
    k1 = tid + kPass < n_cseg ? k1 : 0u;
    const double u0 = r[k0], u1 = r[k1];
    const uint32_t quad = slot_of_quad(tid);
    xs[quad] = x_in.x;
    xs[quad + 2] = x_in.y;
    xs[quad + 4] = x_in.z;
    xs[quad + 6] = x_in.w;
    if (tid == 0) seg0[0] = 0.0;
    if (tid < n_cseg) seg[tid] = u0;
    if (tid + kPass < n_cseg) seg[tid + kPass] = u1;
    for (uint32_t j = tid + 2 * kPass; j < n_cseg; j += kPass) seg[j] = r[c.seg_rank[dc.seg + j]];
    if (n_cseg) {
        __syncthreads();
        auto column = [&](const auto& s, uint32_t j, uint32_t rec) {
            rec = j * 64 + lane < n_col ? rec : 0u;
            const uint32_t n = rec >> 9;
            ColAcc<ACC> a;
            s.each([&](uint32_t unit, uint32_t e) {
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const double u = seg0[(e >> (10 * i)) & 1023u];
                    if (ACC == PCT_ACCUM_KAHAN32) {  // a zero would move the compensation
                        if (3 * unit + i < n) a.add(u);
                    } else {
                        a.add(u);
                    }
                }
            });
            if (n) xs[rec & 511u] += a.mean(n);
        };
        column(c0, j0, v0);
        column(c1, j1, v1);
        column(c2, j2, v2);
        column(c3, j3, v3);
    }
    __syncthreads();
    const float4 v = make_float4(xs[quad], xs[quad + 2], xs[quad + 4], xs[quad + 6]);
    if (n_cseg) xt[tid] = v;
    if (!n_rseg) return;
    // bounds of the tile's values, for every row through it
    int top = -1000, lsb = 1000;
    term_bounds(v.x, top, lsb);
    term_bounds(v.y, top, lsb);
    term_bounds(v.z, top, lsb);
    term_bounds(v.w, top, lsb);
#pragma unroll
    for (int q = 32; q > 0; q >>= 1) {
        const int t = __shfl_xor(top, q, 64), l = __shfl_xor(lsb, q, 64);
        top = t > top ? t : top;
        lsb = l < lsb ? l : lsb;
    }
    if (lane == 0) {
        s_top[wave] = top;
        s_lsb[wave] = lsb;
    }
    __syncthreads();
    RowPart out;
    out.top = s_top[0] > s_top[1] ? s_top[0] : s_top[1];
    out.lsb = s_lsb[0] < s_lsb[1] ? s_lsb[0] : s_lsb[1];
    RowPart* part = w.part + (dr.seg - w.seg0);
    auto row = [&](const auto& s, uint32_t j, uint32_t rec) {
        rec = j * 64 + lane < n_rseg ? rec : 0u;
        const uint32_t n = (rec >> 10) & 255u;
        uint32_t at = rec >> 18;
        double sum = (double)xs[at];
        s.each([&](uint32_t unit, uint32_t e) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                at += (uint32_t)(int32_t)(int8_t)(e >> (8 * i));
                const float f = xs[at];
                sum += 4 * unit + i + 1 < n ? (double)f : 0.0;
            }
        });
        if (n) seg[rec & 1023u] = sum;
    };
    // the bounds of a segment's own values; only tiles whose values span many powers of two take them
    auto own_bounds = [&](const auto& s, uint32_t j, uint32_t rec) {
        const uint32_t n = j * 64 + lane < n_rseg ? (rec >> 10) & 255u : 0u;
        uint32_t at = rec >> 18;
        if (!n) return;
        RowPart p;
        p.top = -1000;
        p.lsb = 1000;
        term_bounds(xs[at], p.top, p.lsb);
        s.each([&](uint32_t unit, uint32_t e) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                at += (uint32_t)(int32_t)(int8_t)(e >> (8 * i));
                if (4 * unit + i + 1 < n) term_bounds(xs[at], p.top, p.lsb);
            }
        });
        p.sum = seg[rec & 1023u];
        part[rec & 1023u] = p;
    };
    const bool wide = (out.top > 1 ? out.top : 1) - out.lsb > kWide;
    row(r0, wave, q0);
    row(r1, wave + 2, q1);
    if (wide) {
        own_bounds(r0, wave, q0);
        own_bounds(r1, wave + 2, q1);
    }
    for (uint32_t j = wave + 4; j * 64 < n_rseg; j += 2) {
        Slice<2> rj;
        rj.load(w.words, dr.row + (j < 8 ? 0u : byte_sum(dr.rw[0])), j < 8 ? dr.rw[0] : dr.rw[1], j & 7u, lane);
        const uint32_t rec = so[j * 64];
        row(rj, j, rec);
        if (wide) own_bounds(rj, j, rec);
    }
    if (wide) return;
    __syncthreads();
    for (uint32_t j = tid; j < n_rseg; j += kPass) {
        out.sum = seg[j];
        part[j] = out;
    }
}

constexpr int kRowLanes = 8;

// per history: its segments' partial sums, or the sum in list order where they may round, and u_i
__global__ void __launch_bounds__(kBlock) k_tile_rows(int64_t proc, const TileRow* __restrict__ rows,
                                                      const uint32_t* __restrict__ place,
                                                      const RowPart* __restrict__ part, uint32_t seg0,
                                                      const uint32_t* __restrict__ vox, const float* __restrict__ x,
                                                      TileIndex at, double lambda, double* __restrict__ r)
{
    constexpr int G = kRowLanes;
    const int lane = threadIdx.x & (G - 1);
    const int64_t k = (int64_t)blockIdx.x * (kBlock / G) + threadIdx.x / G;
    if (k >= proc) return;  // the G lanes of a history leave together
    const TileRow d = rows[k];
    if (d.n_seg == 0) return;  // no column reads this history's update
    double s = 0.0;
    int top = -1000, lsb = 1000;
    for (uint32_t q = lane; q < d.n_seg; q += 2 * G) {
        const bool two = q + G < d.n_seg;
        const uint32_t a = place[d.seg + q], b = two ? place[d.seg + q + G] : a;
        const RowPart p = part[a - seg0], p2 = part[b - seg0];
        s += p.sum;
        if (two) s += p2.sum;
        top = p.top > top ? p.top : top;
        lsb = p.lsb < lsb ? p.lsb : lsb;
        top = p2.top > top ? p2.top : top;
        lsb = p2.lsb < lsb ? p2.lsb : lsb;
    }
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        s += __shfl_xor(s, o, G);
        const int t = __shfl_xor(top, o, G), l = __shfl_xor(lsb, o, G);
        top = t > top ? t : top;
        lsb = l < lsb ? l : lsb;
    }
    const int cnt = (int)d.cnt;
    if (!order_free(top, lsb, cnt)) s = row_sum_ordered<G>(vox + d.off, cnt, x, lane, at);
    if (lane == 0) {
        const double L = d.chord;
        const double ax = s * L;
        const double aa = (double)pct_sqf(L) * (double)cnt;
        r[k] = L * (((double)d.wepl - ax) / aa) * lambda;
    }
}

// (b_i - L_i sum_j x[v_ij])^2 of every history of the plan, in visiting order, from the tiled image
__global__ void __launch_bounds__(kBlock) k_residual_tiles(int64_t n, const TileRow* __restrict__ rows,
                                                           const uint32_t* __restrict__ vox,
                                                           const float* __restrict__ x, TileIndex at, int min_len,
                                                           double* __restrict__ r2)
{
    constexpr int G = 16;
    const int lane = threadIdx.x & (G - 1);
    const int64_t stride = (int64_t)gridDim.x * (blockDim.x / G);
    for (int64_t p = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / G; p < n; p += stride) {
        const TileRow d = rows[p];
        const int cnt = (int)d.cnt;
        const double part = row_sum<G>(vox + d.off, cnt, x, lane, at);
        if (lane == 0) {
            const double e = (double)d.wepl - d.chord * part;
            r2[p] = cnt >= min_len ? e * e : 0.0;
        }
    }
}

int bits_for(int64_t n)  // smallest b with 2^b >= n
{
    int b = 0;
    while ((1ll << b) < n) b++;
    return b;
}

void magic(uint32_t d, uint64_t* m, int* s)
{
    const int l = bits_for(d);
    *s = 31 + l;
    *m = ((1ull << (31 + l)) + d - 1) / d;
}

TileGeom tile_geom(const pct_params& P)
{
    TileGeom g;
    g.C = (uint32_t)P.columns;
    g.R = (uint32_t)P.rows;
    g.ntx = (g.C + 15) / 16;
    g.nty = (g.R + 15) / 16;
    g.nt = g.ntx * g.nty * (uint32_t)((P.slices + 1) / 2);
    magic(g.C, &g.mC, &g.sC);
    magic(g.R, &g.mR, &g.sR);
    return g;
}

template <class T>
int grow(pct_ctx* ctx, T** p, int64_t* cap, int64_t need)
{
    if (need <= *cap && *p) return PCT_OK;
    *cap = 0;
    PCT_TRY(pct_alloc(ctx, p, need));
    *cap = need;
    return PCT_OK;
}
// The segments, tiles and lists of one group (its MLP lists exist).  *fits is false when a tile exceeds the
// limits of the packed lists.
int build_group(pct_ctx* ctx, TilePlan& T, TileGroup& G, const CutArgs& ca, int bin_bits, BlockTotals* totals, bool* fits)
{
    hipStream_t s = ctx->stream;
    TileScratch& W = T.scratch;
    const int64_t H = ca.n;
    *fits = false;
    PCT_TRY(grow(ctx, &W.hkey, &W.cap_hkey, 2 * H));
    PCT_TRY(grow(ctx, &W.hidx, &W.cap_hidx, 2 * H));
    PCT_TRY(grow(ctx, &W.nseg, &W.cap_nseg, H + 1));
    PCT_TRY(grow(ctx, &W.q0, &W.cap_q0, H + 1));
    uint32_t* order = W.hidx + H;
    CutArgs a = ca;
    a.order = order;
    const int n_blocks = (int)((H + a.BS - 1) / a.BS), hbits = bits_for(n_blocks) + bin_bits;
    size_t need = 0, t = 0;
    PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, need, W.hkey, W.hkey + H, W.hidx, order, (int)H, 0,
                                                          hbits, s));
    PCT_CHECK_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, t, W.nseg, W.q0, (int)(H + 1), s));
    PCT_TRY(pct_grow_cub(ctx, std::max(need, t)));
    // visiting order and the histories' segments
    hipLaunchKernelGGL(k_tile_hist_keys, dim3(grid_for(H)), dim3(kBlock), 0, s, a.h0, H, a.BS, a.rb0, a.proc_raw,
                       ctx->bin_num, bin_bits, W.hkey, W.hidx);
    size_t tb = ctx->cub_tmp_bytes;
    PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(ctx->cub_tmp, tb, W.hkey, W.hkey + H, W.hidx, order, (int)H, 0,
                                                          hbits, s));
    PCT_CHECK_HIP(ctx, hipMemsetAsync(W.limits, 0, kLimits * sizeof(uint32_t), s));
    PCT_CHECK_HIP(ctx, hipMemsetAsync(W.nseg + H, 0, sizeof(uint32_t), s));
    const unsigned cg = pct_grid_capped(H * 16, kBlock, 1u << 18);
    hipLaunchKernelGGL(k_tile_cut<false>, dim3(cg), dim3(kBlock), 0, s, a, W.nseg, (const uint32_t*)nullptr,
                       (TileRow*)nullptr, (uint32_t*)nullptr, (uint32_t*)nullptr, (SegRec*)nullptr);
    tb = ctx->cub_tmp_bytes;
    PCT_CHECK_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(ctx->cub_tmp, tb, W.nseg, W.q0, (int)(H + 1), s));
    uint32_t Q = 0;
    PCT_TRY(pct_read(ctx, &Q, W.q0 + H, sizeof(uint32_t)));
    if (Q > (1u << 30)) return PCT_OK;
    G.segs = Q;
    G.n_runs = 0;
    if (Q == 0) {  // nothing to sort, but every history has its row, without segments
        hipLaunchKernelGGL(k_tile_cut<true>, dim3(cg), dim3(kBlock), 0, s, a, (uint32_t*)nullptr, W.q0, T.rows,
                           (uint32_t*)nullptr, (uint32_t*)nullptr, (SegRec*)nullptr);
        PCT_CHECK_HIP(ctx, hipGetLastError());
        *fits = true;
        return PCT_OK;
    }
    PCT_TRY(grow(ctx, &W.keys, &W.cap_keys, 2 * (int64_t)Q));
    PCT_TRY(grow(ctx, &W.idx, &W.cap_idx, 2 * (int64_t)Q));
    PCT_TRY(grow(ctx, &W.recs, &W.cap_recs, 2 * (int64_t)Q));
    PCT_TRY(grow(ctx, &W.runs, &W.cap_runs, 2 * (int64_t)Q));
    PCT_TRY(grow(ctx, &G.seg_rank, &G.cap_seg_rank, (int64_t)Q + kSlack));
    PCT_TRY(grow(ctx, &G.seg_ord, &G.cap_seg_ord, (int64_t)Q + kSlack));
    PCT_TRY(grow(ctx, &G.place, &G.cap_place, (int64_t)Q));
    uint32_t *keys_sorted = W.keys + Q, *idx_sorted = W.idx + Q, *run_start = W.runs + Q;
    SegRec* recs = (SegRec*)W.recs;
    const int kbits = bits_for(n_blocks) + a.tile_bits;
    size_t t2 = 0;
    PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, need, W.keys, keys_sorted, W.idx, idx_sorted, (int)Q,
                                                          0, kbits, s));
    PCT_CHECK_HIP(ctx, hipcub::DeviceRunLengthEncode::Encode(nullptr, t, keys_sorted, W.keys, W.runs, W.n_runs, (int)Q, s));
    PCT_CHECK_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, t2, W.runs, run_start, (int)Q, s));
    PCT_TRY(pct_grow_cub(ctx, std::max(need, std::max(t, t2))));
    hipLaunchKernelGGL(k_tile_cut<true>, dim3(cg), dim3(kBlock), 0, s, a, (uint32_t*)nullptr, W.q0, T.rows, W.keys,
                       W.idx, recs);
    tb = ctx->cub_tmp_bytes;
    PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(ctx->cub_tmp, tb, W.keys, keys_sorted, W.idx, idx_sorted, (int)Q,
                                                          0, kbits, s));
    tb = ctx->cub_tmp_bytes;
    PCT_CHECK_HIP(ctx, hipcub::DeviceRunLengthEncode::Encode(ctx->cub_tmp, tb, keys_sorted, W.keys, W.runs, W.n_runs,
                                                             (int)Q, s));
    uint32_t nr = 0, lim[kLimits] = {};
    PCT_TRY(pct_read(ctx, &nr, W.n_runs, sizeof(uint32_t)));
    if (nr < 1 || nr > Q) {
        ctx->err = "DROP tiles: run count out of range in a group";
        return PCT_E_LIMIT;
    }
    G.n_runs = nr;
    PCT_TRY(grow(ctx, &G.tv, &G.cap_tv, (int64_t)nr * kTileVox));
    PCT_TRY(grow(ctx, &G.runs, &G.cap_runs, (int64_t)nr));
    tb = ctx->cub_tmp_bytes;
    PCT_CHECK_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(ctx->cub_tmp, tb, W.runs, run_start, (int)nr, s));
    SegRec* segs = recs + Q;
    hipLaunchKernelGGL(k_tile_gather, dim3(grid_for(Q)), dim3(kBlock), 0, s, Q, idx_sorted, recs, segs, G.seg_rank,
                       G.place);
    uint32_t* entries = W.keys + Q;  // the sorted keys are spent
    PCT_TRY(grow(ctx, &W.need, &W.cap_need, 4 * (int64_t)nr));
    uint32_t *need_sorted = W.need + nr, *by_need = W.need + 3 * (size_t)nr;
    hipLaunchKernelGGL(k_tile_runs, dim3(grid_for((int64_t)nr * 64)), dim3(kBlock), 0, s, nr, a.tile_bits, W.keys,
                       run_start, W.runs, segs, G.runs, entries, W.need, W.need + 2 * (size_t)nr, T.used);
    PCT_CHECK_HIP(ctx, hipcub::DeviceReduce::Max(nullptr, need, W.runs, W.limits + 1, (int)nr, s));
    PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, t, W.need, need_sorted, W.need + 2 * (size_t)nr, by_need,
                                                          (int)nr, 0, 8, s));
    PCT_TRY(pct_grow_cub(ctx, std::max(need, t)));
    tb = ctx->cub_tmp_bytes;
    PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(ctx->cub_tmp, tb, W.need, need_sorted, W.need + 2 * (size_t)nr,
                                                          by_need, (int)nr, 0, 8, s));
    hipLaunchKernelGGL(k_tile_classes, dim3(1), dim3(64), 0, s, nr, need_sorted, W.limits + 3);
    tb = ctx->cub_tmp_bytes;
    PCT_CHECK_HIP(ctx, hipcub::DeviceReduce::Max(ctx->cub_tmp, tb, W.runs, W.limits + 1, (int)nr, s));
    tb = ctx->cub_tmp_bytes;
    PCT_CHECK_HIP(ctx, hipcub::DeviceReduce::Max(ctx->cub_tmp, tb, entries, W.limits + 2, (int)nr, s));
    PCT_TRY(pct_read(ctx, lim, W.limits, sizeof(lim)));
    if (lim[1] > kMaxSeg || lim[2] > kMaxEnt || lim[2 + kClasses] < nr) return PCT_OK;
    const uint32_t* classes = lim + 3;
    PCT_CHECK_HIP(ctx, hipFuncSetAttribute((const void*)k_tile_fill, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kClassLds[kClasses - 1]));
    T.max_seg = std::max<int64_t>(T.max_seg, lim[1]);
    // the lists, in room for the usual share of padding and of unused slots; again when the cursor passed it
    int64_t want = (int64_t)(1.5 * (double)G.entries_hint) / 128 + 64 + (int64_t)nr;
    for (int attempt = 0; attempt < 2; attempt++) {
        PCT_TRY(grow(ctx, &G.words, &G.cap_words, want * 64 + kSlack));
        PCT_CHECK_HIP(ctx, hipMemsetAsync(W.cursor, 0, sizeof(uint64_t), s));
        if (attempt) PCT_CHECK_HIP(ctx, hipMemsetAsync(totals, 0, n_blocks * sizeof(BlockTotals), s));
        for (int k = kClasses - 1; k >= 0; k--) {  // the largest first
            const uint32_t from = k ? classes[k - 1] : 0u, to = classes[k];
            if (to <= from) continue;
            const FillArgs f{a.g, a.tile_bits, a.slot0, a.vox, segs, by_need + from, (uint64_t)((G.cap_words - kSlack) / 64)};
            hipLaunchKernelGGL(k_tile_fill, dim3(to - from), dim3(kBlock), kClassLds[k], s, f, G.runs, G.tv, G.seg_ord,
                               G.words, (unsigned long long*)W.cursor, W.limits, totals);
        }
        PCT_CHECK_HIP(ctx, hipGetLastError());
        uint64_t total = 0;
        PCT_CHECK_HIP(ctx, hipMemcpyAsync(&total, W.cursor, sizeof(uint64_t), hipMemcpyDeviceToHost, s));
        PCT_TRY(pct_read(ctx, lim, W.limits, sizeof(lim)));
        if (lim[0] || total >= (1ull << 32)) return PCT_OK;
        if ((int64_t)total * 64 + kSlack <= G.cap_words) {
            *fits = true;
            return PCT_OK;
        }
        want = (int64_t)total;
    }
    ctx->err = "DROP tiles: list space";
    return PCT_E_LIMIT;
}

template <typename K, typename... Args>
void timed_launch(K kernel, dim3 g, dim3 blk, size_t lds, hipStream_t s, std::vector<hipEvent_t>* ev, Args... args)
{
    if (!ev) {
        hipLaunchKernelGGL(kernel, g, blk, lds, s, args...);
        return;
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    hipExtLaunchKernelGGL(kernel, g, blk, lds, s, e0, e1, 0, args...);
    ev->push_back(e0);
    ev->push_back(e1);
}

}  // namespace

void pct_tile_plan_free(TilePlan* T)
{
    for (TileGroup& G : T->groups) {
        pct_free(&G.seg_rank);
        pct_free(&G.seg_ord);
        pct_free(&G.place);
        pct_free(&G.tv);
        pct_free(&G.runs);
        pct_free(&G.words);
    }
    T->groups.clear();
    TileScratch& W = T->scratch;
    pct_free(&W.hkey);
    pct_free(&W.hidx);
    pct_free(&W.nseg);
    pct_free(&W.q0);
    pct_free(&W.keys);
    pct_free(&W.idx);
    pct_free(&W.recs);
    pct_free(&W.runs);
    pct_free(&W.cursor);
    pct_free(&W.need);
    pct_free(&W.n_runs);
    pct_free(&W.limits);
    W = TileScratch{};
    pct_free(&T->rows);
    pct_free(&T->used);
    pct_free(&T->index_of);
    pct_free(&T->block_of);
    pct_free(&T->totals);
    pct_free(&T->table);
    pct_free(&T->part);
    pct_free(&T->r);
    pct_free(&T->x);
    const double too_dense = T->too_dense;
    *T = TilePlan{};
    T->too_dense = too_dense;
}

// Whether the tiles take the plan of these flags and sizes (before the lists exist).
bool pct_tiles_wanted(const pct_ctx* ctx)
{
    if (ctx->drop_flags != (PCT_DROP_SPATIAL_ORDER | PCT_DROP_BRICKS | PCT_DROP_COLS_SLICED) || ctx->drop_tiles == 0 ||
        ctx->P.drop_block_size > kMaxBlock || ctx->n_recon <= 0)
        return false;
    return ctx->drop_tiles == 1 || ctx->list_slots >= kMinTotalSlots;
}

int pct_tiles_prepare(pct_ctx* ctx, const MlpLaunch* mlp, bool* done, bool* lists_built)
{
    const pct_params& P = ctx->P;
    hipStream_t s = ctx->stream;
    const int64_t n = ctx->n_recon, BS = P.drop_block_size;
    DropPlan& D = ctx->plan;
    TilePlan& T = D.tile;
    const bool pipe = mlp != nullptr;
    *done = *lists_built = false;
    T.ready = false;
    const TileGeom g = tile_geom(P);
    const int tile_bits = std::max(1, bits_for(g.nt)), bin_bits = bits_for((int64_t)P.num_bins + 1);
    if (tile_bits > 22 || bin_bits > 31) return PCT_OK;
    const int64_t max_blocks = 1ll << (32 - std::max(tile_bits, bin_bits));
    const int64_t n_raw = (n + BS - 1) / BS;

    const double nb_est = std::max(1.0, (double)n / BS);
    // The rule, on list slots of a block and the sampled paths through the tiles (see kMinSlots and the constants after it)
    double density = 0.0;
    if (ctx->drop_tiles != 1) {
        uint32_t* count = nullptr;  // then the reached tiles and the most paths
        PCT_TRY(pct_scratch(ctx, SCR_TILE_COUNT, &count, (size_t)g.nt + 2));
        PCT_CHECK_HIP(ctx, hipMemsetAsync(count, 0, ((size_t)g.nt + 2) * sizeof(uint32_t), s));
        SampleArgs a{n, (n + kSample - 1) / kSample, g, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, pct_geom(P),
                     ctx->list_off, ctx->list_cnt, ctx->list_vox};
        if (pipe) {
            a.x0 = ctx->h[0], a.y0 = ctx->h[1], a.z0 = ctx->h[2];
            a.x1 = ctx->h[3], a.y1 = ctx->h[4], a.z1 = ctx->h[5];
        }
        const dim3 sg(grid_for((n + a.every - 1) / a.every));
        if (g.nt <= kSampleTiles)
            hipLaunchKernelGGL(k_tile_sample<true>, sg, dim3(kBlock), g.nt * sizeof(uint32_t), s, a, count);
        else
            hipLaunchKernelGGL(k_tile_sample<false>, sg, dim3(kBlock), 0, s, a, count);
        hipLaunchKernelGGL(k_tile_reach, dim3(std::min(grid_for(g.nt), 256u)), dim3(kBlock), 0, s, g.nt, count, count + g.nt);
        uint32_t reach[2];
        PCT_TRY(pct_read(ctx, reach, count + g.nt, sizeof(reach)));
        const double block_slots = (double)ctx->list_slots / nb_est, paths = (double)reach[1] * a.every / nb_est;
        density = block_slots / std::max(1u, reach[0]);
        if (density < (block_slots < kSmallBlock ? kMinSlotsSmall : kMinSlots) ||
            (paths >= kManyPaths && block_slots < kMinSpread * paths) || paths >= kMaxPaths || density >= T.too_dense)
            return PCT_OK;
    }

    // processed histories per raw block (DS.cu:9558 floors them) and their list capacities
    std::vector<int32_t> proc(n_raw), block_of(n_raw, -1);
    for (int64_t rb = 0; rb < n_raw; rb++) {
        const int64_t m = std::min(BS, n - rb * BS);
        const int64_t p = P.quirk_a3_drop_floor ? (m / P.histories_per_block) * P.histories_per_block : m;
        proc[rb] = p > 0 ? (int32_t)p : 0;
    }
    int32_t* proc_dev = nullptr;
    int64_t *cap_dev = nullptr, *slot_dev = nullptr;
    PCT_TRY(pct_scratch(ctx, SCR_BLOCK_PROC, &proc_dev, n_raw + 1));
    PCT_TRY(pct_scratch(ctx, SCR_BLOCK_ENTRIES, &cap_dev, n_raw + 1));
    PCT_TRY(pct_scratch(ctx, SCR_BLOCK_SLOTS, &slot_dev, n_raw + 1));
    std::vector<int64_t> cap(n_raw), first_slot(n_raw);
    PCT_CHECK_HIP(ctx, hipMemcpyAsync(proc_dev, proc.data(), n_raw * sizeof(int32_t), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_tile_block_caps, dim3(grid_for(n_raw)), dim3(kBlock), 0, s, n_raw, BS, n,
                       ctx->list_off, cap_dev, slot_dev);
    PCT_CHECK_HIP(ctx, hipMemcpyAsync(cap.data(), cap_dev, n_raw * sizeof(int64_t), hipMemcpyDeviceToHost, s));
    PCT_TRY(pct_read(ctx, first_slot.data(), slot_dev, n_raw * sizeof(int64_t)));

    // groups of whole blocks
    D.blocks.clear();
    D.groups.clear();
    const int64_t max_entries = std::min(ctx->drop_group_entries, kTileGroupEntries);
    std::vector<int64_t> slot0;  // per group: its first list slot
    for (int64_t rb = 0; rb < n_raw; rb++) {
        if (proc[rb] <= 0) continue;
        if (cap[rb] >= (1ll << 30)) return PCT_OK;
        const int64_t start = rb * BS, m = std::min(BS, n - start);
        bool fresh = D.groups.empty();
        if (!fresh) {
            const DropPlan::Group& q = D.groups.back();
            fresh = q.entries + cap[rb] > max_entries || rb - q.hist_begin / BS + 1 > max_blocks ||
                    start + m - q.hist_begin > (1ll << 30);
        }
        if (fresh) {
            D.groups.push_back(DropPlan::Group{(int64_t)D.blocks.size(), 0, 0, 0, start, start});
            slot0.push_back(first_slot[rb]);
        }
        DropPlan::Group& q = D.groups.back();
        q.n_blocks = rb - q.hist_begin / BS + 1;
        q.entries += cap[rb];
        q.hist_end = start + m;
        DropPlan::Block bk{};
        bk.start = start;
        bk.proc = proc[rb];
        bk.group = (int64_t)D.groups.size() - 1;
        block_of[rb] = (int32_t)D.blocks.size();
        D.blocks.push_back(bk);
    }
    const int64_t ng = (int64_t)D.groups.size(), nb = (int64_t)D.blocks.size();
    if (nb == 0) return PCT_OK;
    while ((int64_t)T.groups.size() < ng) T.groups.emplace_back();
    PCT_TRY(grow(ctx, &T.rows, &T.cap_rows, n));
    PCT_TRY(grow(ctx, &T.used, &T.cap_used, g.nt));
    PCT_TRY(grow(ctx, &T.totals, &T.cap_totals, n_raw));
    PCT_TRY(grow(ctx, &T.block_of, &T.cap_block_of, n_raw));
    TileScratch& W = T.scratch;
    if (!W.n_runs) PCT_TRY(pct_alloc(ctx, &W.n_runs, 1));
    if (!W.limits) PCT_TRY(pct_alloc(ctx, &W.limits, kLimits));
    if (!W.cursor) PCT_TRY(pct_alloc(ctx, &W.cursor, 1));
    PCT_CHECK_HIP(ctx, hipMemsetAsync(T.used, 0, g.nt, s));
    PCT_CHECK_HIP(ctx, hipMemsetAsync(T.totals, 0, n_raw * sizeof(BlockTotals), s));

    // With `mlp`, the MLP kernel runs group by group on stream2; a group is cut on `s` once its lists exist.
    // Every return drains stream2.
    struct MlpQueue {
        pct_ctx* ctx;
        std::vector<hipEvent_t> ev;
        hipEvent_t t0 = nullptr, t1 = nullptr;
        ~MlpQueue()
        {
            if (ctx->stream2) (void)hipStreamSynchronize(ctx->stream2);
            for (hipEvent_t e : ev) (void)hipEventDestroy(e);
            if (t0) (void)hipEventDestroy(t0);
            if (t1) (void)hipEventDestroy(t1);
        }
    } q{ctx, {}};
    if (pipe) {
        if (!ctx->stream2) PCT_CHECK_HIP(ctx, hipStreamCreateWithFlags(&ctx->stream2, hipStreamNonBlocking));
        hipStream_t s2 = ctx->stream2;
        hipEvent_t ready = nullptr;
        PCT_CHECK_HIP(ctx, hipEventCreateWithFlags(&ready, hipEventDisableTiming));
        q.ev.push_back(ready);
        PCT_CHECK_HIP(ctx, hipEventRecord(ready, s));
        PCT_CHECK_HIP(ctx, hipStreamWaitEvent(s2, ready, 0));
        PCT_CHECK_HIP(ctx, hipEventCreate(&q.t0));
        PCT_CHECK_HIP(ctx, hipEventCreate(&q.t1));
        PCT_CHECK_HIP(ctx, hipEventRecord(q.t0, s2));
        int64_t prev = 0;
        for (int64_t gi = 0; gi <= ng; gi++) {
            const int64_t h1 = gi < ng ? D.groups[gi].hist_end : n;
            if (h1 > prev) PCT_TRY((*mlp)(prev, h1, s2));
            prev = std::max(prev, h1);
            hipEvent_t e = nullptr;
            PCT_CHECK_HIP(ctx, hipEventCreateWithFlags(&e, hipEventDisableTiming));
            q.ev.push_back(e);
            PCT_CHECK_HIP(ctx, hipEventRecord(e, s2));
        }
        PCT_CHECK_HIP(ctx, hipEventRecord(q.t1, s2));
    }
    T.max_seg = 0;
    bool fits = true;
    for (int64_t gi = 0; gi < ng && fits; gi++) {
        const DropPlan::Group& gr = D.groups[gi];
        if (pipe) PCT_CHECK_HIP(ctx, hipStreamWaitEvent(s, q.ev[gi + 1], 0));
        const int64_t rb0 = gr.hist_begin / BS;
        CutArgs a{gr.hist_begin, gr.hist_end - gr.hist_begin, BS, rb0, slot0[gi], g, tile_bits, P.min_mlp_length,
                  proc_dev, nullptr, ctx->list_off, ctx->list_cnt, ctx->list_vox, ctx->chord, ctx->wepl};
        T.groups[gi].entries_hint = gr.entries;
        PCT_TRY(build_group(ctx, T, T.groups[gi], a, bin_bits, T.totals + rb0, &fits));
    }
    if (pipe) {
        PCT_CHECK_HIP(ctx, hipStreamWaitEvent(s, q.ev[ng + 1], 0));
        PCT_CHECK_HIP(ctx, hipStreamSynchronize(ctx->stream2));
        float ms = 0;
        (void)hipEventElapsedTime(&ms, q.t0, q.t1);
        ctx->t_mlp_kernel = ms;
        *lists_built = true;
    }
    if (!fits) {
        if (density > 0.0) T.too_dense = density;  // lists this dense go to the sort at once from here on
        return PCT_OK;
    }
    int64_t segs = 0;
    for (int64_t gi = 0; gi < ng; gi++) segs += T.groups[gi].segs;
    if (segs == 0) return PCT_OK;  // no history is long enough to update a voxel
    // the tiles any block touches, and the descriptor of every (block, used tile)
    std::vector<uint8_t> used(g.nt);
    std::vector<BlockTotals> totals(n_raw);
    PCT_CHECK_HIP(ctx, hipMemcpyAsync(T.block_of, block_of.data(), n_raw * sizeof(int32_t), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_tile_block_seg, dim3(grid_for(n_raw)), dim3(kBlock), 0, s, n_raw, BS, T.block_of, T.rows, T.totals);
    PCT_CHECK_HIP(ctx, hipMemcpyAsync(used.data(), T.used, g.nt, hipMemcpyDeviceToHost, s));
    PCT_TRY(pct_read(ctx, totals.data(), T.totals, n_raw * sizeof(BlockTotals)));
    std::vector<uint32_t> index_of(g.nt, 0);
    int64_t U = 0;
    for (uint32_t k = 0; k < g.nt; k++)
        if (used[k]) index_of[k] = (uint32_t)U++;
    T.n_used = U;
    if (nb * U > kMaxTable) {
        if (density > 0.0) T.too_dense = density;
        return PCT_OK;
    }
    PCT_TRY(grow(ctx, &T.index_of, &T.cap_index_of, g.nt));
    PCT_TRY(grow(ctx, &T.table, &T.cap_table, (nb + 1) * U + 1));
    PCT_CHECK_HIP(ctx, hipMemcpyAsync(T.index_of, index_of.data(), g.nt * sizeof(uint32_t), hipMemcpyHostToDevice, s));
    PCT_CHECK_HIP(ctx, hipMemsetAsync(T.table, 0, (nb + 1) * U * sizeof(TileDesc), s));  // the last row stays empty
    for (int64_t gi = 0; gi < ng; gi++) {
        const TileGroup& G = T.groups[gi];
        if (G.n_runs)
            hipLaunchKernelGGL(k_tile_table, dim3(grid_for(G.n_runs)), dim3(kBlock), 0, s, G.n_runs, tile_bits, G.runs,
                               T.block_of + D.groups[gi].hist_begin / BS, T.index_of, (uint32_t)U, T.table);
    }
    PCT_CHECK_HIP(ctx, hipGetLastError());
    // first and last segment of every block (its histories' segments are sorted together)
    int64_t max_part = 0, max_proc = 0;
    T.block_seg.assign(nb, 0);
    for (int64_t b = 0; b < nb; b++) {
        DropPlan::Block& bk = D.blocks[b];
        const bool last = b + 1 == nb || D.blocks[b + 1].group != bk.group;
        const BlockTotals& t = totals[bk.start / BS];
        const int64_t end = last ? T.groups[bk.group].segs : totals[D.blocks[b + 1].start / BS].seg;
        T.block_seg[b] = t.seg;
        max_part = std::max(max_part, end - (int64_t)t.seg);
        max_proc = std::max(max_proc, bk.proc);
        bk.n_vox = t.touched;
        bk.entries = t.entries;
    }
    PCT_TRY(grow(ctx, &T.part, &T.cap_part, max_part + 1));
    PCT_TRY(grow(ctx, &T.r, &T.cap_r, max_proc + 1));
    const int64_t nx = (int64_t)g.nt * kTileVox;
    if (T.cap_x < nx || !T.x) {
        PCT_TRY(grow(ctx, &T.x, &T.cap_x, nx));
        PCT_CHECK_HIP(ctx, hipMemsetAsync(T.x, 0, nx * sizeof(float), s));  // padding stays 0
    }
    D.desc_all = D.groups.front().hist_begin == 0 && D.groups.back().hist_end == n;
    for (int64_t gi = 1; gi < ng; gi++) D.desc_all = D.desc_all && D.groups[gi].hist_begin == D.groups[gi - 1].hist_end;
    PCT_CHECK_HIP(ctx, hipStreamSynchronize(s));
    D.groups_bucketed = D.groups_sorted = 0;
    D.flags = ctx->drop_flags;
    D.ready = true;
    T.ready = true;
    *done = true;
    return PCT_OK;
}

int pct_tiles_enter(pct_ctx* ctx, bool enter)
{
    const pct_params& P = ctx->P;
    hipLaunchKernelGGL(k_x_tiles, dim3(grid_for(P.num_voxels)), dim3(kBlock), 0, ctx->stream, (int64_t)P.num_voxels,
                       ctx->x, ctx->plan.tile.x, TileIndex{tile_geom(P)}, enter ? 1 : 0);
    PCT_CHECK_HIP(ctx, hipGetLastError());
    return PCT_OK;
}

// `iterations` DROP iterations on the tiled image.
int pct_tiles_iterate(pct_ctx* ctx, int iterations, DropTiming* timing)
{
    const pct_params& P = ctx->P;
    hipStream_t s = ctx->stream;
    DropPlan& D = ctx->plan;
    TilePlan& T = D.tile;
    const int64_t nb = (int64_t)D.blocks.size();
    if (nb == 0 || iterations <= 0) return PCT_OK;
    std::vector<hipEvent_t> ev_rows, ev_pass;
    std::vector<hipEvent_t>*er = timing ? &ev_rows : nullptr, *ep = timing ? &ev_pass : nullptr;
    const TileIndex at{tile_geom(P)};
    const size_t lds = (size_t)(T.max_seg + 1) * sizeof(double);
    // the arrays of a group without segments do not exist; its descriptors are empty, so another group's serve
    const TileGroup* any = nullptr;
    for (const TileGroup& G : T.groups)
        if (G.words) any = &G;
    auto group = [&](int64_t b) -> const TileGroup& {
        const TileGroup& G = T.groups[D.blocks[b < nb ? b : 0].group];
        return G.words ? G : *any;
    };
    // b == nb: the empty row of descriptors
    auto cols = [&](int64_t b) {
        const TileGroup& G = group(b);
        return PassCols{T.table + b * T.n_used, G.seg_rank, G.tv, G.words};
    };
    auto rows = [&](int64_t b) {
        const TileGroup& G = group(b);
        return PassRows{T.table + b * T.n_used, G.seg_ord, G.words, T.part, b < nb ? T.block_seg[b] : 0u};
    };
    auto pass = [&](const PassCols& c, const PassRows& w) {
        const dim3 grid((unsigned)T.n_used);
        if (P.drop_accum == PCT_ACCUM_FP64)
            timed_launch(k_tile_pass<PCT_ACCUM_FP64>, grid, dim3(kPass), lds, s, ep, c, w, T.r, T.x);
        else if (P.drop_accum == PCT_ACCUM_FP32)
            timed_launch(k_tile_pass<PCT_ACCUM_FP32>, grid, dim3(kPass), lds, s, ep, c, w, T.r, T.x);
        else
            timed_launch(k_tile_pass<PCT_ACCUM_KAHAN32>, grid, dim3(kPass), lds, s, ep, c, w, T.r, T.x);
    };
    pass(cols(nb), rows(0));
    for (int it = 0; it < iterations; it++)
        for (int64_t b = 0; b < nb; b++) {
            const DropPlan::Block& bk = D.blocks[b];
            const TileGroup& G = T.groups[bk.group];
            timed_launch(k_tile_rows, dim3((unsigned)((bk.proc * kRowLanes + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, er, bk.proc, T.rows + bk.start,
                         G.place, T.part, T.block_seg[b], ctx->list_vox, T.x, at, P.lambda, T.r);
            const bool more = b + 1 < nb || it + 1 < iterations;
            pass(cols(b), rows(!more ? nb : b + 1 < nb ? b + 1 : 0));
            if (timing) timing->histories += bk.proc;
        }
    PCT_CHECK_HIP(ctx, hipGetLastError());
    if (timing) {
        PCT_CHECK_HIP(ctx, hipStreamSynchronize(s));
        auto sum = [](std::vector<hipEvent_t>& ev, double* ms, int64_t* launches) {
            for (size_t j = 0; j + 1 < ev.size(); j += 2) {
                float a = 0;
                (void)hipEventElapsedTime(&a, ev[j], ev[j + 1]);
                *ms += a;
                ++*launches;
            }
            for (hipEvent_t e : ev) (void)hipEventDestroy(e);
        };
        sum(ev_rows, &timing->scatter_ms, &timing->scatter_launches);
        sum(ev_pass, &timing->apply_ms, &timing->apply_launches);
    }
    return PCT_OK;
}

// (b - a.x)^2 per history into ctx->res_r2, from the tiled image
int pct_tiles_residual(pct_ctx* ctx)
{
    const pct_params& P = ctx->P;
    PCT_TRY(pct_tiles_enter(ctx, true));
    const int64_t n = ctx->n_recon;
    hipLaunchKernelGGL(k_residual_tiles, dim3(pct_grid_capped(n * 16, kBlock, 1u << 20)), dim3(kBlock), 0, ctx->stream, n,
                       ctx->plan.tile.rows, ctx->list_vox, ctx->plan.tile.x, TileIndex{tile_geom(P)}, P.min_mlp_length,
                       ctx->res_r2);
    PCT_CHECK_HIP(ctx, hipGetLastError());
    return PCT_OK;
}
