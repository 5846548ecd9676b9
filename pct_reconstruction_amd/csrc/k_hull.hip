// k_hull.hip — stage (b): SC / MSC / SM hull carving, edge detection, FBP hull and hull selection.
//
// Carving is one lane per history walking its straight entry->exit chord voxel by voxel (SC_GPU
// DS.cu:6681, MSC_GPU :6799, SM_GPU :6997).  SC clears voxels: here the walk sets bits in a
// bit-packed "carved" mask with 32-bit atomicOr (one word per 32 voxels, 1/8 of the bytes of the
// reference's bool image); the hull is the cylinder mask without the carved bits.  MSC/SM count
// traversals with 32-bit integer atomics, which are exact and order independent.  By default one walk
// serves every method, the histories in sinogram-bin order, with the visits of a workgroup summed in
// LDS first: in a hash table (k_carve_all; 3.4x faster than one walk per method on the head-50M workload), or, for MSC and
// SM counts of many histories on fine grids, in the counts of an image tile that the chords pass through (k_carve_tiles).
#include <hipcub/hipcub.hpp>

#include "internal.h"
#include "walk.h"

namespace {

constexpr int kBlock = 256;
inline unsigned grid_for(int64_t n, int block = kBlock) { return pct_grid_for(n, block); }

// initialize_hull_GPU, DS.cu:6659-6669
__device__ __forceinline__ int inside_cylinder(const DevGeom& g, int column, int row)
{
    double x = (column - g.C / 2 + 0.5) * g.VW;
    double y = (g.R / 2 - row - 0.5) * g.VH;
    return (pct_sqf(x) + pct_sqf(y)) < pct_sqf(g.Rc);
}

__global__ void k_init_counts(DevGeom g, int32_t* counts)
{
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.NV) return;
    int c = (int)(v % g.C), r = (int)((v / g.C) % g.R);
    counts[v] = inside_cylinder(g, c, r);
}

// The chord of a history: take_3D_step's line (DS.cu:11392).
__device__ __forceinline__ void chord_line(float xe, float ye, float ze, float xx, float yx, float zx, Walk3& w)
{
    w.xs = xe;
    w.ys = ye;
    w.zs = ze;
    w.xm = (xe <= xx) - (xe >= xx);
    w.ym = (ye <= yx) - (ye >= yx);
    w.zm = (ze <= zx) - (ze >= zx);
    w.dy_dx = (double)((yx - ye) / (xx - xe));
    w.dz_dx = (double)((zx - ze) / (xx - xe));
    w.dz_dy = (double)((zx - ze) / (yx - ye));
    w.dx_dy = (double)((xx - xe) / (yx - ye));
    w.dx_dz = (double)((xx - xe) / (zx - ze));
    w.dy_dz = (double)((yx - ye) / (zx - ze));
}

// The entry->exit walk of SC/MSC/SM (take_2D_step_GPU :11346, take_3D_step_GPU :11392).  Visits
// every voxel from the entry voxel up to, excluding, the exit voxel.  The walk also stops at a
// negative voxel coordinate or after 4*(C+R+S)+16 steps: there the reference indexes out of bounds
// or does not terminate.
template <class Visit>
__device__ void carve_walk(const DevGeom& g, float xe, float ye, float ze, float xx, float yx, float zx, Visit visit)
{
    const int C = g.C, R = g.R, S = g.S;
    Walk3 w;
    chord_line(xe, ye, ze, xx, yx, zx, w);
    w.ax = w.ay = w.az = w.at = 0;
    w.vx = pct_calc_voxel(g.X0, xe, g.VW);
    w.vy = pct_calc_voxel(g.Y0, ye, g.VH);
    w.vz = pct_calc_voxel(g.Z0, ze, g.VT);
    const int vxo = pct_calc_voxel(g.X0, xx, g.VW), vyo = pct_calc_voxel(g.Y0, yx, g.VH), vzo = pct_calc_voxel(g.Z0, zx, g.VT);
    const int64_t voxel_out = vxo + (int64_t)vyo * C + (int64_t)vzo * C * R;
    auto address = [&] { return w.vx + (int64_t)w.vy * C + (int64_t)w.vz * C * R; };
    int64_t voxel = address();
    bool end_walk = voxel == voxel_out || w.vx >= C || w.vy >= R || w.vz >= S || w.vx < 0 || w.vy < 0 || w.vz < 0;
    const int cap = 4 * (C + R + S) + 16;
    int steps = 0;
    auto stepped = [&] {
        voxel = address();
        end_walk = voxel == voxel_out || w.vx >= C || w.vy >= R || w.vz >= S || w.vx < 0 || w.vy < 0 || ++steps > cap;
    };
    if (w.zm != 0) {
        w.begin(g);
        while (!end_walk) {
            visit(voxel);
            int full;
            bool clamped;
            w.step(g, &full, &clamped);
            stepped();
        }
        return;
    }
    double x = xe, y = ye;
    double x_to_go = pct_dist(g.X0, x, PCT_X_INC, w.xm, g.VW, w.vx);
    double y_to_go = pct_dist(g.Y0, y, PCT_Y_INC, w.ym, g.VH, w.vy);
    while (!end_walk) {
        visit(voxel);
        const double y_ext = fabs(w.dx_dy) * y_to_go;
        if (x_to_go <= y_ext) {
            w.vx += w.xm;
            x = pct_edge(g.X0, w.vx, g.VW, PCT_X_INC, w.xm);
            y = pct_corr(w.dy_dx, x, xe, ye);
            x_to_go = g.VW;
            y_to_go = pct_dist(g.Y0, y, PCT_Y_INC, w.ym, g.VH, w.vy);
        } else {
            w.vy -= w.ym;
            y = pct_edge(g.Y0, w.vy, g.VH, PCT_Y_INC, w.ym);
            x = pct_corr(w.dx_dy, y, ye, xe);
            x_to_go = pct_dist(g.X0, x, PCT_X_INC, w.xm, g.VW, w.vx);
            y_to_go = g.VH;
        }
        if (x_to_go == 0) { x_to_go = g.VW; w.vx += w.xm; }
        if (y_to_go == 0) { y_to_go = g.VH; w.vy -= w.ym; }
        w.vz = w.vz > 0 ? w.vz : 0;
        stepped();
    }
}

struct HistPtrs {
    const float *xe, *ye, *ze, *xx, *yx, *zx, *wepl;
};

// method: 0 SC (WEPL in [SC_LOWER, SC_UPPER], DS.cu:6686), 1 MSC ([MSC_LOWER, MSC_UPPER], :6806),
// 2 SM (WEPL >= SM_LOWER, :7004)
__global__ void k_carve(int64_t n, DevGeom g, HistPtrs hp, int method, double lo, double hi, uint32_t* carved,
                        int32_t* counts)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float w = hp.wepl[i];
    bool take = (method == 2) ? (w >= lo) : ((w <= hi) && (w >= lo));
    if (!take) return;
    if (method == 0) {
        carve_walk(g, hp.xe[i], hp.ye[i], hp.ze[i], hp.xx[i], hp.yx[i], hp.zx[i],
                   [&](int64_t v) { atomicOr(&carved[v >> 5], 1u << (v & 31)); });
    } else {
        carve_walk(g, hp.xe[i], hp.ye[i], hp.ze[i], hp.xx[i], hp.yx[i], hp.zx[i],
                   [&](int64_t v) { atomicAdd(&counts[v], 1); });
    }
}

// One walk per history for every method whose WEPL gate it passes (SC, MSC and SM walk the same chord),
// with the histories taken in sinogram-bin order through `perm`: the 256 histories of a workgroup are then
// neighbouring, nearly parallel chords, and their voxel visits collect in an LDS hash table of the
// workgroup (open addressing, kProbe linear probes) before one global atomic per distinct voxel and method
// at the end.  A visit that finds no slot goes to global memory directly.  The counts are integers, so
// the result does not depend on the order of the visits.
//
// A slot's three counters share one 32-bit word: MSC in bits 0-9, SM in 10-19, SC in 20-29.  A lane that
// reads a field at the spill count or more before its add takes the add back and goes to global memory.
// A field then holds at most `spill` committed visits plus one visit in flight per lane, and the kernel
// caps spill at 1023 - BLOCK, so no field carries into its neighbour.  (A chord visits a voxel once, so a
// field passes BLOCK only on degenerate walks; a small spill count exercises the path.)
constexpr int kProbe = 8;
constexpr uint32_t kEmpty = 0xffffffffu, kField = 1023u;

struct Gates {
    int sc, msc, sm;  // methods on
    double sc_lo, sc_hi, msc_lo, msc_hi, sm_lo;
    uint32_t spill;  // 1..512, capped at 1023 - BLOCK
};

template <int TABLE, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_carve_all(int64_t n, const uint32_t* __restrict__ perm, DevGeom g,
                                                      HistPtrs hp, Gates gt, uint32_t* __restrict__ carved,
                                                      int32_t* __restrict__ msc_counts,
                                                      int32_t* __restrict__ sm_counts)
{
    static_assert(TABLE == 4096 || TABLE == 8192 || TABLE == 16384, "power-of-two table");
    static_assert(BLOCK <= 512, "10-bit fields");
    const uint32_t spill = min(gt.spill, 1023u - BLOCK);
    constexpr int kShift = TABLE == 4096 ? 20 : TABLE == 8192 ? 19 : 18;  // top log2(TABLE) bits of the product
    __shared__ uint32_t keys[TABLE];
    __shared__ uint32_t cnt[TABLE];
    for (int k = threadIdx.x; k < TABLE; k += blockDim.x) {
        keys[k] = kEmpty;
        cnt[k] = 0u;
    }
    __syncthreads();
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) {
        const int64_t i = perm[t];
        const float w = hp.wepl[i];
        const bool sc = gt.sc && w <= gt.sc_hi && w >= gt.sc_lo;
        const bool msc = gt.msc && w <= gt.msc_hi && w >= gt.msc_lo;
        const bool sm = gt.sm && w >= gt.sm_lo;
        const uint32_t inc = (uint32_t)msc | ((uint32_t)sm << 10) | ((uint32_t)sc << 20);
        if (inc) {
            carve_walk(g, hp.xe[i], hp.ye[i], hp.ze[i], hp.xx[i], hp.yx[i], hp.zx[i], [&](int64_t v64) {
                const uint32_t v = (uint32_t)v64;
                uint32_t slot = (v * 2654435761u) >> kShift;
                bool local = false;
                for (int q = 0; q < kProbe; q++) {
                    uint32_t k = keys[slot];
                    if (k == kEmpty) k = atomicCAS(&keys[slot], kEmpty, v);
                    if (k == kEmpty || k == v) {
                        const uint32_t old = atomicAdd(&cnt[slot], inc);
                        local = (old & kField) < spill && ((old >> 10) & kField) < spill && (old >> 20) < spill;
                        if (!local) atomicSub(&cnt[slot], inc);
                        break;
                    }
                    slot = (slot + 1) & (TABLE - 1);
                }
                if (!local) {
                    if (sc) atomicOr(&carved[v >> 5], 1u << (v & 31));
                    if (msc) atomicAdd(&msc_counts[v], 1);
                    if (sm) atomicAdd(&sm_counts[v], 1);
                }
            });
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < TABLE; k += blockDim.x) {
        const uint32_t v = keys[k];
        if (v == kEmpty) continue;
        const uint32_t c = cnt[k];
        if (c >> 20) atomicOr(&carved[v >> 5], 1u << (v & 31));
        if (c & kField) atomicAdd(&msc_counts[v], (int32_t)(c & kField));
        if ((c >> 10) & kField) atomicAdd(&sm_counts[v], (int32_t)((c >> 10) & kField));
    }
}

// ---------------------------------------------------------------- carving by tiles ----
// Counting in LDS needs many visits per voxel and workgroup, and the chords of a workgroup share few voxels when
// bins hold few histories: with 16M head histories the hash table of k_carve_all overflows, and 21 of its 55 ms went
// to visits that missed it, 9 to its flush and 12 to its probes.  Here the image is cut into tiles of 64 x 64 x 2
// voxels, 32 KB of packed counts.  A walk (k_carve_cut) finds where each chord enters a tile, the entries are sorted
// by tile, and a workgroup takes a chunk of one tile's entries (k_carve_tiles), walks each chord on inside the tile
// and adds the tile's counts to memory once: no visit needs a probe, a returned value or a global atomic.  The walk
// is taken twice, but is cheaper (walk.h: 8.9 ms for the cut, 12 before), and both are bound by its FP64 arithmetic.
// 16M histories, 256 x 256 x 48: gather 2.0, cut 8.9, sort 0.7, tiles 6.7 ms, 18.5 in all (54.6 before); 6M: 6.5
// (29.8).
constexpr int kCT = 64, kCTZ = 2, kCTVox = kCT * kCT * kCTZ;
constexpr int kCarveBlock = 512;

__device__ __forceinline__ uint32_t carve_tile(int vx, int vy, int vz, int ntx, int nty)
{
    return ((uint32_t)(vz >> 1) * nty + (uint32_t)(vy >> 6)) * ntx + (uint32_t)(vx >> 6);
}

// The histories of a batch in visiting order, and how many tile entries each may have: one more than the tile steps
// between its first and last voxel, and one for a start on a tile's far edge; none when no method takes it.  cap[n] is
// 0: the scan's total.
__global__ void k_carve_gather(int64_t n, const uint32_t* __restrict__ perm, DevGeom g, HistPtrs hp, Gates gt,
                               CarveRec* __restrict__ recs, uint32_t* __restrict__ cap)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t == n) cap[t] = 0;
    if (t >= n) return;
    const int64_t i = perm[t];
    const float w = hp.wepl[i];
    CarveRec r{hp.xe[i], hp.ye[i], hp.ze[i], hp.xx[i], hp.yx[i], hp.zx[i], 0u, 0.0f};
    if (gt.msc && w <= gt.msc_hi && w >= gt.msc_lo) r.inc |= 1u;
    if (gt.sm && w >= gt.sm_lo) r.inc |= 1u << 15;
    if (gt.sc && w <= gt.sc_hi && w >= gt.sc_lo) r.inc |= 1u << 30;
    recs[t] = r;
    uint32_t c = 0;
    if (r.inc) {
        auto tiles = [](int a, int b, int n, int shift) {
            return abs((min(max(b, 0), n) >> shift) - (min(max(a, 0), n) >> shift));
        };
        c = (uint32_t)(2 + tiles(pct_calc_voxel(g.X0, r.xe, g.VW), pct_calc_voxel(g.X0, r.xx, g.VW), g.C, 6) +
                       tiles(pct_calc_voxel(g.Y0, r.ye, g.VH), pct_calc_voxel(g.Y0, r.yx, g.VH), g.R, 6) +
                       tiles(pct_calc_voxel(g.Z0, r.ze, g.VT), pct_calc_voxel(g.Z0, r.zx, g.VT), g.S, 1));
    }
    cap[t] = c;
}

// The walk of every chord, one entry per tile it passes: key tile, value history | state << 32 (voxel in the tile
// 13 bits, axis 2 bits (3: the start), full 3 bits, visits 14 bits).  What the tile walk does not take is counted
// here with global atomics: chords without a z slope (the 2D walk), what follows once the z voxel was clamped or a
// step left the voxel as it was (voxels can come twice there: an entry's visits are distinct), and what finds no
// room.  Unused room gets the key n_tiles.
__global__ void __launch_bounds__(256) k_carve_cut(int64_t n, DevGeom g, const CarveRec* __restrict__ recs,
                                                   const uint32_t* __restrict__ off, int ntx, int nty, uint32_t n_tiles,
                                                   uint32_t* __restrict__ keys, uint64_t* __restrict__ vals,
                                                   uint32_t* __restrict__ carved, int32_t* __restrict__ msc_counts,
                                                   int32_t* __restrict__ sm_counts)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const CarveRec r = recs[t];
    uint32_t q = off[t];
    const uint32_t end = off[t + 1];
    auto count = [&](int64_t v) {
        if (r.inc >> 30) atomicOr(&carved[v >> 5], 1u << (v & 31));
        if (r.inc & 1u) atomicAdd(&msc_counts[v], 1);
        if (r.inc & (1u << 15)) atomicAdd(&sm_counts[v], 1);
    };
    if (r.inc) {
        Walk3 w;
        chord_line(r.xe, r.ye, r.ze, r.xx, r.yx, r.zx, w);
        if (w.zm == 0) {
            carve_walk(g, r.xe, r.ye, r.ze, r.xx, r.yx, r.zx, count);
        } else {
            w.vx = pct_calc_voxel(g.X0, r.xe, g.VW);
            w.vy = pct_calc_voxel(g.Y0, r.ye, g.VH);
            w.vz = pct_calc_voxel(g.Z0, r.ze, g.VT);
            const int ox = pct_calc_voxel(g.X0, r.xx, g.VW), oy = pct_calc_voxel(g.Y0, r.yx, g.VH),
                      oz = pct_calc_voxel(g.Z0, r.zx, g.VT);
            const int64_t out = ox + (int64_t)oy * g.C + (int64_t)oz * g.C * g.R;
            const int none = -1;  // no voxel of the image: image addresses have 31 bits
            const int at_out = out >= 0 && out < g.NV ? (int)out : none;
            w.ax = w.xm;
            w.ay = -w.ym * g.C;
            w.az = -w.zm * g.C * g.R;
            auto address = [&] { return w.vx + (w.vy + w.vz * g.R) * g.C; };
            auto ended = [&] {
                return w.at == at_out || (uint32_t)w.vx >= (uint32_t)g.C || (uint32_t)w.vy >= (uint32_t)g.R || w.vz >= g.S;
            };
            // a start outside the image has no address
            bool end_walk = (uint32_t)w.vx >= (uint32_t)g.C || (uint32_t)w.vy >= (uint32_t)g.R ||
                            (uint32_t)w.vz >= (uint32_t)g.S;
            w.at = end_walk ? none : address();
            end_walk = end_walk || w.at == at_out;
            w.begin(g);
            int tx = w.vx, ty = w.vy, tz = w.vz;  // where the entry began
            uint32_t state = 3u << 13, visits = 0;
            bool direct = q == end;
            auto flush = [&] {
                if (visits) {
                    keys[q] = carve_tile(tx, ty, tz, ntx, nty);
                    vals[q++] = (uint64_t)t | (uint64_t)(state | visits << 18 | (tz & 1) << 12 | (ty & 63) << 6 |
                                                         (tx & 63)) << 32;
                    visits = 0;
                }
            };
            const int cap = 4 * (g.C + g.R + g.S) + 16;
            int steps = 0;
            while (!end_walk) {
                if (direct) count(w.at);
                else visits++;
                int full;
                bool clamped;
                const int last = w.at, axis = w.step(g, &full, &clamped);
                if (clamped) w.at = address();
                end_walk = ended() || ++steps > cap;
                if (clamped || w.at == last || ((w.vx ^ tx) | (w.vy ^ ty)) >> 6 || (w.vz ^ tz) >> 1) {
                    flush();
                    direct = direct || clamped || w.at == last || q == end;
                    tx = w.vx;
                    ty = w.vy;
                    tz = w.vz;
                    state = (uint32_t)(axis << 13 | full << 15);
                }
            }
            flush();
        }
    }
    for (; q < end; q++) {
        keys[q] = n_tiles;
        vals[q] = 0;
    }
}

// start[t]: first sorted entry of tile t; first_chunk[t]: the chunks of the tiles before t
__global__ void __launch_bounds__(1024) k_carve_chunks(uint32_t n_tiles, uint32_t n, uint32_t chunk,
                                                       const uint32_t* __restrict__ keys, uint32_t* __restrict__ start,
                                                       uint32_t* __restrict__ first_chunk)
{
    __shared__ uint32_t part[1024], total;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    for (uint32_t t0 = 0; t0 <= n_tiles; t0 += 1024) {
        const uint32_t t = t0 + threadIdx.x;
        auto find = [&](uint32_t key) {
            uint32_t lo = 0, hi = n;
            while (lo < hi) {
                const uint32_t mid = lo + (hi - lo) / 2;
                if (keys[mid] < key) lo = mid + 1;
                else hi = mid;
            }
            return lo;
        };
        uint32_t mine = 0;
        if (t <= n_tiles) {
            const uint32_t a = find(t);
            start[t] = a;
            if (t < n_tiles) mine = (find(t + 1) - a + chunk - 1) / chunk;
        }
        part[threadIdx.x] = mine;
        __syncthreads();
        for (uint32_t o = 1; o < 1024; o <<= 1) {
            const uint32_t y = threadIdx.x >= o ? part[threadIdx.x - o] : 0u;
            __syncthreads();
            part[threadIdx.x] += y;
            __syncthreads();
        }
        if (t <= n_tiles) first_chunk[t] = total + part[threadIdx.x] - mine;
        __syncthreads();
        if (threadIdx.x == 1023) total += part[1023];
        __syncthreads();
    }
}

// A chunk of one tile's entries per workgroup: a chord visits a voxel of the tile once (the walk is monotone up to
// a clamp), so a field of 15 bits holds the counts of up to 32767 entries.
__global__ void __launch_bounds__(kCarveBlock) k_carve_tiles(DevGeom g, const CarveRec* __restrict__ recs,
                                                             const uint64_t* __restrict__ vals, uint32_t n_tiles,
                                                             uint32_t chunk, const uint32_t* __restrict__ start,
                                                             const uint32_t* __restrict__ first_chunk, int ntx, int nty,
                                                             uint32_t* __restrict__ carved,
                                                             int32_t* __restrict__ msc_counts,
                                                             int32_t* __restrict__ sm_counts)
{
    __shared__ uint32_t cnt[kCTVox];
    const uint32_t b = blockIdx.x;
    if (b >= first_chunk[n_tiles]) return;
    uint32_t lo = 0, hi = n_tiles;  // first_chunk[lo] <= b < first_chunk[hi]
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (first_chunk[mid] <= b) lo = mid;
        else hi = mid;
    }
    const uint32_t tile = lo, e0 = start[tile] + (b - first_chunk[tile]) * chunk;
    const uint32_t e1 = min(e0 + chunk, start[tile + 1]);
    const int bx = (int)(tile % (uint32_t)ntx) * kCT, by = (int)(tile / (uint32_t)ntx % (uint32_t)nty) * kCT,
              bz = (int)(tile / ((uint32_t)ntx * nty)) * kCTZ;
    for (uint32_t k = threadIdx.x; k < (uint32_t)kCTVox; k += kCarveBlock) cnt[k] = 0u;
    __syncthreads();
    for (uint32_t e = e0 + threadIdx.x; e < e1; e += kCarveBlock) {
        const uint64_t v = vals[e];
        const CarveRec r = recs[(uint32_t)v];
        const uint32_t s = (uint32_t)(v >> 32);
        Walk3 w;
        chord_line(r.xe, r.ye, r.ze, r.xx, r.yx, r.zx, w);
        w.vx = bx + (int)(s & 63u);
        w.vy = by + (int)((s >> 6) & 63u);
        w.vz = bz + (int)((s >> 12) & 1u);
        const int axis = (int)(s >> 13) & 3, full = (int)(s >> 15) & 7;
        if (axis == 3) w.begin(g);
        else w.resume(g, axis, full);
        w.ax = w.xm;
        w.ay = -w.ym * 64;
        w.az = -w.zm * 4096;
        w.at = (int)(s & 8191u);
        for (uint32_t visits = s >> 18;;) {
            if (r.inc & 0x3fffffffu) atomicAdd(&cnt[w.at], r.inc & 0x3fffffffu);
            if (r.inc >> 30) atomicOr(&cnt[w.at], 1u << 30);
            if (--visits == 0) break;
            int f;
            bool clamped;
            w.step(g, &f, &clamped);
        }
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < (uint32_t)kCTVox; k += kCarveBlock) {
        const uint32_t n = cnt[k];
        if (!n) continue;
        const int64_t v = (bx + (int64_t)(k & 63u)) + (by + (int64_t)((k >> 6) & 63u)) * g.C +
                          (bz + (int64_t)(k >> 12)) * g.C * g.R;
        if (n >> 30) atomicOr(&carved[v >> 5], 1u << (v & 31));
        if (n & 0x7fffu) atomicAdd(&msc_counts[v], (int32_t)(n & 0x7fffu));
        if ((n >> 15) & 0x7fffu) atomicAdd(&sm_counts[v], (int32_t)((n >> 15) & 0x7fffu));
    }
}

// SC hull = cylinder mask without the carved voxels
__global__ void k_sc_finish(DevGeom g, const uint32_t* carved, uint8_t* hull)
{
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.NV) return;
    int c = (int)(v % g.C), r = (int)((v / g.C) % g.R);
    bool cut = (carved[v >> 5] >> (v & 31)) & 1u;
    hull[v] = (uint8_t)(inside_cylinder(g, c, r) && !cut);
}

__device__ __forceinline__ bool on_rim(const DevGeom& g, int column, int row)
{
    float x = (float)((column - g.C / 2 + 0.5) * g.VW);
    float y = (float)((g.R / 2 - row - 0.5) * g.VH);
    double m = g.VW > g.VH ? g.VW : g.VH;
    return (x * x + y * y) >= pct_sqf(g.Rc - m / 2);
}

__device__ __forceinline__ int max_diff(const DevGeom& g, const int32_t* counts, int c, int r, int64_t so)
{
    int md = 0;
    if ((r != 0) && (r != g.R - 1) && (c != 0) && (c != g.C - 1)) {
        int32_t own = counts[so + c + r * g.C];
        for (int rr = r - 1; rr <= r + 1; rr++)
            for (int cc = c - 1; cc <= c + 1; cc++) {
                int d = own - counts[so + cc + rr * g.C];
                if (d > md) md = d;
            }
    }
    return md;
}

// MSC_edge_detection_GPU (DS.cu:6911-6957) reading unmodified counts (the race-free semantics of the
// two-buffer version :6958-6985).
__global__ void k_msc_edge(DevGeom g, const int32_t* counts, int32_t* hull, int thresh)
{
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.NV) return;
    int c = (int)(v % g.C), r = (int)((v / g.C) % g.R);
    int64_t so = (v / ((int64_t)g.C * g.R)) * g.C * g.R;
    int md = max_diff(g, counts, c, r, so);
    int32_t out = (md > thresh || counts[v] > thresh) ? 0 : 1;
    if (on_rim(g, c, r)) out = 0;
    hull[v] = out;
}

// carve_differences (DS.cu:6616) + the host threshold scan (:7118-7134): per slice, the count at the
// first pixel (in pixel order) holding the largest 3x3 difference.  One workgroup per slice; ties
// resolved to the lowest pixel index.
__global__ void k_sm_threshold(DevGeom g, const int32_t* counts, int32_t* thr)
{
    __shared__ int s_diff[kBlock];
    __shared__ int s_pix[kBlock];
    const int s = blockIdx.x;
    const int64_t so = (int64_t)s * g.C * g.R;
    int best = 0, best_pix = 0x7fffffff;
    for (int pix = threadIdx.x; pix < g.C * g.R; pix += blockDim.x) {
        int d = max_diff(g, counts, pix % g.C, pix / g.C, so);
        if (d > best || (d == best && d > 0 && pix < best_pix)) {
            best = d;
            best_pix = pix;
        }
    }
    s_diff[threadIdx.x] = best;
    s_pix[threadIdx.x] = best_pix;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            int d2 = s_diff[threadIdx.x + w], p2 = s_pix[threadIdx.x + w];
            int d1 = s_diff[threadIdx.x], p1 = s_pix[threadIdx.x];
            if (d2 > d1 || (d2 == d1 && p2 < p1)) {
                s_diff[threadIdx.x] = d2;
                s_pix[threadIdx.x] = p2;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) thr[s] = (s_diff[0] > 0) ? counts[so + s_pix[0]] : 0;
}

// SM_edge_detection_GPU, DS.cu:7160-7175
__global__ void k_sm_edge(DevGeom g, const int32_t* counts, const int32_t* thr, int32_t* hull, double scale)
{
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.NV) return;
    int c = (int)(v % g.C), r = (int)((v / g.C) % g.R);
    int s = (int)(v / ((int64_t)g.C * g.R));
    int32_t out = (counts[v] > scale * thr[s]) ? 1 : 0;
    if (on_rim(g, c, r)) out = 0;
    hull[v] = out;
}

// FBP_image_2_hull_GPU, DS.cu:6592-6603
__global__ void k_fbp_hull(DevGeom g, const float* image, uint8_t* hull, double threshold)
{
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.NV) return;
    int c = (int)(v % g.C), r = (int)((v / g.C) % g.R);
    double x = -g.Rc + (c + 0.5) * g.VW;
    double y = g.Rc - (r + 0.5) * g.VH;
    double d2 = (double)(pct_sqf(x) + pct_sqf(y));
    hull[v] = (uint8_t)(((double)image[v] > threshold) && (d2 < (double)pct_sqf(g.Rc)));
}

__global__ void k_int_to_bool(int64_t n, const int32_t* in, uint8_t* out)
{
    int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v < n) out[v] = (uint8_t)(in[v] == 1);
}

}  // namespace

DevGeom pct_geom(const pct_params& P)
{
    DevGeom g;
    g.C = P.columns;
    g.R = P.rows;
    g.S = P.slices;
    g.NV = P.num_voxels;
    g.X0 = P.x_zero_coordinate;
    g.Y0 = P.y_zero_coordinate;
    g.Z0 = P.z_zero_coordinate;
    g.VW = P.voxel_width;
    g.VH = P.voxel_height;
    g.VT = P.voxel_thickness;
    g.Rc = P.recon_cyl_radius;
    g.H = P.recon_cyl_height;
    g.PI = P.pi;
    return g;
}

namespace {

// Histories from which the counts of MSC and SM go by tiles.  Preprocessing on a 256 x 256 head grid, table / tiles:
// 0.25M histories 4.1 / 3.0 ms, 2M 20 / 11, 16M 73 / 40; on a 90 x 74 grid 0.15M 1.19 / 1.25 (3.38 / 3.57 in a new
// context, which allocates the scratch), 0.3M 1.63 / 1.53.  SC alone keeps the table at any size: its gate takes few
// histories, and a visit that misses only sets a bit (2M histories on a 200 x 200 cylinder grid, a whole
// reconstruction: 65.3 ms by table, 66.0 by tiles).
constexpr int64_t kCarveTilesMin = 1 << 18;

// On coarse grids a workgroup's chords share their voxels, the table's counts stay in LDS and a chord has too few visits
// to pay for its entries and their sort.  Binning and carve by table | tiles, ms, MSC and SM unless noted, with the
// histories per voxel: 64 x 64 x 24 0.3M (3) 0.51 | 0.52, 4M (41) 1.46 | 2.03; 64 x 64 x 48 1M (5) 0.93 | 0.80, SM alone
// 0.64 | 0.86; 96 x 96 x 64 4M (7) 2.68 | 2.70, 12M (20) 6.1 | 7.7; 128 x 128 x 24 4M (10) 2.99 | 2.89, SM alone
// 2.37 | 2.26, 12M (31) 7.0 | 8.4; 128 x 128 x 96 12M (8) 11.4 | 9.3; 180 x 180 x 24 12M (15) 11.3 | 10.4.
bool carve_tiles_worth(const pct_params& P, int64_t n)
{
    const int64_t methods = (P.msc_on != 0) + (P.sm_on != 0), sides = P.columns + P.rows;
    return n >= kCarveTilesMin && methods * sides >= 200 && 23 * n <= sides * P.num_voxels;
}

void carve_tiles_free(CarveScratch& W)
{
    pct_free(&W.recs);
    pct_free(&W.cap);
    pct_free(&W.off);
    pct_free(&W.keys);
    pct_free(&W.vals);
    pct_free(&W.tiles);
    W = CarveScratch{};
}

// The counts by tiles, in batches of histories (in visiting order ctx->u32_d).  *done: the histories counted; fewer
// than n, with PCT_OK, where there was no memory for the rest or the batches are limited.
int carve_by_tiles(pct_ctx* ctx, const DevGeom& g, const HistPtrs& hp, const Gates& gt, int64_t n, int64_t* done)
{
    hipStream_t s = ctx->stream;
    CarveScratch& W = ctx->carve;
    const int ntx = (g.C + kCT - 1) / kCT, nty = (g.R + kCT - 1) / kCT, ntz = (g.S + kCTZ - 1) / kCTZ;
    const int64_t tiles = (int64_t)ntx * nty * ntz;
    const uint32_t n_tiles = (uint32_t)tiles;
    // 4M histories (0.9 GB on the 256 x 256 head grid), fewer where a chord may pass very many tiles
    const int64_t batch = std::min<int64_t>(ctx->carve_batch, (int64_t)(1 << 28) / (2 + ntx + nty + ntz));
    int bits = 1;
    while ((1ll << bits) < tiles + 1) bits++;
    auto grow = [&](auto** p, int64_t* cap, int64_t need) -> int {
        if (need <= *cap) return PCT_OK;
        *cap = 0;
        PCT_TRY(pct_alloc(ctx, p, need));
        *cap = need;
        return PCT_OK;
    };
    auto no_memory = [&](int rc) {
        if (rc != PCT_E_NOMEM) return rc;
        (void)hipGetLastError();
        ctx->err.clear();
        carve_tiles_free(W);
        return (int)PCT_OK;
    };
    for (*done = 0; *done < n;) {
        if (ctx->carve_tile_batches == ctx->carve_batches) return PCT_OK;
        const int64_t m = std::min(batch, n - *done);
        size_t scan = 0, sort = 0;
        int rc = grow(&W.recs, &W.cap_recs, m);
        if (rc == PCT_OK) rc = grow(&W.cap, &W.cap_cap, m + 1);
        if (rc == PCT_OK) rc = grow(&W.off, &W.cap_off, m + 1);
        if (rc == PCT_OK) rc = grow(&W.tiles, &W.cap_tiles, 2 * (tiles + 1));
        if (rc != PCT_OK) return no_memory(rc);
        PCT_CHECK_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, scan, W.cap, W.off, (int)(m + 1), s));
        rc = pct_grow_cub(ctx, scan);
        if (rc != PCT_OK) return no_memory(rc);
        hipLaunchKernelGGL(k_carve_gather, dim3(grid_for(m + 1)), dim3(kBlock), 0, s, m, ctx->u32_d + *done, g, hp, gt,
                           W.recs, W.cap);
        scan = ctx->cub_tmp_bytes;
        PCT_CHECK_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(ctx->cub_tmp, scan, W.cap, W.off, (int)(m + 1), s));
        uint32_t total = 0;
        PCT_TRY(pct_read(ctx, &total, W.off + m, sizeof(uint32_t)));
        if (total > 0) {
            uint32_t *keys, *sorted_keys, *start = W.tiles, *first_chunk = W.tiles + tiles + 1;
            uint64_t *vals, *sorted_vals;
            const int64_t room = 2 * ((int64_t)total + total / 16);
            rc = grow(&W.keys, &W.cap_keys, room);
            if (rc == PCT_OK) rc = grow(&W.vals, &W.cap_vals, room);
            if (rc != PCT_OK) return no_memory(rc);
            keys = W.keys;
            sorted_keys = keys + total;
            vals = W.vals;
            sorted_vals = vals + total;
            PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, sort, keys, sorted_keys, vals, sorted_vals,
                                                                  (int)total, 0, bits, s));
            rc = pct_grow_cub(ctx, sort);
            if (rc != PCT_OK) return no_memory(rc);
            sort = ctx->cub_tmp_bytes;
            hipLaunchKernelGGL(k_carve_cut, dim3(pct_grid_for(m, 256)), dim3(256), 0, s, m, g, W.recs, W.off, ntx, nty,
                               n_tiles, keys, vals, ctx->sc_carved, ctx->msc_counts, ctx->sm_counts);
            PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(ctx->cub_tmp, sort, keys, sorted_keys, vals,
                                                                  sorted_vals, (int)total, 0, bits, s));
            // several thousand workgroups where there is work for them; 15-bit counts
            const uint32_t chunk = std::min(32767u, std::max(2048u, total / 4096u));
            hipLaunchKernelGGL(k_carve_chunks, dim3(1), dim3(1024), 0, s, n_tiles, total, chunk, sorted_keys, start,
                               first_chunk);
            hipLaunchKernelGGL(k_carve_tiles, dim3(total / chunk + n_tiles + 1), dim3(kCarveBlock), 0, s, g, W.recs,
                               sorted_vals, n_tiles, chunk, start, first_chunk, ntx, nty, ctx->sc_carved,
                               ctx->msc_counts, ctx->sm_counts);
            PCT_CHECK_HIP(ctx, hipGetLastError());
        }
        *done += m;
        ctx->carve_tile_batches++;
    }
    return PCT_OK;
}

}  // namespace

void pct_carve_free(pct_ctx* ctx) { carve_tiles_free(ctx->carve); }

int64_t pct_carve_bytes(const pct_ctx* ctx)
{
    const CarveScratch& W = ctx->carve;
    return W.cap_recs * (int64_t)sizeof(CarveRec) + (W.cap_cap + W.cap_off + W.cap_keys + W.cap_tiles) * 4 + W.cap_vals * 8;
}

// hull_initializations (DS.cu:6636) + the carving counts of hull_detection (:6607)
int pct_carve_counts(pct_ctx* ctx)
{
    const pct_params& P = ctx->P;
    hipStream_t s = ctx->stream;
    DevGeom g = pct_geom(P);
    const int64_t NV = P.num_voxels, n = ctx->n_hist;
    HistPtrs hp{ctx->h[0], ctx->h[1], ctx->h[2], ctx->h[3], ctx->h[4], ctx->h[5], ctx->wepl};
    if (P.sc_on) {
        PCT_TRY(pct_alloc(ctx, &ctx->sc_carved, (NV + 31) / 32));
        PCT_TRY(pct_alloc(ctx, &ctx->sc_hull, NV));
        PCT_CHECK_HIP(ctx, hipMemsetAsync(ctx->sc_carved, 0, ((NV + 31) / 32) * sizeof(uint32_t), s));
    }
    if (P.msc_on) {
        PCT_TRY(pct_alloc(ctx, &ctx->msc_counts, NV));
        hipLaunchKernelGGL(k_init_counts, dim3(grid_for(NV)), dim3(kBlock), 0, s, g, ctx->msc_counts);
    }
    if (P.sm_on) {
        PCT_TRY(pct_alloc(ctx, &ctx->sm_counts, NV));
        hipLaunchKernelGGL(k_init_counts, dim3(grid_for(NV)), dim3(kBlock), 0, s, g, ctx->sm_counts);
    }
    ctx->carve_by_tiles = ctx->carve_tile_batches = ctx->carve_by_walks = 0;
    if (n > 0 && (P.sc_on || P.msc_on || P.sm_on)) {
        ctx->carve_by_walks = n;
        if (ctx->carve_table && NV < (int64_t)kEmpty && n <= 0x7fffffff) {
            // histories in sinogram-bin order (a sort of up to 2^31 - 1); voxel numbers are 32-bit table keys
            // below kEmpty
            const bool tiles = (ctx->carve_tiles == 1 || (ctx->carve_tiles < 0 && carve_tiles_worth(P, n))) &&
                               NV <= 0x7fffffff;
            PCT_TRY(ctx->carve_line_order && !tiles ? pct_line_order(ctx, n) : pct_bin_order(ctx, n));
            Gates gt{P.sc_on, P.msc_on, P.sm_on, P.sc_lower_threshold, P.sc_upper_threshold, P.msc_lower_threshold,
                     P.msc_upper_threshold, P.sm_lower_threshold, (uint32_t)ctx->carve_spill};
            int64_t done = 0;
            if (tiles) {
                ctx->carve.busy = true;
                const int rc = carve_by_tiles(ctx, g, hp, gt, n, &done);
                ctx->carve.busy = false;
                PCT_TRY(rc);
            }
            ctx->carve_by_tiles = done;
            ctx->carve_by_walks = n - done;
            const int tb = ctx->carve_table, bs = ctx->carve_block;
            auto kern = tb == 4096    ? (bs == 512 ? k_carve_all<4096, 512> : k_carve_all<4096, 256>)
                        : tb == 16384 ? (bs == 512 ? k_carve_all<16384, 512> : k_carve_all<16384, 256>)
                                      : (bs == 512 ? k_carve_all<8192, 512> : k_carve_all<8192, 256>);
            if (done < n)
                hipLaunchKernelGGL(kern, dim3(grid_for(n - done, bs)), dim3(bs), 0, s, n - done, ctx->u32_d + done, g, hp,
                                   gt, ctx->sc_carved, ctx->msc_counts, ctx->sm_counts);
        } else {
            if (P.sc_on)
                hipLaunchKernelGGL(k_carve, dim3(grid_for(n)), dim3(kBlock), 0, s, n, g, hp, 0, P.sc_lower_threshold,
                                   P.sc_upper_threshold, ctx->sc_carved, (int32_t*)nullptr);
            if (P.msc_on)
                hipLaunchKernelGGL(k_carve, dim3(grid_for(n)), dim3(kBlock), 0, s, n, g, hp, 1, P.msc_lower_threshold,
                                   P.msc_upper_threshold, (uint32_t*)nullptr, ctx->msc_counts);
            if (P.sm_on)
                hipLaunchKernelGGL(k_carve, dim3(grid_for(n)), dim3(kBlock), 0, s, n, g, hp, 2, P.sm_lower_threshold,
                                   P.sm_upper_threshold, (uint32_t*)nullptr, ctx->sm_counts);
        }
    }
    if (P.sc_on)
        hipLaunchKernelGGL(k_sc_finish, dim3(grid_for(NV)), dim3(kBlock), 0, s, g, ctx->sc_carved, ctx->sc_hull);
    PCT_CHECK_HIP(ctx, hipGetLastError());
    return PCT_OK;
}

// hull_detection_finish, DS.cu:7276-7340
int pct_stage_hull_finish(pct_ctx* ctx)
{
    const pct_params& P = ctx->P;
    hipStream_t s = ctx->stream;
    DevGeom g = pct_geom(P);
    const int64_t NV = P.num_voxels;
    if (P.msc_on) {
        PCT_TRY(pct_alloc(ctx, &ctx->msc_hull, NV));
        hipLaunchKernelGGL(k_msc_edge, dim3(grid_for(NV)), dim3(kBlock), 0, s, g, ctx->msc_counts, ctx->msc_hull,
                           P.msc_diff_thresh);
    }
    if (P.sm_on) {
        PCT_TRY(pct_alloc(ctx, &ctx->sm_hull, NV));
        int32_t* thr = nullptr;
        PCT_TRY(pct_scratch(ctx, SCR_THRESHOLD, &thr, P.slices));
        hipLaunchKernelGGL(k_sm_threshold, dim3(P.slices), dim3(kBlock), 0, s, g, ctx->sm_counts, thr);
        hipLaunchKernelGGL(k_sm_edge, dim3(grid_for(NV)), dim3(kBlock), 0, s, g, ctx->sm_counts, thr, ctx->sm_hull,
                           P.sm_scale_threshold);
    }
    PCT_CHECK_HIP(ctx, hipGetLastError());
    ctx->stage = ST_HULLS;
    return PCT_OK;
}

int pct_fbp_hull(pct_ctx* ctx)
{
    const pct_params& P = ctx->P;
    DevGeom g = pct_geom(P);
    PCT_TRY(pct_alloc(ctx, &ctx->fbp_hull, P.num_voxels));
    hipLaunchKernelGGL(k_fbp_hull, dim3(grid_for(P.num_voxels)), dim3(kBlock), 0, ctx->stream, g, ctx->fbp,
                       ctx->fbp_hull, P.fbp_threshold);
    PCT_CHECK_HIP(ctx, hipGetLastError());
    return PCT_OK;
}

// hull_selection, DS.cu:7351-7393
int pct_stage_select_hull(pct_ctx* ctx)
{
    const pct_params& P = ctx->P;
    hipStream_t s = ctx->stream;
    const int64_t NV = P.num_voxels;
    PCT_TRY(pct_alloc(ctx, &ctx->hull, NV));
    switch (P.hull_type) {
    case PCT_HULL_SC:
        if (!ctx->sc_hull) { ctx->err = "HULL_TYPE = SC requires SC_ON"; return PCT_E_STATE; }
        PCT_CHECK_HIP(ctx, hipMemcpyAsync(ctx->hull, ctx->sc_hull, NV, hipMemcpyDeviceToDevice, s));
        break;
    case PCT_HULL_MSC:
        if (!ctx->msc_hull) { ctx->err = "HULL_TYPE = MSC requires MSC_ON"; return PCT_E_STATE; }
        hipLaunchKernelGGL(k_int_to_bool, dim3(grid_for(NV)), dim3(kBlock), 0, s, NV, ctx->msc_hull, ctx->hull);
        break;
    case PCT_HULL_SM:
        if (!ctx->sm_hull) { ctx->err = "HULL_TYPE = SM requires SM_ON"; return PCT_E_STATE; }
        hipLaunchKernelGGL(k_int_to_bool, dim3(grid_for(NV)), dim3(kBlock), 0, s, NV, ctx->sm_hull, ctx->hull);
        break;
    case PCT_HULL_FBP:
        if (!ctx->fbp_hull) { ctx->err = "HULL_TYPE = FBP requires FBP_ON"; return PCT_E_STATE; }
        PCT_CHECK_HIP(ctx, hipMemcpyAsync(ctx->hull, ctx->fbp_hull, NV, hipMemcpyDeviceToDevice, s));
        break;
    case PCT_HULL_IMPORT:
        if (!ctx->hull_import) { ctx->err = "HULL_TYPE = IMPORT requires a hull set with pct_set_hull"; return PCT_E_STATE; }
        PCT_CHECK_HIP(ctx, hipMemcpyAsync(ctx->hull, ctx->hull_import, NV, hipMemcpyDeviceToDevice, s));
        break;
    default:
        ctx->err = "invalid HULL_TYPE";
        return PCT_E_ARG;
    }
    PCT_CHECK_HIP(ctx, hipGetLastError());
    PCT_TRY(pct_avg_filter_hull(ctx));  // hull_selection, DS.cu:7375-7386
    ctx->stage = ST_HULL_SEL;
    return PCT_OK;
}
