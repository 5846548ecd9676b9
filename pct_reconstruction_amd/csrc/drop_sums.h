// drop_sums.h — the row and column sums of DROP shared by its kernels (k_drop2.hip, k_drop_tiles.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/pct.h"
#include "devmath.h"

constexpr int kUnroll = 8;

// Bounds of a nonzero float term of a row sum: |f| < 2^top, and f is a multiple of 2^lsb (its lowest set
// significand bit).  Zero terms leave the bounds alone.
__device__ __forceinline__ void term_bounds(float f, int& top, int& lsb)
{
    const uint32_t b = __float_as_uint(f) & 0x7fffffffu;
    if (!b) return;
    const int ef = (int)(b >> 23);
    uint32_t m = b & 0x7fffffu;
    int t, l;
    if (ef == 0) {  // subnormal: m * 2^-149
        t = -149 + 32 - __clz(m);
        l = -149 + __ffs(m) - 1;
    } else {        // (2^23 + m) * 2^(ef - 150); Inf and NaN (ef = 255) get top 129 and force the ordered sum
        m |= 0x800000u;
        t = ef - 126;
        l = ef - 150 + __ffs(m) - 1;
    }
    top = t > top ? t : top;
    lsb = l < lsb ? l : lsb;
}

// True where a sum of cnt terms with these bounds is the same in any order (no partial sum rounds).
__device__ __forceinline__ bool order_free(int top, int lsb, int cnt)
{
    const int lg = cnt > 1 ? 32 - __clz((uint32_t)cnt - 1u) : 0;  // ceil(log2 cnt)
    return top + lg - lsb <= 53;
}

// Where the image value of a listed voxel is: at the listed index itself.
struct SameIndex {
    __device__ __forceinline__ uint32_t operator()(uint32_t v) const { return v; }
};

// a_i.x / L_i of one history: the sum of x over its list with the row kernel's lanes and loads
// (G lanes, kUnroll list loads and then kUnroll gathers in flight per lane, lane l summing entries
// l, l + G, l + 2G, ... in order, then a butterfly over the G partial sums).  The reference sums the
// list in order (DS.cu:9245), and the regrouped sum equals the ordered one whenever no partial sum rounds:
// with every term a multiple of 2^lsb and below 2^top in magnitude, any partial sum of at most cnt terms
// is a multiple of 2^lsb below 2^(top + ceil(log2 cnt)), exact in double when top + ceil(log2 cnt) - lsb
// <= 53.  The G lanes of a failing row gather its list again, kUnroll consecutive entries to a lane, and hand the
// running sum from lane to lane: G exchanges for kUnroll * G additions, where an exchange per entry and loads that
// waited for one another took twice the time (a block of a net's image by tiles: 20.7 us, now 11.6).  The sum is
// valid in the G lanes.  (Tracking the bounds this way costs about 1 us per DROP block; comparing raw bit patterns
// instead measured 7 us.)
template <int G, class Map>
__device__ inline double row_sum_ordered(const uint32_t* __restrict__ lst, int cnt, const float* __restrict__ x,
                                         int lane, Map at)
{
    constexpr int E = kUnroll;
    double s = 0.0;
    for (int j = 0; j < cnt; j += E * G) {
        const int first = j + lane * E;
        uint32_t a[E];
        float v[E];
#pragma unroll
        for (int q = 0; q < E; q++) a[q] = lst[first + q < cnt ? first + q : cnt - 1];
#pragma unroll
        for (int q = 0; q < E; q++) v[q] = x[at(a[q])];
#pragma unroll
        for (int q = 0; q < E; q++) v[q] = first + q < cnt ? v[q] : 0.0f;  // a sum from +0 is never -0: + 0 keeps it
        for (int l = 0; l < G; l++) {
            double t = s;
#pragma unroll
            for (int q = 0; q < E; q++) t += (double)v[q];
            s = __shfl(t, l, G);
        }
    }
    return s;
}

template <int G, class Map>
__device__ inline double row_sum(const uint32_t* __restrict__ lst, int cnt, const float* __restrict__ x, int lane,
                                 Map at)
{
    double part = 0.0;
    int top = -1000, lsb = 1000;
    for (int j = lane; j < cnt; j += kUnroll * G) {
        uint32_t a[kUnroll];
        float xv[kUnroll];
#pragma unroll
        for (int q = 0; q < kUnroll; q++) a[q] = j + q * G < cnt ? lst[j + q * G] : 0u;
#pragma unroll
        for (int q = 0; q < kUnroll; q++) xv[q] = j + q * G < cnt ? x[at(a[q])] : 0.0f;
#pragma unroll
        for (int q = 0; q < kUnroll; q++)
            if (j + q * G < cnt) {
                part += (double)xv[q];
                term_bounds(xv[q], top, lsb);
            }
    }
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) {
        part += __shfl_xor(part, o, G);
        const int t = __shfl_xor(top, o, G), l = __shfl_xor(lsb, o, G);
        top = t > top ? t : top;
        lsb = l < lsb ? l : lsb;
    }
    // the same in the G lanes after the butterfly; all-zero rows (top -1000) never fail
    if (!order_free(top, lsb, cnt)) part = row_sum_ordered<G>(lst, cnt, x, lane, at);
    return part;
}

// Running per-voxel sum in history order: FP64 (s = u_1 + u_2 + ...), FP32 (the reference's float
// sums), or FP32 with Kahan compensation (from s = c = 0).
template <int ACC>
struct ColAcc {
    double s64 = 0.0;
    float s32 = 0.0f, c32 = 0.0f;
    bool first = true;
    __device__ __forceinline__ void add(double rv)
    {
        if (ACC == PCT_ACCUM_FP64) {
            s64 = first ? rv : s64 + rv;
        } else if (ACC == PCT_ACCUM_FP32) {
            s32 = first ? (float)rv : s32 + (float)rv;
        } else {
            const float y = (float)rv - c32;
            const float t = s32 + y;
            c32 = (t - s32) - y;
            s32 = t;
        }
        first = false;
    }
    __device__ __forceinline__ float mean(uint32_t n) const
    {
        return ACC == PCT_ACCUM_FP64 ? (float)(s64 / (double)n) : s32 / (float)n;
    }
};
