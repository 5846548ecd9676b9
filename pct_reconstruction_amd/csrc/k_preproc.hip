// k_preproc.hip — stage (a): recon-volume intersections, binning, compaction, per-bin statistics,
// statistical cuts and sinogram sums.
//
// Layout: every per-history quantity is a separate float/int array in HBM (SoA), so each kernel
// streams only the fields it needs with fully coalesced 4-byte loads.  One lane per history.
//
// Determinism: the reference accumulates the per-bin sums with float atomicAdd (DS.cu:5543-5546,
// 5713-5715, 5968-5969), whose order is unspecified.  Here histories are stably sorted by bin
// (LSD radix sort keeps history order inside a bin) and each bin's sums are formed by one lane in
// ascending history order: the sums a single-threaded run of the reference produces, bit for bit,
// on every run.
#include <hipcub/hipcub.hpp>

#include "internal.h"

namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(int64_t n, int block = kBlock) { return pct_grid_for(n, block); }

// convert_mm_2_cm (DS.cu:4070-4089) and apply_tuv_shifts (:4090-4110): float *= 0.1; float += shift.
__global__ void k_units(int64_t n, float* t0, float* t1, float* t2, float* t3, float* v0, float* v1, float* v2,
                        float* v3, float* u0, float* u1, float* u2, float* u3, float* wepl, int mm, double ts,
                        double us, double vs)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (mm) {
        v0[i] = (float)((double)v0[i] * 0.1); v1[i] = (float)((double)v1[i] * 0.1);
        v2[i] = (float)((double)v2[i] * 0.1); v3[i] = (float)((double)v3[i] * 0.1);
        t0[i] = (float)((double)t0[i] * 0.1); t1[i] = (float)((double)t1[i] * 0.1);
        t2[i] = (float)((double)t2[i] * 0.1); t3[i] = (float)((double)t3[i] * 0.1);
        u0[i] = (float)((double)u0[i] * 0.1); u1[i] = (float)((double)u1[i] * 0.1);
        u2[i] = (float)((double)u2[i] * 0.1); u3[i] = (float)((double)u3[i] * 0.1);
        wepl[i] = (float)((double)wepl[i] * 0.1);
    }
    if (ts != 0.0 || us != 0.0 || vs != 0.0) {
        t0[i] = (float)((double)t0[i] + ts); t1[i] = (float)((double)t1[i] + ts);
        t2[i] = (float)((double)t2[i] + ts); t3[i] = (float)((double)t3[i] + ts);
        u0[i] = (float)((double)u0[i] + us); u1[i] = (float)((double)u1[i] + us);
        u2[i] = (float)((double)u2[i] + us); u3[i] = (float)((double)u3[i] + us);
        v0[i] = (float)((double)v0[i] + vs); v1[i] = (float)((double)v1[i] + vs);
        v2[i] = (float)((double)v2[i] + vs); v3[i] = (float)((double)v3[i] + vs);
    }
}

// calculate_intercepts, DS.cu:5286-5372
__device__ __forceinline__ int calc_intercepts(double R, double u, double t, double ut_angle, double* u_int, double* t_int)
{
    const double PI_OVER_4 = atan(1.0), THREE_PI_OVER_4 = 3 * atan(1.0);
    const double FIVE_PI_OVER_4 = 5 * atan(1.0), SEVEN_PI_OVER_4 = 7 * atan(1.0), PI_OVER_2 = 2 * atan(1.0);
    int in_cone = ((ut_angle > PI_OVER_4) && (ut_angle < THREE_PI_OVER_4)) ||
                  ((ut_angle > FIVE_PI_OVER_4) && (ut_angle < SEVEN_PI_OVER_4));
    if (in_cone) {
        double u_temp = u;
        u = -t;
        t = u_temp;
        ut_angle += PI_OVER_2;
    }
    double m = tan(ut_angle);
    double b_in = t - m * u;
    double a = (double)(1 + pct_sqf(m));
    double b = 2 * m * b_in;
    double c = (double)(pct_sqf(b_in) - pct_sqf(R));
    double disc = (double)pct_sqf(b) - (4 * a * c);
    int intersected = (disc > 0);
    if (intersected) {
        double sq = sqrt(disc);
        double u1 = (sq - b) / (2 * a);
        double u2 = (sq + b) / (2 * a);
        double t1 = m * u1 + b_in;
        double t2 = m * u2 - b_in;
        double d1 = (double)(pct_sqf(u1 - u) + pct_sqf(t1 - t));
        double d2 = (double)(pct_sqf(u2 + u) + pct_sqf(t2 + t));
        *u_int = u1 * (double)(d1 <= d2) - u2 * (double)(d1 > d2);
        *t_int = t1 * (double)(d1 <= d2) - t2 * (double)(d1 > d2);
    }
    if (in_cone) {
        double u_temp = *u_int;
        *u_int = *t_int;
        *t_int = -u_temp;
    }
    return intersected;
}

struct RawPtrs {
    const float *t0, *t1, *t2, *t3, *v0, *v1, *v2, *v3, *u0, *u1, *u2, *u3, *ang, *wepl;
};
struct HPtrs {
    float* h[10];
};

// recon_volume_intersections_GPU, DS.cu:4890-5021 (float angles: the _exact_angles variant :5022,
// identical arithmetic for integer gantry angles).
__global__ void k_intersections(int64_t n, RawPtrs r, HPtrs o, float* wepl, float* gantry, uint8_t* missed, double R,
                                double H, double A2R)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float t0 = r.t0[i], t1 = r.t1[i], t2 = r.t2[i], t3 = r.t3[i];
    const float v0 = r.v0[i], v1 = r.v1[i], v2 = r.v2[i], v3 = r.v3[i];
    const float u0 = r.u0[i], u1 = r.u1[i], u2 = r.u2[i], u3 = r.u3[i];
    // WEPL and the gantry angle travel with the histories
    const float ang = r.ang[i];
    wepl[i] = r.wepl[i];
    gantry[i] = ang;
    double rot = (double)ang * A2R;
    double cr = cos(rot), sr = sin(rot);
    double ut_entry_angle = (double)pct_atan2f(t1 - t0, u1 - u0);
    double u_entry = 0.0, t_entry = 0.0;
    int entered = calc_intercepts(R, u1, t1, ut_entry_angle, &u_entry, &t_entry);
    float xya_e = (float)(ut_entry_angle + rot);
    float xe = (float)((cr * u_entry) - (sr * t_entry));
    float ye = (float)((sr * u_entry) + (cr * t_entry));
    double ut_exit_angle = (double)pct_atan2f(t3 - t2, u3 - u2);
    double u_exit = 0.0, t_exit = 0.0;
    int exited = calc_intercepts(R, u2, t2, ut_exit_angle, &u_exit, &t_exit);
    float xya_x = (float)(ut_exit_angle + rot);
    float xx = (float)((cr * u_exit) - (sr * t_exit));
    float yx = (float)((sr * u_exit) + (cr * t_exit));
    double uv_entry_slope = (double)((v1 - v0) / (u1 - u0));
    double uv_exit_slope = (double)((v3 - v2) / (u3 - u2));
    float xza_e = pct_atan2f(v1 - v0, u1 - u0);
    float xza_x = pct_atan2f(v3 - v2, u3 - u2);
    u_entry = (cr * (double)xe) + (sr * (double)ye);
    u_exit = (cr * (double)xx) + (sr * (double)yx);
    float ze = (float)((double)v1 + uv_entry_slope * (u_entry - (double)u1));
    float zx = (float)((double)v2 - uv_exit_slope * ((double)u2 - u_exit));
    if (entered && exited) {
        if ((fabsf(ze) < H * 0.5) && (fabsf(zx) > H * 0.5)) {
            double sgn = (double)((zx >= 0) - (zx < 0));
            double frac = fabs((sgn * H * 0.5 - ze) / (double)(zx - ze));
            xx = (float)((double)xe + frac * (double)(xx - xe));
            yx = (float)((double)ye + frac * (double)(yx - ye));
            zx = (float)(sgn * H * 0.5);
        } else if (fabsf(ze) > H * 0.5) {
            entered = 0;
            exited = 0;
        }
        if ((fabsf(ze) > H * 0.5) && (fabsf(zx) < H * 0.5)) {
            double sgn_x = (double)((zx >= 0) - (zx < 0));
            double sgn_e = (double)((ze >= 0) - (ze < 0));
            double frac = fabs((sgn_x * H * 0.5 - zx) / (double)(zx - ze));
            xe = (float)((double)xx + frac * (double)(xx - xe));
            ye = (float)((double)yx + frac * (double)(yx - ye));
            ze = (float)(sgn_e * H * 0.5);
        }
        if ((fabsf(t2 - t1) > 5) || (fabsf(v2 - v1) > 5)) {
            entered = 0;
            exited = 0;
        }
    }
    o.h[0][i] = xe; o.h[1][i] = ye; o.h[2][i] = ze;
    o.h[3][i] = xx; o.h[4][i] = yx; o.h[5][i] = zx;
    o.h[6][i] = xya_e; o.h[7][i] = xza_e; o.h[8][i] = xya_x; o.h[9][i] = xza_x;
    missed[i] = (uint8_t)(!entered || !exited);
}

// binning_GPU, DS.cu:5482-5553 (bin number only; sums are formed per bin below).
// cos/sin of the angle-bin centres come from a host table so that the values equal the oracle's.
__global__ void k_binning(int64_t n, HPtrs hp, const uint8_t* missed, int32_t* bin_num, uint8_t* in_range,
                          const double* bin_cos, const double* bin_sin, double PI, double abs_deg, double t_bin_size,
                          double v_bin_size, int T, int V, int A)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (missed[i]) {
        bin_num[i] = 0;
        in_range[i] = 0;
        return;
    }
    const float xe = hp.h[0][i], ye = hp.h[1][i], ze = hp.h[2][i], xx = hp.h[3][i], yx = hp.h[4][i], zx = hp.h[5][i];
    double x_mid = (double)((xe + xx) / 2);
    double y_mid = (double)((ye + yx) / 2);
    double z_mid = (double)((ze + zx) / 2);
    double path_angle = (double)pct_atan2f(yx - ye, xx - xe);
    if (path_angle < 0) path_angle += 2 * PI;
    int angle_bin = (int)((path_angle * (180.0 / PI) / abs_deg) + 0.5) % A;
    double tt = y_mid * bin_cos[angle_bin] - x_mid * bin_sin[angle_bin];
    int t_bin = (int)((tt / t_bin_size) + T / 2);
    int v_bin = (int)((z_mid / v_bin_size) + V / 2);
    if ((t_bin >= 0) && (v_bin >= 0) && (t_bin < T) && (v_bin < V)) {
        bin_num[i] = t_bin + angle_bin * T + v_bin * T * A;
        in_range[i] = 1;
    } else {
        bin_num[i] = 0;  // quirk A1 (DS.cu:5380, 5431)
        in_range[i] = 0;
    }
}

// A history's columns: 4-byte values, moved as they are, and the in-range flag.
constexpr int kColumns = 14;
struct Columns {
    const uint32_t* in[kColumns];
    uint32_t* out[kColumns];
    const uint8_t* in8;
    uint8_t* out8;
};

// Moves the kept histories to their positions, all columns at once (one launch per column read the flags and
// positions 14 times: 0.75 ms for 16M histories, now 0.35), and leaves their number in pos[n].
struct Kept {
    uint8_t drop;  // the flag's value of a dropped history is 1 (drop) or 0
    __host__ __device__ __forceinline__ int64_t operator()(uint8_t f) const { return (f != 0) != (drop != 0); }
};
template <int N>
__global__ void k_compact(int64_t n, const uint8_t* __restrict__ flag, Kept kept, int64_t* __restrict__ pos, Columns c)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t keep = kept(flag[i]), p = pos[i];
    if (i == n - 1) pos[n] = p + keep;
    if (!keep) return;
    uint32_t v[N];
#pragma unroll
    for (int k = 0; k < N; k++) v[k] = c.in[k][i];
    const uint8_t v8 = c.in8[i];
#pragma unroll
    for (int k = 0; k < N; k++) c.out[k][p] = v[k];
    c.out8[p] = v8;
}

__global__ void k_iota(int64_t n, uint32_t* out)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (uint32_t)i;
}

// off[b] = the histories in bins below b, from their sorted bins.  (Counting with atomics and a prefix sum took
// 0.9 ms for 16M histories and 1.3M bins, a search per bin takes less than 0.1.)
__global__ void k_bin_offsets(int64_t n, int NB, const uint32_t* __restrict__ sorted, int32_t* __restrict__ off)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b > NB) return;
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (sorted[mid] < (uint32_t)b) lo = mid + 1;
        else hi = mid;
    }
    off[b] = (int32_t)lo;
}

__device__ __forceinline__ double wrap_pi(double a, double PI)
{
    if (a > PI) a -= 2 * PI;
    if (a < -PI) a += 2 * PI;
    return a;
}

// doubles as two arrays of words
struct Words {
    uint32_t *lo, *hi;
};

// The per-history inputs of the bin statistics in bin order (j = position in the sorted order): in-range
// flag, WEPL and the two wrapped angle differences, so that the three passes of k_bin_stats stream
// contiguous memory instead of gathering through the order.
__global__ void k_bin_gather(int64_t n, const uint32_t* __restrict__ perm, const uint8_t* __restrict__ in_range,
                             const float* __restrict__ wepl, const float* __restrict__ xya_e,
                             const float* __restrict__ xza_e, const float* __restrict__ xya_x,
                             const float* __restrict__ xza_x, double PI, uint8_t* __restrict__ g_ir,
                             float* __restrict__ g_w, double* __restrict__ g_ut, Words g_uv)
{
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const uint32_t i = perm[j];
    g_ir[j] = in_range[i];
    g_w[j] = wepl[i];
    g_ut[j] = wrap_pi((double)(xya_x[i] - xya_e[i]), PI);
    const double uv = wrap_pi((double)(xza_x[i] - xza_e[i]), PI);
    g_uv.lo[j] = (uint32_t)__double2loint(uv);
    g_uv.hi[j] = (uint32_t)__double2hiint(uv);
}

// One lane per bin: binning sums (DS.cu:5518-5546), calculate_means_GPU (:5644), the squared
// deviations (:5689-5717), calculate_standard_deviations_GPU (:5737) and statistical_cuts_GPU
// (:5937-5971), each over the bin's histories in ascending history order, read from the bin-ordered
// inputs of k_bin_gather.  The inputs of a wavefront's 64 bins are one contiguous range: it goes to LDS by whole
// lines, kStatChunk entries at a time, once for the three passes where it fits (from memory a lane used 4 or 8 bytes
// of each line that it read: 2.2 ms for 16M histories in 1.3M bins, now 0.35).  A chunk of well-filled bins keeps few
// lanes busy, though: a wavefront with more than `most` entries lets every lane read its bin from memory.
// `failed` is zero on entry.
constexpr int kStatChunk = 1024;
struct BinInputs {
    const uint8_t* ir;
    const float* w;
    const double *ut, *uv;
    Words uv_words;  // where uv is null
    __device__ __forceinline__ double at_uv(int j) const
    {
        return uv ? uv[j] : __hiloint2double((int)uv_words.hi[j], (int)uv_words.lo[j]);
    }
};
__global__ void __launch_bounds__(64) k_bin_stats(int NB, const int32_t* __restrict__ off,
                                                  const uint32_t* __restrict__ perm, const uint8_t* __restrict__ g_ir,
                                                  const float* __restrict__ g_w, const double* __restrict__ g_ut,
                                                  Words g_uv, int32_t* counts_pre, float* m_w,
                                                  float* m_ut, float* m_uv, float* s_w, float* s_ut, float* s_uv,
                                                  int32_t* counts_post, float* sinogram, uint8_t* failed, float k,
                                                  int quirk_a1, int most)
{
    __shared__ double l_ut[kStatChunk], l_uv[kStatChunk];
    __shared__ float l_w[kStatChunk];
    __shared__ uint8_t l_ir[kStatChunk];
    const int b0 = blockIdx.x * 64, b = b0 + (int)threadIdx.x;
    const int32_t lo = off[b0], hi = off[b0 + 64 < NB ? b0 + 64 : NB];
    const int32_t beg = b < NB ? off[b] : hi, end = b < NB ? off[b + 1] : hi;
    const BinInputs staged{l_ir, l_w, l_ut, l_uv, {}}, in_memory{g_ir, g_w, g_ut, nullptr, g_uv};
    const bool direct = hi - lo > most;
    // f(entry, inputs, its place there) over the bin's entries
    auto each = [&](bool first, auto f) {
        if (direct) {
            for (int32_t j = beg; j < end; j++) f(j, in_memory, j);
            return;
        }
        for (int64_t c0 = lo; c0 < hi; c0 += kStatChunk) {
            if (first || hi - lo > kStatChunk) {
                __syncthreads();
                const int m = (int)(hi - c0 < kStatChunk ? hi - c0 : kStatChunk);
#pragma unroll 4
                for (int j = threadIdx.x; j < m; j += 64) {
                    l_ut[j] = g_ut[c0 + j];
                    l_uv[j] = __hiloint2double((int)g_uv.hi[c0 + j], (int)g_uv.lo[c0 + j]);
                    l_w[j] = g_w[c0 + j];
                    l_ir[j] = g_ir[c0 + j];
                }
                __syncthreads();
            }
            const int64_t last = end < c0 + kStatChunk ? end : c0 + kStatChunk;
            for (int64_t j = beg > c0 ? beg : c0; j < last; j++) f((int32_t)j, staged, (int)(j - c0));
        }
    };
    int cnt = 0;
    float sw = 0.0f, su = 0.0f, sv = 0.0f;
    each(true, [&](int32_t, const BinInputs& in, int j) {
        if (!in.ir[j]) return;
        cnt += 1;
        sw += in.w[j];
        su += (float)in.ut[j];
        sv += (float)in.at_uv(j);
    });
    if (cnt > 0) {
        sw /= cnt;
        su /= cnt;
        sv /= cnt;
    }
    float qw = 0.0f, qu = 0.0f, qv = 0.0f;
    each(false, [&](int32_t, const BinInputs& in, int j) {
        if (!quirk_a1 && !in.ir[j]) return;
        double d_w = (double)(in.w[j] - sw);
        double d_ut = in.ut[j] - su;
        double d_uv = in.at_uv(j) - sv;
        qw += pct_sqf(d_w);
        qu += pct_sqf(d_ut);
        qv += pct_sqf(d_uv);
    });
    if (cnt > 1) {
        qw = sqrtf(qw / (cnt - 1));
        qu = sqrtf(qu / (cnt - 1));
        qv = sqrtf(qv / (cnt - 1));
    }
    int cpost = 0;
    float sino = 0.0f;
    each(false, [&](int32_t at, const BinInputs& in, int j) {
        if (!quirk_a1 && !in.ir[j]) {
            failed[perm[at]] = 1;
            return;
        }
        const float w = in.w[j];
        int pass_ut = fabs(in.ut[j] - su) < (double)(k * qu);
        int pass_uv = fabs(in.at_uv(j) - sv) < (double)(k * qv);
        int pass_w = fabsf(sw - w) <= k * qw;
        if (!pass_ut || !pass_uv || !pass_w) {
            failed[perm[at]] = 1;
        } else {
            cpost += 1;
            sino += w;
        }
    });
    if (b >= NB) return;
    counts_pre[b] = cnt;
    m_w[b] = sw;
    m_ut[b] = su;
    m_uv[b] = sv;
    s_w[b] = qw;
    s_ut[b] = qu;
    s_uv[b] = qv;
    counts_post[b] = cpost;
    sinogram[b] = sino;
}

// Entries of 64 bins up to which they go through LDS.  Wavefronts that fill the chip are bound by memory and gain from
// whole lines longer than few ones, which wait for the busiest.  Cuts with LDS | from memory, ms: 16M histories, 71 in a
// bin 2.93 | 4.69, 117 (2139 wavefronts) 3.49 | 4.26, 233 5.99 | 3.49, 462 12.6 | 3.9; 2M, 22 in a bin (1426 wavefronts)
// 0.35 | 0.44, 58 (541) 0.53 | 0.46, 115 1.13 | 0.57; 0.3M, 74 (63 wavefronts) 0.66 | 0.23.
int stat_staged(int bins) { return bins >= 64 * 2048 ? 8192 : 2048; }

}  // namespace

// Keeps the histories whose flag is set, or, with `drop`, those whose flag is not.
int pct_compact(pct_ctx* ctx, const uint8_t* flag, bool drop, int64_t n, int64_t* n_out, bool with_first_voxel)
{
    hipStream_t s = ctx->stream;
    ctx->bin_perm_n = -1;  // the histories move
    if (n == 0) {
        *n_out = 0;
        return PCT_OK;
    }
    // exclusive scan of the kept (as int64) -> positions
    const Kept kept{(uint8_t)drop};
    size_t need = 0;
    hipcub::TransformInputIterator<int64_t, Kept, const uint8_t*> it(flag, kept);
    PCT_CHECK_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(nullptr, need, it, ctx->pos, n, s));
    PCT_TRY(pct_grow_cub(ctx, need));
    need = ctx->cub_tmp_bytes;
    PCT_CHECK_HIP(ctx, hipcub::DeviceScan::ExclusiveSum(ctx->cub_tmp, need, it, ctx->pos, n, s));
    Columns c{};
    int nc = 0;
    auto column = [&](auto*& a, auto*& tmp) {
        c.in[nc] = (const uint32_t*)a;
        c.out[nc++] = (uint32_t*)tmp;
        std::swap(a, tmp);
    };
    for (int k = 0; k < 10; k++) column(ctx->h[k], ctx->h_tmp[k]);
    column(ctx->wepl, ctx->wepl_tmp);
    column(ctx->gantry, ctx->gantry_tmp);
    column(ctx->bin_num, ctx->bin_tmp);
    c.in8 = ctx->in_range;
    c.out8 = ctx->u8_tmp;
    std::swap(ctx->in_range, ctx->u8_tmp);
    if (with_first_voxel) {
        column(ctx->first_voxel, ctx->u32_d);
        hipLaunchKernelGGL(k_compact<14>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, flag, kept, ctx->pos, c);
    } else {
        hipLaunchKernelGGL(k_compact<13>, dim3(grid_for(n)), dim3(kBlock), 0, s, n, flag, kept, ctx->pos, c);
    }
    PCT_CHECK_HIP(ctx, hipGetLastError());
    PCT_TRY(pct_read(ctx, n_out, ctx->pos + n, sizeof(int64_t)));
    return PCT_OK;
}

// Stable sort of the indices of the first n histories by bin number into ctx->u32_d, the sorted bins in ctx->u32_b (an
// LSD radix sort keeps history order inside a bin).  The order stays valid until the next compaction or binning.
int pct_bin_order(pct_ctx* ctx, int64_t n)
{
    if (ctx->bin_perm_n == n) return PCT_OK;
    hipStream_t s = ctx->stream;
    if (n > 0x7fffffff) {
        ctx->err = "bin order: more than 2^31 histories";
        return PCT_E_LIMIT;
    }
    int end_bit = 1;
    while ((1ll << end_bit) < (int64_t)ctx->P.num_bins) end_bit++;
    const uint32_t* keys_in = (const uint32_t*)ctx->bin_num;
    uint32_t* keys_out = ctx->u32_b;
    uint32_t* vals_in = ctx->u32_c;
    uint32_t* perm = ctx->u32_d;
    if (n > 0) {
        hipLaunchKernelGGL(k_iota, dim3(grid_for(n)), dim3(kBlock), 0, s, n, vals_in);
        size_t need = 0;
        PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, need, keys_in, keys_out, vals_in, perm, (int)n, 0,
                                                              end_bit, s));
        PCT_TRY(pct_grow_cub(ctx, need));
        need = ctx->cub_tmp_bytes;
        PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(ctx->cub_tmp, need, keys_in, keys_out, vals_in, perm,
                                                              (int)n, 0, end_bit, s));
        PCT_CHECK_HIP(ctx, hipGetLastError());
    }
    ctx->bin_perm_n = n;
    return PCT_OK;
}

// Sort key of a history's chord: the bin with angle bins a and a + A/2 paired (the same line traversed in
// the opposite direction, at t mirrored), so that histories on one line, either way, become neighbours.
__global__ void k_line_keys(int64_t n, const int32_t* __restrict__ bin_num, int T, int A, uint32_t* __restrict__ key)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t b = (uint32_t)bin_num[i];
    const uint32_t t = b % (uint32_t)T, r = b / (uint32_t)T, a = r % (uint32_t)A, v = r / (uint32_t)A;
    const uint32_t h = (uint32_t)A / 2u, half = a >= h ? 1u : 0u;
    const uint32_t tc = half ? (uint32_t)T - 1u - (t < (uint32_t)T ? t : (uint32_t)T - 1u) : t;
    key[i] = (((v * h + (a - half * h)) * (uint32_t)T + tc) << 1) | half;
}

// History indices ordered by chord line (k_line_keys) into ctx->u32_d.  Replaces a bin order held there.
int pct_line_order(pct_ctx* ctx, int64_t n)
{
    const pct_params& P = ctx->P;
    hipStream_t s = ctx->stream;
    if (n > 0x7fffffff || (P.angular_bins & 1)) return pct_bin_order(ctx, n);
    ctx->bin_perm_n = -1;
    int end_bit = 2;
    while ((1ll << end_bit) < 2ll * P.num_bins) end_bit++;
    if (n > 0) {
        hipLaunchKernelGGL(k_line_keys, dim3(grid_for(n)), dim3(kBlock), 0, s, n, ctx->bin_num, P.t_bins,
                           P.angular_bins, ctx->u32_a);
        hipLaunchKernelGGL(k_iota, dim3(grid_for(n)), dim3(kBlock), 0, s, n, ctx->u32_c);
        size_t need = 0;
        PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, need, ctx->u32_a, ctx->u32_b, ctx->u32_c,
                                                              ctx->u32_d, (int)n, 0, end_bit, s));
        PCT_TRY(pct_grow_cub(ctx, need));
        PCT_CHECK_HIP(ctx, hipcub::DeviceRadixSort::SortPairs(ctx->cub_tmp, need, ctx->u32_a, ctx->u32_b, ctx->u32_c,
                                                              ctx->u32_d, (int)n, 0, end_bit, s));
        PCT_CHECK_HIP(ctx, hipGetLastError());
    }
    return PCT_OK;
}

int pct_ensure_hist_capacity(pct_ctx* ctx, int64_t n)
{
    if (n <= ctx->cap_hist) return PCT_OK;
    ctx->cap_hist = 0;  // until they all are there
    for (int k = 0; k < 10; k++) {
        PCT_TRY(pct_alloc(ctx, &ctx->h[k], n));
        PCT_TRY(pct_alloc(ctx, &ctx->h_tmp[k], n));
    }
    PCT_TRY(pct_alloc(ctx, &ctx->wepl, n));
    PCT_TRY(pct_alloc(ctx, &ctx->wepl_tmp, n));
    PCT_TRY(pct_alloc(ctx, &ctx->gantry, n));
    PCT_TRY(pct_alloc(ctx, &ctx->gantry_tmp, n));
    PCT_TRY(pct_alloc(ctx, &ctx->bin_num, n));
    PCT_TRY(pct_alloc(ctx, &ctx->bin_tmp, n));
    PCT_TRY(pct_alloc(ctx, &ctx->in_range, n));
    PCT_TRY(pct_alloc(ctx, &ctx->u8_tmp, n));
    PCT_TRY(pct_alloc(ctx, &ctx->flag, n));
    PCT_TRY(pct_alloc(ctx, &ctx->pos, n + 1));
    PCT_TRY(pct_alloc(ctx, &ctx->first_voxel, n));
    PCT_TRY(pct_alloc(ctx, &ctx->u32_a, n));
    PCT_TRY(pct_alloc(ctx, &ctx->u32_b, n));
    PCT_TRY(pct_alloc(ctx, &ctx->u32_c, n));
    PCT_TRY(pct_alloc(ctx, &ctx->u32_d, n));
    ctx->cap_hist = n;
    return PCT_OK;
}

int pct_carve_counts(pct_ctx* ctx);  // k_hull.hip

int pct_angle_table(pct_ctx* ctx)
{
    if (ctx->angle_cs) return PCT_OK;
    const pct_params& P = ctx->P;
    const int A = P.angular_bins;
    const double delta = P.angular_bin_size * (P.pi / 180.0);
    std::vector<double> cs(4 * (size_t)A);
    for (int a = 0; a < A; a++) {
        // angle_bin * ANGULAR_BIN_SIZE * ANGLE_TO_RADIANS (DS.cu:5506), and bin_angle = angle_bin * delta (:6362-6364)
        const double binning = a * P.angular_bin_size * (P.pi / 180.0), fbp = a * delta;
        cs[a] = std::cos(binning);
        cs[A + a] = std::sin(binning);
        cs[2 * A + a] = std::cos(fbp);
        cs[3 * A + a] = std::sin(fbp);
    }
    double* d = nullptr;
    PCT_TRY(pct_alloc(ctx, &d, cs.size()));
    if (hipMemcpy(d, cs.data(), cs.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
        pct_free(&d);
        ctx->err = "angle table: copy failed";
        return PCT_E_HIP;
    }
    ctx->angle_cs = d;
    return PCT_OK;
}

int pct_stage_intersect_bin_carve(pct_ctx* ctx)
{
    const pct_params& P = ctx->P;
    hipStream_t s = ctx->stream;
    const int64_t n = ctx->n_loaded;
    ctx->stage = ST_LOADED;  // the histories of an earlier run are overwritten
    PCT_TRY(pct_ensure_hist_capacity(ctx, n));
    ctx->bin_perm_n = -1;
    unsigned g = grid_for(n);
    RawPtrs r{ctx->raw[0], ctx->raw[1], ctx->raw[2], ctx->raw[3], ctx->raw[4], ctx->raw[5], ctx->raw[6],
              ctx->raw[7], ctx->raw[8], ctx->raw[9], ctx->raw[10], ctx->raw[11], ctx->raw[13], ctx->raw[12]};
    HPtrs o;
    for (int k = 0; k < 10; k++) o.h[k] = ctx->h[k];
    uint8_t* missed = ctx->flag;
    if (n > 0) {
        hipLaunchKernelGGL(k_intersections, dim3(g), dim3(kBlock), 0, s, n, r, o, ctx->wepl, ctx->gantry, missed,
                           P.recon_cyl_radius, P.recon_cyl_height, P.pi / 180.0);
        PCT_TRY(pct_angle_table(ctx));
        const double* d_cs = ctx->angle_cs;
        hipLaunchKernelGGL(k_binning, dim3(g), dim3(kBlock), 0, s, n, o, missed, ctx->bin_num, ctx->in_range, d_cs,
                           d_cs + P.angular_bins, P.pi, P.angular_bin_size, P.t_bin_size, P.v_bin_size, P.t_bins,
                           P.v_bins, P.angular_bins);
        PCT_CHECK_HIP(ctx, hipGetLastError());
    }
    // keep histories that traversed the reconstruction volume (DS.cu:5429-5449)
    int64_t kept = 0;
    PCT_TRY(pct_compact(ctx, missed, true, n, &kept, false));
    ctx->n_hist = kept;
    ctx->n_recon_volume = kept;
    // hull-detection counts on the same histories (hull_detection, DS.cu:6607)
    PCT_TRY(pct_carve_counts(ctx));
    ctx->stage = ST_BINNED;
    return PCT_OK;
}

int pct_stage_stats_and_cuts(pct_ctx* ctx)
{
    const pct_params& P = ctx->P;
    hipStream_t s = ctx->stream;
    const int64_t n = ctx->n_hist;
    const int NB = P.num_bins;
    if (n > 0x7fffffff) {
        ctx->err = "statistical cuts: more than 2^31 histories";
        return PCT_E_LIMIT;
    }
    PCT_TRY(pct_alloc(ctx, &ctx->counts_pre, NB));
    PCT_TRY(pct_alloc(ctx, &ctx->counts_post, NB));
    PCT_TRY(pct_alloc(ctx, &ctx->bin_off, NB + 1));
    for (int k = 0; k < 3; k++) {
        PCT_TRY(pct_alloc(ctx, &ctx->mean[k], NB));
        PCT_TRY(pct_alloc(ctx, &ctx->stddev[k], NB));
    }
    PCT_TRY(pct_alloc(ctx, &ctx->sinogram, NB));
    unsigned g = grid_for(n);
    // history indices in bin order (kept from the hull carving when no compaction came between)
    PCT_TRY(pct_bin_order(ctx, n));
    const uint32_t* perm = ctx->u32_d;
    hipLaunchKernelGGL(k_bin_offsets, dim3(grid_for(NB + 1)), dim3(kBlock), 0, s, n, NB, ctx->u32_b, ctx->bin_off);
    uint8_t* failed = ctx->flag;
    if (n > 0) PCT_CHECK_HIP(ctx, hipMemsetAsync(failed, 0, n, s));
    // the gathered inputs lie in columns that the compaction at the end overwrites and in scratch of the bin order
    uint8_t* g_ir = ctx->u8_tmp;
    float* g_w = ctx->wepl_tmp;
    double* g_ut = (double*)ctx->pos;
    const Words g_uv{ctx->u32_a, ctx->u32_c};
    if (n > 0)
        hipLaunchKernelGGL(k_bin_gather, dim3(g), dim3(kBlock), 0, s, n, perm, ctx->in_range, ctx->wepl, ctx->h[6],
                           ctx->h[7], ctx->h[8], ctx->h[9], P.pi, g_ir, g_w, g_ut, g_uv);
    hipLaunchKernelGGL(k_bin_stats, dim3(pct_grid_for(NB, 64)), dim3(64), 0, s, NB, ctx->bin_off, perm, g_ir, g_w,
                       g_ut, g_uv, ctx->counts_pre, ctx->mean[0], ctx->mean[1], ctx->mean[2], ctx->stddev[0],
                       ctx->stddev[1], ctx->stddev[2], ctx->counts_post, ctx->sinogram, failed,
                       (float)P.sigmas_2_keep, P.quirk_a1_bin0, stat_staged(NB));
    PCT_CHECK_HIP(ctx, hipGetLastError());
    // keep the histories that passed (DS.cu:5892-5911)
    int64_t kept = 0;
    PCT_TRY(pct_compact(ctx, failed, true, n, &kept, false));
    ctx->n_hist = kept;
    ctx->n_post_cuts = kept;
    ctx->stage = ST_CUT;
    return PCT_OK;
}

int pct_launch_units(hipStream_t s, int64_t n, float* const raw[14], int mm, double ts, double us, double vs)
{
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_units, dim3(grid_for(n)), dim3(kBlock), 0, s, n, raw[0], raw[1], raw[2], raw[3], raw[4],
                       raw[5], raw[6], raw[7], raw[8], raw[9], raw[10], raw[11], raw[12], mm, ts, us, vs);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}
