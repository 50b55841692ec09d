// adc.hip - adaptive density control (default / ABSGS refine and opacity reset) and the
// row gather it is built on, as data-parallel kernels.
//
// The gsx CPU backend (the parity oracle) runs ADC as sequential loops
// (gsx/src/gsx-cpu/adc/default.c:160-527, gsx/src/gsx-cpu/adc.c:380-559):
//   1. grow candidates in index order until the budget max_num_gaussians - n is spent;
//   2. gather rows [0, n) ++ candidates, zero the optimizer moments of the appended rows;
//   3. duplicate (the gathered copy) or split: 2 children at scale / 1.6, opacity
//      1 - sqrt(1 - sigmoid(o)), offsets R * ((s + 1e-5) * N(0,1)) from one sequential pcg32
//      stream, 6 normals (12 uniforms) per split;
//   4. keep rows with sigmoid(o) > threshold, (size OK or not prune_large) and non-degenerate
//      rotation, in order (stable compaction; at least one row survives);
//   5. zero the auxiliary statistics; in a reset window clamp opacity and reset its moments.
// Here each step is a kernel over rows: ranks come from exclusive scans (so "first-come by
// index" becomes rank < budget), and split k draws from the stream advanced by 12 * k, which
// is exactly where the CPU's sequential stream stands at that split. Classification and keep
// decisions use the glibc-exact expf, so counts and row order match the CPU bit for bit.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <new>

#include "../../include/gsx_hip.h"
#include "common.hpp"

namespace gsx_amd {

// Thread-local message behind gsx_hip_last_error_message (defined in abi.hip).
void set_last_error(const char* what);

constexpr int kAdcThreads = 256;

// gsx_sigmoid / gsx_logit (gsx/src/gsx-core.c:2920-2935), used by the ADC (not the renderer's
// two-branch sigmoid).
__device__ inline float adc_sigmoid(float x) { return 1.0f / (1.0f + gsx_expf(-x)); }

// glibc's logf and cosf, bit for bit (the restatements of gsx_math.h)
__device__ inline float adc_logf(float x) { return gsx_logf(x); }
__device__ inline float adc_cosf(float x) { return gsx_cosf(x); }

__device__ inline float adc_prob_to_logit(float p) {
    // gsx/src/gsx-cpu/adc.c:230-240
    float c = p;
    if (c <= 1e-6f) c = 1e-6f;
    if (c >= 1.0f - 1e-6f) c = 1.0f - 1e-6f;
    return adc_logf(c / (1.0f - c));
}

__device__ inline float adc_next_normal(gsx_amd_pcg32* rng) {
    // gsx/src/gsx-random.c:86-112 (cosine branch, two uniforms)
    float u1 = gsx_pcg32_next_f32(rng);
    const float u2 = gsx_pcg32_next_f32(rng);
    u1 = fmaxf(1e-7f, u1);
    const float mag = sqrtf(-2.0f * adc_logf(u1));
    return mag * adc_cosf(2.0f * (float)3.14159265358979323846264338327950288 * u2);
}

// Number of the workgroup's threads with p, for every thread; two workgroup barriers.
__device__ inline uint32_t adc_block_count(bool p, uint32_t* s_wave) {
    const uint32_t c = (uint32_t)__popcll(wave_ballot(p));
    if (__lane_id() == 0) s_wave[threadIdx.x / kWave] = c;
    __syncthreads();
    uint32_t total = 0;
#pragma unroll
    for (int w = 0; w < kAdcThreads / kWave; ++w) total += s_wave[w];
    __syncthreads();
    return total;
}

// mode: 0 none, 1 duplicate, 2 split (default.c:160-219); per workgroup the number of candidates and,
// in the second array of gridDim.x + 1 words, of splits among them
__global__ __launch_bounds__(kAdcThreads) void adc_classify_kernel(int64_t n, gsx_hip_adc_params p,
                                                                   const float* __restrict__ logscale,
                                                                   const float* __restrict__ grad_acc,
                                                                   const float* __restrict__ visible_counter,
                                                                   uint8_t* __restrict__ mode,
                                                                   uint32_t* __restrict__ partials) {
    __shared__ uint32_t s_wave[kAdcThreads / kWave];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint8_t m = 0;
    if (i < n) {
        const float counter = visible_counter != nullptr ? visible_counter[i] : 1.0f;
        if (counter > 0.0f) {
            const float g = grad_acc[i] / (counter > 1.0f ? counter : 1.0f);
            const float thr = p.algorithm == 1 ? p.duplicate_absgrad_threshold : p.duplicate_grad_threshold;
            if (g > thr) {
                const float sx = gsx_expf(logscale[i * 3 + 0]);
                const float sy = gsx_expf(logscale[i * 3 + 1]);
                const float sz = gsx_expf(logscale[i * 3 + 2]);
                float mx = sx;
                if (sy > mx) mx = sy;
                if (sz > mx) mx = sz;
                m = mx > p.duplicate_scale_threshold * p.scene_scale ? 2 : 1;
            }
        }
        mode[i] = m;
    }
    const uint32_t candidates = adc_block_count(m != 0, s_wave);
    const uint32_t splits = adc_block_count(m == 2, s_wave);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = candidates;
        partials[gridDim.x + 1 + blockIdx.x] = splits;
    }
}

// Rows of a Gaussian set, addressed uniformly: field f has width w[f] floats per row.
struct RowSet {
    float* f[GSX_HIP_ADC_MAX_FIELDS];
    int32_t w[GSX_HIP_ADC_MAX_FIELDS];
    int32_t count;
};

// e / w for the e < 256 * 21 floats of a workgroup's rows, w <= 21: a multiplication by
// ceil(2^18 / w), exact as long as e (w - 1) < 2^18
__device__ inline uint32_t adc_row_of(uint32_t e, uint32_t w) { return e * ((0x3ffffu + w) / w) >> 18; }

// Appends row src as row n + rank for every granted candidate (rank < budget), zeroes the appended
// optimizer moments, then applies the split mutation (default.c:38-158) to both rows. Before the launch,
// partials holds the two exclusive scans of adc_classify_kernel's counts; the workgroup in whose
// candidates the budget ends (the last one if it suffices) stores the granted candidates and splits in
// counts_dev and in host memory. Its granted candidates are listed in LDS first, so that consecutive
// threads copy consecutive floats of the appended (neighbouring) rows and full waves form the splits
// (1M rows, 200k candidates: 42 us with a thread per row, and 77 more to count the granted splits).
__global__ __launch_bounds__(kAdcThreads) void adc_grow_kernel(int64_t n, uint64_t budget, const uint8_t* __restrict__ mode,
                                                               const uint32_t* __restrict__ partials, RowSet rows,
                                                               RowSet moments, uint64_t rng_state, uint64_t rng_inc,
                                                               int32_t mean_f, int32_t rot_f, int32_t ls_f,
                                                               int32_t op_f, uint32_t* __restrict__ counts_dev,
                                                               uint32_t* __restrict__ counts_host) {
    __shared__ uint32_t s_wave[kAdcThreads / kWave];
    __shared__ uint32_t s_row[kAdcThreads];  // granted candidates: row | split rank within the workgroup << 16
    const uint32_t blk = blockIdx.x;
    const int64_t first = (int64_t)blk * kAdcThreads;
    const int64_t i = first + threadIdx.x;
    const uint8_t m = i < n ? mode[i] : 0;
    const uint32_t grow0 = partials[blk], split0 = partials[gridDim.x + 1 + blk];
    const uint64_t grow1 = partials[blk + 1];
    // candidates in the low, splits in the high half (at most 256 each)
    uint32_t total;
    const uint32_t before =
        block_exclusive_scan_256((m != 0 ? 1u : 0u) | (m == 2 ? 0x10000u : 0u), s_wave, total);
    const uint32_t rank = before & 0xffffu;
    const bool granted = m != 0 && (uint64_t)grow0 + rank < budget;
    if (granted) s_row[rank] = threadIdx.x | (m == 2 ? 0x8000u : 0u) | (before & 0xffff0000u);
    const uint32_t here = adc_block_count(granted, s_wave);
    const uint32_t splits = adc_block_count(granted && m == 2, s_wave);
    const bool ends_here = (uint64_t)grow0 <= budget && (grow1 > budget || blk == gridDim.x - 1);
    if (ends_here && threadIdx.x == 0) {
        const uint32_t grown = grow0 + here, all_splits = split0 + splits;
        counts_dev[0] = counts_host[0] = grown;
        counts_dev[1] = counts_host[1] = all_splits;
    }
    if (here == 0) return;  // uniform
    const int64_t to = n + grow0;
    for (int f = 0; f < rows.count; ++f) {
        const uint32_t w = (uint32_t)rows.w[f];
        float* const p = rows.f[f];
        for (uint32_t e = threadIdx.x; e < here * w; e += kAdcThreads) {
            const uint32_t q = adc_row_of(e, w);
            p[to * w + e] = p[(first + (s_row[q] & 0xffu)) * w + (e - q * w)];
        }
    }
    for (int f = 0; f < moments.count; ++f) {
        const uint32_t w = (uint32_t)moments.w[f];
        for (uint32_t e = threadIdx.x; e < here * w; e += kAdcThreads) moments.f[f][to * w + e] = 0.0f;
    }
    __syncthreads();  // the copies stand before a split changes its rows
    const uint32_t entry = threadIdx.x < here ? s_row[threadIdx.x] : 0u;
    if ((entry & 0x8000u) == 0u) return;
    const int64_t src = first + (entry & 0xffu), t = to + threadIdx.x;
    float* mean = rows.f[mean_f];
    float* rot = rows.f[rot_f];
    float* ls = rows.f[ls_f];
    float* op = rows.f[op_f];
    float qx = rot[src * 4 + 0], qy = rot[src * 4 + 1], qz = rot[src * 4 + 2], qw = rot[src * 4 + 3];
    const float sx = gsx_expf(ls[src * 3 + 0]), sy = gsx_expf(ls[src * 3 + 1]), sz = gsx_expf(ls[src * 3 + 2]);
    float so = adc_sigmoid(op[src]);
    const float nsx = sx / 1.6f, nsy = sy / 1.6f, nsz = sz / 1.6f;
    gsx_amd_pcg32 rng;
    rng.state = rng_state;
    rng.inc = rng_inc;
    // in two jumps: the workgroup's (uniform) and the split's short one
    gsx_pcg32_advance(&rng, 12ull * (uint64_t)split0);
    gsx_pcg32_advance(&rng, 12ull * (uint64_t)(entry >> 16));
    const float r1x = adc_next_normal(&rng), r1y = adc_next_normal(&rng), r1z = adc_next_normal(&rng);
    const float r2x = adc_next_normal(&rng), r2y = adc_next_normal(&rng), r2z = adc_next_normal(&rng);
    const float t1x = r1x * (sx + 1e-5f), t1y = r1y * (sy + 1e-5f), t1z = r1z * (sz + 1e-5f);
    const float t2x = r2x * (sx + 1e-5f), t2y = r2y * (sy + 1e-5f), t2z = r2z * (sz + 1e-5f);
    // gsx/src/gsx-cpu/adc.c:290-330
    const float qn = sqrtf(qx * qx + qy * qy + qz * qz + qw * qw);
    if (qn > 1e-8f) {
        const float iq = 1.0f / qn;
        qx *= iq;
        qy *= iq;
        qz *= iq;
        qw *= iq;
    }
    const float m00 = 1.0f - 2.0f * (qy * qy + qz * qz), m01 = 2.0f * (qx * qy - qw * qz),
                m02 = 2.0f * (qx * qz + qw * qy);
    const float m10 = 2.0f * (qx * qy + qw * qz), m11 = 1.0f - 2.0f * (qx * qx + qz * qz),
                m12 = 2.0f * (qy * qz - qw * qx);
    const float m20 = 2.0f * (qx * qz - qw * qy), m21 = 2.0f * (qy * qz + qw * qx),
                m22 = 1.0f - 2.0f * (qx * qx + qy * qy);
    if (so < 0.0f) so = 0.0f;
    if (so > 1.0f - 1e-6f) so = 1.0f - 1e-6f;
    const float sop = 1.0f - sqrtf(1.0f - so);
    const float lx = adc_logf(nsx), ly = adc_logf(nsy), lz = adc_logf(nsz);
    const float lo = adc_prob_to_logit(sop);
    const float mx = mean[src * 3 + 0], my = mean[src * 3 + 1], mz = mean[src * 3 + 2];
    mean[t * 3 + 0] = mx + (m00 * t1x + m01 * t1y + m02 * t1z);
    mean[t * 3 + 1] = my + (m10 * t1x + m11 * t1y + m12 * t1z);
    mean[t * 3 + 2] = mz + (m20 * t1x + m21 * t1y + m22 * t1z);
    ls[t * 3 + 0] = lx;
    ls[t * 3 + 1] = ly;
    ls[t * 3 + 2] = lz;
    op[t] = lo;
    mean[src * 3 + 0] = mx + (m00 * t2x + m01 * t2y + m02 * t2z);
    mean[src * 3 + 1] = my + (m10 * t2x + m11 * t2y + m12 * t2z);
    mean[src * 3 + 2] = mz + (m20 * t2x + m21 * t2y + m22 * t2z);
    ls[src * 3 + 0] = lx;
    ls[src * 3 + 1] = ly;
    ls[src * 3 + 2] = lz;
    op[src] = lo;
}

// default.c:221-273 for the n + *grown rows; max_screen_radius (null: no such test) is that of the rows
// before the growth. Per workgroup the number of kept rows.
__global__ __launch_bounds__(kAdcThreads) void adc_keep_kernel(int64_t n, const uint32_t* __restrict__ grown,
                                                               gsx_hip_adc_params p, int prune_large,
                                                               const float* __restrict__ opacity,
                                                               const float* __restrict__ logscale,
                                                               const float* __restrict__ rotation,
                                                               const float* __restrict__ max_screen_radius,
                                                               uint8_t* __restrict__ keep,
                                                               uint32_t* __restrict__ partials) {
    __shared__ uint32_t s_wave[kAdcThreads / kWave];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool kept = false;
    if (i < n + (int64_t)*grown) {
        const float o = adc_sigmoid(opacity[i]);
        const bool not_transparent = o > p.pruning_opacity_threshold;
        const float sx = gsx_expf(logscale[i * 3 + 0]), sy = gsx_expf(logscale[i * 3 + 1]),
                    sz = gsx_expf(logscale[i * 3 + 2]);
        float mx = sx;
        if (sy > mx) mx = sy;
        if (sz > mx) mx = sz;
        bool not_large_ws = true;
        if (p.max_world_scale > 0.0f) not_large_ws = mx < (p.max_world_scale * p.scene_scale);
        const float rn = fabsf(rotation[i * 4 + 0]) + fabsf(rotation[i * 4 + 1]) + fabsf(rotation[i * 4 + 2]) +
                         fabsf(rotation[i * 4 + 3]);
        const bool not_degenerate = rn > 1.1920928955078125e-07f;  // FLT_EPSILON
        kept = not_transparent && (not_large_ws || !prune_large) && not_degenerate;
        // not_large_ss of default.c:252-254
        if (max_screen_radius != nullptr && i < n && !(max_screen_radius[i] < p.max_screen_scale)) kept = false;
        keep[i] = kept ? 1 : 0;
    }
    const uint32_t count = adc_block_count(kept, s_wave);
    if (threadIdx.x == 0) partials[blockIdx.x] = count;
}

// Out row rank = row i for every kept row (stable compaction of all fields and moments; at least one row
// survives), with the statistics of the result's rows zeroed: out_aux, or rows_aux where every row is
// kept and the result stays in place. partials: the exclusive scan of adc_keep_kernel's counts, the
// total behind it. The workgroup lists its kept rows in LDS; its part of an out array is contiguous, and
// consecutive threads store consecutive floats of it (1M rows with their moments: 134 us with a thread
// per row and array set, 95 so; the bytes alone take 85 at the rate of a large copy).
__global__ __launch_bounds__(kAdcThreads) void adc_compact_kernel(int64_t n, const uint32_t* __restrict__ grown,
                                                                  const uint8_t* __restrict__ keep,
                                                                  const uint32_t* __restrict__ partials, RowSet src,
                                                                  RowSet dst, RowSet src_moments, RowSet dst_moments,
                                                                  RowSet rows_aux, RowSet out_aux) {
    __shared__ uint32_t s_wave[kAdcThreads / kWave];
    __shared__ uint32_t s_row[kAdcThreads];
    const int64_t count = n + (int64_t)*grown;
    const int64_t first = (int64_t)blockIdx.x * kAdcThreads;
    if (first >= count) return;
    const uint32_t survivors = partials[gridDim.x];
    const int64_t all = survivors > 0 ? survivors : 1;  // without a survivor the first row stays
    const uint32_t mine = (uint32_t)min((int64_t)kAdcThreads, count - first);
    if (all == count) {
        for (int f = 0; f < rows_aux.count; ++f)
            if (threadIdx.x < mine) rows_aux.f[f][first + threadIdx.x] = 0.0f;
        return;
    }
    const bool kept = threadIdx.x < mine && (survivors == 0 ? first + threadIdx.x == 0 : keep[first + threadIdx.x] != 0);
    uint32_t here;
    const uint32_t rank = block_exclusive_scan_256(kept ? 1u : 0u, s_wave, here);
    if (kept) s_row[rank] = threadIdx.x;
    __syncthreads();
    const int64_t to = partials[blockIdx.x];
    for (int f = 0; f < src.count; ++f) {
        const uint32_t w = (uint32_t)src.w[f];
        const float* const a = src.f[f] + first * w;
        float* const b = dst.f[f] + to * w;
        for (uint32_t e = threadIdx.x; e < here * w; e += kAdcThreads) {
            const uint32_t q = adc_row_of(e, w);
            b[e] = a[s_row[q] * w + (e - q * w)];
        }
    }
    for (int f = 0; f < src_moments.count; ++f) {
        const uint32_t w = (uint32_t)src_moments.w[f];
        const float* const a = src_moments.f[f] + first * w;
        float* const b = dst_moments.f[f] + to * w;
        for (uint32_t e = threadIdx.x; e < here * w; e += kAdcThreads) {
            const uint32_t q = adc_row_of(e, w);
            b[e] = a[s_row[q] * w + (e - q * w)];
        }
    }
    for (int f = 0; f < out_aux.count; ++f)
        if (threadIdx.x < here) out_aux.f[f][to + threadIdx.x] = 0.0f;
}

__global__ __launch_bounds__(kAdcThreads) void adc_reset_opacity_kernel(int64_t count, float max_logit,
                                                                        float* __restrict__ opacity,
                                                                        float* __restrict__ m, float* __restrict__ v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    // gsx_tensor_clamp_inplace(opacity, -FLT_MAX, logit(c)) then the optimizer group reset
    float o = opacity[i];
    if (o < -3.4028234663852886e+38f) o = -3.4028234663852886e+38f;
    if (o > max_logit) o = max_logit;
    opacity[i] = o;
    if (m != nullptr) m[i] = 0.0f;
    if (v != nullptr) v[i] = 0.0f;
}

// ---- MCMC (gsx/src/gsx-cpu/adc/mcmc.c) ---------------------------------------------------------

// mcmc.c:13-18: logistic gate that lets only nearly transparent Gaussians move
__device__ inline float mcmc_noise_gate(float opacity) {
    const float shifted = (1.0f - opacity) - 0.995f;
    return 1.0f / (1.0f + gsx_expf(-100.0f * shifted));
}

// mcmc.c:345-451 for Gaussian i: three normals from draws 6i..6i+5 of the step's stream, shaped
// by R diag(s^2) R^T, scaled by the gate and noise_strength * lr, added to mean3d. Arithmetic bounds it, the jump to
// draw 6i among it, so a thread takes the rows i, i + gridDim.x * kAdcThreads, ...: it jumps once and goes on by
// `step`, the jump over the rows between. (A step without a refine, 1M / 4M rows: 31.6 / 100 us with a jump for every
// row, 36.2 / 118 with two, the workgroup's on the scalar ALU and the lane's short one behind it; 30.3 / 77 so. With
// 1024 workgroups 30.2 / 92, with 2048 29.8 / 86.)
constexpr int64_t kNoiseBlocks = 3072;
__global__ __launch_bounds__(kAdcThreads) void mcmc_noise_kernel(int64_t n, float noise_lr,
                                                                 float* __restrict__ mean3d,
                                                                 const float* __restrict__ rotation,
                                                                 const float* __restrict__ logscale,
                                                                 const float* __restrict__ opacity,
                                                                 uint64_t rng_state, uint64_t rng_inc,
                                                                 gsx_pcg32_jump step) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    gsx_amd_pcg32 first;
    first.state = rng_state;
    first.inc = rng_inc;
    gsx_pcg32_advance(&first, 6ull * (uint64_t)i);
    for (; i < n; i += (int64_t)gridDim.x * blockDim.x, first.state = step.mult * first.state + step.plus) {
        const float op = adc_sigmoid(opacity[i]);
        const float gate = mcmc_noise_gate(op);
        const float sx = gsx_expf(logscale[i * 3 + 0]), sy = gsx_expf(logscale[i * 3 + 1]),
                    sz = gsx_expf(logscale[i * 3 + 2]);
        float qx = rotation[i * 4 + 0], qy = rotation[i * 4 + 1], qz = rotation[i * 4 + 2], qw = rotation[i * 4 + 3];
        gsx_amd_pcg32 rng = first;
        const float nx = adc_next_normal(&rng), ny = adc_next_normal(&rng), nz = adc_next_normal(&rng);
        const float qn = sqrtf(qx * qx + qy * qy + qz * qz + qw * qw);
        if (qn > 1e-8f) {
            const float iq = 1.0f / qn;
            qx *= iq;
            qy *= iq;
            qz *= iq;
            qw *= iq;
        }
        const float m00 = 1.0f - 2.0f * (qy * qy + qz * qz), m01 = 2.0f * (qx * qy - qw * qz),
                    m02 = 2.0f * (qx * qz + qw * qy);
        const float m10 = 2.0f * (qx * qy + qw * qz), m11 = 1.0f - 2.0f * (qx * qx + qz * qz),
                    m12 = 2.0f * (qy * qz - qw * qx);
        const float m20 = 2.0f * (qx * qz - qw * qy), m21 = 2.0f * (qy * qz + qw * qx),
                    m22 = 1.0f - 2.0f * (qx * qx + qy * qy);
        const float c00 = m00 * m00 * sx * sx + m01 * m01 * sy * sy + m02 * m02 * sz * sz;
        const float c01 = m00 * m10 * sx * sx + m01 * m11 * sy * sy + m02 * m12 * sz * sz;
        const float c02 = m00 * m20 * sx * sx + m01 * m21 * sy * sy + m02 * m22 * sz * sz;
        const float c11 = m10 * m10 * sx * sx + m11 * m11 * sy * sy + m12 * m12 * sz * sz;
        const float c12 = m10 * m20 * sx * sx + m11 * m21 * sy * sy + m12 * m22 * sz * sz;
        const float c22 = m20 * m20 * sx * sx + m21 * m21 * sy * sy + m22 * m22 * sz * sz;
        const float snx = nx * gate * noise_lr, sny = ny * gate * noise_lr, snz = nz * gate * noise_lr;
        mean3d[i * 3 + 0] = mean3d[i * 3 + 0] + (c00 * snx + c01 * sny + c02 * snz);
        mean3d[i * 3 + 1] = mean3d[i * 3 + 1] + (c01 * snx + c11 * sny + c12 * snz);
        mean3d[i * 3 + 2] = mean3d[i * 3 + 2] + (c02 * snx + c12 * sny + c22 * snz);
    }
}

// draw weight sigmoid(opacity) of every row (mcmc.c:502-511); per workgroup the number of dead rows
// (weight <= threshold) and, in the second array of gridDim.x + 1 words, of live rows with a
// positive weight
__global__ __launch_bounds__(kAdcThreads) void mcmc_weight_kernel(int64_t n, float threshold,
                                                                  const float* __restrict__ opacity,
                                                                  float* __restrict__ weight,
                                                                  uint32_t* __restrict__ partials) {
    __shared__ uint32_t s_wave[kAdcThreads / kWave];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float w = 0.0f;
    if (i < n) {
        w = adc_sigmoid(opacity[i]);
        weight[i] = w;
    }
    if (partials == nullptr) return;  // uniform
    const bool dead = i < n && w <= threshold;
    const uint32_t deads = adc_block_count(dead, s_wave);
    const uint32_t positives = adc_block_count(i < n && !dead && w > 0.0f, s_wave);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = deads;
        partials[gridDim.x + 1 + blockIdx.x] = positives;
    }
}

// dead rows in index order to dead_idx, live rows (and their weights) to live_idx / live_w; dead_before:
// the exclusive scan of mcmc_weight_kernel's dead counts
__global__ __launch_bounds__(kAdcThreads) void mcmc_split_kernel(int64_t n, float threshold,
                                                                 const float* __restrict__ weight,
                                                                 const uint32_t* __restrict__ dead_before,
                                                                 uint32_t* __restrict__ dead_idx,
                                                                 uint32_t* __restrict__ live_idx,
                                                                 float* __restrict__ live_w) {
    __shared__ uint32_t s_wave[kAdcThreads / kWave];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const float w = i < n ? weight[i] : 0.0f;
    const bool dead = i < n && w <= threshold;
    uint32_t total;
    const uint32_t r = dead_before[blockIdx.x] + block_exclusive_scan_256(dead ? 1u : 0u, s_wave, total);
    if (i >= n) return;
    if (dead) {
        dead_idx[r] = (uint32_t)i;
    } else {
        live_idx[i - r] = (uint32_t)i;
        live_w[i - r] = w;
    }
}

// source row of draw j (through the live list when given) and the per-row draw counts; sample[j] becomes
// 1 for one draw of every drawn row (the one that counted first), 0 for the others
__global__ __launch_bounds__(kAdcThreads) void mcmc_count_kernel(int64_t draws, int32_t* __restrict__ sample,
                                                                 const uint32_t* __restrict__ live_idx,
                                                                 uint32_t* __restrict__ src,
                                                                 uint32_t* __restrict__ counts) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= draws) return;
    const uint32_t s = live_idx != nullptr ? live_idx[sample[j]] : (uint32_t)sample[j];
    src[j] = s;
    sample[j] = atomicAdd(&counts[s], 1u) == 0u ? 1 : 0;
}

// ---- running float sums ------------------------------------------------------------------------
// cdf[j] = the float sum of max(weight, 0) over [0, j] in index order, each addition rounded to float,
// as the CPU backend's sampler forms it (mcmc.c:137-140); the draws compare against these very
// values. The chain of roundings looks serial, but while the total T stays in one binade
// [2^k, 2^(k+1)) it is T = m 2^(k-23) with an integer m, and adding w takes m to
//   m + round(w 2^(23-k)),
// where the rounding does not depend on m except for a tie, which goes to the even result, i.e. by
// m's parity. So what a run of additions adds to m is a pair of numbers, one per parity of the m it
// starts from, and pairs compose associatively. m only grows: if it ends below 2^24 it never left
// the binade, and the pair gave every sum exactly; otherwise the addition that leaves it is made in
// float and the chain goes on in the next binade (at most some 24 times).
// Totals below 2^-125 count as the binade k = -126 whatever their first bit: m is then below 2^23, the
// weights are whole ulps and nothing is rounded.
//  1. float_sum_maps_kernel: the pair of every 1024-element chunk for each binade from kSumLowest up.
//  2. float_sum_starts_kernel (one workgroup): the total before every chunk, by scans over the chunks'
//     pairs up to the chunk that leaves the binade, whose sum one wave forms. Below kSumLowest the
//     workgroup forms the pairs of its next 16 chunks itself, a wave each: only weights that are
//     tiny for thousands of rows stay there, and the maps of all binades would cost every other sum
//     four times step 1. (A refine of 1M rows of weight 1e-13: 0.56 ms; one chunk after the other
//     2.69, on the host 0.80.)
//  3. float_sums_kernel: every chunk's sums from its start.
// 1M weights: 0.12 ms on the device instead of 0.9 ms for the copy out, a host loop and the copy back.
constexpr int kSumItems = 16;                   // elements per lane
constexpr int kSumChunk = kSumItems * kWave;    // elements per chunk, one wave
constexpr uint32_t kSumLimit = 1u << 24;        // m from which the total has left the binade
constexpr int kSumLowest = -12;                 // lowest binade whose pairs are formed beforehand

struct SumMap {
    uint32_t even, odd;  // what m grows by from an even and from an odd start, at most kSumLimit
};

// first a, then b
__device__ inline SumMap sum_then(SumMap a, SumMap b) {
    SumMap r;
    r.even = min(a.even + ((a.even & 1u) != 0u ? b.odd : b.even), kSumLimit);
    r.odd = min(a.odd + ((a.odd & 1u) != 0u ? b.even : b.odd), kSumLimit);
    return r;
}

// adding w in the binade whose ulp is 1 / scale
__device__ inline SumMap sum_map_of(float w, float scale) {
    const float q = w * scale;  // exact (a power of two); below an ulp's half it counts as 0 either way
    if (!(q < (float)kSumLimit)) return SumMap{kSumLimit, kSumLimit};
    const float f = floorf(q), frac = q - f;
    const uint32_t n = (uint32_t)f;
    if (frac == 0.5f) return SumMap{n + (n & 1u), n + ((n & 1u) ^ 1u)};
    const uint32_t r = n + (frac > 0.5f ? 1u : 0u);
    return SumMap{r, r};
}

// k and m of a total (m 2^(k-23)), and the total of an m below 2^24
__device__ inline int sum_binade(float total) { return max((int)(__float_as_uint(total) >> 23), 1) - 127; }
__device__ inline uint32_t sum_mantissa(float total, int k) {
    return __float_as_uint(total) - ((uint32_t)(k + 126) << 23);
}
__device__ inline float sum_value(uint32_t m, int k) { return __uint_as_float(((uint32_t)(k + 126) << 23) + m); }

// 1 / ulp of binade k, divided by sum_prescale(k) where it would be above the largest float
__device__ inline float sum_prescale(int k) { return k < -100 ? 0x1p64f : 1.0f; }
__device__ inline float sum_scale(int k) { return __uint_as_float((uint32_t)(127 + 23 - k - (k < -100 ? 64 : 0)) << 23); }

// Inclusive composition over the lanes of a wave, lane 0 first.
__device__ inline SumMap wave_sum_scan(SumMap m) {
    const int lane = (int)__lane_id();
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        SumMap before;
        before.even = (uint32_t)__shfl_up((int)m.even, off, kWave);
        before.odd = (uint32_t)__shfl_up((int)m.odd, off, kWave);
        if (lane >= off) m = sum_then(before, m);
    }
    return m;
}

// The lane's 16 weights of a chunk, negative ones, NaN and those past count as 0. weight is 16-byte
// aligned: with single-float loads, whose lanes lie 64 bytes apart, a step of the sums below kSumLowest
// spent 8 of its 10 us on addresses.
__device__ inline void load_sum_chunk(const float* __restrict__ weight, int64_t count, int64_t chunk,
                                      float (&w)[kSumItems]) {
    const int64_t first = chunk * kSumChunk + (int64_t)__lane_id() * kSumItems;
    if (first + kSumItems <= count) {
        const float4* const from = reinterpret_cast<const float4*>(weight + first);
#pragma unroll
        for (int i = 0; i < kSumItems; i += 4) {
            const float4 v = from[i / 4];
            w[i] = v.x, w[i + 1] = v.y, w[i + 2] = v.z, w[i + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < kSumItems; ++i) w[i] = first + i < count ? weight[first + i] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kSumItems; ++i) w[i] = w[i] > 0.0f ? w[i] : 0.0f;
}

// The sums of a chunk whose lanes hold 16 weights each, from `total`: the lane's own in out, the last
// one returned to every lane.
__device__ inline float sum_chunk(float total, const float (&w)[kSumItems], float (&out)[kSumItems]) {
    const int lane = (int)__lane_id();
    int from = 0;  // lanes before it are done
    while (from < kWave) {
        int next;  // the lane to sum in float
        // (uniform) nothing up to the first weight, which leaves whatever binade: no pairs to scan (a refine of 200
        // rows: 139 us with them, 132 so)
        if (total == 0.0f) {
            bool any = false;
#pragma unroll
            for (int i = 0; i < kSumItems; ++i) any |= w[i] > 0.0f;
            const uint64_t some = wave_ballot(any);
            next = some != 0ull ? __builtin_ctzll(some) : kWave;
#pragma unroll
            for (int i = 0; i < kSumItems; ++i)
                if (lane < next) out[i] = 0.0f;
        } else {
            const int k = sum_binade(total);
            const float pre = sum_prescale(k), scale = sum_scale(k);
            const uint32_t m0 = sum_mantissa(total, k);
            SumMap map{0u, 0u};
#pragma unroll
            for (int i = 0; i < kSumItems; ++i) map = sum_then(map, sum_map_of(w[i] * pre, scale));
            if (lane < from) map = SumMap{0u, 0u};
            const SumMap incl = wave_sum_scan(map);
            const uint32_t end = m0 + ((m0 & 1u) != 0u ? incl.odd : incl.even);
            uint32_t start = (uint32_t)__shfl_up((int)end, 1, kWave);
            if (lane == 0) start = m0;
            const uint64_t left = wave_ballot(end >= kSumLimit);
            next = left != 0ull ? __builtin_ctzll(left) : kWave;
            if (lane >= from && lane < next) {
                uint32_t m = start;
#pragma unroll
                for (int i = 0; i < kSumItems; ++i) {
                    const SumMap e = sum_map_of(w[i] * pre, scale);
                    m += (m & 1u) != 0u ? e.odd : e.even;
                    out[i] = sum_value(m, k);
                }
            }
            const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)(next == kWave ? end : start), min(next, kWave - 1));
            total = sum_value(m, k);
        }
        if (next == kWave) break;
#pragma unroll
        for (int i = 0; i < kSumItems; ++i) {
            total += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w[i]), next));
            if (lane == next) out[i] = total;
        }
        from = next + 1;
    }
    return total;
}

// One workgroup per chunk, wave w taking the binades kSumLowest + w, + w + 4, ...; maps[b * chunks + chunk]
// for binade kSumLowest + b.
__global__ __launch_bounds__(kAdcThreads) void float_sum_maps_kernel(const float* __restrict__ weight, int64_t count,
                                                                     int binades, SumMap* __restrict__ maps) {
    float w[kSumItems];
    load_sum_chunk(weight, count, blockIdx.x, w);
    for (int k = (int)(threadIdx.x / kWave); k < binades; k += kAdcThreads / kWave) {
        const float scale = sum_scale(kSumLowest + k);
        SumMap map{0u, 0u};
#pragma unroll
        for (int i = 0; i < kSumItems; ++i) map = sum_then(map, sum_map_of(w[i], scale));
        map = wave_sum_scan(map);
        if (__lane_id() == kWave - 1) maps[(int64_t)k * gridDim.x + blockIdx.x] = map;
    }
}

constexpr int kSumStartThreads = 1024;
__global__ __launch_bounds__(kSumStartThreads) void float_sum_starts_kernel(const float* __restrict__ weight,
                                                                            int64_t count, int binades,
                                                                            const SumMap* __restrict__ maps,
                                                                            int64_t chunks, float* __restrict__ starts) {
    constexpr int kWaves = kSumStartThreads / kWave;
    __shared__ SumMap s_map[kWaves];
    __shared__ uint32_t s_bad[kWaves], s_m;
    __shared__ float s_total;
    const int lane = (int)__lane_id(), wave = (int)(threadIdx.x / kWave);
    float total = 0.0f;
    for (int64_t c = 0; c < chunks;) {
        const int k = sum_binade(total);
        const uint32_t m0 = sum_mantissa(total, k);
        if (k >= kSumLowest && k < kSumLowest + binades) {  // uniform
            const int64_t i = c + threadIdx.x;
            SumMap map{0u, 0u};
            if (i < chunks) map = maps[(int64_t)(k - kSumLowest) * chunks + i];
            map = wave_sum_scan(map);
            if (lane == kWave - 1) s_map[wave] = map;
            __syncthreads();
            SumMap before{0u, 0u};
            for (int w = 0; w < wave; ++w) before = sum_then(before, s_map[w]);
            const uint32_t first = m0 + ((m0 & 1u) != 0u ? before.odd : before.even);  // before this wave's chunks
            const uint32_t end = first + ((first & 1u) != 0u ? map.odd : map.even);
            uint32_t start = (uint32_t)__shfl_up((int)end, 1, kWave);
            if (lane == 0) start = first;
            const uint64_t left = wave_ballot(end >= kSumLimit);
            if (lane == 0) s_bad[wave] = left != 0ull ? (uint32_t)(wave * kWave + __builtin_ctzll(left)) : UINT32_MAX;
            __syncthreads();
            uint32_t bad = UINT32_MAX;
            for (int w = kWaves - 1; w >= 0; --w) bad = s_bad[w] != UINT32_MAX ? s_bad[w] : bad;
            if (i < chunks && threadIdx.x <= bad) starts[i] = sum_value(start, k);
            if (threadIdx.x == min(bad, (uint32_t)kSumStartThreads - 1u)) s_m = bad != UINT32_MAX ? start : end;
            __syncthreads();
            total = sum_value(s_m, k);
            if (bad == UINT32_MAX) {
                c += kSumStartThreads;
                continue;  // uniform
            }
            c += bad;
        } else if (c > 0) {  // (weights of use take the total past the lowest binade in the first chunk)
            const float pre = sum_prescale(k), scale = sum_scale(k);
            const int64_t i = c + wave;
            SumMap map{0u, 0u};
            if (i < chunks) {  // uniform in the wave
                float w[kSumItems];
                load_sum_chunk(weight, count, i, w);
#pragma unroll
                for (int j = 0; j < kSumItems; ++j) map = sum_then(map, sum_map_of(w[j] * pre, scale));
            }
            map = wave_sum_scan(map);
            if (lane == kWave - 1) s_map[wave] = map;
            __syncthreads();
            SumMap before{0u, 0u};
            for (int w = 0; w < wave; ++w) before = sum_then(before, s_map[w]);
            const SumMap own = s_map[wave];
            const uint32_t start = m0 + ((m0 & 1u) != 0u ? before.odd : before.even);
            const uint32_t end = start + ((start & 1u) != 0u ? own.odd : own.even);
            if (lane == 0) s_bad[wave] = end >= kSumLimit ? (uint32_t)wave : UINT32_MAX;
            __syncthreads();
            uint32_t bad = UINT32_MAX;
            for (int w = kWaves - 1; w >= 0; --w) bad = s_bad[w] != UINT32_MAX ? s_bad[w] : bad;
            if (lane == 0 && i < chunks && (uint32_t)wave <= bad) starts[i] = sum_value(start, k);
            if (lane == 0 && (uint32_t)wave == min(bad, (uint32_t)kWaves - 1u)) s_m = bad != UINT32_MAX ? start : end;
            __syncthreads();
            total = sum_value(s_m, k);
            if (bad == UINT32_MAX) {
                c += kWaves;
                continue;  // uniform
            }
            c += bad;
        } else if (threadIdx.x == 0) {
            starts[c] = total;
        }
        // the chunk that leaves the binade (or the first)
        if (wave == 0) {
            float w[kSumItems], out[kSumItems];
            load_sum_chunk(weight, count, c, w);
            const float t = sum_chunk(total, w, out);
            if (lane == 0) s_total = t;
        }
        __syncthreads();
        total = s_total;
        __syncthreads();  // read before the next chunk's is written
        ++c;
    }
}

// One wave per chunk.
__global__ __launch_bounds__(kAdcThreads) void float_sums_kernel(const float* __restrict__ weight, int64_t count,
                                                                 int64_t chunks, const float* __restrict__ starts,
                                                                 float* __restrict__ cdf) {
    const int64_t chunk = (int64_t)blockIdx.x * (kAdcThreads / kWave) + threadIdx.x / kWave;
    if (chunk >= chunks) return;
    float w[kSumItems], out[kSumItems];
    load_sum_chunk(weight, count, chunk, w);
    (void)sum_chunk(starts[chunk], w, out);
    const int64_t first = chunk * kSumChunk + (int64_t)__lane_id() * kSumItems;
#pragma unroll
    for (int i = 0; i < kSumItems; ++i)
        if (first + i < count) cdf[first + i] = out[i];
}

// C(n, k) in double, then float (mcmc.c:20-38)
__device__ inline float mcmc_binom(uint32_t n, uint32_t k) {
    if (k > n) return 0.0f;
    if (k == 0 || k == n) return 1.0f;
    if (k > n - k) k = n - k;
    double v = 1.0;
    for (uint32_t j = 1; j <= k; ++j) v = v * (double)(n - (k - j)) / (double)j;
    return (float)v;
}

// mcmc.c:283-343 for a source row drawn c > 0 times (ratio c + 1, at most 51): the opacity that
// c + 1 copies share, and the scale factor that keeps their summed footprint. A thread per draw, of
// which the one that owns its source row (mcmc_count_kernel) works: most lanes of a wave do, where a
// thread per row leaves one in ten (1M rows, 100k draws: 27 -> 12 us).
__global__ __launch_bounds__(kAdcThreads) void mcmc_relocate_kernel(int64_t draws, float min_opacity,
                                                                    const int32_t* __restrict__ owner,
                                                                    const uint32_t* __restrict__ src,
                                                                    const uint32_t* __restrict__ counts,
                                                                    float* __restrict__ opacity,
                                                                    float* __restrict__ logscale) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= draws || owner[j] == 0) return;
    const int64_t i = src[j];
    const uint32_t c = counts[i];
    const float so = adc_sigmoid(opacity[i]);
    const float sx = gsx_expf(logscale[i * 3 + 0]), sy = gsx_expf(logscale[i * 3 + 1]),
                sz = gsx_expf(logscale[i * 3 + 2]);
    uint32_t ratio = c + 1u;
    if (ratio > 51u) ratio = 51u;
    float clamped = so;
    if (clamped < 0.0f) clamped = 0.0f;
    if (clamped > 1.0f - 1e-6f) clamped = 1.0f - 1e-6f;
    float new_op = 1.0f - gsx_powf(1.0f - clamped, 1.0f / (float)ratio);
    float denom = 0.0f;
    for (uint32_t a = 1; a <= ratio; ++a) {
        for (uint32_t k = 0; k < a; ++k) {
            const float sign = (k % 2u) == 0u ? 1.0f : -1.0f;
            const float coeff = mcmc_binom(a - 1u, k);
            const float power = gsx_powf(new_op, (float)(k + 1u));
            denom += coeff * sign * power / sqrtf((float)(k + 1u));
        }
    }
    const float scale_coeff = fabsf(denom) <= 1e-8f ? 1.0f : so / denom;
    if (new_op < min_opacity) new_op = min_opacity;
    if (new_op > 1.0f - 1e-6f) new_op = 1.0f - 1e-6f;
    opacity[i] = adc_prob_to_logit(new_op);
    logscale[i * 3 + 0] = adc_logf(sx * scale_coeff);
    logscale[i * 3 + 1] = adc_logf(sy * scale_coeff);
    logscale[i * 3 + 2] = adc_logf(sz * scale_coeff);
}

// row dst[j] = row src[j] over the parameter fields (dst = dead_idx for a relocation, or the
// appended rows n + j when dst is null), and the optimizer moments of row zero[j] (the source of
// a relocation, the appended row of a growth) cleared. blockIdx.y names the array; consecutive threads
// take consecutive floats of its rows (and further ones from 2^32 floats on, which no launch has threads for).
__global__ __launch_bounds__(kAdcThreads) void mcmc_copy_kernel(int64_t draws, int64_t n,
                                                                const uint32_t* __restrict__ dst,
                                                                const uint32_t* __restrict__ src, RowSet rows,
                                                                RowSet moments, int zero_source_moments) {
    const bool moment = (int)blockIdx.y >= rows.count;
    const int f = moment ? (int)blockIdx.y - rows.count : (int)blockIdx.y;
    const uint32_t w = (uint32_t)(moment ? moments.w[f] : rows.w[f]);
    float* const a = moment ? moments.f[f] : rows.f[f];
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < draws * w; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = draws * w <= (int64_t)UINT32_MAX ? (int64_t)((uint32_t)e / w) : e / w;
        const int64_t c = e - j * w;
        const int64_t s = src[j];
        const int64_t t = dst != nullptr ? (int64_t)dst[j] : n + j;
        if (moment) a[(zero_source_moments ? s : t) * w + c] = 0.0f;
        else a[t * w + c] = a[s * w + c];
    }
}

__global__ __launch_bounds__(256) void gather_rows_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                          int64_t row_bytes, int64_t row_count,
                                                          const int32_t* __restrict__ index, int64_t src_rows,
                                                          int* __restrict__ out_of_range, int word_rows) {
    // word_rows: row_bytes and both base addresses are multiples of 4 (checked by the host)
    const int64_t words_per_row = row_bytes / 4;
    const int64_t total = word_rows ? row_count * words_per_row : row_count * row_bytes;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = word_rows ? e / words_per_row : e / row_bytes;
        const int64_t k = word_rows ? e % words_per_row : e % row_bytes;
        const int32_t s = index[r];
        if (s < 0 || (int64_t)s >= src_rows) {
            if (out_of_range != nullptr) *out_of_range = 1;
            continue;
        }
        if (word_rows) {
            reinterpret_cast<uint32_t*>(dst)[r * words_per_row + k] =
                reinterpret_cast<const uint32_t*>(src)[(int64_t)s * words_per_row + k];
        } else {
            dst[r * row_bytes + k] = src[(int64_t)s * row_bytes + k];
        }
    }
}

}  // namespace gsx_amd

using namespace gsx_amd;

namespace {

// workgroups of the largest launch: HIP refuses 2^32 threads
constexpr int64_t kAdcMostBlocks = UINT32_MAX / kAdcThreads;

unsigned adc_blocks(int64_t n) {
    int64_t b = (n + kAdcThreads - 1) / kAdcThreads;
    return (unsigned)(b < 1 ? 1 : b);
}

gsx_hip_status adc_fail(gsx_hip_status code, const char* what) {
    set_last_error(what);
    return code;
}

#define ADC_HIP_TRY(expr)                                                        \
    do {                                                                         \
        hipError_t e_ = (expr);                                                  \
        if (e_ != hipSuccess) return adc_fail((gsx_hip_status)e_, #expr);        \
    } while (0)

#define ADC_TRY(expr)                          \
    do {                                       \
        gsx_hip_status s_ = (expr);            \
        if (s_ != GSX_HIP_SUCCESS) return s_;  \
    } while (0)

// Grow-only scratch from the stream-ordered pool (pool.hip); an outgrown or released block returns
// to the pool behind the queued work of the stream of the call that last reserved it.
struct Scratch {
    void* ptr = nullptr;
    size_t bytes = 0;
    hipStream_t stream = nullptr;
    gsx_hip_status reserve(size_t need, hipStream_t s) {
        stream = s;
        if (need <= bytes) return GSX_HIP_SUCCESS;
        if (ptr != nullptr) (void)gsx_hip_pool_free(ptr, s);
        ptr = nullptr;
        bytes = 0;
        const size_t grow = need + need / 4 + 4096;
        gsx_hip_status st = gsx_hip_pool_malloc(&ptr, grow, s);
        if (st != GSX_HIP_SUCCESS) return st;
        bytes = grow;
        return GSX_HIP_SUCCESS;
    }
    void release() {
        if (ptr != nullptr) (void)gsx_hip_pool_free(ptr, stream);
        ptr = nullptr;
        bytes = 0;
    }
};

__global__ void adc_fill_kernel(float* __restrict__ p, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = 0.0f;
}

// Zeroes the first `count` floats of each of a set's arrays (blockIdx.y).
__global__ void adc_fill_rows_kernel(RowSet rows, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) rows.f[blockIdx.y][i] = 0.0f;
}

bool in_refine_window(const gsx_hip_adc_params& p, uint64_t step) {
    const uint64_t s0 = p.start_refine > 0 ? (uint64_t)p.start_refine : 0;
    const uint64_t s1 = p.end_refine > 0 ? (uint64_t)p.end_refine : 0;
    if (p.refine_every == 0) return false;
    if (step % (uint64_t)p.refine_every != 0) return false;
    return !(step < s0 || step > s1);
}

bool in_reset_window(const gsx_hip_adc_params& p, uint64_t step) {
    const uint64_t s0 = p.start_refine > 0 ? (uint64_t)p.start_refine : 0;
    const uint64_t s1 = p.end_refine > 0 ? (uint64_t)p.end_refine : 0;
    if (p.reset_every == 0) return false;
    if (step % (uint64_t)p.reset_every != 0) return false;
    return !(step < s0 || step >= s1);
}

RowSet param_rows(const gsx_hip_gs_rows& r, int* mean_f, int* rot_f, int* ls_f, int* op_f, bool with_aux) {
    RowSet s{};
    s.count = 0;
    auto add = [&](float* p, int w) {
        if (p != nullptr) {
            s.f[s.count] = p;
            s.w[s.count] = w;
            s.count += 1;
        }
    };
    *mean_f = s.count;
    add(r.mean3d, 3);
    *rot_f = s.count;
    add(r.rotation, 4);
    *ls_f = s.count;
    add(r.logscale, 3);
    *op_f = s.count;
    add(r.opacity, 1);
    add(r.sh0, 3);
    if (r.sh_degree >= 1) add(r.sh1, 9);
    if (r.sh_degree >= 2) add(r.sh2, 15);
    if (r.sh_degree >= 3) add(r.sh3, 21);
    if (with_aux) {
        add(r.grad_acc, 1);
        add(r.absgrad_acc, 1);
        add(r.visible_counter, 1);
        add(r.max_screen_radius, 1);
    }
    return s;
}

// The statistics that a refine restarts (one float per row each).
RowSet aux_rows(const gsx_hip_gs_rows& r) {
    RowSet s{};
    for (float* p : {r.grad_acc, r.absgrad_acc, r.visible_counter, r.max_screen_radius}) {
        if (p == nullptr) continue;
        s.f[s.count] = p;
        s.w[s.count] = 1;
        s.count += 1;
    }
    return s;
}

RowSet moment_rows(const gsx_hip_gs_rows& r) {
    static const int widths[8] = {3, 4, 3, 1, 3, 9, 15, 21};
    RowSet s{};
    s.count = 0;
    for (int k = 0; k < 8; ++k) {
        if (k >= 5 && r.sh_degree < k - 4) continue;
        if (r.first_moment[k] != nullptr) {
            s.f[s.count] = r.first_moment[k];
            s.w[s.count] = widths[k];
            s.count += 1;
        }
        if (r.second_moment[k] != nullptr) {
            s.f[s.count] = r.second_moment[k];
            s.w[s.count] = widths[k];
            s.count += 1;
        }
    }
    return s;
}

// Whether two sets bind the same parameter fields and moments (the compaction pairs them in order).
bool same_fields(const gsx_hip_gs_rows& a, const gsx_hip_gs_rows& b) {
    const float* const sh[3][2] = {{a.sh1, b.sh1}, {a.sh2, b.sh2}, {a.sh3, b.sh3}};
    for (int d = 0; d < 3; ++d)
        if (a.sh_degree > d && (sh[d][0] != nullptr) != (sh[d][1] != nullptr)) return false;
    for (int k = 0; k < 8; ++k) {
        if (k >= 5 && a.sh_degree < k - 4) continue;
        if ((a.first_moment[k] != nullptr) != (b.first_moment[k] != nullptr)) return false;
        if ((a.second_moment[k] != nullptr) != (b.second_moment[k] != nullptr)) return false;
    }
    return true;
}

}  // namespace

struct gsx_hip_adc_context {
    gsx_amd_pcg32 rng;
    Scratch scratch;
    uint32_t* host = nullptr;  // pinned counts that kernels of any device write through host_dev
    uint32_t* host_dev = nullptr;
    hipEvent_t counted = nullptr;  // recorded behind the kernel that writes them
    int counted_device = -1;       // the device it belongs to
};

namespace {

// Makes ctx->counted an event of the current device. An event goes with one device and a context with
// none: it may be stepped on another device than it was made on.
hipError_t make_counted(gsx_hip_adc_context* ctx) {
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess || device == ctx->counted_device) return e;
    if (ctx->counted != nullptr) (void)hipEventDestroy(ctx->counted);
    ctx->counted = nullptr;
    ctx->counted_device = -1;
    e = hipEventCreateWithFlags(&ctx->counted, hipEventDisableTiming);
    if (e == hipSuccess) ctx->counted_device = device;
    return e;
}

gsx_hip_status record_counted(gsx_hip_adc_context* ctx, hipStream_t stream) {
    ADC_HIP_TRY(make_counted(ctx));
    ADC_HIP_TRY(hipEventRecord(ctx->counted, stream));
    return GSX_HIP_SUCCESS;
}

// MCMC position noise (gsx/src/gsx-cpu/adc/mcmc.c:345-451): none past end_refine or without
// noise strength; otherwise 6 draws per Gaussian from the context's stream.
gsx_hip_status mcmc_noise(gsx_hip_adc_context* ctx, const gsx_hip_adc_params& p, uint64_t global_step,
                          gsx_hip_gs_rows* rows, hipStream_t stream) {
    const int64_t n = rows->count;
    if (!(p.noise_strength > 0.0f) || n <= 0) return GSX_HIP_SUCCESS;
    if (p.end_refine > 0 && global_step >= (uint64_t)p.end_refine) return GSX_HIP_SUCCESS;
    const float noise_lr = p.noise_strength * p.mean3d_learning_rate;
    const unsigned all = adc_blocks(n), blocks = all < kNoiseBlocks ? all : (unsigned)kNoiseBlocks;
    hipLaunchKernelGGL(mcmc_noise_kernel, dim3(blocks), dim3(kAdcThreads), 0, stream, n, noise_lr, rows->mean3d,
                       rows->rotation, rows->logscale, rows->opacity, ctx->rng.state, ctx->rng.inc,
                       gsx_pcg32_jump_by(ctx->rng.inc, 6ull * blocks * kAdcThreads));
    ADC_HIP_TRY(hipGetLastError());
    gsx_pcg32_advance(&ctx->rng, 6ull * (uint64_t)n);
    return GSX_HIP_SUCCESS;
}

// Binades whose pairs float_sum_maps_kernel forms for `count` weights of at most 1 (whose sum is at
// most count), and the bytes of its pairs and the chunks' starts.
int sum_binades(int64_t count) {
    int b = 1;
    while (b < 32 && ((int64_t)1 << b) <= count) ++b;
    return b - kSumLowest;
}
int64_t sum_chunks(int64_t count) { return (count + kSumChunk - 1) / kSumChunk; }
size_t sum_temp_bytes(int64_t count) {
    return (size_t)sum_chunks(count) * ((size_t)sum_binades(count) * sizeof(SumMap) + sizeof(float));
}

// cdf[0..count) = running float sum of max(w, 0) in index order (see "running float sums" above).
gsx_hip_status mcmc_cdf(const float* weight, int64_t count, float* cdf, void* temp, hipStream_t stream) {
    const int64_t chunks = sum_chunks(count);
    const int binades = sum_binades(count);
    SumMap* maps = static_cast<SumMap*>(temp);
    float* starts = reinterpret_cast<float*>(maps + chunks * binades);
    hipLaunchKernelGGL(float_sum_maps_kernel, dim3((unsigned)chunks), dim3(kAdcThreads), 0, stream, weight, count,
                       binades, maps);
    hipLaunchKernelGGL(float_sum_starts_kernel, dim3(1), dim3(kSumStartThreads), 0, stream, weight, count, binades, maps,
                       chunks, starts);
    hipLaunchKernelGGL(float_sums_kernel, dim3((unsigned)((chunks + 3) / 4)), dim3(kAdcThreads), 0, stream, weight, count,
                       chunks, starts, cdf);
    ADC_HIP_TRY(hipGetLastError());
    return GSX_HIP_SUCCESS;
}

// Draws rows in proportion to the weights, and the relocated or appended rows they make: the sources'
// opacities and scales corrected, the rows copied to dst (or n, n + 1, ... when dst is null).
struct McmcDraws {
    const float* weight;       // [count]
    int64_t count, draws;
    const uint32_t* live_idx;  // rows of the weights (null: the rows themselves)
    const uint32_t* dst;
    float* cdf;
    int32_t* sample;
    uint32_t *src, *counts;    // [draws], [n]
    void* temp;
};
gsx_hip_status mcmc_draw(gsx_hip_adc_context* ctx, const McmcDraws& d, float min_opacity, gsx_hip_gs_rows* rows,
                         const RowSet& prow, const RowSet& mrow, hipStream_t stream) {
    const int64_t n = rows->count;
    ADC_TRY(mcmc_cdf(d.weight, d.count, d.cdf, d.temp, stream));
    ADC_TRY(gsx_hip_multinomial_i32(d.sample, d.draws, d.cdf, d.count, ctx->rng.state, ctx->rng.inc, stream));
    gsx_pcg32_advance(&ctx->rng, (uint64_t)d.draws);
    hipLaunchKernelGGL(adc_fill_kernel, dim3(adc_blocks(n)), dim3(kAdcThreads), 0, stream,
                       reinterpret_cast<float*>(d.counts), n);
    hipLaunchKernelGGL(mcmc_count_kernel, dim3(adc_blocks(d.draws)), dim3(kAdcThreads), 0, stream, d.draws, d.sample,
                       d.live_idx, d.src, d.counts);
    hipLaunchKernelGGL(mcmc_relocate_kernel, dim3(adc_blocks(d.draws)), dim3(kAdcThreads), 0, stream, d.draws, min_opacity,
                       d.sample, d.src, d.counts, rows->opacity, rows->logscale);
    int widest = 1;
    for (int f = 0; f < prow.count; ++f) widest = prow.w[f] > widest ? prow.w[f] : widest;
    const int64_t copy_blocks = (d.draws * widest + kAdcThreads - 1) / kAdcThreads;
    hipLaunchKernelGGL(mcmc_copy_kernel,
                       dim3((unsigned)(copy_blocks < kAdcMostBlocks ? copy_blocks : kAdcMostBlocks),
                            (unsigned)(prow.count + mrow.count)),
                       dim3(kAdcThreads), 0, stream, d.draws, n, d.dst, d.src, prow, mrow, d.dst != nullptr ? 1 : 0);
    ADC_HIP_TRY(hipGetLastError());
    return GSX_HIP_SUCCESS;
}

// MCMC refine (mcmc.c:453-766): relocate the dead rows, then grow; rows are appended in place.
gsx_hip_status mcmc_refine(gsx_hip_adc_context* ctx, const gsx_hip_adc_params& p, gsx_hip_gs_rows* rows,
                           int64_t capacity, int64_t* result_count, int64_t* out_counts, hipStream_t stream) {
    const int64_t n = rows->count;
    // the growth target: floor(n (1 + grow_ratio)) in double, capped at max_num_gaussians
    int64_t target = n;
    if (p.max_num_gaussians > 0 && p.grow_ratio > 0.0f) {
        double t = floor((double)n * (1.0 + (double)p.grow_ratio));
        if (t > (double)p.max_num_gaussians) t = (double)p.max_num_gaussians;
        if (t > (double)n) target = (int64_t)t;
    }
    if (capacity < target) return adc_fail(GSX_HIP_ERROR_OUT_OF_RANGE, "row capacity below the mcmc growth target");
    const int64_t draws_max = n > target - n ? n : target - n;
    // scratch: weight[n] | partials[2][blocks+1] | dead_idx[n] | live_idx[n] | live_w[n] |
    //          cdf[n] | sample[draws] | src[draws] | counts[n] | running sums' temp
    const unsigned blocks = adc_blocks(n);
    const size_t a = 256;
    auto up = [&](size_t x) { return (x + a - 1) / a * a; };
    size_t off = 0;
    const size_t o_w = off;
    off += up((size_t)n * 4);
    const size_t o_part = off;
    off += up(2 * ((size_t)blocks + 1) * 4);
    const size_t o_didx = off;
    off += up((size_t)n * 4);
    const size_t o_lidx = off;
    off += up((size_t)n * 4);
    const size_t o_lw = off;
    off += up((size_t)n * 4);
    const size_t o_cdf = off;
    off += up((size_t)n * 4);
    const size_t o_samp = off;
    off += up((size_t)draws_max * 4);
    const size_t o_src = off;
    off += up((size_t)draws_max * 4);
    const size_t o_cnt = off;
    off += up((size_t)n * 4);
    const size_t o_temp = off;
    off += up(sum_temp_bytes(n));
    ADC_TRY(ctx->scratch.reserve(off, stream));
    uint8_t* base = static_cast<uint8_t*>(ctx->scratch.ptr);
    float* weight = reinterpret_cast<float*>(base + o_w);
    uint32_t* partials = reinterpret_cast<uint32_t*>(base + o_part);
    uint32_t* didx = reinterpret_cast<uint32_t*>(base + o_didx);
    uint32_t* lidx = reinterpret_cast<uint32_t*>(base + o_lidx);
    float* lw = reinterpret_cast<float*>(base + o_lw);
    McmcDraws d{};
    d.cdf = reinterpret_cast<float*>(base + o_cdf);
    d.sample = reinterpret_cast<int32_t*>(base + o_samp);
    d.src = reinterpret_cast<uint32_t*>(base + o_src);
    d.counts = reinterpret_cast<uint32_t*>(base + o_cnt);
    d.temp = base + o_temp;
    int d0, d1, d2, d3;
    const RowSet prow = param_rows(*rows, &d0, &d1, &d2, &d3, false);
    const RowSet mrow = moment_rows(*rows);
    const char* const no_mass = "mcmc weighted sampling requires positive opacity mass";

    hipLaunchKernelGGL(mcmc_weight_kernel, dim3(blocks), dim3(kAdcThreads), 0, stream, n, p.pruning_opacity_threshold,
                       rows->opacity, weight, partials);
    ADC_HIP_TRY(hipGetLastError());
    // the scans' totals go straight to host memory: [0] dead rows, [1] live rows with a positive weight
    ADC_TRY(scan_partials_in_place(partials, blocks, stream, 2, ctx->host_dev));
    ADC_TRY(record_counted(ctx, stream));
    ADC_HIP_TRY(hipEventSynchronize(ctx->counted));
    const int64_t dead_count = ctx->host[0];
    out_counts[0] = dead_count;
    if (dead_count == n) {
        return adc_fail(GSX_HIP_ERROR_INVALID_STATE, "mcmc relocate requires at least one live gaussian");
    }
    if (dead_count > 0) {
        if (ctx->host[1] == 0) return adc_fail(GSX_HIP_ERROR_INVALID_STATE, no_mass);
        hipLaunchKernelGGL(mcmc_split_kernel, dim3(blocks), dim3(kAdcThreads), 0, stream, n, p.pruning_opacity_threshold,
                           weight, partials, didx, lidx, lw);
        ADC_HIP_TRY(hipGetLastError());
        d.weight = lw;
        d.count = n - dead_count;
        d.draws = dead_count;
        d.live_idx = lidx;
        d.dst = didx;
        ADC_TRY(mcmc_draw(ctx, d, p.pruning_opacity_threshold, rows, prow, mrow, stream));
        out_counts[2] += dead_count;
    }
    if (target > n) {
        // the rows that a relocation made have a positive weight, so only without one the mass can be 0
        if (dead_count == 0 && ctx->host[1] == 0) return adc_fail(GSX_HIP_ERROR_INVALID_STATE, no_mass);
        hipLaunchKernelGGL(mcmc_weight_kernel, dim3(blocks), dim3(kAdcThreads), 0, stream, n, p.pruning_opacity_threshold,
                           rows->opacity, weight, nullptr);
        ADC_HIP_TRY(hipGetLastError());
        d.weight = weight;
        d.count = n;
        d.draws = target - n;
        d.live_idx = nullptr;
        d.dst = nullptr;
        ADC_TRY(mcmc_draw(ctx, d, p.pruning_opacity_threshold, rows, prow, mrow, stream));
        out_counts[2] += d.draws;
    }
    *result_count = target;
    // gsx/src/gsx-cpu/adc.c:430-436: the auxiliary statistics restart after a refine
    const RowSet aux = aux_rows(*rows);
    if (aux.count > 0) {
        hipLaunchKernelGGL(adc_fill_rows_kernel, dim3(adc_blocks(target), (unsigned)aux.count), dim3(kAdcThreads), 0, stream,
                           aux, target);
        ADC_HIP_TRY(hipGetLastError());
    }
    return GSX_HIP_SUCCESS;
}

}  // namespace

extern "C" {

gsx_hip_status gsx_hip_adc_context_create(gsx_hip_adc_context** out, uint64_t seed) {
    if (out == nullptr) return adc_fail(GSX_HIP_ERROR_INVALID_ARGUMENT, "out must be non-null");
    gsx_hip_adc_context* ctx = new (std::nothrow) gsx_hip_adc_context();
    if (ctx == nullptr) return adc_fail(GSX_HIP_ERROR_OUT_OF_MEMORY, "adc context allocation");
    // gsx_pcg32_init(seed) -> pcg32_init(seed, seed) (gsx/src/gsx-random.c:25, gsx-cpu/adc.c:466)
    gsx_pcg32_seed2(&ctx->rng, seed, seed);
    hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&ctx->host), 4 * sizeof(uint32_t),
                                 hipHostMallocPortable | hipHostMallocMapped);
    if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&ctx->host_dev), ctx->host, 0);
    if (e == hipSuccess) e = make_counted(ctx);
    if (e != hipSuccess) {
        (void)gsx_hip_adc_context_destroy(ctx);
        return adc_fail((gsx_hip_status)e, "adc context creation");
    }
    *out = ctx;
    return GSX_HIP_SUCCESS;
}

gsx_hip_status gsx_hip_adc_context_destroy(gsx_hip_adc_context* ctx) {
    if (ctx == nullptr) return adc_fail(GSX_HIP_ERROR_INVALID_ARGUMENT, "context must be non-null");
    ctx->scratch.release();
    if (ctx->host != nullptr) (void)hipHostFree(ctx->host);
    if (ctx->counted != nullptr) (void)hipEventDestroy(ctx->counted);
    delete ctx;
    return GSX_HIP_SUCCESS;
}

gsx_hip_status gsx_hip_adc_step(gsx_hip_adc_context* ctx, const gsx_hip_adc_params* params, uint64_t global_step,
                                gsx_hip_gs_rows* rows, int64_t capacity, gsx_hip_gs_rows* out, int32_t* out_result_in_out,
                                int64_t* out_counts, hipStream_t stream) {
    if (ctx == nullptr || params == nullptr || rows == nullptr || out == nullptr || out_result_in_out == nullptr ||
        out_counts == nullptr) {
        return adc_fail(GSX_HIP_ERROR_INVALID_ARGUMENT, "adc arguments must be non-null");
    }
    const gsx_hip_adc_params& p = *params;
    if (p.algorithm != 0 && p.algorithm != 1 && p.algorithm != 2) {
        return adc_fail(GSX_HIP_ERROR_NOT_SUPPORTED, "adc algorithm");
    }
    if (p.algorithm != 2 && !(p.scene_scale > 0.0f)) {
        return adc_fail(GSX_HIP_ERROR_INVALID_ARGUMENT, "scene_scale must be positive");
    }
    const int64_t n = rows->count;
    if (rows->mean3d == nullptr || rows->rotation == nullptr || rows->logscale == nullptr || rows->opacity == nullptr ||
        rows->sh0 == nullptr) {
        return adc_fail(GSX_HIP_ERROR_INVALID_ARGUMENT, "mean3d, rotation, logscale, opacity, sh0 are required");
    }
    out_counts[0] = out_counts[1] = out_counts[2] = out_counts[3] = 0;
    *out_result_in_out = 0;
    out->count = n;
    gsx_hip_gs_rows* result = rows;
    int64_t result_count = n;
    const bool refine = in_refine_window(p, global_step);
    const bool reset = in_reset_window(p, global_step);
    if (p.algorithm == 2) {
        // gsx/src/gsx-cpu/adc.c:515-547: noise every step, then the refine
        ADC_TRY(mcmc_noise(ctx, p, global_step, rows, stream));
        if (refine && n > 0) ADC_TRY(mcmc_refine(ctx, p, rows, capacity, &result_count, out_counts, stream));
    } else if (refine && n > 0) {
        const float* acc = p.algorithm == 1 ? rows->absgrad_acc : rows->grad_acc;
        if (acc == nullptr) return adc_fail(GSX_HIP_ERROR_NOT_SUPPORTED, "refine requires the grad accumulator");
        const uint64_t cap = p.max_num_gaussians > 0 ? (uint64_t)p.max_num_gaussians : 0;
        const uint64_t budget = cap > (uint64_t)n ? cap - (uint64_t)n : 0;
        const int64_t max_rows = n + (int64_t)budget;
        if (capacity < max_rows) return adc_fail(GSX_HIP_ERROR_OUT_OF_RANGE, "row capacity below count + budget");
        // scratch: mode[n] | candidate and split partials [2][blocks + 1] | keep[rows] | keep partials | counts
        const unsigned blocks = adc_blocks(n);
        const int64_t most_rows = n + ((uint64_t)n < budget ? n : (int64_t)budget);
        const unsigned keep_blocks = adc_blocks(most_rows);
        const size_t a = 256;
        auto up = [&](size_t x) { return (x + a - 1) / a * a; };
        size_t off = 0;
        const size_t o_mode = off;
        off += up((size_t)n);
        const size_t o_part = off;
        off += up(2 * ((size_t)blocks + 1) * 4);
        const size_t o_keep = off;
        off += up((size_t)most_rows);
        const size_t o_kpart = off;
        off += up(((size_t)keep_blocks + 1) * 4);
        const size_t o_cnt = off;
        off += a;
        ADC_TRY(ctx->scratch.reserve(off, stream));
        uint8_t* base = static_cast<uint8_t*>(ctx->scratch.ptr);
        uint8_t* mode = base + o_mode;
        uint32_t* partials = reinterpret_cast<uint32_t*>(base + o_part);
        uint8_t* keep = base + o_keep;
        uint32_t* keep_partials = reinterpret_cast<uint32_t*>(base + o_kpart);
        uint32_t* cnt = reinterpret_cast<uint32_t*>(base + o_cnt);

        // everything is queued without the host's knowledge of a count: the kernels read the counts of
        // those before them, and the host reads them (host memory, [0] grown, [1] splits, [2] kept) once
        // the last is there, the compaction still running
        hipLaunchKernelGGL(adc_classify_kernel, dim3(blocks), dim3(kAdcThreads), 0, stream, n, p, rows->logscale, acc,
                           rows->visible_counter, mode, partials);
        ADC_HIP_TRY(hipGetLastError());
        ADC_TRY(scan_partials_in_place(partials, blocks, stream, 2));
        int mean_f, rot_f, ls_f, op_f;
        const RowSet prow = param_rows(*rows, &mean_f, &rot_f, &ls_f, &op_f, true);
        const RowSet mrow = moment_rows(*rows);
        hipLaunchKernelGGL(adc_grow_kernel, dim3(blocks), dim3(kAdcThreads), 0, stream, n, budget, mode, partials, prow, mrow,
                           ctx->rng.state, ctx->rng.inc, mean_f, rot_f, ls_f, op_f, cnt, ctx->host_dev);
        ADC_HIP_TRY(hipGetLastError());
        const int prune_large = global_step > (uint64_t)(p.reset_every > 0 ? p.reset_every : 0);
        hipLaunchKernelGGL(adc_keep_kernel, dim3(keep_blocks), dim3(kAdcThreads), 0, stream, n, cnt, p, prune_large,
                           rows->opacity, rows->logscale, rows->rotation,
                           p.max_screen_scale > 0.0f && prune_large ? rows->max_screen_radius : nullptr, keep,
                           keep_partials);
        ADC_HIP_TRY(hipGetLastError());
        ADC_TRY(scan_partials_in_place(keep_partials, keep_blocks, stream, 1, ctx->host_dev + 2));
        ADC_TRY(record_counted(ctx, stream));
        // out rows that cannot take the result are an error only if rows are pruned
        const bool out_bound = out->mean3d != nullptr && out->rotation != nullptr && out->logscale != nullptr &&
                               out->opacity != nullptr && out->sh0 != nullptr;
        gsx_hip_gs_rows to = *out;
        to.sh_degree = rows->sh_degree;
        int d0, d1, d2, d3;
        const bool out_same = out_bound && same_fields(*rows, to) &&
                              param_rows(to, &d0, &d1, &d2, &d3, true).count == prow.count;
        // the result's statistics restart (gsx/src/gsx-cpu/adc.c:446-452): zeroed, not copied
        const RowSet src = param_rows(*rows, &d0, &d1, &d2, &d3, false);
        if (out_same) {
            hipLaunchKernelGGL(adc_compact_kernel, dim3(keep_blocks), dim3(kAdcThreads), 0, stream, n, cnt, keep,
                               keep_partials, src, param_rows(to, &d0, &d1, &d2, &d3, false), mrow, moment_rows(to),
                               aux_rows(*rows), aux_rows(to));
            ADC_HIP_TRY(hipGetLastError());
        }
        ADC_HIP_TRY(hipEventSynchronize(ctx->counted));
        const uint64_t grown = ctx->host[0], splits = ctx->host[1];
        if (grown > 0) {
            gsx_pcg32_advance(&ctx->rng, 12ull * splits);
            out_counts[1] = (int64_t)(grown - splits);
            out_counts[2] = (int64_t)splits;
        }
        const int64_t grown_count = n + (int64_t)grown;
        const int64_t kept = ctx->host[2] == 0 ? 1 : (int64_t)ctx->host[2];
        if (kept < grown_count) {
            if (!out_bound) return adc_fail(GSX_HIP_ERROR_INVALID_ARGUMENT, "out rows are required when rows are pruned");
            out->sh_degree = rows->sh_degree;
            if (!out_same) return adc_fail(GSX_HIP_ERROR_INVALID_ARGUMENT, "out rows must bind the same fields as rows");
            out_counts[0] = grown_count - kept;
            result = out;
            *out_result_in_out = 1;
        } else if (!out_same) {
            const RowSet aux = aux_rows(*rows);
            if (aux.count > 0) {
                hipLaunchKernelGGL(adc_fill_rows_kernel, dim3(adc_blocks(kept), (unsigned)aux.count), dim3(kAdcThreads), 0,
                                   stream, aux, kept);
                ADC_HIP_TRY(hipGetLastError());
            }
        }
        result_count = kept;
    }
    if (reset && result_count > 0) {
        // default.c:275-314
        float c = p.opacity_clamp_value;
        if (c > 1.0f) c = 1.0f;
        if (c < 1e-6f) c = 1e-6f;
        float cc = c;
        if (cc <= 1e-6f) cc = 1e-6f;
        if (cc >= 1.0f - 1e-6f) cc = 1.0f - 1e-6f;
        const float max_logit = logf(cc / (1.0f - cc));
        hipLaunchKernelGGL(adc_reset_opacity_kernel, dim3(adc_blocks(result_count)), dim3(kAdcThreads), 0, stream,
                           result_count, max_logit, result->opacity, result->first_moment[3], result->second_moment[3]);
        ADC_HIP_TRY(hipGetLastError());
        out_counts[3] = 1;
    }
    result->count = result_count;
    return GSX_HIP_SUCCESS;
}

// Replaces gsx_cuda_gather_rows_kernel_launch (gsx/src/gsx-cuda/internal.h:396-405): out row r =
// src row index[r]. An index outside [0, src_row_count) sets *out_has_out_of_range (device int,
// may be null) and leaves that row unwritten; the host decides when to read the flag, so no
// synchronisation happens here (the CUDA backend syncs per gather, gsx-cuda/buffer.c:1179-1207).
gsx_hip_status gsx_hip_gather_rows_kernel_launch(const void* src, void* dst, int64_t row_bytes, int64_t row_count,
                                                 const int32_t* src_indices, int64_t src_row_count,
                                                 int* out_has_out_of_range, hipStream_t stream) {
    if (row_count <= 0) return GSX_HIP_SUCCESS;
    if (src == nullptr || dst == nullptr || src_indices == nullptr || row_bytes <= 0) {
        return adc_fail(GSX_HIP_ERROR_INVALID_ARGUMENT, "gather arguments must be non-null and sized");
    }
    const bool word_rows = (row_bytes & 3) == 0 && ((reinterpret_cast<uintptr_t>(src) |
                                                      reinterpret_cast<uintptr_t>(dst)) & 3) == 0;
    const int64_t total = word_rows ? row_count * (row_bytes / 4) : row_count * row_bytes;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 16384) blocks = 16384;
    hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, stream,
                       static_cast<const uint8_t*>(src), static_cast<uint8_t*>(dst),
                       row_bytes, row_count, src_indices, src_row_count, out_has_out_of_range, word_rows ? 1 : 0);
    ADC_HIP_TRY(hipGetLastError());
    return GSX_HIP_SUCCESS;
}

}  // extern "C"
