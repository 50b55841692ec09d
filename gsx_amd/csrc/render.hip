// render.hip - the gfx950 render path: preprocess, tile-key emission, tile ranges, blend
// forward, blend backward and projection backward.
//
// Semantics are those of the gsx CPU backend (gsx/src/gsx-cpu/render.c), which is the parity
// oracle: per-pixel order is (depth, Gaussian index), each pixel honours the Gaussian's 3-sigma
// pixel box, the -4.5 power cut, the 1/255 alpha cut and the 1e-4 transmittance cut, and the
// colour clamp max(c + 0.5, 0). The CUDA design this replaces (fastgs, kernels_forward.cuh /
// kernels_backward.cuh) differs in all of those, so none of its arithmetic is used here.
//
// Data layout in HBM (per Gaussian g, written by preprocess, read by emission and both blends),
// 48 B per visible Gaussian in two arrays (culled Gaussians only write tile_count = 0):
//   geo[2g+0] = {mean2d_x, mean2d_y, inv_a, 2*inv_b}      (conic of the dilated 2D covariance)
//   geo[2g+1] = {inv_c, opacity, x_min | x_max << 16, y_min | y_max << 16}   (ints as f32 bits)
//   col[g]    = {color_r, color_g, color_b, depth}
// Emission and tile counting gather records in depth order, one per Gaussian: they need the
// geometry only, a 32 B-aligned read. The blends read both and stage them in LDS as a BlendEntry,
// with the contribution box cbox[g] (8 B, behind the colours).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"

namespace gsx_amd {

constexpr int kBlendThreads = kTilePixels;  // 256: one pixel per thread, 4 waves per tile

// ---------------------------------------------------------------------------------------------
// Preprocess: render.c:850-1016 per Gaussian (culls, EWA projection, box, sigmoid, SH colour),
// plus the tile count of the box and, for TRAIN forwards, visible_counter += 1 (:980-982).
// ---------------------------------------------------------------------------------------------
// ---------------------------------------------------------------------------------------------
// Kept tiles (tile_cull.h): each tile row of a box keeps one contiguous run of tiles, given in
// closed form by the row's band columns. A wave walks the rows of its 64 Gaussians' boxes as one
// flattened sequence, 64 (Gaussian, row) items per step, so lanes stay busy whatever the box
// heights (a near-plane Gaussian's box can span the whole image, most span a row or two). Each
// lane's span constants live in LDS; a lane finds the owner of its item from the wave's
// exclusive prefix of row counts (marks at the lanes where a box's rows start, and a prefix
// maximum over the lanes). Counting adds each run's length to its owner's count; emission writes
// the runs of a step, 64 instances per sub-step, with a second owner search over the runs.
// ---------------------------------------------------------------------------------------------
constexpr int kWavesPerBlock = 4;
// Boxes of more tiles than this are emitted by waves of their own (big_boxes_wave): in depth order
// the near, large boxes are neighbours, and a wave holding many full-image boxes would serialise
// their instances. Counting walks every box in the waves (rows are few).
constexpr uint32_t kBigTiles = 1024;
// preprocess's per-workgroup partials: kept tiles in bits 0..39 (a workgroup keeps fewer than
// 2^34), big boxes in bits 40..51 and visible Gaussians from bit 52 (at most 256 each)
constexpr int kKeptPartBigShift = 40;
constexpr int kKeptPartVisibleShift = 52;

// Sort keys. Gaussians are first sorted by depth: key = (bits(depth) - bits(near)) << index_bits
// | index (visible depths lie in [near, far], where positive floats order like their bit
// patterns, so the offset keeps the order in fewer bits; invisible Gaussians get the offset
// bits(far) - bits(near) + 1 and sort last). Instances are then emitted in that depth order,
// instance_tile[position] = tile, and the tile indices are sorted stably (16-bit keys up to 65536 tiles,
// else 32-bit, the emission positions as values, implicit in the first pass): each tile's run is in (depth, index) order,
// the CPU backend's order, after two passes at 1080p.

__device__ inline uint32_t box_tiles(float4 geo1) {
    const uint32_t bx = __float_as_uint(geo1.z), by = __float_as_uint(geo1.w);
    return ((bx >> 16) / kTile - (bx & 0xffffu) / kTile + 1) * ((by >> 16) / kTile - (by & 0xffffu) / kTile + 1);
}

// The Gaussian's span constants from its geometry record (the record holds 2 * inv_b; halving
// is exact), as every pass that tests tiles forms them.
__device__ inline gsx_tile_span span_of(float4 r0, float4 r1) {
    const uint32_t bx = __float_as_uint(r1.z), by = __float_as_uint(r1.w);
    return gsx_tile_span_make(r0.x, r0.y, r0.z, r0.w * 0.5f, r1.x, r1.y, (int)(bx & 0xffffu), (int)(bx >> 16),
                              (int)(by & 0xffffu), (int)(by >> 16));
}

// A packed pixel box (box_lo / box_ext form, see in_box_packed) that no pixel lies in.
constexpr uint32_t kEmptyBoxLo = 0xffffffffu;

// The box the blend kernels test pixels against, in packed form (x0 | y0 << 16 and
// (x1 - x0) | (y1 - y0) << 16): the rectangle of the record's box that can hold a contributing
// pixel (gsx_contribution_box, from the record's mean, conic, opacity and box). It leaves out the
// corners of the 3-sigma box and, for all but the most opaque Gaussians, its rim, where every pixel
// fails the CPU's power or alpha cut; fewer pixels, and fewer waves of a tile, meet the entry.
// Preprocess stores it per visible Gaussian; key emission keeps using the record's box.
// k receives the Gaussian's span constants (span_of's), shared with the count of its tiles.
__device__ inline uint2 contribution_box_packed(float4 r0, float4 r1, gsx_tile_span& k) {
    const uint32_t bx = __float_as_uint(r1.z), by = __float_as_uint(r1.w);
    int xa, xb, ya, yb;
    gsx_contribution_box_and_span(r0.x, r0.y, r0.z, r0.w * 0.5f, r1.x, r1.y, (int)(bx & 0xffffu), (int)(bx >> 16),
                                  (int)(by & 0xffffu), (int)(by >> 16), &k, &xa, &xb, &ya, &yb);
    if (xa > xb || ya > yb) return make_uint2(kEmptyBoxLo, 0u);
    return make_uint2((uint32_t)xa | ((uint32_t)ya << 16), (uint32_t)(xb - xa) | ((uint32_t)(yb - ya) << 16));
}

// Kept run of tile row ty of a box: len tiles from tile0 (len = 0 when none).
__device__ inline void row_run(const gsx_tile_span& k, uint32_t bx, uint32_t by, uint32_t ty, int32_t tiles_x,
                               uint32_t& len, uint32_t& tile0) {
    const int x0 = (int)(bx & 0xffffu), x1 = (int)(bx >> 16), y0 = (int)(by & 0xffffu), y1 = (int)(by >> 16);
    const int py0 = max((int)ty * kTile, y0), py1 = min((int)ty * kTile + kTile - 1, y1);
    int xa, xb;
    gsx_tile_band_columns(&k, x0, x1, py0, py1, &xa, &xb);
    // (columns of a kept run lie in the box; box coordinates have 16 bits, so both factors have 12)
    const uint32_t ta = (uint32_t)xa / kTile;
    len = xa <= xb ? (uint32_t)xb / kTile - ta + 1u : 0u;
    tile0 = __umul24(ty, (uint32_t)tiles_x) + ta;
}

// One wave's boxes and the walk over their rows. The boxes with rows are held in lane order without
// gaps (slots 0, 1, ..), the non-empty runs of a step likewise.
struct WaveSpans {
    float ml[kWave], mh[kWave], my[kWave], b[kWave], ra[kWave], det[kWave], vr[kWave], aqs[kWave];  // gsx_tile_span
    uint32_t bx[kWave], by[kWave];  // box: x0 | x1 << 16, y0 | y1 << 16
    uint32_t excl[kWave];           // rows of the boxes before it
    uint32_t kept[kWave];           // counting: kept tiles of the box
    uint32_t base[kWave], g[kWave];  // emission: position of the box's first instance less the walked
                                     // instances of the boxes before it; its Gaussian
    uint2 run[kWave];                // emission: a step's runs (first tile less the run's start, Gaussian)
    uint32_t run_pos[kWave];         // .. their positions less their starts, where a wave's boxes are apart
    uint64_t starts[kWave];          // item_starts
};

// The owners of up to 4096 consecutive items (rows of boxes, instances of runs) win, win + 1, ..:
// every lane names the first item (`start`) of its owner, `any` when it has items. Bit i of the 64
// words is set when an owner begins at item win + i + 1, so the number of bits below an item (and
// of those of the windows before it) is its owner's place among the lanes with items: two mask
// counts per item, where marks and a prefix maximum over the lanes took 15 instructions. Lane j
// receives word j (the items 64 j .. of the window).
__device__ inline uint64_t item_starts(WaveSpans& w, bool any, uint32_t start, uint32_t win) {
    const uint32_t lane = __lane_id();
    w.starts[lane] = 0ull;
    wave_lds_sync();
    const uint32_t bit = start - 1u - win;  // wraps past the window for starts up to win
    if (any && bit < kWave * 64u) atomicOr(reinterpret_cast<uint32_t*>(w.starts) + (bit >> 5), 1u << (bit & 31u));
    wave_lds_sync();
    return w.starts[lane];
}

// Owner of the lane's item in the window's j-th 64 items; carry: owners begun before them.
__device__ inline uint32_t item_owner(uint64_t words, uint32_t j, uint32_t& carry) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)words, (int)j);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(words >> 32), (int)j);
    const uint32_t owner = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, carry));
    carry += (uint32_t)__popc(lo) + (uint32_t)__popc(hi);
    return owner;
}

// What a lane keeps of its box while the wave walks: the box's slot, its first row (of the wave's)
// and whether it has any; the wave's row count.
struct WalkLane {
    uint32_t slot, start, wave_rows;
    bool any;
};

// Stores the lane's span constants and box (no rows when !valid).
__device__ inline WalkLane stage_spans(WaveSpans& w, bool valid, const gsx_tile_span& k, float4 r1) {
    const uint32_t bx = __float_as_uint(r1.z), by = __float_as_uint(r1.w);
    const uint32_t rows = valid ? (by >> 16) / kTile - (by & 0xffffu) / kTile + 1 : 0u;
    const uint32_t incl = wave_inclusive_sum_u32(rows);
    const uint64_t m = wave_ballot(valid);
    WalkLane l;
    l.slot = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    l.start = incl - rows;
    l.wave_rows = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
    l.any = valid;
    if (valid) {
        w.ml[l.slot] = k.ml;
        w.mh[l.slot] = k.mh;
        w.my[l.slot] = k.my;
        w.b[l.slot] = k.b;
        w.ra[l.slot] = k.ra;
        w.det[l.slot] = k.det;
        w.vr[l.slot] = k.vr;
        w.aqs[l.slot] = k.aqs;
        w.bx[l.slot] = bx;
        w.by[l.slot] = by;
        w.excl[l.slot] = l.start;
        w.kept[l.slot] = 0;
    }
    wave_lds_sync();
    return l;
}

// The kept run of row p of the wave's rows, a row of the box in slot `owner`.
__device__ inline void staged_row_run(const WaveSpans& w, uint32_t owner, uint32_t p, int32_t tiles_x, uint32_t& len,
                                      uint32_t& tile0) {
    gsx_tile_span k;
    k.ml = w.ml[owner];
    k.mh = w.mh[owner];
    k.my = w.my[owner];
    k.b = w.b[owner];
    k.ra = w.ra[owner];
    k.det = w.det[owner];
    k.vr = w.vr[owner];
    k.aqs = w.aqs[owner];
    const uint32_t by = w.by[owner];
    row_run(k, w.bx[owner], by, (by & 0xffffu) / kTile + (p - w.excl[owner]), tiles_x, len, tile0);
}

// Kept tiles of the lane's box, summed over the wave's flattened rows (64 rows a step).
__device__ inline uint32_t count_wave_rows(WaveSpans& w, const WalkLane& l, int32_t tiles_x) {
    const uint32_t lane = __lane_id();
    uint32_t carry = 0;
    uint64_t words = 0;
    for (uint32_t base = 0; base < l.wave_rows; base += kWave) {
        const uint32_t j = (base / kWave) % kWave;
        if (j == 0) words = item_starts(w, l.any, l.start, base);
        const uint32_t owner = item_owner(words, j, carry);
        const uint32_t p = base + lane;
        if (p < l.wave_rows) {
            uint32_t len, tile0;
            staged_row_run(w, owner, p, tiles_x, len, tile0);
            if (len > 0) atomicAdd(&w.kept[owner], len);
        }
    }
    wave_lds_sync();
    return l.any ? w.kept[l.slot] : 0u;
}

// Writes the kept instances (instance_tile, instance_gaussian) of the wave's boxes, the rows of a
// box in order: instance i of the walk at position base + i of its box, where `base` is each lane's
// base[] and g its Gaussian. A step takes 64 rows, then writes their instances 64 at a time: where
// the boxes' positions follow one another (no big box between them), at one scalar address.
// Vector instructions bound it (about 0.55 wave instructions a ns). Per 64 instances they were ~35
// (marks, a prefix maximum over the lanes, three reads of the run and two 64-bit addresses) and are
// ~13, a row's 64 were ~200 and are ~160: 335M instances of a 1080p image 726 -> 695 us (2 GB are
// written), 5M 36 -> 31.5 us.
template <typename TileT>
__device__ inline void emit_wave_rows(WaveSpans& w, const WalkLane& l, uint32_t base_pos, uint32_t gaussian,
                                      int32_t tiles_x, uint32_t* __restrict__ instance_gaussian,
                                      TileT* __restrict__ instance_tile) {
    const uint32_t lane = __lane_id();
    const uint64_t boxes = wave_ballot(l.any);
    if (boxes == 0ull) return;  // uniform
    const uint32_t first_pos = (uint32_t)__builtin_amdgcn_readlane((int)base_pos, __builtin_ctzll(boxes));
    const bool together = wave_ballot(l.any && base_pos != first_pos) == 0ull;
    if (l.any) {
        w.base[l.slot] = base_pos;
        w.g[l.slot] = gaussian;
    }
    wave_lds_sync();
    uint32_t carry = 0, walked = 0;
    uint64_t words = 0;
    for (uint32_t base = 0; base < l.wave_rows; base += kWave) {
        const uint32_t j = (base / kWave) % kWave;
        if (j == 0) words = item_starts(w, l.any, l.start, base);
        const uint32_t owner = item_owner(words, j, carry);
        const uint32_t p = base + lane;
        uint32_t len = 0, tile0 = 0;
        if (p < l.wave_rows) staged_row_run(w, owner, p, tiles_x, len, tile0);
        const uint32_t incl = wave_inclusive_sum_u32(len);
        const uint32_t start = incl - len;
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        const uint64_t rm = wave_ballot(len > 0);
        const uint32_t slot =
            __builtin_amdgcn_mbcnt_hi((uint32_t)(rm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)rm, 0u));
        wave_lds_sync();  // the previous step's reads of the runs are done
        if (len > 0) {
            w.run[slot] = make_uint2(tile0 - start, w.g[owner]);
            w.run_pos[slot] = w.base[owner] + walked;
        }
        uint32_t* const out_g = instance_gaussian + (first_pos + walked);
        TileT* const out_t = instance_tile + (first_pos + walked);
        uint32_t run_carry = 0;
        uint64_t run_words = 0;
        for (uint32_t base2 = 0; base2 < total; base2 += kWave) {
            const uint32_t j2 = (base2 / kWave) % kWave;
            if (j2 == 0) run_words = item_starts(w, len > 0, start, base2);
            const uint32_t run = item_owner(run_words, j2, run_carry);
            const uint32_t q = base2 + lane;
            if (q < total) {
                const uint2 r = w.run[run];
                if (together) {
                    // (byte offsets below 2^32: a step's runs are at most 64 rows of at most 4096 tiles)
                    *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(out_g) + q * 4u) = r.y;
                    *reinterpret_cast<TileT*>(reinterpret_cast<char*>(out_t) + q * (uint32_t)sizeof(TileT)) =
                        (TileT)(r.x + q);
                } else {
                    const uint32_t pos = w.run_pos[run] + q;
                    instance_gaussian[pos] = r.y;
                    instance_tile[pos] = (TileT)(r.x + q);
                }
            }
        }
        walked += total;
    }
}

// The parameter gradient sinks (mean3d, rotation, logscale, opacity, sh0..sh3: `arrays` of
// them, count[a] floats each), zeroed by the blend backward so that the projection backward
// writes only the rows of Gaussians some tile's backward reached. Workgroup b zeroes slice
// b / arrays of array b % arrays; per[a] floats per slice, a multiple of 4, and vec4 bit a when
// the array is 16-byte aligned (16-byte stores); all set by the host.
struct SinkZeroing {
    float* ptr[8];
    int64_t count[8];
    int64_t per[8];
    int arrays;
    uint32_t vec4;
};

// This workgroup's slice: no load and no wait, so the stores leave beside the kernel's own work.
__device__ inline void zero_sink_slice(const SinkZeroing& z, uint32_t blk) {
    if (z.arrays == 0) return;
    const uint32_t a = blk % (uint32_t)z.arrays;
    float* const p = z.ptr[a];
    const int64_t lo = (int64_t)(blk / (uint32_t)z.arrays) * z.per[a];
    const int64_t hi = min(z.count[a], lo + z.per[a]);
    if (lo >= hi) return;  // uniform
    int64_t done = lo;
    if ((z.vec4 >> a) & 1u) {
        const int vecs = (int)((hi - lo) >> 2);
        float4* const q = reinterpret_cast<float4*>(p + lo);
        for (int i = threadIdx.x; i < vecs; i += blockDim.x) q[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        done = lo + 4 * (int64_t)vecs;
    }
    for (int64_t i = done + threadIdx.x; i < hi; i += blockDim.x) p[i] = 0.0f;
}

// Destination of the retained TRAIN state: each field array copied as the forward reads it
// (null dst[0] in an inference forward). Field order mean3d, rotation, logscale, opacity, sh0..sh3.
struct FieldSnapshot {
    float* dst[8];
};

__device__ inline void copy_floats(const float* __restrict__ src, float* __restrict__ dst, int64_t g, int width) {
    for (int k = 0; k < width; ++k) dst[g * width + k] = src[g * width + k];
}

__global__ __launch_bounds__(256) void preprocess_kernel(
    FieldSnapshot snap, int64_t n, const float* __restrict__ mean3d, const float* __restrict__ rotation,
    const float* __restrict__ logscale, const float* __restrict__ opacity, const float* __restrict__ sh0,
    const float* __restrict__ sh1, const float* __restrict__ sh2, const float* __restrict__ sh3, int sh_degree,
    CameraParams cam, float4* __restrict__ rec, float4* __restrict__ col, uint2* __restrict__ cbox,
    float4* __restrict__ cov_coef, uint32_t* __restrict__ tile_count,
    float* __restrict__ visible_counter, unsigned long long* __restrict__ kept_part,
    uint64_t* __restrict__ depth_keys, uint32_t depth_base, uint32_t depth_max, int index_bits,
    uint64_t big_key_flag, int count_shift, uint8_t* __restrict__ touched) {
    __shared__ WaveSpans s_spans[kWavesPerBlock];
    __shared__ uint32_t s_kept[kWavesPerBlock], s_big[kWavesPerBlock];
    WaveSpans& ws = s_spans[threadIdx.x / kWave];
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    // TRAIN: the blend backward marks the Gaussians it reaches (touched[g] = 1)
    if (touched != nullptr && g < n) touched[g] = 0;
    if (snap.dst[0] != nullptr && g < n) {
        // consecutive lanes copy consecutive rows; preprocess_one then reads them from cache
        copy_floats(mean3d, snap.dst[0], g, 3);
        reinterpret_cast<float4*>(snap.dst[1])[g] = reinterpret_cast<const float4*>(rotation)[g];
        copy_floats(logscale, snap.dst[2], g, 3);
        snap.dst[3][g] = opacity[g];
        copy_floats(sh0, snap.dst[4], g, 3);
        if (sh_degree >= 1) copy_floats(sh1, snap.dst[5], g, 9);
        if (sh_degree >= 2) copy_floats(sh2, snap.dst[6], g, 15);
        if (sh_degree >= 3) copy_floats(sh3, snap.dst[7], g, 21);
    }
    bool visible = false;
    float4 r0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), r1 = r0, r2 = r0;
    gsx_tile_span span = {};
    if (g < n) {
        const Projected p =
            preprocess_one(g, mean3d, rotation, logscale, opacity, sh0, sh1, sh2, sh3, sh_degree, cam, true);
        visible = p.visible;
        if (visible) {
            if (visible_counter != nullptr) visible_counter[g] += 1.0f;
            const float inv_a = p.c * p.inv_det;
            const float inv_b = -p.b * p.inv_det;
            const float inv_c = p.a * p.inv_det;
            const uint32_t bx = (uint32_t)p.x_min | ((uint32_t)p.x_max << 16);
            const uint32_t by = (uint32_t)p.y_min | ((uint32_t)p.y_max << 16);
            r0 = make_float4(p.mx, p.my, inv_a, 2.0f * inv_b);
            r1 = make_float4(inv_c, p.opacity, __uint_as_float(bx), __uint_as_float(by));
            r2 = make_float4(p.color[0], p.color[1], p.color[2], p.depth);
            rec[2 * g + 0] = r0;
            rec[2 * g + 1] = r1;
            col[g] = r2;
            cbox[g] = contribution_box_packed(r0, r1, span);
            if (cov_coef != nullptr) {
                // d(conic)/d(cov2d) coefficients with the CPU's rounding (render.c:1578-1579,
                // 1647-1655): the backward applies them per contribution, as the CPU does,
                // because for near-plane Gaussians with huge footprints the map is close to
                // singular and summing the conic gradients first would round very differently.
                const float det = p.a * p.c - p.b * p.b;
                const float k = 1.0f / (det * det);
                cov_coef[2 * g + 0] =
                    make_float4(-p.c * p.c * k, p.b * p.c * k, -p.b * p.b * k, -(p.a * p.c + p.b * p.b) * k);
                // with the doubled coefficients of the b row (exact: a power-of-two scaling) in the
                // free slots, so the backward forms none of them per pixel
                const float k0y = p.b * p.c * k, k1x = p.a * p.b * k;
                cov_coef[2 * g + 1] = make_float4(k1x, -p.a * p.a * k, 2.0f * k0y, 2.0f * k1x);
            }
        }
    }
    // emitted by big_boxes_wave; rank_gather_kernel lists them. (Appending them here to one list, an
    // atomic per wave on its length, serialised the kernel where a scene holds many: 112k of 6M
    // Gaussians, 790 us against 350 without the list.)
    const bool big = visible && box_tiles(r1) > kBigTiles;
    const uint32_t kept = count_wave_rows(ws, stage_spans(ws, visible, span, r1), cam.tiles_x);
    if (g < n) tile_count[g] = kept;
    // depth key of every Gaussian (~0 for invisible ones, which the depth sort drops);
    // big_key_flag (kBigKeyFlag or 0, see there) marks the big boxes for rank_gather_kernel;
    // count_shift > 0: the kept-tile count rides above the sorted bits, so rank_gather_kernel
    // reads it from the sorted key instead of gathering tile_count at random Gaussians
    if (g < n) {
        uint64_t key = ~0ull;
        if (visible) {
            uint32_t rel = __float_as_uint(r2.w) - depth_base;
            if (rel > depth_max) rel = depth_max;  // only for non-finite depths
            key = ((uint64_t)rel << index_bits) | (uint64_t)g | (big ? big_key_flag : 0ull);
            if (count_shift > 0) key |= (uint64_t)kept << count_shift;
        }
        depth_keys[g] = key;
    }
    // the workgroup's kept tiles, big boxes and visible Gaussians to kept_part[block], host
    // memory that the host sums for the instance count, the big-box launch and the visible count
    // (a wave's kept sum is below 64 * 2^24 tiles, a workgroup's below 2^34)
    const uint32_t wave_kept = wave_reduce_sum_u32(kept);
    const uint32_t wave_big = (uint32_t)__popcll(wave_ballot(big));
    const uint32_t wave_visible = (uint32_t)__popcll(wave_ballot(visible && g < n));
    if (__lane_id() == 0) {
        s_kept[threadIdx.x / kWave] = wave_kept;
        s_big[threadIdx.x / kWave] = wave_big | (wave_visible << 16);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long sum = 0, bigs = 0, vis = 0;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w) {
            sum += s_kept[w];
            bigs += s_big[w] & 0xffffu;
            vis += s_big[w] >> 16;
        }
        kept_part[blockIdx.x] = sum | (bigs << kKeptPartBigShift) | (vis << kKeptPartVisibleShift);
    }
}

// Marks a big box's depth key (big_boxes_wave needs its rank). Used only when the sorted depth
// bits end below bit 63, which holds for fewer than 2^31 Gaussians.
constexpr uint64_t kBigKeyFlag = 1ull << 63;

// Instance runs longer than this are summed in chunks by whole waves in the backward (see
// reduce_long_block), shorter ones by one lane each.
constexpr uint32_t kLaneRun = 32;

// After the depth sort of the V visible Gaussians (V = *depth_count): the Gaussian of every
// depth rank, its kept-tile count, and the rank of each Gaussian whose count exceeds long_chunk
// (the only ranks looked up by Gaussian: by the projection backward, for runs of several chunks).
// Ranks V..n-1 get count 0 and no Gaussian. The ranks of a workgroup's big boxes, each with the sum
// of the workgroup's counts before it, go to big_ranks[256 block ..], in order. Each workgroup also stores four numbers of its 256 ranks, the
// first steps of the scans that emission completes: block_sums[block] the sum of the counts, and
// behind each other in arrays of gridDim.x + 1 the number of counts above kLaneRun, of big boxes
// and of counts above long_chunk. (The lists of big boxes and of runs of several chunks took an
// atomic on one length per wave before: 181 us at 6M ranks with 112k such boxes, half of them serial.)
__global__ __launch_bounds__(256) void rank_gather_kernel(int64_t n, const uint32_t* __restrict__ depth_count,
                                                          const uint64_t* __restrict__ sorted_depth_keys,
                                                          uint64_t index_mask, bool big_flag,
                                                          int count_shift, uint32_t count_mask,
                                                          const uint32_t* __restrict__ tile_count,
                                                          const float4* __restrict__ rec,
                                                          uint32_t* __restrict__ rank_gaussian,
                                                          uint32_t* __restrict__ rank_count,
                                                          uint32_t* __restrict__ gaussian_rank,
                                                          uint32_t long_chunk,
                                                          uint2* __restrict__ big_ranks,
                                                          uint32_t* __restrict__ block_sums) {
    __shared__ uint32_t s_sum[kWavesPerBlock];
    __shared__ uint32_t s_marks[kWavesPerBlock];  // long runs, big boxes, runs of several chunks: a byte each
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t c = 0;
    bool big = false;
    if (r < n) {
        if (r < (int64_t)*depth_count) {
            const uint64_t key = sorted_depth_keys[r];
            const uint32_t g = (uint32_t)(key & index_mask);
            c = count_shift > 0 ? (uint32_t)(key >> count_shift) & count_mask : tile_count[g];
            big = c > 0 && (big_flag ? (key & kBigKeyFlag) != 0 : box_tiles(rec[2 * (size_t)g + 1]) > kBigTiles);
            rank_gaussian[r] = g;
            if (c > long_chunk) gaussian_rank[g] = (uint32_t)r;
        }
        rank_count[r] = c;
    }
    const uint32_t wave_sum = wave_reduce_sum_u32(c);
    const uint64_t longs_m = wave_ballot(c > kLaneRun), bigs = wave_ballot(big), multis_m = wave_ballot(c > long_chunk);
    if (__lane_id() == 0) {
        s_sum[threadIdx.x / kWave] = wave_sum;
        s_marks[threadIdx.x / kWave] = (uint32_t)__popcll(longs_m) | ((uint32_t)__popcll(bigs) << 8) |
                                       ((uint32_t)__popcll(multis_m) << 16);
    }
    __syncthreads();
    if (bigs != 0ull) {  // uniform in the wave
        uint32_t at = blockIdx.x * blockDim.x, before = wave_inclusive_sum_u32(c) - c;
        for (int w = 0; w < (int)(threadIdx.x / kWave); ++w) {
            at += (s_marks[w] >> 8) & 0xffu;
            before += s_sum[w];
        }
        if (big) big_ranks[at + (uint32_t)__popcll(bigs & lanemask_lt())] = make_uint2((uint32_t)r, before);
    }
    if (threadIdx.x == 0) {
        uint32_t sum = 0, longs = 0, big_total = 0, multis = 0;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; ++w) {
            sum += s_sum[w];
            longs += s_marks[w] & 0xffu;
            big_total += (s_marks[w] >> 8) & 0xffu;
            multis += s_marks[w] >> 16;
        }
        const size_t stride = (size_t)gridDim.x + 1;
        block_sums[blockIdx.x] = sum;
        block_sums[stride + blockIdx.x] = longs;
        block_sums[2 * stride + blockIdx.x] = big_total;
        block_sums[3 * stride + blockIdx.x] = multis;
    }
}

// ---------------------------------------------------------------------------------------------
// Instance emission in depth order: the Gaussian of rank r owns positions offset[r] ..
// offset[r+1]) of the instance array, one per kept tile of its box in row-major tile order
// (offsets are the exclusive scan of the counts in rank order). instance_tile[position] = tile
// (the sort's keys; the backward's reduction also looks up each position's tile) and
// instance_gaussian[position] = g. A stable sort of the tiles with the positions as values then
// leaves every tile's run in (depth, index) order, i.e. in ascending position.
// The offsets are finished here: block_prefix[b] is the exclusive scan of rank_gather_kernel's
// 256-rank sums, and emission workgroup b (ranks 256 b .. 256 b + 255, rank_gather_kernel's
// blocking) scans its own 256 counts; offsets[0..n] are stored for the later kernels
// (offsets[n] = total).
// ---------------------------------------------------------------------------------------------
template <typename TileT>
__device__ inline void emit_block(uint32_t b, int64_t n, int64_t rank_end, const float4* __restrict__ rec,
                                  const uint32_t* __restrict__ rank_gaussian, const uint32_t* __restrict__ rank_count,
                                  const uint32_t* __restrict__ block_prefix, uint32_t* __restrict__ offsets,
                                  int32_t tiles_x, uint32_t* __restrict__ instance_gaussian,
                                  TileT* __restrict__ instance_tile,
                                  size_t prefix_stride, uint32_t long_chunk, uint32_t* __restrict__ long_list,
                                  uint32_t* __restrict__ multi_list, WaveSpans* s_spans, uint32_t* s_wave) {
    WaveSpans& ws = s_spans[threadIdx.x / kWave];
    const int64_t r = (int64_t)b * blockDim.x + threadIdx.x;
    // the rank's count and Gaussian load together, then its whole record (one wait each)
    uint32_t cnt = 0, g = 0;
    if (r < n) {
        cnt = rank_count[r];
        g = rank_gaussian[r];
    }
    uint32_t block_total;
    const uint32_t o = block_prefix[b] + block_exclusive_scan_256(cnt, s_wave, block_total);
    if (r < n) offsets[r] = o;
    // offsets[n] (the instance total, read by the ranges pass) from the last rank launched: the
    // launch covers the visible ranks and at least one more, whose counts are 0
    if (r == rank_end - 1) offsets[n] = o + cnt;
    // the lists of long runs and of runs of several chunks, in rank order: the workgroup's scanned
    // start + the rank's place among the workgroup's (s_wave is free again after the scan's last
    // barrier)
    {
        const bool is_long = cnt > kLaneRun, is_multi = cnt > long_chunk;
        const uint64_t lm = wave_ballot(is_long), mm = wave_ballot(is_multi);
        if (__lane_id() == 0)
            s_wave[threadIdx.x / kWave] = (uint32_t)__popcll(lm) | ((uint32_t)__popcll(mm) << 16);
        __syncthreads();
        uint32_t before = 0;  // both counts: at most 192 each
        for (int w = 0; w < (int)(threadIdx.x / kWave); ++w) before += s_wave[w];
        if (is_long)
            long_list[block_prefix[prefix_stride + b] + (before & 0xffffu) + (uint32_t)__popcll(lm & lanemask_lt())] =
                (uint32_t)r;
        if (is_multi)
            multi_list[block_prefix[3 * prefix_stride + b] + (before >> 16) + (uint32_t)__popcll(mm & lanemask_lt())] =
                (uint32_t)r;
    }
    float4 r0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), r1 = r0;
    if (cnt > 0) {
        r0 = rec[2 * (size_t)g + 0];
        r1 = rec[2 * (size_t)g + 1];
    }
    // big boxes are emitted by big_boxes_wave; the walk numbers the wave's other instances
    // consecutively, so a lane's base is its offset less the walked instances of the lanes
    // before it (the counting walk's identical runs gave the counts)
    const bool walked = cnt > 0 && box_tiles(r1) <= kBigTiles;
    const uint32_t wcnt = walked ? cnt : 0u;
    const uint32_t base_pos = o - (wave_inclusive_sum_u32(wcnt) - wcnt);
    emit_wave_rows<TileT>(ws, stage_spans(ws, walked, span_of(r0, r1), r1), base_pos, g, tiles_x, instance_gaussian,
                          instance_tile);
}

// Big boxes first .. first + per_wave - 1 (in rank order, those below big_prefix[blocks]): a wave walks
// their rows as emit_block walks a wave's boxes. It runs beside emit_block in one launch, so each lane
// finds its box's place itself: box i is the (i - big_prefix[b])-th of block b's, the last block with
// big_prefix[b] <= i, and its offset block_prefix[b] plus the counts before it in the block. (The
// lanes past per_wave search along, so that the walk runs with the whole wave.)
template <typename TileT>
__device__ inline void big_boxes_wave(uint32_t first, uint32_t per_wave, const uint2* __restrict__ big_ranks,
                                      const uint32_t* __restrict__ big_prefix, uint32_t blocks,
                                      const float4* __restrict__ rec, int32_t tiles_x,
                                      const uint32_t* __restrict__ rank_gaussian,
                                      const uint32_t* __restrict__ rank_count,
                                      const uint32_t* __restrict__ block_prefix,
                                      uint32_t* __restrict__ instance_gaussian, TileT* __restrict__ instance_tile,
                                      WaveSpans& ws) {
    const uint32_t lane = __lane_id();
    const uint32_t total = big_prefix[blocks];
    if (first >= total) return;  // uniform
    const bool mine = lane < per_wave && first + lane < total;
    const uint32_t i = mine ? first + lane : first;
    uint32_t block = 0, span = blocks;  // the block is one of block .. block + span - 1
    if (per_wave == 1u) {  // uniform: the wave compares 64 counts at a time (3 loads in turn for 6M ranks,
                           // where halving takes 15: 3 us of a launch with a few big boxes)
        while (span > 1) {
            const uint32_t step = (span + kWave - 1) / kWave;
            const uint32_t at = lane * step;  // (lane 0 always counts)
            const uint64_t m = wave_ballot(at < span && big_prefix[min(block + at, blocks)] <= i);
            const uint32_t last = ((uint32_t)__popcll(m) - 1u) * step;
            block += last;
            span = min(step, span - last);
        }
    } else {
        while (span > 1) {
            const uint32_t half = span / 2;
            if (big_prefix[block + half] <= i) block += half;
            span -= half;
        }
    }
    const uint2 rank = big_ranks[block * 256u + (i - big_prefix[block])];
    const uint32_t g = rank_gaussian[rank.x];
    const uint32_t cnt = mine ? rank_count[rank.x] : 0u;
    const float4 r0 = rec[2 * (size_t)g + 0], r1 = rec[2 * (size_t)g + 1];
    // (less the instances of the wave's boxes before it, as in emit_block)
    const uint32_t base_pos = block_prefix[block] + rank.y - (wave_inclusive_sum_u32(cnt) - cnt);
    emit_wave_rows<TileT>(ws, stage_spans(ws, mine, span_of(r0, r1), r1), base_pos, g, tiles_x, instance_gaussian,
                          instance_tile);
}

// All emission in one launch: workgroups [0, big_blocks) hold the waves of big boxes, first so
// that their longer walks start early, big_per_wave boxes each; the rest are the emission workgroups of the ranks.
// block_prefix: rank_gather_kernel's four arrays of `prefix_stride` entries, scanned.
template <typename TileT>
__global__ __launch_bounds__(256) void emit_kernel(int64_t n, const float4* __restrict__ rec,
                                                   const uint32_t* __restrict__ rank_gaussian,
                                                   const uint32_t* __restrict__ rank_count,
                                                   const uint32_t* __restrict__ block_prefix, size_t prefix_stride,
                                                   uint32_t* __restrict__ offsets, int32_t tiles_x,
                                                   const uint2* __restrict__ big_ranks, uint32_t big_blocks,
                                                   uint32_t big_per_wave,
                                                   uint32_t* __restrict__ instance_gaussian,
                                                   TileT* __restrict__ instance_tile, uint32_t long_chunk,
                                                   uint32_t* __restrict__ long_list,
                                                   uint32_t* __restrict__ multi_list) {
    __shared__ WaveSpans s_spans[kWavesPerBlock];
    __shared__ uint32_t s_wave[kWavesPerBlock];
    if (blockIdx.x < big_blocks) {
        // no workgroup barrier on this path: each wave takes its own boxes
        const uint32_t w = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
        big_boxes_wave(w * big_per_wave, big_per_wave, big_ranks, block_prefix + 2 * prefix_stride,
                       (uint32_t)prefix_stride - 1u, rec, tiles_x, rank_gaussian, rank_count, block_prefix,
                       instance_gaussian, instance_tile, s_spans[threadIdx.x / kWave]);
        return;
    }
    // the rank workgroups cover ranks [0, rank_end): the visible ones and at least one past them
    // (ranks of invisible Gaussians emit nothing, and no kernel reads their offsets)
    const int64_t rank_end = min(n, (int64_t)(gridDim.x - big_blocks) * blockDim.x);
    emit_block(blockIdx.x - big_blocks, n, rank_end, rec, rank_gaussian, rank_count, block_prefix, offsets, tiles_x,
               instance_gaussian, instance_tile, prefix_stride, long_chunk, long_list, multi_list, s_spans, s_wave);
}

__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t* __restrict__ p, int64_t count, uint32_t v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = v;
}

__global__ __launch_bounds__(256) void fill_f32_kernel(float* __restrict__ p, int64_t count, float v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = v;
}

// The sorted tiles as 32-bit numbers, for a caller that looks at the retained intermediates.
__global__ __launch_bounds__(256) void widen_tiles_kernel(const uint16_t* __restrict__ in, int64_t count,
                                                          uint32_t* __restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = in[i];
}

// [start, end) of each tile's run in the sorted tile indices. Tiles without instances get
// (0, 0): the thread of the last instance before such a gap (or of the first instance, for the
// tiles before it) writes them, so no fill of all tiles is needed beforehand. count >= 1 (with
// no instances the caller fills the ranges). Each thread takes 4 consecutive sorted tiles (one
// 8- or 16-byte load), plus the tiles just before and after them for the boundaries.
template <typename TileT>
__global__ __launch_bounds__(256) void tile_ranges_kernel(const TileT* __restrict__ sorted_tiles,
                                                          const uint32_t* count_ptr, uint32_t tiles,
                                                          uint2* __restrict__ ranges) {
    const uint32_t count = *count_ptr;
    const uint32_t i0 = 4u * (blockIdx.x * blockDim.x + threadIdx.x);
    if (i0 >= count) return;
    const uint32_t m = min(4u, count - i0);
    // the neighbours load with the thread's own (clamped in-range positions, not branches)
    const uint32_t t_prev = sorted_tiles[i0 == 0 ? 0u : i0 - 1u];
    const uint32_t t_next = sorted_tiles[min(i0 + m, count - 1u)];
    uint32_t t[4];
    if (m == 4) {
        struct alignas(4 * sizeof(TileT)) Four {
            TileT t[4];
        };
        const Four q = *reinterpret_cast<const Four*>(sorted_tiles + i0);
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) t[j] = q.t[j];
    } else {
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) t[j] = j < m ? sorted_tiles[i0 + j] : 0u;
    }
    const uint32_t prev = i0 == 0 ? UINT32_MAX : t_prev;
    const uint32_t next = i0 + m == count ? tiles : t_next;
    if (i0 == 0) {
        for (uint32_t u = 0; u < t[0]; ++u) ranges[u] = make_uint2(0u, 0u);
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        if (j < m) {
            const uint32_t before = j == 0 ? prev : t[j - 1];
            const uint32_t after = j == m - 1 ? next : t[j + 1];
            if (before != t[j]) ranges[t[j]].x = i0 + j;
            if (after != t[j]) {
                ranges[t[j]].y = i0 + j + 1;
                for (uint32_t u = t[j] + 1; u < after; ++u) ranges[u] = make_uint2(0u, 0u);
            }
        }
    }
}

// The same ranges for large instance counts: one thread per tile finds the lower bounds of its
// tile and of the next in the sorted tiles by binary search, the two searches in lockstep
// (ceil(log2(count + 1)) steps of two loads each, the same for every lane) instead of a pass over
// every instance. Tiles without instances get (0, 0).
template <typename TileT>
__global__ __launch_bounds__(256) void tile_ranges_search_kernel(const TileT* __restrict__ sorted_tiles,
                                                                 uint32_t count, uint32_t tiles, int steps,
                                                                 uint2* __restrict__ ranges) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= tiles) return;
    uint32_t lo0 = 0, hi0 = count, lo1 = 0, hi1 = count;
    for (int k = 0; k < steps; ++k) {
        const uint32_t m0 = lo0 + ((hi0 - lo0) >> 1), m1 = lo1 + ((hi1 - lo1) >> 1);
        // both loads in flight (positions clamped into the array; a finished search keeps lo = hi)
        const uint32_t v0 = sorted_tiles[min(m0, count - 1u)], v1 = sorted_tiles[min(m1, count - 1u)];
        if (lo0 < hi0) {
            if (v0 < t) lo0 = m0 + 1u; else hi0 = m0;
        }
        if (lo1 < hi1) {
            if (v1 < t + 1u) lo1 = m1 + 1u; else hi1 = m1;
        }
    }
    ranges[t] = lo0 < lo1 ? make_uint2(lo0, lo1) : make_uint2(0u, 0u);
}

// Workgroup -> tile mapping: consecutive workgroups are dealt round-robin to the 8 XCDs, so give
// each XCD a contiguous band of tiles (neighbouring tiles share Gaussians, and each XCD has its
// own L2).
__device__ inline int xcd_tile_index(int block, int tiles) {
    const int per = (tiles + 7) / 8;
    const int xcd = block & 7;
    const int local = block >> 3;
    const int t = xcd * per + local;
    return t;
}

// Pixel of thread t of a tile's 256-thread workgroup. Each wave takes an 8 x 8 quadrant of the
// tile (wave w: quadrant (w & 1, w >> 1), lane l: pixel (l & 7, l >> 3) in it), not four 16-pixel
// rows: a Gaussian's footprint meets fewer waves of a tile when the waves are square, and each
// wave that meets it works on every lane. The DPP rows of 16 lanes are two pixel rows of a
// quadrant; the backward's per-row partial sums do not depend on which pixels a row holds.
__device__ inline int2 tile_pixel_of_thread(int t) {
    const int w = t >> 6, l = t & 63;
    return make_int2(((w & 1) << 3) | (l & 7), ((w >> 1) << 3) | (l >> 3));
}

// The box test in packed 16-bit halves, three vector instructions: (px, py) lies in
// [x0, x1] x [y0, y1] iff both halves of (px | py << 16) - (x0 | y0 << 16) (each wrapping mod
// 2^16) are at most those of (x1 - x0) | (y1 - y0) << 16. The blend kernels stage each
// contribution box (contribution_box_packed) in this form (kEmptyBoxLo / 0 for none: no pixel
// coordinate is 65535).
typedef uint16_t gsx_u16x2 __attribute__((ext_vector_type(2)));
__device__ inline bool in_box_packed(uint32_t pxy, uint32_t lo, uint32_t ext) {
    const gsx_u16x2 d = __builtin_bit_cast(gsx_u16x2, pxy) - __builtin_bit_cast(gsx_u16x2, lo);
    const gsx_u16x2 m = __builtin_elementwise_min(d, __builtin_bit_cast(gsx_u16x2, ext));
    return __builtin_bit_cast(uint32_t, m) == __builtin_bit_cast(uint32_t, d);
}

// Transmittance checkpoints: the backward needs every contribution's exact T_before (the CPU
// records it, render.c:1501-1506; recomputing it by division perturbs the last bit, which the
// near-singular covariance gradient of near-plane Gaussians amplifies without bound). A TRAIN
// forward therefore stores each pixel's T at the start of every 8-entry bucket of its tile's
// list. Bucket k of a tile whose list starts at position x lives in slot x/8 + tile + k, which
// is collision-free and needs at most I/8 + tiles + 1 slots of 256 floats.
constexpr int kBucket = 8;

__device__ inline size_t checkpoint_slot(uint32_t range_start, int tile, uint32_t position) {
    return (size_t)(range_start / kBucket) + (size_t)tile + (size_t)((position - range_start) / kBucket);
}

// An entry of a tile's list as the blend kernels stage it in LDS, 48 bytes. The conic is stored as
// (-a / 2, -b, -c / 2): the power -(a dx^2 + 2 b dx dy + c dy^2) / 2 then needs no final
// multiplication, and every product rounds as the CPU's (a scaling by powers of two is exact).
struct BlendEntry {
    float4 a;  // mean2d x, y, -inv_a / 2, -inv_b
    float4 b;  // -inv_c / 2, opacity, colour r, g
    float4 c;  // colour b, contribution box low corner and extent (packed halves), next list position
};

__device__ inline BlendEntry blend_entry(float4 geo0, float4 geo1, float4 col, uint2 box, uint32_t next) {
    BlendEntry e;
    e.a = make_float4(geo0.x, geo0.y, -0.5f * geo0.z, -0.5f * geo0.w);
    e.b = make_float4(-0.5f * geo1.x, geo1.y, col.x, col.y);
    e.c = make_float4(col.z, __uint_as_float(box.x), __uint_as_float(box.y), __uint_as_float(next));
    return e;
}

// Whether an entry can contribute to a pixel of the 8 x 8 quadrant whose first pixel is (qx, qy): its
// contribution box meets the quadrant, and so does the ellipse inside the box where the power and
// alpha cuts can pass. Lane l of a wave asks for entry l of 64, so one ballot tells the wave which of
// them it has to look at: an entry that misses the quadrant costs 1/64 of this test instead of a box
// test by every pixel, and the branches of the walk are scalar.
// The power is a concave function of the pixel's offset where the conic is positive definite, so over
// the quadrant it is at most its tangent at the quadrant's point p nearest the mean. The entry is
// skipped when that bound stays below the cut, max(-4.5, ln(1 / (255 opacity))), by 1e-3 and 1e-5 of
// the terms' largest sum (40 times the rounding of the power as the pixels evaluate it; the bound's
// own is about twice that). A conic that is not positive definite by 2^-16 of its terms, and any NaN,
// keeps the entry. Of the entries whose boxes meet a quadrant before its pixels close, 12 to 13% are skipped in
// a cube of long Gaussians (100k and 500k) and 7% of the round ones on a plane: forward 62 -> 57 us (100k,
// 640x480), 97 -> 89 (500k, 720p, TRAIN), backward 185 -> 179. In the clusters a few near Gaussians close the
// tiles, and none is skipped.
__device__ inline bool box_meets_quadrant(const BlendEntry& e, uint32_t qx, uint32_t qy) {
    const uint32_t lo = __float_as_uint(e.c.y), ext = __float_as_uint(e.c.z);
    const uint32_t x0 = lo & 0xffffu, y0 = lo >> 16;
    return (x0 <= qx + 7u) & (x0 + (ext & 0xffffu) >= qx) & (y0 <= qy + 7u) & (y0 + (ext >> 16) >= qy);
}
__device__ inline bool entry_meets_quadrant(const BlendEntry& e, uint32_t qx, uint32_t qy) {
    // (uniform; pinned, so that what is formed from them is formed here and holds no registers in between)
    qx = (uint32_t)__builtin_amdgcn_readfirstlane((int)qx);
    qy = (uint32_t)__builtin_amdgcn_readfirstlane((int)qy);
    asm volatile("" : "+s"(qx), "+s"(qy));
    const float x0 = ((float)qx + 0.5f) - e.a.x, x1 = ((float)qx + 7.5f) - e.a.x;
    const float y0 = ((float)qy + 0.5f) - e.a.y, y1 = ((float)qy + 7.5f) - e.a.y;
    const float px = __builtin_fmaxf(x0, __builtin_fminf(x1, 0.0f)), py = __builtin_fmaxf(y0, __builtin_fminf(y1, 0.0f));
    const float gx = 2.0f * e.a.z * px + e.a.w * py, gy = e.a.w * px + 2.0f * e.b.x * py;
    const float bound = 0.5f * (px * gx + py * gy) + __builtin_fmaxf(gx * (x0 - px), gx * (x1 - px)) +
                        __builtin_fmaxf(gy * (y0 - py), gy * (y1 - py));
    const float far_x = __builtin_fabsf(px) + 7.0f, far_y = __builtin_fabsf(py) + 7.0f;
    const float terms = __builtin_fabsf(e.a.w) * far_x * far_y - e.a.z * far_x * far_x - e.b.x * far_y * far_y;
    const float cut = __builtin_fmaxf(-4.5f, -0.69314718f * __builtin_amdgcn_logf(255.0f * e.b.y));
    const float ac = 4.0f * e.a.z * e.b.x;
    const bool misses = (bound < cut - 1e-3f - 1e-5f * terms) & (e.a.z < 0.0f) & (e.b.x < 0.0f) &
                        ((ac - e.a.w * e.a.w) * 65536.0f >= ac);
    return box_meets_quadrant(e, qx, qy) & !misses;
}

// A regular entry: its 2D covariance has an eigenvalue ratio of at most kRegularRatio and eigenvalues
// of at most kRegularExtent (a standard deviation of 1024 pixels). With trace t and determinant d of
// the conic, ratio <= r iff t^2 <= d (r + 2 + 1 / r), and the covariance's larger eigenvalue is at most
// t / d; from the staged conic (halved: t / 2 and d / 4). A NaN is not regular.
//  * A pixel outside a regular entry's 3-sigma box fails the power cut by itself: it lies at least half
//    a pixel beyond 3 sigma, where the power is below -4.5 (1 + 1 / (3 sigma)) <= -4.5 (1 + 3e-4), and
//    the float evaluation is off by less than 6e-5 of it (the form's terms are at most 2 r = 128 times
//    their sum, each rounded a few times); the rounding of the box's own radius, below 1e-6 of it, is far less. So its pixels need no box test: 3 instructions of some 40,
//    left out where a whole tile is regular (blend_backward_kernel's moments: 934 -> 906 us at 1M
//    Gaussians on a plane; a branch per group in the forward cost more than it saved, 394 -> 417 us).
//  * The map from moments to covariance gradients loses no more digits than the ratio says
//    (blend_backward_kernel).
// The limit: of the entries that a tile's pixels reach, none is above 64 in a cube of 200k or 500k long Gaussians
// (0.4% are above 16, but in 40% of the tiles, one of which takes a whole tile's time: blend backward 230 us
// at 16, 179 at 64 and more) and none above 16 on a plane; all are, at any limit up to 16384, where near-plane
// Gaussians close the tiles (1M in clusters). Only a scene between these would gain from a larger limit:
// 6M at full HD have 6.1% of the entries and 92% of the tiles above 64 (589 us), 1.2 and 40% above 256 (546),
// 0.1 and 7% above 1024 (495). There the gradient's error at such ratios is not measured.
// A tile of fewer than kMomentPixels pixels (at an image's edge) forms every term per contribution all the same: moments
// of a single pixel near an entry's mean leave little of themselves when moved there, and such pixels are then all that
// a gradient comes from (images of 1x1, any scene: 0.5e-6 -> 7.3e-6 off 64 bits in the middle and 1.9e-3 at worst;
// of 2x2 0.6 -> 0.8e-6, of 4x4 and of 49x50 no more than before). Beside whole tiles the few cost nothing.
constexpr int kMomentPixels = 64;
constexpr float kRegularRatio = 64.0f;
constexpr float kRegularExtent = 1048576.0f;
__device__ inline bool entry_is_regular(const BlendEntry& e) {
    const float half_trace = -(e.a.z + e.b.x);
    const float quarter_det = e.a.z * e.b.x - 0.25f * e.a.w * e.a.w;
    return (half_trace * half_trace <= quarter_det * (kRegularRatio + 2.0f + 1.0f / kRegularRatio)) &
           (half_trace <= quarter_det * (2.0f * kRegularExtent));
}

// render.c:1045-1070 for one entry and pixel, without the transmittance: alpha, and whether the
// pixel takes the entry if it is still open. A power above 0 counts as 0 and one below the cut is not
// taken, so the exponential's argument is the power clamped to [cut, 0]; a NaN power is not taken.
template <bool kBoxTest>
__device__ inline bool blend_alpha(const BlendEntry& e, float fpx, float fpy, uint32_t pxy, const uint64_t* s_exp2,
                                   float& gval, float& alpha) {
    const float dx = fpx - e.a.x;
    const float dy = fpy - e.a.y;
    const float power = e.a.z * dx * dx + e.a.w * dx * dy + e.b.x * dy * dy;
    bool near = power >= kPowerThreshold;
    if (kBoxTest) near = near & in_box_packed(pxy, __float_as_uint(e.c.y), __float_as_uint(e.c.z));
    gval = gsx_expf_blend(__builtin_amdgcn_fmed3f(power, kPowerThreshold, 0.0f), s_exp2);
    alpha = fminf(kMaxFragmentAlpha, e.b.y * gval);
    return near & (alpha >= kMinAlpha);
}

// ---------------------------------------------------------------------------------------------
// Blend forward: render.c:1018-1088, per pixel in per-tile (depth, index) order. Records of the
// tile's Gaussians are staged through LDS in batches of 256; a tile stops early once every pixel
// has T < 1e-4. Writes out_rgb (CHW, background composed: C + T*bg), final T, the exclusive end
// of the last contributing position, and (TRAIN) the bucket checkpoints.
// Each wave walks, 64 entries at a time, only the entries whose box meets its quadrant, in groups
// of kGroup whose alphas (independent of the transmittance, some 30 dependent operations and two
// LDS reads each) are evaluated side by side before they are composited in order: a tile's list is a
// serial chain, which sets the time where few waves share a SIMD (4000 Gaussians on 48 tiles: 106 us
// testing every entry one by one, 49 so), and the vector ALUs set it otherwise (1M Gaussians on a plane
// at 1024^2: 506 -> 398 us; full-HD clusters 65 -> 55 us). Groups of 4 need 92 registers with the
// checkpoints (5 waves per SIMD; 2 need 62): the TRAIN forward takes 2 (398 against 426 us).
// ---------------------------------------------------------------------------------------------
template <bool kTrain>
__global__ __launch_bounds__(kBlendThreads) void blend_forward_kernel(
    const uint2* __restrict__ ranges, const uint32_t* __restrict__ values,
    const uint32_t* __restrict__ instance_gaussian, const float4* __restrict__ rec, const float4* __restrict__ col,
    const uint2* __restrict__ cbox, uint32_t* __restrict__ sorted_g,
    CameraParams cam, float* __restrict__ out_rgb,
    float* __restrict__ out_t, uint32_t* __restrict__ out_last, float* __restrict__ ckpt,
    uint32_t* __restrict__ tile_exact) {
    constexpr int kGroup = kTrain ? 2 : 4;
    __shared__ BlendEntry s_entry[kBlendThreads];
    __shared__ uint64_t s_exp2[GSX_EXPF_BLEND_TABLE_SIZE];
    __shared__ uint32_t s_exact;  // TRAIN: few pixels, or an entry that a wave looked at is not regular
    const int tiles = cam.tiles_x * cam.tiles_y;
    const int tile = xcd_tile_index(blockIdx.x, tiles);
    if (tile >= tiles) return;
    if (threadIdx.x < GSX_EXPF_BLEND_TABLE_SIZE) s_exp2[threadIdx.x] = gsx_expf_blend_entry(threadIdx.x);
    const int tx = tile % cam.tiles_x, ty = tile / cam.tiles_x;
    if (kTrain && threadIdx.x == 0)
        s_exact = min(cam.width - tx * kTile, kTile) * min(cam.height - ty * kTile, kTile) < kMomentPixels ? 1u : 0u;
    const int2 tp = tile_pixel_of_thread((int)threadIdx.x);
    const int px = tx * kTile + tp.x;
    const int py = ty * kTile + tp.y;
    const bool inside = px < cam.width && py < cam.height;
    const uint2 range = ranges[tile];
    const float fpx = (float)px + 0.5f;
    const float fpy = (float)py + 0.5f;
    const uint32_t pxy = (uint32_t)px | ((uint32_t)py << 16);  // for in_box_packed
    const uint32_t lane = __lane_id();
    const uint32_t qx = (uint32_t)px & ~7u, qy = (uint32_t)py & ~7u;
    // t only falls, and a pixel is done once an accepted contribution takes it below the
    // threshold, so "done" is t < threshold; pixels outside the image start done (t = 0, never
    // written out)
    float t = inside ? 1.0f : 0.0f, c0 = 0.0f, c1 = 0.0f, c2 = 0.0f;
    uint32_t last = range.x;
    // The first batch is kFirstBatch entries, staged by four threads each: where near Gaussians
    // saturate a tile its list ends there (metric scene: about 50 of some 650 entries per tile), and
    // 256 would mostly be loaded in vain. Later batches are 256, one entry per thread, whose Gaussians
    // are looked up a batch ahead.
    constexpr uint32_t kFirstBatch = kWave;
    uint32_t g_next = 0;
    uint32_t batch = kFirstBatch;
    for (uint32_t base = range.x; base < range.y; base += batch, batch = kBlendThreads) {
        const bool first = base == range.x;
        if (!first && __syncthreads_count(t < kTransmittanceThreshold ? 1 : 0) == kBlendThreads) break;
        const uint32_t slot = first ? threadIdx.x / 4 : threadIdx.x;
        const uint32_t j = base + slot;
        // past the list: the last entry's records, with a box no pixel lies in
        const uint32_t jc = min(j, range.y - 1u);
        const uint32_t g = base <= range.x + kFirstBatch ? instance_gaussian[values[jc]] : g_next;
        if (kTrain && j < range.y && (!first || (threadIdx.x & 3u) == 3u)) sorted_g[j] = g;  // for the backward
        const BlendEntry mine = blend_entry(rec[2 * (size_t)g], rec[2 * (size_t)g + 1], col[g],
                                            j < range.y ? cbox[g] : make_uint2(kEmptyBoxLo, 0u), j + 1u);
        if (!first) {
            s_entry[slot] = mine;
            if (range.y - base > (uint32_t)kBlendThreads)
                g_next = instance_gaussian[values[min(j + (uint32_t)kBlendThreads, range.y - 1u)]];
        } else if ((threadIdx.x & 3u) == 0u) {
            s_entry[slot] = mine;
        }
        __syncthreads();
        // wave-uniform bound, held in a scalar register
        const int count = __builtin_amdgcn_readfirstlane((int)min(batch, range.y - base));
        uint64_t open = wave_ballot(t >= kTransmittanceThreshold);
        // one entry's place in the order: its (independent) alpha composited where the pixel is open
        int bucket = -1;
        auto composite = [&](int k, bool ok, float alpha, const BlendEntry& e) {
            if (kTrain && k / kBucket != bucket) {  // uniform: the first entry of a bucket in this quadrant
                bucket = k / kBucket;
                if (t >= kTransmittanceThreshold)
                    ckpt[checkpoint_slot(range.x, tile, base + (uint32_t)k) * kBlendThreads + threadIdx.x] = t;
            }
            // a lane that does not take the entry uses alpha = 0: it adds (0 * colour) = +-0, which
            // leaves its sums exactly as they are (they start at +0 and stay finite), and multiplies t
            // by 1, so one select serves the colour sums and t
            const bool take = ok & (t >= kTransmittanceThreshold);
            const float a_used = take ? alpha : 0.0f;
            const float w = a_used * t;
            c0 = c0 + w * e.b.z;
            c1 = c1 + w * e.b.w;
            c2 = c2 + w * e.c.x;
            t = t * (1.0f - a_used);
            last = take ? __float_as_uint(e.c.w) : last;
        };
        for (int k0 = 0; k0 < count && !mask_none(open); k0 += kWave) {
            const BlendEntry& mine = s_entry[k0 + lane];
            // (an inference forward takes the boxes alone for the first 64: where pixels close early, the
            // test's latency before the first entry is not made up for: 1M Gaussians in clusters, 56.2 us
            // against 58.8 with it)
            uint64_t todo = !kTrain && base == range.x ? wave_ballot(box_meets_quadrant(mine, qx, qy))
                                                       : wave_ballot(entry_meets_quadrant(mine, qx, qy));
            if (kTrain && !mask_none(wave_ballot(!entry_is_regular(mine)) & todo) && lane == 0u) s_exact = 1u;
            while (todo != 0ull) {
                if (__builtin_popcountll(todo) >= kGroup) {
                    int k[kGroup];
                    bool ok[kGroup];
                    float alpha[kGroup], gval;
                    BlendEntry e[kGroup];
#pragma unroll
                    for (int i = 0; i < kGroup; ++i) {
                        k[i] = k0 + __builtin_ctzll(todo);
                        todo &= todo - 1ull;
                        e[i] = s_entry[k[i]];
                    }
#pragma unroll
                    for (int i = 0; i < kGroup; ++i)
                        ok[i] = blend_alpha<true>(e[i], fpx, fpy, pxy, s_exp2, gval, alpha[i]);
#pragma unroll
                    for (int i = 0; i < kGroup; ++i) composite(k[i], ok[i], alpha[i], e[i]);
                } else {
                    const int k = k0 + __builtin_ctzll(todo);
                    todo &= todo - 1ull;
                    const BlendEntry e = s_entry[k];
                    float alpha, gval;
                    const bool ok = blend_alpha<true>(e, fpx, fpy, pxy, s_exp2, gval, alpha);
                    composite(k, ok, alpha, e);
                }
                open = wave_ballot(t >= kTransmittanceThreshold);
                if (mask_none(open)) break;  // uniform: every pixel of this wave is saturated
            }
        }
        __syncthreads();
    }
    // (an empty list never reaches the barriers that order s_exact; its backward walks nothing)
    if (kTrain && threadIdx.x == 0) tile_exact[tile] = range.x < range.y ? s_exact : 0u;
    if (inside) {
        const size_t pix = (size_t)py * (size_t)cam.width + (size_t)px;
        const size_t plane = (size_t)cam.width * (size_t)cam.height;
        out_rgb[pix] = c0 + t * cam.bg[0];
        out_rgb[plane + pix] = c1 + t * cam.bg[1];
        out_rgb[2 * plane + pix] = c2 + t * cam.bg[2];
        out_t[pix] = t;
        out_last[pix] = last;
    }
}

// Per-Gaussian screen-space gradient accumulator, 9 floats per Gaussian:
//   dmean2d x, y | dcov2d a, b, c | dcolor r, g, b | dopacity (w.r.t. the sigmoid value)
constexpr int kGrad2d = 9;
constexpr int kGradRecord = 8;  // per-instance partials: channels 0-7 in one 32-byte record

// ---------------------------------------------------------------------------------------------
// Blend backward: render.c:1559-1666 restated per pixel, back to front, with the CPU's exact
// T_before: for each 8-entry bucket (last first) the pixel reloads the bucket's checkpointed T,
// replays the bucket forward (same operations as the forward, so T_before, G and the contribution
// set are bit-identical to the CPU's) and then walks it backwards accumulating the suffix colour.
// Each wave looks only at the entries that meet its quadrant, as the forward does.
//
// A tile takes one of two forms of the gradient terms (tile_exact, from the forward):
//  * Moments. Every term of an entry's nine partials is one of two per-pixel scalars, h = dL/dopacity
//    of the pixel and w = alpha T, times something fixed over the list: with dpow = opacity h,
//      dmean2d, d(conic)  are sums of dpow times 1, dx, dy, dx^2, dx dy, dy^2,
//      dcolor             are sums of w times the pixel's image gradient.
//    So the sum over a quadrant's 64 pixels is a product of matrices: 16 rows (h and w of 8 entries)
//    by 64 pixels, times 64 pixels by 16 columns (the monomials of the pixel's offset from an origin near
//    the entry's mean, and the three image gradients): 16 f32 16x16x4 matrix instructions per 8 entries.
//    (On gfx950 an f32 matrix instruction takes the vector ALUs' time, 32 cycles or 8 vector
//    instructions' worth; that is 16 per entry, where the products and their reduction over lanes took
//    some 60.) Once per entry and tile the moments are moved from that origin to the entry's mean, added
//    over the quadrants, and mapped through the conic and the d(conic)/d(cov2d) coefficients. The suffix
//    is one scalar, its product with the image gradient.
//    The move cancels: a second moment about a point at distance d from the mean is larger than the one
//    about the mean by d^2 / sigma^2, and so is its rounding. So the columns hold the moments about four
//    origins, (+/- 2, +/- 2) from the quadrant's centre, which share enough columns to fit the 16, and an
//    entry takes those on its mean's side. (About the centre alone, 9 columns, footprints of a pixel or
//    two lost up to a bit of the scale and rotation gradients: 0.97e-6 -> 1.76e-6 off 64 bits, now 1.03e-6,
//    5000 of sigma 0.6 to 0.8 on a plane. The selection costs 3 to 4% of the kernel.)
//  * Per contribution. That map amplifies rounding by the eigenvalue ratio of the 2D covariance:
//    near-plane Gaussians reach ratios of 1e6 and more, where the CPU's gradient is mostly the
//    rounding of its per-contribution map. A tile with an entry that is not regular forms every term per
//    contribution with the CPU's operations, the suffix colour and its division included, and sums the
//    nine values over the wave with lane swaps and DPP moves. So does a tile of few pixels (kMomentPixels).
//
// Reduction without atomics: every wave leaves one row of nine sums per entry in LDS, four threads
// per entry combine the four waves' rows, and the tile writes one 9-float partial per reached
// instance at its emission position (channels 0-7 as one 32-byte record of instance_grad, channel 8,
// the opacity term, in instance_grad_op) and its cut position (tile_cut: the instances past it were
// not reached and have no partial); reduce_instance_grads_kernel then sums each Gaussian's
// contiguous run of positions. The result is deterministic and immune to the contention of
// full-screen Gaussians (present in every tile), and the instances behind saturated pixels cost the
// backward nothing.
//
// Bound by instruction issue (82% of the SIMDs' cycles at 1M Gaussians on a plane, 73 vector
// instructions per walked quadrant and entry plus the products' 18 such; every term per contribution took 156).
// With every entry tested by every pixel and every term per contribution, and now: that plane at
// 1024^2 1233 -> 892 us; 500k in a cube at 720p 268 -> 184 us; 1M clustered at full HD (per contribution, all
// tiles) 222 -> 227 us: that walk alone would fit 6 waves per SIMD, and both in one kernel leave 5.
// f32 products for the per-contribution sums too were slower (255 us: 8 matrix instructions per entry
// instead of 24 lane operations), as was sharing both forms in one walk (191 us: 105 registers).
// 64-entry batches took 1052 us where 32 took 1174: fewer barriers.
// ---------------------------------------------------------------------------------------------
constexpr int kWavesPerTile = kBlendThreads / kWave;

// Entries per batch: staged together, four threads each, and combined together.
constexpr int kBackBatch = 64;
constexpr int kMomentEntries = 8;  // entries of one matrix product

typedef float gsx_f32x4 __attribute__((ext_vector_type(4)));

// Origins of an entry's moments in a quadrant: (+/- kMomentOrigin, +/- kMomentOrigin) from its centre, on the
// sides of the entry's mean.
constexpr float kMomentOrigin = 2.0f;

// Column c of a product's second factor (blend_backward_walk): its place in a row of sums (1, u, v, u^2, u v, v^2,
// image gradient), and a bit for each of the four sides whose entries take it (bit x + 2 y, x and y 1 where
// the mean lies on the + side). A nibble a column.
__device__ inline uint32_t moment_place(uint32_t c) { return (uint32_t)(0x8764444525231310ull >> (4u * c)) & 15u; }
__device__ inline uint32_t moment_sides(uint32_t c) { return (uint32_t)(0xfff142833cc55aafull >> (4u * c)) & 15u; }

// Sum over the four lanes of a quad, in every lane.
__device__ inline float quad_sum(float v) {
    v += dpp_move<0xb1, 0xf>(v);        // quad_perm [1,0,3,2]
    return v + dpp_move<0x4e, 0xf>(v);  // quad_perm [2,3,0,1]
}

// a's and b's sums over the lane pairs (l, l + 32): a's in lanes 0-31, b's in lanes 32-63.
__device__ inline float merge_halves(float a, float b) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// The same over neighbouring rows of 16 lanes: a's in rows 0 and 2, b's in rows 1 and 3.
__device__ inline float merge_rows(float a, float b) {
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// Sums of v[0..8] over the wave: the returned value of lane l is the sum of v[wave_sum9_index(l)],
// total8 that of v[8] in lane 63. Each merge halves the registers and the lanes a value spreads
// over: 24 lane operations for all nine.
__device__ inline int wave_sum9_index(uint32_t lane) {
    return (int)(((lane >> 1) & 4u) | ((lane >> 3) & 2u) | (lane >> 5));
}
__device__ inline float wave_sum9(const float (&v)[9], float& total8) {
    const float a = merge_rows(merge_halves(v[0], v[1]), merge_halves(v[2], v[3]));  // rows: 0, 2, 1, 3
    const float b = merge_rows(merge_halves(v[4], v[5]), merge_halves(v[6], v[7]));  // rows: 4, 6, 5, 7
    const bool b3 = __builtin_amdgcn_inverse_ballot_w64(0xff00ff00ff00ff00ull);      // lane bit 3
    const float keep = b3 ? b : a;
    const float send = b3 ? a : b;
    float d = keep + dpp_move<0x128, 0xf>(send);  // row_ror:8
    d += dpp_move<0x141, 0xf>(d);                 // row_half_mirror
    d = quad_sum(d);
    float t = quad_sum(v[8]);
    t += dpp_move<0x141, 0xf>(t);  // row_half_mirror
    t += dpp_move<0x140, 0xf>(t);  // row_mirror
    t += dpp_move<0x142, 0xa>(t);  // row_bcast:15 into rows 1 and 3
    t += dpp_move<0x143, 0xc>(t);  // row_bcast:31 into rows 2 and 3
    total8 = t;
    return d;
}

// LDS of a backward workgroup. s_sum: per wave a row of nine sums for each entry that it took, the
// highest entry first (s_used: which); a product writes kMomentEntries rows whatever its fill.
struct BackwardShared {
    BlendEntry entry[kBackBatch];  // c.w: the entry's emission position
    uint64_t exp2[GSX_EXPF_BLEND_TABLE_SIZE];
    uint64_t used[kWavesPerTile];
    alignas(8) uint32_t side[kWavesPerTile][kMomentEntries];  // of a product's entries (see flush)
    uint32_t max_last;
    float sum[kWavesPerTile][(kBackBatch + kMomentEntries) * kGrad2d];
    union {
        // rows 2 i (h) and 2 i + 1 (w) of the i-th entry of a product, 64 pixels each; the 4-float
        // blocks of row r are stored at block index ^ r, so that 16 lanes that read one block of 16
        // rows meet all banks
        alignas(256) float x[kWavesPerTile][2 * kMomentEntries * kWave];
        float4 k[2][kBackBatch];  // d(conic)/d(cov2d) coefficients (per contribution)
    };
};

// What a thread knows of its pixel.
struct BackwardPixel {
    float fpx, fpy;
    uint32_t pxy;
    uint32_t last;      // exclusive end of its contributions (the list's start: none, or outside)
    float t_final;
    float d0, d1, d2;   // image gradient
};

// The tile's list walked back to front: batches, within them the buckets that hold an entry for the
// wave. Workgroup-uniform arguments except pix.
template <bool kMoments>
__device__ inline void blend_backward_walk(BackwardShared& sm, const BackwardPixel& pix, uint2 range, int tile, int tx,
                                           int ty, uint32_t wave_last, uint32_t end_all, uint32_t part_end,
                                           const uint32_t* __restrict__ values, const uint32_t* __restrict__ sorted_g,
                                           const float4* __restrict__ rec, const float4* __restrict__ col,
                                           const uint2* __restrict__ cbox, const float4* __restrict__ cov_coef,
                                           const float* __restrict__ ckpt, const CameraParams& cam,
                                           float* __restrict__ instance_grad, float* __restrict__ instance_grad_op,
                                           uint8_t* __restrict__ touched) {
    const uint32_t lane = __lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const float d0 = pix.d0, d1 = pix.d1, d2 = pix.d2;
    // render.c:1552-1557: the suffix starts as T_final * background (moments: times the gradient)
    float s0 = pix.t_final * cam.bg[0], s1 = pix.t_final * cam.bg[1], s2 = pix.t_final * cam.bg[2];
    if (kMoments) s0 = s0 * d0 + s1 * d1 + s2 * d2;

    // Moments: this lane's column of the products' second factor, one value per step: step s takes the
    // pixels 16 (lane / 16) + s of the quadrant. With u, v the pixel's offset from the quadrant's centre
    // and a = kMomentOrigin the columns are 1; u - a, (u - a)^2, u + a, (u + a)^2; the same of v;
    // (u - a)(v - a), (u - a)(v + a), (u + a)(v - a), (u + a)(v + a); the image gradient. All are exact.
    float* const x = sm.x[wave];
    const uint32_t column = lane & 15u;
    float factor[kMoments ? 16 : 1];
    if constexpr (kMoments) {
        x[lane] = d0;
        x[kWave + lane] = d1;
        x[2 * kWave + lane] = d2;
        wave_lds_sync();
        const float* dcol = x + kWave * (max((int)column, 13) - 13) + 16 * (lane >> 4);
        const float ax = (column - 1u) % 4u < 2u ? kMomentOrigin : -kMomentOrigin;  // columns 1 to 8
        const float bx = column < 11u ? kMomentOrigin : -kMomentOrigin;             // columns 9 to 12
        const float by = (column & 1u) != 0u ? kMomentOrigin : -kMomentOrigin;
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const float u = (float)(s & 7) - 3.5f, v = (float)(2 * (int)(lane >> 4) + (s >> 3)) - 3.5f;
            const float t = (column < 5u ? u : v) - ax;
            float f = dcol[s];
            if (column < 13u) f = (u - bx) * (v - by);
            if (column < 9u) f = (column & 1u) != 0u ? t : t * t;
            if (column == 0u) f = 1.0f;
            factor[s] = f;
        }
        wave_lds_sync();
    }
    // where this lane reads its row of the first factor: row lane % 16, block 4 (lane / 16) of it (and,
    // for t = 1..3, that byte offset ^ 16 t)
    const uint32_t read_at = column * (kWave * 4u) + ((4u * (lane >> 4)) ^ column) * 16u;

    const uint32_t first_batch = range.x + ((end_all - 1u - range.x) / kBackBatch) * kBackBatch;
    // part p of entry e of a batch is staged by thread 4 e + p, its Gaussian and position looked up a batch
    // ahead. sorted_g was written by the TRAIN forward for every batch that it staged, and every entry below
    // part_end lies in one; threads past the batch repeat its first entry, with an empty box.
    const uint32_t e = threadIdx.x >> 2, p = threadIdx.x & 3u;
    uint32_t j = first_batch + e < part_end ? first_batch + e : first_batch;
    uint32_t g = sorted_g[j], position = values[j];
    for (int64_t bstart = first_batch; bstart >= (int64_t)range.x; bstart -= kBackBatch) {
        const int count = (int)min((uint32_t)kBackBatch, part_end - (uint32_t)bstart);
        {
            const bool in = (int)e < count;
            const float4* const first = p < 2 ? rec + 2 * (size_t)g + p : (p == 2 ? col + g : cov_coef + 2 * (size_t)g);
            const float4* const second = p == 3 ? cov_coef + 2 * (size_t)g + 1 : col + g;
            const float4 x0 = *first, x1 = *second;
            const uint2 box = cbox[g];
            if (p == 3) {
                if (!kMoments) {
                    sm.k[0][e] = x0;
                    sm.k[1][e] = x1;
                }
                if (in && j < end_all) touched[g] = 1;
            } else {
                float4 y = make_float4(x0.x, x0.y, -0.5f * x0.z, -0.5f * x0.w);
                if (p == 1) y = make_float4(-0.5f * x0.x, x0.y, x1.x, x1.y);
                if (p == 2)
                    y = make_float4(x0.z, __uint_as_float(in ? box.x : kEmptyBoxLo), __uint_as_float(in ? box.y : 0u),
                                    __uint_as_float(position));
                reinterpret_cast<float4*>(&sm.entry[e])[p] = y;
            }
        }
        const uint32_t g_combine = g;
        if (bstart > (int64_t)range.x) {
            j = (uint32_t)bstart - kBackBatch + e;
            g = sorted_g[j];
            position = values[j];
        }
        __syncthreads();
        // the entries of the batch that meet this quadrant before its pixels' last contribution
        uint64_t todo;
        {
            const BlendEntry& mine = sm.entry[lane];
            todo = wave_ballot((uint32_t)bstart + lane < wave_last &&
                               entry_meets_quadrant(mine, (pix.pxy & 0xffffu) & ~7u, (pix.pxy >> 16) & ~7u));
        }
        // `rows` rows of sums are taken, the last `fill` of them still rows of x
        int rows = 0, fill = 0;
        uint64_t used = 0;
        auto flush = [&]() {
            wave_lds_sync();
            // which side of the quadrant's centre each entry's mean lies on: the product's entries are the lowest
            // `fill` of `used`, the first of them highest. (Formed here by lane = entry: bits collected entry by
            // entry in scalar registers cost 6% of the kernel; a lane's place and sides held in a register gain
            // nothing, and spill others.)
            bool take0, take1;
            {
                uint32_t l = __lane_id();
                asm volatile("" : "+v"(l));
                const float2 mean = *reinterpret_cast<const float2*>(&sm.entry[l].a);
                const uint32_t at = (uint32_t)fill - 1u - __builtin_amdgcn_mbcnt_hi((uint32_t)(used >> 32),
                                                                                   __builtin_amdgcn_mbcnt_lo((uint32_t)used, 0u));
                const uint32_t side = (mean.x >= (float)((pix.pxy & 0xfff8u) + 4u) ? 1u : 0u) |
                                      (mean.y >= (float)((pix.pxy >> 16 & 0xfff8u) + 4u) ? 2u : 0u);
                if (__builtin_amdgcn_inverse_ballot_w64(used) && at < (uint32_t)fill) sm.side[wave][at] = side;
                wave_lds_sync();
                const uint2 both = *reinterpret_cast<const uint2*>(&sm.side[wave][2u * (l >> 4)]);
                const uint32_t sides = moment_sides(l & 15u);
                take0 = ((sides >> (both.x & 3u)) & 1u) != 0u;
                take1 = ((sides >> (both.y & 3u)) & 1u) != 0u;
            }
            // two chains of 32 pixels, not one of 64: half the rounding of the sums
            gsx_f32x4 part[2] = {};
            const char* const xb = reinterpret_cast<const char*>(x);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float4 a = *reinterpret_cast<const float4*>(xb + (read_at ^ (16u * t)));
                gsx_f32x4& to = part[t / 2];
                to = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, factor[kMoments ? 4 * t : 0], to, 0, 0, 0);
                to = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, factor[kMoments ? 4 * t + 1 : 0], to, 0, 0, 0);
                to = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, factor[kMoments ? 4 * t + 2 : 0], to, 0, 0, 0);
                to = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, factor[kMoments ? 4 * t + 3 : 0], to, 0, 0, 0);
            }
            const gsx_f32x4 acc = part[0] + part[1];
            // lane l holds rows 4 (l / 16) .. + 3 of column l % 16: h and w of two entries
            uint32_t l = __lane_id();
            asm volatile("" : "+v"(l));
            float* const to = &sm.sum[wave][(rows - fill + 2 * (int)(l >> 4)) * kGrad2d + (int)moment_place(l & 15u)];
            if (take0) to[0] = (l & 15u) < 13u ? acc.x : acc.y;
            if (take1) to[kGrad2d] = (l & 15u) < 13u ? acc.z : acc.w;
            wave_lds_sync();
            fill = 0;
        };
        // a pixel that needs no checkpoint of a bucket reads one all the same (the slot exists) and drops it
        auto checkpoint = [&](int bucket) {
            return ckpt[checkpoint_slot(range.x, tile, (uint32_t)bstart + (uint32_t)(bucket * kBucket)) * kBlendThreads +
                        threadIdx.x];
        };
        float next_t = 0.0f;
        if (todo != 0ull) next_t = checkpoint((63 - __builtin_clzll(todo)) / kBucket);
        while (todo != 0ull) {
            const int sb = (63 - __builtin_clzll(todo)) / kBucket;
            uint32_t bits = (uint32_t)(todo >> (sb * kBucket));
            const int hits = __builtin_popcount(bits);
            todo &= (1ull << (sb * kBucket)) - 1ull;
            const uint32_t j0 = (uint32_t)bstart + (uint32_t)(sb * kBucket);
            float tt = j0 < pix.last ? next_t : 0.0f;
            if (todo != 0ull) next_t = checkpoint((63 - __builtin_clzll(todo)) / kBucket);
            // forward replay of the bucket from its checkpoint (render.c:1476-1515), two entries' G at a time
            int k[kBucket];
            float tb[kBucket], gv[kBucket];
            uint64_t taken[kBucket];  // the pixels that take the entry
            auto replay = [&](int q, bool ok, float gq, float alpha) {
                ok = ok & ((uint32_t)bstart + (uint32_t)k[q] < pix.last);
                tb[q] = tt;
                taken[q] = wave_ballot(ok);
                gv[q] = ok ? gq : 0.0f;
                tt = ok ? tt * (1.0f - alpha) : tt;
            };
#pragma unroll
            for (int q = 0; q < kBucket; q += 2) {
                if (q >= hits) break;  // uniform
                k[q] = sb * kBucket + __builtin_ctz(bits);
                bits &= bits - 1u;
                float g0, a0, g1, a1;
                if (q + 1 < hits) {  // uniform
                    k[q + 1] = sb * kBucket + __builtin_ctz(bits);
                    bits &= bits - 1u;
                    const bool ok0 = blend_alpha<!kMoments>(sm.entry[k[q]], pix.fpx, pix.fpy, pix.pxy, sm.exp2, g0, a0);
                    const bool ok1 = blend_alpha<!kMoments>(sm.entry[k[q + 1]], pix.fpx, pix.fpy, pix.pxy, sm.exp2, g1, a1);
                    replay(q, ok0, g0, a0);
                    replay(q + 1, ok1, g1, a1);
                } else {
                    const bool ok0 = blend_alpha<!kMoments>(sm.entry[k[q]], pix.fpx, pix.fpy, pix.pxy, sm.exp2, g0, a0);
                    replay(q, ok0, g0, a0);
                }
            }
            // back to front over the bucket (render.c:1559-1666 per contribution)
#pragma unroll
            for (int q = kBucket - 1; q >= 0; --q) {
                if (q >= hits) continue;  // uniform
                if (taken[q] == 0ull) continue;  // uniform: no pixel of this wave
                used |= 1ull << k[q];
                const BlendEntry& en = sm.entry[k[q]];
                const float4 eb = en.b;
                const float cb = en.c.x;
                const float gval = gv[q];
                const float raw = eb.y * gval;
                const float alpha = fminf(kMaxFragmentAlpha, raw);
                const float t_before = tb[q];
                // A lane that does not contribute holds G = 0, hence alpha = 0: its weight w and its
                // opacity term below are (signed) zeros by arithmetic, and it leaves the suffix
                // unchanged, so no per-lane select on the contribution is needed (all values are
                // finite). alpha <= 0.999, so 1 - alpha lies in [0.001, 1]: the CPU's |1 - alpha| > 1e-6
                // guard always holds.
                const float w = alpha * t_before;
                float dalpha;
                if constexpr (kMoments) {
                    const float cd = __builtin_fmaf(eb.z, d0, __builtin_fmaf(eb.w, d1, cb * d2));
                    const float om = 1.0f - alpha;
                    const float y = __builtin_amdgcn_rcpf(om);
                    float quot = s0 * y;
                    quot = __builtin_fmaf(__builtin_fmaf(-om, quot, s0), y, quot);
                    dalpha = __builtin_fmaf(t_before, cd, -quot);
                    s0 = __builtin_fmaf(w, cd, s0);
                } else {
                    // a correctly rounded division as the CPU's: near-plane Gaussians' covariance
                    // gradients amplify even 1-ulp differences of this term (no scaling steps are
                    // needed, and a zero numerator gives a zero quotient)
                    dalpha = t_before * (eb.z * d0 + eb.w * d1 + cb * d2);
                    dalpha -= div_rn_normal(s0 * d0 + s1 * d1 + s2 * d2, 1.0f - alpha);
                    s0 += w * eb.z;
                    s1 += w * eb.w;
                    s2 += w * cb;
                }
                dalpha = raw < kMaxFragmentAlpha ? dalpha : 0.0f;
                const float h = dalpha * gval;
                if constexpr (kMoments) {
                    const uint32_t at = (uint32_t)fill * (2u * kWave * 4u) + ((4u * lane) ^ ((uint32_t)fill * 32u));
                    char* const xb = reinterpret_cast<char*>(x);
                    *reinterpret_cast<float*>(xb + at) = h;
                    *reinterpret_cast<float*>(xb + ((at ^ 16u) + kWave * 4u)) = w;
                    ++rows;
                    if (++fill == kMomentEntries) flush();
                } else {
                    const float4 ea = en.a;
                    const float4 k0 = sm.k[0][k[q]];
                    const float4 k1 = sm.k[1][k[q]];  // k1.z = 2 k0.y, k1.w = 2 k1.x
                    const float dx = pix.fpx - ea.x;
                    const float dy = pix.fpy - ea.y;
                    const float dpow = dalpha * eb.y * gval;
                    const float inv_a = -2.0f * ea.z, inv_b = -ea.w, inv_c = -2.0f * eb.x;
                    const float dia = dpow * (-0.5f * dx * dx);
                    const float dib = dpow * (-dx * dy);
                    const float dic = dpow * (-0.5f * dy * dy);
                    // the mean2d terms may fuse; the covariance terms keep the CPU's rounding
                    const float v[kGrad2d] = {dpow * __builtin_fmaf(inv_a, dx, inv_b * dy),
                                              dpow * __builtin_fmaf(inv_b, dx, inv_c * dy),
                                              dia * k0.x + dib * k0.y + dic * k0.z,
                                              dia * k1.z + dib * k0.w + dic * k1.w,
                                              dia * k0.z + dib * k1.x + dic * k1.y,
                                              w * d0,
                                              w * d1,
                                              w * d2,
                                              h};
                    float total8;
                    const float total = wave_sum9(v, total8);
                    float* const to = &sm.sum[wave][rows * kGrad2d];
                    if ((lane & 7u) == 0u) to[wave_sum9_index(lane)] = total;
                    if (lane == 63u) to[8] = total8;
                    ++rows;
                }
            }
        }
        if (kMoments && fill > 0) flush();
        if (lane == 0u) sm.used[wave] = used;
        __syncthreads();
        // four threads per entry add the waves' rows and write the partial
        if ((int)e < count) {
            const uint64_t mask = sm.used[p];
            const bool hit = ((mask >> e) & 1ull) != 0ull;
            const float* const from = &sm.sum[p][(hit ? __popcll((mask >> e) >> 1) : 0) * kGrad2d];
            float v[kGrad2d];
#pragma unroll
            for (int c = 0; c < kGrad2d; ++c) {
                const float f = from[c];
                v[c] = hit ? f : 0.0f;
            }
            const BlendEntry en = sm.entry[e];
            if constexpr (kMoments) {
                // moments about the entry's origin in the quadrant -> about the mean: the offset is u + ex, v + ey
                const float qcx = (float)(tx * kTile + 8 * (int)(p & 1u) + 4);
                const float qcy = (float)(ty * kTile + 8 * (int)(p >> 1) + 4);
                const float ex = (en.a.x >= qcx ? qcx + kMomentOrigin : qcx - kMomentOrigin) - en.a.x;
                const float ey = (en.a.y >= qcy ? qcy + kMomentOrigin : qcy - kMomentOrigin) - en.a.y;
                const float sx = __builtin_fmaf(ex, v[0], v[1]), sy = __builtin_fmaf(ey, v[0], v[2]);
                v[3] = __builtin_fmaf(ex, v[1] + sx, v[3]);
                v[4] = __builtin_fmaf(ex, v[2], __builtin_fmaf(ey, sx, v[4]));
                v[5] = __builtin_fmaf(ey, v[2] + sy, v[5]);
                v[1] = sx;
                v[2] = sy;
            }
#pragma unroll
            for (int c = 0; c < kGrad2d; ++c) v[c] = quad_sum(v[c]);
            if constexpr (kMoments) {
                const float4 k0 = cov_coef[2 * (size_t)g_combine];
                const float4 k1 = cov_coef[2 * (size_t)g_combine + 1];  // k1.z = 2 k0.y, k1.w = 2 k1.x
                const float op = en.b.y, inv_a = -2.0f * en.a.z, inv_b = -en.a.w, inv_c = -2.0f * en.b.x;
                const float dia = -0.5f * (op * v[3]), dib = -(op * v[4]), dic = -0.5f * (op * v[5]);
                const float h = v[0];
                v[0] = op * __builtin_fmaf(inv_a, v[1], inv_b * v[2]);
                v[1] = op * __builtin_fmaf(inv_b, v[1], inv_c * v[2]);
                v[2] = dia * k0.x + dib * k0.y + dic * k0.z;
                v[3] = dia * k1.z + dib * k0.w + dic * k1.w;
                v[4] = dia * k0.z + dib * k1.x + dic * k1.y;
                v[5] = v[6];
                v[6] = v[7];
                v[7] = v[8];
                v[8] = h;
            }
            const size_t pos = __float_as_uint(en.c.w);
            float4* const dst = reinterpret_cast<float4*>(instance_grad) + 2 * pos;
            if (p == 0) dst[0] = make_float4(v[0], v[1], v[2], v[3]);
            if (p == 1) dst[1] = make_float4(v[4], v[5], v[6], v[7]);
            if (p == 2) instance_grad_op[pos] = v[8];
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBlendThreads, 5) void blend_backward_kernel(
    const uint2* __restrict__ ranges, const uint32_t* __restrict__ values, const uint32_t* __restrict__ sorted_g,
    const float4* __restrict__ rec, const float4* __restrict__ col, const uint2* __restrict__ cbox,
    const float4* __restrict__ cov_coef, const float* __restrict__ ckpt, const uint32_t* __restrict__ tile_exact,
    CameraParams cam, const float* __restrict__ grad_rgb, const float* __restrict__ final_t,
    const uint32_t* __restrict__ last_contrib, float* __restrict__ instance_grad,
    float* __restrict__ instance_grad_op, uint32_t* __restrict__ tile_cut, uint8_t* __restrict__ touched,
    SinkZeroing sinks) {
    __shared__ BackwardShared sm;
    // every workgroup, the padding ones included, zeroes its slice of the gradient sinks first
    zero_sink_slice(sinks, blockIdx.x);
    const int tiles = cam.tiles_x * cam.tiles_y;
    const int tile = xcd_tile_index(blockIdx.x, tiles);
    if (tile >= tiles) return;
    if (threadIdx.x < GSX_EXPF_BLEND_TABLE_SIZE) sm.exp2[threadIdx.x] = gsx_expf_blend_entry(threadIdx.x);
    const int tx = tile % cam.tiles_x, ty = tile / cam.tiles_x;
    const int2 tp = tile_pixel_of_thread((int)threadIdx.x);
    const int px = tx * kTile + tp.x;
    const int py = ty * kTile + tp.y;
    const uint2 range = ranges[tile];
    const uint32_t exact = tile_exact[tile];
    BackwardPixel pix;
    pix.fpx = (float)px + 0.5f;
    pix.fpy = (float)py + 0.5f;
    pix.pxy = (uint32_t)px | ((uint32_t)py << 16);  // for in_box_packed
    pix.last = range.x;
    pix.t_final = pix.d0 = pix.d1 = pix.d2 = 0.0f;
    if (px < cam.width && py < cam.height) {
        const size_t at = (size_t)py * (size_t)cam.width + (size_t)px;
        const size_t plane = (size_t)cam.width * (size_t)cam.height;
        pix.t_final = final_t[at];
        pix.last = last_contrib[at];
        pix.d0 = grad_rgb[at];
        pix.d1 = grad_rgb[plane + at];
        pix.d2 = grad_rgb[2 * plane + at];
    }
    if (threadIdx.x == 0) sm.max_last = range.x;
    const uint32_t wave_last = wave_max_u32(pix.last);
    __syncthreads();
    if (__lane_id() == 0) atomicMax(&sm.max_last, wave_last);
    __syncthreads();
    const uint32_t end_all = sm.max_last;
    // Entries from zero_from on (whole buckets past the last entry any pixel of the tile reaches)
    // get no partial: their gradient is zero. Positions ascend along the tile's run, so the run's
    // entries with a partial are exactly those whose position is below tile_cut[tile], the
    // position of the first entry without one (UINT32_MAX: all have one); the reduction adds +0
    // for the others instead of reading them.
    const uint32_t zero_from =
        end_all <= range.x ? range.x : range.x + ((end_all - range.x + kBucket - 1) / kBucket) * kBucket;
    if (threadIdx.x == 0) tile_cut[tile] = zero_from < range.y ? values[zero_from] : UINT32_MAX;
    if (end_all <= range.x) return;  // uniform
    const uint32_t part_end = min(zero_from, range.y);  // entries below it get a partial
    if (__builtin_amdgcn_readfirstlane((int)exact) != 0)
        blend_backward_walk<false>(sm, pix, range, tile, tx, ty, wave_last, end_all, part_end, values, sorted_g, rec, col,
                                   cbox, cov_coef, ckpt, cam, instance_grad, instance_grad_op, touched);
    else
        blend_backward_walk<true>(sm, pix, range, tile, tx, ty, wave_last, end_all, part_end, values, sorted_g, rec, col,
                                  cbox, cov_coef, ckpt, cam, instance_grad, instance_grad_op, touched);
}

// grad2d[g] = sum of the partials over the emission positions [offset[r], offset[r+1]) of g, r its
// depth rank; every Gaussian's sum is taken in a fixed order, so the result is deterministic.
// Position p has a partial iff p < tile_cut[instance_tile[p]] (the blend backward's cut of p's
// tile); the others count as +0, read from neither array. A Gaussian that no tile reached
// (touched[g] == 0) has no partial at all: its sums are not formed, and projection_backward_kernel
// writes its zero gradients without reading them.
//  * runs of at most kLaneRun instances (reduce_short_block): the 64 runs of a wave's ranks are
//    one contiguous span; the wave stages it through its own LDS piece by piece with coalesced
//    loads, jumping over long runs, and each lane sums its run in position order into grad2d;
//  * longer runs (in depth order the near, large Gaussians sit side by side, and the largest
//    cover nearly every tile) are cut into at most kLongChunks chunks of `chunk` positions, and
//    one wave sums a chunk (DPP tree, reduce_run_chunk). reduce_long_block takes chunk 0 of every
//    long run (long_list, in rank order, written by emit_block) and chunks 1.. of the runs longer
//    than one chunk (multi_list, in rank order), the entries dealt round-robin over the
//    waves: the near, large Gaussians are neighbours in depth order, and a wave of their own
//    would serialise them. A run of one chunk is done; the others leave each chunk's sums in
//    place at its first position, and projection_backward_kernel adds them in chunk order.
// All of it runs in one launch (reduce_instance_grads_kernel).
constexpr uint32_t kShortPiece = 256;  // instances per LDS piece and wave (9 KB)
constexpr uint32_t kLongChunks = 16;

__device__ inline void add_record(float acc[kGrad2d], float4 a, float4 b, float op) {
    acc[0] += a.x;
    acc[1] += a.y;
    acc[2] += a.z;
    acc[3] += a.w;
    acc[4] += b.x;
    acc[5] += b.y;
    acc[6] += b.z;
    acc[7] += b.w;
    acc[8] += op;
}

// Position p's partial (three loads), or +0 where the blend backward wrote none.
struct InstancePartial {
    float4 a, b;
    float op;
};
template <typename TileT>
__device__ inline InstancePartial load_partial(const float4* __restrict__ rec4, const float* __restrict__ instance_grad_op,
                                               const TileT* __restrict__ instance_tile,
                                               const uint32_t* __restrict__ tile_cut, uint32_t p) {
    InstancePartial v;
    const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (p < tile_cut[instance_tile[p]]) {
        v.a = rec4[2 * (size_t)p];
        v.b = rec4[2 * (size_t)p + 1];
        v.op = instance_grad_op[p];
    } else {
        v.a = z;
        v.b = z;
        v.op = 0.0f;
    }
    return v;
}

// Chunk k of the long run [b, e) of Gaussian g, summed by the whole wave (b, e, g, k wave-uniform).
// A run of one chunk gets its sums in grad2d, a longer one its chunk's sums at the chunk's first
// position.
template <typename TileT>
__device__ inline void reduce_run_chunk(uint32_t b, uint32_t e, uint32_t g, uint32_t k, uint32_t chunk,
                                        float* __restrict__ instance_grad, float* __restrict__ instance_grad_op,
                                        const TileT* __restrict__ instance_tile,
                                        const uint32_t* __restrict__ tile_cut, float* __restrict__ grad2d) {
    const uint32_t lane = __lane_id();
    const float4* rec4 = reinterpret_cast<const float4*>(instance_grad);
    const uint32_t cb = b + k * chunk;
    const uint32_t ce = min(e, cb + chunk);
    float acc[kGrad2d];
#pragma unroll
    for (int c = 0; c < kGrad2d; ++c) acc[c] = 0.0f;
    for (uint32_t p0 = cb; p0 < ce; p0 += 4 * kWave) {
        // all loads of the round are in flight together: none sits under a branch (lanes past
        // the chunk re-read its last position and add nothing)
        InstancePartial v[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t p = min(p0 + u * kWave + lane, ce - 1);
            v[u] = load_partial(rec4, instance_grad_op, instance_tile, tile_cut, p);
        }
        // lanes past the chunk add -0, the identity of + (an unconditional use keeps the loads
        // ahead of the adds)
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const bool in = p0 + u * kWave + lane < ce;
            const float4 z = make_float4(-0.0f, -0.0f, -0.0f, -0.0f);
            add_record(acc, in ? v[u].a : z, in ? v[u].b : z, in ? v[u].op : -0.0f);
        }
    }
#pragma unroll
    for (int c = 0; c < kGrad2d; ++c) acc[c] = wave_reduce_sum(acc[c]);
    if (lane != 0) return;
    if (e - b <= chunk) {
#pragma unroll
        for (int c = 0; c < kGrad2d; ++c) grad2d[(size_t)g * kGrad2d + c] = acc[c];
        return;
    }
    // every lane's loads of the chunk fed the sums above, so overwriting position cb is safe
    float4* dst = reinterpret_cast<float4*>(instance_grad) + 2 * (size_t)cb;
    dst[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
    dst[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
    instance_grad_op[cb] = acc[8];
}

// Chunk k of the long runs of the wave's lanes (run [b, e) of Gaussian g where `live`): the
// touched ones are summed by the wave one after another (the untouched ones have no sums: the
// projection backward skips their Gaussians).
template <typename TileT>
__device__ inline void reduce_wave_long_runs(bool live, uint32_t b, uint32_t e, uint32_t g, uint32_t k,
                                             uint32_t chunk, float* __restrict__ instance_grad,
                                             float* __restrict__ instance_grad_op,
                                             const TileT* __restrict__ instance_tile,
                                             const uint32_t* __restrict__ tile_cut,
                                             const uint8_t* __restrict__ touched, float* __restrict__ grad2d) {
    const bool hit = live && touched[g] != 0;
    for (uint64_t todo = __ballot(hit); todo != 0ull; todo &= todo - 1ull) {
        const int src = __builtin_ctzll(todo);
        reduce_run_chunk((uint32_t)__builtin_amdgcn_readlane((int)b, src),
                         (uint32_t)__builtin_amdgcn_readlane((int)e, src),
                         (uint32_t)__builtin_amdgcn_readlane((int)g, src), k, chunk, instance_grad, instance_grad_op,
                         instance_tile, tile_cut, grad2d);
    }
}

template <typename TileT>
__device__ inline void reduce_short_block(uint32_t blk, int64_t n, const uint32_t* __restrict__ depth_count,
                                          const uint32_t* __restrict__ offsets,
                                          const uint32_t* __restrict__ rank_gaussian, uint32_t chunk,
                                          float* __restrict__ instance_grad, float* __restrict__ instance_grad_op,
                                          const TileT* __restrict__ instance_tile,
                                          const uint32_t* __restrict__ tile_cut, const uint8_t* __restrict__ touched,
                                          float* __restrict__ grad2d, float4 (*s_rec)[2 * kShortPiece],
                                          float (*s_op)[kShortPiece]) {
    const uint32_t lane = __lane_id(), wave = threadIdx.x / kWave;
    n = min(n, (int64_t)*depth_count);  // ranks of visible Gaussians
    const int64_t r = (int64_t)blk * blockDim.x + threadIdx.x;
    const int64_t r_first = r - lane;  // first rank of this wave (waves wholly past n find no work)
    const bool valid = r < n;
    uint32_t b = 0, e = 0, g = 0;
    if (valid) {
        b = offsets[r];
        e = offsets[r + 1];
        g = rank_gaussian[r];
    }
    const bool mine = valid && e - b <= kLaneRun;
    const bool has = mine && e > b && touched[g] != 0;
    const uint32_t span_end = offsets[min(r_first + (int64_t)kWave, n)];
    const float4* rec4 = reinterpret_cast<const float4*>(instance_grad);
    float4* sr = s_rec[wave];
    float* so = s_op[wave];
    float acc[kGrad2d];
#pragma unroll
    for (int c = 0; c < kGrad2d; ++c) acc[c] = 0.0f;
    for (uint32_t cur = offsets[min(r_first, n)];;) {
        // the piece starts at the lowest position a short run of the wave still needs
        const uint32_t p0 = wave_min_u32(has && e > cur ? max(b, cur) : UINT32_MAX);
        if (p0 == UINT32_MAX) break;  // uniform
        const uint32_t p1 = min(p0 + kShortPiece, span_end);
        wave_lds_sync();  // the previous piece has been read
        // every load of the piece is issued before the first store waits on one: the loads are
        // not under a branch (lanes past the piece re-read its last position, p1 > p0)
        constexpr int kPieceRounds = (int)(kShortPiece / kWave);
        const uint32_t len = p1 - p0;
        InstancePartial v[kPieceRounds];
#pragma unroll
        for (int u = 0; u < kPieceRounds; ++u) {
            const uint32_t q = min(lane + (uint32_t)u * kWave, len - 1);
            v[u] = load_partial(rec4, instance_grad_op, instance_tile, tile_cut, p0 + q);
        }
        // (unconditional stores: lanes past the piece write its last position's own values again)
#pragma unroll
        for (int u = 0; u < kPieceRounds; ++u) {
            const uint32_t q = min(lane + (uint32_t)u * kWave, len - 1);
            sr[2 * q] = v[u].a;
            sr[2 * q + 1] = v[u].b;
            so[q] = v[u].op;
        }
        wave_lds_sync();
        if (has) {
            const uint32_t lo = max(b, p0), hi = min(e, p1);
            for (uint32_t p = lo; p < hi; ++p) add_record(acc, sr[2 * (p - p0)], sr[2 * (p - p0) + 1], so[p - p0]);
        }
        cur = p1;
    }
    if (has) {
#pragma unroll
        for (int c = 0; c < kGrad2d; ++c) grad2d[(size_t)g * kGrad2d + c] = acc[c];
    }
}

// Chunk k of the runs on `list`, by the gx * 4 waves of the workgroups of column k: lane l of
// wave w takes entries w + W (l + 64 j), j = 0, 1, ... (W waves), so neighbouring entries go to
// different waves.
template <typename TileT>
__device__ inline void reduce_long_block(uint32_t x, uint32_t k, uint32_t gx, const uint32_t* __restrict__ list,
                                         const uint32_t* __restrict__ list_count,
                                         const uint32_t* __restrict__ offsets,
                                         const uint32_t* __restrict__ rank_gaussian, uint32_t chunk,
                                         float* __restrict__ instance_grad, float* __restrict__ instance_grad_op,
                                         const TileT* __restrict__ instance_tile,
                                         const uint32_t* __restrict__ tile_cut, const uint8_t* __restrict__ touched,
                                         float* __restrict__ grad2d) {
    const uint32_t count = *list_count;
    const uint32_t waves = gx * (blockDim.x / kWave);
    const uint32_t w = x * (blockDim.x / kWave) + threadIdx.x / kWave;
    for (uint32_t j = 0; w + waves * j * kWave < count; ++j) {
        const uint32_t i = w + waves * (j * kWave + __lane_id());
        uint32_t b = 0, e = 0, g = 0;
        bool live = false;
        if (i < count) {
            const uint32_t r = list[i];
            b = offsets[r];
            e = offsets[r + 1];
            g = rank_gaussian[r];
            live = b + k * chunk < e;
        }
        reduce_wave_long_runs(live, b, e, g, k, chunk, instance_grad, instance_grad_op, instance_tile, tile_cut,
                              touched, grad2d);
    }
}

// Both reductions in one launch: workgroups [0, gx0) take chunk 0 of the long runs, the next
// gx * (kLongChunks - 1) chunks 1.. of the runs longer than one chunk (x = index % gx, chunk
// k = 1 + index / gx), the rest the short runs of the ranks (256 each).
template <typename TileT>
__global__ __launch_bounds__(256) void reduce_instance_grads_kernel(
    int64_t n, const uint32_t* __restrict__ depth_count, const uint32_t* __restrict__ offsets,
    const uint32_t* __restrict__ rank_gaussian, const uint32_t* __restrict__ long_list,
    const uint32_t* __restrict__ long_count, const uint32_t* __restrict__ multi_list,
    const uint32_t* __restrict__ multi_count, uint32_t gx0, uint32_t gx, uint32_t chunk,
    float* __restrict__ instance_grad,
    float* __restrict__ instance_grad_op, const TileT* __restrict__ instance_tile,
    const uint32_t* __restrict__ tile_cut, const uint8_t* __restrict__ touched, float* __restrict__ grad2d) {
    __shared__ float4 s_rec[kWavesPerBlock][2 * kShortPiece];
    __shared__ float s_op[kWavesPerBlock][kShortPiece];
    if (blockIdx.x < gx0) {
        reduce_long_block(blockIdx.x, 0, gx0, long_list, long_count, offsets, rank_gaussian, chunk, instance_grad,
                          instance_grad_op, instance_tile, tile_cut, touched, grad2d);
        return;
    }
    const uint32_t long_blocks = gx0 + gx * (kLongChunks - 1);
    if (blockIdx.x < long_blocks) {
        const uint32_t bi = blockIdx.x - gx0;
        reduce_long_block(bi % gx, 1 + bi / gx, gx, multi_list, multi_count, offsets, rank_gaussian, chunk,
                          instance_grad, instance_grad_op, instance_tile, tile_cut, touched, grad2d);
        return;
    }
    reduce_short_block(blockIdx.x - long_blocks, n, depth_count, offsets, rank_gaussian, chunk, instance_grad,
                       instance_grad_op, instance_tile, tile_cut, touched, grad2d, s_rec, s_op);
}

__device__ inline void add3(float* p, float x, float y, float z) {
    p[0] += x;
    p[1] += y;
    p[2] += z;
}

// render.c:714-728
__device__ inline void add_dir(float ddir[3], const float dcol[3], const float* coeff, float bx, float by, float bz) {
    const float s = dcol[0] * coeff[0] + dcol[1] * coeff[1] + dcol[2] * coeff[2];
    ddir[0] += s * bx;
    ddir[1] += s * by;
    ddir[2] += s * bz;
}

// ---------------------------------------------------------------------------------------------
// Projection backward: render.c:1667-1969 per Gaussian, from the accumulated screen-space
// gradients. Sinks are overwritten (the CPU zeroes them first, render.c:1537-1550); invisible
// Gaussians get zeros.
// ---------------------------------------------------------------------------------------------
// Instantiated per SH degree (0-3): the higher degrees' gradient arrays then exist only where
// they are used (degree 0 needs 45 fewer live registers).
// Stores the rows of a kWidth-float field for the workgroup's Gaussians [first, first + count)
// (thread t holds row first + t) as whole 16-byte vectors: the rows go through LDS, then
// consecutive threads store consecutive vectors of the block's contiguous span (a row of 3, 9, 15
// or 21 floats would otherwise take that many 4-byte stores at a stride of the row). dst must be
// 16-byte aligned; the span's last floats past its last whole vector are stored one by one. Every
// thread of the workgroup calls it.
template <int kWidth>
__device__ inline void block_store_rows(float* __restrict__ dst, int64_t first, int count, const float (&row)[kWidth],
                                        float* s_stage) {
    __syncthreads();  // the previous field's stores have read s_stage
#pragma unroll
    for (int k = 0; k < kWidth; ++k) s_stage[threadIdx.x * kWidth + k] = row[k];
    __syncthreads();
    const int total = count * kWidth;
    const int vecs = total / 4;
    float* base = dst + first * kWidth;
    for (int i = threadIdx.x; i < vecs; i += blockDim.x)
        reinterpret_cast<float4*>(base)[i] = reinterpret_cast<const float4*>(s_stage)[i];
    for (int i = vecs * 4 + (int)threadIdx.x; i < total; i += blockDim.x) base[i] = s_stage[i];
}

template <int kShDegree>
__global__ __launch_bounds__(256) void projection_backward_kernel(
    int64_t n, const float* __restrict__ mean3d, const float* __restrict__ rotation,
    const float* __restrict__ logscale, const float* __restrict__ opacity, const float* __restrict__ sh0,
    const float* __restrict__ sh1, const float* __restrict__ sh2, const float* __restrict__ sh3,
    CameraParams cam, const float* __restrict__ grad2d, const uint32_t* __restrict__ tile_count,
    const uint32_t* __restrict__ gaussian_rank, const uint32_t* __restrict__ offsets, uint32_t chunk,
    const float* __restrict__ instance_grad, const float* __restrict__ instance_grad_op,
    const uint8_t* __restrict__ touched, float* __restrict__ g_mean3d,
    float* __restrict__ g_rotation, float* __restrict__ g_logscale, float* __restrict__ g_opacity,
    float* __restrict__ g_sh0, float* __restrict__ g_sh1, float* __restrict__ g_sh2, float* __restrict__ g_sh3,
    int vector_stores) {
    constexpr int sh_degree = kShDegree;
    constexpr int kStageWidth = kShDegree >= 3 ? 21 : (kShDegree == 2 ? 15 : (kShDegree == 1 ? 9 : 3));
    // the exp table in LDS: its lookups wait on LDS, not on a global load each
    __shared__ uint64_t s_exp[GSX_EXP2_TABLE_SIZE];
    // the block's rows of one gradient field on their way to whole-vector stores
    __shared__ __align__(16) float s_stage[256 * kStageWidth];
    const int64_t first = (int64_t)blockIdx.x * blockDim.x;
    const int64_t gi = first + threadIdx.x;
    const bool valid = gi < n;  // every thread stays for the block's staged stores
    // a Gaussian that no tile's backward reached (touched[gi] == 0: invisible ones included) has
    // a +0 screen-space gradient and so zero parameter gradients, which the blend backward has
    // already stored in every sink (zero_sink_slice): a block with no reached Gaussian is done
    const bool reached = valid && touched[gi] != 0;
    if (!__syncthreads_or(reached ? 1 : 0)) return;
    // A reached Gaussian was emitted, so preprocess_one found it visible in the forward; of its
    // projection the backward uses only the camera-space mean, the view direction and the clamped
    // colour, recomputed here by the same operations (not the covariance, conic and box, whose
    // dependent chain would set the time of a block holding one of the few reached Gaussians).
    // Every input is loaded before the exp table's barrier, so their latency overlaps it.
    ProjectedView p{};
    p.visible = reached;
    uint32_t run_length = 0;
    uint32_t rank = 0;
    float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float ls[3] = {0.0f, 0.0f, 0.0f};
    if (reached) {
        // the rank is used only by a run of several chunks; read here, coalesced, it takes a load
        // round off that chain
        run_length = tile_count[gi];
        rank = gaussian_rank[gi];
        q = reinterpret_cast<const float4*>(rotation)[gi];
        ls[0] = logscale[gi * 3 + 0];
        ls[1] = logscale[gi * 3 + 1];
        ls[2] = logscale[gi * 3 + 2];
        p = project_view(gi, mean3d, sh0, sh1, sh2, sh3, sh_degree, cam);
    }
    if (threadIdx.x < GSX_EXP2_TABLE_SIZE) s_exp[threadIdx.x] = gsx_exp2_table_entry(threadIdx.x);
    __syncthreads();
    const uint64_t* exp_tab = s_exp;
    __builtin_assume(exp_tab != nullptr);  // no run-time choice of table per lookup
    float gm[3] = {0.0f, 0.0f, 0.0f};
    float gr[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    float gl[3] = {0.0f, 0.0f, 0.0f};
    float gop = 0.0f;
    float gs0[3] = {0.0f, 0.0f, 0.0f};
    float gs1[9];
    float gs2[15];
    float gs3[21];
#pragma unroll
    for (int i = 0; i < 9; ++i) gs1[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < 15; ++i) gs2[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < 21; ++i) gs3[i] = 0.0f;
    float a2[kGrad2d];
#pragma unroll
    for (int c = 0; c < kGrad2d; ++c) a2[c] = 0.0f;
    const bool multi = p.visible && run_length > chunk;
    if (p.visible && !multi) {
#pragma unroll
        for (int c = 0; c < kGrad2d; ++c) a2[c] = grad2d[(size_t)gi * kGrad2d + c];
    }
    {
        // A run of several chunks: the sums of its chunks (reduce_long_block), added in chunk
        // order from +0. The wave loads one such run's chunk sums at once, lane k taking chunk k,
        // and every lane adds them in lane order (the owner keeps the result): one load round per
        // run instead of one per chunk, whose serial latency would set the kernel's time.
        const int lane = (int)(threadIdx.x & (kWave - 1));
        uint32_t rb = 0, re = 0;
        if (multi) {
            rb = offsets[rank];
            re = offsets[rank + 1];
        }
        for (uint64_t runs = wave_ballot(multi); runs != 0; runs &= runs - 1) {
            const int src = __builtin_ctzll(runs);
            const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)rb, src);
            const uint32_t len = (uint32_t)__builtin_amdgcn_readlane((int)re, src) - b;
            float v[kGrad2d];
#pragma unroll
            for (int c = 0; c < kGrad2d; ++c) v[c] = 0.0f;
            if ((uint32_t)lane * chunk < len) {
                const uint32_t cb = b + (uint32_t)lane * chunk;
                const float4* rec4 = reinterpret_cast<const float4*>(instance_grad) + 2 * (size_t)cb;
                const float4 x = rec4[0], y = rec4[1];
                v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
                v[4] = y.x, v[5] = y.y, v[6] = y.z, v[7] = y.w;
                v[8] = instance_grad_op[cb];
            }
            float acc[kGrad2d];
#pragma unroll
            for (int c = 0; c < kGrad2d; ++c) acc[c] = 0.0f;
            for (int k = 0; k < kWave && (uint32_t)k * chunk < len; ++k) {
#pragma unroll
                for (int c = 0; c < kGrad2d; ++c)
                    acc[c] += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[c]), k));
            }
            if (lane == src) {
#pragma unroll
                for (int c = 0; c < kGrad2d; ++c) a2[c] = acc[c];
            }
        }
    }
    if (p.visible) {
        const float dmx = a2[0], dmy = a2[1];
        const float dca = a2[2], dcb = a2[3], dcc = a2[4];
        const float dcx = a2[5], dcy = a2[6], dcz = a2[7];
        const float dop = a2[8];
        const Mat3 w = camera_rotation(cam);
        const Mat3 rot = rotation_from_xyzw(q.x, q.y, q.z, q.w);
        const float sx = gsx_expf_table(ls[0], exp_tab), sy = gsx_expf_table(ls[1], exp_tab),
                    sz = gsx_expf_table(ls[2], exp_tab);
        // R S, and the covariance (R S)(R S)^T by cov3d_from's operations
        Mat3 srot = rot;
#pragma unroll
        for (int row = 0; row < 3; ++row) {
            srot.m[row][0] *= sx;
            srot.m[row][1] *= sy;
            srot.m[row][2] *= sz;
        }
        const Mat3 cov3d = mat3_mul_t(srot, srot);
        const float zc = p.zc, xc = p.xc, yc = p.yc;
        const float j00 = cam.fx / zc;
        const float j02 = -cam.fx * xc / (zc * zc);
        const float j11 = cam.fy / zc;
        const float j12 = -cam.fy * yc / (zc * zc);
        // colour: render.c:1667-1828
        {
            const float dcol[3] = {dcx * (p.color[0] > 0.0f ? 1.0f : 0.0f), dcy * (p.color[1] > 0.0f ? 1.0f : 0.0f),
                                   dcz * (p.color[2] > 0.0f ? 1.0f : 0.0f)};
            float ddir[3] = {0.0f, 0.0f, 0.0f};
            const float x = p.dir[0], y = p.dir[1], z = p.dir[2];
            const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, yz = y * z, xz = x * z;
            gs0[0] = kShC0 * dcol[0];
            gs0[1] = kShC0 * dcol[1];
            gs0[2] = kShC0 * dcol[2];
            if (sh_degree >= 1) {
                const float* c1 = sh1 + gi * 9;
                float s;
                s = -kShC1 * y;
                add3(gs1 + 0, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                s = kShC1 * z;
                add3(gs1 + 3, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                s = -kShC1 * x;
                add3(gs1 + 6, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c1 + 0, 0.0f, -kShC1, 0.0f);
                add_dir(ddir, dcol, c1 + 3, 0.0f, 0.0f, kShC1);
                add_dir(ddir, dcol, c1 + 6, -kShC1, 0.0f, 0.0f);
            }
            if (sh_degree >= 2) {
                const float* c2 = sh2 + gi * 15;
                float s;
                s = kShC2[0] * xy;
                add3(gs2 + 0, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c2 + 0, kShC2[0] * y, kShC2[0] * x, 0.0f);
                s = kShC2[1] * yz;
                add3(gs2 + 3, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c2 + 3, 0.0f, kShC2[1] * z, kShC2[1] * y);
                s = kShC2[2] * (2.0f * zz - xx - yy);
                add3(gs2 + 6, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c2 + 6, -2.0f * kShC2[2] * x, -2.0f * kShC2[2] * y, 4.0f * kShC2[2] * z);
                s = kShC2[3] * xz;
                add3(gs2 + 9, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c2 + 9, kShC2[3] * z, 0.0f, kShC2[3] * x);
                s = kShC2[4] * (xx - yy);
                add3(gs2 + 12, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c2 + 12, 2.0f * kShC2[4] * x, -2.0f * kShC2[4] * y, 0.0f);
            }
            if (sh_degree >= 3) {
                const float* c3 = sh3 + gi * 21;
                float s;
                s = kShC3[0] * y * (3.0f * xx - yy);
                add3(gs3 + 0, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c3 + 0, 6.0f * kShC3[0] * x * y, 3.0f * kShC3[0] * (xx - yy), 0.0f);
                s = kShC3[1] * xy * z;
                add3(gs3 + 3, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c3 + 3, kShC3[1] * y * z, kShC3[1] * x * z, kShC3[1] * xy);
                s = kShC3[2] * y * (4.0f * zz - xx - yy);
                add3(gs3 + 6, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c3 + 6, -2.0f * kShC3[2] * x * y, kShC3[2] * (4.0f * zz - xx - 3.0f * yy),
                        8.0f * kShC3[2] * y * z);
                s = kShC3[3] * z * (2.0f * zz - 3.0f * xx - 3.0f * yy);
                add3(gs3 + 9, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c3 + 9, -6.0f * kShC3[3] * x * z, -6.0f * kShC3[3] * y * z,
                        kShC3[3] * (6.0f * zz - 3.0f * xx - 3.0f * yy));
                s = kShC3[4] * x * (4.0f * zz - xx - yy);
                add3(gs3 + 12, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c3 + 12, kShC3[4] * (4.0f * zz - 3.0f * xx - yy), -2.0f * kShC3[4] * x * y,
                        8.0f * kShC3[4] * x * z);
                s = kShC3[5] * z * (xx - yy);
                add3(gs3 + 15, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c3 + 15, 2.0f * kShC3[5] * x * z, -2.0f * kShC3[5] * y * z, kShC3[5] * (xx - yy));
                s = kShC3[6] * x * (xx - 3.0f * yy);
                add3(gs3 + 18, dcol[0] * s, dcol[1] * s, dcol[2] * s);
                add_dir(ddir, dcol, c3 + 18, 3.0f * kShC3[6] * (xx - yy), -6.0f * kShC3[6] * x * y, 0.0f);
            }
            if (sh_degree >= 1) {
                const float vx = mean3d[gi * 3 + 0] - cam.centre[0];
                const float vy = mean3d[gi * 3 + 1] - cam.centre[1];
                const float vz = mean3d[gi * 3 + 2] - cam.centre[2];
                const float vn = sqrtf(vx * vx + vy * vy + vz * vz);
                if (vn > 0.0f) {
                    const float dd = ddir[0] * x + ddir[1] * y + ddir[2] * z;
                    const float s = 1.0f / vn;
                    gm[0] += (ddir[0] - x * dd) * s;
                    gm[1] += (ddir[1] - y * dd) * s;
                    gm[2] += (ddir[2] - z * dd) * s;
                }
            }
        }
        // opacity: render.c:1830
        {
            const float sg = sigmoid_render(opacity[gi], exp_tab);
            gop += dop * (sg * (1.0f - sg));
        }
        // mean through the projection: render.c:1832-1845
        {
            const float inv_z = 1.0f / zc;
            const float inv_z2 = inv_z * inv_z;
            const float dmc0 = dmx * cam.fx * inv_z;
            const float dmc1 = dmy * cam.fy * inv_z;
            const float dmc2 = dmx * (-cam.fx * xc * inv_z2) + dmy * (-cam.fy * yc * inv_z2);
            gm[0] += w.m[0][0] * dmc0 + w.m[1][0] * dmc1 + w.m[2][0] * dmc2;
            gm[1] += w.m[0][1] * dmc0 + w.m[1][1] * dmc1 + w.m[2][1] * dmc2;
            gm[2] += w.m[0][2] * dmc0 + w.m[1][2] * dmc1 + w.m[2][2] * dmc2;
        }
        // covariance to scale and rotation: render.c:1847-1937
        {
            float mm[2][3];
#pragma unroll
            for (int col = 0; col < 3; ++col) {
                mm[0][col] = j00 * w.m[0][col] + j02 * w.m[2][col];
                mm[1][col] = j11 * w.m[1][col] + j12 * w.m[2][col];
            }
            Mat3 dcov3;
#pragma unroll
            for (int row = 0; row < 3; ++row)
#pragma unroll
                for (int col = 0; col < 3; ++col)
                    dcov3.m[row][col] = mm[0][row] * (dca * mm[0][col] + 0.5f * dcb * mm[1][col]) +
                                        mm[1][row] * (0.5f * dcb * mm[0][col] + dcc * mm[1][col]);
            Mat3 dsum;
#pragma unroll
            for (int row = 0; row < 3; ++row)
#pragma unroll
                for (int col = 0; col < 3; ++col) dsum.m[row][col] = dcov3.m[row][col] + dcov3.m[col][row];
            const Mat3 drs = mat3_mul(dsum, srot);
            gl[0] = (drs.m[0][0] * rot.m[0][0] + drs.m[1][0] * rot.m[1][0] + drs.m[2][0] * rot.m[2][0]) * sx;
            gl[1] = (drs.m[0][1] * rot.m[0][1] + drs.m[1][1] * rot.m[1][1] + drs.m[2][1] * rot.m[2][1]) * sy;
            gl[2] = (drs.m[0][2] * rot.m[0][2] + drs.m[1][2] * rot.m[1][2] + drs.m[2][2] * rot.m[2][2]) * sz;
            Mat3 dr;
#pragma unroll
            for (int row = 0; row < 3; ++row) {
                dr.m[row][0] = drs.m[row][0] * sx;
                dr.m[row][1] = drs.m[row][1] * sy;
                dr.m[row][2] = drs.m[row][2] * sz;
            }
            float nx, ny, nz, nw;
            if (quat_normalize(q.x, q.y, q.z, q.w, nx, ny, nz, nw)) {
                const float inv_norm = 1.0f / sqrtf(q.x * q.x + q.y * q.y + q.z * q.z + q.w * q.w);
                float dqw = 0.0f, dqx = 0.0f, dqy = 0.0f, dqz = 0.0f;
                dqw += dr.m[0][1] * (-2.0f * nz);
                dqw += dr.m[0][2] * (2.0f * ny);
                dqw += dr.m[1][0] * (2.0f * nz);
                dqw += dr.m[1][2] * (-2.0f * nx);
                dqw += dr.m[2][0] * (-2.0f * ny);
                dqw += dr.m[2][1] * (2.0f * nx);
                dqx += dr.m[0][1] * (2.0f * ny);
                dqx += dr.m[0][2] * (2.0f * nz);
                dqx += dr.m[1][0] * (2.0f * ny);
                dqx += dr.m[1][1] * (-4.0f * nx);
                dqx += dr.m[1][2] * (-2.0f * nw);
                dqx += dr.m[2][0] * (2.0f * nz);
                dqx += dr.m[2][1] * (2.0f * nw);
                dqx += dr.m[2][2] * (-4.0f * nx);
                dqy += dr.m[0][0] * (-4.0f * ny);
                dqy += dr.m[0][1] * (2.0f * nx);
                dqy += dr.m[0][2] * (2.0f * nw);
                dqy += dr.m[1][0] * (2.0f * nx);
                dqy += dr.m[1][2] * (2.0f * nz);
                dqy += dr.m[2][0] * (-2.0f * nw);
                dqy += dr.m[2][1] * (2.0f * nz);
                dqy += dr.m[2][2] * (-4.0f * ny);
                dqz += dr.m[0][0] * (-4.0f * nz);
                dqz += dr.m[0][1] * (-2.0f * nw);
                dqz += dr.m[0][2] * (2.0f * nx);
                dqz += dr.m[1][0] * (2.0f * nw);
                dqz += dr.m[1][1] * (-4.0f * nz);
                dqz += dr.m[1][2] * (2.0f * ny);
                dqz += dr.m[2][0] * (2.0f * nx);
                dqz += dr.m[2][1] * (2.0f * ny);
                const float dot = nx * dqx + ny * dqy + nz * dqz + nw * dqw;
                gr[0] = (dqx - nx * dot) * inv_norm;
                gr[1] = (dqy - ny * dot) * inv_norm;
                gr[2] = (dqz - nz * dot) * inv_norm;
                gr[3] = (dqw - nw * dot) * inv_norm;
            }
        }
        // Jacobian's dependence on the camera-space mean: render.c:1939-1969
        {
            const Mat3 cov_cam = mat3_mul_t(mat3_mul(w, cov3d), w);
            const float inv_z = 1.0f / zc;
            const float inv_z2 = inv_z * inv_z;
            const float inv_z3 = inv_z2 * inv_z;
            float dj[2][3];
#pragma unroll
            for (int col = 0; col < 3; ++col) {
                dj[0][col] = 2.0f * dca * (j00 * cov_cam.m[0][col] + j02 * cov_cam.m[2][col]) +
                             dcb * (j11 * cov_cam.m[1][col] + j12 * cov_cam.m[2][col]);
                dj[1][col] = dcb * (j00 * cov_cam.m[0][col] + j02 * cov_cam.m[2][col]) +
                             2.0f * dcc * (j11 * cov_cam.m[1][col] + j12 * cov_cam.m[2][col]);
            }
            const float m0 = dj[0][2] * (-cam.fx * inv_z2);
            const float m1 = dj[1][2] * (-cam.fy * inv_z2);
            const float m2 = dj[0][0] * (-cam.fx * inv_z2) + dj[0][2] * (2.0f * cam.fx * xc * inv_z3) +
                             dj[1][1] * (-cam.fy * inv_z2) + dj[1][2] * (2.0f * cam.fy * yc * inv_z3);
            gm[0] += w.m[0][0] * m0 + w.m[1][0] * m1 + w.m[2][0] * m2;
            gm[1] += w.m[0][1] * m0 + w.m[1][1] * m1 + w.m[2][1] * m2;
            gm[2] += w.m[0][2] * m0 + w.m[1][2] * m1 + w.m[2][2] * m2;
        }
    }
    if (valid) {
        // rows of 16 and 4 bytes: consecutive lanes already store consecutive addresses
        reinterpret_cast<float4*>(g_rotation)[gi] = make_float4(gr[0], gr[1], gr[2], gr[3]);
        g_opacity[gi] = gop;
    }
    if (vector_stores) {  // uniform: every 3-float (and SH) sink is 16-byte aligned
        const int count = (int)min((int64_t)blockDim.x, n - first);
        block_store_rows<3>(g_mean3d, first, count, gm, s_stage);
        block_store_rows<3>(g_logscale, first, count, gl, s_stage);
        block_store_rows<3>(g_sh0, first, count, gs0, s_stage);
        if (sh_degree >= 1) block_store_rows<9>(g_sh1, first, count, gs1, s_stage);
        if (sh_degree >= 2) block_store_rows<15>(g_sh2, first, count, gs2, s_stage);
        if (sh_degree >= 3) block_store_rows<21>(g_sh3, first, count, gs3, s_stage);
        return;
    }
    if (!valid) return;
    g_mean3d[gi * 3 + 0] = gm[0];
    g_mean3d[gi * 3 + 1] = gm[1];
    g_mean3d[gi * 3 + 2] = gm[2];
    g_logscale[gi * 3 + 0] = gl[0];
    g_logscale[gi * 3 + 1] = gl[1];
    g_logscale[gi * 3 + 2] = gl[2];
    g_sh0[gi * 3 + 0] = gs0[0];
    g_sh0[gi * 3 + 1] = gs0[1];
    g_sh0[gi * 3 + 2] = gs0[2];
    if (sh_degree >= 1)
        for (int i = 0; i < 9; ++i) g_sh1[gi * 9 + i] = gs1[i];
    if (sh_degree >= 2)
        for (int i = 0; i < 15; ++i) g_sh2[gi * 15 + i] = gs2[i];
    if (sh_degree >= 3)
        for (int i = 0; i < 21; ++i) g_sh3[gi * 21 + i] = gs3[i];
}

}  // namespace gsx_amd
