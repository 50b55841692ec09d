/*
 * tile_cull.h - the conservative tile test of key emission, shared by the gfx950 kernels and the
 * CPU restatement in oracle/ (both compile it with -ffp-contract=off and correctly rounded
 * division and square root, so they take the same decision bit for bit).
 *
 * The gsx CPU backend visits every pixel of a Gaussian's 3-sigma box (gsx/src/gsx-cpu/render.c:
 * 1042-1079) and skips the pixel when power < -4.5 or opacity * expf(power) < 1/255, with
 * power = -0.5 * (inv_a dx^2 + 2 inv_b dx dy + inv_c dy^2) in float. A tile of the box whose
 * pixels all fail those tests contributes nothing to the image or to any gradient, so its
 * (tile, Gaussian) instance can be left out of the sort. With
 *   thr    = max(-4.5, ln(1/255) - ln(opacity)) - 1e-3     (per Gaussian; the pixel is skipped
 *            when power < thr + 1e-3, and the 1e-3 dwarfs every float rounding in between),
 *   q_cut  = -2 * thr,
 * a pixel that contributes has its quadratic form q = -2 power at most q_cut. The test keeps,
 * for each tile row of the box, the tiles that hold a pixel column where the set {q <= Q}
 * (Q = q_cut plus an allowance for rounding) meets the row's band of pixel rows: one contiguous
 * run of tiles per row, from a closed form (gsx_tile_band_columns). Every dropped tile's pixels
 * therefore fail a cut.
 */
#ifndef GSX_AMD_TILE_CULL_H
#define GSX_AMD_TILE_CULL_H

#include "gsx_math.h"

/* min / max / |x| / clamp as the IEEE operations (one instruction each, or a free source
 * modifier on the GPU). The test's operands are finite, where these equal the compare-and-select
 * forms; a signed zero can differ, and a zero of either sign leaves every quantity below
 * unchanged. lo <= hi in every clamp. */
#if defined(__HIPCC__)
GSX_HD float gsx_cull_minf(float a, float b) { return __builtin_fminf(a, b); }
GSX_HD float gsx_cull_maxf(float a, float b) { return __builtin_fmaxf(a, b); }
GSX_HD float gsx_cull_absf(float a) { return __builtin_fabsf(a); }
#else
GSX_HD float gsx_cull_minf(float a, float b) { return fminf(a, b); }
GSX_HD float gsx_cull_maxf(float a, float b) { return fmaxf(a, b); }
GSX_HD float gsx_cull_absf(float a) { return fabsf(a); }
#endif
/* Correctly rounded square root of x >= 2^-80 (or +inf). On the GPU without the scaling and the class
 * test that sqrtf spends on smaller arguments (half its 18 instructions): the hardware root s is
 * within one unit in the last place, and x <= s (s - ulp) or x > s (s + ulp) tell the neighbour
 * that is nearer (Tuckerman's test). */
#if defined(__HIP_DEVICE_COMPILE__)
GSX_HD float gsx_cull_sqrtf(float x)
{
    const float s = __builtin_amdgcn_sqrtf(x);
    const float below = gsx_f32_from_bits(gsx_f32_bits(s) - 1u), above = gsx_f32_from_bits(gsx_f32_bits(s) + 1u);
    const float r = GSX_FMAF(-below, s, x) <= 0.0f ? below : s;
    return GSX_FMAF(-above, s, x) > 0.0f ? above : r;
}
#else
GSX_HD float gsx_cull_sqrtf(float x) { return sqrtf(x); }
#endif
GSX_HD float gsx_cull_clampf(float v, float lo, float hi) { return gsx_cull_minf(gsx_cull_maxf(v, lo), hi); }

/* Natural logarithm of a positive normal float from IEEE operations only, so the CPU and the
 * GPU agree bit for bit: x = m 2^e with m in [sqrt(1/2), sqrt(2)), ln m = 2 atanh(s),
 * s = (m - 1) / (m + 1), |s| < 0.172, series to s^11 (relative error below 1e-7). */
GSX_HD float gsx_cull_logf(float x)
{
    uint32_t u = gsx_f32_bits(x);
    int e = (int)((u >> 23) & 0xffu) - 127;
    float m = gsx_f32_from_bits((u & 0x007fffffu) | 0x3f800000u);
    float s, s2, t;

    if(m > 1.41421356f) {
        m = m * 0.5f;
        e += 1;
    }
    s = (m - 1.0f) / (m + 1.0f);
    s2 = s * s;
    t = 1.0f / 11.0f;
    t = t * s2 + 1.0f / 9.0f;
    t = t * s2 + 1.0f / 7.0f;
    t = t * s2 + 1.0f / 5.0f;
    t = t * s2 + 1.0f / 3.0f;
    t = t * s2 + 1.0f;
    return 2.0f * s * t + (float)e * 0.693147180559945f;
}

/* q_cut of the Gaussian with activated opacity `opacity` (> 1/255 for every visible one). */
GSX_HD float gsx_tile_qcut(float opacity)
{
    float thr = -5.54126354f - gsx_cull_logf(opacity); /* ln(1/255) - ln(opacity) */

    if(thr < -4.5f) {
        thr = -4.5f;
    }
    return -2.0f * (thr - 1e-3f);
}

/* Per-Gaussian constants of the row-span test. Every kept tile of a tile row of the box is one
 * contiguous run: the pixel centres of the row's band (its pixel rows within the box) that may
 * receive a contribution lie inside the convex set {q(u, v) <= Q}, whose part over the band
 * projects onto one interval of columns. With q = A u^2 + 2 B u v + C v^2 (A, C > 0,
 * det = A C - B^2 > 0) and D(v) = A Q - det v^2, the set's right boundary at height v is
 * u+(v) = (sqrt(D(v)) - B v) / A, a concave function of v largest at vr = -B sqrt(Q / (det C))
 * (the ellipse's rightmost point), so over the band [v0, v1] it is largest at clamp(vr, v0, v1);
 * by symmetry (q(u, v) = q(-u, -v)) the left boundary is least at -clamp(vr, -v1, -v0) mirrored.
 * The band misses the set exactly when D < 0 at that point.
 *   Q    = q_cut + 1e-5 S + 1e-3, S = A X^2 + 2 |B| X Y + C Y^2 with X, Y the largest |offsets| of
 *          the box's pixel centres from the mean: the kernels' power evaluation at a pixel of the
 *          box is within 4 eps S of the exact form (eps = 2^-24), 1e-5 S covers it 40 times over;
 *   aqs  = A Q (1 + 2^-14 + kappa 2^-19), kappa = A C / det: the rounding of D(v) for |v| within
 *          the set is below (3 + 2 kappa) eps A Q, and the factor adds at least 8 times that, so
 *          the computed D is never below the exact one and sqrt(D) never short;
 *   the remaining roundings (of -B v + sqrt(D), of the product with 1 / A) are below
 *          3 eps (sqrt(kappa) + 1) sqrt(Q / A), and the factor widens the span by at least
 *          2^-15 sqrt(Q / A), 8 times more.
 * D is held above 2^-80, which only widens the span.
 * A pixel column x may be contributed to when its centre offset fl(fl(x + 0.5) - mx), the value the
 * kernels evaluate, lies in [u-, u+]. Kept are the columns from ceil(mx - 0.5 - m + u-) to
 * floor(mx - 0.5 + m + u+), m = 2^-6 + 2^-21 |mx|: the roundings of the offset, of mx - 0.5 -/+ m and of
 * the sum are below 2^-22 |mx| + 2^-7 for columns below 2^16. (An exact check of the column on each
 * side instead kept 0.1% fewer tiles and cost 30 of a row's 200 vector instructions.)
 * A Gaussian whose form is not
 * positive definite, whose kappa exceeds 2^16 (det then carries more than 1% rounding) or whose
 * mean lies beyond 2^21 pixels, or any non-finite constant, keeps every column of its box:
 * aqs = +inf, det = vr = B = 0, ra = 1 and a mean of 0 make every band span the box without a branch. */
typedef struct gsx_tile_span {
    float ml, mh; /* mx - 0.5 less and plus the margin m */
    float my;     /* mean2d y */
    float b;      /* inv_b */
    float ra;     /* 1 / inv_a */
    float det;    /* inv_a inv_c - inv_b^2 */
    float vr;     /* v of the rightmost point of the set */
    float aqs;    /* inv_a Q with the rounding allowance */
} gsx_tile_span;

/* The part of a Gaussian's constants that its row spans and its column spans share: Q, det, A C and
 * the rounding allowance of aqs. */
typedef struct gsx_tile_form {
    float q;     /* Q */
    float ac;    /* inv_a inv_c */
    float det;   /* inv_a inv_c - inv_b^2 */
    float slack; /* 2^-14 + kappa 2^-19 */
} gsx_tile_form;

GSX_HD gsx_tile_form gsx_tile_form_make(float mx, float my, float inv_a, float inv_b, float inv_c, float opacity,
    int x0, int x1, int y0, int y1)
{
    gsx_tile_form f;
    const float A = inv_a, B = inv_b, C = inv_c;
    const float dx0 = ((float)x0 + 0.5f) - mx, dx1 = ((float)x1 + 0.5f) - mx;
    const float dy0 = ((float)y0 + 0.5f) - my, dy1 = ((float)y1 + 0.5f) - my;
    const float X = gsx_cull_maxf(gsx_cull_absf(dx0), gsx_cull_absf(dx1));
    const float Y = gsx_cull_maxf(gsx_cull_absf(dy0), gsx_cull_absf(dy1));
    const float S = gsx_cull_absf(A) * X * X + 2.0f * gsx_cull_absf(B) * X * Y + gsx_cull_absf(C) * Y * Y;

    f.q = gsx_tile_qcut(opacity) + (1e-5f * S + 1e-3f);
    f.ac = A * C;
    f.det = f.ac - B * B;
    f.slack = 6.103515625e-05f + (f.ac / f.det) * 1.9073486328125e-06f;
    return f;
}

/* Constants of the Gaussian whose form is f = gsx_tile_form_make(...). With x and y (and inv_a and
 * inv_c) exchanged they are those of its column spans: f is the same up to the rounding of S, which
 * the allowance covers 40 times over. */
GSX_HD gsx_tile_span gsx_tile_span_of_form(const gsx_tile_form *f, float mx, float my, float inv_a, float inv_b,
    float inv_c)
{
    gsx_tile_span k;
    const float A = inv_a, B = inv_b, C = inv_c;

    const float margin = 0.015625f + 4.76837158203125e-07f * gsx_cull_absf(mx);

    k.ml = (mx - 0.5f) - margin;
    k.mh = (mx - 0.5f) + margin;
    k.my = my;
    k.b = B;
    k.ra = 1.0f / A;
    k.det = f->det;
    k.vr = -B * sqrtf(f->q / (f->det * C));
    k.aqs = (A * f->q) * (1.0f + f->slack);
    /* the comparisons are false for NaN, which therefore keeps every column too */
    if(!(A > 0.0f && C > 0.0f && f->det > 0.0f && f->det * 65536.0f >= f->ac && gsx_cull_absf(mx) < 2097152.0f &&
           gsx_cull_absf(my) < 2097152.0f && gsx_cull_absf(k.vr) <= 3.0e38f && k.aqs <= 3.0e38f && k.ra <= 3.0e38f)) {
        k.ml = 0.0f;
        k.mh = 0.0f;
        k.my = 0.0f;
        k.b = 0.0f;
        k.ra = 1.0f;
        k.det = 0.0f;
        k.vr = 0.0f;
        k.aqs = __builtin_inff();
    }
    return k;
}

/* Constants of the Gaussian with conic (inv_a, inv_b, inv_c), activated opacity `opacity` and
 * inclusive pixel box [x0, x1] x [y0, y1]. */
GSX_HD gsx_tile_span gsx_tile_span_make(float mx, float my, float inv_a, float inv_b, float inv_c, float opacity,
    int x0, int x1, int y0, int y1)
{
    const gsx_tile_form f = gsx_tile_form_make(mx, my, inv_a, inv_b, inv_c, opacity, x0, x1, y0, y1);

    return gsx_tile_span_of_form(&f, mx, my, inv_a, inv_b, inv_c);
}

/* The pixel columns [*xa, *xb] of the box [x0, x1] whose centres may receive a contribution in
 * the band of pixel rows [py0, py1] (within the box); *xa > *xb when none. */
GSX_HD void gsx_tile_band_columns(const gsx_tile_span *k, int x0, int x1, int py0, int py1, int *xa, int *xb)
{
    const float v0 = ((float)py0 + 0.5f) - k->my, v1 = ((float)py1 + 0.5f) - k->my;
    const float vh = gsx_cull_clampf(k->vr, v0, v1);
    const float vl = gsx_cull_clampf(k->vr, -v1, -v0);
    const float dh = k->aqs - (k->det * vh) * vh;
    const float dl = k->aqs - (k->det * vl) * vl;
    const float uh = (gsx_cull_sqrtf(gsx_cull_maxf(dh, 8.27180613e-25f)) - k->b * vh) * k->ra;
    const float ul = -((gsx_cull_sqrtf(gsx_cull_maxf(dl, 8.27180613e-25f)) - k->b * vl) * k->ra);

    if(dh < 0.0f) { /* the band misses the set */
        *xa = 1;
        *xb = 0;
        return;
    }
    *xb = (int)floorf(gsx_cull_maxf(gsx_cull_minf(k->mh + uh, (float)x1), (float)x0 - 1.0f));
    *xa = (int)ceilf(gsx_cull_minf(gsx_cull_maxf(k->ml + ul, (float)x0), (float)x1 + 1.0f));
}

/* The pixel rectangle [*xa, *xb] x [*ya, *yb] of the box [x0, x1] x [y0, y1] that holds every
 * pixel centre which may receive a contribution from the Gaussian: the columns from the row-span
 * test with the whole box as one band, the rows from the same test with the roles of x and y
 * exchanged (q(u, v) is the same form with A and C swapped, and the rounding allowances are
 * symmetric in u and v). Empty when *xa > *xb or *ya > *yb. The blend kernels test pixels
 * against this rectangle instead of the 3-sigma box: a pixel outside it fails the CPU's cuts.
 * *k receives the row-span constants (gsx_tile_span_make's), which the tile lists need as well. */
GSX_HD void gsx_contribution_box_and_span(float mx, float my, float inv_a, float inv_b, float inv_c, float opacity, int x0,
    int x1, int y0, int y1, gsx_tile_span *k, int *xa, int *xb, int *ya, int *yb)
{
    const gsx_tile_form f = gsx_tile_form_make(mx, my, inv_a, inv_b, inv_c, opacity, x0, x1, y0, y1);
    const gsx_tile_span ky = gsx_tile_span_of_form(&f, my, mx, inv_c, inv_b, inv_a);

    *k = gsx_tile_span_of_form(&f, mx, my, inv_a, inv_b, inv_c);
    gsx_tile_band_columns(k, x0, x1, y0, y1, xa, xb);
    gsx_tile_band_columns(&ky, y0, y1, x0, x1, ya, yb);
}

GSX_HD void gsx_contribution_box(float mx, float my, float inv_a, float inv_b, float inv_c, float opacity, int x0,
    int x1, int y0, int y1, int *xa, int *xb, int *ya, int *yb)
{
    gsx_tile_span k;

    gsx_contribution_box_and_span(mx, my, inv_a, inv_b, inv_c, opacity, x0, x1, y0, y1, &k, xa, xb, ya, yb);
}

/* Nonzero when some pixel centre of the inclusive pixel rectangle [px0, px1] x [py0, py1] may
 * receive a contribution from the Gaussian (the rectangle taken as its box). */
GSX_HD int gsx_tile_may_contribute(float mx, float my, float inv_a, float inv_b, float inv_c, float opacity, int px0,
    int px1, int py0, int py1)
{
    const gsx_tile_span k = gsx_tile_span_make(mx, my, inv_a, inv_b, inv_c, opacity, px0, px1, py0, py1);
    int xa, xb;

    gsx_tile_band_columns(&k, px0, px1, py0, py1, &xa, &xb);
    return xa <= xb;
}

#endif /* GSX_AMD_TILE_CULL_H */
