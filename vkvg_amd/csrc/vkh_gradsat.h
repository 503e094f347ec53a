// Gradients that are constant over a tile. The fragment math (shaders/vkvg_main.frag:83-144) maps a
// pixel to a coordinate x and mixes the colour stops by smoothstep; where x <= the first stop every mix
// factor is 0 and the colour is the first stop's, where x >= the last stop the last factor is 1 and the
// colour is the last stop's, bit for bit (finite colours, increasing stops). A tile that lies wholly on
// one side needs no per-pixel evaluation. The test below is conservative: it leaves a margin for the
// rounding of the per-pixel float evaluation and for its own, so "outside" is never claimed for a pixel
// whose evaluated x is inside. Shared by the kernels and the CPU test (tests/test_gradsat.py).
//
// Linear: x is affine in the pixel position, so its extremes over a tile are at the corners. The
// evaluation ((py - m px - bb) / sqrt(1 + m m)) / l rounds by at most 5 * 2^-24 (1 + |m| + |bb|) before
// the two divisions and the test's own three products by as much again; the margin is 64 * 2^-24 of
// that, plus 2^-18 (1 + |stop|) for the divisions.
// Radial: x = (|p - c0| - r0) / (t - r0) with t the distance from the focus c0 to the circle (c1, r1)
// along the ray through p. A point outside the circle by a share d of r1 has x - 1 >= d / 2 (it is at
// least d r1 beyond the circle along the ray, and t <= 2 r1). With the focus at most r1 / 2 off centre
// and t - r0 >= r1 / 4, the evaluation's error near x = 1 is below 20 e / r1 + 2^-19, where
// e = 2^-23 (1 + |c0|) bounds the rounding of a coordinate; d = 2^-8 + 128 e / r1 leaves twice that.
// Inside r0 only |p - c0| against r0 matters. Other radial gradients are never taken.
#ifndef VKH_GRADSAT_H
#define VKH_GRADSAT_H

#include <math.h>
#include <stdint.h>

#include "vkvg_hip.h"

#ifdef __HIPCC__
#define VKH_GS __host__ __device__ __forceinline__
#else
#define VKH_GS static inline
#endif

enum { VKH_GS_NONE = 0, VKH_GS_LINEAR = 1, VKH_GS_RADIAL = 2 };
typedef struct {
    uint32_t type;
    float s[6]; // linear: x = s0 X + s1 Y + s2 at pixel centre (X, Y), first colour where x <= s3, last
                // where x >= s4; radial: c1 (s0, s1), outside where the squared distance is >= s2,
                // c0 (s3, s4), inside r0 where it is <= s5
} vkh_grad_sat;

// g's test on a target of W x H pixels
VKH_GS vkh_grad_sat vkh_grad_sat_of(const vkh_gradient *g, float W, float H) {
    vkh_grad_sat r;
    r.type = VKH_GS_NONE;
    for (int k = 0; k < 6; k++)
        r.s[k] = 0.f;
    const uint32_t n = g->count;
    if (n < 2 || n > 16)
        return r;
    int inc = 1; // increasing stops
    double sum = 0.0;
    for (uint32_t i = 0; i < n; i++) {
        for (int c = 0; c < 4; c++)
            sum += fabs((double)g->colors[i][c]);
        sum += fabs((double)g->stops[i]);
        if (i && !(g->stops[i] > g->stops[i - 1]))
            inc = 0;
    }
    if (!inc || !(sum < 1e6))
        return r;
    const double first = g->stops[0], last = g->stops[n - 1];
    if (g->type == 2) {
        // the same float terms as the per-pixel evaluation uses
        const float p0x = g->cp[0][0] / W, p0y = g->cp[0][1] / H, p1x = g->cp[0][2] / W, p1y = g->cp[0][3] / H;
        const float dx = p1x - p0x, dy = p1y - p0y;
        const float l = sqrtf(dx * dx + dy * dy), ux = dx / l, uy = dy / l;
        double a, b, c, e;
        if (uy == 0) {
            const double q = (ux < 0 ? -1.0 : 1.0) / (double)l;
            a = q / (double)W;
            b = 0.0;
            c = -q * (double)p0x;
            e = (1.0 + fabs((double)p0x)) / (double)l;
        } else {
            const float m = -ux / uy, bb = p0y - m * p0x;
            const double q = (uy < 0 ? -1.0 : 1.0) / ((double)sqrtf(1 + m * m) * (double)l);
            a = -q * (double)m / (double)W;
            b = q / (double)H;
            c = -q * (double)bb;
            e = (1.0 + fabs((double)m) + fabs((double)bb)) * fabs(q);
        }
        if (!(l > 1e-12f) || !(e < 1e6) || !(fabs(a) + fabs(b) + fabs(c) < 1e6))
            return r;
        const double u = 1.0 / 262144.0; // 2^-18
        r.s[0] = (float)a;
        r.s[1] = (float)b;
        r.s[2] = (float)c;
        r.s[3] = (float)(first - u * (e + 1.0 + fabs(first)));
        r.s[4] = (float)(last + u * (e + 1.0 + fabs(last)));
        r.type = VKH_GS_LINEAR;
        return r;
    }
    const double c0x = g->cp[0][0] / W, c0y = g->cp[0][1] / H, c1x = g->cp[1][0] / W, c1y = g->cp[1][1] / H;
    const double r0 = g->cp[0][2] / W, r1 = g->cp[1][2] / W;
    const double off = sqrt((c0x - c1x) * (c0x - c1x) + (c0y - c1y) * (c0y - c1y));
    if (!(r1 > 1e-6 && r1 < 1e6 && r0 >= 0.0 && fabs(c0x) + fabs(c0y) < 1e6) || !(off <= 0.5 * r1) ||
        !(r1 - off - r0 >= 0.25 * r1) || !(first >= 0.0 && last <= 1.0))
        return r;
    const double e = (1.0 + fabs(c0x) + fabs(c0y)) / 8388608.0, d = 1.0 / 256.0 + 128.0 * e / r1;
    if (!(d < 0.25))
        return r;
    const double ro = r1 * (1.0 + d), ri = r0 * (1.0 - 1.0 / 256.0) - 4.0 * e;
    r.s[0] = (float)c1x;
    r.s[1] = (float)c1y;
    r.s[2] = (float)(ro * ro);
    r.s[3] = (float)c0x;
    r.s[4] = (float)c0y;
    r.s[5] = ri > 0.0 ? (float)(ri * ri) : -1.f;
    r.type = VKH_GS_RADIAL;
    return r;
}

// For the pixels with centres in [x0, x1] x [y0, y1] (pixels) of a W x H target: 1 where every one has
// the first stop's colour, 2 where every one has the last stop's, else 0
VKH_GS int vkh_grad_sat_tile(uint32_t type, const float *s, float x0, float y0, float x1, float y1, float W, float H) {
    if (type == VKH_GS_LINEAR) {
        const float lo = s[2] + fminf(s[0] * x0, s[0] * x1) + fminf(s[1] * y0, s[1] * y1);
        const float hi = s[2] + fmaxf(s[0] * x0, s[0] * x1) + fmaxf(s[1] * y0, s[1] * y1);
        return hi <= s[3] ? 1 : lo >= s[4] ? 2 : 0;
    }
    if (type == VKH_GS_RADIAL) {
        const float u0 = x0 / W, u1 = x1 / W, v0 = y0 / H, v1 = y1 / H;
        const float dx = fmaxf(fmaxf(u0 - s[0], s[0] - u1), 0.f), dy = fmaxf(fmaxf(v0 - s[1], s[1] - v1), 0.f);
        const float fx = fmaxf(fabsf(u0 - s[3]), fabsf(u1 - s[3])), fy = fmaxf(fabsf(v0 - s[4]), fabsf(v1 - s[4]));
        return fx * fx + fy * fy <= s[5] ? 1 : dx * dx + dy * dy >= s[2] ? 2 : 0;
    }
    return 0;
}

#endif
