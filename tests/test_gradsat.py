"""Tiles that vkvg_amd/csrc/vkh_gradsat.h claims to be constant under a gradient: the fragment math of
shaders/vkvg_main.frag:83-144, restated in C with its float operations, gives every pixel of a claimed
tile exactly the claimed stop's colour. Random linear and radial gradients (degenerate directions, off
centre and out of range foci, tiny and huge radii, unsorted stops) on targets of 1 to 8192 pixels, with
tiles drawn around the places where the claim begins; compiled from the kernels' header with gcc."""
import os
import subprocess
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROG = r"""
#include <stdio.h>
#include <string.h>
#include "vkh_gradsat.h"
static uint64_t rs = 88172645463325252ull;
static double u(void) { rs ^= rs << 13; rs ^= rs >> 7; rs ^= rs << 17; return (double)(rs >> 11) / 9007199254740992.0; }
static double lu(double a, double b) { return exp(log(a) + (log(b) - log(a)) * u()); }
static float cl(float x) { return fminf(fmaxf(x, 0.f), 1.f); }
static void colour(const vkh_gradient *g, float W, float H, float X, float Y, float *col) {
    const float px = X / W, py = Y / H;
    float x;
    if (g->type == 2) {
        float p0x = g->cp[0][0] / W, p0y = g->cp[0][1] / H, p1x = g->cp[0][2] / W, p1y = g->cp[0][3] / H;
        float dx = p1x - p0x, dy = p1y - p0y, l = sqrtf(dx * dx + dy * dy), ux = dx / l, uy = dy / l;
        if (uy == 0) {
            x = (px - p0x) / l;
            if (ux < 0) x = -x;
        } else {
            float m = -ux / uy, bb = p0y - m * p0x;
            x = ((py - m * px - bb) / sqrtf(1 + m * m)) / l;
            if (uy < 0) x = -x;
        }
    } else {
        float c0x = g->cp[0][0] / W, c0y = g->cp[0][1] / H, c1x = g->cp[1][0] / W, c1y = g->cp[1][1] / H;
        float r0 = g->cp[0][2] / W, r1 = g->cp[1][2] / W, dx = c0x - c1x, dy = c0y - c1y;
        float cc = (dx * dx + dy * dy) - r1 * r1, len = 1.f;
        float rx = px - c0x, ry = py - c0y, rl = sqrtf(rx * rx + ry * ry), ex = rx / rl, ey = ry / rl;
        float a = ex * ex + ey * ey, b = 2.f * (ex * dx + ey * dy), disc = b * b - 4.f * a * cc;
        if (disc >= 0.f) {
            float t = (-b + sqrtf(fabsf(disc))) / (2.f * a);
            float qx = (c0x + ex * t) - c0x, qy = (c0y + ey * t) - c0y;
            len = sqrtf(qx * qx + qy * qy) - r0;
        }
        x = (sqrtf(rx * rx + ry * ry) - r0) / len;
    }
    for (int c = 0; c < 4; c++) col[c] = g->colors[0][c];
    for (uint32_t i = 1; i < (g->count > 2 ? g->count : 2); i++) {
        float t = cl((x - g->stops[i - 1]) / (g->stops[i] - g->stops[i - 1]));
        t = t * t * (3.f - 2.f * t);
        for (int c = 0; c < 4; c++) col[c] = col[c] * (1.f - t) + g->colors[i][c] * t;
    }
}
int main(void) {
    long claims[2][3] = {{0}}, bad = 0, pixels = 0;
    for (int it = 0; it < 40000; it++) {
        vkh_gradient g;
        memset(&g, 0, sizeof g);
        const float W = (float)(int)lu(1, 8192), H = (float)(int)lu(1, 8192);
        g.type = u() < 0.5 ? 2 : 3;
        g.count = 2 + (uint32_t)(u() * 5);
        double s = 0;
        for (uint32_t i = 0; i < g.count; i++) { g.stops[i] = (float)s; s += u() < 0.02 ? 0 : u() / g.count; }
        if (u() < 0.6) g.stops[g.count - 1] = 1.f;
        if (u() < 0.05) g.stops[0] = (float)(u() - 0.5);
        for (uint32_t i = 0; i < g.count; i++) for (int c = 0; c < 4; c++) g.colors[i][c] = (float)u();
        const double sc = lu(1, 2.0 * (W > H ? W : H));
        const double cx = W * (u() * 1.4 - 0.2), cy = H * (u() * 1.4 - 0.2);
        if (g.type == 2) {
            const double k = u();
            g.cp[0][0] = (float)cx; g.cp[0][1] = (float)cy;
            g.cp[0][2] = (float)(cx + (k < 0.1 ? 0 : sc * (u() * 2 - 1)));
            g.cp[0][3] = (float)(cy + (k > 0.8 ? 0 : k > 0.7 ? 1e-4 : sc * (u() * 2 - 1)));
        } else {
            const double r1 = sc + 1, off = r1 * u() * (u() < 0.7 ? 0.45 : 1.2), an = 6.2831853 * u();
            g.cp[0][0] = (float)(cx + off * cos(an)); g.cp[0][1] = (float)(cy + off * sin(an));
            g.cp[0][2] = (float)(u() < 0.3 ? 0 : r1 * u() * 0.6);
            g.cp[1][0] = (float)cx; g.cp[1][1] = (float)cy; g.cp[1][2] = (float)r1;
        }
        const vkh_grad_sat t = vkh_grad_sat_of(&g, W, H);
        for (int k = 0; k < 24; k++) {
            const int T = 8 << (int)(u() * 3);
            int X, Y;
            if (k & 1) { // near the gradient's own edge
                const double an = 6.2831853 * u(), q = sc * (1 + (u() - 0.5) * 0.1);
                X = (int)(cx + q * cos(an)) - (int)(u() * T); Y = (int)(cy + q * sin(an)) - (int)(u() * T);
            } else { X = (int)(u() * W); Y = (int)(u() * H); }
            if (X < 0) X = 0;
            if (Y < 0) Y = 0;
            if (X >= W || Y >= H) continue;
            const int X1 = X + T < W ? X + T : (int)W, Y1 = Y + T < H ? Y + T : (int)H;
            const int e = vkh_grad_sat_tile(t.type, t.s, X + 0.5f, Y + 0.5f, X1 - 0.5f, Y1 - 0.5f, W, H);
            claims[g.type - 2][e]++;
            if (!e) continue;
            const float *want = e == 1 ? g.colors[0] : g.colors[g.count - 1];
            for (int y = Y; y < Y1; y++) for (int x = X; x < X1; x++) {
                float c[4];
                colour(&g, W, H, x + 0.5f, y + 0.5f, c);
                pixels++;
                if (c[0] != want[0] || c[1] != want[1] || c[2] != want[2] || c[3] != want[3]) bad++;
            }
        }
    }
    printf("%ld %ld %ld %ld %ld %ld %ld %ld\n", bad, pixels, claims[0][0], claims[0][1], claims[0][2], claims[1][0],
           claims[1][1], claims[1][2]);
    return 0;
}
"""


def test_claimed_tiles_have_the_stops_colour():
    with tempfile.TemporaryDirectory() as t:
        src, exe = os.path.join(t, "g.c"), os.path.join(t, "g")
        open(src, "w").write(PROG)
        subprocess.run(["gcc", "-O2", "-std=c11", "-ffp-contract=off", "-I", os.path.join(ROOT, "vkvg_amd", "csrc"),
                        "-I", os.path.join(ROOT, "include"), "-o", exe, src, "-lm"], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()
    bad, pixels, lin0, lin_lo, lin_hi, rad0, rad_lo, rad_hi = map(int, out)
    assert bad == 0, out
    # both kinds claim both ends, and neither claims everything
    assert min(lin0, lin_lo, lin_hi, rad0, rad_lo, rad_hi) > 1000 and pixels > 10_000_000, out
