// Differentiable renderer of the vkvg HIP backend: analytic area coverage into FP32 RGBA and its
// backward pass (C ABI of include/vkvg_diff.h). Semantics are stated in that header.
//
// Pipeline per forward call:
//   k_dflatten      one thread per polyline point: Bernstein sample of its cubic
//   k_dnormals      one thread per point: unit left normal of the segment leaving it (strokes)
//   k_dedges        one thread per point: the fill edge, or the stroke's rectangle + 2 bevel
//                   triangles (10 edges)
//   k_dpaths        one workgroup per path: bbox of its edges in tiles and how many list entries the
//                   tile rows take; k_dalloc: the paths' positions and the totals, for the host
//   k_dbin          per path: every tile row's list of the edges in it, and from which tile on the row
//                   has coverage; then the coarse pass
//   k_dcmd_of       the command of every path tile
//   k_dcov          one wavefront per (path, tile row): its edges' area deltas are added up in LDS over
//                   the path's whole width, eight tiles at a time, and prefix-summed along the pixel rows
//                   into the coverage buffer (A per command and pixel)
//   k_dcov_split, k_dcov_sum   the same for the rows whose lists are too long or too wide for one workgroup
//   k_work_order    the tiles heaviest first (commands per tile), for k_dcomp and k_dback
//   k_dcomp         one workgroup per 16x16 tile, one thread per pixel: composites the tile's
//                   commands in draw order from the coverage buffer. With checkpoints on, the pixel
//                   state before every batch of 8 commands is kept, and so is the coverage buffer.
// Backward:
//   k_dback         per tile, batches in reverse: reads the batch's coverage, replays the
//                   batch's compositing from its checkpoint and walks it backwards to get dL/dA per
//                   (command, pixel) and the colour gradients
//   k_dedge_grad    one wavefront per 6 points of a stroke or 8 to 60 of a fill: the boundary integral of
//                   dL/dA over every piece of their edges inside a pixel, in all tiles that they
//                   cross, added up to the gradients of the points and normals that the edges hang on
//   k_dg_points, k_dg_ctrl, k_dg_paths: chain rule to points, half-widths, control points, colours and
//                   widths, all as gathers
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "vkh_internal.h"
#include "vkvg_diff.h"

#define VKD_NSEG 16 // polyline segments per cubic
#define VKD_T 16    // tile size in pixels
#define VKD_B 8     // commands per batch of the backward pass (and per compositing checkpoint)
#define VKD_CT 8    // tiles of a row whose coverage a wavefront adds up at a time: 128 columns, two per lane
#define VKD_NO_CMD 0xFFFFFFFFu // a path tile without a command
#define VKD_BIN_MARGIN 0.01f // px added around an edge when binning (rounding safety)

namespace {

__device__ __forceinline__ float2 f2(float x, float y) { return make_float2(x, y); }

// geometry in R = float (product path) or double (the FP64 evaluation used by finite differences)
template <typename R> struct alignas(2 * sizeof(R)) RV2 {
    R x, y;
};
template <typename R> struct alignas(4 * sizeof(R)) RV4 {
    R x, y, z, w;
};
template <typename R> __device__ __forceinline__ RV2<R> r2(R x, R y) { return RV2<R>{x, y}; }

// --------------------------------------------------------------------------------- geometry
template <typename R>
__global__ void k_dflatten(uint32_t n_pts, const uint32_t *__restrict__ pt_path,
                           const uint32_t *__restrict__ path_first_pt, const uint32_t *__restrict__ path_first_ctrl,
                           const uint32_t *__restrict__ path_ncubic, const float2 *__restrict__ ctrl,
                           RV2<R> *__restrict__ pts) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_pts)
        return;
    uint32_t path = pt_path[p];
    uint32_t j = p - path_first_pt[path];
    uint32_t q = j / VKD_NSEG, i = j % VKD_NSEG;
    uint32_t n3 = 3 * path_ncubic[path];
    const float2 *c = ctrl + path_first_ctrl[path];
    const float2 c0 = c[3 * q], c1 = c[3 * q + 1], c2 = c[3 * q + 2], c3 = c[(3 * q + 3) % n3];
    const R t = (R)i / (R)VKD_NSEG, u = (R)1 - t;
    const R b0 = u * u * u, b1 = (R)3 * u * u * t, b2 = (R)3 * u * t * t, b3 = t * t * t;
    pts[p] = r2<R>(b0 * (R)c0.x + b1 * (R)c1.x + b2 * (R)c2.x + b3 * (R)c3.x,
                   b0 * (R)c0.y + b1 * (R)c1.y + b2 * (R)c2.y + b3 * (R)c3.y);
}

__device__ __forceinline__ uint32_t next_pt(uint32_t p, uint32_t first, uint32_t end) {
    return p + 1 == end ? first : p + 1;
}
__device__ __forceinline__ uint32_t prev_pt(uint32_t p, uint32_t first, uint32_t end) {
    return p == first ? end - 1 : p - 1;
}

template <typename R>
__global__ void k_dnormals(uint32_t n_pts, const uint32_t *__restrict__ pt_path,
                           const uint32_t *__restrict__ path_first_pt, const RV2<R> *__restrict__ pts,
                           RV2<R> *__restrict__ nrm) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_pts)
        return;
    uint32_t path = pt_path[p];
    uint32_t nx = next_pt(p, path_first_pt[path], path_first_pt[path + 1]);
    R dx = pts[nx].x - pts[p].x, dy = pts[nx].y - pts[p].y;
    R L = sqrt(dx * dx + dy * dy);
    nrm[p] = L > (R)0 ? r2<R>(-dy / L, dx / L) : r2<R>((R)0, (R)0);
}

template <typename R>
__device__ __forceinline__ RV2<R> vpos(const RV2<R> *pts, const RV2<R> *nrm, R h, uint32_t i, uint32_t k, int s) {
    if (!s)
        return pts[i];
    R sh = (R)s * h;
    return r2<R>(pts[i].x + sh * nrm[k].x, pts[i].y + sh * nrm[k].y);
}

template <typename R>
__global__ void k_dedges(uint32_t n_pts, const uint32_t *__restrict__ pt_path,
                         const uint32_t *__restrict__ path_first_pt, const uint32_t *__restrict__ path_first_edge,
                         const uint32_t *__restrict__ path_stroke, const float *__restrict__ width,
                         const RV2<R> *__restrict__ pts, const RV2<R> *__restrict__ nrm, RV4<R> *__restrict__ edges) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_pts)
        return;
    uint32_t path = pt_path[p];
    uint32_t first = path_first_pt[path], end = path_first_pt[path + 1];
    uint32_t j = p - first;
    uint32_t nx = next_pt(p, first, end);
    if (!path_stroke[path]) {
        uint32_t e = path_first_edge[path] + j;
        edges[e] = RV4<R>{pts[p].x, pts[p].y, pts[nx].x, pts[nx].y};
        return;
    }
    const R h = (R)0.5 * (R)width[path];
    uint32_t e = path_first_edge[path] + 10 * j;
    uint32_t vi[4] = {p, nx, nx, p}, vk[4] = {p, p, p, p};
    int vs[4] = {1, 1, -1, -1};
    for (int a = 0; a < 4; a++) {
        int b = (a + 1) & 3;
        RV2<R> A = vpos(pts, nrm, h, vi[a], vk[a], vs[a]), Bv = vpos(pts, nrm, h, vi[b], vk[b], vs[b]);
        edges[e] = RV4<R>{A.x, A.y, Bv.x, Bv.y};
        e++;
    }
    uint32_t pp = prev_pt(p, first, end);
    RV2<R> n0 = nrm[pp], n1 = nrm[p];
    bool swap = n0.x * n1.y - n0.y * n1.x > (R)0;
    for (int s = 1; s >= -1; s -= 2) {
        uint32_t ti[3] = {p, p, p}, tk[3] = {0, pp, p};
        int ts[3] = {0, s, s};
        if (swap) {
            tk[1] = p;
            tk[2] = pp;
        }
        for (int a = 0; a < 3; a++) {
            int b = a == 2 ? 0 : a + 1;
            RV2<R> A = vpos(pts, nrm, h, ti[a], tk[a], ts[a]), Bv = vpos(pts, nrm, h, ti[b], tk[b], ts[b]);
            edges[e] = RV4<R>{A.x, A.y, Bv.x, Bv.y};
            e++;
        }
    }
}

// ---------------------------------------------------------------------------------- binning
// One workgroup per path lists the edges of every tile row and finds the first tile column of the row
// that an edge reaches: from there to the right end of the bbox the tiles may be covered and get a
// command. A list entry per edge and tile row (1.1 per edge at 3 px edges) replaces one per edge and tile
// from the edge to the right end of the bbox (3.7), so the coverage pass reads a third.
#define VKD_ROWS_MAX 1024 // tile rows of the tallest image (16384)
__device__ __forceinline__ int32_t tile_of(float v) { // clamped before the conversion
    return (int32_t)fminf(fmaxf(floorf(v / VKD_T), -1.0e6f), 1.0e6f);
}
// tile rows and first tile column of an edge, widened by VKD_BIN_MARGIN px; empty (r0 > r1) for
// edges with a NaN coordinate, horizontal ones and those right of the bbox
template <typename R>
__device__ __forceinline__ void dbin_range(const RV4<R> &v, const DrawTiles &dt, int32_t &r0, int32_t &r1,
                                           int32_t &c0) {
    r0 = 1;
    r1 = 0;
    c0 = 0;
    if (v.y == v.w || isnan(v.x) || isnan(v.y) || isnan(v.z) || isnan(v.w))
        return;
    const float ymin = (float)fmin(v.y, v.w) - VKD_BIN_MARGIN, ymax = (float)fmax(v.y, v.w) + VKD_BIN_MARGIN;
    const float xmin = (float)fmin(v.x, v.z) - VKD_BIN_MARGIN;
    c0 = max(tile_of(xmin), dt.bx0);
    if (c0 > dt.bx1)
        return;
    r0 = max(tile_of(ymin), dt.by0);
    r1 = min(tile_of(ymax), dt.by1);
}

// What a path takes: path tiles, tile rows, list entries; then where its own begin
struct PathAlloc {
    uint32_t tiles, rows, segs;
};

// One workgroup per path: bbox of its edges in 24.8 fixed point (floor / ceil) and from it the tiles
template <typename R>
__global__ __launch_bounds__(256) void k_dpaths(const uint32_t *__restrict__ path_first_edge,
                                                const RV4<R> *__restrict__ edges, int32_t tilesW, int32_t tilesH,
                                                DrawTiles *__restrict__ dts, PathAlloc *__restrict__ alloc) {
    __shared__ int32_t red[4][4];
    __shared__ uint32_t s_sum[4];
    const uint32_t d = blockIdx.x, tid = threadIdx.x;
    const uint32_t e0 = path_first_edge[d], e1 = path_first_edge[d + 1];
    float x0 = 3.0e38f, y0 = 3.0e38f, x1 = -3.0e38f, y1 = -3.0e38f;
    for (uint32_t e = e0 + tid; e < e1; e += 256) {
        const RV4<R> v = edges[e];
        if (v.y == v.w || isnan(v.x) || isnan(v.y) || isnan(v.z) || isnan(v.w))
            continue; // horizontal edges contribute nothing
        // widened by the binning margin so that rounding to float never loses a tile
        x0 = fminf(x0, (float)fmin(v.x, v.z) - VKD_BIN_MARGIN);
        x1 = fmaxf(x1, (float)fmax(v.x, v.z) + VKD_BIN_MARGIN);
        y0 = fminf(y0, (float)fmin(v.y, v.w) - VKD_BIN_MARGIN);
        y1 = fmaxf(y1, (float)fmax(v.y, v.w) + VKD_BIN_MARGIN);
    }
    for (int o = 32; o > 0; o >>= 1) {
        x0 = fminf(x0, __shfl_xor(x0, o));
        y0 = fminf(y0, __shfl_xor(y0, o));
        x1 = fmaxf(x1, __shfl_xor(x1, o));
        y1 = fmaxf(y1, __shfl_xor(y1, o));
    }
    auto fx = [](float v, bool up) -> int32_t {
        float s = v * 256.0f;
        s = up ? ceilf(s) : floorf(s);
        return (int32_t)fminf(fmaxf(s, -8.0e6f), 8.0e6f);
    };
    if ((tid & 63) == 0) {
        int w = tid >> 6;
        red[w][0] = x0 > x1 ? INT32_MAX : fx(x0, false);
        red[w][1] = x0 > x1 ? INT32_MAX : fx(y0, false);
        red[w][2] = x0 > x1 ? INT32_MIN : fx(x1, true);
        red[w][3] = x0 > x1 ? INT32_MIN : fx(y1, true);
    }
    __syncthreads();
    int4 b = make_int4(INT32_MAX, INT32_MAX, INT32_MIN, INT32_MIN);
    for (int w = 0; w < 4; w++) {
        b.x = min(b.x, red[w][0]);
        b.y = min(b.y, red[w][1]);
        b.z = max(b.z, red[w][2]);
        b.w = max(b.w, red[w][3]);
    }
    constexpr int SSH = 8 + __builtin_ctz(VKD_T);
    DrawTiles dt;
    dt.bx0 = dt.by0 = 0;
    dt.bx1 = dt.by1 = -1;
    if (b.x <= b.z) {
        dt.bx0 = max(b.x >> SSH, 0);
        dt.by0 = max(b.y >> SSH, 0);
        dt.bx1 = min(b.z >> SSH, tilesW - 1);
        dt.by1 = min(b.w >> SSH, tilesH - 1);
    }
    const bool some = dt.bx0 <= dt.bx1 && dt.by0 <= dt.by1;
    if (!some) {
        dt.bx0 = dt.by0 = 0;
        dt.bx1 = dt.by1 = -1;
    }
    dt.pt_base = 0;
    dt.bw = some ? (uint32_t)(dt.bx1 - dt.bx0 + 1) : 0u;
    uint32_t n = 0;
    if (some)
        for (uint32_t e = e0 + tid; e < e1; e += 256) {
            int32_t r0, r1, c0;
            dbin_range(edges[e], dt, r0, r1, c0);
            n += r0 <= r1 ? (uint32_t)(r1 - r0 + 1) : 0u;
        }
    for (int o = 32; o > 0; o >>= 1)
        n += __shfl_xor(n, o);
    if ((tid & 63) == 0)
        s_sum[tid >> 6] = n;
    __syncthreads();
    if (tid == 0) {
        const uint32_t rows = (uint32_t)(dt.by1 - dt.by0 + 1);
        dts[d] = dt;
        alloc[d] = PathAlloc{dt.bw * rows, rows, s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3]};
    }
}

// Positions of every path's tiles, rows and list entries (exclusive sums, in one workgroup), and the totals
// into the host's memory; clears k_dbin's counters of split rows
__global__ __launch_bounds__(1024) void k_dalloc(uint32_t n_paths, PathAlloc *__restrict__ alloc,
                                                 DrawTiles *__restrict__ dts, uint32_t *__restrict__ split,
                                                 uint32_t *__restrict__ totals) {
    __shared__ uint32_t s_w[16][3];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = tid >> 6;
    uint32_t run[3] = {0, 0, 0};
    for (uint32_t base = 0; base < n_paths; base += 1024) {
        const uint32_t d = base + tid;
        const PathAlloc a = d < n_paths ? alloc[d] : PathAlloc{0, 0, 0};
        const uint32_t v[3] = {a.tiles, a.rows, a.segs};
        uint32_t x[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            x[k] = v[k];
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t y = __shfl_up(x[k], o);
                x[k] += (int)lane >= o ? y : 0u;
            }
            if (lane == 63)
                s_w[wv][k] = x[k];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 3; k++) {
            x[k] += run[k] - v[k];
            for (uint32_t w = 0; w < 16; w++) {
                x[k] += w < wv ? s_w[w][k] : 0u;
                run[k] += s_w[w][k];
            }
        }
        if (d < n_paths) {
            alloc[d] = PathAlloc{x[0], x[1], x[2]};
            dts[d].pt_base = x[0];
        }
        __syncthreads();
    }
    if (tid == 0)
        for (int k = 0; k < 3; k++) {
            totals[k] = run[k];
            split[k] = 0;
        }
}

__device__ __forceinline__ uint32_t block_excl_scan(uint32_t *a, uint32_t n, uint32_t *s_wave) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t per = (n + 255u) / 256u, beg = min(tid * per, n), end = min(beg + per, n);
    uint32_t sum = 0;
    for (uint32_t k = beg; k < end; k++)
        sum += a[k];
    uint32_t x = sum;
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o);
        if ((int)lane >= o)
            x += y;
    }
    if (lane == 63)
        s_wave[w] = x;
    __syncthreads();
    uint32_t run = x - sum, total = 0;
    for (uint32_t k = 0; k < 4; k++) {
        run += k < w ? s_wave[k] : 0u;
        total += s_wave[k];
    }
    for (uint32_t k = beg; k < end; k++) {
        uint32_t v = a[k];
        a[k] = run;
        run += v;
    }
    __syncthreads();
    return total;
}

// A tile row with coverage: path and row within its bbox. Its list is in the row's first path tile
// (seg_off, ntouch); nseg of every path tile says whether it gets a command. acc: VKD_WHOLE, or where the sums
// of a row begin that is split over workgroups (SplitRow).
#define VKD_WHOLE 0xFFFFFFFFu
struct RowUnit {
    uint32_t draw, row, acc;
};
// A row that k_dcov_split shares out: one workgroup per VKD_CT tiles and VKD_SLICE entries of the list,
// from workgroup `first` on
#define VKD_SLICE 1024u
struct SplitRow {
    uint32_t unit, first;
};
// What a tile row costs its workgroup, in steps of some 2 us: one per 256 list entries and eight tiles, mostly entries
// passed over, and four per 256 entries for what they add. A row is split beyond 96 steps (splitting takes 20
// to 50 us itself: 10 strokes of 30 cubics on 1024x1024, 60 steps, 210 us whole and 266 split; 6 paths of 50 cubics on
// 300x40, 112 steps, 332 and 234), and beyond four times what the frame's rows take together on some 2048 workgroups at a
// time: up to there a whole row ends with the others.
__device__ __forceinline__ uint32_t row_steps(uint32_t eights, uint32_t n) { return (eights + 4u) * ((n + 255u) / 256u); }
inline uint32_t split_steps(uint32_t n_ptiles, uint32_t n_rows, uint32_t n_segs) {
    return std::max<uint32_t>(96u, (uint32_t)((n_ptiles / VKD_CT + 4ull * n_rows + n_segs / 64u) / 512u));
}

template <typename R>
__global__ __launch_bounds__(256) void k_dbin(const uint32_t *__restrict__ path_first_edge,
                                              const RV4<R> *__restrict__ edges, const DrawTiles *__restrict__ dts,
                                              const PathAlloc *__restrict__ alloc, PathTile *__restrict__ ptl,
                                              uint32_t *__restrict__ cmd_of, uint32_t *__restrict__ segs,
                                              RowUnit *__restrict__ units, SplitRow *__restrict__ splits,
                                              unsigned long long *__restrict__ n_split, uint32_t *__restrict__ n_acc,
                                              uint32_t max_steps) {
    __shared__ uint32_t s_cnt[VKD_ROWS_MAX]; // edges per row, then offsets, then cursors
    __shared__ int32_t s_col[VKD_ROWS_MAX];  // first tile column reached
    __shared__ uint32_t s_wave[4];
    const uint32_t d = blockIdx.x, tid = threadIdx.x;
    const DrawTiles dt = dts[d];
    if (dt.bw == 0)
        return;
    const uint32_t e0 = path_first_edge[d], e1 = path_first_edge[d + 1], base = alloc[d].segs, unit0 = alloc[d].rows;
    const uint32_t bw = dt.bw, bh = (uint32_t)(dt.by1 - dt.by0 + 1); // at most VKD_ROWS_MAX rows
    for (uint32_t k = tid; k < bh; k += 256) {
        s_cnt[k] = 0;
        s_col[k] = INT32_MAX;
    }
    __syncthreads();
    for (uint32_t e = e0 + tid; e < e1; e += 256) {
        int32_t r0, r1, c0;
        dbin_range(edges[e], dt, r0, r1, c0);
        for (int32_t r = r0; r <= r1; r++) {
            atomicAdd(&s_cnt[r - dt.by0], 1u);
            atomicMin(&s_col[r - dt.by0], c0);
        }
    }
    __syncthreads();
    const uint32_t total = block_excl_scan(s_cnt, bh, s_wave);
    for (uint32_t k = tid; k < bh * bw; k += 256) {
        const uint32_t r = k / bw, off = s_cnt[r], next = r + 1 < bh ? s_cnt[r + 1] : total;
        PathTile pt;
        pt.backdrop = 0;
        pt.nseg = dt.bx0 + (int32_t)(k - r * bw) >= s_col[r] ? 1u : 0u;
        pt.seg_off = base + off;
        pt.ntouch = next - off;
        ptl[dt.pt_base + k] = pt;
        cmd_of[dt.pt_base + k] = VKD_NO_CMD;
    }
    for (uint32_t k = tid; k < bh; k += 256) {
        const uint32_t n = (k + 1 < bh ? s_cnt[k + 1] : total) - s_cnt[k], eights = (bw + VKD_CT - 1) / VKD_CT;
        uint32_t acc = VKD_WHOLE;
        if (row_steps(eights, n) > max_steps) { // rows in the upper half, workgroups in the lower: in one order
            const unsigned long long at =
                atomicAdd(n_split, (1ull << 32) + (unsigned long long)eights * ((n + VKD_SLICE - 1) / VKD_SLICE));
            splits[at >> 32] = SplitRow{unit0 + k, (uint32_t)at};
            acc = atomicAdd(n_acc, eights);
        }
        units[unit0 + k] = RowUnit{d, k, acc};
    }
    __syncthreads();
    for (uint32_t e = e0 + tid; e < e1; e += 256) {
        int32_t r0, r1, c0;
        dbin_range(edges[e], dt, r0, r1, c0);
        for (int32_t r = r0; r <= r1; r++)
            segs[base + atomicAdd(&s_cnt[r - dt.by0], 1u)] = e;
    }
}

// --------------------------------------------------------------------------- edge pieces
// The part of edge v inside pixel row [yr, yr + 1): x range, the edge's parameter at its left and
// right end, and its dy, signed, from the y clip. Parameters at pixel borders are used only
// strictly inside (clamped), which keeps nearly vertical edges well conditioned.
template <typename R> struct RowPart {
    R xl, xr, sL, sR, s0, s1, dy, dxt, dyt, ax;
    __device__ __forceinline__ bool clip(const RV4<R> &v, R yr) {
        const R ay = v.y, by = v.w;
        ax = v.x;
        const R ylo = fmax(fmin(ay, by), yr), yhi = fmin(fmax(ay, by), yr + (R)1);
        if (!(ylo < yhi))
            return false;
        dyt = by - ay;
        dxt = v.z - ax;
        const R sa = (ylo - ay) / dyt, sb = (yhi - ay) / dyt;
        s0 = fmin(sa, sb);
        s1 = fmax(sa, sb);
        const R x0 = ax + s0 * dxt, x1 = ax + s1 * dxt;
        xl = fmin(x0, x1);
        xr = fmax(x0, x1);
        sL = x0 <= x1 ? s0 : s1;
        sR = x0 <= x1 ? s1 : s0;
        dy = dyt > (R)0 ? yhi - ylo : ylo - yhi;
        return true;
    }
    // parameter where the part crosses x: sL left of it, sR right of it
    __device__ __forceinline__ R param(R x) const {
        return x <= xl ? sL : x >= xr ? sR : fmin(fmax((x - ax) / dxt, s0), s1);
    }
    // dy of what lies left of x: 0 and the whole dy outside the part, so the pieces of an edge add up to
    // the y clip's dy and the edges of a closed outline cancel right of it
    __device__ __forceinline__ R dy_left(R x) const {
        return x <= xl ? (R)0 : x >= xr ? dy : fabs(param(x) - sL) * dyt;
    }
};

// Rows shared out over a wavefront: every lane has an edge with cnt (at most 16) pixel rows (or other items) from
// `first` on, and f(lane of the edge, row) is called once for each of all the lanes' rows, 64 at a time. Edges
// cross few rows, some many: a lane doing its own edge's rows would wait for the longest.
struct RowShare {
    uint8_t lane[64 * VKD_T];
    int32_t row[64]; // of the edge's item 0
};
template <class F> __device__ __forceinline__ void share_rows(RowShare &sh, uint32_t lane, int32_t first, uint32_t cnt, F f) {
    uint32_t x = cnt; // inclusive sum over the lanes
#define VKD_DPP(ctrl, rows) (uint32_t) __builtin_amdgcn_update_dpp(0, (int)x, ctrl, rows, 0xf, false)
    x += VKD_DPP(0x111, 0xf); // row_shr:1, 2, 4, 8, then row_bcast:15 and 31
    x += VKD_DPP(0x112, 0xf);
    x += VKD_DPP(0x114, 0xf);
    x += VKD_DPP(0x118, 0xf);
    x += VKD_DPP(0x142, 0xa);
    x += VKD_DPP(0x143, 0xc);
#undef VKD_DPP
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)x, 63), at = x - cnt;
    sh.row[lane] = first - (int32_t)at;
    for (uint32_t k = 0; k < cnt; k++)
        sh.lane[at + k] = (uint8_t)lane;
    // sh is this wavefront's own: its LDS accesses complete in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (uint32_t it = lane; it < total; it += 64) {
        const uint32_t j = sh.lane[it];
        f(j, (int32_t)it + sh.row[j]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// ---------------------------------------------------------------------------------- forward
__device__ __forceinline__ float4 premul(float4 c) { return make_float4(c.x * c.w, c.y * c.w, c.z * c.w, c.w); }

// the command of every path tile that has one
__global__ void k_dcmd_of(uint32_t n_cmds, const Cmd *__restrict__ cmds, uint32_t *__restrict__ cmd_of) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < n_cmds)
        cmd_of[cmds[c].pt] = c;
}

// carry plus the sum of x over the lanes below this one
__device__ __forceinline__ double wave_excl_sum(double x, double carry, uint32_t lane) {
    x = __shfl_up(x, 1);
    if (lane == 0)
        x = carry;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double y = __shfl_up(x, o);
        if ((int)lane >= o)
            x += y;
    }
    return x;
}
// the float one moves data in the adders' operands: a shift by one lane, shifts within rows of 16, then
// the last lane of a row to the next row and that of the lower half to the upper
template <int CTRL, int ROWS> __device__ __forceinline__ float lane_move(float old, float x) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(x), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float wave_excl_sum(float x, float carry, uint32_t) {
    x = lane_move<0x138, 0xf>(carry, x);  // wave_shr:1
    x += lane_move<0x111, 0xf>(0.f, x);   // row_shr:1, 2, 4, 8
    x += lane_move<0x112, 0xf>(0.f, x);
    x += lane_move<0x114, 0xf>(0.f, x);
    x += lane_move<0x118, 0xf>(0.f, x);
    x += lane_move<0x142, 0xa>(0.f, x);   // row_bcast:15 into rows 1 and 3
    x += lane_move<0x143, 0xc>(0.f, x);   // row_bcast:31 into rows 2 and 3
    return x;
}

// Deposits are rounded to 2^-23 and an edge's parts are differences of such numbers, as coordinates from 1 on are.
// While no partial sum exceeds 2 in magnitude float sums of them are therefore exact: they do not depend on
// the order of the atomics, and beside a closed outline that winds once the coverage is exactly 0 or 1. Where a path
// lies over itself more often (a tight bend of a wide stroke) sums are rounded, to 2^-22 from 2 to 4, and their
// last bits depend on the order. Against float64 over 160 scenes of 100x72 to 282x291 the image's relative error is
// 0.4 to 1.7e-6 (0.5 to 1.8e-6 with a list of edges per tile, whose sums were not on a grid), the colour
// gradients' 0.30 to 0.57e-6 (0.34 to 0.61e-6; 1.6 times that without the grid, 1.1 times with 2^-24, exact up to 1 only).
#define VKD_GRID 8388608.0f
__device__ __forceinline__ float deposit(float x) { return rintf(x * VKD_GRID) * (1.0f / VKD_GRID); }
__device__ __forceinline__ double deposit(double x) { return x; }

// Coverage of every command. One workgroup per tile row of a path, VKD_CT tiles at a time: its wavefronts
// share the row's edges, one lane per edge and pixel row adds the area deltas to the row's cells in LDS, then every
// pixel row is prefix-summed (two columns per lane, the sum so far carried on) into cov[c * 256 + pixel]. Each
// edge is so evaluated once per pixel row it crosses (2.7 on edges of 3 px) and not in all 16 rows of every
// tile up to the right end of the path, which the carry covers. Bound by the chains of instructions per row and
// piece. 1024x768 with 3000 paths (1.4 M edges): 121 us (406 with all rows of all tiles); 512x512 with 1024: 55 (180);
// 100x72 with 48: 22 (93).
constexpr int VKD_COLS = VKD_CT * VKD_T, VKD_LD = VKD_COLS + 2; // one more cell takes the last column's overflow
constexpr int VKD_RW = VKD_T / 4;                               // pixel rows that a wavefront prefix-sums
static_assert(VKD_COLS == 128, "two columns per lane");

// adds what the entries [i0, end) of a list, `share` at a time for this wavefront and every fourth such
// share from i0 on, cover of the nt tiles from tile c0 of the row on to acc; ed and rows are the wavefront's own
template <typename R>
__device__ __forceinline__ void dcov_add(R *acc, RV4<R> *ed, RowShare &rows, uint32_t lane, const DrawTiles &dt, int32_t Y0,
                                         uint32_t c0, uint32_t nt, uint32_t i0, uint32_t end, uint32_t share,
                                         const uint32_t *__restrict__ list, const RV4<R> *__restrict__ edges) {
    const R X0 = (R)(dt.bx0 * VKD_T); // x is taken from the path's left tile border: less rounding
    const R XL = (R)(c0 * VKD_T), XR = XL + (R)(nt * VKD_T);
    for (; i0 < end; i0 += 4 * share) {
        int32_t ra = 0, rb = -1;
        if (lane < share && i0 + lane < end) {
            RV4<R> v = edges[list[i0 + lane]];
            v.x -= X0;
            v.z -= X0;
            ed[lane] = v;
            // left of these columns: in the carry
            if (!((c0 && fmax(v.x, v.z) < XL) || fmin(v.x, v.z) > XR)) {
                ra = (int32_t)fmin(fmax(floor(fmin(v.y, v.w)) - (R)Y0, (R)0), (R)VKD_T);
                rb = (int32_t)fmax(fmin(floor(fmax(v.y, v.w)) - (R)Y0, (R)(VKD_T - 1)), (R)-1);
            }
        }
        share_rows(rows, lane, ra, (uint32_t)max(rb - ra + 1, 0), [&](uint32_t j, int32_t r) {
            RowPart<R> p;
            if (!p.clip(ed[j], (R)(Y0 + r)))
                return;
            R *a = acc + r * VKD_LD;
            R done = deposit(p.dy_left(XL));
            if (c0 == 0 && done != (R)0)
                atomicAdd(&a[0], done);
            const R xa0 = fmax(p.xl, XL), xb0 = fmin(p.xr, XR);
            if (!(xa0 <= xb0))
                return;
            const int32_t cl = (int32_t)(floor(xa0) - XL);
            const int32_t cr = min((int32_t)(floor(xb0) - XL), (int32_t)(nt * VKD_T) - 1);
            for (int32_t c = cl; c <= cr; c++) {
                const R cx = XL + (R)c, cn = cx + (R)1;
                const R xa = fmax(p.xl, cx), xb = fmin(p.xr, cn);
                const R upto = deposit(p.dy_left(cn)), dy = upto - done;
                done = upto;
                const R right = deposit(dy * ((R)0.5 * (xa + xb) - cx));
                atomicAdd(&a[c], dy - right);
                atomicAdd(&a[c + 1], right);
            }
        });
    }
}

// prefix sums of this wavefront's pixel rows of acc, onto carry and on, to the commands of the nt tiles from path tile pt
// on; leaves the cells at zero
template <typename R>
__device__ __forceinline__ void dcov_sum(R *acc, R (&carry)[VKD_RW], uint32_t lane, uint32_t wv, uint32_t pt, uint32_t nt,
                                         const uint32_t *__restrict__ cmd_of, R *__restrict__ cov) {
    const uint32_t tl = lane / (64 / VKD_CT); // this lane's tile
    const uint32_t cmd = tl < nt ? cmd_of[pt + tl] : VKD_NO_CMD;
    R *out = cov + (size_t)cmd * 256 + 2 * (lane & (64 / VKD_CT - 1));
#pragma unroll
    for (int q = 0; q < VKD_RW; q++) {
        const int r = (int)wv * VKD_RW + q;
        RV2<R> *cell = (RV2<R> *)&acc[r * VKD_LD + 2 * lane];
        const RV2<R> v = *cell;
        const R over = acc[r * VKD_LD + VKD_COLS];
        *cell = RV2<R>{(R)0, (R)0};
        RV2<R> o;
        o.x = wave_excl_sum(v.x + v.y, carry[q], lane) + v.x;
        o.y = o.x + v.y;
        if (cmd != VKD_NO_CMD)
            *(RV2<R> *)(out + r * VKD_T) = o;
        carry[q] = __shfl(o.y, 63) + over;
    }
    if (lane < VKD_RW)
        acc[(wv * VKD_RW + lane) * VKD_LD + VKD_COLS] = (R)0;
}

template <typename R>
__global__ __launch_bounds__(256) void k_dcov(const RowUnit *__restrict__ units, const DrawTiles *__restrict__ dts,
                                              const PathTile *__restrict__ ptl, const uint32_t *__restrict__ cmd_of,
                                              const uint32_t *__restrict__ segs, const RV4<R> *__restrict__ edges,
                                              R *__restrict__ cov) {
    __shared__ alignas(16) R acc[VKD_T * VKD_LD];
    __shared__ RV4<R> s_edge[4][64];
    __shared__ RowShare s_rows[4];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const RowUnit ru = units[blockIdx.x];
    const DrawTiles dt = dts[ru.draw];
    const uint32_t pt0 = dt.pt_base + ru.row * dt.bw;
    const uint32_t off = ptl[pt0].seg_off, n = ptl[pt0].ntouch;
    if (!n || ru.acc != VKD_WHOLE)
        return;
    for (uint32_t i = threadIdx.x; i < (uint32_t)(VKD_T * VKD_LD); i += 256)
        acc[i] = (R)0;
    __syncthreads();
    const int32_t Y0 = (dt.by0 + (int32_t)ru.row) * VKD_T;
    const uint32_t share = min((n + 3) / 4, 64u); // edges per wavefront and turn
    R carry[VKD_RW];
#pragma unroll
    for (int r = 0; r < VKD_RW; r++)
        carry[r] = (R)0;
    for (uint32_t c0 = 0; c0 < dt.bw; c0 += VKD_CT) {
        const uint32_t nt = min((uint32_t)VKD_CT, dt.bw - c0);
        dcov_add(acc, s_edge[wv], s_rows[wv], lane, dt, Y0, c0, nt, wv * share, n, share, segs + off, edges);
        __syncthreads();
        dcov_sum(acc, carry, lane, wv, pt0 + c0, nt, cmd_of, cov);
        __syncthreads();
    }
}

// Rows too long for one workgroup (row_steps): one workgroup per eight tiles and VKD_SLICE entries adds its cells up in
// LDS and then into the row's in memory, which k_dcov_sum carries on from eight to eight. 8192x64 with one path of
// 200 cubics, forward: 348 us (8878 us with a workgroup per row, 1757 with a list of edges per tile, 64
// entries at a time); four curled strokes of 300 cubics on 256x256: 517 us (970 and 846).
template <typename R>
__global__ __launch_bounds__(256) void k_dcov_split(const SplitRow *__restrict__ splits, uint32_t n_split, uint32_t g0,
                                                    const RowUnit *__restrict__ units, const DrawTiles *__restrict__ dts,
                                                    const PathTile *__restrict__ ptl, const uint32_t *__restrict__ segs,
                                                    const RV4<R> *__restrict__ edges, R *__restrict__ sums) {
    __shared__ alignas(16) R acc[VKD_T * VKD_LD];
    __shared__ RV4<R> s_edge[4][64];
    __shared__ RowShare s_rows[4];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t g = g0 + blockIdx.x;
    uint32_t lo = 0, hi = n_split; // the last row that begins at or before this workgroup
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (splits[mid].first <= g)
            lo = mid;
        else
            hi = mid;
    }
    const RowUnit ru = units[splits[lo].unit];
    const DrawTiles dt = dts[ru.draw];
    const PathTile &pt = ptl[dt.pt_base + ru.row * dt.bw];
    const uint32_t eights = (dt.bw + VKD_CT - 1) / VKD_CT, i = g - splits[lo].first;
    const uint32_t e = i % eights, c0 = e * VKD_CT, first = i / eights * VKD_SLICE, end = min(first + VKD_SLICE, pt.ntouch);
    for (uint32_t k = threadIdx.x; k < (uint32_t)(VKD_T * VKD_LD); k += 256)
        acc[k] = (R)0;
    __syncthreads();
    dcov_add(acc, s_edge[wv], s_rows[wv], lane, dt, (dt.by0 + (int32_t)ru.row) * VKD_T, c0,
             min((uint32_t)VKD_CT, dt.bw - c0), first + wv * 64u, end, 64u, segs + pt.seg_off, edges);
    __syncthreads();
    R *out = sums + (size_t)(ru.acc + e) * (VKD_T * VKD_LD);
    for (uint32_t k = threadIdx.x; k < (uint32_t)(VKD_T * VKD_LD); k += 256)
        if (acc[k] != (R)0)
            unsafeAtomicAdd(&out[k], acc[k]); // device memory
}
template <typename R>
__global__ __launch_bounds__(256) void k_dcov_sum(const SplitRow *__restrict__ splits, const RowUnit *__restrict__ units,
                                                  const DrawTiles *__restrict__ dts, const uint32_t *__restrict__ cmd_of,
                                                  R *__restrict__ sums, R *__restrict__ cov) {
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const RowUnit ru = units[splits[blockIdx.x].unit];
    const DrawTiles dt = dts[ru.draw];
    const uint32_t pt0 = dt.pt_base + ru.row * dt.bw;
    R carry[VKD_RW];
#pragma unroll
    for (int r = 0; r < VKD_RW; r++)
        carry[r] = (R)0;
    R *acc = sums + (size_t)ru.acc * (VKD_T * VKD_LD);
    for (uint32_t c0 = 0; c0 < dt.bw; c0 += VKD_CT, acc += VKD_T * VKD_LD)
        dcov_sum(acc, carry, lane, wv, pt0 + c0, min((uint32_t)VKD_CT, dt.bw - c0), cmd_of, cov);
}

// Compositing in draw order: one workgroup per 16x16 tile, one thread per pixel; coverage comes
// from k_dcov. With checkpoints on, the pixel state before every batch of VKD_B commands is kept
// for the backward pass.
template <typename R>
__global__ __launch_bounds__(256) void k_dcomp(uint32_t W, uint32_t H, uint32_t tilesW, uint32_t nch,
                                               const uint32_t *__restrict__ tile_off, const Cmd *__restrict__ cmds,
                                               const R *__restrict__ cov, const float4 *__restrict__ rgba,
                                               RV4<R> *__restrict__ image, float4 *__restrict__ ckpt,
                                               const uint32_t *__restrict__ batch_off,
                                               const uint32_t *__restrict__ tile_order) {
    const uint32_t t = tile_order[blockIdx.x], tid = threadIdx.x;
    const uint32_t c0 = tile_off[(size_t)t * nch], c1 = tile_off[(size_t)(t + 1) * nch];
    const int32_t px = (int32_t)((t % tilesW) * VKD_T + tid % VKD_T), py = (int32_t)((t / tilesW) * VKD_T + tid / VKD_T);
    RV4<R> st{(R)1, (R)1, (R)1, (R)1};
    for (uint32_t c = c0; c < c1; c++) {
        if (ckpt && ((c - c0) % VKD_B) == 0)
            ckpt[(size_t)(batch_off[t] + (c - c0) / VKD_B) * 256 + tid] =
                make_float4((float)st.x, (float)st.y, (float)st.z, (float)st.w);
        const R A = cov[(size_t)c * 256 + tid];
        const R k = fmin((R)1, fabs(A));
        const float4 cf = rgba[cmds[c].draw];
        const R ca = (R)cf.w;
        const R cx = (R)cf.x * ca, cy = (R)cf.y * ca, cz = (R)cf.z * ca;
        const R ia = (R)1 - ca * k;
        st = RV4<R>{cx * k + st.x * ia, cy * k + st.y * ia, cz * k + st.z * ia, ca * k + st.w * ia};
    }
    if (px < (int32_t)W && py < (int32_t)H)
        image[(size_t)py * W + px] = st;
}

// --------------------------------------------------------------------------------- backward
// sums each of v[0..15] over the 64 lanes of the wavefront; lane l returns the total of value l >> 2. Two
// values take part in one exchange of halves (then of rows) and one addition each; within rows both are
// summed by moves in the adders' operands and a lane keeps the one it is to end up with.
__device__ __forceinline__ float wave_multi_sum16(const float (&v)[16], uint32_t lane) {
    auto swapped = [](auto r) { return __uint_as_float(r[0]) + __uint_as_float(r[1]); };
    float a[8], b[4], c[2];
#pragma unroll
    for (int i = 0; i < 8; i++)
        a[i] = swapped(__builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + 8]), false, false));
#pragma unroll
    for (int i = 0; i < 4; i++)
        b[i] = swapped(__builtin_amdgcn_permlane16_swap(__float_as_uint(a[i]), __float_as_uint(a[i + 4]), false, false));
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const float x = b[i] + lane_move<0x128, 0xf>(0.f, b[i]); // row_ror:8
        const float y = b[i + 2] + lane_move<0x128, 0xf>(0.f, b[i + 2]);
        c[i] = (lane & 8u) ? y : x;
    }
    const float x = c[0] + lane_move<0x141, 0xf>(0.f, c[0]); // row_half_mirror
    const float y = c[1] + lane_move<0x141, 0xf>(0.f, c[1]);
    float d = (lane & 4u) ? y : x;
    d += lane_move<0x4E, 0xf>(0.f, d); // quad_perm [2, 3, 0, 1]
    d += lane_move<0xB1, 0xf>(0.f, d); // quad_perm [1, 0, 3, 2]
    return d;
}

// Compositing backwards: one workgroup per tile, one thread per pixel. dL/dA of every (command, pixel)
// goes to g_cov, in the layout of cov, for k_dedge_grad. Moves 270 MB on 1024x768 with 3000 paths (54 us at
// what a copy reaches) in 64 us; with the sums' values chosen by indexing, which compiled into chains of
// compares over the whole array, it was bound by 280 instructions per command and pixel: 181 us.
__global__ __launch_bounds__(256) void k_dback(uint32_t W, uint32_t H, uint32_t tilesW, uint32_t nch,
                                               const uint32_t *__restrict__ tile_off, const Cmd *__restrict__ cmds,
                                               const float4 *__restrict__ rgba,
                                               const float4 *__restrict__ grad_img, const float4 *__restrict__ ckpt,
                                               const uint32_t *__restrict__ batch_off, const float *__restrict__ cov,
                                               float *__restrict__ g_cov, double *__restrict__ g_col,
                                               const uint32_t *__restrict__ tile_order) {
    __shared__ float s_red2[2][4][32]; // by turns: one barrier a batch
    const uint32_t t = tile_order[blockIdx.x], tid = threadIdx.x, lane = tid & 63;
    const uint32_t c0 = tile_off[(size_t)t * nch], c1 = tile_off[(size_t)(t + 1) * nch];
    if (c0 == c1)
        return;
    const int32_t X0 = (int32_t)(t % tilesW) * VKD_T, Y0 = (int32_t)(t / tilesW) * VKD_T;
    const int32_t px = X0 + (int32_t)(tid % VKD_T), py = Y0 + (int32_t)(tid / VKD_T);
    const bool valid = px < (int32_t)W && py < (int32_t)H;
    float4 g = valid ? grad_img[(size_t)py * W + px] : make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t nbatch = (c1 - c0 + VKD_B - 1) / VKD_B;
    for (uint32_t bb = nbatch; bb-- > 0;) {
        const uint32_t base = c0 + bb * VKD_B;
        const uint32_t nb = min((uint32_t)VKD_B, c1 - base);
        float(*s_red)[32] = s_red2[bb & 1];
        uint32_t c_draw[VKD_B];
#pragma unroll
        for (uint32_t j = 0; j < VKD_B; j++)
            c_draw[j] = cmds[base + min(j, nb - 1)].draw;
        // replay the batch's compositing from its checkpoint, then walk it backwards
        float4 st[VKD_B + 1];
        st[0] = ckpt[(size_t)(batch_off[t] + bb) * 256 + tid];
        float Av[VKD_B];
#pragma unroll
        for (uint32_t j = 0; j < VKD_B; j++) {
            Av[j] = j < nb ? cov[(size_t)(base + j) * 256 + tid] : 0.f;
            if (j < nb) {
                const float k = fminf(1.0f, fabsf(Av[j]));
                const float4 c = premul(rgba[c_draw[j]]);
                const float ia = 1.0f - c.w * k;
                st[j + 1] = make_float4(c.x * k + st[j].x * ia, c.y * k + st[j].y * ia, c.z * k + st[j].z * ia,
                                        c.w * k + st[j].w * ia);
            } else {
                st[j + 1] = st[j];
            }
        }
        auto back4 = [&](auto first) __attribute__((always_inline)) { // four commands, backwards
            constexpr int J0 = decltype(first)::value;
            float gc[16]; // their colour gradients
#pragma unroll
            for (int i = 3; i >= 0; i--) {
                const int j = J0 + i;
                const float A = Av[j];
                const float k = fminf(1.0f, fabsf(A));
                const float fp = fabsf(A) < 1.0f ? (A > 0.f ? 1.f : (A < 0.f ? -1.f : 0.f)) : 0.f;
                const float4 c = premul(rgba[c_draw[j]]);
                const float4 s = st[j];
                const float dk =
                    g.x * (c.x - c.w * s.x) + g.y * (c.y - c.w * s.y) + g.z * (c.z - c.w * s.z) + g.w * (c.w - c.w * s.w);
                const float gs = g.x * s.x + g.y * s.y + g.z * s.z + g.w * s.w;
                const bool on = valid && j < (int)nb;
                gc[4 * i + 0] = on ? g.x * k : 0.f;
                gc[4 * i + 1] = on ? g.y * k : 0.f;
                gc[4 * i + 2] = on ? g.z * k : 0.f;
                gc[4 * i + 3] = on ? g.w * k - gs * k : 0.f;
                if (j < (int)nb) {
                    g_cov[(size_t)(base + j) * 256 + tid] = valid ? dk * fp : 0.f;
                    const float ia = 1.0f - c.w * k;
                    g = make_float4(g.x * ia, g.y * ia, g.z * ia, g.w * ia);
                }
            }
            const float tot = wave_multi_sum16(gc, lane); // summed over the tile's pixels
            if ((lane & 3u) == 0)
                s_red[tid >> 6][4 * J0 + (lane >> 2)] = tot;
        };
        static_assert(VKD_B == 8, "two fours");
        back4(std::integral_constant<int, 4>());
        back4(std::integral_constant<int, 0>());
        __syncthreads();
        if (tid < 4 * nb) { // double: a path's tiles add up in any order
            const double v = ((double)s_red[0][tid] + s_red[1][tid]) + ((double)s_red[2][tid] + s_red[3][tid]);
            if (v != 0.0)
                unsafeAtomicAdd(&g_col[4 * cmds[base + (tid >> 2)].draw + (tid & 3)], v); // device memory
        }
    }
}

// Gradients of the points and normals that the edges hang on. One wavefront takes the edges of 6 points of
// a stroke (60) or 8 to 60 of a fill; one lane per edge and pixel row integrates dL/dA along the edge's pieces in the
// row, over all tiles that it crosses, and adds to the edge's two sums in LDS. The edge's endpoint gradients are
// (-dy, dx) times the sums. Edge layout per path: a fill has edge j = p_j -> p_j+1; a stroke has, per point j, 10
// edges: the rectangle of segment j (p_j + n_j, p_j+1 + n_j, p_j+1 - n_j, p_j - n_j) and two bevel triangles at
// vertex j (p_j, then p_j + s n_j-1 and p_j + s n_j in the order of k_dedges; s = 1, -1), in units of the
// half-width. Per point p the sums go to own[p] (on point p, on the next point) and, for strokes, to own_n[p]
// (on normal p, on the previous normal, without the half-width). Bound by the loads of g_cov that wait for
// the tile's command. With k_dg_points 76 us on 1024x768 with 3000 paths; one lane per edge for all its rows, the
// edges' gradients written (23 MB) and gathered by two kernels, took 125 + 110 us. A lane takes at most VKD_EB columns of
// a row, so that flat edges are shared out too: 8192x64 with one path of 200 cubics, whole backward, 117 us (738 with
// whole rows, 190 with a thread per edge and tile).
#define VKD_EB 32
struct GradUnit {
    uint32_t first_pt, path, n; // n points
};
// Points of a fill per wavefront: 60, fewer where that leaves the scene fewer than some 4096 wavefronts. 64x8192 with 20
// paths of 60 cubics, backward: 280 us with 60 points, 203 with 1024 wavefronts, 148 with 4096; 1024x768 with 3000
// paths: 160, 160 and 153.
inline uint32_t fill_unit_points(uint64_t fill_points) {
    return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(fill_points / 4096u, 8u), 60u);
}
__global__ __launch_bounds__(256) void k_dedge_grad(uint32_t n_units, const GradUnit *__restrict__ units,
                                                    const uint32_t *__restrict__ path_first_pt,
                                                    const uint32_t *__restrict__ path_first_edge,
                                                    const uint32_t *__restrict__ path_stroke,
                                                    const DrawTiles *__restrict__ dts,
                                                    const uint32_t *__restrict__ cmd_of,
                                                    const RV4<float> *__restrict__ edges,
                                                    const float2 *__restrict__ nrm,
                                                    const float *__restrict__ g_cov, float4 *__restrict__ own,
                                                    float4 *__restrict__ own_n) {
    __shared__ float4 s_edge[4][64];
    __shared__ float s_sum[4][64][2];
    __shared__ uint32_t s_blocks[4][64];
    __shared__ RowShare s_rows[4];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6, u = blockIdx.x * 4u + wv;
    if (u >= n_units)
        return;
    const GradUnit gu = units[u];
    const uint32_t d = gu.path, first = path_first_pt[d], end = path_first_pt[d + 1];
    const bool stroke = path_stroke[d] != 0;
    const uint32_t per = stroke ? 10u : 1u, np = gu.n;
    const DrawTiles dt = dts[d];
    float4 *ed = s_edge[wv];
    float(*sum)[2] = s_sum[wv];
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    int32_t r0 = 1, r1 = 0;
    if (lane < np * per) {
        const RV4<float> e = edges[path_first_edge[d] + (gu.first_pt - first) * per + lane];
        v = make_float4(e.x, e.y, e.z, e.w);
        int32_t c0;
        if (dt.bw)
            dbin_range(e, dt, r0, r1, c0);
        if (r0 <= r1) {
            r0 = (int32_t)fmaxf(floorf(fminf(v.y, v.w)), (float)(dt.by0 * VKD_T));
            r1 = (int32_t)fminf(floorf(fmaxf(v.y, v.w)), (float)(dt.by1 * VKD_T + VKD_T - 1));
        }
    }
    ed[lane] = v;
    sum[lane][0] = sum[lane][1] = 0.f;
    const float lo = (float)(dt.bx0 * VKD_T), hi = (float)((dt.bx1 + 1) * VKD_T);
    // blocks of VKD_EB columns that the edge's part in a row spans at most (a column more at each end, and one for
    // rounding); the last block takes what is left
    uint32_t blocks = 1, items = 0;
    if (r0 <= r1) {
        const float dx = fabsf(v.z - v.x), w = fminf(fminf(dx, dx / fabsf(v.w - v.y)), hi - lo);
        blocks = 1u + (uint32_t)((w + 3.f) * (1.f / VKD_EB));
        items = (uint32_t)(r1 - r0 + 1) * blocks;
    }
    const bool wide = __any(blocks > 1u) != 0;
    s_blocks[wv][lane] = blocks;
    uint32_t done = 0;
    while (__any(done < items)) { // up to 16 items of every edge at a time
        const uint32_t cnt = min(items - done, (uint32_t)VKD_T);
        share_rows(s_rows[wv], lane, (int32_t)done + (wide ? 0 : r0), cnt, [&](uint32_t j, int32_t r) {
            const float4 q = ed[j];
            uint32_t b = 0, nb = 1;
            if (wide) { // item r of the edge: row r / nb, block r % nb
                nb = s_blocks[wv][j];
                const uint32_t k = (uint32_t)r / nb;
                b = (uint32_t)r - k * nb;
                r = (int32_t)fmaxf(floorf(fminf(q.y, q.w)), (float)(dt.by0 * VKD_T)) + (int32_t)k;
            }
            RowPart<float> p;
            if (!p.clip(RV4<float>{q.x, q.y, q.z, q.w}, (float)r))
                return;
            const float xa = fmaxf(p.xl, lo), xb = fminf(p.xr, hi);
            if (!(xa <= xb))
                return;
            const uint32_t *co = cmd_of + dt.pt_base + (uint32_t)(r / VKD_T - dt.by0) * dt.bw;
            int32_t cl = (int32_t)floorf(xa), cr = min((int32_t)floorf(xb), (dt.bx1 + 1) * VKD_T - 1);
            float from = p.param(xa), ga = 0.f, gb = 0.f;
            if (wide) {
                cr = b + 1 < nb ? min(cr, cl + (int32_t)(b + 1) * VKD_EB - 1) : cr;
                cl += (int32_t)b * VKD_EB;
                from = b ? p.param((float)cl) : from;
            }
            for (int32_t c = cl; c <= cr; c++) {
                const float to = p.param((float)(c + 1));
                const uint32_t cmd = co[c / VKD_T - dt.bx0];
                const float p0 = fminf(from, to), p1 = fmaxf(from, to);
                from = to;
                if (cmd == VKD_NO_CMD)
                    continue;
                const float Gv = g_cov[(size_t)cmd * 256 + (uint32_t)(r % VKD_T) * VKD_T + (uint32_t)(c % VKD_T)];
                const float I1 = 0.5f * (p1 * p1 - p0 * p0);
                const float I0 = (p1 - p0) - I1;
                ga += Gv * I0;
                gb += Gv * I1;
            }
            if (ga != 0.f || gb != 0.f) {
                atomicAdd(&sum[j][0], ga);
                atomicAdd(&sum[j][1], gb);
            }
        });
        done += cnt;
    }
    const float ga = sum[lane][0], gb = sum[lane][1], dx = v.z - v.x, dy = v.w - v.y;
    const bool any = ga != 0.f || gb != 0.f;
    const float4 ge = any ? make_float4(-dy * ga, dx * ga, -dy * gb, dx * gb) : make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t p = gu.first_pt + lane;
    if (!stroke) {
        if (lane < np)
            own[p] = ge;
        return;
    }
    ed[lane] = ge;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane >= np)
        return;
    const float4 *e = ed + 10 * lane;
    auto vertex = [&](int before, int after) { // where edge `before` ends and edge `after` begins
        return f2(e[after].x + e[before].z, e[after].y + e[before].w);
    };
    const float2 v0 = vertex(3, 0), v1 = vertex(0, 1), v2 = vertex(1, 2), v3 = vertex(2, 3);
    float2 self = f2(v0.x + v3.x, v0.y + v3.y), n_self = f2(v0.x + v1.x - v2.x - v3.x, v0.y + v1.y - v2.y - v3.y);
    float2 n_prev = f2(0.f, 0.f);
    const float2 n0 = nrm[prev_pt(p, first, end)], n1 = nrm[p];
    const bool swap = n0.x * n1.y - n0.y * n1.x > 0.f; // as in k_dedges
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const int b = 4 + 3 * s;
        const float sg = s ? -1.f : 1.f;
        const float2 t0 = vertex(b + 2, b), t1 = vertex(b, b + 1), t2 = vertex(b + 1, b + 2);
        self = f2(self.x + t0.x + t1.x + t2.x, self.y + t0.y + t1.y + t2.y);
        const float2 tp = swap ? t2 : t1, ts = swap ? t1 : t2; // on the previous normal, on this one
        n_prev = f2(n_prev.x + sg * tp.x, n_prev.y + sg * tp.y);
        n_self = f2(n_self.x + sg * ts.x, n_self.y + sg * ts.y);
    }
    own[p] = make_float4(self.x, self.y, v1.x + v2.x, v1.y + v2.y);
    own_n[p] = make_float4(n_self.x, n_self.y, n_prev.x, n_prev.y);
}

// --------------------------------------------------------------------------- chain rule
// gradient of segment a -> b's direction d through its normal n = (-d.y, d.x)/|d|:
// g_d = ((g.y, -g.x) - d (n.g)/|d|)/|d|
__device__ __forceinline__ float2 seg_grad(const float2 *pts, const float2 *nrm, float2 gn, uint32_t a, uint32_t b) {
    const float dx = pts[b].x - pts[a].x, dy = pts[b].y - pts[a].y;
    const float L = sqrtf(dx * dx + dy * dy);
    if (!(L > 0.f) || (gn.x == 0.f && gn.y == 0.f))
        return f2(0.f, 0.f);
    const float ng = nrm[a].x * gn.x + nrm[a].y * gn.y;
    return f2((gn.y - dx * ng / L) / L, (-gn.x - dy * ng / L) / L);
}

// per point p: what its own edges and the previous point's give it, plus, for strokes, the normals'
// dependence on the segments p-1 -> p and p -> p+1, and the half-width's part from normal p
__global__ void k_dg_points(uint32_t n_pts, const uint32_t *__restrict__ pt_path,
                            const uint32_t *__restrict__ path_first_pt, const uint32_t *__restrict__ path_stroke,
                            const float *__restrict__ width, const float4 *__restrict__ own,
                            const float4 *__restrict__ own_n, const float2 *__restrict__ pts,
                            const float2 *__restrict__ nrm, float2 *__restrict__ g_pt, float *__restrict__ g_hp) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_pts)
        return;
    const uint32_t path = pt_path[p];
    const uint32_t first = path_first_pt[path], end = path_first_pt[path + 1];
    const uint32_t pp = prev_pt(p, first, end), nx = next_pt(p, first, end);
    const float4 o = own[p], op = own[pp];
    float gx = op.z + o.x, gy = op.w + o.y;
    if (path_stroke[path]) {
        const float h = 0.5f * width[path];
        const float4 a = own_n[pp], b = own_n[p], c = own_n[nx];
        const float2 sp = f2(a.x + b.z, a.y + b.w), sn = f2(b.x + c.z, b.y + c.w); // sums on normals pp and p
        const float2 din = seg_grad(pts, nrm, f2(h * sp.x, h * sp.y), pp, p);  // segment pp -> p: +g_d at its end p
        const float2 dout = seg_grad(pts, nrm, f2(h * sn.x, h * sn.y), p, nx); // p -> nx: -g_d at its start p
        gx += din.x - dout.x;
        gy += din.y - dout.y;
        g_hp[p] = nrm[p].x * sn.x + nrm[p].y * sn.y;
    }
    g_pt[p] = f2(gx, gy);
}

// one thread per control point: gathers the Bernstein-weighted point gradients of its cubic(s)
__global__ void k_dg_ctrl(uint32_t n_ctrl, const uint32_t *__restrict__ ctrl_path,
                          const uint32_t *__restrict__ path_first_ctrl, const uint32_t *__restrict__ path_first_pt,
                          const uint32_t *__restrict__ path_ncubic, const float2 *__restrict__ g_pt,
                          float2 *__restrict__ g_ctrl) {
    uint32_t ci = blockIdx.x * blockDim.x + threadIdx.x;
    if (ci >= n_ctrl)
        return;
    const uint32_t path = ctrl_path[ci];
    const uint32_t local = ci - path_first_ctrl[path], n = path_ncubic[path];
    const uint32_t q = local / 3, m = local % 3;
    const float2 *gp = g_pt + path_first_pt[path];
    float gx = 0.f, gy = 0.f;
    for (int i = 0; i < VKD_NSEG; i++) {
        const float t = (float)i / (float)VKD_NSEG, u = 1.0f - t;
        const float B[4] = {u * u * u, 3.0f * u * u * t, 3.0f * u * t * t, t * t * t};
        const float2 a = gp[q * VKD_NSEG + i];
        gx += B[m] * a.x;
        gy += B[m] * a.y;
        if (m == 0) { // also the end point of the previous cubic
            const uint32_t qp = (q + n - 1) % n;
            const float2 bq = gp[qp * VKD_NSEG + i];
            gx += B[3] * bq.x;
            gy += B[3] * bq.y;
        }
    }
    g_ctrl[ci] = f2(gx, gy);
}

// one wavefront per path: colour chain c = (r a, g a, b a, a) and width = 2 h
__global__ __launch_bounds__(256) void k_dg_paths(uint32_t n_paths, const float4 *__restrict__ rgba,
                                                  const double *__restrict__ g_col, const float *__restrict__ g_hp,
                                                  const uint32_t *__restrict__ path_first_pt,
                                                  const uint32_t *__restrict__ path_stroke,
                                                  float4 *__restrict__ g_rgba, float *__restrict__ g_width) {
    const uint32_t p = blockIdx.x * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (p >= n_paths)
        return;
    float gh = 0.f;
    if (path_stroke[p])
        for (uint32_t k = path_first_pt[p] + lane; k < path_first_pt[p + 1]; k += 64)
            gh += g_hp[k];
    for (int o = 32; o > 0; o >>= 1)
        gh += __shfl_xor(gh, o);
    if (lane)
        return;
    const float4 c = rgba[p];
    const double g0 = g_col[4 * p], g1 = g_col[4 * p + 1], g2 = g_col[4 * p + 2], g3 = g_col[4 * p + 3];
    g_rgba[p] = make_float4((float)(c.w * g0), (float)(c.w * g1), (float)(c.w * g2),
                            (float)(c.x * g0 + c.y * g1 + c.z * g2 + g3));
    g_width[p] = 0.5f * gh;
}

__global__ void k_dbatches(uint32_t n_tiles, uint32_t nch, const uint32_t *__restrict__ tile_off,
                           uint32_t *__restrict__ nb) {
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n_tiles)
        nb[t] = (tile_off[(size_t)(t + 1) * nch] - tile_off[(size_t)t * nch] + VKD_B - 1) / VKD_B;
}

// the counts that the host sizes its buffers by, written to its memory
__global__ void k_dcounts(const uint32_t *a, const uint32_t *b, const uint32_t *split, uint32_t *__restrict__ out) {
    out[0] = *a;
    out[1] = b ? *b : 0u;
    for (int k = 0; k < 3; k++)
        out[2 + k] = split[k]; // workgroups, rows, eights of tiles
}

__global__ void k_dzero(uint32_t *p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = 0;
}

constexpr uint32_t VKD_LAUNCH = 1u << 23; // workgroups of 256 per launch: a grid holds fewer than 2^32 threads

struct Buf {
    void *p = nullptr;
    size_t cap = 0;
};

} // namespace

struct vkvg_diff_scene_t {
    uint32_t W = 0, H = 0, n_paths = 0, n_pts = 0, n_ctrl = 0, n_edges = 0, tilesW = 0, tilesH = 0, n_tiles = 0;
    uint32_t bin_total = 0, nch = 1, chunk = VKH_COARSE_CHUNK;
    hipStream_t stream = nullptr;
    hipEvent_t ev[4] = {};
    std::string err;
    float ms_fwd = 0, ms_bwd = 0;
    uint32_t n_segs = 0, n_cmds = 0, n_batches = 0, n_grad_units = 0;
    bool have_ckpt = false;
    Buf topology; // the static topology, whose parts follow
    Buf pt_path, ctrl_path, first_pt, first_ctrl, first_edge, ncubic, stroke, draws, tg, grad_units;
    // per call
    Buf pts, nrm, edges, pts64, nrm64, edges64, dtiles, alloc, ptiles, cmd_of, segs, units, sums, tile_cnt, tile_off, cmds,
        nbat, batch_off, ckpt, cov, tile_order, scan_tmp;
    Buf g_cov, own, own_n, g_pt, g_h, g_col;
    uint32_t *counts = nullptr; // pinned: the counts read back
};

namespace {

bool ck(vkvg_diff_scene_t *s, hipError_t e, const char *what) {
    if (e == hipSuccess)
        return true;
    s->err = std::string(what) + ": " + hipGetErrorString(e);
    return false;
}
bool ensure(vkvg_diff_scene_t *s, Buf &b, size_t bytes) {
    if (b.p && bytes <= b.cap)
        return true;
    if (b.p)
        (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
    size_t cap = bytes + bytes / 4 + 256;
    if (!ck(s, hipMalloc(&b.p, cap), "hipMalloc"))
        return false;
    b.cap = cap;
    return true;
}
template <typename T> T *P(Buf &b) { return (T *)b.p; }
bool upload(vkvg_diff_scene_t *s, Buf &b, const void *h, size_t bytes) {
    return ensure(s, b, bytes) && ck(s, hipMemcpy(b.p, h, bytes, hipMemcpyHostToDevice), "upload");
}
bool sync_counts(vkvg_diff_scene_t *s) { // after the kernel that writes s->counts
    return ck(s, hipGetLastError(), "counts") && ck(s, hipStreamSynchronize(s->stream), "sync");
}
bool scan(vkvg_diff_scene_t *s, const uint32_t *in, uint32_t n, uint32_t *out) {
    if (!ensure(s, s->scan_tmp, vkh::scan_temp_words(n) * 4))
        return false;
    vkh::scan_u32(s->stream, in, n, out, P<uint32_t>(s->scan_tmp));
    return ck(s, hipGetLastError(), "scan");
}
void zero(vkvg_diff_scene_t *s, Buf &b, size_t words) {
    if (words)
        hipLaunchKernelGGL(k_dzero, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s->stream, P<uint32_t>(b),
                           words);
}
unsigned blocks(size_t n) { return (unsigned)((n + 255) / 256); }

} // namespace

extern "C" {

VkvgDiffScene vkvg_diff_create(uint32_t width, uint32_t height, uint32_t n_paths, const uint32_t *ncubic,
                               const uint32_t *is_stroke) {
    if (!width || !height || width > 16384 || height > 16384 || !n_paths || !ncubic || !is_stroke)
        return nullptr;
    auto *s = new vkvg_diff_scene_t();
    s->W = width;
    s->H = height;
    s->n_paths = n_paths;
    s->tilesW = (width + VKD_T - 1) / VKD_T;
    s->tilesH = (height + VKD_T - 1) / VKD_T;
    s->n_tiles = s->tilesW * s->tilesH;
    std::vector<uint32_t> first_pt(n_paths + 1), first_ctrl(n_paths + 1), first_edge(n_paths + 1), pt_path, ctrl_path;
    std::vector<uint32_t> stroke(n_paths), nc(n_paths);
    uint64_t np = 0, nctl = 0, ne = 0;
    for (uint32_t i = 0; i < n_paths; i++) {
        if (ncubic[i] == 0 || ncubic[i] > (1u << 20)) {
            delete s;
            return nullptr;
        }
        first_pt[i] = (uint32_t)np;
        first_ctrl[i] = (uint32_t)nctl;
        first_edge[i] = (uint32_t)ne;
        nc[i] = ncubic[i];
        stroke[i] = is_stroke[i] ? 1u : 0u;
        uint64_t m = (uint64_t)ncubic[i] * VKD_NSEG;
        np += m;
        nctl += 3ull * ncubic[i];
        ne += stroke[i] ? 10 * m : m;
        if (np > (1u << 28) || ne > (1u << 30)) {
            delete s;
            return nullptr;
        }
        pt_path.insert(pt_path.end(), (size_t)m, i);
        ctrl_path.insert(ctrl_path.end(), 3 * (size_t)ncubic[i], i);
    }
    first_pt[n_paths] = (uint32_t)np;
    first_ctrl[n_paths] = (uint32_t)nctl;
    first_edge[n_paths] = (uint32_t)ne;
    s->n_pts = (uint32_t)np;
    s->n_ctrl = (uint32_t)nctl;
    s->n_edges = (uint32_t)ne;
    std::vector<GradUnit> gu;
    uint64_t fill_points = 0;
    for (uint32_t i = 0; i < n_paths; i++)
        fill_points += stroke[i] ? 0u : first_pt[i + 1] - first_pt[i];
    const uint32_t per_fill = fill_unit_points(fill_points);
    for (uint32_t i = 0; i < n_paths; i++) {
        const uint32_t per = stroke[i] ? 6u : per_fill;
        for (uint32_t p = first_pt[i]; p < first_pt[i + 1]; p += per)
            gu.push_back(GradUnit{p, i, std::min(per, first_pt[i + 1] - p)});
    }
    s->n_grad_units = (uint32_t)gu.size();
    // draw records for the shared tile / coarse kernels: one target, kind per path
    std::vector<vkh_draw> dr(n_paths);
    memset(dr.data(), 0, sizeof(vkh_draw) * n_paths);
    for (uint32_t i = 0; i < n_paths; i++) {
        dr[i].kind = stroke[i] ? VKH_DRAW_STROKE : VKH_DRAW_FILL_NZ;
        dr[i].target = 0;
        dr[i].grad = -1;
        dr[i].source = -1;
    }
    TargetInfo ti;
    memset(&ti, 0, sizeof(ti));
    ti.width = width;
    ti.height = height;
    ti.tilesW = s->tilesW;
    ti.tilesH = s->tilesH;
    ti.tile_base = 0;
    ti.binsW = (s->tilesW + VKH_BIN_TILES - 1) / VKH_BIN_TILES;
    ti.binsH = (s->tilesH + VKH_BIN_TILES - 1) / VKH_BIN_TILES;
    ti.bin_base = 0;
    ti.draw_begin = 0;
    ti.draw_end = n_paths;
    s->bin_total = ti.binsW * ti.binsH;
    s->chunk = vkh::coarse_chunk(n_paths, s->bin_total);
    s->nch = (n_paths + s->chunk - 1) / s->chunk;
    bool ok = ck(s, hipStreamCreate(&s->stream), "stream") &&
              ck(s, hipHostMalloc((void **)&s->counts, 64, hipHostMallocDefault), "hipHostMalloc");
    for (int k = 0; ok && k < 4; k++)
        ok = ck(s, hipEventCreate(&s->ev[k]), "event");
    // the topology in one allocation and one copy
    struct {
        Buf &b;
        const void *h;
        size_t bytes;
    } parts[] = {{s->pt_path, pt_path.data(), 4ull * np},
                 {s->ctrl_path, ctrl_path.data(), 4ull * nctl},
                 {s->first_pt, first_pt.data(), 4ull * (n_paths + 1)},
                 {s->first_ctrl, first_ctrl.data(), 4ull * (n_paths + 1)},
                 {s->first_edge, first_edge.data(), 4ull * (n_paths + 1)},
                 {s->ncubic, nc.data(), 4ull * n_paths},
                 {s->stroke, stroke.data(), 4ull * n_paths},
                 {s->draws, dr.data(), sizeof(vkh_draw) * n_paths},
                 {s->tg, &ti, sizeof(ti)},
                 {s->grad_units, gu.data(), sizeof(GradUnit) * gu.size()}};
    size_t bytes = 0;
    for (auto &x : parts)
        bytes += (x.bytes + 255) & ~(size_t)255;
    std::vector<char> blob(bytes);
    bytes = 0;
    for (auto &x : parts) {
        memcpy(blob.data() + bytes, x.h, x.bytes);
        bytes += (x.bytes + 255) & ~(size_t)255;
    }
    ok = ok && upload(s, s->topology, blob.data(), bytes);
    bytes = 0;
    for (auto &x : parts) {
        x.b.p = s->topology.p ? (char *)s->topology.p + bytes : nullptr;
        bytes += (x.bytes + 255) & ~(size_t)255;
    }
    ok = ok &&
         ensure(s, s->pts, 8ull * np) && ensure(s, s->nrm, 8ull * np) && ensure(s, s->edges, 16ull * ne) &&
         ensure(s, s->dtiles, sizeof(DrawTiles) * n_paths) && ensure(s, s->alloc, 16 + sizeof(PathAlloc) * n_paths) &&
         ensure(s, s->segs, 4096) && ensure(s, s->tile_cnt, 4ull * ((size_t)s->n_tiles * s->nch + 1)) &&
         ensure(s, s->tile_off, 4ull * ((size_t)s->n_tiles * s->nch + 1)) &&
         ensure(s, s->nbat, 4ull * (s->n_tiles + 1)) && ensure(s, s->batch_off, 4ull * (s->n_tiles + 1)) &&
         ensure(s, s->own, 16ull * np) && ensure(s, s->own_n, 16ull * np) && ensure(s, s->g_pt, 8ull * np) &&
         ensure(s, s->g_h, 4ull * np) && ensure(s, s->g_col, 32ull * n_paths);
    if (!ok) {
        fprintf(stderr, "vkvg_diff_create: %s\n", s->err.c_str());
        vkvg_diff_destroy(s);
        return nullptr;
    }
    return s;
}

void vkvg_diff_destroy(VkvgDiffScene s) {
    if (!s)
        return;
    if (s->stream)
        (void)hipStreamSynchronize(s->stream);
    Buf *bufs[] = {&s->topology, &s->pts, &s->nrm, &s->edges, &s->pts64, &s->nrm64, &s->edges64,
                   &s->dtiles, &s->alloc, &s->ptiles, &s->cmd_of, &s->segs, &s->units, &s->sums, &s->tile_cnt, &s->tile_off,
                   &s->cmds, &s->nbat, &s->batch_off, &s->ckpt, &s->cov, &s->tile_order, &s->scan_tmp, &s->g_cov,
                   &s->own, &s->own_n, &s->g_pt, &s->g_h, &s->g_col};
    for (Buf *b : bufs)
        if (b->p)
            (void)hipFree(b->p);
    if (s->counts)
        (void)hipHostFree(s->counts);
    for (int k = 0; k < 4; k++)
        if (s->ev[k])
            (void)hipEventDestroy(s->ev[k]);
    if (s->stream)
        (void)hipStreamDestroy(s->stream);
    delete s;
}

} // extern "C"

template <typename R>
static int forward_impl(VkvgDiffScene s, const float *ctrl, const float *rgba, const float *width, RV4<R> *image,
                        int keep, Buf &pts, Buf &nrm, Buf &edges) {
    if (!ctrl || !rgba || !width || !image) {
        s->err = "null pointer";
        return -1;
    }
    hipStream_t st = s->stream;
    s->have_ckpt = false;
    if (!ensure(s, pts, 2 * sizeof(R) * (size_t)s->n_pts) || !ensure(s, nrm, 2 * sizeof(R) * (size_t)s->n_pts) ||
        !ensure(s, edges, 4 * sizeof(R) * (size_t)s->n_edges))
        return -1;
    if (!ck(s, hipEventRecord(s->ev[0], st), "event"))
        return -1;
    const uint32_t np = s->n_pts, nd = s->n_paths;
    uint32_t *n_split = P<uint32_t>(s->alloc); // counters of split rows, then the paths' records
    PathAlloc *alloc = (PathAlloc *)(n_split + 4);
    hipLaunchKernelGGL(k_dflatten<R>, dim3(blocks(np)), dim3(256), 0, st, np, P<uint32_t>(s->pt_path),
                       P<uint32_t>(s->first_pt), P<uint32_t>(s->first_ctrl), P<uint32_t>(s->ncubic),
                       (const float2 *)ctrl, P<RV2<R>>(pts));
    hipLaunchKernelGGL(k_dnormals<R>, dim3(blocks(np)), dim3(256), 0, st, np, P<uint32_t>(s->pt_path),
                       P<uint32_t>(s->first_pt), P<RV2<R>>(pts), P<RV2<R>>(nrm));
    hipLaunchKernelGGL(k_dedges<R>, dim3(blocks(np)), dim3(256), 0, st, np, P<uint32_t>(s->pt_path),
                       P<uint32_t>(s->first_pt), P<uint32_t>(s->first_edge), P<uint32_t>(s->stroke), width,
                       P<RV2<R>>(pts), P<RV2<R>>(nrm), P<RV4<R>>(edges));
    hipLaunchKernelGGL(k_dpaths<R>, dim3(nd), dim3(256), 0, st, P<uint32_t>(s->first_edge), P<RV4<R>>(edges),
                       (int32_t)s->tilesW, (int32_t)s->tilesH, P<DrawTiles>(s->dtiles), alloc);
    hipLaunchKernelGGL(k_dalloc, dim3(1), dim3(1024), 0, st, nd, alloc, P<DrawTiles>(s->dtiles), n_split, s->counts);
    if (!sync_counts(s))
        return -1;
    const uint32_t n_ptiles = s->counts[0], n_units = s->counts[1];
    s->n_segs = s->counts[2];
    if (!ensure(s, s->ptiles, sizeof(PathTile) * ((size_t)n_ptiles + 1)) ||
        !ensure(s, s->cmd_of, 4ull * ((size_t)n_ptiles + 1)) ||
        !ensure(s, s->units, (sizeof(RowUnit) + sizeof(SplitRow)) * ((size_t)n_units + 1)) ||
        !ensure(s, s->segs, 4ull * ((size_t)s->n_segs + 1)))
        return -1;
    SplitRow *splits = (SplitRow *)(P<RowUnit>(s->units) + n_units + 1);
    hipLaunchKernelGGL(k_dbin<R>, dim3(nd), dim3(256), 0, st, P<uint32_t>(s->first_edge), P<RV4<R>>(edges),
                       P<DrawTiles>(s->dtiles), alloc, P<PathTile>(s->ptiles),
                       P<uint32_t>(s->cmd_of), P<uint32_t>(s->segs), P<RowUnit>(s->units), splits,
                       (unsigned long long *)n_split, n_split + 2, split_steps(n_ptiles, n_units, s->n_segs));
    const uint32_t n_tc = s->n_tiles * s->nch;
    const bool keep_ckpt = keep && sizeof(R) == sizeof(float);
    zero(s, s->tile_cnt, n_tc + 1);
    vkh::launch_coarse(st, false, s->bin_total, s->nch, s->chunk, P<TargetInfo>(s->tg), 1, P<vkh_draw>(s->draws),
                       P<DrawTiles>(s->dtiles), P<PathTile>(s->ptiles), P<uint32_t>(s->tile_cnt), nullptr, nullptr);
    if (!scan(s, P<uint32_t>(s->tile_cnt), n_tc, P<uint32_t>(s->tile_off)))
        return -1;
    if (keep_ckpt) {
        hipLaunchKernelGGL(k_dbatches, dim3(blocks(s->n_tiles)), dim3(256), 0, st, s->n_tiles, s->nch,
                           P<uint32_t>(s->tile_off), P<uint32_t>(s->nbat));
        if (!scan(s, P<uint32_t>(s->nbat), s->n_tiles, P<uint32_t>(s->batch_off)))
            return -1;
    }
    hipLaunchKernelGGL(k_dcounts, dim3(1), dim3(1), 0, st, P<uint32_t>(s->tile_off) + n_tc,
                       keep_ckpt ? P<uint32_t>(s->batch_off) + s->n_tiles : nullptr, n_split, s->counts);
    if (!sync_counts(s))
        return -1;
    s->n_cmds = s->counts[0];
    const uint32_t split_groups = s->counts[2], split_rows = s->counts[3];
    const size_t sum_words = (size_t)s->counts[4] * (VKD_T * VKD_LD) * (sizeof(R) / 4);
    float4 *ck_ptr = nullptr;
    if (keep_ckpt) {
        s->n_batches = s->counts[1];
        if (!ensure(s, s->ckpt, 16ull * 256 * ((size_t)s->n_batches + 1)))
            return -1;
        ck_ptr = P<float4>(s->ckpt);
    }
    if (!ensure(s, s->cmds, sizeof(Cmd) * ((size_t)s->n_cmds + 1)) ||
        !ensure(s, s->cov, sizeof(R) * 256 * ((size_t)s->n_cmds + 1)) ||
        (sum_words && !ensure(s, s->sums, 4 * sum_words)))
        return -1;
    vkh::launch_coarse(st, true, s->bin_total, s->nch, s->chunk, P<TargetInfo>(s->tg), 1, P<vkh_draw>(s->draws),
                       P<DrawTiles>(s->dtiles), P<PathTile>(s->ptiles), nullptr, P<uint32_t>(s->tile_off),
                       P<Cmd>(s->cmds));
    if (s->n_cmds) {
        hipLaunchKernelGGL(k_dcmd_of, dim3(blocks(s->n_cmds)), dim3(256), 0, st, s->n_cmds, P<Cmd>(s->cmds),
                           P<uint32_t>(s->cmd_of));
        for (uint32_t u0 = 0; u0 < n_units; u0 += VKD_LAUNCH)
            hipLaunchKernelGGL(k_dcov<R>, dim3(std::min(n_units - u0, VKD_LAUNCH)), dim3(256), 0, st,
                               P<RowUnit>(s->units) + u0, P<DrawTiles>(s->dtiles), P<PathTile>(s->ptiles),
                               P<uint32_t>(s->cmd_of), P<uint32_t>(s->segs), P<RV4<R>>(edges), P<R>(s->cov));
    }
    if (s->n_cmds && split_rows) {
        zero(s, s->sums, sum_words);
        for (uint32_t g0 = 0; g0 < split_groups; g0 += VKD_LAUNCH)
            hipLaunchKernelGGL(k_dcov_split<R>, dim3(std::min(split_groups - g0, VKD_LAUNCH)), dim3(256), 0, st, splits,
                               split_rows, g0, P<RowUnit>(s->units), P<DrawTiles>(s->dtiles), P<PathTile>(s->ptiles),
                               P<uint32_t>(s->segs), P<RV4<R>>(edges), P<R>(s->sums));
        hipLaunchKernelGGL(k_dcov_sum<R>, dim3(split_rows), dim3(256), 0, st, splits, P<RowUnit>(s->units),
                           P<DrawTiles>(s->dtiles), P<uint32_t>(s->cmd_of), P<R>(s->sums), P<R>(s->cov));
    }
    // tiles heaviest first (commands per tile vary several-fold), for compositing and the backward
    if (!ensure(s, s->tile_order, 4ull * vkh::order_words(s->n_tiles)))
        return -1;
    vkh::launch_tile_order(st, s->n_tiles, s->nch, P<uint32_t>(s->tile_off), P<uint32_t>(s->tile_order));
    hipLaunchKernelGGL(k_dcomp<R>, dim3(s->n_tiles), dim3(256), 0, st, s->W, s->H, s->tilesW, s->nch,
                       P<uint32_t>(s->tile_off), P<Cmd>(s->cmds), P<R>(s->cov), (const float4 *)rgba, image, ck_ptr,
                       P<uint32_t>(s->batch_off), P<uint32_t>(s->tile_order));
    if (!ck(s, hipGetLastError(), "forward launch") || !ck(s, hipEventRecord(s->ev[1], st), "event") ||
        !ck(s, hipStreamSynchronize(st), "forward"))
        return -1;
    (void)hipEventElapsedTime(&s->ms_fwd, s->ev[0], s->ev[1]);
    s->have_ckpt = ck_ptr != nullptr;
    return 0;
}

extern "C" {

int vkvg_diff_forward(VkvgDiffScene s, const float *ctrl, const float *rgba, const float *width, float *image,
                      int keep) {
    if (!s)
        return -1;
    return forward_impl<float>(s, ctrl, rgba, width, (RV4<float> *)image, keep, s->pts, s->nrm, s->edges);
}

int vkvg_diff_forward_f64(VkvgDiffScene s, const float *ctrl, const float *rgba, const float *width,
                          double *image) {
    if (!s)
        return -1;
    return forward_impl<double>(s, ctrl, rgba, width, (RV4<double> *)image, 0, s->pts64, s->nrm64, s->edges64);
}

int vkvg_diff_backward(VkvgDiffScene s, const float *ctrl, const float *rgba, const float *width,
                       const float *grad_image, float *grad_ctrl, float *grad_rgba, float *grad_width) {
    if (!s)
        return -1;
    if (!s->have_ckpt) {
        s->err = "backward needs a preceding forward with keep != 0";
        return -1;
    }
    if (!ctrl || !rgba || !width || !grad_image || !grad_ctrl || !grad_rgba || !grad_width) {
        s->err = "null pointer";
        return -1;
    }
    (void)ctrl;
    hipStream_t st = s->stream;
    if (!ck(s, hipEventRecord(s->ev[2], st), "event"))
        return -1;
    if (!ensure(s, s->g_cov, 4ull * 256 * ((size_t)s->n_cmds + 1)))
        return -1;
    zero(s, s->g_col, 8ull * s->n_paths);
    hipLaunchKernelGGL(k_dback, dim3(s->n_tiles), dim3(256), 0, st, s->W, s->H, s->tilesW, s->nch,
                       P<uint32_t>(s->tile_off), P<Cmd>(s->cmds), (const float4 *)rgba, (const float4 *)grad_image,
                       P<float4>(s->ckpt), P<uint32_t>(s->batch_off), P<float>(s->cov), P<float>(s->g_cov),
                       P<double>(s->g_col), P<uint32_t>(s->tile_order));
    hipLaunchKernelGGL(k_dedge_grad, dim3((s->n_grad_units + 3) / 4), dim3(256), 0, st, s->n_grad_units,
                       P<GradUnit>(s->grad_units), P<uint32_t>(s->first_pt), P<uint32_t>(s->first_edge),
                       P<uint32_t>(s->stroke), P<DrawTiles>(s->dtiles), P<uint32_t>(s->cmd_of),
                       P<RV4<float>>(s->edges), P<float2>(s->nrm), P<float>(s->g_cov), P<float4>(s->own),
                       P<float4>(s->own_n));
    hipLaunchKernelGGL(k_dg_points, dim3(blocks(s->n_pts)), dim3(256), 0, st, s->n_pts, P<uint32_t>(s->pt_path),
                       P<uint32_t>(s->first_pt), P<uint32_t>(s->stroke), width, P<float4>(s->own),
                       P<float4>(s->own_n), P<float2>(s->pts), P<float2>(s->nrm), P<float2>(s->g_pt),
                       P<float>(s->g_h));
    hipLaunchKernelGGL(k_dg_ctrl, dim3(blocks(s->n_ctrl)), dim3(256), 0, st, s->n_ctrl, P<uint32_t>(s->ctrl_path),
                       P<uint32_t>(s->first_ctrl), P<uint32_t>(s->first_pt), P<uint32_t>(s->ncubic),
                       P<float2>(s->g_pt), (float2 *)grad_ctrl);
    hipLaunchKernelGGL(k_dg_paths, dim3((s->n_paths + 3) / 4), dim3(256), 0, st, s->n_paths, (const float4 *)rgba,
                       P<double>(s->g_col), P<float>(s->g_h), P<uint32_t>(s->first_pt), P<uint32_t>(s->stroke),
                       (float4 *)grad_rgba, grad_width);
    if (!ck(s, hipGetLastError(), "backward launch") || !ck(s, hipEventRecord(s->ev[3], st), "event") ||
        !ck(s, hipStreamSynchronize(st), "backward"))
        return -1;
    (void)hipEventElapsedTime(&s->ms_bwd, s->ev[2], s->ev[3]);
    return 0;
}

float vkvg_diff_last_ms(VkvgDiffScene s, int backward) { return s ? (backward ? s->ms_bwd : s->ms_fwd) : 0.f; }

void vkvg_diff_stats(VkvgDiffScene s, uint32_t out[4]) {
    if (!s || !out)
        return;
    out[0] = s->n_edges;
    out[1] = s->n_segs;
    out[2] = s->n_cmds;
    out[3] = s->n_batches;
}

const char *vkvg_diff_last_error(VkvgDiffScene s) { return s ? s->err.c_str() : "null scene"; }

} // extern "C"
