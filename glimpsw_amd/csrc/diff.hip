// Differentiable texture-sampling resolve for gfx950.
//
// Forward: per covered pixel, the surface from the vis-buffer key, the
// triangle's barycentrics (IntersectTriangle's formula with correctly
// rounded divisions; coverage and barycentrics are constants of the pass),
// then
//   U,V = uv_0 + b1 (uv_1 - uv_0) + b2 (uv_2 - uv_0)
//   col = color_0 + b1 (color_1 - color_0) + b2 (color_2 - color_0)
//   out = Sample(U, V) * col
// with fp32 texel mip chains. Sample keeps the resolve sampler's choices
// (Texture.h:412-459, SurfaceSampler of Shading.cpp:6-10): mip level from the
// UV gradients, one filter per 4x4 tile (any minified pixel -> nearest texel
// of level clamp(mip), else bilinear at level 0), Repeat wrap; the bilinear
// weights are continuous (texel centres at +0.5, clamped at the edges) so
// that the output is differentiable in U and V.
//
// Backward: one pass over the pixels (k_diff_pixels) splits the gradient in
// two.
//
// Vertices. A block covers 16x16 pixels of one view; each of its waves sums,
// per triangle it shows (a run), the 18 products of barycentric weight and
// (dL/dcol, dL/dU, dL/dV) over the run's pixels in lane order, and marks in
// which cells of a grid of up to 16x16 over the view each of its meshlets shows.
// k_diff_vertices walks a meshlet's marked cells in order, adds the meshlet's
// runs per triangle and then the triangles' corners per vertex; a meshlet of
// many cells is split into parts, added in order by the last one to finish.
//
// Texels. Each pixel leaves one record: its base texel (the cell's corner, or
// the nearest texel), dL/dsample and the cell position. The pixels are sorted
// by base texel with a stable radix sort; every run of equal texels is summed
// in pixel order into the four corners of its cell, in 256-record tiles by
// one thread per run piece, then across tiles in tile order. No two cells
// share a corner of the same kind, so four passes add the corners to the
// gradients, one kind at a time, without conflicts. Where the texel ranges of
// two textures overlap and are not the same range, a base texel does not name
// a cell: the pixels are then sorted and summed once per corner, by the
// corner's own texel (backward of three 1280x720 views 630 -> 1,250 us).
//
// The order of every floating-point addition depends only on the inputs, so
// the gradients are bitwise reproducible; no floating-point atomics are used.
#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/iterator/counting_iterator.hpp>

#include "diff.h"
#include "surface.h"

namespace glimp {
namespace {

constexpr uint32_t kTile = 256;

struct PixelState {
    bool active;
    uint32_t mi, tri, vi[3];
    float b1, b2, U, V;
    int32_t tex, level;
    bool linear;
    float fu, fv;                  // U, V minus their wrap period
    int32_t tx, ty;
    bool cx, cy, ex, ey;
    float xs, ys;
};

__device__ __forceinline__ const DiffView& view_at(const DiffParams& p, uint32_t v) {
    return p.views ? p.views[v] : p.view;
}

// View owning global pixel slot t.
__device__ __forceinline__ uint32_t view_of_pixel(const DiffParams& p, uint32_t t) {
    uint32_t lo = 0, hi = p.num_views;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (view_at(p, mid).pixel_base <= t) lo = mid; else hi = mid;
    }
    return lo;
}

// Pixel slot t of the global numbering: its view, and the pixel's row-major
// index and 4x4-tiled index inside that view (slots run over the tiles).
struct PixelSlot {
    uint32_t view, x, y, tiled;
    bool inside;
};

__device__ __forceinline__ PixelSlot pixel_slot(const DiffParams& p, uint32_t t) {
    PixelSlot s;
    s.inside = t < p.total_pixels;
    s.view = s.inside ? view_of_pixel(p, t) : 0;
    const DiffView& V = view_at(p, s.view);
    s.tiled = t - (s.inside ? V.pixel_base : t);
    const uint32_t W = (uint32_t)V.width;
    const uint32_t tile = s.tiled >> 4, q = s.tiled & 15u, tilesX = W / 4;
    uint32_t tx;
    const uint32_t ty = div_small(tile, tilesX, tx);
    s.x = tx * 4 + (q & 3u);
    s.y = ty * 4 + (q >> 2);
    return s;
}

// Pixel of thread `tid` of 16x16-pixel block b: 16 lanes are one 4x4 tile, a
// wave 8x8 pixels (a compact area shows the fewest triangles).
__device__ __forceinline__ PixelSlot block_slot(const DiffParams& p, uint32_t b, uint32_t tid, uint32_t& bx,
                                                uint32_t& by) {
    uint32_t lo = 0, hi = p.num_views;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (view_at(p, mid).block_base <= b) lo = mid; else hi = mid;
    }
    const DiffView& V = view_at(p, lo);
    by = (b - V.block_base) / V.blocks_x;
    bx = (b - V.block_base) - by * V.blocks_x;
    const uint32_t tile = tid >> 4, q = tid & 15u;
    PixelSlot s;
    s.view = lo;
    s.x = bx * 16 + ((tile >> 2) & 1u) * 8 + (tile & 1u) * 4 + (q & 3u);
    s.y = by * 16 + (tile >> 3) * 8 + ((tile >> 1) & 1u) * 4 + (q >> 2);
    s.inside = s.x < (uint32_t)V.width && s.y < (uint32_t)V.height;
    s.tiled = s.inside ? ((s.x & ~3u) << 2) + (s.y & ~3u) * (uint32_t)V.width + q : 0u;
    return s;
}

// Surface, barycentrics and sampler choices of pixel slot t (tiled order:
// 16 lanes = one 4x4 tile of one view). Every lane of the wave must call it.
__device__ void diff_pixel(const DiffParams& p, const PixelSlot& ps, PixelState& S) {
    const DiffView& VW = view_at(p, ps.view);
    const bool inside = ps.inside;
    const uint32_t x = ps.x, y = ps.y;
    const uint32_t lane = __lane_id();
    const unsigned long long groupMask = 0xFFFFull << (lane & 48u);
    const ApproxTables& T = p.tables;

    const unsigned long long key = inside ? VW.keys[ps.tiled] : VW.clear_key;
    const bool active = inside && !(bitsf((uint32_t)(key >> 32)) <= 0.0f);
    S.active = active;
    S.tex = -1;
    S.level = 0;
    S.linear = false;
    S.b1 = S.b2 = S.U = S.V = 0.0f;
    float gradU[2] = { 0, 0 }, gradV[2] = { 0, 0 };
    uint32_t material = 0xFFFFFFFFu;
    if (active) {
        uint32_t tri;
        decode_surface(key, VW.draws, VW.num_draws, S.mi, tri);
        S.tri = tri;
        const uint32_t corners = p.m.triangles[(size_t)S.mi * 128 + tri];
        float c[3][4], uv[3][2];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const uint32_t vi = (corners >> (8 * k)) & 255u;
            S.vi[k] = vi;
            const float4 v = p.m.vertices[(size_t)S.mi * 64 + vi];
#pragma unroll
            for (int j = 0; j < 4; j++) c[k][j] = xform(VW.object_to_clip, j, v.x, v.y, v.z);
            const float2 t2 = p.uv[(size_t)S.mi * 64 + vi];
            uv[k][0] = t2.x;
            uv[k][1] = t2.y;
        }
        material = p.m.material_id[S.mi];
        const float su = __builtin_fmaf((float)(int32_t)x, VW.scale_x, VW.center_x);
        const float sv = __builtin_fmaf((float)(int32_t)y, VW.scale_y, VW.center_y);
        float bary[3], ddx[3], ddy[3];
        intersect_triangle<true>(T, c, su, sv, VW.kx, VW.ky, bary, ddx, ddy);
        S.b1 = bary[1];
        S.b2 = bary[2];
        const float t10x = uv[1][0] - uv[0][0], t10y = uv[1][1] - uv[0][1];
        const float t20x = uv[2][0] - uv[0][0], t20y = uv[2][1] - uv[0][1];
        S.U = __builtin_fmaf(bary[2], t20x, __builtin_fmaf(bary[1], t10x, uv[0][0]));
        S.V = __builtin_fmaf(bary[2], t20y, __builtin_fmaf(bary[1], t10y, uv[0][1]));
        gradU[0] = __builtin_fmaf(t20x, ddx[2], t10x * ddx[1]);
        gradV[0] = __builtin_fmaf(t20y, ddx[2], t10y * ddx[1]);
        gradU[1] = __builtin_fmaf(t20x, ddy[2], t10x * ddy[1]);
        gradV[1] = __builtin_fmaf(t20y, ddy[2], t10y * ddy[1]);
    }

    // material waterfall per 4x4 tile with the tile-wide filter vote
    bool done = !active || material == 0xFFFFFFFFu || material >= p.num_materials;
    for (;;) {
        const unsigned long long todo = __ballot(!done);
        if (!todo) break;
        const unsigned long long mine = todo & groupMask;
        const uint32_t leader = mine ? (uint32_t)__ffsll((long long)mine) - 1 : lane;
        const uint32_t lmat = __shfl(material, (int)leader);
        int32_t texIdx = -1;
        if (mine) texIdx = p.materials[lmat].texture;
        if (texIdx >= (int32_t)p.num_textures) texIdx = -1;
        int32_t mip = -64;
        uint32_t TW = 1, TH = 1, TL = 1;
        if (texIdx >= 0) {
            const DiffTex& D = p.textures[texIdx];
            TW = D.width;
            TH = D.height;
            TL = D.levels;
            const float su2 = (float)TW * (float)TW, sv2 = (float)TH * (float)TH;
            const float dx = __builtin_fmaf(gradU[0], gradU[0], gradV[0] * gradV[0]) * su2;
            const float dy = __builtin_fmaf(gradU[1], gradU[1], gradV[1] * gradV[1]) * sv2;
            const float mx = (dx > dy) ? dx : dy;
            mip = (int32_t)(fbits(mx) - (127u << 23)) >> 24;
        }
        const unsigned long long vote = __ballot(active && mip > 0);
        const bool minify = (vote & groupMask) != 0;
        if (!done && material == lmat) {
            done = true;
            if (texIdx >= 0) {
                S.tex = texIdx;
                S.linear = !minify;
                const float floorU = floorf(S.U), floorV = floorf(S.V);
                S.fu = S.U - floorU;
                S.fv = S.V - floorV;
                if (S.linear) {
                    S.level = 0;
                    S.xs = S.fu * (float)TW - 0.5f;
                    S.ys = S.fv * (float)TH - 0.5f;
                    S.cx = S.xs > 0.0f;
                    S.cy = S.ys > 0.0f;
                    const float xf = S.cx ? S.xs : 0.0f, yf = S.cy ? S.ys : 0.0f;
                    S.tx = (int32_t)xf;
                    S.ty = (int32_t)yf;
                    S.ex = S.tx < (int32_t)TW - 1;
                    S.ey = S.ty < (int32_t)TH - 1;
                    if (!S.ex) S.tx = (int32_t)TW - 1;
                    if (!S.ey) S.ty = (int32_t)TH - 1;
                } else {
                    const int32_t m = min(max(mip, 0), (int32_t)TL - 1);
                    S.level = m;
                    const int32_t Wm = (int32_t)(TW >> m), Hm = (int32_t)(TH >> m);
                    S.tx = min((int32_t)(S.fu * (float)Wm), Wm - 1);
                    S.ty = min((int32_t)(S.fv * (float)Hm), Hm - 1);
                }
            }
        }
    }
}

// Sample value, its texels and weights, and its U/V derivatives.
struct SampleEval {
    float4 val, du, dv;
    uint64_t texel[4];
    float fx, fy;
    int n;
};

__device__ __forceinline__ float4 f4(float a) { return make_float4(a, a, a, a); }
__device__ __forceinline__ float4 operator-(float4 a, float4 b) { return make_float4(a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w); }
__device__ __forceinline__ float4 operator*(float s, float4 a) { return make_float4(s * a.x, s * a.y, s * a.z, s * a.w); }
__device__ __forceinline__ float4 operator*(float4 a, float4 b) { return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w); }
__device__ __forceinline__ float4 fma4(float s, float4 a, float4 b) {
    return make_float4(__builtin_fmaf(s, a.x, b.x), __builtin_fmaf(s, a.y, b.y), __builtin_fmaf(s, a.z, b.z),
                       __builtin_fmaf(s, a.w, b.w));
}
__device__ __forceinline__ float4 add4(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }
__device__ __forceinline__ float dot4(float4 a, float4 b) {
    return __builtin_fmaf(a.x, b.x, __builtin_fmaf(a.y, b.y, __builtin_fmaf(a.z, b.z, a.w * b.w)));
}

__device__ void sample_eval(const DiffParams& p, const PixelState& S, SampleEval& E) {
    E.n = 0;
    E.du = E.dv = f4(0.0f);
    if (S.tex < 0) {
        E.val = f4(1.0f);
        return;
    }
    const DiffTex& D = p.textures[S.tex];
    const uint64_t base = D.level_offset[S.level];
    if (!S.linear) {
        const uint64_t Wm = D.width >> S.level;
        E.n = 1;
        E.texel[0] = base + (uint64_t)S.ty * Wm + (uint64_t)S.tx;
        E.val = p.texels[E.texel[0]];
        return;
    }
    const float xf = S.cx ? S.xs : 0.0f, yf = S.cy ? S.ys : 0.0f;
    const float fx = S.ex ? xf - (float)S.tx : 0.0f, fy = S.ey ? yf - (float)S.ty : 0.0f;
    const uint64_t x0 = (uint64_t)S.tx, y0 = (uint64_t)S.ty;
    const uint64_t x1 = S.ex ? x0 + 1 : x0, y1 = S.ey ? y0 + 1 : y0;
    E.n = 4;
    E.texel[0] = base + y0 * D.width + x0;
    E.texel[1] = base + y0 * D.width + x1;
    E.texel[2] = base + y1 * D.width + x0;
    E.texel[3] = base + y1 * D.width + x1;
    E.fx = fx;
    E.fy = fy;
    const float gx = 1.0f - fx, gy = 1.0f - fy;
    const float4 t00 = p.texels[E.texel[0]], t10 = p.texels[E.texel[1]];
    const float4 t01 = p.texels[E.texel[2]], t11 = p.texels[E.texel[3]];
    const float4 d0 = t10 - t00, d1 = t11 - t01;
    const float4 l0 = fma4(fx, d0, t00), l1 = fma4(fx, d1, t01);
    E.val = fma4(fy, l1 - l0, l0);
    const float sx = (S.cx && S.ex) ? (float)D.width : 0.0f, sy = (S.cy && S.ey) ? (float)D.height : 0.0f;
    E.du = sx * add4(gy * d0, fy * d1);
    E.dv = sy * (l1 - l0);
}

__device__ __forceinline__ float4 vertex_color(const DiffParams& p, const PixelState& S) {
    const float4* C = p.color + (size_t)S.mi * 64;
    const float4 c0 = C[S.vi[0]], c1 = C[S.vi[1]], c2 = C[S.vi[2]];
    return fma4(S.b2, c2 - c0, fma4(S.b1, c1 - c0, c0));
}

__device__ __forceinline__ size_t out_index(const DiffParams& p, const PixelSlot& ps) {
    const DiffView& V = view_at(p, ps.view);
    return (size_t)V.pixel_base + (size_t)ps.y * (uint32_t)V.width + ps.x;
}

__global__ void __launch_bounds__(256) k_diff_forward(DiffParams p) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const PixelSlot ps = pixel_slot(p, t);
    PixelState S;
    diff_pixel(p, ps, S);
    if (!ps.inside) return;
    float4 o = f4(0.0f);
    if (S.active) {
        SampleEval E;
        sample_eval(p, S, E);
        o = E.val * vertex_color(p, S);
    }
    p.out[out_index(p, ps)] = o;
}

// ---------------------------------------------------------------- backward: pixels

constexpr uint32_t kBlockRuns = 256;   // most runs of a block of pixels: 64 a wave
constexpr uint32_t kRunSums = 18;      // 3 corners x (colour, U, V)
constexpr uint32_t kSplitParts = 32768;        // most parts beyond one per meshlet
constexpr uint32_t kPartGrid = 2048;   // 8 blocks a CU
constexpr uint32_t kFillParts = 1024;

// Texel record flags
constexpr uint32_t kTexLinear = 1u, kTexRight = 2u, kTexBelow = 4u;

// Bound by the surface evaluation, as k_diff_forward, and 36 bytes a pixel of
// texel records: 130 us for 2.76 M pixels of three 1280x720 views (forward
// 67). Four texel and three vertex records a pixel, 188 bytes, took 233 us.
// Run sums are per wave, not per block: a block-wide set of triangles cost
// four barriers and a hash table (193 us). Growing a rectangle per meshlet
// with atomic minima instead of marking cells took 177 us: the large
// meshlets' corners are contended.
__global__ void __launch_bounds__(256) k_diff_pixels(DiffParams p) {
    __shared__ float s_val[8][256];              // b1, b2, gcol, gU, gV per pixel
    __shared__ unsigned long long s_mask[kBlockRuns];      // a run's pixels in its wave
    __shared__ uint32_t s_mesh[kBlockRuns], s_pos[kBlockRuns], s_count[4];
    __shared__ uint8_t s_tri[kBlockRuns];
    const uint32_t tid = threadIdx.x, lane = __lane_id(), wid = tid >> 6;
    uint32_t bx, by;
    const PixelSlot ps = block_slot(p, blockIdx.x, tid, bx, by);
    PixelState S;
    diff_pixel(p, ps, S);
    if (ps.inside) {
        const DiffView& V = view_at(p, ps.view);
        const size_t t = (size_t)V.pixel_base + ps.tiled;
        uint32_t texel = p.tex_sentinel;
        if (S.active) {
            SampleEval E;
            sample_eval(p, S, E);
            const float4 g = p.grad_out[out_index(p, ps)];
            const float4 gval = g * vertex_color(p, S);
            const float4 gcol = g * E.val;
            if (E.n) {
                texel = (uint32_t)E.texel[0];
                uint32_t code = 0, width = 0;
                float fx = 0.0f, fy = 0.0f;
                if (E.n == 4) {
                    code = kTexLinear | (S.ex ? kTexRight : 0u) | (S.ey ? kTexBelow : 0u);
                    width = p.textures[S.tex].width;
                    fx = E.fx;
                    fy = E.fy;
                }
                p.tex_recs[2 * t] = gval;
                p.tex_recs[2 * t + 1] = make_float4(fx, fy, __uint_as_float(code), __uint_as_float(width));
            }
            s_val[0][tid] = S.b1;
            s_val[1][tid] = S.b2;
            s_val[2][tid] = gcol.x;
            s_val[3][tid] = gcol.y;
            s_val[4][tid] = gcol.z;
            s_val[5][tid] = gcol.w;
            s_val[6][tid] = dot4(gval, E.du);
            s_val[7][tid] = dot4(gval, E.dv);
        }
        p.tex_keys[t] = texel;
    }
    // the wave's pixels of each triangle: the first of them holds the mask
    const bool active = S.active;          // only inside the view
    unsigned long long todo = __ballot(active), mine = 0;
    while (todo) {
        const int l = __builtin_ctzll(todo);
        const uint32_t m0 = (uint32_t)__builtin_amdgcn_readlane((int)S.mi, l);
        const uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane((int)S.tri, l);
        const unsigned long long m = __ballot(active && S.mi == m0 && S.tri == t0);
        if (lane == (uint32_t)l) mine = m;
        todo &= ~m;
    }
    // the wave's runs in the order of their first pixels, the waves' one after another
    const unsigned long long leaders = __ballot(mine != 0);
    const uint32_t own = (uint32_t)__popcll(leaders);
    if (lane == 0) s_count[wid] = own;
    __syncthreads();
    uint32_t first = 0, runs = 0;
#pragma unroll
    for (uint32_t w = 0; w < 4; w++) {
        if (w < wid) first += s_count[w];
        runs += s_count[w];
    }
    if (mine) {
        const uint32_t r = first + (uint32_t)__popcll(leaders & ((1ull << lane) - 1ull));
        s_mask[r] = mine;
        s_mesh[r] = S.mi;
        s_tri[r] = (uint8_t)S.tri;
    }
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * kBlockRuns;
    if (tid == 0) p.block_runs[blockIdx.x] = runs;
    if (tid < runs) {
        // runs are kept by meshlet, in that order within it
        const uint32_t mesh = s_mesh[tid];
        uint32_t pos = 0, same = 0;
        for (uint32_t r = 0; r < runs; r++) {
            const uint32_t o = s_mesh[r];
            pos += (o < mesh || (o == mesh && r < tid)) ? 1u : 0u;
            same += o == mesh ? 1u : 0u;
        }
        s_pos[tid] = pos;
        p.run_same[base + pos] = (uint8_t)(same - 1);
        p.run_mesh[base + pos] = mesh;
        p.run_tri[base + pos] = s_tri[tid];
        // mark the meshlet's cell (a plain read first: nearly every block finds it marked)
        const DiffView& V = view_at(p, ps.view);
        const uint32_t cell = (by / V.cell_h) * V.cells_x + bx / V.cell_w;
        uint32_t* word = p.cells + ((size_t)ps.view * p.m.count + mesh) * p.cell_words + (cell >> 5);
        const uint32_t bit = 1u << (cell & 31u);
        if (!(__atomic_load_n(word, __ATOMIC_RELAXED) & bit)) atomicOr(word, bit);
    }
    __syncthreads();
    // the wave's (run, value) pairs over its lanes: three corner sums each,
    // over the run's pixels in order
    for (uint32_t i = lane; i < own * 6; i += 64) {
        const uint32_t q = i / 6, c = i - q * 6, r = first + q;
        const float *val = &s_val[2 + c][wid * 64], *w1 = &s_val[0][wid * 64], *w2 = &s_val[1][wid * 64];
        float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
        auto add = [&](float v, float b1, float b2) {
            a0 = __builtin_fmaf((1.0f - b1) - b2, v, a0);
            a1 = __builtin_fmaf(b1, v, a1);
            a2 = __builtin_fmaf(b2, v, a2);
        };
        unsigned long long m = s_mask[r];
        while (m) {       // two pixels a step: their reads overlap
            const uint32_t j = (uint32_t)__builtin_ctzll(m);
            m &= m - 1ull;
            const bool two = m != 0;
            const uint32_t k = two ? (uint32_t)__builtin_ctzll(m) : j;
            m &= m - 1ull;     // 0 stays 0
            const float vj = val[j], b1j = w1[j], b2j = w2[j], vk = val[k], b1k = w1[k], b2k = w2[k];
            add(vj, b1j, b2j);
            if (two) add(vk, b1k, b2k);
        }
        float* out = p.run_sums + (base + s_pos[r]) * kRunSums + c;
        out[0] = a0;
        out[6] = a1;
        out[12] = a2;
    }
}

// ---------------------------------------------------------------- backward: vertices

// Marked cells of each meshlet, and of all together (they set the part size).
// A row of blocks takes about kCountViews of the views (256 views of 16x16
// pixels, 200 meshlets: one block's loop over all of them took 72 us).
constexpr uint32_t kCountViews = 32;

__global__ void __launch_bounds__(256) k_count_cells(DiffParams p) {
    __shared__ uint32_t s_total;
    const uint32_t mi = blockIdx.x * 256 + threadIdx.x;
    if (threadIdx.x == 0) s_total = 0;
    __syncthreads();
    uint32_t n = 0;
    if (mi < p.m.count) {
        for (uint32_t v = blockIdx.y; v < p.num_views; v += gridDim.y) {
            const uint32_t* w = p.cells + ((size_t)v * p.m.count + mi) * p.cell_words;
            if (p.cell_words == 8) {
                const uint4 a = reinterpret_cast<const uint4*>(w)[0], b = reinterpret_cast<const uint4*>(w)[1];
                n += __popc(a.x) + __popc(a.y) + __popc(a.z) + __popc(a.w) + __popc(b.x) + __popc(b.y) +
                     __popc(b.z) + __popc(b.w);
            } else {
                for (uint32_t k = 0; k < p.cell_words; k++) n += __popc(w[k]);
            }
        }
        if (n) atomicAdd(&p.cell_counts[mi], n);
    }
    if (n) atomicAdd(&s_total, n);
    __syncthreads();
    if (threadIdx.x == 0 && s_total) atomicAdd(&p.part_state[0], s_total);
}

// Cells of a part: about kPartBlocks pixel blocks; in scenes of fewer than
// kFillParts meshlets down to a quarter of that, for kFillParts parts; more
// when it could make more than kSplitParts beyond one per meshlet (a meshlet
// of c cells has fewer than c / part_cells of those). 256 views of 16x16
// pixels, 200 meshlets: whole parts 361 us, quarters 274; one 704x512 view,
// 500 meshlets 283 and 236. With 6,000 meshlets the card is full as it is:
// quarters made three 1280x720 views 797 us instead of 732.
__device__ __forceinline__ uint32_t part_cells(const DiffParams& p) {
    const uint32_t total = p.part_state[0];
    const uint32_t g = min(p.part_cells, max(p.part_cells_least, (total + kFillParts - 1) / kFillParts));
    return p.many_parts ? max(g, (total + kSplitParts - 1) / kSplitParts) : g;
}

// The parts of every meshlet (one for a meshlet that shows nowhere: it writes
// zeros); the order of the list does not matter.
__global__ void __launch_bounds__(256) k_list_parts(DiffParams p) {
    const uint32_t mi = blockIdx.x * 256 + threadIdx.x;
    if (mi >= p.m.count) return;
    const uint32_t g = part_cells(p);
    const uint32_t n = max(1u, (p.cell_counts[mi] + g - 1) / g);
    // (the place in the list is the place of the part's sums too, though those
    // of one part have none: a counter of the others alone, one more atomic of
    // all meshlets on one word, made three 1280x720 views 12 us slower)
    const uint32_t at = atomicAdd(&p.part_state[1], n);
    for (uint32_t k = 0; k < n; k++) p.parts[at + k] = make_uint4(mi, k, n, at);
}

// One part a block at a time: the runs of its cells' pixel blocks, 256 blocks
// at a time, are listed in block order and taken in rounds of kRoundRuns:
// their sums are staged in LDS, each triangle's are a bit mask, and a thread
// per (triangle, sum) adds them in order. 2.76 M pixels, 6,000 meshlets: 121 us
// (sorting and reducing 8.3 M vertex records took 574), most of it the
// meshlets at the eye, whose parts list thousands of runs; one block per
// meshlet took 360 us with a linear search for the runs and a thread per
// triangle comparing every run's.
constexpr uint32_t kRoundRuns = 128;
constexpr uint32_t kPartBlocks = 256;

// Cells of a whole part, and the least of one (part_cells)
uint32_t whole_part_cells(const DiffParams& p) { return std::max(1u, kPartBlocks / p.cell_blocks); }
uint32_t least_part_cells(const DiffParams& p) {
    return p.m.count < kFillParts ? std::max(1u, whole_part_cells(p) / 4) : whole_part_cells(p);
}

__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* s_wave, uint32_t& total) {
    const uint32_t lane = __lane_id(), wid = threadIdx.x >> 6;
    uint32_t incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)incl, d);
        if (lane >= (uint32_t)d) incl += o;
    }
    if (lane == 63) s_wave[wid] = incl;
    __syncthreads();
    uint32_t first = incl - v;
    total = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
        if (q < wid) first += s_wave[q];
        total += s_wave[q];
    }
    __syncthreads();
    return first;
}

__global__ void __launch_bounds__(256) k_diff_vertices(DiffParams p, float4* grad_color, float2* grad_uv) {
    __shared__ float s_sum[128][kRunSums];             // per triangle
    __shared__ float s_stage[kRoundRuns][kRunSums];
    __shared__ size_t s_list[kRoundRuns];
    __shared__ unsigned long long s_bits[128][2];      // a triangle's runs of the round
    __shared__ unsigned long long s_corner[64][3][2];  // the triangles a vertex is corner k of
    __shared__ uint32_t s_seen[128], s_ntris, s_wave[4], s_last;
    __shared__ uint8_t s_tris[128];
    __shared__ uint32_t s_cells[kPartBlocks];          // view << 8 | cell
    const uint32_t tid = threadIdx.x, lane = __lane_id(), wid = tid >> 6;
    if (tid < 128) {
        s_bits[tid][0] = s_bits[tid][1] = 0ull;
        s_seen[tid] = 0;
    }
    if (tid == 0) s_ntris = 0;
    const uint32_t nparts = p.part_state[1], group = part_cells(p);
    for (uint32_t item = blockIdx.x; item < nparts; item += gridDim.x) {
        const uint4 part = p.parts[item];
        const uint32_t mi = part.x, cells = p.cell_counts[mi];
        const uint32_t c_lo = part.y * group, c_hi = min(cells, c_lo + group);
        if (c_lo < c_hi) {
            for (uint32_t i = tid; i < 128 * kRunSums; i += 256) s_sum[i / kRunSums][i % kRunSums] = 0.0f;
            for (uint32_t i = tid; i < 384; i += 256) s_corner[i / 6][(i / 2) % 3][i & 1] = 0ull;
            __syncthreads();
            const uint32_t nt = min((uint32_t)p.m.num_triangles[mi], 128u);
            if (tid < nt) {
                const uint32_t corners = p.m.triangles[(size_t)mi * 128 + tid];
#pragma unroll
                for (uint32_t k = 0; k < 3; k++)
                    atomicOr(&s_corner[(corners >> (8 * k)) & 63u][k][tid >> 6], 1ull << (tid & 63u));
            }
        }
        for (uint32_t g0 = c_lo; g0 < c_hi; g0 += kPartBlocks) {
            const uint32_t g1 = min(c_hi, g0 + kPartBlocks);
            // cells [g0, g1) of the meshlet's, in (view, cell) order
            uint32_t seen = 0;
            const uint32_t words = p.num_views * p.cell_words;
            for (uint32_t w0 = 0; w0 < words && seen < g1; w0 += 256) {
                const uint32_t v = (w0 + tid) / p.cell_words, k = w0 + tid - v * p.cell_words;
                uint32_t w = w0 + tid < words ? p.cells[((size_t)v * p.m.count + mi) * p.cell_words + k] : 0u;
                uint32_t total = 0;
                uint32_t rank = seen + block_scan((uint32_t)__popc(w), s_wave, total);
                for (; w && rank < g1; w &= w - 1, rank++)
                    if (rank >= g0) s_cells[rank - g0] = (v << 8) | (k * 32 + (uint32_t)__builtin_ctz(w));
                seen += total;
            }
            __syncthreads();
            const uint32_t candidates = (g1 - g0) * p.cell_blocks;
            for (uint32_t c0 = 0; c0 < candidates; c0 += 256) {
                const uint32_t c = c0 + tid;
                size_t base = 0;
                uint32_t found = 0;
                if (c < candidates) {
                    const uint32_t i = c / p.cell_blocks, q = c - i * p.cell_blocks;
                    const uint32_t vc = s_cells[i];
                    const DiffView& V = view_at(p, vc >> 8);
                    const uint32_t dy = q / V.cell_w, dx = q - dy * V.cell_w;
                    const uint32_t cy = (vc & 255u) / V.cells_x, cx = (vc & 255u) - cy * V.cells_x;
                    const uint32_t x = cx * V.cell_w + dx, y = cy * V.cell_h + dy;
                    if (dy < V.cell_h && x < V.blocks_x && y < V.blocks_y) {
                        const uint32_t b = V.block_base + y * V.blocks_x + x;
                        base = (size_t)b * kBlockRuns;
                        const uint32_t runs = p.block_runs[b];
                        // the runs are sorted by meshlet: find its first
                        uint32_t at = 0;
                        for (uint32_t len = runs; len > 0;) {
                            const uint32_t half_len = len >> 1;
                            const bool up = p.run_mesh[base + at + half_len] < mi;
                            at = up ? at + half_len + 1 : at;
                            len = up ? len - half_len - 1 : half_len;
                        }
                        if (at < runs && p.run_mesh[base + at] == mi) found = p.run_same[base + at] + 1u;
                        base += at;
                    }
                }
                uint32_t total = 0;
                const uint32_t first = block_scan(found, s_wave, total);
                for (uint32_t r0 = 0; r0 < total; r0 += kRoundRuns) {
                    const uint32_t lo = max(first, r0), hi = min(first + found, r0 + kRoundRuns);
                    for (uint32_t k = lo; k < hi; k++) s_list[k - r0] = base + (k - first);
                    __syncthreads();
                    const uint32_t n = min(kRoundRuns, total - r0);
                    if (tid < n) {
                        // the round's runs of each triangle, and the triangles that have some
                        const uint32_t k = p.run_tri[s_list[tid]] & 127u;
                        atomicOr(&s_bits[k][tid >> 6], 1ull << (tid & 63u));
                        if (atomicOr(&s_seen[k], 1u) == 0) s_tris[atomicAdd(&s_ntris, 1u)] = (uint8_t)k;
                    }
                    for (uint32_t i = tid; i < n * kRunSums; i += 256) {
                        const uint32_t e = i / kRunSums, q = i - e * kRunSums;
                        s_stage[e][q] = p.run_sums[s_list[e] * kRunSums + q];
                    }
                    __syncthreads();
                    const uint32_t ntris = s_ntris;
                    for (uint32_t i = tid; i < ntris * kRunSums; i += 256) {
                        const uint32_t e = i / kRunSums, q = i - e * kRunSums, k = s_tris[e];
                        float a = s_sum[k][q];
#pragma unroll
                        for (uint32_t w = 0; w < 2; w++) {
                            unsigned long long m = s_bits[k][w];
                            while (m) {        // two runs a step: their reads overlap
                                const uint32_t j0 = w * 64 + (uint32_t)__builtin_ctzll(m);
                                m &= m - 1ull;
                                const bool two = m != 0;
                                const uint32_t j1 = two ? w * 64 + (uint32_t)__builtin_ctzll(m) : j0;
                                m &= m - 1ull;     // 0 stays 0
                                const float v0 = s_stage[j0][q], v1 = s_stage[j1][q];
                                a += v0;
                                if (two) a += v1;
                            }
                        }
                        s_sum[k][q] = a;
                    }
                    __syncthreads();
                    if (tid < ntris) {
                        const uint32_t k = s_tris[tid];
                        s_bits[k][0] = s_bits[k][1] = 0ull;
                        s_seen[k] = 0;
                    }
                    if (tid == 0) s_ntris = 0;
                    __syncthreads();
                }
            }
        }
        // triangles' corners to vertices: lane = vertex; wave 0-3: channels
        // 0-1, 2-3, 4 and 5 of (colour, U, V)
        const uint32_t ch = wid < 2 ? wid * 2 : wid + 2;
        float g0 = 0.0f, g1 = 0.0f;
        if (c_lo < c_hi) {
#pragma unroll
            for (uint32_t k = 0; k < 3; k++) {
#pragma unroll
                for (uint32_t w = 0; w < 2; w++) {
                    for (unsigned long long m = s_corner[lane][k][w]; m; m &= m - 1ull) {
                        const uint32_t q = w * 64 + (uint32_t)__builtin_ctzll(m);
                        g0 += s_sum[q][k * 6 + ch];
                        if (wid < 2) g1 += s_sum[q][k * 6 + ch + 1];
                    }
                }
            }
        }
        bool write = true;
        if (part.z > 1) {
            // a part of several: the last to finish adds them in order
            float* mine = p.part_sums + (size_t)item * 384;
            mine[ch * 64 + lane] = g0;
            if (wid < 2) mine[(ch + 1) * 64 + lane] = g1;
            __threadfence();
            __syncthreads();
            if (tid == 0) s_last = atomicAdd(&p.parts_done[mi], 1u);
            __syncthreads();
            write = s_last == part.z - 1;
            if (write) {
                __threadfence();
                g0 = g1 = 0.0f;
                for (uint32_t k = 0; k < part.z; k++) {
                    const float* o = p.part_sums + (size_t)(part.w + k) * 384;
                    g0 += __hip_atomic_load(o + ch * 64 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (wid < 2) g1 += __hip_atomic_load(o + (ch + 1) * 64 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        if (write) {
            const size_t vtx = (size_t)mi * 64 + lane;
            if (wid < 2) reinterpret_cast<float2*>(grad_color + vtx)[wid] = make_float2(g0, g1);
            else reinterpret_cast<float*>(grad_uv + vtx)[wid - 2] = g0;
        }
        __syncthreads();       // s_sum, s_corner, s_last
    }
}

// ---------------------------------------------------------------- backward: texels

// Gradients of the four corners of a cell, and the cell's flags and texture
// width (flags 0: a nearest texel only).
struct CellSum {
    float4 c[4];
    uint32_t code, width;

    __device__ void clear() {
#pragma unroll
        for (int k = 0; k < 4; k++) c[k] = f4(0.0f);
        code = width = 0;
    }
    // a pixel's record: dL/dsample g, cell position, flags, texture width
    __device__ void add(float4 g, float fx, float fy, uint32_t cd, uint32_t w) {
        if (!(cd & kTexLinear)) {
            c[0] = add4(c[0], g);
            return;
        }
        const float gx = 1.0f - fx, gy = 1.0f - fy;
        c[0] = fma4(gx * gy, g, c[0]);
        c[1] = fma4(fx * gy, g, c[1]);
        c[2] = fma4(gx * fy, g, c[2]);
        c[3] = fma4(fx * fy, g, c[3]);
        code = cd;
        width = w;
    }
    __device__ void add(const CellSum& o) {
#pragma unroll
        for (int k = 0; k < 4; k++) c[k] = add4(c[k], o.c[k]);
        if (o.code) {
            code = o.code;
            width = o.width;
        }
    }
    // corners past the texture's edge are the cell's own (their weight is 0)
    __device__ void fold() {
        if (!code) return;
        if (!(code & kTexRight)) {
            c[0] = add4(c[0], c[1]);
            c[2] = add4(c[2], c[3]);
        }
        if (!(code & kTexBelow)) {
            c[0] = add4(c[0], c[2]);
            c[1] = add4(c[1], c[3]);
        }
    }
    // the base texel's gradient; the other corners for k_tex_corner. With one
    // corner at a time c[0] is the corner's sum, the first corner's written
    // and the others' added.
    template <int Corner>
    __device__ void write(uint32_t key, float4* grad, float4* cells, size_t start) {
        if constexpr (Corner >= 0) {
            grad[key] = Corner ? add4(grad[key], c[0]) : c[0];
            return;
        }
        fold();
        grad[key] = c[0];
        float4* o = cells + start * 4;
        if (code) {
            o[0] = c[1];
            o[1] = c[2];
            o[2] = c[3];
        }
        o[3] = make_float4(__uint_as_float(code), __uint_as_float(width), 0.0f, 0.0f);
    }
};

// One thread per run piece of a tile of kTile sorted records: 111 us for 2.76 M
// records, bound by the gather of 32 bytes a record in texel order. With the
// sort (125 us, 2.76 M keys instead of 11 M) and the corners (48 us) the
// texel gradients take 289 us, 504 before.
// Corner: every corner of a cell (kWholeCells), or one of them alone, by its
// own texel.
constexpr int kWholeCells = -1;

template <int Corner>
__global__ void __launch_bounds__(kTile) k_tex_reduce(const uint32_t* keys, const uint32_t* idx, const float4* recs,
                                                      uint32_t n, uint32_t sentinel, float4* grad, float4* cells,
                                                      CellSum* part_first, CellSum* part_last, uint2* last,
                                                      uint32_t* spans) {
    __shared__ uint32_t skey[kTile];
    __shared__ float4 sval[kTile], spos[kTile];
    const uint32_t tile = blockIdx.x, tid = threadIdx.x;
    const uint32_t i0 = tile * kTile;
    const uint32_t cnt = min(kTile, n - i0);
    if (tid < cnt) {
        const uint32_t key = keys[i0 + tid];
        skey[tid] = key;
        if (key != sentinel) {
            const size_t r = idx[i0 + tid];
            float4 g = recs[2 * r], q = recs[2 * r + 1];
            if (Corner >= 0 && (__float_as_uint(q.z) & kTexLinear)) {
                g = ((Corner & 1 ? q.x : 1.0f - q.x) * (Corner & 2 ? q.y : 1.0f - q.y)) * g;
                q.z = 0.0f;        // then summed as a nearest texel
            }
            sval[tid] = g;
            spos[tid] = q;
        }
    }
    __syncthreads();
    if (tid >= cnt) return;
    const uint32_t key = skey[tid];
    if (key == sentinel) {
        if (tid == cnt - 1) last[tile] = make_uint2(sentinel, 0u);
        return;
    }
    const uint32_t prev = tid ? skey[tid - 1] : (i0 ? keys[i0 - 1] : sentinel);
    if (tid && prev == key) return;   // not the first record of a piece
    CellSum acc;
    acc.clear();
    uint32_t j = tid;
    for (; j < cnt && skey[j] == key; j++) {
        const float4 q = spos[j];
        acc.add(sval[j], q.x, q.y, __float_as_uint(q.z), __float_as_uint(q.w));
    }
    const bool starts_here = !(tid == 0 && prev == key);
    const bool cont_next = j == cnt && i0 + cnt < n && keys[i0 + cnt] == key;
    if (j == cnt) last[tile] = starts_here && cont_next ? make_uint2(key, i0 + tid) : make_uint2(sentinel, 0u);
    if (starts_here && !cont_next) {
        acc.write<Corner>(key, grad, cells, i0 + tid);
    } else if (starts_here) {
        part_last[tile] = acc;
    } else {
        part_first[tile] = acc;
        spans[tile] = cont_next ? 1u : 0u;
    }
}

// Runs that cross tiles: the tile where a run starts adds the pieces of the
// following tiles in tile order, a thread per tile. Of a run over more than
// kSerialTiles of them the wave adds the rest, 64 pieces a step and then
// across the lanes: one texel for all of 1280x720 pixels (3,600 tiles) took a
// thread 611 us, here 26.
constexpr uint32_t kSerialTiles = 8;

template <int Corner>
__global__ void __launch_bounds__(256) k_tex_fixup(uint32_t tiles, uint32_t sentinel, float4* grad, float4* cells,
                            const CellSum* part_first, const CellSum* part_last, const uint2* last,
                            const uint32_t* spans) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, lane = __lane_id();
    const uint2 l = t < tiles ? last[t] : make_uint2(sentinel, 0u);
    const bool run = l.x != sentinel;
    CellSum acc;
    uint32_t u = t + 1;
    bool more = run;               // tile u has a piece of the run
    if (run) {
        acc = part_last[t];
        for (; more && u - t <= kSerialTiles; u++) {
            acc.add(part_first[u]);
            more = spans[u] != 0;
        }
    }
    for (unsigned long long todo = __ballot(more); todo; todo &= todo - 1ull) {
        const int src = __builtin_ctzll(todo);
        uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)u, src) + lane;
        CellSum sum;
        sum.clear();
        for (;; at += 64) {
            // the run's last piece is the first that does not go on (the array's last tile never does)
            const unsigned long long ends = __ballot(at >= tiles || !spans[at]);
            if (at < tiles && (ends == 0 || lane <= (uint32_t)__builtin_ctzll(ends))) sum.add(part_first[at]);
            if (ends) break;
        }
#pragma unroll
        for (int d = 32; d; d >>= 1) {
#pragma unroll
            for (int k = 0; k < 4; k++)
                sum.c[k] = add4(sum.c[k], make_float4(__shfl_xor(sum.c[k].x, d), __shfl_xor(sum.c[k].y, d),
                                                      __shfl_xor(sum.c[k].z, d), __shfl_xor(sum.c[k].w, d)));
            sum.code |= (uint32_t)__shfl_xor((int)sum.code, d);       // (the pieces' are the same, or 0)
            sum.width |= (uint32_t)__shfl_xor((int)sum.width, d);
        }
        if (lane == (uint32_t)src) acc.add(sum);
    }
    if (run) acc.write<Corner>(l.x, grad, cells, l.y);
}

// Adds the runs' corners of one kind (1 right, 2 below, 3 below right) to the
// gradients: different cells have different corners of a kind.
template <int Corner>
__global__ void __launch_bounds__(256) k_tex_corner(const uint32_t* keys, uint32_t n, uint32_t sentinel,
                                                    const float4* cells, float4* grad) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t key = keys[i];
    if (key == sentinel || (i && keys[i - 1] == key)) return;
    const float4 h = cells[(size_t)i * 4 + 3];
    const uint32_t code = __float_as_uint(h.x), width = __float_as_uint(h.y);
    constexpr uint32_t need = Corner == 1 ? kTexRight : (Corner == 2 ? kTexBelow : kTexRight | kTexBelow);
    if ((code & need) != need) return;
    const size_t at = (size_t)key + (Corner & 1 ? 1u : 0u) + (Corner & 2 ? width : 0u);
    grad[at] = add4(grad[at], cells[(size_t)i * 4 + (Corner - 1)]);
}

// The texel of one corner of each pixel's cell; the sentinel for the corners
// a nearest texel has not. A corner past the texture's edge is the edge's
// texel (its weight is 0).
__global__ void __launch_bounds__(256) k_corner_keys(const uint32_t* base, const float4* recs, uint32_t n,
                                                     uint32_t sentinel, uint32_t corner, uint32_t* keys) {
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    uint32_t key = base[t];
    if (key != sentinel) {
        const float4 q = recs[2 * (size_t)t + 1];
        const uint32_t code = __float_as_uint(q.z);
        if (!(code & kTexLinear)) {
            key = sentinel;
        } else {
            if ((corner & 1u) && (code & kTexRight)) key += 1u;
            if ((corner & 2u) && (code & kTexBelow)) key += __float_as_uint(q.w);
        }
    }
    keys[t] = key;
}

__global__ void k_fill_u32(uint32_t* p, size_t n, uint32_t v) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

__global__ void k_fill_f32(float* p, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0.0f;
}

uint32_t bits_for(uint64_t v) {   // bits needed to hold v
    uint32_t b = 0;
    while (b < 32 && (v >> b) != 0) b++;
    return b;
}

template <class T>
hipError_t grow(T*& p, size_t count) {
    if (p) (void)hipFree(p);
    p = nullptr;
    if (!count) return hipSuccess;
    return hipMalloc((void**)&p, count * sizeof(T));
}

hipError_t fill_zero(void* p, size_t floats, hipStream_t s) {
    if (!floats) return hipSuccess;
    const uint32_t blocks = (uint32_t)std::min<size_t>((floats + 255) / 256, 16384);
    hipLaunchKernelGGL(k_fill_f32, dim3(blocks), dim3(256), 0, s, (float*)p, floats);
    return hipGetLastError();
}

// Sorts the n pixels by key and sums their records per key.
template <int Corner>
hipError_t sum_texels(DiffWorkspace& w, const uint32_t* keys, uint32_t n, uint32_t sentinel, float4* grad,
                      hipStream_t s, Profiler* prof) {
    {
        Profiler::Scope sc(prof, "diff_sort_texels", s);
        size_t bytes = w.sort_temp_bytes;
        const hipError_t e = rocprim::radix_sort_pairs(w.sort_temp, bytes, keys, w.sorted_keys,
                                                       rocprim::counting_iterator<uint32_t>(0), w.sorted_idx, n, 0,
                                                       bits_for(sentinel), s);
        if (e != hipSuccess) return e;
    }
    const uint32_t tiles = (n + kTile - 1) / kTile;
    CellSum* part_first = reinterpret_cast<CellSum*>(w.parts);
    CellSum* part_last = part_first + tiles;
    launch_kernel(prof, "diff_texels", k_tex_reduce<Corner>, dim3(tiles), dim3(kTile), 0, s, w.sorted_keys,
                  w.sorted_idx, w.tex_recs, n, sentinel, grad, w.cells, part_first, part_last, w.last, w.spans);
    launch_kernel(prof, "diff_texels_fixup", k_tex_fixup<Corner>, dim3((tiles + 255) / 256), dim3(256), 0, s, tiles,
                  sentinel, grad, w.cells, part_first, part_last, w.last, w.spans);
    return hipGetLastError();
}

}  // namespace

namespace {

// Parts the meshlets can have beyond one each, kSplitParts at most: with parts
// of whole_part_cells, or up to kFillParts smaller ones. None where the cells
// of all views make one part.
uint32_t split_parts(const DiffParams& p) {
    const size_t cells = (size_t)p.num_views * p.cell_words * 32;
    auto extra = [&](size_t group) { return (size_t)p.m.count * ((cells + group - 1) / group - 1); };
    return (uint32_t)std::max(std::min<size_t>(extra(whole_part_cells(p)), kSplitParts),
                              std::min<size_t>(extra(least_part_cells(p)), kFillParts));
}

size_t cell_mark_words(const DiffParams& p) { return (size_t)p.num_views * p.m.count * p.cell_words; }

// The marks with the counters that start at zero beside them
size_t zeroed_words(const DiffParams& p) { return cell_mark_words(p) + 2 * (size_t)p.m.count + 4; }

}  // namespace

hipError_t diff_workspace_reserve(DiffWorkspace& w, const DiffParams& p) {
    const size_t pixels = p.total_pixels, blocks = p.total_blocks, meshlets = p.m.count;
    hipError_t e = hipSuccess;
    const size_t marks = zeroed_words(p);
    if (marks > w.marks_cap) {
        w.marks_cap = 0;
        e = grow(w.marks, marks);
        if (e != hipSuccess) return e;
        w.marks_cap = marks;
    }
    const size_t splits = split_parts(p);
    if (meshlets + splits > w.parts_cap) {
        w.parts_cap = 0;
        e = grow(w.part_list, meshlets + splits);
        if (e != hipSuccess) return e;
        w.parts_cap = meshlets + splits;
    }
    // (a meshlet of one part writes its gradients at once)
    if (splits && meshlets + splits > w.sums_cap) {
        w.sums_cap = 0;
        e = grow(w.part_sums, (meshlets + splits) * 384);
        if (e != hipSuccess) return e;
        w.sums_cap = meshlets + splits;
    }
    if (blocks > w.blocks) {
        w.blocks = 0;
        e = grow(w.block_runs, blocks);
        if (e == hipSuccess) e = grow(w.run_mesh, blocks * kBlockRuns);
        if (e == hipSuccess) e = grow(w.run_tri, blocks * kBlockRuns);
        if (e == hipSuccess) e = grow(w.run_same, blocks * kBlockRuns);
        if (e == hipSuccess) e = grow(w.run_sums, blocks * kBlockRuns * kRunSums);
        if (e != hipSuccess) return e;
        w.blocks = blocks;
    }
    if (pixels <= w.pixels) return hipSuccess;
    const size_t tiles = (pixels + kTile - 1) / kTile;
    w.pixels = 0;
    e = grow(w.tex_keys, pixels);
    if (e == hipSuccess) e = grow(w.tex_recs, pixels * 2);
    if (e == hipSuccess) e = grow(w.cells, pixels * 4);
    if (e == hipSuccess) e = grow(w.sorted_keys, pixels);
    if (e == hipSuccess) e = grow(w.sorted_idx, pixels);
    if (e == hipSuccess) e = grow(w.parts, tiles * 2 * sizeof(CellSum));
    if (e == hipSuccess) e = grow(w.last, tiles);
    if (e == hipSuccess) e = grow(w.spans, tiles);
    if (e != hipSuccess) return e;
    size_t bytes = 0;
    const uint32_t* keys = w.tex_keys;       // (the sort's argument types: one instance of it)
    e = rocprim::radix_sort_pairs(nullptr, bytes, keys, w.sorted_keys, rocprim::counting_iterator<uint32_t>(0),
                                  w.sorted_idx, (uint32_t)pixels, 0, 32, (hipStream_t)0);
    if (e != hipSuccess) return e;
    if (w.sort_temp) (void)hipFree(w.sort_temp);
    w.sort_temp = nullptr;
    e = hipMalloc(&w.sort_temp, bytes);
    if (e != hipSuccess) return e;
    w.sort_temp_bytes = bytes;
    w.pixels = pixels;
    return hipSuccess;
}

void diff_workspace_release(DiffWorkspace& w) {
    void* ptrs[] = { w.tex_keys, w.tex_recs, w.cells, w.sorted_keys, w.sorted_idx, w.parts,
                     w.last,     w.spans,    w.marks, w.block_runs,  w.run_mesh,   w.run_tri, w.run_same, w.run_sums, w.sort_temp,
                     w.part_list, w.part_sums };
    for (void* q : ptrs)
        if (q) (void)hipFree(q);
    w = DiffWorkspace();
}

hipError_t launch_diff_forward(const DiffParams& p, hipStream_t s, Profiler* prof) {
    const uint32_t n = p.total_pixels;
    launch_kernel(prof, "diff_forward", k_diff_forward, dim3((n + 255) / 256), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_diff_backward(DiffParams p, DiffWorkspace& w, uint64_t num_texels, bool overlapping,
                                float4* grad_texels, float2* grad_uv, float4* grad_color, hipStream_t s,
                                Profiler* prof) {
    const uint32_t n = p.total_pixels;
    p.tex_keys = w.tex_keys;
    p.tex_recs = w.tex_recs;
    p.tex_sentinel = (uint32_t)num_texels;
    p.cells = w.marks;
    p.cell_counts = w.marks + cell_mark_words(p);
    p.parts_done = p.cell_counts + p.m.count;
    p.part_state = p.parts_done + p.m.count;
    p.parts = w.part_list;
    p.part_sums = w.part_sums;
    p.many_parts = split_parts(p) == kSplitParts;
    p.part_cells = whole_part_cells(p);
    p.part_cells_least = least_part_cells(p);
    p.block_runs = w.block_runs;
    p.run_mesh = w.run_mesh;
    p.run_tri = w.run_tri;
    p.run_same = w.run_same;
    p.run_sums = w.run_sums;
    hipError_t e;
    {
        Profiler::Scope sc(prof, "diff_zero_grads", s);
        e = fill_zero(grad_texels, num_texels * 4, s);
        if (e != hipSuccess) return e;
        const size_t words = zeroed_words(p);
        hipLaunchKernelGGL(k_fill_u32, dim3((uint32_t)std::min<size_t>((words + 255) / 256, 4096)), dim3(256), 0, s,
                           w.marks, words, 0u);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    launch_kernel(prof, "diff_pixels", k_diff_pixels, dim3(p.total_blocks), dim3(256), 0, s, p);
    if (p.m.count) {
        const uint32_t mb = (p.m.count + 255) / 256;
        const uint32_t rows = std::min((p.num_views + kCountViews - 1) / kCountViews, 1024u);
        launch_kernel(prof, "diff_cells", k_count_cells, dim3(mb, rows), dim3(256), 0, s, p);
        launch_kernel(prof, "diff_parts", k_list_parts, dim3(mb), dim3(256), 0, s, p);
        launch_kernel(prof, "diff_vertices", k_diff_vertices, dim3(kPartGrid), dim3(256), 0, s, p, grad_color, grad_uv);
    }
    e = hipGetLastError();
    if (e != hipSuccess || !num_texels) return e;
    if (overlapping) {
        // w.cells is free here and holds 64 bytes a pixel
        uint32_t* keys = reinterpret_cast<uint32_t*>(w.cells);
        e = sum_texels<0>(w, w.tex_keys, n, p.tex_sentinel, grad_texels, s, prof);
        for (uint32_t corner = 1; corner < 4 && e == hipSuccess; corner++) {
            launch_kernel(prof, "diff_corner_keys", k_corner_keys, dim3((n + 255) / 256), dim3(256), 0, s, w.tex_keys,
                          w.tex_recs, n, p.tex_sentinel, corner, keys);
            e = corner == 1   ? sum_texels<1>(w, keys, n, p.tex_sentinel, grad_texels, s, prof)
                : corner == 2 ? sum_texels<2>(w, keys, n, p.tex_sentinel, grad_texels, s, prof)
                              : sum_texels<3>(w, keys, n, p.tex_sentinel, grad_texels, s, prof);
        }
        return e;
    }
    e = sum_texels<kWholeCells>(w, w.tex_keys, n, p.tex_sentinel, grad_texels, s, prof);
    if (e != hipSuccess) return e;
    const uint32_t blocks = (n + 255) / 256;
    launch_kernel(prof, "diff_corner_1", k_tex_corner<1>, dim3(blocks), dim3(256), 0, s, w.sorted_keys, n,
                  p.tex_sentinel, w.cells, grad_texels);
    launch_kernel(prof, "diff_corner_2", k_tex_corner<2>, dim3(blocks), dim3(256), 0, s, w.sorted_keys, n,
                  p.tex_sentinel, w.cells, grad_texels);
    launch_kernel(prof, "diff_corner_3", k_tex_corner<3>, dim3(blocks), dim3(256), 0, s, w.sorted_keys, n,
                  p.tex_sentinel, w.cells, grad_texels);
    return hipGetLastError();
}

}  // namespace glimp
