// Differentiable texture-sampling resolve (diff.hip): forward, backward and
// the workspace of the deterministic segmented reduction.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "internal.h"

namespace glimp {

struct DiffTex {                   // fp32 RGBA mip chain, level m row-major at level_offset[m]
    uint32_t width, height, levels, pad;
    uint64_t level_offset[16];     // in texels
};

// One framebuffer of a differentiable resolve. Pixels of all views are
// numbered consecutively (view v owns [pixel_base, pixel_base + W*H)); a
// view's outputs and gradient inputs are row-major at its pixel base.
struct DiffView {
    const unsigned long long* keys;
    int width, height;
    unsigned long long clear_key;
    const DrawEntry* draws;
    uint32_t num_draws;
    uint32_t pixel_base;
    uint32_t block_base, blocks_x, blocks_y;   // 16x16-pixel blocks of the backward, all views' in one numbering
    uint32_t cell_w, cell_h;       // blocks per cell of the grid of up to 16x16 cells over the view
    uint32_t cells_x;              // cells per row of it
    float object_to_clip[16];
    float scale_x, scale_y, center_x, center_y, kx, ky;
};

struct DiffParams {
    DevMeshlets m;
    const DevMaterial* materials;
    uint32_t num_materials;
    const DiffTex* textures;
    uint32_t num_textures;
    ApproxTables tables;
    uint32_t num_views;
    const DiffView* views;         // device table, or null: `view` holds the only view
    DiffView view;
    uint32_t total_pixels;
    const float4* texels;
    const float2* uv;              // [meshlets * 64]
    const float4* color;           // [meshlets * 64]
    float4* out;                   // forward: [total_pixels]
    const float4* grad_out;        // backward: [total_pixels]
    // backward (diff.hip): a texel record per pixel slot ...
    uint32_t* tex_keys;
    float4* tex_recs;              // 2 per pixel: dL/dsample, then cell position, flags and texture width
    uint32_t tex_sentinel;         // key of a pixel without a texel, above every texel index
    // ... and per block of pixels a run per triangle it shows
    uint32_t total_blocks;
    uint32_t* block_runs;          // [total_blocks]
    uint32_t* run_mesh;            // [total_blocks][256] meshlet, ascending
    uint8_t* run_tri;              // [total_blocks][256] triangle
    uint8_t* run_same;             // [total_blocks][256] the block's other runs of the meshlet
    float* run_sums;               // [total_blocks][256][18]
    // the vertex gradients' work list
    uint32_t* cells;               // [views][meshlets][cell_words] a bit per cell of the view the meshlet shows in
    uint32_t* cell_counts;         // [meshlets]
    uint32_t* parts_done;          // [meshlets]
    uint32_t* part_state;          // marked cells; parts
    uint4* parts;                  // meshlet, part of it, its parts, its first part's place
    float* part_sums;              // [parts][6][64], where meshlets can have several
    uint32_t part_cells, part_cells_least, cell_blocks, cell_words;
    bool many_parts;
};

// Device buffers of one backward pass (owned by the context).
struct DiffWorkspace {
    size_t pixels = 0, blocks = 0, marks_cap = 0, parts_cap = 0, sums_cap = 0;
    uint32_t* tex_keys = nullptr;
    float4* tex_recs = nullptr;
    float4* cells = nullptr;       // per run of equal texels, at its first record: three corners, flags and width
    uint32_t* sorted_keys = nullptr;
    uint32_t* sorted_idx = nullptr;
    uint8_t* parts = nullptr;      // per 256-record tile the pieces of runs that cross it
    uint2* last = nullptr;         // per tile its last run (texel, first record) when that goes on
    uint32_t* spans = nullptr;
    uint32_t* marks = nullptr;     // cells, cell_counts, parts_done, part_state
    uint4* part_list = nullptr;
    float* part_sums = nullptr;
    uint32_t* block_runs = nullptr;
    uint32_t* run_mesh = nullptr;
    uint8_t* run_tri = nullptr;
    uint8_t* run_same = nullptr;
    float* run_sums = nullptr;
    void* sort_temp = nullptr;
    size_t sort_temp_bytes = 0;
};

// For the calls of p: its views, blocks, cells and scene.
hipError_t diff_workspace_reserve(DiffWorkspace& w, const DiffParams& p);
void diff_workspace_release(DiffWorkspace& w);
hipError_t launch_diff_forward(const DiffParams& p, hipStream_t s, Profiler* prof);
// grad_texels [num_texels], grad_uv [vertices], grad_color [vertices] are
// overwritten (zeros where nothing contributes). `overlapping`: the level-0
// ranges of two textures overlap and are not the same range.
hipError_t launch_diff_backward(DiffParams p, DiffWorkspace& w, uint64_t num_texels, bool overlapping,
                                float4* grad_texels, float2* grad_uv, float4* grad_color, hipStream_t s,
                                Profiler* prof);

}  // namespace glimp
