// hl_cull.hip -- light preparation and light assignment kernels for gfx950.
//
//  k_prep_lights      GpuLight[] -> HotLight[] (shading) + CullLight[] (culling)
//  k_tile_prep/_cull  reference 16-px tile lists (light_cull.wgsl:123-180) of the
//                     screen's grid, a super-tile per block
//  k_cull_tiles       the same for any tile grid: one wavefront per tile, every
//                     light tested, ballot + prefix-popcount compaction
//  k_cluster_geom     per column: NDC rectangle and lateral planes; per cell:
//                     the view-space AABB; its blocks past the cells prepare
//                     the lights (as k_prep_lights) in the same launch
//                     (this and the next four: grids past the column path's)
//  k_cluster_mark     light-parallel: each light bounds the cells it can reach
//                     (projected bounding box x slice range); a wavefront tests
//                     those candidates 64 at a time with the exact membership
//                     rule and sets the member bits in a two-level bitmask
//                     (bits + a summary bit per non-empty word); past its first
//                     chunks a light queues the rest
//  k_cluster_mark_tail the queued chunks, spread over all CUs
//  k_cluster_count    per cluster (16 lanes): popcount over its non-empty
//                     words; sums of the capped counts per scan tile of 1024
//  k_cluster_fill     per block of 16 clusters: its offsets from the tile
//                     sums and the counts before it (the exclusive scan, no
//                     separate launch), then the ascending indices from the
//                     bitmask, which it clears again for the next call
//  k_col_*            the clustered lists a column of the grid per block (most
//                     grids; see the section)
//  k_cluster_bf_*     the clustered lists by testing every light in every cell
//                     (small problems on wide grids of few slices)
//  k_batch_*          the same steps for many views in one launch each
// Membership is decided by the same exact FP32 tests whatever the order of
// evaluation, so the lists equal the per-cluster brute force bit for bit.
#include <algorithm>

#include "hl_internal.hpp"

namespace hl {

// ------------------------------------------------------------------- prep
// The culling record of a light (view-space centre and range, cone terms).
__device__ __forceinline__ CullLight cull_light(float4 pr, float4 dro, uint32_t type, float range,
                                                const float* __restrict__ v) {
    CullLight c;
    c.vpos = make_float4(hl_x_mat_row(v, 0, pr.x, pr.y, pr.z, 1.0f), hl_x_mat_row(v, 1, pr.x, pr.y, pr.z, 1.0f),
                         hl_x_mat_row(v, 2, pr.x, pr.y, pr.z, 1.0f), range);
    c.cone = make_float4(hl_x_mat_row(v, 0, dro.x, dro.y, dro.z, 0.0f), hl_x_mat_row(v, 1, dro.x, dro.y, dro.z, 0.0f),
                         hl_x_mat_row(v, 2, dro.x, dro.y, dro.z, 0.0f), type == HL_LIGHT_SPOT ? dro.w : kNoCone);
    c.axis = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    c.aux = c.axis;
    if (c.cone.w != kNoCone && !hl_x_cone_light(c.cone, &c.axis, &c.aux.x)) c.cone.w = kNoCone;
    return c;
}

__device__ __forceinline__ CullLight cull_light_at(const GpuLight* __restrict__ lights, uint32_t i,
                                                   const GpuCameraUniforms* __restrict__ cam) {
    const GpuLight* l = &lights[i];
    const float4 pr = *reinterpret_cast<const float4*>(l->position_range);
    const float4 dro = *reinterpret_cast<const float4*>(l->direction_outer);
    const uint32_t type = l->light_type;
    return cull_light(pr, dro, type, type == HL_LIGHT_DIRECTIONAL ? __builtin_inff() : pr.w, cam->view);
}

__device__ __forceinline__ void prep_one(const GpuLight* __restrict__ lights,
                                         const uint32_t* __restrict__ subset, uint32_t n,
                                         const GpuCameraUniforms* __restrict__ cam,
                                         HotLight* __restrict__ hot, CullLight* __restrict__ cull,
                                         uint32_t* __restrict__ flags, uint32_t i) {
    if (i >= n) return;
    const GpuLight* l = &lights[subset ? subset[i] : i];
    const float4 pr = *reinterpret_cast<const float4*>(l->position_range);
    const float4 dro = *reinterpret_cast<const float4*>(l->direction_outer);
    const float4 ci = *reinterpret_cast<const float4*>(l->color_intensity);
    const uint32_t type = l->light_type;
    const float inner = l->inner_angle;
    const float inf = __builtin_inff();
    const float range = type == HL_LIGHT_DIRECTIONAL ? inf : pr.w;
    if (hot)
        hot[i] = make_hot_light(pr.x, pr.y, pr.z, dro.x, dro.y, dro.z, ci, pr.w, dro.w, inner, type,
                                shadow_word(i, type, l->shadow_index), true);
    if (cull) cull[i] = cull_light(pr, dro, type, range, cam->view);
    if (flags) {
        uint32_t f = 0;
        // shadow_factor samples the atlas only below MAX_SHADOW_LIGHTS = 42
        // (deferred_lighting.wgsl:453-459)
        if (l->shadow_index != HL_NO_SHADOW && i < 42u) f |= kFlagShadowIgnored;
        if (l->ies_profile_index >= 0 || l->light_function_index >= 0) f |= kFlagTexturedIgnored;
        if (f) atomicOr(flags, f);
    }
}

__global__ __launch_bounds__(256) void k_prep_lights(const GpuLight* __restrict__ lights,
                                                     const uint32_t* __restrict__ subset,
                                                     uint32_t n,
                                                     const GpuCameraUniforms* __restrict__ cam,
                                                     HotLight* __restrict__ hot,
                                                     CullLight* __restrict__ cull,
                                                     uint32_t* __restrict__ flags) {
    prep_one(lights, subset, n, cam, hot, cull, flags, blockIdx.x * blockDim.x + threadIdx.x);
}

// The adjoint's set-up in one launch: the shading records, the per-light
// gradient accumulators cleared, and the loss (when given) cleared.
__global__ __launch_bounds__(256) void k_prep_zero(const GpuLight* __restrict__ lights, uint32_t n,
                                                   const GpuCameraUniforms* __restrict__ cam,
                                                   HotLight* __restrict__ hot, uint32_t* __restrict__ flags,
                                                   double* __restrict__ acc, size_t acc_n,
                                                   double* __restrict__ loss) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    prep_one(lights, nullptr, n, cam, hot, nullptr, flags, (uint32_t)(i < n ? i : n));
    for (size_t j = i; j < acc_n; j += (size_t)gridDim.x * blockDim.x) acc[j] = 0.0;
    if (i == 0 && loss) *loss = 0.0;
}

// -------------------------------------------------------------- tile cull
// Plane k of a 16x16 tile: left, right, top, bottom (light_cull.wgsl:123-150).
__device__ __forceinline__ float3 tile_plane(const GpuCameraUniforms* __restrict__ cam, const LightCullParams& p,
                                             uint32_t tile_x, uint32_t tile_y, uint32_t k) {
#pragma clang fp contract(off)
    const float fw = (float)p.screen_width, fh = (float)p.screen_height;
    const float ts = (float)HL_TILE_SIZE;
    const float l = ((float)tile_x * ts / fw) * 2.0f - 1.0f;
    const float r = fminf(((float)(tile_x + 1u) * ts / fw) * 2.0f - 1.0f, 1.0f);
    const float t = 1.0f - ((float)tile_y * ts / fh) * 2.0f;
    const float b = fmaxf(1.0f - ((float)(tile_y + 1u) * ts / fh) * 2.0f, -1.0f);
    // (l, b, l, t), (r, t, r, b), (l, t, r, t), (r, b, l, b)
    return hl_x_plane(cam->proj[0], cam->proj[5], (k == 0u || k == 2u) ? l : r, (k == 0u || k == 3u) ? b : t,
                      (k == 0u || k == 3u) ? l : r, (k == 0u || k == 2u) ? t : b);
}
__device__ __forceinline__ void tile_planes(const GpuCameraUniforms* __restrict__ cam, const LightCullParams& p,
                                            uint32_t tile_x, uint32_t tile_y, float3 pl[4]) {
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) pl[k] = tile_plane(cam, p, tile_x, tile_y, k);
}

__device__ __forceinline__ bool tile_pass(const float3 pl[4], float4 c) {
    return hl_x_plane_pass(pl[0], c, c.w) && hl_x_plane_pass(pl[1], c, c.w) && hl_x_plane_pass(pl[2], c, c.w) &&
           hl_x_plane_pass(pl[3], c, c.w);
}

// One wavefront per 16x16 tile; four tiles per 256-thread block; every light
// tested (any tile grid).
__global__ __launch_bounds__(256) void k_cull_tiles(const GpuCameraUniforms* __restrict__ cam,
                                                    LightCullParams p,
                                                    const CullLight* __restrict__ cl,
                                                    uint32_t* __restrict__ lists,
                                                    uint32_t* __restrict__ counts) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t tile = blockIdx.x * 4u + (threadIdx.x >> 6);
    const uint32_t total = p.num_tiles_x * p.num_tiles_y;
    if (tile >= total) return;
    const uint32_t tile_x = tile % p.num_tiles_x, tile_y = tile / p.num_tiles_x;
    float3 pl[4];
    tile_planes(cam, p, tile_x, tile_y, pl);
    uint32_t count = 0;
    uint32_t* out = lists + (size_t)tile * HL_MAX_LIGHTS_PER_TILE;
    for (uint32_t base = 0; base < p.num_lights; base += 64u) {
        const uint32_t i = base + lane;
        bool pass = false;
        if (i < p.num_lights) pass = tile_pass(pl, cl[i].vpos);
        const uint64_t m = hl_ballot(pass);
        const uint32_t pos = count + hl_prefix(m);
        if (pass && pos < HL_MAX_LIGHTS_PER_TILE) out[pos] = i;
        count += (uint32_t)__popcll(m);
        if (count >= HL_MAX_LIGHTS_PER_TILE) break;
    }
    if (lane == 0) counts[tile] = count < HL_MAX_LIGHTS_PER_TILE ? count : HL_MAX_LIGHTS_PER_TILE;
}

// ------------------------------------------------------------ clusters
struct ColumnGeom {
    float3 pl[4];
    float l, r, b, t;
    uint32_t on;
    uint32_t pad[3];
};

struct CellBox {
    float lo[3], hi[3];
};
// chunk_fetch reads both records as words at these offsets
static_assert(sizeof(float3) == 12 && sizeof(ColumnGeom) == 80 && offsetof(ColumnGeom, on) == 64,
              "ColumnGeom layout");
static_assert(sizeof(CellBox) == 24, "CellBox layout");

// geometry scratch: ColumnGeom per column, then (256-B aligned) CellBox per cell
__host__ __device__ inline size_t cluster_geom_offset_boxes_dev(uint32_t ncol) {
    return (sizeof(ColumnGeom) * (size_t)ncol + 255) & ~(size_t)255;
}

__device__ __forceinline__ bool column_rect(const ClusterArgs& a, uint32_t cx, uint32_t cy,
                                            float* l, float* r, float* b, float* t) {
#pragma clang fp contract(off)
    const uint32_t px0 = cx * a.cell_w, py0 = cy * a.cell_h;
    if (px0 >= a.width || py0 >= a.height) return false;
    const uint32_t px1 = min(px0 + a.cell_w, a.width), py1 = min(py0 + a.cell_h, a.height);
    const float fw = (float)a.width, fh = (float)a.height;
    *l = ((float)px0 / fw) * 2.0f - 1.0f;
    *r = ((float)px1 / fw) * 2.0f - 1.0f;
    *t = 1.0f - ((float)py0 / fh) * 2.0f;
    *b = 1.0f - ((float)py1 / fh) * 2.0f;
    return true;
}

// One thread per cell: the cell's view-space AABB (the column's NDC corners
// unprojected at the slice's padded near and far distances); the slice-0
// thread of each column also writes the column's lateral planes (the tile
// cull's construction on the column's pixel rectangle).
// The records of cell (col, k): its view-space box, and with planes its
// column's record.
__device__ __forceinline__ void cell_geometry(const ClusterArgs& a, const GpuCameraUniforms* __restrict__ cam,
                                              uint32_t col, uint32_t k, bool planes, ColumnGeom& g,
                                              CellBox& bx) {
#pragma clang fp contract(off)
    const uint32_t cx = col % a.grid_x, cy = col / a.grid_x;
    float l = 0.0f, r = 0.0f, b = 0.0f, t = 0.0f;
    const bool on = column_rect(a, cx, cy, &l, &r, &b, &t);
    const float p00 = cam->proj[0], p11 = cam->proj[5];
    if (on) {
        const float zn = a.slice_near[k], zf = a.slice_far[k];
        const float x0 = l * zn / p00, x1 = r * zn / p00, x2 = l * zf / p00, x3 = r * zf / p00;
        const float y0 = b * zn / p11, y1 = t * zn / p11, y2 = b * zf / p11, y3 = t * zf / p11;
        bx.lo[0] = fminf(fminf(fminf(x0, x1), x2), x3);
        bx.hi[0] = fmaxf(fmaxf(fmaxf(x0, x1), x2), x3);
        bx.lo[1] = fminf(fminf(fminf(y0, y1), y2), y3);
        bx.hi[1] = fmaxf(fmaxf(fmaxf(y0, y1), y2), y3);
        bx.lo[2] = -zf;
        bx.hi[2] = -zn;
    } else {
        bx.lo[0] = bx.lo[1] = bx.lo[2] = bx.hi[0] = bx.hi[1] = bx.hi[2] = 0.0f;
    }
    if (!planes) return;
    g.on = on ? 1u : 0u;
    g.pad[0] = g.pad[1] = g.pad[2] = 0;
    g.l = l;
    g.r = r;
    g.b = b;
    g.t = t;
    if (on) {
        g.pl[0] = hl_x_plane(p00, p11, l, b, l, t);
        g.pl[1] = hl_x_plane(p00, p11, r, t, r, b);
        g.pl[2] = hl_x_plane(p00, p11, l, t, r, t);
        g.pl[3] = hl_x_plane(p00, p11, r, b, l, b);
    } else {
        for (int i = 0; i < 4; ++i) g.pl[i] = make_float3(0.0f, 0.0f, 0.0f);
    }
}

__device__ __forceinline__ void geom_cell(const ClusterArgs& a,
                                          const GpuCameraUniforms* __restrict__ cam,
                                          ColumnGeom* __restrict__ geom,
                                          CellBox* __restrict__ boxes, uint32_t cell) {
    const uint32_t ncol = a.grid_x * a.grid_y;
    if (cell >= ncol * a.grid_z) return;
    const uint32_t col = cell % ncol, k = cell / ncol;
    ColumnGeom g;
    CellBox bx;
    cell_geometry(a, cam, col, k, k == 0, g, bx);
    boxes[cell] = bx;
    if (k == 0) geom[col] = g;
}

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Membership of light (c) in cell (col, k): the definition of the clustered
// lists -- lateral planes of the column with the column padding, the cell's
// AABB with the slice padding (pad = slice_r_pad[k]), and the cone for spot
// lights.  Every test is evaluated (no short circuit) so that the column and
// box records are loaded together rather than one after another.
__device__ __forceinline__ bool cell_member(const CullLight& c, const ColumnGeom& g,
                                            const CellBox& bx, float pad) {
#pragma clang fp contract(off)
    const float rc = c.vpos.w + pad;
    const float3 lo = make_float3(bx.lo[0], bx.lo[1], bx.lo[2]);
    const float3 hi = make_float3(bx.hi[0], bx.hi[1], bx.hi[2]);
    bool in = g.on != 0u;
    in &= hl_x_plane_pass(g.pl[0], c.vpos, rc);
    in &= hl_x_plane_pass(g.pl[1], c.vpos, rc);
    in &= hl_x_plane_pass(g.pl[2], c.vpos, rc);
    in &= hl_x_plane_pass(g.pl[3], c.vpos, rc);
    in &= hl_x_sphere_aabb(c.vpos, rc, lo, hi);
    if (c.cone.w != kNoCone) in &= hl_x_cone_cell(c.vpos, c.axis, c.aux.x, pad, lo, hi);
    return in;
}

// Candidate cells of a light: the columns and slices left by necessary
// conditions of the membership rule, rounded outwards.
//  * slices: the box test needs slice_near[k] <= zc + rc and slice_far[k] >=
//    zc - rc (zc the light's view distance, rc = |radius| + pad_k, at most rr,
//    the radius plus the largest padding of the slices in reach: paddings do
//    not decrease with k);
//  * columns: a column with NDC edges l < r (|l|, |r| <= 1) passes its left
//    plane (normal (1, 0, l / p00) normalised) only if
//    l <= p00 (cx + rc sqrt(1 + l^2 / p00^2)) / zc <= p00 (cx + rr fx) / zc
//    with fx = sqrt(1 + 1 / p00^2), and its right plane only if
//    r >= p00 (cx - rr fx) / zc (zc > 0, p00 > 0); in pixels, the columns
//    floor(px0 / cell_w) .. floor(px1 / cell_w).  Rows alike with p11.
// The FP32 tests can pass a few ulp beyond these real-number bounds, and the
// bounds are computed with fast reciprocals and square roots (a few ulp of the
// terms): rr is widened by 1e-5 of itself and of |cx| + |cy| + zc, the pixel
// bounds by 1e-5 of their magnitude plus a quarter pixel, the slice limits by
// 1e-5 relative -- each many times those errors.  Directional lights, lights
// with a non-finite centre and a camera with p00 or p11 <= 0 take the whole
// grid (or the whole screen); the exact tests decide there.
struct MarkBox {
    uint32_t x0, y0, s0, nx, ny, nz;
};

// The columns of that bound for a light in front of the camera (centre c,
// view distance zc > 0, widened radius rr; p00, p11 > 0), before clamping to
// the grid: inclusive x and y ranges, each end in [-1, grid].
__device__ __forceinline__ void light_columns(const ClusterArgs& a, float p00, float p11, float4 c, float zc,
                                              float rr, int* x0, int* x1, int* y0, int* y1) {
    const int gx = (int)a.grid_x, gy = (int)a.grid_y;
    const float fx = __builtin_amdgcn_sqrtf(1.0f + hl_f_rcp(p00 * p00));
    const float fy = __builtin_amdgcn_sqrtf(1.0f + hl_f_rcp(p11 * p11));
    const float iz = hl_f_rcp(zc);
    const float nx0 = p00 * (c.x - rr * fx) * iz, nx1 = p00 * (c.x + rr * fx) * iz;
    const float ny0 = p11 * (c.y - rr * fy) * iz, ny1 = p11 * (c.y + rr * fy) * iz;
    const float fw = (float)a.width, fh = (float)a.height;
    float px0 = (nx0 + 1.0f) * 0.5f * fw, px1 = (nx1 + 1.0f) * 0.5f * fw;
    float py0 = (1.0f - ny1) * 0.5f * fh, py1 = (1.0f - ny0) * 0.5f * fh;
    px0 -= 1e-5f * fabsf(px0) + 0.25f;
    px1 += 1e-5f * fabsf(px1) + 0.25f;
    py0 -= 1e-5f * fabsf(py0) + 0.25f;
    py1 += 1e-5f * fabsf(py1) + 0.25f;
    const float icw = hl_f_rcp((float)a.cell_w), ich = hl_f_rcp((float)a.cell_h);
    // clamped to [-1, g] before the conversion (NaN: the whole range)
    *x0 = (int)fminf(fmaxf(floorf(px0 * icw), -1.0f), (float)gx);
    *x1 = (int)fmaxf(fminf(floorf(px1 * icw), (float)gx), -1.0f);
    *y0 = (int)fminf(fmaxf(floorf(py0 * ich), -1.0f), (float)gy);
    *y1 = (int)fmaxf(fminf(floorf(py1 * ich), (float)gy), -1.0f);
}

// Whether a light's cells can be bounded at all (else: the whole grid).
__device__ __forceinline__ bool light_bounded(float4 vpos) {
    return !__builtin_isinf(vpos.w) && __builtin_isfinite(-vpos.z) && __builtin_isfinite(vpos.x) &&
           __builtin_isfinite(vpos.y);
}

// All 64 lanes must be active (the slice limits are found by ballots); sp is
// slice_r_pad[lane] (lanes below grid_z; slice_near, slice_far and the
// paddings are non-decreasing, checked by the host).
__device__ __forceinline__ bool light_cells(const ClusterArgs& a,
                                            const GpuCameraUniforms* __restrict__ cam,
                                            const CullLight& L, float sp, MarkBox& m) {
    const int gx = (int)a.grid_x, gy = (int)a.grid_y, gz = (int)a.grid_z;
    const uint32_t lane = hl_lane();
    const bool sl = (int)lane < gz;
    const float vn = sl ? a.slice_near[lane] : 0.0f, vf = sl ? a.slice_far[lane] : 0.0f;
    const float sn = vn - 1e-5f * fabsf(vn), sf = vf + 1e-5f * fabsf(vf);
    int x0 = 0, x1 = gx - 1, y0 = 0, y1 = gy - 1, s0 = 0, s1 = gz - 1;
    const float zc = -L.vpos.z;
    if (light_bounded(L.vpos)) {
        const float slack = 1e-5f * (fabsf(L.vpos.x) + fabsf(L.vpos.y) + fabsf(zc));
        const float r = fabsf(L.vpos.w);
        // slices in reach under the largest padding, then under the largest
        // padding of those slices
        float rr = (r + hl_readlane(sp, (uint32_t)(gz - 1))) * (1.0f + 1e-5f) + slack;
        s1 = (int)__popcll(hl_ballot(sl && sn <= zc + rr)) - 1;
        if (s1 < 0) return false;
        rr = (r + hl_readlane(sp, (uint32_t)s1)) * (1.0f + 1e-5f) + slack;
        s0 = (int)__popcll(hl_ballot(sl && sf < zc - rr));
        s1 = (int)__popcll(hl_ballot(sl && sn <= zc + rr)) - 1;
        const float p00 = cam->proj[0], p11 = cam->proj[5];
        if (zc > 1e-4f && p00 > 0.0f && p11 > 0.0f)
            light_columns(a, p00, p11, L.vpos, zc, rr, &x0, &x1, &y0, &y1);
    }
    x0 = clampi(x0, 0, gx - 1);
    x1 = clampi(x1, -1, gx - 1);
    y0 = clampi(y0, 0, gy - 1);
    y1 = clampi(y1, -1, gy - 1);
    s0 = clampi(s0, 0, gz - 1);
    s1 = clampi(s1, -1, gz - 1);
    if (x1 < x0 || y1 < y0 || s1 < s0) return false;
    m.x0 = (uint32_t)x0;
    m.y0 = (uint32_t)y0;
    m.s0 = (uint32_t)s0;
    m.nx = (uint32_t)(x1 - x0 + 1);
    m.ny = (uint32_t)(y1 - y0 + 1);
    m.nz = (uint32_t)(s1 - s0 + 1);
    return true;
}

__device__ __forceinline__ uint4 pack_box(const MarkBox& m) {
    return make_uint4(m.x0, m.y0, (m.s0 << 16) | m.nz, (m.nx << 16) | m.ny);
}
__device__ __forceinline__ MarkBox unpack_box(uint4 v) {
    MarkBox m;
    m.x0 = v.x;
    m.y0 = v.y;
    m.s0 = v.z >> 16;
    m.nz = v.z & 0xffffu;
    m.nx = v.w >> 16;
    m.ny = v.w & 0xffffu;
    return m;
}

// Candidate cells chunk*64 .. chunk*64+63 of light li (one per lane, slice
// fastest): the exact membership rule, then the member bit and its summary
// bit (no-return atomics).  Split in a fetch (the lane's cell and its column,
// box and slice-padding records, loaded together) and a test-and-mark, so
// that a wave can have the loads of two chunks in flight at once.
struct ChunkCell {
    ColumnGeom g;
    CellBox bx;
    size_t cell;
    float pad;
    bool on;
};

__device__ __forceinline__ ChunkCell chunk_fetch(const ClusterArgs& a, const MarkBox& m,
                                                 const ColumnGeom* __restrict__ geom,
                                                 const CellBox* __restrict__ boxes, uint32_t chunk) {
    ChunkCell r;
    const uint32_t work = m.nx * m.ny * m.nz;
    const uint32_t t = chunk * 64u + (threadIdx.x & 63u);
    r.on = t < work;
    if (!r.on) return r;
    uint32_t rest, iy;
    if (work <= (1u << 21)) {
        rest = hl_floor_div(t, m.nz);
        iy = hl_floor_div(rest, m.nx);
    } else {
        rest = t / m.nz;
        iy = rest / m.nx;
    }
    const uint32_t kz = t - rest * m.nz, ix = rest - iy * m.nx;
    const uint32_t col = (m.x0 + ix) + a.grid_x * (m.y0 + iy);
    const uint32_t k = m.s0 + kz;
    r.cell = (size_t)col + (size_t)(a.grid_x * a.grid_y) * k;
    // records of a batched view come through pointers read from memory:
    // hl_g keeps their loads global rather than flat
    {
        const hl_gptr<const hl_f32x4> gq = hl_g(reinterpret_cast<const hl_f32x4*>(geom + col));
        const hl_f32x4 q0 = gq[0], q1 = gq[1], q2 = gq[2], q4 = gq[4];
        r.g.pl[0] = make_float3(q0.x, q0.y, q0.z);
        r.g.pl[1] = make_float3(q0.w, q1.x, q1.y);
        r.g.pl[2] = make_float3(q1.z, q1.w, q2.x);
        r.g.pl[3] = make_float3(q2.y, q2.z, q2.w);
        r.g.on = __float_as_uint(q4.x);
        const hl_gptr<const float> bq = hl_g(&boxes[r.cell].lo[0]);
        r.bx.lo[0] = bq[0];
        r.bx.lo[1] = bq[1];
        r.bx.lo[2] = bq[2];
        r.bx.hi[0] = bq[3];
        r.bx.hi[1] = bq[4];
        r.bx.hi[2] = bq[5];
    }
    r.pad = a.slice_r_pad[k];
    return r;
}

__device__ __forceinline__ size_t cluster_cells(const ClusterArgs& a) {
    return (size_t)a.grid_x * a.grid_y * a.grid_z;
}

// The bitmask is stored word-major: word w of cluster c (lights 32 w .. 32 w
// + 31) at bits[w * ncell + c], summary word s (bitmask words 32 s .. 32 s +
// 31) at summary[s * ncell + c].  A light's member cells in one row of one
// slice are then adjacent words (fewer lines for its atomics), and the list
// kernel's 16 consecutive clusters read their words of one light range from
// one line.
__device__ __forceinline__ void chunk_mark(const CullLight& L, const ChunkCell& r, uint32_t li,
                                           uint32_t* __restrict__ bits, uint32_t* __restrict__ summary,
                                           size_t ncell) {
    if (!r.on || !cell_member(L, r.g, r.bx, r.pad)) return;
    const uint32_t word = li >> 5;
    __hip_atomic_fetch_or(hl_g(&bits[(size_t)word * ncell + r.cell]), 1u << (li & 31u), __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_or(hl_g(&summary[(size_t)(word >> 5) * ncell + r.cell]), 1u << (word & 31u),
                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void mark_chunk(const ClusterArgs& a, const CullLight& L,
                                           const MarkBox& m, uint32_t li,
                                           const ColumnGeom* __restrict__ geom,
                                           const CellBox* __restrict__ boxes,
                                           uint32_t* __restrict__ bits,
                                           uint32_t* __restrict__ summary, uint32_t chunk) {
    chunk_mark(L, chunk_fetch(a, m, geom, boxes, chunk), li, bits, summary, cluster_cells(a));
}

__device__ __forceinline__ CullLight load_light_uniform(const CullLight* __restrict__ cl, uint32_t li) {
    CullLight L = cl[li];
    L.vpos = make_float4(hl_uniform(L.vpos.x), hl_uniform(L.vpos.y), hl_uniform(L.vpos.z),
                         hl_uniform(L.vpos.w));
    L.cone = make_float4(hl_uniform(L.cone.x), hl_uniform(L.cone.y), hl_uniform(L.cone.z),
                         hl_uniform(L.cone.w));
    L.axis = make_float4(hl_uniform(L.axis.x), hl_uniform(L.axis.y), hl_uniform(L.axis.z),
                         hl_uniform(L.axis.w));
    L.aux.x = hl_uniform(L.aux.x);
    return L;
}

// One wavefront per light: its candidate box, its first kMarkInline chunks,
// and the rest queued as (qlight, qview << 24 | chunk) entries with the box
// stored at bounds[qlight] (qlight: the light's index in the queue's
// numbering, qview: its view in a batch; chunks stay below 2^20).
// Chunks that do not fit in the light's sub-queue stay with this wave.
__device__ __forceinline__ void mark_light(const ClusterArgs& a,
                                           const GpuCameraUniforms* __restrict__ cam,
                                           const CullLight* __restrict__ cl,
                                           const ColumnGeom* __restrict__ geom,
                                           const CellBox* __restrict__ boxes,
                                           uint32_t* __restrict__ bits,
                                           uint32_t* __restrict__ summary,
                                           uint32_t li, const MarkQueue& q, uint32_t qlight,
                                           uint32_t qview) {
    if (li >= a.num_lights) return;
    const CullLight L = load_light_uniform(cl, li);
    const float sp = hl_lane() < a.grid_z ? a.slice_r_pad[hl_lane()] : 0.0f;
    MarkBox m;
    if (!light_cells(a, cam, L, sp, m)) return;
    const uint32_t nchunk = (m.nx * m.ny * m.nz + 63u) / 64u;
    // chunks 0 and 1 always stay with this wave: their loads go out first,
    // both together, ahead of the queueing of the rest
    static_assert(kMarkInline == 2, "two head chunks fetched together");
    const ChunkCell r0 = chunk_fetch(a, m, geom, boxes, 0u);
    ChunkCell r1;
    if (nchunk > 1u) r1 = chunk_fetch(a, m, geom, boxes, 1u);
    uint32_t qlo = nchunk, qhi = nchunk;  // chunks [qlo, qhi) are queued
    if (nchunk > kMarkInline) {
        const uint32_t extra = nchunk - kMarkInline;
        const uint32_t sub = qlight % kMarkQueues;
        uint32_t base = 0;
        if ((threadIdx.x & 63u) == 0) base = atomicAdd(q.count + sub * kMarkCountStride, extra);
        base = hl_readlane(base, 0);
        // room left in the sub-queue, saturating at zero.  Written as
        // fit = base >= seg ? 0 : min(extra, seg - base), -O3 marked the
        // difference no-wrap and folded the select away, and an overflowing
        // light then took fit = extra and wrote past its segment
        // (tests/test_mark_queue_guard.py checks the compiled form)
        const uint32_t room = __builtin_elementwise_sub_sat(q.seg, base);
        const uint32_t fit = min(extra, room);
        if (fit) {
            if ((threadIdx.x & 63u) == 0) q.bounds[qlight] = pack_box(m);
            uint2* seg = q.entries + (size_t)sub * q.seg + base;
            for (uint32_t j = threadIdx.x & 63u; j < fit; j += 64u)
                seg[j] = make_uint2(qlight, (qview << 24) | (kMarkInline + j));
            qlo = kMarkInline;
            qhi = kMarkInline + fit;
        }
    }
    // chunks [0, qlo) and [qhi, nchunk) stay here (qlo >= 2 whenever nchunk >= 2)
    chunk_mark(L, r0, li, bits, summary, cluster_cells(a));
    if (nchunk > 1u) chunk_mark(L, r1, li, bits, summary, cluster_cells(a));
    for (uint32_t c = 2u; c < qlo; ++c) mark_chunk(a, L, m, li, geom, boxes, bits, summary, c);
    for (uint32_t c = qhi; c < nchunk; ++c) mark_chunk(a, L, m, li, geom, boxes, bits, summary, c);
}

// Count and fill work on 16 lanes per cluster (four clusters per wavefront).
// The non-empty bitmask words of a cluster are first listed in LDS in
// ascending order (lane j of a group owns summary word j (+ 16 r), i.e. bitmask
// words 32 j .. 32 j + 31) and then read together, eight per lane, so that a
// cluster costs one round trip to memory for its words whatever their number
// (up to kWordWin per window).
constexpr uint32_t kCellLanes = 16;
constexpr uint32_t kWordWin = 128;
constexpr uint32_t kWordsPerLane = kWordWin / kCellLanes;
struct CellSmem {
    uint32_t words[256 / kCellLanes][kWordWin];
};

__device__ __forceinline__ uint32_t group_incl_scan(uint32_t v) {
    const uint32_t sl = threadIdx.x & (kCellLanes - 1u);
#pragma unroll
    for (uint32_t o = 1; o < kCellLanes; o <<= 1) {
        const uint32_t u = __shfl_up(v, o, kCellLanes);
        if (sl >= o) v += u;
    }
    return v;
}

// Calls f(list, n) for each window of up to kWordWin non-empty word indices of
// cluster cell (when on), in ascending order, uniformly over the cluster's 16
// lanes (SW is uniform over them).  clear: zero the summary words afterwards.
template <class F>
__device__ __forceinline__ void for_nonempty_words(uint32_t* __restrict__ summary, size_t ncell,
                                                   uint32_t cell, uint32_t SW, bool on, bool clear,
                                                   uint32_t* list, F&& f) {
    const uint32_t sl = threadIdx.x & (kCellLanes - 1u);
    for (uint32_t s0 = 0; s0 < SW; s0 += kCellLanes) {
        const uint32_t j = s0 + sl;
        const bool in = on && j < SW;
        uint32_t* const sp = summary + (in ? (size_t)j * ncell + cell : 0);
        const uint32_t sw = in ? *sp : 0u;
        const uint32_t c = (uint32_t)__popc(sw);
        const uint32_t incl = group_incl_scan(c);
        const uint32_t T = __shfl(incl, kCellLanes - 1u, kCellLanes);
        const uint32_t P = incl - c;
        for (uint32_t wb = 0; wb < T; wb += kWordWin) {
            uint32_t k = P;
            for (uint32_t m = sw; m; m &= m - 1u, ++k)
                if (k >= wb && k < wb + kWordWin) list[k - wb] = 32u * j + (uint32_t)__builtin_ctz(m);
            hl_wave_sync();
            f(list, T - wb < kWordWin ? T - wb : kWordWin);
            hl_wave_sync();
        }
        if (clear && sw) *sp = 0u;
    }
}

// number of members of a cluster (before the cap), returned to every lane of
// the cluster's group; lane 0 of the group also stores it in raw[cell]
__device__ __forceinline__ uint32_t count_cell(uint32_t ncell, uint32_t SW,
                                               const uint32_t* __restrict__ bits,
                                               const uint32_t* __restrict__ summary,
                                               uint32_t* __restrict__ raw, uint32_t cell,
                                               CellSmem& sm) {
    const uint32_t sl = threadIdx.x & (kCellLanes - 1u);
    const bool on = cell < ncell;
    const uint32_t* cb = bits + (on ? cell : 0u);  // word w at cb[w * ncell]
    uint32_t total = 0;
    for_nonempty_words(const_cast<uint32_t*>(summary), ncell, cell, SW, on, false,
                       sm.words[threadIdx.x / kCellLanes], [&](const uint32_t* list, uint32_t n) {
                           uint32_t wv[kWordsPerLane];
#pragma unroll
                           for (uint32_t q = 0; q < kWordsPerLane; ++q) {
                               const uint32_t e = kWordsPerLane * sl + q;
                               wv[q] = cb[(size_t)list[e < n ? e : 0u] * ncell];
                           }
#pragma unroll
                           for (uint32_t q = 0; q < kWordsPerLane; ++q)
                               if (kWordsPerLane * sl + q < n) total += (uint32_t)__popc(wv[q]);
                       });
#pragma unroll
    for (uint32_t o = kCellLanes / 2; o >= 1; o >>= 1) total += __shfl_xor(total, o, kCellLanes);
    if (raw && on && sl == 0) raw[cell] = total;
    return total;
}

// Per block of 16 clusters: adds each cluster's capped count to the sum of
// its scan tile (tile_sum null: no cluster), one atomic per run of equal
// tiles (a block's clusters lie in one tile except at view boundaries of a
// batch).
struct TileSumSmem {
    unsigned long long v[256 / kCellLanes];
    unsigned long long* p[256 / kCellLanes];
};
__device__ __forceinline__ void add_tile_sums(TileSumSmem& sm, unsigned long long* tile_sum,
                                              uint32_t capped) {
    if ((threadIdx.x & (kCellLanes - 1u)) == 0) {
        sm.v[threadIdx.x / kCellLanes] = capped;
        sm.p[threadIdx.x / kCellLanes] = tile_sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long* cur = nullptr;
        unsigned long long acc = 0;
        for (uint32_t i = 0; i < 256u / kCellLanes; ++i) {
            if (sm.p[i] != cur) {
                if (cur && acc) atomicAdd(cur, acc);
                cur = sm.p[i];
                acc = 0;
            }
            acc += sm.v[i];
        }
        if (cur && acc) atomicAdd(cur, acc);
    }
}

constexpr uint32_t kScanVPT = kScanTile / 256u;  // clusters per thread when a block reads a scan tile

// members of a cluster in ascending order, the first cnt of them written to
// dst (its capped, pool-truncated count); clears the cluster's bitmask words
// for the next call
__device__ __forceinline__ void fill_cell_at(uint32_t ncell, uint32_t SW, uint32_t* __restrict__ bits,
                                             uint32_t* __restrict__ summary, uint32_t cell,
                                             uint32_t cnt, uint32_t* __restrict__ dst, CellSmem& sm) {
    const uint32_t sl = threadIdx.x & (kCellLanes - 1u);
    const bool on = cell < ncell;
    uint32_t* cb = bits + (on ? cell : 0u);  // word w at cb[w * ncell]
    uint32_t written = 0;
    for_nonempty_words(summary, ncell, cell, SW, on, true,
                       sm.words[threadIdx.x / kCellLanes], [&](const uint32_t* list, uint32_t n) {
                           uint32_t wi[kWordsPerLane], wv[kWordsPerLane];
#pragma unroll
                           for (uint32_t q = 0; q < kWordsPerLane; ++q) {
                               const uint32_t e = kWordsPerLane * sl + q;
                               wi[q] = list[e < n ? e : 0u];
                               wv[q] = cb[(size_t)wi[q] * ncell];
                           }
                           uint32_t lt = 0;
#pragma unroll
                           for (uint32_t q = 0; q < kWordsPerLane; ++q) {
                               if (kWordsPerLane * sl + q >= n) wv[q] = 0u;
                               lt += (uint32_t)__popc(wv[q]);
                           }
                           const uint32_t incl = group_incl_scan(lt);
                           uint32_t pos = written + incl - lt;
#pragma unroll
                           for (uint32_t q = 0; q < kWordsPerLane; ++q) {
                               if (kWordsPerLane * sl + q >= n) continue;
                               cb[(size_t)wi[q] * ncell] = 0u;
                               for (uint32_t m = wv[q]; m; m &= m - 1u, ++pos)
                                   if (pos < cnt) dst[pos] = 32u * wi[q] + (uint32_t)__builtin_ctz(m);
                           }
                           written += __shfl(incl, kCellLanes - 1u, kCellLanes);
                       });
}

__device__ __forceinline__ void fill_cell(uint32_t ncell, uint32_t SW,
                                          uint32_t* __restrict__ bits,
                                          uint32_t* __restrict__ summary,
                                          const uint32_t* __restrict__ offsets,
                                          const uint32_t* __restrict__ counts,
                                          uint32_t* __restrict__ pool, uint32_t cell, CellSmem& sm) {
    const bool on = cell < ncell;
    fill_cell_at(ncell, SW, bits, summary, cell, on ? counts[cell] : 0u, on ? pool + offsets[cell] : pool, sm);
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// ------------------------------------------------------ scan fused into fill
// A fill block (16 consecutive clusters, in one scan tile of kScanTile) finds
// its clusters' offsets itself: the sums of the preceding scan tiles (from the
// count kernel), the capped raw counts of the tile's clusters before the
// block, and the prefix within the block -- at most 27 + 1008 values at 4K,
// read in one round trip -- then the pool truncation and overflow flags, then
// the lists.  The separate scan launch is gone.
struct ScanFillSmem {
    uint32_t capped[256 / kCellLanes];
    unsigned long long part[4];
    uint32_t flags;
};

__device__ __forceinline__ void scan_fill_block(const uint32_t* __restrict__ raw, uint32_t ncell,
                                                uint32_t SW, uint32_t* __restrict__ bits,
                                                uint32_t* __restrict__ summary, uint32_t cap,
                                                uint32_t pool_cap, uint32_t* __restrict__ offsets,
                                                uint32_t* __restrict__ counts, uint32_t* __restrict__ pool,
                                                uint32_t* __restrict__ flags_out,
                                                uint32_t* __restrict__ flags_out2, uint32_t first,
                                                CellSmem& cs, ScanFillSmem& sm) {
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t grp = t / kCellLanes, sl = t & (kCellLanes - 1u);
    if (first >= ncell) return;  // a batched view's padding cells (uniform)
    const unsigned long long* tile_sums =
        (const unsigned long long*)((const uint8_t*)raw + cluster_tile_sums_offset(ncell));
    const uint32_t tile = first / kScanTile, t0 = tile * kScanTile;
    if (t == 0) sm.flags = 0u;
    // sums of the preceding tiles, and the tile's clusters [t0, first)
    unsigned long long acc = 0;
    for (uint32_t j = t; j < tile; j += 256u) acc += tile_sums[j];
    const uint32_t c0 = t0 + kScanVPT * t;  // 4 clusters per thread, 16-B aligned
    if (c0 < first) {
        const uint4 u = *reinterpret_cast<const uint4*>(raw + c0);  // first <= ncell, a multiple of 16
        const uint32_t v[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) acc += (cap && v[q] > cap) ? cap : v[q];
    }
    acc = wave_sum_u64(acc);
    if (lane == 0) sm.part[wave] = acc;
    // the block's own clusters
    const uint32_t cell = first + grp;
    const bool on = cell < ncell;
    uint32_t n = on ? raw[cell] : 0u;
    uint32_t fl = 0;
    if (cap && n > cap) {
        n = cap;
        fl |= HL_OVERFLOW_CAP;
    }
    if (sl == 0) sm.capped[grp] = n;
    __syncthreads();
    unsigned long long off = sm.part[0] + sm.part[1] + sm.part[2] + sm.part[3];
    for (uint32_t j = 0; j < grp; ++j) off += sm.capped[j];
    const uint32_t o = off > pool_cap ? pool_cap : (uint32_t)off;
    uint32_t cnt = n;
    if (cnt > pool_cap - o) {
        cnt = pool_cap - o;
        fl |= HL_OVERFLOW_POOL;
    }
    if (on && sl == 0) {
        offsets[cell] = o;
        counts[cell] = cnt;
    }
    fill_cell_at(ncell, SW, bits, summary, cell, cnt, pool + o, cs);
    if (fl && sl == 0) atomicOr(&sm.flags, fl);
    __syncthreads();
    if (t == 0 && sm.flags) {
        atomicOr(flags_out, sm.flags);
        if (flags_out2) atomicOr(flags_out2, sm.flags);
    }
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

// ------------------------------------------------------ one view per launch
// The geometry kernel also resets the mark queue, the overflow words and the
// scan tile sums (it runs before every kernel that reads them).  Its blocks past the cells'
// prepare the lights' records (independent work that the mark kernel needs
// too), so that both take one launch.
__global__ __launch_bounds__(256) void k_cluster_geom(ClusterArgs a,
                                                      const GpuCameraUniforms* __restrict__ cam,
                                                      ColumnGeom* __restrict__ geom,
                                                      CellBox* __restrict__ boxes,
                                                      uint32_t* __restrict__ qcount,
                                                      uint32_t* __restrict__ flags,
                                                      uint32_t* __restrict__ flags2,
                                                      unsigned long long* __restrict__ tile_sums,
                                                      uint32_t ntiles,
                                                      const GpuLight* __restrict__ lights,
                                                      HotLight* __restrict__ hot,
                                                      CullLight* __restrict__ cl,
                                                      uint32_t* __restrict__ feature_flags,
                                                      uint32_t geom_blocks) {
    if (blockIdx.x >= geom_blocks) {
        prep_one(lights, nullptr, a.num_lights, cam, hot, cl, feature_flags,
                 (blockIdx.x - geom_blocks) * blockDim.x + threadIdx.x);
        return;
    }
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < kMarkQueues) qcount[g * kMarkCountStride] = 0u;
    if (g == 0) {
        *flags = 0u;
        if (flags2) *flags2 = 0u;
    }
    if (g < ntiles) tile_sums[g] = 0ull;
    geom_cell(a, cam, geom, boxes, g);
}

__global__ __launch_bounds__(256) void k_cluster_mark(ClusterArgs a,
                                                      const GpuCameraUniforms* __restrict__ cam,
                                                      const CullLight* __restrict__ cl,
                                                      const ColumnGeom* __restrict__ geom,
                                                      const CellBox* __restrict__ boxes,
                                                      uint32_t* __restrict__ bits,
                                                      uint32_t* __restrict__ summary, MarkQueue q) {
    const uint32_t li = blockIdx.x * 4u + (threadIdx.x >> 6);
    mark_light(a, cam, cl, geom, boxes, bits, summary, li, q, li, 0u);
}

// Queued chunks over a fixed grid of wavefronts: nw / kMarkQueues waves per
// sub-queue stride over its valid entries, min(count, seg), then exit.
__global__ __launch_bounds__(256) void k_cluster_mark_tail(ClusterArgs a,
                                                           const CullLight* __restrict__ cl,
                                                           const ColumnGeom* __restrict__ geom,
                                                           const CellBox* __restrict__ boxes,
                                                           uint32_t* __restrict__ bits,
                                                           uint32_t* __restrict__ summary, MarkQueue q) {
    const uint32_t w = blockIdx.x * 4u + (threadIdx.x >> 6), nw = gridDim.x * 4u;
    const uint32_t sub = w % kMarkQueues, step = nw / kMarkQueues;  // nw: a multiple of kMarkQueues
    const uint32_t n = min(hl_uniform(q.count[sub * kMarkCountStride]), q.seg);
    const uint2* seg = q.entries + (size_t)sub * q.seg;
    for (uint32_t e = w / kMarkQueues; e < n; e += step) {
        const uint2 en = seg[e];
        const uint32_t li = hl_uniform(en.x), chunk = hl_uniform(en.y) & 0xFFFFFFu;
        const CullLight L = load_light_uniform(cl, li);
        const uint4 pb = q.bounds[li];
        const MarkBox m = unpack_box(make_uint4(hl_uniform(pb.x), hl_uniform(pb.y), hl_uniform(pb.z),
                                                hl_uniform(pb.w)));
        mark_chunk(a, L, m, li, geom, boxes, bits, summary, chunk);
    }
}

__global__ __launch_bounds__(256) void k_cluster_count(uint32_t ncell, uint32_t SW,
                                                       const uint32_t* __restrict__ bits,
                                                       const uint32_t* __restrict__ summary,
                                                       uint32_t* __restrict__ raw, uint32_t cap) {
    __shared__ TileSumSmem sm;
    __shared__ CellSmem cs;
    const uint32_t cell = (blockIdx.x * blockDim.x + threadIdx.x) / kCellLanes;
    const uint32_t n = count_cell(ncell, SW, bits, summary, raw, cell, cs);
    unsigned long long* ts = (unsigned long long*)((uint8_t*)raw + cluster_tile_sums_offset(ncell));
    add_tile_sums(sm, cell < ncell ? ts + cell / kScanTile : nullptr, (cap && n > cap) ? cap : n);
}

__global__ __launch_bounds__(256) void k_cluster_fill(uint32_t ncell, uint32_t SW, const uint32_t* __restrict__ raw,
                                                      uint32_t* __restrict__ bits,
                                                      uint32_t* __restrict__ summary, uint32_t cap,
                                                      uint32_t pool_cap, uint32_t* __restrict__ offsets,
                                                      uint32_t* __restrict__ counts,
                                                      uint32_t* __restrict__ pool,
                                                      uint32_t* __restrict__ flags_out,
                                                      uint32_t* __restrict__ flags_out2) {
    __shared__ CellSmem cs;
    __shared__ ScanFillSmem sm;
    scan_fill_block(raw, ncell, SW, bits, summary, cap, pool_cap, offsets, counts, pool, flags_out, flags_out2,
                    blockIdx.x * (256u / kCellLanes), cs, sm);
}

// ------------------------------------------------- all views in one launch
// base[] holds nviews + 1 prefix offsets; returns the view owning index g.
// Cell ranges start on multiples of kBatchCellAlign, so a block of the
// geometry, count and fill kernels lies in one view: its lookup (and every
// view field it reads) depends on blockIdx only and stays scalar.
__device__ __forceinline__ uint32_t find_view(const uint32_t* __restrict__ base, uint32_t nviews,
                                              uint32_t g) {
    uint32_t lo = 0, hi = nviews;  // base[lo] <= g < base[hi]
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (base[mid] <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ CellBox* view_boxes(const BatchCullView& v) {
    return (CellBox*)((uint8_t*)v.geom + cluster_geom_offset_boxes_dev(v.ca.grid_x * v.ca.grid_y));
}

// ------------------------------------------------- clusters, brute force
// Two launches for small problems (cells x lights <= kSmallTests) on wide grids
// of few slices (cluster_path): every cell tests every light with the
// membership rule (cell_member), one wave per cell and four cells per block,
// the lights' culling records built per block into LDS kBfLights at a time,
// each cell's records built by its own wave in registers.  k_cluster_bf_count
// stores each cell's member count (and the lights' shading records);
// k_cluster_bf_fill finds each cell's offset from the capped counts before
// it, then writes the ascending list.  Membership does not depend on the
// order of evaluation, so the lists are the other paths'.
constexpr uint64_t kSmallTests = 1ull << 22;
constexpr uint32_t kBfCells = 4;  // one per wave
constexpr uint32_t kBfLights = 256;

struct BfSmem {
    CullLight light[kBfLights];
    uint32_t capped[kBfCells];
    unsigned long long part[4];
    uint32_t flags;
};

// The records of the wave's cell (every lane alike).
struct BfCell {
    ColumnGeom g;
    CellBox bx;
    float pad;
};
__device__ __forceinline__ BfCell bf_cell(const ClusterArgs& a, const GpuCameraUniforms* __restrict__ cam,
                                          uint32_t cell, uint32_t ncell) {
    BfCell c;
    const uint32_t ncol = a.grid_x * a.grid_y;
    if (cell < ncell) {
        cell_geometry(a, cam, cell % ncol, cell / ncol, true, c.g, c.bx);
        c.pad = a.slice_r_pad[cell / ncol];
    } else {  // no cell: no member (the records are not read)
        c.g = ColumnGeom{};
        c.bx = CellBox{};
        c.pad = 0.0f;
    }
    return c;
}

// For each light of the LDS chunk [l0, l0 + kBfLights) in ascending order, in
// groups of 64: f(group, pass) with pass this lane's light's membership in
// the wave's cell (uniform calls).
template <class F>
__device__ __forceinline__ void bf_chunk(const ClusterArgs& a, uint32_t l0, const BfCell& c, const BfSmem& sm,
                                         F&& f) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t nl = a.num_lights - l0 < kBfLights ? a.num_lights - l0 : kBfLights;
    for (uint32_t j0 = 0; j0 < nl; j0 += 64u) {
        const uint32_t j = j0 + lane;
        const bool pass = c.g.on != 0u && j < nl && cell_member(sm.light[j], c.g, c.bx, c.pad);
        f(j0, pass);
    }
}

__device__ __forceinline__ void bf_load_lights(const ClusterArgs& a, const GpuCameraUniforms* __restrict__ cam,
                                               const GpuLight* __restrict__ lights, uint32_t l0, BfSmem& sm) {
    __syncthreads();  // the previous chunk is no longer read
    const uint32_t i = l0 + threadIdx.x;
    if (i < a.num_lights) sm.light[threadIdx.x] = cull_light_at(lights, i, cam);
    __syncthreads();
}

__global__ __launch_bounds__(256) void k_cluster_bf_count(ClusterArgs a, const GpuCameraUniforms* __restrict__ cam,
                                                          const GpuLight* __restrict__ lights,
                                                          HotLight* __restrict__ hot,
                                                          uint32_t* __restrict__ feature_flags,
                                                          uint32_t* __restrict__ raw, uint32_t* __restrict__ flags,
                                                          uint32_t* __restrict__ flags2) {
    __shared__ BfSmem sm;
    const uint32_t ncell = a.grid_x * a.grid_y * a.grid_z;
    const uint32_t cell = blockIdx.x * kBfCells + (threadIdx.x >> 6);
    if (blockIdx.x == 0 && threadIdx.x == 0) {  // OR-ed by the fill launch
        *flags = 0u;
        if (flags2) *flags2 = 0u;
    }
    // the shading records, grid-stride over the lights
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < a.num_lights; i += gridDim.x * blockDim.x)
        prep_one(lights, nullptr, a.num_lights, cam, hot, nullptr, feature_flags, i);
    const BfCell c = bf_cell(a, cam, cell, ncell);
    uint32_t cnt = 0u;
    for (uint32_t l0 = 0; l0 < a.num_lights; l0 += kBfLights) {
        bf_load_lights(a, cam, lights, l0, sm);
        bf_chunk(a, l0, c, sm, [&](uint32_t, bool pass) { cnt += (uint32_t)__popcll(hl_ballot(pass)); });
    }
    if ((threadIdx.x & 63u) == 0 && cell < ncell) raw[cell] = cnt;
}

__global__ __launch_bounds__(256) void k_cluster_bf_fill(ClusterArgs a, const GpuCameraUniforms* __restrict__ cam,
                                                         const GpuLight* __restrict__ lights,
                                                         const uint32_t* __restrict__ raw, uint32_t pool_cap,
                                                         uint32_t* __restrict__ offsets, uint32_t* __restrict__ counts,
                                                         uint32_t* __restrict__ pool, uint32_t* __restrict__ flags,
                                                         uint32_t* __restrict__ flags2) {
    __shared__ BfSmem sm;
    const uint32_t ncell = a.grid_x * a.grid_y * a.grid_z, first = blockIdx.x * kBfCells;
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t cell = first + wave, cap = a.cap;
    // capped counts of the cells before the block
    unsigned long long acc = 0;
    for (uint32_t j = t; j < first; j += blockDim.x) {
        const uint32_t v = raw[j];
        acc += (cap && v > cap) ? cap : v;
    }
    acc = wave_sum_u64(acc);
    if (lane == 0) sm.part[wave] = acc;
    if (t == 0) sm.flags = 0u;
    if (t < kBfCells) {
        const uint32_t v = first + t < ncell ? raw[first + t] : 0u;
        sm.capped[t] = (cap && v > cap) ? cap : v;
    }
    const BfCell c = bf_cell(a, cam, cell, ncell);
    __syncthreads();
    // the wave's cell: offset, count after the cap and the pool truncation
    unsigned long long base = sm.part[0] + sm.part[1] + sm.part[2] + sm.part[3];
    for (uint32_t j = 0; j < wave; ++j) base += sm.capped[j];
    const uint32_t o = base > pool_cap ? pool_cap : (uint32_t)base;
    uint32_t cnt = sm.capped[wave], fl = 0u;
    if (cell < ncell && cap && raw[cell] > cap) fl |= HL_OVERFLOW_CAP;
    if (cnt > pool_cap - o) {
        cnt = pool_cap - o;
        fl |= HL_OVERFLOW_POOL;
    }
    if (lane == 0 && cell < ncell) {
        offsets[cell] = o;
        counts[cell] = cnt;
        if (fl) atomicOr(&sm.flags, fl);
    }
    uint32_t written = 0u;
    for (uint32_t l0 = 0; l0 < a.num_lights; l0 += kBfLights) {
        bf_load_lights(a, cam, lights, l0, sm);
        bf_chunk(a, l0, c, sm, [&](uint32_t j0, bool pass) {
            const uint64_t m = hl_ballot(pass);
            const uint32_t pos = written + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            if (pass && pos < cnt) pool[o + pos] = l0 + j0 + lane;
            written += (uint32_t)__popcll(m);
        });
    }
    __syncthreads();
    if (t == 0 && sm.flags) {
        atomicOr(flags, sm.flags);
        if (flags2) atomicOr(flags2, sm.flags);
    }
}

// --------------------------------------------- clusters, column by column
// The path of most grids (cluster_path).  A block owns one column of
// the grid, or kb slices of it when there are few columns (column_plan aims at
// kColBlocks blocks, two to three per CU):
//   k_col_prep   one thread per light: its shading and culling records and
//                its candidate box (light_box: the mark path's bound, packed
//                into 8 bytes);
//   k_col_count  scans the boxes (a compare each) into a bit per candidate
//                light, lists the candidates in LDS in ascending order, tests
//                each one (a lane) against the slices of its box with the
//                membership rule -- the four plane distances once per
//                candidate, as they do not depend on the slice -- and stores
//                the candidates with a bit per member slice, and the counts;
//   k_col_fill   the exclusive prefix of the capped counts, and the lists: the
//                candidates' slice bits transposed into a bit per (slice,
//                candidate) in LDS, each word of which a thread expands.
// Small problems (column_inline) skip k_col_prep: every count block bounds
// all lights itself, which costs less than a launch.
// Nothing is written per (cell, light): the bitmask over cells and lights of
// the mark path (57 MB at 32x18x48 cells and 16384 lights, two atomics per
// member) is not touched, and the geometry of a column lives in its block's
// LDS.  What bounds it is latency: the barriers and memory round trips of one
// block's chain, the fullest columns' (1200 candidates at 4K) above all.
// Measured (kernel times, us): 32x18x48 cells and 16384 lights 32 (prep 6.6,
// count 14.6, fill 10.7) against the mark path's 52 (geometry 5.8, mark 14.7,
// tail 4.5, count 10.5, fill 16.1); 16x9x24 and 1024 lights 21 against 50 for
// two brute-force launches, 256 lights 15 against 23.  1000 blocks aimed at
// instead of 512 made the 4K count 18.8.
constexpr uint32_t kColMaxColumns = 2048;
constexpr uint32_t kColBlocks = 512;
constexpr uint32_t kColChunk = 16384;  // lights scanned at a time
constexpr uint32_t kColThreads = 512;  // of a count block
// of one where there are more blocks than fit the chip at once at 512 threads
// (four per CU): what bounds them is then the rounds of blocks, and eight of half
// the size fit
constexpr uint32_t kColNarrow = 256;
constexpr uint32_t kColResident = 1024;
constexpr uint32_t kColInline = 512;   // lights every block bounds itself
constexpr uint32_t kColInlineCells = 8192;
constexpr uint32_t kColBatch = 512;    // candidates a fill block lists at a time
constexpr uint32_t kColGroup = 16;     // columns per partial sum of counts

// A light's candidate cells (inclusive ranges).  col: its columns, a byte each
// for x0, y0, 127 - x1 and 127 - y1 (in columns >> shift, at most 128 a side),
// so that one subtraction holds a column against all four ends; slice: s0 |
// s1 << 8, the top bit set for a light with a cone test.
struct LightBox {
    uint32_t col, slice;
};
constexpr uint32_t kNoBox = 0x7F7F7F7Fu;  // x >= 127 and x <= 0
constexpr uint32_t kBoxCone = 0x80000000u;
constexpr uint32_t kColMaxSide = 128;
__device__ __forceinline__ uint32_t box_s0(uint32_t s) { return s & 0xFFu; }
__device__ __forceinline__ uint32_t box_s1(uint32_t s) { return (s >> 8) & 0xFFu; }

// Sums of counts fit in 32 bits: cluster_path keeps cells x lights at 2^31.
struct ColumnArgs {
    const GpuCameraUniforms* cam;
    const GpuLight* lights;
    const uint32_t* subset;   // pool indices of the lights, or null
    HotLight* hot;
    CullLight* cull;          // per light (k_col_prep)
    uint32_t* box_col;        // LightBox::col per light, to a multiple of four (k_col_prep)
    uint32_t* box_slice;      // LightBox::slice per light (k_col_prep)
    uint32_t* feature_flags;
    uint32_t* num_cand;       // per block
    uint64_t* cand_slices;    // per block and candidate (n per block): its member slices, bit k: slice k0 + k
    uint32_t* cand;           // the candidate's light
    uint32_t* gsum;           // capped counts per (slice, group of columns) (k_col_prep)
    uint32_t* raw;            // per cell: members before the cap
    uint32_t* offsets;
    uint32_t* counts;
    uint32_t* pool;
    uint32_t pool_cap;
    uint32_t kb;              // slices per block
    uint32_t shift;           // of the columns in box_col
    uint32_t* flags;
    uint32_t* flags2;
};

// The slice tables as the candidate bound reads them: the near and far
// distances rounded outwards, and the paddings.
struct SliceTab {
    float sn[HL_MAX_SLICES], sf[HL_MAX_SLICES], pad[HL_MAX_SLICES];
};
__device__ __forceinline__ void load_slices(const ClusterArgs& a, SliceTab& t) {
    const uint32_t k = threadIdx.x;
    if (k < a.grid_z) {
        const float vn = a.slice_near[k], vf = a.slice_far[k];
        t.sn[k] = vn - 1e-5f * fabsf(vn);
        t.sf[k] = vf + 1e-5f * fabsf(vf);
        t.pad[k] = a.slice_r_pad[k];
    }
}

// Entries of the ascending table v[0, n) that are <= x, or < x (n <= 64).
template <bool kStrict>
__device__ __forceinline__ int count_below(const float* v, int n, float x) {
    int k = 0;
#pragma unroll
    for (int step = 64; step; step >>= 1) {
        const int j = k + step;
        if (j <= n && (kStrict ? v[j - 1] < x : v[j - 1] <= x)) k = j;
    }
    return k;
}

// light_cells for one thread, the slice limits by bisection.
__device__ __forceinline__ LightBox light_box(const ClusterArgs& a, const GpuCameraUniforms* __restrict__ cam,
                                             float4 vpos, bool cone, const SliceTab& t, uint32_t shift) {
    const int gx = (int)a.grid_x, gy = (int)a.grid_y, gz = (int)a.grid_z;
    int x0 = 0, x1 = gx - 1, y0 = 0, y1 = gy - 1, s0 = 0, s1 = gz - 1;
    const LightBox none{kNoBox, 0u};
    if (light_bounded(vpos)) {
        const float zc = -vpos.z;
        const float slack = 1e-5f * (fabsf(vpos.x) + fabsf(vpos.y) + fabsf(zc));
        const float r = fabsf(vpos.w);
        float rr = (r + t.pad[gz - 1]) * (1.0f + 1e-5f) + slack;
        s1 = count_below<false>(t.sn, gz, zc + rr) - 1;
        if (s1 < 0) return none;
        rr = (r + t.pad[s1]) * (1.0f + 1e-5f) + slack;
        s0 = count_below<true>(t.sf, gz, zc - rr);
        while (s1 >= 0 && !(t.sn[s1] <= zc + rr)) --s1;  // seldom any: rr only shrank
        const float p00 = cam->proj[0], p11 = cam->proj[5];
        if (zc > 1e-4f && p00 > 0.0f && p11 > 0.0f)
            light_columns(a, p00, p11, vpos, zc, rr, &x0, &x1, &y0, &y1);
    }
    x0 = clampi(x0, 0, gx - 1);
    x1 = clampi(x1, -1, gx - 1);
    y0 = clampi(y0, 0, gy - 1);
    y1 = clampi(y1, -1, gy - 1);
    s0 = clampi(s0, 0, gz - 1);
    s1 = clampi(s1, -1, gz - 1);
    if (x1 < x0 || y1 < y0 || s1 < s0) return none;
    const uint32_t bx0 = (uint32_t)x0 >> shift, by0 = (uint32_t)y0 >> shift;
    const uint32_t bx1 = (uint32_t)x1 >> shift, by1 = (uint32_t)y1 >> shift;
    return LightBox{bx0 | by0 << 8 | (127u - bx1) << 16 | (127u - by1) << 24,
                    (uint32_t)s0 | (uint32_t)s1 << 8 | (cone ? kBoxCone : 0u)};
}

// Whether the box holds a column, given as column_key: every byte of the key
// (with its top bit as a guard) at least the box's.
constexpr uint32_t kByteTops = 0x80808080u;
__device__ __forceinline__ uint32_t column_key(uint32_t cx, uint32_t cy) {
    return kByteTops | cx | cy << 8 | (127u - cx) << 16 | (127u - cy) << 24;
}
__device__ __forceinline__ bool box_has_column(uint32_t col, uint32_t key) {
    return ((key - col) & kByteTops) == kByteTops;
}
__device__ __forceinline__ bool box_has_slices(uint32_t s, uint32_t k0, uint32_t k1) {
    return box_s0(s) <= k1 && box_s1(s) >= k0;
}

// A cell's box and the padding of its slice, as two 16-byte LDS reads.
struct alignas(16) ColCell {
    float lo[3], hi[3], pad, unused;
};
struct ColGeomSmem {
    float3 pl[4];                 // the column's planes
    ColCell cell[HL_MAX_SLICES];  // the block's cells
    SliceTab tab;
};
template <uint32_t CHUNK, uint32_t NT>
struct ColCountSmem {
    ColGeomSmem g;
    uint32_t words[CHUNK / 32];  // candidate bits of the chunk
    uint16_t list[CHUNK];        // the candidates, ascending, chunk-relative
    uint32_t wave_sum[NT / 64];
    uint32_t cnt[NT / 64][HL_MAX_SLICES];
};
struct ColFillSmem {
    uint32_t bits[HL_MAX_SLICES][kColBatch / 32];  // members of the batch per slice
    uint32_t light[kColBatch];
    uint32_t off[HL_MAX_SLICES], cnt[HL_MAX_SLICES], run[HL_MAX_SLICES];
    uint32_t row[HL_MAX_SLICES], part[HL_MAX_SLICES], base[4];
};

// The block's column and slices: blocks run slice group by slice group over
// the columns.
struct ColBlock {
    uint32_t col, cx, cy, k0, nk, ncol;
};
__device__ __forceinline__ ColBlock col_block(const ClusterArgs& a, uint32_t block, uint32_t kb) {
    ColBlock c;
    c.ncol = a.grid_x * a.grid_y;
    c.col = block % c.ncol;
    c.cx = c.col % a.grid_x;
    c.cy = c.col / a.grid_x;
    c.k0 = block / c.ncol * kb;
    c.nk = min(kb, a.grid_z - c.k0);
    return c;
}

// The planes of the column and the boxes of its cells (cell_geometry's, a
// plane or a box per thread of the block's last two waves, which have no
// lights to bound in the smallest problems) into LDS; the caller
// synchronises.  Returns whether the column covers pixels (uniform).
template <uint32_t NT>
__device__ __forceinline__ bool col_setup(const ClusterArgs& a, const GpuCameraUniforms* __restrict__ cam,
                                          const ColBlock& c, ColGeomSmem& sm) {
    const uint32_t t = threadIdx.x - (NT - 64u);  // wraps: another wave
    if (t < c.nk) {
        ColumnGeom g;
        CellBox bx;
        cell_geometry(a, cam, c.col, c.k0 + t, false, g, bx);
        ColCell& o = sm.cell[t];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            o.lo[i] = bx.lo[i];
            o.hi[i] = bx.hi[i];
        }
        o.pad = a.slice_r_pad[c.k0 + t];
    }
    float l = 0.0f, r = 0.0f, b = 0.0f, tp = 0.0f;
    const bool on = column_rect(a, c.cx, c.cy, &l, &r, &b, &tp);
    const uint32_t p = threadIdx.x - (NT - 128u);
    if (on && p < 4u) {
        // (l, b, l, t), (r, t, r, b), (l, t, r, t), (r, b, l, b)
        const float x0 = (p == 0u || p == 2u) ? l : r, y0 = (p == 0u || p == 3u) ? b : tp;
        const float x1 = (p == 0u || p == 3u) ? l : r, y1 = (p == 0u || p == 2u) ? tp : b;
        sm.pl[p] = hl_x_plane(cam->proj[0], cam->proj[5], x0, y0, x1, y1);
    }
    return on;
}

// Lists the set bits of words[0, nw) (nw <= W) in list, ascending; returns
// their number.  Called by all NT threads; ends with the list visible to them.
template <uint32_t W, uint32_t NT>
__device__ __forceinline__ uint32_t list_bits(const uint32_t* words, uint32_t nw, uint16_t* list,
                                              uint32_t* wave_sum) {
    constexpr uint32_t kPer = (W + NT - 1u) / NT;  // words per thread
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    uint32_t w[kPer], n = 0;
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
        const uint32_t i = t * kPer + q;
        w[q] = i < nw ? words[i] : 0u;
        n += (uint32_t)__popc(w[q]);
    }
    uint32_t incl = n;
#pragma unroll
    for (uint32_t o = 1; o < 64u; o <<= 1) {
        const uint32_t u = __shfl_up(incl, o, 64);
        if (lane >= o) incl += u;
    }
    if (lane == 63u) wave_sum[wave] = incl;
    __syncthreads();
    uint32_t pos = incl - n, total = 0;
#pragma unroll
    for (uint32_t q = 0; q < NT / 64u; ++q) {
        if (q < wave) pos += wave_sum[q];
        total += wave_sum[q];
    }
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q)
        for (uint32_t m = w[q]; m; m &= m - 1u)
            list[pos++] = (uint16_t)(32u * (t * kPer + q) + (uint32_t)__builtin_ctz(m));
    __syncthreads();
    return total;
}

// Sets in words the bits of the lights j < nl whose column box holds the key's
// column (boxes to a multiple of four) and that keep(j) accepts.  A lane takes
// 4 kAhead lights at a time, their boxes loaded together, and sets the bits of
// the few that pass; blocks start at different lights, so that they do not
// all read the same lines at the same time.  Called by all NT threads; the
// caller synchronises before the words are read.
template <uint32_t NT, class F>
__device__ __forceinline__ void scan_boxes(const uint32_t* __restrict__ boxes, uint32_t nl, uint32_t key,
                                           uint32_t block, uint32_t* words, F&& keep) {
    constexpr uint32_t kAhead = 8u;
    const uint32_t t = threadIdx.x;
    for (uint32_t w = t; w < (nl + 31u) / 32u; w += NT) words[w] = 0u;
    __syncthreads();
    const uint4* const cols = reinterpret_cast<const uint4*>(boxes);
    const uint32_t quads = (nl + 3u) / 4u, groups = (quads + NT - 1u) / NT, rot = block % groups;
    for (uint32_t g0 = 0; g0 < groups; g0 += kAhead) {
        uint4 v[kAhead];
#pragma unroll
        for (uint32_t q = 0; q < kAhead; ++q) {
            const uint32_t g = g0 + q + rot, j = (g < groups ? g : g - groups) * NT + t;
            v[q] = make_uint4(kNoBox, kNoBox, kNoBox, kNoBox);
            if (g0 + q < groups && j < quads) v[q] = cols[j];
        }
        uint32_t hits = 0;
#pragma unroll
        for (uint32_t q = 0; q < kAhead; ++q) {
            hits |= box_has_column(v[q].x, key) ? 1u << (4u * q) : 0u;
            hits |= box_has_column(v[q].y, key) ? 2u << (4u * q) : 0u;
            hits |= box_has_column(v[q].z, key) ? 4u << (4u * q) : 0u;
            hits |= box_has_column(v[q].w, key) ? 8u << (4u * q) : 0u;
        }
        for (; hits; hits &= hits - 1u) {
            const uint32_t b = (uint32_t)__builtin_ctz(hits), g = g0 + (b >> 2) + rot;
            const uint32_t j = 4u * ((g < groups ? g : g - groups) * NT + t) + (b & 3u);
            if (keep(j)) atomicOr(&words[j >> 5], 1u << (j & 31u));
        }
    }
}

// The OR of a 64-bit word over the wave, in every lane (scalar).
__device__ __forceinline__ uint64_t wave_or(uint64_t v) {
    const auto red = [](uint32_t x) {
        x |= (uint32_t)hl_dpp_i<0xB1>(0, (int)x);
        x |= (uint32_t)hl_dpp_i<0x4E>(0, (int)x);
        x |= (uint32_t)hl_dpp_i<0x141>(0, (int)x);
        x |= (uint32_t)hl_dpp_i<0x140>(0, (int)x);
        x |= (uint32_t)hl_dpp_i<0x142, 0xA>(0, (int)x);
        x |= (uint32_t)hl_dpp_i<0x143, 0xC>(0, (int)x);
        return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
    };
    return (uint64_t)red((uint32_t)v) | (uint64_t)red((uint32_t)(v >> 32)) << 32;
}

// The slices [k0, k0 + nk) of the column that light L
// (candidate slices box_slice) is a member of: the rule of cell_member.  !(d < -r) for every
// plane is !(min d < -r): the comparison is false for a NaN distance, which
// fminf drops.
__device__ __forceinline__ uint64_t member_slices(const ColBlock& c, const ColGeomSmem& sm, const CullLight& L,
                                                  uint32_t box_slice) {
#pragma clang fp contract(off)
    float d = __builtin_inff();
#pragma unroll
    for (int p = 0; p < 4; ++p)
        d = fminf(d, hl_x_dot3(sm.pl[p].x, sm.pl[p].y, sm.pl[p].z, L.vpos.x, L.vpos.y, L.vpos.z) + 0.0f);
    const uint32_t ka = max(box_s0(box_slice), c.k0), kz = min(box_s1(box_slice), c.k0 + c.nk - 1u);
    uint64_t m = 0;
    for (uint32_t k = ka; k <= kz; ++k) {
        const float4* q = reinterpret_cast<const float4*>(&sm.cell[k - c.k0]);
        const float4 q0 = q[0], q1 = q[1];
        const float rc = L.vpos.w + q1.z;
        const float3 lo = make_float3(q0.x, q0.y, q0.z), hi = make_float3(q0.w, q1.x, q1.y);
        bool in = !(d < -rc) && hl_x_sphere_aabb(L.vpos, rc, lo, hi);
        if (in && (box_slice & kBoxCone)) in = hl_x_cone_cell(L.vpos, L.axis, L.aux.x, q1.z, lo, hi);
        if (in) m |= 1ull << (k - c.k0);
    }
    return m;
}

// A wave per block: the lights' chains (loads, FP64 band, bisections) over all
// CUs rather than over n / 256 of them.
__device__ __forceinline__ void col_prep_block(const ClusterArgs& a, const ColumnArgs& p, uint32_t block,
                                               uint32_t nblocks, uint32_t nsum, SliceTab& tab) {
    load_slices(a, tab);
    __syncthreads();
    const uint32_t i = block * 64u + threadIdx.x;
    if (i == 0) {
        *p.flags = 0u;
        if (p.flags2) *p.flags2 = 0u;
    }
    for (uint32_t j = i; j < nsum; j += nblocks * 64u) p.gsum[j] = 0u;
    if (i >= a.num_lights) {
        if (i < ((a.num_lights + 3u) & ~3u)) p.box_col[i] = kNoBox;
        return;
    }
    const CullLight L = cull_light_at(p.lights, p.subset ? p.subset[i] : i, p.cam);
    p.cull[i] = L;
    const LightBox b = light_box(a, p.cam, L.vpos, L.cone.w != kNoCone, tab, p.shift);
    p.box_col[i] = b.col;
    p.box_slice[i] = b.slice;
    prep_one(p.lights, p.subset, a.num_lights, p.cam, p.hot, nullptr, p.feature_flags, i);
}

__global__ __launch_bounds__(64) void k_col_prep(ClusterArgs a, ColumnArgs p, uint32_t nsum) {
    __shared__ SliceTab tab;
    col_prep_block(a, p, blockIdx.x, gridDim.x, nsum, tab);
}

// INLINE: the block bounds every light itself (a light per thread; the cone
// terms come with the candidate's record), and the blocks share the shading
// records.
template <uint32_t CHUNK, uint32_t NT, bool INLINE>
__device__ __forceinline__ void col_count_block(const ClusterArgs& a, const ColumnArgs& p, uint32_t block,
                                                uint32_t nblocks, ColCountSmem<CHUNK, NT>& sm,
                                                uint32_t* inline_slices) {
    constexpr uint32_t kWaves = NT / 64u;
    static_assert(!INLINE || CHUNK == NT, "a light per thread");
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6, n = a.num_lights;
    const ColBlock c = col_block(a, block, p.kb);
    float4 pr = make_float4(0.0f, 0.0f, 0.0f, 0.0f), dro = pr;
    uint32_t type = 0u;
    if (INLINE && t < n) {  // in flight during the set-up
        pr = *reinterpret_cast<const float4*>(p.lights[t].position_range);
        dro = *reinterpret_cast<const float4*>(p.lights[t].direction_outer);
        type = p.lights[t].light_type;
    }
    if (INLINE) {  // the bounds read the slice tables
        load_slices(a, sm.g.tab);
        __syncthreads();
    }
    const bool on = col_setup<NT>(a, p.cam, c, sm.g);
    const uint32_t key = column_key(c.cx >> p.shift, c.cy >> p.shift), k1 = c.k0 + c.nk - 1u;
    [[maybe_unused]] const bool part_column = c.nk != a.grid_z;
    if (INLINE && block == 0 && t == 0) {
        *p.flags = 0u;
        if (p.flags2) *p.flags2 = 0u;
    }
    uint32_t cnt = 0;  // lane k: members of slice k0 + k among the wave's candidates
    uint32_t done = 0;
    uint32_t* const cand = p.cand + (size_t)block * n;
    uint64_t* const cand_slices = p.cand_slices + (size_t)block * n;
    for (uint32_t l0 = 0; l0 < n; l0 += CHUNK) {
        const uint32_t nl = min(CHUNK, n - l0), nw = (nl + 31u) / 32u;
        if (l0) __syncthreads();  // the previous chunk's list is no longer read
        if (INLINE) {
            bool m = false;
            if (t < n) {
                const float* v = p.cam->view;
                const float4 vp = make_float4(hl_x_mat_row(v, 0, pr.x, pr.y, pr.z, 1.0f),
                                              hl_x_mat_row(v, 1, pr.x, pr.y, pr.z, 1.0f),
                                              hl_x_mat_row(v, 2, pr.x, pr.y, pr.z, 1.0f),
                                              type == HL_LIGHT_DIRECTIONAL ? __builtin_inff() : pr.w);
                const LightBox b = light_box(a, p.cam, vp, type == HL_LIGHT_SPOT, sm.g.tab, p.shift);
                inline_slices[t] = b.slice;
                m = on && box_has_column(b.col, key) && box_has_slices(b.slice, c.k0, k1);
            }
            const uint64_t bal = hl_ballot(m);
            if (lane < 2u) sm.words[2u * wave + lane] = lane ? (uint32_t)(bal >> 32) : (uint32_t)bal;
        } else {
            scan_boxes<NT>(p.box_col + l0, nl, key, block, sm.words, [&](uint32_t j) {
                return on && (!part_column || box_has_slices(p.box_slice[l0 + j], c.k0, k1));
            });
        }
        __syncthreads();
        const uint32_t total = list_bits<CHUNK / 32u, NT>(sm.words, nw, sm.list, sm.wave_sum);
        for (uint32_t j0 = 0; j0 + wave * 64u < total; j0 += NT) {  // uniform over the wave
            const uint32_t j = j0 + t;
            uint64_t m = 0;
            if (j < total) {
                const uint32_t r = sm.list[j], li = l0 + r;
                CullLight L;
                uint32_t slice;
                if (INLINE) {
                    slice = inline_slices[r];
                    L = cull_light_at(p.lights, r, p.cam);
                    if (L.cone.w == kNoCone) slice &= ~kBoxCone;
                } else {
                    const CullLight* cl = p.cull + li;
                    slice = p.box_slice[li];
                    L.vpos = hl_ld4(&cl->vpos);
                    L.axis = L.aux = L.vpos;
                    if (slice & kBoxCone) {
                        L.axis = hl_ld4(&cl->axis);
                        L.aux.x = cl->aux.x;
                    }
                }
                m = member_slices(c, sm.g, L, slice);
                cand[done + j] = li;
                cand_slices[done + j] = m;
            }
            // the slices that some candidate of the wave is a member of
            for (uint64_t any = wave_or(m); any; any &= any - 1ull) {
                const uint32_t k = (uint32_t)__builtin_ctzll(any);
                const uint32_t members = (uint32_t)__popcll(hl_ballot((m >> k) & 1ull));
                cnt += lane == k ? members : 0u;
            }
        }
        done += total;
    }
    sm.cnt[wave][lane] = cnt;
    __syncthreads();
    if (t < c.nk) {
        uint32_t v = 0;
#pragma unroll
        for (uint32_t w = 0; w < kWaves; ++w) v += sm.cnt[w][t];
        p.raw[c.col + c.ncol * (c.k0 + t)] = v;
        const uint32_t capped = (a.cap && v > a.cap) ? a.cap : v;
        if (!INLINE && capped)
            atomicAdd(p.gsum + (size_t)(c.k0 + t) * ((c.ncol + kColGroup - 1u) / kColGroup) + c.col / kColGroup,
                      capped);
    }
    if (t == 0u) p.num_cand[block] = done;
    // the shading records, last: no wait stands on them
    if (INLINE)
        for (uint32_t i = block * NT + t; i < n; i += nblocks * NT)
            prep_one(p.lights, nullptr, n, p.cam, p.hot, nullptr, p.feature_flags, i);
}

// Sum over the aligned groups of 2^lp consecutive lanes.
__device__ __forceinline__ uint32_t part_sum(uint32_t v, uint32_t lp) {
    for (uint32_t o = 1; o < (1u << lp); o <<= 1) v += __shfl_xor(v, (int)o, 64);
    return v;
}

// SUMS: the counts before the block's cells come from the partial sums of
// kColGroup columns and the counts of the column's own group, else from the
// counts of every cell before them.  A thread sums a share of one slice's
// row (256 threads over the block's slices); those loads, the cells' own
// counts and the first candidates go out together.
template <bool SUMS>
__device__ __forceinline__ void col_fill_block(const ClusterArgs& a, const ColumnArgs& p, uint32_t block,
                                               ColFillSmem& sm) {
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6, n = a.num_lights, cap = a.cap;
    const ColBlock c = col_block(a, block, p.kb);
    const auto capped = [&](uint32_t v) { return (cap && v > cap) ? cap : v; };
    const uint32_t* const cand = p.cand + (size_t)block * n;
    const uint64_t* const cand_slices = p.cand_slices + (size_t)block * n;
    const uint32_t total = hl_uniform(p.num_cand[block]);
    const uint32_t own = t < c.nk ? p.raw[c.col + c.ncol * (c.k0 + t)] : 0u;
    uint32_t li[2] = {0u, 0u};
    uint64_t ms[2] = {0ull, 0ull};
    const auto load = [&](uint32_t b0) {
#pragma unroll
        for (uint32_t q = 0; q < 2u; ++q) {
            const uint32_t j = b0 + 256u * q + t;
            ms[q] = 0ull;
            if (j < total) {
                li[q] = cand[j];
                ms[q] = cand_slices[j];
            }
        }
    };
    load(0u);
    // rows before the block's first slice
    const uint32_t ngrp = (c.ncol + kColGroup - 1u) / kColGroup, grp = c.col / kColGroup;
    uint32_t acc = 0;
    if (SUMS) {
#pragma unroll 4
        for (uint32_t i = t; i < c.k0 * ngrp; i += 256u) acc += p.gsum[i];
    } else {
#pragma unroll 8
        for (uint32_t i = t; i < c.k0 * c.ncol; i += 256u) acc += capped(p.raw[i]);
    }
    // the block's rows: 2^lp threads (at most a wave) per row
    uint32_t lp = 2;
    while (lp < 6u && (c.nk << (lp + 1u)) <= 256u) ++lp;
    const uint32_t k = t >> lp, part = t & ((1u << lp) - 1u);
    uint32_t row = 0, before = 0;
    if (k < c.nk) {
        const size_t r = c.k0 + k;
        if (SUMS) {
#pragma unroll 4
            for (uint32_t g = part; g < ngrp; g += 1u << lp) {
                const uint32_t v = p.gsum[r * ngrp + g];
                row += v;
                before += g < grp ? v : 0u;
            }
            for (uint32_t i = grp * kColGroup + part; i < c.col; i += 1u << lp) before += capped(p.raw[r * c.ncol + i]);
        } else {
#pragma unroll 4
            for (uint32_t i = part; i < c.ncol; i += 1u << lp) {
                const uint32_t v = capped(p.raw[r * c.ncol + i]);
                row += v;
                before += i < c.col ? v : 0u;
            }
        }
    }
    if (c.k0) acc = part_sum(acc, 6u);
    row = part_sum(row, lp);
    before = part_sum(before, lp);
    if (lane == 0u) sm.base[wave] = acc;
    if (k < c.nk && part == 0u) {
        sm.row[k] = row;
        sm.part[k] = before;
    }
    for (uint32_t i = t; i < c.nk * (kColBatch / 32u); i += 256u) sm.bits[0][i] = 0u;
    __syncthreads();
    if (t < 64u) {  // the block's slices: at most 64
        const uint32_t v = t < c.nk ? sm.row[t] : 0u;
        uint32_t incl = v;
#pragma unroll
        for (uint32_t o = 1; o < 64u; o <<= 1) {
            const uint32_t u = __shfl_up(incl, o, 64);
            if (lane >= o) incl += u;
        }
        uint32_t fl = 0u;
        if (t < c.nk) {
            const uint32_t off = sm.base[0] + sm.base[1] + sm.base[2] + sm.base[3] + incl - v + sm.part[t];
            const uint32_t cell = c.col + c.ncol * (c.k0 + t);
            uint32_t cnt = capped(own);
            fl = cap && own > cap ? HL_OVERFLOW_CAP : 0u;
            const uint32_t o = off > p.pool_cap ? p.pool_cap : off;
            if (cnt > p.pool_cap - o) {
                cnt = p.pool_cap - o;
                fl |= HL_OVERFLOW_POOL;
            }
            p.offsets[cell] = o;
            p.counts[cell] = cnt;
            sm.off[t] = o;
            sm.cnt[t] = cnt;
            sm.run[t] = 0u;
        }
        const uint32_t any = (hl_ballot(fl & HL_OVERFLOW_CAP) ? HL_OVERFLOW_CAP : 0u) |
                             (hl_ballot(fl & HL_OVERFLOW_POOL) ? HL_OVERFLOW_POOL : 0u);
        if (any && t == 0u) {
            atomicOr(p.flags, any);
            if (p.flags2) atomicOr(p.flags2, any);
        }
    }
    for (uint32_t b0 = 0; b0 < total; b0 += kColBatch) {
        // the candidates' slice bits, transposed
#pragma unroll
        for (uint32_t q = 0; q < 2u; ++q) {
            const uint32_t j = 256u * q + t;
            sm.light[j] = li[q];
            for (uint64_t m = ms[q]; m; m &= m - 1ull)
                atomicOr(&sm.bits[__builtin_ctzll(m)][j >> 5], 1u << (j & 31u));
        }
        if (b0 + kColBatch < total) load(b0 + kColBatch);  // the next batch's, in flight meanwhile
        __syncthreads();
        // a thread per word, 16 lanes per slice
        static_assert(kColBatch == 512, "16 words per slice, two candidates per thread");
        for (uint32_t i = t; i < ((c.nk * 16u + 255u) & ~255u); i += 256u) {
            const uint32_t s = i >> 4, w = i & 15u;
            const bool on = s < c.nk;
            uint32_t m = on ? sm.bits[s][w] : 0u;
            const uint32_t v = (uint32_t)__popc(m);
            uint32_t incl = v;
#pragma unroll
            for (uint32_t o = 1; o < 16u; o <<= 1) {
                const uint32_t u = __shfl_up(incl, o, 16);
                if (w >= o) incl += u;
            }
            if (!on) continue;
            const uint32_t run = sm.run[s], cnt = sm.cnt[s], o = sm.off[s];
            for (uint32_t pos = run + incl - v; m && pos < cnt; ++pos, m &= m - 1u)
                p.pool[o + pos] = sm.light[32u * w + (uint32_t)__builtin_ctz(m)];
            sm.bits[s][w] = 0u;
            hl_wave_sync();  // the slice's 16 lanes have read its run
            if (w == 15u) sm.run[s] = run + incl;
        }
        __syncthreads();  // bits, lights and runs before the next batch's
    }
}

template <uint32_t CHUNK, uint32_t NT, bool INLINE>
__global__ __launch_bounds__(NT) void k_col_count(ClusterArgs a, ColumnArgs p) {
    __shared__ ColCountSmem<CHUNK, NT> sm;
    uint32_t* is = nullptr;
    if constexpr (INLINE) {
        __shared__ uint32_t slices[CHUNK];
        is = slices;
    }
    col_count_block<CHUNK, NT, INLINE>(a, p, blockIdx.x, gridDim.x, sm, is);
}

template <bool SUMS>
__global__ __launch_bounds__(256) void k_col_fill(ClusterArgs a, ColumnArgs p) {
    __shared__ ColFillSmem sm;
    col_fill_block<SUMS>(a, p, blockIdx.x, sm);
}

// Slices per block and blocks: whole columns when there are at least `aim` of
// them, else enough groups of slices.
struct ColumnPlan {
    uint32_t kb, blocks;
};
static uint32_t column_groups(uint32_t ncol) { return (ncol + kColGroup - 1u) / kColGroup; }
static ColumnPlan column_plan(uint32_t ncol, uint32_t gz, uint32_t aim) {
    const uint32_t want = std::min(gz, (aim + ncol - 1u) / ncol);
    const uint32_t kb = (gz + want - 1u) / want;
    return ColumnPlan{kb, ncol * ((gz + kb - 1u) / kb)};
}
// The scan reads 4 bytes per (block, light) and the candidates take 12 bytes
// of scratch each in the worst case: the column path up to 2048 columns (128
// a side) and 2^25 (block, light) pairs, 403 MB (113 MB at 32x18x48 cells and
// 16384 lights, where the mark path's bitmask takes 57).  That is a bound on
// memory, not on speed: calls at it, us, columns / mark path, 64x32x24 cells and
// 16384 lights 84 / 202, 64x32x48 101 / 285, 16x9x24 and 58000 145 / 208.  A
// caller without the memory takes the mark path.
static bool use_columns(uint32_t gx, uint32_t gy, uint32_t gz, uint64_t n) {
    const uint32_t ncol = gx * gy;
    return gx <= kColMaxSide && gy <= kColMaxSide && ncol <= kColMaxColumns &&
           column_plan(ncol, gz, kColBlocks).blocks * n <= (1ull << 25);
}
// Small problems of a single view on wider grids: the brute force where a
// column is only a cell or a few (up to 65536 cells: its fill reads every count
// before its own), else the column path (the lights' boxes in coarser columns);
// the mark path's two atomics per member make it the slowest where lights are
// large, though the fastest where they are small.  Calls, us, brute force /
// columns / mark path with the lights of a scene, and with every light in every
// cell: 256x144x1 cells and 100 lights 144 / 368 / 294, 136 / 447 / 450; 80x45x1
// and 1000 47 / 55 / 79, 43 / 106 / 119; 160x90x1 and 290 71 / 153 / 166, 82 /
// 299 / 217; 128x72x4 and 100 143 / 89 / 31, 135 / 155 / 490; 64x36x8 and 200
// 78 / 35 / 29, 71 / 73 / 288; 80x45x24 and 48 414 / 55 / 36, 407 / 134 / 1020;
// 200x1x1 and 5000 115 / 31 / 56, 86 / 41 / 130.
ClusterPath cluster_path(uint32_t gx, uint32_t gy, uint32_t gz, uint32_t n) {
    const uint32_t ncol = gx * gy;
    const uint64_t ncell = (uint64_t)ncol * gz;
    if (use_columns(gx, gy, gz, n)) return ClusterPath::kColumns;
    if (ncell * n > kSmallTests) return ClusterPath::kMark;
    return gz < 4u && ncol > kColBlocks && ncell <= 65536u ? ClusterPath::kBruteForce : ClusterPath::kColumns;
}
static bool column_inline(uint32_t ncell, uint32_t n) { return n <= kColInline && ncell <= kColInlineCells; }

// Scratch of one view: candidate slices and lights, partial sums, candidate
// numbers, boxes.
static size_t column_scratch(uint8_t* base, uint32_t ncol, uint32_t gz, uint32_t n, uint32_t blocks, ColumnArgs* p) {
    size_t o = 0;
    const auto take = [&](size_t bytes) {
        uint8_t* q = base + o;
        o += (bytes + 255) & ~(size_t)255;
        return q;
    };
    uint8_t* slices = take(8 * (size_t)blocks * n);
    uint8_t* cand = take(4 * (size_t)blocks * n);
    uint8_t* gsum = take(4 * (size_t)column_groups(ncol) * gz);
    uint8_t* num = take(4 * (size_t)blocks);
    uint8_t* box_col = take(4 * ((size_t)n + 3));
    uint8_t* box_slice = take(4 * (size_t)n);
    if (p) {
        p->cand_slices = (uint64_t*)slices;
        p->cand = (uint32_t*)cand;
        p->gsum = (uint32_t*)gsum;
        p->num_cand = (uint32_t*)num;
        p->box_col = (uint32_t*)box_col;
        p->box_slice = (uint32_t*)box_slice;
    }
    return o;
}
size_t column_scratch_bytes(uint32_t gx, uint32_t gy, uint32_t gz, uint32_t n) {
    const uint32_t ncol = gx * gy;
    return column_scratch(nullptr, ncol, gz, n, column_plan(ncol, gz, kColBlocks).blocks, nullptr);
}

// The column path of many views: the same three steps, a launch each, the
// blocks of a view one after the other (base: first block of each view, and
// the end).  The plan aims at a number of blocks for the whole batch, shared
// out by cells x lights.  Lights are scanned kBatchColChunk at a time: the
// smaller list (8 KB against 32) lets four blocks share a CU, or eight of half
// the threads where the plan has more blocks than that (kColNarrow: a 4K frame
// of 2040 columns and 16 lights 59.1 -> 54.1 us, four 1080p views of 2040 and 256
// lights 145 -> 117; with 512 threads frames of many columns and few lights were
// slower than on the mark path, 57.0 and 159).  24 faces of 128^2 with 512 lights
// each and two 1032x1104 eyes with 4096: 7 + 23 + 8 us against the mark path's 51
// (geometry 6, mark 12, tail 11, count 9, fill 12).
struct BatchColumnView {
    ClusterArgs a;
    ColumnArgs p;
    uint32_t nsum, nprep;
};
// read through the constant address space, as k_shade_batch reads its views
typedef const __attribute__((address_space(4))) BatchColumnView* ConstColumnViews;
constexpr uint32_t kBatchColChunk = 4096;
// The view of a block (base strictly ascending): every lane compares one
// entry, one round trip instead of the bisection's log2(nviews).
__device__ __forceinline__ uint32_t view_of_block(const uint32_t* __restrict__ base, uint32_t nviews) {
    uint32_t v = 0;
    for (uint32_t q = 1; q < nviews; q += 64u) {
        const uint32_t i = q + hl_lane();
        v += (uint32_t)__popcll(hl_ballot(i < nviews && base[i] <= blockIdx.x));
    }
    return hl_uniform(v);
}

__global__ __launch_bounds__(64) void k_batch_col_prep(ConstColumnViews __restrict__ views,
                                                       const uint32_t* __restrict__ base, uint32_t nviews) {
    __shared__ SliceTab tab;
    const uint32_t vi = view_of_block(base, nviews);
    const BatchColumnView& v = *(const BatchColumnView*)&views[vi];
    col_prep_block(v.a, v.p, blockIdx.x - base[vi], v.nprep, v.nsum, tab);
}

template <uint32_t NT>
__global__ __launch_bounds__(NT) void k_batch_col_count(ConstColumnViews __restrict__ views,
                                                        const uint32_t* __restrict__ base, uint32_t nviews) {
    __shared__ ColCountSmem<kBatchColChunk, NT> sm;
    const uint32_t vi = view_of_block(base, nviews);
    const BatchColumnView& v = *(const BatchColumnView*)&views[vi];
    col_count_block<kBatchColChunk, NT, false>(v.a, v.p, blockIdx.x - base[vi], 0u, sm, nullptr);
}

__global__ __launch_bounds__(256) void k_batch_col_fill(ConstColumnViews __restrict__ views,
                                                        const uint32_t* __restrict__ base, uint32_t nviews) {
    __shared__ ColFillSmem sm;
    const uint32_t vi = view_of_block(base, nviews);
    const BatchColumnView& v = *(const BatchColumnView*)&views[vi];
    col_fill_block<true>(v.a, v.p, blockIdx.x - base[vi], sm);
}

size_t batch_column_view_size() { return sizeof(BatchColumnView); }

BatchColumnPlan batch_column_plan(uint32_t gx, uint32_t gy, uint32_t gz, uint32_t n, uint32_t aim) {
    BatchColumnPlan r;
    if (!use_columns(gx, gy, gz, n)) return r;
    const ColumnPlan cp = column_plan(gx * gy, gz, aim);
    r.blocks = cp.blocks;
    r.prep_blocks = n ? (n + 63u) / 64u : 1u;
    r.scratch = column_scratch(nullptr, gx * gy, gz, n, cp.blocks, nullptr);
    return r;
}

void batch_column_view(void* dst, const BatchCullView& v, const GpuLight* pool, void* scratch, uint32_t aim) {
    BatchColumnView& o = *(BatchColumnView*)dst;
    const uint32_t ncol = v.ca.grid_x * v.ca.grid_y, gz = v.ca.grid_z, n = v.ca.num_lights;
    const ColumnPlan cp = column_plan(ncol, gz, aim);
    o.a = v.ca;
    o.p = ColumnArgs{};
    o.p.cam = v.cam;
    o.p.lights = pool;
    o.p.subset = v.subset;
    o.p.hot = v.hot;
    o.p.cull = v.cull;
    o.p.raw = v.raw;
    o.p.offsets = v.offsets;
    o.p.counts = v.counts;
    o.p.pool = v.pool;
    o.p.pool_cap = v.pool_cap;
    o.p.kb = cp.kb;
    o.p.flags = v.flags;
    (void)column_scratch((uint8_t*)scratch, ncol, gz, n, cp.blocks, &o.p);
    o.nsum = column_groups(ncol) * gz;
    o.nprep = n ? (n + 63u) / 64u : 1u;
}

hipError_t launch_batch_columns(hipStream_t s, const void* views, const uint32_t* prep_base, const uint32_t* col_base,
                                uint32_t nviews, uint32_t prep_blocks, uint32_t col_blocks) {
    if (nviews == 0) return hipSuccess;
    const ConstColumnViews v = (ConstColumnViews)views;
    hipError_t e;
    k_batch_col_prep<<<prep_blocks, 64, 0, s>>>(v, prep_base, nviews);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (col_blocks > kColResident) k_batch_col_count<kColNarrow><<<col_blocks, kColNarrow, 0, s>>>(v, col_base, nviews);
    else k_batch_col_count<kColThreads><<<col_blocks, kColThreads, 0, s>>>(v, col_base, nviews);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    k_batch_col_fill<<<col_blocks, 256, 0, s>>>(v, col_base, nviews);
    return hipGetLastError();
}

// The mark path of many views.
// Cells of every view, then (blocks past geom_blocks) the lights of every
// view gathered from the pool, in one launch.
__global__ __launch_bounds__(256) void k_batch_geom(const BatchCullView* __restrict__ views,
                                                    const uint32_t* __restrict__ cell_base,
                                                    uint32_t nviews, uint32_t* __restrict__ qcount,
                                                    const GpuLight* __restrict__ pool,
                                                    const uint32_t* __restrict__ light_base,
                                                    uint32_t geom_blocks) {
    // the views' overflow words start each frame at zero (nviews <= 255)
    if (blockIdx.x == 0 && threadIdx.x < nviews) *views[threadIdx.x].flags = 0u;
    if (blockIdx.x >= geom_blocks) {
        const uint32_t l = (blockIdx.x - geom_blocks) * blockDim.x + threadIdx.x;
        if (l >= light_base[nviews]) return;
        const uint32_t vi = find_view(light_base, nviews, l);
        const BatchCullView& v = views[vi];
        prep_one(pool, v.subset, v.ca.num_lights, v.cam, v.hot, v.cull, nullptr, l - light_base[vi]);
        return;
    }
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < kMarkQueues) qcount[g * kMarkCountStride] = 0u;
    const uint32_t vi = find_view(cell_base, nviews, blockIdx.x * blockDim.x);
    const BatchCullView& v = views[vi];
    const uint32_t c = g - cell_base[vi];
    if (c < cluster_scan_tiles_dev(v.ncell))
        ((unsigned long long*)((uint8_t*)v.raw + cluster_tile_sums_offset(v.ncell)))[c] = 0ull;
    geom_cell(v.ca, v.cam, (ColumnGeom*)v.geom, view_boxes(v), c);
}

// one wavefront per light of any view; queue entries carry the global index
__global__ __launch_bounds__(256) void k_batch_mark(const BatchCullView* __restrict__ views,
                                                    const uint32_t* __restrict__ light_base,
                                                    uint32_t nviews, MarkQueue q) {
    const uint32_t g = hl_uniform(blockIdx.x * 4u + (threadIdx.x >> 6));
    if (g >= light_base[nviews]) return;
    const uint32_t vi = find_view(light_base, nviews, g);
    const BatchCullView& v = views[vi];
    mark_light(v.ca, v.cam, v.cull, (const ColumnGeom*)v.geom, view_boxes(v), v.bits, v.summary,
               g - light_base[vi], q, g, vi);
}

__global__ __launch_bounds__(256) void k_batch_mark_tail(const BatchCullView* __restrict__ views,
                                                         const uint32_t* __restrict__ light_base,
                                                         uint32_t nviews, MarkQueue q) {
    const uint32_t w = blockIdx.x * 4u + (threadIdx.x >> 6), nw = gridDim.x * 4u;
    const uint32_t sub = w % kMarkQueues, step = nw / kMarkQueues;  // nw: a multiple of kMarkQueues
    const uint32_t n = min(hl_uniform(q.count[sub * kMarkCountStride]), q.seg);
    const uint2* seg = q.entries + (size_t)sub * q.seg;
    for (uint32_t e = w / kMarkQueues; e < n; e += step) {
        const uint2 en = seg[e];
        const uint32_t g = hl_uniform(en.x), packed = hl_uniform(en.y);
        const uint32_t vi = packed >> 24, chunk = packed & 0xFFFFFFu;
        const BatchCullView& v = views[vi];
        const uint32_t li = g - light_base[vi];
        const CullLight L = load_light_uniform(v.cull, li);
        const uint4 pb = q.bounds[g];
        const MarkBox m = unpack_box(make_uint4(hl_uniform(pb.x), hl_uniform(pb.y), hl_uniform(pb.z),
                                                hl_uniform(pb.w)));
        mark_chunk(v.ca, L, m, li, (const ColumnGeom*)v.geom, view_boxes(v), v.bits, v.summary, chunk);
    }
}

__global__ __launch_bounds__(256) void k_batch_count(const BatchCullView* __restrict__ views,
                                                     const uint32_t* __restrict__ cell_base,
                                                     uint32_t nviews) {
    __shared__ TileSumSmem sm;
    __shared__ CellSmem cs;
    constexpr uint32_t kCellsPerBlock = 256u / kCellLanes;
    const uint32_t vi = find_view(cell_base, nviews, blockIdx.x * kCellsPerBlock);
    const BatchCullView& v = views[vi];
    const uint32_t c = blockIdx.x * kCellsPerBlock + threadIdx.x / kCellLanes - cell_base[vi];
    const uint32_t n = count_cell(v.ncell, v.SW, v.bits, v.summary, v.raw, c, cs);
    unsigned long long* ts = (unsigned long long*)((uint8_t*)v.raw + cluster_tile_sums_offset(v.ncell));
    const uint32_t cap = v.ca.cap;
    add_tile_sums(sm, c < v.ncell ? ts + c / kScanTile : nullptr, (cap && n > cap) ? cap : n);
}

// scan and fill of 16 clusters of one view (scan_fill_block)
__global__ __launch_bounds__(256) void k_batch_fill(const BatchCullView* __restrict__ views,
                                                    const uint32_t* __restrict__ cell_base,
                                                    uint32_t nviews) {
    constexpr uint32_t kCellsPerBlock = 256u / kCellLanes;
    const uint32_t vi = find_view(cell_base, nviews, blockIdx.x * kCellsPerBlock);
    const BatchCullView& v = views[vi];
    __shared__ CellSmem cs;
    __shared__ ScanFillSmem sm;
    scan_fill_block(v.raw, v.ncell, v.SW, v.bits, v.summary, v.ca.cap, v.pool_cap, v.offsets, v.counts, v.pool,
                    v.flags, nullptr, blockIdx.x * kCellsPerBlock - cell_base[vi], cs, sm);
}

// grid of the queued-chunk launches: 64 wavefronts per sub-queue, enough to
// spread the chunks of a few heavy lights over every CU whatever the light
// count (idle waves read one counter and exit); a multiple of kMarkQueues / 4
static uint32_t tail_blocks(uint32_t) { return 16u * kMarkQueues; }

hipError_t launch_batch_cull(hipStream_t s, const GpuLight* pool, const BatchCullView* views,
                             const uint32_t* light_base, const uint32_t* cell_base, uint32_t nviews,
                             uint32_t total_lights, uint32_t total_cells, const MarkQueue& mq) {
    if (nviews == 0) return hipSuccess;
    if (total_cells % kBatchCellAlign) return hipErrorInvalidValue;
    hipError_t e;
    const uint32_t geom_blocks = total_cells / 256u;  // total_cells: kBatchCellAlign multiple
    k_batch_geom<<<geom_blocks + (total_lights + 255) / 256, 256, 0, s>>>(views, cell_base, nviews, mq.count,
                                                                          pool, light_base, geom_blocks);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (total_lights) {
        k_batch_mark<<<(total_lights + 3) / 4, 256, 0, s>>>(views, light_base, nviews, mq);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        k_batch_mark_tail<<<tail_blocks(total_lights), 256, 0, s>>>(views, light_base, nviews, mq);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    const uint32_t cblocks = total_cells / (256u / kCellLanes);  // total_cells: kBatchCellAlign multiple
    k_batch_count<<<cblocks, 256, 0, s>>>(views, cell_base, nviews);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    k_batch_fill<<<cblocks, 256, 0, s>>>(views, cell_base, nviews);
    return hipGetLastError();
}

// ------------------------------------------------------ tile cull, binned
// Candidate tiles of a light for the tile planes' test (inclusive rectangle;
// false when empty).  Necessary conditions of passing a tile's four planes
// (normals (1, 0, l/p00), -(1, 0, r/p00), (0, -1, -t/p11), (0, 1, b/p11),
// normalised by s = sqrt(1 + e^2/p00^2) <= fx for an edge |e| <= 1), with
// the light's centre c, view distance zc = -c.z and radius r (|r| <= rr):
//  - in front (zc > 0): l <= p00 (cx + rr fx) / zc and r >= p00 (cx - rr fx) / zc,
//    rows alike with p11 (the cluster cull's bound);
//  - behind the camera (zc < 0, |zc| = -zc): the planes' half-spaces meet
//    only near the mirrored projection, l >= p00 (-cx - rr fx) / |zc| and
//    r <= p00 (rr fx - cx) / |zc|, t <= p11 (rr fy - cy) / |zc| and
//    b >= p11 (-rr fy - cy) / |zc|;
//  - within 1e-4 of the camera plane, a non-finite centre or radius, or a
//    camera with p00 or p11 <= 0: every tile.
// Rounded outwards as the cluster cull's candidates: rr widened by 1e-5 of
// itself and of |cx| + |cy| + |zc|, the pixel bounds by 1e-5 of their
// magnitude plus a quarter pixel.
__device__ __forceinline__ bool light_tiles(const GpuCameraUniforms* __restrict__ cam, const LightCullParams& p,
                                            float4 c, int* tx0, int* tx1, int* ty0, int* ty1) {
    const int ntx = (int)p.num_tiles_x, nty = (int)p.num_tiles_y;
    *tx0 = 0;
    *tx1 = ntx - 1;
    *ty0 = 0;
    *ty1 = nty - 1;
    const float zc = -c.z, p00 = cam->proj[0], p11 = cam->proj[5];
    if (!__builtin_isfinite(c.w) || !__builtin_isfinite(c.x) || !__builtin_isfinite(c.y) ||
        !__builtin_isfinite(zc) || !(p00 > 0.0f && p11 > 0.0f) || fabsf(zc) <= 1e-4f)
        return ntx > 0 && nty > 0;
    const float slack = 1e-5f * (fabsf(c.x) + fabsf(c.y) + fabsf(zc));
    const float rr = fabsf(c.w) * (1.0f + 1e-5f) + slack;
    const float fx = __builtin_amdgcn_sqrtf(1.0f + hl_f_rcp(p00 * p00));
    const float fy = __builtin_amdgcn_sqrtf(1.0f + hl_f_rcp(p11 * p11));
    const float iz = hl_f_rcp(fabsf(zc));
    float nx0, nx1, nt, nb;  // column edges: l <= nx1, r >= nx0 (front) or l >= nx0, r <= nx1 (behind)
    if (zc > 0.0f) {
        nx0 = p00 * (c.x - rr * fx) * iz;
        nx1 = p00 * (c.x + rr * fx) * iz;
        nb = p11 * (c.y - rr * fy) * iz;  // t >= nb
        nt = p11 * (c.y + rr * fy) * iz;  // b <= nt
    } else {
        nx0 = p00 * (-c.x - rr * fx) * iz;
        nx1 = p00 * (rr * fx - c.x) * iz;
        nt = p11 * (rr * fy - c.y) * iz;   // t <= nt
        nb = p11 * (-rr * fy - c.y) * iz;  // b >= nb
    }
    const float fw = (float)p.screen_width, fh = (float)p.screen_height;
    // in both cases the candidate pixel columns lie in [px0, px1] and rows in
    // [py0, py1]: front, from l <= nx1 and r >= nx0; behind, from l >= nx0 and
    // r <= nx1 (the same interval, reached from the other side)
    float px0 = (nx0 + 1.0f) * 0.5f * fw, px1 = (nx1 + 1.0f) * 0.5f * fw;
    float py0 = (1.0f - nt) * 0.5f * fh, py1 = (1.0f - nb) * 0.5f * fh;
    px0 -= 1e-5f * fabsf(px0) + 0.25f;
    px1 += 1e-5f * fabsf(px1) + 0.25f;
    py0 -= 1e-5f * fabsf(py0) + 0.25f;
    py1 += 1e-5f * fabsf(py1) + 0.25f;
    const float its = 1.0f / (float)HL_TILE_SIZE;  // exact
    // clamped to [-1, n] before the conversion (NaN: the whole range)
    const int x0 = (int)fminf(fmaxf(floorf(px0 * its), -1.0f), (float)ntx);
    const int x1 = (int)fmaxf(fminf(floorf(px1 * its), (float)ntx), -1.0f);
    const int y0 = (int)fminf(fmaxf(floorf(py0 * its), -1.0f), (float)nty);
    const int y1 = (int)fmaxf(fminf(floorf(py1 * its), (float)nty), -1.0f);
    *tx0 = clampi(x0, 0, ntx - 1);
    *tx1 = clampi(x1, -1, ntx - 1);
    *ty0 = clampi(y0, 0, nty - 1);
    *ty1 = clampi(y1, -1, nty - 1);
    return *tx1 >= *tx0 && *ty1 >= *ty0;
}

// A block owns a super-tile of sx x sy tiles (at most 8 x 8; tile_plan): it
// scans the lights' boxes in super-tiles as the column path does, lists the
// candidates in LDS, finds the tiles of each one (a lane) as a bit per tile,
// and a wave per row of tiles lists the candidates of each tile by ballot, the
// first HL_MAX_LIGHTS_PER_TILE, in LDS; whole lists then go out in rows of
// 256 bytes.  It stops when every tile is full.
// A light in front of the camera is held against the columns and rows of the
// super-tile first (tile_mask: the four plane tests are tests of a column or a
// row but for rounding), and only against the planes of the tiles that this
// leaves undecided; a tile's planes are built once, a plane per thread (some
// 200 VALU instructions of exact divisions and square roots each).
// k_tile_prep bounds the lights ahead of it, or every block all of them
// (at most kColInline).
// Measured (kernel times, us): 3840x2160 and 16384 lights 27 (prep 5, cull 22)
// against 78 for the five launches over a bitmask of super-tiles and lights
// that this replaces (prep 5.7, bin 15, count 15, fill 25, lists 17), 1280x720
// and 64 lights 8.3 against 22.  What bounds it is latency, as in the column
// path; half of the 4K launch is tile_mask.  Exact tests of every tile of the
// rectangle in its place, with a store per list entry: 37 (and 8192 lights at
// a time 30: two half-empty batches).
constexpr uint32_t kTileMax = 64;  // tiles per block
struct TileArgs {
    const GpuCameraUniforms* cam;
    const GpuLight* lights;
    HotLight* hot;
    uint32_t* feature_flags;
    LightCullParams p;
    uint32_t sx, sy, nsx;       // tiles per super-tile, super-tiles per row
    uint32_t shift;             // boxes are in super-tiles >> shift (128 a side)
    float4* vpos;               // per light (k_tile_prep): centre and range
    uint2* rect;                // candidate tiles: x0 | y0 << 16, x1 | y1 << 16
    uint32_t* box;              // the same in shifted super-tiles, as LightBox::col
    uint32_t* lists;
    uint32_t* counts;
};

// The candidate tiles of a light, and the super-tiles that hold them.
__device__ __forceinline__ uint32_t tile_box(const TileArgs& a, float4 vpos, uint2* rect) {
    int x0, x1, y0, y1;
    *rect = make_uint2(1u, 0u);
    if (!light_tiles(a.cam, a.p, vpos, &x0, &x1, &y0, &y1)) return kNoBox;
    *rect = make_uint2((uint32_t)x0 | (uint32_t)y0 << 16, (uint32_t)x1 | (uint32_t)y1 << 16);
    const uint32_t fx = a.sx << a.shift, fy = a.sy << a.shift;
    return (uint32_t)x0 / fx | ((uint32_t)y0 / fy) << 8 | (127u - (uint32_t)x1 / fx) << 16 |
           (127u - (uint32_t)y1 / fy) << 24;
}

__device__ __forceinline__ float4 light_vpos(float4 pr, uint32_t type, const float* __restrict__ v) {
    return make_float4(hl_x_mat_row(v, 0, pr.x, pr.y, pr.z, 1.0f), hl_x_mat_row(v, 1, pr.x, pr.y, pr.z, 1.0f),
                       hl_x_mat_row(v, 2, pr.x, pr.y, pr.z, 1.0f),
                       type == HL_LIGHT_DIRECTIONAL ? __builtin_inff() : pr.w);
}

__global__ __launch_bounds__(64) void k_tile_prep(TileArgs a) {
    const uint32_t i = blockIdx.x * 64u + threadIdx.x, n = a.p.num_lights;
    if (i >= n) {
        if (i < ((n + 3u) & ~3u)) a.box[i] = kNoBox;
        return;
    }
    const float4 v = light_vpos(*reinterpret_cast<const float4*>(a.lights[i].position_range), a.lights[i].light_type,
                                a.cam->view);
    uint2 rect;
    a.vpos[i] = v;
    a.box[i] = tile_box(a, v, &rect);
    a.rect[i] = rect;
    prep_one(a.lights, nullptr, n, a.cam, a.hot, nullptr, a.feature_flags, i);
}

// An edge of the super-tile's columns or rows in NDC, and the length
// sqrt(1 + (edge / p)^2) of its plane's unnormalised normal.
struct TileEdge {
    float e, s;
};
template <uint32_t CHUNK>
struct TileSmem {
    alignas(16) float pl[kTileMax][12];  // the tiles' planes, tile y * 8 + x
    TileEdge left[8], right[8], top[8], bottom[8];
    uint32_t words[CHUNK / 32];
    uint16_t list[CHUNK];
    uint8_t tiles[kColBatch][8];         // a byte per row of tiles, a bit per tile
    uint32_t out[kTileMax][HL_MAX_LIGHTS_PER_TILE];
    uint32_t run[kTileMax];
    uint32_t wave_sum[kColThreads / 64];
    uint32_t open[2];                    // waves with a tile that still takes lights, per batch parity
};

// One axis of tile_mask: the tiles k in [k0, k1] that a centre at a = p c / zc
// and a radius b = p r / zc certainly (sure) or possibly (may) pass: the lower
// edge needs lo <= a + b s, the upper hi >= a - b s.
template <class E>
__device__ __forceinline__ void axis_mask(const E* lo, const E* hi, int k0, int k1, float a, float b, float margin,
                                          uint32_t& sure, uint32_t& may) {
    sure = may = 0u;
    for (int k = k0; k <= k1; ++k) {
        const float v = fminf(__builtin_fmaf(b, lo[k].s, a - lo[k].e), __builtin_fmaf(b, hi[k].s, hi[k].e - a));
        const float m = margin + 1e-5f * (fabsf(a) + fabsf(b) * fmaxf(lo[k].s, hi[k].s) + 1.0f);
        sure |= v > m ? 1u << k : 0u;
        may |= !(v < -m) ? 1u << k : 0u;
    }
}

// The bytes of rows set in `rows`, each `cols`.
__device__ __forceinline__ uint64_t mask_product(uint32_t rows, uint32_t cols) {
    uint64_t m = 0;
#pragma unroll
    for (uint32_t y = 0; y < 8u; ++y) m |= (uint64_t)((rows >> y) & 1u ? cols : 0u) << (8u * y);
    return m;
}

// The tiles of the super-tile that light c passes (bit y * 8 + x), of the
// candidate rectangle [x0, x1] x [y0, y1].  In real numbers a light at view
// distance zc > 0 passes a tile's left plane when l <= p00 (cx + r s) / zc
// (s = sqrt(1 + l^2 / p00^2)), a condition of the tile's column alone, and so
// on; the FP32 planes come from a cross product of two rays some theta
// apart, whose components carry an error of at most about 1e-6: the plane
// turns by 1e-6 / theta, moving the distance by that times |c|.  gx and gy
// are four times that per |c| / zc, in NDC; what lies within takes the exact
// test, and so does every tile for the other lights.
template <uint32_t CHUNK>
__device__ __forceinline__ uint64_t tile_mask(const TileSmem<CHUNK>& sm, float p00, float p11, float gx, float gy,
                                              float4 c, int x0, int x1, int y0, int y1) {
    if (x0 > x1 || y0 > y1) return 0ull;
    uint32_t xs = 0u, xm = (2u << x1) - (1u << x0), ys = 0u, ym = (2u << y1) - (1u << y0);
    const float zc = -c.z;
    if (zc > 1e-4f && p00 > 0.0f && p11 > 0.0f && __builtin_isfinite(zc) && __builtin_isfinite(c.x) &&
        __builtin_isfinite(c.y) && __builtin_isfinite(c.w)) {
        const float iz = hl_f_rcp(zc), far = (fabsf(c.x) + fabsf(c.y) + zc) * iz;
        axis_mask(sm.left, sm.right, x0, x1, p00 * c.x * iz, p00 * c.w * iz, gx * far, xs, xm);
        // rows run downwards: the lower edge of the axis is the bottom
        axis_mask(sm.bottom, sm.top, y0, y1, p11 * c.y * iz, p11 * c.w * iz, gy * far, ys, ym);
    }
    uint64_t in = mask_product(ys, xs);
    for (uint64_t m = mask_product(ym, xm) & ~in; m; m &= m - 1ull) {
        const uint32_t tile = (uint32_t)__builtin_ctzll(m);
        const float4* q = reinterpret_cast<const float4*>(sm.pl[tile]);
        const float4 q0 = q[0], q1 = q[1], q2 = q[2];
        const float3 pl[4] = {make_float3(q0.x, q0.y, q0.z), make_float3(q0.w, q1.x, q1.y),
                              make_float3(q1.z, q1.w, q2.x), make_float3(q2.y, q2.z, q2.w)};
        if (tile_pass(pl, c)) in |= 1ull << tile;
    }
    return in;
}

template <uint32_t CHUNK, bool INLINE>
__global__ __launch_bounds__(kColThreads) void k_tile_cull(TileArgs a) {
    constexpr uint32_t NT = kColThreads;
    static_assert(NT == 512, "a wave per row of tiles");
    static_assert(kColBatch == NT, "a candidate per thread");
    static_assert(!INLINE || CHUNK == NT, "a light per thread");
    __shared__ TileSmem<CHUNK> sm;
    float4* s_vpos = nullptr;
    uint2* s_rect = nullptr;
    if constexpr (INLINE) {
        __shared__ float4 v[CHUNK];
        __shared__ uint2 r[CHUNK];
        s_vpos = v;
        s_rect = r;
    }
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = hl_uniform(t >> 6), n = a.p.num_lights;
    const uint32_t sux = blockIdx.x % a.nsx, suy = blockIdx.x / a.nsx;
    const uint32_t tx0 = sux * a.sx, ty0 = suy * a.sy;
    const uint32_t nx = min(a.sx, a.p.num_tiles_x - tx0), ny = min(a.sy, a.p.num_tiles_y - ty0);
    float4 pr = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    uint32_t type = 0u;
    if (INLINE && t < n) {  // in flight while the planes are built
        pr = *reinterpret_cast<const float4*>(a.lights[t].position_range);
        type = a.lights[t].light_type;
    }
    const float p00 = a.cam->proj[0], p11 = a.cam->proj[5];
    float gx, gy;
    {
        const float fw = (float)a.p.screen_width, fh = (float)a.p.screen_height, ts = (float)HL_TILE_SIZE;
        const uint32_t tile = t >> 2, x = tile & 7u, y = tile >> 3;
        if (t < 4u * kTileMax && x < nx && y < ny) {
            const float3 pl = tile_plane(a.cam, a.p, tx0 + x, ty0 + y, t & 3u);
            float* o = &sm.pl[tile][3u * (t & 3u)];
            o[0] = pl.x;
            o[1] = pl.y;
            o[2] = pl.z;
        }
        if (t >= 256u && t < 256u + 32u) {  // the edges, as tile_plane's
            const uint32_t k = t & 7u, side = (t >> 3) & 3u;
            const bool row = side >= 2u;
            const float at = (float)((row ? ty0 : tx0) + k + (side & 1u)) * ts / (row ? fh : fw) * 2.0f;
            const float e = row ? fmaxf(1.0f - at, -1.0f) : fminf(at - 1.0f, 1.0f);
            const float q = e * hl_f_rcp(row ? p11 : p00);
            (side == 0u ? sm.left : side == 1u ? sm.right : side == 2u ? sm.top : sm.bottom)[k] =
                TileEdge{e, __builtin_amdgcn_sqrtf(1.0f + q * q)};
        }
        // the smallest angles under which the block's tiles are seen: their
        // NDC sizes (the screen's last tiles may be narrower), foreshortened
        // at the screen's corners
        const float ix = hl_f_rcp(p00), iy = hl_f_rcp(p11), corner = 1.0f + ix * ix + iy * iy;
        const float wx = fminf((fw - (float)(tx0 + nx - 1u) * ts), ts) * 2.0f * hl_f_rcp(fw);
        const float wy = fminf((fh - (float)(ty0 + ny - 1u) * ts), ts) * 2.0f * hl_f_rcp(fh);
        gx = 4e-6f * p00 * corner * corner * hl_f_rcp(wy * iy);  // a column's planes span the tile's height
        gy = 4e-6f * p11 * corner * corner * hl_f_rcp(wx * ix);
    }
    if (t < kTileMax) sm.run[t] = 0u;
    if (t < 2u) sm.open[t] = 0u;
    uint32_t batch = 0;
    const uint32_t key = column_key(sux >> a.shift, suy >> a.shift);
    bool open = true;  // some tile still takes lights (uniform)
    for (uint32_t l0 = 0; l0 < n && open; l0 += CHUNK) {
        const uint32_t nl = min(CHUNK, n - l0), nw = (nl + 31u) / 32u;
        if (INLINE) {
            bool m = false;
            if (t < n) {
                const float4 v = light_vpos(pr, type, a.cam->view);
                uint2 rect;
                m = box_has_column(tile_box(a, v, &rect), key);
                s_vpos[t] = v;
                s_rect[t] = rect;
            }
            const uint64_t bal = hl_ballot(m);
            if (lane < 2u) sm.words[2u * wave + lane] = lane ? (uint32_t)(bal >> 32) : (uint32_t)bal;
        } else {
            if (l0) __syncthreads();  // the previous chunk's list is no longer read
            scan_boxes<NT>(a.box + l0, nl, key, blockIdx.x, sm.words, [](uint32_t) { return true; });
        }
        __syncthreads();
        const uint32_t total = list_bits<CHUNK / 32u, NT>(sm.words, nw, sm.list, sm.wave_sum);
        for (uint32_t b0 = 0; b0 < total && open; b0 += kColBatch) {
            uint64_t mask = 0;
            if (b0 + t < total) {
                const uint32_t li = sm.list[b0 + t];
                const float4 c = INLINE ? s_vpos[li] : hl_ld4(a.vpos + l0 + li);
                const uint2 r = INLINE ? s_rect[li] : a.rect[l0 + li];
                // empty ranges where the boxes are coarser than the super-tiles
                mask = tile_mask(sm, p00, p11, gx, gy, c, max((int)(r.x & 0xFFFFu) - (int)tx0, 0),
                                 min((int)(r.y & 0xFFFFu) - (int)tx0, (int)nx - 1),
                                 max((int)(r.x >> 16) - (int)ty0, 0), min((int)(r.y >> 16) - (int)ty0, (int)ny - 1));
            }
            *reinterpret_cast<uint64_t*>(sm.tiles[t]) = mask;
            __syncthreads();
            // the next batch's flag: every wave's read of it for the previous
            // batch is before this barrier, the next batch's adds are after
            // the one below
            if (t == 0u) sm.open[(batch + 1u) & 1u] = 0u;
            // the wave's row of tiles
            bool some = false;
            if (wave < ny) {
                uint32_t run[8];
#pragma unroll
                for (uint32_t x = 0; x < 8u; ++x) run[x] = hl_uniform(sm.run[8u * wave + x]);
                for (uint32_t g = 0; g < kColBatch && b0 + g < total; g += 64u) {
                    const uint32_t row = sm.tiles[g + lane][wave];
                    if (hl_ballot(row != 0u) == 0) continue;
                    const uint32_t light = row ? l0 + sm.list[b0 + g + lane] : 0u;
#pragma unroll
                    for (uint32_t x = 0; x < 8u; ++x) {
                        const bool in = (row >> x) & 1u;
                        const uint64_t m = hl_ballot(in);
                        const uint32_t pos = run[x] + hl_prefix(m);
                        if (in && pos < HL_MAX_LIGHTS_PER_TILE) sm.out[8u * wave + x][pos] = light;
                        run[x] += (uint32_t)__popcll(m);
                    }
                }
#pragma unroll
                for (uint32_t x = 0; x < 8u; ++x) {
                    some = some || (x < nx && run[x] < HL_MAX_LIGHTS_PER_TILE);
                    if (lane == x) sm.run[8u * wave + x] = run[x];
                }
            }
            if (some && lane == 0u) atomicAdd(&sm.open[batch & 1u], 1u);
            __syncthreads();  // and the masks and runs before the next batch's
            open = sm.open[batch & 1u] != 0u;
            ++batch;
        }
    }
    __syncthreads();
    // a wave per row again: 64 entries of a tile at a time
    for (uint32_t x = 0; x < nx && wave < ny; ++x) {
        const uint32_t tile = (ty0 + wave) * a.p.num_tiles_x + tx0 + x;
        const uint32_t cnt = min(sm.run[8u * wave + x], (uint32_t)HL_MAX_LIGHTS_PER_TILE);
        static_assert(HL_MAX_LIGHTS_PER_TILE == 64, "an entry per lane");
        if (lane < cnt) a.lists[(size_t)tile * HL_MAX_LIGHTS_PER_TILE + lane] = sm.out[8u * wave + x][lane];
        if (lane == 0u) a.counts[tile] = cnt;
    }
    // the shading records, last: no wait stands on them
    if (INLINE)
        for (uint32_t i = blockIdx.x * NT + t; i < n; i += gridDim.x * NT)
            prep_one(a.lights, nullptr, n, a.cam, a.hot, nullptr, a.feature_flags, i);
}

// ---------------------------------------------------------------- launchers
hipError_t launch_prep(hipStream_t s, const GpuLight* lights, const uint32_t* subset, uint32_t n,
                       const GpuCameraUniforms* cam, HotLight* hot, CullLight* cull,
                       uint32_t* flags) {
    if (n == 0) return hipSuccess;
    k_prep_lights<<<(n + 255) / 256, 256, 0, s>>>(lights, subset, n, cam, hot, cull, flags);
    return hipGetLastError();
}

hipError_t launch_prep_zero(hipStream_t s, const GpuLight* lights, uint32_t n, const GpuCameraUniforms* cam,
                            HotLight* hot, uint32_t* flags, double* acc, size_t acc_n, double* loss) {
    // one thread per light (prep_one), the accumulators grid-stride
    const size_t prep_blocks = ((size_t)n + 255) / 256;
    size_t zero_blocks = (acc_n + 255) / 256;
    if (zero_blocks > 4096) zero_blocks = 4096;
    size_t blocks = prep_blocks > zero_blocks ? prep_blocks : zero_blocks;
    if (blocks == 0) blocks = 1;
    k_prep_zero<<<(unsigned)blocks, 256, 0, s>>>(lights, n, cam, hot, flags, acc, acc_n, loss);
    return hipGetLastError();
}

hipError_t launch_fill_u32(hipStream_t s, uint32_t* p, uint32_t v, size_t n) {
    if (n == 0) return hipSuccess;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    k_fill_u32<<<(unsigned)blocks, 256, 0, s>>>(p, v, n);
    return hipGetLastError();
}

hipError_t launch_cull_tiles(hipStream_t s, const GpuCameraUniforms* cam, const LightCullParams& p,
                             const CullLight* cl, uint32_t* lists, uint32_t* counts) {
    const uint32_t total = p.num_tiles_x * p.num_tiles_y;
    if (total == 0) return hipSuccess;
    k_cull_tiles<<<(total + 3) / 4, 256, 0, s>>>(cam, p, cl, lists, counts);
    return hipGetLastError();
}

// Tiles per super-tile: the smallest power of two that leaves at most
// kTileBlocks blocks, all of them resident at once (two of 59 KB of LDS fit a
// CU), at most kTileMax, at least as wide as high.  Twice as many blocks of half
// the tiles, a quarter of them waiting for a place: 34 us at 4K and 16384
// lights, 11.6 at 720p and 64.
constexpr uint32_t kTileBlocks = 512;
static void tile_plan(TileArgs& a) {
    const uint64_t total = (uint64_t)a.p.num_tiles_x * a.p.num_tiles_y;
    uint32_t log = 0;
    while (log < 6u && total >> log > kTileBlocks) ++log;
    a.sx = 1u << ((log + 1u) / 2u);
    a.sy = 1u << (log / 2u);
    a.nsx = (a.p.num_tiles_x + a.sx - 1u) / a.sx;
    const uint32_t side = std::max(a.nsx, (a.p.num_tiles_y + a.sy - 1u) / a.sy);
    a.shift = 0;
    while ((side + (1u << a.shift) - 1u) >> a.shift > kColMaxSide) ++a.shift;
}

size_t tile_scratch_bytes(uint32_t num_lights) { return 28 * ((size_t)num_lights + 4); }

hipError_t launch_cull_tiles_binned(hipStream_t s, const GpuCameraUniforms* cam, const LightCullParams& p,
                                    const GpuLight* lights, HotLight* hot, uint32_t* feature_flags, void* scratch,
                                    uint32_t* lists, uint32_t* counts) {
    TileArgs a{};
    a.cam = cam;
    a.lights = lights;
    a.hot = hot;
    a.feature_flags = feature_flags;
    a.p = p;
    tile_plan(a);
    const size_t n4 = ((size_t)p.num_lights + 3u) & ~(size_t)3u;
    a.vpos = (float4*)scratch;
    a.rect = (uint2*)(a.vpos + n4);
    a.box = (uint32_t*)(a.rect + n4);
    a.lists = lists;
    a.counts = counts;
    const uint32_t blocks = a.nsx * ((p.num_tiles_y + a.sy - 1u) / a.sy);
    if (p.num_lights <= kColInline) {
        k_tile_cull<kColInline, true><<<blocks, kColThreads, 0, s>>>(a);
        return hipGetLastError();
    }
    k_tile_prep<<<(p.num_lights + 63u) / 64u, 64, 0, s>>>(a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    k_tile_cull<kColChunk, false><<<blocks, kColThreads, 0, s>>>(a);
    return hipGetLastError();
}

size_t cluster_geom_offset_boxes(uint32_t ncol) { return cluster_geom_offset_boxes_dev(ncol); }
size_t cluster_geom_bytes(uint32_t ncol, uint32_t ncell) {
    return cluster_geom_offset_boxes(ncol) + sizeof(CellBox) * (size_t)ncell;
}

hipError_t launch_cluster_cull(hipStream_t s, const ClusterArgs& a, const GpuCameraUniforms* cam,
                               const GpuLight* lights, HotLight* hot, CullLight* cl, uint32_t* feature_flags,
                               ClusterPath path, const ClusterScratch& w, uint32_t* offsets,
                               uint32_t* counts, uint32_t* pool, uint32_t pool_cap,
                               uint32_t* flags, uint32_t* flags2) {
    const uint32_t ncol = a.grid_x * a.grid_y;
    const uint32_t ncell = ncol * a.grid_z;
    if (path == ClusterPath::kBruteForce) {
        const uint32_t blocks = (ncell + kBfCells - 1u) / kBfCells;
        k_cluster_bf_count<<<blocks, 256, 0, s>>>(a, cam, lights, hot, feature_flags, w.raw, flags, flags2);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        k_cluster_bf_fill<<<blocks, 256, 0, s>>>(a, cam, lights, w.raw, pool_cap, offsets, counts, pool, flags,
                                                 flags2);
        return hipGetLastError();
    }
    if (path == ClusterPath::kColumns) {
        const ColumnPlan cp = column_plan(ncol, a.grid_z, kColBlocks);
        ColumnArgs p{};
        p.cam = cam;
        p.lights = lights;
        p.hot = hot;
        p.cull = cl;
        p.feature_flags = feature_flags;
        p.raw = w.raw;
        p.offsets = offsets;
        p.counts = counts;
        p.pool = pool;
        p.pool_cap = pool_cap;
        p.kb = cp.kb;
        while ((std::max(a.grid_x, a.grid_y) - 1u) >> p.shift >= kColMaxSide) ++p.shift;
        p.flags = flags;
        p.flags2 = flags2;
        (void)column_scratch((uint8_t*)w.columns, ncol, a.grid_z, a.num_lights, cp.blocks, &p);
        hipError_t e;
        if (column_inline(ncell, a.num_lights)) {
            k_col_count<kColInline, kColThreads, true><<<cp.blocks, kColThreads, 0, s>>>(a, p);
            if ((e = hipGetLastError()) != hipSuccess) return e;
            k_col_fill<false><<<cp.blocks, 256, 0, s>>>(a, p);
            return hipGetLastError();
        }
        k_col_prep<<<a.num_lights ? (a.num_lights + 63u) / 64u : 1u, 64, 0, s>>>(
            a, p, column_groups(ncol) * a.grid_z);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (ncol <= kColMaxColumns)
            k_col_count<kColChunk, kColThreads, false><<<cp.blocks, kColThreads, 0, s>>>(a, p);
        else  // many blocks with few lights
            k_col_count<kBatchColChunk, kColNarrow, false><<<cp.blocks, kColNarrow, 0, s>>>(a, p);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        k_col_fill<true><<<cp.blocks, 256, 0, s>>>(a, p);
        return hipGetLastError();
    }
    const uint32_t W = (a.num_lights + 31u) / 32u, SW = (W + 31u) / 32u;
    ColumnGeom* geom = (ColumnGeom*)w.geom;
    CellBox* boxes = (CellBox*)((uint8_t*)w.geom + cluster_geom_offset_boxes(ncol));
    const uint32_t ntiles = cluster_scan_tiles(ncell);
    unsigned long long* tile_sums = (unsigned long long*)((uint8_t*)w.raw + cluster_tile_sums_offset(ncell));
    const uint32_t geom_blocks = (ncell + 255) / 256;
    k_cluster_geom<<<geom_blocks + (a.num_lights + 255) / 256, 256, 0, s>>>(
        a, cam, geom, boxes, w.mq.count, flags, flags2, tile_sums, ntiles, lights, hot, cl, feature_flags,
        geom_blocks);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (a.num_lights) {
        k_cluster_mark<<<(a.num_lights + 3) / 4, 256, 0, s>>>(a, cam, cl, geom, boxes, w.bits,
                                                                  w.summary, w.mq);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        k_cluster_mark_tail<<<tail_blocks(a.num_lights), 256, 0, s>>>(a, cl, geom, boxes, w.bits,
                                                                       w.summary, w.mq);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    const uint32_t blocks = (ncell + 256u / kCellLanes - 1u) / (256u / kCellLanes);
    k_cluster_count<<<blocks, 256, 0, s>>>(ncell, SW, w.bits, w.summary, w.raw, a.cap);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    k_cluster_fill<<<blocks, 256, 0, s>>>(ncell, SW, w.raw, w.bits, w.summary, a.cap, pool_cap, offsets, counts,
                                          pool, flags, flags2);
    return hipGetLastError();
}

}  // namespace hl
