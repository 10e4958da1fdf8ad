// kernels.hip -- gfx950 kernels of the triangle path.
//
// Frame = setup -> raster, for one request (the view in the kernel
// argument) or for a batch of requests (views in device memory, each with its
// own target, mesh, uniforms, tiles and bins):
//   k_setup   one lane per shaded vertex (clip position and VertexData of the
//             fixed vertex shader) and one lane per triangle: euc's triangle
//             setup (triangles.rs:55-171) in IEEE f32, culling, and binning of
//             the triangle into every tile its bounding box covers.  Pairs are
//             grouped by tile in an LDS hash so each distinct tile costs one
//             global atomic per workgroup; ranks past a tile's bin capacity go
//             to overflow segments of that tile taken from a pool.  With few
//             triangles per tile (big-triangle mode) and row checkpoints no
//             triangle is binned: span blocks of the same launch set each one
//             up again, walk its rows once and store the row's weights where
//             it enters each tile column, plus per (tile, triangle) the rows
//             that reach into the tile and an occlusion bound (without
//             checkpoints, triangles covering many tiles go on one list).
//   k_raster  256-thread workgroups that each take a tile (256 pixels, one per
//             thread; 32x8, 16x16 or 8x32) of a per-XCD list.  Each pixel
//             keeps a 64-bit key in LDS that encodes the winning fragment; the
//             depth rule becomes an order-independent reduction (atomic min/max
//             of the key) because every fixed shader's blend replaces the old
//             pixel: the winner is a function of the set of fragments, with
//             primitive order as the tie-break (see init_key).  The (triangle,
//             row) pairs of a tile are spread over the lanes, each walking its
//             row exactly as triangles.rs:219-303 does (big triangles from
//             their checkpoints).  The winner is then shaded once and colour
//             and depth are written once per pixel.
//   k_tiny    setup and raster of a small mesh in one launch.
//   k_line_*  the lines rasteriser (lines.rs:15-121) for one request.
#include "internal.hpp"
#include "shade.hpp"

#include <algorithm>

namespace euchip {

EUCHIP_DEV uint32_t lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

// The launch's parameters, read anew from the kernel argument segment: the
// kernels take one reference per phase of their work.  The address passes
// through an empty asm, so a value loaded for one phase is not kept in a
// register through the others (a uniform value that did not fit the scalar
// registers went to vector-register lanes, and every use of it took a
// v_readlane: a quarter of the raster kernels' vector instructions).  Scalar
// loads of a line that the scalar cache holds cost no vector issue at all.  The
// 3840 x 2160 Phong raster issues 48.0M vector instructions instead of 60.4M.
EUCHIP_DEV const FrameParams &args() {
    const EUCHIP_CONST FrameParams *k = (const EUCHIP_CONST FrameParams *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return *(const FrameParams *)__builtin_assume_aligned((const FrameParams *)k, 16);
}

// Bring every line of the parameters into the scalar cache, all in flight at
// once, when a kernel starts: a phase that met its lines cold would wait for
// them again (small frames 3 to 9 % slower).
EUCHIP_DEV void warm_args() {
    const EUCHIP_CONST uint32_t *k = (const EUCHIP_CONST uint32_t *)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr uint32_t lines = (sizeof(FrameParams) + 63u) / 64u;
    static_assert(lines <= 16u, "one load per line below");
#define EUCHIP_LINE(i) k[16u * (i < lines ? i : lines - 1u)]
    asm volatile("" ::"s"(EUCHIP_LINE(0)), "s"(EUCHIP_LINE(1)), "s"(EUCHIP_LINE(2)), "s"(EUCHIP_LINE(3)),
                 "s"(EUCHIP_LINE(4)), "s"(EUCHIP_LINE(5)), "s"(EUCHIP_LINE(6)), "s"(EUCHIP_LINE(7)),
                 "s"(EUCHIP_LINE(8)), "s"(EUCHIP_LINE(9)), "s"(EUCHIP_LINE(10)), "s"(EUCHIP_LINE(11)),
                 "s"(EUCHIP_LINE(12)), "s"(EUCHIP_LINE(13)), "s"(EUCHIP_LINE(14)), "s"(EUCHIP_LINE(15)));
#undef EUCHIP_LINE
}

EUCHIP_DEV bool passes_z_clip(const FrameParams &p, float z) {
    return !p.z_clip || (p.z_min <= z && z <= p.z_max);
}

// Inclusive wave64 prefix sum on DPP lane moves: shifts of 1, 2, 4 and 8 lanes
// inside each 16-lane row (lanes without a source add the `old` operand, 0),
// then row_bcast:15 adds row 0's (row 2's) total to row 1 (row 3) and
// row_bcast:31 adds lane 31's running total to rows 2 and 3.
EUCHIP_DEV uint32_t wave_inclusive_sum(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1, 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2, 3
    return v;
}

// Stream element of corner i of primitive t after the fixed geometry stage
// (Pipeline::geometry, pipeline.rs:221-229): output t % k of input triangle
// t / k, [a, b, c] or [a, c, b].
EUCHIP_DEV uint32_t corner_element(uint32_t geometry, uint32_t t, int i) {
    uint32_t tri = t, rev = 0u;
    if (geometry == GEOM_BOTH_SIDES) tri = t >> 1, rev = t & 1u;
    else if (geometry == GEOM_REVERSED) rev = 1u;
    const uint32_t c = (i == 0 || !rev) ? (uint32_t)i : 3u - (uint32_t)i;
    return 3u * tri + c;
}

// Instance and index within the instance of the corners of primitive t.
EUCHIP_DEV void corner_places(const View &v, uint32_t geometry, uint32_t t, uint32_t inst[3], uint32_t at[3]) {
#pragma unroll
    for (int i = 0; i < 3; i++) inst[i] = 0u, at[i] = corner_element(geometry, t, i);
    if (v.inst_map == INST_TRIANGLES) {
        const uint32_t tri = geometry == GEOM_BOTH_SIDES ? t >> 1 : t;
        const uint32_t q = divide(tri, v.inst_tris);
#pragma unroll
        for (int i = 0; i < 3; i++) inst[i] = q, at[i] -= q * v.count;
    } else if (v.inst_map == INST_CORNERS) {
#pragma unroll
        for (int i = 0; i < 3; i++) inst[i] = at[i] / v.count, at[i] -= inst[i] * v.count;
    }
}

// ---------------------------------------------------------------------------
// triangle setup (triangles.rs:55-171) of primitive t of request v, whole-target
// band clamp, from the vertex shader's clip positions.  Returns false when the
// triangle is culled or its bounding box is empty.
// ---------------------------------------------------------------------------
EUCHIP_DEV bool tri_setup(const FrameParams &p, const View &v, uint32_t t, TriRec &R) {
    float hom[3][4], euc[3][3];
    uint32_t sid[3], inst[3], vi[3];
    const float flip1 = p.y_up ? -1.0f : 1.0f;
    // the corners' clip positions (vertex(): VP * model * (p, 1), or the CLIP
    // input itself), the uniform branches taken outside the corner loop so the
    // loads of all three corners are in flight together
    corner_places(v, p.geometry, t, inst, vi);
    if (v.idx) {
#pragma unroll
        for (int i = 0; i < 3; i++) vi[i] = v.idx[vi[i]];
    }
    float c[3][4];
    if (p.xform == 0u) {
        if (v.pos_comps == 4u) {
#pragma unroll
            for (int i = 0; i < 3; i++) {
                const float *P = v.pos + 4u * vi[i];
                c[i][0] = P[0], c[i][1] = P[1], c[i][2] = P[2], c[i][3] = P[3];
            }
        } else {
#pragma unroll
            for (int i = 0; i < 3; i++) {
                const float *P = v.pos + (size_t)v.pos_comps * vi[i];
                c[i][0] = P[0], c[i][1] = P[1], c[i][2] = P[2], c[i][3] = 1.0f;
            }
        }
    } else {
        float p4[3][4], w[3][4];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const float *P = v.pos + (size_t)v.pos_comps * vi[i];
            p4[i][0] = P[0], p4[i][1] = P[1], p4[i][2] = P[2], p4[i][3] = 1.0f;
        }
        if (v.inst_map == INST_CORNERS) {
#pragma unroll
            for (int i = 0; i < 3; i++) mat4_vec4((const float *)v.models + 16u * inst[i], p4[i], w[i]);
        } else {
            with_model(v, inst[0], [&](const EUCHIP_CONST float *m) {
#pragma unroll
                for (int i = 0; i < 3; i++) mat4_vec4(m, p4[i], w[i]);
            });
        }
#pragma unroll
        for (int i = 0; i < 3; i++) mat4_vec4(v.u + U_VP, w[i], c[i]);
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
        sid[i] = v.sv_base + inst[i] * v.n_vertices + vi[i];
        hom[i][0] = c[i][0] * 1.0f;
        hom[i][1] = c[i][1] * flip1;
        hom[i][2] = c[i][2];
        hom[i][3] = c[i][3];
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
        euc[i][0] = hom[i][0] / hom[i][3];
        euc[i][1] = hom[i][1] / hom[i][3];
        euc[i][2] = hom[i][2] / hom[i][3];
    }
    // winding = cross(e1 - e0, e2 - e0).z
    const float a0 = euc[1][0] - euc[0][0], a1 = euc[1][1] - euc[0][1];
    const float b0 = euc[2][0] - euc[0][0], b1 = euc[2][1] - euc[0][1];
    const float winding = a0 * b1 - a1 * b0;
    if (p.cull == 1u && winding * 1.0f < 0.0f) return false;
    if (p.cull == 2u && winding * -1.0f < 0.0f) return false;
    const bool swapped = winding >= 0.0f;
    if (swapped) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float tmp = hom[0][c];
            hom[0][c] = hom[2][c];
            hom[2][c] = tmp;
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const float tmp = euc[0][c];
            euc[0][c] = euc[2][c];
            euc[2][c] = tmp;
        }
        const uint32_t ts = sid[0];
        sid[0] = sid[2];
        sid[2] = ts;
    }
    const float sx = (float)v.W, sy = (float)v.H;
    const float T[3][3] = {{v.ndc_x, 0.0f, -1.0f}, {0.0f, v.ndc_y, 1.0f}, {0.0f, 0.0f, 1.0f}};
    // coords_to_weights (triangles.rs:86-102)
    const float c3[3] = {hom[2][0], hom[2][1], hom[2][3]};
    const float ca[3] = {hom[0][0] - c3[0], hom[0][1] - c3[1], hom[0][3] - c3[2]};
    const float cb[3] = {hom[1][0] - c3[0], hom[1][1] - c3[1], hom[1][3] - c3[2]};
    const float n[3] = {ca[1] * cb[2] - ca[2] * cb[1], ca[2] * cb[0] - ca[0] * cb[2], ca[0] * cb[1] - ca[1] * cb[0]};
    const float nn = n[0] * n[0] + n[1] * n[1] + n[2] * n[2];
    const float nc = n[0] * c3[0] + n[1] * c3[1] + n[2] * c3[2];
    const float rd = nn > 0.0f ? 1.0f / rmin(nc, -__FLT_EPSILON__) : 1.0f;
    float rows[3][3] = {{cb[1] * c3[2] - cb[2] * c3[1], cb[2] * c3[0] - cb[0] * c3[2], cb[0] * c3[1] - cb[1] * c3[0]},
                        {c3[1] * ca[2] - c3[2] * ca[1], c3[2] * ca[0] - c3[0] * ca[2], c3[0] * ca[1] - c3[1] * ca[0]},
                        {n[0], n[1], n[2]}};
    float M[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
#pragma unroll
        for (int j = 0; j < 3; j++) rows[i][j] = rows[i][j] * rd;
#pragma unroll
        for (int j = 0; j < 3; j++) M[i][j] = rows[i][0] * T[0][j] + rows[i][1] * T[1][j] + rows[i][2] * T[2][j];
    }
    // screen coordinates and bounds (triangles.rs:110-139); the band clamp of y
    // is applied per row by the raster pass, here the clamp is the whole target
    float vs[3][2];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        vs[i][0] = sx * (euc[i][0] * 0.5f + 0.5f);
        vs[i][1] = sy * (euc[i][1] * -0.5f + 0.5f);
    }
    R.xmin = sat_clamp(rmin(rmin(vs[0][0], vs[1][0]), vs[2][0]) + 0.0f, 0u, v.W);
    R.ymin = sat_clamp(rmin(rmin(vs[0][1], vs[1][1]), vs[2][1]) + 0.0f, 0u, v.H);
    R.xmax = sat_clamp(rmax(rmax(vs[0][0], vs[1][0]), vs[2][0]) + 1.0f, 0u, v.W);
    R.ymax = sat_clamp(rmax(rmax(vs[0][1], vs[1][1]), vs[2][1]) + 1.0f, 0u, v.H);
    // w_hom at (0,0) and the per-pixel steps (triangles.rs:142-145)
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const float o = M[i][0] * 0.0f + M[i][1] * 0.0f + M[i][2] * 1.0f;
        const float wx = M[i][0] * 1000.0f + M[i][1] * 0.0f + M[i][2] * 1.0f;
        const float wy = M[i][0] * 0.0f + M[i][1] * 1000.0f + M[i][2] * 1.0f;
        R.o[i] = o;
        R.dx[i] = (wx - o) * (1.0f / 1000.0f);
        R.dy[i] = (wy - o) * (1.0f / 1000.0f);
        R.hz[i] = hom[i][2];
        R.sid[i] = sid[i];
    }
    // verts_by_y (triangles.rs:148-171), ties resolved as the reference does; kept in
    // scalars (a runtime index into a local array would live in scratch memory)
    const float x0 = vs[0][0], y0 = vs[0][1], x1 = vs[1][0], y1 = vs[1][1], x2 = vs[2][0], y2 = vs[2][1];
    const float min_y = rmin(rmin(y0, y1), y2);
    float ax, ay, bx, by, cx, cy;
    if (y0 == min_y) {
        ax = x0, ay = y0;
        if (y1 < y2) bx = x1, by = y1, cx = x2, cy = y2;
        else bx = x2, by = y2, cx = x1, cy = y1;
    } else if (y1 == min_y) {
        ax = x1, ay = y1;
        if (y0 < y2) bx = x0, by = y0, cx = x2, cy = y2;
        else bx = x2, by = y2, cx = x0, cy = y0;
    } else {
        ax = x2, ay = y2;
        if (y0 < y1) bx = x0, by = y0, cx = x1, cy = y1;
        else bx = x1, by = y1, cx = x0, cy = y0;
    }
    R.vby[0] = ax, R.vby[1] = ay, R.vby[2] = bx, R.vby[3] = by, R.vby[4] = cx, R.vby[5] = cy;
    const bool allin = passes_z_clip(p, euc[0][2]) && passes_z_clip(p, euc[1][2]) && passes_z_clip(p, euc[2][2]);
    R.flags = (allin ? TRI_ALL_IN : 0u) | (swapped ? TRI_SWAPPED : 0u);
    return R.xmin < R.xmax && R.ymin < R.ymax;
}

// A segment of n overflow entries of `tile`, taken from the pool and pushed on
// the tile's list: returns the pool index of its first entry, or ~0u when the
// pool ran out (the frame is then dropped and reported; the host re-runs a
// blocking render with a larger pool).
EUCHIP_DEV uint32_t take_segment(const FrameParams &p, uint32_t tile, uint32_t n) {
    const uint32_t words = n + 2u;
    const uint32_t base = atomicAdd(&p.ctr->pool[p.frame & 1u][0], words);
    if (base >= p.pool_cap || p.pool_cap - base < words) {
        atomicOr(&p.ctr->flags[p.frame & 1u][0], FLAG_BIN_OVERFLOW);
        return ~0u;
    }
    p.pool[base] = atomicExch(&p.tile_count[tile].head, base + 1u);
    p.pool[base + 1u] = n;
    return base + 2u;
}

// Bin slot of rank `rank` (below the capacity) of tile `tile` (launch tile space)
// of request v.
EUCHIP_DEV uint32_t *bin_slot(const FrameParams &p, const View &v, uint32_t tile, uint32_t rank) {
    return p.bins + v.bin_base + (size_t)(tile - v.tile_base) * v.tile_cap + rank;
}

// Range [beg, end) of this XCD's tiles: the hardware deals workgroups
// round-robin to the 8 XCDs, so workgroup b runs on XCD b % 8; each XCD gets a
// contiguous run of tiles so triangles shared by neighbouring tiles stay in
// that XCD's L2.
EUCHIP_DEV void xcd_range(uint32_t ntiles, uint32_t xcd, uint32_t &beg, uint32_t &end) {
    const uint32_t q = ntiles >> 3, r = ntiles & 7u;
    beg = xcd * q + (xcd < r ? xcd : r);
    end = beg + q + (xcd < r ? 1u : 0u);
}

// Busy list x: BUSY_BLOCKS lists hold up to ntiles entries at p.busy + x *
// ntiles; BUSY_RANGES list x holds the tiles of range x in that range's own slots.
EUCHIP_DEV void busy_list_span(const FrameParams &p, uint32_t x, uint32_t &base, uint32_t &cap) {
    if (p.busy_map == BUSY_BLOCKS) {
        base = x * p.ntiles, cap = p.ntiles;
    } else {
        uint32_t e;
        xcd_range(p.ntiles, x, base, e);
        cap = e - base;
    }
}

// Busy list of a tile.
EUCHIP_DEV uint32_t busy_list_of(const FrameParams &p, uint32_t tile) {
    if (p.busy_map == BUSY_BLOCKS) {  // one request: blocks of 4 x 4 tiles dealt over the XCDs
        const uint32_t ty = divide(tile, p.v0.row_tiles), tx = tile - ty * p.v0.ntx;
        return ((tx >> 2) + 3u * (ty >> 2)) & 7u;
    }
    // the XCD whose contiguous tile range (xcd_range) holds the tile
    const uint32_t q = p.ntiles >> 3, r = p.ntiles & 7u;
    const uint32_t big = r * (q + 1u);  // tiles of the ranges one longer
    return tile < big ? tile / (q + 1u) : r + (tile - big) / q;
}

// A tile whose count went from `old` to `old + n` may have become heavy.
EUCHIP_DEV void note_heavy(const FrameParams &p, uint32_t tile, uint32_t old, uint32_t n) {
    if (p.heavy_cap && old < kHeavyTile && old + n >= kHeavyTile) {
        const uint32_t k = atomicAdd(&p.ctr->heavy[p.frame & 1u][0], 1u);
        if (k < p.heavy_cap) p.heavy[k] = tile;
    }
}

// Bin append of one pair by a global atomic (the fallback of the LDS-grouped
// path).  maxp: where counts past the capacity are recorded for the host.
EUCHIP_DEV void bin_direct(const FrameParams &p, const View &v, uint32_t tile, uint32_t prim, uint32_t *maxp) {
    const uint32_t rank = atomicAdd(&p.tile_count[tile].count, 1u);
    note_heavy(p, tile, rank, 1u);
    if (p.busy && rank == 0u) {
        const uint32_t x = busy_list_of(p, tile);
        uint32_t lb, lc;
        busy_list_span(p, x, lb, lc);
        const uint32_t k = atomicAdd(&p.ctr->busy[p.frame & 1u][x][0], 1u);
        if (k < lc) p.busy[(size_t)lb + k] = tile;
    }
    if (rank < v.tile_cap) {
        *bin_slot(p, v, tile, rank) = prim;
    } else {
        atomicMax(maxp, rank + 1u);
        const uint32_t e = take_segment(p, tile, 1u);
        if (e != ~0u) p.pool[e] = prim;
    }
}

// The request a workgroup or tile works on: the kernel argument's, or one of
// the batch's in device memory, which no kernel writes: read as constants, by
// scalar loads (r is uniform), and anew for each phase like the parameters.
template <bool BATCH>
EUCHIP_DEV const View &view_of(const FrameParams &p, uint32_t r) {
    if constexpr (BATCH) {
        const EUCHIP_CONST View *k = (const EUCHIP_CONST View *)(const View *)p.views + r;
        asm volatile("" : "+s"(k));
        return *(const View *)__builtin_assume_aligned((const View *)k, 8);
    } else {
        return p.v0;
    }
}

// *q for a uniform q into memory that this launch does not write: a scalar load.
EUCHIP_DEV uint32_t uniform_load(const uint32_t *q) {
    return *(const EUCHIP_CONST uint32_t *)q;
}
EUCHIP_DEV TileBin uniform_load(const TileBin *q) {
    const EUCHIP_CONST uint32_t *k = (const EUCHIP_CONST uint32_t *)q;
    return TileBin{k[0], k[1]};
}

// The key mode of the frame's depth rule (see init_key).
EUCHIP_DEV uint32_t key_mode(const FrameParams &p) {
    return (p.depth_write && p.depth_test == DT_LESS) ? 1u : (p.depth_write && p.depth_test == DT_GREATER) ? 2u : 0u;
}

// Stores that bypass the caches on their way to memory: setup records (read
// back by another launch, usually on another XCD) and the targets (not read
// again by this frame).
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

EUCHIP_DEV void store_stream(uint4 *dst, const uint4 &v) {
    u32x4 x = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(x, reinterpret_cast<u32x4 *>(dst));
}
EUCHIP_DEV void store_stream(uint32_t *dst, uint32_t v) { __builtin_nontemporal_store(v, dst); }
EUCHIP_DEV void store_stream(float *dst, float v) { __builtin_nontemporal_store(v, dst); }

// Setup records (layout in internal.hpp).
EUCHIP_DEV void pack_rec(const TriRec &R, uint4 q0[kRec0Quads], uint4 q1[kRec1Quads]) {
    q0[0] = make_uint4(__float_as_uint(R.o[0]), __float_as_uint(R.o[1]), __float_as_uint(R.o[2]), __float_as_uint(R.dx[0]));
    q0[1] = make_uint4(__float_as_uint(R.dx[1]), __float_as_uint(R.dx[2]), __float_as_uint(R.dy[0]), __float_as_uint(R.dy[1]));
    q0[2] = make_uint4(__float_as_uint(R.dy[2]), __float_as_uint(R.hz[0]), __float_as_uint(R.hz[1]), __float_as_uint(R.hz[2]));
    q0[3] = make_uint4(R.xmin, R.xmax, R.ymin, R.ymax | (R.flags << 30));
    q1[0] = make_uint4(__float_as_uint(R.vby[0]), __float_as_uint(R.vby[1]), __float_as_uint(R.vby[2]), __float_as_uint(R.vby[3]));
    q1[1] = make_uint4(__float_as_uint(R.vby[4]), __float_as_uint(R.vby[5]), 0u, 0u);
}

// o, dx, dy, hz, bounds and flags from a record's first kRec0Quads quads.
EUCHIP_DEV void load_rec0_at(const uint4 *q, TriRec &R) {
    const uint4 a = q[0], b = q[1], c = q[2], d = q[3];
    R.o[0] = __uint_as_float(a.x), R.o[1] = __uint_as_float(a.y), R.o[2] = __uint_as_float(a.z);
    R.dx[0] = __uint_as_float(a.w), R.dx[1] = __uint_as_float(b.x), R.dx[2] = __uint_as_float(b.y);
    R.dy[0] = __uint_as_float(b.z), R.dy[1] = __uint_as_float(b.w), R.dy[2] = __uint_as_float(c.x);
    R.hz[0] = __uint_as_float(c.y), R.hz[1] = __uint_as_float(c.z), R.hz[2] = __uint_as_float(c.w);
    R.xmin = d.x, R.xmax = d.y, R.ymin = d.z, R.ymax = d.w & 0x3fffffffu, R.flags = d.w >> 30;
}

// o, dx, dy, hz, bounds and flags of record `rid`.
EUCHIP_DEV void load_rec0(const FrameParams &p, uint32_t rid, TriRec &R) {
    load_rec0_at(p.rec0 + (size_t)rid * kRec0Quads, R);
}

// verts_by_y from a record's kRec1Quads secondary quads.
EUCHIP_DEV void load_rec1_at(const uint4 *q, TriRec &R) {
    const uint4 a = q[0], b = q[1];
    R.vby[0] = __uint_as_float(a.x), R.vby[1] = __uint_as_float(a.y), R.vby[2] = __uint_as_float(a.z);
    R.vby[3] = __uint_as_float(a.w), R.vby[4] = __uint_as_float(b.x), R.vby[5] = __uint_as_float(b.y);
}

// verts_by_y of record `rid`.
EUCHIP_DEV void load_rec1(const FrameParams &p, uint32_t rid, TriRec &R) {
    load_rec1_at(p.rec1 + (size_t)rid * kRec1Quads, R);
}

// Shaded-vertex ids of primitive t's corners after the winding swap.
EUCHIP_DEV void tri_sids(const View &v, uint32_t geometry, uint32_t t, uint32_t flags, uint32_t sid[3]) {
    uint32_t inst[3], at[3];
    corner_places(v, geometry, t, inst, at);
    if (v.idx) {
#pragma unroll
        for (int i = 0; i < 3; i++) at[i] = v.idx[at[i]];
    }
#pragma unroll
    for (int i = 0; i < 3; i++) sid[i] = v.sv_base + inst[i] * v.n_vertices + at[i];
    if (flags & TRI_SWAPPED) {
        const uint32_t s0 = sid[0];
        sid[0] = sid[2];
        sid[2] = s0;
    }
}

// A triangle's rows all take the bounding-box span ("stupid version",
// triangles.rs:229-233) when its whole-target box is small; band clamping can
// only shrink the box, so then no row needs verts_by_y.
EUCHIP_DEV bool all_rows_boxed(const TriRec &R) {
    const uint32_t bw = R.xmax - R.xmin, bh = R.ymax - R.ymin;
    return bw < 128u && bh < 128u && bw * bh < 128u;
}

// Fragment test of one pixel (triangles.rs:262-301): weights, coverage, z, z-clip.
EUCHIP_DEV bool frag_z(const FrameParams &p, const TriRec &R, float w0, float w1, float w2, float &z) {
    const float u2 = (w2 - w0) - w1;
    if (!(w0 >= 0.0f && w1 >= 0.0f && u2 >= 0.0f)) return false;
    z = (R.hz[0] * w0 + R.hz[1] * w1) + R.hz[2] * u2;
    return (R.flags & TRI_ALL_IN) || passes_z_clip(p, z);
}

// Triangles whose box has at most this many pixels are tested for coverage in
// setup; one that covers no pixel corner emits no fragment and is not binned.
constexpr uint32_t kCoverTestArea = 8;

// Does a boxed triangle (all_rows_boxed) cover any pixel of its box, with the
// raster pass's arithmetic (rows walked from xmin, triangles.rs:257-301)?
EUCHIP_DEV bool covers_any(const FrameParams &p, const TriRec &R) {
    for (uint32_t y = R.ymin; y < R.ymax; y++) {
        const float Y = (float)y, X0 = (float)R.xmin;
        float w0 = (R.o[0] + R.dy[0] * Y) + R.dx[0] * X0;
        float w1 = (R.o[1] + R.dy[1] * Y) + R.dx[1] * X0;
        float w2 = (R.o[2] + R.dy[2] * Y) + R.dx[2] * X0;
        for (uint32_t x = R.xmin; x < R.xmax; x++) {
            float z;
            if (frag_z(p, R, w0, w1, w2, z)) return true;
            w0 = w0 + R.dx[0];
            w1 = w1 + R.dx[1];
            w2 = w2 + R.dx[2];
        }
    }
    return false;
}

constexpr uint32_t kHash = 512;    // LDS hash slots (distinct tiles) per setup workgroup
constexpr uint32_t kPairs = 1024;  // (tile, primitive) pairs grouped in LDS per round, 4 per lane
static_assert(kHash == 512u && kPairs == 4u * 256u, "9-bit hash slots; a lane keeps its 4 pairs in registers");
// A triangle of more tiles than this is binned by its whole wave, a global
// atomic per tile: its tiles are all different, there is nothing to group.
constexpr uint32_t kPairTiles = 4096;

// ---------------------------------------------------------------------------
// k_setup: per-vertex clip position + VertexData (thread t = shaded vertex t)
// and per-triangle culling + binning (thread t = primitive t).
// Binning spreads the workgroup's (tile, primitive) pairs evenly over its lanes,
// kPairs a round, and groups them by tile in an LDS hash table, so each distinct
// tile costs one global atomic per round; ranks inside the group come from LDS.
// (With each lane walking its own triangle's tiles, the lane of the largest set
// the pace, and pairs past one round took an atomic each, one after the other:
// the setup of a 1024x800 frame of 6400 triangles over 12 tiles each took 48 us.)
// ---------------------------------------------------------------------------
// A span block of a checkpoint frame's setup launch (defined with the raster's
// row helpers below).
EUCHIP_DEV void span_item(const FrameParams &p, uint32_t b, void *static_lds);

// LDS of k_setup: the workgroup's records on their way out, then the binning tables.
union SetupShared {
    struct {
        uint4 q0[256 * kRec0Quads];
        uint32_t kept[256];
    } rec;
    struct {
        uint32_t hkey[kHash], hcnt[kHash], hbase[kHash];
        uint32_t hseg[kHash];   // pool index of the slot's overflow entries
        // per triangle: its first pair, first tile, tiles per row and their reciprocal
        uint32_t at[256], tile0[256], nx[256];
        float inv[256];
        uint8_t owner[kPairs];  // triangle of each pair of the round
    } bin;
};

// SPAN: the launch of a checkpoint frame, whose blocks past setup_blocks are
// span blocks (compiled apart so other frames' setup carries none of their code).
template <uint32_t SH, bool BATCH, bool SPAN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_setup(FrameParams) {
    warm_args();
    const FrameParams &p = args();
    __shared__ SetupShared sm;
    __shared__ uint32_t wave_pairs[4];
    __shared__ uint32_t lcnt[9], lbase[9];  // new busy tiles per list (8) and new heavy tiles (8)
    const uint32_t tid = threadIdx.x;
    if constexpr (!BATCH) {
        if (blockIdx.x >= p.tri_blocks) {  // (checkpoint frames: tri_blocks = setup_blocks)
            if constexpr (SPAN) {
                span_item(p, blockIdx.x - p.setup_blocks, &sm);
            } else if constexpr (vd_count(SH) > 0) {  // a vertex block
                const View &v = p.v0;
                const uint32_t t = (blockIdx.x - p.tri_blocks) * 256u + tid;
                if (t < v.n_instances * v.n_vertices) {
                    const uint32_t inst = divide(t, v.inst_verts);
                    float vd[VDN<SH>::N];
                    vertex_data<SH>(p, v, inst, t - inst * v.n_vertices, vd);
#pragma unroll
                    for (uint32_t q = 0; q < vd_count(SH); q++) p.vary[((size_t)v.sv_base + t) * vd_count(SH) + q] = vd[q];
                }
            }
            return;
        }
    }
    uint32_t r = 0, j = blockIdx.x;
    if constexpr (BATCH) {
        const uint2 bj = p.blk[blockIdx.x];
        r = __builtin_amdgcn_readfirstlane(bj.x), j = __builtin_amdgcn_readfirstlane(bj.y);
    }
    const View &v = view_of<BATCH>(p, r);
    const uint32_t tpb = BATCH ? 256u : p.tri_block;  // triangles of this workgroup, one per lane
    const uint32_t t = tid < tpb ? j * tpb + tid : ~0u;
    const uint32_t sx = p.tile_sx, sy = 8u - p.tile_sx;
    bool keep = false;
    uint32_t tx0 = 0, ty0 = 0, nx = 0, ny = 0;
    if (t < v.n_tris) {
        TriRec R;
        keep = tri_setup(p, v, t, R);
        if (keep && all_rows_boxed(R) && (R.xmax - R.xmin) * (R.ymax - R.ymin) <= kCoverTestArea)
            keep = covers_any(p, R);
        if (keep) {
            tx0 = R.xmin >> sx;
            ty0 = R.ymin >> sy;
            nx = ((R.xmax - 1u) >> sx) - tx0 + 1u;
            ny = ((R.ymax - 1u) >> sy) - ty0 + 1u;
            if (p.ck_on) {
                // checkpoint frames: the span blocks walk every triangle (a lane
                // binning a triangle of many tiles here would take them one by
                // one, each behind dependent LDS atomics)
                nx = ny = 0u;
            } else if (p.big_cap && nx * ny > kBigTiles) {  // on the big-triangle list (while it has room)
                const uint32_t k = atomicAdd(&p.ctr->big[p.frame & 1u][0], 1u);
                if (k < p.big_cap) {
                    p.big[k] = t;
                    nx = ny = 0u;
                }
            }
            uint4 q0[kRec0Quads], q1[kRec1Quads];
            pack_rec(R, q0, q1);
#pragma unroll
            for (uint32_t k = 0; k < kRec0Quads; k++) sm.rec.q0[tid * kRec0Quads + k] = q0[k];
            // rec1: this lane's 32 bytes, contiguous with its neighbours' (no
            // staging); only triangles with a span row read it (all_rows_boxed)
            if (!all_rows_boxed(R)) {
#pragma unroll
                for (uint32_t k = 0; k < kRec1Quads; k++)
                    store_stream(&p.rec1[((size_t)v.tri_base + t) * kRec1Quads + k], q1[k]);
            }
        }
    }
    sm.rec.kept[tid] = keep ? 1u : 0u;
    // Batches and checkpoint frames: the vertex stage after the triangles' loads
    // (the VertexData stores would otherwise order those loads behind them);
    // other one-request frames have vertex blocks of their own.
    if constexpr ((BATCH || SPAN) && vd_count(SH) > 0) {  // (their workgroups have 256 triangles)
        if (t < v.n_instances * v.n_vertices) {
            const uint32_t inst = divide(t, v.inst_verts);
            const uint32_t vi = t - inst * v.n_vertices;
            const size_t sv = (size_t)v.sv_base + t;
            float vd[VDN<SH>::N];
            vertex_data<SH>(p, v, inst, vi, vd);
#pragma unroll
            for (uint32_t q = 0; q < vd_count(SH); q++) p.vary[sv * vd_count(SH) + q] = vd[q];
        }
    }
    __syncthreads();
    // the workgroup's records are contiguous: write them out 16 bytes per lane,
    // skipping the culled triangles' slots
    {
        const size_t base = (size_t)v.tri_base + (size_t)j * tpb;
#pragma unroll
        for (uint32_t k = 0; k < kRec0Quads; k++) {
            const uint32_t q = k * 256u + tid;
            if (q < kRec0Quads * tpb && sm.rec.kept[q / kRec0Quads]) store_stream(&p.rec0[base * kRec0Quads + q], sm.rec.q0[q]);
        }
    }
    const uint32_t tbase = v.tile_base;
    uint32_t *maxp = BATCH ? p.req_max + r : &p.ctr->max_count[p.frame & 1u][0];
    uint32_t n = keep ? nx * ny : 0u;  // this triangle's pairs (at most the target's tiles)
    for (uint64_t m = __ballot(n > kPairTiles); m; m &= m - 1u) {
        const int l = __ffsll((unsigned long long)m) - 1;
        const uint32_t bnx = __builtin_amdgcn_readlane(nx, l), bn = __builtin_amdgcn_readlane(n, l);
        const uint32_t b0 = __builtin_amdgcn_readlane(ty0 * v.ntx + tx0, l), prim = __builtin_amdgcn_readlane(t, l);
        for (uint32_t q = lane_id(); q < bn; q += 64u) {
            const uint32_t jy = q / bnx;
            bin_direct(p, v, tbase + b0 + jy * v.ntx + (q - jy * bnx), prim, maxp);
        }
    }
    if (n > kPairTiles) n = 0u;
    const uint32_t incl = wave_inclusive_sum(n);
    if ((tid & 63u) == 63u) wave_pairs[tid >> 6] = incl;
    __syncthreads();  // also: the binning tables reuse the record staging
    uint32_t at = incl - n, total = 0u;
#pragma unroll
    for (uint32_t q = 0; q < 4u; q++) {
        const uint32_t c = wave_pairs[q];
        at += q < (tid >> 6) ? c : 0u;
        total += c;
    }
    total = __builtin_amdgcn_readfirstlane(total);
    sm.bin.at[tid] = at, sm.bin.tile0[tid] = ty0 * v.ntx + tx0, sm.bin.nx[tid] = nx;
    // (m + 0.5) * inv truncates to m / nx for every pair m < 2^12: its error is
    // far below the 0.5 / nx to the next whole number
    sm.bin.inv[tid] = __builtin_amdgcn_rcpf((float)nx);
    for (uint32_t q0 = 0; q0 < total; q0 += kPairs) {
        for (uint32_t i = tid; i < kHash; i += 256u) sm.bin.hkey[i] = 0u, sm.bin.hcnt[i] = 0u;
        if (tid < 9u) lcnt[tid] = 0u;
        // the triangles of this round's pairs: each lane writes its own, a
        // triangle of many pairs the whole wave
        const uint32_t beg = at > q0 ? at : q0, end = at + n < q0 + kPairs ? at + n : q0 + kPairs;
        const bool wide = end > beg + 8u && beg < end;
        if (!wide)
            for (uint32_t q = beg; q < end; q++) sm.bin.owner[q - q0] = (uint8_t)tid;
        for (uint64_t m = __ballot(wide); m; m &= m - 1u) {
            const int l = __ffsll((unsigned long long)m) - 1;
            const uint32_t b = __builtin_amdgcn_readlane(beg, l), e = __builtin_amdgcn_readlane(end, l);
            for (uint32_t q = b + lane_id(); q < e; q += 64u) sm.bin.owner[q - q0] = (uint8_t)((tid & ~63u) + l);
        }
        __syncthreads();
        // each lane's pairs: tile, and hash slot | rank in the slot << 9 (~0: none)
        uint32_t pt[4], ps[4], po[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            ps[i] = ~0u, pt[i] = 0u, po[i] = 0u;
            const uint32_t q = q0 + i * 256u + tid;
            if (q >= total) continue;
            const uint32_t o = sm.bin.owner[q - q0], m = q - sm.bin.at[o], w = sm.bin.nx[o];
            const uint32_t jy = (uint32_t)(((float)m + 0.5f) * sm.bin.inv[o]);
            const uint32_t tile = tbase + sm.bin.tile0[o] + jy * v.ntx + (m - jy * w);
            pt[i] = tile, po[i] = o;
            uint32_t h = (tile * 2654435761u) >> 23;  // 9-bit multiplicative hash
            for (uint32_t probe = 0; probe < 16u; probe++) {
                const uint32_t old = atomicCAS(&sm.bin.hkey[h], 0u, tile + 1u);
                if (old == 0u || old == tile + 1u) {
                    ps[i] = h | (atomicAdd(&sm.bin.hcnt[h], 1u) << 9);
                    break;
                }
                h = (h + 1u) & (kHash - 1u);
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++)  // the table was full here
            if (q0 + i * 256u + tid < total && ps[i] == ~0u) bin_direct(p, v, pt[i], j * tpb + po[i], maxp);
        __syncthreads();
        // One global atomic per distinct tile; tiles that became busy or heavy get a
        // rank among this round's new ones: bits 0-10 busy rank, 11-13 busy list,
        // 14 busy, 15-25 heavy rank, 26 heavy.
        uint32_t code[kHash / 256u], ctile[kHash / 256u];
#pragma unroll
        for (uint32_t c = 0; c < kHash / 256u; c++) {
            const uint32_t i = c * 256u + tid, cn = sm.bin.hcnt[i];
            code[c] = 0u, ctile[c] = 0u;
            if (cn == 0u) continue;
            const uint32_t tile = sm.bin.hkey[i] - 1u;
            const uint32_t old = atomicAdd(&p.tile_count[tile].count, cn);
            sm.bin.hbase[i] = old;
            // ranks past the capacity: one overflow segment for this workgroup's share
            if (old + cn > v.tile_cap) {
                atomicMax(maxp, old + cn);
                const uint32_t first = old > v.tile_cap ? old : v.tile_cap;
                sm.bin.hseg[i] = take_segment(p, tile, old + cn - first);
            }
            ctile[c] = tile;
            if (p.busy && old == 0u) {
                const uint32_t x = busy_list_of(p, tile);
                code[c] |= atomicAdd(&lcnt[x], 1u) | (x << 11) | (1u << 14);
            }
            if (p.heavy_cap && old < kHeavyTile && old + cn >= kHeavyTile) code[c] |= (atomicAdd(&lcnt[8], 1u) << 15) | (1u << 26);
        }
        __syncthreads();
        // list bases (one global atomic per list) in flight while the bins are written
        uint32_t any_new = 0u;
#pragma unroll
        for (uint32_t q = 0; q < 9u; q++) any_new |= lcnt[q];
        uint32_t my_base = 0u;
        if (tid < 9u && lcnt[tid]) {
            my_base = tid < 8u ? atomicAdd(&p.ctr->busy[p.frame & 1u][tid][0], lcnt[tid])
                               : atomicAdd(&p.ctr->heavy[p.frame & 1u][0], lcnt[tid]);
        }
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
            if (ps[i] == ~0u) continue;
            const uint32_t h = ps[i] & (kHash - 1u), base = sm.bin.hbase[h], rank = base + (ps[i] >> 9);
            const uint32_t prim = j * tpb + po[i];
            if (rank < v.tile_cap) {
                *bin_slot(p, v, pt[i], rank) = prim;
            } else {
                const uint32_t first = base > v.tile_cap ? base : v.tile_cap;
                const uint32_t e = sm.bin.hseg[h];
                if (e != ~0u) p.pool[e + (rank - first)] = prim;
            }
        }
        if (any_new) {  // a tile became busy or heavy here (uniform)
            if (tid < 9u) lbase[tid] = my_base;
            __syncthreads();
#pragma unroll
            for (uint32_t c = 0; c < kHash / 256u; c++) {
                if (code[c] & (1u << 14)) {
                    const uint32_t x = (code[c] >> 11) & 7u, k = lbase[x] + (code[c] & 0x7ffu);
                    uint32_t lb, lc;
                    busy_list_span(p, x, lb, lc);
                    if (k < lc) p.busy[(size_t)lb + k] = ctile[c];
                }
                if (code[c] & (1u << 26)) {
                    const uint32_t k = lbase[8] + ((code[c] >> 15) & 0x7ffu);
                    if (k < p.heavy_cap) p.heavy[k] = ctile[c];
                }
            }
        }
        if (q0 + kPairs < total) __syncthreads();  // the next round reuses the tables
    }
}

// ---------------------------------------------------------------------------
// raster
// ---------------------------------------------------------------------------

// Total order of f32 for the winner keys; -0 and +0 map to one value.
EUCHIP_DEV uint32_t zord(float z) {
    const uint32_t u = __float_as_uint(z);
    if ((u & 0x7fffffffu) == 0u) return 0x80000000u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
EUCHIP_DEV float zunord(uint32_t o, uint32_t negzero) {
    if (o == 0x80000000u) return negzero ? -0.0f : 0.0f;
    return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}

// Winner keys.  mode 1 (test Less, write): min of (zord(z), prim+1, sign of zero)
// = the first fragment of the smallest z below D0.  mode 2 (Greater, write):
// the same with ~zord.  mode 0 (every other DepthMode): max of (prim+1, z bits)
// over fragments passing the test against D0 = the last passing fragment.
// In the reference's sequential order (pipeline.rs:519-538) these are exactly
// the fragments whose emit_fragment determines the final pixel and depth.
EUCHIP_DEV uint64_t init_key(uint32_t mode, float D0) {
    if (mode == 0u) return 0ull;
    if (D0 != D0) return 0ull;  // nothing compares with NaN
    const uint32_t o = mode == 1u ? zord(D0) : ~zord(D0);
    return (uint64_t)o << 32;
}

// The winning primitive + 1 of a key, 0 where there is none.
EUCHIP_DEV uint32_t key_prim(uint32_t mode, uint64_t kk) {
    return mode == 0u ? (uint32_t)(kk >> 32) : (uint32_t)kk >> 1;
}

// The depth test of a pixel whose depth before the pass is D0 (not DT_NONE).
EUCHIP_DEV bool passes_depth(uint32_t test, float z, float D0) {
    return test == DT_LESS ? z < D0 : test == DT_EQUAL ? z == D0 : z > D0;
}

// Row span [x0, x1) of row y for a triangle (triangles.rs:219-254); the
// "stupid version" switch uses the band-clamped bounding box.
EUCHIP_DEV void row_span(const TriRec &R, uint32_t y, uint32_t by0, uint32_t by1, uint32_t &x0, uint32_t &x1) {
    const uint32_t bw = R.xmax - R.xmin;
    const uint32_t yl = R.ymin < by0 ? by0 : (R.ymin > by1 ? by1 : R.ymin);
    const uint32_t yh = R.ymax < by0 ? by0 : (R.ymax > by1 ? by1 : R.ymax);
    const uint32_t bh = yh - yl;
    if (bw < 128u && bh < 128u && bw * bh < 128u) {
        x0 = R.xmin;
        x1 = R.xmax;
        return;
    }
    const float Y = (float)y;
    const float ax = R.vby[0], ay = R.vby[1], bx = R.vby[2], byy = R.vby[3], cx = R.vby[4], cy = R.vby[5];
    const float ac = ax + ((Y - ay) / (cy - ay)) * (cx - ax);
    float lo, hi;
    if (Y < byy) {
        const float ab = ax + ((Y - ay) / (byy - ay)) * (bx - ax);
        lo = rmin(ab, ac);
        hi = rmax(ab, ac);
    } else {
        const float bc = bx + ((Y - byy) / (cy - byy)) * (cx - bx);
        lo = rmin(bc, ac);
        hi = rmax(bc, ac);
    }
    const float fl = floorf(lo), ce = ceilf(hi);
    const float fxmin = (float)R.xmin, fxmax = (float)R.xmax;
    x0 = (fl >= fxmin && fl < fxmax) ? (uint32_t)fl : R.xmin;
    x1 = (ce >= fxmin && ce < fxmax) ? (uint32_t)ce : R.xmax;
}

EUCHIP_DEV void band_of(const FrameParams &p, const View &v, uint32_t y, uint32_t &by0, uint32_t &by1) {
    if (p.band_par) {
        by0 = (y / v.G) * v.G;
        by1 = by0 + v.G < v.H ? by0 + v.G : v.H;
    } else {
        by0 = 0;
        by1 = v.H;
    }
}

template <uint32_t SH>
EUCHIP_DEV void v_data(const TriRec &R, const float (*V)[VDN<SH>::N], float X, float Y, float *vd) {
    float w[3];
#pragma unroll
    for (int i = 0; i < 3; i++) w[i] = (R.o[i] + R.dy[i] * Y) + R.dx[i] * X;
    const float u2 = (w[2] - w[0]) - w[1];
    const float r = 1.0f / w[2];
    const float n0 = w[0] * r, n1 = w[1] * r, n2 = u2 * r;
    if constexpr (SH == FLAT) {
        vd[0] = V[0][0];
    } else {
#pragma unroll
        for (uint32_t c = 0; c < vd_count(SH); c++) vd[c] = (V[0][c] * n0 + V[1][c] * n1) + V[2][c] * n2;
    }
}

// VertexData of a record's corners, interpolated at (X, Y), through the fragment
// shader: the deferred shading of a winning fragment (pipeline.rs:539-541), or
// one coarse sample of it (pipeline.rs:541-570).
template <uint32_t SH, bool GS>
EUCHIP_DEV void shade_sample(const FrameParams &p, const View &v, const TriRec &R, const float (*V)[VDN<SH>::N], float X,
                             float Y, float frag[4]) {
    float vd[VDN<SH>::N];
    v_data<SH>(R, V, X, Y, vd);
    fragment_shader<SH, GS>(v, p.sampler, vd, frag);
}

// Tile geometry: TW x TH pixels at (X0, Y0); TW = 1 << sx, TH = 256 >> sx.
struct TileGeom {
    uint32_t X0, Y0, sx, TW, TH;
};

// The tile's pixels [xs, xe) of one row (LDS index pi0 of the first), w_hom at
// xs given: each pixel's fragment updates its winner key.  Rows of small
// triangles where the test reads the depth before the pass (key mode 0 with a
// depth test); the others take walk_span's loops.  One loop per test: with the test
// chosen inside it, a 1280x720 frame of 12 triangles over loaded depth 53.5 us
// instead of 47.8, one of 6000 large triangles 180 instead of 154.
template <uint32_t TEST>
EUCHIP_DEV void walk_row(const FrameParams &p, const TriRec &R, uint32_t prim, uint32_t xs, uint32_t xe, uint32_t pi0,
                         float w0, float w1, float w2, uint64_t *key, const float *d0s) {
    for (uint32_t x = xs; x < xe; x++) {
        float z;
        if (frag_z(p, R, w0, w1, w2, z)) {
            const uint32_t pi = pi0 + (x - xs);
            if (passes_depth(TEST, z, d0s[pi]))
                atomicMax((unsigned long long *)(key + pi), ((uint64_t)(prim + 1u) << 32) | __float_as_uint(z));
        }
        w0 = w0 + R.dx[0];
        w1 = w1 + R.dx[1];
        w2 = w2 + R.dx[2];
    }
}

// The row loop of the write modes and of frames without a depth test: coverage,
// z, z clip and the key of every pixel,
// then one LDS atomic min per pixel, with no branch: an uncovered pixel's
// atomic takes the all-ones key, which changes nothing.  The loop holds no LDS
// read, so nothing waits on the atomics of earlier pixels.
//   * A NaN weight makes z NaN (a NaN factor or term stays NaN), so z == z and
//     the minimum of the three weights >= 0 decide exactly what the three
//     tests w >= 0 and z == z decide.
//   * -0 + 0 = +0 gives both zeros one order value; z + 0 differs from z only
//     for z = -0 (NaN z never wins), in the sign bit alone, so that bit of
//     z ^ (z + 0) shifted in beside (prim + 1) keeps the sign in the key.
//   * An uncovered pixel's key has an all-ones high word: no stored key has
//     one (order values of non-NaN depths stay below it), so it never wins.
//   * MODE 3 (no depth test, no such write): the last fragment wins whatever its
//     z, a NaN among them, so the weights are tested one by one and an uncovered
//     pixel's atomic max takes zero, which changes nothing either.  (Reading the
//     depth before the pass for a test that always passes, with its atomic under
//     a branch, took 9 us for a tile's rows of 32 pixels.)
//   * PAIRS: two pixels per turn (the second atomic at the next address)
//     halve the loop control; a row of odd length ends with one more pixel.
//     It pays for long rows only.
template <uint32_t MODE, bool CLIP, bool PAIRS>
EUCHIP_DEV void walk_keys(const TriRec &R, bool clip, float zlo, float zhi, uint32_t pid, unsigned long long *kp,
                          unsigned long long *const ke, float w0, float w1, float w2) {
    auto pixel = [&](unsigned long long *at) {
        const float u2 = (w2 - w0) - w1;
        const float z = (R.hz[0] * w0 + R.hz[1] * w1) + R.hz[2] * u2;
        bool ok;
        if constexpr (MODE == 3u) ok = (w0 >= 0.0f) & (w1 >= 0.0f) & (u2 >= 0.0f);
        else ok = (__builtin_fminf(__builtin_fminf(w0, w1), u2) >= 0.0f) & (z == z);
        if constexpr (CLIP) ok = ok & (!clip | ((zlo <= z) & (z <= zhi)));
        const uint32_t bz = __float_as_uint(z), u = __float_as_uint(z + 0.0f);
        if constexpr (MODE == 3u) {
            atomicMax(at, ok ? ((uint64_t)pid << 32) | bz : 0ull);
            w0 = w0 + R.dx[0];
            w1 = w1 + R.dx[1];
            w2 = w2 + R.dx[2];
            return;
        }
        const uint32_t o = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
        const uint32_t lo = __builtin_amdgcn_alignbit(pid, bz ^ u, 31u);  // (pid << 1) | (z is -0)
        const uint32_t hi = ok ? (MODE == 1u ? o : ~o) : ~0u;
        atomicMin(at, ((uint64_t)hi << 32) | lo);
        w0 = w0 + R.dx[0];
        w1 = w1 + R.dx[1];
        w2 = w2 + R.dx[2];
    };
    if constexpr (PAIRS) {
        const uint32_t n = (uint32_t)(ke - kp);
        unsigned long long *const pairs_end = kp + (n & ~1u);
        for (; kp < pairs_end; kp += 2) {
            pixel(kp);
            pixel(kp + 1);
        }
        if (n & 1u) pixel(kp);
    } else {
        for (; kp < ke; kp++) pixel(kp);
    }
}

// walk_row without branches on the coverage; the write modes and frames without
// a depth test take walk_keys, with the z clip only where a lane of the wave needs it.
template <uint32_t MODE, bool PAIRS = false>
EUCHIP_DEV void walk_span(const FrameParams &p, const TriRec &R, uint32_t prim, uint32_t xs, uint32_t xe, uint32_t pi0,
                          float w0, float w1, float w2, uint64_t *key, const float *d0s) {
    const bool clip = !(R.flags & TRI_ALL_IN) && p.z_clip;
    if constexpr (MODE != 0u) {
        unsigned long long *kp = (unsigned long long *)(key + pi0);
        unsigned long long *const ke = kp + (xe - xs);
        if (__builtin_amdgcn_ballot_w64(clip) != 0ull)
            walk_keys<MODE, true, PAIRS>(R, clip, p.z_min, p.z_max, prim + 1u, kp, ke, w0, w1, w2);
        else
            walk_keys<MODE, false, PAIRS>(R, clip, p.z_min, p.z_max, prim + 1u, kp, ke, w0, w1, w2);
        return;
    }
    const float zlo = p.z_min, zhi = p.z_max;
    const uint32_t test = p.depth_test;
    const uint32_t pid = prim + 1u;
    for (uint32_t x = xs; x < xe; x++) {
        const float u2 = (w2 - w0) - w1;
        const float z = (R.hz[0] * w0 + R.hz[1] * w1) + R.hz[2] * u2;
        bool ok = (w0 >= 0.0f) & (w1 >= 0.0f) & (u2 >= 0.0f);
        ok = ok & (!clip | ((zlo <= z) & (z <= zhi)));
        const uint32_t pi = pi0 + (x - xs);
        const float D0 = d0s[pi];
        if (ok & passes_depth(test, z, D0)) atomicMax((unsigned long long *)(key + pi), ((uint64_t)pid << 32) | __float_as_uint(z));
        w0 = w0 + R.dx[0];
        w1 = w1 + R.dx[1];
        w2 = w2 + R.dx[2];
    }
}

// One row y of a triangle inside the tile: the row span (triangles.rs:219-254),
// then the walk from the row start exactly as the reference does
// (triangles.rs:257-301), testing the tile's pixels of the span.
template <uint32_t SKIP_UNROLL>
EUCHIP_DEV void raster_row(const FrameParams &p, const TriRec &R, uint32_t prim, uint32_t y, const TileGeom &g,
                           uint32_t mode, uint64_t *key, const float *d0s, const uint32_t *band) {
    uint32_t x0, x1;
    const uint32_t r = y - g.Y0;
    row_span(R, y, band[2 * r], band[2 * r + 1], x0, x1);
    const uint32_t xs = x0 > g.X0 ? x0 : g.X0;
    const uint32_t xe = x1 < g.X0 + g.TW ? x1 : g.X0 + g.TW;
    if (xs >= xe) return;
    const float Y = (float)y, X0 = (float)x0;
    float w0 = (R.o[0] + R.dy[0] * Y) + R.dx[0] * X0;
    float w1 = (R.o[1] + R.dy[1] * Y) + R.dx[1] * X0;
    float w2 = (R.o[2] + R.dy[2] * Y) + R.dx[2] * X0;
    // to the tile's first pixel, one addition per pixel as the reference walks
    // (SKIP_UNROLL pixels per turn: the same additions, less loop control)
    uint32_t x = x0;
    for (; x + SKIP_UNROLL <= xs; x += SKIP_UNROLL) {
#pragma unroll
        for (uint32_t q = 0; q < SKIP_UNROLL; q++) {
            w0 = w0 + R.dx[0];
            w1 = w1 + R.dx[1];
            w2 = w2 + R.dx[2];
        }
    }
    for (; x < xs; x++) {
        w0 = w0 + R.dx[0];
        w1 = w1 + R.dx[1];
        w2 = w2 + R.dx[2];
    }
    const uint32_t pi0 = r * (g.TW + 1u) + (xs - g.X0);
    // the long-row variant (big-triangle kernels) walks two pixels per turn
    if (mode == 1u) walk_span<1u, (SKIP_UNROLL > 4u)>(p, R, prim, xs, xe, pi0, w0, w1, w2, key, d0s);
    else if (mode == 2u) walk_span<2u, (SKIP_UNROLL > 4u)>(p, R, prim, xs, xe, pi0, w0, w1, w2, key, d0s);
    else if (p.depth_test == DT_NONE) walk_span<3u, (SKIP_UNROLL > 4u)>(p, R, prim, xs, xe, pi0, w0, w1, w2, key, d0s);
    else if (p.depth_test == DT_LESS) walk_row<DT_LESS>(p, R, prim, xs, xe, pi0, w0, w1, w2, key, d0s);
    else if (p.depth_test == DT_EQUAL) walk_row<DT_EQUAL>(p, R, prim, xs, xe, pi0, w0, w1, w2, key, d0s);
    else walk_row<DT_GREATER>(p, R, prim, xs, xe, pi0, w0, w1, w2, key, d0s);
}

constexpr uint32_t kMaxTileH = 32;
static_assert(kBatch <= 256u, "a batch is staged one entry per lane");

// Setup of one bin entry of the current batch, kept in LDS (24 words).
struct TriLds {
    float o[3], dx[3], dy[3], hz[3], vby[6];
    uint32_t xmin, xmax, ymin, ymax, flags, prim;
};

struct TileShared {
    // Per pixel of the tile, rows padded by one entry (pixel i at i + i / TW):
    // lanes walking the same column of different rows hit different banks.
    uint64_t key[256 + kMaxTileH];  // winner key
    float d0s[256 + kMaxTileH];     // depth before the pass (the test's reference)
    alignas(16) TriLds tri[kBatch]; // the batch's triangles (also coarse samples, 16 bytes each)
    uint32_t rows_incl[256];        // inclusive prefix sum of their row counts in the tile
    uint8_t owner[256];             // entry of each (entry, row) item of the current 256
    uint32_t wave_rows[4];          // row counts per wave (prefix-sum carry)
    uint32_t band[2 * kMaxTileH];   // [by0, by1) of the render_par band of each row
};

EUCHIP_DEV void put_tri(TriLds &T, const TriRec &R, uint32_t prim) {
#pragma unroll
    for (int i = 0; i < 3; i++) T.o[i] = R.o[i], T.dx[i] = R.dx[i], T.dy[i] = R.dy[i], T.hz[i] = R.hz[i];
#pragma unroll
    for (int i = 0; i < 6; i++) T.vby[i] = R.vby[i];
    T.xmin = R.xmin, T.xmax = R.xmax, T.ymin = R.ymin, T.ymax = R.ymax, T.flags = R.flags, T.prim = prim;
}

// Rows of bin entry `prim` inside the tile, its setup kept in sh.tri[slot].
EUCHIP_DEV uint32_t stage_entry(const FrameParams &p, uint32_t tri_base, TileShared &sh, uint32_t slot, uint32_t prim,
                                const TileGeom &g) {
    TriRec R;
    load_rec0(p, tri_base + prim, R);
    const uint32_t ry0 = R.ymin > g.Y0 ? R.ymin : g.Y0;
    const uint32_t ry1 = R.ymax < g.Y0 + g.TH ? R.ymax : g.Y0 + g.TH;
    const uint32_t xs = R.xmin > g.X0 ? R.xmin : g.X0;
    const uint32_t xe = R.xmax < g.X0 + g.TW ? R.xmax : g.X0 + g.TW;
    if (ry0 >= ry1 || xs >= xe) return 0u;
    if (!all_rows_boxed(R)) {
        load_rec1(p, tri_base + prim, R);
    } else {
#pragma unroll
        for (int i = 0; i < 6; i++) R.vby[i] = 0.0f;  // boxed rows never read verts_by_y
    }
    put_tri(sh.tri[slot], R, prim);
    return ry1 - ry0;
}

// Inclusive prefix sum over the workgroup (4 waves); every thread must call it.
EUCHIP_DEV uint32_t block_inclusive_sum(TileShared &sh, uint32_t tid, uint32_t v) {
    const uint32_t incl = wave_inclusive_sum(v);
    if ((tid & 63u) == 63u) sh.wave_rows[tid >> 6] = incl;
    __syncthreads();
    uint32_t carry = 0;
    for (uint32_t w = 0; w < (tid >> 6); w++) carry += sh.wave_rows[w];
    return incl + carry;
}

// Rank of this thread among the workgroup's threads with `on`, and their number;
// every thread must call it.
EUCHIP_DEV uint32_t block_rank(TileShared &sh, uint32_t tid, bool on, uint32_t &total) {
    const uint64_t bal = __ballot(on);
    if ((tid & 63u) == 0u) sh.wave_rows[tid >> 6] = (uint32_t)__popcll(bal);
    __syncthreads();
    uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
    total = 0u;
#pragma unroll
    for (uint32_t w = 0; w < 4u; w++) {
        const uint32_t c = sh.wave_rows[w];
        at += w < (tid >> 6) ? c : 0u;
        total += c;
    }
    return at;
}

// The rows of up to kBatch triangles staged in LDS, `rows` of this lane's inside
// the tile: the (triangle, row) pairs are spread over all lanes so no lane walks
// much more than one row.  Ends with a barrier.
template <bool OWNER, bool LONG_ROWS>
EUCHIP_DEV void walk_rows(TileShared &sh, uint32_t tid, uint32_t rows, const TileGeom &g) {
    const FrameParams &p = args();
    const uint32_t mode = key_mode(p);
    const uint32_t incl = block_inclusive_sum(sh, tid, rows);
    const uint32_t excl = incl - rows;
    sh.rows_incl[tid] = incl;
    // items [excl, incl) are this entry's rows; the owner table maps the first
    // 256 items back to their entries with one LDS read, later ones (batches
    // past 256 rows) search the prefix sums
    if constexpr (OWNER)
        for (uint32_t k = excl; k < incl && k < 256u; k++) sh.owner[k] = (uint8_t)tid;
    __syncthreads();
    const uint32_t total = sh.rows_incl[255];  // lanes past the batch add nothing
    for (uint32_t k = tid; k < total; k += 256u) {
        uint32_t e;
        if (OWNER && k < 256u) {
            e = sh.owner[k];
        } else {
            uint32_t lo = 0, hi = kBatch - 1u;  // first entry whose inclusive sum exceeds k
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (sh.rows_incl[mid] > k) hi = mid;
                else lo = mid + 1u;
            }
            e = lo;
        }
        const uint32_t base = e ? sh.rows_incl[e - 1u] : 0u;
        const TriLds &T = sh.tri[e];
        TriRec R;
#pragma unroll
        for (int i = 0; i < 3; i++) R.o[i] = T.o[i], R.dx[i] = T.dx[i], R.dy[i] = T.dy[i], R.hz[i] = T.hz[i];
#pragma unroll
        for (int i = 0; i < 6; i++) R.vby[i] = T.vby[i];
        R.xmin = T.xmin, R.xmax = T.xmax, R.ymin = T.ymin, R.ymax = T.ymax, R.flags = T.flags;
        const uint32_t ry0 = R.ymin > g.Y0 ? R.ymin : g.Y0;
        raster_row<LONG_ROWS ? 8u : 4u>(p, R, T.prim, ry0 + (k - base), g, mode, sh.key, sh.d0s, sh.band);
    }
    __syncthreads();  // the next batch reuses sh.tri and sh.rows_incl
}

// One batch of up to 256 bin entries: each lane stages its entry's setup in LDS,
// then the batch's rows are walked.
template <bool OWNER, bool LONG_ROWS>
EUCHIP_DEV void raster_batch(uint32_t tri_base, TileShared &sh, uint32_t tid, bool valid, uint32_t prim,
                             const TileGeom &g) {
    const uint32_t rows = valid ? stage_entry(args(), tri_base, sh, tid, prim, g) : 0u;
    walk_rows<OWNER, LONG_ROWS>(sh, tid, rows, g);
}

// The big triangles of `tile` from their row checkpoints: the tile's list of
// (triangle, rows whose span reaches into the tile), 256 entries at a time
// (one per lane, coalesced; the first 256 issued when the tile starts).  An
// entry whose key-order bound lies above `occl`, the least bound of the tiles'
// full-cover triangles, has no rows here (it loses every pixel).  A
// prefix sum over the row counts places each entry's rows in a task table
// (entry, row), and each lane takes table entries and walks one row from its
// checkpoint (weights and the span inside the tile's column, at the slot of
// triangle, column and row), with the triangle's dx, hz, flags and primitive
// from its big record (two loads beside the checkpoint's).
struct BigTaskLds {
    uint32_t tri[256];        // triangle of each entry of the round
    uint16_t task[256 * 8];   // entry << 3 | row of the tile
};
static_assert(sizeof(BigTaskLds) <= sizeof(TriLds) * kBatch, "big-triangle tasks fit the staging space");

EUCHIP_DEV void big_tasks(const FrameParams &p, TileShared &sh, uint32_t tid, uint32_t tile, uint32_t nbig,
                          uint32_t occl, const TileGeom &g, uint2 e_first) {
    const uint32_t mode = key_mode(p);
    BigTaskLds &bt = *reinterpret_cast<BigTaskLds *>(sh.tri);
    const uint2 *list = p.cktab + (size_t)tile * p.mstride;
    const uint4 *cktile = p.ck + (size_t)(g.X0 >> g.sx) * p.v0.H + g.Y0;  // triangle t's at + t * ntx * H
    const size_t ckstride = (size_t)p.v0.ntx * p.v0.H;
    for (uint32_t s0 = 0; s0 < nbig; s0 += 256u) {
        const uint2 e2 = s0 ? (s0 + tid < nbig ? list[s0 + tid] : make_uint2(0u, 0u)) : e_first;
        const uint32_t e = e2.x;
        // behind the tile's occluder at every pixel: no rows
        const uint32_t m = s0 + tid < nbig && e2.y <= occl ? e & 0xffu : 0u;
        const uint32_t mine = __builtin_popcount(m);
        uint32_t at = block_inclusive_sum(sh, tid, mine) - mine;
        const uint32_t total = sh.wave_rows[0] + sh.wave_rows[1] + sh.wave_rows[2] + sh.wave_rows[3];
        bt.tri[tid] = e >> 8;
        for (uint32_t mm = m; mm; mm &= mm - 1u) bt.task[at++] = (uint16_t)((tid << 3) | (uint32_t)__builtin_ctz(mm));
        __syncthreads();
        // two rows per lane per turn, both rows' loads issued before either walk
        for (uint32_t k0 = 0; k0 < total; k0 += 512u) {
            uint4 c[2], x6[2], x7[2];
            uint32_t r[2];
#pragma unroll
            for (uint32_t h = 0; h < 2u; h++) {
                const uint32_t k = k0 + h * 256u + tid;
                r[h] = 8u;  // no row
                if (k >= total) continue;
                const uint32_t tk = bt.task[k], tri = bt.tri[tk >> 3];
                r[h] = tk & 7u;
                const uint4 *q = p.big_rec + (size_t)tri * kBigRecQuads;
                c[h] = cktile[tri * ckstride + r[h]];
                x6[h] = q[0], x7[h] = q[1];
            }
#pragma unroll
            for (uint32_t h = 0; h < 2u; h++) {
                if (r[h] >= 8u) continue;
                const uint32_t xs = g.X0 + (c[h].w & 0xffffu), xe = g.X0 + (c[h].w >> 16);
                TriRec R;
                R.dx[0] = __uint_as_float(x6[h].z), R.dx[1] = __uint_as_float(x6[h].w);
                R.dx[2] = __uint_as_float(x7[h].x);
                R.hz[0] = __uint_as_float(x7[h].y), R.hz[1] = __uint_as_float(x7[h].z);
                R.hz[2] = __uint_as_float(x7[h].w);
                R.flags = x6[h].y >> 30;
                const uint32_t pi0 = r[h] * (g.TW + 1u) + (xs - g.X0);
                const float w0 = __uint_as_float(c[h].x), w1 = __uint_as_float(c[h].y);
                const float w2 = __uint_as_float(c[h].z);
                if (mode == 1u) walk_span<1u, true>(p, R, x6[h].x, xs, xe, pi0, w0, w1, w2, sh.key, sh.d0s);
                else if (mode == 2u) walk_span<2u, true>(p, R, x6[h].x, xs, xe, pi0, w0, w1, w2, sh.key, sh.d0s);
                else if (p.depth_test == DT_NONE) walk_span<3u, true>(p, R, x6[h].x, xs, xe, pi0, w0, w1, w2, sh.key, sh.d0s);
                else walk_span<0u>(p, R, x6[h].x, xs, xe, pi0, w0, w1, w2, sh.key, sh.d0s);
            }
        }
        __syncthreads();  // the next round reuses the table and the wave totals
    }
}

// A tile's keys resolved: depth and clears stored, the winners' pixels shaded.
// view() is the tile's request, read anew for each phase; sample(v, prim, X, Y,
// frag) is the fragment of primitive prim at (X, Y).
template <uint32_t SH, bool MS, class ViewF, class SampleF>
EUCHIP_DEV void resolve_tile(TileShared &sh, uint32_t tid, const TileGeom &g, ViewF view, SampleF sample) {
    const uint32_t sx = g.sx;
    bool shade = false;  // this lane's pixel has a winner to shade
    {
        const FrameParams &p = args();
        const View &v = view();
        const uint32_t mode = key_mode(p);
        const uint32_t px = g.X0 + (tid & (g.TW - 1u)), py = g.Y0 + (tid >> sx);
        if (px < v.W && py < v.H) {
            const size_t pidx = (size_t)py * v.W + px;
            const uint64_t kk = sh.key[tid + (tid >> sx)];
            bool has;  // a winner (its primitive is read again by the shading lanes)
            float z;
            if (mode == 0u) {
                has = kk != 0ull;
                z = __uint_as_float((uint32_t)kk);
            } else {
                has = ((uint32_t)kk) != 0u;
                const uint32_t o = (uint32_t)(kk >> 32);
                z = zunord(mode == 1u ? o : ~o, (uint32_t)kk & 1u);
            }
            shade = v.pixel && p.pixel_write && has && SH != DEPTH_ONLY;
            if (v.pixel && !shade && v.clear_color_en) store_stream(&v.pixel[pidx], v.clear_color);
            if (v.depth) {
                if (has && p.depth_write) store_stream(&v.depth[pidx], z);
                else if (v.clear_depth_en) store_stream(&v.depth[pidx], v.clear_depth);
            }
        }
    }
    if constexpr (SH != DEPTH_ONLY && (!MS || SH == FLAT)) {  // (FLAT is the same at every coarse sample)
        // The pixels to shade, packed onto the first lanes in tile order: a wave
        // with none of them skips the shader.
        uint32_t total;
        const uint32_t at = block_rank(sh, tid, shade, total);
        if (shade) sh.owner[at] = (uint8_t)tid;
        __syncthreads();
        if (tid < total) {
            const FrameParams &p = args();
            const View &v = view();
            const uint32_t t = sh.owner[tid];
            const uint32_t tx2 = g.X0 + (t & (g.TW - 1u)), ty2 = g.Y0 + (t >> sx);
            const uint32_t prim = key_prim(key_mode(p), sh.key[t + (t >> sx)]) - 1u;
            float frag[4];
            sample(v, prim, (float)tx2, (float)ty2, frag);
            store_stream(&v.pixel[(size_t)ty2 * v.W + tx2], blend_shader<SH>(0u, frag, p.bgra));
        }
    } else if constexpr (SH != DEPTH_ONLY) {
        // Coarse shading (pipeline.rs:541-570): a pixel combines four samples of
        // its winner at the corners of its cell of the band's 2^L grid.  Pixels
        // of a cell with the same winner have the same samples; a 2 x 2 block
        // of even band rows and columns always lies in one cell, so the samples
        // are taken once per block and winner: its first pixel leads.  Each lane
        // takes one sample of a leader, 64 leaders a round, into LDS, and the
        // pixels combine them.  (With four samples per pixel and lane the
        // 1080p terrain's main pass spent three quarters of its vector
        // instructions on samples that its neighbours took as well.)
        const uint32_t mode = key_mode(args());
        const uint32_t tx = tid & (g.TW - 1u), ty = tid >> sx;
        const uint32_t by0 = sh.band[2 * ty], pid = shade ? key_prim(mode, sh.key[tid + ty]) : 0u;
        uint32_t leader = tid;
        if (shade) {
            const uint32_t odd = (g.Y0 + ty - by0) & 1u;  // second row of its block
            const uint32_t x0 = tx & ~1u, row = odd ? ty - 1u : ty;
            const bool above = odd && ty > 0u;  // its first row is in this tile (and then in this band)
            if (tx & 1u && key_prim(mode, sh.key[ty * (g.TW + 1u) + x0]) == pid) leader = (ty << sx) + x0;
            if (above) {
                if (key_prim(mode, sh.key[row * (g.TW + 1u) + x0 + 1u]) == pid) leader = (row << sx) + x0 + 1u;
                if (key_prim(mode, sh.key[row * (g.TW + 1u) + x0]) == pid) leader = (row << sx) + x0;
            }
        }
        uint32_t total;
        const uint32_t at = block_rank(sh, tid, shade && leader == tid, total);
        if (shade && leader == tid) sh.owner[at] = (uint8_t)tid, sh.rows_incl[tid] = at;
        __syncthreads();
        const uint32_t mine = shade ? sh.rows_incl[leader] : ~0u;  // the leader's rank
        float4 *const samples = reinterpret_cast<float4 *>(&sh.tri[kTinyTris]);
        static_assert(sizeof(TriLds) * (kBatch - kTinyTris) >= 256u * sizeof(float4), "a round's samples fit the staging space");
        static_assert(alignof(TileShared) % alignof(float4) == 0u &&
                          (offsetof(TileShared, tri) + kTinyTris * sizeof(TriLds)) % alignof(float4) == 0u,
                      "samples are read and written 16 bytes at a time");
        for (uint32_t b = 0; b < total; b += 64u) {
            const FrameParams &p = args();
            const View &v = view();
            const uint32_t L = p.msaa_level;
            if (b + (tid >> 2) < total) {
                const uint32_t t = sh.owner[b + (tid >> 2)], q = tid & 3u;
                const uint32_t prim = key_prim(mode, sh.key[t + (t >> sx)]) - 1u;
                const uint32_t b0 = sh.band[2 * (t >> sx)];
                const uint32_t cx = (g.X0 + (t & (g.TW - 1u))) >> L, cy = (g.Y0 + (t >> sx) - b0) >> L;
                float frag[4];
                sample(v, prim, (float)((cx + (q & 1u)) << L), (float)(b0 + ((cy + (q >> 1)) << L)), frag);
                samples[tid] = make_float4(frag[0], frag[1], frag[2], frag[3]);
            }
            __syncthreads();
            if (mine - b < 64u) {
                // bilinear reconstruction (pipeline.rs:556-570)
                const float div = 1.0f / (float)(1u << L);
                const float fx = rfract((float)(g.X0 + tx) * div), fy = rfract((float)(g.Y0 + ty - by0) * div);
                const float4 *s4 = samples + 4u * (mine - b);  // t00, t10, t01, t11
                const float4 t00 = s4[0], t10 = s4[1], t01 = s4[2], t11 = s4[3];
                const float c00[4] = {t00.x, t00.y, t00.z, t00.w}, c10[4] = {t10.x, t10.y, t10.z, t10.w};
                const float c01[4] = {t01.x, t01.y, t01.z, t01.w}, c11[4] = {t11.x, t11.y, t11.z, t11.w};
                float frag[4];
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const float t0 = c00[c] * (1.0f - fy) + c01[c] * fy;
                    const float t1 = c10[c] * (1.0f - fy) + c11[c] * fy;
                    frag[c] = t0 * (1.0f - fx) + t1 * fx;
                }
                store_stream(&v.pixel[(size_t)(g.Y0 + ty) * v.W + g.X0 + tx], blend_shader<SH>(0u, frag, p.bgra));
            }
            __syncthreads();  // the next round's samples reuse the space
        }
    }
}

// Waves per SIMD the raster pass is compiled for: what its registers allow
// without spills.  The big-triangle kernels hold two row tasks per lane and take
// 6 (their frames have few tiles, so fewer waves per SIMD than that are resident
// anyway).
constexpr uint32_t raster_waves(uint32_t sh, bool big) {
    return big ? 6u : (sh == PHONG_SHADOW || sh == TEX_SHADOW) ? 7u : 8u;
}

template <uint32_t SH, bool BATCH, bool BIG, bool GS, bool MS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(raster_waves(SH, BIG)))) void k_raster(FrameParams) {
    __shared__ TileShared sh;
    warm_args();
    const uint32_t tid = threadIdx.x;
    // p.heavy_groups workgroups for the heavy tiles, so that the longest tiles start
    // first, then one per tile of the launch (see launch_raster): the w-th of its XCD
    // takes busy tile w of the XCD's list and clears tile t0 + w if it is empty.  The
    // hardware starts them as others end: a queue of tiles for resident workgroups
    // took a returning atomic, a list load and a count load per tile, one after the
    // other, and left the empty tiles to the end.  A workgroup's own chain of loads is
    // short and all of it scalar: counters, list entry and counts cost no vector
    // instruction.  Against that queue: a 1366x768 Gouraud frame 26.7 -> 23.1 us,
    // 1080p Phong 42.8 -> 36.8, 3840x2160 128 -> 126, a batch of 1024 icons 446 ->
    // 416.
    // Where more tiles are heavy than have a workgroup of their own (large triangles
    // in many tiles each, dense meshes), all tiles are taken by the workgroups of the
    // busy lists, none in front, except that twice as many heavy tiles, while they are
    // an eighth of the frame's tiles at most, go in front still, two to a workgroup.
    // With all left to the heavy workgroups / as now, us: a 640x480 frame of 3000
    // large triangles (24 workgroups for 2400 heavy tiles) 2600 / 246, 1280x720 frames
    // of 1.2 million small ones 279 / 143 and of 590,000 51 / 43.  With none in front
    // past one each / as now: the 1080p terrain 110.7 / 106.2, a 1080p torus frame of
    // 590,000 triangles 51.1 / 49.1; without the bound of an eighth that 1280x720
    // frame takes 50.3.
    const uint32_t xcd = blockIdx.x & 7u;
    uint32_t w, per_xcd, nh, nbusy, nbig, pool_used, tile;
    uint32_t t0, t1;   // the XCD's contiguous range of tiles
    uint32_t count;    // bin entries of tile t0 + w
    bool clears;       // it has such a tile and the frame has clears
    bool heavy_apart = !BATCH;  // heavy tiles go to the heavy workgroups, not with the busy ones
    {
        const FrameParams &p = args();
        const uint32_t par = p.frame & 1u, npar = (p.frame + 1u) & 1u;
        const Counters *ctr = p.ctr;
        uint32_t lbase, lcap;
        busy_list_span(p, xcd, lbase, lcap);
        xcd_range(p.ntiles, xcd, t0, t1);
        const bool for_heavy = blockIdx.x < p.heavy_groups;
        per_xcd = (gridDim.x - p.heavy_groups) >> 3;
        w = (blockIdx.x - p.heavy_groups) >> 3;
        // the loads that the work waits for, issued together (list entries and
        // counts at clamped places, used only where they exist)
        const uint32_t flags = uniform_load(&ctr->flags[par][0]);
        pool_used = uniform_load(&ctr->pool[par][0]);
        nh = uniform_load(&ctr->heavy[par][0]);
        // big triangles (with checkpoints any triangle may be on any tile's list)
        nbig = !BIG ? 0u : p.ck_on ? p.v0.n_tris : uniform_load(&ctr->big[par][0]);
        nbusy = uniform_load(&ctr->busy[par][xcd][0]);
        tile = for_heavy ? uniform_load(p.heavy + blockIdx.x) : uniform_load(p.busy + lbase + (w < lcap ? w : 0u));
        clears = !for_heavy && t0 + w < t1;
        count = uniform_load(&p.tile_count[clears ? t0 + w : 0u].count);
        if (p.report && blockIdx.x == 0u && tid == 0u) {
            // this frame's setup counts, for the host (frame number last)
            Report *rp = p.report;
            rp->max_count = p.ctr->max_count[par][0];
            rp->flags = flags;
            rp->pool_used = pool_used;
            if (flags & FLAG_BIN_OVERFLOW) rp->dropped = rp->dropped + 1u;
            __threadfence_system();
            rp->frame = p.frame;
        }
        // The next frame's counters start at zero (its setup counts into them).
        if (blockIdx.x == 0u && tid == 0u) {
            p.ctr->pool[npar][0] = 0u;
            p.ctr->flags[npar][0] = 0u;
            p.ctr->max_count[npar][0] = 0u;
            p.ctr->heavy[npar][0] = 0u;
            p.ctr->big[npar][0] = 0u;
        }
        if (blockIdx.x < 8u && tid == 0u) p.ctr->busy[npar][xcd][0] = 0u;
        for (uint32_t i = blockIdx.x * 256u + tid; i < p.zero_n; i += gridDim.x * 256u) p.count_next[i] = TileBin{0u, 0u};
        if constexpr (BIG)  // after a checkpoint frame: its list counts
            for (uint32_t i = blockIdx.x * 256u + tid; i < p.ck_zero_n; i += gridDim.x * 256u)
                p.ck_count_next[i] = make_uint2(0u, 0u);
        // The pool ran out in setup: entries were lost, the frame is dropped (the
        // host sees the flag and re-runs it with a larger pool).
        if (flags & FLAG_BIN_OVERFLOW) return;
        pool_used = pool_used < p.pool_cap ? pool_used : p.pool_cap;
        if (BIG && !p.ck_on) nbig = nbig < p.big_cap ? nbig : p.big_cap;
        nh = nh < p.heavy_cap ? nh : p.heavy_cap;
        nbusy = nbusy < lcap ? nbusy : lcap;
        if constexpr (!BATCH) {
            heavy_apart = p.heavy_cap && (nh <= p.heavy_groups || (nh <= 2u * p.heavy_groups && nh <= p.ntiles / 8u));
            if (for_heavy && (!heavy_apart || blockIdx.x >= nh)) return;
        }
        // With big triangles every tile may hold fragments: each workgroup then
        // takes its tile of the XCD's contiguous range, none is cleared apart.
        if (BIG && nbig) nbusy = t1 - t0, clears = false, tile = for_heavy ? tile : t0 + w;
        if (!BATCH && !p.v0.clear_color_en && !p.v0.clear_depth_en) clears = false;
        if (!for_heavy && w >= nbusy) tile = ~0u;
    }

    // This workgroup's tile of the XCD's range where it is empty (launches of more
    // tiles than workgroups: its tiles): the clears, stores only.
    for (uint32_t ctile = t0 + w; clears;) {
        if (count == 0u) {
            const FrameParams &p = args();
            const uint32_t sx = p.tile_sx;
            uint32_t r = 0;
            if constexpr (BATCH) r = __builtin_amdgcn_readfirstlane(uniform_load(p.tile_req + ctile));
            const View &v = view_of<BATCH>(p, r);
            const uint32_t lt = ctile - v.tile_base;
            const uint32_t ty = divide(lt, v.row_tiles), tx = lt - ty * v.ntx;
            const uint32_t px = (tx << sx) + (tid & ((1u << sx) - 1u)), py = (ty << (8u - sx)) + (tid >> sx);
            if (px < v.W && py < v.H) {
                const size_t pidx = (size_t)py * v.W + px;
                if (v.pixel && v.clear_color_en) store_stream(&v.pixel[pidx], v.clear_color);
                if (v.depth && v.clear_depth_en) store_stream(&v.depth[pidx], v.clear_depth);
            }
        }
        if (t1 - ctile <= per_xcd) break;
        ctile += per_xcd;
        count = uniform_load(&args().tile_count[ctile].count);
    }

    // One tile with `cnt` bin entries and overflow list `head`: winner keys in
    // LDS, then the resolve.  Ends with a barrier (LDS is reused by a next tile).
    // Loads the bin state `ntb` of the workgroup's next tile on the way.
    auto run_tile = [&](uint32_t tile, uint32_t cnt, uint32_t head, uint32_t ntile, TileBin &ntb) {
        uint32_t r = 0u, lt, sx, nck = 0u, occl = 0u, run, nb, tri_base;
        uint64_t bin_at;  // first bin slot of the tile
        uint32_t ahead = 0u;  // this lane's entry of the next step of the bin, loaded a step ahead
        uint32_t seg = 0u;
        TileGeom g;
        uint2 e_first = make_uint2(0u, 0u);
        bool ckp = false;  // big triangles from their row checkpoints (else walked from the row starts)
        {
            const FrameParams &p = args();
            if constexpr (BATCH) r = __builtin_amdgcn_readfirstlane(uniform_load(p.tile_req + tile));
            const View &v = view_of<BATCH>(p, r);
            lt = tile - v.tile_base;
            tri_base = v.tri_base;
            bin_at = v.bin_base + (uint64_t)lt * v.tile_cap;
            nb = cnt < v.tile_cap ? cnt : v.tile_cap;
            seg = cnt > v.tile_cap ? head : 0u;
            if (tid < kBatch && tid < nb) ahead = p.bins[bin_at + tid];
            const uint32_t ty = divide(lt, v.row_tiles), tx = lt - ty * v.ntx;
            sx = p.tile_sx;
            g.sx = sx, g.TW = 1u << sx, g.TH = 256u >> sx;
            g.X0 = tx << sx, g.Y0 = ty << (8u - sx);
            const uint32_t px = g.X0 + (tid & (g.TW - 1u)), py = g.Y0 + (tid >> sx);
            float D0 = 0.0f;
            if (p.depth_test != DT_NONE || p.depth_write) {
                D0 = v.clear_depth;
                if (!v.clear_depth_en && px < v.W && py < v.H) D0 = v.depth[(size_t)py * v.W + px];
            }
            const uint32_t lp = tid + (tid >> sx);  // padded LDS index of this lane's pixel
            sh.key[lp] = init_key(key_mode(p), D0);
            sh.d0s[lp] = D0;
            if (tid < g.TH) {
                uint32_t by0, by1;
                band_of(p, v, g.Y0 + tid, by0, by1);
                sh.band[2 * tid] = by0;
                sh.band[2 * tid + 1] = by1;
            }
            // the tile's checkpoint list: its length and first 256 entries, loaded
            // now (used after the bin; entries past the length are ignored)
            if constexpr (BIG) {
                ckp = p.ck_on;
                if (ckp) {
                    const uint2 cc = p.ck_count[tile];
                    nck = cc.x, occl = ~cc.y;
                    if (tid < p.mstride) e_first = p.cktab[(size_t)tile * p.mstride + tid];
                }
            }
            run = nb + (ckp ? 0u : nbig);  // entries of the current run
        }
        __syncthreads();
        // Steps of up to kBatch entries: this tile's bin and the big triangles
        // (staging drops those that miss it), then (only when it overflowed) its
        // overflow segments, as many as fill a step together.  Segments were taken
        // from the pool in this frame, each pointing at the one taken before it; a
        // walk of at most pool_used / 3 segments whose every read stays below
        // pool_used ends even on a damaged list.  (There is one segment per setup
        // workgroup that passed the capacity, so often of a few entries: with a
        // step each, a tile of 831 entries ended a batch's launch 110 us after all
        // others.)  One loop, so one copy of raster_batch.
        uint32_t sbase = 0u, slen = 0u, guard = 0u;  // rest of the current segment
        for (uint32_t b = 0;;) {
            bool valid = false;
            uint32_t prim = 0;
            if (b < run) {
                const uint32_t i = b + tid;
                if (tid >= kBatch || i >= run) {
                } else if (i < nb) {
                    valid = true, prim = ahead;
                    if (i + kBatch < nb) ahead = args().bins[bin_at + i + kBatch];
                } else if constexpr (BIG) {
                    valid = true, prim = args().big[i - nb];
                }
                b += kBatch;
            } else {
                if ((seg | slen) == 0u) break;
                const uint32_t *pool = args().pool;
                uint32_t fill = 0u, at = 0u;
                while (fill < kBatch) {  // uniform
                    if (slen == 0u) {
                        if (!seg || guard++ > pool_used / 3u || seg + 1u > pool_used) break;
                        const uint32_t s0 = seg - 1u;
                        seg = uniform_load(pool + s0);
                        slen = uniform_load(pool + s0 + 1u);
                        sbase = s0 + 2u;
                        slen = slen < pool_used - sbase ? slen : pool_used - sbase;
                        continue;
                    }
                    const uint32_t take = slen < kBatch - fill ? slen : kBatch - fill;
                    if (tid - fill < take) at = sbase + (tid - fill);
                    fill += take, sbase += take, slen -= take;
                }
                if (fill == 0u) break;
                // (read once; a plain load would be merged with the bin's into one FLAT load)
                valid = tid < fill;
                if (valid) prim = __builtin_nontemporal_load(&pool[at]);
            }
            raster_batch<!BATCH, BIG>(tri_base, sh, tid, valid, prim, g);
        }
        if (BIG && ckp) {
            nck = __builtin_amdgcn_readfirstlane(nck);
            if (nck) big_tasks(args(), sh, tid, tile, nck, __builtin_amdgcn_readfirstlane(occl), g, e_first);
        }
        if (ntile != ~0u) ntb = uniform_load(&args().tile_count[ntile]);
        // a winner's sample from its setup record and its corners' VertexData
        resolve_tile<SH, MS>(
            sh, tid, g, [&]() -> const View & { return view_of<BATCH>(args(), r); },
            [&](const View &v, uint32_t prim, float X, float Y, float frag[4]) {
                const FrameParams &p = args();
                TriRec R;
                load_rec0(p, tri_base + prim, R);
                tri_sids(v, p.geometry, prim, R.flags, R.sid);
                constexpr uint32_t NV = VDN<SH>::N;
                float V[3][NV];
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const float *src = p.vary + (size_t)R.sid[i] * vd_count(SH);
#pragma unroll
                    for (uint32_t c = 0; c < vd_count(SH); c++) V[i][c] = src[c];
                }
                shade_sample<SH, GS>(p, v, R, V, X, Y, frag);
            });
        __syncthreads();
    };

    // This workgroup's tiles: one, or every per_xcd-th (heavy_groups-th) where the
    // launch has more tiles than workgroups.  The next one's list entry is loaded
    // at the start of a tile, its bin state before the resolve.
    const bool heavy = blockIdx.x < args().heavy_groups;
    uint32_t k = heavy ? blockIdx.x : w;
    const uint32_t stride = heavy ? args().heavy_groups : per_xcd, bound = heavy ? nh : nbusy;
    TileBin tb = tile != ~0u ? uniform_load(&args().tile_count[tile]) : TileBin{0u, 0u};
    while (tile != ~0u) {
        uint32_t ntile = ~0u;
        k += stride;
        if (k < bound) {
            const FrameParams &p = args();
            uint32_t lbase, lcap, b0, b1;
            busy_list_span(p, xcd, lbase, lcap);
            xcd_range(p.ntiles, xcd, b0, b1);
            if (heavy) ntile = uniform_load(p.heavy + k);
            else if (BIG && nbig) ntile = b0 + k;
            else ntile = uniform_load(p.busy + lbase + k);
        }
        TileBin ntb{0u, 0u};
        if (heavy || !heavy_apart || tb.count < kHeavyTile)
            run_tile(tile, tb.count, tb.head, ntile, ntb);
        else if (ntile != ~0u)  // a heavy tile of the busy list: another workgroup's
            ntb = uniform_load(&args().tile_count[ntile]);
        tile = ntile, tb = ntb;
    }
}

// k_tiny: one-request frames of few triangles (the rule and both sides' times are
// at kTinyTris) in one launch.  Every workgroup sets all triangles up itself
// (a lane each) and computes their corners' VertexData, all kept in LDS, then
// takes tile after tile: rows of every triangle that reaches into the tile,
// walked from their starts, and the resolve.  Nothing passes through memory but
// the mesh, the textures and the targets, and no launch waits for another.  (The
// walks from the row starts grow with the square of the width, a checkpoint
// frame's with the width.)
template <uint32_t SH, bool GS, bool MS>
__global__ __launch_bounds__(256) void k_tiny(FrameParams) {
    __shared__ TileShared sh;
    __shared__ float vd[kTinyTris][3][VDN<SH>::N];
    warm_args();
    const uint32_t tid = threadIdx.x;
    {
        const FrameParams &p = args();
        const View &v = p.v0;
        if (tid < kTinyTris) {
            TriRec R;
            R.flags = 0u;
            const bool keep = tid < v.n_tris && tri_setup(p, v, tid, R);
            if (!keep) R.ymin = R.ymax = 0u;  // no row in any tile
            put_tri(sh.tri[tid], R, tid);
        }
        __syncthreads();
        if (tid < 3u * v.n_tris) {  // corner i of triangle t in the order after the winding swap
            const uint32_t t = tid / 3u, i = tid - 3u * t, c = (sh.tri[t].flags & TRI_SWAPPED) && i != 1u ? 2u - i : i;
            uint32_t inst[3], at[3];
            corner_places(v, p.geometry, t, inst, at);
            const uint32_t in = c == 0u ? inst[0] : c == 1u ? inst[1] : inst[2];
            const uint32_t k = c == 0u ? at[0] : c == 1u ? at[1] : at[2];
            vertex_data<SH>(p, v, in, v.idx ? v.idx[k] : k, vd[t][i]);
        }
    }
    for (uint32_t tile = blockIdx.x; tile < args().ntiles; tile += gridDim.x) {
        TileGeom g;
        uint32_t rows = 0u;
        {
            const FrameParams &p = args();
            const View &v = p.v0;
            const uint32_t ty = divide(tile, v.row_tiles), tx = tile - ty * v.ntx;
            g.sx = p.tile_sx, g.TW = 1u << g.sx, g.TH = 256u >> g.sx;
            g.X0 = tx << g.sx, g.Y0 = ty << (8u - g.sx);
            const uint32_t px = g.X0 + (tid & (g.TW - 1u)), py = g.Y0 + (tid >> g.sx);
            float D0 = 0.0f;
            if (p.depth_test != DT_NONE || p.depth_write) {
                D0 = v.clear_depth;
                if (!v.clear_depth_en && px < v.W && py < v.H) D0 = v.depth[(size_t)py * v.W + px];
            }
            const uint32_t lp = tid + (tid >> g.sx);
            sh.key[lp] = init_key(key_mode(p), D0);
            sh.d0s[lp] = D0;
            if (tid < g.TH) {
                uint32_t by0, by1;
                band_of(p, v, g.Y0 + tid, by0, by1);
                sh.band[2 * tid] = by0;
                sh.band[2 * tid + 1] = by1;
            }
            if (tid < v.n_tris) {
                const TriLds &T = sh.tri[tid];
                const uint32_t ry0 = T.ymin > g.Y0 ? T.ymin : g.Y0, ry1 = T.ymax < g.Y0 + g.TH ? T.ymax : g.Y0 + g.TH;
                const bool in = ry0 < ry1 && T.xmin < g.X0 + g.TW && T.xmax > g.X0;
                rows = in ? ry1 - ry0 : 0u;
            }
        }
        walk_rows<true, true>(sh, tid, rows, g);
        resolve_tile<SH, MS>(
            sh, tid, g, [&]() -> const View & { return args().v0; },
            [&](const View &v, uint32_t prim, float X, float Y, float frag[4]) {
                const TriLds &T = sh.tri[prim];
                TriRec R;
#pragma unroll
                for (int i = 0; i < 3; i++) R.o[i] = T.o[i], R.dx[i] = T.dx[i], R.dy[i] = T.dy[i];
                shade_sample<SH, GS>(args(), v, R, vd[prim], X, Y, frag);
            });
        __syncthreads();  // the next tile reuses the keys
    }
}

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t *dst, uint32_t v, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (i < n) dst[i] = v;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline uint32_t blocks_of(size_t n, uint32_t b) { return (uint32_t)((n + b - 1) / b); }

constexpr uint32_t kSmallMesh = 32768;

template <uint32_t SH>
static void launch_setup_t(const FrameParams &p, hipStream_t s, bool batched, uint32_t blocks) {
    if (batched) {
        hipLaunchKernelGGL((k_setup<SH, true, false>), dim3(blocks), dim3(256), 0, s, p);
    } else {
        // triangle blocks, then vertex blocks; checkpoint frames: blocks of
        // triangles and vertices, then span blocks
        FrameParams q = p;
        uint32_t span_blocks = 0;
        size_t lds = 0;
        if (p.ck_on && p.v0.H) {  // span blocks: 4 items of kSpanRows rows per triangle and block
            const uint32_t sy = 8u - p.tile_sx;
            q.span_parts = (p.v0.H + (1u << sy) + kSpanRows - 1u) / kSpanRows;
            span_blocks = p.v0.n_tris * ((q.span_parts + 3u) / 4u);
            const size_t tables = 4u * (size_t)span_table_bytes(sy, p.v0.ntx);  // in the static LDS when it fits
            lds = tables <= sizeof(SetupShared) ? 0u : tables;
        }
        const size_t nv = (size_t)p.v0.n_instances * p.v0.n_vertices;
        if (span_blocks) {
            q.tri_block = 256u;
            q.tri_blocks = q.setup_blocks = blocks_of(std::max<size_t>(p.v0.n_tris, nv), 256);
        } else {
            // Small meshes: 64 triangles a workgroup, so that the chip is not left idle
            // and a workgroup's pairs fit a round or two. With 256 against 64, us per
            // pass: 16 draws of 3000 triangles 295 / 275, a shadowed frame of 6400 54.9
            // / 45.3; tori of 32,768 triangles at 640, 1280 and 1920 columns 22.5 / 23.3,
            // 22.0 / 21.5 and 25.1 / 24.6, of 76,800 23.6 / 24.1, 25.7 / 26.4 and 27.7 /
            // 27.7, of 262,144 27.9 / 33.3, 32.8 / 36.9 and 34.5 / 38.9.
            q.tri_block = p.v0.n_tris <= kSmallMesh ? 64u : 256u;
            q.tri_blocks = blocks_of(p.v0.n_tris, q.tri_block);
            q.setup_blocks = q.tri_blocks + (vd_count(SH) > 0 ? blocks_of(nv, 256) : 0u);
        }
        if (span_blocks)
            hipLaunchKernelGGL((k_setup<SH, false, true>), dim3(q.setup_blocks + span_blocks), dim3(256), lds, s, q);
        else
            hipLaunchKernelGGL((k_setup<SH, false, false>), dim3(q.setup_blocks), dim3(256), 0, s, q);
    }
}

hipError_t launch_setup(const FrameParams &p, hipStream_t s, bool batched, uint32_t blocks) {
    if (batched && blocks == 0) return hipSuccess;
    switch (p.shader) {
    case FLAT: launch_setup_t<FLAT>(p, s, batched, blocks); break;
    case COLOR: launch_setup_t<COLOR>(p, s, batched, blocks); break;
    case GOURAUD: launch_setup_t<GOURAUD>(p, s, batched, blocks); break;
    case PHONG: launch_setup_t<PHONG>(p, s, batched, blocks); break;
    case DEPTH_ONLY: launch_setup_t<DEPTH_ONLY>(p, s, batched, blocks); break;
    case TEXTURED: launch_setup_t<TEXTURED>(p, s, batched, blocks); break;
    case PHONG_SHADOW: launch_setup_t<PHONG_SHADOW>(p, s, batched, blocks); break;
    case TEX_SHADOW: launch_setup_t<TEX_SHADOW>(p, s, batched, blocks); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <uint32_t SH, bool GS, bool MS>
static void launch_raster_m(const FrameParams &p, hipStream_t s, bool batched, uint32_t groups) {
    if (batched) hipLaunchKernelGGL((k_raster<SH, true, false, GS, MS>), dim3(groups), dim3(256), 0, s, p);
    else if (p.big_cap) hipLaunchKernelGGL((k_raster<SH, false, true, GS, MS>), dim3(groups), dim3(256), 0, s, p);
    else hipLaunchKernelGGL((k_raster<SH, false, false, GS, MS>), dim3(groups), dim3(256), 0, s, p);
}

template <uint32_t SH, bool GS>
static void launch_raster_g(const FrameParams &p, hipStream_t s, bool batched, uint32_t groups) {
    if (p.msaa_level) launch_raster_m<SH, GS, true>(p, s, batched, groups);
    else launch_raster_m<SH, GS, false>(p, s, batched, groups);
}

template <uint32_t SH, bool GS>
static void launch_tiny_g(const FrameParams &p, hipStream_t s, uint32_t groups) {
    if (p.msaa_level) hipLaunchKernelGGL((k_tiny<SH, GS, true>), dim3(groups), dim3(256), 0, s, p);
    else hipLaunchKernelGGL((k_tiny<SH, GS, false>), dim3(groups), dim3(256), 0, s, p);
}

// Textured shaders whose sampler is not their own take the kernels that read
// textures through any sampler kind.
template <uint32_t SH>
static void launch_raster_t(const FrameParams &p, hipStream_t s, bool batched, uint32_t groups) {
    if constexpr (SH == TEXTURED || SH == TEX_SHADOW) {
        const uint32_t own = SH == TEX_SHADOW ? (uint32_t)SAMPLER_LINEAR_CLAMPED : (uint32_t)SAMPLER_LINEAR;
        if (p.sampler != own) {
            launch_raster_g<SH, true>(p, s, batched, groups);
            return;
        }
    }
    launch_raster_g<SH, false>(p, s, batched, groups);
}

template <uint32_t SH>
static void launch_tiny_t(const FrameParams &p, hipStream_t s, uint32_t groups) {
    if constexpr (SH == TEXTURED || SH == TEX_SHADOW) {
        const uint32_t own = SH == TEX_SHADOW ? (uint32_t)SAMPLER_LINEAR_CLAMPED : (uint32_t)SAMPLER_LINEAR;
        if (p.sampler != own) {
            launch_tiny_g<SH, true>(p, s, groups);
            return;
        }
    }
    launch_tiny_g<SH, false>(p, s, groups);
}

// ---------------------------------------------------------------------------
// Span blocks of a checkpoint frame's setup launch: block b walks rows of
// triangle t = b % n_tris, its wave w the item 4 * (b / n_tris) + w (kSpanRows
// rows from the triangle's first tile row).  Wave 0 sets the triangle up
// (tri_setup, as the setup blocks do, which write its records and bin none of
// a checkpoint frame's triangles).  A lane takes a row: the row span
// (triangles.rs:219-254, with the row's band), a bit in the wave's LDS mask
// table for every tile column the span touches, then the walk from x0
// (triangles.rs:257-301, the same w += dx additions as the raster's walk)
// storing the weights where the span enters each column; a second table
// keeps a bit per row whose span holds the whole column.  The wave then
// appends the entries of its tiles to their lists, with their key-order
// bounds, and raises the occluder bound of each tile the triangle covers.
// Slots sit at fixed places (layout in internal.hpp), so no block waits for
// another.
// ---------------------------------------------------------------------------

// Key-order bounds of a big triangle over one tile, for the occlusion test
// (write modes).  Every weight the raster computes in the tile comes from the
// walk of its row from x0 (triangles.rs:257-301): the start value and each of
// at most (xmax - xmin) additions round by half an ulp of a partial sum, which
// M bounds (|o| + |dy| y + |dx| x over the triangle's box), so each weight
// stays within err = (xmax - xmin + 8) 2^-23 M of its plane, u2 within the sum
// of those and its two subtractions, and z (three products, two sums) within
// ez of the plane hz . (w0, w1, u2).  The planes are affine, so their extremes
// over the tile's pixels lie at its corners, evaluated in f32 with the
// evaluation's own rounding added to the margins (all terms doubled).
struct TileBounds {
    uint32_t klo;  // key order no fragment of the triangle in the tile goes below
    uint32_t khi;  // key order none goes above (valid where `full`)
    bool full;     // every pixel of the tile is a fragment of the triangle
};

EUCHIP_DEV TileBounds tile_bounds(const FrameParams &p, const TriRec &R, uint32_t mode, uint32_t X0, uint32_t Y0,
                                  uint32_t TW, uint32_t TH) {
    const float Xm = (float)R.xmax + 32.0f, Ym = (float)R.ymax;
    float M[3], e[3];
    const float K = (float)(R.xmax - R.xmin + 8u) * 0x1p-22f;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        M[i] = (fabsf(R.o[i]) + fabsf(R.dy[i]) * Ym + fabsf(R.dx[i]) * Xm) * 1.001f;
        e[i] = K * M[i] + 0x1p-125f;
    }
    const float S = M[0] + M[1] + M[2];
    const float eu = (e[0] + e[1] + e[2]) + 0x1p-21f * S;
    const float h0 = fabsf(R.hz[0]), h1 = fabsf(R.hz[1]), h2 = fabsf(R.hz[2]);
    const float P = h0 * M[0] + h1 * M[1] + h2 * S;
    const float ez = 2.0f * ((h0 * e[0] + h1 * e[1] + h2 * eu) + 0x1p-18f * P) + 0x1p-124f;
    // the corners' weights and z (planes of the reference's setup values)
    const float xs[2] = {(float)X0, (float)(X0 + TW - 1u)}, ys[2] = {(float)Y0, (float)(Y0 + TH - 1u)};
    float zmin = INFINITY, zmax = -INFINITY, wmin[3] = {INFINITY, INFINITY, INFINITY};
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
            float w[3];
#pragma unroll
            for (int i = 0; i < 3; i++) w[i] = (R.o[i] + R.dy[i] * ys[c]) + R.dx[i] * xs[a];
            const float u2 = (w[2] - w[0]) - w[1];
            const float z = (R.hz[0] * w[0] + R.hz[1] * w[1]) + R.hz[2] * u2;
            zmin = fminf(zmin, z), zmax = fmaxf(zmax, z);
            wmin[0] = fminf(wmin[0], w[0]), wmin[1] = fminf(wmin[1], w[1]), wmin[2] = fminf(wmin[2], u2);
        }
    TileBounds b;
    const bool finite = (zmin - zmin == 0.0f) & (zmax - zmax == 0.0f) & (ez - ez == 0.0f);
    const float zlo = zmin - ez, zhi = zmax + ez;
    // order values, as the walk's keys form them (-0 and +0 alike)
    auto ord = [](float z) {
        const uint32_t u = __float_as_uint(z + 0.0f);
        return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
    };
    b.klo = !finite ? 0u : mode == 1u ? ord(zlo) : ~ord(zhi);
    b.khi = mode == 1u ? ord(zhi) : ~ord(zlo);
    const bool clip = !(R.flags & TRI_ALL_IN) && p.z_clip;
    b.full = finite & (wmin[0] > e[0] + 0x1p-21f * M[0]) & (wmin[1] > e[1] + 0x1p-21f * M[1]) &
             (wmin[2] > eu + 0x1p-20f * S) & (!clip | ((p.z_min <= zlo) & (zhi <= p.z_max)));
    return b;
}

EUCHIP_DEV void span_item(const FrameParams &p, uint32_t b, void *static_lds) {
    extern __shared__ uint32_t span_lds[];  // the span tables when the static LDS is too small
    __shared__ TriRec span_tri;              // the block's triangle, set up once by wave 0
    __shared__ uint32_t span_keep;
    const View &v = p.v0;
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t t = b % v.n_tris, part = (b / v.n_tris) * 4u + wv;
    if (wv == 0u) {
        TriRec R0;
        const bool keep = tri_setup(p, v, t, R0);
        if (lane == 0u) span_tri = R0, span_keep = keep ? 1u : 0u;
    }
    __syncthreads();
    if (!span_keep || part >= p.span_parts) return;
    const TriRec R = span_tri;
    const uint32_t sx = p.tile_sx, sy = 8u - sx, TH = 1u << sy, TW = 1u << sx;
    const uint32_t col0 = R.xmin >> sx;
    const uint32_t cols = ((R.xmax - 1u) >> sx) - col0 + 1u;
    if (part == 0u && lane == 0u) {  // what the raster's row tasks read besides the slot
        uint4 *dst = p.big_rec + (size_t)t * kBigRecQuads;
        dst[0] = make_uint4(t, R.flags << 30, __float_as_uint(R.dx[0]), __float_as_uint(R.dx[1]));
        dst[1] = make_uint4(__float_as_uint(R.dx[2]), __float_as_uint(R.hz[0]), __float_as_uint(R.hz[1]),
                            __float_as_uint(R.hz[2]));
    }
    const uint32_t ybase = ((R.ymin >> sy) << sy) + part * kSpanRows;
    if (ybase >= R.ymax) return;
    const uint32_t groups = kSpanRows >> sy, ne = groups * cols;
    // this wave's tables of (tile row, column) bytes: rows reaching into the
    // tile, rows whose span holds all of its columns
    const uint32_t tb = span_table_bytes(sy, v.ntx);
    uint8_t *base = 4u * tb <= sizeof(SetupShared) ? (uint8_t *)static_lds : (uint8_t *)span_lds;
    uint8_t *const tab = base + wv * tb;
    const uint32_t nb = (ne + 3u) & ~3u;
    uint32_t *mw = (uint32_t *)tab, *fw = (uint32_t *)(tab + nb);
    const uint8_t *mb = tab, *fb = tab + nb;
    for (uint32_t i = lane; i < (nb >> 2); i += 64u) mw[i] = 0u, fw[i] = 0u;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint32_t y = ybase + lane;
    uint32_t x0 = 0, x1 = 0;
    if (y >= R.ymin && y < R.ymax) {
        uint32_t by0, by1;
        band_of(p, v, y, by0, by1);
        row_span(R, y, by0, by1, x0, x1);
    }
    if (x0 < x1) {
        const uint32_t at0 = (lane >> sy) * cols - col0, bit = 1u << (y & (TH - 1u));
        for (uint32_t c = x0 >> sx; c <= ((x1 - 1u) >> sx); c++) {
            const uint32_t at = at0 + c, sh = (at & 3u) * 8u;
            atomicOr(&mw[at >> 2], bit << sh);
            if (x0 <= (c << sx) && (c << sx) + TW <= x1) atomicOr(&fw[at >> 2], bit << sh);
        }
        const float Y = (float)y, X0 = (float)x0;
        float w0 = (R.o[0] + R.dy[0] * Y) + R.dx[0] * X0;
        float w1 = (R.o[1] + R.dy[1] * Y) + R.dx[1] * X0;
        float w2 = (R.o[2] + R.dy[2] * Y) + R.dx[2] * X0;
        uint4 *row = p.ck + (size_t)t * v.ntx * v.H + y;  // column c's slot at row + c * H
        for (uint32_t x = x0;;) {
            const uint32_t c = x >> sx, xc = c << sx;
            const uint32_t xe = xc + TW < x1 ? xc + TW : x1;
            row[(size_t)c * v.H] = make_uint4(__float_as_uint(w0), __float_as_uint(w1), __float_as_uint(w2),
                                              (x - xc) | ((xe - xc) << 16));
            if (xe >= x1) break;
            for (; x + 16u <= xe; x += 16u) {
#pragma unroll
                for (uint32_t q = 0; q < 16u; q++) {
                    w0 = w0 + R.dx[0];
                    w1 = w1 + R.dx[1];
                    w2 = w2 + R.dx[2];
                }
            }
            for (; x < xe; x++) {
                w0 = w0 + R.dx[0];
                w1 = w1 + R.dx[1];
                w2 = w2 + R.dx[2];
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // the entries of this item's tiles (every tile row of it is this item's)
    // with their bounds; a tile whose every row's span holds it and whose
    // pixels the triangle covers (tile_bounds) raises its occluder bound.
    // Key order: Less + write takes zord, Greater + write ~zord; other depth
    // modes keep every entry (klo 0) and record no occluder.
    const uint32_t mode = key_mode(p);
    const uint32_t ty0 = ybase >> sy, all_rows = (1u << TH) - 1u;
    for (uint32_t i = lane; i < ne; i += 64u) {
        const uint32_t m = mb[i];
        if (m == 0u) continue;
        const uint32_t gi = i / cols, c = i - gi * cols;
        const size_t tile = (size_t)(ty0 + gi) * v.ntx + col0 + c;
        TileBounds tb{0u, 0u, false};
        if (mode != 0u) tb = tile_bounds(p, R, mode, (col0 + c) << sx, (ty0 + gi) << sy, TW, TH);
        const uint32_t k = atomicAdd(&p.ck_count[tile].x, 1u);  // below mstride: one entry per triangle
        p.cktab[tile * p.mstride + k] = make_uint2((t << 8) | m, tb.klo);
        if (tb.full && fb[i] == all_rows) atomicMax(&p.ck_count[tile].y, ~tb.khi);
    }
}

// Workgroups of a raster launch: one per tile, rounded up to a multiple of the 8
// XCDs, but no more than these; each then takes every n-th tile of its XCD.
// Fewer workgroups start less often (about 1 us of a slot each), more balance
// better.  Measured, us per pass with at most 2048 / 4096 / 8192 / 16384 / any
// number: a 3840x2160 frame (32,400 tiles) 136 / 131 / 126 / 126 / 133, a 2048^2
// depth pass and a 1080p frame 127 / 126 / 124 / 126 / 126, a batch of 111,000 tiles
// 456 / 442 / 430 / 416 / 456, one of 52,000 480 / 455 / 436 / 428 / 416.
constexpr uint32_t kFrameGroups = 8192, kBatchGroups = 16384;
hipError_t launch_raster(const FrameParams &p, hipStream_t s, bool batched) {
    if (p.ntiles == 0) return hipSuccess;
    FrameParams q = p;
    q.heavy_groups = batched ? 0u : heavy_group_count(p.heavy_cap, p.v0.n_tris);
    if (!q.heavy_groups) q.heavy_cap = 0u;  // the busy lists' workgroups take every tile
    const uint32_t g = q.heavy_groups + std::min(batched ? kBatchGroups : kFrameGroups, (uint32_t)(((uint64_t)p.ntiles + 7u) / 8u * 8u));
    switch (p.shader) {
    case FLAT: launch_raster_t<FLAT>(q, s, batched, g); break;
    case COLOR: launch_raster_t<COLOR>(q, s, batched, g); break;
    case GOURAUD: launch_raster_t<GOURAUD>(q, s, batched, g); break;
    case PHONG: launch_raster_t<PHONG>(q, s, batched, g); break;
    case DEPTH_ONLY: launch_raster_t<DEPTH_ONLY>(q, s, batched, g); break;
    case TEXTURED: launch_raster_t<TEXTURED>(q, s, batched, g); break;
    case PHONG_SHADOW: launch_raster_t<PHONG_SHADOW>(q, s, batched, g); break;
    case TEX_SHADOW: launch_raster_t<TEX_SHADOW>(q, s, batched, g); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}


hipError_t launch_tiny(const FrameParams &p, hipStream_t s) {
    if (p.ntiles == 0) return hipSuccess;
    const uint32_t g = std::min(p.ntiles, kTinyGroups);
    switch (p.shader) {
    case FLAT: launch_tiny_t<FLAT>(p, s, g); break;
    case COLOR: launch_tiny_t<COLOR>(p, s, g); break;
    case GOURAUD: launch_tiny_t<GOURAUD>(p, s, g); break;
    case PHONG: launch_tiny_t<PHONG>(p, s, g); break;
    case DEPTH_ONLY: launch_tiny_t<DEPTH_ONLY>(p, s, g); break;
    case TEXTURED: launch_tiny_t<TEXTURED>(p, s, g); break;
    case PHONG_SHADOW: launch_tiny_t<PHONG_SHADOW>(p, s, g); break;
    case TEX_SHADOW: launch_tiny_t<TEX_SHADOW>(p, s, g); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// lines (lines.rs:15-121): one-request frames of LineList / LineTriangleList
// ---------------------------------------------------------------------------

// Clip position and shaded-vertex id of stream element e of request v.
EUCHIP_DEV void element_clip(const FrameParams &p, const View &v, uint32_t e, float c[4], uint32_t &sid) {
    const uint32_t inst = e / v.count;
    uint32_t vi = e - inst * v.count;
    if (v.idx) vi = v.idx[vi];
    const float *P = v.pos + (size_t)v.pos_comps * vi;
    if (p.xform == 0u) {
        c[0] = P[0], c[1] = P[1], c[2] = P[2], c[3] = v.pos_comps == 4u ? P[3] : 1.0f;
    } else {
        const float p4[4] = {P[0], P[1], P[2], 1.0f};
        float w[4];
        mat4_vec4((const float *)v.models + 16u * inst, p4, w);
        mat4_vec4(v.u + U_VP, w, c);
    }
    sid = v.sv_base + inst * v.n_vertices + vi;
}

// `f as isize` clamped to what the record keeps: NaN -> 0, otherwise truncation,
// saturated (coordinates past kLineCoordLimit mark the line undrawn).
EUCHIP_DEV int32_t line_coord(float f, bool &far) {
    if (f != f) return 0;
    if (!(f > -(float)kLineCoordLimit && f < (float)kLineCoordLimit)) {
        far = true;
        return 0;
    }
    return (int32_t)f;
}

// f32::clamp then `as isize` for a bound within [lo, hi] (lo, hi integral, >= 0).
EUCHIP_DEV int32_t clamp_coord(float f, float lo, float hi) {
    if (f < lo) f = lo;
    if (f > hi) f = hi;
    if (f != f) return 0;
    return (int32_t)f;
}

// The Bresenham walk of one line (clipline 0.2's contract: the unclipped line's
// pixels inside the rectangle), clipped to its range of steps along the major axis.
struct LineWalk {
    int32_t M1, m1;      // first end: major and minor coordinate
    uint32_t dM, dm;     // extents
    int32_t sM, sm;      // directions
    int32_t n0, n1;      // clip rectangle along the minor axis
    int32_t klo, khi;    // steps whose major coordinate is inside the rectangle
    bool xmajor, use_x;
    float vs0, norm, ez0, ez1;
};

// Steps k = klo + first, klo + first + stride, ... of line l: each pixel's key is
// raised by its fragment (key 0: no fragment; the greatest key wins).
// LOADS: a depth test reads the target's depth before the pass (not the clear's).
// Kernels of their own: a loop that may load waits in every step for the step
// before's atomic.
template <bool LOADS>
EUCHIP_DEV void walk_line(const FrameParams &p, const View &v, uint32_t l, const LineWalk &W, uint32_t first, uint32_t stride) {
    const uint32_t mode = key_mode(p);
    for (int32_t k = W.klo + (int32_t)first; k <= W.khi; k += (int32_t)stride) {
        // floor((2 k dm + dM - 1) / (2 dM)), in 32 bits where the product fits
        uint32_t j = 0u;
        if (W.dM <= 32767u) j = W.dM ? (2u * (uint32_t)k * W.dm + W.dM - 1u) / (2u * W.dM) : 0u;
        else j = (uint32_t)((2ull * (uint32_t)k * W.dm + W.dM - 1u) / (2ull * W.dM));
        const int32_t M = W.M1 + W.sM * k, m = W.m1 + W.sm * (int32_t)j;
        if (m < W.n0 || m > W.n1) continue;
        const uint32_t x = (uint32_t)(W.xmajor ? M : m), y = (uint32_t)(W.xmajor ? m : M);
        // lines.rs:88-95
        const float frac = (W.use_x ? (float)x - W.vs0 : (float)y - W.vs0) * W.norm;
        const float z = W.ez0 + frac * (W.ez1 - W.ez0);
        if (!passes_z_clip(p, z)) continue;
        const size_t pi = (size_t)y * v.W + x;
        if (p.depth_test != DT_NONE) {
            const float D0 = LOADS ? v.depth[pi] : v.clear_depth;
            if (!passes_depth(p.depth_test, z, D0)) continue;
        }
        // the keys of init_key, those of the write modes complemented
        uint64_t key = ((uint64_t)(l + 1u) << 32) | __float_as_uint(z);
        if (mode != 0u) {
            const uint32_t o = mode == 1u ? zord(z) : ~zord(z), nz = __float_as_uint(z) == 0x80000000u ? 1u : 0u;
            key = ~(((uint64_t)o << 32) | ((l + 1u) << 1) | nz);
        }
        atomicMax((unsigned long long *)&p.lkey[pi], (unsigned long long)key);
    }
}

// k_line_draw: blocks of 256 / LANES lines, then vertex blocks (lane t = shaded
// vertex t).  LANES lanes set a line up (lines.rs:41-86 in f32 over the whole
// target; the band clamp of the clip rectangle only cuts rows other bands draw),
// each for itself, and take its steps k, k + LANES, ...; with 16, lines of more
// than kLongLine pixels are walked by the whole wave, one after the other.  The per-pixel keys are zero
// between frames: the resolve puts back the ones it finds, so no pass initialises
// them.  (A launch for the setup, one for the keys, a wave per line with 64-bit
// divisions and the resolve took 23.5 us for 12,288 lines at 1280x720.)
// Frames of up to kWaveLines lines, whose waves do not fill the chip, give a line
// a whole wave: four long ones in turn are a serial chain, of loads and atomics
// where the depth is read.  16 lanes / a wave, us at 1920x1080: 300 lines of 900
// pixels 32.4 / 18.4, over loaded depth 36.9 / 16.3, 1000 of them 36.6 / 30.5 and
// 39.9 / 18.1; of 30 pixels, 2000 lines 14.2 / 13.8, 8000 20.0 / 20.3, 20,000 32.2 /
// 33.8; of 5 pixels, 1000 lines 11.4 / 11.6, 4000 12.7 / 14.0, 12,000 15.2 / 19.8.
constexpr int32_t kLongLine = 256;
constexpr uint32_t kWaveLines = 2048;

template <uint32_t SH, bool LOADS, uint32_t LANES>
__global__ __launch_bounds__(256) void k_line_draw(FrameParams) {
    warm_args();
    const FrameParams &p = args();
    const View &v = p.v0;
    const uint32_t tid = threadIdx.x;
    if (blockIdx.x >= p.tri_blocks) {
        if constexpr (vd_count(SH) > 0) {
            const uint32_t t = (blockIdx.x - p.tri_blocks) * 256u + tid;
            if (t < v.n_instances * v.n_vertices) {
                const uint32_t inst = divide(t, v.inst_verts);
                float vd[VDN<SH>::N];
                vertex_data<SH>(p, v, inst, t - inst * v.n_vertices, vd);
#pragma unroll
                for (uint32_t q = 0; q < vd_count(SH); q++) p.vary[((size_t)v.sv_base + t) * vd_count(SH) + q] = vd[q];
            }
        }
        return;
    }
    const uint32_t l = p.line_first + blockIdx.x * (256u / LANES) + tid / LANES;
    LineWalk W;
    W.klo = 0, W.khi = -1;
    if (l < p.n_lines) {
        uint32_t e0, e1;
        if (p.primitives == PRIMS_LINE_LIST) {
            e0 = 2u * l, e1 = 2u * l + 1u;
        } else {  // edges a-b, b-c, c-a of stage-output triangle l / 3 (primitives.rs:71-84)
            const uint32_t tri = l / 3u, j = l - 3u * tri;
            e0 = corner_element(p.geometry, tri, (int)j);
            e1 = corner_element(p.geometry, tri, j == 2u ? 0 : (int)j + 1);
        }
        float hom[2][4];
        uint32_t sid[2];
        element_clip(p, v, e0, hom[0], sid[0]);
        element_clip(p, v, e1, hom[1], sid[1]);
        const float flip1 = p.y_up ? -1.0f : 1.0f;
        const float size0 = (float)v.W, size1 = (float)v.H;
        float ez[2], vs[2][2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float x = hom[i][0] * 1.0f, y = hom[i][1] * flip1, z = hom[i][2];
            const float w = rmax(hom[i][3], 0.0001f);
            const float ex = x / w, ey = y / w;
            ez[i] = z / w;
            vs[i][0] = size0 * (ex * 0.5f + 0.5f);
            vs[i][1] = size1 * (ey * -0.5f + 0.5f);
        }
        bool far = false;
        const int32_t x1 = line_coord(vs[0][0], far), y1 = line_coord(vs[0][1], far);
        const int32_t x2 = line_coord(vs[1][0], far), y2 = line_coord(vs[1][1], far);
        const int32_t cx0 = clamp_coord(rmin(vs[0][0], vs[1][0]) + 0.0f, 0.0f, size0);
        const int32_t cy0 = clamp_coord(rmin(vs[0][1], vs[1][1]) + 0.0f, 0.0f, size1);
        const int32_t cx1 = clamp_coord(rmax(vs[0][0], vs[1][0]) + 1.0f, 0.0f, size0) - 1;
        const int32_t cy1 = clamp_coord(rmax(vs[0][1], vs[1][1]) + 1.0f, 0.0f, size1) - 1;
        const uint32_t adx = x1 > x2 ? x1 - x2 : x2 - x1, ady = y1 > y2 ? y1 - y2 : y2 - y1;
        W.use_x = adx > ady, W.xmajor = adx >= ady;
        W.norm = 1.0f / (W.use_x ? vs[1][0] - vs[0][0] : vs[1][1] - vs[0][1]);
        W.vs0 = W.use_x ? vs[0][0] : vs[0][1];
        W.ez0 = ez[0], W.ez1 = ez[1];
        W.M1 = W.xmajor ? x1 : y1, W.m1 = W.xmajor ? y1 : x1;
        W.dM = W.xmajor ? adx : ady, W.dm = W.xmajor ? ady : adx;
        W.sM = (W.xmajor ? x2 < x1 : y2 < y1) ? -1 : 1, W.sm = (W.xmajor ? y2 < y1 : x2 < x1) ? -1 : 1;
        const int32_t c0 = W.xmajor ? cx0 : cy0, c1 = W.xmajor ? cx1 : cy1;
        W.n0 = W.xmajor ? cy0 : cx0, W.n1 = W.xmajor ? cy1 : cx1;
        const int32_t klo = W.sM > 0 ? c0 - W.M1 : W.M1 - c1, khi = W.sM > 0 ? c1 - W.M1 : W.M1 - c0;
        if (!far && cx1 >= cx0 && cy1 >= cy0) {  // (far: an endpoint past the coordinate limit)
            W.klo = klo < 0 ? 0 : klo;
            W.khi = khi > (int32_t)W.dM ? (int32_t)W.dM : khi;
        }
        if (tid % LANES == 0u) {  // what the resolve reads of the line
            uint4 *rq = p.lrec + (size_t)l * kLineRecQuads;
            rq[0] = make_uint4(__float_as_uint(W.vs0), __float_as_uint(W.norm), sid[0], sid[1]);
            rq[1] = make_uint4(W.use_x ? 1u : 0u, 0u, 0u, 0u);
        }
    }
    if constexpr (LANES == 64u) {
        walk_line<LOADS>(p, v, l, W, lane_id(), 64u);
        return;
    }
    const bool wide = W.khi - W.klo >= kLongLine;
    if (!wide) walk_line<LOADS>(p, v, l, W, tid & 15u, 16u);
    for (uint64_t m = __ballot(wide) & 0x0001000100010001ull; m; m &= m - 1u) {
        const int g = __ffsll((unsigned long long)m) - 1;  // the line's first lane
        auto bi = [&](int32_t q) { return __builtin_amdgcn_readlane(q, g); };
        auto bu = [&](uint32_t q) { return (uint32_t)__builtin_amdgcn_readlane((int)q, g); };
        auto bf = [&](float q) { return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(q), g)); };
        LineWalk B;
        B.M1 = bi(W.M1), B.m1 = bi(W.m1), B.dM = bu(W.dM), B.dm = bu(W.dm), B.sM = bi(W.sM), B.sm = bi(W.sm);
        B.n0 = bi(W.n0), B.n1 = bi(W.n1), B.klo = bi(W.klo), B.khi = bi(W.khi);
        B.xmajor = bu(W.xmajor) != 0u, B.use_x = bu(W.use_x) != 0u;
        B.vs0 = bf(W.vs0), B.norm = bf(W.norm), B.ez0 = bf(W.ez0), B.ez1 = bf(W.ez1);
        walk_line<LOADS>(p, v, bu(l), B, lane_id(), 64u);
    }
}

// get_v_data of a line (lines.rs:99-112): weighted_sum2(v0, v1, 1 - frac, frac).
template <uint32_t SH>
EUCHIP_DEV void v_data_line(const float (*V)[VDN<SH>::N], bool use_x, float vs0, float norm, float X, float Y,
                            float *vd) {
    const float frac = (use_x ? X - vs0 : Y - vs0) * norm;
    const float w0 = 1.0f - frac;
    if constexpr (SH == FLAT) {
        vd[0] = V[0][0];
    } else {
#pragma unroll
        for (uint32_t c = 0; c < vd_count(SH); c++) vd[c] = V[0][c] * w0 + V[1][c] * frac;
    }
}

// k_line_resolve: every pixel of the target: the winning line's fragment (shaded
// once, with the coarse-shading combine under MSAA), its depth, or the clears; a
// key found set is zeroed for the next frame.
template <uint32_t SH>
__global__ __launch_bounds__(256) void k_line_resolve(FrameParams) {
    const FrameParams &p = args();
    const View &v = p.v0;
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= (uint64_t)v.W * v.H) return;
    const uint32_t mode = key_mode(p);
    uint64_t kk = p.lkey[i];
    const bool has = kk != 0ull;
    if (has) p.lkey[i] = 0ull;
    if (mode != 0u) kk = ~kk;
    const uint32_t prim = key_prim(mode, kk) - 1u;
    float z = __uint_as_float((uint32_t)kk);
    if (mode != 0u) {
        const uint32_t o = (uint32_t)(kk >> 32);
        z = zunord(mode == 1u ? o : ~o, (uint32_t)kk & 1u);
    }
    if (v.pixel) {
        if (p.pixel_write && has && SH != DEPTH_ONLY) {
            const uint32_t py = divide(i, v.row_pixels), px = i - py * v.W;
            const uint4 *rq = p.lrec + (size_t)prim * kLineRecQuads;
            const uint4 q0 = rq[0];
            const float vs0 = __uint_as_float(q0.x), norm = __uint_as_float(q0.y);
            const bool use_x = rq[1].x & 1u;
            constexpr uint32_t NV = VDN<SH>::N;
            float V[2][NV];
            const uint32_t sid[2] = {q0.z, q0.w};
#pragma unroll
            for (int k = 0; k < 2; k++)
#pragma unroll
                for (uint32_t c = 0; c < vd_count(SH); c++) V[k][c] = p.vary[(size_t)sid[k] * vd_count(SH) + c];
            if constexpr (vd_count(SH) == 0) V[0][0] = V[1][0] = 0.0f;
            float frag[4], vd[NV];
            const uint32_t L = p.msaa_level;
            if (L == 0u) {
                v_data_line<SH>(V, use_x, vs0, norm, (float)px, (float)py, vd);
                fragment_shader<SH, true>(v, p.sampler, vd, frag);
            } else {
                uint32_t by0, by1;
                band_of(p, v, py, by0, by1);
                const float div = 1.0f / (float)(1u << L);
                const uint32_t rx = px, ry = py - by0;
                const float fx = rfract((float)rx * div);
                const float fy = rfract((float)ry * div);
                const uint32_t cx = rx >> L, cy = ry >> L;
                float t[4][4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint32_t ix = cx + (uint32_t)(q & 1), iy = cy + (uint32_t)(q >> 1);
                    v_data_line<SH>(V, use_x, vs0, norm, (float)(ix << L), (float)(by0 + (iy << L)), vd);
                    fragment_shader<SH, true>(v, p.sampler, vd, t[q]);
                }
                if constexpr (SH == FLAT) {
                    frag[0] = t[0][0];
                } else {
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const float t0 = t[0][c] * (1.0f - fy) + t[2][c] * fy;
                        const float t1 = t[1][c] * (1.0f - fy) + t[3][c] * fy;
                        frag[c] = t0 * (1.0f - fx) + t1 * fx;
                    }
                }
            }
            v.pixel[i] = blend_shader<SH>(v.clear_color_en ? v.clear_color : v.pixel[i], frag, p.bgra);
        } else if (v.clear_color_en) {
            v.pixel[i] = v.clear_color;
        }
    }
    if (v.depth) {
        if (has && p.depth_write) v.depth[i] = z;
        else if (v.clear_depth_en) v.depth[i] = v.clear_depth;
    }
}

template <uint32_t SH>
static void launch_lines_t(const FrameParams &p, hipStream_t s) {
    const size_t nsv = (size_t)p.v0.n_instances * p.v0.n_vertices;
    const size_t npx = (size_t)p.v0.W * p.v0.H;
    const bool waves = p.n_lines <= kWaveLines, loads = p.depth_test != DT_NONE && !p.v0.clear_depth_en;
    auto draw = [&](const LineLaunch &l) {
        FrameParams q = p;
        q.line_first = l.first;
        q.tri_blocks = l.line_groups;
        const dim3 blocks(l.line_groups + l.vertex_groups);
        if (loads && waves) hipLaunchKernelGGL((k_line_draw<SH, true, 64>), blocks, dim3(256), 0, s, q);
        else if (loads) hipLaunchKernelGGL((k_line_draw<SH, true, 16>), blocks, dim3(256), 0, s, q);
        else if (waves) hipLaunchKernelGGL((k_line_draw<SH, false, 64>), blocks, dim3(256), 0, s, q);
        else hipLaunchKernelGGL((k_line_draw<SH, false, 16>), blocks, dim3(256), 0, s, q);
    };
    line_launches(p.n_lines, vd_count(SH) > 0 ? nsv : 0u, draw, waves ? 4u : kLinesPerBlock);
    hipLaunchKernelGGL((k_line_resolve<SH>), dim3(blocks_of(npx, 256)), dim3(256), 0, s, p);
}

hipError_t launch_lines(const FrameParams &p, hipStream_t s) {
    if ((size_t)p.v0.W * p.v0.H == 0) return hipSuccess;
    switch (p.shader) {
    case FLAT: launch_lines_t<FLAT>(p, s); break;
    case COLOR: launch_lines_t<COLOR>(p, s); break;
    case GOURAUD: launch_lines_t<GOURAUD>(p, s); break;
    case PHONG: launch_lines_t<PHONG>(p, s); break;
    case DEPTH_ONLY: launch_lines_t<DEPTH_ONLY>(p, s); break;
    case TEXTURED: launch_lines_t<TEXTURED>(p, s); break;
    case PHONG_SHADOW: launch_lines_t<PHONG_SHADOW>(p, s); break;
    case TEX_SHADOW: launch_lines_t<TEX_SHADOW>(p, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t *dst, uint32_t value, size_t n, hipStream_t s) {
    while (n) {
        const uint32_t groups = launch_groups(n, 256u);
        const size_t part = std::min<size_t>(n, (size_t)groups * 256u);
        hipLaunchKernelGGL(k_fill_u32, dim3(groups), dim3(256), 0, s, dst, value, part);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        dst += part, n -= part;
    }
    return hipSuccess;
}

}  // namespace euchip
