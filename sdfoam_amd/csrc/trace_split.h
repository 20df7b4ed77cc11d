// Walks in which G neighbouring lanes share a ray (the forward, the backward's
// lane assignment, the inference render).
#pragma once

#include "trace_kernels.h"

namespace sdfoam_hip {

__device__ __forceinline__ uint32_t split_xor(uint32_t v, int step) {
    // partner of each doubling step: lane ^ 1, lane ^ 2, then the mirror of
    // 8 and of 16 lanes (groups of 4 and 8 hold one value by then)
    switch (step) {
    case 0: return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xb1, 0xf, 0xf, false);
    case 1: return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4e, 0xf, 0xf, false);
    case 2: return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x141, 0xf, 0xf, false);
    default: return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x140, 0xf, 0xf, false);
    }
}

// Position of ray r of wavefront w (of G) in its row of 64: for image rays a
// compact part of the 8x8 tile, else consecutive.
template <int G>
__device__ __forceinline__ uint32_t split_position(uint32_t w, uint32_t r, bool image) {
    if (!image) return w * (64u / G) + r;
    if constexpr (G == 2) {
        return w * 32u + r; // 8x4
    } else if constexpr (G == 4) {
        return ((w >> 1) * 4u + (r >> 2)) * 8u + (w & 1u) * 4u + (r & 3u); // 4x4
    } else if constexpr (G == 8) {
        return ((w >> 1) * 2u + (r >> 2)) * 8u + (w & 1u) * 4u + (r & 3u); // 4x2
    } else {
        return ((w >> 2) * 2u + (r >> 1)) * 8u + (w & 3u) * 2u + (r & 1u); // 2x2
    }
}

// The row of 64 rays that block b of a split launch (of 4 * grid_blocks_for_
// tiles blocks) takes: tiles go round robin over the XCDs, a tile's four rows
// to the same one.
__device__ __forceinline__ uint32_t split_row(uint32_t b) {
    const uint32_t x = b % kXcds, k = b / kXcds;
    return ((k / 4u) * kXcds + x) * 4u + k % 4u;
}

// ray at position l of row `row` (rows of ray_for_lane's wavefronts)
__device__ __forceinline__ uint32_t ray_at(uint32_t row, uint32_t l, uint32_t num_rays,
                                           uint32_t width, uint32_t num_tiles, bool &valid,
                                           const uint32_t *__restrict__ order) {
    const uint32_t t = row / 4u, w = row % 4u;
    valid = false;
    if (t >= num_tiles) return 0u;
    if (width == 0 || order) {
        const uint32_t i = row * 64u + l;
        const uint32_t r = i < num_rays ? (order ? order[i] : i) : num_rays;
        valid = r < num_rays;
        return valid ? r : 0u;
    }
    const uint32_t height = num_rays / width;
    const uint32_t tiles_x = (width + kTile - 1) / kTile;
    const uint32_t x = (t % tiles_x) * kTile + (w & 1u) * 8u + (l & 7u);
    const uint32_t y = (t / tiles_x) * kTile + (w >> 1) * 8u + (l >> 3);
    valid = x < width && y < height;
    return valid ? y * width + x : 0u;
}

// walk_advance<true, ...> over the cell table by the G lanes of a ray (all of
// them active; the results are the same in each).  h: the lane's entries of
// the first batch, loaded by the caller.
template <int G, int U, bool DUAL, uint32_t RB>
__device__ __forceinline__ void walk_advance_split(const SceneView &sc, const RayF &ray,
                                                   uint32_t max_steps, uint32_t sub, uint2 *h,
                                                   WalkState &ws, StepInfo &si) {
    static_assert(G * U <= (int)kDiffPad, "a batch may over-read the table by its padding");
    si.found = false;
    si.agrees = true;
    si.stepped = false;
    si.t1 = ws.t0; // (no exit: what the walk record keeps beside its end mark)
    ++ws.n;
    if (ws.n > max_steps || ws.beg > ws.end || ws.end > sc.num_adj) {
        ws.alive = false;
        return;
    }
    const uint32_t nf = ws.end - ws.beg;
    const float t0 = ws.t0;
    float t1 = __builtin_bit_cast(float, 0x7f800000u);
    float tmin_u = t1;
    bool below = false;
    uint32_t best = kNoIndex, bw = kDeltaNone;
    float t1m = t1;
    const float t0m = t0 * (1.0f - 0x1p-21f);
    const float t0p = t0 * (1.0f + 0x1p-21f);
    const uint2 *__restrict__ row = sc.diff + ws.beg;
    for (uint32_t k0 = 0; k0 < nf; k0 += G * U) {
        if (k0 != 0) {
#pragma unroll
            for (int u = 0; u < U; ++u) h[u] = row[k0 + u * G + sub];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t k = k0 + u * G + sub;
            const float dx = f16_to_f32(h[u].x);
            const float dy = f16_to_f32(h[u].x >> 16);
            const float dz = f16_to_f32(h[u].y);
            const float fx = fmaf(dx, 0.5f, ws.xc[0]);
            const float fy = fmaf(dy, 0.5f, ws.xc[1]);
            const float fz = fmaf(dz, 0.5f, ws.xc[2]);
            const float dp = sdf_dot3(dx, dy, dz, ray.dx, ray.dy, ray.dz);
            const float num = sdf_dot3(fx - ray.ox, fy - ray.oy, fz - ray.oz, dx, dy, dz);
            const bool pos = dp > 0.0f && k < nf;
            // the division filter of walk_advance
            const float lo = fmaf(t0m, dp, -0x1p-126f);
            bool maybe = pos && num < fmaf(t1m, dp, 0x1p-126f) && num > lo;
            if constexpr (DUAL) {
                below = below || (pos && num < lo);
                maybe = maybe || (pos && num >= lo && num <= fmaf(t0p, dp, 0x1p-126f));
            }
            if (maybe) {
                const float t = num / dp;
                if (t > t0 && t < t1) {
                    t1 = t;
                    t1m = fmaf(fabsf(t), 0x1p-21f, t);
                    best = k;
                    bw = h[u].y >> 16;
                }
                if constexpr (DUAL) tmin_u = fminf(tmin_u, t);
            }
        }
    }
    // the first minimum in row order: the smallest t, then the smallest k
    uint32_t bl = below ? 1u : 0u;
#pragma unroll
    for (int s = 0; (1 << s) < G; ++s) {
        const float ot = __builtin_bit_cast(float, split_xor(__builtin_bit_cast(uint32_t, t1), s));
        const uint32_t ob = split_xor(best, s), ow = split_xor(bw, s);
        const bool take = ot < t1 || (ot == t1 && ob < best);
        t1 = take ? ot : t1;
        best = take ? ob : best;
        bw = take ? ow : bw;
        if constexpr (DUAL) {
            bl |= split_xor(bl, s);
            tmin_u = fminf(tmin_u, __builtin_bit_cast(float, split_xor(
                                       __builtin_bit_cast(uint32_t, tmin_u), s)));
        }
    }
    if constexpr (DUAL) si.agrees = !(bl != 0u || tmin_u <= t0);
    if (best == kNoIndex) {
        ws.alive = false;
        return;
    }
    const uint32_t next = bw != kDeltaNone
                              ? (uint32_t)((int32_t)ws.cell + (int32_t)(int16_t)(uint16_t)bw)
                              : sc.adj[ws.beg + best];
    if (next >= sc.num_points) {
        ws.alive = false;
        return;
    }
    si.found = true;
    si.next = next;
    si.t1 = t1;
    load_cell<RB>(sc, next, si.xn, si.beg, si.end);
    si.stepped = t1 > t0;
}

// First wavefront of block b: tiles (4 G wavefronts, G blocks) go round robin
// over the XCDs.
template <int G>
__device__ __forceinline__ uint32_t split_wave(uint32_t b) {
    const uint32_t x = b % kXcds, k = b / kXcds;
    return (((k / G) * kXcds + x) * G + k % G) * 4u;
}

} // namespace sdfoam_hip
