// The inference render (the reference's `benchmark` kernel,
// src/tracing/pipeline.cu:1067-1199) for gfx950.
#include "trace_kernels.h"
#include "trace_split.h"

namespace sdfoam_hip {

namespace {

// One lane (G == 1) or G lanes per pixel, 16x16 pixel tiles as the traced
// kernels.  The step is the forward's compositing without its per-point
// outputs.  CT: the walk reads a cell table and a padded copy of the caller's
// offset table that names each face's neighbour, made for the frame
// (scene_prep_kernel); else the caller's arrays, its unpadded table with
// guarded loads.
template <int L, bool NEUS, typename AT, int G, bool CT>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(CT && G == 1 ? 6 : 1))) void
render_kernel(RenderArgs a) {
    static_assert(G == 1 || CT, "lanes share a pixel over the cell table only");
    constexpr uint32_t RB = CT ? cell_record_bytes(L, sizeof(AT)) : 0u;
    constexpr int nsh = (L + 1) * (L + 1);
    constexpr int D = 1 + 3 * nsh;
    constexpr int U = G == 1 ? 1 : G >= 8 ? 32 / G : 4;
    // with four lanes or more, three of them form one colour channel each
    constexpr bool kByChannel = G >= 4;
    const uint32_t lane = threadIdx.x & 63u, sub = lane % G;
    bool valid;
    uint32_t px;
    if constexpr (G == 1) {
        px = ray_for_lane<kForwardChunk>(a.width * a.height, a.width, a.num_tiles, valid);
    } else {
        const uint32_t wv = split_wave<G>(blockIdx.x) + (threadIdx.x >> 6);
        px = ray_at(wv / G, split_position<G>(wv % G, lane / G, true), a.width * a.height, a.width,
                    a.num_tiles, valid, nullptr);
    }
    const uint32_t pi = valid ? px % a.width : 0u, pj = valid ? px / a.width : 0u;

    RayF ray = {};
    bool masked = false;
    if (valid) {
        float dir[3];
        sdf_cast_ray(a.forward, a.right, a.up, a.fov, a.focal, a.width, a.height, a.model, pi,
                     pj, dir);
        const float n = sqrtf(sdf_dot3(dir[0], dir[1], dir[2], dir[0], dir[1], dir[2]));
        masked = n < 0.1f;
        ray.ox = a.position[0];
        ray.oy = a.position[1];
        ray.oz = a.position[2];
        if (!masked) {
            // ray.direction /= ray.direction.norm()
            ray.dx = dir[0] / n;
            ray.dy = dir[1] / n;
            ray.dz = dir[2] / n;
        }
    }
    float sh[nsh];
    sh_basis<L>(ray.dx, ray.dy, ray.dz, sh);
    const uint32_t ch = sub % 4u < 2u ? sub % 4u : 2u;
    const float sha = a.sharpness[0];
    const int32_t sdf_ch = a.settings.sdf_channel;
    const bool neus_alpha = NEUS && sdf_ch >= 0;
    const float thr = a.settings.weight_threshold;

    float T = 1.0f;
    float C0 = 0.0f, C1 = 0.0f, C2 = 0.0f; // by channel: C0 alone
    WalkState ws;
    walk_init<RB>(a.scene, (valid && !masked) ? a.start[0] : kNoIndex, ws);
    WalkCounters wc = {0u, 0u, 0ull, 0ull};

    while (__ballot(ws.alive) != 0ull) {
        StepInfo si;
        si.stepped = false;
        si.found = false;
        float rowv[kByChannel ? nsh : 1];
        float s = 0.0f, chan = 0.0f;
        const AT *__restrict__ row = nullptr;
        if (ws.alive) {
            row = CT ? reinterpret_cast<const AT *>(reinterpret_cast<const char *>(a.scene.cells) +
                                                    (uint64_t)ws.cell * RB + kCellAttrByte)
                     : static_cast<const AT *>(a.scene.attrs) + (uint64_t)ws.cell * D;
            if constexpr (G == 1) {
                walk_advance<true, false, !CT, false, RB>(a.scene, ray, a.settings.max_intersections,
                                                          ws, si, wc);
            } else {
                // the faces' first batch, then the cell's row, all in flight at once
                uint2 h[U];
#pragma unroll
                for (int u = 0; u < U; ++u) h[u] = make_uint2(0u, 0u);
                if (ws.beg < ws.end && ws.end <= a.scene.num_adj) {
#pragma unroll
                    for (int u = 0; u < U; ++u) h[u] = a.scene.diff[ws.beg + u * G + sub];
                }
                s = (float)row[D - 1];
                chan = neus_alpha ? (float)row[sdf_ch] : s;
                if constexpr (kByChannel) {
#pragma unroll
                    for (int j = 0; j < nsh; ++j) rowv[j] = (float)row[3 * j + ch];
                }
                walk_advance_split<G, U, false, RB>(a.scene, ray, a.settings.max_intersections, sub,
                                                    h, ws, si);
            }
        }
        bool keep = true;
        if (si.stepped) {
            if constexpr (G == 1) {
                s = (float)row[D - 1];
                if (neus_alpha) chan = (float)row[sdf_ch];
            }
            const bool dense = NEUS || s > 1e-6f;
            const float dt = fmaxf(si.t1 - ws.t0, 0.0f);
            if (neus_alpha) {
                const float phi = sdf_sigmoidf(-sha * chan);
                s = sha * phi * (1.0f - phi);
            }
            const float alpha = 1.0f - sdf_expf(-s * dt);
            const float w = T * alpha;
            if constexpr (kByChannel) {
                // sh_rgb_regs' sum for one channel
                float v = 0.5f;
#pragma unroll
                for (int j = 0; j < nsh; ++j) v = fmaf(sh[j], rowv[j], v);
                C0 = fmaf(w, dense ? fmaxf(v, 0.0f) : 0.0f, C0);
            } else {
                float r, g, b;
                if (dense) {
                    sh_rgb_regs<L>(sh, row, r, g, b);
                } else {
                    r = g = b = 0.0f;
                }
                C0 = fmaf(w, r, C0);
                C1 = fmaf(w, g, C1);
                C2 = fmaf(w, b, C2);
            }
            T = T * (1.0f - alpha);
            keep = T > thr;
        }
        if (si.stepped && !keep) ws.alive = false;
        if (ws.alive && si.found) walk_move(ws, si);
    }

    if constexpr (kByChannel) {
        // lanes 1 and 2 of the pixel hold the other channels (all lanes active)
        C1 = __shfl_down(C0, 1, 64);
        C2 = __shfl_down(C0, 2, 64);
    }
    if (!valid || sub != 0) return;
    const uint64_t out_idx = (uint64_t)(a.height - 1u - pj) * a.width + pi;
    if (masked) {
        a.out[out_idx] = sdf_make_rgba8(a.bg[0], a.bg[1], a.bg[2], 1.0f);
        return;
    }
    float bg0 = a.bg[0], bg1 = a.bg[1], bg2 = a.bg[2];
    if (a.checker_bg) {
        const int is = 2 * (int)((pi / 20u) % 2u) - 1;
        const int js = 2 * (int)((pj / 20u) % 2u) - 1;
        bg0 = bg1 = bg2 = (is * js > 0) ? 0.3f : 0.5f;
    }
    a.out[out_idx] = sdf_make_rgba8(fmaf(T, bg0, C0), fmaf(T, bg1, C1), fmaf(T, bg2, C2), 1.0f);
}

} // namespace

// Lanes per pixel: more where few pixels leave the chip idle.  ms with 1, 2, 4, 8
// and 16 lanes (walk and tables; in brackets over the caller's arrays), fp32, SH degree 3:
//   4,096 / 300k points  1.13  0.70  0.43  0.33  0.30  (1.11)
//   77k / 100k           0.94  0.62  0.42  0.40  0.48  (0.91)
//   307k / 300k          1.33  1.40  1.08              (1.29)
//   481k / 1M            3.35  2.97  2.49              (3.40)
//   750k / 1M            4.25  3.93  3.45              (4.36), another scene 3.93 4.74 4.68 (4.50)
//   1.09M / 1M           4.60  4.77  4.57              (4.92), another scene 5.16 6.32 6.36 (5.53)
//   250k / 30k           0.76  0.61  0.48              (0.81)
static int render_lanes(uint32_t pixels, uint32_t num_points) {
    if (pixels < 2ull * num_points) {
        if (pixels <= 16384u) return 16;
        if (pixels <= 49152u) return 8;
        if (pixels <= 400000u) return 4;
        return pixels <= 800000u ? 2 : 1;
    }
    if (pixels <= 8192u) return 8;
    if (pixels <= 65536u) return 4;
    return pixels <= 163840u ? 2 : 1;
}

template <int L, typename AT, int G, bool CT>
static hipError_t launch_render_G(const RenderArgs &a, bool neus, hipStream_t stream) {
    const dim3 grid(grid_blocks_for_tiles(a.num_tiles) * G);
    if (neus) {
        hipLaunchKernelGGL((render_kernel<L, true, AT, G, CT>), grid, dim3(kBlock), 0, stream, a);
    } else {
        hipLaunchKernelGGL((render_kernel<L, false, AT, G, CT>), grid, dim3(kBlock), 0, stream, a);
    }
    return hipGetLastError();
}

template <int L, typename AT>
static hipError_t launch_render_L(const RenderArgs &a, bool neus, hipStream_t stream) {
    if (!a.scene.cells) return launch_render_G<L, AT, 1, false>(a, neus, stream);
    switch (render_lanes(a.width * a.height, a.scene.num_points)) {
    case 16: return launch_render_G<L, AT, 16, true>(a, neus, stream);
    case 8: return launch_render_G<L, AT, 8, true>(a, neus, stream);
    case 4: return launch_render_G<L, AT, 4, true>(a, neus, stream);
    case 2: return launch_render_G<L, AT, 2, true>(a, neus, stream);
    default: return launch_render_G<L, AT, 1, true>(a, neus, stream);
    }
}

template <typename AT>
static hipError_t launch_render_T(int L, const RenderArgs &a, bool neus, hipStream_t stream) {
    switch (L) {
    case 0: return launch_render_L<0, AT>(a, neus, stream);
    case 1: return launch_render_L<1, AT>(a, neus, stream);
    case 2: return launch_render_L<2, AT>(a, neus, stream);
    case 3: return launch_render_L<3, AT>(a, neus, stream);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_render(int L, const RenderArgs &a, bool neus, bool half, hipStream_t stream) {
    return half ? launch_render_T<_Float16>(L, a, neus, stream)
                : launch_render_T<float>(L, a, neus, stream);
}

} // namespace sdfoam_hip
