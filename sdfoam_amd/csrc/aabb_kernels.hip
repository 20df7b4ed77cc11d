// Start-cell lookup: implicit AABB tree over point pairs and an exact
// nearest-neighbour search, for gfx950.
//
// Tree layout (src/aabb_tree/aabb_tree.cuh:35-43): with td = log2(pow2(N)),
// the node (depth d, index i) is box number 2^td - 2^(d+1) + i of a
// [pow2(N), 2, 3] array (min xyz, max xyz); the leaves (depth td-1) bound
// consecutive point pairs, the last point repeated as padding.
//
// The search gives one wave64 to a query.  The wave tests a group of up to
// 64 sibling nodes per step (one per lane), six tree levels apart (depths 6,
// 12, 18, ...), and descends depth first: at each level the children are
// taken in the order of their lower bounds, so the first leaf visit already
// gives a tight bound, and every node whose lower bound exceeds the best
// distance is skipped.  The top two group levels (depth 6: 64 boxes, depth 12:
// 4,096 boxes) are copied into LDS once per block, so a search reads global
// memory only below depth 12.  The fp32 box distance is a lower bound of the
// fp32 point distance (rounding is monotone), so the result is the exact fp32
// nearest neighbour; ties go to the smallest index.
#include "trace_kernels.h"

#include <algorithm>

namespace sdfoam_hip {

__device__ __forceinline__ uint32_t ilog2_u32(uint32_t x) { return x ? 31u - __clz(x) : 0u; }

__device__ __host__ inline uint32_t pow2_up(uint32_t x) {
    if (x <= 1) return 1;
    uint32_t r = 1;
    while (r < x) r <<= 1;
    return r;
}

struct Box {
    float v[6]; // min x, y, z, max x, y, z
};

__device__ __forceinline__ Box join(const Box &a, const Box &b) {
    Box r;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        r.v[c] = fminf(a.v[c], b.v[c]);
        r.v[3 + c] = fmaxf(a.v[3 + c], b.v[3 + c]);
    }
    return r;
}

__device__ __forceinline__ void store_box(float *__restrict__ tree, uint64_t node, const Box &b) {
#pragma unroll
    for (int c = 0; c < 6; ++c) tree[6ull * node + c] = b.v[c];
}

// Eleven tree levels per launch.  A block takes kBuildNodes consecutive nodes
// of the level that starts at node `start` and is `width` nodes wide (a power
// of two): with LEAVES it makes them from point pairs (src/aabb_tree/
// aabb_tree.cu:192-221), else it reads them; each thread joins four of them in
// registers and the block's 256 results go up eight more levels through LDS
// (src/aabb_tree/aabb_tree.cu:254-292, the same pairs).  One launch per level,
// before, was bound by the launches: 20 of them at 1M points, 55 us of GPU
// time and ~100 us of host time, against two launches and 19.5 us.
constexpr uint32_t kBuildNodes = 4 * kBlock;

template <bool LEAVES>
__global__ __launch_bounds__(kBlock) void build_levels_kernel(const float *__restrict__ points,
                                                              uint32_t num_points,
                                                              float *__restrict__ tree,
                                                              uint64_t start, uint32_t width) {
    __shared__ float up[6][kBlock];
    const uint32_t t = threadIdx.x;
    const uint64_t first = (uint64_t)blockIdx.x * kBuildNodes + 4u * t; // of the level
    if (LEAVES && blockIdx.x == 0 && t == 0) {
        // the unused last entry of the [pow2(N), 2, 3] array
        const Box zero = {{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f}};
        store_box(tree, 2ull * width - 1, zero);
    }
    Box n[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const uint64_t i = first + k;
        if (i >= width) break;
        if constexpr (LEAVES) {
            // the last point repeated as padding
            const uint64_t p = 2ull * i;
            const float *a = points + 3ull * (p < num_points ? p : num_points - 1u);
            const float *b = p + 1 < num_points ? points + 3ull * (p + 1) : a;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                n[k].v[c] = fminf(a[c], b[c]);
                n[k].v[3 + c] = fmaxf(a[c], b[c]);
            }
            store_box(tree, i, n[k]);
        } else {
#pragma unroll
            for (int c = 0; c < 6; ++c) n[k].v[c] = tree[6ull * (start + i) + c];
        }
    }
    // two levels in registers (a level of width w has w / 2 parents)
    uint64_t at = start + width;
    uint32_t w = width / 2;
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
        n[k] = join(n[2 * k], n[2 * k + 1]);
        if (first / 2 + k < w) store_box(tree, at + first / 2 + k, n[k]);
    }
    at += w;
    w /= 2;
    n[0] = join(n[0], n[1]);
    if (first / 4 < w) store_box(tree, at + first / 4, n[0]);
#pragma unroll
    for (int c = 0; c < 6; ++c) up[c][t] = n[0].v[c];
    // eight more through LDS: thread t < live joins entries 2 t, 2 t + 1
    for (uint32_t live = kBlock / 2; live >= 1; live /= 2) {
        at += w;
        w /= 2;
        if (w == 0) break; // the whole grid: the root is done
        __syncthreads();
        Box r;
        if (t < live) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                r.v[c] = fminf(up[c][2 * t], up[c][2 * t + 1]);
                r.v[3 + c] = fmaxf(up[3 + c][2 * t], up[3 + c][2 * t + 1]);
            }
            const uint64_t i = (uint64_t)blockIdx.x * live + t;
            if (i < w) store_box(tree, at + i, r);
        }
        __syncthreads();
        if (t < live) {
#pragma unroll
            for (int c = 0; c < 6; ++c) up[c][t] = r.v[c];
        }
    }
}

hipError_t launch_build_aabb_tree(const float *points, uint32_t num_points, float *tree,
                                  hipStream_t stream) {
    uint32_t width = pow2_up(num_points) / 2;
    if (width == 0) return hipSuccess;
    auto grid = [](uint32_t w) { return dim3((w + kBuildNodes - 1) / kBuildNodes); };
    hipLaunchKernelGGL(build_levels_kernel<true>, grid(width), dim3(kBlock), 0, stream, points,
                       num_points, tree, 0ull, width);
    uint64_t start = 0;
    while (width > kBuildNodes) {
        // the launch before ended with one node per block
        for (uint32_t k = kBuildNodes; k > 1; k /= 2) {
            start += width;
            width /= 2;
        }
        hipLaunchKernelGGL(build_levels_kernel<false>, grid(width), dim3(kBlock), 0, stream,
                           points, num_points, tree, start, width);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------

// Blocks of 16 waves share one copy of the top levels (1 block per CU).
constexpr int kNNBlock = 1024;
constexpr int kNNWaves = kNNBlock / 64;
constexpr uint32_t kNNTopA = 64;           // boxes at depth 6
constexpr uint32_t kNNTopB = 4096;         // boxes at depth 12
constexpr uint32_t kNNTop = kNNTopA + kNNTopB;
// Group levels of a descent: depths 6, 12, ..., 30 below the root (tree
// depth <= 32); the points are tested without a level of their own.
constexpr int kNNLevels = 6;
constexpr uint32_t kNNMaxBlocks = 256;

struct NNShared {
    float top[6][kNNTop];              // min x, y, z, max x, y, z (SoA: no bank conflicts)
    float lb[kNNWaves][kNNLevels][64]; // lower bounds of each level's pending nodes
};

__device__ __forceinline__ float point_dist(const float *__restrict__ p, float qx, float qy,
                                            float qz) {
    const float dx = p[0] - qx, dy = p[1] - qy, dz = p[2] - qz;
    return sqrtf(sdf_dot3(dx, dy, dz, dx, dy, dz));
}

// distance from q to the box (0 inside): (min - q).max(0).max(q - max).norm()
// (src/aabb_tree/aabb_tree.cuh:272-275)
__device__ __forceinline__ float box_dist(const float *__restrict__ b, float qx, float qy,
                                          float qz) {
    const float dx = fmaxf(fmaxf(b[0] - qx, 0.0f), qx - b[3]);
    const float dy = fmaxf(fmaxf(b[1] - qy, 0.0f), qy - b[4]);
    const float dz = fmaxf(fmaxf(b[2] - qz, 0.0f), qz - b[5]);
    return sqrtf(sdf_dot3(dx, dy, dz, dx, dy, dz));
}

// wave-wide lexicographic minimum of (value, index)
__device__ __forceinline__ void wave_argmin(float &v, uint32_t &idx) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(v, off, 64);
        const uint32_t oi = __shfl_xor(idx, off, 64);
        if (ov < v || (ov == v && oi < idx)) {
            v = ov;
            idx = oi;
        }
    }
}

__device__ __forceinline__ float box_dist_top(const NNShared &sh, uint32_t b, float qx, float qy,
                                             float qz) {
    const float dx = fmaxf(fmaxf(sh.top[0][b] - qx, 0.0f), qx - sh.top[3][b]);
    const float dy = fmaxf(fmaxf(sh.top[1][b] - qy, 0.0f), qy - sh.top[4][b]);
    const float dz = fmaxf(fmaxf(sh.top[2][b] - qz, 0.0f), qz - sh.top[5][b]);
    return sqrtf(sdf_dot3(dx, dy, dz, dx, dy, dz));
}

// Copies the boxes of depths 6 and 12 (those above the points) into LDS.
// Every thread of the block calls it; it ends with a block barrier.
__device__ void nn_load_top(const float *__restrict__ tree, uint32_t td, NNShared &sh) {
    const uint64_t n2 = 1ull << td;
    for (uint32_t t = threadIdx.x; t < kNNTop; t += kNNBlock) {
        const uint32_t d = t < kNNTopA ? 6u : 12u;
        const uint32_t i = t < kNNTopA ? t : t - kNNTopA;
        if (d >= td) continue; // no boxes at that depth: never read
        const float *b = tree + 6ull * ((n2 - (2ull << d)) + i);
#pragma unroll
        for (int c = 0; c < 6; ++c) sh.top[c][t] = b[c];
    }
    __syncthreads();
}

// Nearest point to q for the whole wavefront (the result is uniform), over
// the tree of depth td (points padded to 2^td).  NaN lower bounds mark nodes
// that are taken, outside the group or not comparable (NaN query): a node is
// pending while lb < best, or lb == best and it holds a smaller index than the
// best (its first one).  0 when no point has a distance (NaN query).
__device__ uint32_t nn_wave(const float *__restrict__ points, const float *__restrict__ tree,
                            uint32_t num_points, uint32_t td, float qx, float qy, float qz,
                            NNShared &sh, uint32_t wave) {
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t n2 = 1ull << td;
    const float kInf = __builtin_bit_cast(float, 0x7f800000u);
    const float kNaN = __builtin_bit_cast(float, 0x7fc00000u);
    float best = kInf;
    uint32_t best_idx = kNoIndex;

    // the points of a group: one per lane
    auto test_points = [&](uint32_t first, uint32_t size) {
        const uint32_t p = first + lane;
        const bool ok = lane < size && p < num_points;
        float dist = ok ? point_dist(points + 3ull * p, qx, qy, qz) : kInf;
        uint32_t idx = ok ? p : kNoIndex;
        wave_argmin(dist, idx);
        if (dist < best || (dist == best && idx < best_idx)) {
            best = dist;
            best_idx = idx;
        }
    };
    // lower bound of node `first + lane` of depth d (NaN outside the group)
    auto bound = [&](uint32_t d, uint32_t first, uint32_t size) {
        const uint32_t node = first + lane;
        if (lane >= size) return kNaN;
        if (d == 6) return box_dist_top(sh, node, qx, qy, qz);
        if (d == 12) return box_dist_top(sh, kNNTopA + node, qx, qy, qz);
        return box_dist(tree + 6ull * ((n2 - (2ull << d)) + node), qx, qy, qz);
    };

    if (td <= 6) { // a single group of points
        test_points(0, 1u << td);
        const uint32_t r = (uint32_t)__builtin_amdgcn_readfirstlane((int)best_idx);
        return r == kNoIndex ? 0u : r;
    }
    float(*lbs)[64] = sh.lb[wave];
    // lane k holds the first node of level k's group (level k at depth
    // min(6 (k + 1), td), all of it below the points' depth)
    uint32_t first_of = 0;
    lbs[0][lane] = bound(6, 0, 64);
    int k = 0;
    while (k >= 0) {
        __builtin_amdgcn_wave_barrier();
        const float lb = lbs[k][lane];
        const uint32_t d = 6u * (uint32_t)(k + 1);
        const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)first_of, k);
        const bool pending =
            lb < best || (lb == best && ((uint64_t)(first + lane) << (td - d)) < best_idx);
        float bl = pending ? lb : kInf;
        uint32_t bi = pending ? lane : 64u;
        wave_argmin(bl, bi);
        if (bi >= 64u) { // level done
            --k;
            continue;
        }
        if (lane == bi) lbs[k][lane] = kNaN; // taken
        const uint32_t node = first + bi;
        const uint32_t dc = d + 6 < td ? d + 6 : td;
        const uint32_t cfirst = node << (dc - d);
        const uint32_t csize = 1u << (dc - d);
        if (dc == td) {
            test_points(cfirst, csize);
            continue;
        }
        ++k; // k + 1 < kNNLevels: dc < td <= 32 makes dc <= 30
        if (lane == (uint32_t)k) first_of = cfirst;
        lbs[k][lane] = bound(dc, cfirst, csize);
    }
    const uint32_t r = (uint32_t)__builtin_amdgcn_readfirstlane((int)best_idx);
    return r == kNoIndex ? 0u : r;
}

__global__ __launch_bounds__(kNNBlock) void nn_kernel(const float *__restrict__ points,
                                                      const float *__restrict__ tree,
                                                      const float *__restrict__ queries,
                                                      uint32_t num_points, uint32_t num_queries,
                                                      uint32_t *__restrict__ indices) {
    __shared__ NNShared sh;
    const uint32_t td = ilog2_u32(pow2_up(num_points));
    nn_load_top(tree, td, sh);
    const uint32_t wave = threadIdx.x >> 6;
    for (uint32_t qi = blockIdx.x * kNNWaves + wave; qi < num_queries; qi += gridDim.x * kNNWaves) {
        const uint32_t r = nn_wave(points, tree, num_points, td, queries[3ull * qi],
                                   queries[3ull * qi + 1], queries[3ull * qi + 2], sh, wave);
        if ((threadIdx.x & 63u) == 0) indices[qi] = r;
    }
}

hipError_t launch_nn(const float *points, const float *tree, const float *queries,
                     uint32_t num_points, uint32_t num_queries, uint32_t *indices,
                     hipStream_t stream) {
    if (num_queries == 0) return hipSuccess;
    const uint32_t blocks = std::min<uint32_t>((num_queries + kNNWaves - 1) / kNNWaves, kNNMaxBlocks);
    hipLaunchKernelGGL(nn_kernel, dim3(blocks), dim3(kNNBlock), 0, stream, points, tree, queries,
                       num_points, num_queries, indices);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Start cells of a ray batch (get_starting_point, sdfoam_model/scene.py:
// 272-282): the nearest point to each ray's origin.  A batch's rays come from
// few camera positions, so the origins are deduplicated on the GPU in an
// open-addressing hash table keyed on their bits (the reference sorts them
// with torch.unique, which synchronises with the host), each distinct
// origin's nearest point is found once, and every ray takes its origin's.
// With at most kStartBrute distinct origins the search is a scan over all
// points (one pass over the points for all of them: the same fp32 distances
// as nn_wave, ties to the smallest index), else nn_wave per origin.  Equal
// results to nn over the distinct origins for finite points and origins.

constexpr uint32_t kStartBrute = 256;
constexpr uint32_t kStartPts = 8;          // points per thread in the scan

__host__ StartLayout start_layout(uint32_t num_rays) {
    StartLayout l;
    uint64_t t = 64;
    while (t < 2ull * num_rays) t *= 2;
    l.table_slots = t;
    auto up = [](uint64_t x) { return (x + 255u) / 256u * 256u; };
    l.table = 256;
    l.uid = l.table + up(4 * t);
    l.ray_slot = l.uid + up(4 * t);
    l.uq_ray = l.ray_slot + up(4ull * num_rays);
    l.best = l.uq_ray + up(4ull * num_rays);
    l.bytes = l.best + up(8ull * num_rays);
    return l;
}

__device__ __forceinline__ uint32_t origin_hash(uint32_t x, uint32_t y, uint32_t z) {
    uint32_t h = x * 0x9e3779b1u ^ (y + 0x7f4a7c15u) * 0x85ebca77u ^ (z + 0x165667b1u) * 0xc2b2ae3du;
    h ^= h >> 15;
    h *= 0x2c1b3c6du;
    h ^= h >> 12;
    return h;
}

__device__ __forceinline__ bool same_origin(const float *__restrict__ rays, uint32_t a, uint32_t b) {
    const uint32_t *ra = reinterpret_cast<const uint32_t *>(rays + 6ull * a);
    const uint32_t *rb = reinterpret_cast<const uint32_t *>(rays + 6ull * b);
    return ra[0] == rb[0] && ra[1] == rb[1] && ra[2] == rb[2];
}

__global__ __launch_bounds__(kBlock) void start_init_kernel(uint32_t *__restrict__ counter,
                                                            uint32_t *__restrict__ table,
                                                            uint64_t slots) {
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < slots;
         i += (uint64_t)gridDim.x * kBlock)
        table[i] = kNoIndex;
    if (blockIdx.x == 0 && threadIdx.x == 0) *counter = 0u;
}

// Each ray claims the first free slot of its probe sequence or finds the
// slot of an equal origin there.  The table has at least twice as many slots
// as rays, so every probe sequence reaches a free slot or its origin's.
// Rays of one block with the bits of its first ray's origin take that ray's
// slot without probing: a batch from one camera makes one probe per 1,024 rays
// instead of every ray contending for the same slot.  (One probe per wavefront,
// before, left 30,000 of them for one line of the table at 1600x1200 rays: 110 us
// against 19 us now.)
constexpr uint32_t kHashBlock = 1024;

__global__ __launch_bounds__(kHashBlock) void start_hash_kernel(const float *__restrict__ rays,
                                                                uint32_t num_rays,
                                                                uint32_t *__restrict__ table,
                                                                uint64_t slots,
                                                                uint32_t *__restrict__ ray_slot) {
    __shared__ uint32_t lead[4]; // the first ray's origin and slot
    const uint32_t i = blockIdx.x * kHashBlock + threadIdx.x;
    uint32_t ox = 0, oy = 0, oz = 0;
    if (i < num_rays) {
        const uint32_t *o = reinterpret_cast<const uint32_t *>(rays + 6ull * i);
        ox = o[0];
        oy = o[1];
        oz = o[2];
    }
    if (threadIdx.x == 0) {
        lead[0] = ox;
        lead[1] = oy;
        lead[2] = oz;
    }
    __syncthreads();
    const bool follower = threadIdx.x != 0 && ox == lead[0] && oy == lead[1] && oz == lead[2];
    uint64_t h = origin_hash(ox, oy, oz) & (slots - 1);
    if (i < num_rays && !follower) {
        for (uint64_t probe = 0; probe < slots; ++probe) {
            uint32_t s = table[h];
            if (s == kNoIndex) {
                s = atomicCAS(table + h, kNoIndex, i);
                if (s == kNoIndex) break; // claimed
            }
            if (same_origin(rays, s, i)) break;
            h = (h + 1) & (slots - 1);
        }
    }
    if (threadIdx.x == 0) lead[3] = (uint32_t)h;
    __syncthreads();
    if (i < num_rays) ray_slot[i] = follower ? lead[3] : (uint32_t)h;
}

// Numbers the claimed slots (the distinct origins) and resets their results.
__global__ __launch_bounds__(kBlock) void start_unique_kernel(const uint32_t *__restrict__ table,
                                                              uint64_t slots,
                                                              uint32_t *__restrict__ counter,
                                                              uint32_t *__restrict__ uid,
                                                              uint32_t *__restrict__ uq_ray,
                                                              uint64_t *__restrict__ best) {
    for (uint64_t h = (uint64_t)blockIdx.x * kBlock + threadIdx.x; h < slots;
         h += (uint64_t)gridDim.x * kBlock) {
        const uint32_t r = table[h];
        if (r == kNoIndex) continue;
        const uint32_t u = atomicAdd(counter, 1u);
        uid[h] = u;
        uq_ray[u] = r;
        best[u] = ~0ull;
    }
}

// Nearest of the block's kBlock * kStartPts points (block `chunk` of them) to
// each of the `count` positions q: per wavefront and position one atomic of the
// smallest (distance bits, index) into slot (LDS).  Lanes keep their own smallest over their
// points; the wave's smallest distance comes by DPP and its index from the
// lanes that hold that distance (one, but for ties).
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
    auto step = [](uint32_t x, uint32_t y) { return x < y ? x : y; };
    v = step(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x111, 0xf, 0xf, false));
    v = step(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x112, 0xf, 0xf, false));
    v = step(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x114, 0xf, 0xf, false));
    v = step(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x118, 0xf, 0xf, false));
    v = step(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xa, 0xf, false));
    v = step(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xc, 0xf, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ void brute_scan(const float *__restrict__ points, uint32_t num_points,
                                           uint32_t chunk, const float (*q)[3], uint32_t count,
                                           unsigned long long *slot) {
    const uint64_t p0 = (uint64_t)chunk * kBlock * kStartPts + threadIdx.x;
    float px[kStartPts], py[kStartPts], pz[kStartPts];
#pragma unroll
    for (uint32_t k = 0; k < kStartPts; ++k) {
        const uint64_t j = p0 + (uint64_t)k * kBlock;
        // past the end: NaN, no candidate
        const bool ok = j < num_points;
        px[k] = ok ? points[3 * j] : __builtin_bit_cast(float, 0x7fc00000u);
        py[k] = ok ? points[3 * j + 1] : 0.0f;
        pz[k] = ok ? points[3 * j + 2] : 0.0f;
    }
    for (uint32_t u = 0; u < count; ++u) {
        const float qx = q[u][0], qy = q[u][1], qz = q[u][2];
        uint32_t dist = 0xffffffffu, at = 0u; // distances are >= 0: their bits sort like them
#pragma unroll
        for (uint32_t k = 0; k < kStartPts; ++k) {
            const float dx = px[k] - qx, dy = py[k] - qy, dz = pz[k] - qz;
            const float d = sqrtf(sdf_dot3(dx, dy, dz, dx, dy, dz));
            const uint32_t b = __builtin_bit_cast(uint32_t, d);
            if (d == d && b < dist) { // points in ascending order: ties keep the first
                dist = b;
                at = k;
            }
        }
        const uint32_t least = wave_min_u32(dist);
        if (least == 0xffffffffu) continue; // no point of the wave has a distance
        const uint32_t j = (uint32_t)(p0 + (uint64_t)at * kBlock);
        const uint32_t first = wave_min_u32(dist == least ? j : 0xffffffffu);
        if ((threadIdx.x & 63u) == 0)
            atomicMin(slot + u, (unsigned long long)least << 32 | first);
    }
}

__device__ __forceinline__ void brute_merge(uint32_t count, const unsigned long long *slot,
                                            uint64_t *__restrict__ best) {
    __syncthreads();
    for (uint32_t u = threadIdx.x; u < count; u += kBlock)
        if (slot[u] != ~0ull) atomicMin(reinterpret_cast<unsigned long long *>(best) + u, slot[u]);
}

// At most kStartBrute distinct origins: every block scans kBlock * kStartPts
// points for all of them.
__global__ __launch_bounds__(kBlock) void start_brute_kernel(const float *__restrict__ points,
                                                             uint32_t num_points,
                                                             const float *__restrict__ rays,
                                                             const uint32_t *__restrict__ counter,
                                                             const uint32_t *__restrict__ uq_ray,
                                                             uint64_t *__restrict__ best) {
    __shared__ float q[kStartBrute][3];
    __shared__ unsigned long long slot[kStartBrute];
    const uint32_t count = *counter;
    if (count == 0 || count > kStartBrute) return; // the whole grid
    for (uint32_t u = threadIdx.x; u < count; u += kBlock) {
        const float *o = rays + 6ull * uq_ray[u];
        q[u][0] = o[0];
        q[u][1] = o[1];
        q[u][2] = o[2];
        slot[u] = ~0ull;
    }
    __syncthreads();
    brute_scan(points, num_points, blockIdx.x, q, count, slot);
    brute_merge(count, slot, best);
}

// The same for nn's queries, `per` of them (at most kScanQueries) per blockIdx.y.
// A block takes its queries one after another, 0.7 us each, so few pairs go to
// many blocks with few queries each: with 64 queries per block whatever the
// sizes, 64 to 1,000 queries over 4,000 to 100k points took 53 us and more.
constexpr uint32_t kScanQueries = 64;
constexpr uint32_t kScanBlocks = 2048; // (8 per CU)

// Up to this many points a block scans all of them and writes the results
// itself: one launch instead of three.
constexpr uint32_t kScanWhole = 4 * kBlock * kStartPts;

__device__ __forceinline__ uint32_t scan_queries(const float *__restrict__ queries,
                                                 uint32_t num_queries, uint32_t per, float (*q)[3],
                                                 unsigned long long *slot) {
    const uint32_t q0 = blockIdx.y * per;
    const uint32_t count = min(per, num_queries - q0);
    if (threadIdx.x < count) {
        const uint32_t u = threadIdx.x;
#pragma unroll
        for (int c = 0; c < 3; ++c) q[u][c] = queries[3ull * (q0 + u) + c];
        slot[u] = ~0ull;
    }
    __syncthreads();
    return count;
}

__global__ __launch_bounds__(kBlock) void nn_whole_kernel(const float *__restrict__ points,
                                                          uint32_t num_points,
                                                          const float *__restrict__ queries,
                                                          uint32_t num_queries, uint32_t per,
                                                          uint32_t *__restrict__ indices) {
    __shared__ float q[kScanQueries][3];
    __shared__ unsigned long long slot[kScanQueries];
    const uint32_t count = scan_queries(queries, num_queries, per, q, slot);
    for (uint32_t chunk = 0; chunk * (kBlock * kStartPts) < num_points; ++chunk)
        brute_scan(points, num_points, chunk, q, count, slot);
    __syncthreads();
    if (threadIdx.x < count) {
        const unsigned long long s = slot[threadIdx.x];
        indices[blockIdx.y * per + threadIdx.x] = s == ~0ull ? 0u : (uint32_t)s;
    }
}

__global__ __launch_bounds__(kBlock) void nn_brute_kernel(const float *__restrict__ points,
                                                          uint32_t num_points,
                                                          const float *__restrict__ queries,
                                                          uint32_t num_queries, uint32_t per,
                                                          uint64_t *__restrict__ best) {
    __shared__ float q[kScanQueries][3];
    __shared__ unsigned long long slot[kScanQueries];
    const uint32_t count = scan_queries(queries, num_queries, per, q, slot);
    brute_scan(points, num_points, blockIdx.x, q, count, slot);
    brute_merge(count, slot, best + blockIdx.y * per);
}

__global__ __launch_bounds__(kBlock) void nn_reset_kernel(uint64_t *__restrict__ best, uint32_t n) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) best[i] = ~0ull;
}

__global__ __launch_bounds__(kBlock) void nn_result_kernel(const uint64_t *__restrict__ best,
                                                           uint32_t n,
                                                           uint32_t *__restrict__ indices) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) indices[i] = best[i] == ~0ull ? 0u : (uint32_t)best[i];
}

hipError_t launch_nn_brute(const float *points, const float *queries, uint32_t num_points,
                           uint32_t num_queries, uint32_t *indices, uint64_t *best,
                           hipStream_t stream) {
    const uint32_t chunks =
        (uint32_t)(((uint64_t)num_points + kBlock * kStartPts - 1) / (kBlock * kStartPts));
    const bool whole = num_points <= kScanWhole;
    const uint32_t per = (uint32_t)std::min<uint64_t>(
        kScanQueries,
        std::max<uint64_t>(1, ((uint64_t)num_queries * (whole ? 1 : chunks) + kScanBlocks - 1) /
                                  kScanBlocks));
    // (nn_route scans for at most 65,536 queries, fewer the more points there are: at most
    // 16,640 groups)
    const dim3 grid(whole ? 1 : chunks, (num_queries + per - 1) / per);
    if (whole) {
        hipLaunchKernelGGL(nn_whole_kernel, grid, dim3(kBlock), 0, stream, points, num_points,
                           queries, num_queries, per, indices);
        return hipGetLastError();
    }
    const dim3 per_query((num_queries + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(nn_reset_kernel, per_query, dim3(kBlock), 0, stream, best, num_queries);
    hipLaunchKernelGGL(nn_brute_kernel, grid, dim3(kBlock), 0, stream, points, num_points, queries,
                       num_queries, per, best);
    hipLaunchKernelGGL(nn_result_kernel, per_query, dim3(kBlock), 0, stream, best, num_queries,
                       indices);
    return hipGetLastError();
}

// More distinct origins: one tree search per origin, the waves of the grid
// taking the origins in turn.
__global__ __launch_bounds__(kNNBlock) void start_tree_kernel(const float *__restrict__ points,
                                                              uint32_t num_points,
                                                              const float *__restrict__ tree,
                                                              const float *__restrict__ rays,
                                                              const uint32_t *__restrict__ counter,
                                                              const uint32_t *__restrict__ uq_ray,
                                                              uint64_t *__restrict__ best) {
    __shared__ NNShared sh;
    const uint32_t count = *counter;
    if (count <= kStartBrute) return; // the whole grid
    const uint32_t td = ilog2_u32(pow2_up(num_points));
    nn_load_top(tree, td, sh);
    const uint32_t wave = threadIdx.x >> 6;
    for (uint32_t u = blockIdx.x * kNNWaves + wave; u < count; u += gridDim.x * kNNWaves) {
        const float *o = rays + 6ull * uq_ray[u];
        const uint32_t r = nn_wave(points, tree, num_points, td, o[0], o[1], o[2], sh, wave);
        if ((threadIdx.x & 63u) == 0) best[u] = r;
    }
}

__global__ __launch_bounds__(kBlock) void start_scatter_kernel(uint32_t num_rays,
                                                               const uint32_t *__restrict__ ray_slot,
                                                               const uint32_t *__restrict__ uid,
                                                               const uint64_t *__restrict__ best,
                                                               uint32_t *__restrict__ start) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= num_rays) return;
    const uint64_t b = best[uid[ray_slot[i]]];
    start[i] = b == ~0ull ? 0u : (uint32_t)b;
}

hipError_t launch_start_points(const float *rays, uint32_t num_rays, const float *points,
                               uint32_t num_points, const float *tree, uint32_t *start,
                               void *scratch, hipStream_t stream) {
    if (num_rays == 0) return hipSuccess;
    const StartLayout l = start_layout(num_rays);
    char *base = static_cast<char *>(scratch);
    uint32_t *counter = reinterpret_cast<uint32_t *>(base);
    uint32_t *table = reinterpret_cast<uint32_t *>(base + l.table);
    uint32_t *uid = reinterpret_cast<uint32_t *>(base + l.uid);
    uint32_t *ray_slot = reinterpret_cast<uint32_t *>(base + l.ray_slot);
    uint32_t *uq_ray = reinterpret_cast<uint32_t *>(base + l.uq_ray);
    uint64_t *best = reinterpret_cast<uint64_t *>(base + l.best);
    const uint32_t slot_blocks = (uint32_t)std::min<uint64_t>((l.table_slots + kBlock - 1) / kBlock, 4096);
    const uint32_t ray_blocks = (num_rays + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(start_init_kernel, dim3(slot_blocks), dim3(kBlock), 0, stream, counter, table,
                       l.table_slots);
    hipLaunchKernelGGL(start_hash_kernel, dim3((num_rays + kHashBlock - 1) / kHashBlock),
                       dim3(kHashBlock), 0, stream, rays, num_rays, table, l.table_slots, ray_slot);
    hipLaunchKernelGGL(start_unique_kernel, dim3(slot_blocks), dim3(kBlock), 0, stream, table,
                       l.table_slots, counter, uid, uq_ray, best);
    const uint32_t point_blocks = (uint32_t)(((uint64_t)num_points + kBlock * kStartPts - 1) /
                                             (kBlock * kStartPts));
    hipLaunchKernelGGL(start_brute_kernel, dim3(point_blocks), dim3(kBlock), 0, stream, points,
                       num_points, rays, counter, uq_ray, best);
    hipLaunchKernelGGL(start_tree_kernel, dim3(kNNMaxBlocks), dim3(kNNBlock), 0, stream, points,
                       num_points, tree, rays, counter, uq_ray, best);
    hipLaunchKernelGGL(start_scatter_kernel, dim3(ray_blocks), dim3(kBlock), 0, stream, num_rays,
                       ray_slot, uid, best, start);
    return hipGetLastError();
}

} // namespace sdfoam_hip
