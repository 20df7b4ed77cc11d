// Exact nearest neighbours of many queries over points sorted along a Z-order
// curve, for gfx950.
//
// The caller's tree bounds consecutive points, and the reference's point order
// (whole-array sorts by one coordinate, then 1,024-point blocks) makes those
// boxes thin slabs across the whole scene: a search over them tests thousands
// of points per query.  Here the points are sorted by Morton code for the call
// (48 bits: cells of the extent / 65,536), and boxes over 64, 64^2, ... of them
// are made, 64 children each.  Queries are sorted by the same code; a wavefront
// takes a run of them, one at a time, and starts each from the distance to the
// previous one's nearest point, so most of the groups it would enter are
// skipped at once.  100,003 scattered queries over 1M points: 14-25 ms by the
// caller's tree, 0.60 ms this way: 0.40 the search (bound by its dependent
// loads, ~50 per query at 8 wavefronts per SIMD), 0.20 the sorts and boxes.
#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>

#include "trace_kernels.h"

namespace sdfoam_hip {

namespace {

constexpr uint32_t kGroup = 64;     // children per box
constexpr int kMaxLevels = 5;       // 64^5 > 2^31 / 64 groups of points
constexpr uint32_t kKeyBits = 48;
constexpr uint32_t kSearchWaves = 8192; // runs of queries at most (8 waves per SIMD)

size_t align256(size_t x) { return (x + 255u) & ~(size_t)255u; }

// levels of boxes: level 0 bounds kGroup points each, the last has at most
// kGroup boxes
struct Levels {
    int count;
    uint64_t width[kMaxLevels + 1];
    uint64_t start[kMaxLevels + 1]; // first box, in boxes
    uint64_t boxes;
};

Levels levels_of(uint32_t n) {
    Levels l = {};
    uint64_t w = ((uint64_t)n + kGroup - 1) / kGroup;
    for (;;) {
        l.width[l.count] = w;
        l.start[l.count] = l.boxes;
        l.boxes += w;
        ++l.count;
        if (w <= kGroup) return l;
        w = (w + kGroup - 1) / kGroup;
    }
}

// 16 bits of x at every third bit
__device__ __forceinline__ uint64_t spread3(uint32_t v) {
    uint64_t x = v & 0xffffu;
    x = (x | (x << 16)) & 0x0000ff0000ffull;
    x = (x | (x << 8)) & 0x00f00f00f00full;
    x = (x | (x << 4)) & 0x0c30c30c30c3ull;
    x = (x | (x << 2)) & 0x249249249249ull;
    return x;
}

// Morton keys of positions in the tree's root box (clamped to it: the keys
// only order the work, any of them gives the same result; NaN sorts as 0)
__global__ __launch_bounds__(kBlock) void key_kernel(const float *__restrict__ x, uint32_t n,
                                                     const float *__restrict__ root,
                                                     uint64_t *__restrict__ keys,
                                                     uint32_t *__restrict__ ids) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float ext = fmaxf(fmaxf(root[3] - root[0], root[4] - root[1]), root[5] - root[2]);
    const float scale = ext > 0.0f ? 65536.0f / ext : 0.0f;
    uint64_t key = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float q = fminf(fmaxf((x[3ull * i + c] - root[c]) * scale, 0.0f), 65535.0f);
        key |= spread3((uint32_t)q) << c;
    }
    keys[i] = key;
    ids[i] = i;
}

// wave-wide minimum of unsigned words, non-negative floats' bits among them
// (result uniform)
__device__ __forceinline__ uint32_t wave_min_bits(uint32_t v) {
    auto less = [](uint32_t x, uint32_t y) { return x < y ? x : y; };
    v = less(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x111, 0xf, 0xf, false));
    v = less(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x112, 0xf, 0xf, false));
    v = less(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x114, 0xf, 0xf, false));
    v = less(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x118, 0xf, 0xf, false));
    v = less(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xa, 0xf, false));
    v = less(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xc, 0xf, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The sorted points (x, y, z, index) and the boxes over 64 of them: one
// wavefront per box.  A box is two float4: its lower corner and the bits of
// its points' smallest index, and its upper corner.
__device__ __forceinline__ float wave_min_f(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off, 64));
    return v;
}

__device__ __forceinline__ void wave_box(float4 lo, float4 hi, float4 *__restrict__ boxes,
                                         uint64_t at) {
    lo.x = wave_min_f(lo.x);
    lo.y = wave_min_f(lo.y);
    lo.z = wave_min_f(lo.z);
    hi.x = -wave_min_f(-hi.x);
    hi.y = -wave_min_f(-hi.y);
    hi.z = -wave_min_f(-hi.z);
    lo.w = __builtin_bit_cast(float, wave_min_bits(__builtin_bit_cast(uint32_t, lo.w)));
    if ((threadIdx.x & 63u) == 0) {
        boxes[2 * at] = lo;
        boxes[2 * at + 1] = hi;
    }
}

__global__ __launch_bounds__(kBlock) void gather_kernel(const float *__restrict__ points,
                                                        const uint32_t *__restrict__ order,
                                                        uint32_t n, float4 *__restrict__ sorted,
                                                        float4 *__restrict__ boxes) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i - (threadIdx.x & 63u) >= n) return; // the whole wavefront
    const uint32_t id = order[i < n ? i : n - 1u]; // the last group repeats the last point
    const float4 p = make_float4(points[3ull * id], points[3ull * id + 1], points[3ull * id + 2],
                                 __builtin_bit_cast(float, id));
    if (i < n) sorted[i] = p;
    wave_box(p, p, boxes, i / kGroup);
}

__global__ __launch_bounds__(kBlock) void level_kernel(float4 *__restrict__ boxes, uint64_t child,
                                                       uint64_t children, uint64_t start) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i - (threadIdx.x & 63u) >= children) return; // the whole wavefront
    const uint64_t c = child + (i < children ? i : children - 1u);
    wave_box(boxes[2 * c], boxes[2 * c + 1], boxes, start + i / kGroup);
}

constexpr uint32_t kNever = 0xffffffffu; // above every distance's bits

struct Search {
    const float4 *sorted;
    const float4 *boxes;
    uint64_t start[kMaxLevels];
    uint64_t width[kMaxLevels];
    uint32_t n;
};

// the query's state: uniform over the wave
struct Nearest {
    float x, y, z;
    uint32_t dist, id; // bits of the best distance, and its smallest index
};

__device__ __forceinline__ void test_group(const Search &s, Nearest &b, uint64_t group) {
    const uint64_t i = group * kGroup + (threadIdx.x & 63u);
    uint32_t dist = kNever, id = kNoIndex;
    if (i < s.n) {
        const float4 p = s.sorted[i];
        const float dx = p.x - b.x, dy = p.y - b.y, dz = p.z - b.z;
        const float d = sqrtf(sdf_dot3(dx, dy, dz, dx, dy, dz));
        if (d == d) { // NaN: no candidate
            dist = __builtin_bit_cast(uint32_t, d);
            id = __builtin_bit_cast(uint32_t, p.w);
        }
    }
    const uint32_t least = wave_min_bits(dist);
    if (least == kNever || least > b.dist) return;
    const uint32_t first = wave_min_bits(dist == least ? id : kNoIndex);
    if (least < b.dist || first < b.id) {
        b.dist = least;
        b.id = first;
    }
}

// The boxes of level LEVEL from `first` on (64 of them), nearest first, while
// their lower bound is below the best distance, or equal to it and they hold a
// smaller index (a tie goes to the smallest one; those go by their smallest
// indices).  The box distance is a lower bound of the fp32 point distance, since
// rounding is monotone.  Entering every equal one made a query with an infinite
// coordinate, or one so far out that all distances round to one value, visit
// every box: with 1% of them 100k queries over 1M points took 120 ms, 0.71 now.
template <int LEVEL>
__device__ __forceinline__ void descend(const Search &s, Nearest &b, uint64_t first) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t lb = kNever;
    if (first + lane < s.width[LEVEL]) {
        const float4 lo = s.boxes[2 * (s.start[LEVEL] + first + lane)];
        const float4 hi = s.boxes[2 * (s.start[LEVEL] + first + lane) + 1];
        const float dx = fmaxf(fmaxf(lo.x - b.x, 0.0f), b.x - hi.x);
        const float dy = fmaxf(fmaxf(lo.y - b.y, 0.0f), b.y - hi.y);
        const float dz = fmaxf(fmaxf(lo.z - b.z, 0.0f), b.z - hi.z);
        const float d = sqrtf(sdf_dot3(dx, dy, dz, dx, dy, dz));
        lb = __builtin_bit_cast(uint32_t, d);
    }
    while (true) {
        const uint32_t least = wave_min_bits(lb);
        uint64_t next = __builtin_amdgcn_ballot_w64(lb == least);
        if (least >= b.dist) { // (kNever is above every distance)
            if (least > b.dist) return;
            // the indices are read where there is a tie
            uint32_t low = kNoIndex;
            if (lb == least)
                low = __builtin_bit_cast(uint32_t, s.boxes[2 * (s.start[LEVEL] + first + lane)].w);
            const uint32_t lowest = wave_min_bits(low);
            if (lowest >= b.id) return;
            next = __builtin_amdgcn_ballot_w64(low == lowest);
        }
        const int at = __builtin_ctzll(next);
        if (lane == (uint32_t)at) lb = kNever; // taken
        if constexpr (LEVEL == 0) {
            test_group(s, b, first + at);
        } else {
            descend<LEVEL - 1>(s, b, (first + at) * kGroup);
        }
    }
}

template <int LEVELS>
__global__ __launch_bounds__(kBlock) void search_kernel(Search s, const float *__restrict__ queries,
                                                        const uint32_t *__restrict__ order,
                                                        uint32_t m, uint32_t run,
                                                        const float *__restrict__ points,
                                                        uint32_t *__restrict__ indices) {
    const uint32_t wave = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    const uint64_t q0 = (uint64_t)wave * run;
    uint32_t near = kNoIndex;
    for (uint64_t k = q0; k < q0 + run && k < m; ++k) {
        const uint32_t q = (uint32_t)__builtin_amdgcn_readfirstlane((int)order[k]);
        Nearest b;
        b.x = queries[3ull * q];
        b.y = queries[3ull * q + 1];
        b.z = queries[3ull * q + 2];
        b.dist = 0x7f800000u; // infinity: a candidate at that distance counts
        b.id = kNoIndex;
        if (near != kNoIndex) {
            // the previous query's nearest point is a candidate
            const float dx = points[3ull * near] - b.x, dy = points[3ull * near + 1] - b.y,
                        dz = points[3ull * near + 2] - b.z;
            const float d = sqrtf(sdf_dot3(dx, dy, dz, dx, dy, dz));
            if (d == d) {
                b.dist = __builtin_bit_cast(uint32_t, d);
                b.id = near;
            }
        }
        b.dist = (uint32_t)__builtin_amdgcn_readfirstlane((int)b.dist);
        b.id = (uint32_t)__builtin_amdgcn_readfirstlane((int)b.id);
        // a query with a NaN has no distance to any point: index 0
        if (b.x == b.x && b.y == b.y && b.z == b.z) descend<LEVELS - 1>(s, b, 0);
        near = b.id;
        if ((threadIdx.x & 63u) == 0) indices[q] = near == kNoIndex ? 0u : near;
    }
}

struct Layout {
    size_t keys_in, keys_out, ids, order, queries, sorted, boxes, temp, temp_bytes, bytes;
};

// 0 bytes: the sort's scratch could not be sized
Layout layout_of(uint32_t n, uint32_t m) {
    Layout l = {};
    const size_t k = std::max(n, m);
    const uint64_t *ki = nullptr;
    uint64_t *ko = nullptr;
    const uint32_t *vi = nullptr;
    uint32_t *vo = nullptr;
    size_t a = 0, b = 0;
    if (rocprim::radix_sort_pairs(nullptr, a, ki, ko, vi, vo, n, 0u, kKeyBits) != hipSuccess ||
        rocprim::radix_sort_pairs(nullptr, b, ki, ko, vi, vo, m, 0u, kKeyBits) != hipSuccess)
        return l;
    auto take = [&l](size_t bytes) {
        const size_t at = l.bytes;
        l.bytes += align256(bytes);
        return at;
    };
    l.keys_in = take(8 * k);
    l.keys_out = take(8 * k);
    l.ids = take(4 * k);
    l.order = take(4ull * n);
    l.queries = take(4ull * m);
    l.sorted = take(16ull * n);
    l.boxes = take(32ull * levels_of(n).boxes);
    l.temp_bytes = std::max(a, b);
    l.temp = take(l.temp_bytes);
    return l;
}

hipError_t sort_positions(const float *x, uint32_t n, const float *root, char *base,
                          const Layout &l, uint32_t *order, hipStream_t stream) {
    uint64_t *keys = reinterpret_cast<uint64_t *>(base + l.keys_in);
    uint64_t *sorted = reinterpret_cast<uint64_t *>(base + l.keys_out);
    uint32_t *ids = reinterpret_cast<uint32_t *>(base + l.ids);
    hipLaunchKernelGGL(key_kernel, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, x, n,
                       root, keys, ids);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    size_t temp = l.temp_bytes;
    return rocprim::radix_sort_pairs(base + l.temp, temp, keys, sorted, ids, order, n, 0u,
                                     kKeyBits, stream);
}

} // namespace

// Which way nn takes when it has scratch, by the times of all three over four
// scenes in the reference's point order and in no order (us: scan / caller's
// tree, lowest to highest / sorted):
//   64 points x 16,384 queries          24 /   7      /  55
//   1,000     x 4,096                   10 /  14-23   /  46
//   1,000     x 65,536                  91 /  94-132  / 112
//   1,000     x 200,000                266 / 245-366  / 232
//   4,000     x 2,048                   14 /  10-14   /  57
//   4,000     x 65,536                 180 /  71-97   / 146
//   8,192     x 16,384                 103 /  88-181  / 104
//   16,384    x 4,096                   56 /  59-146  /  81
//   100,000   x 1,024                   83 /  27-102  / 105
//   100,000   x 8,192                  557 /  43-303  / 133
//   200,003   x 8,192                    - /  47-109  / 151
//   300,000   x 1,024                  231 / 140-2705 / 186
//   1,000,000 x 256                    189 / 211-1180 / 283
//   1,000,000 x 65,536                   - / 1858-5882 / 532
//   2,000,000 x 256                    349 / 178-1294 / 314
// The scan costs 0.7 ps per pair (all of 2,048 points for every block), the sorts
// and boxes 30 to 300 us.  The tree's boxes are the caller's order: up to 4,096
// points two levels of them bound any order's cost; past that it is up to four
// times as fast as the sorted search on good orders and 45 times as slow on
// bad ones (100,000 points in no order x 4,096: 5.0 ms against 0.11), so it is left.
NNRoute nn_route(uint32_t num_points, uint32_t num_queries) {
    if (num_points <= 64) return NNRoute::kTree; // one group of points
    if (num_points <= 2048) return num_queries <= 65536 ? NNRoute::kScan : NNRoute::kSorted;
    if (num_points <= 4096) return num_queries <= 2048 ? NNRoute::kScan : NNRoute::kTree;
    const uint64_t pairs = (uint64_t)num_points * num_queries;
    return pairs <= (1ull << 27) + std::min<uint64_t>(256ull * num_points, 1ull << 28)
               ? NNRoute::kScan
               : NNRoute::kSorted;
}

size_t nn_scratch_bytes(uint32_t num_points, uint32_t num_queries) {
    switch (nn_route(num_points, num_queries)) {
    case NNRoute::kScan: return align256(8ull * std::max(num_queries, 1u));
    case NNRoute::kTree: return 0;
    default: return layout_of(num_points, num_queries).bytes;
    }
}

hipError_t launch_nn_sorted(const float *points, const float *tree, const float *queries,
                            uint32_t num_points, uint32_t num_queries, uint32_t *indices,
                            void *scratch, hipStream_t stream) {
    const Layout l = layout_of(num_points, num_queries);
    if (l.bytes == 0) return hipErrorInvalidValue;
    const Levels lv = levels_of(num_points);
    char *base = static_cast<char *>(scratch);
    uint32_t *order = reinterpret_cast<uint32_t *>(base + l.order);
    uint32_t *qorder = reinterpret_cast<uint32_t *>(base + l.queries);
    float4 *sorted = reinterpret_cast<float4 *>(base + l.sorted);
    float4 *boxes = reinterpret_cast<float4 *>(base + l.boxes);
    // the root box of a tree over 2^td points is its node 2^td - 2
    uint64_t n2 = 1;
    while (n2 < num_points) n2 <<= 1;
    const float *root = tree + 6ull * (n2 - 2);
    hipError_t e = sort_positions(points, num_points, root, base, l, order, stream);
    if (e != hipSuccess) return e;
    e = sort_positions(queries, num_queries, root, base, l, qorder, stream);
    if (e != hipSuccess) return e;
    auto grid = [](uint64_t threads) { return dim3((uint32_t)((threads + kBlock - 1) / kBlock)); };
    hipLaunchKernelGGL(gather_kernel, grid(num_points), dim3(kBlock), 0, stream, points, order,
                       num_points, sorted, boxes);
    for (int k = 1; k < lv.count; ++k)
        hipLaunchKernelGGL(level_kernel, grid(lv.width[k - 1]), dim3(kBlock), 0, stream, boxes,
                           lv.start[k - 1], lv.width[k - 1], lv.start[k]);
    Search s = {};
    s.sorted = sorted;
    s.boxes = boxes;
    s.n = num_points;
    for (int k = 0; k < lv.count; ++k) {
        s.start[k] = lv.start[k];
        s.width[k] = lv.width[k];
    }
    const uint32_t run = (num_queries + kSearchWaves - 1) / kSearchWaves;
    const dim3 waves = grid(((uint64_t)num_queries + run - 1) / run * 64);
    switch (lv.count) {
#define SDF_SEARCH(N)                                                                           \
    case N:                                                                                     \
        hipLaunchKernelGGL(search_kernel<N>, waves, dim3(kBlock), 0, stream, s, queries, qorder, \
                           num_queries, run, points, indices);                                   \
        break
        SDF_SEARCH(1);
        SDF_SEARCH(2);
        SDF_SEARCH(3);
        SDF_SEARCH(4);
        SDF_SEARCH(5);
#undef SDF_SEARCH
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

} // namespace sdfoam_hip
