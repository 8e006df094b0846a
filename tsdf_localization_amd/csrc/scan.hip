// Scan preparation on the device: spatial ordering of the points and the
// per-point score constant.
//
// The evaluation kernel gives each wavefront 64 consecutive points.  Points
// kept in the reference's ring order spread over metres of wall, so one
// wavefront's voxel gathers touch ~60 distinct cache lines; sorted by the
// Morton code of their scanner-frame position (0.25 m cells) they cluster,
// and every particle's rigid transform keeps them clustered.  The order of
// the points only changes the float summation order of the weights (the
// voxel index of every (particle, point) pair is unchanged); perm[j] keeps
// the caller's index of sorted point j for the index trace.
#include <hipcub/hipcub.hpp>

#include "tsl_internal.h"

#include <algorithm>

namespace tsl {

namespace {

// particle-order buckets: kXyBits bits for each of x and y, kYawBits for
// the heading
#ifndef TSL_ORDER_XY_BITS
#define TSL_ORDER_XY_BITS 6
#endif
#ifndef TSL_ORDER_YAW_BITS
#define TSL_ORDER_YAW_BITS 5
#endif
constexpr uint32_t kXyBits = TSL_ORDER_XY_BITS;
constexpr uint32_t kYawBits = TSL_ORDER_YAW_BITS;
constexpr uint32_t kBuckets = 1u << (2 * kXyBits + kYawBits);

__device__ __forceinline__ uint64_t spread3(uint64_t v)
{
    v &= 0x1fffffull;
    v = (v | (v << 32)) & 0x1f00000000ffffull;
    v = (v | (v << 16)) & 0x1f0000ff0000ffull;
    v = (v | (v << 8)) & 0x100f00f00f00f00full;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}

__device__ __forceinline__ uint64_t cell_coord(float x)
{
    // 0.25 m cells, offset so that +-262 km maps into 21 bits; NaN -> 0
    float c = floorf(x * 4.0f) + 1048576.0f;
    c = c > 0.0f ? c : 0.0f;
    c = c < 2097151.0f ? c : 2097151.0f;
    return (uint64_t)c;
}

__device__ __forceinline__ uint64_t morton_key(const tsl_point& p)
{
    return spread3(cell_coord(p.x)) | (spread3(cell_coord(p.y)) << 1) | (spread3(cell_coord(p.z)) << 2);
}

__global__ void k_morton(const tsl_point* __restrict__ in, uint32_t n, uint64_t* __restrict__ keys,
                         uint32_t* __restrict__ vals)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    keys[i] = morton_key(in[i]);
    vals[i] = i;
}

// A point with its constant score term (tsdf_evaluator.cpp:56-65): |p|^2
// evaluated as the reference does.  mark: NaN instead for points that the
// class-grid kernels leave to the exact tiers.
__device__ __forceinline__ float4 scored_point(const tsl_point& p, const ScoreTerm& sc, int mark)
{
    const float d2 = p.x * p.x + p.y * p.y + p.z * p.z;
    float w = d2 < sc.max_range_squared ? sc.range_term : sc.a_max;
    if (mark && !(fabsf(p.x) < kTamePoint && fabsf(p.y) < kTamePoint && fabsf(p.z) < kTamePoint)) w = __builtin_nanf("");
    return make_float4(p.x, p.y, p.z, w);
}

// Sorted point j = input point perm[j].
__global__ void k_prep_sorted(const tsl_point* __restrict__ in, const uint32_t* __restrict__ perm, uint32_t n,
                              ScoreTerm sc, int mark, float4* __restrict__ out)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    out[j] = scored_point(in[perm[j]], sc, mark);
}

// Scans of up to kMergePoints points are sorted in two launches, with the key
// and the score term formed in them: tiles of 256 points by a bitonic network,
// then every point's place from its rank in its own tile and a binary search in
// each of the others (ties in tile order, which is the caller's), staged in LDS
// 8192 keys at a time.  The time is latency: 9 us of kernels at 701 points, 13
// at 2056, 18 at 10,000, where key, radix sort and gather kernels took 24, 27
// and 42 (their merge passes are launches of 5 us each).  The searches grow with
// the square of the points: a whole call that sets a scan is 44 us against 75 at
// 10,000 points, 92 against 116 at 65,536, and the two meet near 100,000.
constexpr uint32_t kSortTile = 256;
constexpr uint32_t kMergeKeys = 8192;  // 64 KB of LDS
constexpr uint32_t kMergePoints = 65536;

// One tile per workgroup: its sorted keys (padded to a whole tile) and caller
// indices.
__global__ __launch_bounds__(kSortTile) void k_sort_tile(const tsl_point* __restrict__ in, uint32_t n,
                                                         uint64_t* __restrict__ keys, uint32_t* __restrict__ vals)
{
    __shared__ uint64_t other_key[kSortTile];
    __shared__ uint32_t other_idx[kSortTile];
    const uint32_t t = threadIdx.x, at = blockIdx.x * kSortTile + t;
    uint64_t key = at < n ? morton_key(in[at]) : ~0ull;  // (keys have 63 bits: the padding comes last)
    uint32_t idx = at;
#pragma unroll
    for (uint32_t k = 2; k <= kSortTile; k <<= 1) {
#pragma unroll
        for (uint32_t j = k >> 1; j; j >>= 1) {
            uint64_t ok;
            uint32_t oi;
            if (j >= 64) {
                __syncthreads();  // the previous exchange has been read
                other_key[t] = key;
                other_idx[t] = idx;
                __syncthreads();
                ok = other_key[t ^ j];
                oi = other_idx[t ^ j];
            } else {
                ok = __shfl_xor((unsigned long long)key, (int)j, 64);
                oi = __shfl_xor(idx, (int)j, 64);
            }
            const bool less = key < ok || (key == ok && idx < oi);
            const bool keep_less = ((t & k) == 0) == ((t & j) == 0);
            if (less != keep_less) {
                key = ok;
                idx = oi;
            }
        }
    }
    if (at < n || gridDim.x > 1) keys[at] = key;  // (2n keys hold two or more whole tiles)
    if (at < n) vals[at] = idx;
}

// A point comes after the keys up to its own in an earlier tile and below its
// own in a later one.
constexpr uint32_t kSearches = 8;     // tiles searched at a time
constexpr uint32_t kMergeGroups = 4;  // groups of threads per tile, each with a share of the searches
__global__ __launch_bounds__(kSortTile * kMergeGroups) void k_merge_tiles(
    const tsl_point* __restrict__ in, uint32_t n, ScoreTerm sc, int mark, const uint64_t* __restrict__ keys,
    const uint32_t* __restrict__ vals, uint32_t* __restrict__ perm, float4* __restrict__ out)
{
    __shared__ uint64_t staged[kMergeKeys];
    const uint32_t t = threadIdx.x % kSortTile, group = threadIdx.x / kSortTile;
    const uint32_t own = blockIdx.x, tiles = gridDim.x, at = own * kSortTile + t;
    const uint64_t key = at < n ? keys[at] : ~0ull;
    const uint32_t idx = at < n ? vals[at] : 0u;
    const tsl_point p = in[idx];
    uint32_t before = 0;
    for (uint32_t t0 = 0; tiles > 1 && t0 < tiles; t0 += kMergeKeys / kSortTile) {
        const uint32_t here = min(tiles - t0, kMergeKeys / kSortTile);
        if (t0) __syncthreads();
        const uint4* src = reinterpret_cast<const uint4*>(keys + t0 * kSortTile);
        uint4* dst = reinterpret_cast<uint4*>(staged);
#pragma unroll 4
        for (uint32_t i = threadIdx.x; i < here * (kSortTile / 2); i += kSortTile * kMergeGroups) dst[i] = src[i];
        __syncthreads();
        for (uint32_t s0 = group; s0 < here; s0 += kSearches * kMergeGroups) {
            uint32_t pos[kSearches];
            uint64_t bound[kSearches];
#pragma unroll
            for (uint32_t q = 0; q < kSearches; ++q) {
                const uint32_t tile = s0 + q * kMergeGroups;
                pos[q] = min(tile, here - 1) * kSortTile;
                bound[q] = key + (t0 + tile < own ? 1u : 0u);
            }
#pragma unroll
            for (uint32_t step = kSortTile / 2; step; step >>= 1) {
#pragma unroll
                for (uint32_t q = 0; q < kSearches; ++q) pos[q] += staged[pos[q] + step - 1] < bound[q] ? step : 0u;
            }
#pragma unroll
            for (uint32_t q = 0; q < kSearches; ++q) {
                const uint32_t tile = s0 + q * kMergeGroups;
                pos[q] += staged[pos[q]] < bound[q] ? 1u : 0u;
                if (tile < here && t0 + tile != own) before += pos[q] - tile * kSortTile;
            }
        }
    }
    __syncthreads();
    uint32_t* parts = reinterpret_cast<uint32_t*>(staged);
    if (group) parts[group * kSortTile + t] = before;
    __syncthreads();
    if (group || at >= n) return;
    uint32_t place = t + before;
#pragma unroll
    for (uint32_t g = 1; g < kMergeGroups; ++g) place += parts[g * kSortTile + t];
    perm[place] = idx;
    out[place] = scored_point(p, sc, mark);
}

// Evaluation order of the particles: a counting sort into Morton-ordered
// buckets of (x, y) cells over the map and yaw sectors.  Particles close in
// position and heading transform the scan onto nearly the same voxels, so
// evaluating them together on one XCD turns most of their voxel gathers
// into L2 hits; the thousands of particles an XCD has in flight at once
// span many buckets, so the order inside a bucket (arrival order of the
// scatter's atomics) does not matter, and no particle's weight depends on
// its slot.
struct BucketGrid {
    float min_x, min_y, inv_x, inv_y, inv_yaw;
};

__device__ __forceinline__ uint32_t bucket_coord(float v, float inv_cell, uint32_t cells)
{
    float c = floorf(v * inv_cell);
    c = c > 0.0f ? c : 0.0f;  // NaN -> 0
    const float top = (float)(cells - 1);
    c = c < top ? c : top;
    return (uint32_t)c;
}

// Morton key: from the lowest bit up, bit k of x, of y (k < kXyBits) and of
// the heading sector (k < kYawBits)
__device__ __forceinline__ uint32_t bucket_of(const tsl_particle& p, const BucketGrid& g)
{
    const uint32_t x = bucket_coord(p.first[0] - g.min_x, g.inv_x, 1u << kXyBits);
    const uint32_t y = bucket_coord(p.first[1] - g.min_y, g.inv_y, 1u << kXyBits);
    const uint32_t a = bucket_coord(p.first[5] + 3.14159265f, g.inv_yaw, 1u << kYawBits);
    uint32_t key = 0, pos = 0;
#pragma unroll
    for (uint32_t k = 0; k < (kXyBits > kYawBits ? kXyBits : kYawBits); ++k) {
        if (k < kXyBits) {
            key |= ((x >> k) & 1u) << pos++;
            key |= ((y >> k) & 1u) << pos++;
        }
        if (k < kYawBits) key |= ((a >> k) & 1u) << pos++;
    }
    return key;
}

__global__ void k_bucket_zero(uint32_t* __restrict__ hist)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kBuckets) hist[i] = 0u;
}

// hist[key] += the number of active lanes with that key, one atomic per
// distinct key of the wavefront (the particles of a tracking filter share a
// few buckets, and per-lane atomics on one counter serialise); returns the
// counter's old value plus the lane's rank among the lanes with its key.
// The lanes are grouped by key first (ballots only), then every group's
// first lane adds its group's size in one atomic instruction for all
// groups, so the wavefront waits for one atomic round trip however many
// keys it holds.  Every lane of the wavefront calls it.
__device__ __forceinline__ uint32_t wave_bucket_add(uint32_t* __restrict__ hist, uint32_t key, bool active)
{
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1ull;
    uint64_t pending = __ballot(active);
    uint32_t leader_of = lane, rank = 0, group = 0;
    while (pending) {
        const int leader = __ffsll((unsigned long long)pending) - 1;  // wavefront-uniform
        const uint32_t lk = __builtin_amdgcn_readlane(key, leader);
        const uint64_t same = __ballot(active && key == lk);
        if (active && key == lk) {
            leader_of = (uint32_t)leader;
            rank = (uint32_t)__popcll(same & below);
            group = (uint32_t)__popcll(same);
        }
        pending &= ~same;
    }
    uint32_t base = 0;
    if (active && leader_of == lane) base = atomicAdd(&hist[key], group);
    base = __shfl(base, (int)leader_of, 64);
    return base + rank;
}

__global__ void k_bucket_count(const tsl_particle* __restrict__ in, const uint32_t* __restrict__ count,
                               BucketGrid g, uint32_t* __restrict__ hist, uint32_t* __restrict__ bucket)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = i < *count;
    uint32_t k = 0;
    if (active) {
        k = bucket_of(in[i], g);
        bucket[i] = k;
    }
    (void)wave_bucket_add(hist, k, active);
}

__global__ void k_bucket_scatter(const uint32_t* __restrict__ count, const uint32_t* __restrict__ bucket,
                                 uint32_t* __restrict__ hist, uint32_t* __restrict__ order)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = i < *count;
    const uint32_t k = active ? bucket[i] : 0u;
    const uint32_t pos = wave_bucket_add(hist, k, active);
    if (active) order[pos] = i;
}

}  // namespace

// Layout of f->pkeys: bucket counts, bucket offsets (their exclusive scan),
// the bucket of each particle, the scan's temporary storage; each part
// 256-byte aligned.
static size_t round256(size_t b) { return (b + 255) / 256 * 256; }

static int bucket_scan_temp_bytes(size_t* bytes)
{
    static size_t t = 0;
    static bool known = false;
    if (!known) {
        TSL_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, t, (uint32_t*)nullptr, (uint32_t*)nullptr,
                                                       (int)kBuckets, (hipStream_t)0));
        known = true;
    }
    *bytes = t;
    return TSL_OK;
}

int particle_order_keys_bytes(size_t n, size_t* bytes)
{
    size_t temp = 0;
    TSL_TRY(bucket_scan_temp_bytes(&temp));
    *bytes = 2 * round256(sizeof(uint32_t) * kBuckets) + round256(sizeof(uint32_t) * n) + round256(temp);
    return TSL_OK;
}

int reserve_particle_order(tsl_filter* f)
{
    const size_t n = f->count_bound;
    size_t keys = 0;
    TSL_TRY(particle_order_keys_bytes(n, &keys));
    TSL_TRY(f->pkeys.reserve(keys));
    TSL_TRY(f->porder.reserve(sizeof(uint32_t) * n));
    return f->pinv.reserve(sizeof(uint32_t) * n);
}

int launch_particle_order(tsl_filter* f, hipStream_t stream)
{
    const uint32_t n = (uint32_t)f->count_bound;
    if (n == 0) return TSL_OK;
    TSL_TRY(reserve_particle_order(f));
    size_t temp = 0;
    TSL_TRY(bucket_scan_temp_bytes(&temp));
    char* at = f->pkeys.as<char>();
    uint32_t* hist = reinterpret_cast<uint32_t*>(at);
    at += round256(sizeof(uint32_t) * kBuckets);
    uint32_t* offsets = reinterpret_cast<uint32_t*>(at);
    at += round256(sizeof(uint32_t) * kBuckets);
    uint32_t* bucket = reinterpret_cast<uint32_t*>(at);
    at += round256(sizeof(uint32_t) * n);
    void* scan_temp = at;
    const uint32_t* count = &f->state.as<FilterState>()->count;
    // x and y cells spanning the map's extent (at least 0.5 m), yaw sectors
    // spanning [-pi, pi)
    const tsl_map_coef& c = f->ev->map->coef;
    const float cells = (float)(1u << kXyBits);
    BucketGrid g;
    g.min_x = c.min_x;
    g.min_y = c.min_y;
    g.inv_x = 1.0f / std::max(0.5f, (c.max_x - c.min_x) / cells);
    g.inv_y = 1.0f / std::max(0.5f, (c.max_y - c.min_y) / cells);
    g.inv_yaw = (float)(1u << kYawBits) / 6.2831853f;
    hipLaunchKernelGGL(k_bucket_zero, dim3(kBuckets / 256), dim3(256), 0, stream, hist);
    TSL_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_bucket_count, dim3((n + 255) / 256), dim3(256), 0, stream, f->particles.as<tsl_particle>(),
                       count, g, hist, bucket);
    TSL_HIP_CHECK(hipGetLastError());
    size_t tb = temp;
    TSL_HIP_CHECK(hipcub::DeviceScan::ExclusiveSum(scan_temp, tb, hist, offsets, (int)kBuckets, stream));
    hipLaunchKernelGGL(k_bucket_scatter, dim3((n + 255) / 256), dim3(256), 0, stream, count, bucket, offsets,
                       f->porder.as<uint32_t>());
    TSL_HIP_CHECK(hipGetLastError());
    return TSL_OK;
}

// Reserve every buffer the scan preparation of up to n points uses, so that
// later preparations allocate nothing (and never synchronise).
int filter_reserve_scan(tsl_filter* f, size_t n)
{
    if (n == 0) n = 1;
    TSL_TRY(filter_reserve_points(f, n));
    TSL_TRY(f->sort_keys.reserve(sizeof(uint64_t) * 2 * n));
    TSL_TRY(f->sort_vals.reserve(sizeof(uint32_t) * n));
    TSL_TRY(f->perm.reserve(sizeof(uint32_t) * n));
    size_t temp = 0;
    uint64_t* keys = f->sort_keys.as<uint64_t>();
    TSL_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, temp, keys, keys + n, f->sort_vals.as<uint32_t>(),
                                                     f->perm.as<uint32_t>(), (int)n, 0, 63, (hipStream_t)0));
    TSL_TRY(f->sort_temp.reserve(temp));
    return TSL_OK;
}

size_t prep_points_temp_bytes(uint32_t n)
{
    size_t temp = 0;
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, temp, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                             (uint32_t*)nullptr, (uint32_t*)nullptr, (int)n, 0, 63, (hipStream_t)0);
    return temp;
}

int launch_prep_points(tsl_filter* f, hipStream_t stream)
{
    const uint32_t n = (uint32_t)f->num_points;
    if (n == 0) return TSL_OK;
    TSL_TRY(f->sort_keys.reserve(sizeof(uint64_t) * 2 * n));
    TSL_TRY(f->sort_vals.reserve(sizeof(uint32_t) * n));
    TSL_TRY(f->perm.reserve(sizeof(uint32_t) * n));
    uint64_t* keys = f->sort_keys.as<uint64_t>();
    uint32_t* vals = f->sort_vals.as<uint32_t>();
    const tsl_evaluator* ev = f->ev;
    if (n <= kMergePoints) {
        const uint32_t tiles = (n + kSortTile - 1) / kSortTile;
        hipLaunchKernelGGL(k_sort_tile, dim3(tiles), dim3(kSortTile), 0, stream, f->points_in.as<tsl_point>(), n, keys,
                           vals);
        TSL_HIP_CHECK(hipGetLastError());
        hipLaunchKernelGGL(k_merge_tiles, dim3(tiles), dim3(kSortTile * kMergeGroups), 0, stream, f->points_in.as<tsl_point>(), n,
                           score_term_of(ev), (int)ev->map->grid.ready, keys, vals, f->perm.as<uint32_t>(),
                           f->points.as<float4>());
        TSL_HIP_CHECK(hipGetLastError());
        return TSL_OK;
    }
    size_t temp = 0;
    TSL_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, temp, keys, keys + n, vals, f->perm.as<uint32_t>(),
                                                     (int)n, 0, 63, stream));
    TSL_TRY(f->sort_temp.reserve(temp));
    const unsigned g = (n + 255) / 256;
    hipLaunchKernelGGL(k_morton, dim3(g), dim3(256), 0, stream, f->points_in.as<tsl_point>(), n, keys, vals);
    TSL_HIP_CHECK(hipGetLastError());
    TSL_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(f->sort_temp.ptr, temp, keys, keys + n, vals,
                                                     f->perm.as<uint32_t>(), (int)n, 0, 63, stream));
    hipLaunchKernelGGL(k_prep_sorted, dim3(g), dim3(256), 0, stream, f->points_in.as<tsl_point>(),
                       f->perm.as<uint32_t>(), n, score_term_of(ev), (int)ev->map->grid.ready, f->points.as<float4>());
    TSL_HIP_CHECK(hipGetLastError());
    return TSL_OK;
}

namespace {

// Sorted position i of scan blockIdx.y: the point and its score constant,
// as k_prep_sorted writes them for one filter.
__global__ void k_prep_sorted_seg(const tsl_point* __restrict__ in, const uint32_t* __restrict__ off,
                                  const uint32_t* __restrict__ sorted_idx, ScoreTerm sc, int mark,
                                  const ScanDest* __restrict__ dst)
{
    const uint32_t r = blockIdx.y;
    const uint32_t b = off[r], n = off[r + 1] - b;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t src = sorted_idx[b + i];
    dst[r].points[i] = scored_point(in[src], sc, mark);
    dst[r].perm[i] = src - b;
}

}  // namespace

size_t prep_points_batch_temp(uint32_t total, uint32_t n)
{
    size_t t1 = 0, t2 = 0;
    if (total == 0 || n == 0) return 0;
    if (hipcub::DeviceRadixSort::SortPairs(nullptr, t1, (uint64_t*)nullptr, (uint64_t*)nullptr, (uint32_t*)nullptr,
                                           (uint32_t*)nullptr, (int)total, 0, 63, (hipStream_t)0) != hipSuccess ||
        hipcub::DeviceRadixSort::SortPairs(nullptr, t2, (uint32_t*)nullptr, (uint32_t*)nullptr, (uint32_t*)nullptr,
                                           (uint32_t*)nullptr, (int)total, 0, 32, (hipStream_t)0) != hipSuccess)
        return 0;
    return std::max(t1, t2);
}

// Sorted position t: the scan (segment of off) that point order[t] belongs
// to (the last r with off[r] <= order[t]; empty scans own no point).
__global__ void k_seg_keys(const uint32_t* __restrict__ off, uint32_t n, const uint32_t* __restrict__ order,
                           uint32_t total, uint32_t* __restrict__ seg)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const uint32_t idx = order[t];
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (off[mid] <= idx) lo = mid; else hi = mid;
    }
    seg[t] = lo;
}

// Every scan of a tick prepared at once: one device-wide stable sort of all
// points by Morton key, then a stable sort by scan.  Within a scan the order
// is by key, ties in point order: the order the per-scan sort gives.
int launch_prep_points_batch(const tsl_evaluator* ev, const tsl_point* pts, const uint32_t* off, const ScanDest* dst,
                             uint32_t n, uint32_t total, uint32_t max_count, uint64_t* keys, uint32_t* vals,
                             void* temp, size_t temp_bytes, hipStream_t stream)
{
    if (n == 0 || total == 0) return TSL_OK;
    const unsigned g = (total + 255) / 256;
    hipLaunchKernelGGL(k_morton, dim3(g), dim3(256), 0, stream, pts, total, keys, vals);
    TSL_HIP_CHECK(hipGetLastError());
    TSL_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(temp, temp_bytes, keys, keys + total, vals, vals + total,
                                                     (int)total, 0, 63, stream));
    // the keys' first half is free again: scan numbers, in and out
    uint32_t* seg = reinterpret_cast<uint32_t*>(keys);
    hipLaunchKernelGGL(k_seg_keys, dim3(g), dim3(256), 0, stream, off, n, vals + total, total, seg);
    TSL_HIP_CHECK(hipGetLastError());
    int bits = 1;
    while ((1u << bits) < n) ++bits;
    TSL_HIP_CHECK(hipcub::DeviceRadixSort::SortPairs(temp, temp_bytes, seg, seg + total, vals + total, vals,
                                                     (int)total, 0, bits, stream));
    hipLaunchKernelGGL(k_prep_sorted_seg, dim3((max_count + 255) / 256, n), dim3(256), 0, stream, pts, off, vals,
                       score_term_of(ev), (int)ev->map->grid.ready, dst);
    TSL_HIP_CHECK(hipGetLastError());
    return TSL_OK;
}

}  // namespace tsl
