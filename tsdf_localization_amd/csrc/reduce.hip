// Scan reduction on the device (TSDFEvaluator::evaluateParticles,
// src/evaluation/tsdf_evaluator.cpp:304-376; CudaEvaluator::evaluate of a
// PointCloud2, src/cuda/cuda_evaluator.cu:78-116): of the points that share a
// reduction cell (and, in the former, a ring) the first stays, and the points
// that stay are ordered by (ring, index).
//
// The first point of every cell comes from an open-addressing hash table of
// entry indices (compare-and-swap into an empty slot, minimum into a slot of
// the same cell), the order from one stable counting pass over 8-bit rings:
// five launches, each a pass over the points, where sorting by cell takes two
// 64-bit sorts and by ring a third.  A 64-beam scan of 250,001 points: 37 us of
// kernels where the sorts took about 300; a 16-beam cloud of 16,384: 28 us
// against about 125.  What bounds them is latency: the insertion's chain of
// table, compare-and-swap and key accesses is 11 us at either size.
#include "tsl_internal.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>

namespace tsl {

namespace {

constexpr uint32_t kRedThreads = 1024, kRedWaves = kRedThreads / 64;
// Workgroups of the ordered passes: each owns one contiguous range of the
// points, and every one of them sums the others' 256 ring counts.
constexpr uint32_t kRedBlocks = 256;
constexpr uint32_t kRedEmpty = 0xffffffffu;  // table: no entry; slot: wins
constexpr uint32_t kRedLoses = 0xfffffffeu;  // slot: a lower entry has the cell

struct RedArgs {
    const tsl_point* raw;
    const void* ring;     // int16 (evaluator) or int32 (cloud), by entry
    uint32_t n, per;      // points; points of a workgroup's range (a multiple of kRedThreads)
    int mode;
    float cell, half;
    uint4* key;           // by entry: x, y, z centre bits, ring in its order
    tsl_point* orig;      // by entry: the point that is written out
    uint32_t* table;      // [mask + 1] entry index or kRedEmpty
    uint32_t* slot;       // by entry: its cell's slot, kRedEmpty or kRedLoses
    uint32_t mask;
    uint32_t* kept;       // [kRedBlocks] kept points of each range
    uint32_t* hist;       // [kRedBlocks][256] winners of each range of entries by ring
    uint32_t* counters;   // reduced points, a ring outside [0, 64), rings of more than 8 bits
};

// The reference skips points closer than 1 m (sqrtf, tsdf_evaluator.cpp:
// 316-322); the cloud reduction keeps every point (cuda_evaluator.cu:84-91).
__device__ __forceinline__ bool red_keep(const RedArgs& a, uint32_t j)
{
    if (a.mode == kReduceCloud) return true;
    const tsl_point p = a.raw[j];
    const float dist = sqrtf(p.x * p.x + p.y * p.y + p.z * p.z);
    return !(dist < 1.0f);
}

// Sum of v over the workgroup, in every thread.
__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t* sh /* kRedWaves */)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t t = 0;
#pragma unroll
    for (uint32_t w = 0; w < kRedWaves; ++w) t += sh[w];
    return t;
}

// Kept points of each range; the table and the counters are cleared.
__global__ __launch_bounds__(kRedThreads) void k_red_count(RedArgs a)
{
    __shared__ uint32_t sh[kRedWaves];
    const uint32_t b = blockIdx.x;
    if (b == 0 && threadIdx.x < 3) a.counters[threadIdx.x] = 0;
    const uint4 empty = make_uint4(kRedEmpty, kRedEmpty, kRedEmpty, kRedEmpty);
    for (uint64_t i = (uint64_t)b * kRedThreads + threadIdx.x; i < ((uint64_t)a.mask + 1) / 4;
         i += (uint64_t)gridDim.x * kRedThreads)
        reinterpret_cast<uint4*>(a.table)[i] = empty;
    const uint64_t end = min((uint64_t)a.n, (uint64_t)(b + 1) * a.per);
    uint32_t c = 0;
    for (uint64_t j = (uint64_t)b * a.per + threadIdx.x; j < end; j += kRedThreads) c += red_keep(a, (uint32_t)j);
    c = block_sum(c, sh);
    if (threadIdx.x == 0) a.kept[b] = c;
}

// Kept point j becomes entry k (its index in the reference): k counts the
// kept points before it, and reads ring[k] because the reference's ring
// iterator only advances on kept points (tsdf_evaluator.cpp:319-331).  Cloud
// mode: rings are int32 (the reference reads the field as int) and used for
// the order only, the centre is computed in double with the literal 0.064 m
// cell (cuda_evaluator.cu:95-97), and the centre itself is the reduced point.
__global__ __launch_bounds__(kRedThreads) void k_red_build(RedArgs a)
{
    __shared__ uint32_t sh[kRedWaves], wave_kept[kRedWaves];
    const uint32_t b = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t base = block_sum(threadIdx.x < b ? a.kept[threadIdx.x] : 0u, sh);
    const uint64_t end = min((uint64_t)a.n, (uint64_t)(b + 1) * a.per);
    for (uint64_t t = (uint64_t)b * a.per; t < end; t += kRedThreads) {
        const uint32_t j = (uint32_t)(t + threadIdx.x);
        const bool keep = t + threadIdx.x < end && red_keep(a, j);
        const uint64_t kept = __ballot(keep);
        __syncthreads();
        if (lane == 0) wave_kept[wave] = (uint32_t)__popcll(kept);
        __syncthreads();
        uint32_t before = 0, all = 0;
#pragma unroll
        for (uint32_t w = 0; w < kRedWaves; ++w) {
            before += w < wave ? wave_kept[w] : 0u;
            all += wave_kept[w];
        }
        const uint32_t k = base + before + (uint32_t)__popcll(kept & ((1ull << lane) - 1ull));
        base += all;
        if (!keep) continue;
        const tsl_point p = a.raw[j];
        uint4 key;
        tsl_point o = p;
        if (a.mode == kReduceCloud) {
            const int32_t* ring = static_cast<const int32_t*>(a.ring);
            const double c = 0.064, h = 0.032;
            o.x = (float)(floor((double)p.x / c) * c + h);
            o.y = (float)(floor((double)p.y / c) * c + h);
            o.z = (float)(floor((double)p.z / c) * c + h);
            key = make_uint4(__float_as_uint(o.x), __float_as_uint(o.y), __float_as_uint(o.z),
                             (uint32_t)ring[k] ^ 0x80000000u);  // signed order
            if ((ring[k] ^ ring[0]) & ~0xff) atomicOr(&a.counters[2], 1u);
        } else {
            const int r = static_cast<const int16_t*>(a.ring)[k];
            if (r < 0 || r >= 64) atomicOr(&a.counters[1], 1u);
            key = make_uint4(__float_as_uint(floorf(p.x / a.cell) * a.cell + a.half),
                             __float_as_uint(floorf(p.y / a.cell) * a.cell + a.half),
                             __float_as_uint(floorf(p.z / a.cell) * a.cell + a.half), (uint32_t)(r & 0xff));
        }
        a.key[k] = key;
        a.orig[k] = o;
    }
}

__device__ __forceinline__ uint32_t red_entries(const RedArgs& a, uint32_t blocks, uint32_t* sh)
{
    return block_sum(threadIdx.x < blocks ? a.kept[threadIdx.x] : 0u, sh);
}

__device__ __forceinline__ bool red_nan(const uint4& k)
{
    const float x = __uint_as_float(k.x), y = __uint_as_float(k.y), z = __uint_as_float(k.z);
    return (x != x) | (y != y) | (z != z);
}

// Same cell (and, in the evaluator's reduction, same ring).
__device__ __forceinline__ bool red_same(const RedArgs& a, const uint4& p, const uint4& q)
{
    return p.x == q.x && p.y == q.y && p.z == q.z && (a.mode == kReduceCloud || p.w == q.w);
}

// Every entry finds or takes its cell's slot and leaves the lowest entry
// there; an entry in the cell of the one before it, as most of a dense scan's
// are, has lost already.  A slot keeps its cell once taken, and there are more
// slots than entries, so the probing ends.  The plain loads may be stale (an
// empty slot is then seen by the compare-and-swap, a higher entry by the
// minimum); where many points share a cell they spare most of them the atomic.
__global__ __launch_bounds__(kRedThreads) void k_red_insert(RedArgs a, uint32_t blocks)
{
    __shared__ uint32_t sh[kRedWaves];
    const uint32_t entries = red_entries(a, blocks, sh);
    const uint64_t step = (uint64_t)gridDim.x * kRedThreads;
    for (uint64_t e64 = (uint64_t)blockIdx.x * kRedThreads + threadIdx.x; e64 < entries; e64 += step) {
        const uint32_t e = (uint32_t)e64;
        const uint4 key = a.key[e];
        if (red_nan(key)) {  // NaN centres match nothing
            a.slot[e] = kRedEmpty;
            continue;
        }
        if (e && red_same(a, key, a.key[e - 1])) {
            a.slot[e] = kRedLoses;
            continue;
        }
        const uint32_t ring = a.mode == kReduceCloud ? 0u : key.w;
        uint32_t h = key.x * 0x9e3779b1u ^ key.y * 0x85ebca77u ^ key.z * 0xc2b2ae3du ^ ring * 0x27d4eb2fu;
        h ^= h >> 15;
        h *= 0x2c1b3c6du;
        h ^= h >> 13;
        uint32_t i = h & a.mask;
        for (;; i = (i + 1) & a.mask) {
            uint32_t cur = *static_cast<volatile const uint32_t*>(&a.table[i]);
            if (cur == kRedEmpty) {
                cur = atomicCAS(&a.table[i], kRedEmpty, e);
                if (cur == kRedEmpty) break;
            }
            if (red_same(a, key, a.key[cur])) {
                if (cur > e) atomicMin(&a.table[i], e);
                break;
            }
        }
        a.slot[e] = i;
    }
}

__device__ __forceinline__ bool red_wins(const RedArgs& a, uint32_t e)
{
    const uint32_t s = a.slot[e];
    return s == kRedEmpty || (s != kRedLoses && a.table[s] == e);
}

// Winners of each range of entries by the ring's low 8 bits.
__global__ __launch_bounds__(kRedThreads) void k_red_mark(RedArgs a)
{
    __shared__ uint32_t sh[kRedWaves], count[256];
    if (threadIdx.x < 256) count[threadIdx.x] = 0;
    const uint32_t b = blockIdx.x;
    const uint32_t entries = red_entries(a, gridDim.x, sh);
    const uint64_t end = min((uint64_t)entries, (uint64_t)(b + 1) * a.per);
    for (uint64_t e = (uint64_t)b * a.per + threadIdx.x; e < end; e += kRedThreads)
        if (red_wins(a, (uint32_t)e)) atomicAdd(&count[a.key[e].w & 0xffu], 1u);
    __syncthreads();
    if (threadIdx.x < 256) a.hist[b * 256 + threadIdx.x] = count[threadIdx.x];
}

// Winners to their places: rings ascending, within a ring by entry.
__global__ __launch_bounds__(kRedThreads) void k_red_scatter(RedArgs a, tsl_point* __restrict__ out)
{
    __shared__ uint32_t sh[kRedWaves], place[256], part[2][4][256], of_wave[kRedWaves][256];
    const uint32_t b = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t entries = red_entries(a, gridDim.x, sh);
    {
        // winners of a ring in the ranges before this one, and in all
        const uint32_t d = threadIdx.x & 255, g = threadIdx.x >> 8;
        uint32_t before = 0, all = 0;
#pragma unroll 8
        for (uint32_t r = g; r < gridDim.x; r += 4) {
            const uint32_t c = a.hist[r * 256 + d];
            before += r < b ? c : 0u;
            all += c;
        }
        part[0][g][d] = before;
        part[1][g][d] = all;
    }
    __syncthreads();
    if (wave == 0) {  // exclusive scan over the 256 rings, four to a lane
        uint32_t all[4], sum = 0;
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint32_t d = lane * 4 + q;
            all[q] = part[1][0][d] + part[1][1][d] + part[1][2][d] + part[1][3][d];
            sum += all[q];
        }
        uint32_t upto = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = __shfl_up(upto, off, 64);
            if (lane >= (uint32_t)off) upto += o;
        }
        if (b == 0 && lane == 63) a.counters[0] = upto;
        uint32_t at = upto - sum;
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint32_t d = lane * 4 + q;
            place[d] = at + part[0][0][d] + part[0][1][d] + part[0][2][d] + part[0][3][d];
            at += all[q];
        }
    }
    const uint64_t end = min((uint64_t)entries, (uint64_t)(b + 1) * a.per);
    for (uint64_t t = (uint64_t)b * a.per; t < end; t += kRedThreads) {
        const uint32_t e = (uint32_t)(t + threadIdx.x);
        const bool win = t + threadIdx.x < end && red_wins(a, e);
        const uint32_t d = win ? a.key[e].w & 0xffu : 0u;
        uint64_t peers = __ballot(win);  // this wavefront's winners of the same ring
#pragma unroll
        for (uint32_t bit = 0; bit < 8; ++bit) {
            const uint64_t set = __ballot(win && (d >> bit & 1u));
            peers &= (d >> bit & 1u) ? set : ~set;
        }
        const uint64_t below = peers & ((1ull << lane) - 1ull);
        __syncthreads();  // the previous tile's counts and places have been read
        for (uint32_t i = threadIdx.x; i < kRedWaves * 256; i += kRedThreads) (&of_wave[0][0])[i] = 0;
        __syncthreads();
        if (win && below == 0) of_wave[wave][d] = (uint32_t)__popcll(peers);
        __syncthreads();
        if (threadIdx.x < 256) {
            uint32_t at = place[threadIdx.x];
#pragma unroll
            for (uint32_t w = 0; w < kRedWaves; ++w) {
                const uint32_t c = of_wave[w][threadIdx.x];
                of_wave[w][threadIdx.x] = at;
                at += c;
            }
            place[threadIdx.x] = at;
        }
        __syncthreads();
        if (win) out[of_wave[wave][d] + (uint32_t)__popcll(below)] = a.orig[e];
    }
}

// (ring, entry) of the winners, for rings of more than 8 bits.
__global__ __launch_bounds__(kRedThreads) void k_red_keys(RedArgs a, uint32_t blocks, uint64_t* __restrict__ keys)
{
    __shared__ uint32_t sh[kRedWaves];
    const uint32_t entries = red_entries(a, blocks, sh);
    const uint64_t step = (uint64_t)gridDim.x * kRedThreads;
    for (uint64_t e = (uint64_t)blockIdx.x * kRedThreads + threadIdx.x; e < a.n; e += step)
        keys[e] = e < entries && red_wins(a, (uint32_t)e) ? ((uint64_t)a.key[e].w << 32) | e : ~0ull;
}

__global__ void k_red_gather(const uint64_t* __restrict__ sorted, const tsl_point* __restrict__ orig,
                             const uint32_t* __restrict__ count, tsl_point* __restrict__ out)
{
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < *count) out[r] = orig[(uint32_t)sorted[r]];
}

// The pass's arguments over the filter's reduction scratch.
int red_args(tsl_filter* f, int mode, const tsl_point* raw, const void* ring, uint32_t n, float cell,
             uint32_t* counters, RedArgs* a, uint32_t* blocks)
{
    uint64_t slots = 4;
    while (slots < 4 * (uint64_t)n && slots < (1ull << 31)) slots *= 2;
    const size_t sizes[] = {sizeof(uint4) * (size_t)n, sizeof(tsl_point) * (size_t)n, sizeof(uint32_t) * slots,
                            sizeof(uint32_t) * (size_t)n, sizeof(uint32_t) * kRedBlocks,
                            sizeof(uint32_t) * kRedBlocks * 256};
    char* at[6];
    size_t total = 0;
    for (size_t b : sizes) total += (b + 255) / 256 * 256;
    TSL_TRY(f->red_scratch.reserve(total));
    char* p = f->red_scratch.as<char>();
    for (int k = 0; k < 6; ++k) {
        at[k] = p;
        p += (sizes[k] + 255) / 256 * 256;
    }
    const uint32_t tiles = (uint32_t)(((uint64_t)n + kRedThreads - 1) / kRedThreads);
    const uint32_t per = (tiles + kRedBlocks - 1) / kRedBlocks * kRedThreads;
    *blocks = (uint32_t)(((uint64_t)n + per - 1) / per);
    *a = RedArgs{raw, ring, n, per, mode, cell, cell / 2, reinterpret_cast<uint4*>(at[0]),
                 reinterpret_cast<tsl_point*>(at[1]), reinterpret_cast<uint32_t*>(at[2]),
                 reinterpret_cast<uint32_t*>(at[3]), (uint32_t)(slots - 1), reinterpret_cast<uint32_t*>(at[4]),
                 reinterpret_cast<uint32_t*>(at[5]), counters};
    return TSL_OK;
}

}  // namespace

// Reduce a raw scan on the device: writes the reduced points to out (room
// for n) and to counters[0] their number, to [1] 1 if a kept point's ring is
// outside [0, 64), to [2] 1 if the points still need launch_reduce_order.
int launch_reduce_scan(tsl_filter* f, int mode, const tsl_point* raw, const void* ring, uint32_t n, float cell,
                       tsl_point* out, uint32_t* counters, hipStream_t stream)
{
    if (n == 0) return TSL_OK;
    RedArgs a;
    uint32_t blocks;
    TSL_TRY(red_args(f, mode, raw, ring, n, cell, counters, &a, &blocks));
    hipLaunchKernelGGL(k_red_count, dim3(blocks), dim3(kRedThreads), 0, stream, a);
    TSL_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_red_build, dim3(blocks), dim3(kRedThreads), 0, stream, a);
    TSL_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_red_insert, dim3(blocks), dim3(kRedThreads), 0, stream, a, blocks);
    TSL_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_red_mark, dim3(blocks), dim3(kRedThreads), 0, stream, a);
    TSL_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_red_scatter, dim3(blocks), dim3(kRedThreads), 0, stream, a, out);
    TSL_HIP_CHECK(hipGetLastError());
    return TSL_OK;
}

// After launch_reduce_scan with the same arguments: the winners in the order
// of rings that differ in more than their low 8 bits (a cloud's ring field may
// hold any int32), by a 64-bit sort of (ring, entry).
int launch_reduce_order(tsl_filter* f, int mode, const tsl_point* raw, const void* ring, uint32_t n, float cell,
                        tsl_point* out, uint32_t* counters, hipStream_t stream)
{
    RedArgs a;
    uint32_t blocks;
    TSL_TRY(red_args(f, mode, raw, ring, n, cell, counters, &a, &blocks));
    TSL_TRY(f->sort_keys.reserve(sizeof(uint64_t) * 2 * (size_t)n));
    uint64_t* keys = f->sort_keys.as<uint64_t>();
    size_t temp = 0;
    TSL_HIP_CHECK(hipcub::DeviceRadixSort::SortKeys(nullptr, temp, keys, keys + n, (int)n, 0, 64, stream));
    TSL_TRY(f->sort_temp.reserve(temp));
    hipLaunchKernelGGL(k_red_keys, dim3(blocks), dim3(kRedThreads), 0, stream, a, blocks, keys);
    TSL_HIP_CHECK(hipGetLastError());
    TSL_HIP_CHECK(hipcub::DeviceRadixSort::SortKeys(f->sort_temp.ptr, temp, keys, keys + n, (int)n, 0, 64, stream));
    hipLaunchKernelGGL(k_red_gather, dim3((n + 255) / 256), dim3(256), 0, stream, keys + n, a.orig, counters, out);
    TSL_HIP_CHECK(hipGetLastError());
    return TSL_OK;
}

}  // namespace tsl
