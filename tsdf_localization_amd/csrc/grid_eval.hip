// Scoring kernels on a map's class grid (class_grid.hip).  A wavefront takes
// two particles x one chunk of the scan, lane l the points base + l; every
// lane adds its points in ascending order and the wavefront sums with the same
// butterfly as eval_kernels.h, so the weights are its bit for bit.
//
// Per pair: the exact float transform, one bucket entry per axis (the class
// boundary and the address terms on its two sides), the sum of the three
// terms, one bitmap bit, and for granules that hold anything the cell and its
// palette value: 43 VALU instructions and no division, block table or negative
// band of its own, where the index arithmetic of eval_kernels.h takes 72.
// Lanes whose cell is the exact tiers' NaN (offsets the table does not hold),
// and points marked by a NaN score term (not finite, or past kTamePoint), are
// recomputed with the reference's arithmetic.
//
// 100,000 particles x 20,000 points of the benchmark's building:
// 2.57 ms against 3.84 (7.8e11 pairs/s against 5.2e11); VALU instructions issue
// on 96 % of the cycles (2.2 ms with the gathers taken out).  Where 85 to 90 % of
// the pairs read a cell (tracking filters) the texture-data path is full
// instead, and a million sparse particles wait for lines beyond the L2.  Two
// particles are in flight per wavefront because more of them
// (4, 8) put more distinct cells in flight than the L2 holds.
//
// The tables take tens of KB of LDS on large maps, so a workgroup has 4, 8 or
// 16 wavefronts, whichever keeps most of them resident (grid_threads), and
// stays.  The points come straight from the caches, one iteration ahead.
#include "eval_kernels.h"

namespace tsl {

namespace {

// Matrices below these bounds and points below kTamePoint keep |t| < 2^22.
constexpr float kTameRotation = 16.0f, kTameShift = 1048576.0f;

struct GridLds {
    uint32_t axis;  // LDS byte address of the bucket tables
};

using Entry4 = uint32_t __attribute__((ext_vector_type(4)));  // an AxisEntry as one load

template <typename T>
__device__ __forceinline__ T lds_at(uint32_t addr)
{
    return *reinterpret_cast<const __attribute__((address_space(3))) T*>((uintptr_t)addr);
}

// The bitmap sits at LDS address 0 and the palette behind it (cells hold the
// LDS addresses of their values), so neither needs a base added per lookup;
// the kernels declare no static LDS.
template <bool kF32>
__device__ __forceinline__ GridLds stage_grid(const DevGrid& g, bool scaled, float a_hit)
{
    extern __shared__ uint4 smem_raw[];
    const uint32_t axis = g.bits_bytes + (kF32 ? 0u : 16u * ((g.palette_size + 3u) / 4u));
    char* base = reinterpret_cast<char*>(smem_raw);
    uint4* dst = reinterpret_cast<uint4*>(base);
    const uint4* src = reinterpret_cast<const uint4*>(g.bits);
    for (uint32_t i = threadIdx.x; i < g.bits_bytes / 16; i += blockDim.x) dst[i] = src[i];
    if (!kF32) {
        float* lut = reinterpret_cast<float*>(base + g.bits_bytes);
        for (uint32_t i = threadIdx.x; i < g.palette_size; i += blockDim.x)
            lut[i] = scaled ? a_hit * g.palette[i] : g.palette[i];
    }
    dst = reinterpret_cast<uint4*>(base + axis);
    src = reinterpret_cast<const uint4*>(g.axis);
    for (uint32_t i = threadIdx.x; i < g.entries; i += blockDim.x) dst[i] = src[i];
    GridLds s;
    s.axis = axis;
    __syncthreads();
    return s;
}

// The bucket entry of coordinate t on one axis, and its address term.
__device__ __forceinline__ Entry4 grid_entry(float t, float scale, float off, float top, uint32_t table)
{
    const float v = __builtin_amdgcn_fmed3f(__builtin_fmaf(t, scale, off), kGridMagic, top);
    // entry address: 16 (bits(v) - bits(kGridMagic)) + table
    return lds_at<Entry4>((__float_as_uint(v) << 4) + table);
}

__device__ __forceinline__ uint32_t grid_term(float t, Entry4 e) { return t >= __uint_as_float(e.x) ? e.z : e.y; }

// Value (times a_hit unless traced) of one pair by the exact tiers.  The map's
// fields are read from device memory here (the empty asm keeps the loads in
// this branch), so that they hold no registers in the loop.
template <bool kF32, bool kScaled>
__device__ __forceinline__ float exact_value(const DevMap* map_dev, float a_hit, float tx, float ty, float tz)
{
    asm volatile("" : "+s"(map_dev));
    const DevMap& map = *map_dev;
    const uint64_t full = slow_index<false, false, false>(map, map.sub_tab, map.neg_tab, nullptr, tx - map.min_x,
                                                          ty - map.min_y, tz - map.min_z);
    float val = map.init;
    if (full < map.data_size) {
        const uint32_t x = (uint32_t)full;
        const uint32_t e = map.brick ? phys_from_linear(map, x) : x;
        if (kF32)
            val = reinterpret_cast<const float*>(map.codes)[e];
        else
            val = map.palette[map.codes[e] >> 2];
    }
    return kScaled ? a_hit * val : val;
}

// Points per buffer descriptor (its offsets have 32 bits), whole iterations.
constexpr uint32_t kSegment = 1u << 24;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t point_buffer(const float4* p, uint32_t n)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float4*>(p), 0, (int)(n * 16u), 0x00020000);
}

// The whole offset goes into the vector operand: a raw buffer's range check
// covers that and the instruction's constant, not a scalar offset, so a load
// past the descriptor's end gives zero and reads nothing.
__device__ __forceinline__ float4 point_at(__amdgpu_buffer_rsrc_t rsrc, uint32_t byte)
{
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)byte, 0, 0);
    return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
}

// The score's point term (tsdf_evaluator.cpp:56-65), as the scan preparation
// forms it.
__device__ __forceinline__ float score_term(const ScoreTerm& sc, const float4& q)
{
    const float d2 = q.x * q.x + q.y * q.y + q.z * q.z;
    return d2 < sc.max_range_squared ? sc.range_term : sc.a_max;
}

// The bucket tables' constants of one kernel: wavefront-uniform bases (entry
// address: 16 bits(v) + base), and the scale in a vector register, since an
// instruction reads one scalar operand.
struct GridTables {
    uint32_t x, y, z;
    float scale;
};

__device__ __forceinline__ GridTables grid_tables(const DevGrid& g, const GridLds& s)
{
    const uint32_t magic = __float_as_uint(kGridMagic) << 4;
    GridTables t{s.axis + 16u * g.first[0] - magic, s.axis + 16u * g.first[1] - magic,
                 s.axis + 16u * g.first[2] - magic, g.scale};
    asm("" : "+s"(t.x), "+s"(t.y), "+s"(t.z));
    asm("" : "+v"(t.scale));
    return t;
}

// tsdf_evaluator.cpp:44-46: ((L0*x + L1*y) + L2*z) + L3, no FMA
__device__ __forceinline__ void transform(const float (&m)[12], const float4& q, float& tx, float& ty, float& tz)
{
    tx = m[0] * q.x + m[1] * q.y + m[2] * q.z + m[3];
    ty = m[4] * q.x + m[5] * q.y + m[6] * q.z + m[7];
    tz = m[8] * q.x + m[9] * q.y + m[10] * q.z + m[11];
}

constexpr int K = (int)kGridParticles;

// Points between two barriers of a workgroup's wavefronts.  In step, the 2 x 16
// neighbouring particles of a workgroup put the same points into the same few
// metres of the map, so that most of their cells come from lines that another
// wavefront has just brought in.  100,000 particles x 20,000 points: 3.05 ms
// without the barriers, 2.59, 2.55, 2.52 ms with one every 128, 256, 512
// points; 1,000,000 x 3989: 18.5 ms, 12.6, 12.8, 13.0.  (Workgroups of an XCD
// waiting for each other as well save more lines than the waiting is worth: 11
// ms there, but 2.7 above.)
constexpr uint32_t kPace = 256;

// One wavefront: particles p0, p0 + 1 x the points [j0, j1) of one chunk
// (kMode 0), or the value of every pair to trace_out in the caller's point
// order (kMode 2).  A wavefront with nothing to do (live false) only meets
// the others at the `paces` barriers.
template <int kMode, bool kF32>
__device__ __forceinline__ void grid_wave(const DevMap* map_dev, const DevGrid& g, const ScoreTerm& sc,
                                          const GridTables& tab, const float* __restrict__ L, uint32_t P, uint32_t p0,
                                          bool live, const float4* __restrict__ pts, uint32_t N, uint32_t j0,
                                          uint32_t j1, uint32_t paces, float a_hit, float* __restrict__ partial_row,
                                          void* __restrict__ trace_out, const uint32_t* __restrict__ perm)
{
    const uint32_t lane = threadIdx.x & 63;
    if (!live) j1 = j0;
    float m[K][12];
    bool tame = true;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t p = min(p0 + k, P - 1);
#pragma unroll
        for (int e = 0; e < 12; ++e) {
            // wavefront-uniform: scalar registers
            m[k][e] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(L[(size_t)p * 12 + e])));
            tame = tame & (fabsf(m[k][e]) < ((e & 3) == 3 ? kTameShift : kTameRotation));
        }
    }
    // all lanes of the exact tiers where a matrix is not tame
    const uint64_t wild = __builtin_amdgcn_readfirstlane(tame ? 1u : 0u) ? 0ull : ~0ull;
    using Cell = std::conditional_t<kF32, float, uint32_t>;
    Cell cell[K];
    uint32_t addr[K];
    bool hit[K];
    float acc[K];
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = 0.0f;
    // Where the pairs of a point read, and whether they read at all.  The
    // stages are kept apart (sched_barrier), so that all of a stage's LDS reads
    // are under way before the first is waited for.
    auto locate = [&](const float4& q) {
        float t[K][3];
        Entry4 e[K][3];
        uint32_t byte[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            transform(m[k], q, t[k][0], t[k][1], t[k][2]);
            e[k][0] = grid_entry(t[k][0], tab.scale, g.off[0], g.top[0], tab.x);
            e[k][1] = grid_entry(t[k][1], tab.scale, g.off[1], g.top[1], tab.y);
            e[k][2] = grid_entry(t[k][2], tab.scale, g.off[2], g.top[2], tab.z);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            addr[k] = grid_term(t[k][0], e[k][0]) + grid_term(t[k][1], e[k][1]) + grid_term(t[k][2], e[k][2]);
            byte[k] = lds_at<uint8_t>(addr[k] >> (g.shift + 3));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            asm("" : "+v"(byte[k]));
            hit[k] = __builtin_amdgcn_ubfe(byte[k], __builtin_amdgcn_ubfe(addr[k], g.shift, 3u), 1u) != 0u;
        }
    };
    // Ask for the cells; granules that hold only init_value are not read.
    auto fetch = [&]() {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const char* at = static_cast<const char*>(g.cells) + addr[k];
            if constexpr (kF32) {
                cell[k] = g.init;
                if (hit[k]) cell[k] = *reinterpret_cast<const float*>(at);
            } else {
                cell[k] = g.init_code;
                if (hit[k]) cell[k] = *reinterpret_cast<const uint16_t*>(at);
            }
        }
    };
    // The points come through a buffer descriptor of at most kSegment of them,
    // whose loads give zero past the chunk's end.
    const uint32_t lane_off = lane * 16u;
    uint32_t met = 0;
    for (uint32_t seg = __builtin_amdgcn_readfirstlane(j0); seg < j1; seg += kSegment) {
        const uint32_t len = min(j1 - seg, kSegment);
        const auto rsrc = point_buffer(pts + seg, len);
        float w;  // score term of the points whose cells are on their way
        auto finish = [&](uint32_t off, auto full_tag) {
            constexpr bool kFull = decltype(full_tag)::value;
            const bool act = kFull || off + lane < len;
            float v[K], sum[K];
            bool nan = false;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if constexpr (kF32)
                    v[k] = kMode == 0 ? a_hit * cell[k] : cell[k];
                else
                    v[k] = lds_at<float>(cell[k]);
                sum[k] = v[k] + w;  // tsdf_evaluator.cpp:56-67 (v = a_hit * value)
                nan = nan | (sum[k] != sum[k]);
            }
            // lanes of the exact tiers and marked points (a NaN value of the
            // map or score term is formed again, with the same result)
            if (__builtin_expect((__builtin_amdgcn_ballot_w64(nan) | wild) != 0, 0)) {
                const float4 q = point_at(rsrc, lane_off + off * 16u);
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (wild || sum[k] != sum[k]) {
                        float tx, ty, tz;
                        transform(m[k], q, tx, ty, tz);
                        v[k] = exact_value<kF32, kMode == 0>(map_dev, a_hit, tx, ty, tz);
                        sum[k] = v[k] + score_term(sc, q);
                    }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if (kMode == 2) {
                    if (act && p0 + k < P)
                        static_cast<float*>(trace_out)[(size_t)(p0 + k) * N + perm[seg + off + lane]] = v[k];
                } else if (act) {
                    acc[k] += sum[k];
                }
            }
        };
        // Software pipeline, two groups of points a turn: while the addresses
        // of one group are formed, the cells of the group before and the
        // points of the group after are on their way (points past the chunk's
        // end read as zeros and are not summed).  The points are waited for
        // before the cells behind them are asked for, so that no wait has to
        // cover loads that some lanes may not have issued.
        auto arrive = [](float4& q) { asm volatile("" : "+v"(q.x), "+v"(q.y), "+v"(q.z), "+v"(q.w)); };
        auto turn = [&](const float4& now, float4& after, uint32_t off, auto full_tag) {
            after = point_at(rsrc, lane_off + (off + 128u) * 16u);
            locate(now);
            finish(off, full_tag);
            w = now.w;
            arrive(after);
            fetch();
        };
        float4 even = point_at(rsrc, lane_off), odd = point_at(rsrc, lane_off + 64u * 16u);
        locate(even);
        w = even.w;
        arrive(odd);
        fetch();
        uint32_t off = 0;
        for (; off + 128 <= len; off += 128) {
            if (off % kPace == 0) {
                __builtin_amdgcn_s_barrier();
                ++met;
            }
            turn(odd, even, off, std::true_type{});
            turn(even, odd, off + 64, std::true_type{});
        }
        for (; off < len; off += 64) {  // the last one or two, by lane
            turn(odd, even, off, std::false_type{});
            odd = even;
        }
    }
    for (; met < paces; ++met) __builtin_amdgcn_s_barrier();
    if (kMode != 0) return;
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = wave_sum(acc[k]);
    if (lane == 0 && live) {
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (p0 + k < P) partial_row[p0 + k] = acc[k];
    }
}

// Items of a workgroup: `per` particles (kGridParticles for each of its
// wavefronts; a few times that where there would be too many items) x one
// chunk, all wavefronts on the same points.  The workgroups of XCD x (dealt to
// the 8 XCDs round-robin by index) take the items of the x-th contiguous
// eighth in order, neighbours in the evaluation order together, so that
// spatially sorted particles share that XCD's L2.  (Dealing the last, partial
// round out by wavefronts instead, a few to every workgroup, measured 2.61 ms
// against 2.54 at 100,000 x 20,000.)
template <int kMode, bool kF32>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_eval_grid(
    const DevMap* __restrict__ map_dev, DevGrid g, ScoreTerm sc, const float* __restrict__ L,
    const uint32_t* __restrict__ count, const float4* __restrict__ pts, uint32_t N, uint32_t per,
    uint32_t chunk_len, uint32_t chunks, float a_hit, float* __restrict__ partial, uint32_t stride,
    void* __restrict__ trace_out, const uint32_t* __restrict__ perm)
{
    const uint32_t P = *count;
    const uint32_t items = (P + per - 1) / per * chunks;
    const uint32_t xcd = blockIdx.x % kXcds;
    const uint32_t q = items / kXcds, rem = items % kXcds;
    const uint32_t first = xcd * q + min(xcd, rem), end = first + q + (xcd < rem ? 1u : 0u);
    const uint32_t waves = blockDim.x >> 6, paces = (chunk_len + kPace - 1) / kPace;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t item = first + blockIdx.x / kXcds;
    if (item >= end) return;  // uniform across the workgroup
    const GridLds s = stage_grid<kF32>(g, kMode == 0, a_hit);
    const GridTables tab = grid_tables(g, s);
    for (; item < end; item += gridDim.x / kXcds) {  // (gridDim.x is a multiple of kXcds)
        const uint32_t row = item / chunks, c = item - row * chunks;
        const uint32_t j0 = c * chunk_len;
        for (uint32_t part = 0; part < per; part += K * waves) {
            const uint32_t p0 = row * per + part + K * wave;
            grid_wave<kMode, kF32>(map_dev, g, sc, tab, L, P, p0, p0 < P, pts, N, j0, min(N, j0 + chunk_len), paces,
                                   a_hit, kMode == 0 ? partial + (size_t)c * stride : nullptr, trace_out, perm);
        }
    }
}

// Batched form: every workgroup claims its items one at a time from its XCD's
// counter, the next one while it works on an item.
template <bool kF32>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_eval_grid_batch(
    const DevMap* __restrict__ map_dev, DevGrid g, ScoreTerm sc, const Member* __restrict__ members,
    BatchPlan* __restrict__ plan, float a_hit, uint32_t per, uint32_t item0, uint32_t count)
{
    const GridLds s = stage_grid<kF32>(g, true, a_hit);
    const GridTables tab = grid_tables(g, s);
    // two claims behind the tables, read and written by turns
    volatile auto* claimed = reinterpret_cast<volatile __attribute__((address_space(3))) uint32_t*>(
        (uintptr_t)(grid_lds_bytes(g) - 16));
    const uint32_t n = plan->n;
    const uint32_t total = min(plan->total, item0 + min(count, 0xffffffffu - item0));
    const uint32_t xcd = blockIdx.x % kPlanXcds;
    const uint32_t waves = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t* counter = &plan->next[xcd * 32];
    if (threadIdx.x == 0) claimed[0] = atomicAdd(counter, 1u);
    for (uint32_t turn = 0;; ++turn) {
        __syncthreads();
        const uint32_t item = item0 + __builtin_amdgcn_readfirstlane(claimed[turn & 1]) * kPlanXcds + xcd;
        if (item >= total) break;
        if (threadIdx.x == 0) claimed[(turn + 1) & 1] = atomicAdd(counter, 1u);
        uint32_t lo = 0, hi = n;  // member: prefix[lo] <= item < prefix[lo + 1]
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (plan->prefix[mid] <= item) lo = mid; else hi = mid;
        }
        const uint32_t f = __builtin_amdgcn_readfirstlane(lo);
        const Member& mb = members[f];
        const uint32_t local = item - plan->prefix[f];
        const uint32_t row = local / mb.chunks, c = local - row * mb.chunks;
        const uint32_t j0 = c * mb.chunk_len, P = mb.st->count, paces = (mb.chunk_len + kPace - 1) / kPace;
        for (uint32_t part = 0; part < per; part += K * waves) {
            const uint32_t p0 = row * per + part + K * wave;
            grid_wave<0, kF32>(map_dev, g, sc, tab, mb.L, P, p0, p0 < P, mb.points, mb.N, j0,
                               min(mb.N, j0 + mb.chunk_len), paces, a_hit, mb.partial + (size_t)c * mb.stride, nullptr,
                               nullptr);
        }
    }
}

template <int kMode, bool kF32>
int launch_grid_t(const tsl_filter* f, const Tile& tile, size_t P, size_t N, hipStream_t stream, float* partial,
                  void* trace_out)
{
    constexpr auto kernel = &k_eval_grid<kMode, kF32>;
    const tsl_map* map = f->ev->map;
    const uint32_t threads = grid_threads(map->grid);
    const uint32_t per = grid_item_particles(map->grid, P * tile.chunks);
    const size_t items = (P + per - 1) / per * tile.chunks;
    uint32_t groups = 0;
    TSL_TRY(resident_groups(reinterpret_cast<const void*>(kernel), (int)threads, grid_lds_bytes(map->grid),
                            map->device, items, &groups));
    FilterState* st = f->state.as<FilterState>();
    hipLaunchKernelGGL(kernel, dim3(groups), dim3(threads), grid_lds_bytes(map->grid), stream,
                       map->dev_copy.as<DevMap>(), map->grid, score_term_of(f->ev), f->L.as<float>(), &st->count,
                       f->points.as<float4>(), (uint32_t)N, per, tile.chunk_len, tile.chunks, f->ev->a_hit, partial,
                       (uint32_t)f->capacity, trace_out, f->perm.as<uint32_t>());
    TSL_HIP_CHECK(hipGetLastError());
    return TSL_OK;
}

template <bool kF32>
int launch_grid_batch_t(const BatchLaunch& b, hipStream_t stream, uint32_t* grid_out)
{
    constexpr auto kernel = &k_eval_grid_batch<kF32>;
    const uint32_t threads = grid_threads(b.map->grid);
    const size_t lds = grid_lds_bytes(b.map->grid);
    if (grid_out)
        return resident_groups(reinterpret_cast<const void*>(kernel), (int)threads, lds, b.map->device, b.max_items,
                               grid_out);
    return launch_slices(b, stream, [&](uint32_t item0, uint32_t count) {
        hipLaunchKernelGGL(kernel, dim3(b.grid), dim3(threads), lds, stream, b.map->dev_copy.as<DevMap>(),
                           b.map->grid, b.score, b.members, b.plan, b.a_hit, b.per, item0, count);
    });
}

}  // namespace

int grid_kernels_init()
{
    const void* kernels[] = {reinterpret_cast<const void*>(&k_eval_grid<0, false>),
                             reinterpret_cast<const void*>(&k_eval_grid<0, true>),
                             reinterpret_cast<const void*>(&k_eval_grid<2, false>),
                             reinterpret_cast<const void*>(&k_eval_grid<2, true>),
                             reinterpret_cast<const void*>(&k_eval_grid_batch<false>),
                             reinterpret_cast<const void*>(&k_eval_grid_batch<true>)};
    for (const void* k : kernels) {
        if (!palette_at_zero(k)) return set_error(TSL_ERR_UNSUPPORTED, "class-grid kernel declares static LDS");
        TSL_HIP_CHECK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGridLdsBudget));
    }
    return TSL_OK;
}

int launch_grid(int mode, const tsl_filter* f, const Tile& tile, size_t P, size_t N, hipStream_t stream,
                float* partial, void* trace_out)
{
    const bool f32 = f->ev->map->dev.f32 != 0;
#define TSL_GRID_ARGS f, tile, P, N, stream, partial, trace_out
    if (mode == 0) return f32 ? launch_grid_t<0, true>(TSL_GRID_ARGS) : launch_grid_t<0, false>(TSL_GRID_ARGS);
    return f32 ? launch_grid_t<2, true>(TSL_GRID_ARGS) : launch_grid_t<2, false>(TSL_GRID_ARGS);
#undef TSL_GRID_ARGS
}

int launch_grid_batch(const BatchLaunch& b, hipStream_t stream, uint32_t* grid_out)
{
    return b.map->dev.f32 ? launch_grid_batch_t<true>(b, stream, grid_out)
                          : launch_grid_batch_t<false>(b, stream, grid_out);
}

}  // namespace tsl
