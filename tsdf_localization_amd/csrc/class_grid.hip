// Class grid of a map: the form of the voxel values that the scoring kernels
// read (grid_eval.hip).
//
// Along one axis the reference's lookup (cuda_sub_voxel_map.tcc:51-137) uses a
// point's coordinate t only through o = fl(t - min): its truncation and the
// truncated quotient of its fraction by the resolution.  Both are step
// functions of t, so the axis falls into intervals ("classes") inside which
// every t gives the same index contribution, and the value read is a function
// of the three classes alone.  Per axis the classes are, in ascending order:
//   - o <= -1: gcc's size_t conversion wraps.  Where every such lookup is
//     rejected the class is "outside"; else there is one class per metre down
//     to kThinDepth (the sub-voxel index is 0 there), and below that "exact":
//     the kernels send those lanes through the exact tiers (tsl_lookup.h);
//   - (-1, 0): the truncated block is 0 and the sub-voxel index runs backwards,
//     one class per index;
//   - one class per voxel of the blocks inside the grid check; in z, none for
//     the layers above the topmost allocated block: "empty", the lowest of
//     them "above", where offsets <= -1 on another axis may reach back into
//     the map and are left to the exact tiers;
//   - beyond the grid check: "outside".
// The values of all class triples are laid out as a dense array of 4x4x4
// bricks (64 voxels, one 128-byte line of 16-bit codes), four bricks to a page
// of 8x8x4, pages in x, y, z order, so an element's byte address is a sum of
// one term per axis.  A bitmap over granules of 2^shift bytes (the finest that
// the LDS budget holds) tells which hold anything but init_value; the kernels
// load only from those.
//
// The class of t comes from a table of buckets: bucket fl(fma(t, scale,
// offset)) holds at most one class boundary (the smallest float of the upper
// class, found with the lookup's own float arithmetic), and the address terms
// on either side of it.
#include "tsl_lookup.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace tsl {

namespace {

constexpr uint32_t kKindVoxel = 0, kKindOutside = 1, kKindExact = 2, kKindEmpty = 3, kKindAbove = 4;

// Metres below a face kept as classes of their own (each costs the bucket
// table a metre of entries, 5 KB of LDS for 16 m at 0.05 m).  On the
// global-localisation workload a fifth of the particles put points below
// -1 m, one in a hundred below -16 m; with no such classes k_eval_grid took
// 5.49 ms there instead of 3.0, its exact lanes more than half of it.
constexpr uint32_t kThinDepth = 16;

// One coordinate of the dense array: its class's contribution to the lookup.
struct ClassDesc {
    int32_t block;   // truncated offset (below 0: an offset <= -1)
    int32_t sub;     // signed sub-voxel index
    uint32_t kind;
};

inline float next_up(float f) { return std::nextafter(f, INFINITY); }

// Order-preserving map between floats and unsigned integers.
inline uint32_t ordered(float f)
{
    uint32_t b;
    std::memcpy(&b, &f, 4);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

inline float unordered(uint32_t o)
{
    const uint32_t b = (o & 0x80000000u) ? (o & 0x7fffffffu) : ~o;
    float f;
    std::memcpy(&f, &b, 4);
    return f;
}

// Smallest t with fl(t - min) >= o (subtraction is monotone in t).
float lower_bound_t(float o, float min)
{
    uint32_t lo = ordered(-3.0e38f), hi = ordered(3.0e38f);
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (unordered(mid) - min >= o) hi = mid; else lo = mid + 1;
    }
    return unordered(lo);
}

struct Axis {
    std::vector<float> bound;        // class i + 1 starts at bound[i]
    std::vector<ClassDesc> classes;  // ascending
};

// The axis's classes and their boundaries in t; thin: metres of classes below
// -1, or none and rejected there.
void build_axis(float min, uint32_t blocks, bool low_out, uint32_t thin, const std::vector<float>& thr, Axis* a)
{
    // sub-voxel thresholds: index >= j from fraction thr[j - 1] on
    const uint32_t n = (uint32_t)thr.size();
    auto add = [&](float o, ClassDesc d) {
        a->bound.push_back(lower_bound_t(o, min));
        a->classes.push_back(d);
    };
    a->classes.push_back(ClassDesc{0, 0, low_out ? kKindOutside : kKindExact});
    if (!low_out)
        for (uint32_t m = thin; m >= 1; --m)  // -(m + 1) < o <= -m
            add(next_up(-(float)(m + 1)), ClassDesc{-(int32_t)m, 0, kKindVoxel});
    // the band (-1, 0): index -j while o <= -thr[j - 1]
    for (uint32_t j = n; j >= 1; --j)
        add(j == n ? next_up(-1.0f) : next_up(-thr[j]), ClassDesc{0, -(int32_t)j, kKindVoxel});
    for (uint32_t b = 0; b < blocks; ++b) {
        // offsets above -thr[0] have index 0 of block 0 already
        add(b == 0 ? (n ? next_up(-thr[0]) : next_up(-1.0f)) : (float)b, ClassDesc{(int32_t)b, 0, kKindVoxel});
        for (uint32_t j = 1; j <= n; ++j) {
            // smallest float o >= b + thr: the fraction of o is exact
            const double edge = (double)b + (double)thr[j - 1];
            float o = (float)edge;
            if ((double)o < edge) o = next_up(o);
            add(o, ClassDesc{(int32_t)b, (int32_t)j, kKindVoxel});
        }
    }
    add((float)blocks, ClassDesc{0, 0, kKindOutside});
}

// The tables of a map's class grid (host only).
struct ClassTables {
    std::vector<AxisEntry> table;        // buckets of x, y, z with address terms
    std::vector<ClassDesc> coords[3];    // class of every coordinate of the dense array
    uint32_t pages[3];
    float scale, off[3], top[3];
    uint32_t first[3];
    uint64_t elems;
};

constexpr uint32_t kPage[3] = {8, 8, 4};

// false: the map has no class grid.  gthr: the grid check's thresholds, R: the
// bound of the 32-bit tiers' offsets, esize: bytes of a cell.
bool class_tables(const tsl_map_coef& c, const int32_t* grid_occ, const uint32_t gthr[3], float R, uint32_t esize,
                  ClassTables* out)
{
    const uint64_t sd = c.sub_dim;
    if (c.data_size == 0) return false;
    // tame lanes (|t| < 2^22) must stay inside the 32-bit tiers' offsets
    const float lim = 4194304.0f;
    if (!(std::fabs(c.min_x) < lim && std::fabs(c.min_y) < lim && std::fabs(c.min_z) < lim)) return false;
    for (int a = 0; a < 3; ++a)
        if (gthr[a] == 0 || gthr[a] > 16384 || (float)gthr[a] >= R) return false;
    // sub-voxel thresholds below 1 from the bucket table of the exact tiers
    SubTable st;
    if (build_sub_table(c.resolution, &st) != TSL_OK) return false;
    std::vector<float> thr;
    for (const SubEntry& e : st.entries)
        if (e.thr != 0x7f800000u) {
            float f;
            std::memcpy(&f, &e.thr, 4);
            thr.push_back(f);
        }
    if (thr.size() > sd || thr.size() > 256) return false;
    // offsets <= -1: rejected for good where the grid check fails, or (even
    // sub_dim: the y and z wrap terms vanish modulo 2^64) on x because the
    // index lands past 2^62, on z because the block index stays negative
    DevMapFull fm{};
    negative_band_constants(c, fm);
    const bool even = fm.neg_y == 0 && fm.neg_z == 0;
    const int64_t plane_top = (int64_t)(gthr[0] - 1) + (int64_t)(gthr[1] - 1) * (int64_t)c.up_dim_x;
    const bool low_out[3] = {!fm.gneg_x || (even && fm.neg_x >= (1ull << 62) && fm.neg_x < (3ull << 62)),
                             !fm.gneg_y, !fm.gneg_z || (even && plane_top < (int64_t)c.up_dim_2)};
    // block layers above the topmost allocated one that a lookup with x and y
    // offsets above -1 can reach
    uint64_t last = 0;
    bool any = false;
    for (uint64_t b = 0; b < c.grid_occ_size; ++b)
        if (grid_occ[b] >= 0) {
            last = b;
            any = true;
        }
    uint64_t layers = any ? std::min<uint64_t>(gthr[2], last / c.up_dim_2 + 1) : 0;
    if (layers == 0) return false;

    const float mins[3] = {c.min_x, c.min_y, c.min_z};
    Axis axis[3];
    const uint64_t ups[3] = {c.up_dim_x, c.up_dim_y, c.up_dim_z};
    uint32_t thin[3];
    for (int a = 0; a < 3; ++a) {
        thin[a] = low_out[a] ? 0 : (uint32_t)std::min<uint64_t>(kThinDepth, ups[a]);
        build_axis(mins[a], gthr[a], low_out[a], thin[a], thr, &axis[a]);
    }
    // one layer above the topmost allocated one can be reached back from
    const uint64_t back = (thin[0] + thin[1] * c.up_dim_x + c.up_dim_2 - 1) / c.up_dim_2;
    for (ClassDesc& k : axis[2].classes)
        if (k.kind == kKindVoxel && k.block >= 0 && (uint64_t)k.block >= layers)
            k = ClassDesc{k.block, 0, (uint64_t)k.block < layers + back ? kKindAbove : kKindEmpty};

    // coordinates of the dense array: the voxel classes in order; from the next
    // page on, one each for "above", "empty" and "outside" (init_value but for
    // few), and on a page of its own "exact"
    std::vector<uint32_t> coord_of[3];
    uint32_t* pages = out->pages;
    for (int a = 0; a < 3; ++a) {
        std::vector<ClassDesc>& co = out->coords[a];
        co.clear();
        coord_of[a].assign(axis[a].classes.size(), 0u);
        for (uint32_t kind : {kKindVoxel, kKindOutside, kKindAbove, kKindEmpty, kKindExact}) {
            bool first = true;
            for (size_t k = 0; k < axis[a].classes.size(); ++k) {
                if (axis[a].classes[k].kind != kind) continue;
                if ((kind == kKindOutside || kind == kKindExact) && first)
                    while (co.size() % kPage[a]) co.push_back(ClassDesc{0, 0, kKindOutside});
                if (kind == kKindVoxel || first) co.push_back(axis[a].classes[k]);
                first = false;
                coord_of[a][k] = (uint32_t)co.size() - 1;
            }
        }
        while (co.size() % kPage[a]) co.push_back(ClassDesc{0, 0, kKindOutside});
        pages[a] = (uint32_t)(co.size() / kPage[a]);
    }
    const uint64_t elems = 256ull * pages[0] * pages[1] * pages[2];
    // the dense array stays within a few times the map's own voxels (all of it
    // counted, also what is never read) and within 32-bit byte addresses
    if (elems * esize >= (1ull << 32) || elems > 4 * c.data_size + (32ull << 20)) return false;
    out->elems = elems;
    // address terms, in bytes
    std::vector<uint32_t> term[3];
    for (int a = 0; a < 3; ++a) {
        const uint64_t stride = a == 0 ? 256ull : a == 1 ? 256ull * pages[0] : 256ull * pages[0] * pages[1];
        for (size_t k = 0; k < coord_of[a].size(); ++k) {
            const uint64_t v = coord_of[a][k];
            const uint64_t in = a == 0 ? (v & 3) + ((v >> 2) & 1) * 64 : a == 1 ? (v & 3) * 4 + ((v >> 2) & 1) * 128
                                                                             : (v & 3) * 16;
            term[a].push_back((uint32_t)(esize * (in + v / kPage[a] * stride)));
        }
    }
    // buckets a little narrower than the narrowest class: at most one boundary each
    float gap = 1.0f;
    for (size_t j = 0; j < thr.size(); ++j) gap = std::min(gap, thr[j] - (j ? thr[j - 1] : 0.0f));
    if (!thr.empty()) gap = std::min(gap, 1.0f - thr.back());
    const float magic = kGridMagic;  // integers are one ulp apart around it
    for (int attempt = 0;; ++attempt) {
        if (attempt == 4) return false;
        const float scale = (float)((1.04 + 0.1 * attempt) / (double)gap);
        std::vector<AxisEntry>& table = out->table;
        table.clear();
        bool ok = true;
        for (int a = 0; a < 3 && ok; ++a) {
            const std::vector<float>& bd = axis[a].bound;
            const double lo = (double)bd.front() * scale, hi = (double)bd.back() * scale;
            if (hi - lo > 65536.0 || std::fabs(lo) > 3e6 || std::fabs(hi) > 3e6) return false;
            const float off = magic + (float)(1.0 - std::floor(lo) + 1.0);
            const uint32_t n = (uint32_t)(std::ceil(hi) - std::floor(lo)) + 5;
            std::vector<AxisEntry> t(n, AxisEntry{0x7fc00000u, 0u, 0u, 0u});
            std::vector<uint8_t> has(n, 0);
            for (size_t j = 0; j < bd.size() && ok; ++j) {
                const int b = (int)(std::fmaf(bd[j], scale, off) - magic);
                if (b < 1 || b > (int)n - 2 || has[b]) {
                    ok = false;
                    break;
                }
                has[b] = 1;
                std::memcpy(&t[b].thr, &bd[j], 4);
                t[b].c_lo = term[a][j];
                t[b].c_hi = term[a][j + 1];
            }
            uint32_t cur = term[a][0];
            for (uint32_t b = 0; b < n && ok; ++b) {
                if (has[b]) cur = t[b].c_hi;
                else t[b].c_lo = t[b].c_hi = cur;
            }
            out->first[a] = (uint32_t)table.size();
            out->off[a] = off;
            out->top[a] = magic + (float)(n - 1);
            table.insert(table.end(), t.begin(), t.end());
        }
        if (!ok) continue;
        out->scale = scale;
        return true;
    }
}

// What a class triple reads: kKindVoxel with *idx its reference index,
// kKindExact (the exact tiers decide), or init_value.
__host__ __device__ __forceinline__ uint32_t class_index(const ClassDesc& dx, const ClassDesc& dy, const ClassDesc& dz,
                                                         const int32_t* grid_occ, uint64_t up_dim_x, uint64_t up_dim_2,
                                                         uint64_t occ, uint64_t data_size, uint64_t sd, uint64_t sd2,
                                                         const uint64_t neg[3], uint64_t* idx)
{
    if (dx.kind == kKindOutside || dy.kind == kKindOutside || dz.kind == kKindOutside) return kKindOutside;
    if (dx.kind == kKindExact || dy.kind == kKindExact || dz.kind == kKindExact) return kKindExact;
    if (dz.kind == kKindEmpty) return kKindEmpty;
    if (dz.kind == kKindAbove) return dx.block < 0 || dy.block < 0 ? kKindExact : kKindEmpty;
    const uint64_t up = (uint64_t)(int64_t)dx.block + (uint64_t)(int64_t)dy.block * up_dim_x +
                        (uint64_t)(int64_t)dz.block * up_dim_2;
    const int32_t s = up < occ ? grid_occ[up] : -1;
    if (s < 0) return kKindEmpty;
    *idx = (uint64_t)((int64_t)s + (int64_t)dx.sub + (int64_t)dy.sub * (int64_t)sd + (int64_t)dz.sub * (int64_t)sd2) +
           (dx.block < 0 ? neg[0] : 0) + (dy.block < 0 ? neg[1] : 0) + (dz.block < 0 ? neg[2] : 0);
    return *idx < data_size ? kKindVoxel : kKindEmpty;
}

struct FillArgs {
    const ClassDesc* desc[3];     // per coordinate of each axis
    uint32_t nx, ny, nz;          // pages per axis
    uint64_t up_dim_x, up_dim_2, occ, data_size, sd, sd2, neg[3];
    const int32_t* grid_occ;
    const void* values;           // the map's voxel array (codes, or floats)
    uint32_t brick, init_code, exact_code;  // the map's code of init_value; the code past its palette
    uint32_t base;                // LDS address of the palette
    float init;
    DevMap map;                   // bricked position of a reference index
};

__host__ __device__ __forceinline__ void grid_coord(uint64_t e, uint32_t nx, uint32_t ny, uint32_t& x, uint32_t& y, uint32_t& z)
{
    const uint32_t in = (uint32_t)(e & 255u);
    const uint64_t page = e >> 8;
    const uint32_t px = (uint32_t)(page % nx), py = (uint32_t)(page / nx % ny), pz = (uint32_t)(page / nx / ny);
    x = px * 8 + ((in >> 6) & 1u) * 4 + (in & 3u);
    y = py * 8 + ((in >> 7) & 1u) * 4 + ((in >> 2) & 3u);
    z = pz * 4 + ((in >> 4) & 3u);
}

// Element e of the dense array (a thread per element, a workgroup per page of
// 256): the value of its class triple as the reference's index arithmetic
// gives it; flags[e / 64] = 1 where a brick holds anything but init_value.
// Bound by the scattered reads of the map (each block's voxels are read from
// the few pages over it): once per map.
template <bool kF32>
__global__ __launch_bounds__(256) void k_grid_fill(FillArgs a, void* __restrict__ cells, uint8_t* __restrict__ flags)
{
    const uint64_t e = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    uint32_t x, y, z;
    grid_coord(e, a.nx, a.ny, x, y, z);
    const ClassDesc dx = a.desc[0][x], dy = a.desc[1][y], dz = a.desc[2][z];
    bool init = true;
    uint32_t code = a.init_code;
    float val = a.init;
    uint64_t idx = 0;
    const uint32_t kind = class_index(dx, dy, dz, a.grid_occ, a.up_dim_x, a.up_dim_2, a.occ, a.data_size, a.sd, a.sd2,
                                      a.neg, &idx);
    if (kind == kKindExact) {
        code = a.exact_code;
        val = __builtin_nanf("");
        init = false;
    } else if (kind == kKindVoxel) {
        const uint32_t at = a.brick ? phys_from_linear(a.map, (uint32_t)idx) : (uint32_t)idx;
        if (kF32) {
            val = static_cast<const float*>(a.values)[at];
            init = __float_as_uint(val) == __float_as_uint(a.init);
        } else {
            code = static_cast<const uint16_t*>(a.values)[at];
            init = code == a.init_code;
        }
    }
    if (kF32)
        static_cast<float*>(cells)[e] = val;
    else
        static_cast<uint16_t*>(cells)[e] = (uint16_t)(a.base + code);
    const uint64_t some = __ballot(!init);
    if ((threadIdx.x & 63u) == 0) flags[e >> 6] = some ? 1 : 0;
}

// Byte b of the bitmap: 8 granules of `per` bricks each.
__global__ void k_grid_bits(const uint8_t* __restrict__ flags, uint64_t bricks, uint32_t per, uint8_t* __restrict__ bits,
                            uint32_t bytes)
{
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= bytes) return;
    uint32_t v = 0;
    for (uint32_t g = 0; g < 8; ++g) {
        const uint64_t first = ((uint64_t)b * 8 + g) * per;
        for (uint64_t k = first; k < first + per && k < bricks; ++k)
            if (flags[k]) {
                v |= 1u << g;
                break;
            }
    }
    bits[b] = (uint8_t)v;
}

// The dense array is a map's second copy and may be larger than the first: it
// takes at most an eighth of the device memory that is free beside the map, so
// that on a card that is nearly full the rest goes to filters, robots and other
// maps as if there were no class grid.
bool leaves_room(uint64_t bytes)
{
    size_t free_bytes = 0, total = 0;
    if (hipMemGetInfo(&free_bytes, &total) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return bytes <= free_bytes / 8;
}

int build(tsl_map* m, const int32_t* grid_occ, uint32_t init_code)
{
    const tsl_map_coef& c = m->coef;
    DevMap& d = m->dev;
    DevGrid& g = m->grid;
    g = DevGrid{};
    const uint32_t gthr[3] = {d.gthr_x, d.gthr_y, d.gthr_z};
    float R;
    std::memcpy(&R, &d.range_bits, 4);
    const uint32_t esize = d.f32 ? 4u : 2u;
    ClassTables ct;
    if (d.wide || !class_tables(c, grid_occ, gthr, R, esize, &ct)) return TSL_OK;
    const std::vector<ClassDesc>* coords = ct.coords;
    const uint32_t* pages = ct.pages;
    const uint64_t elems = ct.elems;
    if (!leaves_room(elems * esize)) return TSL_OK;
    g.scale = ct.scale;
    for (int a = 0; a < 3; ++a) {
        g.off[a] = ct.off[a];
        g.top[a] = ct.top[a];
        g.first[a] = ct.first[a];
    }
    g.entries = (uint32_t)ct.table.size();
    TSL_TRY(m->grid_axis.reserve(sizeof(AxisEntry) * ct.table.size()));
    TSL_HIP_CHECK(hipMemcpy(m->grid_axis.ptr, ct.table.data(), sizeof(AxisEntry) * ct.table.size(),
                            hipMemcpyHostToDevice));
    // the finest granules whose bitmap fits the LDS budget
    const uint64_t bytes = elems * esize;
    const uint32_t brick_shift = d.f32 ? 8u : 7u;
    uint32_t shift = brick_shift;
    for (;; ++shift) {
        g.shift = shift;
        g.bits_bytes = (uint32_t)((((bytes + (1ull << shift) - 1) >> shift) + 127) / 128 * 16);
        g.palette_size = d.f32 ? 0u : d.palette_size + 1;
        // (16-bit cells hold LDS addresses up to the palette's end)
        if (grid_lds_bytes(g) <= kGridLdsBudget && g.bits_bytes + 4 * g.palette_size <= 65536) break;
        if (shift == brick_shift + 6) {
            g = DevGrid{};
            return TSL_OK;
        }
    }
    // palette with the NaN that marks lanes of the exact tiers
    if (!d.f32) {
        const float nan = __builtin_nanf("");
        TSL_TRY(m->grid_palette.reserve(sizeof(float) * g.palette_size));
        TSL_HIP_CHECK(hipMemcpy(m->grid_palette.ptr, d.palette, sizeof(float) * d.palette_size, hipMemcpyDeviceToDevice));
        TSL_HIP_CHECK(hipMemcpy(m->grid_palette.as<float>() + d.palette_size, &nan, sizeof(float), hipMemcpyHostToDevice));
    }
    DevBuf descs, flags;
    TSL_TRY(descs.reserve(sizeof(ClassDesc) * (coords[0].size() + coords[1].size() + coords[2].size())));
    TSL_TRY(flags.reserve(elems / 64));
    TSL_TRY(m->grid_cells.reserve(bytes));
    TSL_TRY(m->grid_bits.reserve(g.bits_bytes));
    FillArgs fa{};
    ClassDesc* at = descs.as<ClassDesc>();
    for (int a = 0; a < 3; ++a) {
        TSL_HIP_CHECK(hipMemcpy(at, coords[a].data(), sizeof(ClassDesc) * coords[a].size(), hipMemcpyHostToDevice));
        fa.desc[a] = at;
        at += coords[a].size();
    }
    fa.nx = pages[0];
    fa.ny = pages[1];
    fa.nz = pages[2];
    fa.up_dim_x = c.up_dim_x;
    fa.up_dim_2 = c.up_dim_2;
    fa.occ = c.grid_occ_size;
    fa.data_size = c.data_size;
    fa.sd = c.sub_dim;
    fa.sd2 = c.sub_dim_2;
    DevMapFull fm{};
    negative_band_constants(c, fm);
    fa.neg[0] = fm.neg_x;
    fa.neg[1] = fm.neg_y;
    fa.neg[2] = fm.neg_z;
    fa.grid_occ = d.grid_occ;
    fa.values = d.codes;
    fa.brick = d.brick;
    fa.init_code = init_code;
    fa.exact_code = d.palette_size * 4u;
    fa.base = g.bits_bytes;
    fa.init = d.init;
    fa.map = d;
    const dim3 grid((unsigned)(elems / 256));
    if (d.f32)
        hipLaunchKernelGGL(k_grid_fill<true>, grid, dim3(256), 0, 0, fa, m->grid_cells.ptr, flags.as<uint8_t>());
    else
        hipLaunchKernelGGL(k_grid_fill<false>, grid, dim3(256), 0, 0, fa, m->grid_cells.ptr, flags.as<uint8_t>());
    TSL_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_grid_bits, dim3((g.bits_bytes + 255) / 256), dim3(256), 0, 0, flags.as<uint8_t>(), elems / 64,
                       1u << (shift - brick_shift), m->grid_bits.as<uint8_t>(), g.bits_bytes);
    TSL_HIP_CHECK(hipGetLastError());
    TSL_HIP_CHECK(hipDeviceSynchronize());
    g.axis = m->grid_axis.as<AxisEntry>();
    g.bits = m->grid_bits.as<uint8_t>();
    g.cells = m->grid_cells.ptr;
    g.palette = m->grid_palette.as<float>();
    g.init_code = g.bits_bytes + init_code;
    g.init = d.init;
    g.ready = 1;
    return grid_kernels_init();
}

}  // namespace

int build_class_grid(tsl_map* m, const int32_t* grid_occ, uint32_t init_code)
{
    const int rc = build(m, grid_occ, init_code);
    if (rc == TSL_ERR_OUT_OF_MEMORY) {  // no room beside the map: it is scored without
        (void)hipGetLastError();
        clear_error();
        m->grid = DevGrid{};
    } else if (rc != TSL_OK) {
        return rc;
    }
    if (!m->grid.ready)
        for (DevBuf* b : {&m->grid_axis, &m->grid_bits, &m->grid_cells, &m->grid_palette}) b->release();
    return TSL_OK;
}

}  // namespace tsl

extern "C" int tsl_check_class_grid(const tsl_map_coef* coef, const int32_t* grid_occ, const float* t, size_t n,
                                    uint64_t* index, int* has_grid)
{
    using namespace tsl;
    if (!coef || !grid_occ || !has_grid || (n && (!t || !index)))
        return set_error(TSL_ERR_INVALID_ARGUMENT, "NULL argument");
    TSL_TRY(validate_coef(coef));
    const tsl_map_coef& c = *coef;
    const uint32_t gthr[3] = {grid_threshold(c.dim_x, c.resolution), grid_threshold(c.dim_y, c.resolution),
                              grid_threshold(c.dim_z, c.resolution)};
    ClassTables ct;
    *has_grid = class_tables(c, grid_occ, gthr, lookup_range(c), 2, &ct) ? 1 : 0;
    if (!*has_grid) return TSL_OK;
    DevMapFull fm{};
    negative_band_constants(c, fm);
    const uint64_t neg[3] = {fm.neg_x, fm.neg_y, fm.neg_z};
    for (size_t i = 0; i < n; ++i) {
        const float* p = t + 3 * i;
        if (!(std::fabs(p[0]) < 4194304.0f && std::fabs(p[1]) < 4194304.0f && std::fabs(p[2]) < 4194304.0f)) {
            index[i] = ~0ull;
            continue;
        }
        uint32_t addr = 0;
        for (int a = 0; a < 3; ++a) {
            const float v = std::min(std::max(std::fmaf(p[a], ct.scale, ct.off[a]), kGridMagic), ct.top[a]);
            const AxisEntry& e = ct.table[ct.first[a] + (uint32_t)(v - kGridMagic)];
            float edge;
            std::memcpy(&edge, &e.thr, 4);
            addr += p[a] >= edge ? e.c_hi : e.c_lo;
        }
        uint32_t x, y, z;
        grid_coord(addr / 2, ct.pages[0], ct.pages[1], x, y, z);
        uint64_t idx = 0;
        switch (class_index(ct.coords[0][x], ct.coords[1][y], ct.coords[2][z], grid_occ, c.up_dim_x, c.up_dim_2,
                            c.grid_occ_size, c.data_size, c.sub_dim, c.sub_dim_2, neg, &idx)) {
        case kKindVoxel: index[i] = idx; break;
        case kKindExact: index[i] = ~0ull; break;
        default: index[i] = c.data_size; break;
        }
    }
    return TSL_OK;
}
