// raycast.hip — rendering-block depth-range prepass and the TSDF raycast
// for gfx950.
//
// Prepass (CreateRenderingBlocks, Mapping/RenderScene.cu:210-289): one thread
// per visible block projects its eight corners, clips the 1/8-resolution box
// and applies the reference's tile coverage directly with integer
// atomicMin / atomicMax on the float bits (all depths are positive, where the
// IEEE bit order is the numeric order) — no rendering-block list, no
// host round trip.
// Raycast (Rendering::operator(), RenderScene.cu:380-488): a first pass of one
// lane per pixel, 8x8-pixel workgroups (one wavefront) so that neighbouring rays
// march through the same voxel blocks, whose lookups they share in LDS; a second
// pass of eight lanes per ray for the rays still marching then. The adjoint runs
// the second pass's march.
#include "map_common.hpp"

namespace sicp {

namespace {

struct PrepassArgs {
    float fx, fy, cx, cy;
    float dmax, dmin;
    int zcols, zrows;
};

__global__ __launch_bounds__(256) void zrange_init_kernel(View<float> zmin, View<float> zmax,
                                                          MapCounters* ctr) {
    const int n = zmin.cols * zmin.rows;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        int y = i / zmin.cols, x = i - y * zmin.cols;
        zmin.at(y, x) = 100.f;
        zmax.at(y, x) = 0.f;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) ctr->render_tiles = 0u;
}

// Projection::projectBlock (RenderScene.cu:54-112).
SICP_DEV bool project_block(const sicp_block& b, const PoseF& pose, const PrepassArgs& g,
                            float voxel, int& ulx, int& uly, int& lrx, int& lry, float& z0,
                            float& z1) {
    ulx = g.zcols;
    uly = g.zrows;
    lrx = -1;
    lry = -1;
    z0 = g.dmax;
    z1 = g.dmin;
    for (int corner = 0; corner < 8; ++corner) {
        int tx = b.x + ((corner & 1) ? 1 : 0);
        int ty = b.y + ((corner & 2) ? 1 : 0);
        int tz = b.z + ((corner & 4) ? 1 : 0);
        v3 p{(float)(tx * kBlockSide) * voxel, (float)(ty * kBlockSide) * voxel,
             (float)(tz * kBlockSide) * voxel};
        p = mv(pose.Rinv, sub(p, pose.t));
        if ((double)p.z < 2e-1) continue;
        float px = (g.fx * p.x / p.z + g.cx) / 8.0f;
        float py = (g.fy * p.y / p.z + g.cy) / 8.0f;
        float fx_ = floorf(px), cx_ = ceilf(px), fy_ = floorf(py), cy_ = ceilf(py);
        if ((float)ulx > fx_) ulx = (int16_t)(int)fx_;
        if ((float)lrx < cx_) lrx = (int16_t)(int)cx_;
        if ((float)uly > fy_) uly = (int16_t)(int)fy_;
        if ((float)lry < cy_) lry = (int16_t)(int)cy_;
        if (z0 > p.z) z0 = p.z;
        if (z1 < p.z) z1 = p.z;
    }
    if (ulx < 0) ulx = 0;
    if (uly < 0) uly = 0;
    if (lrx >= g.zcols) lrx = g.zcols - 1;
    if (lry >= g.zrows) lry = g.zrows - 1;
    if (ulx > lrx) return false;
    if (uly > lry) return false;
    if (z0 < g.dmin) z0 = g.dmin;
    if (z1 < g.dmin) return false;
    return true;
}

// createRenderingBlockList (:114-132) + fillBlocks (:167-190): the tile loop
// runs x < ny and does not offset the tiles' lower-right corner, so a box
// [ul, lr] covers columns ul.x .. min(ul.x+15, lr.x) (+ ul.x+16 when ny >= 2
// and lr.x >= ul.x+16) times rows ul.y .. min(ul.y+15, lr.y) (+ ul.y+16 on
// the same condition). `tile(Y, X, lo, hi)` receives every covered tile with
// the block's depth range as int bit patterns (positive floats order as
// their bits do). Returns whether the block produced tiles.
template <class TileFn>
SICP_DEV bool block_tiles(const sicp_block& b, const PoseF& pose, const PrepassArgs& g,
                          float voxel, TileFn tile) {
    int ulx, uly, lrx, lry;
    float z0, z1;
    if (!project_block(b, pose, g, voxel, ulx, uly, lrx, lry, z0, z1)) return false;
    float dy = (float)lry - (float)uly + 1.0f;
    int ny = (int)ceilf(dy / 16.0f);
    if (ny <= 0) return false;
    const int xe = min(ulx + 15, lrx), ye = min(uly + 15, lry);
    const bool xx = ny >= 2 && lrx >= ulx + 16;
    const bool yy = ny >= 2 && lry >= uly + 16;
    const int lo = __float_as_int(z0), hi = __float_as_int(z1);
    for (int yi = uly; yi <= ye + (yy ? 1 : 0); ++yi) {
        int Y = (yi > ye) ? uly + 16 : yi;
        if (Y >= g.zrows) continue;
        for (int xi = ulx; xi <= xe + (xx ? 1 : 0); ++xi) {
            int X = (xi > xe) ? ulx + 16 : xi;
            if (X >= g.zcols) continue;
            tile(Y, X, lo, hi);
        }
    }
    return true;
}

// What a prepass thread reads before it can decide anything, loaded at once:
// the gate, the counters, the pose, its first visible block (at a clamped
// index, used only below the visible count) and its share of the fusion's
// per-wavefront counts. Each is a round trip to memory the previous launches
// wrote; issued one after another, as early returns would order them, they
// set the length of a launch this small.
struct PrepassIn {
    bool gated;
    uint32_t nvis, heap_used, fuse_sum;
    uint64_t visible_total, heap_total, fusions;
    PoseF pose;
    sicp_block b0;
};
// kThreads, kGrid: the launch's workgroup size and count (constants, so the
// kernel does not load them from the dispatch packet, one more round trip).
template <int kThreads, int kGrid>
SICP_DEV PrepassIn prepass_loads(const MapDev& m, const MapCounters* ctr,
                                 const sicp_block* visible, const PoseArg& pa, const int* gate,
                                 const uint32_t* fuse_counts) {
    PrepassIn in;
    const uint32_t i0 = blockIdx.x * kThreads + threadIdx.x;
    in.nvis = early_load(&ctr->visible);
    in.heap_used = early_load(&ctr->heap_used);
    in.visible_total = early_load(&ctr->visible_total);
    in.heap_total = early_load(&ctr->heap_total);
    in.fusions = early_load(&ctr->fusions);
    in.b0 = visible[i0 < (uint32_t)m.num_blocks ? i0 : 0u];
    static_assert(kThreads * kGrid >= kFuseBlocks * 4, "one fusion count per thread at most");
    in.fuse_sum = fuse_counts && i0 < (uint32_t)(kFuseBlocks * 4) ? fuse_counts[i0] : 0u;
    in.pose = load_pose(pa);
    in.gated = early_load(gate) == 0;  // never null: MapDev::one for an absent gate
    return in;
}

// The fusion's sums (fuse_end_kernel's, updated_voxels reset before the
// fusion) from its kFuseBlocks * 4 per-wavefront counts: integer sums, one
// atomic per wavefront; workgroup 0 also advances the running totals.
SICP_DEV void fusion_sums(MapCounters* ctr, const PrepassIn& in) {
    uint32_t c = in.fuse_sum;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if ((threadIdx.x & 63) == 0 && c) {
        atomicAdd(&ctr->updated_voxels, c);
        atomicAdd(&ctr->updated_total, (unsigned long long)c);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctr->visible_total = in.visible_total + in.nvis;
        ctr->heap_total = in.heap_total + in.heap_used;
        ctr->fusions = in.fusions + 1ull;
    }
}

SICP_DEV void count_render_blocks(MapCounters* ctr, uint32_t valid_blocks) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) valid_blocks += __shfl_xor(valid_blocks, off, 64);
    if ((threadIdx.x & 63) == 0 && valid_blocks) atomicAdd(&ctr->render_tiles, valid_blocks);
}

// The visible blocks of this thread (the first one preloaded), each with
// its tiles passed to `tile`; returns the number that produced tiles.
template <int kThreads, int kGrid, class TileFn>
SICP_DEV uint32_t prepass_blocks(const MapDev& m, const sicp_block* visible, const PrepassIn& in,
                                 const PrepassArgs& g, TileFn tile) {
    uint32_t valid_blocks = 0;
    const uint32_t stride = kGrid * kThreads;
    for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < in.nvis; i += stride)
        valid_blocks += block_tiles(i < stride ? in.b0 : visible[i], in.pose, g, m.voxel, tile);
    return valid_blocks;
}

// The tiles straight into the zRange images: two device-scope atomics per
// covered tile (the fallback for zRange images above kPrepassLdsTiles).
// One-wavefront workgroups: the visible blocks (a thread each) spread over
// more CUs than 256-thread groups would give them.
constexpr int kPrepassGrid = 2048;
__global__ __launch_bounds__(64) void prepass_kernel(MapDev m, MapCounters* ctr,
                                                     const sicp_block* visible, View<float> zmin,
                                                     View<float> zmax, PoseArg pa,
                                                     PrepassArgs g, const int* gate,
                                                     const uint32_t* fuse_counts) {
    const PrepassIn in = prepass_loads<64, kPrepassGrid>(m, ctr, visible, pa, gate, fuse_counts);
    if (in.gated) return;
    if (fuse_counts) fusion_sums(ctr, in);
    auto to_images = [&](int Y, int X, int lo, int hi) {
        atomicMin((int*)&zmin.at(Y, X), lo);
        atomicMax((int*)&zmax.at(Y, X), hi);
    };
    const uint32_t valid_blocks = prepass_blocks<64, kPrepassGrid>(m, visible, in, g, to_images);
    count_render_blocks(ctr, valid_blocks);
}

// The same with the workgroup's tiles gathered in LDS first: its 256
// consecutive visible blocks (heap-slot order, so mostly neighbours) cover
// overlapping tiles, and LDS atomics merge them; the workgroup then applies
// one atomic per touched tile and bound to the zRange images (device-scope
// atomics from eight XCDs are carried out beyond the L2s, one memory
// transaction each). min / max are order-independent, so the images are the
// same as the direct kernel's.
constexpr int kPrepassLdsTiles = 8000;  // 2 x 32000 bytes of LDS
constexpr int kPrepassLdsGrid = 512;
__global__ __launch_bounds__(256) void prepass_lds_kernel(MapDev m, MapCounters* ctr,
                                                          const sicp_block* visible,
                                                          View<float> zmin, View<float> zmax,
                                                          PoseArg pa, PrepassArgs g,
                                                          const int* gate,
                                                          const uint32_t* fuse_counts) {
    __shared__ int tmin[kPrepassLdsTiles], tmax[kPrepassLdsTiles];
    const PrepassIn in =
        prepass_loads<256, kPrepassLdsGrid>(m, ctr, visible, pa, gate, fuse_counts);
    if (in.gated) return;
    if (fuse_counts) fusion_sums(ctr, in);
    if (blockIdx.x * 256 >= in.nvis) return;  // no blocks for this workgroup
    const int ntiles = g.zcols * g.zrows;
    for (int t = threadIdx.x; t < ntiles; t += 256) {
        tmin[t] = 0x7fffffff;
        tmax[t] = 0;
    }
    __syncthreads();
    auto to_lds = [&](int Y, int X, int lo, int hi) {
        atomicMin(&tmin[Y * g.zcols + X], lo);
        atomicMax(&tmax[Y * g.zcols + X], hi);
    };
    const uint32_t valid_blocks =
        prepass_blocks<256, kPrepassLdsGrid>(m, visible, in, g, to_lds);
    count_render_blocks(ctr, valid_blocks);
    __syncthreads();
    for (int t = threadIdx.x; t < ntiles; t += 256) {
        const int lo = tmin[t], hi = tmax[t];
        if (lo == 0x7fffffff) continue;  // untouched (every touch sets both)
        const int Y = t / g.zcols, X = t - Y * g.zcols;
        atomicMin((int*)&zmin.at(Y, X), lo);
        atomicMax((int*)&zmax.at(Y, X), hi);
    }
}

// ------------------------------------------------------------------ raycast --
// Every march iteration is a dependent chain (address, lookup, voxel load,
// decision), run by all of the launch's wavefronts at once (about five share
// each SIMD), so voxel addressing is written for few instructions: floor
// once per distinct float coordinate, block = v >> 3 and
// local = v & 7 (the same values as voxelPosToBlockPos / voxelPosToLocalIdx,
// DeviceMap.cu:169-201, for every int), and one cache compare per block.
struct BlockCache {
    int x, y, z, slot;  // slot -1: empty
};

// make_int3 of one coordinate (VectorMath.h:36-42): the truncation, one less
// where it exceeds the value — the floor, for every float (NaN and values
// past the int range convert as the truncation does). v_floor_f32 and one
// conversion, the floor shared with the fraction of an interpolated read.
SICP_DEV int floor_i(float a) { return (int)floorf(a); }

SICP_DEV int local_of(int vx, int vy, int vz) { return ((vz & 7) << 6) | ((vy & 7) << 3) | (vx & 7); }

SICP_DEV bool cache_has(const BlockCache& c, int bx, int by, int bz) {
    return c.slot >= 0 && bx == c.x && by == c.y && bz == c.z;
}

// DeviceMap::FindVoxel(int3, cache, valid) (DeviceMap.cu:116-133) on integer
// voxel coordinates; the cache starts empty (the reference's default entry
// would match block (0,0,0)).
SICP_DEV long find_voxel_i(const MapDev& m, int vx, int vy, int vz, BlockCache& c, bool& valid) {
    const int bx = vx >> 3, by = vy >> 3, bz = vz >> 3;
    if (cache_has(c, bx, by, bz)) {
        valid = true;
        return (long)c.slot * kBlockVoxels + local_of(vx, vy, vz);
    }
    const int slot = map_lookup(m, bx, by, bz);
    if (slot < 0) {
        valid = false;
        return -1;
    }
    valid = true;
    c = BlockCache{bx, by, bz, slot};
    return (long)slot * kBlockVoxels + local_of(vx, vy, vz);
}

SICP_DEV float sdf_at(const MapDev& m, long k) { return k < 0 ? qnanf() : vox_sdf(m, (size_t)k); }

// One axis of an interpolated read centred at coordinate q: the voxel
// coordinates of q and q + 1 (the reference adds 1.0f to the float point)
// and the fraction q - floor(q).
struct AxisPair {
    int v0, v1;
    float frac;
};
SICP_DEV AxisPair axis_pair(float q) { return AxisPair{floor_i(q), floor_i(q + 1.0f), q - floorf(q)}; }

// Rendering::readSdfInterped (RenderScene.cu:310-343) from its eight corners, NaN
// for a missing block's, in the reference's order.
SICP_DEV float interp_blend(const float (&sd)[8], const AxisPair& X, const AxisPair& Y,
                            const AxisPair& Z) {
    const float fx = X.frac, fy = Y.frac, fz = Z.frac;
    float r0, r1, r2, r3;
    r0 = (1.0f - fx) * sd[0] + fx * sd[1];
    r1 = (1.0f - fx) * sd[2] + fx * sd[3];
    r2 = (1.0f - fy) * r0 + fy * r1;
    r0 = (1.0f - fx) * sd[4] + fx * sd[5];
    r1 = (1.0f - fx) * sd[6] + fx * sd[7];
    r3 = (1.0f - fy) * r0 + fy * r1;
    return (1.0f - fz) * r2 + fz * r3;
}
struct RayArgs {
    float invfx, invfy, cx, cy;
    int cols, rows;
    int tcols, trows;        // raycast_kernel: 8x8-pixel tiles across and down
    int first_pass_samples;  // the first pass's hand-over point (raycast_kernel only)
    int cube_margin;         // ray_cube_margin of it
};

// The ray of pixel (x, y) (RenderScene.cu:393-421): start point and unit
// direction in voxel units, start and end distances along it.
struct Ray {
    v3 start, dir;
    float dist_s, dist_e;
};
SICP_DEV bool ray_setup(const MapDev& m, float z0, float z1, const PoseF& pose, const RayArgs& g,
                        int x, int y, Ray& r) {
    if ((double)z1 < 1e-3 || (double)z0 < 1e-3 || isnan_(z0) || isnan_(z1)) return false;
    v3 p;
    p.z = z0;
    p.x = p.z * ((float)x - g.cx) * g.invfx;
    p.y = p.z * ((float)y - g.cy) * g.invfy;
    r.dist_s = norm(p) * m.voxel_inv;
    const v3 block_s = scale(add(mv(pose.R, p), pose.t), m.voxel_inv);
    p.z = z1;
    p.x = p.z * ((float)x - g.cx) * g.invfx;
    p.y = p.z * ((float)y - g.cy) * g.invfy;
    r.dist_e = norm(p) * m.voxel_inv;
    const v3 block_e = scale(add(mv(pose.R, p), pose.t), m.voxel_inv);
    r.dir = normalised(sub(block_e, block_s));
    r.start = block_s;
    return true;
}
SICP_DEV bool ray_setup(const MapDev& m, const View<float>& zmin, const View<float>& zmax,
                        const PoseF& pose, const RayArgs& g, int x, int y, Ray& r) {
    return ray_setup(m, zmin.at(y >> 3, x >> 3), zmax.at(y >> 3, x >> 3), pose, g, x, y, r);
}

// RayArgs::first_pass_samples is the number of samples one ray marches in
// the first pass; rays still marching then are handed to the second pass.
// Most rays end well before; the few that graze a surface for hundreds of
// one-voxel steps would otherwise set the length of the whole launch.

// ---- first pass: one lane per ray -----------------------------------------
// What bounds it: not bytes (it reads a tenth of what HBM could give it) but
// the instructions and dependent memory round trips of each wavefront's march;
// all wavefronts run at once (4800 at 640x480, up to six a SIMD), and the
// launch lasts as long as the slowest one. Written as the
// reference's loop, every iteration ran every path some lane needed — a
// table probe, an interpolated read with its block lookups, a plain step —
// 450 instructions and up to four dependent round trips, some 20 times. Here
// a lane that needs a table probe or an interpolated read waits while the
// others march on, and the waiting lanes are served together when enough of
// them wait: the same samples, each ray's in the same order. First pass at
// 640x480 / 5 mm 119 to 81 us, at 2 mm 174 to 134, 1280x720 / 4 mm (half)
// 221 to 143, 320x240 / 1 cm 95 to 59.
//
// Blocks are named by a 30-bit tag relative to the wavefront's own origin
// (10 bits an axis: a neighbour's tag is one addition away, and one compare
// tests the lane's cached block), and a missing block by the heap slot
// num_blocks, whose voxels are kept empty (NaN, weight 0), so that no read
// tests for it. Rays whose ends do not lie well inside the 1024-block cube around
// the wavefront's middle (16 m long at 2 mm voxels) are handed to the second
// pass from their first sample on (raycasts of such ranges, 640x480 / 2 mm: 1.6
// ms with depths to 12 m and 7.6 to 60 m; 10.4 and 54.6 as the reference's loop
// over both passes).
constexpr int kRayLdsEntries = 256;  // one 64-bit word each: tag + 1, slot
constexpr uint32_t kTagX = 1u, kTagY = 1u << 10, kTagZ = 1u << 20;
constexpr uint32_t kNoTag = 0xffffffffu;
// Samples of a one-voxel run read together, and the waiting lanes' share that
// has them served: measured (on other frames than above, and before the order
// of tiles below) at 640x480 / 5 mm, 2 mm, 1280x720 / 4 mm and 320x240 / 1 cm,
// first pass in us: two samples 92, 149, 160, 66; one 101, 153, 174, 74; three
// and four 110 to 118 (640x480). Serving the waiting lanes when they are a
// third of the marching ones, as above; only when none marches 135 (640x480);
// in every iteration 113; at half or a quarter the same within 1.
constexpr int kRayAhead = 2, kRayServe = 3;
// Workgroups go to the eight XCDs in turn, each with an L2 of its own:
// super-tiles of 8x8 tiles are given to one XCD, so that neighbouring rays
// find their blocks' lines there (1280x720 160 to 152 us, 320x240 66 to 64,
// the others the same; 4x4 and 2x2 gain less, 16x16 leaves XCDs uneven).
constexpr int kRaySuper = 8;

// The tag of block b relative to the wavefront's origin, and whether a point
// lies inside the cube that tags can name, `margin` blocks from its faces.
SICP_DEV uint32_t block_tag(i3 b, uint32_t otag) {
    return (uint32_t)b.x * kTagX + (uint32_t)b.y * kTagY + (uint32_t)b.z * kTagZ - otag;
}
SICP_DEV bool in_cube(v3 p, i3 o, int margin) {
    const uint32_t x = (uint32_t)((floor_i(p.x) >> 3) - o.x - margin),
                   y = (uint32_t)((floor_i(p.y) >> 3) - o.y - margin),
                   z = (uint32_t)((floor_i(p.z) >> 3) - o.z - margin);
    const uint32_t n = (uint32_t)(kTagSpan - 2 * margin);
    return (x < n) & (y < n) & (z < n);
}

// The wavefront's lookup table: answers of the hash table, missing blocks
// included. One wavefront per workgroup, so its accesses are ordered by its
// own instruction order; entries are written by atomic exchange, so lanes
// storing different blocks at one index leave one complete entry.
template <bool kTable> struct RayTable {
    unsigned long long* t;
    SICP_DEV static uint32_t index(uint32_t tag) { return (tag * 0x9E3779B1u) >> 24; }
    SICP_DEV bool get(uint32_t tag, uint32_t& slot) const {
        if (!kTable) return false;
        const unsigned long long e = t[index(tag)];
        slot = (uint32_t)(e >> 32);
        return (uint32_t)e == tag + 1u;
    }
    SICP_DEV void put(uint32_t tag, uint32_t slot) const {
        if (kTable)
            atomicExch(&t[index(tag)], ((unsigned long long)slot << 32) | (unsigned long long)(tag + 1u));
    }
};

// The hash table's answer, num_blocks for a missing block.
SICP_DEV uint32_t probe_slot(const MapDev& m, int bx, int by, int bz) {
    const int s = map_lookup(m, bx, by, bz);
    return s < 0 ? (uint32_t)m.num_blocks : (uint32_t)s;
}

// sdf (and weight) of a voxel of a slot that exists or is num_blocks.
SICP_DEV float slot_sdf(const MapDev& m, uint32_t slot, uint32_t local) {
    return vox_sdf(m, (size_t)slot * kBlockVoxels + local);
}

// The slots of the blocks (b & 1, b >> 1 & 1, b >> 2) past the block with tag
// `tag0` and coordinates b0, along the axes where `n` is set; the others of
// `s` are not written. `known`: s[0] is given. The table is asked for all of
// them first, then the hash table for those it does not hold.
template <bool kTable>
SICP_DEV void box_slots(const MapDev& m, const RayTable<kTable>& lds, uint32_t tag0, i3 b0,
                        bool nx, bool ny, bool nz, bool known, uint32_t (&s)[8]) {
    uint32_t miss = 0;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool need = (!(b & 1) || nx) && (!(b & 2) || ny) && (!(b & 4) || nz) &&
                          (b != 0 || !known);
        if (need) {
            const uint32_t tag = tag0 + ((b & 1) ? kTagX : 0u) + ((b & 2) ? kTagY : 0u) +
                                 ((b & 4) ? kTagZ : 0u);
            if (!lds.get(tag, s[b])) miss |= 1u << b;
        }
    }
    while (miss) {
        const int b = __ffs((int)miss) - 1;
        miss &= miss - 1u;
        const int dx = b & 1, dy = (b >> 1) & 1, dz = b >> 2;
        const uint32_t sl = probe_slot(m, b0.x + dx, b0.y + dy, b0.z + dz);
        lds.put(tag0 + (uint32_t)dx * kTagX + (uint32_t)dy * kTagY + (uint32_t)dz * kTagZ, sl);
#pragma unroll
        for (int q = 0; q < 8; ++q) s[q] = q == b ? sl : s[q];
    }
}

// Rendering::readSdfInterped (RenderScene.cu:310-343) at p. `known`: the
// block of p's own voxel is `slot`.
template <bool kTable>
SICP_DEV float ray_interp(const MapDev& m, const RayTable<kTable>& lds, v3 p, uint32_t otag,
                          bool known, uint32_t slot) {
    const AxisPair X = axis_pair(p.x), Y = axis_pair(p.y), Z = axis_pair(p.z);
    const i3 b0{X.v0 >> 3, Y.v0 >> 3, Z.v0 >> 3};
    const bool nx = (X.v1 >> 3) != b0.x, ny = (Y.v1 >> 3) != b0.y, nz = (Z.v1 >> 3) != b0.z;
    uint32_t s[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) s[b] = slot;
    box_slots<kTable>(m, lds, block_tag(b0, otag), b0, nx, ny, nz, known, s);
    const uint32_t ox[2] = {(uint32_t)X.v0 & 7u, (uint32_t)X.v1 & 7u};
    const uint32_t oy[2] = {((uint32_t)Y.v0 & 7u) << 3, ((uint32_t)Y.v1 & 7u) << 3};
    const uint32_t oz[2] = {((uint32_t)Z.v0 & 7u) << 6, ((uint32_t)Z.v1 & 7u) << 6};
    float sd[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int cx = i & 1, cy = (i >> 1) & 1, cz = i >> 2;
        // selects, so the slots stay in registers
        const uint32_t a00 = cx && nx ? s[1] : s[0], a10 = cx && nx ? s[3] : s[2];
        const uint32_t a01 = cx && nx ? s[5] : s[4], a11 = cx && nx ? s[7] : s[6];
        const uint32_t c0 = cy && ny ? a10 : a00, c1 = cy && ny ? a11 : a01;
        sd[i] = slot_sdf(m, cz && nz ? c1 : c0, ox[cx] | oy[cy] | oz[cz]);
    }
    return interp_blend(sd, X, Y, Z);
}

// One axis of the normal's reads: the voxel coordinates from the lower
// corner of the read at -1 to the upper corner of the read at +1, four
// consecutive ones. False where rounding makes them differ (p + 1 or p - 1
// rounded to an integer that p's own floor does not lead to).
struct NormalAxis {
    int v;             // the first; the others follow
    float fm, f0, fp;  // the fractions of the reads at -1, 0, +1
};
SICP_DEV bool normal_axis(float p, NormalAxis& a) {
    const AxisPair lo = axis_pair(p + -1.0f), mid = axis_pair(p), hi = axis_pair(p + 1.0f);
    a = NormalAxis{lo.v0, lo.frac, mid.frac, hi.frac};
    const int v = lo.v0;
    return lo.v1 == v + 1 && mid.v0 == v + 1 && mid.v1 == v + 2 && hi.v0 == v + 2 &&
           hi.v1 == v + 3;
}

// Rendering::readNormal (RenderScene.cu:345-378): six interpolated reads
// around p share 32 voxels of a 4x4x4 box in at most eight blocks, each
// looked up and read once. A missing block reads NaN, so a read's value alone
// decides. False without a normal.
template <bool kTable>
SICP_DEV void ray_normal_reads(const MapDev& m, const RayTable<kTable>& lds,
                               const NormalAxis (&A)[3], uint32_t otag, float (&r)[6]) {
    const i3 b0{A[0].v >> 3, A[1].v >> 3, A[2].v >> 3};
    const bool nx = ((A[0].v + 3) >> 3) != b0.x, ny = ((A[1].v + 3) >> 3) != b0.y,
               nz = ((A[2].v + 3) >> 3) != b0.z;
    uint32_t s[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) s[b] = 0u;
    box_slots<kTable>(m, lds, block_tag(b0, otag), b0, nx, ny, nz, false, s);
    // coordinate i of an axis: its offset within its block, and whether that
    // is the second block
    uint32_t o[3][4];
    bool up[3][4];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int bb = a == 0 ? b0.x : (a == 1 ? b0.y : b0.z);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o[a][i] = ((uint32_t)(A[a].v + i) & 7u) << (3 * a);
            up[a][i] = ((A[a].v + i) >> 3) != bb;
        }
    }
    float d[4][4][4];  // [z][y][x]; only the 32 the reads touch are loaded
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const uint32_t s00 = up[0][x] ? s[1] : s[0], s10 = up[0][x] ? s[3] : s[2];
        const uint32_t s01 = up[0][x] ? s[5] : s[4], s11 = up[0][x] ? s[7] : s[6];
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const uint32_t t0 = up[1][y] ? s10 : s00, t1 = up[1][y] ? s11 : s01;
#pragma unroll
            for (int z = 0; z < 4; ++z) {
                const int outer = (x == 0 || x == 3) + (y == 0 || y == 3) + (z == 0 || z == 3);
                if (outer > 1) continue;
                d[z][y][x] = slot_sdf(m, up[2][z] ? t1 : t0, o[0][x] | o[1][y] | o[2][z]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {  // +x, -x, +y, -y, +z, -z
        const int a = k >> 1;
        const int x = a == 0 ? ((k & 1) ? 0 : 2) : 1, y = a == 1 ? ((k & 1) ? 0 : 2) : 1,
                  z = a == 2 ? ((k & 1) ? 0 : 2) : 1;
        AxisPair X{0, 0, A[0].f0}, Y{0, 0, A[1].f0}, Z{0, 0, A[2].f0};
        (a == 0 ? X : (a == 1 ? Y : Z)).frac = (k & 1) ? A[a].fm : A[a].fp;
        const float sd[8] = {d[z][y][x],         d[z][y][x + 1],         d[z][y + 1][x],
                             d[z][y + 1][x + 1], d[z + 1][y][x],         d[z + 1][y][x + 1],
                             d[z + 1][y + 1][x], d[z + 1][y + 1][x + 1]};
        r[k] = interp_blend(sd, X, Y, Z);
    }
}
template <bool kTable>
SICP_DEV bool ray_normal(const MapDev& m, const RayTable<kTable>& lds, v3 p, uint32_t otag,
                         const PoseF& pose, v3& n) {
    float r[6];
    NormalAxis A[3];
    const bool ax = normal_axis(p.x, A[0]), ay = normal_axis(p.y, A[1]),
               az = normal_axis(p.z, A[2]);
    if (ax && ay && az) {
        ray_normal_reads<kTable>(m, lds, A, otag, r);
    } else {
#pragma unroll 1
        for (int k = 0; k < 6; ++k) {
            const float d = (k & 1) ? -1.0f : 1.0f;
            const v3 q{k < 2 ? p.x + d : p.x, (k >> 1) == 1 ? p.y + d : p.y, k > 3 ? p.z + d : p.z};
            const float v = ray_interp<kTable>(m, lds, q, otag, false, 0u);
#pragma unroll
            for (int j = 0; j < 6; ++j) r[j] = j == k ? v : r[j];
        }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k)
        if (isnan_(r[k]) || r[k] == 1.0f) return false;
    n = normalised(mv(pose.Rinv, mk(r[0] - r[1], r[2] - r[3], r[4] - r[5])));
    return true;
}

// 8x8-pixel wavefronts (the zRange tile).
template <bool kHalf, bool kTable>
__global__ __launch_bounds__(64, 5) void raycast_kernel(MapDev map, View<float4> vmap,
                                                     View<float4> nmap, View<float> zmin,
                                                     View<float> zmax, PoseArg pa, RayArgs g,
                                                     const int* gate, const uint32_t* nonempty) {
    MapDev m = map;
    m.half = kHalf;  // a constant: no test of the form per read
    constexpr uint32_t kSuperTiles = kRaySuper * kRaySuper;
    const uint32_t xcd = blockIdx.x & 7u, turn = blockIdx.x >> 3;
    const uint32_t super = turn / kSuperTiles * 8u + xcd, in = turn % kSuperTiles;
    const uint32_t across = ((uint32_t)g.tcols + kRaySuper - 1u) / kRaySuper;
    const int bx = (int)(super % across * kRaySuper + in % kRaySuper);
    const int by = (int)(super / across * kRaySuper + in / kRaySuper);
    if (bx >= g.tcols || by >= g.trows) return;
    const int x = bx * 8 + (threadIdx.x & 7);
    const int y = by * 8 + (threadIdx.x >> 3);
    // the tile's depth range, the pose and the gates, loaded together
    const int ty = min(y, g.rows - 1) >> 3, tx = min(x, g.cols - 1) >> 3;
    const float z0 = early_load(&zmin.at(ty, tx)), z1 = early_load(&zmax.at(ty, tx));
    // gate and nonempty (CreateRenderingBlocks returned true) are never null
    // here: the launch passes MapDev::one for an absent one
    const int open = early_load(gate);
    const uint32_t any = early_load(nonempty);
    const PoseF pose = load_pose(pa);
    if ((open == 0) | (any == 0u)) return;
    __shared__ unsigned long long entries[kTable ? kRayLdsEntries : 1];
    if (kTable) {
#pragma unroll
        for (int i = 0; i < kRayLdsEntries / 64; ++i) entries[threadIdx.x + 64 * i] = 0ull;
    }
    const RayTable<kTable> lds{entries};
    const bool inside = x < g.cols && y < g.rows;
    const float nan = qnanf();
    float4 vout = make_float4(nan, nan, nan, nan);
    float4 nout = vout;
    Ray ray{};
    const bool hits = inside && ray_setup(m, z0, z1, pose, g, x, y, ray);
    // kMarch: takes samples; kProbe, kInterp: waits for a table probe or an
    // interpolated read of its current sample; kEnd: the loop is over
    enum { kMarch, kProbe, kInterp, kEnd };
    int status = hits ? kMarch : kEnd;
    bool deferred = false, back_face = false, crossed = false;
    v3 result{0.f, 0.f, 0.f};
    float dist_s = 0.f, sdf = 1.0f, prev_sdf = 1.0f;
    // The tags' origin: the block in the middle of the first ray, less half
    // the span. A ray whose ends lie ray_cube_margin from the faces stays in
    // the cube for its samples of this pass.
    uint32_t otag = 0;
    i3 o{0, 0, 0};
    {
        const unsigned long long some = __ballot(hits);
        if (some) {
            v3 mid{0.f, 0.f, 0.f};
            if (hits) {
                result = ray.start;
                dist_s = ray.dist_s;
                mid = add(ray.start, scale(0.5f * (ray.dist_e - ray.dist_s), ray.dir));
            }
            const int src = __ffsll((long long)some) - 1;
            o.x = (__builtin_amdgcn_readlane(floor_i(mid.x), src) >> 3) - kTagSpan / 2;
            o.y = (__builtin_amdgcn_readlane(floor_i(mid.y), src) >> 3) - kTagSpan / 2;
            o.z = (__builtin_amdgcn_readlane(floor_i(mid.z), src) >> 3) - kTagSpan / 2;
            otag = (uint32_t)o.x * kTagX + (uint32_t)o.y * kTagY + (uint32_t)o.z * kTagZ;
            if (hits) {
                const v3 e = add(ray.start, scale(ray.dist_e - ray.dist_s, ray.dir));
                if (!in_cube(ray.start, o, g.cube_margin) || !in_cube(e, o, g.cube_margin)) {
                    deferred = true;
                    status = kEnd;
                }
            }
        }
    }
    const v3 dir8 = scale((float)kBlockSide, ray.dir);
    uint32_t tag = kNoTag, slot = 0;  // the lane's last lookup
    int iters = 0;
    for (;;) {
        for (;;) {
            const int marching = __popcll(__ballot(status == kMarch));
            const int waiting = __popcll(__ballot(status == kProbe || status == kInterp));
            if (marching == 0 || waiting * kRayServe > marching) break;
            if (status != kMarch) continue;
            if (!(dist_s < ray.dist_e)) {
                status = kEnd;
            } else if (iters == g.first_pass_samples) {
                deferred = true;
                status = kEnd;
            } else {
                const int vx = floor_i(result.x), vy = floor_i(result.y), vz = floor_i(result.z);
                const uint32_t t = block_tag(i3{vx >> 3, vy >> 3, vz >> 3}, otag);
                bool found = t == tag;
                if (!found) {
                    found = lds.get(t, slot);
                    tag = found ? t : kNoTag;
                }
                if (!found) {
                    status = kProbe;
                } else if (slot == (uint32_t)m.num_blocks) {  // no block here
                    prev_sdf = sdf;
                    sdf = nan;
                    ++iters;
                    result = add(result, dir8);
                    dist_s += (float)kBlockSide;
                } else {
                    // This sample and those that one-voxel steps would take
                    // next in the same block, their loads in flight together
                    v3 P[kRayAhead];
                    bool same[kRayAhead];
                    float s[kRayAhead];
                    uint32_t wt[kRayAhead];
                    P[0] = result;
                    same[0] = true;
                    uint32_t local = (uint32_t)local_of(vx, vy, vz);
#pragma unroll
                    for (int j = 0; j < kRayAhead; ++j) {
                        if (j > 0) {
                            P[j] = add(P[j - 1], ray.dir);
                            const int wx = floor_i(P[j].x), wy = floor_i(P[j].y),
                                      wz = floor_i(P[j].z);
                            same[j] = same[j - 1] &&
                                      (((wx ^ vx) | (wy ^ vy) | (wz ^ vz)) & ~7) == 0;
                            local = same[j] ? (uint32_t)local_of(wx, wy, wz) : local;
                        }
                        vox_load(m, (size_t)slot * kBlockVoxels + local, s[j], wt[j]);
                    }
                    bool plain = true;
#pragma unroll
                    for (int j = 0; j < kRayAhead; ++j) {
                        if (j > 0)
                            plain = plain && same[j] && dist_s < ray.dist_e &&
                                    iters != g.first_pass_samples;
                        if (!plain) continue;
                        prev_sdf = sdf;
                        sdf = s[j];
                        const bool valid = wt[j] != 0u;
                        const bool band = valid && sdf <= 0.1f && sdf >= -0.5f;
                        back_face = valid && prev_sdf < 0.f && sdf >= 0.f;
                        crossed = valid && prev_sdf > 0.f && sdf <= 0.f;
                        plain = valid && !band && !back_face && !crossed;
                        if (band) {
                            status = kInterp;
                        } else {
                            ++iters;
                            if (back_face || crossed) {
                                status = kEnd;
                            } else {
                                const float step = valid ? 1.0f : (float)kBlockSide;
                                result = add(result, scale(step, ray.dir));
                                dist_s += step;
                            }
                        }
                    }
                }
            }
        }
        if (!__any(status != kEnd)) break;
        if (status == kProbe) {
            // In a run of missing blocks the block of the next block-width
            // step is looked up too, both buckets' reads in flight at once
            const bool run = isnan_(sdf);
            const v3 q = add(result, dir8);
            const i3 b{floor_i(result.x) >> 3, floor_i(result.y) >> 3, floor_i(result.z) >> 3};
            i3 c{floor_i(q.x) >> 3, floor_i(q.y) >> 3, floor_i(q.z) >> 3};
            if (!run) c = b;
            const Probe pb = probe_load(m.table, m.nb, m.nb_mask, b.x, b.y, b.z);
            const Probe pc = probe_load(m.table, m.nb, m.nb_mask, c.x, c.y, c.z);
            const int sb = probe_result(pb, m.excess);
            tag = block_tag(b, otag);
            slot = sb < 0 ? (uint32_t)m.num_blocks : (uint32_t)sb;
            lds.put(tag, slot);
            if (run && sb < 0) {  // this sample: no block here
                const int sc = probe_result(pc, m.excess);
                ++iters;
                result = q;
                dist_s += (float)kBlockSide;
                tag = block_tag(c, otag);
                slot = sc < 0 ? (uint32_t)m.num_blocks : (uint32_t)sc;
                lds.put(tag, slot);
            }
            status = kMarch;
        }
        if (status == kInterp) {
            sdf = ray_interp<kTable>(m, lds, result, otag, true, slot);
            ++iters;
            back_face = prev_sdf < 0.f && sdf >= 0.f;
            crossed = prev_sdf > 0.f && sdf <= 0.f;
            if (back_face || crossed) {
                status = kEnd;
            } else {
                result = add(result, ray.dir);
                dist_s += 1.0f;
                status = kMarch;
            }
        }
    }
    if (hits && !deferred && !back_face && sdf <= 0.0f) {
        // the state the second pass would resume from, should it be needed
        const v3 at = result;
        const float sdf_in = crossed ? prev_sdf : sdf;
        result = add(result, scale(sdf * m.step_scale, ray.dir));
        bool ok = in_cube(result, o, kTagReach);
        if (ok) {
            sdf = ray_interp<kTable>(m, lds, result, otag, false, 0u);
            result = add(result, scale(sdf * m.step_scale, ray.dir));
            // (a NaN position has no normal: its reads would be NaN)
            const bool number = !isnan_(result.x) && !isnan_(result.y) && !isnan_(result.z);
            ok = !number || in_cube(result, o, kTagReach);
            v3 normal;
            if (ok && number && ray_normal<kTable>(m, lds, result, otag, pose, normal)) {
                v3 r = mv(pose.Rinv, sub(scale(result, m.voxel), pose.t));
                vout = make_float4(r.x, r.y, r.z, 1.0f);
                nout = make_float4(normal.x, normal.y, normal.z, 1.0f);
            }
        }
        if (!ok) {
            deferred = true;
            result = at;
            sdf = sdf_in;
        }
    }
    // Hand-over: one queue reservation per wavefront.
    const unsigned long long mask = __ballot(deferred);
    if (mask) {
        const int lane = threadIdx.x & 63;
        const int leader = __ffsll((long long)mask) - 1;
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(m.rq_count, (uint32_t)__popcll(mask));
        base = __shfl(base, leader, 64);
        if (deferred) {
            const uint32_t q = base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
            if (q < m.rq_cap)
                m.rq[q] = RayState{y * g.cols + x, result.x, result.y, result.z, dist_s, sdf,
                                   ray.dir.x, ray.dir.y, ray.dir.z, ray.dist_e, {0, 0}};
        }
        if (deferred) return;  // the second pass writes this pixel
    }
    if (!inside) return;
    vmap.at(y, x) = vout;
    nmap.at(y, x) = nout;
}

// ---- second pass: kRayGroup lanes per ray --------------------------------
// Lane k of a group evaluates the sample the scalar loop reaches after k more
// one-voxel steps (result + dir added k times, as the loop adds it). A ballot
// finds the first sample where the scalar loop would do anything but a plain
// one-voxel step — out of range, missing or empty voxel, the interpolation
// band, a sign change — and the group applies the loop body there exactly;
// the samples before it are one-voxel steps taken in one go. Interpolated
// reads and the normal split their corners over the group's lanes.
constexpr int kRayGroup = 8;
static_assert(48 % kRayGroup == 0 && kRayGroup >= 8, "corner split of the normal read");

template <class T> SICP_DEV T gshfl(T v, int src) { return __shfl(v, src, kRayGroup); }
SICP_DEV v3 gshfl3(v3 v, int src) { return v3{gshfl(v.x, src), gshfl(v.y, src), gshfl(v.z, src)}; }

// Rendering::readSdfInterped with corner c on lane c of the group; every lane
// returns the blended value and the validity of the last lookup.
SICP_DEV float coop_interp(const MapDev& m, v3 pt, int k, BlockCache& c, bool& valid) {
    const AxisPair X = axis_pair(pt.x), Y = axis_pair(pt.y), Z = axis_pair(pt.z);
    float mine = qnanf();
    bool ok = false;
    if (k < 8) {
        long idx = find_voxel_i(m, (k & 1) ? X.v1 : X.v0, (k & 2) ? Y.v1 : Y.v0,
                                (k & 4) ? Z.v1 : Z.v0, c, ok);
        mine = sdf_at(m, idx);
    }
    float sd[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sd[i] = gshfl(mine, i);
    valid = gshfl((int)ok, 7) != 0;
    const float fx = X.frac, fy = Y.frac, fz = Z.frac;
    float r0, r1, r2, r3;
    r0 = (1.0f - fx) * sd[0] + fx * sd[1];
    r1 = (1.0f - fx) * sd[2] + fx * sd[3];
    r2 = (1.0f - fy) * r0 + fy * r1;
    r0 = (1.0f - fx) * sd[4] + fx * sd[5];
    r1 = (1.0f - fx) * sd[6] + fx * sd[7];
    r3 = (1.0f - fy) * r0 + fy * r1;
    return (1.0f - fz) * r2 + fz * r3;
}

// Rendering::readNormal with its 48 corners spread over the group's lanes.
SICP_DEV bool coop_normal(const MapDev& m, v3 pt, int k, BlockCache& c, const PoseF& pose,
                          v3& n) {
    const AxisPair xm = axis_pair(pt.x + -1.0f), x0 = axis_pair(pt.x), xp = axis_pair(pt.x + 1.0f);
    const AxisPair ym = axis_pair(pt.y + -1.0f), y0 = axis_pair(pt.y), yp = axis_pair(pt.y + 1.0f);
    const AxisPair zm = axis_pair(pt.z + -1.0f), z0 = axis_pair(pt.z), zp = axis_pair(pt.z + 1.0f);
    constexpr int kPer = 48 / kRayGroup;  // corners per lane
    float val[kPer];
    int ok[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int q = k + kRayGroup * j;  // corner q of the 48: read q / 8, corner q % 8
        const int i = q >> 3, cc = q & 7;
        const AxisPair X = i == 0 ? xp : (i == 1 ? xm : x0);
        const AxisPair Y = i == 2 ? yp : (i == 3 ? ym : y0);
        const AxisPair Z = i == 4 ? zp : (i == 5 ? zm : z0);
        bool v;
        long idx = find_voxel_i(m, (cc & 1) ? X.v1 : X.v0, (cc & 2) ? Y.v1 : Y.v0,
                                (cc & 4) ? Z.v1 : Z.v0, c, v);
        val[j] = sdf_at(m, idx);
        ok[j] = v ? 1 : 0;
    }
    float s[6];
    bool valid[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        float sd[8];
#pragma unroll
        for (int cc = 0; cc < 8; ++cc) {
            const int q = i * 8 + cc;
            sd[cc] = gshfl(val[q / kRayGroup], q % kRayGroup);
        }
        valid[i] = gshfl(ok[(i * 8 + 7) / kRayGroup], (i * 8 + 7) % kRayGroup) != 0;
        const AxisPair X = i == 0 ? xp : (i == 1 ? xm : x0);
        const AxisPair Y = i == 2 ? yp : (i == 3 ? ym : y0);
        const AxisPair Z = i == 4 ? zp : (i == 5 ? zm : z0);
        const float fx = X.frac, fy = Y.frac, fz = Z.frac;
        float r0, r1, r2, r3;
        r0 = (1.0f - fx) * sd[0] + fx * sd[1];
        r1 = (1.0f - fx) * sd[2] + fx * sd[3];
        r2 = (1.0f - fy) * r0 + fy * r1;
        r0 = (1.0f - fx) * sd[4] + fx * sd[5];
        r1 = (1.0f - fx) * sd[6] + fx * sd[7];
        r3 = (1.0f - fy) * r0 + fy * r1;
        s[i] = (1.0f - fz) * r2 + fz * r3;
    }
#pragma unroll
    for (int i = 0; i < 6; ++i)
        if (isnan_(s[i]) || s[i] == 1.0f || !valid[i]) return false;
    n = normalised(mv(pose.Rinv, mk(s[0] - s[1], s[2] - s[3], s[4] - s[5])));
    return true;
}

// The march of a ray by its group of lanes, from any state of the loop: on
// return the state with which the loop ends, or back_face. `k`, `interp` and
// `steps`: the last sample's voxel index (-1: no block), whether it was an
// interpolated read, and the sum of the steps taken (the adjoint's).
struct CoopState {
    v3 result;
    float dist_s, sdf, steps;
    bool back_face, interp;
    long k;
    BlockCache cache;
};
SICP_DEV void coop_march(const MapDev& m, const Ray& ray, int k, int gbase, CoopState& s) {
    const v3 dir8 = scale((float)kBlockSide, ray.dir);
    // After a missing or empty voxel the lanes hold the block-width steps'
    // samples instead, until one of them is a voxel (which the next turn takes).
    bool run = false;
    while (s.dist_s < ray.dist_e) {
        const v3 d = run ? dir8 : ray.dir;
        const float step = run ? (float)kBlockSide : 1.0f;
        v3 P = s.result;
        float D = s.dist_s;
#pragma unroll
        for (int j = 0; j < kRayGroup - 1; ++j)
            if (j < k) {
                P = add(P, d);
                D += step;
            }
        const bool inr = D < ray.dist_e;
        float sv = qnanf();
        int exists = 0, wok = 0;
        long idx = -1;
        if (inr) {
            bool v;
            idx = find_voxel_i(m, floor_i(P.x), floor_i(P.y), floor_i(P.z), s.cache, v);
            if (idx >= 0) {
                uint32_t wt;
                vox_load(m, (size_t)idx, sv, wt);
                exists = 1;
                wok = wt != 0u;
            }
        }
        float sp = __shfl_up(sv, 1, kRayGroup);
        if (k == 0) sp = s.sdf;
        const bool band = wok && sv <= 0.1f && sv >= -0.5f;
        const bool cross = wok && !band && ((sp < 0.f && sv >= 0.f) || (sp > 0.f && sv <= 0.f));
        const bool event = run ? !inr || wok : !inr || !wok || band || cross;
        const uint32_t gm = (uint32_t)(__ballot(event) >> gbase) & ((1u << kRayGroup) - 1u);
        if (gm == 0u) {  // kRayGroup steps
            s.result = add(gshfl3(P, kRayGroup - 1), d);
            s.dist_s = gshfl(D, kRayGroup - 1) + step;
            s.sdf = gshfl(sv, kRayGroup - 1);
            s.k = gshfl(idx, kRayGroup - 1);
            s.steps += step * (float)kRayGroup;
            s.interp = false;
            continue;
        }
        const int ks = __ffs(gm) - 1;
        s.result = gshfl3(P, ks);
        s.dist_s = gshfl(D, ks);
        s.steps += step * (float)ks;
        const float prev = gshfl(sp, ks);
        const long k_prev = gshfl(idx, ks > 0 ? ks - 1 : 0);
        if (ks > 0) {
            s.k = k_prev;
            s.interp = false;
        }
        s.sdf = prev;
        if (!gshfl((int)inr, ks)) break;  // the loop condition fails here
        if (run) {
            run = false;
            continue;
        }
        s.k = gshfl(idx, ks);
        const float sk = gshfl(sv, ks);
        if (!gshfl(wok, ks)) {  // missing block (NaN) or empty voxel: block-width step
            s.sdf = gshfl(exists, ks) ? sk : qnanf();
            s.interp = false;
            s.result = add(s.result, dir8);
            s.dist_s += (float)kBlockSide;
            s.steps += (float)kBlockSide;
            run = true;
            continue;
        }
        float s1 = sk;
        s.interp = gshfl((int)band, ks) != 0;
        if (s.interp) {
            bool v;
            s1 = coop_interp(m, s.result, k, s.cache, v);
        }
        s.sdf = s1;
        if (prev < 0.f && s1 >= 0.f) {
            s.back_face = true;
            break;
        }
        if (prev > 0.f && s1 <= 0.f) break;
        s.result = add(s.result, ray.dir);
        s.dist_s += 1.0f;
        s.steps += 1.0f;
    }
}

constexpr int kRayLongThreads = 256;
__global__ __launch_bounds__(kRayLongThreads) void raycast_long_kernel(
    MapDev m, View<float4> vmap, View<float4> nmap, View<float> zmin, View<float> zmax, PoseArg pa,
    RayArgs g, const int* gate, const uint32_t* nonempty) {
    constexpr uint32_t kGroupsPerWg = kRayLongThreads / kRayGroup;
    const uint32_t i0 = blockIdx.x * kGroupsPerWg + (threadIdx.x / kRayGroup);
    // the queue's count, this group's first entry (at a clamped index, used
    // only below the count) and the gates, loaded together
    const uint32_t queued = early_load(m.rq_count);
    const RayState st0 = m.rq[i0 < m.rq_cap ? i0 : 0u];
    const int open = early_load(gate);  // gate and nonempty: never null here
    const uint32_t any = early_load(nonempty);
    if ((open == 0) | (any == 0u)) return;
    const uint32_t n = min(queued, m.rq_cap);
    const int k = threadIdx.x & (kRayGroup - 1);
    const int gbase = (threadIdx.x & 63) & ~(kRayGroup - 1);  // first lane of the group
    const uint32_t groups = gridDim.x * kGroupsPerWg;
    const float nan = qnanf();
    for (uint32_t i = i0; i < n; i += groups) {
        const RayState st = i == i0 ? st0 : m.rq[i];
        const int x = st.px % g.cols, y = st.px / g.cols;
        Ray ray;  // the first pass's ray_setup
        ray.dir = v3{st.dx, st.dy, st.dz};
        ray.dist_e = st.dist_e;
        CoopState c{v3{st.rx, st.ry, st.rz}, st.dist_s, st.sdf, 0.f, false, false, -1,
                    BlockCache{0, 0, 0, -1}};
        coop_march(m, ray, k, gbase, c);
        v3 result = c.result;
        float sdf = c.sdf;
        float4 vout = make_float4(nan, nan, nan, nan);
        float4 nout = vout;
        if (!c.back_face && sdf <= 0.0f) {
            float step = sdf * m.step_scale;
            result = add(result, scale(step, ray.dir));
            bool v;
            sdf = coop_interp(m, result, k, c.cache, v);
            step = sdf * m.step_scale;
            result = add(result, scale(step, ray.dir));
            v3 normal;
            const PoseF pose = load_pose(pa);  // here: held through the march it spills
            if (coop_normal(m, result, k, c.cache, pose, normal)) {
                v3 r = mv(pose.Rinv, sub(scale(result, m.voxel), pose.t));
                vout = make_float4(r.x, r.y, r.z, 1.0f);
                nout = make_float4(normal.x, normal.y, normal.z, 1.0f);
            }
        }
        if (k == 0) {
            vmap.at(y, x) = vout;
            nmap.at(y, x) = nout;
        }
    }
}

__global__ void ray_queue_reset_kernel(uint32_t* count) { *count = 0u; }

// ------------------------------------------------------------------ adjoint --
// The raycast's vertex and normal as functions of the camera pose and of the
// TSDF values, with the zRange images and every discrete decision of the
// march held fixed. Per sampled pixel the march is recomputed (nothing is
// stored by the forward pass), then the chain
//   r0 = block_s + M dir                      (M: the march's summed steps)
//   r1 = r0 + k s0 dir, s0 = F(r0) or raw voxel (k: stepScale)
//   r2 = r1 + k s1 dir, s1 = F(r1)
//   v  = R^T (voxel r2 - t)
//   n  = normalised(R^T g), g_a = F(r2 + e_a) - F(r2 - e_a)
// is run backwards (F: the trilinear read). The pose perturbation is
// T' = T exp(xi), xi = (translation, rotation) in the camera frame:
// R' = R (I + [w]x), t' = t + R v.

// Eight lanes share a pixel (kRayGroup): they march its ray together, hold a
// corner each of every trilinear read, and scatter its gradient; the values
// and derivatives that follow from the corners are formed by every lane alike.
// One thread per pixel left 160 wavefronts on 1024 SIMDs, each a chain of
// 32000 instructions and 900 dependent reads: 226 us for 10000 pixels at
// 1280x720 / 2 mm, 51 now (500 pixels with the launch's own time 161 and 48,
// 200000 827 and 470, every pixel 2918 and 1969).

// A trilinear read (readSdfInterped, RenderScene.cu:310-343) with this lane's
// corner voxel and weight and the read's gradient in voxel units. The value
// is formed exactly as the forward read forms it.
struct TriRead {
    long k;   // -1: missing
    float w;
    v3 grad;
    float val;
    bool ok;  // every corner exists, the value is not NaN
};
// The corner's lookup, its bucket's read in flight, then the read's rest.
struct TriProbe {
    AxisPair X, Y, Z;
    Probe p;
    int local;
};
SICP_DEV TriProbe tri_probe(const MapDev& m, v3 q, int k) {
    TriProbe t{axis_pair(q.x), axis_pair(q.y), axis_pair(q.z), Probe{}, 0};
    const int vx = (k & 1) ? t.X.v1 : t.X.v0, vy = (k & 2) ? t.Y.v1 : t.Y.v0,
              vz = (k & 4) ? t.Z.v1 : t.Z.v0;
    t.p = probe_load(m.table, m.nb, m.nb_mask, vx >> 3, vy >> 3, vz >> 3);
    t.local = local_of(vx, vy, vz);
    return t;
}
SICP_DEV void tri_corner(const MapDev& m, const TriProbe& t, long& k, float& sd) {
    const int slot = probe_result(t.p, m.excess);
    k = slot < 0 ? -1 : (long)slot * kBlockVoxels + t.local;
    const float v = vox_sdf(m, slot < 0 ? 0 : (size_t)k);
    sd = slot < 0 ? qnanf() : v;
}
SICP_DEV void tri_finish(const TriProbe& q, int k, long kk, float mine, TriRead& t) {
    float sd[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sd[i] = gshfl(mine, i);
    int missing = kk < 0 ? 1 : 0;
#pragma unroll
    for (int o = 1; o < kRayGroup; o <<= 1) missing |= __shfl_xor(missing, o, kRayGroup);
    t.k = kk;
    const float fx = q.X.frac, fy = q.Y.frac, fz = q.Z.frac;
    float r0, r1, r2, r3;
    r0 = (1.0f - fx) * sd[0] + fx * sd[1];
    r1 = (1.0f - fx) * sd[2] + fx * sd[3];
    r2 = (1.0f - fy) * r0 + fy * r1;
    const float a0 = r0, a1 = r1;
    r0 = (1.0f - fx) * sd[4] + fx * sd[5];
    r1 = (1.0f - fx) * sd[6] + fx * sd[7];
    r3 = (1.0f - fy) * r0 + fy * r1;
    t.val = (1.0f - fz) * r2 + fz * r3;
    t.ok = missing == 0 && !isnan_(t.val);
    t.w = ((k & 1) ? fx : 1.0f - fx) * ((k & 2) ? fy : 1.0f - fy) * ((k & 4) ? fz : 1.0f - fz);
    t.grad.x = (1.0f - fz) * ((1.0f - fy) * (sd[1] - sd[0]) + fy * (sd[3] - sd[2])) +
               fz * ((1.0f - fy) * (sd[5] - sd[4]) + fy * (sd[7] - sd[6]));
    t.grad.y = (1.0f - fz) * (a1 - a0) + fz * (r1 - r0);
    t.grad.z = r3 - r2;
}
SICP_DEV void tri_read(const MapDev& m, v3 q, int k, TriRead& t) {
    const TriProbe tp = tri_probe(m, q, k);
    long kk;
    float mine;
    tri_corner(m, tp, kk, mine);
    tri_finish(tp, k, kk, mine, t);
}

// dL/d(values) += g * weights, each lane its corner.
SICP_DEV void tri_scatter(const TriRead& t, float g, float* grad_sdf) {
    if (!grad_sdf || g == 0.0f) return;
    if (t.k >= 0 && t.w != 0.0f) atomicAdd(grad_sdf + t.k, g * t.w);
}

struct AdjointArgs {
    RayArgs g;
    const int32_t* pixels;
    int n;
    const float* grad_v;   // n x 3, d loss / d vertex (camera frame)
    const float* grad_n;   // n x 3, d loss / d normal; may be null
    float* grad_sdf;       // num_blocks x 512, accumulated; may be null
    float* grad_px;        // n x 6 per-pixel pose gradients; may be null
    double* partials;      // 6 x kAdjMaxBlocks
};
constexpr int kAdjThreads = 128;   // 16 pixels: 10000 pixels give each CU two or three
constexpr int kAdjMaxBlocks = 1024;

// One pixel, by the lanes k of a group whose first lane is gbase: false (and
// no gradient) where the forward pass writes NaN. Every lane of the group
// takes the same branches.
SICP_DEV bool adjoint_pixel(const MapDev& m, const View<float>& zmin, const View<float>& zmax,
                            const PoseF& pose, const RayArgs& g, int x, int y, v3 gv, v3 gn,
                            float* grad_sdf, float gxi[6], int k, int gbase) {
    Ray ray;
    if (!ray_setup(m, zmin, zmax, pose, g, x, y, ray)) return false;
    CoopState c{ray.start, ray.dist_s, 1.0f, 0.0f, false, false, -1, BlockCache{0, 0, 0, -1}};
    coop_march(m, ray, k, gbase, c);
    if (c.back_face) return false;
    const v3 result = c.result;
    const float sdf = c.sdf, msum = c.steps;
    const bool interp0 = c.interp;
    const long k0 = c.k;
    if (!(sdf <= 0.0f)) return false;
    const float ks = m.step_scale;
    const v3 r0 = result;
    TriRead t0;
    if (interp0) tri_read(m, r0, k, t0);
    const float s0 = sdf;
    const v3 r1 = add(r0, scale(s0 * ks, ray.dir));
    TriRead t1;
    tri_read(m, r1, k, t1);
    const float s1 = t1.val;
    const v3 r2 = add(r1, scale(s1 * ks, ray.dir));
    // readNormal's six reads: pt.a + 1.0f / pt.a + -1.0f on one axis, pt on
    // the others; a failing one ends the pixel
    auto normal_point = [&](int a) {
        const float d = (a & 1) ? -1.0f : 1.0f;
        const int ax = a >> 1;
        return v3{ax == 0 ? r2.x + d : r2.x, ax == 1 ? r2.y + d : r2.y, ax == 2 ? r2.z + d : r2.z};
    };
    // (all six lookups in flight, then all six reads)
    TriRead tn[6];
    {
        TriProbe tp[6];
        long kk[6];
        float mine[6];
#pragma unroll
        for (int a = 0; a < 6; ++a) tp[a] = tri_probe(m, normal_point(a), k);
#pragma unroll
        for (int a = 0; a < 6; ++a) tri_corner(m, tp[a], kk[a], mine[a]);
#pragma unroll
        for (int a = 0; a < 6; ++a) tri_finish(tp[a], k, kk[a], mine[a], tn[a]);
    }
    float sv[6];
#pragma unroll
    for (int a = 0; a < 6; ++a) {
        sv[a] = tn[a].val;
        if (!tn[a].ok || sv[a] == 1.0f) return false;
    }
    const v3 gvec = mk(sv[0] - sv[1], sv[2] - sv[3], sv[4] - sv[5]);
    const v3 mvec = mv(pose.Rinv, gvec);
    const float mlen = norm(mvec);
    const v3 nrm = divs(mvec, mlen);
    const v3 vout = mv(pose.Rinv, sub(scale(r2, m.voxel), pose.t));
    // ---- backwards ----
    v3 gw{0.f, 0.f, 0.f}, gt{0.f, 0.f, 0.f}, gr2{0.f, 0.f, 0.f}, gdir{0.f, 0.f, 0.f};
    // normal: n = m / |m|, m = R'^T g
    const float ndg = dot(nrm, gn);
    const v3 gm = divs(sub(gn, scale(ndg, nrm)), mlen);
    gw = add(gw, cross(gm, mvec));
    const v3 gg = mv(pose.R, gm);
#pragma unroll
    for (int a = 0; a < 6; ++a) {
        const float ga = (a >> 1) == 0 ? gg.x : ((a >> 1) == 1 ? gg.y : gg.z);
        const float gsa = (a & 1) ? -ga : ga;
        tri_scatter(tn[a], gsa, grad_sdf);
        gr2 = add(gr2, scale(gsa, tn[a].grad));
    }
    // vertex: v = R'^T (voxel r2 - t')
    gr2 = add(gr2, scale(m.voxel, mv(pose.R, gv)));
    gt = sub(gt, gv);
    gw = add(gw, cross(gv, vout));
    // r2 = r1 + k s1 dir
    v3 gr1 = gr2;
    const float gs1 = ks * dot(ray.dir, gr2);
    gdir = add(gdir, scale(ks * s1, gr2));
    tri_scatter(t1, gs1, grad_sdf);
    gr1 = add(gr1, scale(gs1, t1.grad));
    // r1 = r0 + k s0 dir
    v3 gr0 = gr1;
    const float gs0 = ks * dot(ray.dir, gr1);
    gdir = add(gdir, scale(ks * s0, gr1));
    if (interp0) {
        tri_scatter(t0, gs0, grad_sdf);
        gr0 = add(gr0, scale(gs0, t0.grad));
    } else if (grad_sdf && k == 0 && k0 >= 0 && gs0 != 0.0f) {
        atomicAdd(grad_sdf + k0, gs0);
    }
    // r0 = block_s + M dir
    gdir = add(gdir, scale(msum, gr0));
    // dir = R' u, u the ray in the camera frame
    const v3 u = mv(pose.Rinv, ray.dir);
    gw = add(gw, cross(u, mv(pose.Rinv, gdir)));
    // block_s = (R' p_s + t') / voxel
    const float z0 = zmin.at(y >> 3, x >> 3);
    const v3 ps{z0 * ((float)x - g.cx) * g.invfx, z0 * ((float)y - g.cy) * g.invfy, z0};
    const v3 gb = scale(m.voxel_inv, mv(pose.Rinv, gr0));
    gt = add(gt, gb);
    gw = add(gw, cross(ps, gb));
    gxi[0] = gt.x;
    gxi[1] = gt.y;
    gxi[2] = gt.z;
    gxi[3] = gw.x;
    gxi[4] = gw.y;
    gxi[5] = gw.z;
    return true;
}

__global__ __launch_bounds__(kAdjThreads) void raycast_adjoint_kernel(MapDev m, View<float> zmin,
                                                                      View<float> zmax,
                                                                      PoseArg pa, AdjointArgs a) {
    const PoseF pose = load_pose(pa);
    constexpr int kGroups = kAdjThreads / kRayGroup;
    const int k = threadIdx.x & (kRayGroup - 1), gbase = (threadIdx.x & 63) & ~(kRayGroup - 1);
    const int group = threadIdx.x / kRayGroup;
    double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int i = blockIdx.x * kGroups + group; i < a.n; i += gridDim.x * kGroups) {
        const int px = a.pixels[i];
        float gxi[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (px >= 0 && px < a.g.cols * a.g.rows) {  // else outside the image: no gradient
            const int y = px / a.g.cols, x = px - y * a.g.cols;
            const v3 gv{a.grad_v[3 * i], a.grad_v[3 * i + 1], a.grad_v[3 * i + 2]};
            const v3 gn = a.grad_n
                              ? v3{a.grad_n[3 * i], a.grad_n[3 * i + 1], a.grad_n[3 * i + 2]}
                              : v3{0.f, 0.f, 0.f};
            if (!adjoint_pixel(m, zmin, zmax, pose, a.g, x, y, gv, gn, a.grad_sdf, gxi, k, gbase))
                for (int j = 0; j < 6; ++j) gxi[j] = 0.f;
        }
#pragma unroll
        for (int j = 0; j < 6; ++j) acc[j] += (double)gxi[j];
        if (a.grad_px && k < 6) {
            float v = gxi[0];
#pragma unroll
            for (int j = 1; j < 6; ++j) v = k == j ? gxi[j] : v;
            a.grad_px[6 * i + k] = v;
        }
    }
    // fixed-order workgroup sum: one row per group through LDS, thread j sums column j
    __shared__ double tile[kGroups][7];
    if (k == 0) {
#pragma unroll
        for (int j = 0; j < 6; ++j) tile[group][j] = acc[j];
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        double s = 0.0;
        for (int r = 0; r < kGroups; ++r) s += tile[r][threadIdx.x];
        a.partials[threadIdx.x * kAdjMaxBlocks + blockIdx.x] = s;
    }
}

// The workgroups' partial sums in a fixed order: wavefront j adds column j,
// lane l rows l, l + 64, ..., then the lanes fold.
__global__ __launch_bounds__(384) void adjoint_finish_kernel(const double* partials, int nb,
                                                             double* grad_pose) {
    const int j = threadIdx.x >> 6, l = threadIdx.x & 63;
    double s = 0.0;
    for (int b = l; b < nb; b += 64) s += partials[j * kAdjMaxBlocks + b];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (l == 0) grad_pose[j] = s;
}

}  // namespace

int launch_raycast_adjoint(MapDev m, View<float> zmin, View<float> zmax, PoseArg pose,
                           float invfx, float invfy, float cx, float cy, int cols, int rows,
                           const int32_t* pixels, int n, const float* grad_v,
                           const float* grad_n, float* grad_sdf, float* grad_px,
                           double* partials, double* grad_pose, hipStream_t s) {
    AdjointArgs a{RayArgs{invfx, invfy, cx, cy, cols, rows, 0, 0, 0, 0}, pixels, n, grad_v, grad_n,
                  grad_sdf, grad_px, partials};
    int nb = (int)div_up(n > 0 ? n : 1, kAdjThreads / kRayGroup);
    if (nb > kAdjMaxBlocks) nb = kAdjMaxBlocks;
    raycast_adjoint_kernel<<<nb, kAdjThreads, 0, s>>>(m, zmin, zmax, pose, a);
    SICP_LAUNCH_CHECK("raycast_adjoint_kernel");
    adjoint_finish_kernel<<<1, 384, 0, s>>>(partials, nb, grad_pose);
    SICP_LAUNCH_CHECK("adjoint_finish_kernel");
    return SICP_OK;
}

size_t raycast_adjoint_scratch_bytes() { return sizeof(double) * (6 * kAdjMaxBlocks + 8); }

int launch_render_prepass(MapDev m, MapCounters* ctr, const sicp_block* visible, View<float> zmin,
                          View<float> zmax, PoseArg pose, sicp_intrinsics K, float dmax,
                          float dmin, const int* gate, hipStream_t s, bool zrange_cleared,
                          const uint32_t* fuse_counts) {
    int n = zmin.cols * zmin.rows;
    if (!zrange_cleared) {
        zrange_init_kernel<<<div_up(n, 256) > 0 ? div_up(n, 256) : 1, 256, 0, s>>>(zmin, zmax,
                                                                                  ctr);
        SICP_LAUNCH_CHECK("zrange_init_kernel");
    }
    PrepassArgs g{K.fx, K.fy, K.cx, K.cy, dmax, dmin, zmin.cols, zmin.rows};
    if (!gate) gate = m.one;
    if (n <= kPrepassLdsTiles) {
        prepass_lds_kernel<<<kPrepassLdsGrid, 256, 0, s>>>(m, ctr, visible, zmin, zmax, pose, g, gate,
                                               fuse_counts);
        SICP_LAUNCH_CHECK("prepass_lds_kernel");
    } else {
        prepass_kernel<<<kPrepassGrid, 64, 0, s>>>(m, ctr, visible, zmin, zmax, pose, g, gate,
                                           fuse_counts);
        SICP_LAUNCH_CHECK("prepass_kernel");
    }
    return SICP_OK;
}

// Both passes; the queue count is cleared first (unless the caller's
// launch_fuse_count already did).
int launch_raycast_gated(MapDev m, View<float4> vmap, View<float4> nmap, View<float> zmin,
                         View<float> zmax, PoseArg pose, float invfx, float invfy, float cx,
                         float cy, const int* gate, const uint32_t* nonempty, hipStream_t s,
                         bool queue_cleared, RayTuning tune) {
    if ((size_t)vmap.cols * vmap.rows > m.rq_cap) return invalid("raycast: image above the map's max_cols x max_rows");
    if (tune.first_pass_samples < 1 || tune.first_pass_samples > kRayTuneMaxSamples ||
        tune.second_pass_workgroups < 1 || tune.second_pass_workgroups > kRayTuneMaxWorkgroups ||
        (tune.lds_block_table != 0 && tune.lds_block_table != 1))
        return invalid("raycast: tuning outside 1..4096 samples, 1..65536 workgroups, table 0/1");
    const RayArgs g{invfx, invfy, cx, cy, vmap.cols, vmap.rows, (int)div_up(vmap.cols, 8),
                    (int)div_up(vmap.rows, 8), tune.first_pass_samples,
                    ray_cube_margin(tune.first_pass_samples)};
    if (!gate) gate = m.one;
    if (!nonempty) nonempty = reinterpret_cast<const uint32_t*>(m.one);
    if (!queue_cleared) {
        ray_queue_reset_kernel<<<1, 1, 0, s>>>(m.rq_count);
        SICP_LAUNCH_CHECK("ray_queue_reset_kernel");
    }
    // super-tiles rounded up to one for each XCD
    const unsigned grid = div_up((long)div_up(g.tcols, kRaySuper) * div_up(g.trows, kRaySuper), 8) *
                          8u * kRaySuper * kRaySuper;
    auto* first = m.half ? (tune.lds_block_table ? raycast_kernel<true, true> : raycast_kernel<true, false>)
                         : (tune.lds_block_table ? raycast_kernel<false, true>
                                                 : raycast_kernel<false, false>);
    first<<<grid, 64, 0, s>>>(m, vmap, nmap, zmin, zmax, pose, g, gate, nonempty);
    SICP_LAUNCH_CHECK("raycast_kernel");
    raycast_long_kernel<<<tune.second_pass_workgroups, kRayLongThreads, 0, s>>>(
        m, vmap, nmap, zmin, zmax, pose, g, gate, nonempty);
    SICP_LAUNCH_CHECK("raycast_long_kernel");
    return SICP_OK;
}

int launch_raycast(MapDev m, View<float4> vmap, View<float4> nmap, View<float> zmin,
                   View<float> zmax, PoseArg pose, float invfx, float invfy, float cx, float cy,
                   const int* gate, hipStream_t s) {
    return launch_raycast_gated(m, vmap, nmap, zmin, zmax, pose, invfx, invfy, cx, cy, gate,
                                nullptr, s, false, RayTuning{});
}

}  // namespace sicp
