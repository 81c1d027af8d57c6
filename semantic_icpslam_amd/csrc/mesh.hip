// mesh.hip — marching-cubes surface extraction of the TSDF (MeshScene,
// Mapping/MeshScene.cu:4-356) for gfx950.
//
// One workgroup per allocated block, one thread per voxel. The 27 blocks
// around a block are resolved once, and the sdf of the block's voxels and of
// those around it that its cells read is staged in LDS. Two passes: the first
// counts each block's triangles; the second recomputes each voxel's case,
// lists the block's triangles in order, and writes them a vertex per thread at
// the block's offset, which each workgroup forms from the counts before it.
// The output order is therefore canonical (heap slot, then voxel index
// z*64 + y*8 + x, then the table's order), where the reference appends with an
// atomic counter in whatever order the threads arrive.
//
// What bounds it: memory round trips and instructions, not bytes. With every
// voxel reading its 8 corners, 24 neighbours and 8 colours itself, and the few
// voxels on the surface writing up to 15 vertices in turn while the others
// waited, the passes took 68 and 302 us on 6000 blocks (640x480 / 5 mm); a
// block's 1331 staged values, and a thread per vertex, take 45 and 67.
#include <cstdio>
#include <cstring>

#include "map_common.hpp"
#include "sicp_internal.hpp"

namespace sicp {

// ------------------------------------------------------------- tables -----
// Edge j of a voxel cube (its two corners), in the reference's numbering
// (MeshScene.cu:200-291); corner k sits at (x, y, z) = (0,0,0), (1,0,0),
// (1,1,0), (0,1,0), then the same four at z = 1.
static constexpr int kEdge[12][2] = {{0, 1}, {1, 2}, {2, 3}, {3, 0}, {4, 5}, {5, 6},
                                 {6, 7}, {7, 4}, {0, 4}, {1, 5}, {2, 6}, {3, 7}};

struct MeshTables {
    int32_t edge[256];      // bit j: edge j is cut
    int8_t tri[256][16];    // edge triples, -1 terminated
    int32_t nvert[256];     // 3 x triangles
};

// The triangle table is the reference's (the classic published
// marching-cubes table, Mapping/Constant.h:39-296), so the triangles of a
// voxel, and the corner order within each, are the reference's; it is held
// as one hexadecimal string of edge indices per sign case (mc_table.inc,
// written by gen_mc_table.py). The edge table (the cut edges: corners of
// different sign) and the vertex counts follow from it.
#include "mc_table.inc"

static constexpr void build_tables(MeshTables& t) {
    for (int cs = 0; cs < 256; ++cs) {
        int emask = 0;
        for (int j = 0; j < 12; ++j)
            if (((cs >> kEdge[j][0]) & 1) != ((cs >> kEdge[j][1]) & 1)) emask |= 1 << j;
        t.edge[cs] = emask;
        const char* row = kMcTriangles[cs];
        int n = 0;
        while (row[n]) ++n;
        for (int j = 0; j < 16; ++j) {
            const char ch = j < n ? row[j] : 0;
            t.tri[cs][j] = j < n ? (int8_t)(ch <= '9' ? ch - '0' : ch - 'a' + 10) : (int8_t)-1;
        }
        t.nvert[cs] = n;
    }
}

static constexpr MeshTables make_tables() {
    MeshTables t{};
    build_tables(t);
    return t;
}
static const MeshTables& tables() {
    static constexpr MeshTables t = make_tables();
    return t;
}
// What the kernels read of them, part of the code object.
struct CaseTables {
    int8_t tri[256][16];
    uint8_t ntri[256];
};
static constexpr CaseTables make_case_tables() {
    const MeshTables t = make_tables();
    CaseTables c{};
    for (int k = 0; k < 256; ++k) {
        for (int j = 0; j < 16; ++j) c.tri[k][j] = t.tri[k][j];
        c.ntri[k] = (uint8_t)(t.nvert[k] / 3);
    }
    return c;
}
__device__ const CaseTables d_cases = make_case_tables();

namespace {

constexpr int kMeshThreads = 512;  // one per voxel of a block
constexpr uint32_t kMeshGrid = 4096;  // workgroups at most; the blocks are taken in turn

struct MeshOut {
    float* vertices;   // 9 floats per triangle
    float* normals;    // 9 floats per triangle
    uint8_t* colors;   // 9 bytes per triangle
    uint32_t max_triangles;
};

// The 27 blocks around block `b` (offsets -1..1 per axis) into LDS.
SICP_DEV void neighbour_slots(const MapDev& m, const sicp_block& b, int* nslot) {
    const int t = threadIdx.x;
    if (t < 27) {
        const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = t / 9 - 1;
        nslot[t] = map_lookup(m, b.x + dx, b.y + dy, b.z + dz);
    }
}

// A voxel at block-relative voxel coordinates in [-8, 15] (FindVoxel,
// DeviceMap.cu:97-103); -1 when its block is missing.
SICP_DEV long voxel_at(const int* nslot, int x, int y, int z) {
    const int s = nslot[((z >> 3) + 1) * 9 + ((y >> 3) + 1) * 3 + ((x >> 3) + 1)];
    if (s < 0) return -1;
    return (long)s * 512 + ((z & 7) << 6) + ((y & 7) << 3) + (x & 7);
}

// The sdf of the voxels from (-1, -1, -1) to (9, 9, 9) of a block: all that
// its cells and their normals read. A missing block's voxels are NaN.
constexpr int kReach = 11, kTile = kReach * kReach * kReach;
SICP_DEV int tile_index(int x, int y, int z) {
    return ((z + 1) * kReach + y + 1) * kReach + x + 1;
}
SICP_DEV void stage_block(const MapDev& m, const sicp_block& b, int* nslot, float* tile) {
    neighbour_slots(m, b, nslot);
    __syncthreads();
    constexpr int kEach = (kTile + kMeshThreads - 1) / kMeshThreads;
    float v[kEach];
#pragma unroll
    for (int q = 0; q < kEach; ++q) {
        const int i = min((int)threadIdx.x + q * kMeshThreads, kTile - 1);
        const long k = voxel_at(nslot, i % kReach - 1, i / kReach % kReach - 1,
                                i / (kReach * kReach) - 1);
        const float s = vox_sdf(m, k >= 0 ? (size_t)k : 0);
        v[q] = k >= 0 ? s : qnanf();
    }
#pragma unroll
    for (int q = 0; q < kEach; ++q) {
        const int i = (int)threadIdx.x + q * kMeshThreads;
        if (i < kTile) tile[i] = v[q];
    }
    __syncthreads();
}

// MeshEngine::interp (MeshScene.cu:156-164).
SICP_DEV float mc_interp(float v1, float v2) {
    if ((double)fabsf(0 - v1) < 1e-6) return 0;
    if ((double)fabsf(0 - v2) < 1e-6) return 1;
    if ((double)fabsf(v1 - v2) < 1e-6) return 0;
    return (0 - v1) / (v2 - v1);
}

// The corner coordinates on the device, as closed forms of the corner number.
SICP_DEV int d_corner(int k, int axis) {
    return axis == 0 ? ((k == 1 || k == 2 || k == 5 || k == 6) ? 1 : 0)
                     : (axis == 1 ? ((k == 2 || k == 3 || k == 6 || k == 7) ? 1 : 0) : (k >> 2));
}
SICP_DEV int d_edge(int e, int end) {
    // edges 0-3 and 4-7 run round the z = 0 and z = 1 faces, 8-11 are vertical
    if (e < 8) {
        const int base = e & 4, i = e & 3;
        return base + (end ? ((i + 1) & 3) : i);
    }
    return end ? (e - 8) + 4 : e - 8;
}

// readVertexAndColor + readNormal + the case (MeshScene.cu:39-154,166-198): the
// sign case of the cell at voxel (x, y, z), or 0 without triangles. The eight
// corner values are neither NaN nor exactly 1, and none of the voxels either
// side of a corner along an axis is NaN.
SICP_DEV int cell_case(const float* tile, int x, int y, int z) {
    constexpr int kY = kReach, kZ = kReach * kReach;
    const float* c = tile + tile_index(x, y, z);
    float s[8];
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        s[k] = c[d_corner(k, 0) + kY * d_corner(k, 1) + kZ * d_corner(k, 2)];
        ok = ok && !(s[k] == 1.0f || isnan_(s[k]));
    }
    if (!ok) return 0;
    // along each axis the four values before the cell's corners and the four
    // after them, compared in pairs (unordered: either is NaN)
    bool nan = false;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int u = a == 0 ? 1 : (a == 1 ? kY : kZ);
        const int p = a == 0 ? kY : 1, q = a == 2 ? kY : kZ;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int o = (i & 1) * p + (i >> 1) * q;
            nan = nan || __builtin_isunordered(c[o - u], c[o + 2 * u]);
        }
    }
    if (nan) return 0;
    int cube = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) cube |= (s[k] < 0) ? (1 << k) : 0;
    return cube;
}

// One vertex of a triangle, on cut edge `e` of the cell at voxel (x, y, z) of
// block `b` (MeshScene.cu:200-291 and :312-320): the position + the edge's
// corner offsets with the parameter, times the voxel size; the corner normals
// (differences of the voxels either side) interpolated, then normalised; the
// colour of the edge's first corner, or of its second when the parameter is
// exactly 1 (the reference multiplies the uchar3 difference by the float
// parameter converted to int).
SICP_DEV void edge_vertex(const MapDev& m, const int* nslot, const float* tile,
                          const sicp_block& blk, int e, int x, int y, int z, float voxel,
                          float* vo, float* no, uint8_t* co) {
    const int a = d_edge(e, 0), b = d_edge(e, 1);
    const int ca[3] = {d_corner(a, 0), d_corner(a, 1), d_corner(a, 2)};
    const int cb[3] = {d_corner(b, 0), d_corner(b, 1), d_corner(b, 2)};
    const float* pa = tile + tile_index(x + ca[0], y + ca[1], z + ca[2]);
    const float* pb = tile + tile_index(x + cb[0], y + cb[1], z + cb[2]);
    const float val = mc_interp(pa[0], pb[0]);
    const int p[3] = {blk.x * 8 + x, blk.y * 8 + y, blk.z * 8 + z};
    float n[3];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const float comp = ca[ax] == cb[ax] ? (float)ca[ax] : (ca[ax] == 0 ? val : 1 - val);
        vo[ax] = ((float)p[ax] + comp) * voxel;
        const int u = ax == 0 ? 1 : (ax == 1 ? kReach : kReach * kReach);
        const float na = pa[u] - pa[-u], nb = pb[u] - pb[-u];
        n[ax] = na + val * (nb - na);
    }
    const v3 nn = normalised(v3{n[0], n[1], n[2]});
    no[0] = nn.x;
    no[1] = nn.y;
    no[2] = nn.z;
    const int iv = (int)val;
    uint8_t qa[3], qb[3] = {0, 0, 0};
    vox_rgb(m, (size_t)voxel_at(nslot, x + ca[0], y + ca[1], z + ca[2]), qa[0], qa[1], qa[2]);
    if (iv != 0)
        vox_rgb(m, (size_t)voxel_at(nslot, x + cb[0], y + cb[1], z + cb[2]), qb[0], qb[1], qb[2]);
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) {
        const uint8_t d = (uint8_t)(qb[ch] - qa[ch]);
        const uint8_t mm = (uint8_t)(d * iv);
        co[ch] = (uint8_t)(qa[ch] + mm);
    }
}

// Exclusive prefix of `v` over the workgroup (512 threads); `total` gets the
// sum. `part` is LDS for the eight wavefront totals.
SICP_DEV uint32_t block_exclusive_scan(uint32_t v, uint32_t* part, uint32_t& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t up = __shfl_up(inc, o, 64);
        if (lane >= o) inc += up;
    }
    if (lane == 63) part[w] = inc;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
#pragma unroll
    for (int k = 0; k < kMeshThreads / 64; ++k) {
        before += k < w ? part[k] : 0u;
        total += part[k];
    }
    return before + inc - v;
}

// The triangle counts: of every block, and of every chunk of kMeshChunk blocks
// (integer sums by atomics, so their order does not matter).
constexpr uint32_t kMeshChunk = 256;
struct MeshCounts {
    uint32_t *block, *chunk;
    uint32_t nchunks;
};

__global__ __launch_bounds__(256) void mesh_reset_kernel(MeshCounts ct) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < ct.nchunks) ct.chunk[i] = 0u;
}

// Pass 1: the triangle count of every allocated block.
__global__ __launch_bounds__(kMeshThreads) void mesh_count_kernel(MapDev m,
                                                                  const MapCounters* ctr,
                                                                  MeshCounts ct) {
    __shared__ int nslot[27];
    __shared__ float tile[kTile];
    __shared__ uint32_t part[kMeshThreads / 64];
    const uint32_t nblk = ctr->heap_used;
    const int t = threadIdx.x, x = t & 7, y = (t >> 3) & 7, z = t >> 6;
    for (uint32_t b = blockIdx.x; b < nblk; b += gridDim.x) {
        stage_block(m, m.blocks[b], nslot, tile);
        uint32_t total;
        (void)block_exclusive_scan(d_cases.ntri[cell_case(tile, x, y, z)], part, total);
        if (t == 0) {
            ct.block[b] = total;
            if (total) atomicAdd(&ct.chunk[b / kMeshChunk], total);
        }
        __syncthreads();
    }
}

// Pass 2: every triangle at its block's offset plus its rank within the block;
// triangles past `out.max_triangles` are dropped. A block's triangles are
// listed in LDS and its vertices written one per thread, so consecutive
// threads write consecutive vertices. The host reads the number found from
// `host_total`.
__global__ __launch_bounds__(kMeshThreads) void mesh_emit_kernel(MapDev m,
                                                                 const MapCounters* ctr,
                                                                 MeshCounts ct, float voxel,
                                                                 MeshOut out,
                                                                 uint32_t* host_total) {
    __shared__ int nslot[27];
    __shared__ float tile[kTile];
    __shared__ uint32_t part[kMeshThreads / 64];
    __shared__ uint32_t list[kBlockVoxels * 5];  // voxel | case << 9 | triangle << 17
    if (blockIdx.x == 0) {
        uint32_t sum = 0, all;
        for (uint32_t c = threadIdx.x; c < ct.nchunks; c += kMeshThreads) sum += ct.chunk[c];
        (void)block_exclusive_scan(sum, part, all);
        if (threadIdx.x == 0) *host_total = all;
        __syncthreads();  // `part` is used again
    }
    if (out.max_triangles == 0u) return;
    const uint32_t nblk = ctr->heap_used;
    const int t = threadIdx.x, x = t & 7, y = (t >> 3) & 7, z = t >> 6;
    for (uint32_t b = blockIdx.x; b < nblk; b += gridDim.x) {
        if (ct.block[b] == 0u) continue;
        // the triangles of the chunks and of the blocks before this one
        const uint32_t chunk = b / kMeshChunk;
        uint32_t before = 0;
        for (uint32_t c = t; c < chunk; c += kMeshThreads) before += ct.chunk[c];
        if (chunk * kMeshChunk + t < b) before += ct.block[chunk * kMeshChunk + t];
        uint32_t base;
        (void)block_exclusive_scan(before, part, base);
        __syncthreads();  // `part` is used again
        if (base >= out.max_triangles) continue;  // every thread has the sum
        const sicp_block blk = m.blocks[b];
        stage_block(m, blk, nslot, tile);
        const int cube = cell_case(tile, x, y, z);
        const uint32_t n = d_cases.ntri[cube];
        uint32_t total;
        const uint32_t rank = block_exclusive_scan(n, part, total);
        for (uint32_t j = 0; j < n; ++j)
            list[rank + j] = (uint32_t)t | (uint32_t)cube << 9 | j << 17;
        __syncthreads();
        const uint32_t room = out.max_triangles - base;
        const uint32_t nv = 3u * (total < room ? total : room);
        for (uint32_t q = t; q < nv; q += kMeshThreads) {
            const uint32_t e = list[q / 3u];
            const int vox = e & 511, edge = d_cases.tri[(e >> 9) & 255u][(e >> 17) * 3u + q % 3u];
            float vo[3], no[3];
            uint8_t co[3];
            edge_vertex(m, nslot, tile, blk, edge, vox & 7, (vox >> 3) & 7, vox >> 6, voxel, vo,
                        no, co);
            const size_t o = ((size_t)base * 3 + q) * 3;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                out.vertices[o + a] = vo[a];
                out.normals[o + a] = no[a];
                out.colors[o + a] = co[a];
            }
        }
        __syncthreads();
    }
}

}  // namespace

// The counts' device memory and the host word, kept with the map from the
// first call on and lent to one call at a time; a call that finds them lent
// (another thread's) allocates its own for its duration. A call that fails once
// something is queued waits for its stream before it gives them back; where
// that fails too, a kernel may still write them and they are given up.
struct MeshLoan {
    sicp_map* map;
    hipStream_t stream;
    bool kept;
    bool queued = false;  // launches that have not been waited for
    uint32_t* dev = nullptr;
    uint32_t* host = nullptr;
    MeshLoan(sicp_map* m, hipStream_t s)
        : map(m), stream(s), kept(!m->mesh_lent.exchange(true)) {}
    int take(size_t words) {
        if (kept) {
            dev = map->mesh_counts;
            host = map->mesh_total;
        }
        if (!dev) {
            hipError_t e = hipMalloc((void**)&dev, words * sizeof(uint32_t));
            if (e != hipSuccess) return hip_fail(e, "hipMalloc(mesh counts)");
            if (kept) map->mesh_counts = dev;
        }
        if (!host) {
            hipError_t e = hipHostMalloc((void**)&host, sizeof(uint32_t), hipHostMallocDefault);
            if (e != hipSuccess) return hip_fail(e, "hipHostMalloc(mesh total)");
            if (kept) map->mesh_total = host;
        }
        return SICP_OK;
    }
    ~MeshLoan() {
        const bool lost = queued && hipStreamSynchronize(stream) != hipSuccess;
        if (kept) {
            if (lost) map->mesh_counts = map->mesh_total = nullptr;
            map->mesh_lent.store(false);
            return;
        }
        if (lost) return;
        if (dev) (void)hipFree(dev);
        if (host) (void)hipHostFree(host);
    }
};

int launch_mesh(sicp_map* map, float* vertices, float* normals, uint8_t* colors,
                uint32_t max_triangles, uint32_t* n_out, uint32_t* total_out, hipStream_t s) {
    const uint32_t cap = (uint32_t)map->cfg.num_blocks;
    const uint32_t nchunks = div_up(cap, kMeshChunk);
    MeshLoan mem(map, s);
    const int rc = mem.take((size_t)cap + nchunks);
    if (rc) return rc;
    const MeshCounts ct{mem.dev, mem.dev + cap, nchunks};
    mem.queued = true;
    mesh_reset_kernel<<<div_up(nchunks, 256), 256, 0, s>>>(ct);
    SICP_LAUNCH_CHECK("mesh_reset_kernel");
    const int grid = (int)(cap < kMeshGrid ? cap : kMeshGrid);
    mesh_count_kernel<<<grid, kMeshThreads, 0, s>>>(map->dev, map->ctr, ct);
    SICP_LAUNCH_CHECK("mesh_count_kernel");
    const MeshOut out{vertices, normals, colors, max_triangles};
    mesh_emit_kernel<<<max_triangles > 0 ? grid : 1, kMeshThreads, 0, s>>>(
        map->dev, map->ctr, ct, map->cfg.voxel_size, out, mem.host);
    SICP_LAUNCH_CHECK("mesh_emit_kernel");
    SICP_HIP(hipStreamSynchronize(s));
    mem.queued = false;
    const uint32_t tot = *mem.host;
    *n_out = tot < max_triangles ? tot : max_triangles;
    if (total_out) *total_out = tot;
    return SICP_OK;
}

}  // namespace sicp

using namespace sicp;

extern "C" {

int sicp_mesh_tables(int32_t* edge_table, int8_t* triangle_table, int32_t* vertex_table) {
    const MeshTables& t = tables();
    if (edge_table) std::memcpy(edge_table, t.edge, sizeof(t.edge));
    if (triangle_table) std::memcpy(triangle_table, t.tri, sizeof(t.tri));
    if (vertex_table) std::memcpy(vertex_table, t.nvert, sizeof(t.nvert));
    return SICP_OK;
}

int sicp_mesh_scene(sicp_map* map, float* vertices_dev, float* normals_dev, uint8_t* colors_dev,
                    uint32_t max_triangles, uint32_t* n_triangles, uint32_t* n_total,
                    void* stream) {
    if (!map || !n_triangles) return invalid("mesh_scene: null argument");
    if (max_triangles > 0 && (!vertices_dev || !normals_dev || !colors_dev))
        return invalid("mesh_scene: null output buffer");
    return launch_mesh(map, vertices_dev, normals_dev, colors_dev, max_triangles, n_triangles,
                       n_total, (hipStream_t)stream);
}

int sicp_mesh_write_ply(const char* path, const float* vertices, const float* normals,
                        const uint8_t* colors, uint32_t n_triangles) {
    if (!path || (n_triangles > 0 && (!vertices || !normals || !colors)))
        return invalid("mesh_write_ply: null argument");
    FILE* f = std::fopen(path, "w");
    if (!f) return invalid("mesh_write_ply: cannot open the file");
    const unsigned long long nv = 3ull * n_triangles;
    std::fprintf(f,
                 "ply\nformat ascii 1.0\nelement vertex %llu\nproperty float x\nproperty float y\n"
                 "property float z\nproperty float nx\nproperty float ny\nproperty float nz\n"
                 "property uchar red\nproperty uchar green\nproperty uchar blue\n"
                 "element face %u\nproperty list uchar uint vertex_indices\nend_header\n",
                 nv, n_triangles);
    for (unsigned long long i = 0; i < nv; ++i)
        std::fprintf(f, "%g %g %g %g %g %g %d %d %d\n", vertices[3 * i], vertices[3 * i + 1],
                     vertices[3 * i + 2], normals[3 * i], normals[3 * i + 1], normals[3 * i + 2],
                     (int)colors[3 * i], (int)colors[3 * i + 1], (int)colors[3 * i + 2]);
    for (uint32_t i = 0; i < n_triangles; ++i)
        std::fprintf(f, "3 %u %u %u\n", 3 * i, 3 * i + 1, 3 * i + 2);
    const bool ok = std::ferror(f) == 0;
    if (std::fclose(f) != 0 || !ok) return invalid("mesh_write_ply: write failed");
    return SICP_OK;
}

}  // extern "C"
