// unify.hip — neighbour label smoothing after label fusion
// (Fusion::UnifyNeighbor / UpdateNeighborLabel, Mapping/FuseMap.cu:757-948),
// made deterministic, for gfx950.
//
// The reference reads neighbouring voxels while other threads rewrite them,
// so its result depends on timing. Here the pass is double-buffered: a
// snapshot kernel copies the label state (weight != 0, label, count) of
// every voxel of the blocks about to be rewritten, and stamps those blocks;
// the update kernel then reads every neighbour of a stamped block from the
// snapshot and every other neighbour from the map itself (which this pass
// does not write). Each voxel is written only by its own thread, after its
// own reads, so the outcome is that of a serial run in which every voxel sees
// the state before the pass.
//
// One workgroup of 64 threads per block: thread (x, y) walks z = 0..7 in
// order, keeping its neighbour tallies across the walk, as the reference's
// per-thread arrays do (they are declared outside its z loop). The 27 blocks
// around a block are looked up once into LDS, and the label words of the block
// and its surroundings staged there.
//
// What bounds the update: instructions. The reference's probe computes each
// of 26 neighbours' voxels from world coordinates (three divisions each) and
// reads it from memory: 16000 instructions a block. A probe's voxel is the
// same function of one coordinate on each axis, so nine divisions serve a
// whole column's x and y and three each z; the probes then read the staged
// words; and where every neighbour bears the label tallied first (nine blocks
// in ten) one compare, count and maximum per neighbour replace the walk over
// the tallies. 6000 to 7000 visible blocks at 640x480 / 5 mm: 312 us before,
// 91 now; the blocks on a boundary, 43 us each against 11, set the end. Four
// wavefronts a SIMD (the staging loop holds its 21 loads in registers): three
// 92 us, five and more 111 to 127.
#include "map_common.hpp"
#include "sicp_internal.hpp"

namespace sicp {

namespace {

// Snapshot word: bits 0-7 label, bit 8 weight != 0, bits 16-31 count.
SICP_DEV uint32_t pack_label(const MapDev& m, size_t k) {
    const sicp_voxel_sem& s = m.sem[k];
    return (uint32_t)s.label | (vox_weight(m, k) != 0 ? 0x100u : 0u) | ((uint32_t)s.count << 16);
}

__global__ __launch_bounds__(256) void unify_snapshot_kernel(MapDev m, const MapCounters* ctr,
                                                             const sicp_block* visible,
                                                             uint32_t* snap, uint32_t* mark,
                                                             uint32_t* passes,
                                                             const int* gate) {
    if (gate && *gate == 0) return;
    const uint32_t nv = ctr->visible;
    const uint32_t epoch = passes[1] + 1u;
    if (blockIdx.x == 0 && threadIdx.x == 0) passes[0] = epoch;
    for (uint32_t b = blockIdx.x; b < nv; b += gridDim.x) {
        const int slot = visible[b].slot;
        if (threadIdx.x == 0) mark[slot] = epoch;
        const size_t base = (size_t)slot * 512;
        for (int i = threadIdx.x; i < 512; i += blockDim.x)
            snap[base + i] = pack_label(m, base + i);
    }
}

// The 26 neighbour offsets in the order UnifyNeighbor visits them
// (FuseMap.cu:838-892): +x with (y, z) in {0, +y, -y, +z, -z, ++, +-, -+, --}
// order, then -x likewise, then x = 0: +y, +y+z, +y-z, -y, -y+z, -y-z, +z, -z.
SICP_DEV void neighbour_offset(int k, int& dx, int& dy, int& dz) {
    if (k < 18) {
        dx = k < 9 ? 1 : -1;
        const int j = k % 9;
        // (dy, dz) for j = 0..8
        dy = (j == 1 || j == 5 || j == 6) ? 1 : ((j == 2 || j == 7 || j == 8) ? -1 : 0);
        dz = (j == 3 || j == 5 || j == 7) ? 1 : ((j == 4 || j == 6 || j == 8) ? -1 : 0);
    } else {
        dx = 0;
        const int j = k - 18;
        dy = j < 3 ? 1 : (j < 6 ? -1 : 0);
        const int q = j < 6 ? j % 3 : j - 6 + 1;
        dz = q == 1 ? 1 : (q == 2 ? -1 : 0);
    }
}

// Floor of a float coordinate to the voxel lattice (make_int3(float3),
// Utility/VectorMath.h:36-42).
SICP_DEV int floor_f(float a) {
    int b = f2i(a);
    return ((float)b > a) ? b - 1 : b;
}

// The staged label words: kSide^3 voxels from (-2, -2, -2) of the block on. The
// reference's probes at -1, 0, +1 voxel land on voxels -2 to +1 (the quotient of
// a coordinate by the voxel size may fall just short of the integer).
constexpr int kSide = 11, kBelow = 2, kWords = kSide * kSide * kSide;

// The voxels that the probes at -1, 0, +1 of coordinate v land on
// (voxelPosToWorldPos, DeviceMap.cu:165-167, +- VoxelSize, and back through
// FindVoxel(float3, Voxel&), :83-95, 154-163).
SICP_DEV void probe_voxels(int v, float vs, int (&n)[3]) {
    const float p = (float)v * vs, step = vs * (float)1;
    n[0] = floor_f((p - step) / vs);
    n[1] = floor_f(p / vs);
    n[2] = floor_f((p + step) / vs);
}

// One thread's tallies (UpdateNeighborLabel, FuseMap.cu:757-797): labels in
// the order met, each with its count and the largest label count seen.
struct Tallies {
    int label[4], count[4], best[4];
};
SICP_DEV void tally(Tallies& t, uint32_t w) {
    const int tl = (int)(w & 0xffu), tc = (int)(w >> 16);
    const bool weight = (w & 0x100u) != 0u;
    const bool known = t.label[0] == tl || t.label[1] == tl || t.label[2] == tl || t.label[3] == tl;
    bool free_before = false;  // an earlier free place: the places fill in order
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const bool free = t.label[l] == -1;
        const bool here = weight && (t.label[l] == tl || (!known && free && !free_before));
        free_before = free_before || free;
        t.label[l] = here ? tl : t.label[l];
        t.count[l] += here ? 1 : 0;
        t.best[l] = max(t.best[l], here ? tc : 0);
    }
}

__global__ __launch_bounds__(64, 4) void unify_kernel(MapDev m, const MapCounters* ctr,
                                                   const sicp_block* visible,
                                                   const uint32_t* snap, const uint32_t* mark,
                                                   uint32_t* passes, uint32_t count_mask,
                                                   const int* gate) {
    if (gate && *gate == 0) return;
    const uint32_t epoch = passes[0];
    __shared__ int nslot[27];
    __shared__ int nsnap[27];
    __shared__ uint32_t words[kWords];
    const uint32_t nv = ctr->visible;
    const int tx = threadIdx.x & 7, ty = threadIdx.x >> 3;
    const float vs = m.voxel;
    for (uint32_t b = blockIdx.x; b < nv; b += gridDim.x) {
        const sicp_block blk = visible[b];
        if (threadIdx.x < 27) {
            const int t = threadIdx.x;
            const int s = map_lookup(m, blk.x + t % 3 - 1, blk.y + (t / 3) % 3 - 1,
                                     blk.z + t / 9 - 1);
            nslot[t] = s;
            nsnap[t] = s >= 0 && mark[s] == epoch;
        }
        __syncthreads();
        // Every snapshot word's load in flight before the first is stored;
        // the words of blocks outside the snapshot (allocated, not visible)
        // are read from the map afterwards.
        constexpr int kEach = (kWords + 63) / 64;
        uint32_t w[kEach], live = 0u;
#pragma unroll
        for (int q = 0; q < kEach; ++q) {
            const int i = min((int)threadIdx.x + 64 * q, kWords - 1);
            const int x = i % kSide - kBelow, y = i / kSide % kSide - kBelow,
                      z = i / (kSide * kSide) - kBelow;
            const int t = ((z >> 3) + 1) * 9 + ((y >> 3) + 1) * 3 + (x >> 3) + 1;
            const int slot = nslot[t];
            const bool in = slot >= 0 && nsnap[t];
            const uint32_t v =
                snap[in ? (size_t)slot * 512 + ((z & 7) << 6) + ((y & 7) << 3) + (x & 7) : 0];
            w[q] = in ? v : 0u;  // a missing block's voxels count for nothing
            live |= (slot >= 0 && !in) ? 1u << q : 0u;
        }
#pragma unroll
        for (int q = 0; q < kEach; ++q)
            if ((int)threadIdx.x + 64 * q < kWords) words[threadIdx.x + 64 * q] = w[q];
        while (live) {
            const int q = __ffs((int)live) - 1;
            live &= live - 1u;
            const int i = min((int)threadIdx.x + 64 * q, kWords - 1);
            const int x = i % kSide - kBelow, y = i / kSide % kSide - kBelow,
                      z = i / (kSide * kSide) - kBelow;
            const int slot = nslot[((z >> 3) + 1) * 9 + ((y >> 3) + 1) * 3 + (x >> 3) + 1];
            words[i] = pack_label(m, (size_t)slot * 512 + ((z & 7) << 6) + ((y & 7) << 3) + (x & 7));
        }
        __syncthreads();
        Tallies tl;
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            tl.label[l] = -1;
            tl.count[l] = 0;
            tl.best[l] = 0;
        }
        const size_t own = (size_t)blk.slot * 512;
        int nx[3], ny[3], xy[3][3];
        probe_voxels(blk.x * 8 + tx, vs, nx);
        probe_voxels(blk.y * 8 + ty, vs, ny);
        bool staged_xy = true;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int rx = nx[i] - (blk.x * 8 - kBelow), ry = ny[i] - (blk.y * 8 - kBelow);
            staged_xy = staged_xy && (unsigned)rx < (unsigned)kSide && (unsigned)ry < (unsigned)kSide;
        }
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int i = 0; i < 3; ++i)
                xy[j][i] = (ny[j] - (blk.y * 8 - kBelow)) * kSide + nx[i] - (blk.x * 8 - kBelow);
#pragma unroll 1
        for (int z = 0; z < 8; ++z) {
            const int li = z * 64 + ty * 8 + tx;
            const uint32_t cw =
                words[((z + kBelow) * kSide + ty + kBelow) * kSide + tx + kBelow];
            const int cur_label = (cw & 0x100u) ? (int)(cw & 0xffu) : -1;
            if (cur_label == -1) continue;
            int nz[3];
            probe_voxels(blk.z * 8 + z, vs, nz);
            bool staged = staged_xy;
#pragma unroll
            for (int i = 0; i < 3; ++i)
                staged = staged && (unsigned)(nz[i] - (blk.z * 8 - kBelow)) < (unsigned)kSide;
            // Every neighbour without a label, or with the first tallied one
            // (this voxel's own, when there is none yet)?
            const uint32_t want = 0x100u | (uint32_t)(tl.label[0] < 0 ? cur_label : tl.label[0]);
            bool plain = staged;
            if (staged) {
                uint32_t same = 0u, top = 0u, other = 0u;
#pragma unroll 1
                for (int c = 0; c < 3; ++c) {
                    const int vz = c == 0 ? nz[0] : (c == 1 ? nz[1] : nz[2]);
                    const int zo = (vz - (blk.z * 8 - kBelow)) * (kSide * kSide);
#pragma unroll
                    for (int j = 0; j < 3; ++j)
#pragma unroll
                        for (int i = 0; i < 3; ++i) {
                            uint32_t w = words[zo + xy[j][i]];
                            if (j == 1 && i == 1) w = c == 1 ? 0u : w;  // not itself
                            const uint32_t e = (w & 0x1ffu) == want ? w : 0u;
                            same += (e >> 8) & 1u;  // the word's own weight bit
                            top = max(top, e);
                            other |= w ^ e;
                        }
                }
                plain = !(other & 0x100u);
                if (plain && same != 0u) {
                    const int tc = (int)(top >> 16);
                    tl.label[0] = (int)(want & 0xffu);
                    tl.count[0] += (int)same;
                    tl.best[0] = tl.best[0] > tc ? tl.best[0] : tc;
                }
            }
            if (!plain && staged) {  // in the reference's order
                int zo[3];
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    zo[c] = (nz[c] - (blk.z * 8 - kBelow)) * (kSide * kSide);
#pragma unroll
                for (int k = 0; k < 26; ++k) {
                    int dx, dy, dz;
                    neighbour_offset(k, dx, dy, dz);
                    tally(tl, words[zo[dz + 1] + xy[dy + 1][dx + 1]]);
                }
            } else if (!plain) {  // coordinates too large for the voxel size's rounding
#pragma unroll 1
                for (int k = 0; k < 26; ++k) {
                    int dx, dy, dz;
                    neighbour_offset(k, dx, dy, dz);
                    const int vx = dx > 0 ? nx[2] : (dx < 0 ? nx[0] : nx[1]);
                    const int vy = dy > 0 ? ny[2] : (dy < 0 ? ny[0] : ny[1]);
                    const int vz = dz > 0 ? nz[2] : (dz < 0 ? nz[0] : nz[1]);
                    const int slot = map_lookup(m, vx >> 3, vy >> 3, vz >> 3);
                    if (slot < 0) continue;
                    const size_t vi =
                        (size_t)slot * 512 + ((vz & 7) << 6) + ((vy & 7) << 3) + (vx & 7);
                    tally(tl, mark[slot] == epoch ? snap[vi] : pack_label(m, vi));
                }
            }
            // the most frequent neighbour label with a non-zero count
            // (FuseMap.cu:903-917); the first of equals wins
            int nl = -1, nc = 0, nlc = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (tl.label[j] != -1 && tl.best[j] != 0 && tl.count[j] > nc) {
                    nl = tl.label[j];
                    nc = tl.count[j];
                    nlc = tl.best[j];
                }
            // FuseMap.cu:926-944; narrowing to the count's width
            sicp_voxel_sem& cur = m.sem[own + li];
            if (cur_label != nl) {
                const int cur_count = (int)(cw >> 16);
                int tmp;
                if (cur_label == (int)cur.label2)
                    tmp = nlc > (int)cur.count2 ? nlc : ((int)cur.count2 + 5);
                else
                    tmp = nlc;
                cur.label2 = (uint8_t)cur_label;
                cur.count2 = (uint16_t)cur_count;
                cur.label = (uint8_t)nl;
                cur.count = (uint16_t)((uint32_t)tmp & count_mask);
            } else if (((uint32_t)nlc & count_mask) != cw >> 16) {
                cur.count = (uint16_t)((uint32_t)nlc & count_mask);
            }
        }
        __syncthreads();
    }
    // (here: at the start it costs a spilled register)
    if (blockIdx.x == 0 && threadIdx.x == 0) passes[1] = epoch;
}

}  // namespace

int unify_scratch(sicp_map* map) {
    const size_t n = (size_t)map->cfg.num_blocks;
    uint32_t *snap = nullptr, *mark = nullptr;
    hipError_t e = hipMalloc((void**)&snap, n * kBlockVoxels * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMalloc((void**)&mark, (n + 2) * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMemset(mark, 0, (n + 2) * sizeof(uint32_t));
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    if (e != hipSuccess) {
        if (snap) (void)hipFree(snap);
        if (mark) (void)hipFree(mark);
        return hip_fail(e, "hipMalloc(unify scratch)");
    }
    map->unify_snap = snap;
    map->unify_mark = mark;
    map->owned.push_back(snap);
    map->owned.push_back(mark);
    return SICP_OK;
}

int launch_unify(sicp_map* map, const int* gate, hipStream_t s) {
    if (!map->unify_snap) {
        const int rc = unify_scratch(map);
        if (rc) return rc;
    }
    // The pass's number tells the blocks that it stamped from those of earlier
    // passes. It is kept on the device, so that a replayed graph counts on: the
    // snapshot forms it from the passes that ended, [1], and leaves it in [0];
    // the update takes it from there and stores it in [1], so neither launch
    // reads the word that it writes. The marks start at 0, the first pass is 1.
    uint32_t* passes = map->unify_mark + map->cfg.num_blocks;
    const uint32_t mask = map->cfg.max_label_count <= 255 ? 0xffu : 0xffffu;
    unify_snapshot_kernel<<<4096, 256, 0, s>>>(map->dev, map->ctr, map->visible, map->unify_snap,
                                                map->unify_mark, passes, gate);
    SICP_LAUNCH_CHECK("unify_snapshot_kernel");
    unify_kernel<<<8192, 64, 0, s>>>(map->dev, map->ctr, map->visible, map->unify_snap,
                                      map->unify_mark, passes, mask, gate);
    SICP_LAUNCH_CHECK("unify_kernel");
    return SICP_OK;
}

}  // namespace sicp
