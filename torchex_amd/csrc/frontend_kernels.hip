// The callers on either side of the scatter operators: voxel keys from points,
// the unique / inverse / counts triple (from an occupancy map of the key grid, or from
// the same sort the scatter plan uses),
// the rank of an element inside its group, points-in-boxes pooling, and the
// coordinate hash table.
//
// Reference behaviour being replaced: voxelize_single
// (test/test_incremental_mask.py:20-26), ingroup_inds
// (torchex/src/ingroup_inds/ingroup_inds_kernel.cu:17-30), dynamic_point_pool
// (torchex/src/dynamic_point_pool/dynamic_point_pool_kernel.cu:22-170,280-310),
// grid_hash (torchex/src/grid_hash/grid_hash_kernel.cu:19-49,
// torchex/src/utils/functions.cuh:30-64).

#include "key_map.h"
#include "txs_internal.h"

namespace {

using txs_detail::exclusive_scan;
using txs_detail::KeyMap;
using txs_detail::scan_tiles;

__global__ void fill_i32_kernel(int *p, long n, int value) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

// ------------------------------------------------ voxelization front-end --

// torch.div(a, b, rounding_mode='floor') for fp32 (c10::div_floor_floating,
// c10/util/generic_math.h): Python's floor division, not floor(a / b).
__device__ __forceinline__ float div_floor_f32(float a, float b) {
    if (b == 0.0f) return a / b;
    const float mod = fmodf(a, b);
    float div = (a - mod) / b;
    if ((mod != 0.0f) && ((b < 0.0f) != (mod < 0.0f))) div -= 1.0f;
    float fl;
    if (div != 0.0f) {
        fl = floorf(div);
        if (div - fl > 0.5f) fl += 1.0f;
    } else {
        fl = copysignf(0.0f, a / b);
    }
    return fl;
}

// coors = floor((p - lo) / voxel) per axis, key = (x * Y + y) * Z + z
// (test/test_incremental_mask.py:20-26, operator_py/incremental_points.py:18-19)
// flag: set to 1 if a point lies outside the grid; map (may be NULL): the keys' occupancy map, marked
__global__ void voxel_keys_kernel(const float *__restrict__ pts, long n, int stride, float lo0,
                                  float lo1, float lo2, float v0, float v1, float v2, int d0, int d1,
                                  int d2, int *__restrict__ coors, int *__restrict__ keys,
                                  int *__restrict__ flag, unsigned char *__restrict__ map) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float *p = pts + i * stride;
    const int x = (int)div_floor_f32(p[0] - lo0, v0);
    const int y = (int)div_floor_f32(p[1] - lo1, v1);
    const int z = (int)div_floor_f32(p[2] - lo2, v2);
    if (coors) {
        coors[i * 3 + 0] = x;
        coors[i * 3 + 1] = y;
        coors[i * 3 + 2] = z;
    }
    const bool ok = (unsigned)x < (unsigned)d0 && (unsigned)y < (unsigned)d1 && (unsigned)z < (unsigned)d2;
    const int key = ok ? (x * d1 + y) * d2 + z : 0;
    if (!ok) flag[0] = 1;
    keys[i] = key;
    if (map) map[key] = 1;
}

// 1 where a new run of equal keys starts
__global__ void run_flags_kernel(const int *__restrict__ ks, long n, int *__restrict__ flags) {
    long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) flags[j] = (j == 0 || ks[j] != ks[j - 1]) ? 1 : 0;
}

// What torch.unique(keys, return_inverse=True, return_counts=True) returns,
// from the sorted keys and the exclusive scan `ex` of the run-start flags,
// plus the plan arrays: run index rid = ex[j] + flag - 1.
__global__ void unique_finish_kernel(const int *__restrict__ ks, const int *__restrict__ perm,
                                     const int *__restrict__ ex, long n, int *__restrict__ seg,
                                     int *__restrict__ inv, int *__restrict__ unq,
                                     int *__restrict__ preSum, int *__restrict__ stats) {
    long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const bool flag = (j == 0 || ks[j] != ks[j - 1]);
    const int rid = ex[j] + (flag ? 1 : 0) - 1;
    const int row = stats[TXS_STAT_UNSORTED] ? perm[j] : (int)j;
    seg[j] = rid;
    if ((unsigned)row < (unsigned)n) inv[row] = rid;
    if (flag) {
        unq[rid] = ks[j];
        preSum[rid] = (int)j;
    }
    if (j == n - 1) {
        preSum[rid + 1] = (int)n;
        stats[TXS_STAT_NUM_UNQ] = rid + 1;
    }
}


// ---- unique by occupancy map (keys from a bounded grid) ----------------------
// One byte per possible key, set by plain stores (every writer stores the same 1, so no
// atomic is needed; device-scope atomics on a bitmap were measured at 220 us for 1M keys),
// then packed into a cell per 32 keys.  The dense id of a key is the number of occupied keys
// below it: those of the tiles of cells in front, of the cells in front in its tile, and the bits
// below the key inside its cell.  That is the inverse torch.unique returns (ids ascend with the
// keys), found without sorting the keys.

// Where the keys come from: an array of them, or voxel coordinates [n, 3], linearised here
// (x-major, and cut to 32 bits before the range check, as a caller who stores int32 keys would).
template <typename K>
struct FlatKeys {
    const K *p;
    __device__ __forceinline__ long operator()(long i) const { return (long)p[i]; }
};
template <typename K>
struct CoorKeys {
    const K *p;
    long s0, s1;  // strides of x and y in the key
    __device__ __forceinline__ long operator()(long i) const {
        const K *c = p + 3 * i;
        return (long)(int)(unsigned)((unsigned long)c[0] * (unsigned long)s0 + (unsigned long)c[1] * (unsigned long)s1 +
                                     (unsigned long)c[2]);
    }
};

// bad (may be NULL): an int cleared along with the map
__global__ void bytemap_clear_kernel(uint4 *__restrict__ map16, long n16, int *__restrict__ bad) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n16) map16[i] = make_uint4(0u, 0u, 0u, 0u);
    if (bad && i == 0) bad[0] = 0;
}

// bad: set to 1 if a key lies outside [0, key_bound)
template <class Keys>
__global__ void bytemap_mark_kernel(Keys keys, long n, long key_bound, unsigned char *__restrict__ map,
                                    int *__restrict__ bad) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long k = keys(i);
    if (k < 0 || k >= key_bound) {
        bad[0] = 1;
        return;
    }
    map[k] = 1;
}

// 32 map bytes (each 0 or 1) -> one cell of the map: their bits, and how many keys occur in the cells in
// front of it in its tile of kScanTileItems; the number of keys per tile (a workgroup each).  What is in
// front of a tile is added up by those who read the cells: a few hundred numbers, against a scan over
// all cells (5 us of a frame's 16.9M keys, in a launch of its own).
constexpr int kPackThreads = 1024;
__global__ __launch_bounds__(kPackThreads) void bytemap_pack_kernel(const uint4 *__restrict__ map16, long words,
                                                                    uint2 *__restrict__ cells, int *__restrict__ tiles) {
    constexpr int kItems = txs_detail::kScanTileItems / kPackThreads;
    __shared__ int s_sum[kPackThreads / 64];
    // bytes b0..b3 of a word, each 0 or 1 -> bits 0..3: (x * 0x10204080) >> 28 leaves b0 + 2 b1 + 4 b2 + 8 b3
    auto nib = [](unsigned x) -> unsigned { return ((x * 0x10204080u) >> 28) & 15u; };
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long w0 = (long)blockIdx.x * txs_detail::kScanTileItems + (long)threadIdx.x * kItems;
    uint4 lo[kItems], hi[kItems];
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        const bool in = w0 + it < words;
        lo[it] = in ? map16[2 * (w0 + it)] : make_uint4(0u, 0u, 0u, 0u);
        hi[it] = in ? map16[2 * (w0 + it) + 1] : make_uint4(0u, 0u, 0u, 0u);
    }
    unsigned word[kItems];
    int sum = 0;
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        word[it] = nib(lo[it].x) | (nib(lo[it].y) << 4) | (nib(lo[it].z) << 8) | (nib(lo[it].w) << 12) |
                   (nib(hi[it].x) << 16) | (nib(hi[it].y) << 20) | (nib(hi[it].z) << 24) | (nib(hi[it].w) << 28);
        sum += __popc(word[it]);
    }
    const int inc = wave_inclusive_scan(sum);
    if (lane == 63) s_sum[wave] = inc;
    __syncthreads();
    int at = inc - sum, total = 0;
#pragma unroll
    for (int k = 0; k < kPackThreads / 64; ++k) {
        if (k < wave) at += s_sum[k];
        total += s_sum[k];
    }
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
        if (w0 + it < words) cells[w0 + it] = make_uint2(word[it], (unsigned)at);
        at += __popc(word[it]);
    }
    if (threadIdx.x == 0) tiles[blockIdx.x] = total;
}

// the number of distinct keys, by one workgroup
__global__ __launch_bounds__(kThreads) void map_total_kernel(KeyMap m) {
    __shared__ int base_s[txs_detail::kMapTilesSummed];
    const int total = map_tile_bases<kThreads>(m, base_s);
    if (threadIdx.x == 0) m.num_unq[0] = total;
}

// Ids of all keys, and the distinct keys: workgroups behind those of the rows list a part of the cells each.
// Several rows a thread, all of whose loads are in flight together, as every workgroup adds up the map's tiles
// first (plans from 16M sorted keys in 2^20: a row a thread 402 us, eight 374).
constexpr int kAssignItems = 8;
constexpr int kAssignRows = kThreads * kAssignItems;
__global__ __launch_bounds__(kThreads) void map_assign_kernel(KeyMap m, long n, int *__restrict__ inv) {
    __shared__ int base_s[txs_detail::kMapTilesSummed];
    const int total = map_tile_bases<kThreads>(m, base_s);
    if (m.num_unq && blockIdx.x == 0 && threadIdx.x == 0) {
        m.num_unq[0] = total;
        if (m.found) {
            m.found[0] = total;
            m.found[1] = m.bad[0];
        }
    }
    const long row_groups = (n + kAssignRows - 1) / kAssignRows;
    if ((long)blockIdx.x >= row_groups) {
        map_list_part<kThreads>(m, base_s, (long)blockIdx.x - row_groups);
        return;
    }
    const long row0 = (long)blockIdx.x * kAssignRows + threadIdx.x;
    int key[kAssignItems];
    uint2 cell[kAssignItems];
#pragma unroll
    for (int it = 0; it < kAssignItems; ++it) key[it] = map_key(m, min(row0 + it * kThreads, n - 1));
#pragma unroll
    for (int it = 0; it < kAssignItems; ++it) cell[it] = m.cells[key[it] >> 5];
#pragma unroll
    for (int it = 0; it < kAssignItems; ++it)
        if (row0 + it * kThreads < n) inv[row0 + it * kThreads] = map_id(m, base_s, cell[it], key[it]);
}
// workgroups of map_assign_kernel
dim3 assign_grid(long n, const KeyMap &m) { return dim3((unsigned)((n + kAssignRows - 1) / kAssignRows + map_parts(m))); }

// counts of the voxels from their CSR offsets, as int64 (what torch.unique returns)
__global__ void counts_from_presum_kernel(const int *__restrict__ preSum, long U, long long *__restrict__ cnts) {
    const long u = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (u < U) cnts[u] = (long long)(preSum[u + 1] - preSum[u]);
}

// rank of every element inside its group (operator_py/ingroup_inds_op.py,
// src/ingroup_inds/ingroup_inds_kernel.cu:17-30): sorted position minus the
// group's first position; ascending with the element's index, where the
// reference's atomic counter hands ranks out in arbitrary order.
__global__ void ingroup_inds_kernel(const int *__restrict__ seg, const int *__restrict__ perm,
                                    const int *__restrict__ preSum, long n, int U,
                                    long long *__restrict__ out) {
    long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int u = seg[j] & kIdMask;
    const int row = perm ? perm[j] : (int)j;
    if ((unsigned)u < (unsigned)U && (unsigned)row < (unsigned)n) out[row] = (long long)(j - preSum[u]);
}

// the same from a plan whose order flag is still on the device: stats[UNSORTED] says whether
// perm was written (rows already in order leave it unwritten: position == row); a plan that
// was not completed (ids out of range, or handed to the general sequence) is left alone
__global__ void ingroup_inds_auto_kernel(const int *__restrict__ seg, const int *__restrict__ perm,
                                         const int *__restrict__ preSum, const int *__restrict__ stats,
                                         long n, int U, long long *__restrict__ out) {
    long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    if (stats[TXS_STAT_OUT_OF_RANGE] != 0 || stats[TXS_STAT_NEED_GENERAL] != 0) return;
    const int u = seg[j] & kIdMask;
    const int row = stats[TXS_STAT_UNSORTED] != 0 ? perm[j] : (int)j;
    if ((unsigned)u < (unsigned)U && (unsigned)row < (unsigned)n) out[row] = (long long)(j - preSum[u]);
}

// ------------------------------------------------------ dynamic point pool --
// Points inside (enlarged) rotated boxes, with 13 box-relative numbers per hit
// (torchex/src/dynamic_point_pool/dynamic_point_pool_kernel.cu:22-170,280-310).
// The reference compacts the hits with two atomic counters, so their order and,
// when a cap is hit, the surviving subset depend on thread timing.  Here every
// test leaves one bit in a (box, point) bit matrix, with the hits counted per
// (box, tile of 1024 points) and per box, and the set bits are then written in
// (box, point) order: the outcome the reference's own comment calls the usual
// one ("out_roi_idx is automatically sorted"), made deterministic.  The count of
// hits per tile of 256 points and group of 8 boxes, a scan, and a second pass over all results, which
// this replaces, took 34 + 10 + 30 us for 200 boxes and 200k points; the first pass takes 11 now,
// the writing 10.

constexpr int kDppInfo = 13;

struct DppBox {
    float cx, cy, czc, w, l, h, cosa, sina, cz_bottom;
    float half_w, half_l, half_h, half_large_w, half_large_l, half_large_h;  // see half_of
    float r2;  // squared radius of a circle around (cx, cy) that contains the box and its margin
};

// The hits per box are counted by one atomic per tile and box.  Such atomics on one cache line
// complete one after the other, so every box's count has a line of its own: packed, 200 of
// them on 7 lines, they held the first pass up (200 boxes, 200k points: 33-36 -> 27 us).
constexpr int kDppTotalStep = 32;  // ints from one box's count to the next

// The reference compares floats with (double)side / 2.0.  Half a side as a float is the same bound where it is
// exact; the half of an odd multiple of the smallest float is not, and is then rounded `up` for v < half and
// v > -half, down for v > half, which no float v can tell from the exact one.  (Tests in 64 bits: the first pass of
// 32 boxes around all of 100k points 51.5 us, now 47.6.)
__device__ __forceinline__ float half_of(float side, bool up) {
    const float half = 0.5f * side;
    if (up && half + half < side) return nextafterf(half, INFINITY);
    if (!up && half + half > side) return nextafterf(half, -INFINITY);
    return half;
}

// per-box constants, computed once so both passes see identical numbers; the
// rotation terms are evaluated in double and rounded (within an ulp of any cosf)
__global__ void dpp_box_kernel(const float *__restrict__ rois, int B, float extra_w, float extra_l,
                               float extra_h, DppBox *__restrict__ boxes, int *__restrict__ totals) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    totals[(size_t)b * kDppTotalStep] = 0;
    const float *r = rois + (size_t)b * 7;
    DppBox bx;
    bx.cx = r[0];
    bx.cy = r[1];
    bx.cz_bottom = r[2];
    bx.w = r[3];
    bx.l = r[4];
    bx.h = r[5];
    const float large_w = bx.w + extra_w, large_l = bx.l + extra_l, large_h = bx.h + extra_h;
    bx.half_w = half_of(bx.w, true);
    bx.half_l = half_of(bx.l, true);
    bx.half_h = half_of(bx.h, true);
    bx.half_large_w = half_of(large_w, true);
    bx.half_large_l = half_of(large_l, true);
    bx.half_large_h = half_of(large_h, false);
    bx.czc = (float)((double)r[2] + (double)bx.h / 2.0);  // bottom centre -> centre (:46)
    const float rot = (float)((double)r[6] + 3.14159265358979323846 / 2);  // (:24)
    bx.cosa = (float)cos((double)rot);
    bx.sina = (float)sin((double)rot);
    // generous bound (0.1 % + 1 mm^2): a point outside this circle fails the exact
    // test whatever the rounding, so skipping it cannot change the result
    const float hl = 0.5f * fmaxf(fabsf(bx.l), fabsf(large_l));
    const float hw = 0.5f * fmaxf(fabsf(bx.w), fabsf(large_w));
    bx.r2 = (hl * hl + hw * hw) * 1.001f + 1e-6f;
    boxes[b] = bx;
}

// cheap conservative reject in the xy plane; most waves skip the exact test with it
__device__ __forceinline__ bool dpp_near(const DppBox &bx, float x, float y) {
    const float sx = x - bx.cx, sy = y - bx.cy;
    return sx * sx + sy * sy <= bx.r2;
}

// 0: outside the enlarged box, 1: in the margin, 2: inside the box (:33-71)
__device__ __forceinline__ int dpp_test(const DppBox &bx, float x, float y, float z, float &local_x,
                                        float &local_y) {
#pragma clang fp contract(off)
    const float dz = fabsf(z - bx.czc);
    if (dz > bx.half_large_h) return 0;
    const float sx = x - bx.cx, sy = y - bx.cy;
    local_x = sx * bx.cosa + sy * (-bx.sina);
    local_y = sx * bx.sina + sy * bx.cosa;
    const bool in_box = (local_x > -bx.half_l) & (local_x < bx.half_l) & (local_y > -bx.half_w) &
                        (local_y < bx.half_w) & (dz < bx.half_h);
    const bool in_large = (local_x > -bx.half_large_l) & (local_x < bx.half_large_l) &
                          (local_y > -bx.half_large_w) & (local_y < bx.half_large_w);
    return in_box ? 2 : (in_large ? 1 : 0);
}

// What a lane of the wave has written to LDS in front of this, every other lane sees behind it (the hardware keeps
// a wave's LDS accesses in order by itself; this holds the compiler to it).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A workgroup takes 1024 points, four per lane, and kDppGroup boxes.  It lays a grid of kDppCells x kDppCells
// cells over its boxes and marks in every cell the boxes whose circle may reach it; a point looks its
// cell up and meets those boxes alone.  The pairs are queued by wave and tested 64 at a time, whatever their
// boxes.  Every point against every box's circle was bound by the vector units, ten instructions for each of
// 40M pairs of 200 boxes and 200k points, and the exact test behind it ran with few lanes: 27 us, now 11.
// The words of the bit matrix are collected in LDS and leave as whole lines (16 words of a box).
constexpr int kDppItems = 4;
constexpr int kDppTile = kThreads * kDppItems;
constexpr int kDppWords = kDppTile / 64;   // words of a tile per box
constexpr int kDppGroup = 32;              // boxes per workgroup
constexpr int kDppSegTiles = kThreads / kDppWords;  // tiles an emitting workgroup covers: one word per thread
constexpr int kDppCells = 32;
// Hits of a segment that are listed: with room for all 16384 points a compute unit took four of the emitting
// workgroups, of which nearly all list a handful (200 boxes, 200k points, no cap: 56 us, now 53).
constexpr int kDppListed = 8192;
constexpr int kDppDense = 24;              // points of a wave that may lie in a box from which on they are not queued
constexpr float kDppFar = 1e15f;           // boxes further out or larger than this are tested against every point
constexpr int kDppSumBoxes = 2048;         // up to this many boxes the emitting workgroups add up the boxes in front themselves

// (pts_batch / rois_batch, both NULL or both given: a point meets only the boxes of its own
// sample, generate_pts_mask_for_box3d_mixed, dynamic_point_pool_kernel.cu:173-212)
__global__ __launch_bounds__(kThreads) void dpp_mask_kernel(const float *__restrict__ pts, int P,
                                                            const DppBox *__restrict__ boxes, int B, int n_tiles,
                                                            unsigned long long *__restrict__ masks,
                                                            int *__restrict__ counts, int *__restrict__ totals,
                                                            const int *__restrict__ pts_batch,
                                                            const int *__restrict__ rois_batch) {
    __shared__ unsigned long long m_s[kDppGroup][kDppWords];
    __shared__ float pts_s[3][kDppTile];
    __shared__ DppBox boxes_s[kDppGroup];
    __shared__ int box_sample_s[kDppGroup];
    __shared__ unsigned cells_s[kDppCells * kDppCells];     // a bit per box
    __shared__ unsigned short queue_s[kThreads / 64][128];  // box << 10 | point, of the workgroup's boxes and points
    __shared__ float grid_s[4];                             // corner, cells per unit of x and y
    __shared__ unsigned everywhere_s;
    static_assert(kDppTile == 1 << 10 && kDppGroup == 32, "a pair fits in 16 bits, a cell's boxes in 32");
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned long long lanes_below = (1ull << lane) - 1ull;
    const int b0 = blockIdx.y * kDppGroup;
    const int nb = min(kDppGroup, B - b0);
    float x[kDppItems], y[kDppItems];
    int sample[kDppItems];
    bool in[kDppItems];
#pragma unroll
    for (int it = 0; it < kDppItems; ++it) {
        const int at = w * (64 * kDppItems) + it * 64 + lane;
        const long p = (long)blockIdx.x * kDppTile + at;
        in[it] = p < P;
        const size_t q = in[it] ? (size_t)p : 0;
        x[it] = pts_s[0][at] = pts[q * 3];
        y[it] = pts_s[1][at] = pts[q * 3 + 1];
        pts_s[2][at] = pts[q * 3 + 2];
        sample[it] = pts_batch ? pts_batch[q] : 0;
    }
    constexpr int kBoxWords = sizeof(DppBox) / sizeof(int);
    for (int t = threadIdx.x; t < nb * kBoxWords; t += kThreads)
        reinterpret_cast<int *>(boxes_s)[t] = reinterpret_cast<const int *>(boxes + b0)[t];
    if ((int)threadIdx.x < nb) box_sample_s[threadIdx.x] = rois_batch ? rois_batch[b0 + threadIdx.x] : 0;
    for (int t = threadIdx.x; t < kDppGroup * kDppWords; t += kThreads) (&m_s[0][0])[t] = 0ull;
    for (int t = threadIdx.x; t < kDppCells * kDppCells; t += kThreads) cells_s[t] = 0u;
    __syncthreads();
    // ---- the grid.  Eight threads a box; a box's square holds its circle whatever the rounding of its sides
    // (a few parts in 10^7 of the coordinates), and a box of no finite or sensible square, or of most of the grid, is everywhere.
    const int mine = (int)threadIdx.x >> 3, sub = threadIdx.x & 7;
    float lo[2] = {INFINITY, INFINITY}, hi[2] = {-INFINITY, -INFINITY};
    bool far = false;
    if (mine < nb) {
        const DppBox &bx = boxes_s[mine];
        const float r = sqrtf(bx.r2) * 1.0001f;
        const float c[2] = {bx.cx, bx.cy};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            lo[k] = c[k] - r - fabsf(c[k]) * 4e-7f;
            hi[k] = c[k] + r + fabsf(c[k]) * 4e-7f;
            far |= !(lo[k] > -kDppFar && hi[k] < kDppFar);
        }
    }
    if (w == 0) {  // (32 boxes: one wave looks at all of them for the corners)
        float l[2] = {INFINITY, INFINITY}, h[2] = {-INFINITY, -INFINITY};
        bool out = false;
        if (lane < nb) {
            const DppBox &bx = boxes_s[lane];
            const float r = sqrtf(bx.r2) * 1.0001f;
            const float c[2] = {bx.cx, bx.cy};
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                l[k] = c[k] - r - fabsf(c[k]) * 4e-7f;
                h[k] = c[k] + r + fabsf(c[k]) * 4e-7f;
                out |= !(l[k] > -kDppFar && h[k] < kDppFar);
            }
        }
        const unsigned long long outs = __ballot(out);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (out) {
                l[k] = INFINITY;
                h[k] = -INFINITY;
            }
#pragma unroll
            for (int d = 16; d >= 1; d >>= 1) {
                l[k] = fminf(l[k], __shfl_xor(l[k], d, 64));
                h[k] = fmaxf(h[k], __shfl_xor(h[k], d, 64));
            }
        }
        if (lane == 0) {
            everywhere_s = (unsigned)outs;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                grid_s[k] = l[k];
                grid_s[2 + k] = h[k] > l[k] ? kDppCells / (h[k] - l[k]) : 0.0f;
            }
        }
    }
    __syncthreads();
    // a coordinate's place in the grid, and so its cell, ascends with it, rounding included, so that a point inside
    // a box's square lies in one of the cells from that of its lower to that of its upper side.  Either side
    // may round to the grid's very end (with one box far out on the negative side, those of all others do).
    auto place = [&](int axis, float v) { return (v - grid_s[axis]) * grid_s[2 + axis]; };
    auto cell = [](float at) { return min(kDppCells - 1, max(0, (int)at)); };
    if (mine < nb && !far) {
        const int x0 = cell(place(0, lo[0])), x1 = cell(place(0, hi[0]));
        const int y0 = cell(place(1, lo[1])), y1 = cell(place(1, hi[1]));
        if ((x1 - x0 + 1) * (y1 - y0 + 1) > kDppCells * kDppCells / 2) {  // (most points are to be tested anyway)
            if (sub == 0) atomicOr(&everywhere_s, 1u << mine);
        } else {
            for (int cy = y0 + sub; cy <= y1; cy += 8)
                for (int cx = x0; cx <= x1; ++cx) atomicOr(&cells_s[cy * kDppCells + cx], 1u << mine);
        }
    }
    __syncthreads();
    // ---- boxes that are everywhere: every point, one box after the other (heights in registers: read again for
    // every box, each step of this chain waited for LDS as well)
    float z[kDppItems];
#pragma unroll
    for (int it = 0; it < kDppItems; ++it) z[it] = pts_s[2][w * (64 * kDppItems) + it * 64 + lane];
    for (unsigned left = __builtin_amdgcn_readfirstlane(everywhere_s); left != 0u; left &= left - 1u) {
        const int bb = __builtin_ctz(left);
        const DppBox &bx = boxes[b0 + bb];
        const int box_sample = rois_batch ? rois_batch[b0 + bb] : 0;
        bool near[kDppItems], any = false;
#pragma unroll
        for (int it = 0; it < kDppItems; ++it) {
            near[it] = in[it] && sample[it] == box_sample && dpp_near(bx, x[it], y[it]);
            any |= near[it];
        }
        if (__ballot(any) == 0ull) continue;
#pragma unroll
        for (int it = 0; it < kDppItems; ++it) {
            float lx, ly;
            const unsigned long long hits = __ballot(near[it] && dpp_test(bx, x[it], y[it], z[it], lx, ly) != 0);
            if (lane == 0) m_s[bb][w * kDppItems + it] = hits;
        }
    }
    // ---- the others: those of a point's cell
    // the last `count` (at most 64) queued pairs
    auto test = [&](int queued, int count) {
        if (lane >= count) return;
        const int pair = queue_s[w][queued - count + lane], bb = pair >> 10, at = pair & (kDppTile - 1);
        const DppBox &bx = boxes_s[bb];
        const float px = pts_s[0][at], py = pts_s[1][at];
        float lx, ly;
        if (dpp_near(bx, px, py) && dpp_test(bx, px, py, pts_s[2][at], lx, ly) != 0)
            atomicOr(reinterpret_cast<unsigned *>(&m_s[bb][0]) + (at >> 5), 1u << (at & 31));
    };
    int queued = 0;
#pragma unroll
    for (int it = 0; it < kDppItems; ++it) {
        unsigned boxes_here = 0u;
        if (in[it]) {
            const float gx = place(0, x[it]), gy = place(1, y[it]);
            // (a place at the very end may round up to kDppCells; NaN is nowhere)
            const bool inside = gx >= 0.0f && gx < kDppCells + 0.5f && gy >= 0.0f && gy < kDppCells + 0.5f;
            boxes_here = inside ? cells_s[cell(gy) * kDppCells + cell(gx)] : 0u;
        }
        for (unsigned long long left = __ballot(boxes_here != 0u); left != 0ull; left = __ballot(boxes_here != 0u)) {
            // a box that many of the wave's points may lie in is put to the test at once
            const int wide = __builtin_ctz(__shfl((int)boxes_here, __builtin_ctzll(left), 64));  // (uniform)
            const bool mine_too = (boxes_here >> wide & 1u) != 0u;
            if (__popcll(__ballot(mine_too)) >= kDppDense) {
                float lx, ly;
                const DppBox &bx = boxes_s[wide];
                const unsigned long long hits =
                    __ballot(mine_too && sample[it] == box_sample_s[wide] && dpp_near(bx, x[it], y[it]) &&
                             dpp_test(bx, x[it], y[it], pts_s[2][w * (64 * kDppItems) + it * 64 + lane], lx, ly) != 0);
                if (lane == 0 && hits) atomicOr(&m_s[wide][w * kDppItems + it], hits);
                boxes_here &= ~(1u << wide);
                continue;
            }
            const int bb = boxes_here ? __builtin_ctz(boxes_here) : 0;
            const bool meet = boxes_here != 0u && sample[it] == box_sample_s[bb];
            const unsigned long long m = __ballot(meet);
            if (meet) queue_s[w][queued + __popcll(m & lanes_below)] = (unsigned short)(bb << 10 | (w * (64 * kDppItems) + it * 64 + lane));
            queued += __popcll(m);
            boxes_here &= boxes_here - 1u;
            wave_lds_fence();
            if (queued >= 64) {
                test(queued, 64);
                queued -= 64;
                wave_lds_fence();
            }
        }
    }
    test(queued, queued);
    __syncthreads();
    for (int t = threadIdx.x; t < nb * kDppWords; t += kThreads) {
        const int bb = t / kDppWords, k = t % kDppWords;  // (kDppWords lanes per box, all of them here or none)
        const unsigned long long m = m_s[bb][k];
        masks[((size_t)(b0 + bb) * n_tiles + blockIdx.x) * kDppWords + k] = m;
        int c = __popcll(m);
#pragma unroll
        for (int d = kDppWords / 2; d >= 1; d >>= 1) c += __shfl_xor(c, d, 64);
        if (k == 0) {
            counts[(size_t)(b0 + bb) * n_tiles + blockIdx.x] = c;
            if (c) atomicAdd(&totals[(size_t)(b0 + bb) * kDppTotalStep], c);
        }
    }
}

// first output entry of every box (at most max_all: entries from there on are dropped), one workgroup
__global__ __launch_bounds__(kThreads) void dpp_box_base_kernel(const int *__restrict__ totals, int B, int cap,
                                                                int max_all, int *__restrict__ box_base) {
    long carry = 0;
    for (int base = 0; base < B; base += kThreads) {
        const int b = base + threadIdx.x;
        // (a clamped entry leaves the sum of a round, at most 256 of them, inside 64 bits only)
        const int kept = b < B ? min(min(totals[(size_t)b * kDppTotalStep], cap), max_all) : 0;
        int lo_tot, hi_tot;
        const int lo = block_exclusive_scan(kept & 0xffff, &lo_tot), hi = block_exclusive_scan(kept >> 16, &hi_tot);
        if (b < B) box_base[b] = (int)min((long)max_all, carry + lo + ((long)hi << 16));
        carry += lo_tot + ((long)hi_tot << 16);
    }
}

// The set bits of one box in one segment of kDppSegTiles tiles, in point order, as output entries.
// The workgroup of the last box's first segment also writes the number of entries.
__global__ __launch_bounds__(kThreads) void dpp_emit_kernel(
    const float *__restrict__ pts, int P, const DppBox *__restrict__ boxes, int B, int n_tiles,
    const unsigned long long *__restrict__ masks, const int *__restrict__ counts, const int *__restrict__ totals,
    const int *__restrict__ box_base, int cap, int max_all, long long *__restrict__ out_pts_idx,
    long long *__restrict__ out_roi_idx, float *__restrict__ out_feats, int *__restrict__ num_out) {
#pragma clang fp contract(off)
    // the segment's hits: point - first point of the segment; or, where there are more, its words and how many
    // hits lie in front of each
    __shared__ __align__(8) unsigned short hit_s[kDppListed];
    constexpr int kWords = kDppSegTiles * kDppWords;
    static_assert(kWords == kThreads && sizeof(hit_s) >= kWords * (sizeof(unsigned long long) + sizeof(int)), "a word a thread");
    unsigned long long *word_s = reinterpret_cast<unsigned long long *>(hit_s);
    int *first_s = reinterpret_cast<int *>(word_s + kWords);
    const int b = blockIdx.y;
    const int tile0 = blockIdx.x * kDppSegTiles, tile1 = min(n_tiles, tile0 + kDppSegTiles);
    const bool reports = b == B - 1 && blockIdx.x == 0;
    const int *mine = counts + (size_t)b * n_tiles;
    // hits of this box in front of the segment, and in it; entries of the boxes in front, in two halves so
    // that no sum leaves 32 bits.  Asked for and added up together: one after the other, each was a trip
    // to memory or two barriers.
    int sums[4] = {0, 0, 0, 0};
    for (int t = threadIdx.x; t < tile1; t += kThreads) {
        const int c = mine[t];
        if (t < tile0) sums[0] += c; else sums[1] += c;
    }
    if (!box_base) {
        for (int k = threadIdx.x; k < b; k += kThreads) {
            const int kept = min(totals[(size_t)k * kDppTotalStep], cap);
            sums[2] += kept & 0xffff;
            sums[3] += kept >> 16;
        }
    }
    __shared__ int sums_s[kThreads / 64][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) sums[k] += __shfl_xor(sums[k], d, 64);
        if ((threadIdx.x & 63) == 0) sums_s[threadIdx.x >> 6][k] = sums[k];
    }
    __syncthreads();
    int front = 0, here = 0;
    long base = box_base ? box_base[b] : 0;
#pragma unroll
    for (int k = 0; k < kThreads / 64; ++k) {
        front += sums_s[k][0];
        here += sums_s[k][1];
        if (!box_base) base += sums_s[k][2] + ((long)sums_s[k][3] << 16);
    }
    if (!reports && (here == 0 || front >= cap)) return;  // (uniform)
    if (reports && threadIdx.x == 0) num_out[0] = (int)min((long)max_all, base + min(totals[(size_t)b * kDppTotalStep], cap));
    if (here == 0 || front >= cap || base + front >= max_all) return;
    const int word = tile0 * kDppWords + (int)threadIdx.x;
    unsigned long long m = word < tile1 * kDppWords ? masks[(size_t)b * n_tiles * kDppWords + word] : 0ull;
    int total;
    const int at = block_exclusive_scan(__popcll(m), &total);
    const DppBox bx = boxes[b];
    const long kept = min(min((long)total, (long)cap - front), max_all - base - front);
    // point number p as entry number pos
    auto emit = [&](long pos, long p, float x, float y, float z) {
        float lx, ly;
        const int flag = dpp_test(bx, x, y, z, lx, ly);  // the same arithmetic as in the first pass
        const float local_z = (float)((double)z - ((double)bx.cz_bottom + (double)bx.h / 2.0));  // (:103)
        float *f = out_feats + pos * kDppInfo;
        out_pts_idx[pos] = p;
        out_roi_idx[pos] = b;
        f[0] = x;
        f[1] = y;
        f[2] = z;
        f[3] = lx;
        f[4] = ly;
        f[5] = local_z;
        f[6] = lx + bx.l / 2;
        f[7] = ly + bx.w / 2;
        f[8] = local_z + bx.h / 2;
        f[9] = -lx + bx.l / 2;
        f[10] = -ly + bx.w / 2;
        f[11] = -local_z + bx.h / 2;
        f[12] = flag == 1 ? 1.0f : 0.0f;
    };
    if (kept > kDppListed) {
        // (uniform) over half of the segment's points: a lane per point, word by word.  (32 boxes around all of
        // 100k points, the whole call: listed at once, with room for all, 129 us, in two rounds 136, so 123)
        word_s[threadIdx.x] = m;
        first_s[threadIdx.x] = at;
        __syncthreads();
        const int lane = threadIdx.x & 63;
        constexpr int kAhead = 4;  // words a wave asks for the points of at a time
        for (int k0 = (threadIdx.x >> 6) * kAhead; k0 < kWords; k0 += kThreads / 64 * kAhead) {
            float x[kAhead], y[kAhead], z[kAhead];
            int h[kAhead];
#pragma unroll
            for (int r = 0; r < kAhead; ++r) {
                const unsigned long long word = word_s[k0 + r];
                h[r] = (word >> lane & 1ull) != 0ull ? first_s[k0 + r] + __popcll(word & ((1ull << lane) - 1ull)) : 0x7fffffff;
                const long p = (long)tile0 * kDppTile + (h[r] < kept ? (k0 + r) * 64 + lane : 0);
                x[r] = pts[p * 3];
                y[r] = pts[p * 3 + 1];
                z[r] = pts[p * 3 + 2];
            }
#pragma unroll
            for (int r = 0; r < kAhead; ++r)
                if (h[r] < kept) emit(base + front + h[r], (long)tile0 * kDppTile + (k0 + r) * 64 + lane, x[r], y[r], z[r]);
        }
        return;
    }
    for (int place = at; m != 0ull && place < kept; m &= m - 1ull, ++place)
        hit_s[place] = (unsigned short)((int)threadIdx.x * 64 + __builtin_ctzll(m));
    __syncthreads();
    for (int h = threadIdx.x; h < kept; h += kThreads) {
        const long p = (long)tile0 * kDppTile + hit_s[h];
        emit(base + front + h, p, pts[p * 3], pts[p * 3 + 1], pts[p * 3 + 2]);
    }
}

// ------------------------------------------------------------- grid hash --
// Open-addressing table of (key, value) int32 pairs with the reference's probe
// sequence (torchex/src/utils/functions.cuh:30-64, double hashing with an odd
// step over a power-of-two table).  A slot is one 64-bit word (key in the low
// half, value in the high half, as the reference's [size, 2] int32 tensor lays
// them out) claimed with a single 64-bit compare-and-swap, so key and value
// appear together.

// (key % size + i * (2 * key + 1)) % size of the reference, for key >= 0 and a
// power-of-two size: both remainders are bit masks and the 64-bit sum cannot wrap
// (i < size <= 2^30, 2 * key + 1 < 2^32).
__device__ __forceinline__ int grid_hash_slot(int key, int probe_i, int table_size) {
    const unsigned long long mask = (unsigned long long)(table_size - 1);
    const unsigned long long k = (unsigned long long)(unsigned)key;
    return (int)(((k & mask) + (unsigned long long)probe_i * (k * 2ull + 1ull)) & mask);
}

// The probe sequences of a wave's keys are followed together.  While many keys are still looking, each looks at its
// next slot with its own lane; as they become fewer, the wave's lanes are dealt out among them and every key
// looks at more slots of its sequence at a time, in order.  The mean key needs 1.3 - 2.2 slots, but where the grid's
// strides fall badly on the table's size (a frame's 748 x 30 cells a column, 2^18 slots) a few need hundreds.  With a
// lane to a key to the end, the kernels waited for those alone, a trip to memory per slot: 146k keys of a frame built
// in 13 / 218 us and 300k probed in 7 / 100, by the frame, now 13 / 23 and 6 / 9.  (With a lane to a key for 17 slots and the
// wave's lanes for one key after the other from there on, and keys in order spread over all waves, which takes
// a line for each: 16 / 27, and 1M keys in order 50 us against 17 now and with a lane to a key, 3M probes 115 against 86.)
//
// How long a key keeps its own lane, us a call with it / with lanes dealt out at once:
//   placing: while more than 8 keys of the wave look.  A key tries its slot at once, where a group looks first, a trip
//     more: 600k keys 55 / 88, 3M 234 / 361.  In a crowd of long sequences looking ahead is cheaper than trying, the
//     more so the more keys there are: up to kHashFewBuilt keys that lasts kHashCrowd slots (262k keys in 2^18 slots 3010
//     to the end / 1210, so 1230; 30,000 keys 448 apart 88 / 192), above kHashOwnMany (1M keys 448 apart 1240 / 616, so 667).
//   looking: while more than 32 keys look (1M absent keys in a table 0.95 full 290, one by one 272; 300k probes of a frame
//     above).  More than kHashFewProbes keys in as many slots wait for the memory itself, so that what is looked
//     at behind a sequence's end costs time: kHashOwn slots there (3M coordinates 86 / 146, 3M absent keys 194 / 275, 2M
//     in a table 0.95 full 646 / 834; but 1.4M probes of 2^19 slots 43 / 20, of 2^17 47 / 23).
// From kHashLong slots on, the sequences left are long ones, and a lane asks for kHashAhead slots at a time.
constexpr int kHashLong = 32, kHashAhead = 4;
constexpr long kHashFewBuilt = 3L << 17, kHashFewProbes = 1L << 20;
constexpr int kHashCrowd = 64, kHashOwnMany = 8, kHashOwn = 128;

// How a wave's lanes are dealt out among the keys that are still looking: a group of 2^log2 lanes each, the first
// key's first.
struct HashDeal {
    int log2, group, rank;       // the group this lane works in, and the one that works for this lane's key
    unsigned long long members;  // the lanes of a group, shifted to the first one's place
    int from;                    // the lane whose key the group works for
    bool works;                  // the group works for a key
    __device__ __forceinline__ HashDeal(unsigned long long looking) {
        const int lane = threadIdx.x & 63, keys = __popcll(looking);
        const unsigned long long below = (1ull << lane) - 1ull;
        log2 = 6 - (keys > 1 ? 32 - __builtin_clz((unsigned)(keys - 1)) : 0);
        group = lane >> log2;
        const bool looks = (looking >> lane & 1ull) != 0ull;
        rank = looks ? __popcll(looking & below) : 0;
        members = log2 == 6 ? ~0ull : (1ull << (1 << log2)) - 1ull;
        works = group < keys;
        // every lane's number, those that are looking first
        const int place = looks ? rank : keys + __popcll(~looking & below);
        from = __shfl(__builtin_amdgcn_ds_permute(place << 2, lane), group, 64);
    }
    // of a ballot, what the group that works in this lane / for this lane's key has left there
    __device__ __forceinline__ unsigned long long here(unsigned long long ballot) const { return (ballot >> (group << log2)) & members; }
    __device__ __forceinline__ unsigned long long mine(unsigned long long ballot) const { return (ballot >> (rank << log2)) & members; }
};

// A slot as it is now or was a moment ago.  A slot only ever goes from empty to taken, so that one seen taken
// is, and one seen empty may be (the compare-and-swap decides).
__device__ __forceinline__ unsigned long long grid_hash_peek(const unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Slots number t0 + k of a group's key, for k < AHEAD << deal.log2: the first empty one is taken, or the next one
// if that was taken in between, by all groups at a time.  pending: this lane's key has no slot yet.
template <int AHEAD>
__device__ __forceinline__ void hash_place(const HashDeal &deal, int t0, int key, unsigned long long word,
                                           unsigned long long *__restrict__ table, int table_size, bool &pending) {
    constexpr unsigned long long kEmpty = ~0ull;  // (-1, -1)
    const int lane = threadIdx.x & 63, step = 1 << deal.log2, part = lane & (step - 1);
    const int k = __shfl(key, deal.from, 64);
    const unsigned long long w = ((unsigned long long)(unsigned)__shfl((int)(word >> 32), deal.from, 64) << 32) | (unsigned)k;
    unsigned empty = 0u;  // of this lane's slots, a bit each
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
        const int t = t0 + a * step + part;
        const unsigned long long seen = grid_hash_peek(table + grid_hash_slot(k, min(t, table_size - 1), table_size));
        if (deal.works && t < table_size && seen == kEmpty) empty |= 1u << a;
    }
    unsigned long long placed = 0ull;  // lanes that have placed their group's key
    while (__ballot(empty != 0u) != 0ull) {  // (every turn takes a bit from every group that has one)
        // the group's first empty slot
        int first = -1;
        bool tries = false;
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) {
            const unsigned long long here = deal.here(__ballot((empty >> a & 1u) != 0u));
            if (first < 0 && here != 0ull) {
                first = a;
                tries = part == __builtin_ctzll(here);
            }
        }
        bool done = false;
        if (tries) {
            done = atomicCAS(table + grid_hash_slot(k, t0 + first * step + part, table_size), kEmpty, w) == kEmpty;
            empty &= ~(1u << first);
        }
        placed |= __ballot(done);
        if (deal.here(placed) != 0ull) empty = 0u;
    }
    if (pending && deal.mine(placed) != 0ull) pending = false;
}

// values == NULL: key number i gets the value i.  few: at most kHashFewBuilt keys
__global__ __launch_bounds__(kThreads) void grid_hash_build_kernel(const int *__restrict__ keys,
                                                                   const int *__restrict__ values,
                                                                   unsigned long long *__restrict__ table,
                                                                   int table_size, long n, bool few, int *__restrict__ fail) {
    const int lane = threadIdx.x & 63;
    const long wave = (long)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6), waves = (long)gridDim.x * (kThreads / 64);
    // keys next to each other (those with long sequences are, where the keys are in order, and slots too) stay so
    // by four only, where they are few: a wave with many long sequences is what the call waits for
    const int near = few ? 2 : 6;
    const long i = (((lane >> near) * waves + wave) << near) + (lane & ((1 << near) - 1));
    const int key = i < n ? keys[i] : -1;
    const unsigned value = i < n ? (unsigned)(values ? values[i] : (int)i) : 0u;
    const unsigned long long word = ((unsigned long long)value << 32) | (unsigned long long)(unsigned)key;
    bool pending = i < n && key >= 0;
    const bool refused = i < n && key < 0;
    int t = 0;  // (uniform in a wave, as is all that is decided by the ballots)
    for (unsigned long long looking = __ballot(pending); looking != 0ull && t < table_size; looking = __ballot(pending)) {
        if (t < (few ? kHashCrowd : kHashOwnMany) && __popcll(looking) > 8) {
            if (pending) pending = atomicCAS(table + grid_hash_slot(key, t, table_size), ~0ull, word) != ~0ull;
            ++t;
            continue;
        }
        const HashDeal deal(looking);
        if (t < kHashLong && deal.log2 >= 2) {
            hash_place<1>(deal, t, key, word, table, table_size, pending);
            t += 1 << deal.log2;
        } else {
            hash_place<kHashAhead>(deal, t, key, word, table, table_size, pending);
            t += kHashAhead << deal.log2;
        }
    }
    if ((pending || refused) && fail) fail[0] = 1;  // table full or key negative (the reference asserts)
}

// Slots number t0 + k of a group's key, for k < AHEAD << deal.log2, up to the key or an empty slot.  An empty
// slot on the probe sequence proves the key was never inserted (no deletions).  The reference keeps scanning
// all table_size slots before giving up (functions.cuh:54-63), with the same answer.
template <int AHEAD>
__device__ __forceinline__ void hash_look(const HashDeal &deal, int t0, int key, const unsigned long long *__restrict__ table,
                                          int table_size, bool &pending, int &found) {
    const int lane = threadIdx.x & 63, step = 1 << deal.log2;
    const int k = __shfl(key, deal.from, 64);
    unsigned long long word[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a)
        word[a] = table[grid_hash_slot(k, min(t0 + a * step + (lane & (step - 1)), table_size - 1), table_size)];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
        const int slot_key = (int)(unsigned)(word[a] & 0xffffffffull);
        const bool ends = deal.works && t0 + a * step + (lane & (step - 1)) < table_size && (slot_key == k || slot_key == -1);
        const unsigned long long mine = deal.mine(__ballot(ends));
        const int at = pending && mine != 0ull ? (deal.rank << deal.log2) + __builtin_ctzll(mine) : lane;
        const int at_key = __shfl(slot_key, at, 64), at_value = __shfl((int)(unsigned)(word[a] >> 32), at, 64);
        if (pending && mine != 0ull) {
            if (at_key == key) found = at_value;
            pending = false;
        }
    }
}

// Value of the lane's key (-1: absent); a wave at a time, `in`: the lane has a key, and its own lane for `own` slots.
__device__ __forceinline__ int grid_hash_find(int key, bool in, const unsigned long long *__restrict__ table, int table_size,
                                              int own) {
    int found = -1;
    bool pending = in && key >= 0;
    int t = 0;  // (uniform, as above)
    for (unsigned long long looking = __ballot(pending); looking != 0ull && t < table_size; looking = __ballot(pending)) {
        if (t < own || __popcll(looking) > 32) {
            if (pending) {
                const unsigned long long word = table[grid_hash_slot(key, t, table_size)];
                const int slot_key = (int)(unsigned)(word & 0xffffffffull);
                if (slot_key == key) found = (int)(unsigned)(word >> 32);
                pending = slot_key != key && slot_key != -1;
            }
            ++t;
            continue;
        }
        const HashDeal deal(looking);
        if (t < kHashLong) {
            hash_look<1>(deal, t, key, table, table_size, pending, found);
            t += 1 << deal.log2;
        } else {
            hash_look<kHashAhead>(deal, t, key, table, table_size, pending, found);
            t += kHashAhead << deal.log2;
        }
    }
    return found;
}

inline int hash_own(long n, long table_size) { return n > kHashFewProbes && table_size > kHashFewProbes ? kHashOwn : 1; }

template <class Keys>
__global__ void grid_hash_probe_kernel(Keys keys, const unsigned long long *__restrict__ table, int table_size,
                                       long n, int own, int *__restrict__ out) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int value = grid_hash_find(i < n ? (int)keys(i) : -1, i < n, table, table_size, own);
    if (i < n) out[i] = value;
}

// ---- a hash of the distinct voxel coordinates -------------------------------------
// From the occupancy map of the coordinates' grid (as above: distinct keys in ascending order
// without a sort), so that the coordinates are read twice, once for the grid's extents and once
// to mark the map, and never stored as keys.  300k rows of a sweep, 146k of them
// distinct in 16.7M cells, built and probed with another 300k: 307 us of kernels in 44 launches
// (the sort's plan, the linearised keys and the valid slots by library calls) -> 70 us in 12.

// Largest coordinate per axis, one partial [3] per workgroup (the host folds the few of them).
constexpr int kCoorMaxParts = 128;
template <typename K>
__global__ __launch_bounds__(kThreads) void coor_max_kernel(const K *__restrict__ coors, long n,
                                                            long long *__restrict__ parts) {
    __shared__ long long s_max[kThreads / 64][3];
    long long m[3] = {(long long)coors[0], (long long)coors[1], (long long)coors[2]};
    for (long i = (long)blockIdx.x * kThreads + threadIdx.x; i < n; i += (long)kCoorMaxParts * kThreads) {
#pragma unroll
        for (int a = 0; a < 3; ++a) m[a] = max(m[a], (long long)coors[3 * i + a]);
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) m[a] = max(m[a], (long long)__shfl_xor(m[a], d, 64));
        if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6][a] = m[a];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        long long x = s_max[0][threadIdx.x];
        for (int k = 1; k < kThreads / 64; ++k) x = max(x, s_max[k][threadIdx.x]);
        parts[blockIdx.x * 3 + threadIdx.x] = x;
    }
}

// the distinct keys in ascending order (a workgroup per part of the cells), and the table's slots emptied
__global__ __launch_bounds__(kThreads) void grid_hash_prepare_kernel(KeyMap m, unsigned long long *__restrict__ table,
                                                                     long table_size) {
    __shared__ int base_s[txs_detail::kMapTilesSummed];
    map_tile_bases<kThreads>(m, base_s);
    for (long i = (long)blockIdx.x * kThreads + threadIdx.x; i < table_size; i += (long)gridDim.x * kThreads)
        table[i] = ~0ull;
    map_list_part<kThreads>(m, base_s, (long)blockIdx.x);
}

// Occupied slots: a byte per slot, and the occupied ones' (key, value) words in slot order.  Two
// launches: occupied slots per tile, then their words behind those of the tiles in front.
constexpr int kValidItems = 8;
constexpr int kValidTile = kThreads * kValidItems;
constexpr int kValidSumTiles = 1024;  // up to this many tiles the second launch adds up the tiles in front itself
__global__ __launch_bounds__(kThreads) void grid_hash_valid_kernel(const unsigned long long *__restrict__ table,
                                                                   long table_size, unsigned char *__restrict__ valid,
                                                                   int *__restrict__ tile_sums) {
    const long base = (long)blockIdx.x * kValidTile;
    int c = 0;
#pragma unroll
    for (int k = 0; k < kValidItems; ++k) {
        const long i = base + (long)k * kThreads + threadIdx.x;
        if (i >= table_size) continue;
        const bool used = (int)(unsigned)(table[i] & 0xffffffffull) != -1;
        valid[i] = used ? 1 : 0;
        c += used;
    }
    int total;
    block_exclusive_scan(c, &total);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}
__global__ __launch_bounds__(kThreads) void grid_hash_compact_kernel(const unsigned long long *__restrict__ table,
                                                                     long table_size, const int *__restrict__ tile_offs,
                                                                     int offsets_ready,
                                                                     unsigned long long *__restrict__ out, long n_out) {
    const long base = (long)blockIdx.x * kValidTile + (long)threadIdx.x * kValidItems;
    unsigned long long word[kValidItems];
    int c = 0;
#pragma unroll
    for (int k = 0; k < kValidItems; ++k) {
        word[k] = base + k < table_size ? table[base + k] : ~0ull;
        c += (int)(unsigned)(word[k] & 0xffffffffull) != -1;
    }
    int off;
    if (offsets_ready) {
        off = tile_offs[blockIdx.x];
    } else {
        int part = 0;
        for (int t = threadIdx.x; t < (int)blockIdx.x; t += kThreads) part += tile_offs[t];
        block_exclusive_scan(part, &off);
    }
    int total;
    long at = (long)off + block_exclusive_scan(c, &total);
#pragma unroll
    for (int k = 0; k < kValidItems; ++k)
        if ((int)(unsigned)(word[k] & 0xffffffffull) != -1) {
            if (at < n_out) out[at] = word[k];
            ++at;
        }
}

// byte map -> cells of one set of keys.  Layout of the workspace: byte map (8 ints per cell), cells (2),
// the number of distinct keys, a flag for a key outside the bound (used where the caller has no other),
// keys per tile and their scan.
struct BitmapWs {
    long words;
    uint4 *map16;
    uint2 *cells;
    int *total, *bad, *tiles;
};
BitmapWs bitmap_ws_of(const int32_t *ws_in, int64_t key_bound) {
    int32_t *ws = const_cast<int32_t *>(ws_in);
    BitmapWs r;
    r.words = (long)((key_bound + 31) / 32);
    r.map16 = reinterpret_cast<uint4 *>(ws);
    r.cells = reinterpret_cast<uint2 *>(ws + 8 * r.words);
    r.total = ws + 10 * r.words;
    r.bad = r.total + 1;
    r.tiles = r.bad + 1;
    return r;
}
// how the kernels above read a finished map
KeyMap key_map(const BitmapWs &b, const void *keys, int keys64, int64_t key_bound, const int *bad, int *unq_keys, int64_t most) {
    KeyMap m = {};
    m.keys = keys;
    m.keys64 = keys64;
    m.key_bound = (long)key_bound;
    m.cells = b.cells;
    m.tiles = b.tiles;
    m.n_tiles = (int)scan_tiles(b.words);
    m.scanned = m.n_tiles > txs_detail::kMapTilesSummed;
    m.words = b.words;
    m.bad = bad;
    m.unq_keys = unq_keys;
    m.most = (long)most;
    m.num_unq = b.total;
    return m;
}
int64_t most_keys(int64_t n, int64_t key_bound) { return n < key_bound ? n : key_bound; }
// the map, cleared; marked by `mark()`; packed
template <class Mark>
int bitmap_make(const BitmapWs &b, int *clear_flag, hipStream_t st, Mark mark) {
    bytemap_clear_kernel<<<dim3(blocks_for(2 * b.words)), dim3(kThreads), 0, st>>>(b.map16, 2 * b.words, clear_flag);
    mark();
    const long tiles = scan_tiles(b.words);
    bytemap_pack_kernel<<<dim3((unsigned)tiles), dim3(kPackThreads), 0, st>>>(b.map16, b.words, b.cells, b.tiles);
    if (tiles > txs_detail::kMapTilesSummed &&
        exclusive_scan(b.tiles, tiles, b.tiles, tiles + 1, b.tiles + tiles + 1, st) != hipSuccess)
        return TXS_ERR_LAUNCH;
    return status_of(hipGetLastError());
}
template <class Keys>
int bitmap_count(Keys keys, long n, int64_t key_bound, const BitmapWs &b, int *clear_flag, int *bad, hipStream_t st) {
    return bitmap_make(b, clear_flag, st, [&]() {
        bytemap_mark_kernel<Keys><<<dim3(blocks_for(n)), dim3(kThreads), 0, st>>>(
            keys, n, (long)key_bound, reinterpret_cast<unsigned char *>(b.map16), bad);
    });
}

}  // namespace

int txs_detail::unique_map_keys(const void *keys, int key_is_int64, int64_t num_total, int64_t key_bound,
                                int32_t *key_flag, int32_t *bitmap_ws, void *stream) {
    if (!fits_i32(num_total) || num_total == 0 || key_bound <= 0 || key_bound > (1LL << 31)) return TXS_ERR_INVALID_ARG;
    if (!keys || !bitmap_ws || ((uintptr_t)bitmap_ws & 15u) != 0) return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    const BitmapWs b = bitmap_ws_of(bitmap_ws, key_bound);
    int *bad = key_flag ? key_flag : b.bad, *clear_flag = key_flag ? nullptr : b.bad;
    return key_is_int64 ? bitmap_count(FlatKeys<long long>{static_cast<const long long *>(keys)}, num_total, key_bound, b,
                                       clear_flag, bad, st)
                        : bitmap_count(FlatKeys<int>{static_cast<const int *>(keys)}, num_total, key_bound, b, clear_flag,
                                       bad, st);
}

int txs_detail::unique_map_points(const float *points, int64_t num_total, int64_t point_stride, const float *range_lo,
                                  const float *voxel_size, const int32_t *dims, int32_t *coors, int32_t *keys,
                                  int32_t *bitmap_ws, void *stream) {
    if (!fits_i32(num_total) || num_total == 0 || point_stride < 3 || !points || !range_lo || !voxel_size || !dims ||
        !coors || !keys || !bitmap_ws || ((uintptr_t)bitmap_ws & 15u) != 0)
        return TXS_ERR_INVALID_ARG;
    int64_t key_bound = 1;
    for (int a = 0; a < 3; ++a) {
        if (dims[a] <= 0 || dims[a] > 2147483647LL / key_bound) return TXS_ERR_INVALID_ARG;
        key_bound *= dims[a];
    }
    hipStream_t st = (hipStream_t)stream;
    const BitmapWs b = bitmap_ws_of(bitmap_ws, key_bound);
    return bitmap_make(b, b.bad, st, [&]() {
        voxel_keys_kernel<<<dim3(blocks_for(num_total)), dim3(kThreads), 0, st>>>(
            points, num_total, (int)point_stride, range_lo[0], range_lo[1], range_lo[2], voxel_size[0], voxel_size[1],
            voxel_size[2], dims[0], dims[1], dims[2], coors, keys, b.bad, reinterpret_cast<unsigned char *>(b.map16));
    });
}

int txs_detail::unique_plan_of_map(const void *keys, int key_is_int64, int64_t num_total, int64_t key_bound,
                                   const int32_t *key_flag, int32_t *bitmap_ws, int32_t heavy_threshold,
                                   int32_t *plan_ws, int32_t *unq_inv, int32_t *unq_keys, int64_t *unq_cnts,
                                   int32_t *perm, int32_t *seg, int32_t *preSum, int32_t *slot_of, int32_t *heavy_ids,
                                   int32_t *stats, void *stream) {
    if (!unq_inv || !unq_keys || !unq_cnts || !slot_of || !heavy_ids || !stats) return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    const BitmapWs b = bitmap_ws_of(bitmap_ws, key_bound);
    const int64_t most = most_keys(num_total, key_bound);
    KeyMap m = key_map(b, keys, key_is_int64, key_bound, key_flag ? key_flag : b.bad, unq_keys, most);
    m.found = stats + TXS_STATS_LEN;
    if (txs_detail::plan_takes_map(num_total, most))
        return txs_detail::plan_build_mapped(m, unq_inv, num_total, most, heavy_threshold, plan_ws, perm, seg, preSum,
                                             slot_of, heavy_ids, stats, (long long *)unq_cnts, stream);
    map_assign_kernel<<<assign_grid(num_total, m), dim3(kThreads), 0, st>>>(m, num_total, unq_inv);
    return txs_detail::plan_build(unq_inv, num_total, most, heavy_threshold, nullptr, plan_ws, perm, seg, preSum,
                                  slot_of, heavy_ids, stats, nullptr, m.num_unq, (long long *)unq_cnts, nullptr, stream);
}

extern "C" {

int txs_voxel_keys(const float *points, int64_t num_total, int64_t point_stride,
                   const float *range_lo, const float *voxel_size, const int32_t *dims,
                   int32_t *coors, int32_t *keys, int32_t *stats, void *stream) {
    if (!fits_i32(num_total) || point_stride < 3 || !range_lo || !voxel_size || !dims || !stats)
        return TXS_ERR_INVALID_ARG;
    const long long cells = (long long)dims[0] * dims[1] * dims[2];
    if (dims[0] <= 0 || dims[1] <= 0 || dims[2] <= 0 || !fits_i32(cells)) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!points || !keys) return TXS_ERR_INVALID_ARG;
    voxel_keys_kernel<<<dim3(blocks_for(num_total)), dim3(kThreads), 0, (hipStream_t)stream>>>(
        points, num_total, (int)point_stride, range_lo[0], range_lo[1], range_lo[2], voxel_size[0],
        voxel_size[1], voxel_size[2], dims[0], dims[1], dims[2], coors, keys, stats + TXS_STAT_OUT_OF_RANGE, nullptr);
    return status_of(hipGetLastError());
}

int64_t txs_unique_bitmap_workspace_len(int64_t key_bound) {
    if (key_bound <= 0 || key_bound > (1LL << 31)) return -1;
    const int64_t words = (key_bound + 31) / 32;
    // byte map (32 bytes per cell), cells, their number, range flag, keys per tile, scan workspace
    const int64_t tiles = scan_tiles(words);
    return 8 * words + 2 * words + 2 + tiles + 1 + scan_tiles(tiles + 1);
}

int txs_unique_bitmap_count(const void *keys, int key_is_int64, int64_t num_total, int64_t key_bound,
                            int32_t *bitmap_ws, int32_t *stats, void *stream) {
    if (!fits_i32(num_total) || key_bound <= 0 || key_bound > (1LL << 31) || !stats) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!keys || !bitmap_ws || ((uintptr_t)bitmap_ws & 15u) != 0) return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    const BitmapWs b = bitmap_ws_of(bitmap_ws, key_bound);
    int *bad = stats + TXS_STAT_OUT_OF_RANGE;
    const int rc = key_is_int64
                       ? bitmap_count(FlatKeys<long long>{static_cast<const long long *>(keys)}, num_total, key_bound, b,
                                      nullptr, bad, st)
                       : bitmap_count(FlatKeys<int>{static_cast<const int *>(keys)}, num_total, key_bound, b, nullptr,
                                      bad, st);
    if (rc != TXS_OK) return rc;
    KeyMap m = key_map(b, keys, key_is_int64, key_bound, nullptr, nullptr, 0);
    m.num_unq = stats + TXS_STAT_NUM_UNQ;
    map_total_kernel<<<dim3(1), dim3(kThreads), 0, st>>>(m);
    return status_of(hipGetLastError());
}

int txs_coor_max_parts(void) { return kCoorMaxParts; }

int txs_coor_max(const void *coors, int coor_is_int64, int64_t num_total, int64_t *parts, void *stream) {
    if (!fits_i32(num_total) || num_total == 0 || !coors || !parts) return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    if (coor_is_int64)
        coor_max_kernel<long long><<<dim3(kCoorMaxParts), dim3(kThreads), 0, st>>>(
            static_cast<const long long *>(coors), num_total, (long long *)parts);
    else
        coor_max_kernel<int><<<dim3(kCoorMaxParts), dim3(kThreads), 0, st>>>(static_cast<const int *>(coors), num_total,
                                                                            (long long *)parts);
    return status_of(hipGetLastError());
}

int64_t txs_coor_bitmap_count_offset(int64_t key_bound) {
    return key_bound <= 0 || key_bound > (1LL << 31) ? -1 : 10 * ((key_bound + 31) / 32);
}

int txs_coor_bitmap_count(const void *coors, int coor_is_int64, int64_t num_total, const int64_t *dims,
                          int32_t *bitmap_ws, void *stream) {
    if (!fits_i32(num_total) || num_total == 0 || !coors || !dims || !bitmap_ws || ((uintptr_t)bitmap_ws & 15u) != 0)
        return TXS_ERR_INVALID_ARG;
    int64_t key_bound = 1;
    for (int a = 0; a < 3; ++a) {
        if (dims[a] <= 0 || dims[a] > (1LL << 31) / key_bound) return TXS_ERR_INVALID_ARG;
        key_bound *= dims[a];
    }
    hipStream_t st = (hipStream_t)stream;
    const BitmapWs b = bitmap_ws_of(bitmap_ws, key_bound);
    const long s0 = (long)(dims[1] * dims[2]), s1 = (long)dims[2];
    const int rc = coor_is_int64 ? bitmap_count(CoorKeys<long long>{static_cast<const long long *>(coors), s0, s1},
                                                num_total, key_bound, b, b.bad, b.bad, st)
                                 : bitmap_count(CoorKeys<int>{static_cast<const int *>(coors), s0, s1}, num_total,
                                                key_bound, b, b.bad, b.bad, st);
    if (rc != TXS_OK) return rc;
    map_total_kernel<<<dim3(1), dim3(kThreads), 0, st>>>(key_map(b, nullptr, 0, key_bound, nullptr, nullptr, 0));
    return status_of(hipGetLastError());
}

int64_t txs_grid_hash_index_workspace_len(int64_t num_unq, int64_t table_size) {
    if (!fits_i32(num_unq) || !fits_i32(table_size)) return -1;
    const int64_t tiles = (table_size + kValidTile - 1) / kValidTile;
    return num_unq + tiles + scan_tiles(tiles) + 17;
}

int txs_grid_hash_index(const int32_t *bitmap_ws, int64_t key_bound, int64_t num_unq, int32_t *table,
                        int64_t table_size, int32_t *index_ws, unsigned char *valid, int32_t *valid_table,
                        void *stream) {
    if (key_bound <= 0 || key_bound > (1LL << 31) || !fits_i32(num_unq) || num_unq == 0 || !fits_i32(table_size) ||
        num_unq > table_size || (table_size & (table_size - 1)) != 0)
        return TXS_ERR_INVALID_ARG;
    if (!bitmap_ws || !table || !index_ws || !valid || !valid_table || (((uintptr_t)table | (uintptr_t)valid_table) & 7) != 0)
        return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    const BitmapWs b = bitmap_ws_of(bitmap_ws, key_bound);
    auto slots = reinterpret_cast<unsigned long long *>(table);
    int *unq_keys = index_ws, *tile_sums = index_ws + num_unq;
    const KeyMap m = key_map(b, nullptr, 0, key_bound, nullptr, unq_keys, num_unq);
    grid_hash_prepare_kernel<<<dim3((unsigned)map_parts(m)), dim3(kThreads), 0, st>>>(m, slots, table_size);
    grid_hash_build_kernel<<<dim3(blocks_for(num_unq)), dim3(kThreads), 0, st>>>(unq_keys, nullptr, slots,
                                                                                (int)table_size, num_unq, num_unq <= kHashFewBuilt, nullptr);
    const long tiles = (table_size + kValidTile - 1) / kValidTile;
    grid_hash_valid_kernel<<<dim3((unsigned)tiles), dim3(kThreads), 0, st>>>(slots, table_size, valid, tile_sums);
    const bool few = tiles <= kValidSumTiles;
    if (!few && exclusive_scan(tile_sums, tiles, tile_sums, tiles, tile_sums + tiles, st) != hipSuccess)
        return TXS_ERR_LAUNCH;
    grid_hash_compact_kernel<<<dim3((unsigned)tiles), dim3(kThreads), 0, st>>>(
        slots, table_size, tile_sums, !few, reinterpret_cast<unsigned long long *>(valid_table), num_unq);
    return status_of(hipGetLastError());
}

int txs_unique_bitmap_assign(const void *keys, int key_is_int64, int64_t num_total, int64_t key_bound,
                             const int32_t *bitmap_ws, int32_t *unq_inv, int32_t *unq_keys, void *stream) {
    if (!fits_i32(num_total) || key_bound <= 0 || key_bound > (1LL << 31)) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!keys || !bitmap_ws || !unq_inv || !unq_keys) return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    const BitmapWs b = bitmap_ws_of(bitmap_ws, key_bound);
    KeyMap m = key_map(b, keys, key_is_int64, key_bound, nullptr, unq_keys, most_keys(num_total, key_bound));
    m.num_unq = nullptr;  // (txs_unique_bitmap_count has left it where the caller asked for it)
    map_assign_kernel<<<assign_grid(num_total, m), dim3(kThreads), 0, st>>>(m, num_total, unq_inv);
    return status_of(hipGetLastError());
}

int txs_unique_plan(const void *keys, int key_is_int64, int64_t num_total, int64_t key_bound, int32_t *key_flag,
                    int32_t *bitmap_ws, int32_t heavy_threshold, int32_t *plan_ws, int32_t *unq_inv,
                    int32_t *unq_keys, int64_t *unq_cnts, int32_t *perm, int32_t *seg, int32_t *preSum,
                    int32_t *slot_of, int32_t *heavy_ids, int32_t *stats, void *stream) {
    if (!unq_inv || !unq_keys || !unq_cnts || !slot_of || !heavy_ids || !stats) return TXS_ERR_INVALID_ARG;
    const int rc = txs_detail::unique_map_keys(keys, key_is_int64, num_total, key_bound, key_flag, bitmap_ws, stream);
    if (rc != TXS_OK) return rc;
    return txs_detail::unique_plan_of_map(keys, key_is_int64, num_total, key_bound, key_flag, bitmap_ws, heavy_threshold,
                                          plan_ws, unq_inv, unq_keys, unq_cnts, perm, seg, preSum, slot_of, heavy_ids,
                                          stats, stream);
}

int txs_counts_from_presum(const int32_t *preSum, int64_t num_unq, int64_t *unq_cnts, void *stream) {
    if (!fits_i32(num_unq)) return TXS_ERR_INVALID_ARG;
    if (num_unq == 0) return TXS_OK;
    if (!preSum || !unq_cnts) return TXS_ERR_INVALID_ARG;
    counts_from_presum_kernel<<<dim3(blocks_for(num_unq)), dim3(kThreads), 0, (hipStream_t)stream>>>(
        preSum, (long)num_unq, (long long *)unq_cnts);
    return status_of(hipGetLastError());
}

int64_t txs_unique_workspace_len(int64_t num_total) { return num_total + scan_tiles(num_total + 1) + 17; }

int txs_unique_runs(const int32_t *sorted_keys, const int32_t *perm, int64_t num_total,
                    int32_t *unique_ws, int32_t *seg, int32_t *unq_inv, int32_t *unq_keys,
                    int32_t *preSum, int32_t *stats, void *stream) {
    if (!fits_i32(num_total) || !stats || !preSum) return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    if (num_total == 0) {
        fill_i32_kernel<<<dim3(1), dim3(64), 0, st>>>(preSum, 1, 0);
        return status_of(hipGetLastError());
    }
    if (!sorted_keys || !perm || !unique_ws || !seg || !unq_inv || !unq_keys) return TXS_ERR_INVALID_ARG;
    const long n = num_total;
    int *flags = unique_ws;
    int *scan_ws = unique_ws + n;
    run_flags_kernel<<<dim3(blocks_for(n)), dim3(kThreads), 0, st>>>(sorted_keys, n, flags);
    if (exclusive_scan(flags, n, flags, n, scan_ws, st) != hipSuccess) return TXS_ERR_LAUNCH;
    unique_finish_kernel<<<dim3(blocks_for(n)), dim3(kThreads), 0, st>>>(sorted_keys, perm, flags, n, seg,
                                                                       unq_inv, unq_keys, preSum, stats);
    return status_of(hipGetLastError());
}

static int group_ranks(const long long *ids64, const int32_t *group_ids, int64_t num_total, int64_t num_groups,
                       int32_t *plan_ws, int32_t *perm, int32_t *seg, int32_t *preSum, int64_t *out, int32_t *stats,
                       void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_groups) || !stats) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!group_ids || !plan_ws || !perm || !seg || !preSum || !out || num_groups <= 0) return TXS_ERR_INVALID_ARG;
    const int32_t heavy = txs_default_heavy_threshold();
    // the bucket kernels rank while they place; any other route leaves a plan to rank from
    const bool fused = txs_detail::plan_writes_ranks(num_total, num_groups);
    const int rc = txs_detail::plan_build(group_ids, num_total, num_groups, heavy, nullptr, plan_ws, perm, seg, preSum,
                                          nullptr, nullptr, stats, fused ? (long long *)out : nullptr, nullptr, nullptr,
                                          ids64, stream);
    if (rc != TXS_OK || fused) return rc;
    ingroup_inds_auto_kernel<<<dim3(blocks_for(num_total)), dim3(kThreads), 0, (hipStream_t)stream>>>(
        seg, perm, preSum, stats, num_total, (int)num_groups, (long long *)out);
    return status_of(hipGetLastError());
}

int txs_group_ranks(const int32_t *group_ids, int64_t num_total, int64_t num_groups, int32_t *plan_ws,
                    int32_t *perm, int32_t *seg, int32_t *preSum, int64_t *out, int32_t *stats, void *stream) {
    return group_ranks(nullptr, group_ids, num_total, num_groups, plan_ws, perm, seg, preSum, out, stats, stream);
}

int txs_group_ranks_i64(const int64_t *ids, int32_t *group_ids, int64_t num_total, int64_t num_groups,
                        int32_t *plan_ws, int32_t *perm, int32_t *seg, int32_t *preSum, int64_t *out, int32_t *stats,
                        void *stream) {
    if (num_total > 0 && !ids) return TXS_ERR_INVALID_ARG;
    return group_ranks((const long long *)ids, group_ids, num_total, num_groups, plan_ws, perm, seg, preSum, out, stats,
                       stream);
}

int txs_ingroup_inds(const int32_t *seg, const int32_t *perm, const int32_t *preSum,
                     int64_t num_total, int64_t num_unq, int64_t *out, void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_unq)) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!seg || !preSum || !out || num_unq <= 0) return TXS_ERR_INVALID_ARG;
    ingroup_inds_kernel<<<dim3(blocks_for(num_total)), dim3(kThreads), 0, (hipStream_t)stream>>>(
        seg, perm, preSum, num_total, (int)num_unq, (long long *)out);
    return status_of(hipGetLastError());
}

int64_t txs_dpp_workspace_len(int64_t num_pts, int64_t num_boxes) {
    const int64_t tiles = (num_pts + kDppTile - 1) / kDppTile;
    // box constants, hits and first entry per box, hits per (box, tile), the bit matrix (8-byte
    // words); never less than two bits per (point, box), what callers who keep a buffer gave it
    const int64_t head = (int64_t)(sizeof(DppBox) / sizeof(int)) * num_boxes +
                         (kDppTotalStep + 1) * num_boxes + num_boxes * tiles + 2;
    const int64_t bits = 2 * num_boxes * tiles * kDppWords, kept = (num_boxes + 7) / 8 * num_pts / 2 + 1;
    return head + (bits > kept ? bits : kept);
}

int txs_dynamic_point_pool(const float *rois, const float *pts, int64_t num_boxes, int64_t num_pts,
                           const float *extra_wlh, int32_t max_pts_per_box, int64_t max_all_pts,
                           int32_t *workspace, int64_t *out_pts_idx, int64_t *out_roi_idx,
                           float *out_pts_feats, int32_t *num_out, void *stream) {
    return txs_dynamic_point_pool_mixed(rois, nullptr, pts, nullptr, num_boxes, num_pts, extra_wlh,
                                        max_pts_per_box, max_all_pts, workspace, out_pts_idx, out_roi_idx,
                                        out_pts_feats, num_out, stream);
}

int txs_dynamic_point_pool_mixed(const float *rois, const int32_t *rois_batch, const float *pts,
                                 const int32_t *pts_batch, int64_t num_boxes, int64_t num_pts,
                                 const float *extra_wlh, int32_t max_pts_per_box, int64_t max_all_pts,
                                 int32_t *workspace, int64_t *out_pts_idx, int64_t *out_roi_idx,
                                 float *out_pts_feats, int32_t *num_out, void *stream) {
    if (!fits_i32(num_boxes) || !fits_i32(num_pts) || !fits_i32(max_all_pts) || max_pts_per_box < 0 ||
        !extra_wlh || !num_out)
        return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    if (num_boxes == 0 || num_pts == 0) {
        fill_i32_kernel<<<dim3(1), dim3(64), 0, st>>>(num_out, 1, 0);
        return status_of(hipGetLastError());
    }
    if (!rois || !pts || !workspace || !out_pts_idx || !out_roi_idx || !out_pts_feats ||
        ((rois_batch == nullptr) != (pts_batch == nullptr)))
        return TXS_ERR_INVALID_ARG;
    const int B = (int)num_boxes, P = (int)num_pts;
    if (!fits_i32((long)B * ((P + kThreads - 1) / kThreads) + 1) || B > 65535) return TXS_ERR_INVALID_ARG;
    const int n_tiles = (P + kDppTile - 1) / kDppTile;
    DppBox *boxes = reinterpret_cast<DppBox *>(workspace);
    int *totals = workspace + (sizeof(DppBox) / sizeof(int)) * (size_t)B;
    int *box_base = totals + (size_t)kDppTotalStep * B;
    int *counts = box_base + B;
    unsigned long long *masks =
        reinterpret_cast<unsigned long long *>(((uintptr_t)(counts + (size_t)B * n_tiles) + 7u) & ~(uintptr_t)7u);
    dpp_box_kernel<<<dim3(blocks_for(B)), dim3(kThreads), 0, st>>>(rois, B, extra_wlh[0], extra_wlh[1],
                                                                 extra_wlh[2], boxes, totals);
    dpp_mask_kernel<<<dim3(n_tiles, (B + kDppGroup - 1) / kDppGroup), dim3(kThreads), 0, st>>>(
        pts, P, boxes, B, n_tiles, masks, counts, totals, pts_batch, rois_batch);
    const bool summed = B > kDppSumBoxes;
    if (summed)
        dpp_box_base_kernel<<<dim3(1), dim3(kThreads), 0, st>>>(totals, B, max_pts_per_box, (int)max_all_pts, box_base);
    const int segments = (n_tiles + kDppSegTiles - 1) / kDppSegTiles;
    dpp_emit_kernel<<<dim3(segments, B), dim3(kThreads), 0, st>>>(
        pts, P, boxes, B, n_tiles, masks, counts, totals, summed ? box_base : nullptr, max_pts_per_box,
        (int)max_all_pts, (long long *)out_pts_idx, (long long *)out_roi_idx, out_pts_feats, num_out);
    return status_of(hipGetLastError());
}

int txs_grid_hash_build(const int32_t *keys, const int32_t *values, int64_t num_keys, int32_t *table,
                        int64_t table_size, int32_t *fail_flag, void *stream) {
    if (!fits_i32(num_keys) || !fits_i32(table_size) || table_size <= 0 || !table) return TXS_ERR_INVALID_ARG;
    if ((table_size & (table_size - 1)) != 0 || ((uintptr_t)table & 7) != 0) return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    fill_i32_kernel<<<dim3(blocks_for(2 * table_size)), dim3(kThreads), 0, st>>>(table, 2 * table_size, -1);
    if (num_keys > 0) {
        if (!keys || !values || num_keys > table_size) return TXS_ERR_INVALID_ARG;
        grid_hash_build_kernel<<<dim3(blocks_for(num_keys)), dim3(kThreads), 0, st>>>(
            keys, values, (unsigned long long *)table, (int)table_size, num_keys, num_keys <= kHashFewBuilt, fail_flag);
    }
    return status_of(hipGetLastError());
}

int txs_grid_hash_probe(const int32_t *keys, int64_t num_keys, const int32_t *table,
                        int64_t table_size, int32_t *out_values, void *stream) {
    if (!fits_i32(num_keys) || !fits_i32(table_size) || table_size <= 0 || !table) return TXS_ERR_INVALID_ARG;
    if ((table_size & (table_size - 1)) != 0 || ((uintptr_t)table & 7) != 0) return TXS_ERR_INVALID_ARG;
    if (num_keys == 0) return TXS_OK;
    if (!keys || !out_values) return TXS_ERR_INVALID_ARG;
    grid_hash_probe_kernel<<<dim3(blocks_for(num_keys)), dim3(kThreads), 0, (hipStream_t)stream>>>(
        FlatKeys<int>{keys}, (const unsigned long long *)table, (int)table_size, num_keys, hash_own(num_keys, table_size),
        out_values);
    return status_of(hipGetLastError());
}

int txs_grid_hash_probe_coors(const void *coors, int coor_is_int64, int64_t num_coors, int64_t dim1, int64_t dim2,
                              const int32_t *table, int64_t table_size, int32_t *out_values, void *stream) {
    if (!fits_i32(num_coors) || !fits_i32(table_size) || table_size <= 0 || !table) return TXS_ERR_INVALID_ARG;
    if ((table_size & (table_size - 1)) != 0 || ((uintptr_t)table & 7) != 0) return TXS_ERR_INVALID_ARG;
    if (num_coors == 0) return TXS_OK;
    if (!coors || !out_values) return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid(blocks_for(num_coors)), blk(kThreads);
    const long s0 = (long)(dim1 * dim2), s1 = (long)dim2;
    auto slots = (const unsigned long long *)table;
    const int own = hash_own(num_coors, table_size);
    if (coor_is_int64)
        grid_hash_probe_kernel<<<grid, blk, 0, st>>>(CoorKeys<long long>{static_cast<const long long *>(coors), s0, s1},
                                                     slots, (int)table_size, num_coors, own, out_values);
    else
        grid_hash_probe_kernel<<<grid, blk, 0, st>>>(CoorKeys<int>{static_cast<const int *>(coors), s0, s1}, slots,
                                                     (int)table_size, num_coors, own, out_values);
    return status_of(hipGetLastError());
}

}  // extern "C"
