// The occupancy map of a grid of keys, as the kernels that make it (frontend_kernels.hip) leave it and those
// that turn keys into dense ids (there, and plan_kernels.hip while it sorts the rows) read it.
#pragma once

#include "txs_common.h"

namespace txs_detail {

// Dense ids of keys from an occupancy map of the grid they come from (frontend_kernels.hip): the id of a
// key is the number of occurring keys below it.
struct KeyMap {
    const void *keys;      // int32, or int64
    int keys64;
    long key_bound;
    const uint2 *cells;    // per 32 keys: (a bit for each that occurs, how many occur in its tile's cells in front)
    const int *tiles;      // occurring keys per tile of kScanTileItems cells; with `scanned` their exclusive
    int n_tiles, scanned;  // scan and the total (more than kMapTilesSummed tiles)
    long words;            // cells
    const int *bad;        // set if a key lies outside [0, key_bound)
    int *unq_keys;         // out: the occurring keys, ascending, the first `most` of them
    long most;
    int *num_unq, *found;  // out: their number; the same and *bad once more (found may be NULL)
};
constexpr int kMapTilesSummed = 1024;

// plan_build with the ids looked up by key: unq_inv is written, and so is what the map says of the keys.  Only
// where plan_takes_map() says so; the voxel count is map->num_unq.
int plan_build_mapped(const KeyMap &map, int32_t *unq_inv, int64_t num_total, int64_t num_unq, int32_t heavy_threshold,
                      int32_t *plan_ws, int32_t *perm, int32_t *seg, int32_t *preSum, int32_t *slot_of,
                      int32_t *heavy_ids, int32_t *stats, long long *cnts_out, void *stream);
bool plan_takes_map(long num_total, long num_unq);

}  // namespace txs_detail

namespace {

// Occurring keys in the map's tiles in front of every tile, into base_s (kMapTilesSummed ints; not used
// where the tiles are scanned already); returns their total.  The whole workgroup, which synchronises.
template <int THREADS>
__device__ __forceinline__ int map_tile_bases(const txs_detail::KeyMap &m, int *base_s) {
    if (m.scanned) return m.tiles[m.n_tiles];
    constexpr int kMost = txs_detail::kMapTilesSummed / THREADS;
    __shared__ int wave_s[THREADS / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, t0 = (int)threadIdx.x * kMost;
    int c[kMost], sum = 0;
#pragma unroll
    for (int k = 0; k < kMost; ++k) c[k] = t0 + k < m.n_tiles ? m.tiles[t0 + k] : 0;
#pragma unroll
    for (int k = 0; k < kMost; ++k) sum += c[k];
    const int inc = wave_inclusive_scan(sum);
    if (lane == 63) wave_s[w] = inc;
    __syncthreads();
    int off = 0, total = 0;
#pragma unroll
    for (int k = 0; k < THREADS / 64; ++k) {
        const int x = wave_s[k];
        if (k < w) off += x;
        total += x;
    }
    int at = off + inc - sum;
#pragma unroll
    for (int k = 0; k < kMost; ++k) {
        base_s[t0 + k] = at;
        at += c[k];
    }
    __syncthreads();
    return total;
}
__device__ __forceinline__ int map_tile_base(const txs_detail::KeyMap &m, const int *base_s, long tile) {
    return m.scanned ? m.tiles[tile] : base_s[tile];
}
// key as an index of the map; one outside the bound (which the caller refuses) counts as 0
__device__ __forceinline__ int map_key(const txs_detail::KeyMap &m, long i) {
    const long k = m.keys64 ? (long)static_cast<const long long *>(m.keys)[i] : (long)static_cast<const int *>(m.keys)[i];
    return k >= 0 && k < m.key_bound ? (int)k : 0;
}
__device__ __forceinline__ int map_id(const txs_detail::KeyMap &m, const int *base_s, uint2 cell, int key) {
    return map_tile_base(m, base_s, (long)(unsigned)key / (32 * txs_detail::kScanTileItems)) + (int)cell.y +
           __popc(cell.x & ((1u << (key & 31)) - 1u));
}
// The occurring keys of the cells of part number `part`, in their places among all.  A part is short: a cell
// with many keys is written by one lane, and more cells to a lane left too few in flight (a part of
// 2048 cells for 256 threads: grid_hash_prepare_kernel 10.7 us of 16.8M cells, of 512 cells 6).
constexpr int kMapPart = 512;
template <int THREADS>
__device__ __forceinline__ void map_list_part(const txs_detail::KeyMap &m, const int *base_s, long part) {
    const int base = map_tile_base(m, base_s, part * kMapPart / txs_detail::kScanTileItems);
    constexpr int kPer = kMapPart / THREADS;
    uint2 cell[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const long c = part * kMapPart + k * THREADS + threadIdx.x;
        cell[k] = c < m.words ? m.cells[c] : make_uint2(0u, 0u);
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const long c = part * kMapPart + k * THREADS + threadIdx.x;
        long r = (long)base + (int)cell[k].y;
        for (unsigned bits = cell[k].x; bits != 0u && r < m.most; bits &= bits - 1u, ++r)
            m.unq_keys[r] = (int)(c * 32 + __builtin_ctz(bits));
    }
}
inline int map_parts(const txs_detail::KeyMap &m) { return (int)((m.words + kMapPart - 1) / kMapPart); }

}  // namespace
