// What the extension module calls of libtorchex_scatter.so beside its C ABI: txs_unique_plan in two
// halves, so that the map of the keys is under way while the rest is being allocated, and the
// first half straight from points.  Arguments and results as described for txs_unique_plan and
// txs_voxel_keys in torchex_scatter.h.
#pragma once

#include <stdint.h>

namespace txs_detail {

// The occupancy map of the keys.
int unique_map_keys(const void *keys, int key_is_int64, int64_t num_total, int64_t key_bound, int32_t *key_flag,
                    int32_t *bitmap_ws, void *stream);
// Coordinates and linear keys of the points, and the map of those: key_bound is dims[0] * dims[1] * dims[2], at
// most 2^31.  A point outside the grid is told of by the workspace's own flag (key_flag == NULL below).
int unique_map_points(const float *points, int64_t num_total, int64_t point_stride, const float *range_lo,
                      const float *voxel_size, const int32_t *dims, int32_t *coors, int32_t *keys, int32_t *bitmap_ws,
                      void *stream);
// The rest, from the map that either left in the workspace.
int unique_plan_of_map(const void *keys, int key_is_int64, int64_t num_total, int64_t key_bound, const int32_t *key_flag,
                       int32_t *bitmap_ws, int32_t heavy_threshold, int32_t *plan_ws, int32_t *unq_inv,
                       int32_t *unq_keys, int64_t *unq_cnts, int32_t *perm, int32_t *seg, int32_t *preSum,
                       int32_t *slot_of, int32_t *heavy_ids, int32_t *stats, void *stream);

}  // namespace txs_detail
