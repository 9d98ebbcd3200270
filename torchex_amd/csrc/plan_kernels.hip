// Index preparation for the voxel scatter kernels (built once per ScatterData and
// reused by every forward/backward call): a two-level bucket sort of (voxel id, row) for up
// to 2^22 voxels that yields CSR offsets, the table of special voxels and the
// per-position voxel ids on the way; for anything else a general sequence of
// sortedness/range check, stable LSD radix sort, CSR offsets from run boundaries and the
// same tables.  No histogram atomics on global memory and no inter-block spinning anywhere.
//
// Reference behaviour being replaced: ScatterData.__init__
// (torchex/operator_py/scatter_op.py:7-21) and getPreSum
// (torchex/src/scatter/scatter_kernel.cu:85-100).

#include "key_map.h"

#include <atomic>

namespace {

// -------------------------------------------------------------- small utils --

// Reference getPreSum (scatter_kernel.cu:85-100) for sorted ids.
__global__ void get_presum_kernel(const int *__restrict__ inv, int *__restrict__ preSum, long n,
                                  long num_presum) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int v = inv[i];
    bool boundary = (i == n - 1) || (inv[i + 1] != v);
    long slot = (long)v + 1;
    if (boundary && slot >= 0 && slot < num_presum) preSum[slot] = (int)(i + 1);
}

// Order and range flags of unq_inv (no histogram: counts come from the run
// boundaries of the sorted ids, which needs no atomics).
__global__ void plan_check_kernel(const int *__restrict__ inv, long n, int U,
                                  int *__restrict__ stats) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int v = inv[i];
    if ((unsigned)v >= (unsigned)U) stats[TXS_STAT_OUT_OF_RANGE] = 1;
    if (i + 1 < n && inv[i + 1] < v) stats[TXS_STAT_UNSORTED] = 1;
}

// ids that are already sorted are their own sorted keys
__global__ void copy_if_sorted_kernel(const int *__restrict__ inv, long n,
                                      const int *__restrict__ stats, int *__restrict__ keys) {
    if (stats[TXS_STAT_UNSORTED] != 0) return;
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) keys[i] = inv[i];
}

// CSR offsets from sorted keys: preSum[u] = first position whose key is >= u.
// Thread j owns the boundary in front of position j, i.e. the ids in (key[j-1], key[j]]
// (more than one only across empty voxels).  A long run of empty voxels is not walked by
// its one owner: the aligned blocks of kGapBlock ids that lie wholly inside a gap are left to
// presum_gap_blocks_kernel, and the owner fills only the two ragged ends.
constexpr int kGapBlock = 256;
__global__ void presum_from_sorted_kernel(const int *__restrict__ keys, long n, int U,
                                          int *__restrict__ preSum) {
    long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j > n) return;
    long lo = (j == 0) ? -1 : (long)(keys[j - 1] & kIdMask);
    long hi = (j == n) ? (long)U : (long)(keys[j] & kIdMask);
    if (hi > U) hi = U;
    // whole blocks [b0, b1) of ids inside (lo, hi]
    const long b0 = (lo + 1 + kGapBlock - 1) / kGapBlock * kGapBlock;
    const long b1 = (hi + 1) / kGapBlock * kGapBlock;
    if (b1 > b0) {
        for (long u = lo + 1; u < b0; ++u) preSum[u] = (int)j;
        for (long u = b1; u <= hi; ++u) preSum[u] = (int)j;
    } else {
        for (long u = lo + 1; u <= hi; ++u) preSum[u] = (int)j;
    }
}

// One workgroup per aligned block of kGapBlock ids: if no key falls inside the block (and
// none equals its last id's successor boundary), every id of it has the same offset, the
// first position whose key is at or above the block.
__global__ __launch_bounds__(kGapBlock) void presum_gap_blocks_kernel(const int *__restrict__ keys, long n, int U,
                                                                      int *__restrict__ preSum) {
    __shared__ long s_pos;
    const long bs = (long)blockIdx.x * kGapBlock, be = bs + kGapBlock;  // ids [bs, be)
    if (be - 1 > (long)U) return;                                       // not wholly inside [0, U]
    if (threadIdx.x == 0) {
        long a = 0, b = n;  // first position whose key is >= bs
        while (a < b) {
            const long m = (a + b) >> 1;
            if ((long)(keys[m] & kIdMask) < bs) a = m + 1; else b = m;
        }
        // the block lies wholly inside one gap iff the key at that position (or the end of
        // the ids, U) is at or beyond the block's last id
        const long next = a < n ? (long)(keys[a] & kIdMask) : (long)U;
        s_pos = next >= be - 1 ? a : -1;
    }
    __syncthreads();
    const long pos = s_pos;
    if (pos >= 0) preSum[bs + threadIdx.x] = (int)pos;
}

// ------------------------------------------------------------ exclusive scan --
// out[i] = sum_{k<i} in[k] for i in [0, n_out), where in[k] = 0 for k >= n_in.
// Three launches, no inter-block waiting: tile sums, scan of tile sums by one
// workgroup, tile-local scan plus tile offset.

constexpr int kScanItems = 8;
constexpr int kScanTile = kThreads * kScanItems;
static_assert(kScanTile == txs_detail::kScanTileItems, "producers of tile sums use the same tile");
constexpr int kScanFusedTiles = 1024;  // up to this many tiles the apply kernel sums the tile totals itself

__global__ __launch_bounds__(kThreads) void scan_tile_sums_kernel(const int *__restrict__ in,
                                                                  long n_in,
                                                                  int *__restrict__ tile_sums) {
    long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        long i = base + k;
        if (i < n_in) s += in[i];
    }
    int tot;
    block_exclusive_scan(s, &tot);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(kThreads) void scan_tile_offsets_kernel(int *__restrict__ tile_sums,
                                                                     long n_tiles) {
    int carry = 0;
    for (long base = 0; base < n_tiles; base += kThreads) {
        long i = base + threadIdx.x;
        int x = (i < n_tiles) ? tile_sums[i] : 0;
        int tot;
        int ex = block_exclusive_scan(x, &tot);
        if (i < n_tiles) tile_sums[i] = carry + ex;
        carry += tot;
    }
}

// in and out may be the same array: a thread reads its items before any write.
// With offsets_ready == 0, tile_offs still holds the plain tile sums and the
// workgroup adds up the ones in front of its own tile itself (cheaper than a
// launch of its own while there are few tiles).
// heads (may be NULL): receives every stride-th output on its own, heads[k] = out[k * stride].
__global__ __launch_bounds__(kThreads) void scan_apply_kernel(const int *in, long n_in, int *out,
                                                              long n_out, const int *tile_offs,
                                                              int offsets_ready, int *__restrict__ heads,
                                                              int stride) {
    long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
    int x[kScanItems];
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        long i = base + k;
        x[k] = (i < n_in) ? in[i] : 0;
        s += x[k];
    }
    int tile_off;
    if (offsets_ready) {
        tile_off = tile_offs[blockIdx.x];
    } else {
        int part = 0;
        for (int t = threadIdx.x; t < (int)blockIdx.x; t += kThreads) part += tile_offs[t];
        block_exclusive_scan(part, &tile_off);
    }
    int tot;
    int run = block_exclusive_scan(s, &tot) + tile_off;
    long head = heads ? (base + stride - 1) / stride : 0;  // the next one at or after `base`
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        long i = base + k;
        if (i < n_out) {
            out[i] = run;
            if (heads && i == head * stride) heads[head++] = run;
        }
        run += x[k];
    }
}

}  // namespace

namespace txs_detail {

long scan_tiles(long n_out) { return (n_out + kScanTile - 1) / kScanTile; }

hipError_t exclusive_scan(const int *in, long n_in, int *out, long n_out, int *ws,
                          hipStream_t st, int *heads, int stride) {
    if (n_out <= 0) return hipSuccess;
    const long tiles = scan_tiles(n_out);
    scan_tile_sums_kernel<<<dim3((unsigned)tiles), dim3(kThreads), 0, st>>>(in, n_in, ws);
    return scan_from_tile_sums(in, n_in, out, n_out, ws, st, heads, stride);
}

hipError_t scan_from_tile_sums(const int *in, long n_in, int *out, long n_out, int *ws, hipStream_t st, int *heads,
                               int stride) {
    if (n_out <= 0) return hipSuccess;
    const long tiles = scan_tiles(n_out);
    const int few = tiles <= kScanFusedTiles;
    if (!few) scan_tile_offsets_kernel<<<dim3(1), dim3(kThreads), 0, st>>>(ws, tiles);
    scan_apply_kernel<<<dim3((unsigned)tiles), dim3(kThreads), 0, st>>>(in, n_in, out, n_out, ws, !few, heads, stride);
    return hipGetLastError();
}

}  // namespace txs_detail

namespace {

using txs_detail::exclusive_scan;
using txs_detail::KeyMap;
using txs_detail::scan_tiles;

__device__ __forceinline__ int wave_max_i32(int x) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) x = max(x, __shfl_xor(x, d, 64));
    return x;
}

// Special-voxel table, max_cnt, and the check of the caller's counts against
// the histogram.  Launched with 1024-thread workgroups: the statistics are
// reduced across the workgroup first, because device-scope atomics on one
// address complete one after the other (~10 ns each) and one per wavefront
// would dominate the kernel.
constexpr int kSpecialThreads = 1024;
__global__ __launch_bounds__(kSpecialThreads) void plan_special_kernel(
    const int *__restrict__ preSum, int U_arg, int heavy_threshold,
    const long long *__restrict__ unq_cnts, int *__restrict__ slot_of,
    int *__restrict__ heavy_ids, int *__restrict__ stats, const int *__restrict__ num_unq_dev,
    long long *__restrict__ cnts_out) {
    __shared__ int s_max[kSpecialThreads / 64], s_bad[kSpecialThreads / 64];
    // the voxel count may only be known on the device (unique path): U_arg is then an upper bound
    const int U = num_unq_dev ? min(U_arg, *num_unq_dev) : U_arg;
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = u < U;
    const int c = in ? preSum[u + 1] - preSum[u] : 0;
    const int wmax = wave_max_i32(c);
    const bool mismatch = in && unq_cnts && unq_cnts[u] != (long long)c;
    const int any_mismatch = __ballot(mismatch) != 0ull;
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        s_max[w] = wmax;
        s_bad[w] = any_mismatch;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int m = 0, b = 0;
        for (int k = 0; k < kSpecialThreads / 64; ++k) {
            m = max(m, s_max[k]);
            b |= s_bad[k];
        }
        if (m > 0) atomicMax(&stats[TXS_STAT_MAX_CNT], m);
        if (b) stats[TXS_STAT_COUNT_MISMATCH] = 1;
    }
    if (in && cnts_out) cnts_out[u] = (long long)c;
    // Slots: heavy voxels fill heavy_ids from the front (their slot is also their row in
    // the scratch table), empty voxels from the back of the U-entry array (they own no
    // scratch).  One atomic per wave and kind hands out a contiguous range.
    const bool heavy = in && c > heavy_threshold;
    const bool empty = in && c == 0;
    const unsigned long long mh = __ballot(heavy), me = __ballot(empty);
    const int lane = threadIdx.x & 63;
    const unsigned long long below = (1ull << lane) - 1ull;
    int base_h = 0, base_e = 0;
    if (lane == 0) {
        if (mh) base_h = atomicAdd(&stats[TXS_STAT_NUM_HEAVY], __popcll(mh));
        if (me) base_e = atomicAdd(&stats[TXS_STAT_NUM_EMPTY], __popcll(me));
        if (mh | me) atomicAdd(&stats[TXS_STAT_NUM_SPECIAL], __popcll(mh) + __popcll(me));
    }
    base_h = __shfl(base_h, 0, 64);
    base_e = __shfl(base_e, 0, 64);
    if (!in) return;
    int slot = -1;
    if (heavy) {
        slot = base_h + __popcll(mh & below);
        if (slot < U_arg) heavy_ids[slot] = u;
    } else if (empty) {
        slot = U_arg - 1 - (base_e + __popcll(me & below));
        if (slot >= 0) heavy_ids[slot] = u;
    }
    slot_of[u] = slot;
}

// ----------------------------------------------------------- stable radix sort --
// One pass = per-tile digit histogram, exclusive scan of the digit-major
// histogram, stable scatter.  Inside a tile the order is (wave, item, lane),
// i.e. ascending input index, so each pass is stable.

constexpr int kSortItems = 8;
constexpr int kSortTile = kThreads * kSortItems;  // 2048 keys per workgroup
constexpr int kSortWaves = kThreads / 64;
constexpr int kSortWaveSpan = 64 * kSortItems;    // 512 consecutive keys per wave

__global__ __launch_bounds__(kThreads) void sort_hist_kernel(const int *__restrict__ keys, long n,
                                                             int shift, int rbits,
                                                             int *__restrict__ hist, int n_tiles,
                                                             const int *__restrict__ stats) {
    __shared__ int h[256];
    if (stats[TXS_STAT_UNSORTED] == 0) return;  // nothing to sort
    const int R = 1 << rbits;
    h[threadIdx.x] = 0;
    __syncthreads();
    long base = (long)blockIdx.x * kSortTile;
#pragma unroll
    for (int it = 0; it < kSortItems; ++it) {
        long i = base + (long)it * kThreads + threadIdx.x;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & (R - 1)], 1);
    }
    __syncthreads();
    if ((int)threadIdx.x < R) hist[(long)threadIdx.x * n_tiles + blockIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(kThreads) void sort_scatter_kernel(
    const int *__restrict__ keys_in, const int *__restrict__ vals_in, int *__restrict__ keys_out,
    int *__restrict__ vals_out, long n, int shift, int rbits, const int *__restrict__ hist_scanned,
    int n_tiles, const int *__restrict__ stats) {
    __shared__ int wcount[kSortWaves][256];
    if (stats[TXS_STAT_UNSORTED] == 0) return;  // nothing to sort
    __shared__ int woff[kSortWaves][256];
    const int R = 1 << rbits;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned long long lanes_below = (1ull << lane) - 1ull;
    for (int k = threadIdx.x; k < kSortWaves * 256; k += kThreads) (&wcount[0][0])[k] = 0;
    __syncthreads();

    const long base = (long)blockIdx.x * kSortTile + (long)w * kSortWaveSpan;
    int key[kSortItems], lrank[kSortItems];
    volatile int *wc = &wcount[w][0];
#pragma unroll
    for (int it = 0; it < kSortItems; ++it) {
        long i = base + (long)it * 64 + lane;
        bool valid = i < n;
        key[it] = valid ? keys_in[i] : 0;
        int digit = (key[it] >> shift) & (R - 1);
        unsigned long long mask = __ballot(valid);
        for (int b = 0; b < rbits; ++b) {
            bool bit = (digit >> b) & 1;
            unsigned long long bal = __ballot(bit);
            mask &= bit ? bal : ~bal;
        }
        int below = __popcll(mask & lanes_below);
        int prev = wc[digit];
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0) wc[digit] = prev + __popcll(mask);
        __builtin_amdgcn_wave_barrier();
        lrank[it] = prev + below;
    }
    __syncthreads();
    if ((int)threadIdx.x < R) {
        int run = hist_scanned[(long)threadIdx.x * n_tiles + blockIdx.x];
#pragma unroll
        for (int k = 0; k < kSortWaves; ++k) {
            woff[k][threadIdx.x] = run;
            run += wcount[k][threadIdx.x];
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kSortItems; ++it) {
        long i = base + (long)it * 64 + lane;
        if (i < n) {
            int digit = (key[it] >> shift) & (R - 1);
            long dst = (long)woff[w][digit] + lrank[it];
            if (dst >= 0 && dst < n) {
                keys_out[dst] = key[it];
                vals_out[dst] = vals_in ? vals_in[i] : (int)i;
            }
        }
    }
}

// seg[j] = id | special bit
__global__ void seg_flag_kernel(const int *ids, long n, int U, const int *__restrict__ slot_of,
                                int *seg) {
    long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    int u = ids[j] & kIdMask;
    int flag = ((unsigned)u < (unsigned)U && slot_of[u] >= 0) ? kSpecialBit : 0;
    seg[j] = u | flag;
}

// seg by binary search of each position in preSum (largest u with preSum[u] <= j)
__global__ void seg_from_presum_kernel(const int *__restrict__ preSum, long n, int U,
                                       const int *__restrict__ slot_of, int *__restrict__ seg) {
    long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    int lo = 0, hi = U;  // invariant: preSum[lo] <= j < preSum[hi]
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if ((long)preSum[mid] <= j) lo = mid; else hi = mid;
    }
    int flag = (slot_of[lo] >= 0) ? kSpecialBit : 0;
    seg[j] = lo | flag;
}

// ------------------------------------------------ two-level plan (bucket sort) --
//
// For up to 2^22 voxels the whole index preparation is four kernels:
//   (1) tile_sort_kernel: a tile of 1024 - 8192 rows is sorted by the HIGH digit of the voxel id
//       (the "bucket") in LDS and written back in place of itself, four bytes a row (the LOW digit
//       and the row's number inside the tile), with the tile's first row of every bucket and its
//       order / range flags;
//   (2) bucket_start_kernel: the first rows of a bucket, added up over the tiles, are the rows of all
//       buckets in front of it: where the bucket starts.  Flags of the whole input;
//   (3) bucket_count_kernel: a bucket is cut into slices; where one has very many, each is counted
//       per voxel (low digit, <= 11 bits) by a workgroup and the counts are written out.  Returns
//       at once for ordinary inputs;
//   (4) bucket_plan_kernel: a workgroup per slice gathers its rows from the tiles (a short run of
//       each, found by a scan over the tiles' counts) and counts them, and the bucket's other
//       slices, per voxel, which at the same time yields the bucket's share of everything else the
//       plan holds: CSR offsets, per-voxel counts (checked against the caller's), the special-voxel
//       table and its slots, max_cnt; then it places its slice by the low digit, stably, writing
//       the flagged per-position ids next to the permutation.
// No kernel needs the histogram of the whole input before it can write, so that neither a pass
// over the ids for it nor its scan is there, and every write up to the last kernel's is a stream.
// Above kTiledRows rows a bucket's runs would lie in too many tiles: the rows are then moved to
// bucket order, as (id, row) pairs, by bucket_hist_kernel, an exclusive scan of the digit-major
// histogram and bucket_scatter_kernel, and (3) and (4) read them there.

constexpr int kBucketHighBits = 9;      // high digit of the rows moved to bucket order
constexpr int kBucketLowBitsMax = 11;   // also the largest high digit
constexpr int kBucketBitsMax = 22;
constexpr int kHistThreads = 512;
// rows per tile of the histogram and scatter kernels: the instances of 4 and 8 items a thread
// served inputs that tile_sort_kernel takes now
constexpr int kHistItems = 16;
constexpr int kHistWaves = kHistThreads / 64;
constexpr int kBktItems = 8;                           // rows of its slice a thread places
constexpr long kBktGiant = 262144;                     // rows in one bucket beyond which the general sequence runs
// A bucket of up to this many slices is counted as a whole by each of its workgroups; above, the
// counts come from bucket_count_kernel.
constexpr int kSelfSlices = 2;
constexpr int kFlagUnsorted = 1, kFlagOutOfRange = 2;

// Bits of ids below U, and of them the low digit where the bucket digit may take high_bits.
__host__ __device__ __forceinline__ int radix_bits(int U) { return U > 2 ? 32 - __builtin_clz((unsigned)(U - 1)) : 1; }
__device__ __forceinline__ int low_bits_of(int U, int high_bits) { return max(0, radix_bits(U) - high_bits); }
// The voxel count a kernel works with: num_unq_dev (may be NULL) holds it where the host knows an
// upper bound only.  The digits are split by this count, not by the bound: ids of 2000 voxels among
// a million rows would all lie in the first bucket of the bound's split.
__device__ __forceinline__ int voxel_count(int U_arg, const int *__restrict__ num_unq_dev) {
    return num_unq_dev ? min(U_arg, *num_unq_dev) : U_arg;
}

// How the rows are cut into tiles and the ids into digits, for ids of `bits` bits.  Short tiles keep workgroups
// short and many, long ones leave fewer runs of a bucket to find.  Plans of a sweep, of rows in clusters of 4 and of 50, us
// a call with their host read, on either side of the lines:
//   2^18 rows (tiles of 1024 / 2048): 60k rows 48 / 48, 49 / 49, 50 / 50; 2^18 53 / 53, 51 / 51, 53 / 52.  256 threads, which
//     serve a slice best up to here (below), look at 256 tiles at most.
//   5 * 2^18 rows (2048 / 4096): plans gain 1 - 4 % from the longer tiles from 600k rows on (1M 74 / 72, 62 / 60, 66 / 63; 1.5M
//     80 / 78, 81 / 77, 74 / 74), plans from keys, whose ids are looked up on the way, lose up to 9 % (1M 116 / 117,
//     105 / 111, 103 / 107; 1.3M 114 / 116, 103 / 110, 114 / 115).
//   2^21 rows (4096 / 8192): 2.1M 87 / 88, 89 / 87, 86 / 85; 4M 123 / 118, 138 / 125, 114 / 106.
constexpr int kTileRowsMax = 8192;
constexpr int kTilesMax = 2048;
constexpr long kTiledRows = (long)kTileRowsMax * kTilesMax;
constexpr long kMappedRows = 1L << 21;  // rows up to which ids are looked up by the kernel that sorts the tiles
struct TileSplit {
    int tile_bits;   // log2(rows per tile)
    int high_bits;
    int tiles;
    int pitch;       // entries of a tile's row of first rows: one per bucket, the tile's valid rows, padding
};
TileSplit tile_split(long n, int bits) {
    TileSplit r;
    r.tile_bits = n <= (1L << 18) ? 10 : (n <= (5L << 18) ? 11 : (n <= kMappedRows ? 12 : 13));
    r.high_bits = bits <= kBucketLowBitsMax ? bits : min(max(kBucketHighBits, bits - 10), kBucketLowBitsMax);
    if (r.high_bits > 10 && r.tile_bits < 11) r.tile_bits = 11;  // (256 threads scan at most 1024 buckets)
    r.tiles = (int)((n + (1L << r.tile_bits) - 1) >> r.tile_bits);
    r.pitch = max(1 << r.high_bits, 4) + 4;
    return r;
}
// Threads of the workgroups that serve a slice of kBktItems rows per thread: 256 while they can look at all tiles
// (256 of them; 2^19 rows) and at all of a bucket's voxels (four a thread).  256 / 512: 60k rows in 1500 voxels 47 / 56 us a
// plan, grouped 51 / 61; 262k in 1500 voxels 52 / 60, a sweep 53 / 50; 2^19 rows 62 / 63 and 56 / 63.  Ranks come with the
// number of rows for a bound, so that few groups crowd one bucket, whose slices each look at all others' counts: 2000
// rows 35 - 40 / 36 - 48 us, 100k 40 - 52 / 41 - 49, 200k in 64 groups 72 / 55, in 66,000 46 / 45, 350k in 1500 113 / 69.
int slice_threads_for(long n, int low_bits, bool ranks) { return n > (ranks ? 1L << 17 : 1L << 19) || low_bits > 10 ? 512 : 256; }

// exclusive scan of one int per thread across a workgroup of WAVES wavefronts
template <int WAVES>
__device__ __forceinline__ int wide_exclusive_scan(int x, int *total) {
    __shared__ int wsum[WAVES];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int inc = wave_inclusive_scan(x);
    __syncthreads();  // wsum may still be read by a previous call
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    int off = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) {
        const int v = wsum[k];
        if (k < w) off += v;
        tot += v;
    }
    *total = tot;
    return off + inc - x;
}

// Lanes of the wavefront whose `digit` (of `bits` bits) equals this lane's, among those with
// `valid` set; all 64 lanes take part.
__device__ __forceinline__ unsigned long long wave_match(int digit, int bits, bool valid) {
    const unsigned long long all = __ballot(valid);
    unsigned lo = (unsigned)all, hi = (unsigned)(all >> 32);
    for (int b = 0; b < bits; ++b) {
        const unsigned mine = (unsigned)((int)((unsigned)digit << (31 - b)) >> 31);  // the bit in every position
        const unsigned long long bal = __ballot(mine != 0u);
        lo &= ~((unsigned)bal ^ mine);
        hi &= ~((unsigned)(bal >> 32) ^ mine);
    }
    return ((unsigned long long)hi << 32) | lo;
}

// Rank of every row among its wave's rows of the same digit (`bits` bits of the key from bit `shift` on, the
// key's highest ones), in (item, lane) order: turn[k] for the rows with key[k] >= 0.  counts2: the wave's own 16-bit counts, one per digit, zero on entry; the wave's
// rows per digit on return.  The items advance bit by bit side by side: an item's chain of ballots depends on
// itself all the way, and one item after the other left the vector units idle for most of it (eight
// items of eight bits, in a workgroup of 256 threads: 3.1 us, now 2.1).
template <int COUNT>
__device__ __forceinline__ void wave_rank(const int (&key)[COUNT], int shift, int bits, unsigned *counts2, int (&turn)[COUNT]) {
    const int lane = threadIdx.x & 63;
    const unsigned below_lo = lane < 32 ? (1u << lane) - 1u : 0xffffffffu;
    const unsigned below_hi = lane < 32 ? 0u : (1u << (lane - 32)) - 1u;
    unsigned lo[COUNT], hi[COUNT];
#pragma unroll
    for (int k = 0; k < COUNT; ++k) {
        const unsigned long long all = __ballot(key[k] >= 0);
        lo[k] = (unsigned)all;
        hi[k] = (unsigned)(all >> 32);
    }
#pragma unroll 1
    for (int b = 0; b < bits; ++b) {
#pragma unroll
        for (int k = 0; k < COUNT; ++k) {
            const unsigned mine = (unsigned)__builtin_amdgcn_sbfe(key[k], shift + b, 1);  // the bit in every position
            const unsigned long long bal = __ballot(mine != 0u);
            lo[k] &= ~((unsigned)bal ^ mine);
            hi[k] &= ~((unsigned)(bal >> 32) ^ mine);
        }
    }
    // The first row of each group adds the group to the count, two 16-bit counts to a word, and hands
    // the count before it round: the adds of all items are in flight together (LDS serves a wave's
    // instructions in order, so they count up item by item); the other rows add nothing to a word of
    // their own, so that no add is under a branch.  The stages are kept apart to bound the registers.
    __shared__ unsigned sink_s[64];
    unsigned before[COUNT];
#pragma unroll
    for (int k = 0; k < COUNT; ++k) {
        const int below = __popc(lo[k] & below_lo) + __popc(hi[k] & below_hi), group = __popc(lo[k]) + __popc(hi[k]);
        const int leader = lo[k] ? __builtin_ctz(lo[k]) : 32 + __builtin_ctz(hi[k] | 0x80000000u);
        turn[k] = below | leader << 8 | group << 16;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < COUNT; ++k) {
        const bool first = key[k] >= 0 && (turn[k] & 255) == 0;
        before[k] = atomicAdd(first ? counts2 + (key[k] >> (shift + 1)) : &sink_s[lane],
                              first ? (unsigned)(turn[k] >> 16) << ((key[k] >> shift & 1) << 4) : 0u);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < COUNT; ++k)
        turn[k] = (turn[k] & 255) + (int)((__shfl(before[k], (turn[k] >> 8) & 255, 64) >> ((key[k] >> shift & 1) << 4)) & 0xffffu);
    __builtin_amdgcn_sched_barrier(0);
}

// A tile's rows in bucket order: rows_out[tile's first row + k] = low digit << tile bits | row inside
// the tile; offs[tile][d] = the tile's rows in buckets below d (d up to the number of buckets).
// K = long long: ids as torch.unique returns them, cut to 32 bits and left in `ids32` for later readers.
// K = KeyMap: the ids are looked up by key and left in `ids32` (a kernel of its own for that, which this one
// then read again, took 6 us of 200k rows in 16.9M cells); the workgroups behind those of the tiles list
// the occurring keys.
// stats and ctl are cleared for the kernels that follow.
// Ranking is by wave ballots on the digit's bits and a 16-bit count per wave and bucket; the rows pass
// through LDS so that they leave as one stream.
template <int THREADS, int ITEMS, typename K>
__global__ __launch_bounds__(THREADS) void tile_sort_kernel(
    std::conditional_t<std::is_same_v<K, KeyMap>, KeyMap, const K *> ids, long n, int n_tiles, int U_arg, int high_bits,
    unsigned *__restrict__ rows_out, unsigned short *__restrict__ offs, int pitch, int *__restrict__ tile_flags,
    int *__restrict__ ids32, int *__restrict__ stats, int *__restrict__ ctl, const int *__restrict__ num_unq_dev) {
    constexpr int WAVES = THREADS / 64, kRows = THREADS * ITEMS, kTileBits = __builtin_ctz(kRows);
    // [bins] first place of every bucket, then the larger of [WAVES][bins] counts and the staged rows
    extern __shared__ __align__(16) uint2 lds_tile[];
    constexpr bool kMap = std::is_same_v<K, KeyMap>;
    __shared__ int s_flags;
    __shared__ int base_s[kMap ? txs_detail::kMapTilesSummed : 1];
    int U;
    if constexpr (kMap) {
        U = min(U_arg, map_tile_bases<THREADS>(ids, base_s));
        if ((int)blockIdx.x >= n_tiles) {
            map_list_part<THREADS>(ids, base_s, (int)blockIdx.x - n_tiles);
            return;
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            ids.num_unq[0] = U;
            if (ids.found) {
                ids.found[0] = U;
                ids.found[1] = ids.bad[0];
            }
        }
    } else {
        U = voxel_count(U_arg, num_unq_dev);
    }
    const int low_bits = low_bits_of(U, high_bits);
    const int quads = max(1 << high_bits, 4) >> 2;  // bins / 4
    uint2 *first4 = lds_tile, *cnt4 = lds_tile + quads;
    const unsigned short *first = reinterpret_cast<const unsigned short *>(first4);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long tile0 = (long)blockIdx.x * kRows;
    const long wbase = tile0 + (long)w * (64 * ITEMS);
    if (blockIdx.x == 0) {
        if (threadIdx.x < TXS_STATS_LEN) stats[threadIdx.x] = 0;
        if (threadIdx.x == 0) ctl[0] = 0;
    }
    int key[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const long i = wbase + (long)it * 64 + lane;
        if constexpr (kMap) key[it] = i < n ? map_key(ids, i) : 0x7fffffff;
        else key[it] = i < n ? (int)ids[i] : 0x7fffffff;
    }
    // the id (or key: they ascend together) behind the wave's rows
    int behind = 0x7fffffff;
    if (lane == 63 && wbase + 64 * ITEMS < n) {
        if constexpr (kMap) behind = map_key(ids, wbase + 64 * ITEMS);
        else behind = (int)ids[wbase + 64 * ITEMS];
    }
    uint2 cell[kMap ? ITEMS : 1];
    if constexpr (kMap) {
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) cell[it] = ids.cells[wbase + (long)it * 64 + lane < n ? key[it] >> 5 : 0];
    }
    if (threadIdx.x == 0) s_flags = 0;
    for (int k = threadIdx.x; k < WAVES * quads; k += THREADS) cnt4[k] = make_uint2(0u, 0u);
    __syncthreads();
    bool bad_range = false, bad_order = false;
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const long i = wbase + (long)it * 64 + lane;
        if (std::is_same_v<K, long long> && i < n) ids32[i] = key[it];
        int next = __shfl_down(key[it], 1, 64);
        const int wrap = it + 1 < ITEMS ? __builtin_amdgcn_readfirstlane(key[it + 1 < ITEMS ? it + 1 : 0]) : behind;
        if (lane == 63) next = wrap;
        bad_order |= next < key[it];  // (rows behind the last one compare as the largest id)
        if constexpr (kMap) {
            if (i < n) ids32[i] = key[it] = map_id(ids, base_s, cell[it], key[it]);
        }
        if ((unsigned)key[it] >= (unsigned)U) {
            bad_range |= i < n;
            key[it] = -1;  // out-of-range ids are dropped (and flagged)
        }
    }
    const int f = (__ballot(bad_order) != 0ull ? kFlagUnsorted : 0) | (__ballot(bad_range) != 0ull ? kFlagOutOfRange : 0);
    if (f && lane == 0) atomicOr(&s_flags, f);
    int place[ITEMS];
    wave_rank<ITEMS>(key, low_bits, high_bits, reinterpret_cast<unsigned *>(cnt4 + w * quads), place);
    __syncthreads();
    const unsigned short *wc = reinterpret_cast<const unsigned short *>(cnt4 + w * quads);
    // counts per wave -> rows of the waves in front; totals -> first place of every bucket.  Four
    // buckets a thread, two 16-bit numbers to a word: no sum passes the tile's 8192 rows.
    uint2 run = make_uint2(0u, 0u);
    const int q = threadIdx.x;
    if (q < quads) {
#pragma unroll
        for (int k = 0; k < WAVES; ++k) {
            const uint2 c = cnt4[k * quads + q];
            cnt4[k * quads + q] = run;
            run.x += c.x;
            run.y += c.y;
        }
    }
    const int c0 = run.x & 0xffff, c1 = run.x >> 16, c2 = run.y & 0xffff, c3 = run.y >> 16;
    int total;
    const int at = wide_exclusive_scan<WAVES>(c0 + c1 + c2 + c3, &total);
    uint2 *offs4 = reinterpret_cast<uint2 *>(offs + (long)blockIdx.x * pitch);
    if (q < quads) {
        const uint2 o = make_uint2((unsigned)at | (unsigned)(at + c0) << 16,
                                   (unsigned)(at + c0 + c1) | (unsigned)(at + c0 + c1 + c2) << 16);
        first4[q] = o;
        offs4[q] = o;
    }
    if (threadIdx.x == 0) {
        offs4[quads] = make_uint2((unsigned)total * 0x10001u, (unsigned)total * 0x10001u);
        tile_flags[blockIdx.x] = s_flags;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) place[it] += (int)first[max(key[it], 0) >> low_bits] + (int)wc[max(key[it], 0) >> low_bits];
    __syncthreads();
    unsigned *stage = reinterpret_cast<unsigned *>(cnt4);
    const unsigned low_mask = (1u << low_bits) - 1u;
#pragma unroll
    for (int it = 0; it < ITEMS; ++it)
        if (key[it] >= 0)
            stage[place[it]] = ((unsigned)key[it] & low_mask) << kTileBits | (unsigned)(w * (64 * ITEMS) + it * 64 + lane);
    __syncthreads();
    for (int p = threadIdx.x; p < total; p += THREADS) rows_out[tile0 + p] = stage[p];
}

// What a plan holds per voxel (any of it may be NULL but preSum; slot_of and heavy_ids go together).
struct VoxelArgs {
    int heavy_threshold;
    const long long *unq_cnts;  // the caller's counts
    int *preSum, *slot_of, *heavy_ids;
    long long *cnts_out;
};
// Special voxels and their slots, as plan_special_kernel: COUNT consecutive voxels a lane, from `u` on, as
// far as they lie below `end`.  One atomic per wave and kind.
template <int COUNT>
__device__ __forceinline__ void voxel_slots(const VoxelArgs &v, int U, int u, int end, const int (&count)[COUNT],
                                            int *__restrict__ stats) {
    const int lane = threadIdx.x & 63;
    const unsigned long long lanes_below = (1ull << lane) - 1ull;
    int heavy = 0, empty = 0, heavy_below[COUNT], empty_below[COUNT];  // of the wave; in front of this voxel
#pragma unroll
    for (int k = 0; k < COUNT; ++k) {
        const bool valid = u + k < end;
        const unsigned long long mh = __ballot(valid && count[k] > v.heavy_threshold), me = __ballot(valid && count[k] == 0);
        heavy_below[k] = heavy + __popcll(mh & lanes_below);
        empty_below[k] = empty + __popcll(me & lanes_below);
        heavy += __popcll(mh);
        empty += __popcll(me);
    }
    int base_h = 0, base_e = 0;
    if (heavy + empty > 0) {
        if (lane == 0) {
            if (heavy) base_h = atomicAdd(&stats[TXS_STAT_NUM_HEAVY], heavy);
            if (empty) base_e = atomicAdd(&stats[TXS_STAT_NUM_EMPTY], empty);
            atomicAdd(&stats[TXS_STAT_NUM_SPECIAL], heavy + empty);
        }
        base_h = __shfl(base_h, 0, 64);
        base_e = __shfl(base_e, 0, 64);
    }
#pragma unroll
    for (int k = 0; k < COUNT; ++k) {
        if (u + k >= end) continue;
        int slot = -1;
        if (count[k] > v.heavy_threshold) {
            slot = base_h + heavy_below[k];
            if (slot < U) v.heavy_ids[slot] = u + k;
        } else if (count[k] == 0) {
            slot = U - 1 - (base_e + empty_below[k]);
            if (slot >= 0) v.heavy_ids[slot] = u + k;
        }
        v.slot_of[u + k] = slot;
    }
}

// The same and the rest of it where a bucket is a voxel: a wave of voxels u, those with `in`, whose rows
// start at `start`.
__device__ __forceinline__ void bucket_voxel(const VoxelArgs &v, int U, int n, int u, bool in, int start, int rows,
                                             int *__restrict__ stats) {
    if (in) {
        v.preSum[u] = start;
        if (v.cnts_out) v.cnts_out[u] = (long long)rows;
        if (u == U - 1) v.preSum[U] = n;
    }
    if (v.slot_of == nullptr) return;
    const int count[1] = {rows};
    voxel_slots<1>(v, U, u, in ? U : 0, count, stats);
    const bool mismatch = in && v.unq_cnts && v.unq_cnts[u] != (long long)rows;
    const int most = wave_max_i32(in ? rows : 0);
    if (__ballot(mismatch) != 0ull && (threadIdx.x & 63) == 0) stats[TXS_STAT_COUNT_MISMATCH] = 1;
    if ((threadIdx.x & 63) == 0 && most > 0) atomicMax(&stats[TXS_STAT_MAX_CNT], most);
}
__global__ __launch_bounds__(64) void bucket_voxels_kernel(const int *__restrict__ bucket_start, int n, int U_arg,
                                                           int high_bits, int *__restrict__ stats,
                                                           const int *__restrict__ num_unq_dev, VoxelArgs v) {
    const int U = voxel_count(U_arg, num_unq_dev), u = (int)(blockIdx.x * 64 + threadIdx.x);
    if (low_bits_of(U, high_bits) > 0 || stats[TXS_STAT_NEED_GENERAL] != 0) return;
    const bool in = u < U;
    const int start = in ? bucket_start[u] : 0;
    bucket_voxel(v, U, n, u, in, start, in ? bucket_start[u + 1] - start : 0, stats);
}

// bucket_start[d] = rows in buckets below d, for d up to the number of buckets: the sum over the tiles
// of offs[.][d].  A workgroup reads 32 neighbouring columns (a 64-byte sector per tile) and owns the
// first 30 of them, so that it also sees where each of its buckets ends.
// Where a bucket is a voxel (ids of at most 11 bits), what the plan holds per voxel is left here too: the
// statistics take one atomic per 30 voxels, where bucket_plan_kernel's workgroups, one or more per voxel,
// would queue up for the same few words (index preparation of 1M rows in 1000 Zipf voxels: 88 us with
// that, 65 so).
// Sets stats[NEED_GENERAL] for a bucket above kBktGiant rows (the kernels that follow step aside; not
// where so few voxels have so many rows that the low digit has next to nothing left) and ctl[0] for
// one of more than kSelfSlices slices; workgroup 0 also the flags of the whole input.
constexpr int kStartThreads = 1024, kStartColumns = 32, kStartOwned = 30;
__global__ __launch_bounds__(kStartThreads) void bucket_start_kernel(
    const unsigned short *__restrict__ offs, int pitch, int n_tiles, int n, int U_arg, int high_bits, int self_rows,
    const int *__restrict__ tile_flags, int *__restrict__ bucket_start, int *__restrict__ stats,
    int *__restrict__ ctl, const int *__restrict__ num_unq_dev, VoxelArgs v) {
    constexpr int kLanes = kStartColumns / 2, kGroups = kStartThreads / kLanes;  // two columns a thread
    __shared__ int sum_s[kGroups][kStartColumns + 2];
    __shared__ int start_s[kStartColumns];
    const int x = threadIdx.x % kLanes, y = threadIdx.x / kLanes;
    const int word = (int)blockIdx.x * (kStartOwned / 2) + x, words = pitch / 2;
    const unsigned *offs2 = reinterpret_cast<const unsigned *>(offs);
    int lo = 0, hi = 0;
    if (word < words) {
#pragma unroll 4
        for (int t = y; t < n_tiles; t += kGroups) {
            const unsigned two = offs2[(long)t * words + word];
            lo += (int)(two & 0xffffu);
            hi += (int)(two >> 16);
        }
    }
    sum_s[y][2 * x] = lo;
    sum_s[y][2 * x + 1] = hi;
    if (blockIdx.x == 0) {
        int f = 0;
        for (int t = threadIdx.x; t < n_tiles; t += kStartThreads) f |= tile_flags[t];
        if (f & kFlagUnsorted) stats[TXS_STAT_UNSORTED] = 1;
        if (f & kFlagOutOfRange) stats[TXS_STAT_OUT_OF_RANGE] = 1;
    }
    __syncthreads();
    // 32 threads per column
    const int c = threadIdx.x >> 5, part = threadIdx.x & 31;
    int s = 0;
    for (int k = part; k < kGroups; k += 32) s += sum_s[k][c];
#pragma unroll
    for (int d = 16; d >= 1; d >>= 1) s += __shfl_xor(s, d, 64);
    if (part == 0) start_s[c] = s;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const int col = (int)blockIdx.x * kStartOwned + (int)threadIdx.x;
    const int bins = 1 << high_bits, U = voxel_count(U_arg, num_unq_dev);
    const bool owned = threadIdx.x < kStartOwned, bucket = owned && col < bins;
    const int start = owned ? start_s[threadIdx.x] : 0;
    const int rows = bucket ? start_s[threadIdx.x + 1] - start : 0;
    if (owned && col <= bins) bucket_start[col] = start;
    if (low_bits_of(U, high_bits) > 0) {
        if (rows > kBktGiant && U > 1 << kBucketLowBitsMax) stats[TXS_STAT_NEED_GENERAL] = 1;
        if (rows > self_rows) ctl[0] = 1;
        return;
    }
    bucket_voxel(v, U, n, col, bucket && col < U, start, rows, stats);
}

// hist: [high_bins][n_tiles] digit-major (the order its exclusive scan needs); tile_flags: [n_tiles]
// K = long long: ids as torch.unique returns them, cut to 32 bits and left in `ids32` for the
// kernels that follow (a conversion of its own reads and writes them once more: 16 us of 4M ids,
// 5 us of 1M)
template <typename K>
__global__ __launch_bounds__(kHistThreads) void bucket_hist_kernel(
    const K *__restrict__ inv, long n, int U_arg, int high_bits, int *__restrict__ hist,
    int *__restrict__ tile_flags, int n_tiles, int *__restrict__ ids32, const int *__restrict__ num_unq_dev) {
    __shared__ int h[1 << kBucketLowBitsMax];
    __shared__ int s_flags;
    const int U = voxel_count(U_arg, num_unq_dev), low_bits = low_bits_of(U, high_bits), high_bins = 1 << high_bits;
    for (int d = threadIdx.x; d < high_bins; d += kHistThreads) h[d] = 0;
    if (threadIdx.x == 0) s_flags = 0;
    __syncthreads();
    const long base = (long)blockIdx.x * (kHistThreads * kHistItems);
    int v[kHistItems];
#pragma unroll
    for (int it = 0; it < kHistItems; ++it) {
        const long i = base + (long)it * kHistThreads + threadIdx.x;
        v[it] = i < n ? (int)inv[i] : 0x7fffffff;
        if (sizeof(K) == 8 && i < n) ids32[i] = v[it];
    }
    bool bad_range = false, bad_order = false;
#pragma unroll
    for (int it = 0; it < kHistItems; ++it) {
        const long i = base + (long)it * kHistThreads + threadIdx.x;
        if (i >= n) continue;
        if ((unsigned)v[it] >= (unsigned)U) {
            bad_range = true;
        } else {
            atomicAdd(&h[v[it] >> low_bits], 1);
        }
        // neighbour in memory = the next thread's element of the same round
        int nb = __shfl_down(v[it], 1, 64);
        if ((threadIdx.x & 63) == 63) nb = (i + 1 < n) ? (int)inv[i + 1] : 0x7fffffff;
        if (i + 1 < n && nb < v[it]) bad_order = true;
    }
    const int f = (__ballot(bad_order) != 0ull ? kFlagUnsorted : 0) | (__ballot(bad_range) != 0ull ? kFlagOutOfRange : 0);
    if (f && (threadIdx.x & 63) == 0) atomicOr(&s_flags, f);
    __syncthreads();
    for (int d = threadIdx.x; d < high_bins; d += kHistThreads) hist[(long)d * n_tiles + blockIdx.x] = h[d];
    if (threadIdx.x == 0) tile_flags[blockIdx.x] = s_flags;
}

__global__ void narrow_ids_kernel(const long long *__restrict__ ids64, long n, int *__restrict__ ids32) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) ids32[i] = (int)ids64[i];
}

// Stable scatter by the high digit.  hist: the exclusive scan of the digit-major tile histograms.
//   bucket_start [high_bins + 1] (from the scan): first position of every bucket.
//   stats: zero-filled here (workgroup 0), then UNSORTED / OUT_OF_RANGE of the whole input
//   and NEED_GENERAL (a bucket above kBktGiant rows: the bucket kernels step aside; not where so few
//   voxels have so many rows that the low digit has next to nothing left).
// Rows already in order are not moved: the next kernel reads unq_inv itself.  out_pairs: (id, row) per
// position, one 8-byte store.
__global__ __launch_bounds__(kHistThreads) void bucket_scatter_kernel(
    const int *__restrict__ inv, long n, int U_arg, int high_bits,
    const int *__restrict__ hist, const int *__restrict__ tile_flags, int n_tiles,
    const int *__restrict__ bucket_start, int *__restrict__ stats, int2 *__restrict__ out_pairs,
    const int *__restrict__ num_unq_dev) {
    // [bins] base_s: first destination of this tile's rows, per digit; then the larger of
    // [kHistWaves][bins] wave counts and the tile's staged (id, row) pairs
    extern __shared__ __align__(8) int lds_base[];
    __shared__ int s_flags;
    const int U = voxel_count(U_arg, num_unq_dev), low_bits = low_bits_of(U, high_bits);
    const bool may_overfill = U > 1 << kBucketLowBitsMax;
    const int bins = 1 << high_bits;
    int *base_s = lds_base, *lds_scatter = lds_base + bins, *wcount = lds_scatter;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned long long lanes_below = (1ull << lane) - 1ull;
    if (threadIdx.x == 0) s_flags = 0;
    for (int k = threadIdx.x; k < kHistWaves * bins; k += kHistThreads) wcount[k] = 0;
    __syncthreads();

    // ---- flags of the whole input
    int f = 0;
    for (int t = threadIdx.x; t < n_tiles; t += kHistThreads) f |= tile_flags[t];
    if (f) atomicOr(&s_flags, f);

    // ---- first destination of this tile's rows per digit (from the scanned histogram) and the
    // test for an overfull bucket.  The bucket boundaries lie side by side for it: read from the
    // histogram, two lines of it per bucket, they cost every workgroup more (1M ids 13.7 -> 15.4 us).
    for (int d = threadIdx.x; d < bins; d += kHistThreads) {
        base_s[d] = hist[(long)d * n_tiles + blockIdx.x];
        if (may_overfill && (long)bucket_start[d + 1] - bucket_start[d] > kBktGiant) atomicOr(&s_flags, 4);
    }
    __syncthreads();
    const int flags = s_flags;
    if (blockIdx.x == 0) {
        for (int k = threadIdx.x; k < TXS_STATS_LEN; k += kHistThreads) {
            int val = 0;
            if (k == TXS_STAT_UNSORTED) val = (flags & kFlagUnsorted) ? 1 : 0;
            if (k == TXS_STAT_OUT_OF_RANGE) val = (flags & kFlagOutOfRange) ? 1 : 0;
            if (k == TXS_STAT_NEED_GENERAL) val = (flags & 4) ? 1 : 0;
            stats[k] = val;
        }
    }
    if (flags & 4) return;  // the caller re-plans with the general sequence
    const long tile0 = (long)blockIdx.x * (kHistThreads * kHistItems);
    if (!(flags & kFlagUnsorted)) return;

    // ---- stable ranking inside the tile
    const long wbase = tile0 + (long)w * (64 * kHistItems);
    int key[kHistItems], lrank[kHistItems];
#pragma unroll
    for (int it = 0; it < kHistItems; ++it) {
        const long i = wbase + (long)it * 64 + lane;
        const int v = i < n ? inv[i] : -1;
        key[it] = (unsigned)v < (unsigned)U ? v : -1;  // out-of-range ids are dropped (and flagged)
    }
    volatile int *wc = wcount + w * bins;
#pragma unroll
    for (int it = 0; it < kHistItems; ++it) {
        const bool valid = key[it] >= 0;
        const unsigned long long mask = wave_match(valid ? key[it] >> low_bits : 0, high_bits, valid);
        // rows of the same bucket in front of this one among the wave's 64, and the group's size
        lrank[it] = __popcll(mask & lanes_below) | (__popcll(mask) << 8);
    }
#pragma unroll
    for (int it = 0; it < kHistItems; ++it) {
        const bool valid = key[it] >= 0;
        const int digit = valid ? (key[it] >> low_bits) : 0;
        const int below = lrank[it] & 255, group = lrank[it] >> 8;
        const int prev = wc[digit];
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0) wc[digit] = prev + group;
        __builtin_amdgcn_wave_barrier();
        lrank[it] = prev + below;
    }
    __syncthreads();
    // ---- the tile's rows in bucket order: wcount[k][d] becomes the place, inside the tile, of
    // the first row that wave k has for bucket d, base_s[d] the step from there to its destination
    int total = 0;
    {
        const int per = (bins + kHistThreads - 1) / kHistThreads;
        const int d0 = (int)threadIdx.x * per;
        int mine = 0;
        for (int d = d0; d < min(d0 + per, bins); ++d)
            for (int k = 0; k < kHistWaves; ++k) mine += wcount[k * bins + d];
        int run = wide_exclusive_scan<kHistWaves>(mine, &total);
        for (int d = d0; d < min(d0 + per, bins); ++d) {
            base_s[d] -= run;
            for (int k = 0; k < kHistWaves; ++k) {
                const int c = wcount[k * bins + d];
                wcount[k * bins + d] = run;
                run += c;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kHistItems; ++it)
        if (key[it] >= 0) lrank[it] += wcount[w * bins + (key[it] >> low_bits)];
    __syncthreads();
    // ---- through LDS (over the wave counts, which are done with): the tile's rows leave in
    // bucket order, so that neighbouring lanes write neighbouring addresses.  Written straight
    // from the ranking, every 8-byte pair was a memory request of its own.  (4M ids in
    // 1024 buckets: 37.6 -> 28.5 us; 1M ids, whose tiles hold four rows per bucket only: 15.2 -> 15.6)
    int2 *stage = reinterpret_cast<int2 *>(lds_scatter);
#pragma unroll
    for (int it = 0; it < kHistItems; ++it)
        if (key[it] >= 0) stage[lrank[it]] = make_int2(key[it], (int)(wbase + (long)it * 64 + lane));
    __syncthreads();
    for (int p = threadIdx.x; p < total; p += kHistThreads) {
        const int2 kr = stage[p];
        const long dst = (long)base_s[kr.x >> low_bits] + p;
        if (dst < 0 || dst >= n) continue;
        out_pairs[dst] = kr;
    }
}

// A bucket is cut into slices of slice_rows rows.  The first `more` workgroups (an upper bound) serve the
// further slices of all buckets, bucket by bucket, and start first, because theirs are the full buckets;
// those behind them serve the first slice of a bucket each.
__device__ __forceinline__ int slices_of(int rows, int slice_rows) { return max(1, (rows + slice_rows - 1) / slice_rows); }

// Where the counts of a bucket's slices lie, one row each: no two slices share a row, and there are as
// many rows as buckets and slice_rows rows.
__device__ __forceinline__ int count_row(int bucket, int start, int slice_rows) { return bucket + start / slice_rows; }

// (bucket, slice) of further slice number `extra` into s_pick, or (-1, .) if there are no more; the whole
// workgroup.
template <int THREADS>
__device__ __forceinline__ void find_slice(const int *__restrict__ bucket_start, int bins, int slice_rows, int extra,
                                           int *s_pick) {
    constexpr int kMost = (1 << kBucketLowBitsMax) / THREADS;
    const int per = (bins + THREADS - 1) / THREADS;
    const int d0 = (int)threadIdx.x * per;
    int start[kMost + 1];
#pragma unroll
    for (int k = 0; k <= kMost; ++k) start[k] = bucket_start[min(d0 + min(k, per), bins)];
    if (threadIdx.x == 0) s_pick[0] = -1;
    int more = 0;
#pragma unroll
    for (int k = 0; k < kMost; ++k) more += slices_of(start[k + 1] - start[k], slice_rows) - 1;
    int total;
    int first = wide_exclusive_scan<THREADS / 64>(more, &total);  // (synchronises the workgroup)
#pragma unroll
    for (int k = 0; k < kMost; ++k) {
        const int m = slices_of(start[k + 1] - start[k], slice_rows) - 1;
        if (extra >= first && extra < first + m) {
            s_pick[0] = d0 + k;
            s_pick[1] = 1 + extra - first;
        }
        first += m;
    }
    __syncthreads();
}

// Where a bucket's rows come from: the tiles (TILED), a short run of each, or (id, row) pairs in
// bucket order / the ids themselves where the rows are in order.
// seen_s[t] rows of the bucket lie in tiles in front of tile t (none lies in the padding, up to a power of
// two, behind the last tile), and rows[from_s[t] + p] is the row at position p of the bucket if that
// lies in tile t.
template <bool TILED>
struct BucketRows {
    const unsigned *rows;  // TILED
    const int *keys;       // pairs (packed) or ids
    bool packed;
    const int *seen_s, *from_s;
    int top, tile_bits;    // top: half the padded number of tiles
    int u_lo, start;
    // Low digits and rows at COUNT positions inside the bucket.  Nothing here is under a branch, so that
    // the searches advance side by side and all loads are in flight before the first is used (each under
    // its own condition, one after the other: ranks of 1M ids 77 us in bucket_plan_kernel as it was then, 46 so; 25 by now).
    template <int COUNT>
    __device__ __forceinline__ void get(const int (&p)[COUNT], int (&dig)[COUNT], int (&row)[COUNT]) const {
        if (TILED) {
            int t[COUNT];
            unsigned r[COUNT];
#pragma unroll
            for (int k = 0; k < COUNT; ++k) t[k] = 0;
#pragma unroll 1
            for (int step = top; step > 0; step >>= 1) {
#pragma unroll
                for (int k = 0; k < COUNT; ++k) t[k] += seen_s[t[k] + step] <= p[k] ? step : 0;
            }
#pragma unroll
            for (int k = 0; k < COUNT; ++k) r[k] = rows[from_s[t[k]] + p[k]];
#pragma unroll
            for (int k = 0; k < COUNT; ++k) {
                dig[k] = (int)(r[k] >> tile_bits);
                row[k] = (t[k] << tile_bits) + (int)(r[k] & ((1u << tile_bits) - 1u));
            }
        } else if (packed) {
            int2 kr[COUNT];
#pragma unroll
            for (int k = 0; k < COUNT; ++k) kr[k] = reinterpret_cast<const int2 *>(keys)[(long)start + p[k]];
#pragma unroll
            for (int k = 0; k < COUNT; ++k) {
                dig[k] = kr[k].x - u_lo;
                row[k] = kr[k].y;
            }
        } else {
#pragma unroll
            for (int k = 0; k < COUNT; ++k) {
                dig[k] = keys[(long)start + p[k]] - u_lo;
                row[k] = start + p[k];
            }
        }
    }
};
__host__ __device__ __forceinline__ int padded_tiles(int n_tiles) {
    return n_tiles > 1 ? 2 << (31 - __builtin_clz((unsigned)(n_tiles - 1))) : 1;
}
// Fills seen_s / from_s (padded_tiles entries each) for bucket b; the whole workgroup.  All loads are
// requested before the first is used.
template <int THREADS>
__device__ __forceinline__ void find_rows(const unsigned short *__restrict__ offs, int pitch, int n_tiles, int padded,
                                          int tile_bits, int b, int *seen_s, int *from_s) {
    constexpr int kMost = (THREADS == 512 ? kTilesMax : 256) / THREADS;  // (256 threads serve up to 2^19 rows)
    const int per = (padded + THREADS - 1) / THREADS;
    const int t0 = (int)threadIdx.x * per;
    int a[kMost], c[kMost], sum = 0;
#pragma unroll
    for (int k = 0; k < kMost; ++k) {
        const bool in = k < per && t0 + k < n_tiles;
        // both ends of the tile's run in one load (at a short's alignment)
        typedef unsigned word __attribute__((aligned(2)));
        const unsigned o = *reinterpret_cast<const word *>(offs + (long)(in ? t0 + k : 0) * pitch + b);
        a[k] = in ? (int)(o & 0xffffu) : 0;
        c[k] = in ? (int)(o >> 16) - (int)(o & 0xffffu) : 0;
    }
#pragma unroll
    for (int k = 0; k < kMost; ++k) sum += c[k];
    int total;
    int seen = wide_exclusive_scan<THREADS / 64>(sum, &total);
#pragma unroll
    for (int k = 0; k < kMost; ++k) {
        if (k < per && t0 + k < padded) {
            seen_s[t0 + k] = t0 + k < n_tiles ? seen : 0x7fffffff;
            from_s[t0 + k] = ((t0 + k) << tile_bits) + a[k] - seen;
        }
        seen += c[k];
    }
}
// Arguments the count and the plan kernel share.
struct BucketArgs {
    const int *inv;               // ids, in row order
    const unsigned *rows;         // TILED: the tiles' rows and
    const unsigned short *offs;   // first rows per bucket
    const int *pairs;             // otherwise: (id, row) in bucket order
    const int *bucket_start, *ctl, *num_unq_dev;
    int *part_hist;
    int n, U, high_bits, pitch, n_tiles, padded, tile_bits;
    int more;                     // workgroups for further slices
    int self_slices;              // buckets of more slices than this are counted by bucket_count_kernel
};

// Counts, per voxel (low digit) of its bucket, the rows of one slice of a bucket of more than
// self_slices slices: part_hist[workgroup][*].
template <int THREADS, bool TILED>
__global__ __launch_bounds__(THREADS) void bucket_count_kernel(BucketArgs g, const int *__restrict__ stats) {
    constexpr int kSlice = THREADS * kBktItems;
    extern __shared__ int lds_count[];  // [padded] seen, [padded] from (TILED), [low_bins] counts
    __shared__ int s_pick[2];
    if (TILED && g.ctl[0] == 0) return;
    if (stats[TXS_STAT_NEED_GENERAL] != 0) return;
    const int U = voxel_count(g.U, g.num_unq_dev), low_bits = low_bits_of(U, g.high_bits);
    const int bins = 1 << g.high_bits, low_bins = 1 << low_bits;
    int b = (int)blockIdx.x - g.more, j = 0;
    if (b < 0) {
        find_slice<THREADS>(g.bucket_start, bins, kSlice, (int)blockIdx.x, s_pick);
        b = s_pick[0];
        j = s_pick[1];
        if (b < 0) return;
    }
    const int s = g.bucket_start[b], cnt_b = g.bucket_start[b + 1] - s;
    if (low_bits == 0 || slices_of(cnt_b, kSlice) <= g.self_slices) return;  // (uniform)
    int *seen_s = lds_count, *from_s = lds_count + (TILED ? g.padded : 0), *cnt_s = from_s + (TILED ? g.padded : 0);
    if (TILED) find_rows<THREADS>(g.offs, g.pitch, g.n_tiles, g.padded, g.tile_bits, b, seen_s, from_s);
    for (int k = threadIdx.x; k < low_bins; k += THREADS) cnt_s[k] = 0;
    __syncthreads();
    const bool packed = stats[TXS_STAT_UNSORTED] != 0;
    const BucketRows<TILED> src{g.rows, packed ? g.pairs : g.inv, packed, seen_s, from_s, g.padded >> 1, g.tile_bits,
                                b << low_bits, s};
    const int p0 = j * kSlice + (int)threadIdx.x;
    int at[kBktItems], dig[kBktItems], row[kBktItems];
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) at[it] = min(p0 + it * THREADS, cnt_b - 1);
    src.get(at, dig, row);
#pragma unroll
    for (int it = 0; it < kBktItems; ++it)
        if (p0 + it * THREADS < cnt_b && (unsigned)dig[it] < (unsigned)low_bins) atomicAdd(&cnt_s[dig[it]], 1);
    __syncthreads();
    int *mine = g.part_hist + ((long)(count_row(b, s, kSlice) + j) << low_bits);
    for (int k = threadIdx.x; k < low_bins; k += THREADS) mine[k] = cnt_s[k];
}

// One slice.  Its rows, in input order (a wave owns neighbouring positions), are ranked among those of
// their voxel by wave ballots on the low digit and a 16-bit count per wave and voxel; a scan over
// the counts then gives every voxel's place in the slice, and a bucket of several slices adds what
// the other slices hold.  The rows pass through LDS so that they leave in voxel order, neighbouring
// lanes to neighbouring addresses; ranks leave at once.
// What bounds it is the chain of dependent steps inside a workgroup, about 10 us for a slice (bounds 0.5,
// runs in the tiles 1.5, rows 2-3, ranking 2-3, scans 1.5, slots 1, places and stores 1.5), far more
// than bytes: 66 vector registers, seven waves a SIMD, keep three workgroups of 512 threads on a compute unit.
// Index preparation in all, us a call with its host read, against rows moved to bucket order first and a
// voxel's rows ranked by counting the smaller ones: sweeps 200k 72 -> 52, 1M 93 -> 74, 4M 138 -> 123,
// pillars 1M 95 -> 68, 1M ids of 4 / 50 / 400 rows per voxel 80 -> 62, 93 -> 66, 91 -> 67, 2M of 20,000 Zipf
// voxels (through the general sequence) 201 -> 186, 2000 ids 78 -> 45; ranks of 1M 80 -> 69.
template <int THREADS>
constexpr int plan_stage_ints() { return THREADS * kBktItems + THREADS * kBktItems / 2; }
struct PlanLds {
    int counts, first, step, seen, from, tot, front, ints;  // offsets in ints; counts: shared with the staged rows
};
template <int THREADS>
__host__ __device__ __forceinline__ constexpr PlanLds plan_lds(int low_bins, int padded) {
    const int bins = low_bins > 4 ? low_bins : 4, counts = bins / 2 * (THREADS / 64);
    PlanLds l = {};
    l.first = counts > plan_stage_ints<THREADS>() ? counts : plan_stage_ints<THREADS>();  // [bins] shorts
    l.tot = (l.first + bins / 2 + 3) & ~3;  // [bins] rows in the other slices
    l.front = l.tot + bins;                 // [bins] ... and of those in front
    l.step = l.tot;                         // [bins] (in their place, by the thread that read them)
    l.seen = l.front + bins;
    l.from = l.seen + padded;
    l.ints = l.from + padded;
    return l;
}
// counts and first places are read two words at a time, the other three arrays four
template <int THREADS>
constexpr bool plan_lds_aligned() {
    for (int bits = 0; bits <= kBucketLowBitsMax; ++bits)
        for (int padded = 0; padded <= kTilesMax; padded = padded ? 2 * padded : 1) {
            const PlanLds l = plan_lds<THREADS>(1 << bits, padded);
            if (l.counts % 2 || l.first % 2 || l.tot % 4 || l.front % 4 || l.step % 4) return false;
        }
    return true;
}
static_assert(plan_lds_aligned<256>() && plan_lds_aligned<512>(), "vector accesses lie at their alignment");
template <int THREADS, bool TILED>
__global__ __launch_bounds__(THREADS) void bucket_plan_kernel(
    BucketArgs g, VoxelArgs v, int *__restrict__ perm, int *__restrict__ seg, int *__restrict__ stats,
    long long *__restrict__ ranks) {
    constexpr int kWaves = THREADS / 64, kSlice = THREADS * kBktItems, kWaveRows = 64 * kBktItems;
    constexpr unsigned kHeavyMark = 0x8000u;  // in a first place (at most kSlice) and a staged digit (11 bits)
    static_assert(kSlice < (int)kHeavyMark, "first places leave the mark's bit free");
    extern __shared__ __align__(16) int lds_plan[];
    __shared__ int s_red[kWaves], s_bad[kWaves], s_pick[2];
    // ranks != NULL: the caller wants the rank of every row inside its voxel and nothing else
    // (ingroup_inds): the placement writes ranks[row] in place of the permutation and the ids
    const bool rank_mode = ranks != nullptr;
    const int bins = 1 << g.high_bits;
    // (asked for together: each is a trip to memory)
    int b = (int)blockIdx.x - g.more, j = 0, s = g.bucket_start[max(b, 0)], e = g.bucket_start[max(b, 0) + 1];
    const bool step_aside = stats[TXS_STAT_NEED_GENERAL] != 0, unsorted = stats[TXS_STAT_UNSORTED] != 0;
    const int U = voxel_count(g.U, g.num_unq_dev), low_bits = low_bits_of(U, g.high_bits);
    if (step_aside) return;
    const int low_bins = 1 << low_bits;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (b < 0) {
        find_slice<THREADS>(g.bucket_start, bins, kSlice, (int)blockIdx.x, s_pick);
        b = s_pick[0];
        j = s_pick[1];
        if (b < 0) return;
        s = g.bucket_start[b];
        e = g.bucket_start[b + 1];
    }
    const int u_lo = b << low_bits, u_hi = min(U, u_lo + low_bins);
    if (u_lo >= U) return;  // (uniform; such a bucket has no rows)
    const int cnt_b = e - s, nsl = slices_of(cnt_b, kSlice);
    // what is left per voxel comes from the bucket's first slice (or has been left, where a bucket is a voxel)
    const bool voxels = j == 0 && low_bits > 0;
    if (cnt_b == 0 && !voxels) return;

    const PlanLds l = plan_lds<THREADS>(low_bins, TILED ? g.padded : 0);
    const int quads = max(low_bins, 4) >> 2;
    uint2 *cnt4 = reinterpret_cast<uint2 *>(lds_plan + l.counts), *first4 = reinterpret_cast<uint2 *>(lds_plan + l.first);
    int4 *step4 = reinterpret_cast<int4 *>(lds_plan + l.step), *tot4 = reinterpret_cast<int4 *>(lds_plan + l.tot),
         *front4 = reinterpret_cast<int4 *>(lds_plan + l.front);
    const unsigned short *first_s = reinterpret_cast<const unsigned short *>(first4);
    const int *step_s = lds_plan + l.step;
    int *tot_s = lds_plan + l.tot, *front_s = lds_plan + l.front;
    int *seen_s = lds_plan + l.seen, *from_s = lds_plan + l.from;

    const int q = threadIdx.x;  // this thread's four voxels: low digits 4 q .. 4 q + 3
    for (int k = threadIdx.x; k < kWaves * quads; k += THREADS) cnt4[k] = make_uint2(0u, 0u);
    if (nsl > 1 && q < quads) {
        tot4[q] = make_int4(0, 0, 0, 0);
        front4[q] = make_int4(0, 0, 0, 0);
    }
    if (TILED && cnt_b > 0) find_rows<THREADS>(g.offs, g.pitch, g.n_tiles, g.padded, g.tile_bits, b, seen_s, from_s);
    __syncthreads();
    const BucketRows<TILED> src{g.rows, unsorted ? g.pairs : g.inv, unsorted, seen_s, from_s, g.padded >> 1, g.tile_bits,
                                u_lo, s};
    const int my_s = j * kSlice, my_e = min(cnt_b, my_s + kSlice);  // the slice's positions in the bucket
    const int w_s = my_s + w * kWaveRows;
    const unsigned short *wc = reinterpret_cast<const unsigned short *>(cnt4 + w * quads);
    int dig[kBktItems], row[kBktItems], turn[kBktItems];
    if (cnt_b > 0) {  // (uniform)
        int at[kBktItems];
#pragma unroll
        for (int it = 0; it < kBktItems; ++it) at[it] = min(w_s + it * 64 + lane, cnt_b - 1);
        src.get(at, dig, row);
        // ---- rank inside the wave
#pragma unroll
        for (int it = 0; it < kBktItems; ++it)
            if (w_s + it * 64 + lane >= my_e || (unsigned)dig[it] >= (unsigned)low_bins) dig[it] = -1;
        if (w_s < my_e) wave_rank<kBktItems>(dig, 0, low_bits, reinterpret_cast<unsigned *>(cnt4 + w * quads), turn);  // (uniform in a wave)
    }
    // ---- several slices: counts of the bucket's voxels in the other slices, and in those in front
    if (nsl > 1 && low_bits == 0) {
        if (threadIdx.x == 0) {
            tot_s[0] = cnt_b - (my_e - my_s);
            front_s[0] = my_s;
        }
    } else if (nsl > g.self_slices) {
        // sums over the per-slice counts of the bucket's workgroups, four loads in flight per thread
        const int total = nsl << low_bits;
        constexpr int kGather = 4;
        for (int i0 = threadIdx.x; i0 < total; i0 += THREADS * kGather) {
            int c[kGather];
#pragma unroll
            for (int r = 0; r < kGather; ++r) {
                const int i = min(i0 + r * THREADS, total - 1), k = i >> low_bits;
                c[r] = g.part_hist[((long)(count_row(b, s, kSlice) + k) << low_bits) + (i & (low_bins - 1))];
            }
#pragma unroll
            for (int r = 0; r < kGather; ++r) {
                const int i = i0 + r * THREADS, d = i & (low_bins - 1), k = i >> low_bits;
                if (i >= total || c[r] == 0 || k == j) continue;
                atomicAdd(&tot_s[d], c[r]);
                if (k < j) atomicAdd(&front_s[d], c[r]);
            }
        }
    } else if (nsl > 1) {
        // the bucket's other rows once more, four in flight per thread
        constexpr int kAgain = 4;
        const int others = cnt_b - (my_e - my_s);
        for (int i0 = threadIdx.x; i0 < others; i0 += THREADS * kAgain) {
            int at[kAgain], d[kAgain], ignored_rows[kAgain];
#pragma unroll
            for (int r = 0; r < kAgain; ++r) {
                const int i = min(i0 + r * THREADS, others - 1);
                at[r] = i < my_s ? i : i + kSlice;
            }
            src.get(at, d, ignored_rows);
#pragma unroll
            for (int r = 0; r < kAgain; ++r) {
                if (i0 + r * THREADS >= others || (unsigned)d[r] >= (unsigned)low_bins) continue;
                atomicAdd(&tot_s[d[r]], 1);
                if (i0 + r * THREADS < my_s) atomicAdd(&front_s[d[r]], 1);
            }
        }
    }
    __syncthreads();
    // ---- counts per wave -> rows of the waves in front; scans over the voxels of the slice's counts
    // and (the same where there is one slice) of the bucket's
    uint2 run = make_uint2(0u, 0u);
    int4 more = make_int4(0, 0, 0, 0);
    if (q < quads) {
#pragma unroll
        for (int k = 0; k < kWaves; ++k) {
            const uint2 c = cnt4[k * quads + q];
            cnt4[k * quads + q] = run;
            run.x += c.x;
            run.y += c.y;
        }
        if (nsl > 1) more = tot4[q];
    }
    const int c[4] = {(int)(run.x & 0xffff), (int)(run.x >> 16), (int)(run.y & 0xffff), (int)(run.y >> 16)};
    const int all[4] = {c[0] + more.x, c[1] + more.y, c[2] + more.z, c[3] + more.w};
    int placed, ignored;
    int at = wide_exclusive_scan<kWaves>(c[0] + c[1] + c[2] + c[3], &placed);
    int at_all = nsl > 1 ? wide_exclusive_scan<kWaves>(all[0] + all[1] + all[2] + all[3], &ignored) : at;
    {
        int4 front = make_int4(0, 0, 0, 0);
        if (nsl > 1 && q < quads) front = front4[q];
        const int in_front[4] = {front.x, front.y, front.z, front.w};
        int first[4], step[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int u = u_lo + 4 * q + k;
            first[k] = at | (all[k] > v.heavy_threshold ? (int)kHeavyMark : 0);
            // ranks count from the voxel's first row, positions from the bucket's start
            step[k] = (rank_mode ? 0 : s + at_all) + in_front[k] - at;
            if (voxels && 4 * q + k < low_bins && u < u_hi) {
                v.preSum[u] = s + at_all;
                if (v.cnts_out) v.cnts_out[u] = (long long)all[k];
                if (u == U - 1) v.preSum[U] = g.n;
            }
            at += c[k];
            at_all += all[k];
        }
        if (q < quads) {
            first4[q] = make_uint2((unsigned)first[0] | (unsigned)first[1] << 16, (unsigned)first[2] | (unsigned)first[3] << 16);
            step4[q] = make_int4(step[0], step[1], step[2], step[3]);
        }
    }
    // ---- statistics, special voxels and their slots (first slice only; as plan_special_kernel)
    const bool slots = voxels && v.slot_of != nullptr;
    if (slots) {
        int most = 0;
        bool mismatch = false;
        if (w * 256 < low_bins) {  // (uniform in a wave)
            const int u = u_lo + 4 * q;
            const bool in = 4 * q < low_bins;
            long long given[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) given[k] = v.unq_cnts && in && u + k < u_hi ? v.unq_cnts[u + k] : 0;
            voxel_slots<4>(v, U, u, in ? u_hi : 0, all, stats);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int cnt = in && u + k < u_hi ? all[k] : 0;
                if (v.unq_cnts) mismatch |= given[k] != (long long)cnt;
                most = max(most, cnt);
            }
        }
        most = wave_max_i32(most);
        const bool any_mismatch = __ballot(mismatch) != 0ull;
        if (lane == 0) {
            s_red[w] = most;
            s_bad[w] = any_mismatch;
        }
    }
    __syncthreads();
    if (slots && threadIdx.x == 0) {
        int m = 0, bad = 0;
        for (int k = 0; k < kWaves; ++k) {
            m = max(m, s_red[k]);
            bad |= s_bad[k];
        }
        if (m > 0) atomicMax(&stats[TXS_STAT_MAX_CNT], m);
        if (bad) stats[TXS_STAT_COUNT_MISMATCH] = 1;
    }
    if (cnt_b == 0) return;  // (uniform)
    // ---- places
    int step[kBktItems];
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) {
        const int d = max(dig[it], 0);
        const unsigned f = first_s[d];
        step[it] = rank_mode ? step_s[d] : (int)(f & kHeavyMark);
        turn[it] += (int)(f & (kHeavyMark - 1u)) + (int)wc[d];
    }
    if (rank_mode) {
#pragma unroll
        for (int it = 0; it < kBktItems; ++it)
            if (dig[it] >= 0 && (unsigned)row[it] < (unsigned)g.n) ranks[row[it]] = (long long)(step[it] + turn[it]);
        return;
    }
    __syncthreads();  // (the rows take the counts' space)
    int *row_s = lds_plan + l.counts;
    unsigned short *dig_s = reinterpret_cast<unsigned short *>(row_s + kSlice);
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) {
        if (dig[it] < 0) continue;
        row_s[turn[it]] = row[it];
        dig_s[turn[it]] = (unsigned short)(dig[it] | step[it]);
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) {
        dig[it] = dig_s[it * THREADS + (int)threadIdx.x];  // (what lies behind the last row is not used)
        row[it] = row_s[it * THREADS + (int)threadIdx.x];
    }
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) turn[it] = step_s[min(dig[it] & (int)(kHeavyMark - 1u), max(low_bins, 4) - 1)];
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) {
        const int p = it * THREADS + (int)threadIdx.x, dst = turn[it] + p;
        if (p >= placed || dst < s || dst >= e) continue;
        seg[dst] = (u_lo + (dig[it] & (int)(kHeavyMark - 1u))) | ((dig[it] & (int)kHeavyMark) ? kSpecialBit : 0);
        if (unsorted) perm[dst] = row[it];
    }
}

__global__ void stats_clear_kernel(int *__restrict__ stats) {
    if (threadIdx.x < TXS_STATS_LEN) stats[threadIdx.x] = 0;
}

// Heavy voxel number blockIdx.x of the list becomes an ordinary one again: the special bit
// comes off its positions and it gives up its slot.
__global__ void demote_heavy_kernel(const int *__restrict__ preSum, int *__restrict__ seg,
                                    int *__restrict__ slot_of, const int *__restrict__ heavy_ids,
                                    int N, int U, int *__restrict__ stats) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        stats[TXS_STAT_NUM_HEAVY] = 0;
        stats[TXS_STAT_NUM_SPECIAL] = stats[TXS_STAT_NUM_EMPTY];
    }
    const int u = heavy_ids[blockIdx.x];
    if ((unsigned)u >= (unsigned)U) return;
    const int lo = max(preSum[u], 0), hi = min(preSum[u + 1], N);
    for (int p = lo + (int)threadIdx.x; p < hi; p += (int)blockDim.x) seg[p] &= kIdMask;
    if (threadIdx.x == 0) slot_of[u] = -1;
}

int plan_general(const int32_t *unq_inv, int64_t num_total, int64_t num_unq, int32_t heavy_threshold,
                 const int64_t *unq_cnts, int32_t *plan_ws, int32_t *perm, int32_t *seg, int32_t *preSum,
                 int32_t *slot_of, int32_t *heavy_ids, int32_t *stats, const int *num_unq_dev, long long *cnts_out,
                 void *stream);

// Workspace of the bucket sort, in int32 entries from the (8-byte aligned) start.
struct PlanLayout {
    bool tiled;
    TileSplit split;                     // tiled
    int high_bits, hist_tiles, slice_threads;
    int64_t slices_more;                 // an upper bound of the further slices of all buckets
    int64_t rows, offs;                  // tiled; the other route starts with the (id, row) pairs
    int64_t hist, scan_ws;               // otherwise
    int64_t tile_flags, bucket_start, ctl, part_hist, len;
};
// ranks: for the ranks alone (which need no more than the plan does)
PlanLayout plan_layout(int64_t n, int bits, bool ranks) {
    PlanLayout l = {};
    l.tiled = n <= kTiledRows;
    int64_t at = 0;
    auto take = [&at](int64_t entries) {
        const int64_t here = at;
        at += entries;
        return here;
    };
    if (l.tiled) {
        l.split = tile_split((long)n, bits);
        l.high_bits = l.split.high_bits;
        l.rows = take(n);
        at = (at + 1) & ~(int64_t)1;
        l.offs = take((int64_t)l.split.tiles * l.split.pitch / 2);
        l.tile_flags = take(l.split.tiles);
    } else {
        take(2 * n);
        // the bucket digit has 9 bits (narrower, and the buckets of a spatially sorted id space get too
        // uneven; wider, and a tile sends too few rows to a bucket for the scatter to write whole cache
        // lines) and the low digit takes the rest, at most 11
        l.high_bits = bits <= kBucketLowBitsMax ? bits : max(kBucketHighBits, bits - kBucketLowBitsMax);
        l.hist_tiles = (int)((n + kHistThreads * kHistItems - 1) / (kHistThreads * kHistItems));
        const int64_t hist = ((int64_t)1 << l.high_bits) * l.hist_tiles + 1;
        l.hist = take(hist);
        l.scan_ws = take(scan_tiles((long)hist) + 17);
        l.tile_flags = take(l.hist_tiles);
    }
    l.bucket_start = take(((int64_t)1 << l.high_bits) + 1);
    l.ctl = take(1);
    const int low_bits = bits - l.high_bits;
    l.slice_threads = slice_threads_for((long)n, low_bits, ranks);
    l.slices_more = n / (l.slice_threads * kBktItems);
    l.part_hist = take(low_bits > 0 ? (((int64_t)1 << l.high_bits) + l.slices_more) << low_bits : 0);
    l.len = at;
    return l;
}

}  // namespace

extern "C" {

int txs_get_presum(const int32_t *unq_inv, int32_t *preSum, int64_t num_total, int64_t num_presum,
                   void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_presum)) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!unq_inv || !preSum) return TXS_ERR_INVALID_ARG;
    get_presum_kernel<<<dim3(blocks_for(num_total)), dim3(kThreads), 0, (hipStream_t)stream>>>(
        unq_inv, preSum, num_total, num_presum);
    return status_of(hipGetLastError());
}

int txs_plan_check(const int32_t *unq_inv, int64_t num_total, int64_t num_unq, int32_t *stats,
                   void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_unq) || !stats) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!unq_inv) return TXS_ERR_INVALID_ARG;
    plan_check_kernel<<<dim3(blocks_for(num_total)), dim3(kThreads), 0, (hipStream_t)stream>>>(
        unq_inv, num_total, (int)num_unq, stats);
    return status_of(hipGetLastError());
}

int64_t txs_sort_workspace_len(int64_t num_total, int64_t num_unq) {
    const int64_t tiles = (num_total + kSortTile - 1) / kSortTile;
    const int64_t hist = 256 * (tiles > 0 ? tiles : 1);
    (void)num_unq;
    // two ping-pong arrays, the digit-major histogram, and the scan workspace
    return 2 * num_total + hist + scan_tiles(hist + 1) + 17;
}

int txs_plan_sort(const int32_t *unq_inv, int64_t num_total, int64_t num_unq, const int32_t *stats,
                  int32_t *perm, int32_t *keys, int32_t *sort_ws, void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_unq)) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!unq_inv || !stats || !perm || !keys || !sort_ws || num_unq <= 0) return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    const long n = num_total;
    const int n_tiles = (int)((n + kSortTile - 1) / kSortTile);
    const long hist_len = 256L * n_tiles;
    int *tmp_keys = sort_ws;
    int *tmp_vals = sort_ws + n;
    int *hist = sort_ws + 2 * n;
    int *scan_ws = hist + hist_len;

    copy_if_sorted_kernel<<<dim3(blocks_for(n)), dim3(kThreads), 0, st>>>(unq_inv, n, stats, keys);
    const int bits = radix_bits(num_unq);
    const int passes = (bits + 7) / 8;
    const int rbits = (bits + passes - 1) / passes;
    const int *kin = unq_inv;
    const int *vin = nullptr;  // identity
    for (int p = 0; p < passes; ++p) {
        const bool to_final = ((passes - 1 - p) % 2) == 0;
        int *kout = to_final ? keys : tmp_keys;
        int *vout = to_final ? perm : tmp_vals;
        const int shift = p * rbits;
        sort_hist_kernel<<<dim3(n_tiles), dim3(kThreads), 0, st>>>(kin, n, shift, rbits, hist, n_tiles,
                                                                  stats);
        const long used = (1L << rbits) * n_tiles;
        if (exclusive_scan(hist, used, hist, used, scan_ws, st) != hipSuccess) return TXS_ERR_LAUNCH;
        sort_scatter_kernel<<<dim3(n_tiles), dim3(kThreads), 0, st>>>(kin, vin, kout, vout, n, shift,
                                                                     rbits, hist, n_tiles, stats);
        kin = kout;
        vin = vout;
    }
    return status_of(hipGetLastError());
}

int txs_plan_presum(const int32_t *sorted_keys, int64_t num_total, int64_t num_unq, int32_t *preSum,
                    void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_unq) || !preSum) return TXS_ERR_INVALID_ARG;
    if (num_total > 0 && !sorted_keys) return TXS_ERR_INVALID_ARG;
    presum_from_sorted_kernel<<<dim3(blocks_for(num_total + 1)), dim3(kThreads), 0,
                                (hipStream_t)stream>>>(sorted_keys, num_total, (int)num_unq, preSum);
    // long runs of empty voxels, one workgroup per 256 ids (only where there can be any)
    if (num_unq + 1 >= kGapBlock)
        presum_gap_blocks_kernel<<<dim3((unsigned)((num_unq + 1) / kGapBlock)), dim3(kGapBlock), 0,
                                   (hipStream_t)stream>>>(sorted_keys, num_total, (int)num_unq, preSum);
    return status_of(hipGetLastError());
}

int txs_plan_special(const int32_t *preSum, int64_t num_unq, int32_t heavy_threshold,
                     const int64_t *unq_cnts, int32_t *slot_of, int32_t *heavy_ids, int32_t *stats,
                     const int32_t *num_unq_dev, int64_t *cnts_out, void *stream) {
    if (!fits_i32(num_unq) || !preSum || !stats || heavy_threshold < kChunk) return TXS_ERR_INVALID_ARG;
    if (num_unq == 0) return TXS_OK;
    if (!slot_of || !heavy_ids) return TXS_ERR_INVALID_ARG;
    plan_special_kernel<<<dim3(blocks_for(num_unq, kSpecialThreads)), dim3(kSpecialThreads), 0,
                          (hipStream_t)stream>>>(
        preSum, (int)num_unq, heavy_threshold, (const long long *)unq_cnts, slot_of, heavy_ids, stats,
        num_unq_dev, (long long *)cnts_out);
    return status_of(hipGetLastError());
}

int txs_plan_seg_flag(int32_t *keys_to_seg, int64_t num_total, int64_t num_unq,
                      const int32_t *slot_of, void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_unq)) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!keys_to_seg || !slot_of) return TXS_ERR_INVALID_ARG;
    seg_flag_kernel<<<dim3(blocks_for(num_total)), dim3(kThreads), 0, (hipStream_t)stream>>>(
        keys_to_seg, num_total, (int)num_unq, slot_of, keys_to_seg);
    return status_of(hipGetLastError());
}

int txs_plan_demote_heavy(const int32_t *preSum, int32_t *seg, int32_t *slot_of, const int32_t *heavy_ids,
                          int64_t num_heavy, int64_t num_total, int64_t num_unq, int32_t *stats, void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_unq) || num_heavy < 0 || num_heavy > num_unq)
        return TXS_ERR_INVALID_ARG;
    if (num_heavy == 0) return TXS_OK;
    if (!preSum || !seg || !slot_of || !heavy_ids || !stats) return TXS_ERR_INVALID_ARG;
    demote_heavy_kernel<<<dim3((unsigned)num_heavy), dim3(128), 0, (hipStream_t)stream>>>(
        preSum, seg, slot_of, heavy_ids, (int)num_total, (int)num_unq, stats);
    return status_of(hipGetLastError());
}

int txs_plan_seg_from_presum(const int32_t *preSum, int64_t num_total, int64_t num_unq,
                             const int32_t *slot_of, int32_t *seg, void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_unq)) return TXS_ERR_INVALID_ARG;
    if (num_total == 0) return TXS_OK;
    if (!preSum || !slot_of || !seg || num_unq <= 0) return TXS_ERR_INVALID_ARG;
    seg_from_presum_kernel<<<dim3(blocks_for(num_total)), dim3(kThreads), 0, (hipStream_t)stream>>>(
        preSum, num_total, (int)num_unq, slot_of, seg);
    return status_of(hipGetLastError());
}

int64_t txs_plan_workspace_len(int64_t num_total, int64_t num_unq) {
    if (!fits_i32(num_total) || !fits_i32(num_unq)) return -1;
    const int64_t general = txs_sort_workspace_len(num_total, num_unq);
    const int bits = radix_bits((int)(num_unq > 1 ? num_unq : 1));
    if (bits > kBucketBitsMax) return general;
    const PlanLayout l = plan_layout(num_total, bits, false);
    return general > l.len ? general : l.len;
}

int txs_plan_build_general(const int32_t *unq_inv, int64_t num_total, int64_t num_unq, int32_t heavy_threshold,
                           const int64_t *unq_cnts, int32_t *plan_ws, int32_t *perm, int32_t *seg,
                           int32_t *preSum, int32_t *slot_of, int32_t *heavy_ids, int32_t *stats, void *stream) {
    return plan_general(unq_inv, num_total, num_unq, heavy_threshold, unq_cnts, plan_ws, perm, seg, preSum, slot_of,
                        heavy_ids, stats, nullptr, nullptr, stream);
}

int txs_plan_build(const int32_t *unq_inv, int64_t num_total, int64_t num_unq, int32_t heavy_threshold,
                   const int64_t *unq_cnts, int32_t *plan_ws, int32_t *perm, int32_t *seg, int32_t *preSum,
                   int32_t *slot_of, int32_t *heavy_ids, int32_t *stats, void *stream) {
    return txs_detail::plan_build(unq_inv, num_total, num_unq, heavy_threshold, unq_cnts, plan_ws, perm, seg, preSum,
                                  slot_of, heavy_ids, stats, nullptr, nullptr, nullptr, nullptr, stream);
}

int txs_plan_build_i64(const int64_t *ids, int32_t *unq_inv, int64_t num_total, int64_t num_unq,
                       int32_t heavy_threshold, const int64_t *unq_cnts, int32_t *plan_ws, int32_t *perm, int32_t *seg,
                       int32_t *preSum, int32_t *slot_of, int32_t *heavy_ids, int32_t *stats, void *stream) {
    if (num_total > 0 && !ids) return TXS_ERR_INVALID_ARG;
    return txs_detail::plan_build(unq_inv, num_total, num_unq, heavy_threshold, unq_cnts, plan_ws, perm, seg, preSum,
                                  slot_of, heavy_ids, stats, nullptr, nullptr, nullptr, (const long long *)ids, stream);
}

}  // extern "C"

namespace {

// num_unq_dev, cnts_out: as for txs_plan_special
int plan_general(const int32_t *unq_inv, int64_t num_total, int64_t num_unq, int32_t heavy_threshold,
                 const int64_t *unq_cnts, int32_t *plan_ws, int32_t *perm, int32_t *seg, int32_t *preSum,
                 int32_t *slot_of, int32_t *heavy_ids, int32_t *stats, const int *num_unq_dev, long long *cnts_out,
                 void *stream) {
    if (!fits_i32(num_total) || !fits_i32(num_unq) || !stats || !preSum || heavy_threshold < kChunk)
        return TXS_ERR_INVALID_ARG;
    const long n = num_total;
    const int U = (int)num_unq;
    if (n > 0 && (!unq_inv || !plan_ws || !perm || !seg)) return TXS_ERR_INVALID_ARG;
    if (U > 0 && ((slot_of == nullptr) != (heavy_ids == nullptr))) return TXS_ERR_INVALID_ARG;
    // order/range flags, three-kernel radix passes, CSR offsets, special table, flags
    int rc = txs_plan_check(unq_inv, n, U, stats, stream);
    if (rc == TXS_OK && n > 0 && U > 0) rc = txs_plan_sort(unq_inv, n, U, stats, perm, seg, plan_ws, stream);
    if (rc == TXS_OK) rc = txs_plan_presum(seg, U > 0 ? n : 0, U, preSum, stream);
    if (slot_of == nullptr) return rc;  // order and offsets only
    if (rc == TXS_OK)
        rc = txs_plan_special(preSum, U, heavy_threshold, unq_cnts, slot_of, heavy_ids, stats, num_unq_dev,
                              (int64_t *)cnts_out, stream);
    if (rc == TXS_OK) rc = txs_plan_seg_flag(seg, U > 0 ? n : 0, U, slot_of, stream);
    return rc;
}

}  // namespace

// txs_plan_build, or with `ranks` the in-voxel rank of every row and no special-voxel table.
// Ranks are written by the bucket kernels only: txs_detail::plan_writes_ranks tells a caller
// whether they apply to the extents (otherwise it ranks from the plan this call leaves).
bool txs_detail::plan_writes_ranks(long num_total, long num_unq) {
    const int bits = radix_bits(num_unq > 1 ? num_unq : 1);
    return num_total > 0 && num_unq > 0 && bits <= kBucketBitsMax;
}

// Up to kMappedRows rows the lookup on the way saves a pass and a launch (sweeps, pillars, clusters, grouped rows; looked up
// on the way / apart: 140k keys 79 - 89 / 84 - 92 us, 1M 91 - 115 / 97 - 118, 2M 105 - 127 / 110 - 131).  Above, in tiles of 8192,
// a thread would hold 16 rows' keys and cells: 199 registers, one workgroup on a compute unit.  A kernel for the ids
// alone, which the sorting kernel then reads, is faster there: 2.2M keys in
// 2^20 139 -> 132 us, 8M 295 -> 276, 16M 582 -> 517 (8M of 2048 keys 265 -> 238, 16M 462 -> 405).
bool txs_detail::plan_takes_map(long num_total, long num_unq) {
    return num_total > 0 && num_total <= kMappedRows && num_unq > 0 && radix_bits((int)(num_unq > 1 ? num_unq : 1)) <= kBucketBitsMax;
}

namespace {

// map (may be NULL): see plan_build_mapped
int build(const int32_t *unq_inv, int64_t num_total, int64_t num_unq, int32_t heavy_threshold, const int64_t *unq_cnts,
          int32_t *plan_ws, int32_t *perm, int32_t *seg, int32_t *preSum, int32_t *slot_of, int32_t *heavy_ids,
          int32_t *stats, long long *ranks, const int *num_unq_dev, long long *cnts_out, const long long *ids64,
          const KeyMap *map, void *stream) {
    if (map && !txs_detail::plan_takes_map(num_total, num_unq)) return TXS_ERR_INVALID_ARG;
    if (!fits_i32(num_total) || !fits_i32(num_unq) || !stats || !preSum || heavy_threshold < kChunk)
        return TXS_ERR_INVALID_ARG;
    hipStream_t st = (hipStream_t)stream;
    const long n = num_total;
    const int U = (int)num_unq;
    if (n > 0 && (!unq_inv || !plan_ws || !perm || !seg)) return TXS_ERR_INVALID_ARG;
    if (U > 0 && ((slot_of == nullptr) != (heavy_ids == nullptr))) return TXS_ERR_INVALID_ARG;
    if (((uintptr_t)plan_ws & 7u) != 0) return TXS_ERR_INVALID_ARG;
    if (slot_of == nullptr) heavy_threshold = 0x7fffffff;  // no special voxels: no flag bit in seg
    const int bits = radix_bits(U > 1 ? U : 1);
    if (n == 0 || U == 0 || (num_unq_dev && bits > kBucketBitsMax)) {
        // the general sequence adds to `stats`, which this call promises to initialise itself
        // where there is nothing to sort, and the unique path always
        stats_clear_kernel<<<dim3(1), dim3(64), 0, st>>>(stats);
        if (hipGetLastError() != hipSuccess) return TXS_ERR_LAUNCH;
    }
    int *ids32 = const_cast<int *>(unq_inv);  // written only where ids64 is given
    if (n == 0 || U == 0 || bits > kBucketBitsMax) {
        if (ids64 && n > 0) narrow_ids_kernel<<<dim3(blocks_for(n)), dim3(kThreads), 0, st>>>(ids64, n, ids32);
        return plan_general(unq_inv, num_total, num_unq, heavy_threshold, unq_cnts, plan_ws, perm, seg, preSum, slot_of,
                            heavy_ids, stats, num_unq_dev, cnts_out, stream);
    }
    // (the attribute belongs to the current device's copy of a kernel: once per device)
    constexpr int kMaxDevices = 64;
    static std::atomic<bool> lds_allowed[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return TXS_ERR_LAUNCH;
    if (!lds_allowed[dev].load(std::memory_order_acquire)) {
        for (const void *k : {reinterpret_cast<const void *>(bucket_scatter_kernel),
                              reinterpret_cast<const void *>(bucket_plan_kernel<512, true>)})
            if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024) != hipSuccess)
                return TXS_ERR_LAUNCH;
        lds_allowed[dev].store(true, std::memory_order_release);
    }
    const PlanLayout l = plan_layout(n, bits, ranks != nullptr);
    const int low_most = bits - l.high_bits;  // (of the voxels there are at most; the kernels know their number)
    int *bucket_start = plan_ws + l.bucket_start;
    const int threads = l.slice_threads;
    BucketArgs g = {};
    g.inv = unq_inv;
    g.bucket_start = bucket_start;
    g.ctl = plan_ws + l.ctl;
    g.num_unq_dev = num_unq_dev;
    g.part_hist = plan_ws + l.part_hist;
    g.n = (int)n;
    g.U = U;
    g.high_bits = l.high_bits;
    g.more = (int)l.slices_more;
    const VoxelArgs voxels = {heavy_threshold, (const long long *)unq_cnts, preSum, slot_of, heavy_ids, cnts_out};
    if (l.tiled) {
        auto rows = reinterpret_cast<unsigned *>(plan_ws + l.rows);
        auto offs = reinterpret_cast<unsigned short *>(plan_ws + l.offs);
        int *tile_flags = plan_ws + l.tile_flags, *ctl = plan_ws + l.ctl;
        const TileSplit &t = l.split;
        const int tile_threads = t.tile_bits == 10 ? 256 : 512;
        const size_t bins = (size_t)t.pitch - 4;
        const size_t lds = 2 * bins + max(2 * bins * (tile_threads / 64), sizeof(int) << t.tile_bits);
        auto sort_tiles = [&](auto ids, int more) {
            using K = std::remove_const_t<std::remove_pointer_t<decltype(ids)>>;
            auto kernel = t.tile_bits == 10   ? tile_sort_kernel<256, 4, K>
                          : t.tile_bits == 11 ? tile_sort_kernel<512, 4, K>
                                              : tile_sort_kernel<512, 8, K>;
            if constexpr (!std::is_same_v<K, KeyMap>)
                if (t.tile_bits == 13) kernel = tile_sort_kernel<512, 16, K>;
            kernel<<<dim3(t.tiles + more), dim3(tile_threads), lds, st>>>(ids, n, t.tiles, U, t.high_bits, rows, offs, t.pitch,
                                                                          tile_flags, ids32, stats, ctl, num_unq_dev);
        };
        if (map) sort_tiles(*map, map_parts(*map));
        else if (ids64) sort_tiles(ids64, 0);
        else sort_tiles(unq_inv, 0);
        bucket_start_kernel<<<dim3(((1 << t.high_bits) + kStartOwned) / kStartOwned), dim3(kStartThreads), 0, st>>>(
            offs, t.pitch, t.tiles, (int)n, U, t.high_bits, (threads == 512 ? 1 : kSelfSlices) * threads * kBktItems, tile_flags, bucket_start, stats, ctl, num_unq_dev,
            voxels);
        g.rows = rows;
        g.offs = offs;
        g.pitch = t.pitch;
        g.n_tiles = t.tiles;
        g.padded = padded_tiles(t.tiles);
        g.tile_bits = t.tile_bits;
        g.self_slices = threads == 512 ? 1 : kSelfSlices;
    } else {
        const int high_bins = 1 << l.high_bits;
        int *hist = plan_ws + l.hist, *tile_flags = plan_ws + l.tile_flags, *scan_ws = plan_ws + l.scan_ws;
        const long used = (long)high_bins * l.hist_tiles;
        if (ids64)
            bucket_hist_kernel<long long><<<dim3(l.hist_tiles), dim3(kHistThreads), 0, st>>>(
                ids64, n, U, l.high_bits, hist, tile_flags, l.hist_tiles, ids32, num_unq_dev);
        else
            bucket_hist_kernel<int><<<dim3(l.hist_tiles), dim3(kHistThreads), 0, st>>>(
                unq_inv, n, U, l.high_bits, hist, tile_flags, l.hist_tiles, nullptr, num_unq_dev);
        // one entry more than the histogram: it receives the total, the end of the last bucket.  A
        // bucket's first entry (that of tile 0) is where it starts.
        if (exclusive_scan(hist, used, hist, used + 1, scan_ws, st, bucket_start, l.hist_tiles) != hipSuccess)
            return TXS_ERR_LAUNCH;
        const size_t lds = (size_t)high_bins * sizeof(int) + max((size_t)kHistWaves * high_bins * sizeof(int),
                                                                 (size_t)kHistThreads * kHistItems * sizeof(int2));
        bucket_scatter_kernel<<<dim3(l.hist_tiles), dim3(kHistThreads), lds, st>>>(
            unq_inv, n, U, l.high_bits, hist, tile_flags, l.hist_tiles, bucket_start, stats,
            reinterpret_cast<int2 *>(plan_ws), num_unq_dev);
        // (a bucket is a voxel where there are at most 2^11 of them, which the host may not know)
        if (bits <= kBucketLowBitsMax || num_unq_dev)
            bucket_voxels_kernel<<<dim3((high_bins + 63) / 64), dim3(64), 0, st>>>(bucket_start, (int)n, U, l.high_bits,
                                                                                  stats, num_unq_dev, voxels);
        g.pairs = plan_ws;
        g.self_slices = 1;
    }
    // A bucket so full that its workgroups would run long after all others have finished (only a few
    // voxels holding most of the rows do that) sends the call to the general sequence.
    const int low_bins = 1 << low_most, tiles = l.tiled ? g.padded : 0;
    const dim3 grid((unsigned)(((int64_t)1 << l.high_bits) + l.slices_more));
    const size_t lds_count = sizeof(int) * (size_t)(low_bins + 2 * tiles);
    auto place = [&](auto count_kernel, auto plan_kernel, size_t lds) {
        if (low_most > 0) count_kernel<<<grid, dim3(threads), lds_count, st>>>(g, stats);
        plan_kernel<<<grid, dim3(threads), lds, st>>>(g, voxels, perm, seg, stats, ranks);
    };
    if (!l.tiled)
        place(bucket_count_kernel<512, false>, bucket_plan_kernel<512, false>, sizeof(int) * plan_lds<512>(low_bins, 0).ints);
    else if (threads == 512)
        place(bucket_count_kernel<512, true>, bucket_plan_kernel<512, true>, sizeof(int) * plan_lds<512>(low_bins, tiles).ints);
    else
        place(bucket_count_kernel<256, true>, bucket_plan_kernel<256, true>, sizeof(int) * plan_lds<256>(low_bins, tiles).ints);
    return status_of(hipGetLastError());
}

}  // namespace

int txs_detail::plan_build(const int32_t *unq_inv, int64_t num_total, int64_t num_unq, int32_t heavy_threshold,
                           const int64_t *unq_cnts, int32_t *plan_ws, int32_t *perm, int32_t *seg,
                           int32_t *preSum, int32_t *slot_of, int32_t *heavy_ids, int32_t *stats,
                           long long *ranks, const int *num_unq_dev, long long *cnts_out,
                           const long long *ids64, void *stream) {
    return build(unq_inv, num_total, num_unq, heavy_threshold, unq_cnts, plan_ws, perm, seg, preSum, slot_of, heavy_ids,
                 stats, ranks, num_unq_dev, cnts_out, ids64, nullptr, stream);
}

int txs_detail::plan_build_mapped(const KeyMap &map, int32_t *unq_inv, int64_t num_total, int64_t num_unq,
                                  int32_t heavy_threshold, int32_t *plan_ws, int32_t *perm, int32_t *seg,
                                  int32_t *preSum, int32_t *slot_of, int32_t *heavy_ids, int32_t *stats,
                                  long long *cnts_out, void *stream) {
    return build(unq_inv, num_total, num_unq, heavy_threshold, nullptr, plan_ws, perm, seg, preSum, slot_of, heavy_ids,
                 stats, nullptr, map.num_unq, cnts_out, nullptr, &map, stream);
}
