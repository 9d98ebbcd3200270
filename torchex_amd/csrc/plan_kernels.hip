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

#include "txs_common.h"

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
// For up to 2^22 voxels the whole index preparation is four kernels and a scan:
//   (1) bucket_hist_kernel: per tile of 2048 - 8192 rows, the histogram of the HIGH digit of the
//       voxel id (the "bucket") and the tile's order / range flags;
//   (2) exclusive scan of the digit-major histogram;
//   (3) bucket_scatter_kernel: flags of the whole input and the stable scatter of (id, row) pairs
//       by bucket (wave-ballot ranking, then through LDS);
//   (4) bucket_count_kernel: a bucket is cut into slices of 4096 rows, one workgroup per slice;
//       where there are several, each counts its slice's rows per voxel (LOW digit, <= 11 bits)
//       in LDS and writes the counts out;
//   (5) bucket_plan_kernel: the same workgroups count their slice again, or add up the counts of
//       their bucket's slices (a voxel's count, and its rows in the slices in front), which at the
//       same time yields the bucket's share of everything else the plan holds: CSR offsets,
//       per-voxel counts (checked against the caller's), the special-voxel table and its slots,
//       max_cnt; then each places its slice by the low digit, stably, writing the flagged
//       per-position ids next to the permutation.
// Ids of at most 11 bits need no low digit: (3) already gives the final order, and the
// elementwise kernels used by the general sequence finish the plan.
// Measured alternatives (1M ids of 19 bits): an 11-bit bucket digit made the scatter, then without
// staging through LDS, write 16-byte runs and cost 30 us instead of 20; folding the scan into the
// scatter (every workgroup adding up the tile histograms itself) saves two launches but costs
// more than it saves from about 100 tiles on.

#ifndef TXS_BUCKET_HIGH_BITS
#define TXS_BUCKET_HIGH_BITS 9
#endif
constexpr int kBucketHighBits = TXS_BUCKET_HIGH_BITS;
constexpr int kBucketLowBitsMax = 11;   // also the largest high digit
constexpr int kBucketBitsMax = 22;
constexpr int kHistThreads = 512;
// rows per tile of the histogram and scatter kernels: 512 * {4, 8, 16}, the largest that still
// gives every compute unit a tile
int hist_items_for(long n) {
    return n >= 256L * kHistThreads * 16 ? 16 : (n >= 256L * kHistThreads * 8 ? 8 : 4);
}
constexpr int kHistWaves = kHistThreads / 64;
constexpr int kBktThreads = 512;
constexpr int kBktItems = 8;
constexpr int kBktWaves = kBktThreads / 64;
constexpr int kBktSlice = kBktThreads * kBktItems;     // rows one workgroup places
constexpr long kBktGiant = 64L * kBktSlice;            // rows in one bucket beyond which the general sequence runs
// Rows of one voxel in a slice beyond which they are ranked by ballots.  bucket_plan_kernel, us, with
// 64 (and one read at a time) / 63 / 31 / 24 / 21: 1M ids of pillars 37.2 / 29.5 / 22.9 / 22.8 / 22.1, 1M
// ids of 50 rows per voxel 46.3 / 39.6 / 31.0 / 29.7 / 29.4, of 25 rows 33.7 / 30.3 / 28.4 / 27.7 / 27.8, of 10
// rows 20.9 / 17.6 / 18.8 / 20.9 / 21.4, of a sweep 21.5 / 19.5 / 20.8 / 21.8 / 21.9.
constexpr int kLongRun = 24;
constexpr int kMaxLongRuns = kBktSlice / (kLongRun + 1);
static_assert(kMaxLongRuns < 256 && kBktSlice / 64 == 64, "eight bits number a slice's long runs, a wave scans their chunk counts");
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

// hist: [high_bins][n_tiles] digit-major (the order its exclusive scan needs); tile_flags: [n_tiles]
// K = long long: ids as torch.unique returns them, cut to 32 bits and left in `ids32` for the
// kernels that follow (a conversion of its own reads and writes them once more: 16 us of 4M ids,
// 5 us of 1M)
template <int ITEMS, typename K>
__global__ __launch_bounds__(kHistThreads) void bucket_hist_kernel(
    const K *__restrict__ inv, long n, int U_arg, int high_bits, int *__restrict__ hist,
    int *__restrict__ tile_flags, int n_tiles, int *__restrict__ ids32, const int *__restrict__ num_unq_dev) {
    __shared__ int h[1 << kBucketLowBitsMax];
    __shared__ int s_flags;
    const int U = voxel_count(U_arg, num_unq_dev), low_bits = low_bits_of(U, high_bits), high_bins = 1 << high_bits;
    for (int d = threadIdx.x; d < high_bins; d += kHistThreads) h[d] = 0;
    if (threadIdx.x == 0) s_flags = 0;
    __syncthreads();
    const long base = (long)blockIdx.x * (kHistThreads * ITEMS);
    int v[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const long i = base + (long)it * kHistThreads + threadIdx.x;
        v[it] = i < n ? (int)inv[i] : 0x7fffffff;
        if (sizeof(K) == 8 && i < n) ids32[i] = v[it];
    }
    bool bad_range = false, bad_order = false;
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
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

// id at position i: of unq_inv itself (rows in order) or of the (id, row) pairs the bucket scatter wrote
__device__ __forceinline__ int kread(const int *keys, long i, bool packed) {
    return packed ? keys[2 * i] : keys[i];
}

// Stable scatter by the high digit.  hist: the exclusive scan of the digit-major tile histograms.
//   bucket_start [high_bins + 1] (from the scan): first position of every bucket.
//   stats: zero-filled here (workgroup 0), then UNSORTED / OUT_OF_RANGE of the whole input
//   and NEED_GENERAL (a bucket above kBktGiant rows: the bucket kernels step aside; not where so few
//   voxels have so many rows that the low digit has next to nothing left).
// Rows already in order are not moved: out_keys (if given) receives a copy of the ids, and
// the next kernel reads unq_inv itself.  out_pairs: (id, row) per position, one 8-byte
// store; or out_keys / out_rows as two arrays when the order is already final.
template <int ITEMS>
__global__ __launch_bounds__(kHistThreads) void bucket_scatter_kernel(
    const int *__restrict__ inv, long n, int U_arg, int high_bits,
    const int *__restrict__ hist, const int *__restrict__ tile_flags, int n_tiles,
    const int *__restrict__ bucket_start, int *__restrict__ stats, int *__restrict__ out_keys,
    int *__restrict__ out_rows, int2 *__restrict__ out_pairs, const int *__restrict__ num_unq_dev) {
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
    const long tile0 = (long)blockIdx.x * (kHistThreads * ITEMS);
    if (!(flags & kFlagUnsorted)) {
        if (out_keys)
            for (int it = 0; it < ITEMS; ++it) {
                const long i = tile0 + (long)it * kHistThreads + threadIdx.x;
                if (i < n) out_keys[i] = inv[i];
            }
        return;
    }

    // ---- stable ranking inside the tile
    const long wbase = tile0 + (long)w * (64 * ITEMS);
    int key[ITEMS], lrank[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const long i = wbase + (long)it * 64 + lane;
        const int v = i < n ? inv[i] : -1;
        key[it] = (unsigned)v < (unsigned)U ? v : -1;  // out-of-range ids are dropped (and flagged)
    }
    volatile int *wc = wcount + w * bins;
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const bool valid = key[it] >= 0;
        const unsigned long long mask = wave_match(valid ? key[it] >> low_bits : 0, high_bits, valid);
        // rows of the same bucket in front of this one among the wave's 64, and the group's size
        lrank[it] = __popcll(mask & lanes_below) | (__popcll(mask) << 8);
    }
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
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
    for (int it = 0; it < ITEMS; ++it)
        if (key[it] >= 0) lrank[it] += wcount[w * bins + (key[it] >> low_bits)];
    __syncthreads();
    // ---- through LDS (over the wave counts, which are done with): the tile's rows leave in
    // bucket order, so that neighbouring lanes write neighbouring addresses.  Written straight
    // from the ranking, every 8-byte pair was a memory request of its own.  (4M ids in
    // 1024 buckets: 37.6 -> 28.5 us; 1M ids, whose tiles hold four rows per bucket only: 15.2 -> 15.6)
    int2 *stage = reinterpret_cast<int2 *>(lds_scatter);
#pragma unroll
    for (int it = 0; it < ITEMS; ++it)
        if (key[it] >= 0) stage[lrank[it]] = make_int2(key[it], (int)(wbase + (long)it * 64 + lane));
    __syncthreads();
    for (int p = threadIdx.x; p < total; p += kHistThreads) {
        const int2 kr = stage[p];
        const long dst = (long)base_s[kr.x >> low_bits] + p;
        if (dst < 0 || dst >= n) continue;
        if (out_pairs) {
            out_pairs[dst] = kr;
        } else {
            out_keys[dst] = kr.x;
            out_rows[dst] = kr.y;
        }
    }
}

// Rows of bucket b that slice j of it covers.  A bucket is cut into slices of kBktSlice rows.
struct BucketSlice {
    long s, e;        // the bucket's rows [s, e) in bucket order
    long my_s, my_e;  // the slice's rows
    int nsl;          // slices of the bucket
};
__device__ __forceinline__ int slices_of(long cnt_b) {
    return (int)max(1L, (cnt_b + kBktSlice - 1) / kBktSlice);
}
__device__ __forceinline__ BucketSlice bucket_slice(long s, long e, int j) {
    BucketSlice r;
    r.s = s;
    r.e = e;
    r.nsl = slices_of(e - s);
    r.my_s = s + (long)j * kBktSlice;
    r.my_e = min(e, r.my_s + kBktSlice);
    return r;
}

// Workgroup g serves slice j of bucket b; (b, j) follows from the bucket sizes and is kept with
// the bucket's bounds in wg_pick[g] = (b, j, start, end) (b = -1: no work) for the kernel that
// follows, which so learns its work from one load.  Where a bucket has several slices, each
// workgroup counts the rows of ITS slice per voxel (low digit) and writes the counts to
// part_hist[g][*]: the slices of a bucket sit in consecutive workgroups, so the next kernel gets a
// voxel's count in the whole bucket, and in the slices in front of its own, from one short
// read per slice instead of every workgroup of a crowded bucket counting all of its rows.
__global__ __launch_bounds__(kBktThreads) void bucket_count_kernel(
    const int *__restrict__ inv, const int *__restrict__ pairs1, long n, int U_arg, int high_bits,
    const int *__restrict__ bucket_start, const int *__restrict__ stats, int4 *__restrict__ wg_pick,
    int *__restrict__ part_hist, const int *__restrict__ num_unq_dev) {
    const int U = voxel_count(U_arg, num_unq_dev), low_bits = low_bits_of(U, high_bits), high_bins = 1 << high_bits;
    extern __shared__ int cnt_s[];  // [low_bins]
    __shared__ int s_pick[2];
    const int low_bins = 1 << low_bits;
    if (stats[TXS_STAT_NEED_GENERAL] != 0) return;
    {
        if (threadIdx.x == 0) s_pick[0] = -1;
        int carried = 0;
        for (int bb0 = 0; bb0 < high_bins; bb0 += kBktThreads) {
            const int bb = bb0 + (int)threadIdx.x;
            int nsl = 0;
            if (bb < high_bins && ((long)bb << low_bits) < (long)U)
                nsl = slices_of((long)bucket_start[bb + 1] - bucket_start[bb]);
            int total;
            const int first = carried + wide_exclusive_scan<kBktWaves>(nsl, &total);  // (synchronises the workgroup)
            if ((int)blockIdx.x >= first && (int)blockIdx.x < first + nsl) {
                s_pick[0] = bb;
                s_pick[1] = (int)blockIdx.x - first;
            }
            carried += total;
        }
        __syncthreads();
    }
    const int b = s_pick[0], j = s_pick[1];
    if (b < 0) {
        if (threadIdx.x == 0) wg_pick[blockIdx.x] = make_int4(-1, 0, 0, 0);
        return;
    }
    const int u_lo = b << low_bits;
    const bool packed = stats[TXS_STAT_UNSORTED] != 0;
    const int *keys = packed ? pairs1 : inv;
    const BucketSlice sl = bucket_slice(bucket_start[b], bucket_start[b + 1], j);
    if (threadIdx.x == 0) wg_pick[blockIdx.x] = make_int4(b, j, (int)sl.s, (int)sl.e);
    if (sl.nsl == 1) return;  // (uniform) the next kernel counts the bucket itself
    for (int k = threadIdx.x; k < low_bins; k += kBktThreads) cnt_s[k] = 0;
    __syncthreads();
    int v[kBktItems];
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) {
        const long i = sl.my_s + (long)it * kBktThreads + threadIdx.x;
        v[it] = i < sl.my_e ? kread(keys, i, packed) : -1;
    }
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) {
        const int d = v[it] - u_lo;
        if (v[it] >= 0 && (unsigned)d < (unsigned)low_bins) atomicAdd(&cnt_s[d], 1);
    }
    __syncthreads();
    int *mine = part_hist + (long)blockIdx.x * low_bins;
    for (int k = threadIdx.x; k < low_bins; k += kBktThreads) mine[k] = cnt_s[k];
}

// One slice: its rows are counted per voxel by LDS atomics, whose returned values put them, voxel
// by voxel, into LDS in whatever order the atomics ran; each row then finds its place among its
// voxel's rows of the slice by counting the smaller row numbers there (rows ascend along a bucket,
// so that is the stable order).  That costs as many reads, four in flight, as the voxel has rows in
// the slice: runs above kLongRun rows (at most kMaxLongRuns of them in a slice) are ranked by wave
// ballots on their number instead, with a count per run and 64 rows in input order.  Rows leave in
// voxel order, neighbouring lanes to neighbouring addresses.
// What bounds it is the chain of dependent steps inside a workgroup, far more than bytes: 45 KB of
// LDS keep 24 waves on a compute unit (the ballots on all 11 bits that this replaces needed a count
// per wave and voxel as well, left 12, and wrote every row as a request of its own).  Then -> now, us:
// 4M ids of four sweeps (1.3M voxels, 64 MB moved) 131 -> 47, 1M of one 26.2 -> 21.8, of pillars 21.9 ->
// 22.8, 1M ids of 50 / 25 / 10 rows per voxel 27.5 -> 29.7, 23.7 -> 27.7, 28.2 -> 20.9.
__global__ __launch_bounds__(kBktThreads) void bucket_plan_kernel(
    const int *__restrict__ inv, const int *__restrict__ pairs1, long n, int U_arg,
    int high_bits, int heavy_threshold,
    const long long *__restrict__ unq_cnts, int *__restrict__ perm, int *__restrict__ seg,
    int *__restrict__ preSum, int *__restrict__ slot_of, int *__restrict__ heavy_ids,
    int *__restrict__ stats, const int4 *__restrict__ wg_pick, const int *__restrict__ part_hist,
    long long *__restrict__ ranks, const int *__restrict__ num_unq_dev, long long *__restrict__ cnts_out) {
    const int U = voxel_count(U_arg, num_unq_dev), low_bits = low_bits_of(U, high_bits);
    // ranks != NULL: the caller wants the rank of every row inside its voxel and nothing else
    // (ingroup_inds): the placement writes ranks[row] in place of the permutation and the ids
    const bool rank_mode = ranks != nullptr;
    constexpr int kBins = 1 << kBucketLowBitsMax;
    // one after the other: the bucket's counts; a long run's rows per 64 rows of the slice; the slice's
    // rows in voxel order and their voxels (low digits)
    __shared__ int pool_s[kBktSlice + kBktSlice / 2];
    __shared__ int first_s[kBins + 1];            // the slice's counts, then the first place of every voxel in row_s
    __shared__ int step_s[kBins];                 // rows of the voxel in front of this slice, then place -> destination
    __shared__ unsigned short mark_s[kBins];      // bits 0-7: number of a long run + 1 (0: short); bit 15: heavy voxel
    __shared__ int s_red[kBktWaves], s_bad[kBktWaves], s_long;
    static_assert(kBins <= kBktSlice && kMaxLongRuns * 64 * sizeof(short) <= sizeof(pool_s), "what shares a space fits");
    int *tot = pool_s, *row_s = pool_s;
    unsigned short *dig_s = reinterpret_cast<unsigned short *>(pool_s + kBktSlice);
    auto chunk_s = reinterpret_cast<unsigned short(*)[64]>(pool_s);
    const int low_bins = 1 << low_bits;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned long long lanes_below = (1ull << lane) - 1ull;
    if (stats[TXS_STAT_NEED_GENERAL] != 0) return;
    const int4 pick = wg_pick[blockIdx.x];
    const int b = pick.x, j = pick.y;
    if (b < 0) return;
    const int u_lo = b << low_bits;
    const int u_hi = min(U, u_lo + low_bins);
    const bool unsorted = stats[TXS_STAT_UNSORTED] != 0;
    const BucketSlice sl = bucket_slice(pick.z, pick.w, j);
    const long s = sl.s, e = sl.e, my_s = sl.my_s, my_e = sl.my_e;

    // Everything the workgroup reads from memory is requested here, in one go: the slice's rows
    // and the caller's counts of this bucket's voxels (first slice only; compared once the
    // kernel's own counts are complete).
    int dig[kBktItems], row[kBktItems];
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) {
        const long i = my_s + (long)it * kBktThreads + threadIdx.x;
        int v = -1;
        row[it] = (int)i;
        if (i < my_e) {
            if (unsorted) {
                const int2 kr = reinterpret_cast<const int2 *>(pairs1)[i];
                v = kr.x;
                row[it] = kr.y;
            } else {
                v = inv[i];
            }
        }
        dig[it] = (i < my_e && (unsigned)(v - u_lo) < (unsigned)low_bins) ? v - u_lo : -1;
    }
    constexpr int kCntPer = kBins / kBktThreads;
    long long given[kCntPer];
    const bool check_counts = j == 0 && unq_cnts != nullptr;
    if (check_counts) {
#pragma unroll
        for (int k = 0; k < kCntPer; ++k) {
            const int d = k * kBktThreads + (int)threadIdx.x;
            given[k] = (d < low_bins && u_lo + d < u_hi) ? unq_cnts[u_lo + d] : -1;
        }
    }
    for (int k = threadIdx.x; k < low_bins; k += kBktThreads) {
        tot[k] = 0;
        first_s[k] = 0;
        step_s[k] = 0;
    }
    if (threadIdx.x == 0) s_long = 0;
    __syncthreads();
    // ---- the slice's rows per voxel; a row's turn among them, for now in any order
    int turn[kBktItems];
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) turn[it] = dig[it] >= 0 ? atomicAdd(&first_s[dig[it]], 1) : 0;
    // ---- several slices: counts of the bucket's voxels, and of the rows in front of this slice, as
    // sums over the per-slice counts of the bucket's workgroups (blockIdx.x - j is the bucket's
    // first), eight loads in flight per thread
    if (sl.nsl > 1) {
        const int *first = part_hist + ((long)blockIdx.x - j) * low_bins;
        const int total = sl.nsl << low_bits;
        constexpr int kGather = 8;
        for (int i0 = threadIdx.x; i0 < total; i0 += kBktThreads * kGather) {
            int c[kGather];
#pragma unroll
            for (int q = 0; q < kGather; ++q) {
                const int i = i0 + q * kBktThreads;
                c[q] = i < total ? first[i] : 0;
            }
#pragma unroll
            for (int q = 0; q < kGather; ++q) {
                const int i = i0 + q * kBktThreads;
                if (c[q] == 0) continue;
                const int d = i & (low_bins - 1), k = i >> low_bits;
                atomicAdd(&tot[d], c[q]);
                if (k < j) atomicAdd(&step_s[d], c[q]);
            }
        }
    }
    __syncthreads();
    // ---- exclusive scans over the voxels of the bucket, a run of consecutive voxels per thread:
    // of the slice's counts and (the same where there is one slice) of the bucket's
    const int per = (low_bins + kBktThreads - 1) / kBktThreads;
    const int d0 = (int)threadIdx.x * per, d1 = min(d0 + per, low_bins);
    int mine = 0, mine_all = 0;
    for (int d = d0; d < d1; ++d) {
        mine += first_s[d];
        if (sl.nsl > 1) mine_all += tot[d];
    }
    int placed, ignored;
    int run = wide_exclusive_scan<kBktWaves>(mine, &placed);
    int run_all = sl.nsl > 1 ? wide_exclusive_scan<kBktWaves>(mine_all, &ignored) : run;
    for (int d = d0; d < d1; ++d) {
        const int c = first_s[d];
        const int c_all = sl.nsl > 1 ? tot[d] : c;
        if (sl.nsl == 1) tot[d] = c;
        int mark = c_all > heavy_threshold ? 0x8000 : 0;
        if (c > kLongRun) mark |= 1 + atomicAdd(&s_long, 1);
        mark_s[d] = (unsigned short)mark;
        first_s[d] = run;
        // ranks count from the voxel's first row, positions from the bucket's start
        step_s[d] += (rank_mode ? 0 : (int)s + run_all) - run;
        if (j == 0 && u_lo + d < u_hi) {
            preSum[u_lo + d] = (int)s + run_all;
            if (cnts_out) cnts_out[u_lo + d] = (long long)c_all;
            if (u_lo + d == U - 1) preSum[U] = (int)n;
        }
        run += c;
        run_all += c_all;
    }
    if (threadIdx.x == 0) first_s[low_bins] = placed;
    __syncthreads();
    // ---- statistics, special voxels and their slots (first slice only; as plan_special_kernel)
    if (j == 0 && slot_of != nullptr) {
        int vmax = 0;
        bool mismatch = false;
        if (check_counts) {
#pragma unroll
            for (int k = 0; k < kCntPer; ++k) {
                const int d = k * kBktThreads + (int)threadIdx.x;
                if (d < low_bins && u_lo + d < u_hi) mismatch |= given[k] != (long long)tot[d];
            }
        }
        for (int dd = 0; dd < low_bins; dd += kBktThreads) {
            const int d = dd + (int)threadIdx.x;
            const int u = u_lo + d;
            const bool in = d < low_bins && u < u_hi;
            const int cnt = in ? tot[d] : 0;
            vmax = max(vmax, cnt);
            const bool heavy = in && cnt > heavy_threshold;
            const bool empty = in && cnt == 0;
            const unsigned long long mh = __ballot(heavy), me = __ballot(empty);
            int base_h = 0, base_e = 0;
            if (lane == 0) {
                if (mh) base_h = atomicAdd(&stats[TXS_STAT_NUM_HEAVY], __popcll(mh));
                if (me) base_e = atomicAdd(&stats[TXS_STAT_NUM_EMPTY], __popcll(me));
                if (mh | me) atomicAdd(&stats[TXS_STAT_NUM_SPECIAL], __popcll(mh) + __popcll(me));
            }
            base_h = __shfl(base_h, 0, 64);
            base_e = __shfl(base_e, 0, 64);
            if (in) {
                int slot = -1;
                if (heavy) {
                    slot = base_h + __popcll(mh & lanes_below);
                    if (slot < U) heavy_ids[slot] = u;
                } else if (empty) {
                    slot = U - 1 - (base_e + __popcll(me & lanes_below));
                    if (slot >= 0) heavy_ids[slot] = u;
                }
                slot_of[u] = slot;
            }
        }
        const int wmax = wave_max_i32(vmax);
        const bool any_mismatch = __ballot(mismatch) != 0ull;
        if (lane == 0) {
            s_red[w] = wmax;
            s_bad[w] = any_mismatch;
        }
        __syncthreads();  // (also: the last read of tot, whose space the rows take next)
        if (threadIdx.x == 0) {
            int m = 0, bad = 0;
            for (int k = 0; k < kBktWaves; ++k) {
                m = max(m, s_red[k]);
                bad |= s_bad[k];
            }
            if (m > 0) atomicMax(&stats[TXS_STAT_MAX_CNT], m);
            if (bad) stats[TXS_STAT_COUNT_MISMATCH] = 1;
        }
    }

    // what is known of a row once its place p in voxel order is: p's destination
    auto put = [&](int d, int p, int row_i) {
        const long dst = (long)step_s[d] + p;
        if (rank_mode) {
            if ((unsigned)row_i < (unsigned)n) ranks[row_i] = dst;
        } else if (unsorted && dst >= s && dst < e) {
            perm[dst] = row_i;
        }
    };
    // ---- long runs: straight from the registers, ranked by 64 rows in input order at a time
    const int n_long = s_long;  // (uniform)
    if (n_long > 0) {
        const int id_bits = 32 - __builtin_clz((unsigned)n_long);
        for (int k = threadIdx.x; k < n_long * 64; k += kBktThreads) (&chunk_s[0][0])[k] = 0;
        __syncthreads();
#pragma unroll
        for (int it = 0; it < kBktItems; ++it) {
            const int id = dig[it] >= 0 ? (mark_s[dig[it]] & 255) : 0;
            const unsigned long long mask = wave_match(id, id_bits, id > 0);
            const int below = __popcll(mask & lanes_below);
            if (id > 0) {
                turn[it] = below;
                if (below == 0) chunk_s[id - 1][it * kBktWaves + w] = (unsigned short)__popcll(mask);
            }
        }
        __syncthreads();
        for (int k = w; k < n_long; k += kBktWaves) {
            const int c = chunk_s[k][lane];
            chunk_s[k][lane] = (unsigned short)(wave_inclusive_scan(c) - c);
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < kBktItems; ++it) {
            const int id = dig[it] >= 0 ? (mark_s[dig[it]] & 255) : 0;
            if (id == 0) continue;
            turn[it] += chunk_s[id - 1][it * kBktWaves + w];
            put(dig[it], first_s[dig[it]] + turn[it], row[it]);
        }
        __syncthreads();  // (the rows take the chunk counts' space)
    }
    // ---- short runs: into voxel order, then by the number of smaller rows in the run
#pragma unroll
    for (int it = 0; it < kBktItems; ++it) {
        if (dig[it] < 0) continue;
        const int p = first_s[dig[it]] + turn[it];
        row_s[p] = row[it];
        dig_s[p] = (unsigned short)dig[it];
    }
    __syncthreads();
    for (int p = threadIdx.x; p < placed; p += kBktThreads) {
        const int d = dig_s[p];
        const int mark = mark_s[d];
        if (!rank_mode) {
            const long dst = (long)step_s[d] + p;
            if (dst >= s && dst < e) seg[dst] = (u_lo + d) | ((mark & 0x8000) ? kSpecialBit : 0);
        }
        if ((mark & 255) != 0 || (!rank_mode && !unsorted)) continue;
        const int a = first_s[d], z = first_s[d + 1], row_i = row_s[p];
        int smaller = 0;
        for (int q = a; q < z; q += 4) {
            int other[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) other[e] = row_s[min(q + e, kBktSlice - 1)];
#pragma unroll
            for (int e = 0; e < 4; ++e) smaller += (q + e < z && other[e] < row_i) ? 1 : 0;
        }
        put(d, a + smaller, row_i);
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
    const int64_t tile = (int64_t)kHistThreads * hist_items_for(num_total);
    const int64_t tiles = (num_total + tile - 1) / tile;
    const int64_t bins = (int64_t)1 << kBucketLowBitsMax;
    // (id, row) pairs after the bucket scatter, the digit-major histogram, tile flags, bucket
    // boundaries, the scan workspace
    const int64_t hist = bins * (tiles > 0 ? tiles : 1) + 1;
    // per-slice voxel counts of the bucket kernels: (slices + buckets) * voxels per bucket, for
    // the digit split txs_plan_build uses
    const int ubits = radix_bits(num_unq > 1 ? num_unq : 1);
    int low_bits = ubits <= kBucketLowBitsMax ? 0 : ubits - kBucketHighBits;
    if (low_bits > kBucketLowBitsMax) low_bits = kBucketLowBitsMax;
    int64_t counts = 0;
    if (low_bits > 0 && ubits <= kBucketBitsMax) {
        const int64_t groups = num_total / kBktSlice + ((int64_t)1 << (ubits - low_bits));
        counts = 4 + 4 * groups + groups * ((int64_t)1 << low_bits);
    }
    const int64_t bucket = 2 * num_total + hist + tiles + bins + 1 + scan_tiles(hist + 1) + 17 + counts;
    return general > bucket ? general : bucket;
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
    return num_total > 0 && num_unq > 0 && bits <= kBucketBitsMax && bits > kBucketLowBitsMax;
}

int txs_detail::plan_build(const int32_t *unq_inv, int64_t num_total, int64_t num_unq, int32_t heavy_threshold,
                           const int64_t *unq_cnts, int32_t *plan_ws, int32_t *perm, int32_t *seg,
                           int32_t *preSum, int32_t *slot_of, int32_t *heavy_ids, int32_t *stats,
                           long long *ranks, const int *num_unq_dev, long long *cnts_out,
                           const long long *ids64, void *stream) {
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
    // ids of up to 11 bits are sorted by the bucket pass alone; beyond that the bucket digit has
    // 9 bits (narrower, and the buckets of a spatially sorted id space get too uneven: every
    // workgroup of a crowded bucket adds up the counts of all its slices, and above kBktGiant rows the
    // plan is left to the general sequence; wider, and a tile sends too few rows to a bucket for
    // the scatter to write whole cache lines) and the low digit takes the rest, at most 11
    const int low_bits = bits <= kBucketLowBitsMax ? 0 : min(bits - kBucketHighBits, kBucketLowBitsMax);
    const int high_bits = bits - low_bits;
    const int high_bins = 1 << high_bits;
    const int items = hist_items_for(n);
    const long tile = (long)kHistThreads * items;
    const int n_tiles = (int)((n + tile - 1) / tile);
    int *pairs1 = plan_ws;  // (id, row) after the bucket scatter, 8-byte aligned
    int *hist = plan_ws + 2 * n;
    const long used = (long)high_bins * n_tiles;
    int *tile_flags = hist + used + 1;
    int *bucket_start = tile_flags + n_tiles;
    int *scan_ws = bucket_start + high_bins + 1;
    // an upper bound of the (bucket, slice) pairs; workgroups beyond the last pair return at once
    const long groups = n / kBktSlice + high_bins;
    int *wg_pick = reinterpret_cast<int *>(  // 16-byte records
        ((uintptr_t)(scan_ws + scan_tiles(used + 1) + 17) + 15u) & ~(uintptr_t)15u);
    int *part_hist = wg_pick + 4 * groups;
    // (the attribute belongs to the current device's copy of a kernel: once per device)
    constexpr int kMaxDevices = 64;
    static std::atomic<bool> lds_allowed[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return TXS_ERR_LAUNCH;
    if (!lds_allowed[dev].load(std::memory_order_acquire)) {
        for (const void *k : {reinterpret_cast<const void *>(bucket_scatter_kernel<4>),
                              reinterpret_cast<const void *>(bucket_scatter_kernel<8>),
                              reinterpret_cast<const void *>(bucket_scatter_kernel<16>)})
            if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024) != hipSuccess)
                return TXS_ERR_LAUNCH;
        lds_allowed[dev].store(true, std::memory_order_release);
    }
    auto hist32 = items == 16 ? bucket_hist_kernel<16, int>
                              : (items == 8 ? bucket_hist_kernel<8, int> : bucket_hist_kernel<4, int>);
    auto hist64 = items == 16 ? bucket_hist_kernel<16, long long>
                              : (items == 8 ? bucket_hist_kernel<8, long long> : bucket_hist_kernel<4, long long>);
    auto scatter_kernel =
        items == 16 ? bucket_scatter_kernel<16> : (items == 8 ? bucket_scatter_kernel<8> : bucket_scatter_kernel<4>);
    if (ids64)
        hist64<<<dim3(n_tiles), dim3(kHistThreads), 0, st>>>(ids64, n, U, high_bits, hist, tile_flags, n_tiles, ids32,
                                                             num_unq_dev);
    else
        hist32<<<dim3(n_tiles), dim3(kHistThreads), 0, st>>>(unq_inv, n, U, high_bits, hist, tile_flags, n_tiles, nullptr,
                                                             num_unq_dev);
    // one entry more than the histogram: it receives the total, the end of the last bucket.  A
    // bucket's first entry (that of tile 0) is where it starts.
    if (exclusive_scan(hist, used, hist, used + 1, scan_ws, st, bucket_start, n_tiles) != hipSuccess) return TXS_ERR_LAUNCH;
    const size_t lds_scatter = (size_t)high_bins * sizeof(int) +
                               max((size_t)kHistWaves * high_bins * sizeof(int), (size_t)tile * sizeof(int2));
    if (low_bits == 0) {
        // a bucket is a voxel: the scatter already gives the final order
        scatter_kernel<<<dim3(n_tiles), dim3(kHistThreads), lds_scatter, st>>>(
            unq_inv, n, U, high_bits, hist, tile_flags, n_tiles, bucket_start, stats, seg, perm, nullptr, num_unq_dev);
        int rc = txs_plan_presum(seg, n, U, preSum, stream);
        if (slot_of == nullptr) return rc;
        if (rc == TXS_OK)
            rc = txs_plan_special(preSum, U, heavy_threshold, unq_cnts, slot_of, heavy_ids, stats, num_unq_dev,
                                  (int64_t *)cnts_out, stream);
        if (rc == TXS_OK) rc = txs_plan_seg_flag(seg, n, U, slot_of, stream);
        return rc;
    }
    // a bucket so full that its workgroups would run long after all others have finished
    // (only a few voxels holding most of the rows do that) sends the call to the general sequence
    scatter_kernel<<<dim3(n_tiles), dim3(kHistThreads), lds_scatter, st>>>(
        unq_inv, n, U, high_bits, hist, tile_flags, n_tiles, bucket_start, stats, nullptr, nullptr,
        reinterpret_cast<int2 *>(pairs1), num_unq_dev);
    const int low_bins = 1 << low_bits;
    bucket_count_kernel<<<dim3((unsigned)groups), dim3(kBktThreads), (size_t)low_bins * sizeof(int), st>>>(
        unq_inv, pairs1, n, U, high_bits, bucket_start, stats, reinterpret_cast<int4 *>(wg_pick), part_hist, num_unq_dev);
    bucket_plan_kernel<<<dim3((unsigned)groups), dim3(kBktThreads), 0, st>>>(
        unq_inv, pairs1, n, U, high_bits, heavy_threshold,
        (const long long *)unq_cnts, perm, seg, preSum, slot_of, heavy_ids, stats,
        reinterpret_cast<const int4 *>(wg_pick), part_hist, ranks, num_unq_dev, cnts_out);
    return status_of(hipGetLastError());
}
