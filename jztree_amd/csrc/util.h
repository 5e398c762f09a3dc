// Device-wide scan / fill / compaction helpers shared by the jztree_amd ops.
// All launches are stream-ordered, allocate nothing and are graph-capturable (fills are kernels,
// never hipMemsetAsync).
#pragma once
#include "common.h"

namespace jzt {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;  // 2048

// number of int32 temp words a scan of n elements needs
inline int64_t scan_tmp_words(int64_t n) { return div_up(n, kScanTile) + 1; }

// out[i] = sum_{j<i} in[j] (exclusive) or sum_{j<=i} (inclusive); in may alias out.
// tmp must hold scan_tmp_words(n) int32.
int scan_i32(hipStream_t s, const int32_t* in, int32_t* out, int64_t n, bool inclusive, int32_t* tmp);

// process-wide tuning knobs (set through jzt_set_tuning; the values the kernels were written for
// are the defaults)
enum TuneKnob { kTuneLeafWaves = 0, kTuneSortKpt = 1, kTuneXcd = 2, kTuneCount = 3 };
int tune_get(int knob);

// byte offsets of the regions inside one scratch buffer are kept 256-byte aligned
inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// fill n 32-bit words with v
int fill_u32(hipStream_t s, void* p, uint32_t v, int64_t n);
int clear_flag(hipStream_t s, uint8_t* p);

// Stable compaction: out[j] = index of the j-th nonzero flag (j < size), remaining out = fill
// (or *fill_dev when given);
// *count_out (device) = number of nonzero flags (may exceed size).  tmp: scan_tmp_words(n) + n words.
int where_flags_i8(hipStream_t s, const int8_t* flags, int64_t n, int32_t* out, int64_t size, int32_t fill,
                   const int32_t* fill_dev, int32_t* count_out, int32_t* tmp);

// exclusive scan of n words in place by one workgroup; the total goes to p[n]
void scan_tiles_i32(hipStream_t s, int32_t* p, int64_t n);

// flags[i] |= lvl[i] >= *lvl_max && i <= *npart, as 0/1 bytes
int flags_or_level_i8(hipStream_t s, int8_t* flags, const int32_t* lvl, int64_t n, const int32_t* lvl_max,
                      const int32_t* npart);

// wave64 inclusive prefix sum of an int (all 64 lanes active)
__device__ __forceinline__ int wave_incl_scan(int v) {
  int lane = __lane_id();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int t = __shfl_up(v, o, 64);
    v += (lane >= o) ? t : 0;
  }
  return v;
}

// block-wide exclusive scan for blockDim.x == NT (multiple of 64); returns exclusive prefix and
// writes the block total to *total.  `sbuf` needs NT/64 ints of shared memory.
template <int NT>
__device__ __forceinline__ int block_excl_scan(int v, int* sbuf, int* total) {
  constexpr int NW = NT / 64;
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = wave_incl_scan(v);
  if (lane == 63) sbuf[w] = inc;
  __syncthreads();
  int off = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < NW; i++) {
    int x = sbuf[i];
    off += (i < w) ? x : 0;
    tot += x;
  }
  __syncthreads();
  *total = tot;
  return off + inc - v;
}

// Grid-stride kernels over the segments of a split array spl[0..n] (non-decreasing, as every
// split array of the tree and its lists is, with padded slots repeating the final value): the
// segments from the first index where spl reaches its final value on are empty, so the loop stops
// there instead of striding through a padded allocation.  Found by a binary search at kernel start
// (the same value in every lane).
__device__ __forceinline__ int64_t active_items(const int32_t* __restrict__ spl, int64_t n) {
  const int32_t last = spl[n];
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (spl[mid] < last) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// XCD-aware order of a grid-stride loop over n items.  The chip deals workgroups to its 8 XCDs
// round-robin (workgroup b runs on XCD b % 8) and every XCD has its own L2, so the plain order
// (block b takes items b, b + grid, ...) spreads neighbouring items over all eight L2s.  With `on`
// (and a grid that is a multiple of 8), XCD x takes the x-th eighth of the items and its blocks
// stride through that range: the items an XCD has in flight are neighbours, which in z-order share
// most of their sources.  The item set is the same either way.
struct ItemRange {
  int64_t first, end, step;
};
__device__ __forceinline__ ItemRange xcd_items(int64_t n, bool on) {
  const int64_t g = gridDim.x;
  if (!on || (g & 7) != 0) return {(int64_t)blockIdx.x, n, g};
  const int64_t x = blockIdx.x & 7, per = (n + 7) >> 3;
  return {x * per + (int64_t)(blockIdx.x >> 3), n < (x + 1) * per ? n : (x + 1) * per, g >> 3};
}
// Walk over the items of xcd_items by one-wave workgroups, in that fixed order or (counters given, zeroed
// before the launch) dynamically: the blocks of an XCD take the items of its eighth from a shared
// counter, so they finish together however uneven the items are; the item set and the XCD-contiguous
// order are the same.  It pays where items are expensive and uneven (kNN query leaves); for the cheap,
// even FoF leaves every fetch order tried was slower than the static one.
//
// An atomic on a counter that all waves share takes about 11 ns, one after the other on all XCDs: item by
// item, with 50,000 waves that each make one more to find the queue empty, 32,000 leaves of k = 8 waited
// 0.9 ms for it (1.13 ms the kernel, 0.70 now).  queue_grid therefore launches no more waves than the
// chip holds, and where there are 16 pairs of items for each wave they are taken in pairs over the first
// three quarters (eights cost more in L2 hits and balance than they saved: 2^26 points, learned kNN,
// 63.7 ms against 62.6).
constexpr int kQueueStride = 8;  // words from counter to counter
struct ItemWalk {
  int64_t at, end;  // the item in hand; all 64 lanes call the functions (wave-uniform results)
  int64_t step, begin, big, stop, fresh;
  uint32_t* ctr;
  uint32_t chunk, got, count;
  __device__ __forceinline__ ItemWalk(int64_t n, bool on, uint32_t* counters) {
    const ItemRange r = xcd_items(n, on);
    at = r.first;
    end = r.end;
    step = r.step;
    ctr = counters;
    if (ctr) {
      const int64_t g = gridDim.x;
      const bool split = on && (g & 7) == 0;
      const int64_t per = split ? (n + 7) >> 3 : n, waves = split ? g >> 3 : g;
      begin = split ? (blockIdx.x & 7) * per : 0;
      if (split) ctr += (blockIdx.x & 7) * kQueueStride;
      big = begin + per / 4 * 3;
      chunk = (uint32_t)min(max(per / (16 * waves), (int64_t)1), (int64_t)2);
      take(begin);
      next();
    }
  }
  __device__ __forceinline__ bool more() const { return at < end; }
  // to be called when the work on an item begins: the next ones are asked for meanwhile
  __device__ __forceinline__ void started() {
    if (ctr && at >= fresh) {
      fresh = stop;
      take(at);
    }
  }
  __device__ __forceinline__ void advance() {
    if (!ctr) at += step;
    else if (++at >= stop) next();
  }

 private:
  __device__ __forceinline__ void take(int64_t pos) {
    count = pos < big ? chunk : 1u;
    got = 0;
    if (threadIdx.x == 0) got = atomicAdd(ctr, count);
  }
  __device__ __forceinline__ void next() {
    at = fresh = begin + (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane(got);
    stop = at + (int64_t)count;
  }
};
// grid of a kernel of one-wave workgroups that walk a queue, `per_cu` of which a compute unit holds
inline unsigned queue_grid(int64_t n, int per_cu) {
  const int64_t most = 256 * (int64_t)per_cu;
  return (unsigned)(((n <= 0 ? 8 : n < most ? n : most) + 7) & ~(int64_t)7);
}
// grid for xcd_items: at most kMaxGrid blocks, a multiple of 8
inline unsigned grid_for8(int64_t n) {
  int64_t g = n <= 0 ? 8 : (n < kMaxGrid ? n : kMaxGrid);
  return (unsigned)((g + 7) & ~(int64_t)7);
}

}  // namespace jzt
