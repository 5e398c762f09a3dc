// Leaf and node construction from z-sorted positions (replaces jztree's tree.cuh kernels).
//
//  FlagLeafBoundaries  tree.cuh:13-98    boundary b (between particles b-1 and b) is a leaf split if
//                                        the binary Morton cell it separates holds > max_size
//                                        particles (counted in an LDS window of scan_size boundaries)
//  FindNodeBoundaries  tree.cuh:104-199  per boundary of the leaf representatives: its level and the
//                                        [lbound, rbound) extent of the node it splits (binary search)
//  GetNodeGeometry     tree.cuh:312-372  level, centre and extent of the smallest cell holding a range
//
// All integer/bit exact.  Launch: 256 threads (4 waves) per workgroup, one node per lane (four
// boundaries per lane in FlagLeafBoundaries).
#include "util.h"
#include "../../include/jztree_amd.h"

namespace jzt {
namespace {

constexpr int kTreeThreads = 256;
constexpr int kFlagPer = 4;  // boundaries per thread in k_flag_leaf: the LDS window's halo is shared by more of them
constexpr int kFlagSpan = kTreeThreads * kFlagPer;
constexpr int kFlagChunk = 8;  // levels per block in k_flag_leaf's outward scans
constexpr int kFlagPad = 8 * kFlagChunk + kFlagChunk;  // slots past either end of its LDS window

template <int D, typename T>
__global__ __launch_bounds__(kTreeThreads) void k_flag_leaf(const T* __restrict__ posz, const uint8_t* __restrict__ ptype,
                                                            const int32_t* __restrict__ lvl_bound,
                                                            const int32_t* __restrict__ npart_p,
                                                            int8_t* __restrict__ split_flags, int32_t* __restrict__ lvl,
                                                            int64_t size_part, int max_size, int scan_size,
                                                            int num_types, const int32_t* __restrict__ seg) {
  extern __shared__ int32_t s_mem[];
  const int nload = kFlagSpan + 2 * scan_size + 1;
  const int nslot = nload + 2 * kFlagPad;
  // levels, and the maximum of each run of kFlagChunk levels ending at a slot; kFlagPad slots on
  // either side hold INT_MIN (the scans may read past the window: those reads never hit)
  int32_t* const s_level = s_mem + kFlagPad;
  int32_t* const s_max8 = s_mem + nslot + kFlagPad;
  uint8_t* s_types = reinterpret_cast<uint8_t*>(s_mem + 2 * nslot);
  const int64_t nump = npart_p[0];
  const int lb_l = lvl_bound[0], lb_r = lvl_bound[1];
  const int64_t ioff = (int64_t)blockIdx.x * kFlagSpan - scan_size - 1;

  // s_level[i] = level of boundary ioff+i+1, i.e. between particles ioff+i and ioff+i+1
  for (int i = threadIdx.x; i < nload - 1; i += kTreeThreads) {
    int64_t ip = ioff + i;
    int L;
    uint8_t ty = 0;
    if (ip < 0) {
      L = lb_l;
    } else if (ip + 1 >= nump) {
      L = lb_r;
    } else {
      L = (seg && seg[ip] != seg[ip + 1]) ? kLvlSet
                                          : msb_diff_level<D, T>(load_vec<D, T>(posz, ip), load_vec<D, T>(posz, ip + 1));
      if (num_types > 1) ty = ptype[ip];
    }
    s_level[i] = L;
    s_types[i] = ty;
  }
  for (int i = threadIdx.x; i < 2 * kFlagPad + 1; i += kTreeThreads) {
    const int j = i < kFlagPad ? i - kFlagPad : nload - 1 + (i - kFlagPad);
    s_level[j] = INT32_MIN;
    s_max8[j] = INT32_MIN;
  }
  __syncthreads();
  if (num_types == 1) {
    for (int i = threadIdx.x; i < nload - 1; i += kTreeThreads) {
      int m = s_level[i];
#pragma unroll
      for (int u = 1; u < kFlagChunk; u++) m = max(m, s_level[i - u]);
      s_max8[i] = m;
    }
    __syncthreads();
  }

  for (int rep = 0; rep < kFlagPer; rep++) {
    const int64_t node_idx = (int64_t)blockIdx.x * kFlagSpan + rep * kTreeThreads + threadIdx.x;
    const int idx = rep * kTreeThreads + threadIdx.x + scan_size;
    const int my = s_level[idx];
    bool is_split = false;
    if (num_types == 1) {
      // one type: lsize = idx - (the nearest i < idx in the window with s_level[i] >= my), or the whole
      // window if there is none -- what the reset-and-count loop below leaves -- i.e. the distance
      // to the nearest level >= my on the left, capped at scan_size (likewise rsize to the right).
      // The scan goes by blocks of kFlagChunk levels: eight block maxima per step (one LDS round
      // trip covers 64 levels), then the levels of the first block that holds a hit.  Reads past
      // the window land in the INT_MIN pads or beyond scan_size, where the cap hides them.
      const int32_t* const here = s_level + idx;
      const int32_t* const here8 = s_max8 + idx;
      auto nearest = [&](auto right_c) {
        constexpr bool R = decltype(right_c)::value;
        for (int d0 = 1; d0 <= scan_size; d0 += 8 * kFlagChunk) {
          int mb[8];
#pragma unroll
          for (int u = 0; u < 8; u++) {
            const int d = d0 + u * kFlagChunk;  // block of distances [d, d + kFlagChunk - 1]
            mb[u] = R ? here8[d + kFlagChunk - 1] : here8[-d];
          }
          int blk = -1;
#pragma unroll
          for (int u = 7; u >= 0; u--) blk = mb[u] >= my ? u : blk;
          if (blk >= 0) {
            const int d = d0 + blk * kFlagChunk;
            int lv[kFlagChunk];
#pragma unroll
            for (int v = 0; v < kFlagChunk; v++) lv[v] = R ? here[d + v] : here[-(d + v)];
            int hit = d + kFlagChunk - 1;  // the block max is a hit, so some v matches
#pragma unroll
            for (int v = kFlagChunk - 1; v >= 0; v--) hit = lv[v] >= my ? d + v : hit;
            return min(hit, scan_size);
          }
        }
        return scan_size;
      };
      const int lsize = nearest(std::false_type());
      const int rsize = nearest(std::true_type());
      is_split |= (lsize + rsize > max_size);
      is_split |= (my > lb_l) && (node_idx - lsize <= 0);
      is_split |= (my > lb_r) && (node_idx + rsize >= nump);
    } else {
      for (int type = 0; type < num_types; type++) {
        int lsize = 0;
        for (int i = idx - scan_size; i < idx; i++) lsize = (s_level[i] < my ? lsize : 0) + (s_types[i] == type ? 1 : 0);
        int rsize = 0;
        for (int i = idx + scan_size; i > idx; i--) rsize = (s_level[i] < my ? rsize : 0) + (s_types[i] == type ? 1 : 0);
        is_split |= (lsize + rsize > max_size);
        is_split |= (my > lb_l) && (node_idx - lsize <= 0);
        is_split |= (my > lb_r) && (node_idx + rsize >= nump);
      }
    }
    is_split |= my >= kLvlSet;  // set boundary of a batch
    is_split &= node_idx <= nump;
    is_split |= node_idx == 0;
    is_split |= node_idx == nump;
    if (node_idx < size_part + 1) {
      split_flags[node_idx] = (int8_t)is_split;
      lvl[node_idx] = my;
    }
  }
}

template <int D, typename T>
__global__ __launch_bounds__(kTreeThreads) void k_find_node_bounds(const T* __restrict__ pos_in,
                                                                   const T* __restrict__ pos_boundary,
                                                                   const int32_t* __restrict__ nleaves_p,
                                                                   int32_t* __restrict__ levels, int32_t* __restrict__ lbound,
                                                                   int32_t* __restrict__ rbound, int64_t size_nodes,
                                                                   int lvl_invalid, const int32_t* __restrict__ seg) {
  int64_t idx = (int64_t)blockIdx.x * kTreeThreads + threadIdx.x;
  const int n = nleaves_p[0];
  const int nnodes = n + 1;
  if (idx >= size_nodes) return;
  if (idx >= nnodes) {
    levels[idx] = lvl_invalid;
    lbound[idx] = n;
    rbound[idx] = n;
    return;
  }
  // the points past either end: pos_boundary, or NaN without it
  auto end_point = [&](int i) {
    Vec<D, T> r;
#pragma unroll
    for (int d = 0; d < D; d++) r[d] = pos_boundary ? pos_boundary[i * D + d] : (T)__builtin_nan("");
    return r;
  };
  Vec<D, T> p1 = (idx == 0) ? end_point(0) : load_vec<D, T>(pos_in, idx - 1);
  Vec<D, T> p2 = (idx == nnodes - 1) ? end_point(1) : load_vec<D, T>(pos_in, idx);
  if (n <= 0) {  // no leaves: the single boundary spans nothing (the reference would read pos_in[-1])
    levels[idx] = msb_diff_level<D, T>(p1, p2);
    lbound[idx] = 0;
    rbound[idx] = 0;
    return;
  }
  // batch sets: points of different sets are separated at kLvlSet; the array ends take the set of
  // their neighbour.  Sets are contiguous, so levels stay monotone along the searches below.
  const int64_t ia = idx > 0 ? idx - 1 : 0, ib = idx < n ? idx : n - 1;
  auto level = [&](int64_t i, const Vec<D, T>& a, int64_t j, const Vec<D, T>& b) {
    return (seg && seg[i] != seg[j]) ? kLvlSet : msb_diff_level<D, T>(a, b);
  };
  const int target = level(ia, p1, ib, p2);
  int lb, rb;
  if (level(0, load_vec<D, T>(pos_in, 0), ib, p2) <= target) {
    lb = 0;
  } else {
    int ibefore = 0, iinside = (int)idx;
    while (ibefore + 1 < iinside) {
      int it = (ibefore + iinside) / 2;
      if (level(it, load_vec<D, T>(pos_in, it), ib, p2) > target) ibefore = it;
      else iinside = it;
    }
    lb = iinside;
  }
  if (level(ia, p1, n - 1, load_vec<D, T>(pos_in, n - 1)) <= target) {
    rb = n;
  } else {
    int iinside = (int)idx - 1, iafter = n - 1;
    while (iinside + 1 < iafter) {
      int it = (iinside + iafter) / 2;
      if (level(ia, p1, it, load_vec<D, T>(pos_in, it)) > target) iafter = it;
      else iinside = it;
    }
    rb = iafter;
  }
  levels[idx] = target;
  lbound[idx] = lb;
  rbound[idx] = rb;
}

template <typename T> __device__ __forceinline__ T quiet_nan();
template <> __device__ __forceinline__ float quiet_nan<float>() { return __uint_as_float(0x7fc00000u); }
template <> __device__ __forceinline__ double quiet_nan<double>() { return __longlong_as_double(0x7ff8000000000000ll); }

template <int D, typename T>
__global__ __launch_bounds__(kTreeThreads) void k_node_geometry(const T* __restrict__ pos, const int32_t* __restrict__ lbound,
                                                                const int32_t* __restrict__ rbound,
                                                                const int32_t* __restrict__ nnodes_p,
                                                                int32_t* __restrict__ level, T* __restrict__ center,
                                                                T* __restrict__ extent, int64_t size_nodes,
                                                                int64_t size_part, int lvl_invalid, uint32_t mode,
                                                                int upper) {
  int64_t idx = (int64_t)blockIdx.x * kTreeThreads + threadIdx.x;
  if (idx >= size_nodes) return;
  if (idx >= nnodes_p[0]) {
    if (mode & 1u) level[idx] = lvl_invalid;
#pragma unroll
    for (int d = 0; d < D; d++) {
      if (mode & 2u) center[idx * D + d] = quiet_nan<T>();
      if (mode & 4u) extent[idx * D + d] = T(0);
    }
    return;
  }
  auto clip = [&](int64_t a) { return a < 0 ? (int64_t)0 : (a > size_part - 1 ? size_part - 1 : a); };
  const int64_t lb = lbound[idx], rb = rbound[idx];
  Vec<D, T> x0b = load_vec<D, T>(pos, clip(lb));
  Vec<D, T> x1a = load_vec<D, T>(pos, clip(rb - 1));
  int lvl;
  if (!upper) {
    lvl = msb_diff_level<D, T>(x0b, x1a);
  } else {
    Vec<D, T> x0a = load_vec<D, T>(pos, clip(lb - 1));
    Vec<D, T> x1b = load_vec<D, T>(pos, clip(rb));
#pragma unroll
    for (int d = 0; d < D; d++) {
      if (lb - 1 < 0) x0a[d] = -INFINITY;
      if (rb >= size_part) x1b[d] = INFINITY;
    }
    lvl = min(msb_diff_level<D, T>(x0a, x0b), msb_diff_level<D, T>(x1a, x1b)) - 1;
  }
  int l[D];
  lvl_vec<D>(lvl, l);
  if (mode & 1u) level[idx] = lvl;
#pragma unroll
  for (int d = 0; d < D; d++) {
    if (mode & 2u) center[idx * D + d] = round_pow2_cent(x0b[d], l[d]);
    if (mode & 4u) extent[idx * D + d] = pow2<T>(T(1), l[d]);
  }
}

template <int D, typename T>
int flag_leaf_impl(hipStream_t s, const void* posz, const uint8_t* ptype, const int32_t* lvl_bound, const int32_t* npart,
                   int8_t* flags, int32_t* lvl, int64_t size_part, int max_size, int scan_size, int num_types,
                   const int32_t* seg) {
  int64_t nb = size_part + 1;
  int nload = kFlagSpan + 2 * scan_size + 1;
  size_t shmem = (size_t)(2 * (nload + 2 * kFlagPad)) * sizeof(int32_t) + (size_t)nload;
  if (shmem > 60000) return fail("FlagLeafBoundaries: scan_size too large");
  hipLaunchKernelGGL((k_flag_leaf<D, T>), dim3((unsigned)div_up(nb, kFlagSpan)), dim3(kTreeThreads), shmem, s,
                     (const T*)posz, ptype, lvl_bound, npart, flags, lvl, size_part, max_size, scan_size, num_types,
                     seg);
  return check_launch("FlagLeafBoundaries");
}

template <int D, typename T>
int find_node_impl(hipStream_t s, const void* pos_in, const void* pos_boundary, const int32_t* nleaves, int32_t* lv,
                   int32_t* lb, int32_t* rb, int64_t size_nodes, int lvl_invalid, const int32_t* seg) {
  hipLaunchKernelGGL((k_find_node_bounds<D, T>), dim3((unsigned)div_up(size_nodes, kTreeThreads)), dim3(kTreeThreads),
                     0, s, (const T*)pos_in, (const T*)pos_boundary, nleaves, lv, lb, rb, size_nodes, lvl_invalid, seg);
  return check_launch("FindNodeBoundaries");
}

template <int D, typename T>
int geometry_impl(hipStream_t s, const void* pos, const int32_t* lbound, const int32_t* rbound, const int32_t* nnodes,
                  int32_t* level, void* center, void* extent, int64_t size_nodes, int64_t size_part, int lvl_invalid,
                  uint32_t mode, int upper) {
  hipLaunchKernelGGL((k_node_geometry<D, T>), dim3((unsigned)div_up(size_nodes, kTreeThreads)), dim3(kTreeThreads), 0,
                     s, (const T*)pos, lbound, rbound, nnodes, level, (T*)center, (T*)extent, size_nodes, size_part,
                     lvl_invalid, mode, upper);
  return check_launch("GetNodeGeometry");
}

// ------------------------------------------------------------------------------------------------
// regularization level (tree.py:55-68 _level_histogram, :160-187 find_regularization_level)
// ------------------------------------------------------------------------------------------------
// Block-private histogram in LDS (levels cluster on a few bins: global atomics alone would
// serialise on them), merged with one global atomic per nonzero bin and block.  Level ranges past
// kRegLdsLevels bins (float64 positions in 4 or more dims: 2099 levels per dim) count straight
// into the global histogram.
constexpr int kRegLdsLevels = 8192;  // 64 KB of u64 bins
__global__ __launch_bounds__(256) void k_reg_hist(const int32_t* __restrict__ lvl, const int32_t* __restrict__ w,
                                                  int64_t n, int min_lvl, int nlvl,
                                                  unsigned long long* __restrict__ hist) {
  extern __shared__ unsigned long long s_hist[];
  const bool lds = nlvl <= kRegLdsLevels;
  unsigned long long* h = lds ? s_hist : hist;
  if (lds) {
    for (int j = threadIdx.x; j < nlvl; j += blockDim.x) s_hist[j] = 0ull;
    __syncthreads();
  }
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    int b = lvl[i] - min_lvl;
    b = b < 0 ? 0 : b;  // jnp.bincount clips below and drops above
    const int64_t wi = w ? (int64_t)w[i] : 1;
    if (b < nlvl && wi != 0) atomicAdd(&h[b], (unsigned long long)wi);
  }
  if (lds) {
    __syncthreads();
    for (int j = threadIdx.x; j < nlvl; j += blockDim.x)
      if (s_hist[j]) atomicAdd(&hist[j], s_hist[j]);
  }
}

// FP32 evaluation in ascending level order (the reference reduces under XLA's order; only
// borderline ties can differ).  One thread forms the running sums in that order over the nonzero bins
// alone (leaves and nodes sit on a few tens of the 838 levels of 3-D float32, and adding 0 changes no
// sum); the two "first level whose running sum reaches ..." searches go over the same bins, the levels
// between two of them taking the value of the lower one.  71 us with a serial pass over all levels
// (500 us for float64), 9 us (42).  One workgroup per histogram (blockIdx.x).
constexpr int kRegThreads = 256;
__global__ __launch_bounds__(kRegThreads) void k_reg_level(const unsigned long long* __restrict__ hist_all, int nlvl,
                                                           int min_lvl, int max_lvl, float fac, float frac,
                                                           int32_t* __restrict__ bins_all, int32_t* out) {
  __shared__ int sbuf[kRegThreads / 64];
  __shared__ int s_bin[kRegThreads];    // a chunk of nonzero bins
  __shared__ float s_cnt[kRegThreads];  // and their counts
  const unsigned long long* const hist = hist_all + (int64_t)blockIdx.x * nlvl;
  int32_t* const bins = bins_all + (int64_t)blockIdx.x * nlvl;
  const int tid = threadIdx.x;
  // nonzero bins in ascending order
  int nz = 0;
  for (int b0 = 0; b0 < nlvl; b0 += kRegThreads) {
    const int b = b0 + tid;
    const int f = b < nlvl && hist[b] != 0ull ? 1 : 0;
    int tot;
    const int o = block_excl_scan<kRegThreads>(f, sbuf, &tot);
    if (f) bins[nz + o] = b;
    nz += tot;
  }
  __syncthreads();
  // every thread runs the same serial passes, on chunks staged in LDS; body(bin, count) returns false to stop
  auto each = [&](auto body) {
    for (int c0 = 0; c0 < nz; c0 += kRegThreads) {
      __syncthreads();
      if (c0 + tid < nz) {
        const int b = bins[c0 + tid];
        s_bin[tid] = b;
        s_cnt[tid] = (float)(int64_t)hist[b];
      }
      __syncthreads();
      const int m = min(kRegThreads, nz - c0);
      for (int i = 0; i < m; i++)
        if (!body(s_bin[i], s_cnt[i])) return;
    }
  };
  float total = 0.f;
  each([&](int, float c) {
    total += c;
    return true;
  });
  const float thresh = frac * total;
  // the first level whose running sum reaches the threshold: level 0 if an empty sum does
  int first = 0.f >= thresh && nlvl > 0 ? 0 : INT_MAX;
  float cum = 0.f;
  if (first == INT_MAX)
    each([&](int b, float c) {
      cum += c;
      if (cum >= thresh) first = b;
      return first == INT_MAX;
    });
  const int ref = first == INT_MAX ? max_lvl : first + min_lvl;
  float vol_sum = 0.f, cts_sum = 0.f;
  each([&](int b, float c) {
    if (b + min_lvl > ref) return false;
    const float v = ldexpf(1.0f, b + min_lvl - ref);
    vol_sum += v * c;
    cts_sum += c;
    return true;
  });
  const float avg = vol_sum / cts_sum;
  const float lim = fac * avg;
  // the first level from `first` on whose cell volume reaches the limit (volumes grow with the level,
  // running sums past `first` stay past the threshold)
  __shared__ int s_first;
  if (tid == 0) s_first = INT_MAX;
  __syncthreads();
  if (first != INT_MAX)
    for (int b = first + tid; b < nlvl; b += kRegThreads)
      if (ldexpf(1.0f, b + min_lvl - ref) >= lim) atomicMin(&s_first, b);
  __syncthreads();
  if (tid == 0) out[blockIdx.x] = s_first == INT_MAX ? max_lvl : s_first + min_lvl;
}

// Node geometry of a float64 tree for float32 distance kernels on the float32-rounded points.
// The node's Morton cell (c, level) holds its float64 points.  It is replaced by the smallest
// enclosing Morton cell whose per-dim sides are at least 2^(E_i - 23), where every coordinate of
// the cell has magnitude <= 2^E_i: the boundaries of that cell (multiples of its side) and its
// centre (multiples of half a side) are then float32 numbers, so rounding to float32, which is
// monotone and leaves those boundaries fixed, keeps every point inside it.  The float32 cell is
// therefore a conservative bound for the rounded points, as the float64 cell is for the originals.
// Levels past the float32 range (a node spanning signs) become the float32 "whole space" level.
template <int D>
__global__ void k_geometry_to_f32(const double* __restrict__ cent, const int32_t* __restrict__ lvl, int64_t n,
                                  int lvl_invalid, float* __restrict__ cent_out, int32_t* __restrict__ lvl_out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int level = lvl[i];
  double c[D];
  bool finite = true;
#pragma unroll
  for (int d = 0; d < D; d++) {
    c[d] = cent[i * D + d];
    finite &= __builtin_isfinite(c[d]);
  }
  const int top32 = 128 * D;  // float32: cells spanning signs or infinities
  if (level == lvl_invalid || !finite || level >= top32) {
#pragma unroll
    for (int d = 0; d < D; d++) cent_out[i * D + d] = (float)c[d];
    lvl_out[i] = (level == lvl_invalid || !finite) ? level : top32;
    return;
  }
  int L = level;
  for (int guard = 0; guard < 64 * D; guard++) {
    int l[D];
    lvl_vec<D>(L, l);
    bool ok = true;
#pragma unroll
    for (int d = 0; d < D; d++) {
      // |x| <= |centre| + side for x in the cell; E = exponent with that bound <= 2^E
      const double m = fabs(round_pow2_cent(c[d], l[d])) + ldexp(1.0, l[d]);
      int e;
      frexp(m, &e);  // m < 2^e
      ok &= l[d] >= max(e - 23, -149);
    }
    if (ok) break;
    L++;
  }
  if (L >= top32) L = top32;
  int l[D];
  lvl_vec<D>(L, l);
#pragma unroll
  for (int d = 0; d < D; d++) cent_out[i * D + d] = (float)round_pow2_cent(c[d], l[d]);
  lvl_out[i] = L;
}


// ------------------------------------------------------------------------------------------------
// the whole hierarchy of one set or a batch in one call (tree.py:189-262, :600-829)
// ------------------------------------------------------------------------------------------------
// FlagLeafBoundaries, FindNodeBoundaries and GetNodeGeometry are the kernels above; the steps between
// them (compactions, level histograms, plane activity, prefix sums, scatters into the packed arrays) ran as
// ~130 array operations of a few microseconds each, most of them launch-bound.  With them as kernels that handle
// all planes at once, kNN of 1000 points went from 189 launches and 1.60 ms to 54 and 0.43 ms, FoF of 12,800
// from 1.65 to 0.42 ms, kNN of 65,536 from 1.74 to 0.58.
// A boundary's activity on up to kMaxPlanes planes is one bit mask, so each step reads it once for all planes.
constexpr int kMaxPlanes = 32;
constexpr int kBuildThreads = 256;
constexpr int kBuildPer = 4;  // boundaries per thread of the plane passes
constexpr int kBuildTile = kBuildThreads * kBuildPer;
// words of the small device state: npart, lvl_bound[2], leaf splits found, leaves, first row with a NaN
enum { kBsNpart = 0, kBsLvlBound = 1, kBsFilled = 3, kBsLeaves = 4, kBsTail = 5, kBsWords = 16 };
// rows up to which the workgroup that finds the first NaN row also looks through those after it; above, they
// get a launch of their own (k_build_tail)
constexpr int64_t kBuildTailHere = 16384;

struct PlaneSizes {
  int32_t v[kMaxPlanes];
};

// npart: the given count, or the rows whose first coordinate is not NaN.  Rows with a NaN are the last ones of
// z-sorted positions, so only those are looked at, here (tail_here) or by k_build_tail.  Also clears the
// histograms.
template <int D, typename T>
__global__ __launch_bounds__(kBuildThreads) void k_build_init(const T* __restrict__ posz, int64_t n,
                                                              const int32_t* __restrict__ npart_in, int64_t npart_host,
                                                              int tail_here, int lvl_bound, int32_t* __restrict__ state,
                                                              uint32_t* __restrict__ hist, int64_t hist_words) {
  for (int64_t i = (int64_t)blockIdx.x * kBuildThreads + threadIdx.x; i < hist_words; i += (int64_t)gridDim.x * kBuildThreads)
    hist[i] = 0u;
  if (blockIdx.x != 0) return;
  __shared__ int s_num;
  if (threadIdx.x == 0) s_num = 0;
  __syncthreads();
  if (npart_in == nullptr && npart_host < 0) {
    auto has_nan = [&](int64_t i) {
      const Vec<D, T> x = load_vec<D, T>(posz, i);
      bool r = false;
#pragma unroll
      for (int d = 0; d < D; d++) r |= x[d] != x[d];
      return r;
    };
    int64_t lo = 0, hi = n;  // rows before lo hold no NaN, rows from hi on do
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (has_nan(mid)) hi = mid;
      else lo = mid + 1;
    }
    if (tail_here) {
      int c = 0;
      for (int64_t i = lo + threadIdx.x; i < n; i += kBuildThreads) {
        const T x = posz[i * D];
        c += x == x ? 1 : 0;
      }
      if (c) atomicAdd(&s_num, c);
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      state[kBsTail] = (int32_t)lo;
      state[kBsNpart] = (int32_t)lo + s_num;
    }
  } else if (threadIdx.x == 0) {
    state[kBsNpart] = npart_in ? npart_in[0] : (int32_t)npart_host;
  }
  if (threadIdx.x == 0) {
    state[kBsLvlBound] = lvl_bound;
    state[kBsLvlBound + 1] = lvl_bound;
  }
}

// Adds the rows from the first NaN row on whose first coordinate is not NaN.  One workgroup for the 5.6e6 NaN
// rows of 2^24 took 9.4 ms; this 14 us, and 4 if there are none.
template <int D, typename T>
__global__ __launch_bounds__(kBuildThreads) void k_build_tail(const T* __restrict__ posz, int64_t n,
                                                              int32_t* __restrict__ state) {
  int c = 0;
  for (int64_t i = state[kBsTail] + (int64_t)blockIdx.x * kBuildThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBuildThreads) {
    const T x = posz[i * D];
    c += x == x ? 1 : 0;
  }
  c = __syncthreads_or(c) ? wave_reduce(c, [](int a, int b) { return a + b; }) : 0;
  if (c && (threadIdx.x & 63) == 0) atomicAdd(&state[kBsNpart], c);
}

// level histogram of the leaves, weighted with their particles (tree.py:236-240)
__global__ __launch_bounds__(kBuildThreads) void k_build_leaf_hist(const int32_t* __restrict__ spl, int64_t nleaf,
                                                                   const int32_t* __restrict__ lvl, int min_lvl, int nlvl,
                                                                   int use_lds, unsigned long long* __restrict__ hist) {
  extern __shared__ unsigned long long s_hist[];
  unsigned long long* const h = use_lds ? s_hist : hist;
  if (use_lds) {
    for (int j = threadIdx.x; j < nlvl; j += kBuildThreads) s_hist[j] = 0ull;
    __syncthreads();
  }
  for (int64_t i = (int64_t)blockIdx.x * kBuildThreads + threadIdx.x; i < nleaf;
       i += (int64_t)gridDim.x * kBuildThreads) {
    const int a = spl[i], b = spl[i + 1];
    if (b != a) {
      const int L = max(min(lvl[b], lvl[a]) - 1 - min_lvl, 0);
      if (L < nlvl) atomicAdd(&h[L], (unsigned long long)(int64_t)(b - a));
    }
  }
  if (use_lds) {
    __syncthreads();
    for (int j = threadIdx.x; j < nlvl; j += kBuildThreads)
      if (s_hist[j]) atomicAdd(&hist[j], s_hist[j]);
  }
}

// first particle (and set) of every leaf slot, and the number of leaves
template <int D, typename T>
__global__ void k_build_reps(const T* __restrict__ posz, int64_t n, const int32_t* __restrict__ spl, int64_t A,
                             const int32_t* __restrict__ set_id, T* __restrict__ reps, int32_t* __restrict__ leaf_set,
                             int32_t* __restrict__ state) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) state[kBsLeaves] = (int32_t)(min((int64_t)state[kBsFilled], A) - 1);
  if (i >= A - 1) return;
  const int64_t p = min((int64_t)spl[i], n - 1);
  store_vec<D, T>(reps, i, load_vec<D, T>(posz, p));
  if (set_id) leaf_set[i] = set_id[p];
}

// particles and plane activity of every leaf boundary (tree.py:664-700)
__global__ void k_build_mask(const int32_t* __restrict__ spl, const int32_t* __restrict__ lvl,
                             const int32_t* __restrict__ lb, const int32_t* __restrict__ rb, int64_t A, int nplanes,
                             PlaneSizes sizes, const int32_t* __restrict__ state, int sets, int32_t* __restrict__ npins,
                             uint32_t* __restrict__ mask) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A) return;
  const int nleaves = state[kBsLeaves];
  const int np = spl[rb[i]] - spl[lb[i]];
  bool always = (lb[i] <= 0 && lvl[i] > state[kBsLvlBound]) || (rb[i] >= nleaves && lvl[i] > state[kBsLvlBound + 1]);
  // set boundaries split every plane, and so do the two ends of a batch: a single-set tree only splits
  // those through the size or level tests, which can miss a small end set
  if (sets) always = always || lvl[i] >= kLvlSet || i == 0 || i == nleaves;
  uint32_t m = 0;
  for (int p = 0; p < nplanes; p++) m |= (always || np > sizes.v[p]) ? 1u << p : 0u;
  npins[i] = np;
  mask[i] = m;
}

// level histograms of the nodes of planes 1 ... (blockIdx.y + 1), weighted with their particles (tree.py:702-712)
__global__ __launch_bounds__(kBuildThreads) void k_build_node_hist(
    const int32_t* __restrict__ lvl, const int32_t* __restrict__ lb, const int32_t* __restrict__ rb,
    const int32_t* __restrict__ npins, const uint32_t* __restrict__ mask, int64_t A, const int32_t* __restrict__ state,
    int min_lvl, int nlvl, int use_lds, unsigned long long* __restrict__ hist_all) {
  extern __shared__ unsigned long long s_hist[];
  const int p = blockIdx.y + 1;
  unsigned long long* const hist = hist_all + (int64_t)p * nlvl;
  unsigned long long* const h = use_lds ? s_hist : hist;
  if (use_lds) {
    for (int j = threadIdx.x; j < nlvl; j += kBuildThreads) s_hist[j] = 0ull;
    __syncthreads();
  }
  const int64_t nb = min((int64_t)state[kBsLeaves], A);
  for (int64_t i = (int64_t)blockIdx.x * kBuildThreads + threadIdx.x; i < nb; i += (int64_t)gridDim.x * kBuildThreads) {
    const int l = lb[i], r = rb[i];
    if ((mask[i] >> p & 1u) || !(mask[l] >> p & 1u) || !(mask[r] >> p & 1u) || npins[i] == 0) continue;
    const int L = max(min(lvl[l], lvl[r]) - 1 - min_lvl, 0);
    if (L < nlvl) atomicAdd(&h[L], (unsigned long long)(int64_t)npins[i]);
  }
  if (use_lds) {
    __syncthreads();
    for (int j = threadIdx.x; j < nlvl; j += kBuildThreads)
      if (s_hist[j]) atomicAdd(&hist[j], s_hist[j]);
  }
}

// final activity (with the regularization levels), and its count per plane and tile
__global__ __launch_bounds__(kBuildThreads) void k_build_count(const int32_t* __restrict__ lvl,
                                                               const int32_t* __restrict__ npins,
                                                               uint32_t* __restrict__ mask, int64_t A, int nplanes,
                                                               const int32_t* __restrict__ state,
                                                               const int32_t* __restrict__ reg_lvl, int64_t ntiles,
                                                               int32_t* __restrict__ tiles) {
  __shared__ int s_n[kMaxPlanes];
  if (threadIdx.x < kMaxPlanes) s_n[threadIdx.x] = 0;
  __syncthreads();
  const int nleaves = state[kBsLeaves];
  for (int u = 0; u < kBuildPer; u++) {
    const int64_t i = (int64_t)blockIdx.x * kBuildTile + u * kBuildThreads + threadIdx.x;
    uint32_t m = 0;
    if (i < A) {
      m = mask[i];
      if (reg_lvl) {
        if (npins[i] > 0) m |= 1u;
        for (int p = 1; p < nplanes; p++)
          if (lvl[i] > reg_lvl[p] && i <= nleaves) m |= 1u << p;
        mask[i] = m;
      }
    }
    for (int p = 0; p < nplanes; p++) {
      const uint64_t b = __ballot(m >> p & 1u);
      if ((threadIdx.x & 63) == 0 && b) atomicAdd(&s_n[p], __popcll(b));
    }
  }
  __syncthreads();
  if (threadIdx.x < nplanes) tiles[threadIdx.x * ntiles + blockIdx.x] = s_n[threadIdx.x];
}

// the packed split arrays: an active boundary's slot is its rank among the active ones, plane after plane
__global__ __launch_bounds__(kBuildThreads) void k_build_splits(
    const int32_t* __restrict__ spl, const uint32_t* __restrict__ mask, int64_t A, int nplanes,
    const int32_t* __restrict__ tiles, int64_t ntiles, int32_t* __restrict__ n2l, int32_t* __restrict__ n2n) {
  __shared__ int sbuf[kBuildThreads / 64];
  const int64_t i0 = (int64_t)blockIdx.x * kBuildTile + (int64_t)threadIdx.x * kBuildPer;
  uint32_t m[kBuildPer];
  int off0[kBuildPer], prev[kBuildPer];
#pragma unroll
  for (int u = 0; u < kBuildPer; u++) m[u] = i0 + u < A ? mask[i0 + u] : 0u;
  const int total = tiles[nplanes * ntiles];
  int prev_start = 0;
  for (int p = 0; p < nplanes; p++) {
    int c = 0, tot;
#pragma unroll
    for (int u = 0; u < kBuildPer; u++) c += m[u] >> p & 1u;
    int o = tiles[p * ntiles + blockIdx.x] + block_excl_scan<kBuildThreads>(c, sbuf, &tot);
#pragma unroll
    for (int u = 0; u < kBuildPer; u++) {
      const bool on = m[u] >> p & 1u;
      const int slot = on ? o : (int)A;
      if (p == 0) off0[u] = slot;
      if (on && slot < A) {
        n2l[slot] = off0[u];
        n2n[slot] = p == 0 ? spl[i0 + u] : prev[u] - prev_start;
      }
      prev[u] = slot;
      o += on ? 1 : 0;
    }
    prev_start = tiles[p * ntiles];
  }
#pragma unroll
  for (int u = 0; u < kBuildPer; u++)
    if (i0 + u >= total && i0 + u < A) n2l[i0 + u] = n2n[i0 + u] = 0;
}

// level and cell centre of every packed node, without the slots between two planes, and the small arrays
template <int D, typename T>
__global__ void k_build_nodes(const T* __restrict__ posz, int64_t n, const int32_t* __restrict__ spl,
                              const int32_t* __restrict__ n2l, int64_t A, int nplanes, const int32_t* __restrict__ tiles,
                              int64_t ntiles, const int32_t* __restrict__ state, int lvl_invalid, int32_t* __restrict__ lvl,
                              T* __restrict__ cent, int32_t* __restrict__ level_spl, int32_t* __restrict__ n2l_fill,
                              int32_t* __restrict__ n2n_fill, int32_t* __restrict__ prop_spl, int32_t* __restrict__ lvl_fill,
                              T* __restrict__ cent_fill, int32_t* __restrict__ counts, uint8_t* __restrict__ err) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int total = tiles[nplanes * ntiles];
  if (i == 0) {
    int prop = 0;
    for (int p = 0; p < nplanes; p++) {
      const int a = tiles[p * ntiles], nodes = tiles[(p + 1) * ntiles] - a - 1;
      level_spl[p] = a;
      prop_spl[p] = prop;
      prop += nodes;
      n2l_fill[p] = tiles[ntiles] - 1;
      n2n_fill[p] = p == 0 ? spl[A - 1] : a - tiles[(p - 1) * ntiles] - 1;
      lvl_fill[p] = lvl_invalid;
      cent_fill[p] = quiet_nan<T>();
    }
    level_spl[nplanes] = total;
    prop_spl[nplanes] = prop;
    counts[0] = state[kBsFilled];
    counts[1] = nplanes;
    err[0] = state[kBsFilled] > A ? 1 : 0;
    err[1] = total > A ? 1 : 0;
  }
  if (i >= A - 1) return;
  // the slot at the end of a plane spans two planes: its row is left out (indices in range even after an
  // overflow, which is reported)
  int before = 0;
  int64_t last = -1;
  for (int p = 1; p < nplanes; p++) {
    const int64_t seam = min(max((int64_t)tiles[p * ntiles] - 1, (int64_t)0), A - 2);
    if (seam == i) return;
    before += seam < i && seam != last ? 1 : 0;
    last = seam;
  }
  const int64_t o = i - before;
  if (o >= A - nplanes) return;
  if (i >= total - 1) {
    lvl[o] = lvl_invalid;
#pragma unroll
    for (int d = 0; d < D; d++) cent[o * D + d] = quiet_nan<T>();
    return;
  }
  auto clip = [&](int64_t a, int64_t m) { return a < 0 ? (int64_t)0 : (a > m - 1 ? m - 1 : a); };
  const int64_t a = spl[clip(n2l[i], A)], b = spl[clip(n2l[i + 1], A)];
  const Vec<D, T> x0 = load_vec<D, T>(posz, clip(a, n)), x1 = load_vec<D, T>(posz, clip(b - 1, n));
  const int lv = msb_diff_level<D, T>(x0, x1);
  int l[D];
  lvl_vec<D>(lv, l);
  lvl[o] = lv;
#pragma unroll
  for (int d = 0; d < D; d++) cent[o * D + d] = round_pow2_cent(x0[d], l[d]);
}

// Per plane: the child splits (padded with the plane's fill value), and of every node the centre with the
// level's bits in the last column, the level and the particle count (data.py:199-239 of the reference).
template <int D, typename T>
__global__ void k_plane_tables(const int32_t* __restrict__ n2n, const int32_t* __restrict__ n2l,
                               const int32_t* __restrict__ level_spl, const int32_t* __restrict__ n2n_fill,
                               const int32_t* __restrict__ n2l_fill, const int32_t* __restrict__ lvl_in,
                               const T* __restrict__ cent, const int32_t* __restrict__ prop_spl,
                               const int32_t* __restrict__ spl, int64_t nspl, int64_t size, int64_t stride,
                               int32_t* __restrict__ out_spl, T* __restrict__ out_nodes, int32_t* __restrict__ out_lvl,
                               int32_t* __restrict__ out_npart) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int p = blockIdx.y;
  if (i > size) return;
  const int64_t a = level_spl[p], b = level_spl[p + 1];
  const int64_t A = size + 1;  // packed slots
  out_spl[p * stride + i] = a + i < b ? n2n[min(a + i, A - 1)] : n2n_fill[p];
  const int64_t pa = prop_spl[p], pb = prop_spl[p + 1];
  // rows past the plane's nodes are not read (nor are there rows for them after a reported overflow)
  if (i >= size || pa + i >= pb || pa + i >= A - (int64_t)gridDim.y) return;
  using TI = typename IntOf<T>::type;
  const int lv = lvl_in[pa + i];
#pragma unroll
  for (int d = 0; d < D; d++) out_nodes[(p * stride + i) * (D + 1) + d] = cent[(pa + i) * D + d];
  const TI bits = (TI)lv;
  out_nodes[(p * stride + i) * (D + 1) + D] = *reinterpret_cast<const T*>(&bits);
  out_lvl[p * stride + i] = lv;
  auto first = [&](int64_t j) {
    const int64_t leaf = a + j < b ? (int64_t)n2l[min(a + j, A - 1)] : (int64_t)n2l_fill[p];
    return spl[min(leaf, nspl - 1)];
  };
  out_npart[p * stride + i] = first(i + 1) - first(i);
}

struct BuildLayout {
  size_t flags, lvl, where, reps, lset, blvl, lb, rb, npins, mask, state, reg, hist, bins, tiles, total;
  int64_t ntiles;
  int nlvl;
};

BuildLayout build_layout(int64_t n, int64_t A, int nplanes, int dim, int dtype, bool reg) {
  BuildLayout L;
  const size_t es = dtype == JZT_F64 ? 8 : 4;
  size_t o = 0;
  auto take = [&](size_t b) {
    const size_t r = o;
    o = align256(o + b);
    return r;
  };
  L.ntiles = div_up(A, kBuildTile);
  L.nlvl = reg ? (dtype == JZT_F64 ? max_level<double>(dim) - min_level<double>(dim)
                                   : max_level<float>(dim) - min_level<float>(dim)) + 1 : 0;
  L.flags = take((size_t)n + 1);
  L.lvl = take(4 * (size_t)(n + 1));
  L.where = take(4 * (size_t)scan_tmp_words(n + 1));
  L.reps = take(es * dim * (size_t)A);
  L.lset = take(4 * (size_t)A);
  L.blvl = take(4 * (size_t)A);
  L.lb = take(4 * (size_t)A);
  L.rb = take(4 * (size_t)A);
  L.npins = take(4 * (size_t)A);
  L.mask = take(4 * (size_t)A);
  L.state = take(4 * kBsWords);
  L.reg = take(4 * (size_t)nplanes);
  L.hist = take(8 * (size_t)L.nlvl * nplanes);
  L.bins = take(4 * (size_t)L.nlvl * nplanes);
  L.tiles = take(4 * ((size_t)nplanes * L.ntiles + 1));
  L.total = o;
  return L;
}

struct BuildOut {
  int32_t *spl, *n2l, *n2n, *lvl;
  void* cent;
  int32_t *level_spl, *n2l_fill, *n2n_fill, *prop_spl, *lvl_fill;
  void* cent_fill;
  int32_t *counts, *leaf_set;
  uint8_t* err;
};

template <int D, typename T>
int build_tree_impl(hipStream_t s, const void* posz_v, const int32_t* set_id, const int32_t* npart_in, int64_t npart_host,
                    int64_t n, int dtype, const int32_t* node_sizes, int nplanes, int64_t A, int reg, float max_vol_fac,
                    float min_percentile, const BuildOut& out, char* tmp) {
  const BuildLayout L = build_layout(n, A, nplanes, D, dtype, reg != 0);
  const T* posz = (const T*)posz_v;
  int8_t* flags = (int8_t*)(tmp + L.flags);
  int32_t* lvl = (int32_t*)(tmp + L.lvl);
  int32_t* wtmp = (int32_t*)(tmp + L.where);
  T* reps = (T*)(tmp + L.reps);
  int32_t* lset = set_id ? out.leaf_set : nullptr;
  int32_t *blvl = (int32_t*)(tmp + L.blvl), *lb = (int32_t*)(tmp + L.lb), *rb = (int32_t*)(tmp + L.rb);
  int32_t* npins = (int32_t*)(tmp + L.npins);
  uint32_t* mask = (uint32_t*)(tmp + L.mask);
  int32_t* state = (int32_t*)(tmp + L.state);
  int32_t* reg_lvl = reg ? (int32_t*)(tmp + L.reg) : nullptr;
  unsigned long long* hist = (unsigned long long*)(tmp + L.hist);
  int32_t* bins = (int32_t*)(tmp + L.bins);
  int32_t* tiles = (int32_t*)(tmp + L.tiles);
  const int min_lvl = min_level<T>(D), max_lvl = max_level<T>(D);
  const int64_t hist_words = (int64_t)L.nlvl * nplanes * 2;
  const int lds = L.nlvl <= kRegLdsLevels ? 1 : 0;
  const size_t hshm = lds ? (size_t)L.nlvl * 8 : 0;
  const float frac = (float)(0.01 * (double)min_percentile);
  const unsigned gA = (unsigned)div_up(A, kBuildThreads);
  hipLaunchKernelGGL((k_build_init<D, T>), dim3((unsigned)(hist_words ? min(div_up(hist_words, kBuildThreads), (int64_t)64) : 1)),
                     dim3(kBuildThreads), 0, s, posz, n, npart_in, npart_host, n <= kBuildTailHere ? 1 : 0, max_lvl, state,
                     (uint32_t*)hist, hist_words);
  if (npart_in == nullptr && npart_host < 0 && n > kBuildTailHere)
    hipLaunchKernelGGL((k_build_tail<D, T>), dim3((unsigned)min(div_up(n, 4 * kBuildThreads), (int64_t)1024)),
                       dim3(kBuildThreads), 0, s, posz, n, state);
  if (flag_leaf_impl<D, T>(s, posz, nullptr, state + kBsLvlBound, state + kBsNpart, flags, lvl, n, node_sizes[0],
                           node_sizes[0] + 1, 1, set_id))
    return 1;
  if (reg) {
    if (where_flags_i8(s, flags, n + 1, out.spl, A, 0, state + kBsNpart, state + kBsFilled, wtmp)) return 1;
    hipLaunchKernelGGL(k_build_leaf_hist, dim3((unsigned)min((int64_t)gA, (int64_t)512)), dim3(kBuildThreads), hshm, s, out.spl,
                       A - 1, lvl, min_lvl, L.nlvl, lds, hist);
    hipLaunchKernelGGL(k_reg_level, dim3(1), dim3(kRegThreads), 0, s, hist, L.nlvl, min_lvl, max_lvl, max_vol_fac, frac, bins,
                       reg_lvl);
    if (flags_or_level_i8(s, flags, lvl, n + 1, reg_lvl, state + kBsNpart)) return 1;
  }
  if (where_flags_i8(s, flags, n + 1, out.spl, A, 0, state + kBsNpart, state + kBsFilled, wtmp)) return 1;
  hipLaunchKernelGGL((k_build_reps<D, T>), dim3(gA), dim3(kBuildThreads), 0, s, posz, n, out.spl, A, set_id, reps, lset, state);
  if (find_node_impl<D, T>(s, reps, nullptr, state + kBsLeaves, blvl, lb, rb, A, -2000, lset)) return 1;
  PlaneSizes ps;
  for (int p = 0; p < kMaxPlanes; p++) ps.v[p] = p < nplanes ? node_sizes[p] : 0;
  hipLaunchKernelGGL(k_build_mask, dim3(gA), dim3(kBuildThreads), 0, s, out.spl, blvl, lb, rb, A, nplanes, ps, state,
                     set_id ? 1 : 0, npins, mask);
  if (reg && nplanes > 1) {
    hipLaunchKernelGGL(k_build_node_hist, dim3((unsigned)min((int64_t)gA, (int64_t)256), (unsigned)(nplanes - 1)),
                       dim3(kBuildThreads), hshm, s, blvl, lb, rb, npins, mask, A, state, min_lvl, L.nlvl, lds, hist);
    hipLaunchKernelGGL(k_reg_level, dim3((unsigned)(nplanes - 1)), dim3(kRegThreads), 0, s, hist + L.nlvl, L.nlvl, min_lvl,
                       max_lvl, max_vol_fac, frac, bins + L.nlvl, reg_lvl + 1);
  }
  hipLaunchKernelGGL(k_build_count, dim3((unsigned)L.ntiles), dim3(kBuildThreads), 0, s, blvl, npins, mask, A, nplanes, state,
                     reg_lvl, L.ntiles, tiles);
  scan_tiles_i32(s, tiles, nplanes * L.ntiles);
  hipLaunchKernelGGL(k_build_splits, dim3((unsigned)L.ntiles), dim3(kBuildThreads), 0, s, out.spl, mask, A, nplanes, tiles,
                     L.ntiles, out.n2l, out.n2n);
  hipLaunchKernelGGL((k_build_nodes<D, T>), dim3(gA), dim3(kBuildThreads), 0, s, posz, n, out.spl, out.n2l, A, nplanes, tiles,
                     L.ntiles, state, -2000, out.lvl, (T*)out.cent, out.level_spl, out.n2l_fill, out.n2n_fill, out.prop_spl,
                     out.lvl_fill, (T*)out.cent_fill, out.counts, out.err);
  return check_launch("BuildTree");
}

template <int D, typename T>
int plane_tables_impl(hipStream_t s, const int32_t* n2n, const int32_t* n2l, const int32_t* level_spl,
                      const int32_t* n2n_fill, const int32_t* n2l_fill, const int32_t* lvl, const void* cent,
                      const int32_t* prop_spl, const int32_t* spl, int64_t nspl, int nplanes, int64_t size,
                      int32_t* out_spl, void* out_nodes, int32_t* out_lvl, int32_t* out_npart) {
  hipLaunchKernelGGL((k_plane_tables<D, T>), dim3((unsigned)div_up(size + 1, 256), (unsigned)nplanes), dim3(256), 0, s, n2n,
                     n2l, level_spl, n2n_fill, n2l_fill, lvl, (const T*)cent, prop_spl, spl, nspl, size, size + 1, out_spl,
                     (T*)out_nodes, out_lvl, out_npart);
  return check_launch("PlaneTables");
}

}  // namespace
}  // namespace jzt

using namespace jzt;

extern "C" int jzt_geometry_to_f32(jzt_stream_t stream, const double* cent, const int32_t* lvl, int64_t n, int dim,
                                   int lvl_invalid, float* cent_out, int32_t* lvl_out) {
  hipStream_t s = (hipStream_t)stream;
  if (n <= 0) return 0;
  const unsigned g = (unsigned)div_up(n, 256);
#define JZT_G2F(D)                                                                                                 \
  case D:                                                                                                          \
    hipLaunchKernelGGL(k_geometry_to_f32<D>, dim3(g), dim3(256), 0, s, cent, lvl, n, lvl_invalid, cent_out, lvl_out); \
    break;
  switch (dim) {
    JZT_G2F(2) JZT_G2F(3) JZT_G2F(4) JZT_G2F(5) JZT_G2F(6) JZT_G2F(7) JZT_G2F(8) JZT_G2F(9) JZT_G2F(10)
    default:
      return fail("GeometryToF32: unsupported dim");
  }
#undef JZT_G2F
  return check_launch("GeometryToF32");
}

extern "C" size_t jzt_regularization_tmp_bytes(int min_lvl, int max_lvl) {
  // the u64 histogram and the list of its nonzero bins
  const size_t nlvl = (size_t)(max_lvl - min_lvl + 1);
  return nlvl * 8 + nlvl * 4;
}

extern "C" int jzt_regularization_level(jzt_stream_t stream, const int32_t* lvl, const int32_t* weights, int64_t n,
                                        int32_t* out_level, int min_lvl, int max_lvl, float max_volume_fac,
                                        float min_percentile, void* tmp, size_t tmp_bytes) {
  hipStream_t s = (hipStream_t)stream;
  const int nlvl = max_lvl - min_lvl + 1;
  if (tmp_bytes < jzt_regularization_tmp_bytes(min_lvl, max_lvl)) return fail("regularization: tmp too small");
  if (nlvl < 1 || nlvl > (1 << 24)) return fail("regularization: level range out of bounds");
  const bool lds = nlvl <= kRegLdsLevels;
  if (fill_u32(s, tmp, 0u, (int64_t)nlvl * 2)) return 1;
  if (n > 0)
    hipLaunchKernelGGL(k_reg_hist, dim3((unsigned)min(div_up(n, 256), (int64_t)512)), dim3(256),
                       lds ? (size_t)nlvl * sizeof(unsigned long long) : 0, s, lvl, weights, n, min_lvl, nlvl,
                       (unsigned long long*)tmp);
  // 0.01*percentile is formed in double and rounded to float, as the reference's weak typing does
  const float frac = (float)(0.01 * (double)min_percentile);
  hipLaunchKernelGGL(k_reg_level, dim3(1), dim3(kRegThreads), 0, s, (const unsigned long long*)tmp, nlvl, min_lvl,
                     max_lvl, max_volume_fac, frac, (int32_t*)((char*)tmp + (size_t)nlvl * 8), out_level);
  return check_launch("regularization level");
}

// CenterOfMass (tree.cuh:378-429): per node, the mass-weighted mean of the points of its range
// [isplit[i], isplit[i+1]) and their total mass, out = (centre[D], mass) per node.  One thread per
// node sums its points in order, with Kahan compensation when `kahan` (the reference's default):
// y = m * x - c for a coordinate (formed as one fused multiply-add, the form a contracting
// compiler gives the reference's m * x followed by "add - c"), y = m - c for the mass, then
// t = sum + y, c = (t - sum) - y, sum = t.  The centre is (1 / mass) * sum.  An empty range or a
// non-positive total mass gives NaN in every slot.
template <int D, typename T>
__global__ void k_center_of_mass(const int32_t* __restrict__ isplit, const T* __restrict__ pos,
                                 const T* __restrict__ mass, T* __restrict__ out, int64_t nnodes, int kahan) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnodes) return;
  const int s0 = isplit[i], s1 = isplit[i + 1];
  const T nan = (T)__builtin_nan("");
  T sum[D + 1], c[D + 1];
#pragma unroll
  for (int d = 0; d <= D; d++) sum[d] = c[d] = T(0);
  for (int p = s0; p < s1; p++) {
    const T m = mass[p];
#pragma unroll
    for (int d = 0; d <= D; d++) {
      const T x = d < D ? pos[(int64_t)p * D + d] : T(1);
      if (kahan) {
        const T y = d < D ? fmaT(m, x, -c[d]) : m - c[d];
        const T t = sum[d] + y;
        c[d] = (t - sum[d]) - y;
        sum[d] = t;
      } else {
        sum[d] = d < D ? fmaT(m, x, sum[d]) : sum[d] + m;
      }
    }
  }
  if (s0 < s1 && sum[D] > T(0)) {
    const T inv = T(1) / sum[D];
#pragma unroll
    for (int d = 0; d < D; d++) out[i * (D + 1) + d] = inv * sum[d];
    out[i * (D + 1) + D] = sum[D];
  } else {
#pragma unroll
    for (int d = 0; d <= D; d++) out[i * (D + 1) + d] = nan;
  }
}

template <int D, typename T>
int com_impl(hipStream_t s, const int32_t* isplit, const void* pos, const void* mass, void* out, int64_t nnodes,
             int kahan) {
  if (nnodes <= 0) return 0;
  hipLaunchKernelGGL((k_center_of_mass<D, T>), dim3((unsigned)div_up(nnodes, 256)), dim3(256), 0, s, isplit,
                     (const T*)pos, (const T*)mass, (T*)out, nnodes, kahan);
  return check_launch("CenterOfMass");
}

// single-set tree kernels: dims 2-10 (the reference's instances, _generate_ffi.py:9-21)
#define JZT_DISPATCH_ND(fn, ...)                                                  \
  do {                                                                            \
    switch ((dtype == JZT_F64 ? 100 : 0) + dim) {                                 \
      case 2: return fn<2, float>(__VA_ARGS__);                                   \
      case 3: return fn<3, float>(__VA_ARGS__);                                   \
      case 4: return fn<4, float>(__VA_ARGS__);                                   \
      case 5: return fn<5, float>(__VA_ARGS__);                                   \
      case 6: return fn<6, float>(__VA_ARGS__);                                   \
      case 7: return fn<7, float>(__VA_ARGS__);                                   \
      case 8: return fn<8, float>(__VA_ARGS__);                                   \
      case 9: return fn<9, float>(__VA_ARGS__);                                   \
      case 10: return fn<10, float>(__VA_ARGS__);                                 \
      case 102: return fn<2, double>(__VA_ARGS__);                                \
      case 103: return fn<3, double>(__VA_ARGS__);                                \
      case 104: return fn<4, double>(__VA_ARGS__);                                \
      case 105: return fn<5, double>(__VA_ARGS__);                                \
      case 106: return fn<6, double>(__VA_ARGS__);                                \
      case 107: return fn<7, double>(__VA_ARGS__);                                \
      case 108: return fn<8, double>(__VA_ARGS__);                                \
      case 109: return fn<9, double>(__VA_ARGS__);                                \
      case 110: return fn<10, double>(__VA_ARGS__);                               \
      default: break;                                                             \
    }                                                                             \
    return fail(std::string(#fn) + ": unsupported dim/dtype");                    \
  } while (0)

#define JZT_DISPATCH(fn, ...)                                                     \
  do {                                                                            \
    if (dtype == JZT_F32 && dim == 3) return fn<3, float>(__VA_ARGS__);           \
    if (dtype == JZT_F32 && dim == 2) return fn<2, float>(__VA_ARGS__);           \
    if (dtype == JZT_F64 && dim == 3) return fn<3, double>(__VA_ARGS__);          \
    if (dtype == JZT_F64 && dim == 2) return fn<2, double>(__VA_ARGS__);          \
    return fail(std::string(#fn) + ": unsupported dim/dtype");                    \
  } while (0)

extern "C" int jzt_flag_leaf_boundaries(jzt_stream_t stream, const void* posz, const uint8_t* ptype,
                                        const int32_t* lvl_bound, const int32_t* npart, int8_t* split_flags,
                                        int32_t* lvl, int64_t size_part, int dim, int dtype, int max_size,
                                        int scan_size, int num_types) {
  if (num_types > 1 && ptype == nullptr) return fail("FlagLeafBoundaries: ptype required for num_types > 1");
  JZT_DISPATCH_ND(flag_leaf_impl, (hipStream_t)stream, posz, ptype, lvl_bound, npart, split_flags, lvl, size_part,
                  max_size, scan_size, num_types, (const int32_t*)nullptr);
}

extern "C" int jzt_flag_leaf_boundaries_sets(jzt_stream_t stream, const void* posz, const int32_t* set_id,
                                             const int32_t* lvl_bound, const int32_t* npart, int8_t* split_flags,
                                             int32_t* lvl, int64_t size_part, int dim, int dtype, int max_size,
                                             int scan_size) {
  if (set_id == nullptr) return fail("FlagLeafBoundaries (sets): set_id is required");
  JZT_DISPATCH(flag_leaf_impl, (hipStream_t)stream, posz, (const uint8_t*)nullptr, lvl_bound, npart, split_flags, lvl,
               size_part, max_size, scan_size, 1, set_id);
}

extern "C" int jzt_find_node_boundaries(jzt_stream_t stream, const void* pos_in, const void* pos_boundary,
                                        const int32_t* nleaves, int32_t* nodes_levels, int32_t* nodes_lbound,
                                        int32_t* nodes_rbound, int64_t size_nodes, int dim, int dtype, int lvl_max,
                                        int lvl_invalid) {
  (void)lvl_max;  // the reference passes it but its kernel never reads it outside dead stores (tree.cuh:144-196)
  if (size_nodes <= 0) return 0;
  JZT_DISPATCH_ND(find_node_impl, (hipStream_t)stream, pos_in, pos_boundary, nleaves, nodes_levels, nodes_lbound,
                  nodes_rbound, size_nodes, lvl_invalid, (const int32_t*)nullptr);
}

extern "C" int jzt_find_node_boundaries_sets(jzt_stream_t stream, const void* pos_in, const int32_t* set_id,
                                             const void* pos_boundary, const int32_t* nleaves, int32_t* nodes_levels,
                                             int32_t* nodes_lbound, int32_t* nodes_rbound, int64_t size_nodes, int dim,
                                             int dtype, int lvl_invalid) {
  if (set_id == nullptr) return fail("FindNodeBoundaries (sets): set_id is required");
  if (size_nodes <= 0) return 0;
  JZT_DISPATCH(find_node_impl, (hipStream_t)stream, pos_in, pos_boundary, nleaves, nodes_levels, nodes_lbound,
               nodes_rbound, size_nodes, lvl_invalid, set_id);
}

extern "C" int jzt_get_node_geometry(jzt_stream_t stream, const void* pos, const int32_t* lbound, const int32_t* rbound,
                                     const int32_t* nnodes, int32_t* level, void* center, void* extent,
                                     int64_t size_nodes, int64_t size_part, int dim, int dtype, int lvl_invalid,
                                     uint32_t mode_flags, int upper_extent) {
  if (size_nodes <= 0) return 0;
  JZT_DISPATCH_ND(geometry_impl, (hipStream_t)stream, pos, lbound, rbound, nnodes, level, center, extent, size_nodes,
                  size_part, lvl_invalid, mode_flags, upper_extent);
}

extern "C" size_t jzt_where_tmp_bytes(int64_t n) { return (size_t)(scan_tmp_words(n) + n) * 4; }

extern "C" int jzt_where_flags(jzt_stream_t stream, const int8_t* flags, int64_t n, int32_t* out, int64_t size,
                               int32_t fill, const int32_t* fill_dev, int32_t* count, void* tmp, size_t tmp_bytes) {
  if (tmp_bytes < jzt_where_tmp_bytes(n)) return fail("jzt_where_flags: tmp too small");
  return where_flags_i8((hipStream_t)stream, flags, n, out, size, fill, fill_dev, count, (int32_t*)tmp);
}

extern "C" int jzt_center_of_mass(jzt_stream_t stream, const int32_t* isplit, const void* pos, const void* mass,
                                  void* com_out, int64_t nnodes, int kahan, int dim, int dtype) {
  JZT_DISPATCH_ND(com_impl, (hipStream_t)stream, isplit, pos, mass, com_out, nnodes, kahan);
}

extern "C" size_t jzt_build_tree_tmp_bytes(int64_t size_part, int64_t alloc_size, int nplanes, int dim, int dtype,
                                           int regularize) {
  if (size_part < 0 || alloc_size < 1 || nplanes < 1 || dim < 1) return 0;
  return build_layout(size_part, alloc_size, nplanes, dim, dtype, regularize != 0).total;
}

extern "C" int jzt_build_tree(jzt_stream_t stream, const void* posz, const int32_t* set_id, const int32_t* npart,
                              int64_t npart_host, int64_t size_part, int dim, int dtype, const int32_t* node_sizes,
                              int nplanes, int64_t alloc_size, int regularize, float max_volume_fac,
                              float min_percentile, int32_t* leaf_spl, int32_t* n2l, int32_t* n2n, int32_t* level_spl,
                              int32_t* n2l_fill, int32_t* n2n_fill, int32_t* lvl, void* cent, int32_t* prop_spl,
                              int32_t* lvl_fill, void* cent_fill, int32_t* counts, int32_t* leaf_set, uint8_t* err,
                              void* tmp, size_t tmp_bytes) {
  if (size_part < 1 || nplanes < 1 || nplanes > kMaxPlanes || alloc_size < nplanes + 1)
    return fail("BuildTree: empty input, too many planes or too small an allocation");
  if (set_id != nullptr && (leaf_set == nullptr || regularize)) return fail("BuildTree: batches need leaf_set and take no regularization");
  if (dim < 2 || dim > 10 || (dtype != JZT_F32 && dtype != JZT_F64)) return fail("BuildTree: unsupported dim/dtype");
  if (tmp_bytes < jzt_build_tree_tmp_bytes(size_part, alloc_size, nplanes, dim, dtype, regularize))
    return fail("BuildTree: tmp too small");
  const BuildOut out{leaf_spl, n2l, n2n, lvl, cent, level_spl, n2l_fill, n2n_fill, prop_spl, lvl_fill, cent_fill,
                     counts, leaf_set, err};
  JZT_DISPATCH_ND(build_tree_impl, (hipStream_t)stream, posz, set_id, npart, npart_host, size_part, dtype, node_sizes,
                  nplanes, alloc_size, regularize, max_volume_fac, min_percentile, out, (char*)tmp);
}

extern "C" int jzt_plane_tables(jzt_stream_t stream, const int32_t* n2n, const int32_t* n2l, const int32_t* level_spl,
                                const int32_t* n2n_fill, const int32_t* n2l_fill, const int32_t* lvl, const void* cent,
                                const int32_t* prop_spl, const int32_t* leaf_spl, int64_t size_leaf_spl, int nplanes,
                                int64_t size_nodes, int dim, int dtype, int32_t* out_spl, void* out_nodes,
                                int32_t* out_lvl, int32_t* out_npart) {
  if (nplanes < 1 || size_nodes < 1 || size_leaf_spl < 1) return fail("PlaneTables: empty tree");
  JZT_DISPATCH_ND(plane_tables_impl, (hipStream_t)stream, n2n, n2l, level_spl, n2n_fill, n2l_fill, lvl, cent, prop_spl,
                  leaf_spl, size_leaf_spl, nplanes, size_nodes, out_spl, out_nodes, out_lvl, out_npart);
}
