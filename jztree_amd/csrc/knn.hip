// Exact k-nearest-neighbour search (replaces jztree's knn.cuh).
//
// KnnNode2Node (knn.cuh:435-694): for every child node Q of a parent, walk the parent's
//   r2-sorted interaction list and
//     find      the smallest maxdist2 within which >= k particles are guaranteed; that radius
//               (times 1 + 2^-16) bounds the k-th neighbour of every point in Q
//     count,    then, after a scan of the counts, list every child T of the listed parents with
//     insert    mindist2(Q,T) <= rmax2(Q)
//     sort      each node's list ascending by (r2, src)
//   node_tiles.h has the work split.
//
// KnnLeaf2Leaf (knn.cuh:203-356): one wave64 per query leaf, one query per lane.  The leaf's
//   interaction list is walked in ascending r2 and stops once no lane could still accept
//   (r2T > kth*(1+2^-16) on all lanes).  Source particles are read at wave-uniform addresses
//   (scalar loads, broadcast to all lanes); each lane keeps its k best (r2, id) pairs sorted in
//   VGPRs as 64-bit keys (r2 bits << 32 | id), inserted with a static compare/select network.
//   k > 64 runs ceil(k/64) passes, each resuming after the previous pass's last key.
//
// Order: ascending by (canonical FP32 r2, reported id).  The reference inserts with strict '<' in
// visit order (knn.cuh:84-102), so its tie order depends on the traversal; here it does not.
#include "util.h"
#include "knn_common.h"
#include "knn_nd.h"
#include "node_tiles.h"
#include "../../include/jztree_amd.h"

namespace jzt {
namespace {

constexpr float kRmaxSlack = 1.0f + kBoundSlack;

template <int D, typename T> struct NodeT {
  Vec<D, T> cent;
  int level;
};

template <int D, typename T>
__device__ __forceinline__ NodeT<D, T> load_node(const T* __restrict__ nodes, int64_t i) {
  NodeT<D, T> n;
#pragma unroll
  for (int d = 0; d < D; d++) n.cent[d] = nodes[i * (D + 1) + d];
  T lv = nodes[i * (D + 1) + D];
  if constexpr (sizeof(T) == 4) n.level = __float_as_int(lv);
  else n.level = (int)__double_as_longlong(lv);
  return n;
}

template <int D, typename T>
__device__ __forceinline__ Vec<D, T> add(const Vec<D, T>& a, const Vec<D, T>& b) {
  Vec<D, T> r;
#pragma unroll
  for (int d = 0; d < D; d++) r[d] = a[d] + b[d];
  return r;
}

// ------------------------------------------------------------------------------------------------
// guaranteed k-neighbour radius of a node, and the nodes within it
// ------------------------------------------------------------------------------------------------
// The guaranteed radius^2 of a child Q is the smallest R such that the nodes T with maxdist2(Q, T) <= R
// hold at least k particles (knn.cuh:106-191 keeps 8 to 32 bins of (maxdist2, count) per child and
// merges the rest; here the selection is exact).  A node that holds k particles itself starts at its
// own squared diagonal.  Candidates below the current radius go into the child's LDS buffer; a wave
// then sums, for every buffered entry, the particles of the entries up to it, and the smallest entry
// that reaches k is the new radius; entries beyond it are dropped.
//
// Cost: about 40 VALU instructions per child pair, and the latency of the list walk (entry, children
// range, node) where a parent has few pairs.  KnnNode2Node of 2^24 clustered points, leaf 48, k = 32: the
// leaf plane (8e8 child pairs, 1.4e8 list entries) takes 3.0 ms for the radii and counts and 1.2 ms for the
// lists, the top plane (1.5e8 pairs) 0.7 and 0.3 ms; one wave per parent, walking its list entry by entry,
// took 18.2 and 12.0 ms for the two planes without the list sort.
constexpr int kNodeKeep = 64;   // entries a child keeps after a reduction
constexpr int kNodeLazy = 32;   // new entries that trigger one

template <int D, typename T> struct NodeChild {
  Vec<D, T> c, e;
};

template <int NT> struct RadiusLds {
  static constexpr int kCap = kNodeKeep + kNodeLazy + NT;
  float r[kNodeChildren][kCap];
  int w[kNodeChildren][kCap];
  int n[kNodeChildren];       // entries in the buffer
  int kept[kNodeChildren];    // of them left by the last reduction
};

// Smallest radius^2 among the wave's entries (radius r, w particles; w = 0: none) up to which they hold at
// least k particles; +inf if they hold fewer.  `in`: the lanes with an entry.  Every entry is broadcast
// with readlane and added where it does not lie beyond the lane's own: about six instructions per
// entry and no wait for LDS (broadcast from LDS, the same loop waited 64 times for a read).
__device__ __forceinline__ float wave_select(float r, int w, uint64_t in, int k) {
  int sum = 0;
  for (uint64_t b = in; b; b &= b - 1ull) {
    const int j = __builtin_ctzll(b);
    const float rj = rdlane(r, j);
    const int wj = rdlane(w, j);
    sum += rj <= r ? wj : 0;
  }
  return wave_minf(w > 0 && sum >= k ? r : INFINITY);
}

// One wave reduces the buffer of child c: returns the smallest radius^2 that its entries guarantee
// (+inf if they hold fewer than k particles) and compacts the buffer to the entries below it and one
// entry for the radius itself.  At most k entries stay (every entry holds a particle); with k > kNodeKeep
// they are merged in order, each group taking its largest radius, which is still guaranteed.
template <int NT> __device__ __forceinline__ float node_radius_reduce(RadiusLds<NT>& s, int c, int k) {
  constexpr int E = (RadiusLds<NT>::kCap + 63) / 64;
  const int lane = threadIdx.x & 63;
  const int m = __builtin_amdgcn_readfirstlane(s.n[c]);
  float r[E];
  int w[E];
#pragma unroll
  for (int i = 0; i < E; i++) {
    const int me = i * 64 + lane;
    r[i] = me < m ? s.r[c][me] : INFINITY;
    w[i] = me < m ? s.w[c][me] : 0;
  }
  float best = INFINITY;
  if (m <= 64) {
    best = wave_select(r[0], w[0], m == 64 ? ~0ull : (1ull << m) - 1ull, k);
  } else {
    int sum[E];
#pragma unroll
    for (int i = 0; i < E; i++) sum[i] = 0;
#pragma unroll
    for (int i2 = 0; i2 < E; i2++) {
      for (int j = 0; j < min(64, m - i2 * 64); j++) {
        const float rj = rdlane(r[i2], j);
        const int wj = rdlane(w[i2], j);
#pragma unroll
        for (int i = 0; i < E; i++) sum[i] += rj <= r[i] ? wj : 0;
      }
    }
#pragma unroll
    for (int i = 0; i < E; i++)
      if (w[i] > 0 && sum[i] >= k) best = fminf(best, r[i]);
    best = wave_minf(best);
  }
  // entries that stay: strictly below the radius
  int kept = 0;
  const uint64_t lt_mask = (1ull << lane) - 1ull;
#pragma unroll
  for (int i = 0; i < E; i++) {
    const bool keep = w[i] > 0 && r[i] < best;
    const uint64_t b = __ballot(keep);
    if (keep) {
      const int o = kept + __popcll(b & lt_mask);
      s.r[c][o] = r[i];
      s.w[c][o] = w[i];
    }
    kept += __popcll(b);
  }
  if (best < INFINITY) {
    if (lane == 0) {
      s.r[c][kept] = best;
      s.w[c][kept] = k;
    }
    kept++;
  }
  if (kept > kNodeKeep) {
    // merge groups of q entries that are consecutive in (radius, slot) order
    const int q = (kept + kNodeKeep - 1) / kNodeKeep;
    int slot[E];
    bool top[E];
#pragma unroll
    for (int i = 0; i < E; i++) {
      const int me = i * 64 + lane;
      int rank = 0;
      r[i] = me < kept ? s.r[c][me] : INFINITY;
      w[i] = me < kept ? s.w[c][me] : 0;
      if (i * 64 < kept) {
        for (int j = 0; j < kept; j++) {
          const float rj = s.r[c][j];
          rank += (rj < r[i] || (rj == r[i] && j < me)) ? 1 : 0;
        }
      }
      slot[i] = rank / q;
      top[i] = rank % q == q - 1 || rank == kept - 1;
    }
    const int groups = (kept + q - 1) / q;
    if (lane < groups) s.w[c][lane] = 0;  // groups <= kNodeKeep = 64
#pragma unroll
    for (int i = 0; i < E; i++) {
      if (i * 64 + lane < kept) {
        atomicAdd(&s.w[c][slot[i]], w[i]);
        if (top[i]) s.r[c][slot[i]] = r[i];
      }
    }
    kept = groups;
  }
  if (lane == 0) {
    s.n[c] = kept;
    s.kept[c] = kept;
  }
  return best;
}

// RADIUS: find the guaranteed radii (written to rmax2, slack included), else read them from rmax2; in both
// cases count, for every child, the children of the listed parents within its radius.
template <bool RADIUS, int NT, int D, typename T>
__global__ __launch_bounds__(NT) void k_node_count(
    const int32_t* __restrict__ pil_spl, const int32_t* __restrict__ pil_src, const float* __restrict__ pil_r2,
    const int32_t* __restrict__ parent_spl, const T* __restrict__ nodes, const int32_t* __restrict__ npart,
    const float* __restrict__ parent_rmax2, float* __restrict__ rmax2, int32_t* __restrict__ count_out, int k, T boxsize, int64_t pil_size, int64_t nitems,
    int nnodes, NodeQueue queue) {
  __shared__ TileLds<NT> s_t;
  __shared__ NodeChild<D, T> s_q[kNodeChildren];
  __shared__ float s_R[kNodeChildren];
  __shared__ int s_cnt[kNodeChildren];
  __shared__ typename std::conditional<RADIUS, RadiusLds<NT>, int>::type s_b;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint64_t lt_mask = (1ull << lane) - 1ull;
  // one-wave workgroups take all parents but those with long lists, the larger ones the queue's
  const int64_t nact = NT == 64 ? active_items(parent_spl, nitems) : min((int64_t)queue.q[0], queue.most);
  const NodeGroups ng = NT == 64 ? node_groups(nact) : NodeGroups{4, kNodeChildren};
  for (int64_t item = blockIdx.x; item < nact * ng.groups; item += gridDim.x) {
    const int grp = (int)(item / nact), ip = (int)(item - grp * nact);  // see node_groups
    const int pq = NT == 64 ? ip : queue.q[1 + ip];
    const int q1 = min(parent_spl[pq + 1], nnodes);
    const int e0 = pil_spl[pq], e1 = (int)min((int64_t)pil_spl[pq + 1], pil_size);
    if (NT == 64 && queue.is_long(e1 - e0)) {
      if (grp == 0 && tid == 0) queue.push(pq);
      continue;
    }
    for (int q0 = parent_spl[pq] + grp * ng.width; q0 < q1; q0 += ng.groups * ng.width) {
      const int nc = min(q1 - q0, ng.width);
      __syncthreads();  // the previous round's readers are done
      if (tid < nc) {
        const NodeT<D, T> nq = load_node<D, T>(nodes, q0 + tid);
        NodeChild<D, T> q;
        q.c = nq.cent;
        q.e = lvl_half_ext<D, T>(nq.level);
        s_q[tid] = q;
        s_cnt[tid] = 0;
        if constexpr (RADIUS) {
          s_b.n[tid] = 0;
          s_b.kept[tid] = 0;
          // radii known before any list entry: the parent's (it holds for every point of the parent) and,
          // if the node holds k particles itself, its squared diagonal
          float r0 = parent_rmax2 ? parent_rmax2[pq] : INFINITY;
          if (npart[q0 + tid] >= k) r0 = fminf(r0, (float)maxdist2<D, T>(q.c, q.c, add<D, T>(q.e, q.e), boxsize));
          s_R[tid] = r0;
        } else {
          s_R[tid] = rmax2[q0 + tid];
        }
      }
      __syncthreads();
      if constexpr (RADIUS) {
        bool first = true;
        for (int eb = e0; eb < e1; eb += NT) {
          float rtop = s_R[0];
          for (int c = 1; c < nc; c++) rtop = fmaxf(rtop, s_R[c]);
          rtop *= kRmaxSlack;
          const int ne = min(NT, e1 - eb);
          int t0 = 0, cnt = 0, tot;
          float r2t = INFINITY;
          if (tid < ne) {
            r2t = pil_r2[eb + tid];
            if (r2t <= rtop) {
              const int pt = pil_src[eb + tid];
              t0 = parent_spl[pt];
              cnt = max(min(parent_spl[pt + 1], nnodes) - t0, 0);
            }
          }
          const int pre = block_excl_scan<NT>(cnt, s_t.scan, &tot);
          s_t.pre[tid] = pre;
          s_t.off[tid] = t0 - pre;
          int act = __syncthreads_count(tid < ne && r2t <= rtop);  // entries ascend by r2: a prefix
          int lim = tot;
          for (int base = 0; base < lim;) {
            // the first tile (the node, its siblings and its nearest neighbours) is a short one:
            // its reduction gives a radius that keeps nearly all later targets out of the buffer
            const int width = first ? 64 : NT;
            const int j = base + tid;
            const bool valid = tid < width && j < lim;
            const int e = tile_entry<NT>(s_t, ne, valid ? j : 0);
            int np = 0;
            NodeChild<D, T> t;
            if (valid) {
              const int it = j + s_t.off[e];
              const NodeT<D, T> nt = load_node<D, T>(nodes, it);
              t.c = nt.cent;
              t.e = lvl_half_ext<D, T>(nt.level);
              np = npart[it];
            }
            for (int c = 0; c < nc; c++) {
              bool cand = false;
              float r2 = 0.f;
              if (np > 0) {
                r2 = (float)maxdist2<D, T>(t.c, s_q[c].c, add<D, T>(s_q[c].e, t.e), boxsize);
                cand = r2 < s_R[c];
              }
              uint64_t hits = __ballot(cand);
              if (hits) {
                if (first) {  // one wave holds the whole first tile: select before anything is stored
                  const float rn = wave_select(cand ? r2 : INFINITY, cand ? np : 0, hits, k);
                  cand = cand && (r2 < rn || rn == INFINITY);
                  hits = __ballot(cand);
                  if (rn < INFINITY) {
                    if (lane == 0) {
                      s_R[c] = rn;
                      s_b.r[c][0] = rn;
                      s_b.w[c][0] = k;
                      s_b.n[c] = 1;
                    }
                  }
                }
                int o = 0;
                if (lane == 0) o = atomicAdd(&s_b.n[c], __popcll(hits));
                o = __builtin_amdgcn_readfirstlane(o) + __popcll(hits & lt_mask);
                if (cand) {
                  s_b.r[c][o] = r2;
                  s_b.w[c][o] = np;
                }
                if (first && lane == 0) s_b.kept[c] = s_b.n[c];
              }
            }
            __syncthreads();
            bool any = false;
            for (int c = 0; c < nc; c++) any |= first || s_b.n[c] - s_b.kept[c] >= kNodeLazy;
            __syncthreads();  // all have read the fills before the reductions change them
            if (any) {
              for (int c = w; c < nc; c += NT / 64) {
                if (s_b.n[c] > s_b.kept[c]) {
                  const float rn = node_radius_reduce(s_b, c, k);
                  if (lane == 0) s_R[c] = fminf(s_R[c], rn);
                }
              }
              __syncthreads();
              rtop = s_R[0];
              for (int c = 1; c < nc; c++) rtop = fmaxf(rtop, s_R[c]);
              rtop *= kRmaxSlack;
              act = __syncthreads_count(tid < ne && r2t <= rtop);
              lim = act < ne ? min(lim, s_t.pre[act]) : lim;
            }
            base += width;
            first = false;
          }
          const bool more = act == ne;
          __syncthreads();
          if (!more) break;
        }
        for (int c = w; c < nc; c += NT / 64) {
          float rn = INFINITY;
          if (s_b.n[c] > s_b.kept[c]) rn = node_radius_reduce(s_b, c, k);
          if (lane == 0) {
            rn = fminf(s_R[c], rn) * kRmaxSlack;
            s_R[c] = rn;
            rmax2[q0 + c] = rn;
          }
        }
        __syncthreads();
      }
      float rtop = s_R[0];
      for (int c = 1; c < nc; c++) rtop = fmaxf(rtop, s_R[c]);
      for_target_tiles<NT>(
          s_t, e0, e1,
          [&](int e, int& t0, int& cnt) {
            const bool in = pil_r2[e] <= rtop;
            if (in) {
              const int pt = pil_src[e];
              t0 = parent_spl[pt];
              cnt = max(min(parent_spl[pt + 1], nnodes) - t0, 0);
            }
            return in;
          },
          [&](bool valid, int it) {
            const NodeT<D, T> nt = load_node<D, T>(nodes, it);
            const Vec<D, T> te = lvl_half_ext<D, T>(nt.level);
            for (int c = 0; c < nc; c++) {
              const float r2 = (float)mindist2<D, T>(nt.cent, s_q[c].c, add<D, T>(s_q[c].e, te), boxsize);
              const uint64_t hits = __ballot(valid && r2 <= s_R[c]);
              if (hits && lane == 0) atomicAdd(&s_cnt[c], __popcll(hits));
            }
          });
      if (tid < nc) count_out[q0 + tid] = s_cnt[tid];
    }
  }
}

// The same pairs as k_node_count's, written to the children's lists.  A child's slots are handed out by
// an LDS counter, a wave's hits at a time, so the order inside a list is arbitrary; every list is sorted by
// (r2, src) afterwards and its pairs are unique, so the lists do not depend on it.
template <int NT, int D, typename T>
__global__ __launch_bounds__(NT) void k_node_insert(
    const int32_t* __restrict__ pil_spl, const int32_t* __restrict__ pil_src, const float* __restrict__ pil_r2,
    const int32_t* __restrict__ parent_spl, const T* __restrict__ nodes, const float* __restrict__ rmax2,
    const int32_t* __restrict__ out_spl, int32_t* __restrict__ out_src, float* __restrict__ out_r2, int64_t nmax,
    T boxsize, int64_t pil_size, int64_t nitems, int nnodes, uint8_t* __restrict__ overflow, NodeQueue queue) {
  __shared__ TileLds<NT> s_t;
  __shared__ NodeChild<D, T> s_q[kNodeChildren];
  __shared__ float s_R[kNodeChildren];
  __shared__ int s_run[kNodeChildren];  // hits so far
  __shared__ int s_out[kNodeChildren];  // first list slot
  if (NT == 64 && overflow && blockIdx.x == 0 && threadIdx.x == 0) *overflow = (int64_t)out_spl[nnodes] > nmax ? 1 : 0;
  const int tid = threadIdx.x, lane = tid & 63;
  const uint64_t lt_mask = (1ull << lane) - 1ull;
  // one-wave workgroups take all parents but those with long lists, the larger ones the queue's
  const int64_t nact = NT == 64 ? active_items(parent_spl, nitems) : min((int64_t)queue.q[0], queue.most);
  const NodeGroups ng = NT == 64 ? node_groups(nact) : NodeGroups{4, kNodeChildren};
  for (int64_t item = blockIdx.x; item < nact * ng.groups; item += gridDim.x) {
    const int grp = (int)(item / nact), ip = (int)(item - grp * nact);  // see node_groups
    const int pq = NT == 64 ? ip : queue.q[1 + ip];
    const int q1 = min(parent_spl[pq + 1], nnodes);
    const int e0 = pil_spl[pq], e1 = (int)min((int64_t)pil_spl[pq + 1], pil_size);
    if (NT == 64 && queue.is_long(e1 - e0)) {
      continue;
    }
    for (int q0 = parent_spl[pq] + grp * ng.width; q0 < q1; q0 += ng.groups * ng.width) {
      const int nc = min(q1 - q0, ng.width);
      __syncthreads();
      if (tid < nc) {
        const NodeT<D, T> nq = load_node<D, T>(nodes, q0 + tid);
        NodeChild<D, T> q;
        q.c = nq.cent;
        q.e = lvl_half_ext<D, T>(nq.level);
        s_q[tid] = q;
        s_R[tid] = rmax2[q0 + tid];
        s_run[tid] = 0;
        s_out[tid] = out_spl[q0 + tid];
      }
      __syncthreads();
      float rtop = s_R[0];
      for (int c = 1; c < nc; c++) rtop = fmaxf(rtop, s_R[c]);
      for_target_tiles<NT>(
          s_t, e0, e1,
          [&](int e, int& t0, int& cnt) {
            const bool in = pil_r2[e] <= rtop;
            if (in) {
              const int pt = pil_src[e];
              t0 = parent_spl[pt];
              cnt = max(min(parent_spl[pt + 1], nnodes) - t0, 0);
            }
            return in;
          },
          [&](bool valid, int it) {
            const NodeT<D, T> nt = load_node<D, T>(nodes, it);
            const Vec<D, T> te = lvl_half_ext<D, T>(nt.level);
            for (int c = 0; c < nc; c++) {
              const Vec<D, T> ew = add<D, T>(s_q[c].e, te);
              float r2 = (float)mindist2<D, T>(nt.cent, s_q[c].c, ew, boxsize);
              const bool hit = valid && r2 <= s_R[c];
              const uint64_t hits = __ballot(hit);
              if (hits) {
                int o = 0;
                if (lane == 0) o = atomicAdd(&s_run[c], __popcll(hits));
                const int64_t slot =
                    (int64_t)s_out[c] + __builtin_amdgcn_readfirstlane(o) + __popcll(hits & lt_mask);
                // Touching nodes are listed with a negative radius, -1 / maxdist2: they sort before every
                // node at a positive distance, the node itself first among them (smallest maxdist2), and
                // a consumer's "r2 <= k-th distance" test keeps them even when the k-th distance is
                // exactly 0 (k or more copies of a point): such a node may hold copies with smaller ids.
                // (A tiny positive radius, 1e-10 * maxdist2, failed that test and lost those ties.)
                if (hit && r2 == 0.f)
                  r2 = -1.0f / fmaxf((float)maxdist2<D, T>(nt.cent, s_q[c].c, ew, boxsize), 1e-30f);
                if (hit && slot < nmax) {
                  out_r2[slot] = r2;
                  out_src[slot] = it;
                }
              }
            }
          });
    }
  }
}

// ------------------------------------------------------------------------------------------------
// segmented sort by (key, val)
// ------------------------------------------------------------------------------------------------
// A (key, val) pair P of a node list, whose keys are distances and never NaN, is one double with the key's
// own bits as its high word: up to float infinity (0x7f800000) the double's exponent field stays below 0x7ff,
// and the double order is the float total order; below zero the order of the low word is reversed, so
// val is stored complemented there.  Denormal doubles are kept by the FP64 mode.  A compare-exchange is
// then one FP64 compare (or v_min_f64 + v_max_f64) instead of a 64-bit integer one.
// Keys of a caller (jzt_segment_sort) can be any bits: NaN patterns from 0x7ff00000 on would make the
// double a NaN, and -0 with val -1 would be -0.0, equal to +0 with val 0.  Their pairs are 64-bit integers in
// the same order.
constexpr int kSegThreads = 256;
constexpr int kSegLds = 4096;        // entries a workgroup of kSegThreads sorts in LDS (32 KB)
constexpr int kSegBigThreads = 1024;
constexpr int kSegBigLds = 16384;    // entries a workgroup of kSegBigThreads sorts in LDS (128 KB)
constexpr int kWaveSortMax = 1024;   // entries one wave sorts in registers

template <typename P> constexpr bool kAnyKey = std::is_same<P, uint64_t>::value;
template <typename P> __device__ __forceinline__ P kv_pack(float k, int32_t v) {
  const uint32_t kb = __float_as_uint(k);
  if constexpr (kAnyKey<P>) return ((uint64_t)((kb >> 31) ? ~kb : kb | 0x80000000u) << 32) | (uint32_t)v;
  else return __longlong_as_double((long long)(((uint64_t)kb << 32) | ((kb >> 31) ? ~(uint32_t)v : (uint32_t)v)));
}
template <typename P> __device__ __forceinline__ float kv_key(P p) {
  const uint32_t h = (uint32_t)(__builtin_bit_cast(uint64_t, p) >> 32);
  if constexpr (kAnyKey<P>) return __uint_as_float((h >> 31) ? h & 0x7fffffffu : ~h);
  else return __uint_as_float(h);
}
template <typename P> __device__ __forceinline__ int32_t kv_val(P p) {
  const uint64_t b = __builtin_bit_cast(uint64_t, p);
  if constexpr (kAnyKey<P>) return (int32_t)(uint32_t)b;
  else return (int32_t)((b >> 63) ? ~(uint32_t)b : (uint32_t)b);
}
// no pair is above it
template <typename P> __device__ __forceinline__ P kv_last() {
  if constexpr (kAnyKey<P>) return ~0ull;
  else return __longlong_as_double(0x7fefffffffffffffll);
}

// Bitonic network with only ascending comparators (the first stage of each merge compares mirrored
// pairs), so lengths need not be powers of two (virtual +inf tail).
template <typename Arr>
__device__ __forceinline__ void bitonic_sort_asc(Arr a, int len) {
  int np2 = 1;
  while (np2 < len) np2 <<= 1;
  for (int size = 2; size <= np2; size <<= 1) {
    // mirrored compare within each block of `size`
    for (int t = threadIdx.x; t < np2 / 2; t += blockDim.x) {
      int blk = t / (size / 2), off = t % (size / 2);
      int i = blk * size + off;
      int j = blk * size + size - 1 - off;
      if (j < len) {
        const auto x = a.load(i), y = a.load(j);
        if (y < x) {
          a.store(i, y);
          a.store(j, x);
        }
      }
    }
    __syncthreads();
    for (int stride = size / 4; stride > 0; stride >>= 1) {
      for (int t = threadIdx.x; t < np2 / 2; t += blockDim.x) {
        int blk = t / stride, off = t % stride;
        int i = blk * 2 * stride + off;
        int j = i + stride;
        if (j < len) {
          const auto x = a.load(i), y = a.load(j);
          if (y < x) {
            a.store(i, y);
            a.store(j, x);
          }
        }
      }
      __syncthreads();
    }
  }
}

template <typename P> struct LdsArr {
  P* p;
  __device__ __forceinline__ P load(int i) const { return p[i]; }
  __device__ __forceinline__ void store(int i, P x) const { p[i] = x; }
};
// (key, val) pairs sorted in place in global memory
template <typename P> struct GlobalKV {
  float* k;
  int32_t* v;
  __device__ __forceinline__ P load(int i) const { return kv_pack<P>(k[i], v[i]); }
  __device__ __forceinline__ void store(int i, P x) const {
    k[i] = kv_key(x);
    v[i] = kv_val(x);
  }
};

// ---- wave-level segment sort ---------------------------------------------------------------
// One wave per segment of up to 64*E entries, entry lane*E + i in register i of lane `lane`: the
// short strides, which a bitonic network uses most, stay inside a lane (v_min_f64 / v_max_f64), and
// the lane strides go through DPP and, from 16 on, permlane swaps, so nothing waits for LDS
// (exchanged with ds_bpermute, entry i*64 + lane, the sort was bound by LDS: 2.0 ms for the
// 548,000 lists of 257 entries of 2^24 clustered points at leaf 48, 0.97 now).
// lane l's value of lane l ^ M, for M = 1, 2, 4, 8, 16, 32 (strides) and 3, 7, 15, 31, 63 (mirrors)
template <int M> __device__ __forceinline__ uint32_t lane_xor(uint32_t x) {
  if constexpr (M == 1) return dpp<0xB1>(x);         // quad_perm 1,0,3,2
  else if constexpr (M == 2) return dpp<0x4E>(x);    // quad_perm 2,3,0,1
  else if constexpr (M == 3) return dpp<0x1B>(x);    // quad_perm 3,2,1,0
  else if constexpr (M == 7) return dpp<0x141>(x);   // row_half_mirror
  else if constexpr (M == 15) return dpp<0x140>(x);  // row_mirror
  else if constexpr (M == 8) return dpp<0x128>(x);   // row_ror:8
  else if constexpr (M == 4) return lane_xor<3>(lane_xor<7>(x));
  else if constexpr (M == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return (__lane_id() & 16) ? r[0] : r[1];
  } else if constexpr (M == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return (__lane_id() & 32) ? r[0] : r[1];
  } else if constexpr (M == 31) return lane_xor<16>(lane_xor<15>(x));
  else return lane_xor<32>(lane_xor<31>(x));  // 63
}
template <int M, typename P> __device__ __forceinline__ P pair_xor(P v) {
  return on_words(v, [](uint32_t x) { return lane_xor<M>(x); });
}
// keeps the smaller of v and o where `low`, else the larger (of equal ones either)
template <typename P> __device__ __forceinline__ P keep_side(P v, P o, bool low) { return (o < v) == low ? o : v; }

__device__ __forceinline__ void kv_order(double& a, double& b) {
  const double lo = __builtin_fmin(a, b), hi = __builtin_fmax(a, b);
  a = lo;
  b = hi;
}
__device__ __forceinline__ void kv_order(uint64_t& a, uint64_t& b) {
  const uint64_t lo = a < b ? a : b, hi = a < b ? b : a;
  a = lo;
  b = hi;
}

// entries x ^ S for register strides S < E (the whole wave is in blocks of 2S)
template <int E, int S, typename P> __device__ __forceinline__ void half_clean(P (&v)[E], int lane) {
  if constexpr (S < E) {
#pragma unroll
    for (int i = 0; i < E; i++)
      if (!(i & S)) kv_order(v[i], v[i | S]);
  } else {
    const bool low = (lane & (S / E)) == 0;
#pragma unroll
    for (int i = 0; i < E; i++) v[i] = keep_side(v[i], pair_xor<S / E>(v[i]), low);
  }
  if constexpr (S > 1) half_clean<E, S / 2>(v, lane);
}
// merges sorted blocks of SIZE/2 entries into sorted blocks of SIZE, from SIZE = 2 up to 64 * E
template <int E, int SIZE, typename P> __device__ __forceinline__ void wave_merge(P (&v)[E], int lane) {
  if constexpr (SIZE <= E) {
#pragma unroll
    for (int i = 0; i < E; i++) {
      const int j = i ^ (SIZE - 1);
      if (j > i) kv_order(v[i], v[j]);
    }
  } else {
    constexpr int M = SIZE / E - 1;  // mirrored partner: lane ^ M, register E - 1 - i
    const bool low = (lane & (SIZE / E / 2)) == 0;
    P o[E];
#pragma unroll
    for (int i = 0; i < E; i++) o[i] = pair_xor<M>(v[E - 1 - i]);
#pragma unroll
    for (int i = 0; i < E; i++) v[i] = keep_side(v[i], o[i], low);
  }
  if constexpr (SIZE > 2) half_clean<E, SIZE / 4>(v, lane);
  if constexpr (SIZE < 64 * E) wave_merge<E, SIZE * 2>(v, lane);
}

template <int E, typename P>
__device__ __forceinline__ void wave_sort_segment(float* key, int32_t* val, const float* key_in, const int32_t* val_in,
                                                  int64_t b, int len, int lane) {
  P v[E];
#pragma unroll
  for (int i = 0; i < E; i++) {
    const int idx = i * 64 + lane;  // any assignment will do before the sort: the coalesced one
    v[i] = idx < len ? kv_pack<P>(key_in[b + idx], val_in[b + idx]) : kv_last<P>();
  }
  wave_merge<E, 2>(v, lane);
#pragma unroll
  for (int i = 0; i < E; i++) {
    const int idx = lane * E + i;
    if (idx < len) {
      key[b + idx] = kv_key(v[i]);
      val[b + idx] = kv_val(v[i]);
    }
  }
}

// Segments too long for one wave: n, then their indices (a segment of more than kWaveSortMax entries
// each, so nmax / kWaveSortMax of them at most).  Null: the long-segment kernels look at every segment.
inline int64_t seg_queue_words(int64_t nmax) { return nmax / kWaveSortMax + 1; }

// Segments of up to kWaveSortMax entries, one wave each (in place allowed: a wave reads its whole
// segment into registers before writing); longer ones are queued for k_segment_sort.
template <typename P>
__global__ __launch_bounds__(64) void k_segment_sort_wave(const int32_t* __restrict__ spl, float* key, int32_t* val,
                                                          const float* key_in, const int32_t* val_in, int64_t nmax,
                                                          int64_t nitems, int32_t* __restrict__ queue) {
  const int64_t nact_ = active_items(spl, nitems);
  const int lane = threadIdx.x;
  for (int64_t seg = blockIdx.x; seg < nact_; seg += gridDim.x) {
    int64_t b = spl[seg], e = spl[seg + 1];
    if (e > nmax) e = nmax;
    if (b >= e) continue;
    const int64_t len = e - b;
    if (len > kWaveSortMax) {
      if (queue && lane == 0) queue[1 + atomicAdd(queue, 1)] = (int32_t)seg;
      continue;
    }
    if (len <= 64) wave_sort_segment<1, P>(key, val, key_in, val_in, b, (int)len, lane);
    else if (len <= 128) wave_sort_segment<2, P>(key, val, key_in, val_in, b, (int)len, lane);
    else if (len <= 256) wave_sort_segment<4, P>(key, val, key_in, val_in, b, (int)len, lane);
    else if (len <= 512) wave_sort_segment<8, P>(key, val, key_in, val_in, b, (int)len, lane);
    else wave_sort_segment<16, P>(key, val, key_in, val_in, b, (int)len, lane);
  }
}

// One workgroup per segment of more than LO entries: up to CAP in LDS; longer ones, where BIG, in
// place in the output arrays (global memory, visible within the workgroup across barriers).
template <typename P, int NT, int LO, int CAP, bool BIG>
__global__ __launch_bounds__(NT) void k_segment_sort(const int32_t* __restrict__ spl, float* key, int32_t* val,
                                                     const float* key_in, const int32_t* val_in, int64_t nmax,
                                                     int64_t nitems, const int32_t* __restrict__ queue) {
  __shared__ P s_a[CAP];
  const int64_t nseg = queue ? (int64_t)queue[0] : active_items(spl, nitems);
  for (int64_t it = blockIdx.x; it < nseg; it += gridDim.x) {
    const int64_t seg = queue ? (int64_t)queue[1 + it] : it;
    int64_t b = spl[seg], e = spl[seg + 1];
    if (e > nmax) e = nmax;
    if (e - b <= LO || (!BIG && e - b > CAP)) continue;
    const int len = (int)(e - b);
    if (len <= CAP) {
      for (int i = threadIdx.x; i < len; i += NT) s_a[i] = kv_pack<P>(key_in[b + i], val_in[b + i]);
      __syncthreads();
      bitonic_sort_asc(LdsArr<P>{s_a}, len);
      for (int i = threadIdx.x; i < len; i += NT) {
        key[b + i] = kv_key(s_a[i]);
        val[b + i] = kv_val(s_a[i]);
      }
    } else {
      if (key != key_in) {
        for (int i = threadIdx.x; i < len; i += NT) {
          key[b + i] = key_in[b + i];
          val[b + i] = val_in[b + i];
        }
        __syncthreads();
      }
      bitonic_sort_asc(GlobalKV<P>{key + b, val + b}, len);
    }
    __syncthreads();  // the next segment reuses s_a
  }
}

// ------------------------------------------------------------------------------------------------
// leaf-vs-leaf top-k
// ------------------------------------------------------------------------------------------------
// Bounding box of a leaf's particles (dims 2 and 3; unused dims are not read).
struct alignas(16) LeafBox {
  float lo[4], hi[4];
};

// Eight lanes per leaf; bound by the read of the positions (12 B a point).
template <int D>
__global__ __launch_bounds__(256) void k_leaf_boxes(const int32_t* __restrict__ spl, const float* __restrict__ x,
                                                    int64_t nleaves, LeafBox* __restrict__ boxes) {
  const int sub = threadIdx.x & 7;
  const int64_t step = (int64_t)gridDim.x * (blockDim.x / 8);
  for (int64_t l0 = (int64_t)blockIdx.x * (blockDim.x / 8); l0 < nleaves; l0 += step) {
    const int64_t leaf = l0 + (threadIdx.x >> 3);
    int a = 0, b = 0;
    if (leaf < nleaves) {
      a = spl[leaf];
      b = spl[leaf + 1];
    }
    float lo[D], hi[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
      lo[d] = INFINITY;
      hi[d] = -INFINITY;
    }
    for (int i = a + sub; i < b; i += 8) {
      const Vec<D, float> p = load_vec<D, float>(x, i);
#pragma unroll
      for (int d = 0; d < D; d++) {
        lo[d] = fminf(lo[d], p[d]);
        hi[d] = fmaxf(hi[d], p[d]);
      }
    }
    for (int o = 4; o > 0; o >>= 1) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        lo[d] = fminf(lo[d], __shfl_xor(lo[d], o, 8));
        hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], o, 8));
      }
    }
    if (sub == 0 && a < b) {
      LeafBox bx = {};
#pragma unroll
      for (int d = 0; d < D; d++) {
        bx.lo[d] = lo[d];
        bx.hi[d] = hi[d];
      }
      boxes[leaf] = bx;
    }
  }
}

// Smallest canonical r2 between a point in [qlo, qhi] and one in the box, from below: fl(q - p) lies in
// [fl(qlo - hi), fl(qhi - lo)], the wrap moves the whole interval one box over or (where it could go
// either way) the dimension counts as 0, and every step of the FMA chain rounds monotonically.
// wrapped: some difference may need the wrap.
template <bool PER, int D>
__device__ __forceinline__ float box_gap2(const Vec<D, float>& qlo, const Vec<D, float>& qhi, const LeafBox& bx,
                                          float boxsize, float half, bool& wrapped) {
  float g2 = 0.f;
  wrapped = false;
#pragma unroll
  for (int d = 0; d < D; d++) {
    float a = qlo[d] - bx.hi[d], b = qhi[d] - bx.lo[d];
    float gap;
    if (PER) {
      const bool up = b < -half, down = a >= half, no = a >= -half && b < half;
      wrapped |= !no;
      const float sh = up ? boxsize : -boxsize;
      a = no ? a : a + sh;
      b = no ? b : b + sh;
      gap = (no || up || down) ? fmaxf(0.f, fmaxf(a, -b)) : 0.f;
    } else {
      gap = fmaxf(0.f, fmaxf(a, -b));
    }
    g2 = fmaf(gap, gap, g2);
  }
  return g2;
}

// One wave per query leaf.  Interaction-list metadata (source leaf, r2, particle range) is loaded
// 64 entries at a time, one per lane, and broadcast with readlane.  Source particles move in
// chunks of <= 64: the next chunk is loaded into registers (one particle per lane) while the
// current chunk is consumed from LDS, where every lane reads the same record (broadcast).
//
// Periodic boxes: a chunk is streamed without the wrap selects when, for every staged particle p
// and every dim, fl(qlo - p) >= -half and fl(qhi - p) < half, with [qlo, qhi] the query chunk's
// bounding box.  Rounding is monotone, so then every difference fl(q - p) lies in [-half, half)
// and the canonical wrap leaves it unchanged: the distances are bit-identical.
//
// boxes (the source leaves' bounding boxes, optional): an entry is dropped when its box is out of the
// k-th distance's reach of the query chunk's box (tested for 64 entries at once) or of every single
// query (tested when its turn comes); both bounds are exact by monotone rounding.  Without the second
// test a leaf in a void next to a halo streamed the whole halo past queries of which none was near it:
// 224,000 particles for one wave of 10^6 clustered points at k = 64 (now 2,122; 1,903 -> 866 on
// average), and that wave set the time of the launch.
//
// Two lanes per query while 32 queries or fewer are left of the leaf (half of the leaves at the default
// size of 48: a leaf holds 30 points on average): each half of the wave takes every other source into
// a list of its own, both accept up to what bounds the k nearest of the union, and the lists are merged
// at the end.  Half of the lanes idled before, and the work for a source is the same for any number of
// active lanes.
//
// Query leaves come from a per-XCD item queue (ItemWalk) when the caller's tmp holds its eight
// counters (jzt_knn_leaf2leaf_tmp_bytes includes them), else in the fixed xcd_items order: the
// leaves' costs vary widely, and with a fixed stride the last waves of the launch ran long after
// the others had finished (plain kNN at 2^26: 92.4 -> 87.8 ms with the queue).
//
// Optional start bound (init_r2, per query leaf, K <= 64 single pass): the slots start at
// (r2_0, id = 2^32-1), so only candidates with r2 <= r2_0 enter.  A leaf with r2_0 < 0 is skipped
// entirely (its rows and retry flags are not written), so a later pass can redo selected leaves.  A query that ends with fewer
// than K real neighbours is flagged in `retry` (its row holds the sentinel entries); every other
// query's row is exact, because all its K neighbours lie within r2_0 and the list holds every
// leaf within r2_0 (the caller's contract).
template <int K, bool PER, bool FLOOR, int D, int W>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(W))) void k_knn_leaf(const int32_t* __restrict__ il_spl, const int32_t* __restrict__ il_src,
                                                 const float* __restrict__ il_r2, const int32_t* __restrict__ splT,
                                                 const float* __restrict__ xT, const int32_t* __restrict__ splQ,
                                                 const float* __restrict__ xQ, const int32_t* __restrict__ src_ids,
                                                 const int32_t* __restrict__ dst_rows,
                                                 const float* __restrict__ init_r2, int32_t* __restrict__ retry,
                                                 float* __restrict__ rad_out, int32_t* __restrict__ id_out,
                                                 uint64_t* __restrict__ resume, int koff, int ktot, float boxsize,
                                                 int64_t il_size, int64_t out_rows, int64_t nitems, int xcd,
                                                 uint32_t* __restrict__ queue, const LeafBox* __restrict__ boxes) {
  __shared__ SrcRec s_rec[64];
  __shared__ uint64_t s_buf[64 * kBufStride<K>];
  const int lane = threadIdx.x;
  const int64_t nact = active_items(splQ, nitems);
  for (ItemWalk walk(nact, xcd != 0, queue); walk.more(); walk.advance()) {
    const int64_t lq = walk.at;
    walk.started();
    uint64_t* const row = s_buf + lane * kBufStride<K>;
    const uint64_t lt_mask = (1ull << lane) - 1ull;
    const int q0 = splQ[lq], q1 = splQ[lq + 1];
    const int e0 = il_spl[lq], e1 = (int)min((int64_t)il_spl[lq + 1], il_size);
    const float half = 0.5f * boxsize;
    // a negative (or NaN) start bound marks a leaf that this launch leaves untouched
    const float r2_0 = init_r2 ? init_r2[lq] : 0.f;
    if (init_r2 && !(r2_0 >= 0.f)) continue;
    const uint64_t start_key = init_r2 ? (((uint64_t)__float_as_uint(r2_0) << 32) | 0xffffffffull) : kEmptyKey;
    for (int qoff = q0, g = 1; qoff < q1; qoff += 64 / g) {
      g = q1 - qoff <= 32 ? 2 : 1;  // lanes per query
      const int sub = g == 2 ? lane >> 5 : 0, ql = qoff + (g == 2 ? lane & 31 : lane);
      const int iq = min(ql, q1 - 1);
      const Vec<D, float> q = load_vec<D, float>(xQ, iq);
      const int64_t orow = dst_rows ? (int64_t)dst_rows[iq] : (int64_t)iq;
      const uint64_t floor_key = FLOOR ? resume[iq] : 0ull;
      Vec<D, float> qlo, qhi;  // bounding box of the query chunk, in scalar registers
  #pragma unroll
      for (int d = 0; d < D; d++) {
        qlo[d] = rdlane(wave_minf(q[d]), 0);
        qhi[d] = rdlane(wave_maxf(q[d]), 0);
      }
      uint64_t best[K];
  #pragma unroll
      for (int i = 0; i < K; i++) best[i] = start_key;
      int cnt = 0;  // entries in this lane's buffer row
      // largest r2 that can still be among the query's k nearest; best[] changes only on flushes
      auto bound = [&]() -> float {
        // two lists: K of the union are within either's last, and within both their K/2-th (no branch:
        // one here cost 27 registers)
        const float r = key_r2(best[K - 1]), m = key_r2(best[K / 2 - 1]);
        const float ro = __uint_as_float(other_half(__float_as_uint(r)));
        const float mo = __uint_as_float(other_half(__float_as_uint(m)));
        const float both = fminf(fminf(r, ro), fmaxf(m, mo));
        return g == 2 ? both : r;
      };
      float kr = key_r2(start_key);
      float kmax = wave_maxf(kr) * kRmaxSlack;  // of the wave, slack included
      float n_r2 = INFINITY;
      int n_src = 0;
      if (e0 + lane < e1) {
        n_r2 = il_r2[e0 + lane];
        n_src = il_src[e0 + lane];
      }
      for (int eb = e0; eb < e1; eb += 64) {
        const int ne = min(64, e1 - eb);
        // one entry per lane: its particles, and whether its box is within reach of the query chunk's
        int m_t0 = 0, m_t1 = 0;
        float m_r2 = INFINITY;
        LeafBox m_box;
        bool m_in = false, m_wrap = false;
        if (lane < ne) {
          m_r2 = n_r2;
          m_in = m_r2 <= kmax;
          if (m_in) {
            const int src = n_src;
            m_t0 = splT[src];
            m_t1 = splT[src + 1];
            m_in = m_t0 < m_t1;
            if (boxes) {
              m_box = boxes[src];
              const float g2 = box_gap2<PER, D>(qlo, qhi, m_box, boxsize, half, m_wrap);
              m_in = m_in && g2 <= kmax;
            }
          }
        }
        if (eb + 64 + lane < e1) {  // the next batch's, in flight while this one is worked off
          n_r2 = il_r2[eb + 64 + lane];
          n_src = il_src[eb + 64 + lane];
        }
        // ascending by r2: none further on is in reach either
        if (!(rdlane(m_r2, 0) <= kmax)) break;
        uint64_t em = __ballot(m_in);
        const uint64_t wm = __ballot(m_wrap);
        int E = -1, t0 = 0, t1 = 0;  // the entry and the range of its particles that are left
        // the next entry that some lane's k-th distance reaches
        auto next_entry = [&]() -> bool {
          while (em) {
            E = __builtin_ctzll(em);
            em &= em - 1ull;
            bool want = rdlane(m_r2, E) <= kr * kRmaxSlack;
            if (boxes) {
              LeafBox bx;
#pragma unroll
              for (int d = 0; d < D; d++) {
                bx.lo[d] = rdlane(m_box.lo[d], E);
                bx.hi[d] = rdlane(m_box.hi[d], E);
              }
              float g2;
              bool w;
              if (PER && ((wm >> E) & 1ull)) g2 = box_gap2<true, D>(q, q, bx, boxsize, half, w);
              else g2 = box_gap2<false, D>(q, q, bx, boxsize, half, w);
              want = want && g2 <= kr;
            }
            if (wave_any(want)) {
              t0 = rdlane(m_t0, E);
              t1 = rdlane(m_t1, E);
              return true;
            }
          }
          return false;
        };
        // the next chunk: up to 64 particles of as many entries as that takes, one per lane
        SrcRec cr;
        auto load_chunk = [&]() -> int {
          int n = 0, it = 0;
          while (n < 64 && (t0 < t1 || next_entry())) {
            if (lane >= n) it = t0 + lane - n;
            const int c = min(64 - n, t1 - t0);
            n += c;
            t0 += c;
          }
          if (lane < n) {
            const Vec<D, float> p = load_vec<D, float>(xT, it);
  #pragma unroll
            for (int d = 0; d < D; d++) cr.p[d] = p[d];
            cr.id = src_ids ? (uint32_t)src_ids[it] : (uint32_t)it;
          }
          return n;
        };
        for (int cn = load_chunk(); cn;) {
          const int n_cur = cn;
          // Source filter: p can enter some lane's top-k only if its gap to the query box is within
          // the largest current k-th distance of the wave (or a periodic wrap is possible); the
          // kept records are compacted into LDS.  Exact: by monotone rounding every canonical r2
          // from the box is >= the gap^2 computed here with the same FMA chain.
          bool need = false, reach = false;
          if (lane < n_cur) {
            float g2 = 0.f;
  #pragma unroll
            for (int d = 0; d < D; d++) {
              const float dlo = qlo[d] - cr.p[d], dhi = qhi[d] - cr.p[d];
              if (PER) need |= !(dlo >= -half) || !(dhi < half);
              const float gap = fmaxf(0.f, fmaxf(dlo, -dhi));
              g2 = fmaf(gap, gap, g2);
            }
            reach = need || g2 <= kmax;
          }
          const uint64_t keep = __ballot(reach);
          const bool wrap = PER && wave_any(need);
          // the halves of the wave take every other source: those of odd rank from slot 32 on.  Slots
          // past the last source hold NaN positions (a wave's LDS writes keep their order)
          const int n_keep = (__popcll(keep) + g - 1) / g;
          const int rank = __popcll(keep & lt_mask);
          s_rec[lane].p[0] = __builtin_nanf("");
          if (reach) s_rec[g == 2 ? (rank >> 1) + ((rank & 1) << 5) : rank] = cr;
          __syncthreads();
          cn = load_chunk();  // in flight while this chunk is consumed
          if (consume_chunk<K, PER, FLOOR, D>(best, q, s_rec + 32 * sub, n_keep, wrap, boxsize, half, floor_key, row,
                                              cnt, kr, bound))
            kmax = wave_maxf(kr) * kRmaxSlack;
          __syncthreads();
        }
      }
      if (wave_any(cnt > 0)) topk_flush<K>(best, row, cnt);
      if (g == 2) merge_halves<K>(best);
      if (sub == 0 && ql < q1) {
        if (orow >= 0 && orow < out_rows) write_row<K>(best, rad_out, id_out, orow * ktot + koff, ktot - koff);
        // the last slot this pass reports (k need not be a power of two: slots past it may
        // keep the start key even when the query has all its neighbours)
        const int last = min(K, ktot - koff) - 1;
        uint64_t lk = best[0];
  #pragma unroll
        for (int i = 0; i < K; i++) lk = (i == last) ? best[i] : lk;
        if (retry) retry[iq] = (lk == start_key && init_r2) ? 1 : 0;
        if (resume) resume[iq] = lk;
      }
    }
  
  }
}

// Sort each segment by (key, val): segments of up to kWaveSortMax entries one wave each in registers,
// longer ones by a workgroup (in LDS up to kSegBigLds entries, else in place in global memory).
// queue (seg_queue_words(nmax) words, or null): the long segments, found by the first kernel.  A segment
// has no more than max_len entries, so kernels for longer ones than that are not launched.  Lists of 4096
// to 16384 entries (the nodes around a void; 200 of 548,000 at 2^24, leaf 48) are sorted in 128 KB of LDS:
// in global memory they took 3.1 ms together, 0.9 now.
template <typename P>
int segment_sort(hipStream_t s, const int32_t* spl, float* key, int32_t* val, const float* key_in,
                 const int32_t* val_in, int64_t nseg, int64_t nmax, int64_t max_len, int32_t* queue, const char* what) {
  if (nseg <= 0) return 0;
  if (queue && max_len > kWaveSortMax && fill_u32(s, queue, 0u, 1)) return 1;
  // four times the waves that the chip holds: workgroups stride over the segments
  const unsigned gw = (unsigned)(nseg < 32768 ? nseg : 32768);
  hipLaunchKernelGGL(k_segment_sort_wave<P>, dim3(gw), dim3(64), 0, s, spl, key, val, key_in, val_in, nmax, nseg,
                     max_len > kWaveSortMax ? queue : nullptr);
  if (check_launch(what)) return 1;
  // the kernels touch disjoint segments; without a queue their workgroups go over all of them
  if (max_len > kWaveSortMax)
    hipLaunchKernelGGL((k_segment_sort<P, kSegThreads, kWaveSortMax, kSegLds, false>),
                       dim3((unsigned)(nseg < 4096 ? nseg : 4096)), dim3(kSegThreads), 0, s, spl, key, val, key_in,
                       val_in, nmax, nseg, queue);
  if (max_len > kSegLds)
    hipLaunchKernelGGL((k_segment_sort<P, kSegBigThreads, kSegLds, kSegBigLds, true>),
                       dim3((unsigned)(nseg < 1024 ? nseg : 1024)), dim3(kSegBigThreads), 0, s, spl, key, val, key_in,
                       val_in, nmax, nseg, queue);
  return check_launch(what);
}

// ------------------------------------------------------------------------------------------------
// distances for the dense top-plane list
// ------------------------------------------------------------------------------------------------
// The dense list pairs every super-node (about 32 consecutive top-plane nodes) with every other, at no
// distance: each of the three passes over the top plane tested all pairs of its nodes (2048 to 13,000),
// and the radius search met the node's own neighbourhood only when the list came to it.  With the
// distances of the super-nodes' bounding boxes, sorted, the passes stop where the radius ends.  A
// distance is lowered by 2^-15 of itself and the boxes are widened by 2^-20 of their coordinates, which
// covers the rounding of the nodes' own distances: the nodes' lists are the same.
template <int D, typename T>
__global__ __launch_bounds__(256) void k_super_boxes(const T* __restrict__ nodes, const int32_t* __restrict__ spl,
                                                     const int32_t* __restrict__ nsuper, int64_t nmax, int64_t nnodes,
                                                     T* __restrict__ boxes) {
  const int sub = threadIdx.x & 31;
  const int64_t ns = min((int64_t)nsuper[0], nmax);
  for (int64_t i = (int64_t)blockIdx.x * (blockDim.x / 32) + (threadIdx.x >> 5); i < ns;
       i += (int64_t)gridDim.x * (blockDim.x / 32)) {
    const int64_t a = spl[i], b = min((int64_t)spl[i + 1], nnodes);
    T lo[D], hi[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
      lo[d] = (T)INFINITY;
      hi[d] = -(T)INFINITY;
    }
    for (int64_t j = a + sub; j < b; j += 32) {
      const NodeT<D, T> n = load_node<D, T>(nodes, j);
      const Vec<D, T> e = lvl_half_ext<D, T>(n.level);
#pragma unroll
      for (int d = 0; d < D; d++) {
        lo[d] = min(lo[d], n.cent[d] - e[d]);
        hi[d] = max(hi[d], n.cent[d] + e[d]);
      }
    }
    for (int o = 16; o > 0; o >>= 1) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        lo[d] = min(lo[d], __shfl_xor(lo[d], o, 32));
        hi[d] = max(hi[d], __shfl_xor(hi[d], o, 32));
      }
    }
    if (sub == 0) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        const T c = T(0.5) * lo[d] + T(0.5) * hi[d];
        boxes[i * 2 * D + d] = c;
        boxes[i * 2 * D + D + d] = (T(0.5) * hi[d] - T(0.5) * lo[d]) + (abs(lo[d]) + abs(hi[d])) * T(1.0 / 1048576.0);
      }
    }
  }
}

// r2 given: the distance of every entry (negative for touching super-nodes, nearest first, as in
// k_node_insert); else entries beyond `limit` are replaced by -1, which the FoF passes skip.
template <int D, typename T>
__global__ __launch_bounds__(256) void k_dense_r2(const T* __restrict__ boxes, const int32_t* __restrict__ nsuper,
                                                  int64_t nmax, int64_t size_ilist, T boxsize, float limit,
                                                  int32_t* __restrict__ ilist, float* __restrict__ r2) {
  const int64_t ns = nsuper[0];
  if (ns > nmax) return;  // reported by the list's own check
  const int64_t m = min(ns * ns, size_ilist);
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < m; j += (int64_t)gridDim.x * blockDim.x) {
    const int64_t a = j / ns, b = j - a * ns;
    Vec<D, T> ca, cb, w;
#pragma unroll
    for (int d = 0; d < D; d++) {
      ca[d] = boxes[a * 2 * D + d];
      cb[d] = boxes[b * 2 * D + d];
      w[d] = boxes[a * 2 * D + D + d] + boxes[b * 2 * D + D + d];
    }
    const float g2 = (float)mindist2<D, T>(ca, cb, w, boxsize) * (1.0f - 2.f * kBoundSlack);
    if (!r2) {
      if (g2 > limit) ilist[j] = -1;
    } else {
      r2[j] = g2 > 0.f ? g2 : a == b ? -INFINITY : -1.0f / fmaxf((float)maxdist2<D, T>(ca, cb, w, boxsize), 1e-30f);
    }
  }
}

__global__ void k_scale_rmax2(const float* __restrict__ in, float* __restrict__ out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[i] * kRmaxSlack;
}

// Guaranteed k-neighbour radius^2 of the nodes of one plane, planes taken from the top down:
// cap[c] = squared cell diagonal of node c if it holds >= k particles, else its parent's cap (the
// parent: the last node P of the plane above with n2c_up[P] <= c, clamped into [0, size)), +inf
// at the top plane.  npart[c] = spl[n2l[c+1]] - spl[n2l[c]] (indices clamped to the spl array).
// The diagonal^2 sums 4^l_i over the per-dim levels of lvl_vec, in float64 (exact).
__global__ void k_plane_cap(const int32_t* __restrict__ n2l, const int32_t* __restrict__ spl, int64_t nspl,
                            const int32_t* __restrict__ lvl, const int32_t* __restrict__ n2c_up,
                            const double* __restrict__ cap_up, int64_t size, int k, int dim, double* __restrict__ cap) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= size) return;
  const int64_t a = min((int64_t)n2l[c], nspl - 1), b = min((int64_t)n2l[c + 1], nspl - 1);
  const int64_t np = (int64_t)spl[b] - (int64_t)spl[a];
  double r;
  if (np >= k) {
    const int o = (lvl[c] + 2000 * dim) / dim - 2000;
    const int rem = lvl[c] - o * dim;
    r = 0.0;
    for (int i = 0; i < dim; i++) r += ldexp(1.0, 2 * (o + (rem >= dim - i ? 1 : 0)));
  } else if (!n2c_up) {
    r = INFINITY;
  } else {
    int64_t lo = 0, hi = size + 1;  // count of n2c_up entries <= c
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (n2c_up[mid] <= c) lo = mid + 1;
      else hi = mid;
    }
    const int64_t parent = min(max(lo - 1, (int64_t)0), size - 1);
    r = cap_up[parent];
  }
  cap[c] = r;
}

// out[i] = max of v over the segment [spl[i], spl[i+1]) (clamped to [0, nv)), `empty` if it is empty
__global__ void k_segment_max(const int32_t* __restrict__ spl, const float* __restrict__ v, int64_t nv,
                              float* __restrict__ out, int64_t nseg, float empty) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nseg) return;
  const int64_t a = min(max((int64_t)spl[i], (int64_t)0), nv), b = min(max((int64_t)spl[i + 1], (int64_t)0), nv);
  float m = empty;
  for (int64_t j = a; j < b; j++) m = fmaxf(m, v[j]);
  out[i] = m;
}

template <int D, typename T>
int node2node_impl(hipStream_t s, const int32_t* pil_spl, const int32_t* pil_src, const float* pil_r2,
                   const int32_t* parent_spl, const void* nodes, const int32_t* npart, const float* parent_rmax2,
                   const float* rmax2_in,
                   float* rmax2, int32_t* il_spl, int32_t* il_src, float* il_r2, int64_t size_parents,
                   int64_t size_nodes, int64_t pil_size, int64_t il_size, int k, float boxsize, void* tmp,
                   size_t tmp_bytes, uint8_t* overflow) {
  const T* nd = (const T*)nodes;
  if (fill_u32(s, il_spl, 0u, size_nodes + 1)) return 1;
  if (size_nodes >= INT32_MAX) return fail("KnnNode2Node: too many nodes");
  if (size_parents <= 0) return overflow ? clear_flag(s, overflow) : 0;  // empty lists
  const dim3 g(node_grid(size_parents, 64)), b(64), gl(node_grid(size_parents, kNodeThreads)), bl(kNodeThreads);
  // without room for the queue, one-wave workgroups run the long lists too
  const bool split = tmp && tmp_bytes >= 4 * (size_t)node_queue_words(size_parents);
  const NodeQueue queue{split ? (int32_t*)tmp : nullptr, size_parents};
  if (split && fill_u32(s, tmp, 0u, 1)) return 1;
#define JZT_NODE_COUNT(RADIUS)                                                                                        \
  do {                                                                                                                \
    hipLaunchKernelGGL((k_node_count<RADIUS, 64, D, T>), g, b, 0, s, pil_spl, pil_src, pil_r2, parent_spl, nd, npart, \
                       parent_rmax2, rmax2, il_spl + 1, k, (T)boxsize, pil_size, size_parents, (int)size_nodes, queue);             \
    if (split)                                                                                                        \
      hipLaunchKernelGGL((k_node_count<RADIUS, kNodeThreads, D, T>), gl, bl, 0, s, pil_spl, pil_src, pil_r2,          \
                         parent_spl, nd, npart, parent_rmax2, rmax2, il_spl + 1, k, (T)boxsize, pil_size,             \
                         size_parents, (int)size_nodes, queue);                                                       \
  } while (0)
  if (rmax2_in) {
    if (size_nodes > 0)
      hipLaunchKernelGGL(k_scale_rmax2, dim3((unsigned)div_up(size_nodes, 256)), dim3(256), 0, s, rmax2_in, rmax2,
                         size_nodes);
    JZT_NODE_COUNT(false);
  } else {
    JZT_NODE_COUNT(true);
  }
#undef JZT_NODE_COUNT
  if (check_launch("KnnNode2Node count")) return 1;
  // inclusive scan of the counts in place; the scan temp lives in the (not yet written) list
  if (scan_tmp_words(size_nodes) > il_size) return fail("KnnNode2Node: interaction list too small for scan temp");
  if (scan_i32(s, il_spl + 1, il_spl + 1, size_nodes, true, il_src)) return 1;
  hipLaunchKernelGGL((k_node_insert<64, D, T>), g, b, 0, s, pil_spl, pil_src, pil_r2, parent_spl, nd, rmax2, il_spl,
                     il_src, il_r2, il_size, (T)boxsize, pil_size, size_parents, (int)size_nodes, overflow, queue);
  if (split)
    hipLaunchKernelGGL((k_node_insert<kNodeThreads, D, T>), gl, bl, 0, s, pil_spl, pil_src, pil_r2, parent_spl, nd, rmax2,
                       il_spl, il_src, il_r2, il_size, (T)boxsize, pil_size, size_parents, (int)size_nodes, overflow,
                       queue);
  if (check_launch("KnnNode2Node insert")) return 1;
  // sort each node's list by (r2, src) in place
  // (a list names every node at most once)
  const size_t qoff = align256(4 * (size_t)node_queue_words(size_parents));
  int32_t* sq = tmp && tmp_bytes >= qoff + 4 * (size_t)seg_queue_words(il_size) ? (int32_t*)((char*)tmp + qoff) : nullptr;
  return segment_sort<double>(s, il_spl, il_r2, il_src, il_r2, il_src, size_nodes, il_size, size_nodes, sq, "KnnNode2Node sort");
}

template <int D>
int leaf2leaf_impl(hipStream_t s, const int32_t* il_spl, const int32_t* il_src, const float* il_r2, const int32_t* splT,
                   const void* xT, const int32_t* splQ, const void* xQ, const int32_t* src_ids,
                   const int32_t* dst_rows, const float* init_r2, int32_t* retry, void* rad, int32_t* ids, void* tmp,
                   size_t tmp_bytes, int64_t nleaves_q, int64_t npart_q, int64_t out_rows, int64_t il_size, int k,
                   float boxsize, const LeafBox* boxes) {
  if (nleaves_q <= 0) return 0;
  if (init_r2 && k > 64) return fail("KnnLeaf2Leaf: a start bound needs k <= 64");
  uint64_t* resume = k > 64 ? (uint64_t*)tmp : nullptr;
  // item queue counters after the resume keys, when the caller's tmp holds them
  const size_t qoff = align256(knn_leaf_nd_tmp_bytes(npart_q, k, false));
  uint32_t* queue = tmp && tmp_bytes >= qoff + 256 ? (uint32_t*)((char*)tmp + qoff) : nullptr;
  const dim3 b(64);
  const float* xt = (const float*)xT;
  const float* xq = (const float*)xQ;
  const int xcd = tune_get(kTuneXcd);
  for (int koff = 0; koff < k; koff += 64) {
    const int kn = min(k - koff, 64);
    const bool floor = resume && koff > 0;
    if (queue && fill_u32(s, queue, 0u, 8 * kQueueStride)) return 1;
    // waves that a compute unit holds, by registers
    const dim3 g(queue ? queue_grid(nleaves_q, kn <= 8 ? 20 : kn <= 16 ? 16 : kn <= 32 ? 12 : 8) : grid_for8(nleaves_q));
#define JZT_KNN_LAUNCH(KK, PER, FLOOR, W)                                                                              \
  hipLaunchKernelGGL((k_knn_leaf<KK, PER, FLOOR, D, W>), g, b, 0, s, il_spl, il_src, il_r2, splT, xt, splQ, xq, src_ids, \
                     dst_rows, init_r2, retry, (float*)rad, ids, resume, koff, k, boxsize, il_size, out_rows, nleaves_q, xcd, \
                     queue, boxes)
  // waves per EU (the register budget of the kernel).  K <= 8 takes 89 registers and K <= 16 122 with any
  // budget that holds them; at K = 32, 4 waves spilled 29, in the flush (2^26 points, learned: 65.6 ms against
  // 61.9 at 3); at K = 64, 2 spill 12 and hide more than 1 (1,000,003 points, k = 64: 4.5 ms against 5.1)
#define JZT_KNN_LAUNCH_K(KK)                                                      \
  do {                                                                            \
    constexpr int w = KK > 32 ? 2 : KK > 16 ? 3 : 4, wf = KK > 32 ? 1 : w;        \
    if (boxsize > 0.f) {                                                          \
      if (floor) JZT_KNN_LAUNCH(KK, true, true, wf);                              \
      else JZT_KNN_LAUNCH(KK, true, false, w);                                    \
    } else {                                                                      \
      if (floor) JZT_KNN_LAUNCH(KK, false, true, wf);                             \
      else JZT_KNN_LAUNCH(KK, false, false, w);                                   \
    }                                                                             \
  } while (0)
    if (kn <= 8) JZT_KNN_LAUNCH_K(8);
    else if (kn <= 16) JZT_KNN_LAUNCH_K(16);
    else if (kn <= 32) JZT_KNN_LAUNCH_K(32);
    else JZT_KNN_LAUNCH_K(64);
#undef JZT_KNN_LAUNCH_K
#undef JZT_KNN_LAUNCH
    if (check_launch("KnnLeaf2Leaf")) return 1;
  }
  return 0;
}

}  // namespace
}  // namespace jzt

using namespace jzt;

extern "C" int jzt_knn_node2node(jzt_stream_t stream, const int32_t* parent_ilist_spl, const int32_t* parent_ilist_isrc,
                                 const float* parent_ilist_r2, const int32_t* parent_spl, const void* nodes,
                                 const int32_t* nodes_npart, float* node_rmax2, int32_t* node_ilist_spl,
                                 int32_t* node_ilist_isrc, float* node_ilist_r2, int64_t size_parents,
                                 int64_t size_nodes, int64_t parent_ilist_size, int64_t node_ilist_size, int k,
                                 float boxsize, int dim, int dtype) {
  return jzt_knn_node2node_ex(stream, parent_ilist_spl, parent_ilist_isrc, parent_ilist_r2, parent_spl, nodes,
                              nodes_npart, nullptr, node_rmax2, node_ilist_spl, node_ilist_isrc, node_ilist_r2,
                              size_parents, size_nodes, parent_ilist_size, node_ilist_size, k, boxsize, dim, dtype);
}

extern "C" size_t jzt_knn_node2node_tmp_bytes(int64_t size_parents, int64_t node_ilist_size) {
  return align256(4 * (size_t)node_queue_words(size_parents)) + 4 * (size_t)seg_queue_words(node_ilist_size);
}

extern "C" int jzt_knn_node2node_ex(jzt_stream_t stream, const int32_t* parent_ilist_spl,
                                    const int32_t* parent_ilist_isrc, const float* parent_ilist_r2,
                                    const int32_t* parent_spl, const void* nodes, const int32_t* nodes_npart,
                                    const float* node_r2_in, float* node_rmax2, int32_t* node_ilist_spl,
                                    int32_t* node_ilist_isrc, float* node_ilist_r2, int64_t size_parents,
                                    int64_t size_nodes, int64_t parent_ilist_size, int64_t node_ilist_size, int k,
                                    float boxsize, int dim, int dtype) {
  return jzt_knn_node2node_tmp(stream, parent_ilist_spl, parent_ilist_isrc, parent_ilist_r2, parent_spl, nodes,
                               nodes_npart, nullptr, node_r2_in, node_rmax2, node_ilist_spl, node_ilist_isrc, node_ilist_r2,
                               size_parents, size_nodes, parent_ilist_size, node_ilist_size, k, boxsize, dim, dtype,
                               nullptr, 0, nullptr);
}

extern "C" int jzt_knn_node2node_tmp(jzt_stream_t stream, const int32_t* parent_ilist_spl,
                                    const int32_t* parent_ilist_isrc, const float* parent_ilist_r2,
                                    const int32_t* parent_spl, const void* nodes, const int32_t* nodes_npart,
                                    const float* parent_rmax2, const float* node_r2_in, float* node_rmax2, int32_t* node_ilist_spl,
                                    int32_t* node_ilist_isrc, float* node_ilist_r2, int64_t size_parents,
                                    int64_t size_nodes, int64_t parent_ilist_size, int64_t node_ilist_size, int k,
                                    float boxsize, int dim, int dtype, void* tmp, size_t tmp_bytes,
                                     uint8_t* overflow) {
  hipStream_t s = (hipStream_t)stream;
  if (k < 1) return fail("KnnNode2Node: k must be >= 1");
  // dims 2-10, float or double node geometry (_generate_ffi.py:9-21)
#define JZT_N2N(D, T)                                                                                              \
  return node2node_impl<D, T>(s, parent_ilist_spl, parent_ilist_isrc, parent_ilist_r2, parent_spl, nodes,         \
                              nodes_npart, parent_rmax2, node_r2_in, node_rmax2, node_ilist_spl, node_ilist_isrc, node_ilist_r2, \
                              size_parents, size_nodes, parent_ilist_size, node_ilist_size, k, boxsize, tmp, tmp_bytes, overflow)
#define JZT_N2N_DIM(D)                  \
  case D:                               \
    if (dtype == JZT_F32) JZT_N2N(D, float); \
    JZT_N2N(D, double);
  if (dtype == JZT_F32 || dtype == JZT_F64) {
    switch (dim) {
      JZT_N2N_DIM(2) JZT_N2N_DIM(3) JZT_N2N_DIM(4) JZT_N2N_DIM(5) JZT_N2N_DIM(6) JZT_N2N_DIM(7) JZT_N2N_DIM(8)
      JZT_N2N_DIM(9) JZT_N2N_DIM(10)
      default: break;
    }
  }
#undef JZT_N2N_DIM
#undef JZT_N2N
  return fail("KnnNode2Node: unsupported dim/dtype");
}

extern "C" size_t jzt_dense_ilist_r2_tmp_bytes(int64_t size_super, int dim, int dtype) {
  return (size_t)size_super * 2 * dim * (dtype == JZT_F64 ? 8 : 4);
}

extern "C" int jzt_dense_ilist_r2(jzt_stream_t stream, const void* nodes, int64_t nnodes, const int32_t* spl_super,
                                  const int32_t* ispl, int64_t size_super, const int32_t* nsuper, int32_t* ilist,
                                  float* r2, int64_t size_ilist, float boxsize, float limit, int dim, int dtype,
                                  void* tmp, size_t tmp_bytes) {
  hipStream_t s = (hipStream_t)stream;
  if (size_super <= 0 || nnodes <= 0) return 0;
  if (nnodes >= INT32_MAX) return fail("DenseIlistR2: too many nodes");
  if (tmp_bytes < jzt_dense_ilist_r2_tmp_bytes(size_super, dim, dtype)) return fail("DenseIlistR2: tmp buffer too small");
#define JZT_DENSE_R2(D, T)                                                                                          \
  hipLaunchKernelGGL((k_super_boxes<D, T>), dim3((unsigned)std::min(div_up(size_super, 8), (int64_t)256)), dim3(256), \
                     0, s, (const T*)nodes, spl_super, nsuper, size_super, nnodes, (T*)tmp);                         \
  hipLaunchKernelGGL((k_dense_r2<D, T>), dim3((unsigned)std::min(div_up(size_ilist, 256), (int64_t)1024)), dim3(256), \
                     0, s, (const T*)tmp, nsuper, size_super, size_ilist, (T)boxsize, limit, ilist, r2)
  if (dim == 3 && dtype == JZT_F32) { JZT_DENSE_R2(3, float); }
  else if (dim == 3 && dtype == JZT_F64) { JZT_DENSE_R2(3, double); }
  else if (dim == 2 && dtype == JZT_F32) { JZT_DENSE_R2(2, float); }
  else if (dim == 2 && dtype == JZT_F64) { JZT_DENSE_R2(2, double); }
  else return fail("DenseIlistR2: unsupported dim/dtype");
#undef JZT_DENSE_R2
  if (check_launch("DenseIlistR2")) return 1;
  if (!r2) return 0;
  // rows past the last super-node are empty
  return segment_sort<double>(s, ispl, r2, ilist, r2, ilist, size_super, size_ilist, size_super, nullptr, "DenseIlistR2 sort");
}

extern "C" int jzt_segment_max_f32(jzt_stream_t stream, const int32_t* spl, const float* vals, int64_t nvals,
                                   float* out, int64_t nseg, float empty) {
  if (nseg <= 0) return 0;
  hipLaunchKernelGGL(k_segment_max, dim3((unsigned)div_up(nseg, 256)), dim3(256), 0, (hipStream_t)stream, spl, vals,
                     nvals, out, nseg, empty);
  return check_launch("SegmentMax");
}

extern "C" int jzt_plane_cap(jzt_stream_t stream, const int32_t* n2l, const int32_t* spl, int64_t nspl,
                             const int32_t* lvl, const int32_t* n2c_up, const double* cap_up, int64_t size, int k,
                             int dim, double* cap) {
  if (size <= 0) return 0;
  if (nspl < 1 || dim < 1) return fail("PlaneCap: empty splits or dim < 1");
  if ((n2c_up == nullptr) != (cap_up == nullptr)) return fail("PlaneCap: n2c_up and cap_up go together");
  hipLaunchKernelGGL(k_plane_cap, dim3((unsigned)div_up(size, 256)), dim3(256), 0, (hipStream_t)stream, n2l, spl, nspl,
                     lvl, n2c_up, cap_up, size, k, dim, cap);
  return check_launch("PlaneCap");
}

extern "C" size_t jzt_knn_leaf2leaf_tmp_bytes(int64_t size_part_query, int k, int dtype) {
  // float: the packed kernel's u64 resume key, or the (r2, id) pair of the any-dim kernel, both 8
  // bytes per query past 64 neighbours; double: a (double r2, u32 id) pair past 32
  // ... then 256 bytes of item-queue counters for the packed kernel
  return align256(knn_leaf_nd_tmp_bytes(size_part_query, k, dtype == JZT_F64)) + 256;
}

extern "C" int jzt_knn_leaf2leaf(jzt_stream_t stream, const int32_t* ilist_spl, const int32_t* ilist_isrc,
                                 const float* ilist_r2, int64_t ilist_size, const int32_t* splT, const void* xT,
                                 const int32_t* splQ, const void* xQ, const int32_t* src_ids, void* knn_rad,
                                 int32_t* knn_id, void* tmp, size_t tmp_bytes, int64_t size_leaves_query,
                                 int64_t size_part_query, int k, float boxsize, int dim, int dtype) {
  return jzt_knn_leaf2leaf_ex(stream, ilist_spl, ilist_isrc, ilist_r2, ilist_size, splT, xT, splQ, xQ, src_ids,
                              nullptr, nullptr, nullptr, knn_rad, knn_id, tmp, tmp_bytes, size_leaves_query,
                              size_part_query, size_part_query, k, boxsize, dim, dtype);
}

extern "C" int jzt_leaf_boxes(jzt_stream_t stream, const int32_t* spl, const float* x, int64_t nleaves, int dim,
                              float* leaf_boxes) {
  if (nleaves <= 0) return 0;
  if ((uintptr_t)leaf_boxes & 15) return fail("LeafBoxes: leaf boxes must be 16-byte aligned");
  const dim3 g((unsigned)std::min(div_up(nleaves, 32), (int64_t)16384)), b(256);
  hipStream_t s = (hipStream_t)stream;
  if (dim == 3) hipLaunchKernelGGL(k_leaf_boxes<3>, g, b, 0, s, spl, x, nleaves, (LeafBox*)leaf_boxes);
  else if (dim == 2) hipLaunchKernelGGL(k_leaf_boxes<2>, g, b, 0, s, spl, x, nleaves, (LeafBox*)leaf_boxes);
  else return fail("LeafBoxes: unsupported dim");
  return check_launch("LeafBoxes");
}

extern "C" int jzt_knn_leaf2leaf_boxes(jzt_stream_t stream, const int32_t* ilist_spl, const int32_t* ilist_isrc,
                                    const float* ilist_r2, int64_t ilist_size, const int32_t* splT, const void* xT,
                                    const int32_t* splQ, const void* xQ, const int32_t* src_ids,
                                    const int32_t* dst_rows, const float* init_r2, int32_t* retry, void* knn_rad,
                                    int32_t* knn_id, void* tmp, size_t tmp_bytes, int64_t size_leaves_query,
                                    int64_t size_part_query, int64_t out_rows, int k, float boxsize, int dim,
                                    int dtype, const float* leaf_boxes) {
  hipStream_t s = (hipStream_t)stream;
  const LeafBox* boxes = (const LeafBox*)leaf_boxes;
  if ((uintptr_t)leaf_boxes & 15) return fail("KnnLeaf2Leaf: leaf boxes must be 16-byte aligned");
  if (k < 1) return fail("KnnLeaf2Leaf: k must be >= 1");
  // the multi-pass state is required; the work-queue counters after it are optional
  if (tmp_bytes < knn_leaf_nd_tmp_bytes(size_part_query, k, dtype == JZT_F64))
    return fail("KnnLeaf2Leaf: tmp too small");
  if (dtype != JZT_F32 && dtype != JZT_F64) return fail("KnnLeaf2Leaf: positions must be float32 or float64");
  if (dtype == JZT_F64 || dim > 3)
    return (dtype == JZT_F64 ? knn_leaf_nd_f64 : knn_leaf_nd_f32)(
        s, ilist_spl, ilist_isrc, ilist_r2, splT, xT, splQ, xQ, src_ids, dst_rows, init_r2, retry, knn_rad, knn_id, tmp,
        tmp_bytes, size_leaves_query, size_part_query, out_rows, ilist_size, k, boxsize, dim);
  if (dim == 3)
    return leaf2leaf_impl<3>(s, ilist_spl, ilist_isrc, ilist_r2, splT, xT, splQ, xQ, src_ids, dst_rows, init_r2, retry,
                             knn_rad, knn_id, tmp, tmp_bytes, size_leaves_query, size_part_query, out_rows, ilist_size, k,
                             boxsize, boxes);
  if (dim == 2)
    return leaf2leaf_impl<2>(s, ilist_spl, ilist_isrc, ilist_r2, splT, xT, splQ, xQ, src_ids, dst_rows, init_r2, retry,
                             knn_rad, knn_id, tmp, tmp_bytes, size_leaves_query, size_part_query, out_rows, ilist_size, k,
                             boxsize, boxes);
  return fail("KnnLeaf2Leaf: unsupported dim");
}

extern "C" int jzt_knn_leaf2leaf_ex(jzt_stream_t stream, const int32_t* ilist_spl, const int32_t* ilist_isrc,
                                    const float* ilist_r2, int64_t ilist_size, const int32_t* splT, const void* xT,
                                    const int32_t* splQ, const void* xQ, const int32_t* src_ids,
                                    const int32_t* dst_rows, const float* init_r2, int32_t* retry, void* knn_rad,
                                    int32_t* knn_id, void* tmp, size_t tmp_bytes, int64_t size_leaves_query,
                                    int64_t size_part_query, int64_t out_rows, int k, float boxsize, int dim,
                                    int dtype) {
  return jzt_knn_leaf2leaf_boxes(stream, ilist_spl, ilist_isrc, ilist_r2, ilist_size, splT, xT, splQ, xQ, src_ids,
                                 dst_rows, init_r2, retry, knn_rad, knn_id, tmp, tmp_bytes, size_leaves_query,
                                 size_part_query, out_rows, k, boxsize, dim, dtype, nullptr);
}

extern "C" int jzt_segment_sort(jzt_stream_t stream, const int32_t* spl, const float* key, const int32_t* val,
                                float* key_out, int32_t* val_out, int64_t size_segs, int64_t size_keys) {
  hipStream_t s = (hipStream_t)stream;
  if (size_segs <= 0) return 0;
  return segment_sort<uint64_t>(s, spl, key_out, val_out, key, val, size_segs, size_keys, size_keys, nullptr,
                      "SegmentSort");
}
