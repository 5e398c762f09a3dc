// Work split of the node-vs-node passes (KnnNode2Node, FofNode2Node).
//
// A parent node's interaction list names other parents; its children are tested against the children
// of every one of them.  How much work that is varies by orders of magnitude: the dense list of the
// top plane pairs ~400 parents with all others (390,000 child pairs each, 2^24 points), while the
// parents of the planes below number 10^4 to 10^5 with 10^3 to 10^5 pairs.  One wave per parent
// walking the list entry by entry left most of the chip idle on the top plane and waited for a
// few long lists on the others.  Here
//   - a work item is (parent, group of at most kNodeChildren children); the groups per parent
//     (node_groups) grow as the parents get fewer, so a plane of 64 parents still fills the chip;
//   - items of up to kNodeLong list entries are run by one wave each, longer ones by workgroups of
//     kNodeThreads from a queue (the nodes around a void list 100 times as many as the others);
//   - the workgroup flattens the list: NT entries at a time, an exclusive scan of their child counts,
//     and every thread finds its target child by a binary search of the scan, so all lanes hold a
//     target whatever the entries' sizes are;
//   - a thread keeps its target in registers and runs over the group's children, which are read
//     from LDS at wave-uniform addresses.
#pragma once
#include "util.h"

namespace jzt {

constexpr int kNodeChildren = 8;
constexpr int kNodeLong = 256;      // list entries from which on a parent gets workgroups of kNodeThreads
constexpr int kNodeThreads = 256;

// Child groups per parent with `nact` parents: four of eight children, and more of fewer children
// where the parents would not fill the chip (a dense top plane of 64 super-nodes of 32 children: 2048
// items of one child).  Children past groups * width are taken in further rounds of the same groups.
// Items are numbered group by group: most parents have no more than eight children, and with the group
// in the low bits every first group went to two of the eight XCDs (workgroup b runs on XCD b % 8).
struct NodeGroups {
  int groups, width;
};
__device__ __forceinline__ NodeGroups node_groups(int64_t nact) {
  if (nact >= 1024) return {4, 8};
  if (nact >= 256) return {8, 4};
  if (nact >= 128) return {16, 2};
  return {32, 1};
}

// Parents with long lists, left by the one-wave workgroups to workgroups of kNodeThreads: n, then
// their indices.  Null: every parent is handled by one wave per child group.
struct NodeQueue {
  int32_t* q;
  int64_t most;
  __device__ __forceinline__ bool is_long(int len) const { return q != nullptr && len > kNodeLong; }
  __device__ __forceinline__ void push(int p) const {
    const int o = atomicAdd(q, 1);
    if (o < most) q[1 + o] = p;
  }
};
inline int64_t node_queue_words(int64_t nparents) { return nparents + 1; }

// Grid of the node passes: workgroups stride over the items, so that the search for the number of
// parents (active_items) is paid per workgroup and not per item; four times what the chip holds, so
// that the last ones to start do not leave it idle.
inline unsigned node_grid(int64_t nparents, int threads) {
  const int64_t most = 4 * 256 * (2048 / threads);
  const int64_t items = nparents * 32;
  return (unsigned)(items <= 0 ? 1 : (items < most ? items : most));
}

template <int NT> struct TileLds {
  int pre[NT];   // exclusive scan of the batch's target counts
  int off[NT];   // first target of the entry minus its scan value
  int scan[NT / 64];
};

// index of the entry that flattened target j belongs to: the last one with pre <= j (entries without
// targets share their successor's value and are never the last); n >= 1 entries, pre[0] = 0
template <int NT> __device__ __forceinline__ int tile_entry(const TileLds<NT>& s, int n, int j) {
  int lo = 0, hi = n;  // pre[lo] <= j < pre[hi]
#pragma unroll
  for (int it = 0; (1 << it) < NT; it++) {
    const int mid = (lo + hi) >> 1;
    const bool le = mid > lo && s.pre[mid] <= j;
    lo = le ? mid : lo;
    hi = le ? hi : max(mid, lo + 1);
  }
  return lo;
}

// Runs tile(valid, target index) over the children of the entries [e0, e1), NT targets at a time, in
// list order.  entry(e, t0, cnt) gives entry e's children [t0, t0 + cnt) and returns whether the list
// goes on past it: a batch in which some entry says no is the last one.
template <int NT, typename EntryFn, typename TileFn>
__device__ __forceinline__ void for_target_tiles(TileLds<NT>& s, int e0, int e1, EntryFn entry, TileFn tile) {
  const int tid = threadIdx.x;
  for (int eb = e0; eb < e1; eb += NT) {
    int t0 = 0, cnt = 0, tot;
    bool more = true;
    if (eb + tid < e1) more = entry(eb + tid, t0, cnt);
    const int pre = block_excl_scan<NT>(cnt, s.scan, &tot);
    s.pre[tid] = pre;
    s.off[tid] = t0 - pre;
    const bool last = __syncthreads_or(!more);
    const int ne = min(NT, e1 - eb);
    for (int base = 0; base < tot; base += NT) {
      const int j = base + tid;
      const bool valid = j < tot;
      const int e = tile_entry<NT>(s, ne, valid ? j : 0);
      tile(valid, valid ? j + s.off[e] : 0);
    }
    if (last) break;
    __syncthreads();  // pre / off are rewritten
  }
  __syncthreads();
}

}  // namespace jzt
