// Sorted bulk load of an empty tree (reference gpu_blink_tree sorted-input
// constructor, gpu_blink_tree.hpp:85-136, bulk_build_kernel
// btree_kernels.hpp:915-1025; available there only for the plain tree with the
// bump allocator, here for both tree kinds and every node width).
//
// The tree is laid out level by level with `fill` entries per node:
//   node 0                 the root (fixed, internal), over the top level
//   nodes 1 .. c0          leaves: leaf m holds keys [m*fill, (m+1)*fill)
//   then levels 1 .. top   internal nodes, node m of level k over children
//                          [m*fill, (m+1)*fill) of level k-1
// A node's first entry routes keys down from its low bound (pivot 0 for the
// left-most node of a level), its high key is the low bound of its right
// sibling, and the last node of a level has no sibling and high key kEmpty:
// the shape the insert path's splits produce, so later writes continue on it.
// Each tile writes one node with one coalesced store; no node depends on
// another, so the whole build is one grid-stride pass over the nodes.
#pragma once
#include "mvbt_sort.hpp"
#include "mvbt_tree.hpp"

namespace mvbt {

constexpr uint32_t kMaxBulkLevels = 34;  // fill >= 2 and n < 2^32 need at most 32

struct bulk_plan {
  unsigned long long n;      // keys
  unsigned long long total;  // nodes written, root included (= new bump frontier)
  uint32_t fill;             // entries per leaf and per internal node
  uint32_t levels;           // levels below the root; level 0 = leaves
  unsigned long long count[kMaxBulkLevels];  // nodes of each level
  unsigned long long base[kMaxBulkLevels];   // index of each level's first node
  unsigned long long span[kMaxBulkLevels];   // keys under one full node of each level
  unsigned long long extra;  // 1: a last, empty leaf in node 1 behind the keys (a first insert)
};

// The level plan for n keys, leaves from node `first` on, or false when
// `root_cap` entries cannot hold the top level within kMaxBulkLevels levels.
// extra = 1 adds an empty last leaf (node 1, not among those laid out).
MVBT_HD bool make_bulk_plan(unsigned long long n, uint32_t fill, uint32_t root_cap, bulk_plan* p,
                            unsigned long long first = 1, unsigned long long extra = 0) {
  *p = bulk_plan{};
  p->n = n;
  p->fill = fill;
  p->extra = extra;
  unsigned long long c = (n + fill - 1) / fill + extra, span = fill, base = first;
  uint32_t lv = 0;
  for (;;) {
    if (lv >= kMaxBulkLevels) return false;
    p->count[lv] = c;
    p->base[lv] = base;
    p->span[lv] = span;
    base += lv == 0 ? c - extra : c;
    ++lv;
    if (c <= root_cap) break;
    c = (c + fill - 1) / fill;
    span *= fill;
  }
  p->levels = lv;
  p->total = base;
  return true;
}

// Strictly ascending, no reserved key: *bad receives 1 otherwise.
__global__ void bulk_check_kernel(const uint32_t* keys, unsigned long long n, unsigned long long* bad) {
  bool b = false;
  for (unsigned long long i = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; i < n;
       i += (unsigned long long)gridDim.x * blockDim.x) {
    const uint32_t k = keys[i];
    b |= (k == 0u || k == kEmpty || (i + 1 < n && keys[i + 1] <= k));
  }
  if (__builtin_amdgcn_ballot_w64(b) != 0 && __lane_id() == 0) *bad = 1ull;
}

// Index of node m of level lv.
MVBT_DEV uint32_t bulk_index(const bulk_plan& plan, uint32_t lv, unsigned long long m) {
  return lv == 0 && plan.extra && m + 1 == plan.count[0] ? 1u : (uint32_t)(plan.base[lv] + m);
}
// Key i, or past the last one the lowest key of the empty last leaf.
MVBT_DEV uint32_t bulk_key(const bulk_plan& plan, const uint32_t* keys, unsigned long long i) {
  return i < plan.n ? keys[i] : keys[plan.n - 1] + 1;
}

// Lane r's pair of node `id` of the plan (0 is the root).
template <int NW, bool VER>
MVBT_DEV uint64_t bulk_pair(const bulk_plan& plan, unsigned long long id, uint32_t r, const uint32_t* keys,
                            const uint32_t* values, uint32_t stamp) {
  using node_t = node<NW, VER>;
  const uint32_t fill = plan.fill;
  uint64_t p = node_t::kEmptyPair;
  if (id == 0) {
    // root: one entry per node of the top level
    const uint32_t top = plan.levels - 1;
    if (r < plan.count[top]) {
      const unsigned long long first = (unsigned long long)r * plan.span[top];
      p = pack(r == 0 ? 0u : bulk_key(plan, keys, first), bulk_index(plan, top, r));
    } else if (r == node_t::kMetaLane) {
      p = pack(kEmpty, kNoSibling | (plan.levels == 1 ? kAboveLeaves : 0u));
    } else if (VER && r == node_t::kVerLane) {
      p = pack(0u, kNone);
    }
    return p;
  }
  uint32_t lv = 0;
  while (lv + 1 < plan.levels && id >= plan.base[lv + 1]) ++lv;
  const unsigned long long m = id - plan.base[lv];
  const bool last = m + 1 == plan.count[lv];
  const uint32_t sib = last ? kNoSibling : bulk_index(plan, lv, m + 1);
  if (lv == 0) {
    const unsigned long long first = m * fill;
    const unsigned long long cnt = plan.n - first < fill ? plan.n - first : fill;
    if (r < cnt) {
      p = pack(keys[first + r], values[first + r]);
    } else if (r == node_t::kMetaLane) {
      p = pack(last ? kEmpty : bulk_key(plan, keys, first + fill), sib | kLeafBit);
    } else if (VER && r == node_t::kVerLane) {
      p = pack(stamp, kNone);
    }
  } else {
    const unsigned long long below = plan.count[lv - 1], span = plan.span[lv - 1];
    const unsigned long long c0 = m * fill;
    const unsigned long long cnt = last ? below - c0 : fill;
    if (r < cnt) {
      const unsigned long long c = c0 + r;
      p = pack(c == 0 ? 0u : bulk_key(plan, keys, c * span), bulk_index(plan, lv - 1, c));
    } else if (r == node_t::kMetaLane) {
      p = pack(last ? kEmpty : bulk_key(plan, keys, (c0 + fill) * span), sib | (lv == 1 ? kAboveLeaves : 0u));
    } else if (VER && r == node_t::kVerLane) {
      p = pack(0u, kNone);
    }
  }
  return p;
}

template <int NW, bool VER>
__global__ void __launch_bounds__(256) bulk_build_kernel(tree_view<NW, VER> tv, const uint32_t* keys,
                                                         const uint32_t* values, bulk_plan plan) {
  tile<NW> t;
  const unsigned long long tiles = (unsigned long long)gridDim.x * (blockDim.x / NW);
  const uint32_t stamp = VER ? ld32_coherent(&tv.st->clock) : 0u;
  for (unsigned long long id = blockIdx.x * (unsigned long long)(blockDim.x / NW) + threadIdx.x / NW;
       id < plan.total; id += tiles)
    st_coherent(tv.at((uint32_t)id) + t.rank(), bulk_pair<NW, VER>(plan, id, t.rank(), keys, values, stamp));
  if (blockIdx.x == 0 && threadIdx.x == 0) tv.st->bump = plan.total;
}

// ---- A large insert into an empty tree -----------------------------------------
// The first insert of a tree is loaded like a sorted build: its pairs are
// sorted by key (mvbt_sort.hpp, stable, so of equal keys the last one of the
// call is kept), reserved keys are flagged and dropped, and the nodes are
// laid out level by level. Inserted key by key they would all meet on a few
// leaves at first: 1M keys at 16 pairs took 2.28 ms in four growing launches.
// The sort's buffers and the plan lie in the part of the node pool behind the
// nodes the build can need. A reader on another stream (MVBT_CONCURRENT) may
// run meanwhile: it reads the old root and the old, empty leaf (node 1), until
// the last kernel writes the root. Node 1 stays as it is, as an empty last leaf
// behind the largest key (out of use if that is the largest key there is).

// Segment counts of the sorted pairs that stay (radix segments of n).
MVBT_DEV bool first_insert_keeps(const uint32_t* keys, uint32_t i, uint32_t n) {
  const uint32_t k = keys[i];
  return valid_key(k) && (i + 1 == n || keys[i + 1] != k);
}
// 1 if the sorted keys leave a key above the largest valid one (reserved keys sort first and last).
MVBT_DEV unsigned long long largest_key_free(const uint32_t* keys, uint32_t n) {
  uint32_t lo = 0, hi = n;  // first position holding 0xFFFFFFFE or more
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (keys[mid] < kEmpty - 1) lo = mid + 1;
    else hi = mid;
  }
  return lo < n && keys[lo] == kEmpty - 1 ? 0ull : 1ull;
}
__global__ void __launch_bounds__(kSortBlock)
    first_insert_count_kernel(tree_state* st, const uint32_t* keys, uint32_t n, uint32_t* seg) {
  __shared__ uint32_t part[kSortBlock / 64];
  uint32_t a, b, c = 0;
  bool reserved = false;
  segment_of(n, blockIdx.x, gridDim.x, a, b);
  for (uint32_t i = a + threadIdx.x; i < b; i += kSortBlock) {
    c += first_insert_keeps(keys, i, n) ? 1u : 0u;
    reserved |= !valid_key(keys[i]);
  }
  if (__builtin_amdgcn_ballot_w64(reserved) != 0 && __lane_id() == 0) atomic_or32(&st->error_flags, kErrInvalidKey);
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tot = 0;
    for (uint32_t w = 0; w < kSortBlock / 64; ++w) tot += part[w];
    seg[blockIdx.x] = tot;
  }
}

// (after radix_scan_kernel: seg holds each segment's first position, *kept the
// total) Moves the pairs that stay together; block 0 also writes the plan.
__global__ void __launch_bounds__(kSortBlock)
    first_insert_pack_kernel(const uint32_t* keys, const uint32_t* values, uint32_t n, const uint32_t* seg,
                             const uint32_t* kept, uint32_t fill, uint32_t root_cap, uint32_t* out_keys,
                             uint32_t* out_values, bulk_plan* plan) {
  constexpr uint32_t kWaves = kSortBlock / 64;
  __shared__ uint32_t wsum[kWaves];
  const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint64_t below = (1ull << lane) - 1;
  uint32_t a, b;
  segment_of(n, blockIdx.x, gridDim.x, a, b);
  uint32_t run = seg[blockIdx.x];
  for (uint32_t c = a; c < b; c += kSortBlock) {
    const uint32_t i = c + tid;
    const bool keep = i < b && first_insert_keeps(keys, i, n);
    const uint64_t m = __builtin_amdgcn_ballot_w64(keep);
    if (lane == 0) wsum[w] = (uint32_t)__builtin_popcountll(m);
    __syncthreads();
    uint32_t pos = run + (uint32_t)__builtin_popcountll(m & below), tot = 0;
#pragma unroll
    for (uint32_t v = 0; v < kWaves; ++v) {
      if (v < w) pos += wsum[v];
      tot += wsum[v];
    }
    if (keep) {
      out_keys[pos] = keys[i];
      out_values[pos] = values[i];
    }
    run += tot;
    __syncthreads();
  }
  if (blockIdx.x == 0 && tid == 0) make_bulk_plan(*kept, fill, root_cap, plan, 2, largest_key_free(keys, n));
}

// Every node but the root.
template <int NW, bool VER>
__global__ void __launch_bounds__(256) first_insert_nodes_kernel(tree_view<NW, VER> tv, const uint32_t* keys,
                                                                 const uint32_t* values, const bulk_plan* dplan) {
  __shared__ bulk_plan plan;
  for (uint32_t i = threadIdx.x; i < sizeof(bulk_plan) / 4; i += blockDim.x)
    reinterpret_cast<uint32_t*>(&plan)[i] = reinterpret_cast<const uint32_t*>(dplan)[i];
  __syncthreads();
  if (plan.n == 0) return;
  tile<NW> t;
  const unsigned long long tiles = (unsigned long long)gridDim.x * (blockDim.x / NW);
  const uint32_t stamp = VER ? ld32_coherent(&tv.st->clock) : 0u;
  for (unsigned long long id = 2 + blockIdx.x * (unsigned long long)(blockDim.x / NW) + threadIdx.x / NW;
       id < plan.total; id += tiles)
    st_coherent(tv.at((uint32_t)id) + t.rank(), bulk_pair<NW, VER>(plan, id, t.rank(), keys, values, stamp));
}

// The root (one tile), once every other node is in memory.
template <int NW, bool VER>
__global__ void first_insert_root_kernel(tree_view<NW, VER> tv, const uint32_t* keys, const uint32_t* values,
                                         const bulk_plan* plan) {
  if (blockIdx.x != 0 || threadIdx.x >= (unsigned)NW || plan->n == 0) return;
  tile<NW> t;
  st_coherent(tv.at(0) + t.rank(), bulk_pair<NW, VER>(*plan, 0, t.rank(), keys, values, 0u));
  if (t.leader()) tv.st->bump = plan->total;
}

}  // namespace mvbt
