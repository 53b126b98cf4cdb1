// Batched form: many batches of mixed operations in one call.
//
// Semantics (identical to issuing the batches one by one through the plain
// per-batch API with a snapshot before each): batch b reads (find, range) at
// snapshot clock0 + b, i.e. it sees exactly the writes of batches < b; its
// writes (insert, erase) are stamped clock0 + b + 1. The call reserves the
// nb snapshot ids by advancing the tree clock by nb.
//
// Two forms. The sorted form (worker modes 2 and 3; calls of up to kSmallOps
// operations in fewer launches) applies all writes of a window of batches first,
// leaf by leaf in batch order, then answers all its reads at their snapshots; it
// is described from batch_slice_kernel on. The persistent worker (modes 0 and 1,
// which only the autotuner and callers that ask for them use) works through one
// queue of the call's operations:
//
// Scheduling: tiles claim operations one at a time from the queue, in order
// (see the worker). An operation of batch b may run once every write of batches < b has
// completed (a device frontier F = last batch whose writes are all done). A
// write of batch b must also wait for that, because leaf version chains are
// stamp-ordered: a late write of batch b-1 must never follow a copy made by
// batch b. Reads of batch b then overlap writes of batch b and later work.
// The lowest unexecuted operation is always runnable, so the queue drains.
// A tile that must wait polls F once per pass of its outer loop and never
// spins inside a branch (the tiles of a wave run in lockstep).
//
// A batch's writes must name distinct keys: two writes of one key inside a
// batch would make the result depend on which tile runs first. Both forms
// check this with a hash table over (batch, key) of the call's write
// operations and reject the whole call (kErrBadBatch; nothing is applied,
// results are left as they were) when a key repeats, an operation type is
// unknown, or the offsets disagree with the operation count.
//
// Reference counterpart: the ratio-partitioned mixed kernels
// concurrent_insert_range_kernel / concurrent_find_erase_kernel_versioned
// (btree_kernels.hpp:31-306), which take per-tile snapshots inside the
// kernel and are therefore not deterministic.
#pragma once
#include "mvbt_kernels.hpp"
#include "mvbt_sort.hpp"
#include "mvbt_tree.hpp"

namespace mvbt {

enum : uint32_t { kOpFind = 0, kOpInsert = 1, kOpErase = 2, kOpRange = 3 };

// One operation: {type, key or range lower bound, value or range upper
// bound, output slot of a range (pairs at pairs + slot * L)}.
struct op_record {
  uint32_t type, key, arg, slot;
};

// A write of the sorted form: one 16-byte record, so that the gather into
// sorted order touches one line per write.
struct alignas(16) write_rec {
  uint32_t key, arg;
  uint32_t rel;    // index - first_op, bit 31: erase
  uint32_t batch;
};

struct alignas(128) batch_job {
  // per-call parameters (written by batch_setup_kernel or batch_small_begin_kernel)
  const op_record* ops;
  unsigned long long nops;  // one past the last op index (= offsets[nb])
  const unsigned long long* offsets;  // nb + 1 absolute op indices into ops
  uint32_t nb;
  uint32_t L;
  uint32_t* results;     // one word per op
  uint64_t* pairs;       // range output
  unsigned long long pair_slots;  // capacity of `pairs` in slots of L pairs
  uint32_t clock0;
  uint32_t hash_mask;    // conflict table size - 1: a power of two >= 2 * writes (batch_mask_kernel)
  unsigned long long first_op;  // offsets[0]
  // library-owned scratch: capacity batches each, and the conflict table
  uint32_t* nwrites;
  uint32_t* done;
  int32_t* advance;
  uint32_t* hash;        // hash_mask + 1 entries: 0 empty, else 1 + op index - first_op
  uint32_t* op_batch;    // batch of op first_op + i, written by the count pass
  uint32_t bad;          // nonzero: the call was rejected and runs nothing
  uint32_t pad1[1];
  // hot runtime words, one line each
  unsigned long long next_op;  // next unclaimed operation index
  unsigned long long pad2[15];
  // kFrontierCopies replicas of the frontier, one line each: waiting waves
  // poll the replica of their wave id, so polling spreads over L2 channels.
  // Replicas only grow (atomic max), so no replica ever moves backwards.
  int32_t frontier[8 * 32];
  // Sorted form (worker mode 2): library-owned scratch, one entry per
  // operation unless stated.
  uint32_t* list;        // the call's finds, then its ranges (index - first_op), in operation order
  write_rec* writes;     // the call's writes, in operation order
  uint32_t* w_par;       // parent hint of each write of the window; after the gather the lent
                         // slots (lend_slots)
  uint32_t* sort_k[2];   // leaf hints (sort keys), two buffers; the spare one then holds the
                         // sorted writes' parent hints
  uint32_t* sort_v[2];   // positions in the window's writes (sort payloads), two buffers; the
                         // spare one then holds the sorted writes' copy slots (lent: and the first
                         // one their groups)
  write_rec* sorted;     // the window's writes in sorted order
  uint32_t* seg;         // segment counts: kOpClasses * kSliceWaves
  uint32_t* hist;        // kRadix * kSortSegments histogram + kRadix digit totals
  // counts of the current call (zeroed by batch_setup_kernel), one line
  uint32_t n_writes;     // of the current window
  uint32_t n_finds;
  uint32_t n_ranges;
  uint32_t n_planned;    // lent slots: (leaf, batch) groups of the window's writes, each one's slot in w_par
  uint32_t cp_valid;     // planned slots that exist (the rest: pool exhausted)
  uint32_t cp_got;       // of them, taken from the free stack
  uint32_t total_writes;  // write operations of the call (sizes the conflict table)
  uint32_t hash_cap_mask;  // the conflict table's capacity - 1
  long long cp_top;                 // free-stack top before the reservation
  unsigned long long cp_bump;       // first never-used index of the reservation
  unsigned long long cp_ring;       // first retire-ring position of the reservation
  // windows of the sorted form: the call's batches in `windows` consecutive
  // groups of about equal operation count
  uint32_t windows;
  uint32_t reclaim;
  uint32_t first[3];     // the window's first write, find and range in their part of `list`
  uint32_t total[3];     // the call's writes, finds and ranges
  uint32_t lend;         // 1: copy slots are lent to the call (lend_slots)
  uint32_t pad4[9];
};
constexpr uint32_t kFrontierCopies = 8;

struct batch_params {
  const op_record* ops;
  unsigned long long nops;
  const unsigned long long* offsets;
  uint32_t nb;
  uint32_t L;
  uint32_t* results;
  uint64_t* pairs;
  unsigned long long pair_slots;
  uint32_t* base_out;
  uint32_t hash_mask;
  uint32_t windows;  // sorted form: windows of batches the call runs in (>= 1)
  uint32_t reclaim;  // sorted form: free every retired copy after each window
  uint32_t lend;     // sorted form: see lend_slots (small calls: always)
};

// 1. Parameters in, clock range reserved, queue reset.
__global__ void batch_setup_kernel(batch_job* job, tree_state* st, batch_params p) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  job->ops = p.ops;
  job->offsets = p.offsets;
  job->nb = p.nb;
  job->L = p.L;
  job->results = p.results;
  job->pairs = p.pairs;
  job->pair_slots = p.pair_slots;
  job->clock0 = __hip_atomic_fetch_add(&st->clock, p.nb, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
  job->hash_cap_mask = p.hash_mask;
  job->hash_mask = 1023u;
  job->total_writes = 0;
  // Operation indices are absolute: batch b covers ops [offsets[b], offsets[b+1]),
  // results go to the same indices; offsets[nb] - offsets[0] must equal the op
  // count the caller passed (the size its buffers were checked against).
  const unsigned long long first = p.offsets[0], last = p.offsets[p.nb];
  const bool ok = last >= first && last - first == p.nops;
  job->first_op = first;
  job->next_op = first;
  job->nops = ok ? last : first;
  job->bad = ok ? 0u : 1u;
  job->n_writes = 0;
  job->n_finds = 0;
  job->n_ranges = 0;
  job->n_planned = 0;
  job->lend = p.lend;
  job->windows = p.windows > 0 ? p.windows : 1u;
  job->reclaim = p.reclaim;
  if (p.base_out) *p.base_out = job->clock0;  // clock0 goes back to the caller
  if (!ok) atomic_or32(&st->error_flags, kErrBadBatch);
  for (uint32_t c = 0; c < kFrontierCopies; ++c) job->frontier[c * 32] = -1;
}

// 0. Points a job descriptor at its scratch arrays from the device side (the
// allocation-free entry point: the job and its scratch all lie in one static
// device array, so no host copy is needed).
constexpr uint32_t kSortedPtrs = 10;  // list .. hist of batch_job
struct scratch_layout {
  uint32_t* nwrites;
  uint32_t* done;
  int32_t* advance;
  uint32_t* hash;
  uint32_t* op_batch;
  uint32_t* sorted[kSortedPtrs];  // list .. hist, in the order of batch_job
};
__global__ void batch_bind_kernel(batch_job* job, scratch_layout l) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  job->nwrites = l.nwrites;
  job->done = l.done;
  job->advance = l.advance;
  job->hash = l.hash;
  job->op_batch = l.op_batch;
  job->list = l.sorted[0];
  job->writes = reinterpret_cast<write_rec*>(l.sorted[1]);
  job->w_par = l.sorted[2];
  job->sort_k[0] = l.sorted[3];
  job->sort_k[1] = l.sorted[4];
  job->sort_v[0] = l.sorted[5];
  job->sort_v[1] = l.sorted[6];
  job->sorted = reinterpret_cast<write_rec*>(l.sorted[7]);
  job->seg = l.sorted[8];
  job->hist = l.sorted[9];
}

// 1'. Clears the conflict table (a fill kernel, so the launch graph holds no
// memset node).
__global__ void batch_clear_kernel(batch_job* job) {
  const uint32_t n = job->hash_mask + 1;
  uint32_t* h = job->hash;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) h[i] = 0;
}

MVBT_DEV uint32_t batch_of(const unsigned long long* offsets, uint32_t nb, unsigned long long i);

MVBT_DEV uint32_t conflict_hash(uint32_t key, uint32_t b) {
  uint32_t h = key * 0x9E3779B1u ^ (b * 0x7FEB352Du + 0x165667B1u);
  h ^= h >> 15;
  h *= 0x846CA68Bu;
  h ^= h >> 16;
  return h;
}

// Records write op i (batch b, valid key) in the conflict table; false when
// batch b already writes `key`. Linear probing; the table has at least twice
// as many entries as the call has operations, so a free entry always exists.
MVBT_DEV bool claim_write(const batch_job* job, unsigned long long i, uint32_t b, uint32_t key) {
  const uint32_t mask = job->hash_mask;
  uint32_t* table = job->hash;
  const uint32_t me = (uint32_t)(i - job->first_op) + 1u;
  uint32_t h = conflict_hash(key, b) & mask;
  for (uint32_t probe = 0; probe <= mask; ++probe) {
    uint32_t cur = ld32_coherent(table + h);
    if (cur == 0) {
      cur = atomic_cas32(table + h, 0u, me);
      if (cur == 0) return true;
    }
    const unsigned long long j = job->first_op + cur - 1u;
    if (job->ops[j].key == key && job->op_batch[cur - 1u] == b) return false;
    h = (h + 1) & mask;
  }
  return true;
}

// 2. Writes per batch (one block per batch, grid-stride over batches), each
// operation's batch, the call's write count, and the first checks: known op
// types, ordered offsets.
__global__ void batch_count_kernel(batch_job* job, tree_state* st) {
  __shared__ uint32_t partial[4];
  const uint32_t nb = job->nb;
  if (ld32_coherent(&job->bad)) return;  // offsets disagree with the op count
  for (uint32_t b = blockIdx.x; b < nb; b += gridDim.x) {
    const unsigned long long lo = job->offsets[b], hi = job->offsets[b + 1];
    uint32_t c = 0;
    bool bad = hi < lo;
    for (unsigned long long i = lo + threadIdx.x; i < hi; i += blockDim.x) {
      const op_record o = job->ops[i];
      const bool w = o.type == kOpInsert || o.type == kOpErase;
      c += w ? 1u : 0u;
      job->op_batch[i - job->first_op] = b;
      if (o.type > kOpRange) bad = true;
    }
    if (bad) {
      atomic_or32(&job->bad, 1u);
      atomic_or32(&st->error_flags, kErrBadBatch);
    }
    // wave reduction via ballot-free shuffles
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t tot = 0;
      for (uint32_t w = 0; w < (blockDim.x + 63) / 64; ++w) tot += partial[w];
      job->nwrites[b] = tot;
      job->done[b] = 0;
      if (tot) atomic_add32(&job->total_writes, tot);
    }
    __syncthreads();
  }
}

// Operation classes of the sorted form: writes (insert, erase), finds, ranges.
MVBT_DEV uint32_t op_class(uint32_t ty) {
  return (ty == kOpInsert || ty == kOpErase) ? 0u : ty == kOpFind ? 1u : ty == kOpRange ? 2u : 3u;
}
constexpr uint32_t kOpClasses = 3;

// 2 (sorted form). Each operation's batch, the checks, and the operations of
// each class, over equal slices of the operations, one to a wave
// (seg[class * kSliceWaves + slice]): the batches differ in size by three
// orders of magnitude, and a workgroup to a batch waits for the largest (480
// batches of 4M operations: 129 us). A workgroup looks its slices' batches up
// in a copy of their offsets in LDS where it has at most kSliceBatches.
constexpr uint32_t kSliceBatches = 2048;
constexpr uint32_t kSliceBlocks = 1024, kSliceWaves = kSliceBlocks * (kSortBlock / 64);
MVBT_DEV uint32_t batch_in(const unsigned long long* offsets, uint32_t lo, uint32_t hi, unsigned long long i) {
  while (hi - lo > 1) {  // offsets[lo] <= i < offsets[hi]
    const uint32_t mid = (lo + hi) >> 1;
    if (offsets[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}
__global__ void __launch_bounds__(kSortBlock) batch_slice_kernel(batch_job* job, tree_state* st) {
  constexpr uint32_t kWaves = kSortBlock / 64;
  __shared__ unsigned long long off[kSliceBatches + 1];
  __shared__ uint32_t bounds[2];
  const uint32_t nb = job->nb, tid = threadIdx.x, lane = tid & 63, w = blockIdx.x * kWaves + tid / 64;
  const unsigned long long first = job->first_op;
  const uint32_t n = (uint32_t)(job->nops - first);  // 0 if the offsets disagree with the op count
  bool bad = false;
  if (n)
    for (uint32_t b = blockIdx.x * kSortBlock + tid; b < nb; b += gridDim.x * kSortBlock)
      bad |= job->offsets[b + 1] < job->offsets[b];
  uint32_t a, e, unused, c[kOpClasses] = {0, 0, 0};
  segment_of(n, blockIdx.x * kWaves, kSliceWaves, a, unused);
  segment_of(n, blockIdx.x * kWaves + kWaves - 1, kSliceWaves, unused, e);
  if (a < e) {
    if (tid < 2) bounds[tid] = batch_in(job->offsets, 0, nb, first + (tid ? e - 1 : a));
    __syncthreads();
    // (offsets out of order may give any batches here: the call is rejected)
    const uint32_t b0 = bounds[0], b1 = bounds[1] < b0 ? b0 : bounds[1];
    const bool local = b1 - b0 < kSliceBatches;
    if (local) {
      for (uint32_t k = tid; k <= b1 - b0 + 1; k += kSortBlock) off[k] = job->offsets[b0 + k];
      __syncthreads();
    }
    segment_of(n, w, kSliceWaves, a, e);
    for (uint32_t i0 = a; i0 < e; i0 += 64) {
      const uint32_t i = i0 + lane;
      uint32_t k = kOpClasses;
      if (i < e) {
        k = op_class(job->ops[first + i].type);
        bad |= k == kOpClasses;
        job->op_batch[i] =
            local ? b0 + batch_in(off, 0, b1 - b0 + 1, first + i) : batch_in(job->offsets, b0, b1 + 1, first + i);
      }
#pragma unroll
      for (uint32_t q = 0; q < kOpClasses; ++q) c[q] += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(k == q));
    }
  }
  if (lane < kOpClasses) job->seg[lane * kSliceWaves + w] = lane == 0 ? c[0] : lane == 1 ? c[1] : c[2];
  if (bad) {
    atomic_or32(&job->bad, 1u);
    atomic_or32(&st->error_flags, kErrBadBatch);
  }
}

// 2b. One workgroup per class: slice counts to positions, the call's totals,
// and (a call in one window) the window's counts. The first one also sizes
// the conflict table: the smallest power of two >= twice the call's writes
// (at least 1024, at most its capacity), so a table that fits the caches
// serves a call whose operations are mostly reads.
__global__ void __launch_bounds__(kSortBlock) batch_class_scan_kernel(batch_job* job) {
  static_assert(kSliceWaves <= kScanMax, "one row");
  __shared__ scan_lds l;
  const uint32_t q = blockIdx.x;
  const uint32_t total = scan_row(job->seg + q * kSliceWaves, kSliceWaves, l);
  if (threadIdx.x != kSortBlock - 1) return;
  job->total[q] = total;
  job->first[q] = 0;
  (q == 0 ? job->n_writes : q == 1 ? job->n_finds : job->n_ranges) = total;
  if (q == 0) {
    unsigned long long e = 1024;
    while (e < 2ull * total) e *= 2;
    const unsigned long long cap = (unsigned long long)job->hash_cap_mask + 1;
    job->hash_mask = (uint32_t)((e < cap ? e : cap) - 1);
  }
}

// 2c. Every class to its list, in operation order (a stable scatter per slice;
// no shared counter); the conflict table is cleared.
__global__ void __launch_bounds__(kSortBlock) batch_split_kernel(batch_job* job) {
  if (ld32_coherent(&job->bad)) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63, w = blockIdx.x * (kSortBlock / 64) + tid / 64;
  const uint32_t n = (uint32_t)(job->nops - job->first_op);
  const op_record* ops = job->ops + job->first_op;
  const uint32_t* op_batch = job->op_batch;
  const uint64_t below = (1ull << lane) - 1;
  uint32_t a, e, run[kOpClasses];
  segment_of(n, w, kSliceWaves, a, e);
#pragma unroll
  for (uint32_t q = 0; q < kOpClasses; ++q)
    run[q] = job->seg[q * kSliceWaves + w] + (q == 2 ? job->total[1] : 0u);  // ranges behind the finds
  for (uint32_t i0 = a; i0 < e; i0 += 64) {
    const uint32_t i = i0 + lane;
    op_record o{};
    uint32_t k = kOpClasses, b = 0;
    if (i < e) {
      o = ops[i];
      b = op_batch[i];
      k = op_class(o.type);
    }
#pragma unroll
    for (uint32_t q = 0; q < kOpClasses; ++q) {
      const uint64_t m = __builtin_amdgcn_ballot_w64(k == q);
      const uint32_t pos = run[q] + (uint32_t)__builtin_popcountll(m & below);
      if (k == q) {
        if (q == 0) job->writes[pos] = write_rec{o.key, o.arg, i | (o.type == kOpErase ? 0x80000000u : 0u), b};
        else job->list[pos] = i;
      }
      run[q] += (uint32_t)__builtin_popcountll(m);
    }
  }
  const uint32_t mask = job->hash_mask;
  for (uint32_t i = blockIdx.x * kSortBlock + tid; i <= mask; i += gridDim.x * kSortBlock) job->hash[i] = 0;
}

// 2d. Distinct write keys per batch: every write of a valid key claims
// (batch, key) in the conflict table (an entry is 1 + the write's position);
// a second claim rejects the call. The table has at least twice as many
// entries as the call has writes, so a free entry always exists.
__global__ void __launch_bounds__(kSortBlock) batch_claim_kernel(batch_job* job, tree_state* st) {
  if (ld32_coherent(&job->bad)) return;
  const uint32_t n = job->total[0], mask = job->hash_mask;
  const write_rec* writes = job->writes;
  uint32_t* table = job->hash;
  bool bad = false;
  for (uint32_t i = blockIdx.x * kSortBlock + threadIdx.x; i < n; i += gridDim.x * kSortBlock) {
    const uint32_t key = writes[i].key, b = writes[i].batch;
    if (!valid_key(key)) continue;
    uint32_t h = conflict_hash(key, b) & mask;
    for (uint32_t probe = 0; probe <= mask; ++probe) {
      const uint32_t cur = atomic_cas32(table + h, 0u, i + 1);  // most entries are free: no look before
      if (cur == 0) break;
      if (writes[cur - 1].key == key && writes[cur - 1].batch == b) {
        bad = true;
        break;
      }
      h = (h + 1) & mask;
    }
  }
  if (bad) {
    atomic_or32(&job->bad, 1u);
    atomic_or32(&st->error_flags, kErrBadBatch);
  }
}

// 2' (modes 0 and 1). The conflict table's size: the smallest power of two >= twice the
// call's writes (at least 1024, at most its capacity), so a table that fits
// the caches serves a call whose operations are mostly reads.
__global__ void batch_mask_kernel(batch_job* job) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  unsigned long long e = 1024;
  while (e < 2ull * job->total_writes) e *= 2;
  const unsigned long long cap = (unsigned long long)job->hash_cap_mask + 1;
  job->hash_mask = (uint32_t)((e < cap ? e : cap) - 1);
}

// 2''. (after batch_clear_kernel) Distinct write keys per batch: every write
// of a valid key claims (batch, key) in the conflict table; a second claim
// rejects the call.
__global__ void batch_conflict_kernel(batch_job* job, tree_state* st) {
  if (ld32_coherent(&job->bad)) return;
  const unsigned long long first = job->first_op, n = job->nops - first;
  bool bad = false;
  for (unsigned long long r = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; r < n;
       r += (unsigned long long)gridDim.x * blockDim.x) {
    const op_record o = job->ops[first + r];
    if ((o.type == kOpInsert || o.type == kOpErase) && valid_key(o.key) &&
        !claim_write(job, first + r, job->op_batch[r], o.key))
      bad = true;
  }
  if (bad) {
    atomic_or32(&job->bad, 1u);
    atomic_or32(&st->error_flags, kErrBadBatch);
  }
}

// 3. advance[b] = frontier value once batch b's writes are done: the last
// batch of the run of write-free batches that follows b.
__global__ void batch_frontier_kernel(batch_job* job) {
  const uint32_t nb = job->nb;
  for (uint32_t b = blockIdx.x * blockDim.x + threadIdx.x; b < nb; b += gridDim.x * blockDim.x) {
    uint32_t j = b + 1;
    while (j < nb && job->nwrites[j] == 0) ++j;
    job->advance[b] = (int32_t)j - 1;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    uint32_t j = 0;
    while (j < nb && job->nwrites[j] == 0) ++j;
    for (uint32_t c = 0; c < kFrontierCopies; ++c) job->frontier[c * 32] = (int32_t)j - 1;
  }
}

// Batch of op i (offsets[0] <= i < offsets[nb]), by bisection.
MVBT_DEV uint32_t batch_of(const unsigned long long* offsets, uint32_t nb, unsigned long long i) {
  uint32_t lo = 0, hi = nb;  // offsets[lo] <= i < offsets[hi] (i in [offsets[0], offsets[nb]))
  while (hi - lo > 1) {
    uint32_t mid = (lo + hi) >> 1;
    if (offsets[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

// 4. The persistent worker. Each tile holds one operation at a time, so a
// batch spreads over as many tiles as it has operations and a batch's writes
// finish after about one write latency. The idle tiles of a wave claim the
// next operations of the single queue together, with one atomic (ranked by
// tile order). Claims are in operation order, so the lowest unexecuted
// operation is always held by a running tile and runnable: the queue drains
// without deadlock however many of the launch's blocks are resident (a block
// claims only while it runs). Per-wave home queues would lose this: ops of a
// queue whose waves are not resident could block every resident tile.
template <int NW>
__global__ void __launch_bounds__(256) batch_worker_kernel(tree_ptrs tp, batch_job* job) {
  if (ld32_coherent(&job->bad)) return;  // rejected call: nothing runs
  const tree_view<NW, true> tv(tp);
  using node_t = node<NW, true>;
  tile<NW> t;
  const unsigned long long nops = job->nops;
  const uint32_t L = job->L, clock0 = job->clock0;
  const op_record* ops = job->ops;
  uint32_t* results = job->results;
  uint64_t* pairs = job->pairs;
  const unsigned long long pair_slots = job->pair_slots;
  const uint32_t lane = __lane_id();
  const uint32_t my_tile = lane / NW;  // tile index within the wave
  const uint32_t wave = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
  int32_t* const my_frontier = job->frontier + (wave % kFrontierCopies) * 32;
  uint32_t backoff = 1;  // s_sleep units while the whole wave waits
  write_ctx ctx = tv.begin_writes(t);
  ctx.track = 0;          // stamps are fixed per batch: clock0 + b + 1
  int32_t seen = -1;      // last frontier value observed (tile-uniform)
  bool have = false;      // tile holds an operation (tile-uniform)
  unsigned long long idx = 0;
  op_record op{};
  uint32_t b = 0;
  uint32_t waits = 0;     // consecutive passes without progress
  for (;;) {
    // Idle tiles of this wave claim operations together.
    const uint64_t idle = __builtin_amdgcn_ballot_w64(!have && t.leader());
    if (idle) {
      const uint32_t n_idle = (uint32_t)__builtin_popcountll(idle);
      const uint32_t first = (uint32_t)__builtin_ctzll(idle);
      unsigned long long base = 0;
      if (lane == first) base = atomic_add64(&job->next_op, (unsigned long long)n_idle);
      base = ((unsigned long long)__builtin_amdgcn_readlane((int)(uint32_t)(base >> 32), (int)first) << 32) |
             (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)base, (int)first);
      if (!have) {
        // rank of this tile among the idle tiles (tile leaders are lanes my_tile*NW)
        const uint64_t below = (my_tile == 0) ? 0ull : (idle & ((1ull << (my_tile * NW)) - 1));
        idx = base + (unsigned long long)__builtin_popcountll(below);
        if (idx >= nops) break;  // queue drained
        op = ops[idx];
        b = job->op_batch[idx - job->first_op];
        have = true;
      }
    }
    // Tiles whose batch is not yet open refresh their view of the frontier:
    // one load per wave (the first such tile leader's), shared by readlane.
    const bool blocked = (int32_t)b - 1 > seen;
    const uint64_t need = __builtin_amdgcn_ballot_w64(blocked && t.leader());
    if (need) {
      const uint32_t poller = (uint32_t)__builtin_ctzll(need);
      int32_t f = 0;
      if (lane == poller) f = __hip_atomic_load(my_frontier, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      f = __builtin_amdgcn_readlane(f, (int)poller);
      if (f > seen) seen = f;
    }
    if ((int32_t)b - 1 > seen) {
      if (++waits > (1u << 21)) {  // seconds: the frontier never moved
        tv.flag(kErrCorrupt, t);
        break;
      }
      // back off only when no tile of the wave can work
      if (__builtin_amdgcn_ballot_w64(!((int32_t)b - 1 > seen)) == 0) {
        for (uint32_t i = 0; i < backoff; ++i) __builtin_amdgcn_s_sleep(8);
        if (backoff < 16) backoff *= 2;
      }
      continue;
    }
    waits = 0;
    backoff = 1;
    // Every operation starts with a root-to-leaf walk, so the tiles of a wave
    // take it together whatever their operation types: their node loads
    // overlap instead of running type by type. Only the short leaf-side parts
    // below diverge.
    uint32_t rkey = op.key;
    if (op.type == kOpRange && rkey == 0) rkey = 1;
    const bool route = valid_key(rkey) && !(op.type == kOpRange && op.arg <= rkey);
    node_t n;
    uint32_t leaf = kNone, par = kNone;
    if (route) leaf = tv.template descend<true, true>(rkey, n, t, &par);
    uint32_t r;
    if (op.type == kOpFind) {
      r = route ? tv.template find_in<true, false>(op.key, clock0 + b, n, leaf, t) : kEmpty;
    } else if (op.type == kOpRange) {
      uint64_t* out = (pairs && op.slot < pair_slots) ? pairs + (size_t)op.slot * L : nullptr;
      if (pairs && op.slot >= pair_slots) tv.flag(kErrCorrupt, t);
      r = route ? tv.template range_in<true, false>(rkey, op.arg, clock0 + b, n, leaf, out, L, t) : 0u;
      if (r > L) tv.flag(kErrRangeOverflow, t);
    } else {
      ctx.cur = clock0 + b + 1;
      ctx.want = NW;  // refills grow with demand (write_ctx::grow)
      r = (op.type == kOpInsert) ? tv.template write<0>(op.key, op.arg, ctx, t, leaf, par)
                                 : tv.template write<1>(op.key, 0u, ctx, t, leaf, par);
      order_release();  // this write's stores complete before it is counted
      if (t.leader()) {
        uint32_t prev = atomic_add32(job->done + b, 1u);
        if (prev + 1 == job->nwrites[b]) {
          const int32_t adv = job->advance[b];
          for (uint32_t c = 0; c < kFrontierCopies; ++c)
            __hip_atomic_fetch_max(job->frontier + c * 32, adv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
    if (t.leader()) results[idx] = r;
    have = false;
  }
  tv.finish(ctx, t);
}

// 4'. The chunked worker. A tile claims a run of C consecutive operations
// (lane j holds operation start + j) and routes all of them at once, before
// their batches open: every key stops one level above the leaves and takes
// its leaf from the parent's entry (routing reads only the latest internal
// nodes, which need no frontier). The run is then worked through batch
// segment by batch segment, each once its batch is open (the frontier rule of
// the single-op worker), with only the leaf side left to do: inserts and
// erases go through the batched leaf phase (write_chunk) from the leaf hints,
// finds run a pass engine that starts at the hints and moves right or down
// as the tree has changed since (find_chunk_from), ranges start there one at
// a time; the segment's writes are counted with one atomic. So the walk from
// the root, about half of an operation's dependent loads, overlaps the wait
// for earlier batches instead of following it.
// C follows the size of the batch the wave claimed from last: batch size /
// tiles in the grid, clamped to [1, W], so small batches still spread one
// operation per tile and large ones are taken W at a time. Claims stay in
// operation order and each tile finishes its segments in order, so the
// lowest unfinished operation is always held by a running tile whose earlier
// segments are done: the queue drains as in the single-op worker.
template <int NW>
__global__ void __launch_bounds__(256) batch_chunk_worker_kernel(tree_ptrs tp, batch_job* job) {
  if (ld32_coherent(&job->bad)) return;  // rejected call: nothing runs
  const tree_view<NW, true> tv(tp);
  using node_t = node<NW, true>;
  tile<NW> t;
  const unsigned long long nops = job->nops, first_op = job->first_op;
  const uint32_t L = job->L, clock0 = job->clock0;
  const op_record* ops = job->ops;
  const unsigned long long* offsets = job->offsets;
  const uint32_t* op_batch = job->op_batch;
  uint32_t* results = job->results;
  uint64_t* pairs = job->pairs;
  const unsigned long long pair_slots = job->pair_slots;
  const uint32_t lane = __lane_id(), r = t.rank();
  const uint32_t my_tile = lane / NW;
  const uint32_t wave = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
  int32_t* const my_frontier = job->frontier + (wave % kFrontierCopies) * 32;
  const unsigned long long tiles_total = (unsigned long long)gridDim.x * (blockDim.x / NW);
  uint32_t backoff = 1;
  // The top levels in LDS (as in write_kernel, at 32-pair nodes only), copied
  // once per block of the persistent launch: used when the job gives every
  // tile several operations (the copy delays the block's first one) and the
  // tree's nodes can hold the whole job (its splits then leave the images
  // about one right move stale at most).
  __shared__ route_cache<NW, 16384> rc;
  if constexpr (NW == 32)
    tv.build_route_cache(rc, nops - first_op >= 4 * tiles_total ? (nops - first_op) / node_t::kData + 1 : ~0ull);
  write_ctx ctx = tv.begin_writes(t);
  ctx.exact = 1;
  ctx.track = 0;  // stamps are fixed per batch: clock0 + b + 1
  int32_t seen = -1;
  bool have = false;          // tile holds an unfinished run (tile-uniform)
  uint64_t pending = 0;       // lanes of the run not yet done (tile-uniform)
  unsigned long long cstart = 0;
  uint32_t wave_b = 0;        // batch of the wave's last claim (run sizing)
  op_record op{};             // lane j: operation cstart + j
  uint32_t ob = 0;            // lane j: its batch
  uint32_t hint = kNone, hint_par = kNone;  // lane j: leaf hint and its parent
  bool routed = false;        // lane j: its key was routed
  uint32_t waits = 0;
  for (;;) {
    const uint64_t idle = __builtin_amdgcn_ballot_w64(!have && t.leader());
    bool fresh = false;  // tile-uniform: claimed a run in this pass
    if (idle) {
      const uint32_t n_idle = (uint32_t)__builtin_popcountll(idle);
      const uint32_t first = (uint32_t)__builtin_ctzll(idle);
      const unsigned long long bsz = offsets[wave_b + 1] - offsets[wave_b];
      const unsigned long long cq = bsz / tiles_total;
      const uint32_t C = cq < 1 ? 1u : (cq > (unsigned long long)NW ? (uint32_t)NW : (uint32_t)cq);
      unsigned long long base = 0;
      if (lane == first) base = atomic_add64(&job->next_op, (unsigned long long)n_idle * C);
      base = ((unsigned long long)__builtin_amdgcn_readlane((int)(uint32_t)(base >> 32), (int)first) << 32) |
             (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)base, (int)first);
      if (!have) {
        const uint64_t below = (my_tile == 0) ? 0ull : (idle & ((1ull << (my_tile * NW)) - 1));
        cstart = base + (unsigned long long)__builtin_popcountll(below) * C;
        if (cstart >= nops) break;  // queue drained
        const unsigned long long end = cstart + C < nops ? cstart + C : nops;
        const bool mine = cstart + r < end;
        if (mine) {
          op = ops[cstart + r];
          ob = op_batch[cstart + r - first_op];
        }
        pending = t.ballot(mine);
        have = true;
        fresh = true;
      }
      // size the wave's next runs from the batch its claim started in
      if (base < nops) wave_b = op_batch[base - first_op];
    }
    // route the operations just claimed, whatever their batch
    if (__builtin_amdgcn_ballot_w64(fresh)) {
      uint32_t rkey = op.key;
      if (op.type == kOpRange && rkey == 0) rkey = 1;
      const bool route = fresh && ((pending >> r) & 1) && valid_key(rkey) && !(op.type == kOpRange && op.arg <= rkey);
      const uint64_t todo = t.ballot(route);
      uint32_t st0 = kNone, sp0 = kNone;
      if constexpr (NW == 32) {
        if (route) st0 = tv.route_lane(rc, rkey, sp0);
      }
      uint32_t lf = kNone, pr = kNone;
      tv.template descend_chunk<true>(rkey, todo, lf, pr, t, todo, st0, sp0);
      if (fresh) {
        hint = lf;
        hint_par = pr;
        routed = route && lf < tv.cap_;
      }
    }
    if (!have) continue;
    // the run's next segment: its pending operations of the lowest pending batch
    const uint32_t b = t.shfl(ob, (uint32_t)lowest_bit(pending));
    const bool blocked = (int32_t)b - 1 > seen;
    const uint64_t need = __builtin_amdgcn_ballot_w64(blocked && t.leader());
    if (need) {
      const uint32_t poller = (uint32_t)__builtin_ctzll(need);
      int32_t f = 0;
      if (lane == poller) f = __hip_atomic_load(my_frontier, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      f = __builtin_amdgcn_readlane(f, (int)poller);
      if (f > seen) seen = f;
    }
    if ((int32_t)b - 1 > seen) {
      if (++waits > (1u << 21)) {  // seconds: the frontier never moved
        tv.flag(kErrCorrupt, t);
        break;
      }
      if (__builtin_amdgcn_ballot_w64(have && !((int32_t)b - 1 > seen)) == 0) {
        for (uint32_t i = 0; i < backoff; ++i) __builtin_amdgcn_s_sleep(8);
        if (backoff < 16) backoff *= 2;
      }
      continue;
    }
    waits = 0;
    backoff = 1;
    const uint32_t ts = clock0 + b;
    const bool mine = ((pending >> r) & 1) && ob == b;
    const uint64_t seg = t.ballot(mine);
    const bool is_w = mine && (op.type == kOpInsert || op.type == kOpErase);
    const bool is_rd = mine && !is_w;
    uint32_t res = 0;
    // writes: batched leaf phase from the hints, then the keys it hands back one by one
    ctx.cur = ts + 1;
    const uint64_t qw = t.ballot(is_w);
    for (int w = 0; w < 2; ++w) {
      uint64_t q = t.ballot(is_w && op.type == (w == 0 ? kOpInsert : kOpErase));
      if (!q) continue;
      ctx.want = (uint32_t)__builtin_popcountll(q);
      q = (w == 0) ? tv.template write_chunk<0>(op.key, op.arg, q, hint, res, ctx, t)
                   : tv.template write_chunk<1>(op.key, 0u, q, hint, res, ctx, t);
      while (q) {
        const uint32_t j = (uint32_t)lowest_bit(q);
        ctx.want = (uint32_t)__builtin_popcountll(q);
        q &= q - 1;
        const uint32_t k = t.shfl(op.key, j);
        const uint32_t lf = t.shfl(hint, j), pr = t.shfl(hint_par, j);
        const uint32_t v = (w == 0) ? tv.template write<0>(k, t.shfl(op.arg, j), ctx, t, lf, pr)
                                    : tv.template write<1>(k, 0u, ctx, t, lf, pr);
        if (r == j) res = v;
      }
    }
    // reads at the batch's snapshot, from the hints: finds together, ranges one by one
    const uint64_t ok = t.ballot(routed);
    {
      const uint64_t qf = t.ballot(is_rd && op.type == kOpFind);
      if (qf) {
        const uint32_t v = tv.find_chunk_from(op.key, hint, ts, qf & ok, t);
        if ((qf >> r) & 1) res = v;
      }
    }
    uint64_t qr = t.ballot(is_rd && op.type == kOpRange);
    while (qr) {
      const uint32_t j = (uint32_t)lowest_bit(qr);
      qr &= qr - 1;
      const uint32_t k = t.shfl(op.key, j), a = t.shfl(op.arg, j), lf = t.shfl(hint, j);
      const uint32_t sl = t.shfl(op.slot, j);
      uint64_t* out = (pairs && sl < pair_slots) ? pairs + (size_t)sl * L : nullptr;
      if (pairs && sl >= pair_slots) tv.flag(kErrCorrupt, t);
      uint32_t v = 0;
      if ((ok >> j) & 1) v = tv.template range<true, false>(k == 0 ? 1u : k, a, ts, out, L, t, lf);
      if (v > L) tv.flag(kErrRangeOverflow, t);
      if (r == j) res = v;
    }
    if (mine) results[cstart + r] = res;
    // count the segment's writes: one atomic; the batch's last one opens the next
    if (qw) {
      order_release();  // the segment's stores complete before they are counted
      if (t.leader()) {
        const uint32_t cnt = (uint32_t)__builtin_popcountll(qw);
        const uint32_t prev = atomic_add32(job->done + b, cnt);
        if (prev + cnt == job->nwrites[b]) {
          const int32_t adv = job->advance[b];
          for (uint32_t c = 0; c < kFrontierCopies; ++c)
            __hip_atomic_fetch_max(job->frontier + c * 32, adv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
    pending &= ~seg;
    if (!pending) have = false;
  }
  tv.finish(ctx, t);
}

// ---- The sorted form (worker mode 2) ------------------------------------------
// The whole stream is known when the call starts, so it need not run batch
// after batch. Because every read names its snapshot and the tree keeps
// versions, a read of batch b gives the same answer after every write of the
// call as before the writes of batch b: it reads the version stamped <=
// clock0 + b. So the call applies all its writes first and then answers all
// its reads in one parallel pass. The writes only have to keep, per leaf,
// the order of their batches (version chains are stamp-ordered); writes to
// different leaves are independent. The pipeline:
//   split  the writes, in operation order, into one list; finds and ranges
//          into two more (any order);
//   route  every write to its leaf (the tree is quiescent: no writer runs);
//   sort   the writes by leaf, stably (mvbt_sort.hpp), so each leaf's
//          writes are contiguous and in operation order, i.e. batch order;
//   write  each tile owns the leaf groups that start in its window of the
//          sorted list (a group that runs past the window stays with the
//          tile that holds its start), and applies each group's writes
//          batch by batch: one round writes, for every group, the writes of
//          its earliest remaining batch through the batched leaf phase with
//          that batch's stamp (write_chunk_at); keys it hands back (split,
//          moved right) go one by one. No other tile writes a group's leaves
//          or the leaves split from them, so no leaf lock is ever contended;
//   read   finds and ranges, each at its batch's snapshot, as plain
//          snapshot reads (no writer runs any more).
// No frontier and no per-batch wait: a call costs a few bulk passes however
// many batches it holds. Results are identical to the per-batch path.

// 5'. Window k of the sorted form: the batches whose first operation lies in
// the k-th of `windows` equal slices of the call's operations (a batch is
// never split). Windows run one after another; a read of a window sees the
// writes of the earlier windows, which have been applied, and of its own
// earlier batches, as in the whole-call form.
MVBT_DEV uint32_t window_start(const batch_job* job, uint32_t k) {
  const uint32_t nb = job->nb, K = job->windows;
  if (k == 0) return 0;
  if (k >= K) return nb;
  const unsigned long long n = job->nops - job->first_op;
  const unsigned long long target = job->first_op + (n * k) / K;
  uint32_t lo = 0, hi = nb;  // the first batch starting at or after target
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (job->offsets[mid] < target) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// (calls of several windows only) The window's part of each class: its first
// and last position by bisection, one lane each.
__global__ void batch_window_begin_kernel(batch_job* job, uint32_t k) {
  if (blockIdx.x != 0 || threadIdx.x >= 2 * kOpClasses) return;
  if (ld32_coherent(&job->bad)) return;
  const uint32_t q = threadIdx.x >> 1, at_end = threadIdx.x & 1;
  const uint32_t target = (uint32_t)(job->offsets[window_start(job, k + at_end)] - job->first_op);
  const uint32_t* part = job->list + (q > 1 ? job->total[1] : 0u);
  uint32_t lo = 0, hi = job->total[q];  // the first entry of an operation >= target
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if ((q == 0 ? job->writes[mid].rel & 0x7FFFFFFFu : part[mid]) < target) lo = mid + 1;
    else hi = mid;
  }
  const uint32_t other = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((threadIdx.x ^ 1u) << 2), (int)lo);
  if (at_end) return;
  job->first[q] = lo;
  (q == 0 ? job->n_writes : q == 1 ? job->n_finds : job->n_ranges) = other - lo;
}

// End of a window: every read of the call at a snapshot below the next
// window's first batch is done, so - when the call may reclaim (no snapshot
// outside it is live) - every retired copy is garbage: the window's own copies
// hold contents that only those reads could see. Frees them (appending an
// epoch to the memory timeline) and merges parked slots either way.
__global__ void __launch_bounds__(kReclaimBlock)
    batch_window_end_kernel(batch_job* job, tree_state* st, epoch_stat* series, uint32_t* ring,
                            const uint32_t* spill, uint32_t* free_stack) {
  if (ld32_coherent(&job->bad)) return;
  const bool r = job->reclaim != 0;
  reclaim_grid(st, r ? ~0ull : 0ull, r ? series : nullptr, ring, spill, free_stack, {job->w_par, job->n_planned});
}

// How the sorted form's kernels divide n operations, a count only the device
// knows: one to a tile while that leaves tiles idle, then as few as keep
// `tiles` of them busy (as split_for does for the plain launches).
MVBT_DEV uint32_t per_tile(uint32_t n, uint32_t tiles, uint32_t width) {
  const uint32_t p = (n + tiles - 1) / tiles;
  return p < 1 ? 1u : p < width ? p : width;
}

// 7. Routes every write of the window to its leaf: sort key = leaf (cap_ for a
// key that is not routed: reserved keys, which fail in the write pass), payload
// = the write's position in the window; the parent goes to w_par. T: routing tile
// width (T < NW: NW / T pairs per lane, mvbt_wide.hpp).
template <int NW, int T = NW>
__global__ void __launch_bounds__(256) batch_route_kernel(tree_ptrs tp, batch_job* job) {
  if (ld32_coherent(&job->bad)) return;
  const tree_view<NW, true> tv(tp);
  tile<T> t;
  const uint32_t n = job->n_writes;
  chunking<T> c(per_tile(n, gridDim.x * (blockDim.x / T) / 2, T));  // half the grid's tiles are resident
  if (c.block_ops(n) == 0) return;
  __shared__ route_cache<NW, kRangeCacheBytes> rc;
  tv.build_route_cache(rc, c.per >= kCachedFrom ? 0ull : ~0ull);
  const write_rec* writes = job->writes + job->first[0];
  uint32_t* hint = job->sort_k[0];
  uint32_t* pos = job->sort_v[0];
  uint32_t* w_par = job->w_par;
  for (uint64_t base = c.first; base < n; base += c.stride) {
    const uint64_t i = base + t.rank();
    const bool act = c.holds(base, t.rank(), n);
    const uint32_t key = act ? writes[i].key : 0u;
    const bool go = act && valid_key(key);
    const uint64_t q = t.ballot(go);
    uint32_t st0 = kNone, sp0 = kNone, leaf = kNone, par = kNone;
    if (go) st0 = tv.route_lane(rc, key, sp0);
    if constexpr (T < NW)
      descend_chunk_wide<T, false, kWideRouteGroup<NW / T>>(tv, key, q, leaf, par, t, q, st0, sp0);
    else
      tv.template descend_chunk<false>(key, q, leaf, par, t, q, st0, sp0);
    if (act) {
      const bool routed = go && leaf < tv.cap_;
      hint[i] = routed ? leaf : tv.cap_;
      pos[i] = (uint32_t)i;
      w_par[i] = routed ? par : kNone;
    }
  }
}

// 7'. The sorted writes' fields in sorted order, so that the write pass reads
// them with coalesced loads instead of chasing the position and the write one
// dependent load after another, and the copy planning: every (leaf, batch)
// group of the sorted writes may copy its leaf once, so the groups are counted
// here and numbered below (a stable count / scan / assign over the sorted
// list), and one reservation takes a slot for each from the free stack and the
// never-used frontier, and enters them all in the retire ring: the write pass
// then copies into its group's slot without touching the shared allocation and
// retirement counters. A slot its group does not use (no change, or the
// per-key path took over) is simply freed by the next reclamation.
__global__ void __launch_bounds__(kSortBlock) batch_gather_kernel(batch_job* job, uint32_t which) {
  __shared__ uint32_t part[kSortBlock / 64];
  const uint32_t n = ld32_coherent(&job->bad) ? 0u : job->n_writes;
  const uint32_t *hint = job->sort_k[which], *pos = job->sort_v[which];
  const write_rec* writes = job->writes + job->first[0];
  const uint32_t lane = threadIdx.x & 63;
  uint32_t a, e, c = 0;
  segment_of(n, blockIdx.x, gridDim.x, a, e);
  for (uint32_t i0 = a; i0 < e; i0 += kSortBlock) {
    const uint32_t i = i0 + threadIdx.x;
    const bool act = i < e;
    uint32_t b = 0, h = 0;
    if (act) {
      const uint32_t p = pos[i];
      h = hint[i];
      const write_rec r = writes[p];
      b = r.batch;
      job->sorted[i] = r;
      job->sort_k[which ^ 1u][i] = job->w_par[p];
    }
    // the write before this one in sorted order: the lane below, or a load
    uint32_t hb = (uint32_t)__shfl_up((int)h, 1, 64), bb = (uint32_t)__shfl_up((int)b, 1, 64);
    if (act && lane == 0 && i > 0) {
      hb = hint[i - 1];
      bb = writes[pos[i - 1]].batch;
    }
    const bool start = act && (i == 0 || h != hb || b != bb);
    if (act) job->sort_v[which ^ 1u][i] = start ? 1u : 0u;  // read, then replaced, by batch_assign_kernel
    c += start ? 1u : 0u;
  }
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if (lane == 0) part[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tot = 0;
    for (uint32_t w = 0; w < kSortBlock / 64; ++w) tot += part[w];
    job->seg[blockIdx.x] = tot;
  }
}

// Calls that keep their copies until mvbt_reclaim however small they are (mode 3
// below 16384 operations), and all small calls, must not hold more slots than
// they make copies: there a group's slot is only lent to the call. sort_v holds
// each write's slot in one buffer and its group in the other, w_par each group's
// slot; the write pass sets kSlotUsed there when a copy lies in it, and the end
// of the window (settle_planned) retires those slots and gives the others back.
// Until then the call holds a slot per group, so none is planned where its
// writes could run short of slots for that: a write may take a copy, a new leaf,
// a new node on each level above, and its tile as many again before it uses
// them. The write pass then takes slots only for the copies it makes, a few at a
// time, as a batch-by-batch call would.
constexpr unsigned long long kPlanRoom = 16;  // free slots a write of the window, plus kPlanRoomBase
constexpr unsigned long long kPlanRoomBase = 256;
MVBT_DEV bool lend_slots(const tree_ptrs& tp, uint32_t writes) {
  const long long on_stack = (long long)ld_coherent((const uint64_t*)&tp.st->free_top);
  const unsigned long long bump = ld_coherent((const uint64_t*)&tp.st->bump);
  const unsigned long long fresh = bump < tp.cap_ ? tp.cap_ - bump : 0ull;
  return fresh + (on_stack > 0 ? (unsigned long long)on_stack : 0ull) >= kPlanRoom * writes + kPlanRoomBase;
}

// One workgroup: seg to each segment's first group number; its last thread,
// which holds the number of groups, reserves a slot for each (free stack first,
// then the frontier) and, unless they are lent, as many retire-ring positions as
// slots exist.
__global__ void __launch_bounds__(kSortBlock)
    batch_copy_reserve_kernel(batch_job* job, tree_ptrs tp, uint32_t segments) {
  __shared__ scan_lds l;
  if (ld32_coherent(&job->bad)) return;
  const uint32_t groups = scan_row(job->seg, segments, l);
  if (threadIdx.x != kSortBlock - 1) return;
  const bool lend = job->lend != 0;
  const uint32_t E = !lend || lend_slots(tp, job->n_writes) ? groups : 0u;
  job->n_planned = lend ? E : 0u;
  tree_state* st = tp.st;
  long long top = atomic_add_s64(&st->free_top, -(long long)E);
  const uint32_t got = (uint32_t)(top < 0 ? 0 : (top > (long long)E ? (long long)E : top));
  unsigned long long b = 0;
  if (got < E) b = atomic_add64(&st->bump, (unsigned long long)(E - got));
  const unsigned long long fresh = b < (unsigned long long)tp.cap_ ? (unsigned long long)tp.cap_ - b : 0ull;
  const uint32_t valid = got + (uint32_t)((unsigned long long)(E - got) < fresh ? (E - got) : fresh);
  if (valid < E) atomic_or32(&st->error_flags, kErrPoolExhausted);
  const unsigned long long ring = lend ? 0ull : atomic_add64(&st->retire_tail, (unsigned long long)valid);
  job->cp_top = top;
  job->cp_got = got;
  job->cp_bump = b;
  job->cp_valid = valid;
  job->cp_ring = ring;
}

// The slot of every sorted write's group (kNone past the pool); the existing
// ones go to the retire ring (lent ones to w_par), each by its group's first
// write.
__global__ void __launch_bounds__(kSortBlock) batch_assign_kernel(batch_job* job, tree_ptrs tp, uint32_t which) {
  constexpr uint32_t kWaves = kSortBlock / 64;
  __shared__ uint32_t wsum[kWaves];
  if (ld32_coherent(&job->bad)) return;
  const uint32_t n = job->n_writes, got = job->cp_got, valid = job->cp_valid;
  const long long top = job->cp_top;
  const unsigned long long bump = job->cp_bump, ring = job->cp_ring, mask = tp.retire_cap - 1;
  uint32_t* slots = job->sort_v[which ^ 1u];
  const bool lent = job->n_planned != 0;
  const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint64_t below = (1ull << lane) - 1;
  uint32_t a, e;
  segment_of(n, blockIdx.x, gridDim.x, a, e);
  uint32_t run = job->seg[blockIdx.x];  // groups started before this segment
  for (uint32_t c = a; c < e; c += kSortBlock) {
    const uint32_t i = c + tid;
    const bool act = i < e;
    const bool start = act && slots[i] != 0;
    const uint64_t m = __builtin_amdgcn_ballot_w64(start);
    if (lane == 0) wsum[w] = (uint32_t)__builtin_popcountll(m);
    __syncthreads();
    uint32_t before = run + (uint32_t)__builtin_popcountll(m & below), tot = 0;
#pragma unroll
    for (uint32_t v = 0; v < kWaves; ++v) {
      if (v < w) before += wsum[v];
      tot += wsum[v];
    }
    if (act) {
      const uint32_t k = before + (start ? 1u : 0u) - 1u;  // the write's group: starts at or before it, minus one
      uint32_t slot = kNone;
      if (k < got) slot = ld32_coherent(tp.free_stack + (top - 1 - (long long)k));
      else if (k < valid) slot = (uint32_t)(bump + (k - got));
      slots[i] = slot;
      if (lent) {
        job->sort_v[which][i] = k;
        if (start) job->w_par[k] = slot;
      } else if (start && k < valid) {
        tp.retire_ring[(ring + k) & mask] = slot;
      }
    }
    run += tot;
    __syncthreads();
  }
}

// ---- small calls of the sorted form ----------------------------------------
// A call of at most kSmallOps operations in at most kSmallBatches batches: a
// launch costs 4-5 us whatever it does, and the launches above, 13 and 3 more a
// radix pass, are most of such a call (3 batches of 3000 operations: no less than
// the 146 us of the batch-after-batch worker). One workgroup therefore does the
// checks and the split, and after the routing one workgroup sorts the writes in
// LDS and plans their copies: the call is 7 launches (89 us), besides the
// maintenance launch that a call after another write begins with.
constexpr uint32_t kSmallOps = 16384, kSmallBatches = 4096, kSmallBlock = 1024;

// Exclusive prefix of `v` over the workgroup's threads; *total: its sum. `w`:
// kSmallBlock / 64 words of LDS.
MVBT_DEV uint32_t block_prefix(uint32_t v, uint32_t* w, uint32_t* total) {
  constexpr uint32_t kWaves = kSmallBlock / 64;
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t incl = v;
#pragma unroll
  for (uint32_t d = 1; d < 64; d <<= 1) {
    const uint32_t up = (uint32_t)__shfl_up((int)incl, (int)d, 64);
    if (lane >= d) incl += up;
  }
  if (lane == 63) w[wave] = incl;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (uint32_t k = 0; k < kWaves; ++k) {
    if (k < wave) before += w[k];
    all += w[k];
  }
  __syncthreads();
  *total = all;
  return before + incl - v;
}

// S1. Setup, batches, checks and split of a small call, by one workgroup.
__global__ void __launch_bounds__(kSmallBlock) batch_small_begin_kernel(batch_job* job, tree_state* st, batch_params p) {
  constexpr uint32_t kWaves = kSmallBlock / 64;
  __shared__ uint32_t table[2 * kSmallOps];
  __shared__ uint32_t off[kSmallBatches + 1];
  __shared__ uint32_t wsum[kOpClasses][kWaves];
  // Two words: every wave reads the first one below, while others that are ahead
  // of it may already set the second.
  __shared__ uint32_t bad_offsets, bad;
  const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nb = p.nb, n = (uint32_t)p.nops;
  const unsigned long long first = p.offsets[0];
  if (tid == 0) {
    bad_offsets = p.offsets[nb] - first == p.nops ? 0u : 1u;  // (last < first differs as well)
    bad = 0;
  }
  __syncthreads();
  for (uint32_t b = tid; b <= nb; b += kSmallBlock) {
    const unsigned long long o = p.offsets[b] - first;
    if (o > n || (b > 0 && p.offsets[b] < p.offsets[b - 1])) bad_offsets = 1;
    off[b] = (uint32_t)o;
  }
  __syncthreads();
  const bool ordered = bad_offsets == 0;
  uint32_t run[kOpClasses] = {0, 0, 0};
  const op_record* ops = p.ops + first;
  const uint64_t below = (1ull << lane) - 1;
  // finds and ranges share `list`: the ranges go in behind n - 1 downwards and are turned round below
  for (uint32_t i0 = 0; ordered && i0 < n; i0 += kSmallBlock) {
    const uint32_t i = i0 + tid;
    op_record o{};
    uint32_t k = kOpClasses, b = 0;
    if (i < n) {
      o = ops[i];
      uint32_t hi = nb;
      while (hi - b > 1) {  // off[b] <= i < off[hi]
        const uint32_t mid = (b + hi) >> 1;
        if (off[mid] <= i) b = mid;
        else hi = mid;
      }
      job->op_batch[i] = b;
      k = op_class(o.type);
      if (k == kOpClasses) bad = 1;
    }
    uint64_t m[kOpClasses];
#pragma unroll
    for (uint32_t q = 0; q < kOpClasses; ++q) {
      m[q] = __builtin_amdgcn_ballot_w64(k == q);
      if (lane == 0) wsum[q][w] = (uint32_t)__builtin_popcountll(m[q]);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < kOpClasses; ++q) {
      uint32_t pos = run[q] + (uint32_t)__builtin_popcountll(m[q] & below), tot = 0;
#pragma unroll
      for (uint32_t v = 0; v < kWaves; ++v) {
        if (v < w) pos += wsum[q][v];
        tot += wsum[q][v];
      }
      if (k == q) {
        if (q == 0) job->writes[pos] = write_rec{o.key, o.arg, i | (o.type == kOpErase ? 0x80000000u : 0u), b};
        else job->list[q == 1 ? pos : n - 1 - pos] = i;
      }
      run[q] += tot;
    }
    __syncthreads();
  }
  // distinct write keys per batch (as batch_claim_kernel, with the table in LDS)
  uint32_t mask = 1023;
  while (mask + 1 < 2 * run[0]) mask = 2 * mask + 1;
  for (uint32_t i = tid; i <= mask; i += kSmallBlock) table[i] = 0;
  __syncthreads();
  for (uint32_t i = tid; i < run[0]; i += kSmallBlock) {
    const write_rec r = job->writes[i];
    if (!valid_key(r.key)) continue;
    uint32_t h = conflict_hash(r.key, r.batch) & mask;
    for (uint32_t probe = 0; probe <= mask; ++probe) {
      const uint32_t cur = atomicCAS(&table[h], 0u, i + 1);
      if (cur == 0) break;
      if (job->writes[cur - 1].key == r.key && job->writes[cur - 1].batch == r.batch) {
        bad = 1;
        break;
      }
      h = (h + 1) & mask;
    }
  }
  // the ranges, turned round, behind the finds (each pair of entries by one thread)
  __syncthreads();
  const uint32_t nf = run[1], nr = run[2];
  uint32_t mine[(kSmallOps + kSmallBlock - 1) / kSmallBlock];
#pragma unroll
  for (uint32_t j = 0; j < (kSmallOps + kSmallBlock - 1) / kSmallBlock; ++j) {
    const uint32_t r = tid + j * kSmallBlock;
    if (r < nr) mine[j] = job->list[n - 1 - r];
  }
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < (kSmallOps + kSmallBlock - 1) / kSmallBlock; ++j) {
    const uint32_t r = tid + j * kSmallBlock;
    if (r < nr) job->list[nf + r] = mine[j];
  }
  if (tid == 0) {
    const uint32_t clock0 = __hip_atomic_fetch_add(&st->clock, nb, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
    if (p.base_out) *p.base_out = clock0;
    job->ops = p.ops;
    job->offsets = p.offsets;
    job->nb = nb;
    job->L = p.L;
    job->results = p.results;
    job->pairs = p.pairs;
    job->pair_slots = p.pair_slots;
    job->clock0 = clock0;
    job->first_op = first;
    job->nops = ordered ? first + n : first;
    job->bad = bad | bad_offsets;
    job->windows = 1;
    job->n_planned = 0;
    job->lend = 1;
    job->reclaim = p.reclaim;
    for (uint32_t q = 0; q < kOpClasses; ++q) {
      job->first[q] = 0;
      job->total[q] = run[q];
    }
    job->n_writes = run[0];
    job->n_finds = nf;
    job->n_ranges = nr;
    if (bad | bad_offsets) atomic_or32(&st->error_flags, kErrBadBatch);
  }
}

// S2. Sort by leaf, gather and copy planning of a small call's writes, by one
// workgroup: an 8-bit radix pass for every eight bits of the pool's size (three
// below 2^24 nodes) with leaf and position in LDS, each wave ranking its own
// stretch; then the gather
// and the groups as in batch_gather_kernel. The sorted leaf hints end in
// sort_k[1], as after an odd number of passes.
__global__ void __launch_bounds__(kSmallBlock) batch_small_plan_kernel(batch_job* job, tree_ptrs tp, uint32_t bits) {
  constexpr uint32_t kWaves = kSmallBlock / 64, kItems = kSmallOps / kSmallBlock;
  __shared__ uint32_t key[kSmallOps];
  __shared__ uint16_t pos[kSmallOps];
  __shared__ uint16_t bat[kSmallOps];
  __shared__ uint32_t cnt[kWaves][kRadix];
  __shared__ uint32_t wsum[kWaves];
  __shared__ long long s_top;
  __shared__ unsigned long long s_bump;
  __shared__ uint32_t s_got, s_planned;
  if (ld32_coherent(&job->bad)) return;
  const uint32_t n = job->n_writes;
  if (n == 0) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const uint64_t below = (1ull << lane) - 1;
  const write_rec* writes = job->writes;
  for (uint32_t i = tid; i < n; i += kSmallBlock) {
    key[i] = job->sort_k[0][i];
    pos[i] = (uint16_t)i;
  }
  __syncthreads();
  // wave w ranks items [w * S, (w + 1) * S), 64 at a time
  const uint32_t S = ((n + kWaves - 1) / kWaves + 63) / 64 * 64, a = w * S;
  for (uint32_t shift = 0; shift < bits; shift += 8) {
    volatile uint32_t* my = cnt[w];  // this wave's alone until the barrier; its LDS operations run in order
    for (uint32_t d = lane; d < kRadix; d += 64) my[d] = 0;
    uint32_t k[kItems], v[kItems], rank[kItems];
#pragma unroll
    for (uint32_t j = 0; j < kItems; ++j) {
      const uint32_t i = a + j * 64 + lane;
      const bool act = j * 64 < S && i < n;
      if (__builtin_amdgcn_ballot_w64(act) == 0) continue;
      k[j] = act ? key[i] : 0u;
      v[j] = act ? pos[i] : 0u;
      const uint32_t d = (k[j] >> shift) & (kRadix - 1);
      uint64_t same = __builtin_amdgcn_ballot_w64(act);
#pragma unroll
      for (uint32_t bit = 0; bit < 8; ++bit) {
        const uint64_t ones = __builtin_amdgcn_ballot_w64(((d >> bit) & 1u) != 0);
        same &= ((d >> bit) & 1u) ? ones : ~ones;
      }
      const uint32_t before = my[d];  // this wave's earlier items with the digit
      rank[j] = before + (uint32_t)__builtin_popcountll(same & below);
      if (act && (same & below) == 0) my[d] = before + (uint32_t)__builtin_popcountll(same);
    }
    __syncthreads();
    {  // exclusive prefix over (digit, wave): thread t holds waves 4 (t & 3) .. of digit t / 4
      const uint32_t d = tid >> 2, w0 = (tid & 3) * (kWaves / 4);
      uint32_t c[kWaves / 4], s = 0, total;
#pragma unroll
      for (uint32_t q = 0; q < kWaves / 4; ++q) {
        c[q] = cnt[w0 + q][d];
        s += c[q];
      }
      uint32_t r = block_prefix(s, wsum, &total);
#pragma unroll
      for (uint32_t q = 0; q < kWaves / 4; ++q) {
        cnt[w0 + q][d] = r;
        r += c[q];
      }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kItems; ++j) {
      const uint32_t i = a + j * 64 + lane;
      if (j * 64 < S && i < n) {
        const uint32_t to = cnt[w][(k[j] >> shift) & (kRadix - 1)] + rank[j];
        key[to] = k[j];
        pos[to] = (uint16_t)v[j];
      }
    }
    __syncthreads();
  }
  // sorted position i: the write's record and parent, and its batch
  for (uint32_t i = tid; i < n; i += kSmallBlock) {
    const write_rec r = writes[pos[i]];
    job->sorted[i] = r;
    bat[i] = (uint16_t)r.batch;
    job->sort_k[1][i] = key[i];
    job->sort_k[0][i] = job->w_par[pos[i]];
  }
  __syncthreads();
  // groups started at or before each position; the slots are reserved in between
  uint32_t group[kItems], run = 0;
  bool start[kItems];
#pragma unroll
  for (uint32_t j = 0; j < kItems; ++j) {
    if (j * kSmallBlock >= n) continue;
    const uint32_t i = j * kSmallBlock + tid;
    start[j] = i < n && (i == 0 || key[i] != key[i - 1] || bat[i] != bat[i - 1]);
    uint32_t total;
    group[j] = run + block_prefix(start[j] ? 1u : 0u, wsum, &total) + (start[j] ? 1u : 0u) - 1u;
    run += total;
  }
  if (tid == 0) {
    tree_state* st = tp.st;
    s_got = 0;
    s_planned = lend_slots(tp, n) ? run : 0u;
    if (s_planned) {  // (no other writer runs beside the call: what was left is still there)
      const long long top = atomic_add_s64(&st->free_top, -(long long)run);
      const uint32_t got = (uint32_t)(top < 0 ? 0 : (top > (long long)run ? (long long)run : top));
      s_top = top;
      s_got = got;
      if (got < run) s_bump = atomic_add64(&st->bump, (unsigned long long)(run - got));
    }
    job->n_planned = s_planned;
  }
  __syncthreads();
  const bool planned = s_planned != 0;
#pragma unroll
  for (uint32_t j = 0; j < kItems; ++j) {
    const uint32_t i = j * kSmallBlock + tid;
    if (i >= n) continue;
    uint32_t slot = kNone;
    if (planned) {
      slot = group[j] < s_got ? ld32_coherent(tp.free_stack + (s_top - 1 - (long long)group[j]))
                              : (uint32_t)(s_bump + (group[j] - s_got));
      job->sort_v[1][i] = group[j];
      if (start[j]) job->w_par[group[j]] = slot;
    }
    job->sort_v[0][i] = slot;
  }
}

// 8. The write pass over the sorted writes (buffers sort_k/v[which]). LEND: slots
// are lent to the call (lend_slots), and leaves are locked, for latest reads on
// other streams: such calls once ran on the persistent worker, which locks them.
// It is 1% of a small call's time and 4.6% of 4M operations' (1273 -> 1332 us),
// whose leaves were never locked: mvbt_run_batches forbids such reads beside them.
template <int NW, bool LEND>
MVBT_DEV void sorted_writes(const tree_ptrs& tp, batch_job* job, uint32_t which) {
  const tree_view<NW, true> tv(tp);
  tile<NW> t;
  const uint32_t r = t.rank();
  const uint32_t n = job->n_writes;
  const chunking<NW> c(per_tile(n, gridDim.x * (blockDim.x / NW), NW));
  const uint32_t* hint = job->sort_k[which];
  const write_rec* recs = job->sorted;
  const uint32_t *pars = job->sort_k[which ^ 1u], *slots = job->sort_v[which ^ 1u];
  uint32_t* results = job->results + job->first_op;
  const uint32_t clock0 = job->clock0;
  const bool lent = LEND && job->n_planned != 0;  // slots that a copy takes are marked
  write_ctx ctx = tv.begin_writes(t);
  ctx.exact = !LEND || lent;  // else few slots are left
  ctx.track = 0;  // stamps are fixed per batch: clock0 + b + 1
  for (uint64_t p = c.first; p < n; p += c.stride) {
    uint64_t i = p + r;
    bool start = c.holds(p, r, n) && (i == 0 || hint[i] != hint[i - 1]);
    const uint64_t starts = t.ballot(start);
    if (!starts) continue;  // the window lies inside a group that started earlier
    // sub-windows of NW positions from the first group start in the window (of c.per positions) to
    // the first group start at or past its end
    const uint64_t wend = p + c.per;
    for (uint64_t a = p + (uint64_t)lowest_bit(starts);; a += NW) {
      i = a + r;
      const bool in = i < n;
      const uint32_t h = in ? hint[i] : kNone;
      start = in && (i == 0 || h != hint[i - 1]);
      uint64_t mine = t.ballot(in);
      const uint64_t foreign = t.ballot(start && i >= wend);
      bool last = a + NW >= n;
      if (foreign) {
        mine &= (1ull << lowest_bit(foreign)) - 1;
        last = true;
      }
      if (!mine) break;
      const bool act = (mine >> r) & 1;
      op_record op{};
      uint32_t rel = 0, b = 0, par = kNone, planned = kNone;
      if (act) {
        const write_rec w = recs[i];
        op.key = w.key;
        op.arg = w.arg;
        rel = w.rel & 0x7FFFFFFFu;
        op.type = (w.rel >> 31) ? kOpErase : kOpInsert;
        b = w.batch;
        par = pars[i];
        planned = slots[i];
      }
      const uint32_t cur = clock0 + b + 1;
      const uint32_t leaf = (act && h < tv.cap_) ? h : kNone;
      // lane r's group begins at glead (lane 0 or a group start of this sub-window)
      const uint64_t gs = t.ballot(start) | 1ull;
      const uint64_t upto = (r == 63) ? ~0ull : ((2ull << r) - 1);
      const uint64_t from_lead = ~((1ull << highest_bit(gs & upto)) - 1);
      uint32_t res = 0;
      // rounds: every group writes its earliest remaining batch (a group's
      // lanes are in batch order, so that is its lowest remaining lane's)
      for (uint64_t R = mine; R;) {
        const uint64_t ahead = R & from_lead;
        const uint32_t front = ahead ? (uint32_t)lowest_bit(ahead) : r;
        const uint32_t fb = t.shfl(b, front);
        const bool sel = ((R >> r) & 1) && b == fb;
        const uint64_t S = t.ballot(sel);
        for (int w = 0; w < 2; ++w) {
          uint64_t q = t.ballot(sel && op.type == (w == 0 ? kOpInsert : kOpErase));
          if (!q) continue;
          ctx.want = (uint32_t)__builtin_popcountll(q);
          q = (w == 0) ? tv.template write_chunk_at<0, true, LEND>(op.key, op.arg, q, leaf, cur, res, ctx, t, planned)
                       : tv.template write_chunk_at<1, true, LEND>(op.key, 0u, q, leaf, cur, res, ctx, t, planned);
          while (q) {
            const uint32_t j = (uint32_t)lowest_bit(q);
            ctx.want = (uint32_t)__builtin_popcountll(q);
            q &= q - 1;
            ctx.cur = t.shfl(cur, j);
            const uint32_t k = t.shfl(op.key, j), lf = t.shfl(leaf, j), pr = t.shfl(par, j);
            const uint32_t v = (w == 0) ? tv.template write<0>(k, t.shfl(op.arg, j), ctx, t, lf, pr)
                                        : tv.template write<1>(k, 0u, ctx, t, lf, pr);
            if (r == j) res = v;
          }
        }
        R &= ~S;
      }
      if (act) results[rel] = res;
      if (lent && planned == kTaken) job->w_par[job->sort_v[which][i]] = slots[i] | kSlotUsed;
      if (last) break;
    }
  }
  tv.finish(ctx, t);
}
template <int NW>
__global__ void __launch_bounds__(256) batch_sorted_write_kernel(tree_ptrs tp, batch_job* job, uint32_t which) {
  if (ld32_coherent(&job->bad)) return;
  if (job->lend) sorted_writes<NW, true>(tp, job, which);
  else sorted_writes<NW, false>(tp, job, which);
}

// 9. Finds, each at its batch's snapshot (no writer runs). T: read tile
// width (T < NW: P = NW / T pairs per lane, mvbt_wide.hpp).
template <int NW, int T = NW>
__global__ void __launch_bounds__(kFindBlock) __attribute__((amdgpu_waves_per_eu(8)))
batch_sorted_find_kernel(tree_ptrs tp, const batch_job* job) {
  if (ld32_coherent(&job->bad)) return;
  const tree_view<NW, true> tv(tp);
  tile<T> t;
  const uint32_t n = job->n_finds;
  chunking<T> c(per_tile(n, gridDim.x * (blockDim.x / T), T));
  if (c.block_ops(n) == 0) return;
  __shared__ route_cache<NW, kFindCacheBytes> rc;
  tv.build_route_cache(rc, c.per >= kCachedFrom ? 0ull : ~0ull);
  const uint32_t* list = job->list + job->first[1];
  const uint32_t* op_batch = job->op_batch;
  const op_record* ops = job->ops + job->first_op;
  uint32_t* results = job->results + job->first_op;
  const uint32_t clock0 = job->clock0;
  for (uint64_t base = c.first; base < n; base += c.stride) {
    const uint64_t i = base + t.rank();
    const bool act = c.holds(base, t.rank(), n);
    const uint32_t rel = act ? list[i] : 0u;
    const uint32_t key = act ? ops[rel].key : 0u;
    const uint32_t ts = act ? clock0 + op_batch[rel] : 0u;
    uint32_t result = kEmpty;
    if constexpr (T == 16) {
      const bool go = act && valid_key(key);
      uint32_t start = tv.root_, unused;
      if (go) start = tv.route_lane(rc, key, unused);
      result = find_rows(tv, key, ts, start, (uint32_t)t.ballot(go), c.per);
    } else if constexpr (T < NW) {
      result = read_chunk_wide<T, false, true, kWideFindGroup<NW / T>>(tv, key, 0u, ts, nullptr, 0u, t.ballot(act), t,
                                                                        &rc);
    } else if constexpr (NW >= 32) {
      // as in find_kernel: the pass-based engine keeps more walks in flight
      result = tv.template read_chunk<false, route_cache<NW, kFindCacheBytes>, true, tree_view<NW, true>::kFindGroup>(
          key, 0u, ts, nullptr, 0u, t.ballot(act), t, &rc);
    }
    if (act) results[rel] = result;
  }
}

// 10. Ranges, each at its batch's snapshot: the pass-based reader with a
// snapshot and an output slot per lane (T: read tile width, as above).
template <int NW, int T = NW>
__global__ void __launch_bounds__(256) batch_sorted_range_kernel(tree_ptrs tp, const batch_job* job) {
  if (ld32_coherent(&job->bad)) return;
  using rc_t = route_cache<NW, kRangeCacheBytes>;
  const tree_view<NW, true> tv(tp);
  tile<T> t;
  const uint32_t n = job->n_ranges, L = job->L;
  chunking<T> c(per_tile(n, gridDim.x * (blockDim.x / T) / 2, T));  // half the grid's tiles are resident
  if (c.block_ops(n) == 0) return;
  __shared__ rc_t rc;
  tv.build_route_cache(rc, c.per >= kCachedFrom ? 0ull : ~0ull);
  const uint32_t* list = job->list + job->total[1] + job->first[2];
  const uint32_t* op_batch = job->op_batch;
  const op_record* ops = job->ops + job->first_op;
  uint32_t* results = job->results + job->first_op;
  uint64_t* pairs = job->pairs;
  const unsigned long long pair_slots = job->pair_slots;
  const uint32_t clock0 = job->clock0;
  bool overflow = false, bad_slot = false;
  for (uint64_t base = c.first; base < n; base += c.stride) {
    const uint64_t i = base + t.rank();
    const bool act = c.holds(base, t.rank(), n);
    const uint32_t rel = act ? list[i] : 0u;
    op_record op{};
    if (act) op = ops[rel];
    const uint32_t ts = act ? clock0 + op_batch[rel] : 0u;
    uint64_t* out = nullptr;
    if (act && pairs) {
      if (op.slot < pair_slots) out = pairs + (size_t)op.slot * L;
      else bad_slot = true;
    }
    const uint32_t k0 = op.key == 0 ? 1u : op.key;
    uint32_t cnt;
    if constexpr (T == 16) {
      const bool go = act && valid_key(k0) && op.arg > k0;
      uint32_t start = tv.root_, unused;
      if (go) start = tv.route_lane(rc, k0, unused);
      cnt = range_rows(tv, k0, op.arg, ts, start, out, L, (uint32_t)t.ballot(go));
    } else if constexpr (T < NW) {
      cnt = read_chunk_wide<T, true, true, kWideRangeGroup<NW / T>>(tv, k0, op.arg, ts, out, L, t.ballot(act), t, &rc);
    } else {
      cnt = tv.template read_chunk<true, rc_t, true>(k0, op.arg, ts, out, L, t.ballot(act), t, &rc);
    }
    if (act) results[rel] = cnt;
    overflow |= act && cnt > L;
  }
  const uint32_t err = (t.any(overflow) ? kErrRangeOverflow : 0u) | (t.any(bad_slot) ? kErrCorrupt : 0u);
  if (err && t.leader()) atomic_or32(&tv.st->error_flags, err);
}

}  // namespace mvbt
