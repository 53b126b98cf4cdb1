// Stable LSD radix sort of 32-bit keys with 32-bit payloads, for the sorted
// batched form (mvbt_batch.hpp): it groups a call's writes by the leaf they
// route to while keeping operation order inside each group.
//
// The element count is read from device memory (`n`), so the kernels can sit
// in a graph whose parameters never change while the count does. Every pass
// splits the input into gridDim.x contiguous segments, one per workgroup:
//   1. radix_hist_kernel    per-segment histogram of one 8-bit digit
//                           (hist[digit * G + segment]);
//   2. radix_scan_kernel    one workgroup per digit: exclusive scan of its G
//                           segment counts in place, and the digit's total;
//   3. radix_scatter_kernel each segment writes its elements, in input
//                           order, at digit base + earlier segments' count +
//                           rank inside the segment (stable).
// Passes alternate between two buffer pairs. Memory traffic per pass is one
// read of the keys (histogram) and one read plus one scattered write of
// keys and payloads (scatter): 20 bytes per element.
#pragma once
#include "mvbt_common.hpp"

namespace mvbt {

constexpr uint32_t kSortSegments = 512;  // workgroups (segments) per pass
constexpr uint32_t kSortBlock = 256;     // threads per workgroup
constexpr uint32_t kRadix = 256;         // 8-bit digits
constexpr uint32_t kSortEach = 8;        // elements of a thread in flight
// Sorts take fewer elements than this: the division below and the indices of the
// passes' loops, which run up to a chunk past a segment's end, are 32-bit.
constexpr uint64_t kSortMax = 1ull << 31;

MVBT_HD void segment_of(uint32_t n, uint32_t g, uint32_t G, uint32_t& a, uint32_t& b) {
  const uint32_t seg = (n + G - 1) / G;
  const uint64_t lo = (uint64_t)g * seg;
  a = lo < n ? (uint32_t)lo : n;
  b = (uint64_t)a + seg < n ? a + seg : n;
}

__global__ void set_word_kernel(uint32_t* p, uint32_t v) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *p = v;
}

__global__ void __launch_bounds__(kSortBlock)
    radix_hist_kernel(const uint32_t* keys, const uint32_t* n_ptr, uint32_t shift, uint32_t* hist) {
  __shared__ uint32_t h[kRadix];
  const uint32_t tid = threadIdx.x;
  h[tid] = 0;
  __syncthreads();
  uint32_t a, b;
  segment_of(*n_ptr, blockIdx.x, gridDim.x, a, b);
  for (uint32_t i = a + tid; i < b; i += kSortEach * kSortBlock) {
    uint32_t k[kSortEach];  // all loaded before the first is counted
#pragma unroll
    for (uint32_t j = 0; j < kSortEach; ++j)
      if (i + j * kSortBlock < b) k[j] = keys[i + j * kSortBlock];
#pragma unroll
    for (uint32_t j = 0; j < kSortEach; ++j)
      if (i + j * kSortBlock < b) atomicAdd(&h[(k[j] >> shift) & (kRadix - 1)], 1u);
  }
  __syncthreads();
  hist[tid * gridDim.x + blockIdx.x] = h[tid];
}

// Exclusive scan of a row of at most kScanMax in place by one workgroup, read
// and written coalesced through LDS (one word of padding a bank row); returns
// the row's total on its last thread.
constexpr uint32_t kScanMax = 4096;
struct scan_lds {
  uint32_t part[kSortBlock];
  uint32_t row[kScanMax + kScanMax / 32];
};
MVBT_DEV uint32_t scan_row(uint32_t* row, uint32_t n, scan_lds& l) {
  const uint32_t tid = threadIdx.x;
  for (uint32_t i = tid; i < n; i += kSortBlock) l.row[i + i / 32] = row[i];
  __syncthreads();
  const uint32_t per = (n + kSortBlock - 1) / kSortBlock;
  const uint32_t a = tid * per, b = a + per < n ? a + per : n;
  uint32_t s = 0;
  for (uint32_t i = a; i < b; ++i) s += l.row[i + i / 32];
  l.part[tid] = s;
  __syncthreads();
  for (uint32_t off = 1; off < kSortBlock; off <<= 1) {  // inclusive scan (Hillis-Steele)
    const uint32_t v = tid >= off ? l.part[tid - off] : 0u;
    __syncthreads();
    l.part[tid] += v;
    __syncthreads();
  }
  uint32_t run = l.part[tid] - s;  // exclusive
  for (uint32_t i = a; i < b; ++i) {
    const uint32_t c = l.row[i + i / 32];
    l.row[i + i / 32] = run;
    run += c;
  }
  __syncthreads();
  for (uint32_t i = tid; i < n; i += kSortBlock) row[i] = l.row[i + i / 32];
  return l.part[tid];
}

// One workgroup per digit (gridDim.x = 256), G = `segments` counts each.
__global__ void __launch_bounds__(kSortBlock)
    radix_scan_kernel(uint32_t* hist, uint32_t segments, uint32_t* totals) {
  __shared__ scan_lds l;
  const uint32_t total = scan_row(hist + (size_t)blockIdx.x * segments, segments, l);
  if (threadIdx.x == kSortBlock - 1) totals[blockIdx.x] = total;
}

// Exclusive scan over the workgroup's kRadix threads; wsum: a word a wave, free
// again after the caller's next barrier.
MVBT_DEV uint32_t scan_digits(uint32_t mine, uint32_t* wsum) {
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t incl = mine;
#pragma unroll
  for (uint32_t off = 1; off < 64; off <<= 1) {
    const uint32_t v = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((lane - off) << 2), (int)incl);
    incl += lane >= off ? v : 0u;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  uint32_t s = incl - mine;
  for (uint32_t v = 0; v < w; ++v) s += wsum[v];
  return s;
}

// What bounds it is the number of lines its stores touch: written from the lane
// that read it, each element's key and value went to lines of their own, and 1M
// pairs took 20.3 us (0.8 TB/s) on MI355X, 17.4 with several elements of a
// thread in flight. So a chunk of kSortEach elements a thread is first put in
// digit order in LDS, and neighbouring lanes store the runs of a digit: 11.4 us
// (1.4 TB/s; chunks of half the size 12.9). 26K pairs, a chunk of one element a
// thread: 4.8 us either way.
__global__ void __launch_bounds__(kSortBlock)
    radix_scatter_kernel(const uint32_t* kin, const uint32_t* vin, uint32_t* kout, uint32_t* vout,
                         const uint32_t* n_ptr, uint32_t shift, const uint32_t* hist, const uint32_t* totals) {
  constexpr uint32_t kWaves = kSortBlock / 64, kChunk = kSortEach * kSortBlock;
  __shared__ uint32_t wcnt[kWaves][kRadix];  // a wave's elements of each digit, then where they start in the chunk
  __shared__ uint32_t to[kRadix];            // output position of a digit's run less its start in the chunk
  __shared__ uint32_t wsum[2][kWaves];
  __shared__ uint64_t sorted[kChunk];        // the chunk's pairs in digit order
  const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, G = gridDim.x;
  uint32_t a, b;
  segment_of(*n_ptr, blockIdx.x, G, a, b);
  if (a >= b) return;  // (the same for the whole workgroup)
  // digit tid's base: the digits before it, plus its elements in earlier segments
  const uint32_t earlier = hist[tid * G + blockIdx.x];
  uint32_t base = scan_digits(totals[tid], wsum[0]) + earlier;
  const uint64_t below = (1ull << lane) - 1;
  for (uint32_t c = a; c < b; c += kChunk) {
    const uint32_t m = b - c < kChunk ? b - c : kChunk;  // elements of this chunk
    uint32_t k[kSortEach], v[kSortEach], rank[kSortEach];
    const uint32_t each = (m + kSortBlock - 1) / kSortBlock;  // elements a thread of this chunk
    const uint32_t i0 = w * (each * 64) + lane;               // a wave's share is contiguous
#pragma unroll
    for (uint32_t j = 0; j < kSortEach; ++j) {
      if (j < each && i0 + j * 64 < m) {
        k[j] = kin[c + i0 + j * 64];
        v[j] = vin[c + i0 + j * 64];
      }
    }
#pragma unroll
    for (uint32_t x = 0; x < kWaves; ++x) wcnt[x][tid] = 0;
    __syncthreads();
    // rank of each element among its wave's of the same digit
#pragma unroll
    for (uint32_t j = 0; j < kSortEach; ++j) {
      if (j >= each) break;
      const bool act = i0 + j * 64 < m;
      const uint32_t d = act ? (k[j] >> shift) & (kRadix - 1) : 0u;
      uint64_t same = __builtin_amdgcn_ballot_w64(act);  // lanes of this wave holding the same digit
#pragma unroll
      for (uint32_t bit = 0; bit < 8; ++bit) {
        const uint64_t ones = __builtin_amdgcn_ballot_w64(((d >> bit) & 1u) != 0);
        same &= ((d >> bit) & 1u) ? ones : ~ones;
      }
      const uint32_t r = (uint32_t)__builtin_popcountll(same & below);
      const uint32_t so_far = wcnt[w][d];
      rank[j] = so_far + r;
      __builtin_amdgcn_wave_barrier();  // every lane has read the count before the first lane raises it,
      if (act && r == 0) wcnt[w][d] = so_far + (uint32_t)__builtin_popcountll(same);
      __builtin_amdgcn_wave_barrier();  // and the next element of the wave reads it raised
    }
    __syncthreads();
    // thread d: digit d's run in the chunk, each wave's part of it, and its place in the output
    uint32_t count = 0;
#pragma unroll
    for (uint32_t x = 0; x < kWaves; ++x) count += wcnt[x][tid];
    uint32_t start = scan_digits(count, wsum[1]);
    to[tid] = base - start;
    base += count;
#pragma unroll
    for (uint32_t x = 0; x < kWaves; ++x) {
      const uint32_t part = wcnt[x][tid];
      wcnt[x][tid] = start;
      start += part;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kSortEach; ++j)
      if (j < each && i0 + j * 64 < m) sorted[wcnt[w][(k[j] >> shift) & (kRadix - 1)] + rank[j]] = pack(k[j], v[j]);
    __syncthreads();
    for (uint32_t i = tid; i < m; i += kSortBlock) {
      const uint64_t x = sorted[i];
      const uint32_t pos = to[(lo32(x) >> shift) & (kRadix - 1)] + i;
      kout[pos] = lo32(x);
      vout[pos] = hi32(x);
    }
    // (the next chunk clears wcnt, whose readers the barrier above has seen off;
    // its `sorted` and `to` are written two barriers and more from here)
  }
}

}  // namespace mvbt
