// Reads by 16-lane tiles in launches in which no writer runs: the reader of the
// find and range launches at 16-pair nodes, of the 16-lane read tiles at 32 and
// 64 pairs, and of the sorted batched form's read passes.
//
// What bounds them is the number of vector instructions (on MI355X a 64-lane
// instruction holds its SIMD for four cycles): the pass-based reader that kept
// each walk's state in its own lane (read_chunk_wide) took 69 a node visit, and
// 1M finds at 40M keys kept the vector units busy 96% of their time. So here
//   * a walk's key, node, snapshot and counts are tile-uniform registers: no
//     shuffle fetches or updates them;
//   * a tile is one DPP row, so metadata and version words are broadcast by one
//     row_newbcast each instead of a pair of LDS permutes;
//   * nodes are sorted, so the pairs at or below a key are a prefix of the node:
//     one ballot and a bit count find its end;
//   * the walks of a group go down in step. The tree is quiescent: all leaves
//     are on one level and every node is in its parent, so no walk moves right
//     on its way (a walk that does meet a key at or above its leaf's high key
//     moves right there).
// P = NW / 16 pairs per lane, pair g in lane g / P, slot g % P.
#pragma once
#include "mvbt_tree.hpp"
#include "mvbt_wide.hpp"

namespace mvbt {

// Lane SRC of each 16-lane row to the whole row.
template <uint32_t SRC>
MVBT_DEV uint32_t row_bcast(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 | SRC, 0xf, 0xf, true);
}
// Lane (i + N) % 16 of the row to lane i.
template <uint32_t N>
MVBT_DEV uint32_t row_rotate(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 | (16 - N), 0xf, 0xf, true);
}
// The 16 bits of a wave's ballot that belong to this lane's row.
MVBT_DEV uint32_t row_bits(uint64_t ballot, uint32_t lane) {
  return __builtin_amdgcn_ubfe((lane & 32) ? hi32(ballot) : lo32(ballot), lane & 16, 16);
}

// Calls f(integral constant J) for J = 0 .. N - 1.
template <int J, int N, class F>
MVBT_DEV void each_walk(F&& f) {
  if constexpr (J < N) {
    f(std::integral_constant<int, J>{});
    each_walk<J + 1, N>(f);
  }
}

// Lane j of the tile: key lo (find) or range [lo, hi) with lo >= 1, its snapshot
// ts, its first node (from the route cache, or the root) and, for a range, its
// output (at most cap pairs; null counts only). Returns lane j's value or
// kEmpty, or its true count. Lanes not in `todo` return kEmpty or 0. RG walks of
// the tile are in flight at once.
template <bool RANGE, int RG, int NW, bool VER>
MVBT_DEV uint32_t read_rows(const tree_view<NW, VER>& tv, uint32_t lo, uint32_t hi, uint32_t ts, uint32_t start,
                            uint64_t* out, uint32_t cap, uint32_t todo) {
  using node_t = node<NW, VER>;
  constexpr int P = NW / 16;
  constexpr uint32_t kVerLane = (NW - 2) / P, kVerSlot = (NW - 2) % P;
  static_assert(16 % RG == 0, "groups of the tile's lanes");
  if (todo == 0) return RANGE ? 0u : kEmpty;
  const uint32_t lane = __lane_id(), r = lane & 15, row4 = (lane & 48) << 2;
  const uint32_t below = (1u << r) - 1;
  const bool mine = (todo >> r) & 1;
  {  // lanes without an operation walk with the tile's first one, and write nothing
    const int any = (int)(row4 + ((uint32_t)__builtin_ctz(todo) << 2));
    const uint32_t l0 = (uint32_t)__builtin_amdgcn_ds_bpermute(any, (int)lo);
    const uint32_t s0 = (uint32_t)__builtin_amdgcn_ds_bpermute(any, (int)start);
    const uint32_t t0 = (uint32_t)__builtin_amdgcn_ds_bpermute(any, (int)ts);
    const uint32_t h0 = RANGE ? (uint32_t)__builtin_amdgcn_ds_bpermute(any, (int)hi) : 0u;
    if (!mine) {
      lo = l0;
      start = s0;
      ts = t0;
      hi = h0;
      out = nullptr;
    }
  }
  const uint64_t* const pairs = tv.nodes + r * P;  // this lane's pairs of node 0
  const uint32_t last = tv.cap_ - 1;
  uint32_t res = RANGE ? 0u : kEmpty, err = 0, furthest = 0;  // furthest: the largest index followed
  uint32_t o_lo = lo32(reinterpret_cast<uint64_t>(out)), o_hi = hi32(reinterpret_cast<uint64_t>(out));
  for (uint32_t g = 0; g < 16 && (todo >> g) != 0; g += RG) {
    uint32_t k[RG], cur[RG], at[RG], h[RG], cnt[RG];
    uint64_t o[RG];
    uint64_t q[RG][P];
    each_walk<0, RG>([&](auto J) {
      constexpr int j = J.value;
      k[j] = row_bcast<j>(lo);
      cur[j] = row_bcast<j>(start);
      at[j] = row_bcast<j>(ts);
      cnt[j] = 0;
      if constexpr (RANGE) {
        h[j] = row_bcast<j>(hi);
        o[j] = pack(row_bcast<j>(o_lo), row_bcast<j>(o_hi));
      }
    });
    auto load = [&](int j) {
      const uint64_t* n = pairs + (uint64_t)cur[j] * NW;
      if constexpr (P == 1) {
        q[j][0] = *n;
      } else {
#pragma unroll
        for (int s = 0; s < P / 2; ++s) {
          const u64x2 v = reinterpret_cast<const u64x2*>(n)[s];
          q[j][2 * s] = v.x;
          q[j][2 * s + 1] = v.y;
        }
      }
    };
    auto meta_lo = [&](int j) { return row_bcast<15>(lo32(q[j][P - 1])); };
    auto meta_hi = [&](int j) { return row_bcast<15>(hi32(q[j][P - 1])); };
    auto follow = [&](int j, uint32_t next) {  // (an index past the pool is flagged at the end)
      furthest = next > furthest ? next : furthest;
      cur[j] = next < last ? next : last;
    };
    // Down to the leaves, the group's walks one level at a time.
    for (uint32_t step = 0;; ++step) {
#pragma unroll
      for (int j = 0; j < RG; ++j) load(j);
      if (meta_hi(0) & kLeafBit) break;
      if (step >= kMaxReadSteps) {
        err |= kErrCorrupt;
        break;
      }
#pragma unroll
      for (int j = 0; j < RG; ++j) {
        uint32_t v = hi32(q[j][0]);
        uint64_t b = 0;
#pragma unroll
        for (int s = 0; s < P; ++s) {
          // pivots <= key: an empty pair's key is above every key, and the
          // version and metadata pairs have the bound 0
          const bool m = lo32(q[j][s]) < ((uint32_t)(r * P + s) < node_t::kData ? k[j] + 1 : 0u);
          if (s == 0) b = __builtin_amdgcn_ballot_w64(m);
          else if (m) v = hi32(q[j][s]);
        }
        // they are a prefix: its last lane holds the child (lane 0 if it is empty)
        const uint32_t n = (uint32_t)__builtin_popcount(row_bits(b, lane));
        follow(j, (uint32_t)__builtin_amdgcn_ds_bpermute((int)(row4 - 4 + ((n > 1 ? n : 1u) << 2)), (int)v));
      }
    }
    // At the leaves: right moves, version chains and scans, all nodes of a pass
    // loaded before any is used. Bit j of `in`: walk j has reached its leaf.
    uint32_t act = (1u << RG) - 1, in = 0;
    for (uint32_t step = 0;;) {
#pragma unroll
      for (int j = 0; j < RG; ++j) {
        if (!((act >> j) & 1)) continue;
        const uint32_t high = meta_lo(j);
        if (!((in >> j) & 1) && k[j] >= high) {
          follow(j, meta_hi(j) & kPtrMask);
          continue;
        }
        in |= 1u << j;
        if constexpr (VER) {
          if (at[j] != kLatest && row_bcast<kVerLane>(lo32(q[j][kVerSlot])) > at[j]) {  // stamped later
            const uint32_t older = row_bcast<kVerLane>(hi32(q[j][kVerSlot]));
            if (older == kNone) {  // no version old enough
              err |= kErrVersionGap;
              act &= ~(1u << j);
            } else {
              follow(j, older);
            }
            continue;
          }
        }
        if constexpr (!RANGE) {
          uint32_t v = 0;
          bool f = false;
#pragma unroll
          for (int s = 0; s < P; ++s) {
            const bool m = lo32(q[j][s]) == k[j] && (uint32_t)(r * P + s) < node_t::kData;
            if (m) v = hi32(q[j][s]);
            f |= m;
          }
          const uint32_t bits = row_bits(__builtin_amdgcn_ballot_w64(f), lane);
          const uint32_t l = (uint32_t)__builtin_ctz(bits | 0x8000u);
          v = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(row4 + (l << 2)), (int)v);
          if (r == g + (uint32_t)j) res = bits ? v : kEmpty;
          act &= ~(1u << j);
        } else {
          // pairs of [k, h): a contiguous run of the sorted node
          uint32_t before = cnt[j], total = cnt[j];
          bool m[P];
#pragma unroll
          for (int s = 0; s < P; ++s) {
            m[s] = lo32(q[j][s]) - k[j] < ((uint32_t)(r * P + s) < node_t::kData ? h[j] - k[j] : 0u);
            const uint32_t bits = row_bits(__builtin_amdgcn_ballot_w64(m[s]), lane);
            before += (uint32_t)__builtin_popcount(bits & below);
            total += (uint32_t)__builtin_popcount(bits);
          }
          if (o[j] != 0) {
            uint64_t* slot = reinterpret_cast<uint64_t*>(o[j]);
#pragma unroll
            for (int s = 0; s < P; ++s) {
              if (m[s] && before < cap) slot[before] = q[j][s];
              before += m[s] ? 1u : 0u;
            }
          }
          cnt[j] = total;
          const uint32_t sib = meta_hi(j) & kPtrMask;
          if (h[j] <= high || sib == kNoSibling) act &= ~(1u << j);
          else follow(j, sib);
        }
      }
      if (act == 0) break;
      if (++step >= kMaxReadSteps) {
        err |= kErrCorrupt;
        break;
      }
#pragma unroll
      for (int j = 0; j < RG; ++j)
        if ((act >> j) & 1) load(j);
    }
    if constexpr (RANGE) {
#pragma unroll
      for (int j = 0; j < RG; ++j)
        if (r == g + (uint32_t)j) res = cnt[j];
    }
    lo = row_rotate<RG>(lo);
    start = row_rotate<RG>(start);
    ts = row_rotate<RG>(ts);
    if constexpr (RANGE) {
      hi = row_rotate<RG>(hi);
      o_lo = row_rotate<RG>(o_lo);
      o_hi = row_rotate<RG>(o_hi);
    }
  }
  if (furthest > last) err |= kErrCorrupt;
  if (err && r == 0) atomic_or32(&tv.st->error_flags, err);
  return mine ? res : RANGE ? 0u : kEmpty;
}

// Finds of a tile that takes `per` keys at a time. Walks in flight, measured on
// MI355X: at 32 pairs two (1M finds at 40M keys 94 us; one 100, four 98); at 16
// pairs four where tiles are full (1M at 10M keys 60 us; two 70, eight 78), two
// where a tile has at most four keys (64K: 11.2 against 15.4 us with four, of
// which most then repeat another's loads).
template <int NW, bool VER>
MVBT_DEV uint32_t find_rows(const tree_view<NW, VER>& tv, uint32_t key, uint32_t ts, uint32_t start, uint32_t todo,
                            uint32_t per) {
  if constexpr (NW == 16) {
    if (per > 4) return read_rows<false, 4>(tv, key, 0u, ts, start, nullptr, 0u, todo);
  }
  return read_rows<false, NW == 64 ? 1 : 2>(tv, key, 0u, ts, start, nullptr, 0u, todo);
}
// Ranges, one walk in flight: walks of one group end at different passes, and a
// pass costs its instructions for every walk of the group. 500K of 32 pairs at
// 40M keys, 32-pair nodes: 165 us (two 245, four 216, the pass-based reader 223);
// at 10M keys, 16-pair nodes: 170 (two 194, four 252, pass-based 249).
template <int NW, bool VER>
MVBT_DEV uint32_t range_rows(const tree_view<NW, VER>& tv, uint32_t lo, uint32_t hi, uint32_t ts, uint32_t start,
                             uint64_t* out, uint32_t cap, uint32_t todo) {
  return read_rows<true, 1>(tv, lo, hi, ts, start, out, cap, todo);
}

}  // namespace mvbt
