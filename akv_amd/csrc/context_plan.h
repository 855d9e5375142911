// How the keys of a prefill batch are shared out over workgroups
// (context_attention.hip, the split launch).  Host and device code, so that
// the cuts can be checked without a GPU.
//
// A KV head's work is a line of cost units: segments in order, a segment's
// token blocks in order, a block's key tiles in order; the heads follow each
// other.  2^k workgroups take equal stretches of that line, cut at tile
// boundaries.  Costs are 64-bit: segments whose queries and prefix keys each
// fit 31 bits have a plan (sixty-four of the longest would take a head's line
// past 63 bits only at groups of 64 q heads and more, and years).
#pragma once

#include <cstdint>

namespace akv {

#if defined(__HIPCC__)
#define AKV_HD __host__ __device__ __forceinline__
#else
#define AKV_HD inline
#endif

// Cost units of one key tile of a full token block.  The waves of a block
// with at most half its rows share the tile's keys, so it takes about half the
// time; with at most a quarter, less again where a tile has quarters enough
// (128 keys).
constexpr int kFullTile = 8, kHalfTile = 5, kQuarterTile = 3;
// The smallest stretch given to a workgroup, in full tiles of 128 keys (twice
// as many of 64).
constexpr int kMinStretch = 2;

struct SplitShape {
  int32_t token_shift;  // log2 of the tokens of a block
  int32_t key_shift;    // log2 of the keys of a tile: 6 or 7
};

// What a block costs beside its tiles (its queries, the first tile's latency,
// the result), half of it at each end: a cut that falls there moves to the
// block's end (a cut among its tiles stays, be it next to the first or last).
AKV_HD int32_t block_cost(const SplitShape& s) { return (4 * kFullTile) >> (s.key_shift - 6); }

// Extend-key tiles of a segment's first b blocks (block j sees the segment's
// first (j + 1) blocks of own keys).
AKV_HD int64_t ext_tiles_before(const SplitShape& s, int32_t b) {
  const int64_t n = b;
  if (s.token_shift >= s.key_shift) return (n * (n + 1) / 2) << (s.token_shift - s.key_shift);
  const int r = s.key_shift - s.token_shift;  // 2^r blocks share a tile count
  const int64_t a = b >> r, e = b & ((1 << r) - 1);
  return ((a * (a + 1) / 2) << r) + e * (a + 1);
}

// (n + 2^shift - 1) >> shift without the sum's overflow near 2^31
AKV_HD int32_t shift_up(int32_t n, int shift) { return (n >> shift) + ((n & ((1 << shift) - 1)) != 0); }

AKV_HD int32_t split_blocks(const SplitShape& s, int32_t q) { return shift_up(q, s.token_shift); }

AKV_HD int32_t key_tiles(const SplitShape& s, int32_t n) { return shift_up(n, s.key_shift); }

// Tiles of block b of a segment with q queries and p prefix keys.
AKV_HD int32_t block_tiles(const SplitShape& s, int32_t q, int32_t p, int32_t b) {
  const int32_t left = q - (b << s.token_shift), full = 1 << s.token_shift;
  return key_tiles(s, p) + key_tiles(s, left < full ? q : (b + 1) << s.token_shift);
}

// Cost of one tile of block b: only a segment's last block can be short.
AKV_HD int32_t tile_cost(const SplitShape& s, int32_t q, int32_t b) {
  const int32_t tokens = q - (b << s.token_shift), full = 1 << s.token_shift;
  if (tokens > full / 2) return kFullTile;
  return s.key_shift < 7 || tokens > full / 4 ? kHalfTile : kQuarterTile;
}

// Cost of the segment's blocks before b (b < blocks: all of them full).
AKV_HD int64_t cost_before(const SplitShape& s, int32_t p, int32_t b) {
  return kFullTile * (static_cast<int64_t>(b) * key_tiles(s, p) + ext_tiles_before(s, b)) +
         static_cast<int64_t>(b) * block_cost(s);
}

AKV_HD int64_t segment_cost(const SplitShape& s, int32_t q, int32_t p) {
  if (q <= 0) return 0;
  const int32_t last = split_blocks(s, q) - 1;
  return cost_before(s, p, last) + static_cast<int64_t>(tile_cost(s, q, last)) * block_tiles(s, q, p, last) +
         block_cost(s);
}

// A bound of any head's cost for a batch of these sums.
AKV_HD int64_t cost_bound(const SplitShape& s, int64_t segments, int64_t queries, int64_t prefix) {
  const int64_t blocks = (queries >> s.token_shift) + segments;
  const int64_t tiles = ((queries + prefix) >> s.key_shift) + 2;
  return blocks * (kFullTile * tiles + block_cost(s));
}

// log2 of the number of stretches: as many as there are workgroups, unless
// they would be shorter than kMinStretch.
AKV_HD int32_t parts_shift(const SplitShape& s, int64_t total, int32_t heads, int32_t max_shift) {
  const int64_t least = static_cast<int64_t>(kMinStretch * kFullTile) << (7 - s.key_shift);
  const int64_t enough = least << max_shift;
  const int64_t cost = (total < enough ? total : enough) * heads;
  int32_t k = 0;
  while (k < max_shift && (least << (k + 1)) <= cost) ++k;
  return k;
}

// A place on the line: tile `tile` of block `block` of segment `seg` for KV
// head `head`.
struct Place {
  int32_t head, seg, block, tile;
};

AKV_HD bool same_block(const Place& x, const Place& y) {
  return x.head == y.head && x.seg == y.seg && x.block == y.block;
}

// Where boundary r of 2^k stretches lies.  get(s, &q, &p, &before) gives
// segment s (in order; live: the ones with queries) and the cost before it;
// total is one head's cost.
template <typename Get>
AKV_HD Place place_of(const SplitShape& s, Get get, uint64_t live, int64_t total, int32_t heads, int32_t k, int32_t r) {
  const uint32_t hr = static_cast<uint32_t>(heads) * static_cast<uint32_t>(r);
  Place at;
  at.head = static_cast<int32_t>(hr >> k);
  const int64_t part = hr & ((1u << k) - 1);
  int64_t x = (total >> k) * part + (((total & ((1 << k) - 1)) * part) >> k);  // total * part / 2^k
  for (;;) {
    int32_t q = 0, p = 0;
    int64_t before = 0;
    at.seg = 0;
    for (uint64_t rest = live; rest; rest &= rest - 1) {
      const int i = __builtin_ctzll(rest);
      int32_t qi, pi;
      int64_t bi;
      get(i, &qi, &pi, &bi);
      if (bi <= x) {
        at.seg = i;
        q = qi;
        p = pi;
        before = bi;
      }
    }
    int32_t lo = 0, hi = split_blocks(s, q) - 1;
    while (lo < hi) {
      const int32_t mid = lo + ((hi - lo + 1) >> 1);
      if (before + cost_before(s, p, mid) <= x) lo = mid; else hi = mid - 1;
    }
    at.block = lo;
    const int64_t off = x - before - cost_before(s, p, lo) - block_cost(s) / 2;
    const int32_t cost = tile_cost(s, q, lo), tiles = block_tiles(s, q, p, lo);
    // off is within one block here, whose cost fits 31 bits
    at.tile = off < 0 ? 0 : static_cast<int32_t>(static_cast<uint32_t>(off) / static_cast<uint32_t>(cost));
    if (at.tile < tiles) return at;
    // past the last tile: the next block's beginning
    x = x - off + static_cast<int64_t>(tiles) * cost + block_cost(s) / 2;
    if (x == total) {
      ++at.head;
      x = 0;
    }
  }
}

// A workgroup's stretch: the block it is at, and where it starts and ends.
struct SplitState {
  Place cur, first, end;
  uint64_t live;  // segments with queries
  int32_t rank;
  int32_t last;  // the part left for last is the one being done
};

// The next block, segment or head after s.cur in its stretch, then the part
// left for last; false when the stretch is done.  qlen: s.cur's segment.
AKV_HD bool next_piece(const SplitShape& shape, int32_t heads, SplitState& s, int32_t qlen) {
  if (s.last) return false;
  bool done = same_block(s.cur, s.end);
  if (!done) {
    s.cur.tile = 0;
    if (s.cur.block + 1 < split_blocks(shape, qlen)) {
      ++s.cur.block;
    } else {
      s.cur.block = 0;
      const uint64_t later = s.cur.seg < 63 ? s.live >> (s.cur.seg + 1) << (s.cur.seg + 1) : 0;
      if (!later) ++s.cur.head;
      s.cur.seg = __builtin_ctzll(later ? later : s.live);
    }
    done = s.cur.head >= heads || (same_block(s.cur, s.end) && s.end.tile == 0);
  }
  if (!done) return true;
  if (s.first.tile == 0 || same_block(s.first, s.end)) return false;
  s.cur = s.first;
  s.last = 1;
  return true;
}

}  // namespace akv
