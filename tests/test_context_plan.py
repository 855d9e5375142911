"""The split prefill launch's cuts (``context_plan.h``) on the CPU: every tile
of a batch is done once, boundaries ascend, parts and the merge's walk over
them agree, and batches whose costs pass 32 bits have a plan too.  Signed
overflow aborts the program."""

import hostcpp

COMMON = r"""
#include "context_plan.h"

#include <algorithm>
#include <cstdio>
#include <map>
#include <random>
#include <tuple>
#include <vector>

using namespace akv;

#define CHECK(c)                                              \
  if (!(c)) {                                                 \
    std::printf("line %d (batch %d): %s\n", __LINE__, id, #c); \
    return false;                                             \
  }

// shape: the two instances' (512 rows, 128 keys) or (256 rows, 64 keys), group 2^gs
SplitShape shape_of(bool wide, int gs) { return SplitShape{(wide ? 8 : 9) - gs, wide ? 6 : 7}; }

struct Batch {
  SplitShape sh;
  int heads;
  std::vector<int32_t> q, p;
};

struct Plan {
  std::vector<int64_t> before;
  int64_t total = 0;
  uint64_t live = 0;
  int k = 0;
};

Plan plan_of(const Batch& b) {
  Plan pl;
  for (size_t s = 0; s < b.q.size(); ++s) {
    const int64_t cost = segment_cost(b.sh, b.q[s], b.p[s]);
    pl.before.push_back(pl.total);
    pl.total += cost;
    if (cost > 0) pl.live |= uint64_t(1) << s;
  }
  pl.k = pl.total ? parts_shift(b.sh, pl.total, b.heads, 8) : 0;
  return pl;
}

Place place(const Batch& b, const Plan& pl, int r) {
  return place_of(b.sh, [&](int i, int32_t* q, int32_t* p, int64_t* before) {
    *q = b.q[i]; *p = b.p[i]; *before = pl.before[i];
  }, pl.live, pl.total, b.heads, pl.k, r);
}

using Key = std::tuple<int, int, int, int>;
Key key(const Place& x) { return {x.head, x.seg, x.block, x.tile}; }

// boundaries ascend from the line's beginning to its end and lie on tiles
bool boundaries(int id, const Batch& b, const Plan& pl) {
  for (int s = 0; s < int(b.q.size()); ++s) CHECK(b.q[s] == 0 || (pl.live >> s & 1));
  CHECK(pl.total > 0);
  Place last = place(b, pl, 0);
  CHECK(key(last) == Key(0, __builtin_ctzll(pl.live), 0, 0));
  for (int r = 1; r <= 1 << pl.k; ++r) {
    const Place at = place(b, pl, r);
    CHECK(key(last) <= key(at));
    if (r == 1 << pl.k) {
      CHECK(at.head == b.heads);
      break;
    }
    CHECK(at.head < b.heads && at.seg < int(b.q.size()) && at.block < split_blocks(b.sh, b.q[at.seg]));
    CHECK(at.tile >= 0 && at.tile < block_tiles(b.sh, b.q[at.seg], b.p[at.seg], at.block));
    last = at;
  }
  return true;
}

// walks every workgroup's pieces as the kernel does, then the merge
bool walk(int id, const Batch& b, const Plan& pl) {
  const int groups = 1 << pl.k;
  std::map<std::tuple<int, int, int>, std::vector<std::pair<int, int>>> done;
  std::map<int, std::tuple<int, int, int, int, int>> parts;
  for (int rank = 0; rank < groups; ++rank) {
    SplitState s{};
    s.first = s.cur = place(b, pl, rank);
    s.end = place(b, pl, rank + 1);
    s.live = pl.live;
    if (same_block(s.first, s.end) ? s.first.tile == s.end.tile
                                   : s.first.tile > 0 && !next_piece(b.sh, b.heads, s, b.q[s.first.seg]))
      continue;
    do {
      const Place at = s.cur;
      const int n = block_tiles(b.sh, b.q[at.seg], b.p[at.seg], at.block);
      const int stop = same_block(at, s.end) ? s.end.tile : n;
      CHECK(at.tile < stop && stop <= n);
      done[{at.head, at.seg, at.block}].push_back({at.tile, stop});
      if (at.tile > 0 || stop < n) {
        const int slot = 2 * rank + (at.tile > 0 ? 0 : 1);
        CHECK(!parts.count(slot));
        parts[slot] = {at.head, at.seg, at.block, at.tile, stop};
      }
    } while (next_piece(b.sh, b.heads, s, b.q[s.cur.seg]));
  }
  size_t blocks = 0;
  for (size_t s = 0; s < b.q.size(); ++s) blocks += size_t(split_blocks(b.sh, b.q[s])) * b.heads;
  CHECK(done.size() == blocks);
  for (auto& [at, runs] : done) {
    std::sort(runs.begin(), runs.end());
    int from = 0;
    for (auto& r : runs) {
      CHECK(r.first == from);
      from = r.second;
    }
    CHECK(from == block_tiles(b.sh, b.q[std::get<1>(at)], b.p[std::get<1>(at)], std::get<2>(at)));
  }
  size_t merged = 0;
  for (int r0 = 1; r0 < groups; ++r0) {
    const Place at = place(b, pl, r0), prev = place(b, pl, r0 - 1);
    if (at.tile == 0 || (same_block(prev, at) && prev.tile > 0)) continue;  // not a block's first cut
    const int n = block_tiles(b.sh, b.q[at.seg], b.p[at.seg], at.block);
    int from = 0, to = at.tile;
    for (int r = r0;; ++r) {
      if (from < to) {
        const int slot = from == 0 ? 2 * (r - 1) + 1 : 2 * (r - 1);
        CHECK(parts.count(slot) && parts[slot] == std::make_tuple(at.head, at.seg, at.block, from, to));
        ++merged;
      }
      if (to == n) break;
      from = to;
      const Place next = r + 1 < groups ? place(b, pl, r + 1) : Place{b.heads, 0, 0, 0};
      to = same_block(next, at) ? next.tile : n;
    }
  }
  CHECK(merged == parts.size());
  return true;
}
"""

RANDOM = COMMON + r"""
int main() {
  std::mt19937 g(1);
  for (int id = 0; id < 6000; ++id) {
    Batch b;
    b.sh = shape_of(g() % 2, g() % 8);
    b.heads = 1 + g() % (id % 7 ? 12 : 33);
    const int n = 1 + g() % (id % 10 ? 5 : 64);
    for (int s = 0; s < n; ++s) {
      b.q.push_back(g() % 4 ? g() % (1 + (1 << g() % 10)) : 0);  // a quarter without queries
      b.p.push_back(g() % 3 ? g() % (1 + (1 << g() % 14)) : 0);
    }
    const Plan pl = plan_of(b);
    if (!pl.total) continue;
    int64_t queries = 0, prefix = 0;
    for (int s = 0; s < n; ++s) queries += b.q[s], prefix += b.p[s];
    if (pl.total > cost_bound(b.sh, n, queries, prefix)) return std::printf("bound, batch %d\n", id), 1;
    // the closed forms against the sums they stand for
    for (int s = 0; s < n; ++s) {
      int64_t sum = 0;
      for (int k = 0; k < split_blocks(b.sh, b.q[s]); ++k) {
        if (cost_before(b.sh, b.p[s], k) != sum) return std::printf("cost before, batch %d\n", id), 1;
        sum += int64_t(block_tiles(b.sh, b.q[s], b.p[s], k)) * tile_cost(b.sh, b.q[s], k) + block_cost(b.sh);
      }
      if (segment_cost(b.sh, b.q[s], b.p[s]) != sum) return std::printf("cost, batch %d\n", id), 1;
    }
    if (!boundaries(id, b, pl) || !walk(id, b, pl)) return 1;
  }
  std::puts("ok");
}
"""

LARGE = COMMON + r"""
int main() {
  // costs past 32 bits: one segment of 1.5M queries and prefixes up to 2^30,
  // walked; the largest lengths a segment can have, boundaries only
  const int32_t top = 0x7fffffff;
  const std::vector<Batch> walked = {
      {shape_of(true, 2), 1, {1500000}, {0}},
      {shape_of(true, 2), 3, {700000, 0, 800001}, {1 << 30, 5, 77}},
      {shape_of(false, 3), 2, {1500000, 3}, {100000000, 1 << 30}},
      {shape_of(true, 7), 1, {40000}, {top}},
  };
  int id = 0;
  for (const Batch& b : walked) {
    const Plan pl = plan_of(b);
    if (pl.total <= top) return std::printf("batch %d is not large\n", id), 1;
    if (pl.k != 8 || !boundaries(id, b, pl) || !walk(id, b, pl)) return 1;
    ++id;
  }
  for (int gs = 0; gs < 8; ++gs)
    for (bool wide : {false, true})
      for (int n : {1, 64}) {
        if (n == 64 && gs > 5) continue;  // their sum passes 63 bits
        Batch b{shape_of(wide, gs), 33, std::vector<int32_t>(n, top), std::vector<int32_t>(n, top)};
        if (n == 64) b.q[7] = 0;
        if (!boundaries(id++, b, plan_of(b))) return 1;
      }
  std::puts("ok");
}
"""


def test_cuts_cover_every_tile_once(tmp_path):
    assert hostcpp.run(tmp_path, RANDOM, "-ftrapv") == "ok\n"


def test_costs_past_32_bits(tmp_path):
    assert hostcpp.run(tmp_path, LARGE, "-ftrapv") == "ok\n"
