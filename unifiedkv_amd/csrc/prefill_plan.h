// Block plan of the tiled prefill (host only, no HIP): how many wide and narrow query blocks each
// (sequence, KV group) pair takes and how many parts its keys are cut into. A launch runs in rounds of
// one block per slot (CU, or half a CU where two workgroups share one); each XCD's slots take the XCD's
// blocks in the kernel's order, each slot the next block once free, and the plan with the shortest
// predicted launch is taken.
//
// It runs on the calling thread before a launch of ~30 us or more, and a serving engine's chunks rarely have
// the shape of an earlier one, so a plan not yet known has to be cheap: whole blocks are timed in closed form,
// part counts are ranked by a lower bound and the best few simulated. 400 random
// chunks on 28/4 heads take 23 us on average and 130 at most on a 2.7 GHz Xeon (one KV head 45 and 170), within
// 0.3 % of the best of every mix and part count on average; simulating them all on every XCD took 0.8 ms.
#pragma once

#include <algorithm>
#include <array>
#include <cstdint>
#include <map>
#include <mutex>
#include <tuple>

namespace ukv {

constexpr int kTileKeys = 32;

struct BlockPlan {
  int n3, n2;             // wide and narrow query blocks of each pair
  int parts, part_tiles;  // parts of the keys, and the tiles of one
  int whole3, whole2;     // the blocks of a pair whose keys fill one part (the table may be wider than they)
};

// A launch: pairs of (sequence, KV group) whose longest chunk has max_cols columns (query, head), blocks
// of w2 / w3 columns, tables of `tiles` key tiles.
struct PlanShape {
  int64_t max_cols, pairs, part_row_bytes;  // part_row_bytes: one part's partials of the whole call
  int w2, w3, n_rep, slots_per_xcd, tiles;
  double narrow;  // cost of a narrow block relative to a wide one
  bool allow_parts;
};

// Cost of a narrow block relative to a wide one: single blocks timed over the same 32768 keys (3 and
// 2 column blocks), and estimated from the instruction counts (2 and 1).
constexpr double kNarrowCost = 0.79, kNarrowCostFine = 0.62;
// Key parts: a block's fixed cost (first loads, page ids, the output) and the merge launch, in tile
// times of a wide block (1.16 us), the bytes of partials merged per tile time (read at 4 TB/s and
// half of them again for the blocks' stores), and the fewest tiles a part is worth a block for.
constexpr double kStartTiles = 5.0, kMergeTiles = 4.0, kMergeBytesPerTile = 3.1e6;
constexpr int kMinPartTiles = 12, kMaxParts = 16;
constexpr int kMaxSlots = 128, kMaxPlanItems = 2048, kMaxPlanSteps = 2000;

// The range of work items [start, end) that XCD xcd runs of `total` (the kernel's xcd_range).
inline void plan_xcd_range(int64_t total, int xcd, int64_t& start, int64_t& end) {
  const int64_t per = total / 8, rem = total % 8;
  start = xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per;
  end = start + per + (xcd < rem ? 1 : 0);
}

// Items numbered below `start` (pair after pair, n to a pair) that are among the first nl of their pair.
inline int64_t wide_below(int64_t start, int n, int nl) {
  return start / n * nl + std::min<int64_t>(start % n, nl);
}

// Whole blocks that all stream equally many keys: n3 of cost 1, dispatched first, and n2 of cost c.
// Slots hold q or q + 1 wide blocks; the narrow ones then finish at the earliest of the times
// (slot's wide blocks) + k c, so the last of N finishes at the N-th of them.
inline double flat_makespan(int64_t pairs, int n3, int n2, double c, int slots) {
  const int n = n3 + n2;
  double worst = 0.0;
  for (int x = 0; x < 8; ++x) {
    int64_t start, end;
    plan_xcd_range(pairs * n, x, start, end);
    const int64_t wide = wide_below(end, n, n3) - wide_below(start, n, n3), narrow = end - start - wide;
    const int64_t q = wide / slots, r = wide % slots;
    double t = (double)(q + (r > 0));
    if (narrow > 0) {
      auto finished = [&](double at) {  // narrow blocks finished by then
        const double k0 = (at - q) / c + 1e-9, k1 = (at - q - 1) / c + 1e-9;
        return (slots - r) * (int64_t)std::max(0.0, k0) + r * (int64_t)std::max(0.0, k1);
      };
      const double least = (wide + narrow * c) / slots;  // no slot idle
      double last = 0.0;
      for (int slow = 0; slow < 2; ++slow) {
        const double from = (double)(q + slow);
        int64_t k = std::max<int64_t>(1, (int64_t)((least - from) / c));
        while (finished(from + k * c) < narrow) ++k;
        if (last == 0.0 || from + k * c < last) last = from + k * c;
      }
      t = std::max(t, last);
    }
    worst = std::max(worst, t);
  }
  return worst;
}

// Slots as a binary heap of the times they are free: give() puts the next item on the first free one.
struct SlotHeap {
  std::array<double, kMaxSlots> at{};
  int n;
  double last = 0.0;
  explicit SlotHeap(int slots) : n(std::min(slots, kMaxSlots)) {}
  void give(double cost) {
    const double t = at[0] + cost;
    last = std::max(last, t);
    int i = 0;
    for (;;) {
      int c = 2 * i + 1;
      if (c >= n) break;
      if (c + 1 < n && at[c + 1] < at[c]) ++c;
      if (at[c] >= t) break;
      at[i] = at[c];
      i = c;
    }
    at[i] = t;
  }
};

// A mix of blocks with causal key counts: each streams the keys up to its last query's own.
struct CausalBlocks {
  const PlanShape& f;
  int n3 = 0, n2 = 0;
  std::array<int, kMaxPlanItems> seen;          // key tiles each block sees
  std::array<double, kMaxPlanItems + 1> below;  // all_parts(0 .. j - 1)

  explicit CausalBlocks(const PlanShape& shape) : f(shape) {}
  void set(int wide, int narrow) {
    n3 = wide;
    n2 = narrow;
    for (int j = 0; j < n3 + n2; ++j) {
      const int64_t after = j < n3 ? (int64_t)f.w3 * j : (int64_t)f.w3 * n3 + (int64_t)f.w2 * (j - n3);
      seen[j] = (int)std::max<int64_t>(1, f.tiles - after / f.n_rep / kTileKeys);
    }
  }
  int first_tile(int s, int parts) const { return (int)((int64_t)s * f.tiles / parts); }
  // Block j's time on tiles [t0, t1) (a part), in tile times of a wide block.
  double cost(int j, int t0, int t1) const {
    return seen[j] > t0 ? kStartTiles + (std::min(seen[j], t1) - t0) * (j < n3 ? 1.0 : f.narrow) : 0.3;
  }
  // Block j's times summed over the parts.
  double all_parts(int j, int parts) const {
    const int in = (int)std::min<int64_t>(parts, ((int64_t)seen[j] * parts + f.tiles - 1) / f.tiles);  // parts it sees
    return in * kStartTiles + seen[j] * (j < n3 ? 1.0 : f.narrow) + 0.3 * (parts - in);
  }
  // No schedule is shorter: every slot busy, and the longest item (block 0 sees every tile).
  double lower_bound(int parts) const {
    double pair = 0.0;
    for (int j = 0; j < n3 + n2; ++j) pair += all_parts(j, parts);
    const double longest = kStartTiles + ((f.tiles + parts - 1) / parts) * (n3 > 0 ? 1.0 : f.narrow);
    return std::max(longest, f.pairs * pair / (8.0 * f.slots_per_xcd));
  }
  // The XCDs' slots taking their pairs' blocks part after part, wide ones first; the ranges with an item more go
  // round the XCDs. The most loaded XCD alone, or, where that is below `limit`, the slowest of all eight.
  double makespan(int parts, double limit) {
    const int n = n3 + n2, rem = (int)(f.pairs * n % 8);
    below[0] = 0.0;
    for (int j = 0; j < n; ++j) below[j + 1] = below[j] + all_parts(j, parts);
    std::array<double, 8> load;  // of each range, over the parts' average
    std::array<int64_t, 8> start, end;
    for (int y = 0; y < 8; ++y) {
      plan_xcd_range(f.pairs * n, y, start[y], end[y]);
      load[y] = (end[y] / n - start[y] / n) * below[n] + below[end[y] % n] - below[start[y] % n];
    }
    int loaded = 0;
    double most = -1.0;
    for (int x = 0; x < 8; ++x) {
      double all = 0.0;
      for (int s = 0; s < parts; ++s) all += load[(x + s * rem) & 7];
      if (all > most) {
        most = all;
        loaded = x;
      }
    }
    double t = makespan_of(loaded, rem, parts, start, end);
    const bool alike = f.pairs % 8 == 0;  // every XCD runs whole pairs, as many
    for (int x = 0; x < 8 && t < limit && !alike; ++x)
      if (x != loaded) t = std::max(t, makespan_of(x, rem, parts, start, end));
    return t;
  }
  double makespan_of(int xcd, int rem, int parts, const std::array<int64_t, 8>& start,
                     const std::array<int64_t, 8>& end) const {
    const int n = n3 + n2;
    SlotHeap slots(f.slots_per_xcd);
    for (int s = 0; s < parts; ++s) {
      const int y = (xcd + s * rem) & 7;
      if (end[y] == start[y]) continue;
      const int t0 = first_tile(s, parts), t1 = first_tile(s + 1, parts);
      for (int pass = 0; pass < 2; ++pass)
        for (int64_t p = start[y] / n; p <= (end[y] - 1) / n; ++p) {
          const int j0 = (int)std::max<int64_t>(pass ? n3 : 0, start[y] - p * n);
          const int j1 = (int)std::min<int64_t>(pass ? n : n3, end[y] - p * n);
          for (int j = j0; j < j1; ++j) slots.give(cost(j, t0, t1));
        }
    }
    return slots.last;
  }
};

inline double merge_tiles(const PlanShape& f, int parts) {
  return kMergeTiles + parts * (double)f.part_row_bytes / kMergeBytesPerTile;
}

inline BlockPlan compute_plan(const PlanShape& f, bool parts_ok) {
  const int n3_max = (int)((f.max_cols + f.w3 - 1) / f.w3);
  BlockPlan best{n3_max, 0, 1, std::max(1, f.tiles), n3_max, 0};
  auto narrow_blocks = [&](int n3) { return (int)((f.max_cols - (int64_t)n3 * f.w3 + f.w2 - 1) / f.w2); };
  // Each wide block traded for narrow ones adds work: a dozen trades fill any last round.
  double best_t = flat_makespan(f.pairs, n3_max, 0, f.narrow, f.slots_per_xcd);
  for (int n3 = n3_max - 1; n3 >= std::max(0, n3_max - 12); --n3) {
    const int n2 = narrow_blocks(n3);
    const double t = flat_makespan(f.pairs, n3, n2, f.narrow, f.slots_per_xcd);
    if (t < best_t - 1e-9) {
      best_t = t;
      best.n3 = n3;
      best.n2 = n2;
    }
  }
  best.whole3 = best.n3;
  best.whole2 = best.n2;
  if (!parts_ok || n3_max + 4 > kMaxPlanItems || best.n3 + best.n2 > kMaxPlanItems) return best;
  CausalBlocks blocks(f);
  blocks.set(best.n3, best.n2);
  const double whole = blocks.makespan(1, 1e30);
  // Every part count with wide blocks alone, one or two of them traded, and the whole blocks' mix: those
  // that some count is best with. Ranked by the bound, then simulated until the next bound is no better.
  struct Candidate {
    double bound;
    int n3, n2, parts;
  };
  std::array<Candidate, 4 * kMaxParts> c;
  int n = 0;
  auto add = [&](int n3, int n2) {
    blocks.set(n3, n2);
    for (int parts = 2; parts <= std::min(kMaxParts, f.tiles / kMinPartTiles); ++parts) {
      if (merge_tiles(f, parts) >= 0.97 * whole) break;
      const double bound = merge_tiles(f, parts) + blocks.lower_bound(parts);
      if (bound < 0.97 * whole) c[n++] = {bound, n3, n2, parts};
    }
  };
  for (int n3 = n3_max; n3 >= std::max(0, n3_max - 2); --n3) add(n3, n3 == n3_max ? 0 : narrow_blocks(n3));
  // (Not where the chunk holds half of the keys or more: its later blocks see the first parts alone, and the
  // workgroups that exit in their place leave shader engines idle, which take workgroups in turn. One 2048-token
  // prompt on 16 heads without GQA in three parts: 54 us with wide blocks, 65 with eight narrow ones.)
  const int64_t chunk_tiles = f.max_cols / f.n_rep / kTileKeys;
  if (best.n3 < n3_max - 2 && 2 * chunk_tiles <= f.tiles) add(best.n3, best.n2);
  std::sort(c.begin(), c.begin() + n, [](const Candidate& a, const Candidate& b) { return a.bound < b.bound; });
  best_t = 0.97 * whole;
  int64_t steps = kMaxPlanSteps;
  for (int i = 0; i < n && c[i].bound < best_t && steps > 0; ++i) {
    blocks.set(c[i].n3, c[i].n2);
    const double merge = merge_tiles(f, c[i].parts), t = merge + blocks.makespan(c[i].parts, best_t - merge);
    steps -= f.pairs * (c[i].n3 + c[i].n2) * c[i].parts / 8;
    if (t < best_t) {
      best_t = t;
      best.n3 = c[i].n3;
      best.n2 = c[i].n2;
      best.parts = c[i].parts;
    }
  }
  return best;
}

// x up to the next multiple of 1/16 to 1/32 of itself.
inline int64_t plan_step(int64_t x) {
  int64_t step = 1;
  while (x / step >= 32) step *= 2;
  return (x + step - 1) / step * step;
}

inline BlockPlan choose_plan(PlanShape f) {
  const int n3_max = (int)((f.max_cols + f.w3 - 1) / f.w3);
  // Large launches run many rounds, where the last one matters little: keep wide blocks.
  if (f.pairs * n3_max > (1 << 16) || f.slots_per_xcd <= 0 || n3_max == 0)
    return BlockPlan{n3_max, 0, 1, std::max(1, f.tiles), n3_max, 0};
  // Parts are considered for launches of few blocks: there whole blocks leave CUs idle.
  const bool parts_ok =
      f.allow_parts && f.tiles >= 2 * kMinPartTiles && f.pairs * n3_max < 16 * f.slots_per_xcd;
  // Ragged chunks share a plan: columns to the blocks' common divisor (the same block counts), partials to steps
  // of 3-6 %. Tiles stay exact: where a round of items just fits, the last part's few tiles decide it.
  const int tiles = f.tiles, unit = f.w3 - f.w2;
  f.max_cols = (f.max_cols + unit - 1) / unit * unit;
  f.tiles = parts_ok ? f.tiles : 0;
  f.part_row_bytes = parts_ok ? plan_step(f.part_row_bytes) : 0;
  static std::mutex mu;
  static std::map<std::tuple<int64_t, int64_t, int64_t, int, int, int, int>, BlockPlan> cache;
  const auto key = std::make_tuple(f.max_cols, f.pairs, f.part_row_bytes, f.w2, f.n_rep, f.slots_per_xcd, f.tiles);
  BlockPlan plan;
  bool known = false;
  {
    std::lock_guard<std::mutex> lock(mu);
    const auto hit = cache.find(key);
    if (hit != cache.end()) {
      plan = hit->second;
      known = true;
    }
  }
  if (!known) {
    plan = compute_plan(f, parts_ok);
    std::lock_guard<std::mutex> lock(mu);
    if (cache.size() >= 4096) cache.clear();  // a caller cycling through many shapes recomputes
    try {
      cache.emplace(key, plan);
    } catch (...) {  // (no memory for the entry: the plan itself needs none)
    }
  }
  plan.part_tiles = std::max(1, (tiles + plan.parts - 1) / plan.parts);
  return plan;
}

}  // namespace ukv
