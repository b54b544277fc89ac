"""The prefill's block plan (csrc/prefill_plan.h, host code without HIP), compiled for the CPU with a device
of 32 slots an XCD (64 at 64 dims) given.

Against an exhaustive search (every mix of wide and narrow blocks, every part count, every XCD simulated with
a priority queue): the plan's predicted time is close to the best, planning is cheap, ragged chunks share
a plan, and large launches stay whole.
"""
import ctypes
import random
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

HARNESS = r"""
#include <chrono>
#include <queue>
#include <vector>
#include "prefill_plan.h"
using namespace ukv;

static PlanShape shape(const int64_t* p) {  // batch, rows, max_chunk, groups, dim, n_rep, pages
  const bool fine = p[4] != 128 || 16 % p[5];
  const int cb = fine ? 2 : 3;
  PlanShape f{};
  f.max_cols = p[2] * p[5];
  f.pairs = p[3] * p[0];
  f.part_row_bytes = p[1] * p[4] * 4;
  f.w2 = 8 * (cb - 1) * 16;
  f.w3 = 8 * cb * 16;
  f.n_rep = (int)p[5];
  f.slots_per_xcd = p[4] == 64 ? 64 : 32;
  f.tiles = (int)(p[6] + 1) / 2;
  f.narrow = fine ? kNarrowCostFine : kNarrowCost;
  f.allow_parts = true;
  return f;
}

// Every XCD's slots take its range's items, part after part, wide blocks first.
static double simulate(const PlanShape& f, int n3, int n2, int parts) {
  const int n = n3 + n2;
  const int64_t total = f.pairs * n, rem = total % 8;
  double worst = 0.0;
  for (int x = 0; x < 8; ++x) {
    std::priority_queue<double, std::vector<double>, std::greater<double>> slot;
    for (int i = 0; i < f.slots_per_xcd; ++i) slot.push(0.0);
    for (int s = 0; s < parts; ++s) {
      const int y = (int)((x + s * rem) % 8);
      const int64_t start = y * (total / 8) + std::min<int64_t>(y, rem), end = start + total / 8 + (y < rem);
      const int t0 = (int)((int64_t)s * f.tiles / parts), t1 = (int)((int64_t)(s + 1) * f.tiles / parts);
      for (int narrow = 0; narrow < 2; ++narrow)
        for (int64_t i = start; i < end; ++i) {
          const int j = (int)(i % n);
          if ((j >= n3) != (narrow == 1)) continue;
          const int64_t after = j < n3 ? (int64_t)f.w3 * j : (int64_t)f.w3 * n3 + (int64_t)f.w2 * (j - n3);
          const int seen = (int)std::max<int64_t>(1, f.tiles - after / f.n_rep / kTileKeys);
          const double c = seen > t0 ? kStartTiles + (std::min(seen, t1) - t0) * (j < n3 ? 1.0 : f.narrow) : 0.3;
          const double t = slot.top() + c;
          slot.pop();
          slot.push(t);
          worst = std::max(worst, t);
        }
    }
  }
  return worst + (parts > 1 ? merge_tiles(f, parts) : 0.0);
}

extern "C" void plan(const int64_t* p, int* out) {
  const BlockPlan b = choose_plan(shape(p));
  const int v[6] = {b.n3, b.n2, b.parts, b.part_tiles, b.whole3, b.whole2};
  std::copy(v, v + 6, out);
}
extern "C" double predicted(const int64_t* p, int n3, int n2, int parts) { return simulate(shape(p), n3, n2, parts); }
extern "C" double best(const int64_t* p) {
  const PlanShape f = shape(p);
  const int most = (int)((f.max_cols + f.w3 - 1) / f.w3);
  double t = 1e30;
  for (int n3 = most; n3 >= std::max(0, most - 12); --n3) {
    const int n2 = n3 == most ? 0 : (int)((f.max_cols - (int64_t)n3 * f.w3 + f.w2 - 1) / f.w2);
    for (int parts = 1; parts <= std::max(1, std::min(kMaxParts, f.tiles / kMinPartTiles)); ++parts)
      t = std::min(t, simulate(f, n3, n2, parts));
  }
  return t;
}
extern "C" double compute_us(const int64_t* p) {  // not from the cache; the fastest of five
  const PlanShape f = shape(p);
  double least = 1e30;
  for (int i = 0; i < 5; ++i) {
    const auto a = std::chrono::steady_clock::now();
    volatile int parts = compute_plan(f, true).parts;
    (void)parts;
    least = std::min(least, std::chrono::duration<double>(std::chrono::steady_clock::now() - a).count() * 1e6);
  }
  return least;
}
extern "C" double flat_error(int64_t pairs, int n3, int n2, double narrow, int slots) {
  double worst = 0.0;
  const int64_t n = n3 + n2, total = pairs * n, rem = total % 8;
  for (int x = 0; x < 8; ++x) {
    std::priority_queue<double, std::vector<double>, std::greater<double>> slot;
    for (int i = 0; i < slots; ++i) slot.push(0.0);
    const int64_t start = x * (total / 8) + std::min<int64_t>(x, rem), end = start + total / 8 + (x < rem);
    for (int pass = 0; pass < 2; ++pass)
      for (int64_t i = start; i < end; ++i) {
        if ((i % n >= n3) != (pass == 1)) continue;
        const double t = slot.top() + (pass ? narrow : 1.0);
        slot.pop();
        slot.push(t);
        worst = std::max(worst, t);
      }
  }
  return flat_makespan(pairs, n3, n2, narrow, slots) - worst;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{ROOT / 'unifiedkv_amd' / 'csrc'}",
                    str(d / "plan.cpp"), "-o", str(d / "plan.so")], check=True)
    lib = ctypes.CDLL(str(d / "plan.so"))
    for name in ("predicted", "best", "compute_us", "flat_error"):
        getattr(lib, name).restype = ctypes.c_double
    lib.flat_error.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_double, ctypes.c_int]
    return lib


def _shape(*p):
    return (ctypes.c_int64 * 7)(*p)


def _plan(lib, p):
    out = (ctypes.c_int * 6)()
    lib.plan(p, out)
    return list(out)  # n3, n2, parts, part_tiles, whole3, whole2


def _chunks(rng, groups, n_rep, dim):
    """A random chunked-prefill call: (batch, query rows, longest chunk, groups, dim, n_rep, table pages)."""
    batch = rng.choice([1, 2, 4, 4, 4, 8, 16])
    chunk = [rng.randint(1, rng.choice([512, 2048])) for _ in range(batch)]
    longest = max(c + rng.randint(0, rng.choice([4000, 16000, 32000])) for c in chunk)
    return _shape(batch, sum(chunk) * groups * n_rep, max(chunk), groups, dim, n_rep, -(-longest // 16))


HEADS = [(8, 4, 128), (4, 7, 128), (1, 4, 128), (2, 4, 128), (8, 1, 128), (8, 4, 64)]


@pytest.mark.parametrize("groups,n_rep,dim", HEADS)
def test_plan_is_close_to_the_best_of_every_mix_and_part_count(lib, groups, n_rep, dim):
    rng = random.Random(groups * 100 + n_rep + dim)
    ratios = []
    for _ in range(40):
        p = _chunks(rng, groups, n_rep, dim)
        n3, n2, parts, part_tiles, whole3, whole2 = _plan(lib, p)
        tiles = (p[6] + 1) // 2
        assert 1 <= parts <= 16 and parts * part_tiles >= tiles
        cb = 2 if dim == 64 or 16 % n_rep else 3
        for wide, narrow in ((n3, n2), (whole3, whole2)):  # both cover the longest chunk's columns
            assert (wide * cb + narrow * (cb - 1)) * 128 >= p[2] * n_rep
        assert parts == 1 or parts * (n3 + n2) >= whole3 + whole2  # the whole blocks fit the items of every part
        if groups * p[0] * -(-p[2] * n_rep // (cb * 128)) < 16 * (64 if dim == 64 else 32):
            ratios.append(lib.predicted(p, n3, n2, parts) / lib.best(p))
    # (a plan in parts has to be 3 % better than a whole one, partials are planned in steps of 3-6 %)
    assert len(ratios) > 10 and max(ratios) < 1.1 and sum(ratios) / len(ratios) < 1.02, sorted(ratios)[-5:]


def test_planning_a_new_shape_is_cheap(lib):
    """0.6-3 ms a shape where every part count and XCD is simulated; here 10-40 us (100 allowed for slow hosts)."""
    rng = random.Random(7)
    times = sorted(lib.compute_us(_chunks(rng, *rng.choice(HEADS))) for _ in range(200))
    assert sum(times) / len(times) < 100 and times[-1] < 400, times[-5:]


def test_ragged_chunks_share_a_plan(lib):
    """The same blocks and table, query rows a few per cent apart: one plan (its partials are sized by the call)."""
    plans = [_plan(lib, _shape(2, (900 + i) * 32, 500 + i // 3, 8, 128, 4, 1000)) for i in range(0, 30, 3)]
    assert len({tuple(p) for p in plans}) == 1 and plans[0][2] > 1


def test_only_launches_short_of_blocks_are_cut(lib):
    """Sixteen whole blocks a slot (8 x 32 slots) and more stay whole; the same keys with fewer blocks are cut."""
    assert _plan(lib, _shape(64, 64 * 2048 * 32, 2048, 8, 128, 4, 1000))[2] == 1
    assert _plan(lib, _shape(8, 8 * 768 * 32, 768, 8, 128, 4, 2048))[2] == 1  # 64 pairs of 8 blocks: 512
    assert _plan(lib, _shape(1, 512 * 32, 512, 8, 128, 4, 2048))[2] > 1
    assert _plan(lib, _shape(1, 512 * 32, 512, 8, 128, 4, 46))[2] == 1  # 23 key tiles: no two parts of 12


def test_closed_form_of_whole_blocks(lib):
    rng = random.Random(3)
    for _ in range(300):
        n3, n2 = rng.randint(0, 9), rng.randint(0, 14)
        if n3 + n2:
            assert abs(lib.flat_error(rng.randint(1, 200), n3, n2, rng.choice([0.79, 0.62]), rng.choice([32, 64]))) < 1e-9


def test_whole_mix_is_cut_only_behind_a_prefix(lib):
    """Narrow blocks alone, the mix of whole blocks here, are a candidate for parts where the chunk holds at most half
    of the keys; a prompt without a prefix keeps wide blocks."""
    n3, n2, parts, _, whole3, whole2 = _plan(lib, _shape(2, 2 * 512 * 32, 512, 8, 128, 4, 1024))
    assert parts > 1 and (n3, n2) == (whole3, whole2) == (0, 8)
    n3, _, parts, _, whole3, _ = _plan(lib, _shape(1, 2048 * 16, 2048, 16, 128, 1, 128))
    assert parts > 1 and whole3 == 0 and n3 >= 4  # of six
