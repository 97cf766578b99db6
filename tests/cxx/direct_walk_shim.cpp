// C entry points for the CPU test tests/test_direct_walk.py, which builds this
// file with g++ beside tal_sh_amd/csrc/plan.cpp and direct_args.cpp: the walk
// of a direct contraction kernel through its K steps.
#include <cstdint>
#include <cstring>
#include <set>
#include <vector>

#include "direct_args.hpp"
#include "plan.hpp"

using namespace tal;

extern "C" {

// The kernel's reads and writes of the table of contracted offsets, for a K
// range of `len` in steps of kb with pf steps in flight.  A phase is what lies
// between two barriers: within one, waves run in any order, so an entry that is
// written there must not be read there, and one that is read must have been
// written in an earlier phase.  Returns 0; 1: an entry is read while it is
// written over; 2: an entry does not hold the contracted index that is wanted.
int table_walk(int len, int kb, int half, int pf, int ahead) {
  const int steps = (len + kb - 1) / kb;
  std::vector<int> table(2 * half, -1);  // which contracted index an entry holds
  std::vector<std::pair<int, int>> pending;
  std::set<int> reads, writes;
  int bad = 0;
  auto fill = [&](int h) {
    for (int i = 0; i < half; ++i) {
      pending.emplace_back((h & 1) * half + i, h * half + i);
      writes.insert((h & 1) * half + i);
    }
  };
  auto read = [&](int at) {
    for (int i = 0; i < kb; ++i) {
      const int e = (at & (2 * half - 1)) + i;
      reads.insert(e);
      if (table[e] != at + i && !bad) bad = 2;
    }
  };
  auto barrier = [&] {
    for (int e : reads)
      if (writes.count(e)) bad = 1;
    for (auto &w : pending) table[w.first] = w.second;
    pending.clear();
    reads.clear();
    writes.clear();
  };
  int at = 0;
  auto load = [&] {
    if (!ahead) read(at);
    if (at + kb < len) {
      at += kb;
      const int h = table_refill(at, len, kb, half, ahead != 0);
      if (h >= 0) fill(h);
      if (ahead) read(at);
    }
  };
  fill(0);
  if (half < len) fill(1);
  barrier();
  if (ahead) read(at);
  for (int q = 0; q < pf; ++q) load();
  barrier();
  for (int t = 0; t < steps && !bad; ++t) {
    load();
    barrier();
  }
  return bad;
}

// Mode, tile and K range (in K) that a contraction gets straight from the
// tensors on a GPU of `cus` compute units, with tile's K step.
int direct_variant(const char *pattern, const int *ddims, const int *ldims, const int *rdims, int dk, int cus, int *out) {
  DigitalPattern p;
  ContractPlan plan;
  if (parse_pattern(pattern, &p) || plan_contraction(p, ddims, ldims, rdims, 1, &plan) || !plan.direct_ok) return -1;
  const DirectForm &f = plan.direct;
  const DirectChoice c = direct_choose(dk, f.M, f.N, f.K, f.batch, cus);
  DirectArgs a;
  DirectVariant v;
  const int kb = direct_tiles(dk)[c.tile].kb;
  if (!direct_args(c.swap ? direct_swapped(f) : f, direct_elem(dk), direct_width(dk), kb, &a, &v)) return -1;
  out[0] = v.mode;
  out[1] = c.tile;
  out[2] = c.rem ? (int)(c.ksteps * kb) : (int)f.K;
  return 0;
}

}  // extern "C"
