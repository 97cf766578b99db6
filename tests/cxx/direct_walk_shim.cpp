// C entry points for the CPU test tests/test_direct_walk.py, which builds this
// file with g++ beside tal_sh_amd/csrc/plan.cpp, direct_args.cpp and route.cpp: the walk
// of a direct contraction kernel through its K steps.
#include <cstdint>
#include <cstring>
#include <set>
#include <vector>

#include "direct_args.hpp"
#include "plan.hpp"
#include "route.hpp"

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

namespace {

// The lane offsets that one operand's loads form, against the addresses they
// mean: `rows` / rs its group and stride of rows, t its place in k's strides.
struct Operand {
  const DirectGroup &g;
  bool grouped;
  int64_t stride, kstride, nrows;
  const std::vector<DirectDim> &rdims;
  int t, tile;
};

int64_t true_row(const Operand &o, int esz, int64_t r) {
  int64_t x = 0;
  for (const DirectDim &d : o.rdims) {
    x += r % d.ext * d.s[0] * esz;
    r /= d.ext;
  }
  return x;
}
int64_t true_k(const DirectForm &f, int esz, int t, int64_t k) {
  int64_t x = 0;
  for (const DirectDim &d : f.k) {
    x += k % d.ext * d.s[t] * esz;
    k /= d.ext;
  }
  return x;
}

// 0: every load of the walk reads what it means to (past the edge: nothing);
// 1: a load inside the operand misses the range of its resource or its address;
// 2: a row past the edge comes back into the range.
int check_operand(const DirectForm &f, const DirectArgs &a, const DirectVariant &v, const Operand &o, int esz, int kb,
                  int width) {
  if (v.mode == 3) return 0;  // 64-bit addresses
  const int64_t tiles = (o.nrows + o.tile - 1) / o.tile;
  std::set<int64_t> which = {0, tiles / 2, tiles - 1};
  for (int64_t tile : which) {
    const int64_t r0 = tile * o.tile, base0 = o.grouped ? 0 : r0 * o.stride;
    std::vector<uint32_t> ro(o.tile);
    for (int64_t r = r0; r < r0 + o.tile; ++r)
      ro[r - r0] = r >= o.nrows ? kOutside
                   : o.grouped  ? group_offset32(o.g, (uint32_t)r)
                                : (uint32_t)(r - r0) * (uint32_t)o.stride;
    RunWalk w = run_walk(a.k);
    int kr = 0, kd1 = 0;
    int64_t at[2] = {0, 0};
    if (v.mode == 1) run_start(a.k, 0, &at[0], &at[1], &kr, &kd1);
    const int64_t whole = f.K / kb * kb;
    uint32_t advance = 0;
    for (int64_t k0 = 0; k0 < f.K; k0 += kb) {
      const bool lin = v.mode == 0 || (v.mode == 1 && a.k.nd == 1), tail = k0 >= whole && v.mode != 2;
      const bool wrap = a.k.nd > 2 && kd1 + 1 == (int)a.k.ext[1];
      const int d = wrap ? w.wrap[o.t] : w.next[o.t], cross = w.e0 - kr;
      int64_t base = base0;
      if (tail) base += lin ? k0 * o.kstride : 0;
      else if (v.mode == 1) base += at[o.t] + (d < 0 ? d : 0);
      // elements of a load along k; the last, partial step is loaded one by one
      const int wide = !tail && (o.t ? v.kb : v.ka) ? width : 1;
      for (int kk = 0; kk < kb; kk += wide) {
        uint64_t ko;
        if (v.mode == 2 || tail) {
          uint32_t x[2] = {kOutside, kOutside};
          if (k0 + kk < f.K) {
            if (v.mode != 2 && lin) x[0] = x[1] = (uint32_t)kk * (uint32_t)o.kstride;
            else pair_offsets32(a.k, (uint32_t)(k0 + kk), &x[0], &x[1]);
          }
          ko = x[o.t];
        } else if (v.mode == 0) {
          ko = (uint64_t)(uint32_t)kk * (uint32_t)o.kstride + advance;
        } else {
          ko = (uint64_t)(uint32_t)kk * (uint32_t)o.kstride + (uint32_t)(kk >= cross ? (d > 0 ? d : 0) : (d < 0 ? -(int64_t)d : 0));
        }
        for (int r = 0; r < o.tile; ++r) {
          const uint64_t off = ro[r] + ko;
          const bool in = r0 + r < o.nrows && k0 + kk < f.K;
          if (!in && (off < kOutside || off >> 32)) return 2;
          if (!in) continue;
          if (off + (uint64_t)(esz * wide) > kOutside) return 1;
          if (base + (int64_t)off != true_row(o, esz, r0 + r) + true_k(f, esz, o.t, k0 + kk)) return 1;
        }
      }
      if (v.mode == 0 && k0 + 2 * kb <= f.K) advance += (uint32_t)kb * (uint32_t)o.kstride;
      if (v.mode == 1 && k0 + 2 * kb <= f.K) {
        const bool over = kr + kb >= w.e0;
        for (int t = 0; t < 2; ++t)
          at[t] += kb * (t ? a.kb1 : a.ka1) + (over ? (wrap ? w.wrap[t] : w.next[t]) : 0);
        kr += over ? kb - w.e0 : kb;
        kd1 = !over ? kd1 : wrap ? 0 : kd1 + 1;
      }
    }
  }
  return 0;
}

}  // namespace

// Lane offsets of a contraction read straight from the tensors, at every tile
// of the kind, both ways round.  Returns 0, -1 where the form is not taken by
// any tile, else 16 * (tile * 2 + swap) + 4 * operand + code.  modes: bits of the modes met.
int lane_offsets(const char *pattern, const int *ddims, const int *ldims, const int *rdims, int dk, int *modes) {
  DigitalPattern p;
  ContractPlan plan;
  if (parse_pattern(pattern, &p) || plan_contraction(p, ddims, ldims, rdims, 1, &plan) || !plan.direct_ok) return -1;
  *modes = 0;
  const int esz = direct_elem(dk);
  for (int tile = 0; tile < kDirectTiles; ++tile)
    for (int swap = 0; swap < 2; ++swap) {
      const DirectTile &ti = direct_tiles(dk)[tile];
      const DirectForm f = swap ? direct_swapped(plan.direct) : plan.direct;
      DirectArgs a;
      DirectVariant v;
      if (!direct_args(f, esz, direct_width(dk), ti.kb, &a, &v)) continue;
      *modes |= 1 << v.mode;
      const Operand A{a.am, (a.flags & kDirectGroupA) != 0, a.am1, a.ka1, f.M, f.m, 0, ti.bm};
      const Operand B{a.bn, (a.flags & kDirectGroupB) != 0, a.bn1, a.kb1, f.N, f.n, 1, ti.bn};
      if (int e = check_operand(f, a, v, A, esz, ti.kb, v.width)) return 16 * (tile * 2 + swap) + e;
      if (int e = check_operand(f, a, v, B, esz, ti.kb, v.width)) return 16 * (tile * 2 + swap) + 4 + e;
    }
  return *modes ? 0 : -1;
}

// Whether the product on the planner's operands (copied where it copies them)
// is one that the direct kernels take; *in_place: D is written where it lies.
int mat_addressable(const char *pattern, const int *ddims, const int *ldims, const int *rdims, int dk, int *in_place) {
  DigitalPattern p;
  ContractPlan plan;
  if (parse_pattern(pattern, &p) || plan_contraction(p, ddims, ldims, rdims, 1, &plan)) return -1;
  *in_place = plan.mat_d_in_place;
  DirectVariant v;
  return direct_addressable(plan.mat, dk, &v) ? 1 : 0;
}

// The route of a contraction without fast math on a GPU of `cus` compute units;
// out: mode and width of the product that it runs, and its tile.
int route_of(const char *pattern, const int *ddims, const int *ldims, const int *rdims, int dk, int cus, int *out) {
  DigitalPattern p;
  ContractPlan plan;
  if (parse_pattern(pattern, &p) || plan_contraction(p, ddims, ldims, rdims, 1, &plan)) return -1;
  static int on;
  on = cus;
  const Route r = contract_route(plan, dk, [](int kind, int64_t M, int64_t N, int64_t K, int64_t batch) {
    return direct_choose(kind, M, N, K, batch, on);
  });
  const DirectForm &f = r == kRouteDirect ? plan.direct : plan.mat;
  const DirectChoice c = direct_choose(dk, f.M, f.N, f.K, f.batch, cus);
  DirectArgs a;
  DirectVariant v;
  if (!direct_args(c.swap ? direct_swapped(f) : f, direct_elem(dk), direct_width(dk), direct_tiles(dk)[c.tile].kb, &a, &v))
    return r;
  out[0] = v.mode;
  out[1] = v.width;
  out[2] = c.tile;
  return r;
}

// Units of the launch that begins at unit `at`.
long long launch_units(long long units, long long at, unsigned threads) { return direct_launch_units(units, at, threads); }

// Whether a product has a tile shape, and its number of workgroups and threads of each.
int choose_units(int dk, long long M, long long N, long long K, int cus, long long *units) {
  const DirectChoice c = direct_choose(dk, M, N, K, 1, cus);
  *units = c.whole + c.rem * c.ksplit;
  return c.us >= 0;
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
