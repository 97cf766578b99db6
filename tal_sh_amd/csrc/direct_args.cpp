// Layout arguments of the direct contraction kernels, and the choice of tile
// shape and K split.
#include "direct_args.hpp"

#include <algorithm>
#include <cstring>

namespace tal {

int direct_elem(int dk) { return dk == 4 ? 4 : dk == 8 ? 8 : dk == 14 ? 8 : dk == 18 ? 16 : 0; }
int direct_width(int dk) { return dk == 4 ? 4 : dk == 8 || dk == 14 ? 2 : 1; }

DirectForm direct_swapped(const DirectForm &f) {
  DirectForm g = f;
  std::swap(g.M, g.N);
  std::swap(g.m, g.n);
  std::swap(g.sa, g.sb);
  std::swap(g.avol, g.bvol);
  for (DirectDim &d : g.k) std::swap(d.s[0], d.s[1]);
  return g;
}

namespace {

// One number in one tensor: neighbouring dimensions that chain there fused.
bool single_group(const std::vector<DirectDim> &dims, int t, int esz, DirectGroup *g) {
  int64_t ext[kDirectDims];
  g->nd = 0;
  for (const DirectDim &d : dims) {
    if (g->nd > 0 && g->s[g->nd - 1] * ext[g->nd - 1] == d.s[t] * esz) {
      ext[g->nd - 1] *= d.ext;
      continue;
    }
    if (g->nd == kDirectDims) return false;
    ext[g->nd] = d.ext;
    g->s[g->nd++] = d.s[t] * esz;
  }
  if (g->nd == 0) g->nd = 1;
  for (int i = 0; i + 1 < g->nd; ++i) {
    const Divider dv = make_divider((uint32_t)ext[i]);
    g->ext[i] = (uint32_t)ext[i];
    g->mg[i] = dv.magic;
    g->sh[i] = dv.shift;
  }
  return true;
}

bool pair_group(const std::vector<DirectDim> &dims, int esz, DirectPair *g) {
  if ((int)dims.size() > kDirectDims) return false;
  g->nd = std::max<int>(1, (int)dims.size());
  for (size_t i = 0; i < dims.size(); ++i) {
    g->s[0][i] = dims[i].s[0] * esz;
    g->s[1][i] = dims[i].s[1] * esz;
    if (i + 1 == dims.size()) break;
    const Divider dv = make_divider((uint32_t)dims[i].ext);
    g->ext[i] = (uint32_t)dims[i].ext;
    g->mg[i] = dv.magic;
    g->sh[i] = dv.shift;
  }
  return true;
}

// Whether an operand's loads may be `w` elements wide: 16-byte aligned, and
// no vector leaves its contiguous run.  t: the operand's place in k's strides.
bool wide(const std::vector<DirectDim> &rows, const std::vector<DirectDim> &k, int t, bool along_k, int64_t batch_stride,
          int w) {
  if (batch_stride % w) return false;
  const std::vector<DirectDim> &c = along_k ? k : rows, &o = along_k ? rows : k;
  const int tc = along_k ? t : 0, to = along_k ? 0 : t;
  if (c.empty() || c[0].s[tc] != 1) return false;
  // along k the last, partial step is loaded by elements: a single run needs no divisibility
  if (!(along_k && c.size() == 1) && c[0].ext % w) return false;
  for (size_t i = 1; i < c.size(); ++i)
    if (c[i].s[tc] % w) return false;
  for (const DirectDim &d : o)
    if (d.s[to] % w) return false;
  return true;
}

}  // namespace

bool direct_args(const DirectForm &f, int esz, int full_width, int kstep, DirectArgs *a, DirectVariant *v) {
  std::memset(a, 0, sizeof(*a));
  constexpr int64_t kMax = 0x7fffffff - 127;  // a tile past the edge is still numbered in 31 bits
  if (f.M < 1 || f.N < 1 || f.K < 0 || f.batch < 1 || f.M > kMax || f.N > kMax || f.K > kDirectMaxK) return false;
  if (!single_group(f.m, 0, esz, &a->am) || !single_group(f.n, 0, esz, &a->bn) || !single_group(f.m, 1, esz, &a->dm) ||
      !single_group(f.n, 1, esz, &a->dn) || !pair_group(f.k, esz, &a->k))
    return false;
  a->am1 = a->am.s[0];
  a->bn1 = a->bn.s[0];
  a->dm1 = a->dm.s[0];
  a->dn1 = a->dn.s[0];
  a->ka1 = a->k.s[0][0];
  a->kb1 = a->k.s[1][0];
  // D is stored along the number that holds its contiguous index
  const bool along_n = !(!f.m.empty() && f.m[0].s[1] == 1) && !f.n.empty() && f.n[0].s[1] == 1;
  a->flags = (a->am.nd > 1 ? kDirectGroupA : 0) | (a->bn.nd > 1 ? kDirectGroupB : 0) |
             (a->dm.nd > 1 ? kDirectGroupDm : 0) | (a->dn.nd > 1 ? kDirectGroupDn : 0) |
             (along_n ? kDirectAlongN : 0);
  a->M = (int32_t)f.M;
  a->N = (int32_t)f.N;
  a->K = (int32_t)f.K;
  a->sa = f.sa * esz;
  a->sb = f.sb * esz;
  a->sd = f.sd * esz;
  v->ka = !f.k.empty() && f.k[0].s[0] == 1;
  v->kb = !f.k.empty() && f.k[0].s[1] == 1;
  v->width = wide(f.m, f.k, 0, v->ka, f.batch > 1 ? f.sa : 0, full_width) &&
                     wide(f.n, f.k, 1, v->kb, f.batch > 1 ? f.sb : 0, full_width)
                 ? full_width
                 : 1;
  // 32-bit addressing of the operands: whole ones from their first element,
  // or, where a tile's origin can go into the 64-bit base (one dimension in
  // both numbers), a tile's rows over one K step; else, with one dimension in
  // both, a 64-bit address per load: k 64 MiB apart or more (8.4 million rows
  // of R8), or 128 rows that span 2 GiB (2.1 million contracted indices)
  const int64_t abytes = f.avol * esz, bbytes = f.bvol * esz;
  const bool small = abytes < (int64_t)kOutside && bbytes < (int64_t)kOutside;
  auto reach = [&](const DirectGroup &g, int64_t rows, int64_t kstride, int64_t bytes) {
    if (bytes < (int64_t)kOutside) return true;
    if (a->k.nd > 1 || g.nd > 1) return false;
    return (std::min<int64_t>(rows, 128) - 1) * g.s[0] + 32 * kstride + 64 * esz < (int64_t)kOutside;
  };
  // loads of rows past the edge: what is added to kOutside stays below 2^31
  if (!reach(a->am, f.M, a->ka1, abytes) || !reach(a->bn, f.N, a->kb1, bbytes) ||
      32 * a->ka1 >= (int64_t)kOutside || 32 * a->kb1 >= (int64_t)kOutside) {
    v->mode = 3;
    return a->k.nd == 1 && a->am.nd == 1 && a->bn.nd == 1;
  }
  // Mode 1 puts the way to a step's next run into the base where it is
  // negative, and gives it back in the offsets of the lanes before the crossing:
  // up to |way| beyond the operand's own span.  Where that could leave the range
  // (or, past the edge, wrap round into it), offsets go by table: they are those
  // in the operand.
  auto walks = [&](const DirectGroup &g, bool grouped, const std::vector<DirectDim> &rows, int64_t nrows, int t) {
    int64_t span = (int64_t)(kstep - 1) * a->k.s[t][0] + 16, way = 0;
    if (!grouped) span += (std::min<int64_t>(nrows, 128) - 1) * g.s[0];
    else
      for (const DirectDim &d : rows) span += (d.ext - 1) * d.s[0] * esz;
    const int64_t past = f.k[0].ext * a->k.s[t][0], next = a->k.s[t][1] - past;
    way = next < 0 ? -next : next;
    if (a->k.nd > 2) {
      const int64_t wrap = a->k.s[t][2] - (f.k[1].ext - 1) * a->k.s[t][1] - past;
      way = std::max(way, wrap < 0 ? -wrap : wrap);
    }
    return span + way < (int64_t)kOutside;
  };
  if (a->k.nd == 1) v->mode = small ? 0 : 1;
  else
    v->mode = a->k.nd <= 3 && f.k[0].ext >= kstep && walks(a->am, a->am.nd > 1, f.m, f.M, 0) &&
                      walks(a->bn, a->bn.nd > 1, f.n, f.N, 1)
                  ? 1
                  : 2;
  return true;
}

bool direct_addressable(const DirectForm &f, int dk, DirectVariant *v) {
  DirectArgs a;
  if (f.K > kDirectMaxK) {
    if (f.k.size() != 1) return false;
    DirectForm g = f;
    g.K = g.k[0].ext = kDirectMaxK;
    return direct_addressable(g, dk, v);
  }
  return direct_args(f, direct_elem(dk), direct_width(dk), 16, &a, v);
}

const DirectTile *direct_tiles(int dk) {
  // unit: 256 tiles of K = 1024 on 256 CUs; stream: products of 4096^3 (complex 2048^3)
  static const DirectTile r8[kDirectTiles] = {
      {128, 128, 16, 133, 119}, {64, 64, 16, 38.5, 32}, {64, 32, 16, 24, 17.3}, {32, 32, 16, 13, 9.4}};
  static const DirectTile r4[kDirectTiles] = {
      {128, 128, 16, 76, 63}, {64, 64, 32, 18.5, 16.3}, {64, 32, 32, 12.5, 8.4}, {32, 32, 32, 5.6, 4.5}};
  static const DirectTile c8[kDirectTiles] = {
      {64, 64, 16, 139, 127}, {64, 64, 16, 139, 127}, {64, 32, 8, 86, 66}, {32, 32, 8, 48, 33}};
  static const DirectTile c4[kDirectTiles] = {
      {64, 64, 16, 77.5, 64}, {64, 64, 16, 77.5, 64}, {64, 32, 16, 56, 34}, {32, 32, 16, 29.4, 18}};
  return dk == 8 ? r8 : dk == 4 ? r4 : dk == 18 ? c8 : c4;
}

// Every tile shape is tried, both ways round.  A CU that gets u tiles (u may
// be a fraction where tiles are split along K) takes max(unit, u * stream)
// per 1024 of K.  The tiles that do not fill a last round over the CUs are cut
// into ksplit ranges of K, which costs the partial sums' way through memory
// and a second launch (about 5 us).
DirectChoice direct_choose(int dk, int64_t M, int64_t N, int64_t K, int64_t batch, int cus) {
  const DirectTile *tiles = direct_tiles(dk);
  const int esz = direct_elem(dk);
  K = std::min(K, kDirectMaxK);  // of the first of several launches
  DirectChoice best;
  best.us = -1;  // stays where every tile shape makes too many
  for (int swap = 0; swap < 2; ++swap) {
    const int64_t m = swap ? N : M, n = swap ? M : N;
    for (int t = 0; t < kDirectTiles; ++t) {
      const DirectTile &ti = tiles[t];
      if (swap && ti.bm == ti.bn) continue;
      const int64_t gx = (m + ti.bm - 1) / ti.bm, gy = (n + ti.bn - 1) / ti.bn, T = gx * gy;
      const int64_t nk = std::max<int64_t>(1, (K + ti.kb - 1) / ti.kb);
      const double k = (double)nk * ti.kb / 1024;
      if (T > 0x7fffffff - 64 * (int64_t)cus) continue;  // units are numbered in 31 bits, K ranges of `rem` < cus tiles included
      auto consider = [&](int64_t whole, int64_t rem, int ks, int64_t steps, double us, size_t bytes) {
        if (best.us >= 0 && us >= best.us) return;
        best.swap = swap != 0;
        best.tile = t;
        best.gx = gx;
        best.gy = gy;
        best.whole = whole;
        best.rem = rem;
        best.ksplit = ks;
        best.ksteps = (int)steps;
        best.us = us;
        best.part_bytes = bytes;
      };
      const int64_t all = T * batch;
      const double u = (double)((all + cus - 1) / cus);
      consider(T, 0, 1, nk, std::max(ti.unit, u * ti.stream) * k, 0);
      if (batch != 1) continue;
      const int64_t rem = T % cus, whole = T - rem;
      if (rem == 0) continue;
      for (int want = 2; want <= 64; want += want < 8 ? 1 : want < 16 ? 2 : 8) {
        const int64_t steps = (nk + want - 1) / want, ks = (nk + steps - 1) / steps;
        if (ks < 2 || steps < 2) continue;
        const double part = (double)steps / nk;  // of a tile's K
        const double us = (double)(whole / cus) + (double)((rem * ks + cus - 1) / cus) * part;
        const double one = whole ? ti.unit : ti.unit * part;
        const size_t bytes = (size_t)rem * ks * ti.bm * ti.bn * esz;
        if (bytes > kSumsBytes) continue;
        consider(whole, rem, (int)ks, steps, std::max(one, us * ti.stream) * k + 5.0 + 2.0 * bytes / 3.5e6, bytes);
      }
    }
  }
  return best;
}

}  // namespace tal
