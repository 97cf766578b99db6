// C entry points over the planning of direct contractions (tal_sh_amd/csrc/
// plan.cpp and direct_args.cpp) for the CPU test tests/test_direct_plan.py,
// which builds this file with g++.
//
// direct_check plans a contraction and evaluates it element by element with
// the addresses the kernel would form (direct_index.hpp), walking k in the
// kernel's steps, and compares it with the pattern's own loop nest.
#include <cstdint>
#include <cstring>
#include <vector>

#include "direct_args.hpp"
#include "plan.hpp"

using namespace tal;

namespace {

std::vector<int64_t> dlf(int rank, const int *dims) {
  std::vector<int64_t> s(rank);
  int64_t a = 1;
  for (int i = 0; i < rank; ++i) {
    s[i] = a;
    a *= dims[i];
  }
  return s;
}
int64_t volume(int rank, const int *dims) {
  int64_t v = 1;
  for (int i = 0; i < rank; ++i) v *= dims[i];
  return v;
}
int64_t value(int64_t i, int seed) { return (i * 2654435761LL + seed * 40503) % 17 - 8; }

std::vector<int64_t> permuted(const std::vector<int64_t> &x, int rank, const int *dims, const std::vector<int> &o2n) {
  std::vector<int> od(rank);
  for (int i = 0; i < rank; ++i) od[o2n[i]] = dims[i];
  const std::vector<int64_t> os = dlf(rank, od.data());
  std::vector<int64_t> y(x.size());
  for (int64_t e = 0; e < (int64_t)x.size(); ++e) {
    int64_t r = e, o = 0;
    for (int i = 0; i < rank; ++i) {
      o += (r % dims[i]) * os[o2n[i]];
      r /= dims[i];
    }
    y[o] = x[e];
  }
  return y;
}

}  // namespace

extern "C" {

// form 0: straight from the tensors; 1: on the transposed copies.  kstep: the
// kernel's K step.  swap: A and B exchanged.  info: [mode, width, ka, kb].
// Returns 0 when every element agrees, -1 when the form is not available,
// positive codes for the first disagreement.
int direct_check(const char *pattern, const int *ddims, const int *ldims, const int *rdims, int dk, int form,
                 int kstep, int swap, int *info) {
  DigitalPattern p;
  ContractPlan plan;
  if (parse_pattern(pattern, &p) || plan_contraction(p, ddims, ldims, rdims, 1, &plan)) return 1;
  if (form == 0 && !plan.direct_ok) return -1;
  std::vector<int64_t> L(volume(p.lrank, ldims)), R(volume(p.rrank, rdims)), D(volume(p.drank, ddims), 0);
  for (size_t i = 0; i < L.size(); ++i) L[i] = value((int64_t)i, 1);
  for (size_t i = 0; i < R.size(); ++i) R[i] = value((int64_t)i, 2);
  // the pattern's loop nest: D indices and contracted pairs
  const std::vector<int64_t> ds = dlf(p.drank, ddims), ls = dlf(p.lrank, ldims), rs = dlf(p.rrank, rdims);
  struct Index {
    int64_t ext, d, l, r;
  };
  std::vector<Index> idx(p.drank);
  for (int i = 0; i < p.drank; ++i) idx[i] = Index{ddims[i], ds[i], 0, 0};
  for (int i = 0; i < p.lrank; ++i) {
    const int c = p.dig[i];
    if (c > 0) idx[c - 1].l += ls[i];
    else idx.push_back(Index{ldims[i], 0, ls[i], rs[-c - 1]});
  }
  for (int j = 0; j < p.rrank; ++j)
    if (p.dig[p.lrank + j] > 0) idx[p.dig[p.lrank + j] - 1].r += rs[j];
  int64_t total = 1;
  for (const Index &x : idx) total *= x.ext;
  std::vector<int64_t> want(D.size(), 0);
  for (int64_t e = 0; e < total; ++e) {
    int64_t q = e, od = 0, ol = 0, orr = 0;
    for (const Index &x : idx) {
      const int64_t v = q % x.ext;
      q /= x.ext;
      od += v * x.d;
      ol += v * x.l;
      orr += v * x.r;
    }
    want[od] += L[ol] * R[orr];
  }
  // operands of the form
  std::vector<int64_t> A = L, B = R, C = D;
  DirectForm f = plan.direct;
  if (form == 1) {
    const std::vector<int64_t> &X = plan.swap ? R : L, &Y = plan.swap ? L : R;
    const int xr = plan.swap ? p.rrank : p.lrank, yr = plan.swap ? p.lrank : p.rrank;
    A = plan.a.transpose ? permuted(X, xr, plan.swap ? rdims : ldims, plan.a.o2n) : X;
    B = plan.b.transpose ? permuted(Y, yr, plan.swap ? ldims : rdims, plan.b.o2n) : Y;
    f = plan.mat;
  }
  if (swap) {
    f = direct_swapped(f);
    A.swap(B);
  }
  const int esz = direct_elem(dk);
  DirectArgs a;
  DirectVariant v;
  if (!direct_args(f, esz, direct_width(dk), kstep, &a, &v)) return -1;
  info[0] = v.mode;
  info[1] = v.width;
  info[2] = v.ka;
  info[3] = v.kb;
  auto row = [&](bool grouped, const DirectGroup &g, int64_t one, int64_t x) {
    return grouped ? (int64_t)group_offset32(g, (uint32_t)x) : x * one;
  };
  for (int64_t b = 0; b < f.batch; ++b) {
    const int64_t ab = b * a.sa, bb = b * a.sb, db = b * a.sd;
    for (int64_t m = 0; m < f.M; ++m) {
      const int64_t am = row(a.flags & kDirectGroupA, a.am, a.am1, m);
      for (int64_t n = 0; n < f.N; ++n) {
        const int64_t bn = row(a.flags & kDirectGroupB, a.bn, a.bn1, n);
        int64_t sum = 0, oa = 0, ob = 0;
        RunWalk w = run_walk(a.k);
        int kr = 0, kd1 = 0;
        if (v.mode == 1) run_start(a.k, 0, &oa, &ob, &kr, &kd1);
        const int64_t whole = f.K / kstep * kstep;
        for (int64_t k0 = 0; k0 < f.K; k0 += kstep) {
          const bool wrap = a.k.nd > 2 && kd1 + 1 == (int)a.k.ext[1];
          const int da = wrap ? w.wrap[0] : w.next[0], dbk = wrap ? w.wrap[1] : w.next[1], cross = w.e0 - kr;
          for (int64_t k = k0; k < f.K && k < k0 + kstep; ++k) {
            int64_t ka, kb;
            if (v.mode == 0) {
              ka = k * a.ka1;
              kb = k * a.kb1;
            } else if (v.mode == 1 && k0 < whole) {
              const int64_t kk = k - k0;
              ka = oa + kk * a.ka1 + (kk >= cross ? da : 0);
              kb = ob + kk * a.kb1 + (kk >= cross ? dbk : 0);
            } else {
              uint32_t x, y;
              pair_offsets32(a.k, (uint32_t)k, &x, &y);
              ka = x;
              kb = y;
            }
            const int64_t ea = ab + am + ka, eb = bb + bn + kb;
            if (ea < 0 || eb < 0 || ea % esz || eb % esz || ea / esz >= (int64_t)A.size() || eb / esz >= (int64_t)B.size())
              return 2;
            // a wide load along k: its elements are neighbours in memory
            if (v.width > 1 && k0 < whole && (k - k0) % v.width) {
              uint32_t x0, y0, x1, y1;
              pair_offsets32(a.k, (uint32_t)(k - 1), &x0, &y0);
              pair_offsets32(a.k, (uint32_t)k, &x1, &y1);
              if ((v.ka && x1 != x0 + esz) || (v.kb && y1 != y0 + esz)) return 3;
            }
            if (v.width > 1 && ((v.ka && k == k0 && ea % 16) || (!v.ka && m % v.width == 0 && ea % 16))) return 4;
            sum += A[ea / esz] * B[eb / esz];
          }
          if (v.mode == 1 && k0 + 2 * kstep <= f.K) {
            const bool over = kr + kstep >= w.e0;
            oa += (int64_t)kstep * a.ka1 + (over ? da : 0);
            ob += (int64_t)kstep * a.kb1 + (over ? dbk : 0);
            kr += over ? kstep - w.e0 : kstep;
            kd1 = !over ? kd1 : wrap ? 0 : kd1 + 1;
          }
        }
        // rows of a wide load along m or n
        if (v.width > 1 && !v.ka && m % v.width && am != row(a.flags & kDirectGroupA, a.am, a.am1, m - 1) + esz) return 5;
        if (v.width > 1 && !v.kb && n % v.width && bn != row(a.flags & kDirectGroupB, a.bn, a.bn1, n - 1) + esz) return 5;
        if (v.width > 1 && ((!v.ka && f.M % v.width) || (!v.kb && f.N % v.width))) return 6;
        const int64_t ed = db + d_row(a, (int)m) + d_col(a, (int)n);
        if (ed < 0 || ed % esz || ed / esz >= (int64_t)C.size()) return 7;
        C[ed / esz] += sum;
      }
    }
  }
  std::vector<int64_t> out = C;
  if (form == 1 && plan.d_transpose && !plan.mat_d_in_place)
    out = permuted(C, (int)plan.dprime_dims.size(), plan.dprime_dims.data(), plan.d_back_o2n);
  return std::memcmp(out.data(), want.data(), want.size() * sizeof(int64_t)) ? 8 : 0;
}

// Tile choice: out = [swap, tile, gx, gy, whole, rem, ksplit, ksteps, part bytes].
int direct_choice(int dk, long long M, long long N, long long K, long long batch, int cus, long long *out) {
  const DirectChoice c = direct_choose(dk, M, N, K, batch, cus);
  const DirectTile &t = direct_tiles(dk)[c.tile];
  const long long v[] = {c.swap, c.tile, c.gx, c.gy, c.whole, c.rem, c.ksplit, c.ksteps, (long long)c.part_bytes};
  std::memcpy(out, v, sizeof(v));
  const int64_t m = c.swap ? N : M, n = c.swap ? M : N;
  // every tile once, every K step once
  if (c.gx * t.bm < m || (c.gx - 1) * t.bm >= m || c.gy * t.bn < n || (c.gy - 1) * t.bn >= n) return 1;
  if (c.whole + c.rem != c.gx * c.gy || c.whole < 0 || c.rem < 0) return 2;
  const int64_t nk = (K + t.kb - 1) / t.kb;
  if (c.rem && ((int64_t)c.ksplit * c.ksteps < nk || (int64_t)(c.ksplit - 1) * c.ksteps >= nk)) return 3;
  if (c.rem && (batch != 1 || c.part_bytes != (size_t)c.rem * c.ksplit * t.bm * t.bn * direct_elem(dk))) return 4;
  if (!c.rem && c.part_bytes) return 5;
  return 0;
}

}  // extern "C"
