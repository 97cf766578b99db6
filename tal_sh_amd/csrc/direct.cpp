// Launch of the direct contraction kernels.
#include "direct.hpp"

#include <algorithm>

namespace tal {

namespace {

int device_cus() {
  static int cache[64] = {0};
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cache[dev]) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) return 256;
    cache[dev] = cus;
  }
  return cache[dev];
}

}  // namespace

// A call asks several times for its product's choice: the last one is kept per thread.
DirectChoice direct_choose(int dk, int64_t M, int64_t N, int64_t K, int64_t batch) {
  struct Last {
    int dk = 0, cus = 0;
    int64_t m = 0, n = 0, k = 0, b = 0;
    DirectChoice c;
  };
  static thread_local Last l;
  const int cus = device_cus();
  if (l.dk != dk || l.cus != cus || l.m != M || l.n != N || l.k != K || l.b != batch) {
    l.c = direct_choose(dk, M, N, K, batch, cus);
    l.dk = dk, l.cus = cus, l.m = M, l.n = N, l.k = K, l.b = batch;
  }
  return l.c;
}

int launch_direct(int dk, const DirectForm &f, const void *A, const void *B, void *D, double ar, double ai, bool conja,
                  bool conjb, bool accumulate, void *sums, hipStream_t s) {
  const int esz = direct_elem(dk);
  if (!esz || !A || !B || !D) return -1;
  if (f.K > kDirectMaxK) {
    if (f.k.size() != 1) return -4;
    DirectForm g = f;
    for (int64_t k0 = 0; k0 < f.K; k0 += g.K) {
      g.K = g.k[0].ext = std::min(kDirectMaxK, f.K - k0);
      if (int e = launch_direct(dk, g, (const char *)A + k0 * f.k[0].s[0] * esz, (const char *)B + k0 * f.k[0].s[1] * esz,
                                D, ar, ai, conja, conjb, accumulate || k0 > 0, sums, s))
        return e;
    }
    return 0;
  }
  DirectChoice c = direct_choose(dk, f.M, f.N, f.K, f.batch);
  if (c.part_bytes && !sums) {  // no room for partial sums: whole tiles
    c.whole = c.gx * c.gy;
    c.rem = 0;
    c.ksplit = 1;
    c.ksteps = 0;
  }
  if (c.us < 0) return -4;  // more tiles than 31 bits number
  DirectForm swapped;
  const DirectForm *p = &f;
  if (c.swap) {
    swapped = direct_swapped(f);
    p = &swapped;
    std::swap(A, B);
    std::swap(conja, conjb);
  }
  DirectArgs a;
  DirectVariant v;
  if (!direct_args(*p, esz, direct_width(dk), direct_tiles(dk)[c.tile].kb, &a, &v)) return -4;
  a.gx = (int32_t)c.gx;
  a.gy = (int32_t)c.gy;
  a.whole = (int32_t)c.whole;
  a.rem = (int32_t)c.rem;
  a.ksplit = c.ksplit;
  a.ksteps = c.ksteps;
  a.ar = ar;
  a.ai = ai;
  a.part = sums;
  for (int cus = device_cus(); cus > 1; cus >>= 1) a.flags += 1 << kDirectCuShift;
  a.flags |= (accumulate ? kDirectBeta : 0) | (conja ? kDirectConjA : 0) | (conjb ? kDirectConjB : 0);
  const DirectLaunch launch =
      dk == 8 ? direct_launch_r8 : dk == 4 ? direct_launch_r4 : dk == 18 ? direct_launch_c8 : direct_launch_c4;
  for (int64_t b0 = 0; b0 < f.batch; b0 += 65535) {  // batch entries go to grid.y, at most 65535 per launch
    a.A = (const char *)A + b0 * a.sa;
    a.B = (const char *)B + b0 * a.sb;
    a.D = (char *)D + b0 * a.sd;
    if (!launch(c.tile, v, a, (unsigned)std::min<int64_t>(65535, f.batch - b0), s)) return -4;
  }
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace tal
