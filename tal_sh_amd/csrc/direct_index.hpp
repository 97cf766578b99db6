// Index groups of the direct contraction kernel (direct_kernel.hpp), shared by
// the device code, the host that fills its arguments (direct.cpp) and the CPU
// tests, so that every address the kernel forms comes from the functions below.
//
// The kernel computes D(m, n) (+)= alpha * sum_k A(m, k) * B(k, n), where m, n
// and k are mixed-radix numbers over tensor dimensions: the offset of m in A is
// the sum of its digits times A's strides, and so on.  Each (number, tensor)
// pair has its own group, with the dimensions that chain in that tensor fused,
// so a number that is linear in a tensor needs no division.
#pragma once

#include <cstdint>

#include "batch_item.hpp"
#include "direct_form.hpp"

// Inlined before anything else is done, so that the kernel's arguments stay scalar loads.
#define TAL_INLINE __attribute__((always_inline))

namespace tal {

// Digits x -> (d0, ..., d[nd-1]) over ext[0..nd-2], the last digit unbounded.
struct DirectGroup {
  int32_t nd;
  uint32_t ext[kDirectDims - 1], mg[kDirectDims - 1], sh[kDirectDims - 1];
  int64_t s[kDirectDims];  // byte strides
};
// k over the dimensions it has in both operands (strides below 2^31 bytes when nd > 1).
struct DirectPair {
  int32_t nd;
  uint32_t ext[kDirectDims - 1], mg[kDirectDims - 1], sh[kDirectDims - 1];
  int64_t s[2][kDirectDims];
};

// Byte offset of x: 64-bit (D), and 32-bit for operands shorter than kOutside bytes.
TAL_HD TAL_INLINE inline int64_t group_offset64(const DirectGroup &g, uint32_t x) {
  int64_t o = 0;
#if defined(__HIPCC__)
#pragma unroll
#endif
  for (int i = 0; i + 1 < kDirectDims; ++i) {
    if (i + 1 >= g.nd) return o + (int64_t)x * g.s[i];
    const uint32_t q = divide(x, g.mg[i], g.sh[i]);
    o += (int64_t)(x - q * g.ext[i]) * g.s[i];
    x = q;
  }
  return o + (int64_t)x * g.s[kDirectDims - 1];
}
TAL_HD TAL_INLINE inline uint32_t group_offset32(const DirectGroup &g, uint32_t x) {
  uint32_t o = 0;
#if defined(__HIPCC__)
#pragma unroll
#endif
  for (int i = 0; i + 1 < kDirectDims; ++i) {
    if (i + 1 >= g.nd) return o + x * (uint32_t)g.s[i];
    const uint32_t q = divide(x, g.mg[i], g.sh[i]);
    o += (x - q * g.ext[i]) * (uint32_t)g.s[i];
    x = q;
  }
  return o + x * (uint32_t)g.s[kDirectDims - 1];
}
TAL_HD TAL_INLINE inline void pair_offsets32(const DirectPair &g, uint32_t x, uint32_t *oa, uint32_t *ob) {
  uint32_t a = 0, b = 0;
#if defined(__HIPCC__)
#pragma unroll
#endif
  for (int i = 0; i + 1 < kDirectDims; ++i) {
    if (i + 1 >= g.nd) {
      *oa = a + x * (uint32_t)g.s[0][i];
      *ob = b + x * (uint32_t)g.s[1][i];
      return;
    }
    const uint32_t q = divide(x, g.mg[i], g.sh[i]), d = x - q * g.ext[i];
    a += d * (uint32_t)g.s[0][i];
    b += d * (uint32_t)g.s[1][i];
    x = q;
  }
  *oa = a + x * (uint32_t)g.s[0][kDirectDims - 1];
  *ob = b + x * (uint32_t)g.s[1][kDirectDims - 1];
}

// Walking k in steps no longer than its leading run, k of up to three
// dimensions (or one).  next / wrap: how much further on than the position
// just past a run's end the next run starts in A and B, where the second
// dimension goes on / wraps; direct_args lets only those walk whose ways, with
// what the lanes add, stay within 32-bit offsets.
struct RunWalk {
  int32_t e0;
  int32_t next[2], wrap[2];
};
TAL_HD TAL_INLINE inline RunWalk run_walk(const DirectPair &g) {
  RunWalk w;
  w.e0 = g.nd > 1 ? (int32_t)g.ext[0] : 0x7fffffff;
  for (int t = 0; t < 2; ++t) {
    const int64_t past = g.nd > 1 ? (int64_t)g.ext[0] * g.s[t][0] : 0;
    w.next[t] = g.nd > 1 ? (int32_t)(g.s[t][1] - past) : 0;
    w.wrap[t] = g.nd > 2 ? (int32_t)(g.s[t][2] - (int64_t)(g.ext[1] - 1) * g.s[t][1] - past) : 0;
  }
  return w;
}
// Offsets of k, its place r in its run and the run's digit in the second dimension.
TAL_HD TAL_INLINE inline void run_start(const DirectPair &g, int k, int64_t *oa, int64_t *ob, int *r, int *d1) {
  if (g.nd == 1) {
    *oa = (int64_t)k * g.s[0][0];
    *ob = (int64_t)k * g.s[1][0];
    *r = *d1 = 0;  // never reaches the run's end
    return;
  }
  const uint32_t q = divide((uint32_t)k, g.mg[0], g.sh[0]);
  const uint32_t y = g.nd > 2 ? divide(q, g.mg[1], g.sh[1]) : 0;
  *r = (int)((uint32_t)k - q * g.ext[0]);
  *d1 = (int)(g.nd > 2 ? q - y * g.ext[1] : q);
  *oa = (int64_t)*r * g.s[0][0] + (int64_t)*d1 * g.s[0][1] + (int64_t)y * g.s[0][2];
  *ob = (int64_t)*r * g.s[1][0] + (int64_t)*d1 * g.s[1][1] + (int64_t)y * g.s[1][2];
}

// Offset tables of contracted indices: two halves of `half` entries, in which
// half h of a K range takes the place of half h - 2.  The walk has advanced to
// step offset `at` of a range of `len` (steps of kb): the half to fill now, or
// -1.  Between two calls lies a barrier, but none within one, so the half that
// is written over must be one that no wave reads any more in this call.  A
// kernel that reads a step's entries a call ahead has read the last ones of
// half h - 1 in the call before it comes to half h; one that reads them in the
// call that uses them reads those in the very call that comes to half h, and
// fills one call later.
TAL_HD TAL_INLINE inline int table_refill(int at, int len, int kb, int half, bool ahead) {
  const int h = at / half;
  if (h < 1 || at % half != (ahead ? 0 : kb) || (h + 1) * half >= len) return -1;
  return h + 1;
}

// Arguments of one launch.  Byte strides and sizes throughout.  What every
// launch reads comes first; a group is read only where its flag says that the
// number has more than one dimension in that tensor (kernel arguments come
// from memory far away: each line of them costs a workgroup about a
// microsecond before its first load).
enum DirectFlags {
  kDirectBeta = 1,    // D is accumulated
  kDirectConjA = 2, kDirectConjB = 4,
  kDirectAlongN = 8,  // D is stored along n (its contiguous index is an n index), else along m
  kDirectGroupA = 16, kDirectGroupB = 32, kDirectGroupDm = 64, kDirectGroupDn = 128,
  kDirectCuShift = 8  // from this bit on: log2 of the GPU's compute units (a power of two in every partition mode)
};
struct DirectArgs {
  const void *A, *B;
  void *D, *part;
  int32_t M, N, K, flags;
  int32_t gx, gy;               // tiles along m and n
  int32_t whole;                // tiles [0, whole) take all of K, one workgroup each
  int32_t rem, ksplit, ksteps;  // the rem tiles after them are cut into ksplit ranges of ksteps K steps
  int32_t first;                // unit of the launch's first workgroup (a grid holds fewer than 2^32 threads)
  int32_t pad0;
  int64_t am1, bn1, dm1, dn1;   // strides of m and n where they have one dimension
  int64_t ka1, kb1;             // strides of k's first dimension
  double ar, ai;
  int64_t sa, sb, sd;           // batch strides (grid.y)
  DirectPair k;                 // k in A and B
  DirectGroup am, bn;           // m in A, n in B
  DirectGroup dm, dn;           // m and n in D
};

TAL_HD TAL_INLINE inline int64_t d_row(const DirectArgs &p, int m) {
  return p.flags & kDirectGroupDm ? group_offset64(p.dm, (uint32_t)m) : (int64_t)m * p.dm1;
}
TAL_HD TAL_INLINE inline int64_t d_col(const DirectArgs &p, int n) {
  return p.flags & kDirectGroupDn ? group_offset64(p.dn, (uint32_t)n) : (int64_t)n * p.dn1;
}

}  // namespace tal
