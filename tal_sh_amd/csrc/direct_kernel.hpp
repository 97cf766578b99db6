// Direct contraction kernel (gfx950): D(m, n) (+)= alpha * sum_k A(m, k) * B(k, n)
// for tensors in any dense layout, m, n and k being groups of tensor indices.
// Replaces the GEMM call of gpu_tensor_block_contract_dlf
// (tensor_algebra_gpu_nvidia.cu:6851-7060, cuBLAS/hipBLAS), its in-house
// fallback gpu_matrix_multiply_tn__ (:2263-2312) and, where an operand or D
// would only be transposed for its sake, the transposes around it.
//
// A workgroup of WM x WN waves computes a BM x BN tile of D (or one of the K
// ranges of it) from 16x16x4 MFMAs:
//   R8/C8: v_mfma_f64_16x16x4_f64   R4/C4: v_mfma_f32_16x16x4_f32
// Complex products are four real MFMAs per step (re += ar*br - ai*bi, im +=
// ar*bi + ai*br); conjugation is a sign put on while staging.  Operand lanes:
// A lane l holds row l % 16, B lane l column l % 16; accumulator register r of
// lane l holds C[4*(l/16)+r][l%16] for f32 and C[4*r+l/16][l%16] for f64.
//
// What bounds it: large products, the matrix cores (75 TFLOP/s at 9216^3 FP64
// with the last round split along K, of 78.6 nominal); products of a few
// tiles per CU, the latency of their K steps; narrow products, memory.  Hence:
//  - K steps of KB are loaded PF steps ahead into registers and staged through
//    two LDS buffers, one barrier per step.  The loads are pinned to the head
//    of the step: left to itself the scheduler sinks them next to their use
//    (1024^3 FP64, 64 x 64 tiles: 56 us with one step in flight, 38-42 with
//    three pinned).  128 x 128 tiles have two workgroups per CU to hide
//    latency and run best with one step in flight.
//  - Each operand keeps the order it has in memory: rows of k for one that is
//    contiguous along k, rows of m (n) otherwise, padded so that fragment
//    reads are free of bank conflicts.  A lane reads KQ consecutive k of a
//    k-contiguous tile at once (16 bytes) and uses them in KQ MFMA steps; the
//    other operand follows the same order of k.  So neither layout is
//    scattered while staging (4096^3 FP64: 72.4 TFLOP/s with both operands
//    contiguous along k, 72.9 with both along their rows; the kernel before
//    this one 65 and 48).
//  - The K loop holds no branch and no bounds check: loads are buffer loads
//    whose range check returns 0 for rows past the edge (offset kOutside), and
//    the last, partial K step is peeled off and loaded element by element.
//  - Tiles that do not fill a last round over the CUs are cut into K ranges in
//    the same launch (direct_choose), their sums added in order by
//    direct_reduce.  Uncut and cut, us: R8 9216^3 21,740 and 20,840, 189 x 278
//    by 147864 (27 tiles) 3,408 and 316, R4 4224 x 4224 by 4096 1,293 and 1,122,
//    C8 1920 x 1848 by 1720 863 and 744.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "direct_index.hpp"

namespace tal {

namespace direct {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// The kernels read their arguments where they lie.  As a by-value parameter
// the compiler keeps a private copy of all of them wherever a branch picks one
// of two groups: 784 bytes of scratch memory a lane, and launches that took
// 17-33 us longer.
__device__ TAL_INLINE inline const DirectArgs &kernel_args() {
  return *(const DirectArgs *)__builtin_amdgcn_kernarg_segment_ptr();
}

template <typename S>
struct Mfma;
template <>
struct Mfma<double> {
  using acc_t = f64x4;
  __device__ static int row(int lane, int r) { return 4 * r + (lane >> 4); }
  __device__ static acc_t op(double a, double b, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
};
template <>
struct Mfma<float> {
  using acc_t = f32x4;
  __device__ static int row(int lane, int r) { return 4 * (lane >> 4) + r; }
  __device__ static acc_t op(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

__device__ inline __amdgpu_buffer_rsrc_t rsrc(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, (int)bytes, 0x00020000);
}

template <int BYTES>
struct Raw;
template <>
struct Raw<4> {
  using type = unsigned int;
  __device__ static type load(__amdgpu_buffer_rsrc_t r, uint32_t o) { return __builtin_amdgcn_raw_buffer_load_b32(r, (int)o, 0, 0); }
};
template <>
struct Raw<8> {
  using type = u32x2;
  __device__ static type load(__amdgpu_buffer_rsrc_t r, uint32_t o) { return __builtin_amdgcn_raw_buffer_load_b64(r, (int)o, 0, 0); }
};
template <>
struct Raw<16> {
  using type = u32x4;
  __device__ static type load(__amdgpu_buffer_rsrc_t r, uint32_t o) { return __builtin_amdgcn_raw_buffer_load_b128(r, (int)o, 0, 0); }
};

template <typename S, int N>
struct Vec {
  S v[N];
};
template <typename S, int N>
__device__ inline Vec<S, N> bload(__amdgpu_buffer_rsrc_t r, uint32_t o) {
  const typename Raw<(int)sizeof(S) * N>::type u = Raw<(int)sizeof(S) * N>::load(r, o);
  Vec<S, N> v;
  __builtin_memcpy(&v, &u, sizeof(v));
  return v;
}
// The same from a 64-bit address in device memory.
template <typename S, int N>
__device__ inline Vec<S, N> gload(const char *a) {
  typedef typename Raw<(int)sizeof(S) * N>::type __attribute__((address_space(1), aligned(sizeof(S)))) G;
  const auto u = *(const G *)(uintptr_t)a;
  Vec<S, N> v;
  __builtin_memcpy(&v, &u, sizeof(v));
  return v;
}
// Tile t of C -> (bx, by): tiles are walked in groups of 8 tile-rows, column
// by column inside a group (a bijection of [0, gx*gy)).
__device__ inline void tile_xy(int t, int gx, int gy, int &bx, int &by) {
  constexpr int G = 8;
  const int group = t / (G * gy), first = group * G;
  const int rows = min(G, gx - first), in = t - group * G * gy;
  bx = first + in % rows;
  by = in / rows;
}

// Unit u of n in dispatch order -> a number such that the units of one XCD
// (workgroups are dealt round-robin over the 8 XCDs) are neighbours: XCD x
// gets the x-th contiguous share (a bijection of [0, n)).
__device__ inline int xcd_order(int u, int n) {
  const int q = n >> 3, r = n & 7, x = u & 7;
  return x * q + min(x, r) + (u >> 3);
}

template <typename S, int NC>
__device__ TAL_INLINE inline void old_values(const char *__restrict__ D, const int64_t (&off)[4], Vec<S, NC> (&d)[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (off[r] >= 0) d[r] = *reinterpret_cast<const Vec<S, NC> *>(D + off[r]);
}

// Values of one 16x16 accumulator block of this lane to D.  Along m (dn = 0):
// the block is turned round through a wave-private LDS patch so that a store
// covers 16 consecutive rows of 4 columns; along n the accumulator layout
// already has 16 consecutive columns of 4 rows.  LDS accesses of one wave
// complete in order, so the patch needs no barrier.
// off[r]: byte offset of the lane's r-th element, negative when it is outside D.
// old: D's values there (beta), read before.
template <typename S, int NC, typename ACC>
__device__ TAL_INLINE inline void emit_block(S *patch, int lane, const ACC (&acc)[NC], bool turn, char *__restrict__ D,
                                             const int64_t (&off)[4], S ar, S ai, bool beta, const Vec<S, NC> (&old)[4]) {
  constexpr int TP = 17;
  const int tl = lane & 15, tg = lane >> 4;
  Vec<S, NC> v[4];
  if (turn) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
#pragma unroll
      for (int r = 0; r < 4; ++r) patch[tl * TP + Mfma<S>::row(lane, r)] = acc[c][r];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r].v[c] = patch[(4 * r + tg) * TP + tl];
      __builtin_amdgcn_wave_barrier();
    }
  } else {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r].v[c] = acc[c][r];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    Vec<S, NC> x;
    if (NC == 1) {
      x.v[0] = ar * v[r].v[0];
    } else {
      const S xr = v[r].v[0], xi = v[r].v[NC - 1];
      x.v[0] = ar * xr - ai * xi;
      x.v[NC - 1] = ar * xi + ai * xr;
    }
    if (beta) {
#pragma unroll
      for (int c = 0; c < NC; ++c) x.v[c] = old[r].v[c] + x.v[c];
    }
    if (off[r] >= 0) *reinterpret_cast<Vec<S, NC> *>(D + off[r]) = x;
  }
}

// D offsets of rows and columns; past the edge, a value whose sum with any offset is negative (|offsets| < 2^62).
constexpr int64_t kNone = -((int64_t)1 << 62);
__device__ TAL_INLINE inline int64_t row_or_none(const DirectArgs &p, int m) { return m < p.M ? d_row(p, m) : kNone; }
__device__ TAL_INLINE inline int64_t col_or_none(const DirectArgs &p, int n) { return n < p.N ? d_col(p, n) : kNone; }

// D offsets of a wave's TM x TN slab, one 16x16 block at a time.
// DN: stored along n.  A template parameter: with indexes that depend on a
// variable the arrays would live in scratch memory.
template <typename S, int SM, int SN, bool DN>
struct SlabOffsets {
  static constexpr int RR = DN ? 4 : 1, CC = DN ? 1 : 4;
  int64_t rows[SM * RR], cols[SN * CC];
  // row(m), col(n): offsets of the slab's m-th row and n-th column
  template <class R, class C>
  __device__ TAL_INLINE SlabOffsets(int lane, R row, C col) {
    const int fl = lane & 15, fg = lane >> 4;
#pragma unroll
    for (int i = 0; i < SM * RR; ++i) rows[i] = row(DN ? (i / RR) * 16 + Mfma<S>::row(lane, i % RR) : i * 16 + fl);
#pragma unroll
    for (int j = 0; j < SN * CC; ++j) cols[j] = col(DN ? j * 16 + fl : (j / CC) * 16 + 4 * (j % CC) + fg);
  }
  __device__ TAL_INLINE void block(int i, int j, int64_t (&off)[4]) const {
#pragma unroll
    for (int r = 0; r < 4; ++r) off[r] = DN ? rows[i * RR + r % RR] + cols[j] : rows[i] + cols[j * CC + r % CC];
  }
};

// KA / KBC: operand A / B is contiguous along k (else along its rows); WA /
// WB: elements per load along that direction.  MODE says how a K step is
// addressed:
//   0  k is linear in both operands: 32-bit offsets advance by a constant
//   1  k starts with a run of at least KB (or an operand is 2 GiB or more): a
//      scalar base per step and, where the step crosses into the next run, one
//      more scalar for the lanes past the crossing
//   2  any k: offsets by table.  The offsets of each row, column and contracted
//      index are worked out once, by one thread, and read from LDS, those of k a
//      step ahead of the loads that use them and with offsets outside the
//      operands past k's end, so that the last, partial step is like the others.
//      Worked out for every load they took 6 KB of code a step, and a small
//      product ran as long as its code took to arrive: 77 x 72 by 60 R8 9.7 ->
//      8.1 us of kernel, 399 x 440 by 195 18.0 -> 13.6 (R4, whose compilation
//      needed scratch memory, 50 -> 14).
//   3  rows and k linear, operands whose rows or contracted indices lie too far
//      apart for 32-bit offsets within a tile: a 64-bit address per load and
//      lane, advanced by a constant. Rows past the edge read the last row again
//      (their products are never stored).
//      R8, in us, by the kernel with 64-bit index arithmetic before and now: 208^3
//      rows by 208 and 208 24,400 -> 18,000, 9,000,000 by 24 and 24 3,090 ->
//      1,460; C8 8,000,000 by 32 and 32 4,990 -> 2,430; R8 130 x 130 by
//      2,200,000 along k, one tile there and cut into K ranges here, 364,000 ->
//      3,300.
template <typename S, int NC, int KA, int KBC, int WA, int WB, int BM, int BN, int KB, int WM, int WN, int PF, int OCC,
          int MODE>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(OCC))) void direct_kernel(DirectArgs) {
  const DirectArgs &p = kernel_args();
  using MF = Mfma<S>;
  using acc_t = typename MF::acc_t;
  constexpr int NT = 64 * WM * WN;
  constexpr int TM = BM / WM, TN = BN / WN, SM = TM / 16, SN = TN / 16;
  constexpr int KQ = sizeof(S) == 8 ? 2 : 4;  // consecutive k per fragment read of a k-contiguous tile
  constexpr int KPAD = KQ, RPAD = sizeof(S) == 8 ? 8 : 4;
  // LDS tiles: [plane][row][k] for a k-contiguous operand, [plane][k][row] otherwise
  constexpr int AL = KA ? BM : KB, AR = KA ? KB + KPAD : BM + RPAD;
  constexpr int BL = KBC ? BN : KB, BR = KBC ? KB + KPAD : BN + RPAD;
  __shared__ __attribute__((aligned(16))) S As[2][NC][AL][AR];
  __shared__ __attribute__((aligned(16))) S Bs[2][NC][BL][BR];
  constexpr int ALINE = (KA ? KB : BM) / WA, BLINE = (KBC ? KB : BN) / WB;
  constexpr int NVA = BM * KB / WA / NT, NVB = BN * KB / WB / NT;
  constexpr int ASTEP = NT / ALINE, BSTEP = NT / BLINE;
  static_assert(NVA >= 1 && NVB >= 1 && NT % ALINE == 0 && NT % BLINE == 0, "tile split");
  static_assert(KB % (4 * KQ) == 0, "fragment depth");

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  // units: the whole tiles, then the K ranges of the others
  int u = p.first + (int)blockIdx.x, tile, kpart = 0;
  const bool part = u >= p.whole;
  if (!part) {
    tile = u = xcd_order(u, p.whole);
  } else {
    // by K range, then by tile: the tiles of one range read the same panels,
    // side by side on an XCD, so its L2 serves them.  A call by tile first and
    // by range first, us: 189 x 278 by 147864 R8 (27 tiles in 56 ranges) 600 and
    // 443, 240 x 264 by 70400 322 and 236, 300 x 400 by 60000 R4 281 and 160; 76
    // x 5254 by 20952, whose tiles share one panel only, 478 and 504.
    u = xcd_order(u - p.whole, p.rem * p.ksplit);
    kpart = u / p.rem;
    tile = u - kpart * p.rem;
    u = tile * p.ksplit + kpart;  // place of the partial sums
    tile += p.whole;
  }
  int bx, by;
  tile_xy(tile, p.gx, p.gy, bx, by);
  const int m0 = bx * BM, n0 = by * BN;
  const int kbeg = kpart * p.ksteps * KB;
  const int kend = part ? min(p.K, kbeg + p.ksteps * KB) : p.K;
  // The second workgroup of each CU gets the matrix cores first: equals, the two
  // go through their K steps together and wait together (4096^3 R4 993 -> 985
  // us, 4026 x 3990 by 3654 982 -> 968, R8 1913 -> 1903; no difference for the
  // smaller tiles, and four levels of priority cost R4 23 %).  Every other round
  // over the CUs is taken to be the second workgroups: so the first two rounds
  // are dealt, later workgroups go where one ended and may meet an equal.
  if (BM * BN == 128 * 128 && (blockIdx.x >> (p.flags >> kDirectCuShift) & 1)) __builtin_amdgcn_s_setprio(1);
  // A number with one dimension in an operand is linear there, and its offset
  // from the tile's origin fits 32 bits (the host checks): the origin goes
  // into the 64-bit base.
  const bool ga = p.flags & kDirectGroupA, gb = p.flags & kDirectGroupB;
  const int am0 = ga ? 0 : m0, bn0 = gb ? 0 : n0;
  const char *abase = (const char *)p.A + (int64_t)blockIdx.y * p.sa + (int64_t)am0 * p.am1;
  const char *bbase = (const char *)p.B + (int64_t)blockIdx.y * p.sb + (int64_t)bn0 * p.bn1;
  if (MODE == 0) {
    abase += (int64_t)kbeg * p.ka1;
    bbase += (int64_t)kbeg * p.kb1;
  }

  // load j of a thread: vector at ac of line al + j * ASTEP (line = row of a
  // k-contiguous operand, else k); a line of 64 or more threads is uniform per wave
  const int ac = (tid % ALINE) * WA, bc = (tid % BLINE) * WB;
  const int al = ALINE % 64 == 0 ? __builtin_amdgcn_readfirstlane(tid / ALINE) : tid / ALINE;
  const int bl = BLINE % 64 == 0 ? __builtin_amdgcn_readfirstlane(tid / BLINE) : tid / BLINE;
  // Mode 2: offsets by table.  Rows, columns and D's of both once; k in two
  // halves of kHalf, one filled while loads read the other.
  constexpr bool TAB = MODE == 2, FAR = MODE == 3;
  constexpr int kHalf = 256;
  static_assert(!TAB || (WA == 1 && WB == 1 && kHalf % KB == 0 && kHalf <= NT && kHalf > (PF + 1) * KB), "tables");
  __shared__ uint32_t arow_t[TAB ? BM : 1], brow_t[TAB ? BN : 1];
  __shared__ int64_t drow_t[TAB ? BM : 1], dcol_t[TAB ? BN : 1];
  __shared__ uint2 k_t[TAB ? 2 * kHalf : 1];
  auto arow = [&](int r) TAL_INLINE -> uint32_t {
    return r >= p.M ? kOutside : ga ? group_offset32(p.am, (uint32_t)r) : (uint32_t)(r - am0) * (uint32_t)p.am1;
  };
  auto brow = [&](int r) TAL_INLINE -> uint32_t {
    return r >= p.N ? kOutside : gb ? group_offset32(p.bn, (uint32_t)r) : (uint32_t)(r - bn0) * (uint32_t)p.bn1;
  };
  auto fill_k = [&](int h) TAL_INLINE {  // half h of this K range; past its end, offsets outside both operands
    if (kHalf == NT || tid < kHalf) {
      const int k = kbeg + h * kHalf + tid;
      uint2 o = make_uint2(kOutside, kOutside);
      if (k < kend) pair_offsets32(p.k, (uint32_t)k, &o.x, &o.y);
      k_t[(h & 1) * kHalf + tid] = o;
    }
  };
  if (TAB) {
    fill_k(0);
    if (kbeg + kHalf < kend) fill_k(1);
    static_assert(!TAB || BM + BN <= NT, "a thread per row and column");
    if (tid < BM) {
      arow_t[tid] = arow(m0 + tid);
      drow_t[tid] = row_or_none(p, m0 + tid);
    } else if (tid < BM + BN) {
      brow_t[tid - BM] = brow(n0 + tid - BM);
      dcol_t[tid - BM] = col_or_none(p, n0 + tid - BM);
    }
    __syncthreads();
  }
  uint32_t aro[KA ? NVA : 1], bro[KBC ? NVB : 1];
  // Mode 3: the address of load j of row r0 (clamped to the operand) and contracted index k.
  auto afar = [&](int j, int k) TAL_INLINE {
    const int r = min(m0 + (KA ? al + j * ASTEP : ac), p.M - (KA ? 1 : WA));
    return (const char *)p.A + (int64_t)blockIdx.y * p.sa + (int64_t)r * p.am1 + (int64_t)k * p.ka1;
  };
  auto bfar = [&](int j, int k) TAL_INLINE {
    const int r = min(n0 + (KBC ? bl + j * BSTEP : bc), p.N - (KBC ? 1 : WB));
    return (const char *)p.B + (int64_t)blockIdx.y * p.sb + (int64_t)r * p.bn1 + (int64_t)k * p.kb1;
  };
  const char *af[FAR ? NVA : 1], *bf[FAR ? NVB : 1];
  if (FAR) {
#pragma unroll
    for (int j = 0; j < NVA; ++j) af[FAR ? j : 0] = afar(j, kbeg + (KA ? ac : al + j * ASTEP));
#pragma unroll
    for (int j = 0; j < NVB; ++j) bf[FAR ? j : 0] = bfar(j, kbeg + (KBC ? bc : bl + j * BSTEP));
  } else {
#pragma unroll
    for (int j = 0; j < (KA ? NVA : 1); ++j) {
      const int r = KA ? al + j * ASTEP : ac;
      aro[j] = TAB ? arow_t[r] : arow(m0 + r);
    }
#pragma unroll
    for (int j = 0; j < (KBC ? NVB : 1); ++j) {
      const int r = KBC ? bl + j * BSTEP : bc;
      bro[j] = TAB ? brow_t[r] : brow(n0 + r);
    }
  }

  Vec<S, WA * NC> ra[PF][NVA];
  Vec<S, WB * NC> rb[PF][NVB];
  uint32_t av[NVA], bv[NVB];
  if (MODE < 2) {
#pragma unroll
    for (int j = 0; j < NVA; ++j) av[j] = aro[KA ? j : 0] + (uint32_t)(KA ? ac : al + j * ASTEP) * (uint32_t)p.ka1;
#pragma unroll
    for (int j = 0; j < NVB; ++j) bv[j] = bro[KBC ? j : 0] + (uint32_t)(KBC ? bc : bl + j * BSTEP) * (uint32_t)p.kb1;
  }
  // mode 1: the leading run's extent, the offset from past its end to the next
  // run (also where the second dimension wraps), k's place in its run and run's digit
  RunWalk rw;
  int kr = 0, kd1 = 0;
  if (MODE == 1) {
    rw = run_walk(p.k);
    int64_t oa, ob;
    run_start(p.k, kbeg, &oa, &ob, &kr, &kd1);
    abase += oa;
    bbase += ob;
  }
  // What the K loop needs of the arguments, held in scalar registers: read again
  // in the loop, they come with branches around the loads (4096^3 R4 987 -> 1013 us).
  uint32_t astep = KB * (uint32_t)p.ka1, bstep = KB * (uint32_t)p.kb1;
  int64_t abase_step = KB * p.ka1, bbase_step = KB * p.kb1;
  uint32_t kext1 = MODE == 1 ? p.k.ext[1] : 0;
  asm volatile("" : "+s"(astep), "+s"(bstep), "+s"(abase_step), "+s"(bbase_step), "+s"(kext1));
  // The next whole K step into a register set.  Past the last whole step the
  // same step is loaded again and never multiplied.
  int kload = kbeg;
  // mode 2: the table's offsets for the step at kload, read a step ahead of
  // their use (but by 128 x 128 tiles, which have no registers for that)
  constexpr bool AHEAD = BM * BN < 128 * 128;
  auto next_k = [&]() TAL_INLINE {
    const uint2 *t = k_t + ((kload - kbeg) & (2 * kHalf - 1));
#pragma unroll
    for (int j = 0; j < NVA; ++j) av[j] = t[KA ? ac : al + j * ASTEP].x;
#pragma unroll
    for (int j = 0; j < NVB; ++j) bv[j] = t[KBC ? bc : bl + j * BSTEP].y;
  };
  if (TAB && AHEAD) next_k();
  auto load = [&](int set) TAL_INLINE {
    const bool more = kload + 2 * KB <= kend;
    if (MODE == 0) {
      const auto rsa = rsrc(abase, kOutside), rsb = rsrc(bbase, kOutside);
#pragma unroll
      for (int j = 0; j < NVA; ++j) ra[set][j] = bload<S, WA * NC>(rsa, av[j]);
#pragma unroll
      for (int j = 0; j < NVB; ++j) rb[set][j] = bload<S, WB * NC>(rsb, bv[j]);
      const uint32_t sa = more ? astep : 0, sb = more ? bstep : 0;
#pragma unroll
      for (int j = 0; j < NVA; ++j) av[j] += sa;
#pragma unroll
      for (int j = 0; j < NVB; ++j) bv[j] += sb;
    } else if (MODE == 1) {
      const bool wrap = kd1 + 1 == (int)kext1;
      const int da = wrap ? rw.wrap[0] : rw.next[0], db = wrap ? rw.wrap[1] : rw.next[1];
      const int cross = rw.e0 - kr;  // the step's elements from here on are in the next run: da / db further on
      const auto rsa = rsrc(abase + min(da, 0), kOutside), rsb = rsrc(bbase + min(db, 0), kOutside);
      const uint32_t a0 = (uint32_t)max(-da, 0), a1 = (uint32_t)max(da, 0);
      const uint32_t b0 = (uint32_t)max(-db, 0), b1 = (uint32_t)max(db, 0);
#pragma unroll
      for (int j = 0; j < NVA; ++j)
        ra[set][j] = bload<S, WA * NC>(rsa, av[j] + ((KA ? ac : al + j * ASTEP) >= cross ? a1 : a0));
#pragma unroll
      for (int j = 0; j < NVB; ++j)
        rb[set][j] = bload<S, WB * NC>(rsb, bv[j] + ((KBC ? bc : bl + j * BSTEP) >= cross ? b1 : b0));
      const bool over = kr + KB >= rw.e0;
      if (more) {
        abase += abase_step + (over ? da : 0);
        bbase += bbase_step + (over ? db : 0);
        kr += over ? KB - rw.e0 : KB;
        kd1 = !over ? kd1 : wrap ? 0 : kd1 + 1;
      }
    } else if (FAR) {
#pragma unroll
      for (int j = 0; j < NVA; ++j) ra[set][j] = gload<S, WA * NC>(af[FAR ? j : 0]);
#pragma unroll
      for (int j = 0; j < NVB; ++j) rb[set][j] = gload<S, WB * NC>(bf[FAR ? j : 0]);
      const int64_t sa = more ? abase_step : 0, sb = more ? bbase_step : 0;
#pragma unroll
      for (int j = 0; j < NVA; ++j) af[FAR ? j : 0] += sa;
#pragma unroll
      for (int j = 0; j < NVB; ++j) bf[FAR ? j : 0] += sb;
    } else {
      const auto rsa = rsrc(abase, kOutside), rsb = rsrc(bbase, kOutside);
      if (!AHEAD) next_k();
#pragma unroll
      for (int j = 0; j < NVA; ++j) ra[set][j] = bload<S, WA * NC>(rsa, aro[KA ? j : 0] + av[j]);
#pragma unroll
      for (int j = 0; j < NVB; ++j) rb[set][j] = bload<S, WB * NC>(rsb, bro[KBC ? j : 0] + bv[j]);
      const int next = kload + KB;
      if (next < kend) {
        kload = next;
        const int h = table_refill(kload - kbeg, kend - kbeg, KB, kHalf, AHEAD);
        if (h >= 0) fill_k(h);
        if (AHEAD) next_k();
      }
      return;
    }
    kload += more ? KB : 0;
  };
  // the last, partial K step, from k0: element by element, zeros past kend
  auto load_tail = [&](int k0) TAL_INLINE {
    if (FAR) {  // indices past kend read the last one, and count as zeros in both operands
#pragma unroll
      for (int j = 0; j < NVA; ++j)
#pragma unroll
        for (int w = 0; w < (KA ? WA : 1); ++w) {
          const int k = k0 + (KA ? ac + w : al + j * ASTEP);
          constexpr int L = KA ? NC : WA * NC;
          const Vec<S, L> x = gload<S, L>(afar(j, min(k, kend - 1)));
#pragma unroll
          for (int c = 0; c < L; ++c) ra[0][j].v[w * L + c] = k < kend ? x.v[c] : (S)0;
        }
#pragma unroll
      for (int j = 0; j < NVB; ++j)
#pragma unroll
        for (int w = 0; w < (KBC ? WB : 1); ++w) {
          const int k = k0 + (KBC ? bc + w : bl + j * BSTEP);
          constexpr int L = KBC ? NC : WB * NC;
          const Vec<S, L> x = gload<S, L>(bfar(j, min(k, kend - 1)));
#pragma unroll
          for (int c = 0; c < L; ++c) rb[0][j].v[w * L + c] = k < kend ? x.v[c] : (S)0;
        }
      return;
    }
    const bool lin = MODE == 0 || (MODE == 1 && p.k.nd == 1);
    const char *at = (const char *)p.A + (int64_t)blockIdx.y * p.sa + (int64_t)am0 * p.am1;
    const char *bt = (const char *)p.B + (int64_t)blockIdx.y * p.sb + (int64_t)bn0 * p.bn1;
    if (lin) {
      at += (int64_t)k0 * p.ka1;
      bt += (int64_t)k0 * p.kb1;
    }
    const auto rsa = rsrc(at, kOutside), rsb = rsrc(bt, kOutside);
    auto off = [&](int k, int t) TAL_INLINE -> uint32_t {
      if (k >= kend) return kOutside;
      if (lin) return (uint32_t)(k - k0) * (uint32_t)(t ? p.kb1 : p.ka1);
      uint32_t o[2];
      pair_offsets32(p.k, (uint32_t)k, &o[0], &o[1]);
      return o[t];
    };
#pragma unroll
    for (int j = 0; j < NVA; ++j) {
      if (KA) {
#pragma unroll
        for (int w = 0; w < WA; ++w) {
          const Vec<S, NC> x = bload<S, NC>(rsa, aro[KA ? j : 0] + off(k0 + ac + w, 0));
#pragma unroll
          for (int c = 0; c < NC; ++c) ra[0][j].v[w * NC + c] = x.v[c];
        }
      } else {
        ra[0][j] = bload<S, WA * NC>(rsa, aro[0] + off(k0 + al + j * ASTEP, 0));
      }
    }
#pragma unroll
    for (int j = 0; j < NVB; ++j) {
      if (KBC) {
#pragma unroll
        for (int w = 0; w < WB; ++w) {
          const Vec<S, NC> x = bload<S, NC>(rsb, bro[KBC ? j : 0] + off(k0 + bc + w, 1));
#pragma unroll
          for (int c = 0; c < NC; ++c) rb[0][j].v[w * NC + c] = x.v[c];
        }
      } else {
        rb[0][j] = bload<S, WB * NC>(rsb, bro[0] + off(k0 + bl + j * BSTEP, 1));
      }
    }
  };
  const S sgna = p.flags & kDirectConjA ? (S)-1 : (S)1, sgnb = p.flags & kDirectConjB ? (S)-1 : (S)1;
  auto stage = [&](int buf, int set) TAL_INLINE {
#pragma unroll
    for (int j = 0; j < NVA; ++j) {
      const int line = al + j * ASTEP;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        Vec<S, WA> x;
#pragma unroll
        for (int w = 0; w < WA; ++w) x.v[w] = c ? sgna * ra[set][j].v[w * NC + c] : ra[set][j].v[w * NC + c];
        __builtin_memcpy(__builtin_assume_aligned(&As[buf][c][line][ac], sizeof(S) * WA), &x, sizeof(x));
      }
    }
#pragma unroll
    for (int j = 0; j < NVB; ++j) {
      const int line = bl + j * BSTEP;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        Vec<S, WB> x;
#pragma unroll
        for (int w = 0; w < WB; ++w) x.v[w] = c ? sgnb * rb[set][j].v[w * NC + c] : rb[set][j].v[w * NC + c];
        __builtin_memcpy(__builtin_assume_aligned(&Bs[buf][c][line][bc], sizeof(S) * WB), &x, sizeof(x));
      }
    }
  };

  acc_t acc[SM][SN][NC];
#pragma unroll
  for (int i = 0; i < SM; ++i)
#pragma unroll
    for (int j = 0; j < SN; ++j)
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[i][j][c] = acc_t{0, 0, 0, 0};

  // Where a wave has one block and offsets come from tables, it reads D ahead of its products.
  constexpr bool EARLY = TAB && SM * SN == 1;
  const bool dn = p.flags & kDirectAlongN, beta = p.flags & kDirectBeta;
  char *D = (char *)p.D + (int64_t)blockIdx.y * p.sd;
  auto drow = [&](int m) TAL_INLINE { return TAB ? drow_t[wm * TM + m] : row_or_none(p, m0 + wm * TM + m); };
  auto dcol = [&](int n) TAL_INLINE { return TAB ? dcol_t[wn * TN + n] : col_or_none(p, n0 + wn * TN + n); };
  int64_t off0[4];
  Vec<S, NC> old[4];
  auto read_old = [&]() TAL_INLINE {
    if (EARLY && !part) {
      if (dn) SlabOffsets<S, SM, SN, true>(lane, drow, dcol).block(0, 0, off0);
      else SlabOffsets<S, SM, SN, false>(lane, drow, dcol).block(0, 0, off0);
      if (beta) old_values(D, off0, old);
    }
  };

  const int fl = lane & 15, fg = lane >> 4;
  auto compute = [&](int buf) TAL_INLINE {
#pragma unroll
    for (int q = 0; q < KB / (4 * KQ); ++q) {
      // lane group g holds k = 4 KQ q + KQ g + h in MFMA step h, in both operands
      const int kk = q * 4 * KQ + fg * KQ;
      Vec<S, KQ> fa[NC][SM], fb[NC][SN];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
#pragma unroll
        for (int i = 0; i < SM; ++i) {
          const int r = wm * TM + i * 16 + fl;
          if (KA) __builtin_memcpy(&fa[c][i], __builtin_assume_aligned(&As[buf][c][r][kk], 16), 16);
          else
#pragma unroll
            for (int h = 0; h < KQ; ++h) fa[c][i].v[h] = As[buf][c][kk + h][r];
        }
#pragma unroll
        for (int j = 0; j < SN; ++j) {
          const int r = wn * TN + j * 16 + fl;
          if (KBC) __builtin_memcpy(&fb[c][j], __builtin_assume_aligned(&Bs[buf][c][r][kk], 16), 16);
          else
#pragma unroll
            for (int h = 0; h < KQ; ++h) fb[c][j].v[h] = Bs[buf][c][kk + h][r];
        }
      }
#pragma unroll
      for (int h = 0; h < KQ; ++h)
#pragma unroll
        for (int i = 0; i < SM; ++i)
#pragma unroll
          for (int j = 0; j < SN; ++j) {
            if (NC == 1) {
              acc[i][j][0] = MF::op(fa[0][i].v[h], fb[0][j].v[h], acc[i][j][0]);
            } else {
              const S ar = fa[0][i].v[h], ai = fa[NC - 1][i].v[h], br = fb[0][j].v[h], bi = fb[NC - 1][j].v[h];
              acc[i][j][0] = MF::op(ar, br, acc[i][j][0]);
              acc[i][j][0] = MF::op(-ai, bi, acc[i][j][0]);
              acc[i][j][NC - 1] = MF::op(ar, bi, acc[i][j][NC - 1]);
              acc[i][j][NC - 1] = MF::op(ai, br, acc[i][j][NC - 1]);
            }
          }
    }
  };

  // whole K steps; in mode 2 the last step may be a partial one like any other
  const int nfull = TAB ? (max(0, kend - kbeg) + KB - 1) / KB : max(0, kend - kbeg) / KB;
  if (nfull > 0) {
#pragma unroll
    for (int q = 0; q < PF; ++q) load(q);
    read_old();
    stage(0, 0);
    __syncthreads();
  } else {
    read_old();
  }
  // K step kt: the loads of step kt + PF go out, step kt + 1 (loaded PF - 1
  // steps ago) is staged into the other LDS buffer, step kt is multiplied
  auto step = [&](int q, int buf) TAL_INLINE {
    load(q);
    __builtin_amdgcn_sched_barrier(0);  // the loads go out first
    if (PF > 1) stage(buf ^ 1, (q + 1) % PF);
    compute(buf);
    if (PF == 1) stage(buf ^ 1, 0);
    __syncthreads();
  };
  constexpr int U = PF % 2 == 0 ? PF : 2 * PF;  // steps per loop round: register set and LDS buffer are constants
  int kt = 0;
  for (; kt + U <= nfull; kt += U) {
#pragma unroll
    for (int q = 0; q < U; ++q) step(q % PF, q & 1);
  }
#pragma unroll
  for (int q = 0; q < U - 1; ++q)
    if (kt + q < nfull) step(q % PF, q & 1);
  if (!TAB && kbeg + nfull * KB < kend) {
    load_tail(kbeg + nfull * KB);
    stage(0, 0);
    __syncthreads();
    compute(0);
    __syncthreads();
  }

  if (part) {  // raw partial sums in accumulator order: element e of lane l at e * 64 + l
    S *pb = (S *)p.part + ((int64_t)u * WM * WN + wave) * (SM * SN * NC * 4 * 64) + lane;
#pragma unroll
    for (int i = 0; i < SM; ++i)
#pragma unroll
      for (int j = 0; j < SN; ++j)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int r = 0; r < 4; ++r) pb[(((i * SN + j) * NC + c) * 4 + r) * 64] = acc[i][j][c][r];
    return;
  }
  static_assert(sizeof(As) >= sizeof(S) * WM * WN * 16 * 17, "patches fit the A tiles' space");
  S *patch = &As[0][0][0][0] + wave * 16 * 17;
  if constexpr (EARLY) {
    emit_block<S, NC, acc_t>(patch, lane, acc[0][0], !dn, D, off0, (S)p.ar, (S)p.ai, beta, old);
  } else {
    auto emit = [&](auto along_n) TAL_INLINE {
      constexpr bool DN = decltype(along_n)::value;
      const SlabOffsets<S, SM, SN, DN> so(lane, drow, dcol);
      // D's old values are read DIST blocks before theirs are stored: a wave that
      // reads and stores block by block waits for memory at every block (C4
      // rank-6 product of K = 24, 755 MB of D: 541 -> 516 us).  The largest real
      // tiles have no registers for it (R8: 313 us, 463 with DIST = 4), but more
      // waves that wait in turn.
      constexpr int NBLK = SM * SN, DIST = NC == 1 && NBLK > 2 ? 0 : NBLK < 4 ? NBLK : 4;
      int64_t off[DIST + 1][4];
      Vec<S, NC> d[DIST + 1][4];
      auto fetch = [&](int b) TAL_INLINE {
        so.block(b / SN, b % SN, off[b % (DIST + 1)]);
        if (beta) old_values(D, off[b % (DIST + 1)], d[b % (DIST + 1)]);
      };
#pragma unroll
      for (int b = 0; b < DIST; ++b) fetch(b);
#pragma unroll
      for (int b = 0; b < NBLK; ++b) {
        if (b + DIST < NBLK) fetch(b + DIST);
        emit_block<S, NC, acc_t>(patch, lane, acc[b / SN][b % SN], !DN, D, off[b % (DIST + 1)], (S)p.ar, (S)p.ai, beta,
                                 d[b % (DIST + 1)]);
      }
    };
    if (dn) emit(std::true_type());
    else emit(std::false_type());
  }
}

// Sums the ksplit partial blocks of each split tile in order; one wave per 16x16 block.
template <typename S, int NC, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(256) void direct_reduce(DirectArgs) {
  const DirectArgs &p = kernel_args();
  using acc_t = typename Mfma<S>::acc_t;
  constexpr int TM = BM / WM, TN = BN / WN, SM = TM / 16, SN = TN / 16, PER = SM * SN * NC * 4 * 64;
  __shared__ S patches[4][16 * 17];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = blockIdx.x * 4 + w;  // block index: (tile, wave, i, j)
  constexpr int BPT = WM * WN * SM * SN;
  const int tile = blk / BPT, in = blk % BPT;
  if (tile >= p.rem) return;
  const int wave = in / (SM * SN), ij = in % (SM * SN), i = ij / SN, j = ij % SN;
  int bx, by;
  tile_xy(p.whole + tile, p.gx, p.gy, bx, by);
  const int mb = bx * BM + (wave % WM) * TM + i * 16, nb = by * BN + (wave / WM) * TN + j * 16;
  auto drow = [&](int m) TAL_INLINE { return row_or_none(p, mb + m); };
  auto dcol = [&](int n) TAL_INLINE { return col_or_none(p, nb + n); };
  const bool dn = p.flags & kDirectAlongN, beta = p.flags & kDirectBeta;
  int64_t off[4];
  if (dn) SlabOffsets<S, 1, 1, true>(lane, drow, dcol).block(0, 0, off);
  else SlabOffsets<S, 1, 1, false>(lane, drow, dcol).block(0, 0, off);
  Vec<S, NC> old[4];
  if (beta) old_values((const char *)p.D, off, old);
  acc_t acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = acc_t{0, 0, 0, 0};
  const S *pb = (const S *)p.part + ((int64_t)tile * p.ksplit * WM * WN + wave) * PER + (int64_t)ij * NC * 256 + lane;
#pragma unroll 4
  for (int q = 0; q < p.ksplit; ++q, pb += (int64_t)WM * WN * PER) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[c][r] += pb[(c * 4 + r) * 64];
  }
  emit_block<S, NC, acc_t>(patches[w], lane, acc, !dn, (char *)p.D, off, (S)p.ar, (S)p.ai, beta, old);
}

}  // namespace direct
}  // namespace tal
