// Split R4 GEMMs (fast math, gfx950).
//
// Contract (the GEMM call of gpu_tensor_block_contract_dlf,
// tensor_algebra_gpu_nvidia.cu:6851-7060):
//   C(MxN, column-major, ldc) = alpha * op(A) * op(B) + beta * C,  beta in {0,1}
// with op(A) in {A, A^T} and op(B) in {B, B^T}.  All other products run on the
// direct contraction kernels (direct_kernel.hpp).  Blocks are renumbered so that
// each XCD (dispatch round-robins workgroups over the 8 XCDs) walks a compact
// band of C tiles and the operand panels it streams stay in its own L2.
#include "kernels.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace tal {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kXcds = 8;

// Tile t of C -> (bx, by): tiles are walked in groups of 8 tile-rows, column
// by column inside a group (a bijection of [0, gx*gy)).
__device__ inline void tile_xy(int64_t t, int64_t gx, int64_t gy, int64_t &bx, int64_t &by) {
  constexpr int64_t G = 8;  // tile-rows per group
  const int64_t group = t / (G * gy);
  const int64_t first = group * G;
  const int64_t rows = min(G, gx - first);
  const int64_t in = t - group * G * gy;
  bx = first + in % rows;
  by = in / rows;
}

// Unit u of n in dispatch order -> a number such that the units of one XCD are
// neighbours, for any n (a bijection of [0, n)).
__device__ inline int64_t xcd_order(int64_t u, int64_t n) {
  const int64_t q = n / kXcds, r = n % kXcds, x = u % kXcds;
  return x * q + min(x, r) + u / kXcds;
}

// ---------------------------------------------------------------------------
// R4 GEMM as 3-term split-BF16 products (bf16x6): every FP32 operand value x
// is split exactly into x = h + m + l with h = bf16(x), m = bf16(x - h),
// l = bf16(x - h - m) (each residual is exact in FP32), and
//   a*b ~ ah*bh + ah*bm + am*bh + ah*bl + am*bm + al*bh
// is accumulated in FP32 by v_mfma_f32_16x16x32_bf16 (method of Henry, Tang,
// Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", ARITH 2019).  The dropped terms are below
// 2^-24 relative; with FP32 accumulation the normwise error at K = 9216 is a
// few 1e-7 (cf. ~1e-6 for the FP32 MFMA path).  Both operands are split once
// into swizzled BF16 planes in a workspace by split_planes_kernel, then 256 x
// 128 tiles of 8 waves stream the planes with no VALU split work in the K
// loop; a partial last round of tiles is split along K into partials summed by
// presplit_reduce_kernel.  MFMA 16x16x32 bf16
// layout: A lane l holds A[l%16][8*(l/16)..+7], B lane l holds
// B[8*(l/16)..+7][l%16], accumulator register r of lane l holds
// C[4*(l/16)+r][l%16].
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------------------
// Pre-split GEMMs.  split_planes_kernel writes the planes of an operand once
// into a workspace (layout: plane_chunk; rows padded to the GEMM tile, K padded
// to 32, zeros in the padding), so the GEMM's inner loop only moves bytes and
// issues MFMAs: no split arithmetic and no bounds checks.  The dominant product of the leading terms goes to one accumulator
// and the small products to a second, so the main accumulator is rounded once
// per K step of 32 without any VALU adds; the two are summed in the epilogue.
//
// Two splits share the kernel body (NP = planes per operand):
//  - NP = 3, bf16x6: three BF16 planes h, m, l (x = h + m + l exactly) and six
//    products per block, as described above;
//  - NP = 2, fp16x3: every row of op(A) and every column of op(B) is scaled
//    by a power of two 2^-e, e the exponent of the row's largest magnitude
//    (so the row lies in (-1, 1)), then split into two FP16 planes
//    h = fp16(y), m = fp16(y - h) (y - h is exact in FP32).  FP16 keeps 11
//    significant bits, so |y - h - m| <= 2^-22 |y| for normal m, and the
//    three products ah*bh + ah*bm + am*bh (v_mfma_f32_16x16x32_f16, the same
//    rate as BF16) carry about 22 bits of each operand: normwise relative
//    error a few 1e-7, like bf16x6, for half of its MFMA work.  The dropped
//    am*bm is below 2^-22 relative.  An element below 2^-24 of its row's
//    largest keeps only an absolute accuracy of 2^-25 of that largest (FP16
//    subnormals), so rows that mix magnitudes over more than about 2^10 lose
//    relative accuracy on their small elements; bf16x6, whose planes keep
//    FP32's exponent range, has no such limit.  The epilogue multiplies by
//    2^(ea + eb), which is exact.
//
// Block tile 256 x 128, 8 waves of 64 x 64 (two per SIMD), K steps of 32.  The
// planes lie in memory as the blocks an LDS stage holds (plane_chunk), so a
// stage is filled by loads straight to LDS, 1 KB a wave and instruction, with
// no registers, no address arithmetic and no LDS store instructions; fragment
// reads are free of bank conflicts.  What bounds it: fp16x3, where a step is 48
// MFMAs a wave, the latency of the next step's loads and the LDS (1,400 of
// 1,536 cycles a step); hence three stages, two steps in flight.  bf16x6 has
// twice the MFMAs and room for two stages.  One barrier per K step.  Rates of
// the 16-bit products: fp16x3 at 5184^3 772 -> 1,100 TFLOP/s (1080 -> 757 us
// with the last round split), bf16x6 at 9216^3 1,146 -> 1,376 (8.19 -> 6.82 ms),
// against loads through registers one step ahead of rows with a stride of K; a
// bf16 library product reaches 1,230-1,320 on this card.
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ inline void split3_finite(float x, __bf16 &h, __bf16 &m, __bf16 &l) {
  h = (__bf16)x;
  if (!__builtin_isfinite(x)) {  // Inf/NaN carried by the leading term alone
    m = l = (__bf16)0.0f;
    return;
  }
  const float r = x - (float)h;
  m = (__bf16)r;
  l = (__bf16)(r - (float)m);
}

// Exponent e with max * 2^-e in [0.5, 1) for the bit pattern u of a row's
// largest magnitude; 0 for an all-zero row or one holding Inf/NaN.
__device__ inline int row_exp(uint32_t u) {
  const float v = __uint_as_float(u);
  if (!(v > 0.0f) || !__builtin_isfinite(v)) return 0;
  int e;
  (void)frexpf(v, &e);
  return e;
}

__device__ inline void split2_scaled(float x, int e, _Float16 &h, _Float16 &m) {
  const float y = ldexpf(x, -e);
  h = (_Float16)y;
  m = __builtin_isfinite(y) ? (_Float16)(y - (float)h) : (_Float16)0.0f;  // Inf/NaN: leading term alone
}

__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t *__restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

__device__ inline uint32_t abs_bits(float x) { return __float_as_uint(x) & 0x7fffffffu; }

// U[r] = max over k < K of the bit pattern of |X(r, k)| with X(r, k) at
// X[r + k*ld] (for non-negative floats the pattern orders as the value; NaN
// patterns sort above Inf), U zeroed beforehand.  Block = 4 waves, lanes along
// r; grid.x = row groups, grid.y = K segments of kseg, which the four waves share.
__global__ __launch_bounds__(256) void row_absmax_kernel(const float *__restrict__ X, int64_t ld, int64_t R, int64_t K,
                                                         int64_t kseg, uint32_t *__restrict__ U) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t k0 = (int64_t)blockIdx.y * kseg, k1 = min(K, k0 + kseg);
  uint32_t m = 0;
  const int64_t r = (int64_t)blockIdx.x * 64 + lane;
  if (r >= R) return;
#pragma unroll 8
  for (int64_t k = k0 + wave; k < k1; k += 4) m = max(m, abs_bits(X[r + k * ld]));
  if (m) atomicMax(U + r, m);
}

// Plane layout: blocks of kPRows rows x PBK contracted indices, 8 KB each and
// contiguous, along K first; in a block row r holds its four 16-byte chunks at
// slots c ^ pswz(r).  A K step of the GEMM reads whole blocks, as they lie, and
// they are the image its LDS stage needs.
constexpr int kPRows = 128, PBK = 32;
__device__ inline int pswz(int r) { return ((r >> 1) ^ (r >> 3)) & 3; }
// Address of chunk kc (8 contracted indices) of row r, in chunks; nks: K steps of the plane.
__device__ inline int64_t plane_chunk(int64_t r, int64_t kc, int64_t nks) {
  const int rr = (int)(r % kPRows), c = (int)(kc & 3);
  return ((r / kPRows * nks + (kc >> 2)) * kPRows + rr) * 4 + (c ^ pswz(rr));
}

// 8 consecutive k of row x (contiguous along k), zeros past n.
__device__ inline void load8(const float *x, int64_t k0, int64_t n, bool vec, float (&v)[8]) {
  if (vec && k0 + 8 <= n) {
    const float4 a = *reinterpret_cast<const float4 *>(x + k0);
    const float4 b = *reinterpret_cast<const float4 *>(x + k0 + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = k0 + i < n ? x[k0 + i] : 0.0f;
  }
}

// The NP planes of 8 values to their chunk; e: exponent of the row (NP = 2).
template <int NP>
__device__ inline void split_store(const float (&v)[8], int e, uint4 *__restrict__ P, int64_t plane, int64_t at) {
  uint4 u;
  if constexpr (NP == 3) {
    __bf16 h[8], m[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) split3_finite(v[i], h[i], m[i], l[i]);
    __builtin_memcpy(&u, h, 16);
    P[at] = u;
    __builtin_memcpy(&u, m, 16);
    P[plane + at] = u;
    __builtin_memcpy(&u, l, 16);
    P[2 * plane + at] = u;
  } else {
    _Float16 h[8], m[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) split2_scaled(v[i], e, h[i], m[i]);
    __builtin_memcpy(&u, h, 16);
    P[at] = u;
    __builtin_memcpy(&u, m, 16);
    P[plane + at] = u;
  }
}

// fp16x3 planes of op(X) when its rows are K-contiguous (X(r, k) at
// X[r*ld + k]).  A block takes 2^rows_log padded rows: it finds their largest
// magnitudes (U[r], 0 for padding rows) and splits them, four threads on the 32
// k of a row's part of a plane block (128 bytes read, 64 written, the block's
// rows side by side).  The first kHeld chunks of a thread stay in registers
// between the two, so rows of up to 8,192 are read once; longer ones' other
// chunks are read again.  vec: X 16-byte aligned and ld a multiple of 4.
// Memory-bound: 5184 x 5184, two rows a block, in 46 us, 4.7 TB/s (two passes
// over a row per block: 60).  Short rows go many to a block, as long as their
// chunks stay in registers and there are blocks for all CUs (split_rows_log).
constexpr int kSplitThreads = 512, kHeld = 4;
int split_rows_log(int64_t nks, int64_t Rp) {
  int l = 1;
  while (l < 7 && (kSplitThreads / 8 >> l) * kHeld >= nks && Rp >> l > 1024) ++l;
  return l;
}
__global__ __launch_bounds__(kSplitThreads) void split_rows_f16_kernel(const float *__restrict__ X, int64_t ld,
                                                                       int64_t R, int64_t K, int64_t nks,
                                                                       uint4 *__restrict__ P, int64_t plane, int vec,
                                                                       uint32_t *__restrict__ U, int rows_log,
                                                                       int64_t first) {
  __shared__ uint32_t red[kSplitThreads / 4];
  const int tid = threadIdx.x, c = tid & 3, row = tid >> 2 & ((1 << rows_log) - 1);
  const int ks0 = tid >> (2 + rows_log), round = kSplitThreads / 4 >> rows_log;  // K steps per round of the block
  const int64_t r = ((first + blockIdx.x) << rows_log) + row, n = r < R ? K : 0;
  const float *x = X + r * ld;
  if (tid < kSplitThreads / 4) red[tid] = 0;
  float v[kHeld][8];
  uint32_t m = 0;
#pragma unroll
  for (int q = 0; q < kHeld; ++q) load8(x, (int64_t)(ks0 + q * round) * PBK + c * 8, n, vec, v[q]);
#pragma unroll
  for (int q = 0; q < kHeld; ++q)
#pragma unroll
    for (int i = 0; i < 8; ++i) m = max(m, abs_bits(v[q][i]));
  for (int64_t ks = ks0 + kHeld * round; ks < nks; ks += round) {
    float w[8];
    load8(x, ks * PBK + c * 8, n, vec, w);
#pragma unroll
    for (int i = 0; i < 8; ++i) m = max(m, abs_bits(w[i]));
  }
  // the four threads of a chunk row, then the wave's and the block's others in LDS
  m = max(m, (uint32_t)__shfl_xor((int)m, 1));
  m = max(m, (uint32_t)__shfl_xor((int)m, 2));
  __syncthreads();
  if (c == 0) atomicMax(&red[row], m);
  __syncthreads();
  m = red[row];
  if (ks0 == 0 && c == 0) U[r] = m;
  const int e = row_exp(m);
#pragma unroll
  for (int q = 0; q < kHeld; ++q) {
    const int64_t ks = ks0 + q * round;
    if (ks < nks) split_store<2>(v[q], e, P, plane, plane_chunk(r, ks * 4 + c, nks));
  }
  for (int64_t ks = ks0 + kHeld * round; ks < nks; ks += round) {
    float w[8];
    load8(x, ks * PBK + c * 8, n, vec, w);
    split_store<2>(w, e, P, plane, plane_chunk(r, ks * 4 + c, nks));
  }
}

// KC = 1: source element (r, k) at X[r*ld + k]; KC = 0: at X[r + k*ld].  A
// thread splits 8 consecutive k of one row.  KC = 1: a block covers kSplitRows
// rows of 64 / kSplitRows K steps, four threads on a row's 32 k (9216 x 9216 in
// 141 us, 6.0 TB/s; 2, 4, 16 and 64 rows 149, 147, 147 and 165); KC = 0: 64
// rows of one K step, lanes along the rows; so source reads are coalesced
// either way.  NP = 3: BF16 planes; NP = 2: FP16 planes of the row scaled by
// the exponent from U.
constexpr int kSplitRows = 8;
template <int KC, int NP>
__global__ __launch_bounds__(256) void split_planes_kernel(const float *__restrict__ X, int64_t ld, int64_t R,
                                                           int64_t K, int64_t nks, uint4 *__restrict__ P,
                                                           int64_t plane, int vec, const uint32_t *__restrict__ U,
                                                           int64_t first) {
  const int tid = threadIdx.x;
  constexpr int ROWS = KC ? kSplitRows : 64, STEPS = 64 / ROWS;  // of a block
  const int64_t block = first + blockIdx.x, nkb = (nks + STEPS - 1) / STEPS, rg = block / nkb;
  const int64_t r = rg * ROWS + (KC ? (tid >> 2) % ROWS : tid & 63);
  const int64_t ks = (block - rg * nkb) * STEPS + (KC ? tid / (4 * ROWS) : 0);
  const int c = KC ? tid & 3 : tid >> 6;
  if (ks >= nks) return;
  const int64_t k0 = ks * PBK + c * 8;
  float v[8];
  if (KC) {
    load8(X + r * ld, k0, r < R ? K : 0, vec, v);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (r < R && k0 + i < K) ? X[r + (k0 + i) * ld] : 0.0f;
  }
  const int e = NP == 2 && r < R ? row_exp(U[r]) : 0;
  split_store<NP>(v, e, P, plane, plane_chunk(r, ks * 4 + c, nks));
}

constexpr int PBM = 256, PBN = 128;

template <int NP>
__device__ inline f32x4 pmfma(uint4 a, uint4 b, f32x4 c) {
  if constexpr (NP == 3)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
}

struct SplitArgs {
  const uint4 *a, *b;      // planes of op(A) and op(B)
  int64_t apl, bpl, nks;   // chunks per plane, K steps
  float *C;
  const int64_t *cmap;     // element offsets of C's rows, then its columns; null: m + n * ldc
  float *part;             // partial sums of the tiles cut into K ranges, PBM x PBN each
  const uint32_t *ua, *ub; // NP = 2: row maxima of op(A), column maxima of op(B)
  int64_t M, N, ldc;
  int64_t gx, gy, whole;   // tiles; the first `whole` are computed by one workgroup each
  int64_t rem, ksteps;     // the others by ksplit workgroups, `ksteps` K steps each
  int ksplit;
  int beta_one;
  float alpha;
};

// 16 bytes a lane from base + off to the LDS bytes from `lds` on, lane after
// lane: no registers, no LDS store instructions.  The compiler neither knows
// the load nor waits for it; presplit_gemm_kernel's loop does.
__device__ inline void dma16(uint32_t lds, const char *base, uint32_t off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}

template <int N>
__device__ inline void wait_dma() {  // at most N of the wave's loads in flight, its LDS reads done
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

template <int NP>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void presplit_gemm_kernel(SplitArgs p) {
  constexpr int NS = NP == 2 ? 3 : 2;             // LDS stages
  constexpr int PIECE = kPRows * 4, PIECES = 3;   // chunks of a plane block; blocks of a plane: two of A, one of B
  constexpr int LOADS = NP * PIECES;              // a wave's loads per K step
  __shared__ uint4 S[NS][NP][PIECES][PIECE];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 3, wn = wave >> 2;
  // units: the whole tiles, then the K ranges of the others
  const int64_t whole = p.whole;
  int64_t tile, kt0 = 0, kt1 = p.nks, unit = (int64_t)blockIdx.x - whole;
  const bool range = unit >= 0;
  if (!range) {
    tile = xcd_order(blockIdx.x, whole);
  } else {
    // by K range, then by tile: the tiles of one range share panels in an XCD's L2
    unit = xcd_order(unit, p.rem * p.ksplit);
    const int64_t kpart = unit / p.rem;
    tile = unit - kpart * p.rem;
    unit = tile * p.ksplit + kpart;  // place of the partial sums
    kt0 = kpart * p.ksteps;
    kt1 = min(kt1, kt0 + p.ksteps);
    tile += whole;
  }
  int64_t bx, by;
  tile_xy(tile, p.gx, p.gy, bx, by);
  const int64_t nk = kt1 - kt0;  // may be <= 0 for a trailing K range: its partial sums are zeros

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint4 *)&S[0][0][0][0] + wave * 1024;
  const uint32_t voff = (uint32_t)lane * 16;
  const char *ab = reinterpret_cast<const char *>(p.a + (2 * bx * p.nks + kt0) * PIECE) + wave * 1024;
  const char *bb = reinterpret_cast<const char *>(p.b + (by * p.nks + kt0) * PIECE) + wave * 1024;
  const int64_t ablk = p.nks * PIECE * 16, apl = p.apl * 16, bpl = p.bpl * 16;
  auto load = [&](int st) {
    const uint32_t l = lds0 + (uint32_t)st * (NP * PIECES * PIECE * 16);
#pragma unroll
    for (int t = 0; t < NP; ++t) {
      dma16(l + (t * PIECES + 0) * PIECE * 16, ab + t * apl, voff);
      dma16(l + (t * PIECES + 1) * PIECE * 16, ab + t * apl + ablk, voff);
      dma16(l + (t * PIECES + 2) * PIECE * 16, bb + t * bpl, voff);
    }
  };

  f32x4 big[4][4], small[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) big[i][j] = small[i][j] = f32x4{0, 0, 0, 0};

  // fragment slot of row 16*x + (lane & 15), chunk lane >> 4: the swizzle of
  // that row is pswz(lane & 15), with bit 1 flipped when x is odd
  const int fc = lane >> 4, fr = lane & 15;
  const int fs[2] = {fr * 4 + (fc ^ pswz(fr)), fr * 4 + (fc ^ pswz(fr) ^ 2)};
  const int am = (wm >> 1) * PIECE + (wm & 1) * 256, bn = 2 * PIECE + wn * 256;  // the wave's rows and columns
  auto compute = [&](int st) {
    const uint4 *s = &S[st][0][0][0];
    uint4 fb[NP][4];
#pragma unroll
    for (int t = 0; t < NP; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) fb[t][j] = s[t * PIECES * PIECE + bn + j * 64 + fs[j & 1]];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint4 fa[NP];
#pragma unroll
      for (int t = 0; t < NP; ++t) fa[t] = s[t * PIECES * PIECE + am + i * 64 + fs[i & 1]];
      // B is the first operand, so that a lane's column of the accumulators is a row of C
      if constexpr (NP == 3) {
#pragma unroll
        for (int j = 0; j < 4; ++j) small[i][j] = pmfma<NP>(fb[0][j], fa[2], small[i][j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) small[i][j] = pmfma<NP>(fb[1][j], fa[1], small[i][j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) small[i][j] = pmfma<NP>(fb[2][j], fa[0], small[i][j]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) small[i][j] = pmfma<NP>(fb[0][j], fa[1], small[i][j]);
#pragma unroll
      for (int j = 0; j < 4; ++j) small[i][j] = pmfma<NP>(fb[1][j], fa[0], small[i][j]);
#pragma unroll
      for (int j = 0; j < 4; ++j) big[i][j] = pmfma<NP>(fb[0][j], fa[0], big[i][j]);
    }
  };

  // K step kt is multiplied while the loads of step kt + NS - 1 are in flight.
  // A stage is loaded again only behind the barrier that every wave reaches
  // after its reads of it.  Past the last step that step is loaded again, into
  // stages nobody reads, so that the number of loads in flight is a constant.
  if (nk > 0) {
    int64_t left = nk - 1;  // steps whose loads have not gone out
    auto next = [&] {
      const int64_t d = left > 0 ? PIECE * 16 : 0;
      ab += d;
      bb += d;
      left -= left > 0;
    };
#pragma unroll
    for (int q = 0; q < NS - 1; ++q) {
      load(q);
      next();
    }
    int64_t kt = 0;
    for (; kt + NS <= nk; kt += NS) {
#pragma unroll
      for (int q = 0; q < NS; ++q) {
        wait_dma<(NS - 2) * LOADS>();
        load((q + NS - 1) % NS);
        next();
        __builtin_amdgcn_sched_barrier(0);
        compute(q);
      }
    }
#pragma unroll
    for (int q = 0; q < NS - 1; ++q) {
      if (kt + q < nk) {
        wait_dma<(NS - 2) * LOADS>();
        load((q + NS - 1) % NS);
        next();
        compute(q);
      }
    }
    wait_dma<0>();  // LDS is given back only when nothing writes to it any more
  }

  // NP = 2: exponents of this lane's 4 rows (i) and 16 columns (j, r); every
  // index is below the padded sizes of ua / ub
  const int64_t m0 = bx * PBM + wm * 64 + fr, n0 = by * PBN + wn * 64 + 4 * fc;
  int ea[4] = {}, eb[4][4] = {};
  if constexpr (NP == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) ea[i] = row_exp(p.ua[m0 + i * 16]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) eb[j][r] = row_exp(p.ub[n0 + j * 16 + r]);
  }
  if (range) {
    float *pb = p.part + unit * PBM * PBN;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int ml = wm * 64 + i * 16 + fr, nl = wn * 64 + j * 16 + 4 * fc + r;
          const float x = big[i][j][r] + small[i][j][r];
          pb[ml + nl * PBM] = NP == 2 ? ldexpf(x, ea[i] + eb[j][r]) : x;
        }
    return;
  }
  int64_t om[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) om[i] = m0 + i * 16 >= p.M ? -1 : p.cmap ? p.cmap[m0 + i * 16] : m0 + i * 16;
  // The columns' offsets are read together and the old values of four columns
  // while the four before are stored: one after the other, a lone tile's 16
  // columns wait for memory 32 times (products of 300 x 280 by 500 53 us each).
  int64_t on[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t n = n0 + j * 16 + r;
      on[j][r] = n >= p.N ? -1 : p.cmap ? p.cmap[p.M + n] : n * p.ldc;
    }
  float old[2][4][4];
  auto fetch = [&](int j) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) old[j & 1][r][i] = on[j][r] >= 0 && om[i] >= 0 ? p.C[on[j][r] + om[i]] : 0.0f;
  };
  if (p.beta_one) fetch(0);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (p.beta_one && j < 3) fetch(j + 1);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = big[i][j][r] + small[i][j][r];
        const float v = p.alpha * (NP == 2 ? ldexpf(x, ea[i] + eb[j][r]) : x);
        if (on[j][r] >= 0 && om[i] >= 0) p.C[on[j][r] + om[i]] = p.beta_one ? old[j & 1][r][i] + v : v;
      }
  }
}

// Sums the ksplit partial blocks of the tiles cut into K ranges in order and applies C = alpha * sum (+ C).
__global__ __launch_bounds__(kThreads) void presplit_reduce_kernel(SplitArgs p) {
  const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (e >= p.rem * PBM * PBN) return;
  const int64_t q = e / (PBM * PBN);
  const int in = (int)(e % (PBM * PBN)), ml = in % PBM, nl = in / PBM;
  int64_t bx, by;
  tile_xy(p.whole + q, p.gx, p.gy, bx, by);
  const int64_t m = bx * PBM + ml, n = by * PBN + nl;
  if (m >= p.M || n >= p.N) return;
  const float *pb = p.part + q * p.ksplit * (PBM * PBN) + in;
  float x = 0.0f;
#pragma unroll 4
  for (int ch = 0; ch < p.ksplit; ++ch) x += pb[(int64_t)ch * (PBM * PBN)];
  float *c = p.C + (p.cmap ? p.cmap[m] + p.cmap[p.M + n] : m + n * p.ldc);
  const float v = p.alpha * x;
  *c = p.beta_one ? *c + v : v;
}

int64_t round_up(int64_t x, int64_t q) { return (x + q - 1) / q * q; }

__global__ __launch_bounds__(256) void offset_map_kernel(OffsetMap map, int64_t *__restrict__ out) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= map.M + map.N) return;
  const bool row = e < map.M;
  int64_t x = row ? e : e - map.M, off = 0;
  const int t0 = row ? 0 : map.nm, t1 = row ? map.nm : map.nm + map.nn;
  for (int t = t0; t < t1; ++t) {
    off += (x % map.ext[t]) * map.str[t];
    x /= map.ext[t];
  }
  out[e] = off;
}

// Splits op(X) (rows R, depth K) into NP planes at P (NP = 2: also the row
// maxima into U, Rp entries, used for the scaling); returns 0 or a launch error.
template <int NP>
int split_operand(bool kcont, const float *X, int64_t ld, int64_t R, int64_t K, int64_t Rp, int64_t Kp, uint4 *P,
                  uint32_t *U, hipStream_t s) {
  const int64_t nks = Kp / PBK, plane = Rp * Kp / 8;
  const int64_t steps = kcont ? 64 / kSplitRows : 1, nblk = Rp / (64 / steps) * ((nks + steps - 1) / steps);
  const int vec = ((uintptr_t)X % 16 == 0) && ld % 4 == 0;
  if (NP == 2 && kcont) {  // maxima and planes in one pass over HBM
    if (Rp / 2 > 0x7fffffffLL) return -4;  // blocks are numbered in 31 bits
    const int rows_log = split_rows_log(nks, Rp);  // at most the 128 rows that Rp is a multiple of
    launch_grids(Rp >> rows_log, kSplitThreads, [&](int64_t first, dim3 grid, bool) {
      split_rows_f16_kernel<<<grid, dim3(kSplitThreads), 0, s>>>(X, ld, R, K, nks, P, plane, vec, U, rows_log, first);
    });
    return hipGetLastError() == hipSuccess ? 0 : -2;
  }
  if constexpr (NP == 2) {
    fill_u32_kernel<<<dim3((unsigned)((Rp + 255) / 256)), dim3(256), 0, s>>>(U, Rp);
    if (R > 0 && K > 0) {
      const int64_t kseg = std::max<int64_t>(512, round_up((K + 65534) / 65535, 256));
      launch_grids((R + 63) / 64, 256, [&](int64_t first, dim3 grid, bool) {
        grid.y = (unsigned)((K + kseg - 1) / kseg);
        row_absmax_kernel<<<grid, dim3(256), 0, s>>>(X + first * 64, ld, R - first * 64, K, kseg, U + first * 64);
      });
    }
  }
  // short rows fill a block to an eighth: 134 million of them take two grids
  launch_grids(nblk, 256, [&](int64_t first, dim3 grid, bool) {
    if (kcont) split_planes_kernel<1, NP><<<grid, dim3(256), 0, s>>>(X, ld, R, K, nks, P, plane, vec, U, first);
    else split_planes_kernel<0, NP><<<grid, dim3(256), 0, s>>>(X, ld, R, K, nks, P, plane, vec, U, first);
  });
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

// The tiles of C are dealt to the resident workgroups in rounds.  The `rem`
// tiles of a partial last round may be computed as ksplit K ranges each; ksplit
// = 1 means no split.
struct TailSplit {
  int64_t rem = 0;
  int ksplit = 1;
};

int op_code(char t) {
  switch (t) {
    case 'N': case 'n': return 0;
    case 'T': case 't': return 1;
    default: return -1;
  }
}

}  // namespace

bool gemm_split_bf16_available() { return true; }

// Resident workgroups of the pre-split GEMM kernel with NP planes on the
// current device, cached per device.
template <int NP>
static int64_t presplit_slots() {
  static int64_t cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (!cache[dev]) {
    int cus = 0, per = 0;
    hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess)
      e = NP == 3 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, presplit_gemm_kernel<3>, 512, 0)
                  : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, presplit_gemm_kernel<2>, 512, 0);
    if (e != hipSuccess) return 0;
    cache[dev] = (int64_t)cus * std::max(per, 1);
  }
  return cache[dev];
}

// K split of a partial last round of tiles: as many ranges as make it shortest,
// counted in K steps.  A range costs about 4 steps beside its own (its first
// loads) and the way of its partial sums through memory, 128 KB written and read
// again (a step is 1.3 us of fp16x3, 2.3 of bf16x6): 5184^3 in fp16x3 has 861
// tiles on 256 slots, and its 93 last ones run as 5 ranges each, 0.5 of a round
// instead of a whole one (and 20 us of summing against 110 saved).  All ranges'
// sums have to fit into kSumsBytes, two rounds of them.
template <int NP>
static TailSplit presplit_tail(int64_t M, int64_t N, int64_t K, bool room) {
  TailSplit t;
  if (M <= 0 || N <= 0 || !room) return t;
  const int64_t T = (round_up(M, PBM) / PBM) * (round_up(N, PBN) / PBN), slots = presplit_slots<NP>();
  if (slots <= 0) return t;
  const int64_t rem = T % slots, nks = round_up(std::max<int64_t>(K, 1), PBK) / PBK;
  if (rem == 0) return t;
  double best = (double)nks;
  for (int64_t ks = 2; ks <= 16 && ks * 8 <= nks && rem * ks * PBM * PBN * 4 <= (int64_t)kSumsBytes; ++ks) {
    const double cost = (double)((rem * ks + slots - 1) / slots * ((nks + ks - 1) / ks + 4)) +
                        (NP == 2 ? 0.033 : 0.019) * (double)(rem * ks);
    if (cost < best) {
      best = cost;
      t.rem = rem;
      t.ksplit = (int)ks;
    }
  }
  return t;
}

// Workspace of the pre-split GEMM: the planes of op(A) and op(B) (NP planes
// of 2-byte values each) and for NP = 2 the row / column maxima; each part
// starts on 256 bytes.
struct SplitLayout {
  int64_t Mp, Np, Kp;
  size_t a, b, ua, ub, total;
};

template <int NP>
static SplitLayout split_layout(int64_t M, int64_t N, int64_t K) {
  SplitLayout l;
  l.Mp = round_up(std::max<int64_t>(M, 1), PBM);
  l.Np = round_up(std::max<int64_t>(N, 1), PBN);
  l.Kp = round_up(std::max<int64_t>(K, 1), PBK);
  l.a = 0;
  l.b = l.a + (size_t)round_up(2 * NP * l.Mp * l.Kp, 256);
  l.ua = l.b + (size_t)round_up(2 * NP * l.Np * l.Kp, 256);
  l.ub = l.ua + (NP == 2 ? (size_t)round_up(4 * l.Mp, 256) : 0);
  l.total = l.ub + (NP == 2 ? (size_t)round_up(4 * l.Np, 256) : 0);
  return l;
}

template <int NP>
static int launch_presplit(int opa, int opb, int64_t M, int64_t N, int64_t K, double ar, const void *A, int64_t lda,
                           const void *B, int64_t ldb, int beta_one, void *C, int64_t ldc, void *ws,
                           void *sums, const int64_t *cmap, hipStream_t s) {
  const SplitLayout l = split_layout<NP>(M, N, K);
  const TailSplit tail = presplit_tail<NP>(M, N, K, sums != nullptr);
  char *w = (char *)ws;
  uint4 *pa = (uint4 *)(w + l.a), *pb = (uint4 *)(w + l.b);
  uint32_t *ua = NP == 2 ? (uint32_t *)(w + l.ua) : nullptr, *ub = NP == 2 ? (uint32_t *)(w + l.ub) : nullptr;
  // A 'T' (KxM) and B 'N' (KxN) already have K contiguous per row of the plane
  if (int e = split_operand<NP>(opa == 1, (const float *)A, lda, M, K, l.Mp, l.Kp, pa, ua, s)) return e;
  if (int e = split_operand<NP>(opb == 0, (const float *)B, ldb, N, K, l.Np, l.Kp, pb, ub, s)) return e;
  SplitArgs p;
  p.a = pa;
  p.b = pb;
  p.apl = l.Mp * l.Kp / 8;
  p.bpl = l.Np * l.Kp / 8;
  p.nks = l.Kp / PBK;
  p.C = (float *)C;
  p.cmap = cmap;
  p.part = (float *)sums;
  p.ua = ua;
  p.ub = ub;
  p.M = M;
  p.N = N;
  p.ldc = ldc;
  p.gx = l.Mp / PBM;
  p.gy = l.Np / PBN;
  p.rem = tail.rem;
  p.whole = p.gx * p.gy - p.rem;
  p.ksplit = tail.ksplit;
  p.ksteps = (p.nks + p.ksplit - 1) / p.ksplit;
  p.beta_one = beta_one;
  p.alpha = (float)ar;
  if (p.gx * p.gy > 0x7fffffffLL - 16 * p.rem) return -4;
  const dim3 grid((unsigned)(p.whole + p.rem * p.ksplit)), block(512);
  if (p.rem == 0) {
    launch_last(presplit_gemm_kernel<NP>, grid, block, s, p);
  } else {
    presplit_gemm_kernel<NP><<<grid, block, 0, s>>>(p);
    launch_last(presplit_reduce_kernel, dim3((unsigned)(p.rem * PBM * PBN / kThreads)), dim3(kThreads), s, p);
  }
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_offset_map(const OffsetMap &map, int64_t *out, hipStream_t s) {
  if (map.nm < 0 || map.nn < 0 || map.nm + map.nn > kMaxMapDims || !out) return -1;
  for (int t = 0; t < map.nm + map.nn; ++t)
    if (map.ext[t] < 1) return -1;
  const int64_t n = map.M + map.N, nblk = (n + 255) / 256;
  if (nblk > 0x7fffffffLL) return -4;
  offset_map_kernel<<<dim3((unsigned)nblk), dim3(256), 0, s>>>(map, out);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

size_t gemm_split_workspace(int method, int64_t M, int64_t N, int64_t K) {
  return method == SPLIT_FP16X3 ? split_layout<2>(M, N, K).total : split_layout<3>(M, N, K).total;
}

int launch_gemm_split(int method, char ta, char tb, int64_t M, int64_t N, int64_t K, double ar, const void *A,
                      int64_t lda, const void *B, int64_t ldb, int beta_one, void *C, int64_t ldc, void *ws,
                      void *sums, hipStream_t s, const int64_t *cmap) {
  const int opa = op_code(ta), opb = op_code(tb);
  if (opa < 0 || opb < 0 || M < 0 || N < 0 || K < 0 || !A || !B || !C || !ws || (uintptr_t)ws % 16) return -1;
  if (method != SPLIT_BF16X6 && method != SPLIT_FP16X3) return -1;
  if (M == 0 || N == 0) return 0;
  if (ldc < std::max<int64_t>(1, M)) return -1;
  if (lda < std::max<int64_t>(1, opa == 0 ? M : K)) return -1;
  if (ldb < std::max<int64_t>(1, opb == 0 ? K : N)) return -1;
  return method == SPLIT_FP16X3
             ? launch_presplit<2>(opa, opb, M, N, K, ar, A, lda, B, ldb, beta_one, C, ldc, ws, sums, cmap, s)
             : launch_presplit<3>(opa, opb, M, N, K, ar, A, lda, B, ldb, beta_one, C, ldc, ws, sums, cmap, s);
}

}  // namespace tal
