// Instantiates the direct contraction kernels of one data kind: included by
// direct_r4.hip, direct_r8.hip, direct_c4.hip and direct_c8.hip.
#pragma once

#include "direct.hpp"
#include "direct_kernel.hpp"
#include "kernels.hpp"

namespace tal {
namespace direct {

// A tile shape's kernel: BM x BN x KB by WM x WN waves, PF K steps of loads
// in flight, OCC waves per SIMD.
template <int BM_, int BN_, int KB_, int WM_, int WN_, int PF_, int OCC_>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, KB = KB_, WM = WM_, WN = WN_, PF = PF_, OCC = OCC_;
};

template <typename S, int NC, class T, int KA, int KBC, int W, int MODE>
void run(DirectArgs a, unsigned batch, hipStream_t s) {
  constexpr unsigned NT = 64 * T::WM * T::WN;
  constexpr auto kernel =
      direct_kernel<S, NC, KA, KBC, W, W, T::BM, T::BN, T::KB, T::WM, T::WN, T::PF, T::OCC, MODE>;
  const int64_t units = a.whole + (int64_t)a.rem * a.ksplit;
  int64_t at = 0;
  for (int64_t n; (n = direct_launch_units(units, at, NT)) > 0; at += n) {
    const dim3 grid((unsigned)n, batch), block(NT);
    a.first = (int32_t)at;
    if (a.rem == 0 && at + n == units) launch_last(kernel, grid, block, s, a);
    else kernel<<<grid, block, 0, s>>>(a);
  }
  if (a.rem == 0) return;
  constexpr int kBlocks = (T::BM / 16) * (T::BN / 16);  // 16 x 16 blocks of a tile
  launch_last(direct_reduce<S, NC, T::BM, T::BN, T::WM, T::WN>, dim3((unsigned)(((int64_t)a.rem * kBlocks + 3) / 4)),
              dim3(256), s, a);
}

template <typename S, int NC, class T, int W, int MODE>
void run_layout(const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s) {
  if (v.ka && v.kb) run<S, NC, T, 1, 1, W, MODE>(a, batch, s);
  else if (v.ka) run<S, NC, T, 1, 0, W, MODE>(a, batch, s);
  else if (v.kb) run<S, NC, T, 0, 1, W, MODE>(a, batch, s);
  else run<S, NC, T, 0, 0, W, MODE>(a, batch, s);
}

// Mode 2 (any k, offsets by table) is for small problems: element loads only.
// 32 x 32 tiles take it for every k of several dimensions, also where its
// leading run would do for mode 1, whose steps carry more code (418 x 420 by
// 475 R8 22.7 -> 19.2 us, by 105 C8 17.4 -> 15.8, by 665 R4 20.5 -> 18.4; with
// one dimension mode 0 is the faster one, 9.0 against 9.8).
template <typename S, int NC, class T, int W>
bool run_tile(const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s) {
  const bool tables = v.mode == 2 || (v.mode == 1 && a.k.nd > 1 && T::BM * T::BN == 32 * 32);
  if (tables) run_layout<S, NC, T, 1, 2>(v, a, batch, s);
  else if (v.mode == 3 && v.width == W) run_layout<S, NC, T, W, 3>(v, a, batch, s);
  else if (v.mode == 3) run_layout<S, NC, T, 1, 3>(v, a, batch, s);
  else if (v.mode == 1 && v.width == W) run_layout<S, NC, T, W, 1>(v, a, batch, s);
  else if (v.mode == 1) run_layout<S, NC, T, 1, 1>(v, a, batch, s);
  else if (v.width == W) run_layout<S, NC, T, W, 0>(v, a, batch, s);
  else run_layout<S, NC, T, 1, 0>(v, a, batch, s);
  return true;
}

}  // namespace direct
}  // namespace tal
