// Kernel arguments, variant, tile shape and K split of a direct contraction.
// No HIP: planned and tested on the CPU.
#pragma once

#include <cstddef>
#include <cstdint>

#include "direct_form.hpp"
#include "direct_index.hpp"

namespace tal {

// The form with A and B (m and n) exchanged: the same product.
DirectForm direct_swapped(const DirectForm &f);

// The kernel's variant for a form.
struct DirectVariant {
  bool ka = false, kb = false;  // the operand is contiguous along k
  int width = 1;                // elements per load
  int mode = 0;                 // how a K step is addressed (direct_kernel.hpp), for K steps of kb
};

// Fills the layout part of the kernel arguments and the variant for elements
// of esz bytes, loads of up to full_width elements and K steps of kstep;
// false when the kernel cannot address the form (more than kDirectDims
// dimensions in a group, extents past 31 bits, strides past 32 bits where rows
// or k have several dimensions).
bool direct_args(const DirectForm &f, int esz, int full_width, int kstep, DirectArgs *a, DirectVariant *v);
// Longest K of one launch: a longer product (k of one dimension) is summed into D range after range.
constexpr int64_t kDirectMaxK = (int64_t)1 << 30;

// Whether the direct kernels take the form for data kind dk at every tile, either way round; the variant at K steps of 16.
bool direct_addressable(const DirectForm &f, int dk, DirectVariant *v);

// Units of one launch of workgroups of `threads`, from unit `at` of `units` on: a
// grid may not hold 2^32 threads or more (products of more than 2^30 rows).
inline int64_t direct_launch_units(int64_t units, int64_t at, unsigned threads) {
  const int64_t most = (int64_t)(0xffffffffu / threads) / 8 * 8;  // whole rounds over the XCDs
  return units - at < most ? units - at : most;
}

// Tile shapes of a kind, largest first.  unit / stream: microseconds that one
// tile of K = 1024 takes alone on a CU, and per tile when several share the CU.
constexpr int kDirectTiles = 4;
struct DirectTile {
  int bm, bn, kb;
  double unit, stream;
};
const DirectTile *direct_tiles(int dk);

// Most memory that the partial sums of a product's K ranges may take.
constexpr size_t kSumsBytes = (size_t)64 << 20;

// Tile shape and K split of a product on a GPU of `cus` compute units; depends on nothing else.
struct DirectChoice {
  bool swap = false;  // A and B exchange roles
  int tile = 0;
  int64_t gx = 0, gy = 0, whole = 0, rem = 0;
  int ksplit = 1, ksteps = 0;
  size_t part_bytes = 0;
  double us = 0;  // estimate
};
DirectChoice direct_choose(int dk, int64_t M, int64_t N, int64_t K, int64_t batch, int cus);

// Element size and elements per 16-byte load of a data kind.
int direct_elem(int dk);
int direct_width(int dk);

}  // namespace tal
