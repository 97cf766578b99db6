// Direct contraction kernels: D(m, n) (+)= alpha * sum_k A(m, k) * B(k, n)
// read from and written to any dense tensor layout.  Internal.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "direct_args.hpp"

namespace tal {

// direct_choose on the current device.
DirectChoice direct_choose(int dk, int64_t M, int64_t N, int64_t K, int64_t batch);

// Enqueues the product on stream s; sums: room for kSumsBytes bytes of
// partial sums, or null (tiles are not cut along K).  Nonzero: it was not launched.
int launch_direct(int dk, const DirectForm &f, const void *A, const void *B, void *D, double ar, double ai, bool conja,
                  bool conjb, bool accumulate, void *sums, hipStream_t s);

// One kind's kernels (direct_r4.hip ... direct_c8.hip).  false: no such variant.
using DirectLaunch = bool (*)(int tile, const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s);
bool direct_launch_r4(int tile, const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s);
bool direct_launch_r8(int tile, const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s);
bool direct_launch_c4(int tile, const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s);
bool direct_launch_c8(int tile, const DirectVariant &v, const DirectArgs &a, unsigned batch, hipStream_t s);

}  // namespace tal
