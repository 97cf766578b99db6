// Contractions as the direct kernels see them.  No HIP: planned and tested on the CPU.
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

namespace tal {

// A contraction (or a plain matrix product) in elements: m, n and k as lists
// of (fused) tensor dimensions, first fastest, with each one's stride in the
// two tensors that have it; batch entries at fixed strides.
struct DirectDim {
  int64_t ext;
  int64_t s[2];  // m: (A, D), n: (B, D), k: (A, B)
};
struct DirectForm {
  int64_t M = 1, N = 1, K = 1, batch = 1;
  std::vector<DirectDim> m, n, k;
  int64_t sa = 0, sb = 0, sd = 0;  // batch strides
  int64_t avol = 0, bvol = 0;      // elements of A and B (at least the span of one batch entry)
};

// Appends a dimension, fused with the one before where both tensors chain; unit extents are dropped.
inline void direct_dim(std::vector<DirectDim> *v, int64_t ext, int64_t s0, int64_t s1) {
  if (ext == 1) return;
  if (!v->empty()) {
    DirectDim &l = v->back();
    if (l.s[0] * l.ext == s0 && l.s[1] * l.ext == s1) {
      l.ext *= ext;
      return;
    }
  }
  v->push_back(DirectDim{ext, {s0, s1}});
}

// Most dimensions a number may have in one tensor, neighbours that chain there counted as one.
constexpr int kDirectDims = 6;
inline int direct_chains(const std::vector<DirectDim> &v, int t) {
  int n = 0;
  for (size_t i = 0; i < v.size(); ++i) n += i == 0 || v[i - 1].s[t] * v[i - 1].ext != v[i].s[t];
  return n;
}

}  // namespace tal
