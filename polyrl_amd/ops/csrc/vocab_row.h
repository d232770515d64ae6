// Reading a row of vocabulary logits in 16-byte words.
//
// A row need not start at a 16-byte address (odd vocabularies).  Its groups
// are the whole words at 16-byte addresses, one short group of ``lead``
// numbers before them and one short group behind; entries outside the row
// read as -inf.
#pragma once

#include "common.h"

template <typename T>
struct VocabRow {
  static constexpr int VEC = 16 / sizeof(T);
  const T* x;
  int V, lead;

  DEV_INLINE VocabRow(const T* row, int V_) : x(row), V(V_) {
    const int n = (int)((16 - ((uintptr_t)row & 15)) & 15) / (int)sizeof(T);
    lead = n < V_ ? n : V_;
  }
  DEV_INLINE int groups() const { return 1 + (V - lead + VEC - 1) / VEC; }
  // index of a group's first entry (below 0 in a short first group)
  DEV_INLINE int first(int g) const { return lead + (g - 1) * VEC; }
  DEV_INLINE void load(int g, float (&v)[VEC]) const {
    const int i0 = first(g);
    if (i0 >= 0 && i0 + VEC <= V) {
      if constexpr (sizeof(T) == 2) {
        const bf16x8 w = *reinterpret_cast<const bf16x8*>(x + i0);
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = bf2f(w.v[j]);
      } else {
        const f32x4v w = *reinterpret_cast<const f32x4v*>(x + i0);
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = w.v[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const int i = i0 + j;
        v[j] = i >= 0 && i < V ? (float)x[i] : -INFINITY;
      }
    }
  }
};
