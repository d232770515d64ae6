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
  typedef __attribute__((ext_vector_type(4))) uint32_t Word;
  // a whole word's group, and its numbers
  DEV_INLINE Word word(int g) const {
    return *reinterpret_cast<const Word*>(x + first(g));
  }
  DEV_INLINE static void numbers(const Word& w, float (&v)[VEC]) {
#pragma unroll
    for (int j = 0; j < VEC; ++j)
      v[j] = __uint_as_float(sizeof(T) == 4 ? w[j % 4]
                             : j % 2 ? w[j / 2] & 0xffff0000u
                                     : w[j / 2] << 16);
  }
  DEV_INLINE void load(int g, float (&v)[VEC]) const {
    const int i0 = first(g);
    if (i0 >= 0 && i0 + VEC <= V) {
      numbers(word(g), v);
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const int i = i0 + j;
        v[j] = i >= 0 && i < V ? (float)x[i] : -INFINITY;
      }
    }
  }
};
