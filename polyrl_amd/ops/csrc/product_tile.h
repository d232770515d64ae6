// Products of bf16 matrices by tiles of 256 x 256 outputs (linear_backward.hip,
// linear_prompt.hip).
//
// Split.  A block has four waves, 128 x 128 outputs each: 256 accumulator registers a
// lane, 128 more for the fragments of two steps, one wave a SIMD, one block a CU.  (Tiles
// of fewer rows, 32 J, where the left operand is LINES: a wave has J row parts for eight.)
// A step is 32 inner numbers.  Two steps of an operand, 32 KiB, are loaded as one unit
// straight into LDS, five units' room, three of both operands for tiles of up to 160 rows,
// whose short steps would wait for their loads; a barrier every two steps.  Where an operand's
// inner dimension is its memory's rows' own (LINES: x and W in x W^T, dY in dY W) a unit
// is 256 rows of 128 bytes, whole lines, and fragments are read as they are; where it
// runs over the memory's rows (COLUMNS: W in dY W, both in dY^T X) a unit is 64 rows of 512
// bytes and fragments come by transposed reads (ds_read_b64_tr_b16).  Both leave a
// lane eight inner numbers from 8 * (lane / 16) of 32.
//
// Schedule.  One wave a SIMD has nobody to take its turn: the order is fixed instruction
// by instruction (order()).  Behind each of a step's 64 v_mfma_f32_16x16x32_bf16, 16
// cycles each, stands at most one of the next step's fragment reads, of the unit's
// loads, of the words that say where a load goes, or of the next addresses, a fragment
// to three products (two: 3% slower, 582 for 566 us at 7168 x 14336 x 4096).  A block's
// tiles are one stream of units: at a tile's end the next one's first are there, and its
// sums are read, rounded and stored between the products of the next one's first step,
// which start from 0 instead of from a cleared accumulator.
#pragma once

#include <utility>

#include "attention_tile.h"

namespace product {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;
template <int J = 8>
using Acc = f32x4_t[8][J];             // columns, rows: 16 x 16 outputs each

constexpr int SIDE = 256;              // outputs of a tile, each way
constexpr int PAIR = 64;               // inner numbers of a unit
constexpr int UNIT = SIDE * PAIR * 2;  // bytes
constexpr int LDS_BYTES = 5 * UNIT;
constexpr int CUS = 256;
constexpr int GROUP = 8;               // rows of tiles that a die walks together

// f(0), f(1), .., as constants
template <typename F, int... K>
DEV_INLINE void each(std::integer_sequence<int, K...>, F f) {
  (f(std::integral_constant<int, K>()), ...);
}

DEV_INLINE void order() { __builtin_amdgcn_sched_barrier(0); }

DEV_INLINE void aim(unsigned to) {
  asm volatile("s_mov_b32 m0, %0" ::"s"(to) : "m0");
}

// Sums of an accumulator, read where they are asked for: left to the compiler all are
// read at once, into registers that the next tile's fragments hold
DEV_INLINE f32x4_t sums_of(const f32x4_t& c) {
  f32x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float x;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(c[e]));
    v[e] = x;
  }
  return v;
}

// all but N loads of this wave are there, and all waves are here
template <int N>
DEV_INLINE void arrived() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// An operand of one tile: its first unit's address, the bytes from there to the
// operand's end, the units
struct Units {
  const void* at;
  long bytes;
  int n;
};

// P: 16-row parts of a wave's half
template <bool LINES, int P = 8>
struct Operand {
  static_assert(LINES || P == 8, "COLUMNS are 256");
  static constexpr int FRAGS = LINES ? 2 : 8;
  u32x4_t from;                        // descriptor of the unit to load
  unsigned step, left;                 // bytes to the next one; units to the tile's end
  unsigned after_lo, after_hi, after_bytes, after_n;   // the next tile
  unsigned load_at[P];                 // of this lane's loads
  int frag_at[FRAGS];  // this lane's place, slot 0, of 16 columns (LINES: of a step)

  // COLUMNS: a row's 512 bytes stand in windows of 32, turned by the row, so that
  // eight rows of a window meet no bank twice
  DEV_INLINE static int turn(int r) { return (r & 3) | ((r >> 3) & 1) << 2; }
  // LINES: a row's granules are turned by the row, so that 16 rows of a granule meet
  // no bank twice
  DEV_INLINE static int place(int g, int r) { return g ^ (r >> 1 & 7); }

  // ld: numbers of a memory row; half: which 128 of the outer numbers are the wave's
  DEV_INLINE Operand(const char* lds, long ld, int half) {
    pitch(ld);
    const int lane = threadIdx.x & 63;
    const int lds0 = (int)(uintptr_t)(lds_p)lds, c = lane & 15, h = lane >> 4;
#pragma unroll
    for (int d = 0; d < FRAGS; ++d) {
      if (LINES) {
        frag_at[d] = lds0 + half * (P * 2048) + c * 128 + (place(4 * d + h, c) << 4);
      } else {
        const int r = 8 * h + (c >> 2);
        frag_at[d] = lds0 + half * 256 + r * 512 + ((d ^ turn(r)) << 5) +
                     (c & 3) * 8;
      }
    }
  }
  DEV_INLINE void pitch(long ld) {
    const unsigned ldb = (unsigned)ld * 2;
    step = LINES ? 2 * PAIR : PAIR * ldb;
    const int lane = threadIdx.x & 63, wid = wave_id();
#pragma unroll
    for (int i = 0; i < P; ++i) {
      if (LINES) {
        const int r = wid * (8 * P) + i * 8 + (lane >> 3);
        load_at[i] = r * ldb + (place(lane & 7, r) << 4);
      } else {
        const int r = wid * 16 + i * 2 + (lane >> 5);
        load_at[i] = r * ldb + (((lane & 31) ^ (turn(r) << 1)) << 4);
      }
    }
  }
  // The tile that follows; what is behind ``bytes`` reads as 0
  DEV_INLINE void follow(const Units& u) {
    const uint64_t b = (uint64_t)u.at;
    after_lo = (unsigned)uniform((int)b);
    after_hi = (unsigned)uniform((int)(b >> 32)) & 0xffffu;
    after_bytes = (unsigned)uniform((int)u.bytes), after_n = uniform(u.n);
    // (a scalar that a vector instruction wrote is not to be used at once)
    asm volatile("s_nop 4"
                 : "+s"(after_lo), "+s"(after_hi), "+s"(after_bytes),
                   "+s"(after_n));
  }
  DEV_INLINE void start() {
    from = {after_lo, after_hi, after_bytes, 0x00020000u};
    left = after_n;
    asm volatile("s_nop 4" : "+s"(from), "+s"(left), "+s"(step));
  }
  // In assembly, so that the compiler does not wait for it on its own account; no
  // register is written.
  DEV_INLINE void go(int i) const {
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(load_at[i]),
                 "s"(from)
                 : "memory");
  }
  // on to the next unit, in three parts
  template <int PART>
  DEV_INLINE void next() {
    unsigned lo = from[0], hi = from[1], bytes = from[2];
    if (PART == 0)
      asm volatile("s_add_u32 %0, %0, %2\n\ts_addc_u32 %1, %1, 0"
                   : "+s"(lo), "+s"(hi)
                   : "s"(step)
                   : "scc");
    if (PART == 1)
      asm volatile(
          "s_sub_u32 %0, %0, %2\n\ts_cselect_b32 %0, 0, %0\n\ts_sub_u32 %1, %1, 1"
          : "+s"(bytes), "+s"(left)
          : "s"(step)
          : "scc");
    if (PART == 2)
      asm volatile(
          "s_cmp_eq_u32 %3, 0\n\ts_cselect_b32 %0, %4, %0\n\t"
          "s_cselect_b32 %1, %5, %1\n\ts_cselect_b32 %2, %6, %2\n\t"
          "s_cselect_b32 %3, %7, %3"
          : "+s"(lo), "+s"(hi), "+s"(bytes), "+s"(left)
          : "s"(after_lo), "s"(after_hi), "s"(after_bytes), "s"(after_n)
          : "scc");
    from[0] = lo, from[1] = hi, from[2] = bytes;
  }
  DEV_INLINE void load(unsigned to) {  // a unit, at once
#pragma unroll
    for (int i = 0; i < P; ++i) {
      aim(to + i * 1024);
      asm volatile("s_nop 0");
      go(i);
    }
    next<0>(), next<1>(), next<2>();
  }
};

// 16 outer numbers, a step's 32 inner ones: of lane l number l % 16, inner ones from
// 8 * (l / 16)
template <bool LINES>
struct Frag {
  i16x8_t all;
  i16x4_t half[2];
  // frag_at[] of the unit; d: which 16 of the wave's 128
  template <int STEP, int H>
  DEV_INLINE void read(const int* at, int d) {
    typedef __attribute__((address_space(3))) const i16x8_t* lds_i16x8_p;
    if constexpr (!LINES)
      half[H] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_i16x4_p)(uintptr_t)(at[d] + STEP * 16384 + H * 2048));
    else if constexpr (H == 0)
      all = *(lds_i16x8_p)(uintptr_t)(at[STEP] + d * 2048);
  }
  DEV_INLINE i16x8_t whole() const {
    return LINES ? all
                 : __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

// Row and column of a tile: GROUP rows of tiles, one column after the other, so that
// the blocks that run on a die at once share 8 x 4 tiles' operands
struct Place {
  int row, col, share;                 // (share: of the tile's inner numbers)
  DEV_INLINE Place() {}
  DEV_INLINE Place(int tile, int row_tiles, int col_tiles, int share_ = 0)
      : share(share_) {
    const int group = tile / (GROUP * col_tiles);
    const int rest = tile - group * GROUP * col_tiles;
    const int high = min(GROUP, row_tiles - group * GROUP);
    row = uniform(group * GROUP + rest % high), col = uniform(rest / high);
  }
};

// Tiles r = 0, 1, ..: units(r, left, right, place) says where tile r and its operands
// are, false behind the last one.  Its sums go to ``sink``: sink.tile(place), then for each
// row part j sink.rows(j), and sink.put(j, q, sums) of each of its groups of COLS column
// parts, columns_of(q, e) for e = 0, 1, ..  Accumulator e of column part i, row part j is
// column 16 i + 4 (lane / 16) + e of row 16 j + lane % 16 of the wave's 16 J x 128 (row half
// wave % 2, column half wave / 2).  A row part is STORES stores in every wave, whatever of
// it is within the matrix: the waits count them.  A tile that another one follows has four
// units and more.
//
// PARTS > 1: the sum of that many products, part p of tile t as number PARTS t + p, whose
// left operand's rows may be of another length each (left_ld(part)).  Each starts anew,
// which costs some 2 us.
template <bool LL, bool RL, int J = 8, int PARTS = 1, typename LeftLd,
          typename UnitsOf, typename Sink>
DEV_INLINE void run(char* lds, LeftLd left_ld, long right_ld, UnitsOf units,
                    Sink& sink) {
  const int wid = wave_id();
  Operand<LL, J> a(lds, left_ld(0), wid & 1);
  Operand<RL> b(lds, right_ld, wid >> 1);
  // (of a unit a wave loads 1 KiB for each of its row parts)
  // DEEP: three pairs' units fit
  constexpr int LEFT = J * 4096, THIRD = LEFT + UNIT;
  constexpr bool DEEP = LL && RL && 3 * THIRD <= LDS_BYTES;
  constexpr int B0 = DEEP ? LEFT : UNIT;
  // Loads that may be on their way when the next pair's units have to be there: of the pair
  // after that the left operand's, and (DEEP) the right one's
  constexpr int YOUNG = DEEP ? J + 8 : J;
  const unsigned to_a = (unsigned)(uintptr_t)(lds_p)lds + wid * (J * 1024);
  const unsigned to_b = (unsigned)(uintptr_t)(lds_p)lds + wid * 8192;
  Units ua, ub;
  Place last, here, next;              // the tiles behind, at and ahead of this step
  int now = 0, pairs = 0;
  bool more = units(0, ua, ub, here);
  if (!more) return;
  auto look_ahead = [&] {              // (behind the last tile nothing is read)
    more = units(now + 1, ua, ub, next);
    if (!more || PARTS > 1) {
      ua.bytes = ub.bytes = 0;
      if (PARTS == 1) ua.n = ub.n = 1 << 30;
    }
    a.follow(ua), b.follow(ub);
  };
  Acc<J> acc;
  Frag<LL> fa[2][J];
  Frag<RL> fb[2][8];
  int na[a.FRAGS], nb[b.FRAGS];        // where the next fragments are
  // the first units and fragments
  auto begin = [&] {
    a.follow(ua), b.follow(ub);
    a.start(), b.start();
    pairs = ua.n;
    look_ahead();
    a.load(to_a), b.load(to_b + B0);
    if constexpr (DEEP) {
      a.load(to_a + THIRD), b.load(to_b + THIRD + B0), a.load(to_a + 2 * THIRD);
      arrived<J + YOUNG>();
    } else {
      a.load(to_a + 2 * UNIT), b.load(to_b + 3 * UNIT);
      arrived<J + 8>();
    }
#pragma unroll
    for (int d = 0; d < a.FRAGS; ++d) na[d] = a.frag_at[d];
#pragma unroll
    for (int d = 0; d < b.FRAGS; ++d) nb[d] = b.frag_at[d] + B0;
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      if (d < J) {
        fa[0][d < J ? d : 0].template read<0, 0>(na, d);
        fa[0][d < J ? d : 0].template read<0, 1>(na, d);
      }
      fb[0][d].template read<0, 0>(nb, d), fb[0][d].template read<0, 1>(nb, d);
    }
  };
  begin();

  constexpr int COLS = Sink::COLS, GROUPS = 8 / COLS;
  // The products of a step, whose fragments are registers N, the reads of the next one's,
  // and the loads of a unit to ``slot``.  (Loads behind the end read nothing: the
  // count of them is the same in every step.)  ENDS: the first pair of steps of a tile,
  // which take the last one's sums out of the accumulators and start them anew; columns
  // go fastest there, as the sink has them.
  auto step = [&](auto n_, auto ends_, auto& load, unsigned slot, int a_next,
                  int b_next) {
    constexpr int N = decltype(n_)::value, O = 1 - N;
    constexpr bool ENDS = decltype(ends_)::value;
    constexpr int FRAGS = 8 + J, LOADS = (N == 0) == DEEP ? 8 : J, ALL = 8 * J;
    // instructions of a fragment (and a load's two, or with the load's first; few row
    // parts leave room for two)
    constexpr int PER = LL && RL && J < 6 ? 2 : 3;
    static_assert(PER == 2 ? LOADS <= FRAGS : 2 * LOADS <= FRAGS + 2, "the order");
    static_assert(PER * FRAGS + 2 <= ALL, "the order");
    __builtin_amdgcn_s_waitcnt(0xc07f);            // fragments: lgkmcnt(0)
    // The next unit of both is there, and this one's, read to the end, make room.  (The
    // last tile's stores are as young as this step's loads, and still on their way.)
    if constexpr (N == 1)
      arrived<ENDS ? std::min(63, YOUNG + J * Sink::STORES) : YOUNG>();
    constexpr bool FIRST = ENDS && N == 0;
    f32x4_t sums[COLS];
    each(std::make_integer_sequence<int, ALL>(), [&](auto k_) {
      constexpr int k = decltype(k_)::value;
      constexpr int q = k / COLS % GROUPS, e = k % COLS;
      constexpr int i = FIRST ? Sink::column_of(q, e) : k / J;
      constexpr int j = FIRST ? k / 8 : i & 1 ? J - 1 - k % J : k % J;
      order();
      // (in assembly, else the compiler moves accumulators about)
      if constexpr (FIRST) {
        if constexpr (k % 8 == 0) sink.rows(j);
        sums[e] = sums_of(acc[i][j]);
        order();
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0"
                     : "+a"(acc[i][j])
                     : "v"(fb[N][i].whole()), "v"(fa[N][j].whole()));
        order();
        if constexpr (e == COLS - 1) sink.put(j, q, sums);
      } else {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[i][j])
                     : "v"(fb[N][i].whole()), "v"(fa[N][j].whole()));
      }
      order();
      constexpr int f = k / PER;       // fragment: one column's, all rows', the rest
      if constexpr (f < FRAGS) {
        constexpr int H = k % PER;
        if constexpr (H < 2 && f >= 1 && f <= J)
          fa[O][f - 1].template read<O, H>(na, f - 1);
        else if constexpr (H < 2)
          fb[O][f == 0 ? 0 : f - J].template read<O, H>(nb, f == 0 ? 0 : f - J);
        if constexpr (PER == 2 && f < LOADS) {
          if constexpr (H == 0) aim(slot + f * 1024);
          else load.go(f);
        } else if constexpr (PER == 3 && H == 2 && f / 2 < LOADS) {
          if constexpr (f % 2 == 0) aim(slot + f / 2 * 1024);
          else load.go(f / 2);
        }
      } else {
        // the addresses of the pair that comes next, and the next unit to load
        constexpr int d = k - PER * FRAGS, REST = ALL - PER * FRAGS;
        constexpr int FA = Operand<LL, J>::FRAGS, FB = Operand<RL>::FRAGS;
        // (what of the loads had no place beside a fragment)
        if constexpr (PER == 3 && (FRAGS + d) / 2 < LOADS) {
          if constexpr ((FRAGS + d) % 2 == 0) aim(slot + (FRAGS + d) / 2 * 1024);
          else load.go((FRAGS + d) / 2);
        }
        if constexpr (N == 0)
          each(std::make_integer_sequence<int, FA + FB>(), [&](auto e_) {
            constexpr int e = decltype(e_)::value;
            if constexpr (e * REST / (FA + FB) == d && e < FA) {
              na[e] = a.frag_at[e] + a_next;
              asm volatile("" : "+v"(na[e]));
            } else if constexpr (e * REST / (FA + FB) == d) {
              nb[e - FA] = b.frag_at[e - FA] + b_next;
              asm volatile("" : "+v"(nb[e - FA]));
            }
          });
        if constexpr (d == REST / 5) load.template next<0>();
        if constexpr (d == REST / 2) load.template next<1>();
        if constexpr (d == REST * 4 / 5) load.template next<2>();
      }
    });
  };

  // slots: this pair's units, the next pair's, the left one behind that
  int s0 = 0, s1 = UNIT, s2 = 2 * UNIT, s3 = 3 * UNIT, s4 = 4 * UNIT;
  // (DEEP: where they, the next pair and the one behind that are)
  int d0 = 0, d1 = THIRD, d2 = 2 * THIRD;
  auto pair = [&](auto ends) {
    if constexpr (DEEP) {
      step(std::integral_constant<int, 0>(), ends, b, to_b + d2 + B0, d1, d1 + B0);
      step(std::integral_constant<int, 1>(), ends, a, to_a + d0, d1, d1 + B0);
      const int t = d0;
      d0 = d1, d1 = d2, d2 = t;
    } else {
      step(std::integral_constant<int, 0>(), ends, a, to_a + s4, s2, s3);
      step(std::integral_constant<int, 1>(), ends, b, to_b + s0, s2, s3);
      const int t0 = s0, t1 = s1;
      s0 = s2, s1 = s3, s2 = s4, s3 = t0, s4 = t1;
    }
  };
  if constexpr (PARTS > 1) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  for (;;) {
    int p = 0;
    if (PARTS == 1 && now > 0) {
      sink.tile(last);
      pair(std::true_type());
      p = 1;
    } else if (PARTS == 1) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    for (; p < pairs; ++p) pair(std::false_type());
    if (!more || (PARTS > 1 && now % PARTS == PARTS - 1)) {
      // (the compiler does not know that these are products, whose results take a
      // while; they are read by sums_of())
      asm volatile("s_nop 15\n\ts_nop 15");
      sink.tile(here);
      each(std::make_integer_sequence<int, J * GROUPS>(), [&](auto g_) {
        constexpr int j = decltype(g_)::value / GROUPS, q = decltype(g_)::value % GROUPS;
        order();
        if constexpr (q == 0) sink.rows(j);
        f32x4_t sums[COLS];
#pragma unroll
        for (int e = 0; e < COLS; ++e) sums[e] = sums_of(acc[Sink::column_of(q, e)][j]);
        sink.put(j, q, sums);
      });
      // (here and not where the next one begins: the compiler keeps numbers that nobody
      // reads and spills others)
      if constexpr (PARTS > 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int j = 0; j < J; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
    if (!more) break;
    ++now;
    last = here, here = next;
    if constexpr (PARTS == 1) {
      pairs = ua.n;
      look_ahead();
    } else {
      // (no load on its way, no wave at the last fragments)
      __builtin_amdgcn_s_waitcnt(0xc07f);
      arrived<0>();
      a.pitch(left_ld(now % PARTS));
      units(now, ua, ub, here);
      s0 = 0, s1 = UNIT, s2 = 2 * UNIT, s3 = 3 * UNIT, s4 = 4 * UNIT;
      begin();
    }
  }
  // (no load is on its way to LDS when the block ends)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Item r of this block: blocks go to the dies in turn, each die takes one stretch of
// the items, its blocks every ``blocks / dies``-th of it; -1 behind the last
DEV_INLINE int item_of(int r, int items, int blocks) {
  const int per = (items + ATTN_XCDS - 1) / ATTN_XCDS;
  const int in = (int)blockIdx.x / ATTN_XCDS + r * (blocks / ATTN_XCDS);
  const int item = (int)(blockIdx.x % ATTN_XCDS) * per + in;
  return in < per && item < items ? item : -1;
}

// Units of rows from ``first`` of an operand in LINES: inner numbers from inner0 on
DEV_INLINE Units lines(const bf16_t* p, long outer, long inner, long first,
                       long inner0, int n) {
  const long skip = first * inner + inner0;
  return {p + skip, min(2 * (outer * inner - skip), 2 * SIDE * inner), n};
}
// of 256 columns of one in COLUMNS.  (Columns behind the last one are the next row's,
// and whoever reads them stores nothing.)
DEV_INLINE Units columns(const bf16_t* p, long outer, long inner, long first,
                         long inner0, int n) {
  const long skip = inner0 * outer + first;
  return {p + skip, 2 * (inner * outer - skip), n};
}

// Two column parts of a row part as rows of bf16 numbers: this lane's 8 columns are 16 i +
// 8 (lane / 16) of the wave's, of row 16 j + lane % 16
DEV_INLINE u32x4_t eight_columns(const f32x4_t& c0, const f32x4_t& c1) {
  u32x4_t out;
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    union { bf16_t h[2]; unsigned u; } x, y;
    x.h[0] = f2bf(c0[2 * w]), x.h[1] = f2bf(c0[2 * w + 1]);
    y.h[0] = f2bf(c1[2 * w]), y.h[1] = f2bf(c1[2 * w + 1]);
    const auto p = __builtin_amdgcn_permlane32_swap(x.u, y.u, false, false);
    const auto q = __builtin_amdgcn_permlane16_swap(p[0], p[1], false, false);
    out[w] = q[0], out[2 + w] = q[1];
  }
  return out;
}

// Rows of a matrix (rows, cols), cols in 8s, from a wave's first one on, 16 at a time, as a
// buffer: what would be behind the last row is not written, nor are columns behind the last
// one, whose offsets are behind every buffer's end.  In every wave each store is an
// instruction that is counted.
//
// Outputs that the L2s hold, 4 MiB each, go past them (``past``), so that the kernel's end
// has nothing to write back (us, through and past them: 5135 rows, 1024 -> 1536 18.2 and
// 16.3, 1024 -> 1024 15.0 and 13.8; gate, up and activation of 1024 -> 4096 68.6 and 66.9, of
// 8192 rows 103.5 and 101.0).  Not as nontemporal ones, which the next kernel would have to
// read from memory (the rotation behind 1024 -> 1536 10.1 us for 8.1).  Larger ones pass
// through them: repeated alone they gain too where the 256 MB behind hold them (8192 rows,
// 4096 -> 16384 736 and 696), but not in a trainer's step (input gradients of 7168 rows
// through 4096 x 4096 and 4096 x 14336 together 747 and 790), nor where nothing does (4096
// rows, 4096 -> 128256 2816 and 2992; the trainer's gate, up and activation of 7168 x 14336
// each 1166 and 1288).
constexpr long L2_OUT = ATTN_XCDS * (4L << 20);
struct OutRows {
  char* at;
  long left, pitch;                    // bytes: to the matrix's end, of 16 rows
  __amdgpu_buffer_rsrc_t buffer;
  DEV_INLINE void start(bf16_t* out, long rows, long cols, long row0) {
    pitch = 32 * cols, at = (char*)(out + row0 * cols) - pitch;
    left = 2 * cols * (rows - row0) + pitch;
  }
  DEV_INLINE void next() {
    at += pitch, left -= pitch;
    buffer = __builtin_amdgcn_make_buffer_rsrc(
        at, 0, (int)max(0L, min(left, 0x7fffffffL)), 0x00020000);
  }
  // this lane's 8 columns from col on of row lane % 16
  DEV_INLINE static unsigned offset(long cols, long col) {
    return col < cols ? (unsigned)((threadIdx.x & 15) * cols + col) * 2 : 0x80000000u;
  }
  DEV_INLINE u32x4_t get(unsigned offset) const {
    return __builtin_amdgcn_raw_buffer_load_b128(buffer, offset, 0, 0);
  }
  DEV_INLINE void put(unsigned offset, const u32x4_t& w, bool past) const {
    constexpr int PAST = 17;           // (sc0 and sc1)
    if (past) __builtin_amdgcn_raw_buffer_store_b128(w, buffer, offset, 0, PAST);
    else __builtin_amdgcn_raw_buffer_store_b128(w, buffer, offset, 0, 0);
  }
};

// A tile's sums as rows of bf16 numbers
template <int J>
struct TileRows {
  static constexpr int COLS = 2, STORES = 4;
  static constexpr int column_of(int q, int e) { return 2 * q + e; }
  OutRows to;
  unsigned offset[4];
  bool past;
  DEV_INLINE void start(bf16_t* out, long rows, long cols, const Place& at, long col0) {
    const int lane = threadIdx.x & 63, wid = wave_id();
    to.start(out, rows, cols, (long)at.row * (32 * J) + (wid & 1) * (16 * J));
    past = 2 * rows * cols < L2_OUT;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      offset[q] = OutRows::offset(
          cols, col0 + (wid >> 1) * 128 + 32 * q + 8 * (lane >> 4));
  }
  DEV_INLINE void rows(int) { to.next(); }
  DEV_INLINE void put(int, int q, const f32x4_t (&sums)[2]) const {
    to.put(offset[q], eight_columns(sums[0], sums[1]), past);
  }
};

// Rows of a tile whose left operand is LINES, in 32s from LEAST on (6 where the right one
// is COLUMNS): as many as end the last round of 256 tiles earliest.  A unit of 64 inner
// numbers costs 0.105 us a row part and 0.25 for the columns' fragments and loads (0.19 of
// the tiles with three pairs of units in LDS), a tile 5 us more.  (1024 -> 4096, tiles of 128, 192, 224 and 256 rows: 5135 rows 89.2, 81.4,
// 74.0, 81.0 us; 1500 rows 30.0, 24.7, 26.8, 28.8; 1024 rows 18.5, 22.8, 24.0, 25.8; 3072
// rows, 1536 -> 8960, 145, 142, 136, 147; 5135 rows, 4096 -> 14336, 1068, 875, 868, 888; the
// gradient of 7168 rows through 14336 x 4096, 192 to 256 rows a tile, 703, 539, 573, of 8192
// 767, 748, 615.)
struct Rows {
  int parts;
  long cost;
};
inline long cost_of(int parts, long inner) {
  return inner / PAIR * (10 * parts + (parts <= 5 ? 18 : 24)) + 480;
}
inline Rows rows_of(long rows, long cols, long inner, int least) {
  Rows best{8, -1};
  for (int j = least; j <= 8; ++j) {
    const long items = (rows + 32 * j - 1) / (32 * j) * cols;
    const long cost = (items + CUS - 1) / CUS * cost_of(j, inner);
    if (best.cost < 0 || cost <= best.cost) best = {j, cost};
  }
  return best;
}

// Blocks: as many as run at once, each with its tiles one after the other, but of few
// units a tile a block each
inline long blocks_of(long items, long inner) {
  const long most = inner >= 4 * PAIR ? CUS : items;
  return (std::min(items, most) + ATTN_XCDS - 1) / ATTN_XCDS * ATTN_XCDS;
}

}  // namespace product
