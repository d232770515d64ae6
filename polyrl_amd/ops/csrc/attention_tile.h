// Tiles of the matrix-core attention kernels (attention_prefill.hip,
// attention_backward_v3.hip, seq_gqa_mfma.hip; the swizzle in
// attention_decode.hip): 64 rows x D bf16 numbers in LDS, their
// fragments for v_mfma_f32_32x32x16_bf16, and the table of row tiles.
//
// Layout.  A tile row is D numbers in 16-byte granules; granule g of row r
// lies at place g ^ swz(r).  Two kinds of reads are free of bank conflicts
// (64 banks of 4 bytes):
//   * rows as they are (frag_rows, ds_read_b128): 16 neighbouring rows read
//     the same granule, so the places of 16 rows must differ;
//   * columns (frag_cols, ds_read_b64_tr_b16): four neighbouring rows read
//     the same 64 bytes, so their 64-byte windows must differ: the window
//     bits of swz come from the row's lowest bits.
//
// Operands.  32x32x16: lane l holds row (A) or column (B) l % 32 and eight
// numbers of the inner dimension from 8 * (l / 32); accumulator register r
// is row 8 * (r / 4) + 4 * (l / 32) + r % 4 of column l % 32.  A product's
// inner order is free as long as both operands use the same one, so an
// accumulator, rounded to bf16, is at once the B operand of the next product:
// registers 8s .. 8s+7 are inner step s, in the order that frag_cols reads.
#pragma once

#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) int i32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4_t;
typedef __attribute__((ext_vector_type(4))) short i16x4_t;
typedef __attribute__((ext_vector_type(8))) short i16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((address_space(3))) i16x4_t* lds_i16x4_p;
typedef __attribute__((address_space(3))) void* lds_p;
typedef __attribute__((address_space(1))) const void* global_p;

#define ATILE 64                      // rows of a tile
#define ATTN_XCDS 8                   // dies, each with an L2 of its own

DEV_INLINE int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

template <int D>
struct AttnTile {
  static constexpr int BYTES = ATILE * D * 2;
  static constexpr int GR = D / 8;    // granules of a row
  static constexpr int LOADS = ATILE * GR / 256;  // granules per thread

  DEV_INLINE static int swz(int r) {
    return D == 128 ? ((r & 3) << 2) | ((r >> 2) & 3)
                    : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
  }

  // Rows [0, min(live, 64)) of one head straight into a tile, zeros behind them
  // (a weight of 0 meets them, and 0 * inf is NaN): the buffer ends with the last
  // row's granules of this head, and what a lane asks for behind it is not read
  // and is 0.  No registers on the way: a wave's lanes write neighbouring
  // granules, so the swizzle is in which granule of its row a lane asks for.  In
  // flight until wait_loads().  The tiles that are read meanwhile have to be
  // another array, else the compiler waits before it reads.
  DEV_INLINE static void copy(char* tile, const bf16_t* rows0, long ld,
                              int live) {
    const int ldb = (int)ld * 2;
    const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(rows0), 0,
        live > 0 ? (min(live, ATILE) - 1) * ldb + 2 * D : 0, 0x00020000);
    const int r = threadIdx.x / GR, g = threadIdx.x % GR;
    int at = r * ldb + ((g ^ swz(r)) << 4);
    char* to = tile + uniform(threadIdx.x >> 6) * 1024;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          from, (lds_p)(to + i * 4096), 16, at, 0, 0, 0);
      at += 256 / GR * ldb;              // (whole periods of the swizzle)
    }
  }

  // The same from 64 rows that start ``start[r]`` numbers behind ``base``
  DEV_INLINE static void gather(char* tile, const bf16_t* base,
                                const long* start) {
    // (heads of 128 have no registers left for these through a kernel's loop:
    // new to the compiler they are derived again for every tile)
    int tid = threadIdx.x;
    if constexpr (D == 128) asm volatile("" : "+v"(tid));
    const int r = tid / GR, g = tid % GR;
    const bf16_t* from = base + (g ^ swz(r)) * 8;
    char* to = tile + uniform(threadIdx.x >> 6) * 1024;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds(
          (global_p)(from + start[r + i * (256 / GR)]), (lds_p)(to + i * 4096),
          16, 0, 0);
  }

  // 32 rows of a wave's own, laid out like a tile's, to rows [0, min(live, 32)) of
  // memory: the buffer ends with the last one, and what is behind it is not written.
  // Offsets have 32 bits: ld is below STORE_LD.
  static constexpr long STORE_LD = 1L << 25;
  DEV_INLINE static void store32(const char* rows, bf16_t* to, long ld,
                                 int live) {
    constexpr int RS = 64 / GR;         // rows of a step
    const int ldb = (int)ld * 2;
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
        to, 0, live > 0 ? (min(live, 32) - 1) * ldb + 2 * D : 0, 0x00020000);
    const int lane = threadIdx.x & 63, r = lane / GR, g = lane % GR;
    const int from = r * (2 * D) + ((g ^ swz(r)) << 4);
    int at = r * ldb + (g << 4);
#pragma unroll
    for (int i = 0; i < 32 / RS; ++i) {
      __builtin_amdgcn_raw_buffer_store_b128(
          *reinterpret_cast<const u32x4_t*>(rows + i * RS * (2 * D) +
                                            (from ^ (swz(i * RS) << 4))),
          out, at, 0, 0);
      at += RS * ldb;
    }
  }

  // zeros for this thread's granules of the rows from ``live`` on
  DEV_INLINE static void clear_from(char* tile, int live) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      if ((int)(threadIdx.x + i * 256) / GR >= live)
        *reinterpret_cast<i32x4_t*>(tile + (threadIdx.x + i * 256) * 16) =
            i32x4_t{0, 0, 0, 0};
  }
};

// Per-lane offsets of the two kinds of fragments.  renew() makes them new to
// the compiler: called once per tile it keeps the sixteen and more derived
// addresses from living in registers through the whole loop.
template <int D>
struct FragAt {
  int rows, cols0, cols1;
  DEV_INLINE FragAt() {
    const int lane = threadIdx.x & 63;
    const int h = lane >> 5, r = lane & 31, c = lane & 15;
    rows = r * (2 * D) + ((h ^ AttnTile<D>::swz(r)) << 4);
    const int ra = 4 * h + (c >> 2), rb = ra + 8;
    const int g = ((lane >> 4) & 1) * 2 + ((c & 3) >> 1);
    cols0 = ra * (2 * D) + ((g ^ AttnTile<D>::swz(ra)) << 4) + (c & 1) * 8;
    cols1 = rb * (2 * D) + ((g ^ AttnTile<D>::swz(rb)) << 4) + (c & 1) * 8;
  }
  DEV_INLINE void renew() {
    asm volatile("" : "+v"(rows), "+v"(cols0), "+v"(cols1));
  }
};

// A operand with the tile's rows [32 * sub, +32) as its rows, inner step ks
// over D
template <int D>
DEV_INLINE bf16x8_t frag_rows(const char* tile, const FragAt<D>& at, int sub,
                              int ks) {
  return *reinterpret_cast<const bf16x8_t*>(
      tile + sub * 32 * (2 * D) + (at.rows ^ (ks << 5)));
}

// A operand with the tile's columns [32 * dt, +32) as its rows, inner step s
// over the tile's rows [16 * s, +16) in the accumulators' order
template <int D>
DEV_INLINE bf16x8_t frag_cols(const char* tile, const FragAt<D>& at, int dt,
                              int s) {
  const char* p = tile + s * 16 * (2 * D);
  const i16x4_t a = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_i16x4_p)(p + (at.cols0 ^ (dt << 6))));
  const i16x4_t b = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_i16x4_p)(p + (at.cols1 ^ (dt << 6))));
  const i16x8_t v = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8_t, v);
}

// row (or column) fragments of one head straight from memory: lane l holds
// row l % 32 of 32 rows, numbers 16 * ks + 8 * (l / 32) ..
template <int D>
DEV_INLINE void frag_global(bf16x8_t (&f)[D / 16], const bf16_t* row) {
  const int h = (threadIdx.x & 63) >> 5;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
    f[ks] = *reinterpret_cast<const bf16x8_t*>(row + ks * 16 + h * 8);
}

// B operand from accumulator registers 8s .. 8s+7
DEV_INLINE bf16x8_t acc_operand(const f32x16_t& c, int s) {
  bf16x8_t v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (__bf16)c[8 * s + j];
  return v;
}

// the larger / the sum of a lane's value and that of the lane 32 away
DEV_INLINE float half_max(float x) {
  const auto p = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
DEV_INLINE float half_sum(float x) {
  const auto p = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}

// a * b, never fused with what it is added to
DEV_INLINE float rounded_product(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}

// 2^x in one instruction; results below 2^-126 become 0
DEV_INLINE float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

// Order of a stretch of straight-line code: ``n`` of the named kind next.  Left
// to itself the compiler reads one fragment, waits for it and multiplies, so
// that every product pays the LDS latency.
#define SCHED_MFMA(n) __builtin_amdgcn_sched_group_barrier(0x008, n, 0)
#define SCHED_LDS(n) __builtin_amdgcn_sched_group_barrier(0x100, n, 0)

// all loads so far are there.  Before a loop with loads in flight: the wait
// for a register that was loaded before the loop would otherwise stand inside
// it and catch the loop's own loads.
DEV_INLINE void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// all but the last N (at most 15)
template <int N>
DEV_INLINE void wait_all_but() { __builtin_amdgcn_s_waitcnt(0x0F70 | N); }

// Sequence and first row of row tile ``tile``.  With a table it is looked
// up; without one the tiles are the sequences' 64-row pieces in order, found
// from cu_q by one scan (64 sequences a step), so that a caller that does
// not know the lengths on the host launches rows / 64 + sequences tiles and
// the ones past the last return false.
DEV_INLINE bool find_tile(int tile, const int* tile_seq, const int* tile_r0,
                          const int* cu, int nseq, int& seq, int& r0) {
  if (tile_seq != nullptr) {
    seq = uniform(tile_seq[tile]);
    r0 = uniform(tile_r0[tile]);
    return true;
  }
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int s0 = 0; s0 < nseq; s0 += 64) {
    const int s = s0 + lane;
    const int n = s < nseq ? (cu[s + 1] - cu[s] + ATILE - 1) / ATILE : 0;
    int upto = n;                      // tiles of sequences s0 .. s
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(upto, off, 64);
      if (lane >= off) upto += o;
    }
    const unsigned long long past = __ballot(before + upto > tile);
    if (past) {
      const int l = __ffsll((long long)past) - 1;
      seq = uniform(s0 + l);
      r0 = (tile - __builtin_amdgcn_readlane(before + upto - n, l)) * ATILE;
      return true;
    }
    before += __builtin_amdgcn_readlane(upto, 63);
  }
  return false;
}

// sum over the wave's lanes, the same in all of them
DEV_INLINE int wave_total(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false); // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false); // row_bcast:31
  return __builtin_amdgcn_readlane(x, 63);
}

// Row tile of block ``t`` of ``ntiles``, and its sequence's rows and keys; false
// past the last.
//
// Of at most 64 sequences: in the order of their walks, longest first.  A causal
// walk is as long as the row tile is late (EARLY: the walk over the query tiles
// that see a key tile, as it is early), so the order of the table, sequence after
// sequence, starts a longest block when most of the chip is done: two sequences of
// 3500 .. 4096, 28/4 heads of 128, kept 1.3 of two waves a SIMD on average.
// ``above(L)`` counts the tiles whose walk is longer than L tiles.  A table of as
// many tiles as the sequences have is read at the place that this tile has in
// the sequences' order, so that every entry is taken once, whatever it names (the
// lengths are on their way meanwhile, in case it names this tile: one wait after
// the other cost 64 sequences of 33 .. 128, 32/8 heads of 128, 95.8 -> 100.7 us).
// Up to 16 sequences the count is taken for 64 lengths at once, one a lane, five
// instructions a sequence; of more a search by halves sums over the lanes ten times.
// (With blocks that find their heads and parts without divisions, and rows written
// by stores that end with the buffer, timed in turn on one card: eight prompts of 1200
// .. 2048, 32/8 heads of 64, 149.7 -> 147.5 us; 16 sequences of 300 .. 512, 32/8 of 128,
// forward and backward 225 -> 221; one prompt of 512 15.4 -> 14.7.)
//
// In the table's order, from the end where late tiles walk longest: tables of
// another length (of some of the tiles), more sequences than lanes, and calls
// whose blocks all start at once, no two on a CU, or whose walks are one tile
// each, where order is worth less than the time to find it (backward of one
// sequence of 300, 8/8 heads of 128: 25.8 us in the order of the walks, 25.1; 64
// sequences of 17 .. 64, 16/4 heads of 64, 24.6 and 24.1; with the line at 512
// blocks 8 of 63 .. 250, 32/8 heads of 128, would take 47.8 for 45.3).
struct RowTile {
  int seq, r0, qbeg, Lq, kbeg, Lk;

  DEV_INLINE void lengths(const int* cu_q, const int* cu_k) {
    qbeg = cu_q[seq], Lq = cu_q[seq + 1] - qbeg;
    kbeg = cu_k[seq], Lk = cu_k[seq + 1] - kbeg;
  }
};

template <bool EARLY>
DEV_INLINE bool row_tile(int t, int ntiles, const int* tile_seq,
                         const int* tile_r0, const int* cu_q, const int* cu_k,
                         int nseq, RowTile& at) {
  auto in_order = [&] {
    if (!find_tile(EARLY ? t : ntiles - 1 - t, tile_seq, tile_r0, cu_q, nseq,
                   at.seq, at.r0))
      return false;
    at.lengths(cu_q, cu_k);
    return true;
  };
  if (nseq > 64 ||
      (tile_seq != nullptr && (gridDim.x <= 256 || ntiles <= nseq)))
    return in_order();
  const int lane = threadIdx.x & 63;
  int n = 0, h = 0;                    // row tiles; key tiles before the first
  if (lane < nseq) {
    const int lq = max(cu_q[lane + 1] - cu_q[lane], 0);
    n = (lq + ATILE - 1) / ATILE;
    if (!EARLY) h = max(cu_k[lane + 1] - cu_k[lane] - lq, 0) / ATILE;
  }
  auto above = [&](int L) { return wave_total(min(max(h + n - L, 0), n)); };
  int lo, longer, total;               // the walk's length less one; above(lo + 1)
  if (nseq <= 16) {
    // 64 lengths at a time, one a lane
    for (int base = 0;; base += 64) {
      int sum = 0;
      for (int s = 0; s < nseq; s += 4)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int ns = __builtin_amdgcn_readlane(n, s + i);
          const int end = __builtin_amdgcn_readlane(h, s + i) + ns;
          sum += min(max(end - (base + lane), 0), ns);
        }
      if (base == 0) {
        total = __builtin_amdgcn_readlane(sum, 0);
        if (total <= t || (tile_seq != nullptr && ntiles != total)) break;
      }
      const unsigned long long more = __ballot(sum > t);
      if (more == ~0ull) continue;
      const int c = __popcll(more);
      lo = base + c - 1;
      longer = __builtin_amdgcn_readlane(sum, c);
      break;
    }
    if (tile_seq != nullptr && ntiles != total) return in_order();
    if (total <= t) return false;
  } else {
    total = above(0);
    if (tile_seq != nullptr && ntiles != total) return in_order();
    if (total <= t) return false;
    lo = 0;
    int hi = 1;
    while (above(hi) > t) lo = hi, hi *= 2;
    while (hi - lo > 1) {
      const int mid = (lo + hi) / 2;
      if (above(mid) > t) lo = mid;
      else hi = mid;
    }
    longer = above(lo + 1);
  }
  // of the sequences with a tile of this length, the one that t stands for
  const int which = t - longer;
  const unsigned long long has = __ballot(h <= lo && lo < h + n);
  const int rank = __builtin_amdgcn_mbcnt_hi(
      (unsigned)(has >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)has, 0));
  const unsigned long long me =
      __ballot((has >> lane & 1) && rank == which);
  at.seq = __ffsll((long long)me) - 1;
  const int nth = EARLY ? __builtin_amdgcn_readlane(n, at.seq) - 1 - lo
                        : lo - __builtin_amdgcn_readlane(h, at.seq);
  at.r0 = nth * ATILE;
  at.lengths(cu_q, cu_k);
  if (tile_seq != nullptr) {
    const int i = wave_total(lane < at.seq ? n : 0) + nth;
    const int seq = uniform(tile_seq[i]), r0 = uniform(tile_r0[i]);
    if (seq != at.seq || r0 != at.r0) {
      at.seq = seq, at.r0 = r0;
      at.lengths(cu_q, cu_k);
    }
  }
  return true;
}

// id / n and id % n of uniform numbers (heads and parts are mostly powers of two)
DEV_INLINE int split_id(int id, int n, int& rest) {
  if ((n & (n - 1)) == 0) {
    rest = id & (n - 1);
    return id >> __builtin_ctz(n);
  }
  rest = (unsigned)id % (unsigned)n;
  return (unsigned)id / (unsigned)n;
}

// Tile, part of it and key/value head of a block: the head innermost, and the
// parts, which are not equal, turning from tile to tile
struct BlockItem {
  int tile, part, head;
  DEV_INLINE BlockItem(int heads, int parts) {
    int turn;
    tile = split_id(split_id(blockIdx.x, heads, head), parts, turn);
    split_id(turn + tile, parts, part);
  }
};

// wave of the block, known to the compiler to be the same for all its lanes
DEV_INLINE int wave_id() {
  return uniform(threadIdx.x >> 6);
}

// Work item of a block of the window kernel.  Blocks go to the dies in turn
// (id % 8); each die takes one stretch of the items, whose order is key/value
// head, row tile, part, so the tiles that read the same keys share an L2.
DEV_INLINE int die_item(int items) {
  const int per = (items + ATTN_XCDS - 1) / ATTN_XCDS;
  return (int)(blockIdx.x % ATTN_XCDS) * per + (int)(blockIdx.x / ATTN_XCDS);
}

// Rows for AttnTile::copy, 16 bytes a lane: a tensor whose rows do not all start
// at 16-byte addresses is laid out again.
inline torch::Tensor rows_by16(const torch::Tensor& t) {
  const bool ok = ((uintptr_t)t.data_ptr() & 15) == 0 &&
                  (t.stride(0) % 8 == 0 || t.size(0) < 2);
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}
