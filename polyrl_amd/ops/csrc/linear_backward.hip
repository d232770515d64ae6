// Products of the trainer's backward pass, bf16 with fp32 sums: weight gradients dW =
// dY^T X, (N, K) from (M, N) and (M, K), and input gradients dX = dY W, (M, K) from (M, N)
// and (N, K).
//
// Reference capability: the gradients of the update loop's projections.
//
// Split.  A block owns 256 x 256 outputs, four waves 128 x 128 each: 256 accumulator
// registers a lane, 128 more for the fragments of two steps, one wave a SIMD, one block
// a CU.  A step is 32 inner numbers, 16 KiB of each operand, straight into LDS, four
// steps ahead.  Where the inner dimension runs over the memory's rows (COLUMNS: W, and
// both operands of dW) fragments come from LDS by transposed loads
// (ds_read_b64_tr_b16); where it is the rows' own (LINES: dY in dX) as they are, and
// two steps' are loaded as one, so that a row's piece is a whole line of 128 bytes
// (pieces of 64, loads of one step alone, take 30% longer).
//
// Schedule.  One wave a SIMD has nobody to take its turn: the order is fixed instruction
// by instruction (order()).  Behind each of a step's 64 v_mfma_f32_16x16x32_bf16, 16
// cycles each, stands at most one of the next step's fragment reads, of the 8 loads four
// steps ahead, of the words that say where a load goes, or of the next step's
// addresses; a barrier a step.
//
// What bounds it: the power that the card may draw.  Of random numbers 8192^3 (dW)
// takes 707 us (1550 TFLOP/s), matrix cores busy in 80% of the cycles at 1.85 GHz; of
// zeros 541 at 2.34 GHz.  v_mfma_f32_32x32x16_bf16 in such a loop is as busy (83%), but
// the clock falls to 1.63 GHz: 763 us; with order and addresses left to the compiler 865.
// The library's best algorithm takes 1028.  8192 rows, dW of 14336 x 4096, 4096 x 4096,
// 8960 x 1536, 1024 x 4096: 702, 175, 160, 68 us for 887, 227, 234, 84; dX through 14336 x
// 4096, 4096 x 4096, 8960 x 1536, 128256 x 2048: 614, 184, 159, 2760 for 690, 202, 179, 3149,
// of 256 rows through the latter 137 for 343.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "attention_tile.h"

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int SIDE = 256;              // outputs of a block, each way
constexpr int INNER = 32;              // inner numbers of a step
constexpr int PART = SIDE * INNER * 2; // bytes of an operand's step
constexpr int STAGES = 4;              // steps of COLUMNS in LDS
constexpr int PAIRS = 3;               // pairs of steps of LINES in LDS
constexpr int LOADS = 8;               // of a wave and step, 1 KiB each
constexpr int CUS = 256;
constexpr int GROUP = 8;               // rows of tiles that a die walks together

// One of a product's operands, 256 of its outer numbers from ``first`` on.  LINES: its
// inner numbers are the memory's rows'; COLUMNS: they run over the memory's rows.
// What is behind the operand's end is 0; columns behind the last one are the next
// row's, and whoever reads them stores nothing.
template <bool LINES>
struct Operand {
  static constexpr int CHUNKS = LINES ? 8 : 4;     // loads that differ
  static constexpr int FRAGS = LINES ? 2 : 8;
  u32x4_t from;                        // buffer descriptor
  unsigned step;                       // bytes to the next step (LINES: two steps)
  unsigned at[CHUNKS];                 // of this lane's loads
  int frag_at[FRAGS];  // this lane's place, slot 0, in 16 columns (LINES: in a half)

  // COLUMNS: a row's 512 bytes stand in windows of 32, turned by the row, so that
  // eight rows of a window meet no bank twice
  DEV_INLINE static int turn(int r) { return (r & 3) | ((r >> 3) & 1) << 2; }
  // LINES: rows of 64 inner numbers, 128 bytes, whose granules are turned by the row,
  // so that 16 rows of a granule meet no bank twice
  DEV_INLINE static int place(int g, int r) { return g ^ (r >> 1 & 7); }

  DEV_INLINE Operand(const bf16_t* p, long outer, long inner, long first,
                     long inner0, const char* tile, int half) {
    const long skip = LINES ? first * inner + inner0 : inner0 * outer + first;
    const uint64_t base = (uint64_t)(p + skip);
    const long bytes = 2 * (outer * inner - skip);
    const unsigned ldb = (unsigned)(LINES ? inner : outer) * 2;
    step = LINES ? 4 * INNER : INNER * ldb;
    from = {(unsigned)uniform((int)base),
            (unsigned)uniform((int)(base >> 32)) & 0xffffu,
            (unsigned)uniform((int)(LINES ? min(bytes, (long)SIDE * ldb) : bytes)),
            0x00020000u};
    // (a scalar that a vector instruction wrote is not to be used at once)
    asm volatile("s_nop 4" : "+s"(from), "+s"(step));
    const int lane = threadIdx.x & 63, wid = wave_id();
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
      if (LINES) {
        const int r = wid * 64 + i * 8 + (lane >> 3);
        at[i] = r * ldb + (place(lane & 7, r) << 4);
      } else {
        const int r = wid * 8 + i * 2 + (lane >> 5);
        at[i] = r * ldb + (((lane & 31) ^ (turn(r) << 1)) << 4);
      }
    }
    const int tile_at = (int)(uintptr_t)(lds_p)tile, c = lane & 15, h = lane >> 4;
#pragma unroll
    for (int d = 0; d < FRAGS; ++d) {
      if (LINES) {
        frag_at[d] = tile_at + half * 16384 + c * 128 + (place(4 * d + h, c) << 4);
      } else {
        const int r = 8 * h + (c >> 2);
        frag_at[d] = tile_at + half * 256 + r * 512 + ((d ^ turn(r)) << 5) +
                     (c & 3) * 8;
      }
    }
  }

  // A load in two instructions, both in assembly, so that the compiler does not
  // wait for it on its own account; no register is written.
  DEV_INLINE void go(int i) const {
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(at[i]), "s"(from)
                 : "memory");
  }
  // four of them at once
  template <int FIRST>
  DEV_INLINE void load(unsigned to) const;
  DEV_INLINE void next() {
    unsigned lo = from[0], hi = from[1], left = from[2];
    asm volatile(
        "s_add_u32 %0, %0, %3\n\ts_addc_u32 %1, %1, 0\n\t"
        "s_sub_u32 %2, %2, %3\n\ts_cselect_b32 %2, 0, %2"
        : "+s"(lo), "+s"(hi), "+s"(left)
        : "s"(step)
        : "scc");
    from[0] = lo, from[1] = hi, from[2] = left;
  }
};

DEV_INLINE void aim(unsigned to) {
  asm volatile("s_mov_b32 m0, %0" ::"s"(to) : "m0");
}

template <bool LINES>
template <int FIRST>
DEV_INLINE void Operand<LINES>::load(unsigned to) const {
#pragma unroll
  for (int i = FIRST; i < FIRST + 4; ++i) {
    aim(to + i * 1024);
    asm volatile("s_nop 0");
    go(i);
  }
}

// 16 outer numbers, 32 inner ones: of lane l number l % 16, inner ones from 8 * (l / 16)
struct Frag {
  i16x8_t all;
  i16x4_t half[2];
  template <bool LINES, int H>
  DEV_INLINE void read(int at) {
    typedef __attribute__((address_space(3))) const i16x8_t* lds_i16x8_p;
    if constexpr (!LINES)
      half[H] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_i16x4_p)(uintptr_t)(at + H * 2048));
    else if constexpr (H == 0)
      all = *(lds_i16x8_p)(uintptr_t)at;
  }
  template <bool LINES>
  DEV_INLINE i16x8_t whole() const {
    return LINES ? all
                 : __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

// all but N loads of this wave are there, and all waves are here
template <int N>
DEV_INLINE void arrived() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

DEV_INLINE void order() { __builtin_amdgcn_sched_barrier(0); }

// Row and column of a tile: GROUP rows of tiles, one column after the other
struct Place {
  int row, col;
  DEV_INLINE Place(int tile, int row_tiles, int col_tiles) {
    const int group = tile / (GROUP * col_tiles);
    const int rest = tile - group * GROUP * col_tiles;
    const int high = min(GROUP, row_tiles - group * GROUP);
    row = uniform(group * GROUP + rest % high), col = uniform(rest / high);
  }
};

// out (R, C): sums over inner of left(row, inner) right(inner, column), right in
// COLUMNS.  ``ways`` blocks share a tile's inner numbers, whose fp32 sums (tiles, ways,
// SIDE * SIDE) are added up afterwards.
template <bool LINES>
__global__ __launch_bounds__(256, 1) void product_kernel(
    bf16_t* __restrict__ out, float* __restrict__ shares,
    const bf16_t* __restrict__ left, const bf16_t* __restrict__ right, long R,
    long C, long inner, int row_tiles, int col_tiles, int ways) {
  constexpr int SLOT = LINES ? 2 * PART : PART;    // of the left operand
  constexpr int B0 = LINES ? PAIRS * SLOT : STAGES * SLOT;
  __shared__ __attribute__((aligned(1024))) char lds[B0 + STAGES * PART];
  const int tiles = row_tiles * col_tiles, item = die_item(tiles * ways);
  if (item >= tiles * ways) return;
  const int part = item / tiles, tile = item - part * tiles;
  const Place at_tile(tile, row_tiles, col_tiles);
  const long r0 = (long)at_tile.row * SIDE, c0 = (long)at_tile.col * SIDE;
  // (an even number of steps; in COLUMNS what is behind the last row is 0)
  const int all = (int)((inner + 2 * INNER - 1) / (2 * INNER));
  const int p0 = (int)((long)all * part / ways);
  const int pairs = (int)((long)all * (part + 1) / ways) - p0;

  const int lane = threadIdx.x & 63, wid = wave_id();
  const int wr = wid & 1, wc = wid >> 1;
  Operand<LINES> a(left, R, inner, r0, p0 * (2L * INNER), lds, wr);
  Operand<false> b(right, C, inner, c0, p0 * (2L * INNER), lds + B0, wc);
  const unsigned lds0 = (unsigned)(uintptr_t)(lds_p)lds;
  const unsigned a_to = lds0 + wid * (LINES ? 8192 : 4096);
  const unsigned b_to = lds0 + B0 + wid * 4096;

  f32x4_t acc[8][8];                   // columns, rows
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // The loads that the steps before the first would have started, in their order:
  // of LINES two pairs and the first half of a third, of COLUMNS four steps'
  if constexpr (LINES) {
    a.template load<0>(a_to), a.template load<4>(a_to), a.next();
    a.template load<0>(a_to + SLOT);
    b.template load<0>(b_to), b.next();
    b.template load<0>(b_to + PART), b.next();
    a.template load<4>(a_to + SLOT), a.next();
    b.template load<0>(b_to + 2 * PART), b.next();
    a.template load<0>(a_to + 2 * SLOT);
    b.template load<0>(b_to + 3 * PART), b.next();
  } else {
#pragma unroll
    for (int i = 0; i < STAGES; ++i) {
      a.template load<0>(a_to + i * SLOT), a.next();
      b.template load<0>(b_to + i * PART), b.next();
    }
  }
  Frag fa[2][8], fb[2][8];
  int na[LINES ? 1 : 8], nb[8];        // where the next step's fragments are
  arrived<LOADS * (STAGES - 2) + (LINES ? 4 : LOADS)>();
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    const int at = LINES ? a.frag_at[0] + d * 2048 : a.frag_at[LINES ? 0 : d];
    fa[0][d].template read<LINES, 0>(at), fa[0][d].template read<LINES, 1>(at);
    fb[0][d].template read<false, 0>(b.frag_at[d]);
    fb[0][d].template read<false, 1>(b.frag_at[d]);
    if (!LINES) na[LINES ? 0 : d] = a.frag_at[LINES ? 0 : d] + SLOT;
    nb[d] = b.frag_at[d] + PART;
  }
  if (LINES) na[0] = a.frag_at[LINES];

  // The products of a step, whose fragments are registers N, the reads of the next
  // one's, and loads: the left operand's to ``a_slot``, the right one's, of the step
  // four ahead, to ``b_slot``, this step's own, which all waves have read.  ``a_after``,
  // ``b_after``: where the fragments of the step two ahead are.  (Loads behind the end
  // read nothing: the count of them is the same in every step.)
  auto step = [&](auto n_, unsigned a_slot, unsigned b_slot, int a_after,
                  int b_after) {
    constexpr int N = decltype(n_)::value, O = 1 - N;
    constexpr int FIRST = LINES && N == 0 ? 4 : 0;   // (a pair's later half)
    __builtin_amdgcn_s_waitcnt(0xc07f);            // fragments: lgkmcnt(0)
    arrived<LOADS * (STAGES - 2)>();
#pragma unroll
    for (int k = 0; k < 64; ++k) {
      const int i = k >> 3, j = i & 1 ? 7 - (k & 7) : k & 7;
      order();
      // In assembly, else the compiler moves accumulators about; but the last eight,
      // of whose results it has to know that they take a while.
      if (i < 7)
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[i][j])
                     : "v"(fb[N][i].template whole<false>()),
                       "v"(fa[N][j].template whole<LINES>()));
      else
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, fb[N][i].template whole<false>()),
            __builtin_bit_cast(bf16x8_t, fa[N][j].template whole<LINES>()),
            acc[i][j], 0, 0, 0);
      order();
      const int f = k / 3;             // fragment: one column's, all rows', the rest
      if (k < 48 && k % 3 < 2) {
        if (f >= 1 && f <= 8) {
          const int d = f - 1;
          const int at = LINES ? na[0] + d * 2048 : na[LINES ? 0 : d];
          if (k % 3 == 0) fa[O][d].template read<LINES, 0>(at);
          else fa[O][d].template read<LINES, 1>(at);
        } else {
          const int d = f == 0 ? 0 : f - 8;
          if (k % 3 == 0) fb[O][d].template read<false, 0>(nb[d]);
          else fb[O][d].template read<false, 1>(nb[d]);
        }
      } else if (k < 48) {
        const int l = f / 2;
        if (f % 2 == 0)
          aim(l < 4 ? a_slot + (FIRST + l) * 1024 : b_slot + (l - 4) * 1024);
        else if (l < 4)
          a.go(FIRST + l);
        else
          b.go(l - 4);
      } else {
        const int d = k & 7;
        if (k >= 56) {
          nb[d] = b.frag_at[d] + b_after;
          asm volatile("" : "+v"(nb[d]));
        } else if (!LINES || d == 0) {
          // (of a pair's halves the next step but one has this step's)
          int& next = na[LINES ? 0 : d];
          next = a.frag_at[LINES ? N : d] + a_after;
          asm volatile("" : "+v"(next));
        }
        if (k == 50 && (!LINES || N == 0)) a.next();
        if (k == 54) b.next();
      }
    }
  };
  static_assert(STAGES == 4 && PAIRS == 3, "the slots of a pair of steps");
  int bs = 0;                          // the right operand's slot of this pair
  if (LINES) {
    int s0 = 0, s1 = SLOT, s2 = 2 * SLOT;          // this pair's, the next ones'
    for (int p = 0; p < pairs; ++p) {
      const int other = bs ^ (2 * PART);
      step(std::integral_constant<int, 0>(), a_to + s2, b_to + bs, s1, other);
      step(std::integral_constant<int, 1>(), a_to + s0, b_to + bs + PART, s1,
           other + PART);
      bs = other;
      const int s = s0;
      s0 = s1, s1 = s2, s2 = s;
    }
  } else {
    for (int p = 0; p < pairs; ++p) {
      const int other = bs ^ (2 * PART);
      step(std::integral_constant<int, 0>(), a_to + bs, b_to + bs, other, other);
      step(std::integral_constant<int, 1>(), a_to + bs + PART, b_to + bs + PART,
           other + PART, other + PART);
      bs = other;
    }
  }
  arrived<0>();

  // Accumulator r of column part i, row part j: column 16 i + 4 (lane / 16) + r of row
  // 16 j + lane % 16
  if (ways > 1) {
    f32x4_t* p = reinterpret_cast<f32x4_t*>(
                     shares + ((long)tile * ways + part) * SIDE * SIDE) +
                 wid * 4096 + lane;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) p[(i * 8 + j) * 64] = acc[i][j];
    return;
  }
  // through the wave's own 32 KiB to whole rows
  char* mine = lds + wid * 32768;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    order();                           // (else it reads them all first, and spills)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int row = j * 16 + (lane & 15);
      bf16x4 w;
#pragma unroll
      for (int t = 0; t < 4; ++t) w.v[t] = f2bf(acc[i][j][t]);
      *reinterpret_cast<bf16x4*>(mine + row * 256 +
                                 (((i * 2 + (lane >> 5)) ^ (row & 15)) << 4) +
                                 ((lane >> 4) & 1) * 8) = w;
    }
  }
  const int g = lane & 15;
  const long c = c0 + wc * 128 + g * 8;
  if (c >= C) return;
#pragma unroll 8
  for (int k = 0; k < 32; ++k) {
    const int row = k * 4 + (lane >> 4);
    const long r = r0 + wr * 128 + row;
    if (r < R)
      *reinterpret_cast<u32x4_t*>(out + r * C + c) =
          *reinterpret_cast<const u32x4_t*>(mine + row * 256 +
                                            ((g ^ (row & 15)) << 4));
  }
}

// Sums of the shares: a wave takes 16 rows of 32 outputs
__global__ __launch_bounds__(256) void product_sum_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ shares, long R, long C,
    int row_tiles, int col_tiles, int ways) {
  const int lane = threadIdx.x & 63;
  const int sub = (blockIdx.x & 31) * 4 + wave_id();   // (wave, i / 2, j) of a tile
  const int tile = blockIdx.x >> 5;
  const int wid = sub >> 5, i = sub >> 3 & 3, j = sub & 7;
  const Place at_tile(tile, row_tiles, col_tiles);
  const long r = (long)at_tile.row * SIDE + (wid & 1) * 128 + j * 16 + (lane & 15);
  const long c = (long)at_tile.col * SIDE + (wid >> 1) * 128 + i * 32;
  const f32x4_t* p =
      reinterpret_cast<const f32x4_t*>(shares + (long)tile * ways * SIDE * SIDE) +
      wid * 4096 + (i * 16 + j) * 64 + lane;
  f32x4_t sum[2] = {p[0], p[512]};
#pragma unroll 2
  for (int w = 1; w < ways; ++w) {
    p += SIDE * SIDE / 4;
    sum[0] += p[0], sum[1] += p[512];
  }
  if (r >= R) return;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const long at = c + 16 * h + 4 * (lane >> 4);
    bf16x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w.v[e] = f2bf(sum[h][e]);
    if (at < C) *reinterpret_cast<bf16x4*>(out + r * C + at) = w;
  }
}

void check_operands(const torch::Tensor& dy, const torch::Tensor& other) {
  for (const auto* t : {&dy, &other})
    TORCH_CHECK(t->is_cuda() && t->device() == dy.device() && t->dim() == 2 &&
                    t->is_contiguous() && t->dtype() == torch::kBFloat16,
                "linear backward: contiguous 2-D bf16 of one device");
}

bool at_granules(const torch::Tensor& dy, const torch::Tensor& other) {
  return (((uintptr_t)dy.data_ptr() | (uintptr_t)other.data_ptr()) & 15) == 0;
}

// 16-byte granules, offsets of 32 bits
bool wgrad_fits(const torch::Tensor& dy, const torch::Tensor& x) {
  const long M = dy.size(0), N = dy.size(1), K = x.size(1);
  return M > 0 && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0 &&
         M * std::max(N, K) * 2 < (1L << 32) && at_granules(dy, x);
}

// and whole pairs of steps, behind which are the next row's numbers
bool dgrad_fits(const torch::Tensor& dy, const torch::Tensor& w) {
  const long M = dy.size(0), N = dy.size(1), K = w.size(1);
  return M > 0 && N > 0 && K > 0 && N % (2 * INNER) == 0 && K % 8 == 0 &&
         N < (1L << 22) && N * K * 2 < (1L << 32) && at_granules(dy, w);
}

long tiles_of(long R, long C) {
  return ((R + SIDE - 1) / SIDE) * ((C + SIDE - 1) / SIDE);
}

// Blocks of a tile: as many as run at once, but each with some hundred inner numbers,
// for the shares' trip through memory (weight gradients of 8192 rows: 64 tiles 130, 83,
// 69, 68 us with 1 to 4 blocks a tile; 16 tiles 74, 45, 34, 34, 39 with 2, 4, 8, 12, 16)
long ways_of(long tiles, long inner) {
  return std::max(1L, std::min(CUS / tiles, inner / 640));
}

template <bool LINES>
torch::Tensor product(const torch::Tensor& left, const torch::Tensor& right, long R,
                      long C, long inner) {
  auto out = torch::empty({R, C}, left.options());
  const long row_tiles = (R + SIDE - 1) / SIDE, col_tiles = (C + SIDE - 1) / SIDE;
  const long tiles = row_tiles * col_tiles, ways = ways_of(tiles, inner);
  const long items = tiles * ways;
  const long grid = (items + ATTN_XCDS - 1) / ATTN_XCDS * ATTN_XCDS;
  TORCH_CHECK(grid < (1L << 31), "grid too large");
  torch::Tensor shares;
  if (ways > 1)
    shares = torch::empty({items * SIDE * SIDE},
                          out.options().dtype(torch::kFloat32));
  float* sums = ways > 1 ? shares.data_ptr<float>() : nullptr;
  auto stream = at::hip::getCurrentHIPStream();
  product_kernel<LINES><<<dim3((unsigned)grid), dim3(256), 0, stream>>>(
      (bf16_t*)out.data_ptr(), sums, (const bf16_t*)left.data_ptr(),
      (const bf16_t*)right.data_ptr(), R, C, inner, (int)row_tiles,
      (int)col_tiles, (int)ways);
  if (ways > 1)
    product_sum_kernel<<<dim3((unsigned)tiles * 32), dim3(256), 0, stream>>>(
        (bf16_t*)out.data_ptr(), sums, R, C, (int)row_tiles, (int)col_tiles,
        (int)ways);
  HIP_CHECK_KERNEL();
  return out;
}

}  // namespace

// Whether linear_wgrad has these operands (contiguous bf16 matrices) and is the better
// choice than the library's best algorithm.  From 160 tiles on, which fill the chip,
// and 512 rows it takes 0.67 to 1.01 of the library's time (14336 x 4096 of 512, 2048
// and 8192 rows: 76, 193, 702 us for 81, 242, 887; 5120 x 2048, 160 tiles, 21, 45, 146
// for 30, 48, 175); fewer tiles are shared among blocks, which pays with many rows
// (1024 x 4096 of 2048, 4096, 8192 rows: 35, 46, 68 for 27, 46, 84; 1536 x 1536 29, 36, 49
// for 25, 44, 80; 4096 x 2048 43, 71, 112 for 39, 69, 132).
bool linear_wgrad_takes(const torch::Tensor& dy, const torch::Tensor& x) {
  const long M = dy.size(0);
  return wgrad_fits(dy, x) &&
         (tiles_of(dy.size(1), x.size(1)) >= 160 ? M >= 512 : M >= 5120);
}

// The same for linear_dgrad, where the library does better.  Tiles that fill two thirds
// of each round of 256 take 0.78 to 1.02 of its time, less full ones up to 1.19 (of 2816,
// 3072, 4096, 4608, 5376 rows through 4096 x 4096, 176 to 336 tiles: 78, 80, 95, 157, 159 us
// for 80, 85, 103, 135, 159); fewer tiles pay where the inner dimension is long enough
// to be shared (256, 1024, 2048 rows through 14336 x 4096 46, 98, 176 for 69, 134, 209;
// through 8192 x 2048 26, 46, 70 for 37, 60, 75; through 4096 x 4096 26, 47, 70 for 25,
// 42, 63).
bool linear_dgrad_takes(const torch::Tensor& dy, const torch::Tensor& w) {
  if (!dgrad_fits(dy, w)) return false;
  const long M = dy.size(0), N = dy.size(1), tiles = tiles_of(M, w.size(1));
  if (tiles <= CUS / 2) return N >= 8192 && M >= 64;
  const long rounds = (tiles + CUS - 1) / CUS;
  return 3 * tiles >= 2 * rounds * CUS - 16;
}

// dW (N, K) = dY^T X of dY (M, N), X (M, K)
torch::Tensor linear_wgrad(torch::Tensor dy, torch::Tensor x) {
  check_operands(dy, x);
  TORCH_CHECK(x.size(0) == dy.size(0) && wgrad_fits(dy, x),
              "linear_wgrad: rows in 16-byte granules, at most 4 GiB");
  return product<false>(dy, x, dy.size(1), x.size(1), dy.size(0));
}

// dX (M, K) = dY W of dY (M, N), W (N, K)
torch::Tensor linear_dgrad(torch::Tensor dy, torch::Tensor w) {
  check_operands(dy, w);
  TORCH_CHECK(w.size(0) == dy.size(1) && dgrad_fits(dy, w),
              "linear_dgrad: N in 64s, rows in 16-byte granules, W at most 4 GiB");
  return product<true>(dy, w, dy.size(0), w.size(1), dy.size(1));
}
