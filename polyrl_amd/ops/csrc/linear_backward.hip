// Weight gradients of the trainer's projections, bf16 with fp32 sums: dW = dY^T X,
// (N, K) from (M, N) and (M, K).
//
// Reference capability: the weight gradients of the update loop's projections.
//
// Split.  A block owns 256 x 256 outputs, four waves 128 x 128 each: 256 accumulator
// registers a lane, 128 more for the fragments of two steps, one wave a SIMD, one block
// a CU.  The inner dimension runs over the memory's rows in both operands.  A stage is 32
// rows of 256 columns of both, 32 KiB, straight into LDS, four stages' room; fragments
// come from there by transposed loads (ds_read_b64_tr_b16) that leave a lane eight rows
// of its column.  A row's 512 bytes stand in windows of 32 that are turned by the row,
// so that eight rows of a window meet no bank twice.
//
// Schedule.  One wave a SIMD has nobody to take its turn: the order is fixed instruction
// by instruction (order()).  Behind each of a step's 64 v_mfma_f32_16x16x32_bf16, 16
// cycles each, stands at most one of the next step's 32 fragment reads, of the 8 loads
// four stages ahead, of the words that say where a load goes, or of the next step's
// addresses; a barrier a step.
//
// What bounds it: the power that the card may draw.  Of random numbers 8192^3 takes 707
// us (1550 TFLOP/s), matrix cores busy in 80% of the cycles at 1.85 GHz; of zeros 541 at
// 2.34 GHz.  v_mfma_f32_32x32x16_bf16 in such a loop is as busy (83%), but the clock
// falls to 1.63 GHz: 763 us; with order and addresses left to the compiler 865.  The
// library's best algorithm takes 1028.  8192 rows, 14336 x 4096, 4096 x 4096, 8960 x
// 1536, 1024 x 4096: 702, 175, 160, 68 us for 887, 227, 234, 84.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "attention_tile.h"

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int SIDE = 256;              // outputs of a block, each way
constexpr int INNER = 32;              // rows of a stage
constexpr int STAGES = 4;
constexpr int PART = SIDE * INNER * 2; // bytes of an operand's stage
constexpr int STAGE = 2 * PART;
constexpr int LOADS = 8;               // of a wave and stage, 1 KiB each
constexpr int CUS = 256;
constexpr int GROUP = 8;               // rows of tiles that a die walks together

// 256 columns from ``first`` of an operand's rows from ``row0`` on.  Rows behind the
// last are 0; columns behind the last one are the next row's, and whoever reads them
// stores nothing.
struct Columns {
  u32x4_t from;                        // buffer descriptor
  unsigned step;                       // bytes from stage to stage
  unsigned at[LOADS / 2];              // of this lane's loads
  int frag_at[8];                      // this lane's place in 16 columns, slot 0

  // place of a 32-byte window: its number, turned by this
  DEV_INLINE static int turn(int r) { return (r & 3) | ((r >> 3) & 1) << 2; }

  DEV_INLINE Columns(const bf16_t* p, long rows, long cols, long row0, long first,
                     const char* tile, int half) {
    const long skip = row0 * cols + first;
    const uint64_t base = (uint64_t)(p + skip);
    const unsigned ldb = (unsigned)cols * 2;
    step = INNER * ldb;
    from = {(unsigned)uniform((int)base),
            (unsigned)uniform((int)(base >> 32)) & 0xffffu,
            (unsigned)uniform((int)(2 * (rows * cols - skip))), 0x00020000u};
    // (a scalar that a vector instruction wrote is not to be used at once)
    asm volatile("s_nop 4" : "+s"(from), "+s"(step));
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < LOADS / 2; ++i) {
      const int r = wave_id() * 8 + i * 2 + (lane >> 5);
      at[i] = r * ldb + (((lane & 31) ^ (turn(r) << 1)) << 4);
    }
    const int c = lane & 15, r = 8 * (lane >> 4) + (c >> 2);
#pragma unroll
    for (int d = 0; d < 8; ++d)
      frag_at[d] = (int)(uintptr_t)(lds_p)tile + half * 256 + r * 512 +
                   ((d ^ turn(r)) << 5) + (c & 3) * 8;
  }

  // A load in two instructions, both in assembly, so that the compiler does not
  // wait for it on its own account; no register is written.
  DEV_INLINE static void aim(unsigned to) {
    asm volatile("s_mov_b32 m0, %0" ::"s"(to) : "m0");
  }
  DEV_INLINE void go(int i) const {
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(at[i]), "s"(from)
                 : "memory");
  }
  DEV_INLINE void load(unsigned to) {  // a stage
#pragma unroll
    for (int i = 0; i < LOADS / 2; ++i) {
      aim(to + i * 1024);
      asm volatile("s_nop 0");
      go(i);
    }
    next();
  }
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

// 16 columns, 32 rows: of lane l column l % 16, rows from 8 * (l / 16)
struct Frag {
  i16x4_t half[2];
  template <int H>
  DEV_INLINE void read(int at) {
    half[H] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_i16x4_p)(uintptr_t)(at + H * 2048));
  }
  DEV_INLINE i16x8_t whole() const {
    return __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
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

// out (N, K) = L (M, N)^T R (M, K).  ``ways`` blocks share a tile's rows, whose fp32
// sums (tiles, ways, SIDE * SIDE) are added up afterwards.
__global__ __launch_bounds__(256, 1) void wgrad_kernel(
    bf16_t* __restrict__ out, float* __restrict__ shares,
    const bf16_t* __restrict__ left, const bf16_t* __restrict__ right, long M,
    long N, long K, int row_tiles, int col_tiles, int ways) {
  __shared__ __attribute__((aligned(1024))) char lds[STAGES * STAGE];
  const int tiles = row_tiles * col_tiles, item = die_item(tiles * ways);
  if (item >= tiles * ways) return;
  const int part = item / tiles, tile = item - part * tiles;
  const Place place(tile, row_tiles, col_tiles);
  const long r0 = (long)place.row * SIDE, c0 = (long)place.col * SIDE;
  // (an even number of stages; what is behind the last row is 0)
  const int all = (int)((M + 2 * INNER - 1) / (2 * INNER));
  const int s0 = 2 * (int)((long)all * part / ways);
  const int s1 = 2 * (int)((long)all * (part + 1) / ways);

  const int lane = threadIdx.x & 63, wid = wave_id();
  const int wr = wid & 1, wc = wid >> 1;
  Columns a(left, M, N, (long)s0 * INNER, r0, lds, wr);
  Columns b(right, M, K, (long)s0 * INNER, c0, lds + PART, wc);
  const unsigned to0 = (unsigned)(uintptr_t)(lds_p)lds + wid * 4096;

  f32x4_t acc[8][8];                   // columns, rows
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int i = 0; i < STAGES; ++i) {
    a.load(to0 + i * STAGE);
    b.load(to0 + i * STAGE + PART);
  }
  Frag fa[2][8], fb[2][8];
  int na[8], nb[8];                    // where the next step's fragments are
  arrived<LOADS * (STAGES - 1)>();
#pragma unroll
  for (int d = 0; d < 8; ++d) {
    fa[0][d].read<0>(a.frag_at[d]), fa[0][d].read<1>(a.frag_at[d]);
    fb[0][d].read<0>(b.frag_at[d]), fb[0][d].read<1>(b.frag_at[d]);
    na[d] = a.frag_at[d] + STAGE, nb[d] = b.frag_at[d] + STAGE;
  }

  // The products of a stage, whose fragments are registers N, and the reads of the
  // next one's.  Its slot, ``slot``, which all waves have read, takes the stage four
  // ahead; ``after`` is the slot of the stage two ahead.  (Loads behind the last row
  // read nothing: the count of them is the same in every step.)
  auto step = [&](auto n_, int slot, int after) {
    constexpr int N_ = decltype(n_)::value, O = 1 - N_;
    __builtin_amdgcn_s_waitcnt(0xc07f);            // fragments: lgkmcnt(0)
    arrived<LOADS * (STAGES - 2)>();
    const unsigned to = to0 + slot;
#pragma unroll
    for (int k = 0; k < 64; ++k) {
      const int i = k >> 3, j = i & 1 ? 7 - (k & 7) : k & 7;
      order();
      // In assembly, else the compiler moves accumulators about; but the last eight,
      // of whose results it has to know that they take a while.
      if (i < 7)
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[i][j])
                     : "v"(fb[N_][i].whole()), "v"(fa[N_][j].whole()));
      else
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, fb[N_][i].whole()),
            __builtin_bit_cast(bf16x8_t, fa[N_][j].whole()), acc[i][j], 0, 0, 0);
      order();
      const int f = k / 3;             // fragment: one column's, all rows', the rest
      if (k < 48 && k % 3 < 2) {
        if (f >= 1 && f <= 8) {
          if (k % 3 == 0) fa[O][f - 1].template read<0>(na[f - 1]);
          else fa[O][f - 1].template read<1>(na[f - 1]);
        } else {
          const int d = f == 0 ? 0 : f - 8;
          if (k % 3 == 0) fb[O][d].template read<0>(nb[d]);
          else fb[O][d].template read<1>(nb[d]);
        }
      } else if (k < 48) {
        const int l = f / 2;
        if (f % 2 == 0)
          Columns::aim(to + l % 4 * 1024 + (l >= 4 ? PART : 0));
        else if (l < 4)
          a.go(l);
        else
          b.go(l - 4);
      } else {
        const int d = k & 7;
        int& next = k < 56 ? na[d] : nb[d];
        next = (k < 56 ? a : b).frag_at[d] + after;
        asm volatile("" : "+v"(next));
        if (k == 50) a.next();
        if (k == 54) b.next();
      }
    }
  };
  static_assert(STAGES == 4, "the slots of a pair of steps");
  int slot = 0;
  for (int s = s0; s < s1; s += 2) {
    const int other = slot ^ (2 * STAGE);
    step(std::integral_constant<int, 0>(), slot, other);
    step(std::integral_constant<int, 1>(), slot + STAGE, other + STAGE);
    slot = other;
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
  if (c >= K) return;
#pragma unroll 8
  for (int k = 0; k < 32; ++k) {
    const int row = k * 4 + (lane >> 4);
    const long r = r0 + wr * 128 + row;
    if (r < N)
      *reinterpret_cast<u32x4_t*>(out + r * K + c) =
          *reinterpret_cast<const u32x4_t*>(mine + row * 256 +
                                            ((g ^ (row & 15)) << 4));
  }
}

// Sums of the shares: a wave takes 16 rows of 32 outputs
__global__ __launch_bounds__(256) void wgrad_sum_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ shares, long N, long K,
    int row_tiles, int col_tiles, int ways) {
  const int lane = threadIdx.x & 63;
  const int sub = (blockIdx.x & 31) * 4 + wave_id();   // (wave, i / 2, j) of a tile
  const int tile = blockIdx.x >> 5;
  const int wid = sub >> 5, i = sub >> 3 & 3, j = sub & 7;
  const Place place(tile, row_tiles, col_tiles);
  const long r = (long)place.row * SIDE + (wid & 1) * 128 + j * 16 + (lane & 15);
  const long c = (long)place.col * SIDE + (wid >> 1) * 128 + i * 32;
  const f32x4_t* p =
      reinterpret_cast<const f32x4_t*>(shares + (long)tile * ways * SIDE * SIDE) +
      wid * 4096 + (i * 16 + j) * 64 + lane;
  f32x4_t sum[2] = {p[0], p[512]};
#pragma unroll 2
  for (int w = 1; w < ways; ++w) {
    p += SIDE * SIDE / 4;
    sum[0] += p[0], sum[1] += p[512];
  }
  if (r >= N) return;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const long at = c + 16 * h + 4 * (lane >> 4);
    bf16x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w.v[e] = f2bf(sum[h][e]);
    if (at < K) *reinterpret_cast<bf16x4*>(out + r * K + at) = w;
  }
}

// 16-byte granules, offsets of 32 bits
bool operands_fit(const torch::Tensor& dy, const torch::Tensor& x) {
  const long M = dy.size(0), N = dy.size(1), K = x.size(1);
  return M > 0 && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0 &&
         M * std::max(N, K) * 2 < (1L << 32) &&
         (((uintptr_t)dy.data_ptr() | (uintptr_t)x.data_ptr()) & 15) == 0;
}

// Blocks of a tile: as many as run at once, but each with some hundred rows, for the
// shares' trip through memory (8192 rows: 64 tiles 130, 83, 69, 68 us with 1 to 4 blocks
// a tile; 16 tiles 74, 45, 34, 34, 39 with 2, 4, 8, 12, 16)
long wgrad_ways(long tiles, long M) {
  return std::max(1L, std::min(CUS / tiles, M / 640));
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
  if (!operands_fit(dy, x)) return false;
  const long M = dy.size(0), N = dy.size(1), K = x.size(1);
  const long tiles = ((N + SIDE - 1) / SIDE) * ((K + SIDE - 1) / SIDE);
  return tiles >= 160 ? M >= 512 : M >= 5120;
}

// dW = dY^T X
torch::Tensor linear_wgrad(torch::Tensor dy, torch::Tensor x) {
  for (const auto* t : {&dy, &x})
    TORCH_CHECK(t->is_cuda() && t->device() == dy.device() && t->dim() == 2 &&
                    t->is_contiguous() && t->dtype() == torch::kBFloat16,
                "linear_wgrad: contiguous 2-D bf16 of one device");
  TORCH_CHECK(x.size(0) == dy.size(0) && operands_fit(dy, x),
              "linear_wgrad: rows in 16-byte granules, at most 4 GiB");
  const long M = dy.size(0), N = dy.size(1), K = x.size(1);
  auto dw = torch::empty({N, K}, dy.options());
  const long row_tiles = (N + SIDE - 1) / SIDE, col_tiles = (K + SIDE - 1) / SIDE;
  const long tiles = row_tiles * col_tiles, ways = wgrad_ways(tiles, M);
  const long items = tiles * ways;
  const long grid = (items + ATTN_XCDS - 1) / ATTN_XCDS * ATTN_XCDS;
  TORCH_CHECK(grid < (1L << 31), "grid too large");
  torch::Tensor shares;
  if (ways > 1)
    shares = torch::empty({items * SIDE * SIDE},
                          dw.options().dtype(torch::kFloat32));
  float* sums = ways > 1 ? shares.data_ptr<float>() : nullptr;
  auto stream = at::hip::getCurrentHIPStream();
  wgrad_kernel<<<dim3((unsigned)grid), dim3(256), 0, stream>>>(
      (bf16_t*)dw.data_ptr(), sums, (const bf16_t*)dy.data_ptr(),
      (const bf16_t*)x.data_ptr(), M, N, K, (int)row_tiles, (int)col_tiles,
      (int)ways);
  if (ways > 1)
    wgrad_sum_kernel<<<dim3((unsigned)tiles * 32), dim3(256), 0, stream>>>(
        (bf16_t*)dw.data_ptr(), sums, N, K, (int)row_tiles, (int)col_tiles,
        (int)ways);
  HIP_CHECK_KERNEL();
  return dw;
}
