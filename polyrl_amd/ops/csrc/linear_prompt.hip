// Products of prompts (hundreds of rows and more) with a weight's rows, bf16:
// x W^T, and silu(x Wg^T) * (x Wu^T), the gated MLP's two products and its
// activation, in one kernel.
//
// Reference capability: the engine-side projections and the fused gate/up
// projection with its activation.
//
// Split.  A block owns 32 JT rows and 256 columns of the product: those of two
// stretches of 128 rows of the weight, next to each other, or (GLU) 128 of the gate
// and 128 of the up projection, of which it makes 128 outputs.  Eight waves = two
// row groups x four column groups: a wave holds up to 128 rows x (32 + 32 columns)
// in 128 registers, so gate and up of an output meet in one lane.  Weights are
// the A operand of v_mfma_f32_32x32x16_bf16, so that a lane's accumulators are
// neighbouring columns of one row.  Waves w and w + 4 share a SIMD: where JT is
// odd the one has a row tile more than the other and every SIMD the same.
// Tiles of 64 inner numbers, the layout of attention_tile.h (rows of 128
// bytes, no bank conflicts), go straight into LDS, those of W two tiles ahead: one
// block per CU, two waves per SIMD.  Nothing is rounded but the result (the
// products and the activation used to round gate, up and out).
//
// What bounds it: LDS reads and matrix instructions, each about 60% of the cycles,
// and the clock under them; per block 2 to 4 us for the first tiles and the
// activation.  Measured (us in a graph, inputs of twelve layers in turn, against the
// library's product and the activation's pass): 1024 -> 4096 of 513, 1024, 5135 and
// 16384 rows 15.2, 20.0, 85.6, 259 for 21.2, 26.0, 103, 297; 1536 -> 8960 35.9, 64, 263,
// 788 for 42, 81, 288, 867; 2048 -> 8192 44, 62, 313, 930 for 47, 67, 323, 925.  With W
// one tile ahead 5135 rows, 1024 -> 4096, 88.9, 513 rows 16.3, 1024 rows, 1536 -> 8960,
// 71.6.  Reading the fragments of the next 16 inner numbers ahead of the barrier
// takes 5% more, rows in groups of 64 (four row groups, two column groups) the
// same.  x W^T alone, for the library: 1024 -> 1024 of 1024, 4096, 5135 and 8192 rows
// 12.3, 16.6, 19.1, 23.9 for 9.1, 14.7, 21.3, 22.6; 512 -> 1536 8.3, 13.2, 14.8, 21.2 for 9.3,
// 15.0, 16.8, 28.7; 1024 -> 4096 16.3, 37.1, 53.4, 71.5 for 14.4, 31.8, 49.4, 58.2; 2048 -> 3072
// of 1024 and 4096 22, 54 for 20, 47.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "attention_tile.h"

namespace {

typedef AttnTile<64> InTile;           // 64 inner numbers of a row
typedef AttnTile<128> OutTile;         // 128 columns of a row
constexpr int LIN_GROUP = 4;           // column tiles that a die walks together

// ROWS rows of an operand, 64 inner numbers at a time, straight into LDS; rows
// past ``live`` are zeros
template <int ROWS>
struct RowsFrom {
  const char* base;
  int records, ldb, at;

  DEV_INLINE RowsFrom(const bf16_t* rows0, int inner, int live)
      : base(reinterpret_cast<const char*>(rows0)), ldb(inner * 2) {
    records = live > 0 ? min(live, ROWS) * ldb : 0;
    const int r = threadIdx.x / InTile::GR, g = threadIdx.x % InTile::GR;
    at = r * ldb + ((g ^ InTile::swz(r)) << 4);
  }
  // the next tile; zeros, without a look at memory, where there is none
  DEV_INLINE void copy(char* tile, bool more) {
    // In assembly, so that the compiler does not wait for it on its own account:
    // what it knows of such loads tells three buffers apart in some places only, and
    // elsewhere it waits for the next tile before it reads this one.  No register
    // is written; wait_and_meet is the wait.  (Words of the buffer: address,
    // bytes, raw; the pause is for a word that came through a vector register.)
    const uint64_t b = (uint64_t)base;
    const u32x4_t from = {(unsigned)uniform((int)b),
                          (unsigned)uniform((int)(b >> 32)) & 0xffffu,
                          (unsigned)uniform(more ? records : 0), 0x00020000u};
    const unsigned to =
        (unsigned)(uintptr_t)(lds_p)tile + uniform(threadIdx.x >> 6) * 1024;
    int a = at;
#pragma unroll
    for (int i = 0; i < (ROWS + 63) / 64; ++i) {
      asm volatile(
          "s_nop 4\n\t"
          "buffer_load_dwordx4 %1, %2, 0 offen lds" ::"{m0}"(to + i * 8192),
          "v"(a), "s"(from)
          : "memory");
      a += 64 * ldb;                   // (whole periods of the swizzle)
    }
    base += 2 * ATILE;
    records = max(records - 2 * ATILE, 0);
  }
};

// All but the last N loads of this wave are there, and all waves are here: what
// they read from LDS has been read.  (A barrier of the compiler's waits for every
// load that writes LDS; the wait is one that the compiler knows, else it waits
// again before it reads.)
template <int N>
DEV_INLINE void wait_and_meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070 | N);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// LDS: buffers of X, then three of W; when all is multiplied the outputs, rows of 128
// columns of each stretch.  Two buffers of X where three do not fit: its rows come
// from the caches, again for every column tile, W's from memory.
template <int JT>
struct LinTile {
  static constexpr int BM = 32 * JT;
  static constexpr int X_LOADS = (BM + 63) / 64, W_LOADS = 4;  // of a thread
  static constexpr int X_STAGES = JT <= 4 ? 3 : 2, W_STAGES = 3;
  static constexpr int X_BYTES = X_LOADS * 8192, W_BYTES = 32768;
  static constexpr int W0 = X_STAGES * X_BYTES, BYTES = W0 + W_STAGES * W_BYTES;
  static constexpr int OUT0 = BYTES - 65536;
  static constexpr int OUT1 = JT <= 4 ? OUT0 + 32768 : OUT0 - 65536;
  // loads behind those of a tile when it is read
  static constexpr int BEHIND = (X_STAGES == 3 ? X_LOADS : 0) + W_LOADS;
  static_assert(BYTES <= 160 * 1024 && (JT <= 4 || BYTES >= 131072), "LDS");
};

// A wave's part: J row tiles from ``row0``.  Its outputs are left in LDS.
template <int J, int JT, bool GLU, typename FetchX, typename FetchW>
DEV_INLINE void linear_wave(char* lds, int row0, int tiles, FetchX fetch_x,
                            FetchW fetch_w) {
  typedef LinTile<JT> L;
  const int lane = threadIdx.x & 63, wn = wave_id() & 3;
  FragAt<64> at;
  f32x16_t acc[2][J];                  // the stretches
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  int xo = 0, wo = L::W0, xn = (L::X_STAGES - 1) * L::X_BYTES,
      wn_o = L::W0 + 2 * L::W_BYTES;   // this tile's buffers, the next ones' to come
  for (int t = 0; t < tiles; ++t) {
    // The tile is there when the loads behind it alone are on their way; the
    // buffers of the one before it, which all have read, take the next ones.  (Under
    // no condition, so that the count is the same in every step.)
    wait_and_meet<L::BEHIND>();
    fetch_x(lds + xn, t + L::X_STAGES - 1 < tiles);
    fetch_w(lds + wn_o, t + 2 < tiles);
    at.renew();
    const char* xb = lds + xo + row0 * (2 * ATILE);
    const char* wb = lds + wo + wn * 32 * (2 * ATILE);
    xn = xo, wn_o = wo;
    xo = xo + L::X_BYTES < L::W0 ? xo + L::X_BYTES : 0;
    wo = wo + L::W_BYTES < L::BYTES ? wo + L::W_BYTES : L::W0;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      bf16x8_t wf[2], xf[J];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        wf[i] = frag_rows<64>(wb + i * (L::W_BYTES / 2), at, 0, ks);
#pragma unroll
      for (int j = 0; j < J; ++j) xf[j] = frag_rows<64>(xb, at, j, ks);
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[i], xf[j],
                                                              acc[i][j], 0, 0, 0);
    }
    constexpr int FIRST = 2 + J, REST = 3 * FIRST, PRODUCTS = 8 * J;
    constexpr int BOTH = REST < PRODUCTS ? REST : PRODUCTS;
    SCHED_LDS(FIRST);
#pragma unroll
    for (int i = 0; i < BOTH; ++i) {
      SCHED_MFMA(1);
      SCHED_LDS(1);
    }
    if constexpr (REST > BOTH) SCHED_LDS(REST - BOTH);
    if constexpr (PRODUCTS > BOTH) SCHED_MFMA(PRODUCTS - BOTH);
  }
  wait_and_meet<0>();

#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int r0 = row0 + j * 32;
#pragma unroll
    for (int i = 0; i < (GLU ? 1 : 2); ++i) {
      char* rows = lds + (i == 0 ? L::OUT0 : L::OUT1) + r0 * 256;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        bf16x4 v;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float g = acc[i][j][4 * q + t];
          // (the activation first: gate times up may be beyond 32 bits where the
          // sigmoid is 0)
          v.v[t] = f2bf(GLU ? g * __builtin_amdgcn_rcpf(
                                      1.f + exp2_hw(g * -1.4426950408889634f)) *
                                  acc[1][j][4 * q + t]
                            : g);
        }
        *reinterpret_cast<bf16x4*>(
            rows + (lane & 31) * 256 +
            (((wn * 4 + q) ^ OutTile::swz(lane & 31)) << 4) +
            (lane >> 5) * 8) = v;
      }
    }
  }
}

template <int JT, bool GLU>
__global__ __launch_bounds__(512, 2) void linear_kernel(
    bf16_t* __restrict__ out,          // (M, N)
    const bf16_t* __restrict__ x,      // (M, K)
    const bf16_t* __restrict__ w,      // (N, K), or (2 N, K): gate, up
    int M, int N, int K, int row_tiles, int col_tiles) {
  typedef LinTile<JT> L;
  constexpr int BM = L::BM, J0 = (JT + 1) / 2, J1 = JT / 2;
  __shared__ __attribute__((aligned(16))) char lds[L::BYTES];
  // each die takes one stretch of the tiles; within groups of columns, whose
  // weights its L2 holds, rows come first
  const int items = row_tiles * col_tiles;
  const int item = die_item(items);
  if (item >= items) return;
  const int group = item / (row_tiles * LIN_GROUP);
  const int rest = item - group * row_tiles * LIN_GROUP;
  const int width = min(LIN_GROUP, col_tiles - group * LIN_GROUP);
  const int m0 = uniform(rest / width * BM);
  const int n0 =
      uniform((group * LIN_GROUP + rest % width) * (GLU ? 128 : 256));

  RowsFrom<BM> xr(x + (long)m0 * K, K, M - m0);
  RowsFrom<128> first(w + (long)n0 * K, K, 128);
  RowsFrom<128> second(w + ((long)n0 + (GLU ? N : 128)) * K, K, 128);
  auto fetch_x = [&](char* to, bool more) { xr.copy(to, more); };
  auto fetch_w = [&](char* to, bool more) {
    first.copy(to, more);
    second.copy(to + L::W_BYTES / 2, more);
  };
  const int wid = wave_id(), tiles = K / ATILE;
  fetch_x(lds, true);
  fetch_w(lds + L::W0, true);
  if (L::X_STAGES == 3) fetch_x(lds + L::X_BYTES, tiles > 1);
  fetch_w(lds + L::W0 + L::W_BYTES, tiles > 1);
  if (J0 == J1)
    linear_wave<J0, JT, GLU>(lds, wid / 4 * (J0 * 32), tiles, fetch_x, fetch_w);
  else if (wid < 4)                    // (the same barriers on both sides)
    linear_wave<J0, JT, GLU>(lds, 0, tiles, fetch_x, fetch_w);
  else
    linear_wave<J1, JT, GLU>(lds, J0 * 32, tiles, fetch_x, fetch_w);
  __syncthreads();
  if (wid >= JT) return;
  const int r = m0 + wid * 32, from = wid * (32 * 256);
  bf16_t* to = out + (long)r * N + n0;
  OutTile::store32(lds + L::OUT0 + from, to, N, M - r);
  if (!GLU) OutTile::store32(lds + L::OUT1 + from, to + 128, N, M - r);
}

template <bool GLU>
torch::Tensor linear_prompt(const torch::Tensor& x, const torch::Tensor& w) {
  for (const auto* t : {&x, &w})
    TORCH_CHECK(t->is_cuda() && t->device() == x.device() && t->dim() == 2 &&
                    t->is_contiguous() && t->dtype() == torch::kBFloat16 &&
                    ((uintptr_t)t->data_ptr() & 15) == 0,
                "linear: contiguous 2-D bf16 at 16-byte addresses of one device");
  const long M = x.size(0), K = x.size(1), N = w.size(0) / (GLU ? 2 : 1);
  TORCH_CHECK(w.size(1) == K && K % 64 == 0 && K > 0 && w.size(0) % 256 == 0 &&
                  K < (1L << 20) && N < OutTile::STORE_LD && M < (1L << 30),
              "linear: inner numbers in 64s, the weight's rows in 256s, outputs "
              "below 2^25");
  auto out = torch::empty({M, N}, x.options());
  if (M == 0 || N == 0) return out;
  // Rows of a block: as many as end the last round of 256 blocks, one per CU,
  // earliest.  64 inner numbers cost what their row tiles do and one more for the
  // weights' fragments, a block 20 times as much as one of these.  (1024 -> 4096,
  // tiles of 96, 192, 224 and 256 rows: 5135 rows 105, 85.5, 80, 83 us; 1500 rows 31.5, 24,
  // 25.4, 25.7; 513 rows 13.9, 17.3, 19.8, 20.9; 3000 rows, 1536 -> 8960, 206, 157, 146,
  // 154.)
  const long cols = w.size(0) / 256;
  int best = 8;
  long least = -1;
  for (int jt = 2; jt <= 8; ++jt) {
    const long items = (M + 32 * jt - 1) / (32 * jt) * cols;
    const long cost = (items + 255) / 256 * ((jt + 1) * (K / 64) + 20);
    if (least < 0 || cost < least) least = cost, best = jt;
  }
  const long rows = (M + 32 * best - 1) / (32 * best), items = rows * cols;
  TORCH_CHECK(items < (1L << 31) - 8, "grid too large");
  const dim3 grid((unsigned)((items + ATTN_XCDS - 1) / ATTN_XCDS * ATTN_XCDS));
  auto stream = at::hip::getCurrentHIPStream();
  auto launch = [&](auto kern) {
    kern<<<grid, dim3(512), 0, stream>>>(
        (bf16_t*)out.data_ptr(), (const bf16_t*)x.data_ptr(),
        (const bf16_t*)w.data_ptr(), (int)M, (int)N, (int)K, (int)rows,
        (int)cols);
  };
  switch (best) {
    case 2: launch(linear_kernel<2, GLU>); break;
    case 3: launch(linear_kernel<3, GLU>); break;
    case 4: launch(linear_kernel<4, GLU>); break;
    case 5: launch(linear_kernel<5, GLU>); break;
    case 6: launch(linear_kernel<6, GLU>); break;
    case 7: launch(linear_kernel<7, GLU>); break;
    default: launch(linear_kernel<8, GLU>);
  }
  HIP_CHECK_KERNEL();
  return out;
}

}  // namespace

// x (M, K), w (N, K)
torch::Tensor linear_rows(torch::Tensor x, torch::Tensor w) {
  return linear_prompt<false>(x, w);
}

// x (M, K), w (2 N, K): rows of the gate, then of the up projection
torch::Tensor linear_swiglu(torch::Tensor x, torch::Tensor w) {
  return linear_prompt<true>(x, w);
}
