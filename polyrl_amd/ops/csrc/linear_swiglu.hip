// out = silu(x Wg^T) * (x Wu^T), bf16: the gated MLP's two products and its
// activation in one kernel, for prompts (hundreds of rows and more).
//
// Reference capability: the engine-side fused gate/up projection and activation.
//
// Split.  A block owns 32 JT rows and 128 output columns, whose 128 gate and 128 up
// rows of the weight are its 256 columns of the product.  Eight waves = two row
// groups x four column groups: a wave holds up to 128 rows x (32 gate + 32 up)
// in 128 registers, so gate and up of an output meet in one lane.  Weights are
// the A operand of v_mfma_f32_32x32x16_bf16, so that a lane's accumulators are
// neighbouring columns of one row.  Waves w and w + 4 share a SIMD: where JT is
// odd the one has a row tile more than the other and every SIMD the same.
// Tiles of 64 inner numbers, the layout of attention_tile.h (rows of 128
// bytes, no bank conflicts), go straight into LDS, two buffers of each operand,
// 128 KiB: one block per CU, two waves per SIMD.  Nothing is rounded but the
// result (the products and the activation used to round gate, up and out).
//
// What bounds it: LDS reads and matrix instructions, each about 60% of the cycles,
// and the clock under them; per block 2 to 4 us for the first tiles and the
// activation.  Measured, against the library's product and the activation's pass:
// 5135 rows, 1024 -> 4096 79.8 us and 101.6; 4096 rows, 2048 -> 8192 213 and 224; 3000
// rows, 1536 -> 8960 147 and 162; 1500 rows, 1024 -> 4096 24 and 32; 513 rows 13.6
// and 27.9.  Reading the fragments of the next 16 inner numbers ahead of the barrier
// takes 5% more, rows in groups of 64 (four row groups, two column groups) the
// same.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "attention_tile.h"

namespace {

typedef AttnTile<64> InTile;           // 64 inner numbers of a row
typedef AttnTile<128> OutTile;         // 128 columns of a row
constexpr int LIN_BUFFER = 256 * 128;  // bytes of 256 rows of a tile
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
  DEV_INLINE void copy(char* tile) {
    const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(base), 0, records, 0x00020000);
    char* to = tile + uniform(threadIdx.x >> 6) * 1024;
    int a = at;
#pragma unroll
    for (int i = 0; i < (ROWS + 63) / 64; ++i) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (lds_p)(to + i * 8192), 16,
                                               a, 0, 0, 0);
      a += 64 * ldb;                   // (whole periods of the swizzle)
    }
    base += 2 * ATILE;
    records = max(records - 2 * ATILE, 0);
  }
};

// A wave's part: J row tiles from ``row0``.  Its outputs are left in x0_s and x1_s,
// rows of 128 columns.
template <int J, typename Fetch>
DEV_INLINE void swiglu_wave(char* x0_s, char* w0_s, char* x1_s, char* w1_s,
                            int row0, int tiles, Fetch fetch) {
  const int lane = threadIdx.x & 63, wn = wave_id() & 3;
  FragAt<64> at;
  f32x16_t acc[2][J];                  // gate and up
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  auto step = [&](const char* xs, const char* ws, char* xn, char* wn_s,
                  bool more) {
    if (more) fetch(xn, wn_s);
    at.renew();
    const char* xb = xs + row0 * (2 * ATILE);
    const char* wb = ws + wn * 32 * (2 * ATILE);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      bf16x8_t wf[2], xf[J];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        wf[i] = frag_rows<64>(wb + i * (LIN_BUFFER / 2), at, 0, ks);
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
    wait_loads();
    __syncthreads();
  };
  for (int t = 0; t < tiles; t += 2) {
    step(x0_s, w0_s, x1_s, w1_s, t + 1 < tiles);
    if (t + 1 < tiles) step(x1_s, w1_s, x0_s, w0_s, t + 2 < tiles);
  }

#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int r0 = row0 + j * 32;
    char* rows = (r0 < 128 ? x0_s : x1_s) + (r0 & 127) * 256;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bf16x4 v;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float g = acc[0][j][4 * q + t];
        v.v[t] = f2bf(g * acc[1][j][4 * q + t] *
                      __builtin_amdgcn_rcpf(
                          1.f + exp2_hw(g * -1.4426950408889634f)));
      }
      *reinterpret_cast<bf16x4*>(
          rows + (lane & 31) * 256 +
          (((wn * 4 + q) ^ OutTile::swz(lane & 31)) << 4) + (lane >> 5) * 8) = v;
    }
  }
}

template <int JT>
__global__ __launch_bounds__(512, 2) void linear_swiglu_kernel(
    bf16_t* __restrict__ out,          // (M, N)
    const bf16_t* __restrict__ x,      // (M, K)
    const bf16_t* __restrict__ w,      // (2 N, K): gate, up
    int M, int N, int K, int row_tiles, int col_tiles) {
  constexpr int BM = 32 * JT, J0 = (JT + 1) / 2, J1 = JT / 2;
  __shared__ __attribute__((aligned(16))) char x0_s[LIN_BUFFER],
      w0_s[LIN_BUFFER], x1_s[LIN_BUFFER], w1_s[LIN_BUFFER];
  // each die takes one stretch of the tiles; within groups of columns, whose
  // weights its L2 holds, rows come first
  const int items = row_tiles * col_tiles;
  const int item = die_item(items);
  if (item >= items) return;
  const int group = item / (row_tiles * LIN_GROUP);
  const int rest = item - group * row_tiles * LIN_GROUP;
  const int width = min(LIN_GROUP, col_tiles - group * LIN_GROUP);
  const int m0 = rest / width * BM;
  const int n0 = (group * LIN_GROUP + rest % width) * 128;

  RowsFrom<BM> xr(x + (long)m0 * K, K, M - m0);
  RowsFrom<128> gr(w + (long)n0 * K, K, 128);
  RowsFrom<128> ur(w + ((long)N + n0) * K, K, 128);
  auto fetch = [&](char* xs, char* ws) {
    xr.copy(xs);
    gr.copy(ws);
    ur.copy(ws + LIN_BUFFER / 2);
  };
  fetch(x0_s, w0_s);
  wait_loads();
  __syncthreads();
  const int wid = wave_id(), tiles = K / ATILE;
  if (J0 == J1)
    swiglu_wave<J0>(x0_s, w0_s, x1_s, w1_s, wid / 4 * (J0 * 32), tiles, fetch);
  else if (wid < 4)                    // (the same barriers on both sides)
    swiglu_wave<J0>(x0_s, w0_s, x1_s, w1_s, 0, tiles, fetch);
  else
    swiglu_wave<J1>(x0_s, w0_s, x1_s, w1_s, J0 * 32, tiles, fetch);
  __syncthreads();
  if (wid >= JT) return;
  const int r = m0 + wid * 32;
  OutTile::store32((wid < 4 ? x0_s : x1_s) + (wid & 3) * (32 * 256),
                   out + (long)r * N + n0, N, M - r);
}

}  // namespace

// x (M, K), w (2 N, K): rows of the gate, then of the up projection
torch::Tensor linear_swiglu(torch::Tensor x, torch::Tensor w) {
  for (const auto* t : {&x, &w})
    TORCH_CHECK(t->is_cuda() && t->dim() == 2 && t->is_contiguous() &&
                    t->dtype() == torch::kBFloat16 &&
                    ((uintptr_t)t->data_ptr() & 15) == 0,
                "linear_swiglu: contiguous 2-D bf16 at a 16-byte address");
  const long M = x.size(0), K = x.size(1), N = w.size(0) / 2;
  TORCH_CHECK(w.size(1) == K && K % 64 == 0 && K > 0 && w.size(0) % 256 == 0 &&
                  K < (1L << 20) && N < (1L << 30) && M < (1L << 30),
              "linear_swiglu: inner numbers in 64s, columns in 128s");
  auto out = torch::empty({M, N}, x.options());
  if (M == 0 || N == 0) return out;
  // Rows of a block: as many as end the last round of 256 blocks, one per CU,
  // earliest.  64 inner numbers cost what their row tiles do and one more for the
  // weights' fragments, a block 20 times as much as one of these.  (5135 rows, 1024 -> 4096, tiles of 96, 192, 224 and
  // 256 rows 105, 85.5, 80, 83 us; 1500 rows 31.5, 24, 25.4, 25.7; 513 rows 13.9,
  // 17.3, 19.8, 20.9; 3000 rows, 1536 -> 8960, 206, 157, 146, 154.)
  const long cols = N / 128;
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
    case 2: launch(linear_swiglu_kernel<2>); break;
    case 3: launch(linear_swiglu_kernel<3>); break;
    case 4: launch(linear_swiglu_kernel<4>); break;
    case 5: launch(linear_swiglu_kernel<5>); break;
    case 6: launch(linear_swiglu_kernel<6>); break;
    case 7: launch(linear_swiglu_kernel<7>); break;
    default: launch(linear_swiglu_kernel<8>);
  }
  HIP_CHECK_KERNEL();
  return out;
}
