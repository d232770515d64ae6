// Products of prompts (hundreds of rows and more) with a weight's rows, bf16:
// x W^T, and silu(x Wg^T) * (x Wu^T), the gated MLP's two products and its
// activation, in one kernel.
//
// Reference capability: the engine-side projections and the fused gate/up
// projection with its activation.
//
// Tiles, schedule and layouts: product_tile.h, both operands in LINES.  A tile is 32 J
// rows by 256 columns of the product, or (GLU) 128 of the gate's and 128 of the up
// projection's, of which it makes 128 outputs: each wave has 64 of both, so gate and up
// of an output meet in one lane.  Nothing is rounded but the result.
//
// What bounds it: the matrix cores and, in few rounds of tiles, how full the last one
// is (rows_of).  Measured (us, beside the kernel that this replaces, eight waves of
// 128 x 64 and a block a tile, and the library's product with the activation's pass):
// 1024 -> 4096 of 513, 1024, 5135 and 8192 rows 15.0, 18.5, 74.0, 113 for 15.8, 20.1, 86.9,
// 128 and 23.8, 28.2, 103, 149; 2048 -> 8192 34.1, 51.8, 256, 391 for 39.0, 60.8, 310, 461
// and 44.7, 69.0, 316, 472; 4096 -> 14336 117, 183, 868, 1301 for 136, 210, 1035, 1544 and
// 131, 207, 996, 1408.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "product_tile.h"

namespace {

using namespace product;

template <int J, bool GLU>
__global__ __launch_bounds__(256, 1) void linear_kernel(
    bf16_t* __restrict__ out,          // (M, N)
    const bf16_t* __restrict__ x,      // (M, K)
    const bf16_t* __restrict__ w,      // (N, K), or (2 N, K): gate, up
    long M, long N, long K, int row_tiles, int col_tiles) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  constexpr int ROWS = 32 * J, COLS = GLU ? 128 : 256;
  const int items = row_tiles * col_tiles, n = (int)(K / PAIR);
  auto units = [&](int r, Units& a, Units& b) {
    const int item = item_of(r, items, gridDim.x);
    if (item < 0) return false;
    const Place at(item, row_tiles, col_tiles);
    a = lines(x, M, K, (long)at.row * ROWS, 0, n);
    if (GLU) {
      // a wave loads the 64 rows of its number: gate, up, gate, up
      const int wid = wave_id();
      const long row = (long)at.col * COLS + (wid >> 1) * 64 + (wid & 1) * N;
      b = lines(w, 2 * N, K, row - wid * 64, 0, n);
    } else {
      b = lines(w, N, K, (long)at.col * COLS, 0, n);
    }
    return true;
  };
  auto finish = [&](int r, Acc<J>& acc) {
    const int lane = threadIdx.x & 63, wid = wave_id();
    const Place at(item_of(r, items, gridDim.x), row_tiles, col_tiles);
    const long r0 = (long)at.row * ROWS + (wid & 1) * (16 * J) + (lane & 15);
    const long c0 = (long)at.col * COLS + (wid >> 1) * (COLS / 2) + 8 * (lane >> 4);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const long row = r0 + 16 * j;
      order();
#pragma unroll
      for (int i = 0; i < (GLU ? 4 : 8); i += 2) {
        f32x4_t y[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          y[h] = sums_of(acc[i + h][j]);
          if (!GLU) continue;
          const f32x4_t u = sums_of(acc[(i + h + 4) % 8][j]);
          // (the activation first: gate times up may be beyond 32 bits where the
          // sigmoid is 0)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            y[h][e] = y[h][e] *
                      __builtin_amdgcn_rcpf(
                          1.f + exp2_hw(y[h][e] * -1.4426950408889634f)) *
                      u[e];
        }
        const u32x4_t v = eight_columns(y[0], y[1]);
        if (row < M && (GLU || c0 + 16 * i < N))
          *reinterpret_cast<u32x4_t*>(out + row * N + c0 + 16 * i) = v;
      }
    }
  };
  run<true, true, J>(lds, K, K, units, finish);
}

template <bool GLU>
void launch_linear(torch::Tensor& out, const torch::Tensor& x, const torch::Tensor& w) {
  const long M = x.size(0), K = x.size(1), N = out.size(1);
  if (M == 0 || N == 0) return;
  const long cols = (w.size(0) + SIDE - 1) / SIDE;
  const int best = rows_of(M, cols, K, 3).parts;
  const long rows = (M + 32 * best - 1) / (32 * best), items = rows * cols;
  TORCH_CHECK(items < (1L << 31) - ATTN_XCDS, "grid too large");
  const dim3 grid((unsigned)blocks_of(items, K));
  auto stream = at::hip::getCurrentHIPStream();
  auto launch = [&](auto kern) {
    kern<<<grid, dim3(256), 0, stream>>>(
        (bf16_t*)out.data_ptr(), (const bf16_t*)x.data_ptr(),
        (const bf16_t*)w.data_ptr(), M, N, K, (int)rows, (int)cols);
  };
  switch (best) {
    case 3: launch(linear_kernel<3, GLU>); break;
    case 4: launch(linear_kernel<4, GLU>); break;
    case 5: launch(linear_kernel<5, GLU>); break;
    case 6: launch(linear_kernel<6, GLU>); break;
    case 7: launch(linear_kernel<7, GLU>); break;
    default: launch(linear_kernel<8, GLU>);
  }
  HIP_CHECK_KERNEL();
}

template <bool GLU>
torch::Tensor linear_prompt(const torch::Tensor& x, const torch::Tensor& w) {
  for (const auto* t : {&x, &w})
    TORCH_CHECK(t->is_cuda() && t->device() == x.device() && t->dim() == 2 &&
                    t->is_contiguous() && t->dtype() == torch::kBFloat16 &&
                    ((uintptr_t)t->data_ptr() & 15) == 0,
                "linear: contiguous 2-D bf16 at 16-byte addresses of one device");
  const long M = x.size(0), K = x.size(1), N = w.size(0) / (GLU ? 2 : 1);
  TORCH_CHECK(w.size(1) == K && K % PAIR == 0 && K > 0 && w.size(0) % 256 == 0 &&
                  K < (1L << 20) && N < (1L << 25) && M < (1L << 30),
              "linear: inner numbers in 64s, the weight's rows in 256s, outputs "
              "below 2^25");
  auto out = torch::empty({M, N}, x.options());
  launch_linear<GLU>(out, x, w);
  return out;
}

}  // namespace

// Whether linear_rows_into has these contiguous bf16 matrices: as linear_rows, but the
// weight's rows, which are whole 16-byte granules of the output, in 8s
bool linear_rows_fits(const torch::Tensor& x, const torch::Tensor& w) {
  const long M = x.size(0), K = x.size(1), N = w.size(0);
  return M > 0 && M < (1L << 30) && K > 0 && K % PAIR == 0 && K < (1L << 20) && N > 0 &&
         N % 8 == 0 && N < (1L << 25) &&
         (((uintptr_t)x.data_ptr() | (uintptr_t)w.data_ptr()) & 15) == 0;
}

void linear_rows_into(torch::Tensor& out, const torch::Tensor& x,
                      const torch::Tensor& w) {
  for (const auto* t : {(const torch::Tensor*)&out, &x, &w})
    TORCH_CHECK(t->is_cuda() && t->device() == x.device() && t->dim() == 2 &&
                    t->is_contiguous() && t->dtype() == torch::kBFloat16,
                "linear: contiguous 2-D bf16 of one device");
  TORCH_CHECK(w.size(1) == x.size(1) && out.size(0) == x.size(0) &&
                  out.size(1) == w.size(0) && linear_rows_fits(x, w) &&
                  ((uintptr_t)out.data_ptr() & 15) == 0,
              "linear: inner numbers in 64s, outputs in 8s, 16-byte addresses");
  launch_linear<false>(out, x, w);
}

// Whether linear_rows is the better choice than the library's own: tiles that fill
// rounds of 256 to 0.74 of what whole ones would cost, but not whole tiles of 256 rows,
// which the library multiplies 1 to 4% faster.  (us, beside the library's, of 2600, 4096,
// 5135 and 7168 rows: 2048 -> 2048 25.0, 29.8, 36.0, 44.0 and 29.1, 32.8, 48.6, 45.1;
// 8192 -> 2048 81.5, 99.6, 123, 151 and 82.0, 107, 146, 156; 8960 -> 1536 94.7, 98.3,
// 108, 138 and 72.5, 96.7, 117, 151, whose first two fill 0.44 and 0.6; 4096 of 14336 ->
// 4096 296 and 289.)
bool linear_rows_pays(long M, long N, long K) {
  if (M <= 0 || N <= 0 || K < PAIR) return false;
  const Rows best = rows_of(M, (N + SIDE - 1) / SIDE, K, 3);
  const double whole = (double)M * N / (CUS * SIDE * SIDE) * cost_of(8, K);
  return best.cost <= 1.35 * whole && (best.parts < 8 || M % SIDE != 0);
}

// x (M, K), w (N, K)
torch::Tensor linear_rows(torch::Tensor x, torch::Tensor w) {
  return linear_prompt<false>(x, w);
}

// x (M, K), w (2 N, K): rows of the gate, then of the up projection
torch::Tensor linear_swiglu(torch::Tensor x, torch::Tensor w) {
  return linear_prompt<true>(x, w);
}
