// Products of the trainer's backward pass, bf16 with fp32 sums: weight gradients dW =
// dY^T X, (N, K) from (M, N) and (M, K), and input gradients dX = dY W, (M, K) from (M, N)
// and (N, K).
//
// Reference capability: the gradients of the update loop's projections.
//
// Tiles, schedule and layouts: product_tile.h.
//
// What bounds it: the power that the card may draw.  Of random numbers 8192^3 (dW)
// takes 691 us (1590 TFLOP/s), of zeros 530: matrix cores busy in 80% of the cycles at
// 1.85 and 2.34 GHz.  v_mfma_f32_32x32x16_bf16 in such a loop is as busy, but the clock
// falls to 1.63 GHz: 763 us; with order and addresses left to the compiler 865; with a
// block a tile, each waiting for its first units and turning its outputs through LDS,
// 744 (14336 x 4096 of 7168 rows 603 for 584; 512 rows, 128256 x 2048, 333 for 289).  The
// library's best algorithm takes 1028.  8192 rows, dW of 14336 x 4096, 4096 x 4096, 8960 x
// 1536, 1024 x 4096: 672, 170, 157, 66 us for 887, 227, 234, 84; dX through 14336 x 4096, 4096
// x 4096, 8960 x 1536, 128256 x 2048: 610, 182, 158, 2730 for 690, 202, 179, 3149, of 256
// rows through the latter 137 for 343.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <climits>

#include "product_tile.h"

namespace {

using namespace product;

// A second product of the same size and right operand: its row tiles are those from
// ``first`` on
struct Twin {
  bf16_t* out;
  const bf16_t* left;
  int first;
};

// A tile's outputs, or where blocks share its inner numbers its fp32 sums, which are added
// up afterwards: (tiles, ways, SIDE * SIDE)
template <int J>
struct Outputs : TileRows<J> {
  bf16_t* const out;
  float* const shares;
  const long R, C;
  const Twin twin;
  f32x4_t* to_share;
  DEV_INLINE Outputs(bf16_t* out_, float* shares_, long R_, long C_, const Twin& twin_)
      : out(out_), shares(shares_), R(R_), C(C_), twin(twin_) {}
  DEV_INLINE void tile(const Place& at) {
    if (J == 8 && shares != nullptr) {
      to_share = reinterpret_cast<f32x4_t*>(shares + (long)at.share * SIDE * SIDE) +
                 wave_id() * 4096 + (threadIdx.x & 63);
    } else {
      Place in = at;
      if (at.row >= twin.first) in.row -= twin.first;
      this->start(at.row >= twin.first ? twin.out : out, R, C, in, (long)at.col * SIDE);
    }
  }
  DEV_INLINE void rows(int) {
    if (J < 8 || shares == nullptr) this->to.next();
  }
  // (a share's block has no other tile: nothing counts these stores)
  DEV_INLINE void put(int j, int q, const f32x4_t (&sums)[2]) const {
    if (J == 8 && shares != nullptr) {
#pragma unroll
      for (int e = 0; e < 2; ++e) to_share[((2 * q + e) * 8 + j) * 64] = sums[e];
    } else {
      TileRows<J>::put(j, q, sums);
    }
  }
};

// out (R, C): sums over inner of left(row, inner) right(inner, column), right in
// COLUMNS.  ``ways`` blocks share a tile's inner numbers.  LINES: tiles of 32 J rows.
template <bool LINES, int J>
__global__ __launch_bounds__(256, 1) void product_kernel(
    bf16_t* __restrict__ out, float* __restrict__ shares,
    const bf16_t* __restrict__ left, const bf16_t* __restrict__ right,
    const Twin twin, long R, long C, long inner, int row_tiles, int col_tiles,
    int ways) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  constexpr int ROWS = 32 * J;
  const int tiles = row_tiles * col_tiles, items = tiles * ways;
  const int all = (int)((inner + PAIR - 1) / PAIR);
  auto units = [&](int r, Units& a, Units& b, Place& at) {
    const int item = item_of(r, items, gridDim.x);
    if (item < 0) return false;
    const int part = item / tiles, tile = item - part * tiles;
    at = Place(tile, row_tiles, col_tiles, tile * ways + part);
    const int p0 = (int)((long)all * part / ways);
    const int n = (int)((long)all * (part + 1) / ways) - p0;
    const bool second = !LINES && at.row >= twin.first;
    const bf16_t* l = second ? twin.left : left;
    const long r0 = (long)(at.row - (second ? twin.first : 0)) * ROWS;
    const long c0 = (long)at.col * SIDE, i0 = (long)p0 * PAIR;
    a = LINES ? lines(l, R, inner, r0, i0, n) : columns(l, R, inner, r0, i0, n);
    b = columns(right, C, inner, c0, i0, n);
    return true;
  };
  Outputs<J> outputs(out, shares, R, C, twin);
  run<LINES, false, J>(
      lds, [&](int) { return LINES ? inner : R; }, C, units, outputs);
}

// out (R, C): the sum of left_p(row, inner) right_p(inner, column) over the parts, the
// input's gradient of layers that share it.  In a layer of 7168 and of 8192 rows: through
// gate and up, 14336 x 4096 each, 1101 and 1245 us for 1132 and 1283 of two products and an
// addition, through q, k and v 238 and 275 for 321 and 363 of three.
constexpr int MOST = 3;
struct Parts {
  const bf16_t *left[MOST], *right[MOST];
  long inner[MOST];
};

template <int J, int PARTS>
__global__ __launch_bounds__(256, 1) void parts_kernel(
    bf16_t* __restrict__ out, const Parts parts, long R, long C, int row_tiles,
    int col_tiles) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  const int items = row_tiles * col_tiles;
  auto inner_of = [&](int p) {
    return p == 0 ? parts.inner[0] : p == 1 ? parts.inner[1] : parts.inner[2];
  };
  auto units = [&](int r, Units& a, Units& b, Place& at) {
    const int item = item_of(r / PARTS, items, gridDim.x), p = r % PARTS;
    if (item < 0) return false;
    at = Place(item, row_tiles, col_tiles);
    const bf16_t* left = p == 0 ? parts.left[0] : p == 1 ? parts.left[1] : parts.left[2];
    const bf16_t* right =
        p == 0 ? parts.right[0] : p == 1 ? parts.right[1] : parts.right[2];
    const long inner = inner_of(p);
    a = lines(left, R, inner, (long)at.row * (32 * J), 0, (int)(inner / PAIR));
    b = columns(right, C, inner, (long)at.col * SIDE, 0, (int)(inner / PAIR));
    return true;
  };
  Outputs<J> outputs(out, nullptr, R, C, {nullptr, nullptr, INT_MAX});
  run<true, false, J, PARTS>(lds, inner_of, C, units, outputs);
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
  return M > 0 && N > 0 && K > 0 && N % PAIR == 0 && K % 8 == 0 &&
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
torch::Tensor product_of(const torch::Tensor& left, const torch::Tensor& right, long R,
                      long C, long inner) {
  auto out = torch::empty({R, C}, left.options());
  const long col_tiles = (C + SIDE - 1) / SIDE;
  const long ways = ways_of(tiles_of(R, C), inner);
  const int parts = LINES && ways == 1 ? rows_of(R, col_tiles, inner, 6).parts : 8;
  const long row_tiles = (R + 32 * parts - 1) / (32 * parts);
  const long tiles = row_tiles * col_tiles, items = tiles * ways;
  TORCH_CHECK(items < (1L << 31) - ATTN_XCDS, "grid too large");
  const long grid = blocks_of(items, inner / ways);
  torch::Tensor shares;
  if (ways > 1)
    shares = torch::empty({items * SIDE * SIDE},
                          out.options().dtype(torch::kFloat32));
  float* sums = ways > 1 ? shares.data_ptr<float>() : nullptr;
  auto stream = at::hip::getCurrentHIPStream();
  auto launch = [&](auto kern) {
    kern<<<dim3((unsigned)grid), dim3(256), 0, stream>>>(
        (bf16_t*)out.data_ptr(), sums, (const bf16_t*)left.data_ptr(),
        (const bf16_t*)right.data_ptr(), Twin{nullptr, nullptr, INT_MAX}, R, C, inner,
        (int)row_tiles, (int)col_tiles, (int)ways);
  };
  if (LINES && parts == 6) launch(product_kernel<LINES, LINES ? 6 : 8>);
  else if (LINES && parts == 7) launch(product_kernel<LINES, LINES ? 7 : 8>);
  else launch(product_kernel<LINES, 8>);
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

// The same for linear_dgrad, where the library does better.  Where tiles fill rounds of
// 256 to 0.69 of what whole ones would cost it takes 0.61 to 1.02 of the library's time (at
// 0.67 to 0.69 of it, through 18944 x 3584 of 2600 and 5120 rows 327 and 688 us for 320 and
// 640, through 1536 x 1536 of 6144 34.6 for 34.1; through 4096 x 4096 of 2600, 5120, 7168 rows,
// 0.77, 0.76, 0.96 of it, 79, 140, 164 for 89, 164, 204); half a chip's tiles and less pay
// where the inner dimension is long enough to be shared (256, 1024, 2048 rows through 14336 x
// 4096 61, 110, 190 for 77, 150, 241; through 4096 x 4096 26, 47, 70 for 25, 42, 63), unless
// two blocks a tile at most leave much of the chip idle (through 8192 x 28672 of 64 and 130
// rows 121 and 124 for 93 and 107, through 28672 x 8192 of 513, 700, 768 290, 310, 317 for 266,
// 331, 336: 0.22, 0.44, 0.50, 0.68, 0.75 of it), and but for the fewest rows (64 and 130
// through 8192 x 8192 49, 51 for 46, 65; 64 through 14336 x 4096 47 for 70).  Weights in turn
// from memory.
bool linear_dgrad_takes(const torch::Tensor& dy, const torch::Tensor& w) {
  if (!dgrad_fits(dy, w)) return false;
  const long M = dy.size(0), N = dy.size(1), K = w.size(1), tiles = tiles_of(M, K);
  const double rounds = (double)M * K / (CUS * SIDE * SIDE);
  if (tiles <= CUS / 2) {
    const long ways = ways_of(tiles, N);
    return N >= 8192 && M >= (N > K ? 64 : 128) && (ways > 2 || rounds * ways >= 0.6);
  }
  return rows_of(M, (K + SIDE - 1) / SIDE, N, 6).cost <= 1.45 * rounds * cost_of(8, N);
}

// dW (N, K) = dY^T X of dY (M, N), X (M, K)
torch::Tensor linear_wgrad(torch::Tensor dy, torch::Tensor x) {
  check_operands(dy, x);
  TORCH_CHECK(x.size(0) == dy.size(0) && wgrad_fits(dy, x),
              "linear_wgrad: rows in 16-byte granules, at most 4 GiB");
  return product_of<false>(dy, x, dy.size(1), x.size(1), dy.size(0));
}

// Whether linear_wgrad_pair has these operands and is the better choice than a product
// each: two of one size whose tiles are not shared.  Their tiles fill rounds of 256
// together (7168 rows, 14336 x 4096 each: 7 rounds for 4 and 4, 1120 us for 1224; 7168
// rows, 11008 x 2048 458 for 542; 512 rows, 14336 x 4096 119 for 136; 3000 rows, 8960 x 1536
// 126 for 131; 5135 rows, 5120 x 2048, whose rounds are as many, 191 both).
bool linear_wgrad_pair_takes(const torch::Tensor& dy0, const torch::Tensor& dy1,
                             const torch::Tensor& x) {
  return dy0.sizes() == dy1.sizes() && wgrad_fits(dy1, x) && linear_wgrad_takes(dy0, x) &&
         tiles_of(dy0.size(1), x.size(1)) >= 160;
}

// dW_p (N, K) = dY_p^T X of dY_p (M, N), X (M, K)
std::vector<torch::Tensor> linear_wgrad_pair(torch::Tensor dy0, torch::Tensor dy1,
                                             torch::Tensor x) {
  check_operands(dy0, x);
  check_operands(dy1, x);
  TORCH_CHECK(x.size(0) == dy0.size(0) && linear_wgrad_pair_takes(dy0, dy1, x),
              "linear_wgrad_pair: operands that it does not take");
  const long R = dy0.size(1), C = x.size(1), inner = dy0.size(0);
  std::vector<torch::Tensor> outs;
  for (int i = 0; i < 2; ++i) outs.push_back(torch::empty({R, C}, x.options()));
  const long rows = (R + SIDE - 1) / SIDE, cols = (C + SIDE - 1) / SIDE;
  const long items = 2 * rows * cols;
  TORCH_CHECK(items < (1L << 31) - ATTN_XCDS, "grid too large");
  product_kernel<false, 8><<<dim3((unsigned)blocks_of(items, inner)), dim3(256), 0,
                             at::hip::getCurrentHIPStream()>>>(
      (bf16_t*)outs[0].data_ptr(), nullptr, (const bf16_t*)dy0.data_ptr(),
      (const bf16_t*)x.data_ptr(),
      Twin{(bf16_t*)outs[1].data_ptr(), (const bf16_t*)dy1.data_ptr(), (int)rows}, R, C,
      inner, (int)(2 * rows), (int)cols, 1);
  HIP_CHECK_KERNEL();
  return outs;
}

// dX (M, K) = dY W of dY (M, N), W (N, K)
torch::Tensor linear_dgrad(torch::Tensor dy, torch::Tensor w) {
  check_operands(dy, w);
  TORCH_CHECK(w.size(0) == dy.size(1) && dgrad_fits(dy, w),
              "linear_dgrad: N in 64s, rows in 16-byte granules, W at most 4 GiB");
  return product_of<true>(dy, w, dy.size(0), w.size(1), dy.size(1));
}

namespace {

long inner_of(const std::vector<torch::Tensor>& dys) {
  long sum = 0;
  for (const auto& dy : dys) sum += dy.size(1);
  return sum;
}

}  // namespace

// Whether linear_dgrad_sum has these operands and is the better choice than a product
// each and additions: not where tiles leave rounds emptier than linear_dgrad's may, which
// shares them.  (Rounds' cost by whole ones', us for a product each, weights in turn from
// memory: gate and up 1.46, 1.48 635, 1333 for 642, 1326 of 2600 and 5120 rows of 3584; 1.62,
// 1.62, 1.73, 1.85 266, 928, 300, 630 for 269, 795, 297, 585; 2.16 471 for 355.  q, k and v,
// whose products alone are small, would gain beyond the line too: 1.63, 1.65, 1.78 112, 59,
// 44 for 137, 91, 75, from 2.2 on as much.)
bool linear_dgrad_sum_takes(const std::vector<torch::Tensor>& dys,
                            const std::vector<torch::Tensor>& ws) {
  if (dys.size() < 2 || dys.size() > MOST || dys.size() != ws.size()) return false;
  for (size_t i = 0; i < dys.size(); ++i)
    if (!dgrad_fits(dys[i], ws[i])) return false;
  const long M = dys[0].size(0), K = ws[0].size(1), N = inner_of(dys);
  const double whole = (double)M * K / (CUS * SIDE * SIDE) * cost_of(8, N);
  return rows_of(M, (K + SIDE - 1) / SIDE, N, 6).cost <= 1.5 * whole;
}

// dX (M, K) = the sum of dY_p W_p, of dY_p (M, N_p), W_p (N_p, K): rounded once
torch::Tensor linear_dgrad_sum(std::vector<torch::Tensor> dys,
                               std::vector<torch::Tensor> ws) {
  const int n = (int)dys.size();
  TORCH_CHECK((n == 2 || n == 3) && ws.size() == dys.size(),
              "linear_dgrad_sum: two or three products");
  Parts parts = {};
  for (int i = 0; i < n; ++i) {
    check_operands(dys[i], ws[i]);
    TORCH_CHECK(dys[i].device() == dys[0].device() &&
                    dys[i].size(0) == dys[0].size(0) &&
                    ws[i].size(0) == dys[i].size(1) &&
                    ws[i].size(1) == ws[0].size(1) && dgrad_fits(dys[i], ws[i]),
                "linear_dgrad_sum: N in 64s, rows in 16-byte granules, W at most 4 GiB");
    parts.left[i] = (const bf16_t*)dys[i].data_ptr();
    parts.right[i] = (const bf16_t*)ws[i].data_ptr();
    parts.inner[i] = dys[i].size(1);
  }
  const long R = dys[0].size(0), C = ws[0].size(1), inner = inner_of(dys);
  auto out = torch::empty({R, C}, dys[0].options());
  const long col_tiles = (C + SIDE - 1) / SIDE;
  const int j = rows_of(R, col_tiles, inner, 6).parts;
  const long row_tiles = (R + 32 * j - 1) / (32 * j), items = row_tiles * col_tiles;
  TORCH_CHECK(items < (1L << 31) / MOST - ATTN_XCDS, "grid too large");
  const dim3 grid((unsigned)blocks_of(items, inner));
  auto stream = at::hip::getCurrentHIPStream();
  auto launch = [&](auto kern) {
    kern<<<grid, dim3(256), 0, stream>>>((bf16_t*)out.data_ptr(), parts, R, C,
                                         (int)row_tiles, (int)col_tiles);
  };
  if (n == 2)
    launch(j == 6 ? parts_kernel<6, 2> : j == 7 ? parts_kernel<7, 2> : parts_kernel<8, 2>);
  else
    launch(j == 6 ? parts_kernel<6, 3> : j == 7 ? parts_kernel<7, 3> : parts_kernel<8, 3>);
  HIP_CHECK_KERNEL();
  return out;
}
