// Products of prompts (hundreds of rows and more) with a weight's rows, bf16:
// x W^T of one weight or several, and silu(x Wg^T) * (x Wu^T), the gated MLP's two
// products and its activation, in one kernel.
//
// Reference capability: the engine-side projections and the fused gate/up
// projection with its activation.
//
// Tiles, schedule and layouts: product_tile.h, both operands in LINES.  A tile is 32 J
// rows by 256 columns of the product, or (GLU) 128 of the gate's and 128 of the up
// projection's, of which it makes 128 outputs: each wave has 64 of both, so gate and up
// of an output meet in one lane.  Nothing is rounded but what is stored: the result, and
// for the trainer the two products (KEPT).
//
// In a layer of the trainer of 7168 rows (its kernels one after the other): gate, up and
// activation of 4096 -> 14336 1200 us for 585 + 585 + 112 of two products and a pass, q, k
// and v of 4096 -> 4096, 1024, 1024 244 for 175 + 59 + 58.
//
// What bounds it: the matrix cores and, in few rounds of tiles, how full the last one
// is (rows_of).  Measured (us, beside the kernel that this replaces, eight waves of
// 128 x 64 and a block a tile, and the library's product with the activation's pass):
// 1024 -> 4096 of 513, 1024, 5135 and 8192 rows 15.0, 18.5, 74.0, 113 for 15.8, 20.1, 86.9,
// 128 and 23.8, 28.2, 103, 149; 2048 -> 8192 34.1, 51.8, 256, 391 for 39.0, 60.8, 310, 461
// and 44.7, 69.0, 316, 472; 4096 -> 14336 117, 183, 868, 1301 for 136, 210, 1035, 1544 and
// 131, 207, 996, 1408.  Since then a tile's sums are taken out beside the next one's
// products and outputs go past the L2s: 1024 -> 4096 of 5135 and 8192 rows 70.3, 105 ->
// 66.7, 101 (on another card), 1024 -> 1536 and 1024 of 5135 19.0, 15.2 -> 17.0, 14.0.  What
// is left above the products' own time in 1024 -> 4096 of 7168 rows, one tile a block: the
// stores 2 us and the activation 1 of 26.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "product_tile.h"

namespace {

using namespace product;

// Outputs of one matrix of weights; of several products of the same rows each but the
// last has whole tiles of columns
struct Part {
  bf16_t* out;                         // (M, n)
  const bf16_t* w;                     // (n, K)
  long n;
};
constexpr int MOST = 3;
struct Parts {
  Part p[MOST];
};

// part of a column of the products together, and which of its columns
DEV_INLINE Part part_of(const Parts& parts, long& col) {
  Part p = parts.p[0];
  if (col >= p.n) {
    col -= p.n, p = parts.p[1];
    if (col >= p.n) col -= p.n, p = parts.p[2];
  }
  return p;
}

// PLAIN: the products.  GATED: out = silu(gate) * up of the products with p[0], gate, and
// p[1], up.  KEPT: the products too.  ADDED: the product added to what its output holds.
enum Kind { PLAIN, GATED, KEPT, ADDED };
constexpr bool halves(Kind kind) { return kind == GATED || kind == KEPT; }

// Where a tile's outputs go
template <int J, Kind KIND>
struct Outputs;

template <int J>
struct Outputs<J, PLAIN> : TileRows<J> {
  const Parts& parts;
  const long M;
  DEV_INLINE Outputs(bf16_t*, const Parts& parts_, long M_) : parts(parts_), M(M_) {}
  DEV_INLINE void tile(const Place& at) {
    long col = (long)at.col * SIDE;
    const Part p = part_of(parts, col);
    this->start(p.out, M, p.n, at, col);
  }
};

// Two row parts' old numbers are on their way at once (all of a tile's: no gain)
template <int J>
struct Outputs<J, ADDED> : TileRows<J> {
  const Part part;
  const long M;
  OutRows old;
  static constexpr int AHEAD = 2;
  u32x4_t held[AHEAD][4];
  DEV_INLINE Outputs(bf16_t*, const Parts& parts, long M_) : part(parts.p[0]), M(M_) {}
  DEV_INLINE void load(int j) {
    old.next();
#pragma unroll
    for (int q = 0; q < 4; ++q) held[j % AHEAD][q] = old.get(this->offset[q]);
  }
  DEV_INLINE void tile(const Place& at) {
    this->start(part.out, M, part.n, at, (long)at.col * SIDE);
    old = this->to;
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) load(j);
  }
  // (the part before is stored)
  DEV_INLINE void rows(int j) {
    this->to.next();
    if (j > 0 && j - 1 + AHEAD < J) load(j - 1 + AHEAD);
  }
  DEV_INLINE void put(int j, int q, const f32x4_t (&sums)[2]) const {
    // the old numbers where the sums' lanes have theirs: lanes exchanged as in
    // eight_columns, the other way
    f32x4_t c[2] = {sums[0], sums[1]};
    const u32x4_t& now = held[j % AHEAD][q];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const auto p = __builtin_amdgcn_permlane16_swap(now[w], now[2 + w], false, false);
      const auto x = __builtin_amdgcn_permlane32_swap(p[0], p[1], false, false);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        c[h][2 * w] += __uint_as_float(x[h] << 16);
        c[h][2 * w + 1] += __uint_as_float(x[h] & 0xffff0000u);
      }
    }
    this->to.put(this->offset[q], eight_columns(c[0], c[1]), this->past);
  }
};

// Gate's and up projection's column parts are four apart
template <int J, Kind KIND>
struct Outputs {
  static constexpr int COLS = 4, STORES = KIND == KEPT ? 6 : 2;
  static constexpr int column_of(int q, int e) { return 2 * q + (e & 1) + 4 * (e >> 1); }
  bf16_t* const out;
  const Parts& parts;
  const long M;
  OutRows to, gate, up;
  unsigned offset[2];
  DEV_INLINE Outputs(bf16_t* out_, const Parts& parts_, long M_)
      : out(out_), parts(parts_), M(M_) {}
  DEV_INLINE void tile(const Place& at) {
    const int lane = threadIdx.x & 63, wid = wave_id();
    const long N = parts.p[0].n;
    const long row0 = (long)at.row * (32 * J) + (wid & 1) * (16 * J);
    to.start(out, M, N, row0);
    if (KIND == KEPT)
      gate.start(parts.p[0].out, M, N, row0), up.start(parts.p[1].out, M, N, row0);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      offset[q] = OutRows::offset(
          N, (long)at.col * 128 + (wid >> 1) * 64 + 32 * q + 8 * (lane >> 4));
  }
  DEV_INLINE void rows(int) {
    to.next();
    if (KIND == KEPT) gate.next(), up.next();
  }
  DEV_INLINE void put(int, int q, const f32x4_t (&sums)[4]) const {
    f32x4_t y[2];
    // (the activation first: gate times up may be beyond 32 bits where the sigmoid is 0)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        y[h][e] = sums[h][e] *
                  __builtin_amdgcn_rcpf(1.f +
                                        exp2_hw(sums[h][e] * -1.4426950408889634f)) *
                  sums[2 + h][e];
    // (a choice at each store costs the prompts' tiles 1.2 us of 67 together; 16384 rows,
    // 2048 -> 8192, 268 MB, 754 us through the L2s and 726 past them)
    to.put(offset[q], eight_columns(y[0], y[1]), KIND == GATED);
    if (KIND == KEPT) {
      gate.put(offset[q], eight_columns(sums[0], sums[1]), false);
      up.put(offset[q], eight_columns(sums[2], sums[3]), false);
    }
  }
};

template <int J, Kind KIND>
__global__ __launch_bounds__(256, 1) void linear_kernel(
    bf16_t* __restrict__ out,          // (M, n), GATED and KEPT
    const bf16_t* __restrict__ x,      // (M, K)
    const Parts parts, long M, long K, int row_tiles, int col_tiles) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  constexpr int ROWS = 32 * J, COLS = halves(KIND) ? 128 : 256;
  const int items = row_tiles * col_tiles, n = (int)(K / PAIR);
  const long N = parts.p[0].n;
  auto units = [&](int r, Units& a, Units& b, Place& at) {
    const int item = item_of(r, items, gridDim.x);
    if (item < 0) return false;
    at = Place(item, row_tiles, col_tiles);
    a = lines(x, M, K, (long)at.row * ROWS, 0, n);
    long col = (long)at.col * COLS;
    if (halves(KIND)) {
      // a wave loads the 64 rows of its number: gate, up, gate, up
      const int wid = wave_id();
      b = lines(wid & 1 ? parts.p[1].w : parts.p[0].w, N, K,
                col + (wid >> 1) * 64 - wid * 64, 0, n);
    } else {
      const Part p = part_of(parts, col);
      b = lines(p.w, p.n, K, col, 0, n);
    }
    return true;
  };
  Outputs<J, KIND> outputs(out, parts, M);
  run<true, true, J>(lds, [&](int) { return K; }, K, units, outputs);
}

// cols: tiles of columns of the weights together
template <Kind KIND>
void launch_linear(bf16_t* out, const torch::Tensor& x, const Parts& parts, long cols) {
  const long M = x.size(0), K = x.size(1);
  if (M == 0 || cols == 0) return;
  // (what is kept of the trainer's few rows is no path of its own)
  const int best = rows_of(M, cols, K, KIND == KEPT ? 6 : 3).parts;
  const long rows = (M + 32 * best - 1) / (32 * best), items = rows * cols;
  TORCH_CHECK(items < (1L << 31) - ATTN_XCDS, "grid too large");
  const dim3 grid((unsigned)blocks_of(items, K));
  auto stream = at::hip::getCurrentHIPStream();
  auto launch = [&](auto kern) {
    kern<<<grid, dim3(256), 0, stream>>>(out, (const bf16_t*)x.data_ptr(), parts, M, K,
                                         (int)rows, (int)cols);
  };
  if constexpr (KIND != KEPT) {
    if (best == 3) launch(linear_kernel<3, KIND>);
    if (best == 4) launch(linear_kernel<4, KIND>);
    if (best == 5) launch(linear_kernel<5, KIND>);
  }
  if (best == 6) launch(linear_kernel<6, KIND>);
  if (best == 7) launch(linear_kernel<7, KIND>);
  if (best == 8) launch(linear_kernel<8, KIND>);
  HIP_CHECK_KERNEL();
}

Part part(const torch::Tensor* out, const torch::Tensor& w, long first, long n) {
  return {out ? (bf16_t*)out->data_ptr() : nullptr,
          (const bf16_t*)w.data_ptr() + first * w.size(1), n};
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
  if (GLU)
    launch_linear<GATED>((bf16_t*)out.data_ptr(), x,
                         {{part(nullptr, w, 0, N), part(nullptr, w, N, N)}}, N / 128);
  else
    launch_linear<PLAIN>(nullptr, x, {{part(&out, w, 0, N)}}, N / SIDE);
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
  const long N = w.size(0);
  launch_linear<PLAIN>(nullptr, x, {{part(&out, w, 0, N)}}, (N + SIDE - 1) / SIDE);
}

// Whether linear_rows is the better choice than the library's own: tiles that fill
// rounds of 256 to 0.53 of what whole ones would cost, but not whole tiles of 256 rows,
// which the library multiplies 1 to 6% faster where it has no long inner dimension to
// choose for.  Weights beyond 16 MB come from memory: tiles of 96 rows, whose steps are
// shorter than that takes, are left to the library, ones of 128 where there are few of them.
// (us, beside the library's, weights in turn from memory: 4096 -> 1024 of 5135, 6145, 8192
// rows 46, 46, 54 and 46, 51, 58; 2048 -> 2048 of 2300, 3072, 5135 26, 27, 38 and 30, 28, 49;
// 96 rows a tile, 14336 -> 4096 of 1024, 28672 -> 8192 of 600, 8192 -> 8192 of 560, 8960 ->
// 1536 of 3072 169, 324, 107, 105 and 132, 259, 87, 93; 128, 4096 -> 6144 of 1024 and 4096, 8960
// -> 1536 of 4096, 4096 -> 4096 of 2048 56, 169, 114, 58 and 53, 156, 107, 63; 3584 -> 3584 of
// 8192 152 and 146, 18944 -> 3584 of 4096 363 and 539.  Of 399 shapes the 149 within the line
// take 0.52 to 1.06 of the library's time, 0.89 on average, six of them more than 1.02.)
bool linear_rows_pays(long M, long N, long K) {
  if (M <= 0 || N <= 0 || K < PAIR) return false;
  const long cols = (N + SIDE - 1) / SIDE;
  const Rows best = rows_of(M, cols, K, 3);
  const double whole = (double)M * N / (CUS * SIDE * SIDE) * cost_of(8, K);
  if (best.cost > 1.9 * whole) return false;
  if (best.parts == 8)
    return best.cost >= 1.05 * whole && (M % SIDE != 0 || K > 2 * N);
  if (best.parts > 4 || N * K <= 1L << 23) return true;
  const long tiles = (M + 32 * best.parts - 1) / (32 * best.parts) * cols;
  return best.parts == 4 && M > 1024 && best.cost <= 1.5 * whole && tiles <= 2 * CUS;
}

// Row parts of a tile, 32 rows each, of M rows by ``cols`` tiles of columns with K inner
// numbers, at least ``least`` (6 where products are kept or an operand is in COLUMNS, else
// 3), and what the rounds cost
std::vector<long> product_rows(long M, long cols, long K, long least) {
  TORCH_CHECK(M > 0 && cols > 0 && K > 0 && least > 0 && least <= 8, "product_rows");
  const Rows r = rows_of(M, cols, K, (int)least);
  return {r.parts, r.cost};
}

// x (M, K), w (N, K)
torch::Tensor linear_rows(torch::Tensor x, torch::Tensor w) {
  return linear_prompt<false>(x, w);
}

// out += x W^T, rounded once: what follows need not add it.  (us, the product and a norm
// that adds, and this and a norm: 1024 -> 1024 of 1024, 3072, 4096, 8192 rows 14.7, 17.2, 19.0,
// 26.6 and 16.2, 18.0, 19.2, 25.3; 4096 -> 1024 of 5135, 8192 45.5, 62.4 and 45.7, 60.0; 2048 ->
// 2048 of 2600, 4096 28.7, 38.0 and 28.3, 36.4; 4096 -> 4096 of 1300, 2048, 6145 45.1, 62.0, 174
// and 45.9, 60.7, 166; 14336 -> 4096 of 1300, 2600 135, 242 and 135, 224)
void linear_rows_add(torch::Tensor out, torch::Tensor x, torch::Tensor w) {
  for (const auto* t : {&out, &x, &w})
    TORCH_CHECK(t->is_cuda() && t->device() == x.device() && t->dim() == 2 &&
                    t->is_contiguous() && t->dtype() == torch::kBFloat16,
                "linear: contiguous 2-D bf16 of one device");
  TORCH_CHECK(w.size(1) == x.size(1) && out.size(0) == x.size(0) &&
                  out.size(1) == w.size(0) && linear_rows_fits(x, w) &&
                  ((uintptr_t)out.data_ptr() & 15) == 0,
              "linear: inner numbers in 64s, outputs in 8s, 16-byte addresses");
  const long N = w.size(0);
  launch_linear<ADDED>(nullptr, x, {{part(&out, w, 0, N)}}, (N + SIDE - 1) / SIDE);
}

// x (M, K), w (2 N, K): rows of the gate, then of the up projection
torch::Tensor linear_swiglu(torch::Tensor x, torch::Tensor w) {
  return linear_prompt<true>(x, w);
}

namespace {

// of weights of one input: the operands' form, and whether the tiles fill their rounds
bool joint_takes(const torch::Tensor& x, const std::vector<torch::Tensor>& ws, long each) {
  if (ws.size() < 2 || ws.size() > MOST || x.dim() != 2 || !x.is_cuda() ||
      !x.is_contiguous() || x.dtype() != torch::kBFloat16)
    return false;
  long N = 0;
  for (const auto& w : ws) {
    if (!w.is_cuda() || w.device() != x.device() || w.dim() != 2 || !w.is_contiguous() ||
        w.dtype() != torch::kBFloat16 || w.size(1) != x.size(1) ||
        w.size(0) % each != 0 || !linear_rows_fits(x, w))
      return false;
    N += w.size(0);
  }
  const long M = x.size(0), K = x.size(1);
  const double whole = (double)M * N / (CUS * SIDE * SIDE) * cost_of(8, K);
  return M > 512 && N < (1L << 25) &&
         rows_of(M, (N + SIDE - 1) / SIDE, K, 6).cost <= 1.35 * whole;
}

}  // namespace

// Whether linear_joint has these operands (contiguous bf16 matrices, the weights' rows in
// 256s) and is the better choice than a product each: rounds that cost up to 1.35 of whole
// ones.  (That, us and a product each, weights in turn from memory: 4096 -> 4096, 1024, 1024
// of 7168, 4096, 2048 rows, 1.04, 1.21, 1.21, 249, 169, 80 and 291, 181, 125; 8192 -> 8192, 1024,
// 1024 of 2048, 1.30, 288 and 280.  Beyond the line it would gain as well: 4096 of 3072 and
// 1536 rows, both 1.46, 131, 65 and 150, 107, 1536 -> 1536, 256, 256 of 4096, 1.68, 25 and 57.)
bool linear_joint_takes(const torch::Tensor& x, const std::vector<torch::Tensor>& ws) {
  return joint_takes(x, ws, SIDE);
}

// x W_p^T of two or three weights (N_p, K)
std::vector<torch::Tensor> linear_joint(torch::Tensor x, std::vector<torch::Tensor> ws) {
  TORCH_CHECK(joint_takes(x, ws, SIDE), "linear_joint: operands that it does not take");
  std::vector<torch::Tensor> outs;
  Parts parts = {};
  long cols = 0;
  for (size_t i = 0; i < ws.size(); ++i) {
    outs.push_back(torch::empty({x.size(0), ws[i].size(0)}, x.options()));
    parts.p[i] = part(&outs[i], ws[i], 0, ws[i].size(0));
    cols += ws[i].size(0) / SIDE;
  }
  launch_linear<PLAIN>(nullptr, x, parts, cols);
  return outs;
}

// The same for linear_gated: rows of weights in 128s, as many of both.  (With the products
// stored, us and two products with the activation's pass: 2048 -> 8192 of 8192 rows, 1.00, 462
// and 468, 4096 -> 14336 of 2048, 7168, 1.14, 1.04, 382, 1186 and 384, 1323; beyond the line
// 4096 -> 14336 of 700 and 520, 1.37, 1.85, 157, 151 and 181, 145, 1024 -> 4096 of 1024, 1.70, 26
// and 43.)
bool linear_gated_takes(const torch::Tensor& x, const torch::Tensor& wg,
                        const torch::Tensor& wu) {
  return wg.dim() == 2 && wu.dim() == 2 && wg.size(0) == wu.size(0) &&
         joint_takes(x, {wg, wu}, 128);
}

// silu(gate) * up, and with keep gate = x Wg^T and up = x Wu^T behind it
std::vector<torch::Tensor> linear_gated(torch::Tensor x, torch::Tensor wg,
                                        torch::Tensor wu, bool keep) {
  TORCH_CHECK(linear_gated_takes(x, wg, wu),
              "linear_gated: operands that it does not take");
  const long N = wg.size(0);
  std::vector<torch::Tensor> outs;
  for (int i = 0; i < (keep ? 3 : 1); ++i)
    outs.push_back(torch::empty({x.size(0), N}, x.options()));
  const Parts parts = {{part(keep ? &outs[1] : nullptr, wg, 0, N),
                        part(keep ? &outs[2] : nullptr, wu, 0, N)}};
  (keep ? launch_linear<KEPT> : launch_linear<GATED>)((bf16_t*)outs[0].data_ptr(), x,
                                                      parts, N / 128);
  return outs;
}
