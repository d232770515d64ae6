// The trainer's packed rows: which tokens of a padded batch (B, L) are real, their
// rows in one packed sequence of sequences, hidden rows back to the places that are
// asked for, and the gradient of the embedding.
//
// Reference capability: remove-padding (unpad / pad) around the packed forward, and
// the embedding's backward.
//
// A boolean index is a count, a wait of the host for it, a scan and a gather, each
// time it is used (two gathers in, one scatter out, one gather in the backward pass:
// 30 launches and five waits of an actor step's start).  Here the rows' lengths and the
// largest position come back to the host in one copy, and every map in one launch
// after it.
//
// What bounds it: the launches (5 us each) and, where hidden rows move, memory: 8192
// rows of 4096 numbers of bf16 are read and written once.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "attention_tile.h"

namespace {

// ------------------------------------------------------------------ lengths
// info (2, B): tokens of a row; the largest of their positions (-1: none)
__global__ __launch_bounds__(256) void pack_lengths_kernel(
    int* __restrict__ info, const bool* __restrict__ mask,
    const int64_t* __restrict__ pos, int B, long L) {
  const long row = (long)blockIdx.x * L;
  int n = 0, most = -1;
  for (long l = threadIdx.x; l < L; l += 256)
    if (mask[row + l]) {
      ++n;
      most = max(most, (int)pos[row + l]);
    }
  __shared__ int ns[4], ms[4];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    n += __shfl_xor(n, off, 64);
    most = max(most, __shfl_xor(most, off, 64));
  }
  if ((threadIdx.x & 63) == 0) ns[wave_id()] = n, ms[wave_id()] = most;
  __syncthreads();
  if (threadIdx.x == 0) {
    info[blockIdx.x] = ns[0] + ns[1] + ns[2] + ns[3];
    info[B + blockIdx.x] = max(max(ms[0], ms[1]), max(ms[2], ms[3]));
  }
}

// --------------------------------------------------------------------- maps
// Block b < B: the tokens of row b to their packed rows, and the packed row of every
// place in [lo, hi) (-1: none); block B: the rows that fill up to ``padded``, tokens 0
// at positions 0, 1, ..  place[t]: where in the rows of [lo, hi) packed row t goes.
__global__ __launch_bounds__(256) void pack_rows_kernel(
    int64_t* __restrict__ ids_out, int64_t* __restrict__ pos_out,
    int* __restrict__ packed, int* __restrict__ place,
    const bool* __restrict__ mask, const int64_t* __restrict__ ids,
    const int64_t* __restrict__ pos, const int* __restrict__ cu, int B, long L,
    long lo, long hi, int total, int padded) {
  const int b = blockIdx.x, lane = threadIdx.x & 63, wid = wave_id();
  if (b == B) {
    for (int t = total + threadIdx.x; t < padded; t += 256)
      ids_out[t] = 0, pos_out[t] = t - total, place[t] = -1;
    return;
  }
  const long row = (long)b * L;
  int at = cu[b];
  __shared__ int count[2][4];
  int turn = 0;
  for (long l0 = 0; l0 < L; l0 += 256, turn ^= 1) {
    const long l = l0 + threadIdx.x;
    const bool live = l < L && mask[row + l];
    const unsigned long long all = __ballot(live);
    if (lane == 0) count[turn][wid] = __popcll(all);
    __syncthreads();                   // (the other turn's are read before the next)
    int t = at + __popcll(all & ((1ull << lane) - 1));
    for (int w = 0; w < wid; ++w) t += count[turn][w];
    const bool asked = l >= lo && l < hi;
    const long out = (long)b * (hi - lo) + l - lo;
    if (live) {
      ids_out[t] = ids[row + l];
      pos_out[t] = pos[row + l];
      place[t] = asked ? (int)out : -1;
    }
    if (asked) packed[out] = live ? t : -1;
    at += count[turn][0] + count[turn][1] + count[turn][2] + count[turn][3];
  }
}

// ------------------------------------------------------------------- gather
// out[r] = from[map[r]], zeros where map[r] < 0; rows of ``words`` 16-byte words
__global__ __launch_bounds__(256) void gather_rows_kernel(
    u32x4_t* __restrict__ out, const u32x4_t* __restrict__ from,
    const int* __restrict__ map, long rows, int words) {
  const long n = rows * words, stride = (long)gridDim.x * 256;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    const long r = i / words;
    const int t = map[r];
    out[i] = t < 0 ? u32x4_t{0, 0, 0, 0} : from[(long)t * words + (i - r * words)];
  }
}

// -------------------------------------------------------- embedding gradient
// Tokens in the order (id, row): a token's place is the number of tokens before it
// in that order, counted by comparing it with all, 256 of them and a stretch of the
// others a block; the counts add up the same in any order.  (7168 tokens, rows of 4096
// numbers, 128256 ids: ranks 11 us, order 5, sums 39, shares 5, the fill 139; a sort's
// scans and merges, sums and their scatter took 300 beside the fill.  The whole, beside
// the library's backward, which sorts, of 512, 2048, 7168 and 32768 tokens 172, 180, 208, 403
// and 202, 336, 429, 1276; an id that a fourth, half and all of 32768 tokens have 692, 969,
// 1538 and 1188, 1424, 1529, of 7168 all 450 and 487: its shares are added up one after the
// other.  32768 tokens of 32000 ids, 1024 numbers, 157 and 248, ids by Zipf's law 211 and 222:
// comparisons grow with the square of the tokens, and beyond that it is the library's.)
constexpr int STRETCH = 256;

__global__ __launch_bounds__(256) void embed_rank_kernel(
    int* __restrict__ rank, const int64_t* __restrict__ ids, int T) {
  __shared__ __attribute__((aligned(16))) int other[STRETCH];
  const int t = blockIdx.x * 256 + threadIdx.x, o0 = blockIdx.y * STRETCH;
  for (int i = threadIdx.x; i < STRETCH; i += 256)
    other[i] = o0 + i < T ? (int)ids[o0 + i] : 0x7fffffff;
  const int id = t < T ? (int)ids[t] : 0;
  __syncthreads();
  int n = 0;
  // an earlier row of the same id counts, a later one does not
  const int same = min(max(t - o0, 0), STRETCH);
#pragma unroll 8
  for (int i = 0; i < STRETCH; i += 4) {
    const i32x4_t o = *reinterpret_cast<const i32x4_t*>(other + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) n += o[j] < id + (i + j < same ? 1 : 0);
  }
  if (t < T && n > 0) atomicAdd(rank + t, n);
}

__global__ void embed_order_kernel(int* __restrict__ order,
                                   int* __restrict__ sorted,
                                   const int* __restrict__ rank,
                                   const int64_t* __restrict__ ids, int T) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= T) return;
  order[rank[t]] = t;
  sorted[rank[t]] = (int)ids[t];
}

constexpr int WINDOW = 32;             // rows that one block adds up

// Block p: where an id's rows start at p, or go on at a window's start, the sum of
// them up to the window's end: the gradient's row, or a share of it.  Shares: of the
// id that goes on at window w's start at place w, of the one that starts in it and
// goes on behind it at windows + w.
__global__ __launch_bounds__(256) void embed_sum_kernel(
    bf16_t* __restrict__ dw, float* __restrict__ shares,
    const bf16_t* __restrict__ dy, const int* __restrict__ order,
    const int* __restrict__ sorted, int T, int H, int V) {
  const int p = blockIdx.x, lane = threadIdx.x & 63;
  const int border = min((p / WINDOW + 1) * WINDOW, T);
  // lane l < 32: place p + l and its row; lane 63: the place before
  const int at = lane == 63 ? p - 1 : p + lane;
  int own = -1, row = 0;
  if (at >= 0 && at <= border && at < T) own = sorted[at], row = order[at];
  const int id = uniform(own);
  const bool starts = p == 0 || __builtin_amdgcn_readlane(own, 63) != id;
  if ((!starts && p % WINDOW != 0) || (unsigned)id >= (unsigned)V) return;
  const unsigned long long same = __ballot(own == id && lane <= WINDOW);
  const int n = min(__ffsll((long long)~same) - 1, border - p);
  const bool goes_on = border < T && (same >> (border - p) & 1) &&
                       n == border - p;
  const int windows = (T + WINDOW - 1) / WINDOW;
  for (int h = threadIdx.x * 8; h < H; h += 256 * 8) {
    float sum[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sum[e] = 0.f;
    int r = 0;
    for (; r + 4 <= n; r += 4) {       // (four rows on their way at once)
      bf16x8_t v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] = *reinterpret_cast<const bf16x8_t*>(
            dy + (long)__builtin_amdgcn_readlane(row, r + i) * H + h);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] += (float)v[i][e];
    }
    for (; r < n; ++r) {
      const bf16x8_t v = *reinterpret_cast<const bf16x8_t*>(
          dy + (long)__builtin_amdgcn_readlane(row, r) * H + h);
#pragma unroll
      for (int e = 0; e < 8; ++e) sum[e] += (float)v[e];
    }
    if (starts && !goes_on) {
      bf16x8_t w;
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = (__bf16)sum[e];
      *reinterpret_cast<bf16x8_t*>(dw + (long)id * H + h) = w;
    } else {
      float* to = shares + (long)(p / WINDOW + (starts ? windows : 0)) * H + h;
#pragma unroll
      for (int e = 0; e < 8; ++e) to[e] = sum[e];
    }
  }
}

// Block w: the sum of the shares of the id that starts in window w and goes on
// behind it
__global__ __launch_bounds__(256) void embed_shares_kernel(
    bf16_t* __restrict__ dw, const float* __restrict__ shares,
    const int* __restrict__ sorted, int T, int H, int V) {
  const int w = blockIdx.x, windows = (T + WINDOW - 1) / WINDOW;
  const int border = (w + 1) * WINDOW;
  if (border >= T) return;
  const int id = sorted[border - 1];
  if (sorted[border] != id || (unsigned)id >= (unsigned)V) return;
  if (w > 0 && sorted[w * WINDOW - 1] == id) return;   // it started before
  int last = w + 1;                    // last window that it reaches
  while ((last + 1) * WINDOW < T && sorted[(last + 1) * WINDOW] == id) ++last;
  for (int h = threadIdx.x * 4; h < H; h += 256 * 4) {
    f32x4v sum = *reinterpret_cast<const f32x4v*>(shares + (long)(windows + w) * H + h);
#pragma unroll 4
    for (int o = w + 1; o <= last; ++o) {
      const f32x4v v = *reinterpret_cast<const f32x4v*>(shares + (long)o * H + h);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum.v[e] += v.v[e];
    }
    bf16x4 out;
#pragma unroll
    for (int e = 0; e < 4; ++e) out.v[e] = f2bf(sum.v[e]);
    *reinterpret_cast<bf16x4*>(dw + (long)id * H + h) = out;
  }
}

void check_tokens(const torch::Tensor& t, const torch::Tensor& like,
                  torch::ScalarType type, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.dim() == 2 && t.is_contiguous() &&
                  t.scalar_type() == type && t.sizes() == like.sizes(),
              "pack: ", name);
}

}  // namespace

// (2, B) int32: tokens of every row of mask (B, L) bool, the largest of their
// positions
torch::Tensor pack_lengths(torch::Tensor mask, torch::Tensor pos) {
  check_tokens(mask, mask, torch::kBool, "mask (B, L) bool");
  check_tokens(pos, mask, torch::kInt64, "positions (B, L) int64");
  const long B = mask.size(0);
  TORCH_CHECK(mask.numel() < (1L << 31), "pack: too many places");
  auto info = torch::empty({2, B}, pos.options().dtype(torch::kInt32));
  if (B == 0) return info;
  pack_lengths_kernel<<<dim3((unsigned)B), dim3(256), 0,
                        at::hip::getCurrentHIPStream()>>>(
      info.data_ptr<int>(), mask.data_ptr<bool>(), pos.data_ptr<int64_t>(),
      (int)B, mask.size(1));
  HIP_CHECK_KERNEL();
  return info;
}

// Packed tokens and positions (padded), the packed rows of places [lo, hi) of every
// row (B, hi - lo), the place of every packed row.  cu: where the rows' tokens start.
std::vector<torch::Tensor> pack_rows(torch::Tensor mask, torch::Tensor ids,
                                     torch::Tensor pos, torch::Tensor cu,
                                     int64_t total, int64_t padded, int64_t lo,
                                     int64_t hi) {
  check_tokens(mask, mask, torch::kBool, "mask (B, L) bool");
  check_tokens(ids, mask, torch::kInt64, "ids (B, L) int64");
  check_tokens(pos, mask, torch::kInt64, "positions (B, L) int64");
  const long B = mask.size(0), L = mask.size(1);
  TORCH_CHECK(cu.is_cuda() && cu.scalar_type() == torch::kInt32 &&
                  cu.is_contiguous() && cu.numel() > B,
              "pack: cu (B + 1) int32");
  TORCH_CHECK(0 <= lo && lo <= hi && hi <= L && 0 <= total && total <= padded &&
                  total <= B * L && padded < (1L << 31) && B * L < (1L << 31),
              "pack: sizes");
  auto i32 = cu.options();
  std::vector<torch::Tensor> out = {
      torch::empty({padded}, ids.options()), torch::empty({padded}, ids.options()),
      torch::empty({B, hi - lo}, i32), torch::empty({padded}, i32)};
  pack_rows_kernel<<<dim3((unsigned)B + 1), dim3(256), 0,
                     at::hip::getCurrentHIPStream()>>>(
      out[0].data_ptr<int64_t>(), out[1].data_ptr<int64_t>(),
      out[2].data_ptr<int>(), out[3].data_ptr<int>(), mask.data_ptr<bool>(),
      ids.data_ptr<int64_t>(), pos.data_ptr<int64_t>(), cu.data_ptr<int>(),
      (int)B, L, lo, hi, (int)total, (int)padded);
  HIP_CHECK_KERNEL();
  return out;
}

// x (T, H) rows map (int32, any shape) names; zeros where it is negative
torch::Tensor gather_rows(torch::Tensor x, torch::Tensor map) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.is_contiguous() &&
                  x.scalar_type() == torch::kBFloat16 && x.size(1) % 8 == 0 &&
                  ((uintptr_t)x.data_ptr() & 15) == 0,
              "gather_rows: contiguous (T, H) bf16 in 16-byte words");
  TORCH_CHECK(map.is_cuda() && map.is_contiguous() &&
                  map.scalar_type() == torch::kInt32,
              "gather_rows: int32 map");
  auto shape = map.sizes().vec();
  shape.push_back(x.size(1));
  auto out = torch::empty(shape, x.options());
  const long rows = map.numel();
  const int words = x.size(1) / 8;
  if (rows * words == 0) return out;
  const long blocks = std::min((rows * words + 255) / 256, 8192L);
  gather_rows_kernel<<<dim3((unsigned)blocks), dim3(256), 0,
                       at::hip::getCurrentHIPStream()>>>(
      (u32x4_t*)out.data_ptr(), (const u32x4_t*)x.data_ptr(),
      map.data_ptr<int>(), rows, words);
  HIP_CHECK_KERNEL();
  return out;
}

// Gradient (V, H) of an embedding whose rows ``ids`` (T) got gradients dy (T, H):
// fp32 sums in the order of the rows
torch::Tensor embed_grad(torch::Tensor dy, torch::Tensor ids, int64_t V) {
  TORCH_CHECK(dy.is_cuda() && dy.dim() == 2 && dy.is_contiguous() &&
                  dy.scalar_type() == torch::kBFloat16 && dy.size(1) % 8 == 0 &&
                  ((uintptr_t)dy.data_ptr() & 15) == 0,
              "embed_grad: contiguous (T, H) bf16 in 16-byte words");
  TORCH_CHECK(ids.is_cuda() && ids.dim() == 1 && ids.is_contiguous() &&
                  ids.scalar_type() == torch::kInt64 &&
                  ids.size(0) == dy.size(0) && V < (1L << 31) - 1,
              "embed_grad: ids (T) int64");
  const long T = dy.size(0), H = dy.size(1);
  TORCH_CHECK(T <= 32768, "embed_grad: at most 32768 rows");
  auto dw = torch::zeros({V, H}, dy.options());
  if (T == 0 || H == 0) return dw;
  auto i32 = ids.options().dtype(torch::kInt32);
  auto rank = torch::zeros({T}, i32);
  auto order = torch::empty({2, T}, i32);
  const long windows = (T + WINDOW - 1) / WINDOW;
  auto shares = torch::empty({2 * windows, H}, dy.options().dtype(torch::kFloat32));
  int* sorted = order.data_ptr<int>() + T;
  auto stream = at::hip::getCurrentHIPStream();
  const unsigned blocks = (T + 255) / 256;
  embed_rank_kernel<<<dim3(blocks, (unsigned)((T + STRETCH - 1) / STRETCH)),
                      dim3(256), 0, stream>>>(rank.data_ptr<int>(),
                                              ids.data_ptr<int64_t>(), (int)T);
  embed_order_kernel<<<dim3(blocks), dim3(256), 0, stream>>>(
      order.data_ptr<int>(), sorted, rank.data_ptr<int>(),
      ids.data_ptr<int64_t>(), (int)T);
  embed_sum_kernel<<<dim3((unsigned)T), dim3(256), 0, stream>>>(
      (bf16_t*)dw.data_ptr(), shares.data_ptr<float>(),
      (const bf16_t*)dy.data_ptr(), order.data_ptr<int>(), sorted, (int)T, (int)H,
      (int)V);
  embed_shares_kernel<<<dim3((unsigned)windows), dim3(256), 0, stream>>>(
      (bf16_t*)dw.data_ptr(), shares.data_ptr<float>(), sorted, (int)T, (int)H,
      (int)V);
  HIP_CHECK_KERNEL();
  return dw;
}
