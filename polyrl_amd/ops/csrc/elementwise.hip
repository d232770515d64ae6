// Memory-bound decoder-layer kernels: RMSNorm, fused add+RMSNorm, SiLU-mul,
// RoPE (NEOX rotate-half, table-driven).
//
// All bf16 I/O is vectorized as bf16x8 (16 B/lane, guide G13); accumulation
// in fp32.  Reference semantics: polyrl_amd/ops/ref.py.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"

// ------------------------------------------------------------------ RMSNorm
// One block per row; D multiple of 8.  V > 0: a row is at most V words of 16 bytes a
// thread, which stay in registers between the sum of squares and the output, and the
// block has as many waves as that takes; 0: longer rows, read twice.
//
// What bounds it: memory, in few rows the chain of load, sum and store.  (us, the sum with
// a residual, by a block of 256 threads that reads what it wrote again, and now: 1, 128,
// 2048, 5135 rows of 1024 2.1, 2.4, 4.1, 7.3 and 1.8, 2.2, 3.7, 6.2; 1, 128, 512, 16384 rows of
// 4096 2.6, 3.2, 4.3, 96 and 2.0, 2.6, 3.8, 88; 1, 5135 rows of 8192 3.7, 60 and 2.5, 48.)
template <bool FUSED_ADD, int NT, int V>
__global__ __launch_bounds__(NT) void rmsnorm_kernel(
    bf16_t* __restrict__ out,
    bf16_t* __restrict__ residual,     // inout if FUSED_ADD
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ weight, int D,
    float eps) {
  __shared__ float red[NT / 64];
  const int row = blockIdx.x;
  const bf16x8* xr = reinterpret_cast<const bf16x8*>(x + (long)row * D);
  bf16x8* rr =
      FUSED_ADD ? reinterpret_cast<bf16x8*>(residual + (long)row * D) : nullptr;
  const bf16x8* wr = reinterpret_cast<const bf16x8*>(weight);
  bf16x8* outr = reinterpret_cast<bf16x8*>(out + (long)row * D);
  const int nvec = D / 8;
  float ss = 0.f;
  // a word of the row, the residual added to it and written back
  auto summed = [&](int i) {
    bf16x8 v = xr[i];
    if (FUSED_ADD) {
      const bf16x8 r = rr[i];
#pragma unroll
      for (int j = 0; j < 8; ++j) v.v[j] = f2bf(bf2f(v.v[j]) + bf2f(r.v[j]));
      rr[i] = v;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float f = bf2f(v.v[j]);
      ss += f * f;
    }
    return v;
  };
  auto scaled = [&](int i, const bf16x8& v, const bf16x8& w, float inv) {
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o.v[j] = f2bf(bf2f(v.v[j]) * inv * bf2f(w.v[j]));
    outr[i] = o;
  };
  if constexpr (V > 0) {
    bf16x8 v[V], w[V];
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const int i = threadIdx.x + u * NT;
      if (i < nvec) w[u] = wr[i], v[u] = summed(i);
    }
    const float inv = rsqrtf(block_reduce_sum<NT / 64>(ss, red) / D + eps);
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const int i = threadIdx.x + u * NT;
      if (i < nvec) scaled(i, v[u], w[u], inv);
    }
  } else {
    for (int i = threadIdx.x; i < nvec; i += NT) summed(i);
    const float inv = rsqrtf(block_reduce_sum<NT / 64>(ss, red) / D + eps);
    for (int i = threadIdx.x; i < nvec; i += NT)
      scaled(i, FUSED_ADD ? rr[i] : xr[i], wr[i], inv);
  }
}

template <bool FUSED_ADD>
static void launch_rmsnorm(torch::Tensor& out, bf16_t* residual,
                           const torch::Tensor& x, const torch::Tensor& weight,
                           double eps) {
  const int D = x.size(-1);
  TORCH_CHECK(D % 8 == 0, "hidden dim must be a multiple of 8");
  const long rows = x.numel() / D;
  auto stream = at::hip::getCurrentHIPStream();
  auto launch = [&](auto kern, int threads) {
    kern<<<dim3(rows), dim3(threads), 0, stream>>>(
        (bf16_t*)out.data_ptr(), residual, (const bf16_t*)x.data_ptr(),
        (const bf16_t*)weight.data_ptr(), D, (float)eps);
  };
  if (D <= 512) launch(rmsnorm_kernel<FUSED_ADD, 64, 1>, 64);
  else if (D <= 1024) launch(rmsnorm_kernel<FUSED_ADD, 128, 1>, 128);
  else if (D <= 2048) launch(rmsnorm_kernel<FUSED_ADD, 256, 1>, 256);
  // (rows of 3072 to 8192 numbers, 10 to 20 MiB of them, are read again the faster: 2048 of
  // 3072 and 4096, 1792 of 4608, 1536 of 5120, 1024 of 8192 6.4, 9.0, 8.7, 8.4, 8.9 us, from
  // registers 7.5, 10.7, 10.4, 9.5, 9.5; 1792 of 5632 12.0 and 12.5; not of 1280 x 4096, 1024 x
  // 5120 6.0, 6.3 and 5.9, 5.8, 3072 x 4096, 2304 x 5120 15.8, 15.7 and 15.3, 14.6, nor 2048 to
  // 4096 rows of 2560 6.1, 14.0 and 6.1, 13.3)
  else if (FUSED_ADD && D >= 3072 && D <= 8192 && rows * D >= 21 << 18 &&
           rows * D <= 10 << 20)
    launch(rmsnorm_kernel<FUSED_ADD, 256, 0>, 256);
  else if (D <= 4096) launch(rmsnorm_kernel<FUSED_ADD, 512, 1>, 512);
  else if (D <= 8192) launch(rmsnorm_kernel<FUSED_ADD, 512, 2>, 512);
  else launch(rmsnorm_kernel<FUSED_ADD, 256, 0>, 256);
  HIP_CHECK_KERNEL();
}

void rmsnorm(torch::Tensor out, torch::Tensor x, torch::Tensor weight,
             double eps) {
  TORCH_CHECK(x.is_cuda() && x.dtype() == torch::kBFloat16);
  TORCH_CHECK(x.is_contiguous() && out.is_contiguous());
  launch_rmsnorm<false>(out, nullptr, x, weight, eps);
}

void fused_add_rmsnorm(torch::Tensor out, torch::Tensor residual,
                       torch::Tensor x, torch::Tensor weight, double eps) {
  TORCH_CHECK(x.is_cuda() && x.dtype() == torch::kBFloat16);
  TORCH_CHECK(x.is_contiguous() && residual.is_contiguous() && out.is_contiguous());
  launch_rmsnorm<true>(out, (bf16_t*)residual.data_ptr(), x, weight, eps);
}

// ----------------------------------------------------------------- SiLU-mul
// gate/up may be strided row views into a fused (N, 2I) gate_up projection
// (row stride ldg/ldu elements, inner dim contiguous) — avoids the
// .contiguous() copies in the engine forward.
__global__ void silu_mul_kernel(bf16_t* __restrict__ out,
                                const bf16_t* __restrict__ gate,
                                const bf16_t* __restrict__ up, long rows,
                                int cvec /* cols/8 */, long ldg, long ldu) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long stride = (long)gridDim.x * blockDim.x;
  const long nvec = rows * cvec;
  for (; i < nvec; i += stride) {
    const long r = i / cvec;
    const long c = i % cvec;
    bf16x8 g = *reinterpret_cast<const bf16x8*>(gate + r * ldg + c * 8);
    bf16x8 u = *reinterpret_cast<const bf16x8*>(up + r * ldu + c * 8);
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float gf = bf2f(g.v[j]);
      float s = gf / (1.f + __expf(-gf));
      o.v[j] = f2bf(s * bf2f(u.v[j]));
    }
    reinterpret_cast<bf16x8*>(out)[i] = o;
  }
}

// training backward of silu(gate)*up: one pass, contiguous operands
// dgate = dy * up * (sig + g*sig*(1-sig)); dup = dy * silu(g)
__global__ void silu_mul_bwd_kernel(bf16_t* __restrict__ dgate,
                                    bf16_t* __restrict__ dup,
                                    const bf16_t* __restrict__ dy,
                                    const bf16_t* __restrict__ gate,
                                    const bf16_t* __restrict__ up,
                                    long nvec) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long stride = (long)gridDim.x * blockDim.x;
  for (; i < nvec; i += stride) {
    bf16x8 d = reinterpret_cast<const bf16x8*>(dy)[i];
    bf16x8 g = reinterpret_cast<const bf16x8*>(gate)[i];
    bf16x8 u = reinterpret_cast<const bf16x8*>(up)[i];
    bf16x8 og, ou;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float gf = bf2f(g.v[j]);
      const float df = bf2f(d.v[j]);
      const float sig = 1.f / (1.f + __expf(-gf));
      const float silu = gf * sig;
      og.v[j] = f2bf(df * bf2f(u.v[j]) * (sig + gf * sig * (1.f - sig)));
      ou.v[j] = f2bf(df * silu);
    }
    reinterpret_cast<bf16x8*>(dgate)[i] = og;
    reinterpret_cast<bf16x8*>(dup)[i] = ou;
  }
}

void silu_mul_bwd(torch::Tensor dgate, torch::Tensor dup, torch::Tensor dy,
                  torch::Tensor gate, torch::Tensor up) {
  TORCH_CHECK(dy.is_cuda() && dy.dtype() == torch::kBFloat16);
  TORCH_CHECK(dy.is_contiguous() && gate.is_contiguous() &&
              up.is_contiguous() && dgate.is_contiguous() &&
              dup.is_contiguous());
  TORCH_CHECK(gate.numel() % 8 == 0);
  const long nvec = gate.numel() / 8;
  const long blocks = std::min<long>((nvec + 255) / 256,
                                     MAX_RESIDENT_BLOCKS);
  auto stream = at::hip::getCurrentHIPStream();
  silu_mul_bwd_kernel<<<dim3(blocks), dim3(256), 0, stream>>>(
      (bf16_t*)dgate.data_ptr(), (bf16_t*)dup.data_ptr(),
      (const bf16_t*)dy.data_ptr(), (const bf16_t*)gate.data_ptr(),
      (const bf16_t*)up.data_ptr(), nvec);
  HIP_CHECK_KERNEL();
}

void silu_mul(torch::Tensor out, torch::Tensor gate, torch::Tensor up) {
  TORCH_CHECK(gate.is_cuda() && gate.dtype() == torch::kBFloat16);
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(gate.dim() == 2 && up.dim() == 2);
  TORCH_CHECK(gate.stride(1) == 1 && up.stride(1) == 1,
              "inner dim must be contiguous");
  const long rows = gate.size(0);
  const long cols = gate.size(1);
  TORCH_CHECK(cols % 8 == 0);
  const long nvec = rows * (cols / 8);
  int blocks = (int)std::min<long>((nvec + 255) / 256, MAX_RESIDENT_BLOCKS);
  auto stream = at::hip::getCurrentHIPStream();
  silu_mul_kernel<<<dim3(blocks), dim3(256), 0, stream>>>(
      (bf16_t*)out.data_ptr(), (const bf16_t*)gate.data_ptr(),
      (const bf16_t*)up.data_ptr(), rows, (int)(cols / 8), gate.stride(0),
      up.stride(0));
  HIP_CHECK_KERNEL();
}

// --------------------------------------------------------------------- RoPE
// NEOX rotate-half, in place on q and k. cos/sin tables precomputed on host
// (guide App. B: never on-device trig), fp32, indexed by per-token position.
// q: (N, Hq, D) k: (N, Hk, D) contiguous; cos/sin: (max_pos, D/2).
// One block per token; threads cover (head, d) pairs; d pairs are
// (d, d + D/2). Loads are bf16x4 (8 B) on each half.
__global__ void rope_kernel(bf16_t* __restrict__ q, bf16_t* __restrict__ k,
                            const int* __restrict__ positions,
                            const float* __restrict__ cos_tab,
                            const float* __restrict__ sin_tab, int Hq, int Hk,
                            int D, long ldq, long ldk /* token strides */) {
  const int tok = blockIdx.x;
  const int pos = positions[tok];
  const int half = D / 2;
  const float* c = cos_tab + (long)pos * half;
  const float* s = sin_tab + (long)pos * half;
  const int H = Hq + Hk;
  // each thread handles 4 consecutive rotary pairs of one head
  const int quads_per_head = half / 4;
  for (int t = threadIdx.x; t < H * quads_per_head; t += blockDim.x) {
    const int h = t / quads_per_head;
    const int qd = (t % quads_per_head) * 4;
    bf16_t* base = (h < Hq) ? q + (long)tok * ldq + (long)h * D
                            : k + (long)tok * ldk + (long)(h - Hq) * D;
    bf16x4 x1 = *reinterpret_cast<bf16x4*>(base + qd);
    bf16x4 x2 = *reinterpret_cast<bf16x4*>(base + half + qd);
    float4 cv = *reinterpret_cast<const float4*>(c + qd);
    float4 sv = *reinterpret_cast<const float4*>(s + qd);
    const float cc[4] = {cv.x, cv.y, cv.z, cv.w};
    const float ss[4] = {sv.x, sv.y, sv.z, sv.w};
    bf16x4 o1, o2;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float a = bf2f(x1.v[j]), b = bf2f(x2.v[j]);
      o1.v[j] = f2bf(a * cc[j] - b * ss[j]);
      o2.v[j] = f2bf(b * cc[j] + a * ss[j]);
    }
    *reinterpret_cast<bf16x4*>(base + qd) = o1;
    *reinterpret_cast<bf16x4*>(base + half + qd) = o2;
  }
}

void rope_inplace(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
                  torch::Tensor cos_tab, torch::Tensor sin_tab) {
  // q: (N, Hq, D), k: (N, Hk, D); token stride may exceed Hq*D (views into a
  // fused qkv projection), heads/dims must be contiguous.
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16);
  TORCH_CHECK(q.stride(2) == 1 && k.stride(2) == 1);
  TORCH_CHECK(q.stride(1) == q.size(2) && k.stride(1) == k.size(2),
              "head dim must be packed");
  TORCH_CHECK(positions.dtype() == torch::kInt32);
  const int N = q.size(0), Hq = q.size(1), D = q.size(2);
  const int Hk = k.size(1);
  TORCH_CHECK((D / 2) % 4 == 0, "head_dim/2 must be a multiple of 4");
  auto stream = at::hip::getCurrentHIPStream();
  rope_kernel<<<dim3(N), dim3(256), 0, stream>>>(
      (bf16_t*)q.data_ptr(), (bf16_t*)k.data_ptr(),
      positions.data_ptr<int>(), cos_tab.data_ptr<float>(),
      sin_tab.data_ptr<float>(), Hq, Hk, D, q.stride(0), k.stride(0));
  HIP_CHECK_KERNEL();
}

// ------------------------------------------------------ RoPE + KV cache rows
// rope_kernel on q and k, and the token's rotated k and its v into their page
// slot, in one launch: a prompt or decode step's k row is read and turned once
// and goes to both places from registers (two launches read it twice).
// Measured, 5700 tokens, 16/4 heads of 64: 7.1 + 5.0 us, 8.4 us.
__global__ void rope_kv_append_kernel(
    bf16_t* __restrict__ q, bf16_t* __restrict__ k,
    const bf16_t* __restrict__ v, const int* __restrict__ positions,
    const float* __restrict__ cos_tab, const float* __restrict__ sin_tab,
    bf16_t* __restrict__ k_cache, bf16_t* __restrict__ v_cache,
    const int* __restrict__ slot_mapping, int Hq, int Hk, int D, long ldq,
    long ldk, long ldv /* token strides */) {
  const long tok = blockIdx.x;
  const int half = D / 2, quads = half / 4;
  const float* c = cos_tab + (long)positions[tok] * half;
  const float* s = sin_tab + (long)positions[tok] * half;
  const long slot = slot_mapping[tok];   // < 0: a padding token
  bf16_t* kc = k_cache + slot * Hk * D;
  bf16_t* vc = v_cache + slot * Hk * D;
  const int nrope = (Hq + Hk) * quads;
  for (int t = threadIdx.x; t < nrope + Hk * D / 8; t += blockDim.x) {
    if (t >= nrope) {
      const int at = (t - nrope) * 8;
      if (slot >= 0)
        *reinterpret_cast<bf16x8*>(vc + at) =
            *reinterpret_cast<const bf16x8*>(v + tok * ldv + at);
      continue;
    }
    const int h = t / quads;
    const int d = (t % quads) * 4;
    bf16_t* base = h < Hq ? q + tok * ldq + (long)h * D
                          : k + tok * ldk + (long)(h - Hq) * D;
    const bf16x4 x1 = *reinterpret_cast<bf16x4*>(base + d);
    const bf16x4 x2 = *reinterpret_cast<bf16x4*>(base + half + d);
    const f32x4v cv = *reinterpret_cast<const f32x4v*>(c + d);
    const f32x4v sv = *reinterpret_cast<const f32x4v*>(s + d);
    bf16x4 o1, o2;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = bf2f(x1.v[j]), b = bf2f(x2.v[j]);
      // (fused as the compiler fuses rope_kernel's: the same bits)
      o1.v[j] = f2bf(__fmaf_rn(a, cv.v[j], -(b * sv.v[j])));
      o2.v[j] = f2bf(__fmaf_rn(a, sv.v[j], b * cv.v[j]));
    }
    *reinterpret_cast<bf16x4*>(base + d) = o1;
    *reinterpret_cast<bf16x4*>(base + half + d) = o2;
    if (h >= Hq && slot >= 0) {
      bf16_t* to = kc + (h - Hq) * D + d;
      *reinterpret_cast<bf16x4*>(to) = o1;
      *reinterpret_cast<bf16x4*>(to + half) = o2;
    }
  }
}

void rope_kv_append(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                    torch::Tensor positions, torch::Tensor cos_tab,
                    torch::Tensor sin_tab, torch::Tensor k_cache,
                    torch::Tensor v_cache, torch::Tensor slot_mapping) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16 &&
              k.dtype() == torch::kBFloat16 && v.dtype() == torch::kBFloat16);
  TORCH_CHECK(k_cache.is_cuda() && k_cache.dtype() == torch::kBFloat16 &&
              v_cache.dtype() == torch::kBFloat16 &&
              k_cache.is_contiguous() && v_cache.is_contiguous());
  TORCH_CHECK(q.dim() == 3 && k.dim() == 3 && v.dim() == 3);
  for (const auto* t : {&q, &k, &v})
    TORCH_CHECK(t->stride(2) == 1 && t->stride(1) == t->size(2),
                "heads and head dim must be packed");
  TORCH_CHECK(positions.dtype() == torch::kInt32 &&
              slot_mapping.dtype() == torch::kInt32);
  const int N = q.size(0), Hq = q.size(1), D = q.size(2), Hk = k.size(1);
  TORCH_CHECK(D % 8 == 0, "head_dim must be a multiple of 8");
  TORCH_CHECK(k_cache.size(2) == Hk && k_cache.size(3) == D &&
              v.size(1) == Hk && v.size(2) == D);
  if (N == 0) return;
  // a thread per rotary quad and value word, in whole waves
  const int work = (Hq + Hk) * (D / 8) + Hk * D / 8;
  const int threads = std::min(256, (work + 63) / 64 * 64);
  auto stream = at::hip::getCurrentHIPStream();
  rope_kv_append_kernel<<<dim3(N), dim3(threads), 0, stream>>>(
      (bf16_t*)q.data_ptr(), (bf16_t*)k.data_ptr(),
      (const bf16_t*)v.data_ptr(), positions.data_ptr<int>(),
      cos_tab.data_ptr<float>(), sin_tab.data_ptr<float>(),
      (bf16_t*)k_cache.data_ptr(), (bf16_t*)v_cache.data_ptr(),
      slot_mapping.data_ptr<int>(), Hq, Hk, D, q.stride(0), k.stride(0),
      v.stride(0));
  HIP_CHECK_KERNEL();
}
