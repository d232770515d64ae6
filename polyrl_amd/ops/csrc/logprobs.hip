// Fused per-token log-prob gather (+ entropy) over the vocab dim.
//
// Replaces the logprobs_from_logits / entropy_from_logits pair (consumed by
// compute_log_prob and the rollout logprob capture).  One streaming pass:
// online max + sum-exp + weighted-sum for entropy, then lp = x[label] - LZ.
//
// What bounds it: memory.  A thread takes four 16-byte words at a time: their
// largest number first, then one rescale if it beats the running maximum and
// one exponential per number (a compare, a branch and two-byte loads per
// number ran at 1.7 TB/s).  Rows that do not start at a 16-byte address are
// read from the next one, their first numbers apart.  Measured, 4096 x 128256
// bf16: log-probabilities and entropies 600 us with two-byte loads, 183 with
// words, 162 (6.5 TB/s) past the caches; forward and backward 995, 615, 534: dx
// through the caches drove out the rows that the backward had still to read, and
// its blocks of 256 threads read ahead too little (1024: 546 for 551).
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"

typedef __attribute__((ext_vector_type(4))) uint32_t Word16;

// a 16-byte word, ONCE: of what will not be read again while a cache could hold it
template <bool ONCE>
DEV_INLINE Word16 load16(const void* p) {
  const Word16* w = reinterpret_cast<const Word16*>(p);
  return ONCE ? __builtin_nontemporal_load(w) : *w;
}

template <typename T>
DEV_INLINE void unpack16(const Word16& w, float (&v)[16 / sizeof(T)]) {
#pragma unroll
  for (int j = 0; j < (int)(16 / sizeof(T)); ++j)
    v[j] = __uint_as_float(sizeof(T) == 4 ? w[j % 4]
                           : j % 2 ? w[j / 2] & 0xffff0000u
                                   : w[j / 2] << 16);
}

// numbers before a row's first 16-byte address
template <typename T>
DEV_INLINE int lead_of(const T* x, int V) {
  const int n = (int)((16 - ((uintptr_t)x & 15)) & 15) / (int)sizeof(T);
  return n < V ? n : V;
}

// running maximum and sums over numbers relative to it
template <bool ENT>
struct Online {
  float m = -INFINITY, s = 0.f, t = 0.f;
  template <int N>
  DEV_INLINE void add(const float (&v)[N]) {
    float c = v[0];
#pragma unroll
    for (int j = 1; j < N; ++j) c = fmaxf(c, v[j]);
    if (c > m) {
      const float f = __expf(m - c);   // 0 at the first numbers
      s *= f;
      if (ENT) t *= f;
      m = c;
    }
    if (m == -INFINITY) {              // nothing but -inf (and NaN) so far
#pragma unroll
      for (int j = 0; j < N; ++j) s += v[j] != v[j] ? v[j] : 0.f;
      return;
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float e = __expf(v[j] - m);
      s += e;
      if (ENT) t += e * v[j];
    }
  }
};

// one block per row; the last rows first: in training they are the ones that
// the vocabulary product wrote last, and the backward pass starts with the
// ones that are read last here (the 256 MB cache behind the L2s holds a
// quarter of them)
template <typename T, bool ENT, int NT>
__global__ __launch_bounds__(NT) void gather_logprobs_kernel(
    float* __restrict__ out_lp, float* __restrict__ out_lse,
    float* __restrict__ out_ent, const T* __restrict__ logits,
    const int64_t* __restrict__ labels, int V, long kept) {
  constexpr int VEC = 16 / sizeof(T), UN = 4, NW = NT / 64;
  __shared__ float red[NW];
  const long row = gridDim.x - 1 - (long)blockIdx.x;
  const T* x = logits + row * V;
  const int lead = lead_of(x, V);
  const T* xv = x + lead;
  const int nvec = (V - lead) / VEC;
  Online<ENT> a;
  auto words = [&](auto once) {
    constexpr bool ONCE = decltype(once)::value;
    int i = threadIdx.x;
    for (; i + (UN - 1) * NT < nvec; i += UN * NT) {
      Word16 w[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u)
        w[u] = load16<ONCE>(xv + (long)(i + u * NT) * VEC);
      // (else the first word is waited for before the others are on their way:
      // 2000 x 32000 24.7 us for 23.5; past the caches it makes no difference)
      if constexpr (!ONCE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        float v[VEC];
        unpack16<T>(w[u], v);
        a.add(v);
      }
    }
    for (; i < nvec; i += NT) {
      float v[VEC];
      unpack16<T>(load16<ONCE>(xv + (long)i * VEC), v);
      a.add(v);
    }
  };
  if (row >= kept) words(std::true_type());
  else words(std::false_type());
  // the numbers before the first and behind the last whole word
  const int rest = V - lead - nvec * VEC;
  if ((int)threadIdx.x < lead + rest) {
    const int at = (int)threadIdx.x < lead
        ? threadIdx.x : lead + nvec * VEC + threadIdx.x - lead;
    const float v[1] = {(float)x[at]};
    a.add(v);
  }
  const float gm = block_reduce_max<NW>(a.m, red);
  __syncthreads();
  const float f = a.m == -INFINITY ? (a.s == a.s ? 0.f : 1.f)
                                   : __expf(a.m - gm);
  const float gs = block_reduce_sum<NW>(a.s * f, red);
  float gt = 0.f;
  if (ENT) {
    __syncthreads();
    gt = block_reduce_sum<NW>(a.t * f, red);
    // a banned entry (-inf) has no part in the entropy, but gave 0 * inf: such
    // rows are summed again (a check of every number costs all rows 3 to 14%)
    if (gt != gt && gs == gs) {
      float t = 0.f;
      for (int at = threadIdx.x; at < V; at += NT) {
        const float v = (float)x[at];
        if (v != -INFINITY) t += __expf(v - gm) * v;
      }
      __syncthreads();
      gt = block_reduce_sum<NW>(t, red);
    }
  }
  if (threadIdx.x == 0) {
    const float lz = gm + __logf(gs);
    out_lp[row] = (float)x[labels[row]] - lz;
    if (out_lse != nullptr) out_lse[row] = lz;
    if (ENT) out_ent[row] = lz - gt / gs;
  }
}

// ---------------------------------------------------- training backward
// d lp / d logits = onehot(label) - softmax(logits); chain with dlp.
// One streaming pass per row using the forward-saved logsumexp.  Large dx go past
// the caches (DX_ONCE), which keep the rows that the forward read last for as long
// as they are needed; the logits too, where they are more than fits (ONCE).
template <bool ONCE, bool DX_ONCE>
__global__ __launch_bounds__(1024) void gather_logprobs_bwd_kernel(
    bf16_t* __restrict__ dlogits,
    const bf16_t* __restrict__ logits,
    const int64_t* __restrict__ labels,
    const float* __restrict__ lse,
    const float* __restrict__ dlp,
    int V) {
  const long row = blockIdx.x;
  const bf16_t* x = logits + row * V;
  bf16_t* dx = dlogits + row * V;
  const float g = dlp[row];
  const float l = lse[row];
  const long lab = labels[row];
  // 16-byte words of dx from its first 16-byte address on, as in the forward;
  // those of x too, unless the two stand differently (x may be a slice)
  const int lead = lead_of(dx, V);
  const int n8 = (V - lead) / 8;
  const bool same = (((uintptr_t)(x + lead)) & 15) == 0;
  for (int i = threadIdx.x; i < n8; i += blockDim.x) {
    const bf16_t* at = x + lead + (long)i * 8;
    float v[8];
    if (same) {
      unpack16<bf16_t>(load16<ONCE>(at), v);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = bf2f(at[j]);
    }
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o.v[j] = f2bf(-g * __expf(v[j] - l));
    const Word16 w = __builtin_bit_cast(Word16, o);
    Word16* to = reinterpret_cast<Word16*>(dx + lead + (long)i * 8);
    if (DX_ONCE) __builtin_nontemporal_store(w, to);
    else *to = w;
  }
  // the numbers before the first and behind the last whole word
  const int rest = V - lead - n8 * 8;
  if ((int)threadIdx.x < lead + rest) {
    const int i = (int)threadIdx.x < lead ? threadIdx.x
                                          : n8 * 8 + threadIdx.x;
    dx[i] = f2bf(-g * __expf(bf2f(x[i]) - l));
  }
  // add the onehot term after every softmax write landed
  __syncthreads();
  if (threadIdx.x == 0)
    dx[lab] = f2bf(bf2f(dx[lab]) + g);
}

template <typename T, bool ENT>
static void launch_gather(float* lp, float* lse, float* ent,
                          const torch::Tensor& logits,
                          const torch::Tensor& labels, long kept) {
  const long N = logits.size(0);
  if (N == 0) return;
  const int V = logits.size(1);
  auto stream = at::hip::getCurrentHIPStream();
  const T* x = (const T*)logits.data_ptr();
  const int64_t* lab = labels.data_ptr<int64_t>();
  // with too few rows to fill the chip with small blocks a row gets four
  // times the threads
  if (N >= 1024)
    gather_logprobs_kernel<T, ENT, 256>
        <<<dim3(N), dim3(256), 0, stream>>>(lp, lse, ent, x, lab, V, kept);
  else
    gather_logprobs_kernel<T, ENT, 1024>
        <<<dim3(N), dim3(1024), 0, stream>>>(lp, lse, ent, x, lab, V, kept);
  HIP_CHECK_KERNEL();
}

// Rows of logits that the 256 MB cache behind the L2s holds.  The rows that the
// forward reads last stay there for the backward; the others are read past the
// caches.  Measured, 4096 x 128256 forward and backward: with 160 MB kept 542 us,
// 200 535, 240 534, 300 529, none 554.  Where no backward follows, logits that fit
// are read through the caches, which may hold them from the product that wrote
// them (written and read, 1024 x 50257 bf16: 49 us, past the caches 58; 1 x 128256
// fp32, read alone, 10.9 and 14.6), and larger ones past them (1023 x 151936, 310
// MB: 142 us for 150; 4096 x 128256 504 for 562).
static long cached_rows(const torch::Tensor& logits) {
  return (256L << 20) /
         std::max<long>(1, logits.size(1) * (long)logits.element_size());
}

// training fwd: lp + logsumexp (for the hand-written backward)
void gather_logprobs_train_fwd(torch::Tensor out_lp, torch::Tensor out_lse,
                               torch::Tensor logits, torch::Tensor labels) {
  TORCH_CHECK(logits.is_cuda() && logits.dim() == 2 &&
              logits.is_contiguous() &&
              logits.dtype() == torch::kBFloat16);
  TORCH_CHECK(labels.dtype() == torch::kInt64);
  launch_gather<bf16_t, false>(out_lp.data_ptr<float>(),
                               out_lse.data_ptr<float>(), nullptr, logits,
                               labels, cached_rows(logits));
}

torch::Tensor gather_logprobs_train_bwd(torch::Tensor logits,
                                        torch::Tensor labels,
                                        torch::Tensor lse,
                                        torch::Tensor dlp) {
  TORCH_CHECK(logits.is_cuda() && logits.is_contiguous() &&
              logits.dtype() == torch::kBFloat16);
  const long N = logits.size(0);
  const int V = logits.size(1);
  auto dlogits = torch::empty_like(logits);
  auto stream = at::hip::getCurrentHIPStream();
  if (N == 0) return dlogits;
  // dx stays in the caches for its next reader where it fits there beside the
  // logits (4096 x 5000, dx read again: 54 us, past the caches 60; 1000 x 50257 109
  // and 120, but the call alone 54 and 51; 2000 x 32000, 128 MB, 134 and 146, alone
  // 78 and 62; 1000 x 128256, 256 MB, 296 and 273, alone 153 and 126)
  const long rows = cached_rows(logits);
  auto kern = N > rows            ? gather_logprobs_bwd_kernel<true, true>
              : N > rows * 7 / 16 ? gather_logprobs_bwd_kernel<false, true>
                                  : gather_logprobs_bwd_kernel<false, false>;
  // 1024 threads of rows that give each two words or more (of 16384 entries and
  // more: 4096 x 20000 84 us with 1024, 88 with 256; 16000 x 10000 165 and 156,
  // 4096 x 5000 28 and 26, 4096 x 500 16.4 and 11.4, forward and backward)
  const int threads = V < 16384 ? 256 : 1024;
  kern<<<dim3(N), dim3(threads), 0, stream>>>(
      (bf16_t*)dlogits.data_ptr(), (const bf16_t*)logits.data_ptr(),
      labels.data_ptr<int64_t>(), lse.data_ptr<float>(),
      dlp.contiguous().data_ptr<float>(), V);
  HIP_CHECK_KERNEL();
  return dlogits;
}

void gather_logprobs(torch::Tensor out_lp, torch::Tensor out_ent,
                     torch::Tensor logits, torch::Tensor labels,
                     bool want_entropy) {
  TORCH_CHECK(logits.is_cuda() && logits.dim() == 2 && logits.is_contiguous());
  TORCH_CHECK(labels.dtype() == torch::kInt64);
  TORCH_CHECK(out_lp.dtype() == torch::kFloat32);
  float* lp = out_lp.data_ptr<float>();
  float* ent = want_entropy ? out_ent.data_ptr<float>() : nullptr;
  const long kept =
      logits.size(0) <= cached_rows(logits) ? logits.size(0) : 0;
  if (logits.dtype() == torch::kBFloat16) {
    (want_entropy ? launch_gather<bf16_t, true> : launch_gather<bf16_t, false>)(
        lp, nullptr, ent, logits, labels, kept);
  } else if (logits.dtype() == torch::kFloat32) {
    (want_entropy ? launch_gather<float, true> : launch_gather<float, false>)(
        lp, nullptr, ent, logits, labels, kept);
  } else {
    TORCH_CHECK(false, "gather_logprobs: dtype must be bf16 or fp32");
  }
}
