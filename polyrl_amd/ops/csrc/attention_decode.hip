// Paged decode attention (continuous-batching, one new token per sequence).
//
// Reference capability: the paged/continuous-batching decode attention the
// reference reaches through its inference engine.
//
// A block serves one key/value head of one sequence (or a stretch of its
// context) for all G query heads of the group; each of its four waves takes
// 32 keys at a time, on its own: no barrier until the waves' results meet.
//   * S^T = K Q^T on v_mfma_f32_16x16x32_bf16, 16 keys x 16 head columns (G of
//     them in use): a lane's K fragment is 16 bytes of one cached row, loaded
//     straight from the page, and its accumulators are keys of ONE head, so
//     maximum and sum take two lane exchanges per 32 keys.
//   * O^T += V^T P^T: V rows go through 8 KiB of LDS of the wave's own and come
//     back turned (ds_read_b64_tr_b16); the weights are the operand as they
//     stand in the accumulators.  They stay the 32-bit numbers they are: each
//     is the sum of three bf16 numbers, and all three are multiplied.
// What bounds it: reading K and V once.  (With per-key dot products, shuffles
// and exponentials on the vector units the kernel was bound by those: 1.4 TB/s
// at seven heads a group, 4.1 at four.)  Measured: 128 rows of 257 .. 512
// tokens, 32/8 heads of 128, 59.5 -> 45.2 us, with V read past the caches 41 (5.1
// TB/s; on inputs that no cache holds 43.9 and 41.2); 33 rows of 1900 .. 8192, 28/4
// heads, 264 -> 86.5 -> 82 us, 77 in ten stretches.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "attention_tile.h"

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int DEC_KEYS = 32;          // keys of a wave's round
constexpr int DEC_HEADS = 8;          // most query heads of a group

// the larger / the sum of the four lanes l, l+16, l+32, l+48
DEV_INLINE float quad_max(float x) {
  const auto p = __builtin_amdgcn_permlane16_swap(
      __float_as_uint(x), __float_as_uint(x), false, false);
  return half_max(fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1])));
}
DEV_INLINE float quad_sum(float x) {
  const auto p = __builtin_amdgcn_permlane16_swap(
      __float_as_uint(x), __float_as_uint(x), false, false);
  return half_sum(__uint_as_float(p[0]) + __uint_as_float(p[1]));
}

// WAVES: of a SIMD, at least; ONCE: values are read past the caches
template <int D, int WAVES, bool ONCE>
__global__ __launch_bounds__(256, WAVES) void paged_decode_attn_kernel(
    bf16_t* __restrict__ out,              // (B, Hq, D)
    float* __restrict__ partial,           // (B, Hq, S, D+2) when nsplit>1
    const bf16_t* __restrict__ q,          // (B, Hq, D)
    const bf16_t* __restrict__ k_cache,    // (num_pages, page_size, Hk, D)
    const bf16_t* __restrict__ v_cache,
    const int* __restrict__ page_table,    // (B, max_pages)
    const int* __restrict__ context_lens,  // (B,)
    int Hq, int Hk, int page_size, int max_pages, float scale, long ldq,
    int nsplit) {
  typedef AttnTile<D> T;
  constexpr int KS = D / 32, DT = D / 16;
  constexpr int RPI = 64 / T::GR;          // V rows of one load instruction
  constexpr int NV = DEC_KEYS / RPI;
  __shared__ __attribute__((aligned(16))) char lds[4][DEC_KEYS * D * 2];
  __shared__ float ml[4][DEC_HEADS][2];

  const int b = blockIdx.x / (Hk * nsplit);
  const int rem = blockIdx.x % (Hk * nsplit);
  const int hk = rem / nsplit;
  const int sp = rem % nsplit;
  const int G = Hq / Hk;
  const int L = context_lens[b];
  // a stretch per block, in whole rounds of a wave
  const int Lc = ((L + nsplit - 1) / nsplit + DEC_KEYS - 1) / DEC_KEYS *
                 DEC_KEYS;
  const int cbeg = sp * Lc;
  const int cend = min(cbeg + Lc, L);
  const int lane = threadIdx.x & 63;
  const int wid = wave_id();
  const int l15 = lane & 15, lhi = lane >> 4;

  // Q of head l15 (columns past the group repeat its last head)
  bf16x8_t qf[KS];
  {
    const bf16_t* qp = q + (long)b * ldq +
                       (long)(hk * G + min(l15, G - 1)) * D + lhi * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = *reinterpret_cast<const bf16x8_t*>(qp + ks * 32);
  }
  const float s2 = scale * 1.4426950408889634f;
  // m starts at a large negative FINITE value: an empty stretch then weighs
  // 2^(m - largest) = 0 in the merges instead of inf - inf
  float m_run = -1e30f, l_run = 0.f;
  f32x4_t o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = {0.f, 0.f, 0.f, 0.f};

  const long kv_stride = (long)Hk * D;
  const int* ptab = page_table + (long)b * max_pages;
  char* vs = lds[wid];
  // turned reads of V: rows 4 * lhi + l15 / 4 (+16), columns 16 dt + ..
  const int ra = 4 * lhi + (l15 >> 2), rb = ra + 16;
  const int vg = (l15 & 3) >> 1;
  const int va = ra * (2 * D) + ((vg ^ T::swz(ra)) << 4) + (l15 & 1) * 8;
  const int vb = rb * (2 * D) + ((vg ^ T::swz(rb)) << 4) + (l15 & 1) * 8;
  const int vrow = lane / T::GR, vcol = lane % T::GR;

  // cache row of key t0 + lane % 32 (keys past the stretch: its last)
  auto slot_of = [&](int t0) {
    const int t = min(t0 + (lane & 31), cend - 1);
    const int pg = t / page_size;
    return ptab[pg] * page_size + (t - pg * page_size);
  };
  int t0 = cbeg + wid * DEC_KEYS;
  int slot = t0 < cend ? slot_of(t0) : 0;
  for (; t0 < cend; t0 += 4 * DEC_KEYS) {
    bf16x8_t kf[2][KS];
    i32x4_t vv[NV];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const bf16_t* kp = k_cache + __shfl(slot, n * 16 + l15, 64) * kv_stride +
                         hk * D + lhi * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kf[n][ks] = *reinterpret_cast<const bf16x8_t*>(kp + ks * 32);
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const i32x4_t* vp = reinterpret_cast<const i32x4_t*>(
          v_cache + __shfl(slot, i * RPI + vrow, 64) * kv_stride + hk * D +
          vcol * 8);
      vv[i] = ONCE ? __builtin_nontemporal_load(vp) : *vp;
    }
    if (t0 + 4 * DEC_KEYS < cend) slot = slot_of(t0 + 4 * DEC_KEYS);

    // ---- S^T: 32 keys x 16 heads; this lane: head l15, keys 4 lhi + r -------
    f32x4_t s[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      s[n] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        s[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[n][ks], qf[ks], s[n],
                                                       0, 0, 0);
    }
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[n][r] *= s2;
    if (t0 + DEC_KEYS > cend) {
      const int last = cend - 1 - t0;
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n * 16 + 4 * lhi + r > last) s[n][r] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[n][r]);
    const float mn = fmaxf(m_run, quad_max(mx));
    const float alpha = exp2_hw(m_run - mn);
    m_run = mn;
    l_run *= alpha;
    // weights as the sum of three bf16 numbers, the 24 bits of a 32-bit one in
    // groups of eight.  None is 0 unless the weight is (the smallest bf16
    // number stands in), so that an infinite value stays infinite.
    i16x8_t w3[3];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = exp2_hw(s[n][r] - mn);
        l_run += p;
        float rest = p;
        unsigned least = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const unsigned bits = __float_as_uint(rest);
          w3[i][4 * n + r] = (short)max(bits >> 16, least);
          if (i == 0) least = min(bits, 1u);
          rest -= __uint_as_float(bits & 0xFFFF0000u);
        }
      }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[dt][r] *= alpha;

    // ---- V rows into the wave's LDS, turned fragments back --------------------
    // (zeros past the stretch: its last row, which stands in, need not be
    // finite, and 0 * inf is NaN)
    if (t0 + DEC_KEYS > cend) {
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if (t0 + i * RPI + vrow >= cend) vv[i] = {0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int r = i * RPI + vrow;
      *reinterpret_cast<i32x4_t*>(vs + r * (2 * D) +
                                  ((vcol ^ T::swz(r)) << 4)) = vv[i];
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const i16x4_t a = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_i16x4_p)(vs + (va ^ (dt << 5))));
      const i16x4_t c = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_i16x4_p)(vs + (vb ^ (dt << 5))));
      const bf16x8_t vt = __builtin_bit_cast(
          bf16x8_t, __builtin_shufflevector(a, c, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
      for (int i = 0; i < 3; ++i)
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            vt, __builtin_bit_cast(bf16x8_t, w3[i]), o[dt], 0, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  }
  l_run = quad_sum(l_run);

  // ---- the four waves' shares meet in LDS ------------------------------------
  if (l15 < G) {
    float* mine = reinterpret_cast<float*>(vs) + l15 * D + lhi * 4;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      *reinterpret_cast<f32x4_t*>(mine + dt * 16) = o[dt];
    if (lhi == 0) {
      ml[wid][l15][0] = m_run;
      ml[wid][l15][1] = l_run;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < G * D; i += 256) {
    const int h = i / D, d = i % D;
    float gm = ml[0][h][0];
#pragma unroll
    for (int w = 1; w < 4; ++w) gm = fmaxf(gm, ml[w][h][0]);
    float l = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float a = exp2_hw(ml[w][h][0] - gm);
      l += ml[w][h][1] * a;
      acc += reinterpret_cast<const float*>(lds[w])[i] * a;
    }
    const long row = (long)b * Hq + hk * G + h;
    if (nsplit == 1) {
      out[row * D + d] = f2bf(l > 0.f ? acc / l : 0.f);
    } else {
      float* pp = partial + (row * nsplit + sp) * (D + 2);
      pp[d] = acc;
      if (d == 0) {
        pp[D] = gm * 0.6931471805599453f;
        pp[D + 1] = l;
      }
    }
  }
}

// One query head per key/value head, many blocks or short contexts: matrix
// products use one column in sixteen, and with two or three of their blocks
// resident on a CU a short context is all latency.  Here a wave streams keys
// with D / 8 lanes each, and dot products and softmax run on the vector units
// in 32 bits: 53 registers, eight blocks to a CU.  Bound by latency, from a few
// hundred keys on by memory.  Measured, 300 rows of 32 heads of 128: 5 keys 14.4
// us (51 on the matrix cores), 100 keys 90 (100), 500 keys 432 (421).
template <int D>
__global__ __launch_bounds__(256) void paged_decode_attn_one_kernel(
    bf16_t* __restrict__ out,              // (B, H, D)
    float* __restrict__ partial,           // (B, H, S, D+2) when nsplit>1
    const bf16_t* __restrict__ q,          // (B, H, D)
    const bf16_t* __restrict__ k_cache,    // (num_pages, page_size, H, D)
    const bf16_t* __restrict__ v_cache,
    const int* __restrict__ page_table,    // (B, max_pages)
    const int* __restrict__ context_lens,  // (B,)
    int H, int /* Hk */, int page_size, int max_pages, float scale, long ldq,
    int nsplit) {
  constexpr int GL = D / 8;                // lanes of a key
  constexpr int KPW = 64 / GL;             // keys of a wave's round
  __shared__ float mrg[4][GL][10];         // per wave: o, m, l

  const int b = blockIdx.x / (H * nsplit);
  const int rem = blockIdx.x % (H * nsplit);
  const int h = rem / nsplit;
  const int sp = rem % nsplit;
  const int L = context_lens[b];
  const int Lc = (L + nsplit - 1) / nsplit;
  const int cbeg = sp * Lc;
  const int cend = min(cbeg + Lc, L);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int grp = lane / GL, gl = lane % GL;
  const int d0 = gl * 8;                   // this lane's numbers of a row

  float qr[8];
  {
    const bf16x8 qv = *reinterpret_cast<const bf16x8*>(
        q + (long)b * ldq + (long)h * D + d0);
#pragma unroll
    for (int j = 0; j < 8; ++j) qr[j] = bf2f(qv.v[j]) * scale;
  }
  // (m starts finite, as above)
  float m = -1e30f, l = 0.f, o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = 0.f;

  const long row = (long)H * D;
  const int* ptab = page_table + (long)b * max_pages;
  for (int t0 = cbeg + wid * KPW + grp; t0 < cend; t0 += 4 * KPW) {
    const long slot =
        (long)ptab[t0 / page_size] * page_size + t0 % page_size;
    const bf16x8 kv = *reinterpret_cast<const bf16x8*>(
        k_cache + slot * row + h * D + d0);
    const bf16x8 vv = *reinterpret_cast<const bf16x8*>(
        v_cache + slot * row + h * D + d0);
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) s += qr[j] * bf2f(kv.v[j]);
#pragma unroll
    for (int off = GL / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    const float mn = fmaxf(m, s);
    const float alpha = __expf(m - mn), p = __expf(s - mn);
    l = l * alpha + p;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = o[j] * alpha + p * bf2f(vv.v[j]);
    m = mn;
  }

  // the wave's key groups meet
#pragma unroll
  for (int off = GL; off < 64; off <<= 1) {
    const float om = __shfl_xor(m, off, 64), ol = __shfl_xor(l, off, 64);
    const float mn = fmaxf(m, om);
    const float a = __expf(m - mn), c = __expf(om - mn);
    l = l * a + ol * c;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = o[j] * a + __shfl_xor(o[j], off, 64) * c;
    m = mn;
  }
  // and the four waves
  if (grp == 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) mrg[wid][gl][j] = o[j];
    mrg[wid][gl][8] = m;
    mrg[wid][gl][9] = l;
  }
  __syncthreads();
  if (wid != 0 || grp != 0) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) m = fmaxf(m, mrg[w][gl][8]);
  l = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float a = __expf(mrg[w][gl][8] - m);
    l += mrg[w][gl][9] * a;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] += mrg[w][gl][j] * a;
  }
  const long at = (long)b * H + h;
  if (nsplit == 1) {
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    bf16x8 w;
#pragma unroll
    for (int j = 0; j < 8; ++j) w.v[j] = f2bf(o[j] * inv);
    *reinterpret_cast<bf16x8*>(out + at * D + d0) = w;
  } else {
    float* pp = partial + (at * nsplit + sp) * (D + 2);
#pragma unroll
    for (int j = 0; j < 8; ++j) pp[d0 + j] = o[j];
    if (gl == 0) {
      pp[D] = m;
      pp[D + 1] = l;
    }
  }
}

// combine the nsplit context partials of one (b, hq): sum-exp merge
template <int D>
__global__ void paged_decode_merge_kernel(
    bf16_t* __restrict__ out,              // (B, Hq, D)
    const float* __restrict__ partial,     // (B*Hq, S, D+2)
    int nsplit) {
  constexpr int EPL = D / 64;              // d-elems per lane (64 threads)
  const long row = blockIdx.x;             // b*Hq + hq
  const int lane = threadIdx.x;
  const float* base = partial + row * (long)nsplit * (D + 2);
  // stretch lane: its maximum and sum (nsplit <= 64)
  const float m = lane < nsplit ? base[lane * (D + 2) + D] : -1e30f;
  const float w = __expf(m - wave_reduce_max(m));
  const float gl_sum = wave_reduce_sum(
      lane < nsplit ? base[lane * (D + 2) + D + 1] * w : 0.f);
  float acc[EPL];
#pragma unroll
  for (int j = 0; j < EPL; ++j) acc[j] = 0.f;
  for (int sp = 0; sp < nsplit; ++sp) {
    const float* pp = base + sp * (D + 2);
    const float a = __shfl(w, sp, 64);
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      acc[j] += pp[lane + j * 64] * a;
  }
  const float inv = (gl_sum > 0.f) ? 1.0f / gl_sum : 0.f;
#pragma unroll
  for (int j = 0; j < EPL; ++j)
    out[row * D + lane + j * 64] = f2bf(acc[j] * inv);
}

template <int D>
static void dispatch_g(torch::Tensor& out, const torch::Tensor& q,
                       const torch::Tensor& k_cache, const torch::Tensor& v_cache,
                       const torch::Tensor& page_table,
                       const torch::Tensor& context_lens, int Hq, int Hk,
                       int page_size, int max_pages, float scale,
                       hipStream_t stream) {
  const int G = Hq / Hk;
  const long B = q.size(0);
  // Context split: from the sizes alone, not from the lengths on the device,
  // so that a captured graph may replay it with longer contexts.  No stretch
  // under 128 keys (a round of the four waves) of the longest context that the
  // page table holds: there the merging launch costs more than the split gains
  // (37 cached tokens: 16.8 us in 16 stretches, 6.8 in one).
  //
  // Contexts of up to 1024: up to 512 blocks (two per CU), more cost more in the
  // merging launch than they give (64 of 12/2 heads of 128 19.0 us in eight, 15.6
  // in four; 16 of 64/8 heads 20.3 in eight, 17.0 in four; 64 of 32/8 heads of 64,
  // 500 .. 1000, 22.6 in two, 19.8 in one; 56 of 128 35.5, 36.5, 35.9, 38.0 in one to
  // four).  Where less than half of the CUs have a second block the others wait for
  // it: in three (33 rows of 500 .. 1000, 32/8 heads of 128, in one to four 30.4,
  // 28.0, 26.7, 27.8; of 257 .. 1024 tokens and heads of 64 19.8, 19.5, 16.9, 17.8;
  // of 300 .. 600 tokens 17.5, 18.9, 18.8, 19.6; 50 of 500 .. 1000 33.4, 34.8, 33.0,
  // 35.7, of 450 .. 900 29.9, 32.2, 31.2, 33.4).
  //
  // Longer ones: 1024 blocks (25 rows of 1024 .. 2048, 32/8 heads of 128, in 5, 6,
  // 8 and 10: 39.3, 41.4, 43.9, 44.3; 50 in 2, 3, 4 and 5: 67.9, 65.4, 69.1, 65.9;
  // inputs of several layers in turn), but five stretches where four are 1024 to
  // 1364 (33 rows of 2049 .. 8192 in 4, 5 and 6: 137, 130, 129; of 1024 .. 2048 53.1,
  // 52.5, 53.1), and ten of the longest where seven or eight are 1024 to 1272
  // (33 rows of 1900 .. 8192, 28/4 heads, in 8, 9, 10, 11 and 15: 82, 76, 76, 76, 78).
  const long base_blocks = B * Hk;
  const long most = (long)max_pages * page_size;
  int nsplit = 1;
  if (base_blocks < 1024) {
    const long want =
        most <= 1024 ? (most > 700 && base_blocks > 256 && base_blocks < 384
                            ? 3 : 512 / base_blocks)
        : base_blocks >= 256 && base_blocks <= 341 ? 5
        : most > 4096 && base_blocks >= 128 && base_blocks < 160
            ? 10 : (1024 + base_blocks - 1) / base_blocks;
    nsplit = (int)std::max<long>(
        1, std::min<long>({want, 16, (most + 127) / 128}));
  }
  torch::Tensor ws;                     // per call: any stream, any capture
  float* ppart = nullptr;
  if (nsplit > 1) {
    ws = torch::empty({B * Hq * (long)nsplit * (D + 2)},
                      q.options().dtype(torch::kFloat32));
    ppart = ws.data_ptr<float>();
  }
  const dim3 grid(B * Hk * nsplit), block(256);
  auto args = [&](auto kern) {
    kern<<<grid, block, 0, stream>>>(
        (bf16_t*)out.data_ptr(), ppart, (const bf16_t*)q.data_ptr(),
        (const bf16_t*)k_cache.data_ptr(), (const bf16_t*)v_cache.data_ptr(),
        page_table.data_ptr<int>(), context_lens.data_ptr<int>(), Hq, Hk,
        page_size, max_pages, scale, q.stride(0), nsplit);
    if (nsplit > 1)
      paged_decode_merge_kernel<D><<<dim3(B * Hq), dim3(64), 0, stream>>>(
          (bf16_t*)out.data_ptr(), ppart, nsplit);
  };
  TORCH_CHECK(G >= 1 && G <= DEC_HEADS, "GQA group size ", G,
              " unsupported (1..8)");
  // One head a group: the vector kernel from four rounds of the matrix kernel's
  // blocks on (heads of 128: 64 rows of 32 heads, 40 keys 9.7 us and 12.4, 300
  // keys 52 and 55; 32 rows 300 keys 26.4 both, 3000 keys 306 and 278; heads
  // of 64: 300 rows of 16, 40 keys 12.8 and 15.0, 300 keys 75.7 and 72.4, 128
  // rows 1000 keys 97.7 and 103), and where the page table holds short contexts
  // only (128 wide, 4 heads, 128 rows of 300 keys: 18.2 and 20.0).
  // Values go past the caches, read once in whole rows: that leaves the ways of the
  // 256 MB cache behind the L2s to K, whose lines two instructions read (K past the
  // caches too 45.9 us where V alone gave 37.6).  On inputs that no cache holds, as
  // the layers of a model come in turn, it takes 3 to 8% less time at every size
  // (128 rows of 257 .. 512, 32/8 heads of 128, 43.9 -> 41.2; 56 of 1024 .. 2048,
  // 77.6 -> 72.3).  Small calls keep V in the caches for those who repeat them on
  // the same tensors: up to 10% slower past them with two of up to 128 MiB in turn
  // (128 to 192 MiB: 11% slower to 2% faster; 256 MiB: 10 to 17% faster).
  const bool once = B * most * Hk * D * 4 > (128L << 20);
  // Groups of two and three heads of 128 keep three blocks on a CU, which short
  // contexts need (300 rows of 16 groups of two, 5 keys: 28 us with two, 19.7
  // with three); at larger groups the registers that this takes cost more (32
  // rows of 8000 keys, 28/4 heads: 106 and 110 us).
  if (G == 1 && (base_blocks >= 2048 || most <= (D == 128 ? 512 : 64)))
    args(paged_decode_attn_one_kernel<D>);
  else if (D == 128 && G <= 3)
    once ? args(paged_decode_attn_kernel<D, 3, true>)
         : args(paged_decode_attn_kernel<D, 3, false>);
  else
    once ? args(paged_decode_attn_kernel<D, 1, true>)
         : args(paged_decode_attn_kernel<D, 1, false>);
}

void paged_attention_decode(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor page_table,
                            torch::Tensor context_lens, double scale) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16);
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == q.size(2),
              "q heads/dims must be packed (token stride free)");
  TORCH_CHECK(page_table.dtype() == torch::kInt32 && page_table.is_contiguous());
  TORCH_CHECK(context_lens.dtype() == torch::kInt32);
  const int Hq = q.size(1), D = q.size(2);
  const int Hk = k_cache.size(2);
  const int page_size = k_cache.size(1);
  const int max_pages = page_table.size(1);
  TORCH_CHECK(Hq % Hk == 0);
  auto stream = at::hip::getCurrentHIPStream();
  if (D == 128) {
    dispatch_g<128>(out, q, k_cache, v_cache, page_table, context_lens, Hq,
                    Hk, page_size, max_pages, (float)scale, stream);
  } else if (D == 64) {
    dispatch_g<64>(out, q, k_cache, v_cache, page_table, context_lens, Hq, Hk,
                   page_size, max_pages, (float)scale, stream);
  } else {
    TORCH_CHECK(false, "head_dim ", D, " unsupported (64 or 128)");
  }
  HIP_CHECK_KERNEL();
}
