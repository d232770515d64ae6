// Paged decode attention (continuous-batching, one new token per sequence).
//
// Reference capability: the paged/continuous-batching decode attention the
// reference reaches through its inference engine.
//
// A block serves one key/value head of one sequence (or a stretch of its
// context) for all G query heads of the group; each of its four waves takes
// 32 keys at a time, on its own: no barrier until the waves' results meet.
//   * S^T = K Q^T on v_mfma_f32_16x16x32_bf16, 16 keys x 16 columns: a lane's
//     accumulators are keys of ONE head, so maximum and sum take two lane
//     exchanges per 32 keys.  Large calls read K in whole rows past the caches and
//     take the fragments from LDS; small ones, which the caches may hold, load
//     them straight from the page, 64 bytes of a row at a time.
//   * O^T += V^T P^T: V rows go through 8 KiB of LDS of the wave's own and come
//     back turned (ds_read_b64_tr_b16); the weights are the operand as they
//     stand in the accumulators.  They stay the 32-bit numbers they are: each
//     is the sum of three bf16 numbers, and all three are multiplied, in columns
//     that the heads leave free: one product for up to four heads, two for eight.
// What bounds it: reading K and V once, at the rate that this order of pages and
// heads reaches (the same loads alone, 128 rows of 257 .. 512 tokens, 32/8 heads of
// 128: 35.7 us; 33 rows of 1900 .. 8192, 28/4: 59).  Loads of the next round ahead of
// this one's products, and three blocks of large calls on a CU, change nothing
// (38.2 and 68.0 us with, 38.6 and 68.4 without; both together 38.0 and 76).
// Measured (inputs of three layers in turn): those 128 rows 41.2 us with K in 64-byte
// pieces through the caches, 38.0 now (5.3 TB/s); those 33 rows 77.1, 68.0, of which
// the merge's loads one after the other were 2.5.  (With per-key dot products,
// shuffles and exponentials on the vector units it was bound by those: 1.4 TB/s at
// seven heads a group, 4.1 at four.)
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "attention_tile.h"

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int DEC_KEYS = 32;          // keys of a wave's round
constexpr int DEC_HEADS = 8;          // most query heads of a group
constexpr int DEC_SPLITS = 16;        // most stretches of a row

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

// FEW: four heads or less; ONCE: keys and values are read past the caches
template <int D, bool FEW, bool ONCE>
__global__ __launch_bounds__(256, ONCE ? 2 : 3) void paged_decode_attn_kernel(
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
  constexpr int RPI = 64 / T::GR;          // cache rows of one load instruction
  constexpr int NV = DEC_KEYS / RPI;
  constexpr int HC = FEW ? 4 : DEC_HEADS;  // columns of a part of the weights
  // a wave's values, and at the end its sums; its keys
  __shared__ __attribute__((aligned(16))) char lds[4][DEC_KEYS * D * 2],
      keys[ONCE ? 4 : 1][ONCE ? DEC_KEYS * D * 2 : 16];
  __shared__ float ml[4][DEC_HEADS][2];

  int rem, sp, none;
  const int b = split_id(blockIdx.x, Hk * nsplit, rem);
  const int hk = split_id(rem, nsplit, sp);
  const int G = split_id(Hq, Hk, none);
  const int lane = threadIdx.x & 63;
  const int wid = wave_id();
  const int l15 = lane & 15, lhi = lane >> 4;
  const int vrow = lane / T::GR, vcol = lane % T::GR;

  // Cache rows of keys t0 + lane % 32.  The table of a row that is not divided is
  // read before its length is known; an entry past the stretch may be anything, and
  // the round's first key stands in for it.
  const int* ptab = page_table + (long)b * max_pages;
  const bool pow2 = (page_size & (page_size - 1)) == 0;
  const int shift = 31 - __builtin_clz(page_size);
  auto look_up = [&](int t0) {
    const int t = t0 + (lane & 31);
    return ptab[min(pow2 ? t >> shift : t / page_size, max_pages - 1)];
  };
  int page = 0;
  if (nsplit == 1 && max_pages > 0) page = look_up(wid * DEC_KEYS);
  const int L = max(context_lens[b], 0);
  // a stretch per block, in whole rounds of a wave
  const int Lc = nsplit == 1 ? L : ((L + nsplit - 1) / nsplit + DEC_KEYS - 1) /
                                       DEC_KEYS * DEC_KEYS;
  const int cbeg = sp * Lc;
  const int cend = min(cbeg + Lc, L);
  auto rows_of = [&](int page, int t0) {
    const int t = t0 + (lane & 31);
    const int slot =
        page * page_size + (pow2 ? t & (page_size - 1) : t % page_size);
    // (outside the choice: in it the first lane would be one past the stretch)
    const int first = uniform(slot);
    return t < cend ? slot : first;
  };
  int t0 = cbeg + wid * DEC_KEYS;
  if (nsplit > 1 && max_pages > 0) page = look_up(t0);

  // Q of this column's head (columns past the group repeat its last head)
  bf16x8_t qf[KS];
  {
    const bf16_t* qp = q + (long)b * ldq +
                       (long)(hk * G + min(l15 % HC, G - 1)) * D + lhi * 8;
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

  const unsigned row_bytes = (unsigned)(Hk * D) * 2;
  char* vs = lds[wid];
  char* kt = keys[ONCE ? wid : 0];
  // turned reads of V: rows 4 * lhi + l15 / 4 (+16), columns 16 dt + ..
  const int ra = 4 * lhi + (l15 >> 2), rb = ra + 16;
  const int vg = (l15 & 3) >> 1;
  int va = ra * (2 * D) + ((vg ^ T::swz(ra)) << 4) + (l15 & 1) * 8;
  int vb = rb * (2 * D) + ((vg ^ T::swz(rb)) << 4) + (l15 & 1) * 8;
  // rows of K: l15 (+16), numbers 32 ks + 8 lhi ..
  int ka = l15 * (2 * D) + ((lhi ^ T::swz(l15)) << 4);
  // whole rows to their places
  int to = vrow * (2 * D) + ((vcol ^ T::swz(vrow)) << 4);

  // the round's rows into registers, and from there to the wave's LDS
  auto load_rows = [&](i32x4_t (&w)[NV], const bf16_t* cache, int slot) {
    const char* base =
        reinterpret_cast<const char*>(cache + hk * D + vcol * 8);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const i32x4_t* p = reinterpret_cast<const i32x4_t*>(
          base + (uint64_t)(unsigned)__shfl(slot, i * RPI + vrow, 64) *
                     row_bytes);
      w[i] = ONCE ? __builtin_nontemporal_load(p) : *p;
    }
  };
  auto store_rows = [&](char* tile, const i32x4_t (&w)[NV]) {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      *reinterpret_cast<i32x4_t*>(tile + i * RPI * (2 * D) +
                                  (to ^ (T::swz(i * RPI) << 4))) = w[i];
    __builtin_amdgcn_wave_barrier();
  };

  for (; t0 < cend; t0 += 4 * DEC_KEYS) {
    // (new to the compiler: else the addresses derived from them live in
    // registers through the loop)
    asm volatile("" : "+v"(to), "+v"(ka), "+v"(va), "+v"(vb));
    const int slot = rows_of(page, t0);
    bf16x8_t kf[2][KS];
    i32x4_t kk[NV], vv[NV];
    if constexpr (ONCE) {
      load_rows(kk, k_cache, slot);
    } else {
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const char* kp =
            reinterpret_cast<const char*>(k_cache + hk * D + lhi * 8) +
            (uint64_t)(unsigned)__shfl(slot, n * 16 + l15, 64) * row_bytes;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          kf[n][ks] = *reinterpret_cast<const bf16x8_t*>(kp + ks * 64);
      }
    }
    load_rows(vv, v_cache, slot);
    if (t0 + 4 * DEC_KEYS < cend) page = look_up(t0 + 4 * DEC_KEYS);
    if constexpr (ONCE) {
      __builtin_amdgcn_sched_barrier(0);
      store_rows(kt, kk);
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          kf[n][ks] = *reinterpret_cast<const bf16x8_t*>(
              kt + n * 16 * (2 * D) + (ka ^ (ks << 6)));
    }

    // ---- S^T: 32 keys x 16 columns; this lane: column l15, keys 4 lhi + r ----
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
    if (__any(mn > m_run)) {
      const float alpha = exp2_hw(m_run - mn);
      m_run = mn;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[dt][r] *= alpha;
    }
    // Weights as the sum of three bf16 numbers, the 24 bits of a 32-bit one in
    // groups of eight.  None is 0 unless the weight is (the smallest bf16
    // number stands in), so that an infinite value stays infinite.  The columns
    // past the heads take the second and third part of the same heads; of eight
    // heads the third part and, beside it, that smallest number make a second
    // product.
    i16x8_t w3[FEW ? 1 : 2];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = exp2_hw(s[n][r] - m_run);
        l_run += p;
        const unsigned b0 = __float_as_uint(p);
        const float r1 = p - __uint_as_float(b0 & 0xFFFF0000u);
        const unsigned b1 = __float_as_uint(r1);
        const float r2 = r1 - __uint_as_float(b1 & 0xFFFF0000u);
        const unsigned b2 = __float_as_uint(r2);
        const unsigned least = min(b0, 1u);
        if constexpr (FEW) {
          const unsigned w = l15 < 4 ? b0 : l15 < 8 ? b1 : b2;
          w3[0][4 * n + r] = (short)max(w >> 16, least);
        } else {
          w3[0][4 * n + r] = (short)max((l15 < 8 ? b0 : b1) >> 16, least);
          w3[1][4 * n + r] =
              (short)(l15 < 8 ? max(b2 >> 16, least) : least);
        }
      }

    // ---- V rows into the wave's LDS, turned fragments back --------------------
    // (zeros past the stretch: the row that stands in need not be finite, and
    // 0 * inf is NaN)
    if (t0 + DEC_KEYS > cend) {
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if (t0 + i * RPI + vrow >= cend) vv[i] = {0, 0, 0, 0};
    }
    store_rows(vs, vv);
    bf16x8_t vt[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const i16x4_t a = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_i16x4_p)(vs + (va ^ (dt << 5))));
      const i16x4_t c = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_i16x4_p)(vs + (vb ^ (dt << 5))));
      vt[dt] = __builtin_bit_cast(
          bf16x8_t, __builtin_shufflevector(a, c, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    // (small calls, whose rounds are a chain of waits: all reads on their way before
    // the first product; 256 rows of 100 .. 300, 12/2 heads of 128, 14.1 -> 13.9 us)
    if constexpr (!ONCE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < (FEW ? 1 : 2); ++i)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            vt[dt], __builtin_bit_cast(bf16x8_t, w3[i]), o[dt], 0, 0, 0);
    __builtin_amdgcn_wave_barrier();
  }
  l_run = quad_sum(l_run);

  // ---- the four waves' shares meet in LDS ------------------------------------
  {
    float* mine = reinterpret_cast<float*>(vs) + l15 * D + lhi * 4;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      *reinterpret_cast<f32x4_t*>(mine + dt * 16) = o[dt];
    if (lhi == 0 && l15 < G) {
      ml[wid][l15][0] = m_run;
      ml[wid][l15][1] = l_run;
    }
  }
  __syncthreads();
  // Neighbouring sums of a thread, as many as take all threads once: in rounds of one
  // sum a thread the reads were half a microsecond of the smallest calls (64 rows of
  // 19 .. 31, 64/8 heads of 128, 5.9 -> 5.3 us; 58 of 14 .. 36, 12/2 heads, 4.7 -> 4.2).
  constexpr int N = (FEW ? 4 : 8) * D / 256;
  typedef __attribute__((ext_vector_type(N))) float part_t;
  const int i = threadIdx.x * N;
  if (i < G * D) {
    const int h = i / D, d = i % D;
    float gm = ml[0][h][0];
#pragma unroll
    for (int w = 1; w < 4; ++w) gm = fmaxf(gm, ml[w][h][0]);
    float l = 0.f, acc[N];
#pragma unroll
    for (int t = 0; t < N; ++t) acc[t] = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float a = exp2_hw(ml[w][h][0] - gm);
      const part_t* part = reinterpret_cast<const part_t*>(lds[w]) + threadIdx.x;
      const part_t p0 = part[0], p1 = part[HC * D / N],
                   p2 = FEW ? part[2 * HC * D / N] : p1;
      l += ml[w][h][1] * a;
#pragma unroll
      for (int t = 0; t < N; ++t) {
        float sum = p0[t] + p1[t];
        if (FEW) sum += p2[t];
        acc[t] += sum * a;
      }
    }
    const long row = (long)b * Hq + hk * G + h;
    if (nsplit == 1) {
      struct alignas(2 * N) { bf16_t v[N]; } to;
#pragma unroll
      for (int t = 0; t < N; ++t) to.v[t] = f2bf(l > 0.f ? acc[t] / l : 0.f);
      *reinterpret_cast<decltype(to)*>(out + row * D + d) = to;
    } else {
      float* pp = partial + (row * nsplit + sp) * (D + 2);
#pragma unroll
      for (int t = 0; t < N; ++t) pp[d + t] = acc[t];
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
  static_assert(DEC_SPLITS <= 64, "a stretch a lane");
  // stretch lane: its maximum and sum
  const float m = lane < nsplit ? base[lane * (D + 2) + D] : -1e30f;
  const float w = __expf(m - wave_reduce_max(m));
  const float gl_sum = wave_reduce_sum(
      lane < nsplit ? base[lane * (D + 2) + D + 1] * w : 0.f);
  // (all stretches on their way at once: 5.5 us one after the other, 3)
  float acc[EPL], part[DEC_SPLITS][EPL];
#pragma unroll
  for (int sp = 0; sp < DEC_SPLITS; ++sp)
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      part[sp][j] = sp < nsplit ? base[sp * (D + 2) + lane + j * 64] : 0.f;
#pragma unroll
  for (int j = 0; j < EPL; ++j) acc[j] = 0.f;
#pragma unroll
  for (int sp = 0; sp < DEC_SPLITS; ++sp) {
    const float a = __shfl(w, sp, 64);
#pragma unroll
    for (int j = 0; j < EPL; ++j)
      if (sp < nsplit) acc[j] += part[sp][j] * a;
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
  // page table holds.
  //
  // Contexts of up to 1024 are divided where the blocks leave half of the CUs
  // idle, but not up to 384: a second launch costs as much (us in a graph, rows of
  // 2/3 of the longest and more; 8 rows of 32/8 heads of 128, up to 256 in one and
  // two stretches 7.0 and 8.5, 384 in one and three 9.0 and 8.9, 512 in one and four
  // 10.7 and 9.3, 1024 in one, four and eight 16.3, 12.2, 12.4; 16 rows 7.9 and 9.7, 9.4
  // and 11.3, 11.0 and 12.0, 16.7, 17.0, 16.9; 24 rows 1024 in one and two 19.8 and
  // 22.9).  Where less than half of the CUs have a second block the others wait for
  // it: heads of 128 in three (33 rows of 682 .. 1024, 32/8 heads, 31.9, 30.6, 29.2 in
  // one to three; of 512 .. 768 24.1, 23.2, 21.9; heads of 64 13.7, 18.4, 17.4).
  //
  // Longer ones: 1024 blocks (25 rows of 1024 .. 2048, 32/8 heads of 128, in 5, 6,
  // 8 and 10: 34.8, 35.4, 37.4, 38.3), but never in eight: blocks go to the eight dies
  // in turn, so that a stretch of every row would go to one die, and the last ones
  // are the shorter (128, 132, 136, 140 and 144 rows and heads of 28/4, 1900 .. 8192, in
  // 7, 8, 9 and 10: 65.2, 66.9, 63.1, 63.3; 69.2, 72.3, 68.2, 69.0; 72.9, 74.5, 73.3, 74.3;
  // 67.4, 68.8, 66.8, 66.7; 72.4, 73.9, 72.2, 72.1; of 1025 .. 5000 45.8, 47.0, 44.4, 45.4
  // at 132; of heads of 64, 32/8, 1900 .. 8192, 38.3, 39.3, 37.6, 37.6 at 136).  From 256
  // rows and heads on an odd number for the same reason: five (33 rows of 2049 ..
  // 8192, 32/8 heads of 128, in 4, 5, 6: 127, 121, 120; 64 of 2000 .. 4096, heads of 64, in
  // 1 to 6: 85, 89, 77, 85, 75, 77; 100 of 1500 .. 3000 102, 96, 84, 94, 84, 87), of heads
  // of 128 three where five are too many (56 of 1024 .. 2048 in 2 to 5: 68.0, 65.0, 67.2,
  // 65.1; 90 of 2000 .. 4096 194, 192, 196, 194).  Of 320 to 960 rows and heads of 1280
  // to 4096 keys that is 2% from the best of one to seven on average; most of it is
  // lost up to 2048 keys, where one is up to 15% quicker (heads of 128 from 512 rows
  // and heads on, of 64 up to 383).
  const long base_blocks = B * Hk;
  const long most = (long)max_pages * page_size;
  int nsplit = 1;
  if (most > 384 && base_blocks < 1024) {
    const long fill = (1024 + base_blocks - 1) / base_blocks;
    const long want =
        most <= 1024
            ? (base_blocks < 128 ? 512 / base_blocks
               : D == 128 && most > 700 && base_blocks > 256 &&
                         base_blocks < 384 ? 3 : 1)
        : base_blocks >= 256 ? (D == 64 || base_blocks <= 341 ? 5 : 3)
        : fill == 8 ? 9 : fill;
    nsplit = (int)std::max<long>(
        1, std::min<long>({want, DEC_SPLITS, (most + 127) / 128}));
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
  // Keys and values go past the caches, read once in whole rows: on inputs that no
  // cache holds, as the layers of a model come in turn, that is the faster the
  // larger the call (128 rows of 257 .. 512, 32/8 heads of 128, 40.4 us with K
  // through the caches in pieces of rows, 44.1 in whole rows, 38.6 past them; 56 of
  // 1024 .. 2048 69.8, 74.6, 65.0; 64 of 257 .. 1024, 64/8 heads, 33.9 and 35.7).  Small
  // calls keep both in the caches for those who repeat them on the same tensors.
  const bool once = B * most * Hk * D * 4 > (128L << 20);
  if (G == 1 && (base_blocks >= 2048 || most <= (D == 128 ? 512 : 64)))
    args(paged_decode_attn_one_kernel<D>);
  else if (G <= 4)
    once ? args(paged_decode_attn_kernel<D, true, true>)
         : args(paged_decode_attn_kernel<D, true, false>);
  else
    once ? args(paged_decode_attn_kernel<D, false, true>)
         : args(paged_decode_attn_kernel<D, false, false>);
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
