// Varlen causal prefill attention, bf16, head_dim 64/128, GQA — MFMA forward.
//
// Reference capability: chunked-prefill flash attention.  Flash-style online
// softmax, no score matrix in memory.
//
// Split.  A wave owns 32 query rows of one head; a block is four such units
// of one 64-row tile and one key/value head, heads of the group first (four
// heads x 32 rows with a group of four), so the four waves read the same
// keys and end at the same causal border.  K and V tiles of 64 keys go straight
// into LDS (AttnTile::copy), the next tile during this one's products.  Heads of
// 64: two buffers of both, 32 KiB, and no more than 128 registers, so that four
// blocks run per CU.  Heads of 128: two of K and one of V, whose next tile is
// on its way from the last value product to the next softmax (a second barrier
// a tile, where the next keys have to be there too), 48 KiB and 165 registers:
// three blocks.
//
// Products.  Scores are computed as S^T = K Q^T with the queries held in
// registers: a lane's accumulators are 16 keys of ONE row, so the softmax
// takes one lane exchange per tile, the row's maximum and sum are scalars of
// the lane, and the weights, rounded to bf16, are at once the operand of
// O^T += V^T P^T, whose V^T comes from the row-major tile by transposed LDS
// reads (layouts: attention_tile.h).  The output is rescaled in tiles that
// lift some row's maximum; only tiles that touch the causal border or the
// sequence's end are masked.
//
// What bounds it: at 64 the vector instructions, 76% of the cycles, 87% of those in which
// a CU has a wave, beside matrix instructions at 38 and 44 (185 vector instructions a tile of
// a wave: exponential, scale, sum, maximum, rounding, and the rescaling of the
// output); at 128 those and the matrix instructions, 58% and 44%, and what is
// left of their taking turns (the 16-row score tiles with scalar LDS gathers for
// V that this replaces ran at 160 TFLOP/s).  Blocks of a second row half that
// holds no row still fetch the tiles (7% of the walks of 16 sequences of up to
// 512 rows).  Measured, eight ragged prompts of 1200 .. 2048 tokens, 32/8 heads
// of 64: 671 us a call with those and the tile table's trip through the host (50
// us), 154 with tiles through registers and three blocks per CU, 141 now (757
// TFLOP/s of live pairs); of 128: 283 in the sequences' order, 280, 243 now; two
// sequences of 3500 .. 4096, 28/4 heads of 128, 323, 265, 222.  Where the prompts took
// 147.5 (another card) they took 128 with no tile loaded after the first and 128
// without exponentials, of 128 248, 205 and 231.  Up to 64 sequences
// run in the order of their walks, more in the table's (as all did before: 100
// prompts of 21 .. 80 take what they took).  A maximum that may lag by 2^6 saves
// the rescaling in most tiles (5 to 7%), but then a row's largest weight is no
// longer exactly 1 and takes part in the rounding to bf16: the error against 64
// bits grows by 2 to 3% (2.03e-3 for 1.98e-3, rms, 1024 keys).
//
// Chunked-prefill semantics: query block aligned to the END of the keys
// (q row i at absolute kv position (Lk - Lq) + i), matching ops/ref.py.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "attention_tile.h"

// ONE_V: one buffer of values
template <int D, bool ONE_V>
__global__ __launch_bounds__(256, D == 64 ? 4 : ONE_V ? 3 : 2)
void prefill_attn_kernel(
    bf16_t* __restrict__ out,        // (total_q, Hq, D)
    float* __restrict__ lse,         // (total_q, Hq) log-sum-exp, or null
    const bf16_t* __restrict__ q,    // (total_q, Hq, D)
    const bf16_t* __restrict__ k,    // (total_k, Hk, D)
    const bf16_t* __restrict__ v,    // (total_k, Hk, D)
    const int* __restrict__ cu_q,    // (B+1,)
    const int* __restrict__ cu_k,
    const int* __restrict__ tile_seq,  // (ntiles,) or null
    const int* __restrict__ tile_q0,   // (ntiles,) local first q row
    int nseq, int ntiles, int nparts, int Hq, int Hk, int G, float scale,
    int causal,
    long ldq, long ldk, long ldv) {
  typedef AttnTile<D> T;
  // two buffers of K and V each; at the end the waves' rows of the output
  __shared__ __attribute__((aligned(16))) char k0_s[T::BYTES], v0_s[T::BYTES],
      k1_s[T::BYTES], vx_s[ONE_V ? 16 : T::BYTES];
  char* const v1_s = ONE_V ? v0_s : vx_s;

  // Blocks go to the dies in turn (id % 8): with the key/value head innermost a
  // die has one head or few, and every die a share of every length.  The parts
  // of a tile are not equal (the last may have fewer heads): they turn from tile
  // to tile, so that no die has only the short ones
  const BlockItem item(Hk, nparts);
  const int hk = item.head, part = item.part;
  RowTile tile;
  if (!row_tile<false>(item.tile, ntiles, tile_seq, tile_q0, cu_q, cu_k, nseq, tile))
    return;
  const int q0 = tile.r0, qbeg = tile.qbeg, Lq = tile.Lq;
  const int kbeg = tile.kbeg, Lk = tile.Lk;
  const int qk_off = Lk - Lq;                      // chunked-prefill alignment

  const int lane = threadIdx.x & 63;
  const int wid = wave_id();
  constexpr int KS = D / 16, DT = D / 32;
  const int unit = part * 4 + wid;        // (row half, head)
  const int half = (unit >= G) + (unit >= 2 * G);
  const int hq = hk * G + unit - half * G;
  const int wq0 = q0 + half * 32;                  // this wave's first row
  const bool busy = unit < 2 * G && wq0 < Lq;
  const int row = wq0 + (lane & 31);               // this lane's row
  const int qpos = causal ? qk_off + row : Lk;     // last key it sees

  // keys that this wave and this block walk
  const int seen = causal ? min(Lk, qk_off + min(wq0 + 32, Lq)) : Lk;
  const int wend = busy ? seen : 0;
  const int last_half = min(part * 4 + 3, 2 * G - 1) >= G;
  const int bend = causal
      ? min(Lk, qk_off + min(q0 + last_half * 32 + 32, Lq)) : Lk;

  bf16x8_t qf[KS];
  frag_global<D>(qf, q + (long)(qbeg + min(busy ? row : 0, Lq - 1)) * ldq +
                         (long)hq * D * (busy ? 1 : 0));

  FragAt<D> at;
  // scores in powers of two.  Hidden keys are marked before the scale is
  // multiplied in, so a scale of 0 becomes the smallest number: every score is
  // then 0 all the same, but a hidden one -inf and not -inf * 0
  const float s2 = scale != 0.f ? scale * 1.4426950408889634f : 0x1p-126f;
  const float hidden = s2 >= 0.f ? -INFINITY : INFINITY;
  float m_run = -1e30f, l_run = 0.f;               // l: this lane's keys only
  f32x16_t o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;

  const bf16_t* kb = k + (long)kbeg * ldk + (long)hk * D;
  const bf16_t* vb = v + (long)kbeg * ldv + (long)hk * D;
  if (bend > 0) {
    T::copy(k0_s, kb, ldk, Lk);
    T::copy(v0_s, vb, ldv, Lk);
  }
  wait_loads();
  __syncthreads();

  auto tile_step = [&](const char* ks_, const char* vs_, char* kn, char* vn,
                       int t0) {
    const bool more = t0 + ATILE < bend;
    if (more) {
      kb += ATILE * ldk;
      T::copy(kn, kb, ldk, Lk - t0 - ATILE);
      if (!ONE_V) {
        vb += ATILE * ldv;
        T::copy(vn, vb, ldv, Lk - t0 - ATILE);
      }
    }
    at.renew();
    f32x16_t s[2];
    if (t0 < wend) {
      // ---- S^T: 64 keys x 32 rows ------------------------------------------
#pragma unroll
      for (int r = 0; r < 16; ++r) s[0][r] = 0.f, s[1][r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int n = 0; n < 2; ++n)
          s[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              frag_rows<D>(ks_, at, n, ks), qf[ks], s[n], 0, 0, 0);
      SCHED_LDS(3);
#pragma unroll
      for (int i = 0; i < 2 * KS - 3; ++i) {
        SCHED_MFMA(1);
        SCHED_LDS(1);
      }
      SCHED_MFMA(3);
      // ---- mask (wave-uniform: some key of the tile is hidden) --------------
      if (t0 + ATILE > Lk || (causal && t0 + ATILE - 1 > qk_off + wq0)) {
        // (in this lane's rows of the accumulators, so that the numbers it is
        // compared with are literals: else they live in 32 registers)
        const int last = min(qpos, Lk - 1) - t0 - 4 * (lane >> 5);
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (n * 32 + 8 * (r >> 2) + (r & 3) > last) s[n][r] = hidden;
      }
      // ---- online softmax -----------------------------------------------------
      // (largest score: the smallest product where the scale is negative)
      float mx = s[0][0];
      if (s2 >= 0.f) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[n][r]);
      } else {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int r = 0; r < 16; ++r) mx = fminf(mx, s[n][r]);
      }
      const float mn = fmaxf(m_run, half_max(mx * s2));
      // the largest weight is exactly 1, so bf16 does not round it
      if (__any(mn > m_run)) {
        const float alpha = exp2_hw(m_run - mn);
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
        m_run = mn;
      }
      // (very large scores are rounded like their maximum: what it lost to
      // rounding would pass the exponential's range)
      float by = s2, less = m_run;
      if (__any(fabsf(m_run) >= 0x1p24f)) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s[n][r] = rounded_product(s[n][r], s2) - m_run;
        by = 1.f, less = 0.f;
      }
      float sum = 0.f;
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          s[n][r] = exp2_hw(__builtin_fmaf(s[n][r], by, -less));
          sum += s[n][r];
        }
      l_run += sum;
    }
    if (ONE_V) {
      // this tile's values are there.  (The next keys need not be, but the barrier
      // waits for them too: the compiler sees copies that write LDS.)
      if (more) wait_all_but<T::LOADS>();
      else wait_loads();
      __syncthreads();
    }
    if (t0 < wend) {
      // ---- O^T += V^T P^T ------------------------------------------------------
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const bf16x8_t p = acc_operand(s[st >> 1], st & 1);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              frag_cols<D>(vs_, at, dt, st), p, o[dt], 0, 0, 0);
      }
      SCHED_LDS(4);
#pragma unroll
      for (int i = 0; i < 4 * DT - 2; ++i) {
        SCHED_MFMA(1);
        SCHED_LDS(2);
      }
      SCHED_MFMA(2);
    }
    wait_loads();
    __syncthreads();
    if (ONE_V && more) {
      vb += ATILE * ldv;
      T::copy(vn, vb, ldv, Lk - t0 - ATILE);
    }
  };
  for (int t0 = 0; t0 < bend; t0 += 2 * ATILE) {
    tile_step(k0_s, v0_s, k1_s, v1_s, t0);
    if (t0 + ATILE < bend)
      tile_step(k1_s, v1_s, k0_s, v0_s, t0 + ATILE);
  }

  // ---- out = O / l, turned through LDS to whole rows; lse = m + log l --------
  const float l = half_sum(l_run);
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  char* mine = (wid < 2 ? k0_s : v0_s) + wid % 2 * (32 * D * 2);
  if (busy) {
    if (lse != nullptr && lane < 32 && row < Lq)
      lse[((long)qbeg + row) * Hq + hq] =
          l > 0.f ? m_run * 0.6931471805599453f + __logf(l) : -1e30f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bf16x4 w;
#pragma unroll
        for (int t = 0; t < 4; ++t) w.v[t] = f2bf(o[dt][4 * i + t] * inv);
        const int d = dt * 32 + 8 * i + 4 * (lane >> 5);
        *reinterpret_cast<bf16x4*>(
            mine + (lane & 31) * (2 * D) +
            (((d >> 3) ^ T::swz(lane & 31)) << 4) + (d & 4) * 2) = w;
      }
  }
  __syncthreads();
  if (!busy) return;
  T::store32(mine, out + (((long)qbeg + wq0) * Hq + hq) * D, (long)Hq * D,
             Lq - wq0);
}

// tile_seq / tile_q0: the 64-row tiles of the packed rows to compute (all or some
// of them), or empty: the kernel then finds all from cu_seqlens_q itself.
void varlen_prefill_attention(torch::Tensor out, torch::Tensor q,
                              torch::Tensor k, torch::Tensor v,
                              torch::Tensor cu_seqlens_q,
                              torch::Tensor cu_seqlens_k,
                              torch::Tensor tile_seq, torch::Tensor tile_q0,
                              double scale, bool causal,
                              torch::Tensor lse /* undefined or (tq,Hq) f32 */) {
  const bool want_lse = lse.defined() && lse.numel() > 0;
  if (want_lse) {
    TORCH_CHECK(lse.dtype() == torch::kFloat32 && lse.is_contiguous());
    TORCH_CHECK(lse.size(0) == q.size(0) && lse.size(1) == q.size(1));
  }
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16);
  auto packed = [](const torch::Tensor& t) {
    return t.stride(2) == 1 && t.stride(1) == t.size(2);
  };
  TORCH_CHECK(packed(q) && packed(k) && packed(v),
              "q/k/v heads and dims must be packed (token stride free)");
  TORCH_CHECK(out.is_contiguous());
  TORCH_CHECK(cu_seqlens_q.dtype() == torch::kInt32);
  const bool table = tile_seq.defined() && tile_seq.numel() > 0;
  if (table)
    TORCH_CHECK(tile_seq.dtype() == torch::kInt32 &&
                tile_q0.dtype() == torch::kInt32);
  k = rows_by16(k);
  v = rows_by16(v);
  const int Hq = q.size(1), D = q.size(2), Hk = k.size(1);
  TORCH_CHECK(D == 128 || D == 64, "prefill kernel supports head_dim 64/128");
  TORCH_CHECK(Hq % Hk == 0 && (long)Hq * D < AttnTile<64>::STORE_LD);
  const int nseq = cu_seqlens_q.size(0) - 1;
  const long ntiles = table ? tile_seq.size(0)
                            : q.size(0) / ATILE + nseq;
  if (ntiles == 0 || q.size(0) == 0) return;
  const int nparts = (2 * (Hq / Hk) + 3) / 4;      // blocks of a tile's units
  const long items = ntiles * Hk * nparts;
  TORCH_CHECK(items < (1L << 31), "grid too large");
  auto stream = at::hip::getCurrentHIPStream();
  // One buffer of values costs a wait in the middle of a tile, which only a third
  // block per CU makes up for, so not where two per CU are all of them: one prompt
  // of 1200, 28/4 heads of 128 (300 blocks), 31.3 us with one and 29.8 with two; one
  // of 512, 32/8 heads 15.8 and 15.0; eight of 1200 .. 2048 (3400) 243 and 259.
  auto kern = D == 64        ? prefill_attn_kernel<64, false>
              : items <= 512 ? prefill_attn_kernel<128, false>
                             : prefill_attn_kernel<128, true>;
  kern<<<dim3((unsigned)items), dim3(256), 0, stream>>>(
      (bf16_t*)out.data_ptr(),
      want_lse ? lse.data_ptr<float>() : nullptr,
      (const bf16_t*)q.data_ptr(),
      (const bf16_t*)k.data_ptr(), (const bf16_t*)v.data_ptr(),
      cu_seqlens_q.data_ptr<int>(), cu_seqlens_k.data_ptr<int>(),
      table ? tile_seq.data_ptr<int>() : nullptr,
      table ? tile_q0.data_ptr<int>() : nullptr, nseq, (int)ntiles, nparts,
      Hq, Hk, Hq / Hk, (float)scale, causal ? 1 : 0, q.stride(0), k.stride(0),
      v.stride(0));
  HIP_CHECK_KERNEL();
}
