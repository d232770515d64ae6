// Varlen causal flash-attention backward v3 (bf16, head_dim 64/128, MFMA).
//
// Reference capability: the training-side flash-attn backward the reference
// reaches through the flash-attn package.
//
// Two kernels that each OWN the rows they write: no atomics, no zero-fill,
// the same bits on every run; gradients are rounded to bf16 once, as they are
// written.  The recompute of S and dP in both is 7 products instead of 5.
// Layouts and operands: attention_tile.h.
//
//  * dq kernel — units, blocks and tiles of the forward kernel
//    (attention_prefill.hip): a wave holds Q and dO of 32 rows of one head in
//    registers and walks the keys; S^T = K Q^T and dP^T = V dO^T, whose
//    difference dS^T, rounded to bf16, is at once the operand of
//    dQ^T += K^T dS^T (K^T by transposed LDS reads of the K tile).  It
//    starts with delta = rowsum(dO * O) of its rows, from the fragments it
//    loads anyway, and leaves it for the other kernel: it runs first.
//  * dkv kernel — a block owns 64 keys of one key/value head and walks the
//    64-row query tiles of the group's heads; wave = (32 keys, 32 rows).
//    S = Q K^T and dP = dO V^T have keys as columns, so P and dS are the
//    operands of dV^T += dO^T P and dK^T += Q^T dS.  256 registers a wave
//    (two waves per SIMD, so that one's exponentials run beside the other's
//    products; at 64 166 and three) hold both gradients and K at D = 128 but not
//    V, which is read from LDS.  Tiles go straight into LDS (AttnTile::copy): Q has
//    two buffers, dO one (two blocks with two of each are 162 KiB), whose next tile
//    arrives beside one step's dK and the next step's S products.  The two waves of
//    a key half meet at the end: each adds the other's share of one gradient.
//    With few blocks the group's heads are divided among several (their
//    shares then pass through fp32 and one summing kernel).
//
// What bounds it: matrix instructions (about 40% of the cycles) and exponentials
// with what surrounds them, of two waves in turn.  Measured, forward and
// backward of packed sequences: 16 of up to 512, 32/8 heads of 128, 727 us with
// kernels that turned Q, dO, K and dS into LDS two bytes at a time and wrote fp32
// gradients for a cast to read, 231 with tiles through registers (whose loads and
// stores took a fifth of the forward kernel's time), 220 now; 2 of up to 4096,
// 28/4 heads, 4000, 1138 and 1015; 8 of up to 1024, 32/8 heads of 64, 200 and 190.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "attention_tile.h"

// ------------------------------------------------------------------- dQ
template <int D>
__global__ __launch_bounds__(256, D == 64 ? 4 : 2) void attn_bwd_dq_kernel(
    bf16_t* __restrict__ dq,         // (total_q, Hq, D)
    float* __restrict__ delta,       // (total_q, Hq)
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
    const bf16_t* __restrict__ v, const bf16_t* __restrict__ out,
    const bf16_t* __restrict__ dout, // (total_q, Hq, D) contiguous, like out
    const float* __restrict__ lse, const int* __restrict__ cu_q,
    const int* __restrict__ cu_k, const int* __restrict__ tile_seq,
    const int* __restrict__ tile_q0, int nseq, int ntiles, int nparts, int Hq,
    int Hk, int G, float scale, int causal, long ldq, long ldk, long ldv) {
  typedef AttnTile<D> T;
  // two buffers of K and V each; at the end the waves' rows of the gradient
  __shared__ __attribute__((aligned(16))) char k0_s[T::BYTES], v0_s[T::BYTES],
      k1_s[T::BYTES], v1_s[T::BYTES];

  const BlockItem item(Hk, nparts);
  const int hk = item.head, part = item.part;
  RowTile tile;
  if (!row_tile<false>(item.tile, ntiles, tile_seq, tile_q0, cu_q, cu_k, nseq, tile))
    return;
  const int q0 = tile.r0, qbeg = tile.qbeg, Lq = tile.Lq;
  const int kbeg = tile.kbeg, Lk = tile.Lk;
  const int qk_off = Lk - Lq;

  const int lane = threadIdx.x & 63;
  const int wid = wave_id();
  constexpr int KS = D / 16, DT = D / 32;
  const int unit = part * 4 + wid;        // (row half, head)
  const int half = (unit >= G) + (unit >= 2 * G);
  const int wq0 = q0 + half * 32;
  const bool busy = unit < 2 * G && wq0 < Lq;
  const int hq = busy ? hk * G + unit - half * G : hk * G;
  const int row = wq0 + (lane & 31);
  const int qpos = causal ? qk_off + row : Lk;

  const int seen = causal ? min(Lk, qk_off + min(wq0 + 32, Lq)) : Lk;
  const int wend = busy ? seen : 0;
  const int last_half = min(part * 4 + 3, 2 * G - 1) >= G;
  const int bend = causal
      ? min(Lk, qk_off + min(q0 + last_half * 32 + 32, Lq)) : Lk;

  const bf16_t* kb = k + (long)kbeg * ldk + (long)hk * D;
  const bf16_t* vb = v + (long)kbeg * ldv + (long)hk * D;
  if (bend > 0) {
    T::copy(k0_s, kb, ldk, Lk);
    T::copy(v0_s, vb, ldv, Lk);
  }
  const long tok = qbeg + min(busy ? row : 0, Lq - 1);
  bf16x8_t qf[KS], df[KS];
  frag_global<D>(df, dout + (tok * Hq + hq) * D);
  float del = 0.f;
  {
    bf16x8_t of[KS];
    frag_global<D>(of, out + (tok * Hq + hq) * D);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) del += (float)df[ks][j] * (float)of[ks][j];
    del = half_sum(del);
  }
  if (busy && lane < 32 && row < Lq) delta[tok * Hq + hq] = del;
  del *= scale;                      // dS is rounded with the scale in it
  frag_global<D>(qf, q + tok * ldq + (long)hq * D);
  const float s2 = scale * 1.4426950408889634f;
  const float lse2 = lse[tok * Hq + hq] * 1.4426950408889634f;

  FragAt<D> at;
  f32x16_t acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;

  wait_loads();
  __syncthreads();

  // one tile; the next one is on its way into the other buffers, whose readers
  // passed the last barrier.  (The compiler loads Q's fragments behind the barrier
  // above and waits for them, and so for the copies, in every other tile.  Held
  // before it the loop has no such wait and takes no less: 2 sequences of 3500 ..
  // 4096, 28/4 heads, forward and backward 1010 us and 1018; 64 of 33 .. 128, 32/8
  // heads, backward 95.8 and 97.2.)
  auto tile_step = [&](const char* ks_, const char* vs_, char* kn, char* vn,
                       int t0) {
    if (t0 + ATILE < bend) {
      kb += ATILE * ldk;
      vb += ATILE * ldv;
      T::copy(kn, kb, ldk, Lk - t0 - ATILE);
      T::copy(vn, vb, ldv, Lk - t0 - ATILE);
    }
    at.renew();
#pragma unroll
    for (int n = 0; n < 2; ++n) {                  // 32 keys at a time
      const int k0 = t0 + n * 32;
      if (k0 >= wend) continue;
      f32x16_t s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.f, dp[r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            frag_rows<D>(ks_, at, n, ks), qf[ks], s, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            frag_rows<D>(vs_, at, n, ks), df[ks], dp, 0, 0, 0);
      }
      SCHED_LDS(6);
#pragma unroll
      for (int i = 0; i < 2 * KS - 6; ++i) {
        SCHED_MFMA(1);
        SCHED_LDS(1);
      }
      SCHED_MFMA(6);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] = exp2_hw(__builtin_fmaf(s[r], s2, -lse2));
      if (k0 + 32 > Lk || (causal && k0 + 31 > qk_off + wq0)) {
        // (compared with literals, in this lane's rows of the accumulators)
        const int last = min(qpos, Lk - 1) - k0 - 4 * (lane >> 5);
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + (r & 3) > last) s[r] = 0.f;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] *= __builtin_fmaf(dp[r], scale, -del);
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bf16x8_t ds = acc_operand(s, st);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              frag_cols<D>(ks_, at, dt, n * 2 + st), ds, acc[dt], 0, 0, 0);
      }
      SCHED_LDS(8);
#pragma unroll
      for (int i = 0; i < 2 * DT - 4; ++i) {
        SCHED_MFMA(1);
        SCHED_LDS(2);
      }
      SCHED_MFMA(4);
    }
    wait_loads();
    __syncthreads();
  };
  for (int t0 = 0; t0 < bend; t0 += 2 * ATILE) {
    tile_step(k0_s, v0_s, k1_s, v1_s, t0);
    if (t0 + ATILE < bend)
      tile_step(k1_s, v1_s, k0_s, v0_s, t0 + ATILE);
  }

  // ---- dQ, turned through LDS to whole rows ---------------------------------
  char* mine = (wid < 2 ? k0_s : v0_s) + wid % 2 * (32 * D * 2);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      bf16x4 w;
#pragma unroll
      for (int t = 0; t < 4; ++t) w.v[t] = f2bf(acc[dt][4 * i + t]);
      const int d = dt * 32 + 8 * i + 4 * (lane >> 5);
      *reinterpret_cast<bf16x4*>(
          mine + (lane & 31) * (2 * D) +
          (((d >> 3) ^ T::swz(lane & 31)) << 4) + (d & 4) * 2) = w;
    }
  __syncthreads();
  if (!busy) return;
  T::store32(mine, dq + (((long)qbeg + wq0) * Hq + hq) * D, (long)Hq * D,
             Lq - wq0);
}

// ---------------------------------------------------------------- dK/dV
template <int D>
__global__ __launch_bounds__(256, 2) void attn_bwd_dkv_kernel(
    bf16_t* __restrict__ dk,         // (total_k, Hk, D); nsplit == 1
    bf16_t* __restrict__ dv,
    float* __restrict__ part,        // (nsplit, 2, total_k, Hk, D), else
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k,
    const bf16_t* __restrict__ v, const bf16_t* __restrict__ dout,
    const float* __restrict__ lse, const float* __restrict__ delta,
    const int* __restrict__ cu_q, const int* __restrict__ cu_k,
    const int* __restrict__ tile_seq, const int* __restrict__ tile_k0,
    int nseq, int ntiles, int nsplit, long total_k, int Hq, int Hk, int G,
    float scale, int causal, long ldq, long ldk, long ldv) {
  typedef AttnTile<D> T;
  constexpr bool V_LDS = D == 128;   // V does not fit beside the gradients
  __shared__ __attribute__((aligned(16))) char q0_s[T::BYTES], q1_s[T::BYTES],
      do_s[T::BYTES], v_s[T::BYTES];
  // log-sum-exp (in powers of two) and scale * delta of the rows
  __shared__ __attribute__((aligned(16))) float r0_s[2][ATILE], r1_s[2][ATILE];

  const BlockItem item(Hk, nsplit);
  const int hk = item.head, split = item.part;
  const int g0 = G * split / nsplit, g1 = G * (split + 1) / nsplit;
  RowTile tile;
  if (!row_tile<true>(item.tile, ntiles, tile_seq, tile_k0, cu_q, cu_k, nseq, tile))
    return;
  const int t0 = tile.r0, qbeg = tile.qbeg, Lq = tile.Lq;
  const int kbeg = tile.kbeg, Lk = tile.Lk;
  const int qk_off = Lk - Lq;
  if (t0 >= Lk) return;

  const int lane = threadIdx.x & 63;
  const int wid = wave_id();
  const int kh = wid & 1, qh = wid >> 1;           // key half, row half
  constexpr int KS = D / 16, DT = D / 32;
  const int wk0 = t0 + kh * 32;                    // this wave's first key
  const int key = wk0 + (lane & 31);               // this lane's key
  const int krow = kbeg + min(key, Lk - 1);

  bf16x8_t kf[KS], vf[V_LDS ? 1 : KS];
  frag_global<D>(kf, k + (long)krow * ldk + (long)hk * D);
  if constexpr (!V_LDS)
    frag_global<D>(vf, v + (long)krow * ldv + (long)hk * D);
  const float s2 = scale * 1.4426950408889634f;

  FragAt<D> at;
  f32x16_t ak[DT], av[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) ak[dt][r] = 0.f, av[dt][r] = 0.f;

  // query tiles that see key t0, one head after the other
  const int qs = causal ? max(t0 - qk_off, 0) / ATILE * ATILE : 0;
  const int nq = qs < Lq ? (Lq - qs + ATILE - 1) / ATILE : 0;
  const int steps = (g1 - g0) * nq;
  const bf16_t* qb0 = q + (long)qbeg * ldq + (long)hk * G * D;
  const bf16_t* db0 = dout + ((long)qbeg * Hq + (long)hk * G) * D;

  float rowv = 0.f;                                // lse or delta of a row
  bool rlive = false;
  int fg = g0, fq = qs;               // head and first row of the next tile
  auto fetch_rows = [&]() {           // the first two waves' are stored
    const int r = fq + lane;
    const long i = ((long)qbeg + min(r, Lq - 1)) * Hq + hk * G +
                   min(fg, g1 - 1);
    rlive = r < Lq;
    rowv = (wid == 0 ? lse : delta)[i];
  };
  auto store_rows = [&](float (*row_s)[ATILE]) {
    // rows past the end weigh nothing: 2^(s - inf) = 0
    if (wid == 0) row_s[0][lane] = rlive ? rowv * 1.4426950408889634f : INFINITY;
    if (wid == 1) row_s[1][lane] = rlive ? rowv * scale : 0.f;
  };
  auto copy_q = [&](char* to) {
    T::copy(to, qb0 + (long)fg * D + fq * ldq, ldq, Lq - fq);
  };
  auto copy_do = [&]() {              // and on to the next tile
    T::copy(do_s, db0 + (long)fg * D + (long)fq * Hq * D, (long)Hq * D,
            Lq - fq);
    fq += ATILE;
    if (fq >= Lq) fq = qs, ++fg;
  };
  if (steps > 0) {
    if constexpr (V_LDS)
      T::copy(v_s, v + ((long)kbeg + t0) * ldv + (long)hk * D, ldv, Lk - t0);
    fetch_rows();
    copy_q(q0_s);
    copy_do();
    store_rows(r0_s);
  }
  wait_loads();
  __syncthreads();

  // One row tile.  S needs Q alone: the dO tile, whose one buffer was free only
  // after the last step's dV product, arrives beside that step's dK and this
  // step's S products (first barrier); the next Q tile beside the rest, up to
  // the dV product (second).
  int q0 = qs;
  auto step = [&](const char* qs_, char* qn, float (*row_s)[ATILE],
                  float (*row_n)[ATILE], bool more) {
    const int wq0 = q0 + qh * 32;                     // this wave's rows
    q0 = q0 + ATILE < Lq ? q0 + ATILE : qs;
    const bool work = wq0 < Lq && wk0 < Lk &&
                      (!causal || qk_off + wq0 + 31 >= wk0);
    at.renew();
    f32x16_t s, dp;
    bf16x8_t p[2], ds[2];
    const int r0 = qh * 32 + 4 * (lane >> 5);
    // The weights need no dO: at 64 they come before the barrier that waits for it
    // (8 sequences of 300 .. 1024, 32/8 heads, forward and backward 163.4 us behind
    // it, 160.3 before), at 128 their exponentials do better beside dP (2 of 3500 ..
    // 4096, 28/4 heads, 986 and 996).
    auto weights = [&] {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4 le = *reinterpret_cast<const float4*>(&row_s[0][r0 + 8 * i]);
        const float l4[4] = {le.x, le.y, le.z, le.w};
#pragma unroll
        for (int t = 0; t < 4; ++t)
          s[4 * i + t] = __builtin_fmaf(s[4 * i + t], s2, -l4[t]);
      }
      // rows before this lane's key (compared with literals), whatever their
      // log-sum-exp: it may be NaN
      if (causal && qk_off + wq0 < wk0 + 31) {
        const int border = key - (qk_off + wq0) - 4 * (lane >> 5);
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (8 * (r >> 2) + (r & 3) < border) s[r] = -INFINITY;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = exp2_hw(s[r]);
    };
    if (work) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            frag_rows<D>(qs_, at, qh, ks), kf[ks], s, 0, 0, 0);
      SCHED_LDS(3);
#pragma unroll
      for (int i = 0; i < KS - 3; ++i) {
        SCHED_MFMA(1);
        SCHED_LDS(1);
      }
      SCHED_MFMA(3);
      if constexpr (D == 64) weights();
    }
    wait_loads();
    __syncthreads();
    if (more) {
      fetch_rows();
      copy_q(qn);
    }
    if (work) {
#pragma unroll
      for (int r = 0; r < 16; ++r) dp[r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            frag_rows<D>(do_s, at, qh, ks),
            V_LDS ? frag_rows<D>(v_s, at, kh, ks) : vf[V_LDS ? 0 : ks], dp, 0,
            0, 0);
      constexpr int PER = V_LDS ? 2 : 1;           // fragments of a product
      SCHED_LDS(3 * PER);
#pragma unroll
      for (int i = 0; i < KS - 3; ++i) {
        SCHED_MFMA(1);
        SCHED_LDS(PER);
      }
      SCHED_MFMA(3);
      if constexpr (D == 128) weights();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4 de = *reinterpret_cast<const float4*>(&row_s[1][r0 + 8 * i]);
        const float d4[4] = {de.x, de.y, de.z, de.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int r = 4 * i + t;
          dp[r] = s[r] * __builtin_fmaf(dp[r], scale, -d4[t]);
        }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        p[h] = acc_operand(s, h);
        ds[h] = acc_operand(dp, h);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          av[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              frag_cols<D>(do_s, at, dt, qh * 2 + h), p[h], av[dt], 0, 0, 0);
    }
    if (more) store_rows(row_n);
    wait_loads();
    __syncthreads();
    if (more) copy_do();
    if (work) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          ak[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              frag_cols<D>(qs_, at, dt, qh * 2 + h), ds[h], ak[dt], 0, 0, 0);
      SCHED_LDS(6);
#pragma unroll
      for (int i = 0; i < 2 * DT - 3; ++i) {
        SCHED_MFMA(1);
        SCHED_LDS(2);
      }
      SCHED_MFMA(3);
    }
  };
  for (int st = 0; st < steps; st += 2) {
    step(q0_s, q1_s, r0_s, r1_s, st + 1 < steps);
    if (st + 1 < steps) step(q1_s, q0_s, r1_s, r0_s, st + 2 < steps);
  }
  __syncthreads();

  // ---- the two waves of a key half: one completes dV, the other dK ----------
  auto share = [&](int w) {
    return reinterpret_cast<float*>(w == 0 ? q0_s : w == 1 ? q1_s
                                    : w == 2 ? do_s : v_s);
  };
  float* mine = share(wid);
  const float* other = share(wid ^ 2);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      mine[(dt * 16 + r) * 64 + lane] = qh == 0 ? ak[dt][r] : av[dt][r];
  __syncthreads();
  const bool ok = key < Lk;
  const long o = ((long)krow * Hk + hk) * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f32x4v w;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int r = 4 * i + t;
        w.v[t] = (qh == 0 ? av[dt][r] : ak[dt][r]) +
                 other[(dt * 16 + r) * 64 + lane];
      }
      const int d = dt * 32 + 8 * i + 4 * (lane >> 5);
      if (!ok) continue;
      if (part != nullptr) {
        *reinterpret_cast<f32x4v*>(
            part + (split * 2 + (qh == 0 ? 1 : 0)) * (total_k * Hk * D) + o +
            d) = w;
      } else {
        bf16x4 b;
#pragma unroll
        for (int t = 0; t < 4; ++t) b.v[t] = f2bf(w.v[t]);
        *reinterpret_cast<bf16x4*>((qh == 0 ? dv : dk) + o + d) = b;
      }
    }
}

// dK, dV = sums over the head shares
__global__ void attn_bwd_sum_kernel(bf16_t* __restrict__ dk,
                                    bf16_t* __restrict__ dv,
                                    const float* __restrict__ part,
                                    int nsplit, long n /* of one gradient */) {
  const long i = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= n) return;
  bf16_t* const to[2] = {dk, dv};
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    f32x4v a = *reinterpret_cast<const f32x4v*>(part + w * n + i);
    for (int s = 1; s < nsplit; ++s) {
      const f32x4v b =
          *reinterpret_cast<const f32x4v*>(part + (2 * s + w) * n + i);
#pragma unroll
      for (int t = 0; t < 4; ++t) a.v[t] += b.v[t];
    }
    bf16x4 o;
#pragma unroll
    for (int t = 0; t < 4; ++t) o.v[t] = f2bf(a.v[t]);
    *reinterpret_cast<bf16x4*>(to[w] + i) = o;
  }
}

// ---------------------------------------------------------------- launcher
template <int D>
static void launch_bwd(torch::Tensor& dq, torch::Tensor& dk,
                       torch::Tensor& dv, const torch::Tensor& q,
                       const torch::Tensor& k, const torch::Tensor& v,
                       const torch::Tensor& out, const torch::Tensor& dout,
                       const torch::Tensor& lse, const torch::Tensor& cu_q,
                       const torch::Tensor& cu_k, const torch::Tensor& t_seq,
                       const torch::Tensor& t_q0, float scale, bool causal) {
  const int Hq = q.size(1), Hk = k.size(1), G = Hq / Hk;
  const long ntiles = t_seq.size(0), total_k = k.size(0);
  auto stream = at::hip::getCurrentHIPStream();
  const int nseq = cu_q.size(0) - 1;
  auto blocks = [&](long items) {
    TORCH_CHECK(items < (1L << 31), "grid too large");
    return dim3((unsigned)items);
  };
  auto delta = torch::empty_like(lse);
  const int nparts = (2 * G + 3) / 4;
  attn_bwd_dq_kernel<D>
      <<<blocks(ntiles * Hk * nparts), dim3(256), 0, stream>>>(
          (bf16_t*)dq.data_ptr(), delta.data_ptr<float>(),
          (const bf16_t*)q.data_ptr(), (const bf16_t*)k.data_ptr(),
          (const bf16_t*)v.data_ptr(), (const bf16_t*)out.data_ptr(),
          (const bf16_t*)dout.data_ptr(), lse.data_ptr<float>(),
          cu_q.data_ptr<int>(), cu_k.data_ptr<int>(), t_seq.data_ptr<int>(),
          t_q0.data_ptr<int>(), nseq, (int)ntiles, nparts, Hq, Hk, G, scale,
          causal ? 1 : 0, q.stride(0), k.stride(0), v.stride(0));
  // Blocks of the dkv kernel are as long as their key is early and run longest
  // first, 512 at a time (two per CU).  For all to end together the longest may
  // not exceed a slot's share of the steps: in a sequence of m tiles the longest
  // block takes m steps a head, a slot's share is G * base * m / 2 / 512, so a
  // block takes 0.9 of G * base / 1024 heads of its group.  Sequences of less
  // than 16 tiles are cut less fine: the shares' trip through fp32 costs as much
  // whatever the length.  Measured, forward and backward: 2 sequences of 3500 ..
  // 4096, 28/4 heads (476 key tiles), blocks of 1, 2, 3 and 4 heads 1041, 1015,
  // 1015, 1037 us; one of 4096, 32/8 heads (512), of 1, 2 and 4 668, 669, 735; 3 of
  // 4096, 28/4 (768), of 3, 4 and 7 1830, 1828, 1837.  Sequences of 800 .. 1024,
  // 64/8 heads (480), of 2, 3 and 4 389, 384, 376; 16 of 130 .. 512, 28/4 heads
  // (372), of 2, 3 and 4 170, 161, 155.
  // The shares take 64 KiB a block at D = 128 while the call runs: at most 48 MiB
  // times the heads of a group.
  const long base = ntiles * Hk;
  const bool lengthy = ntiles >= 16 * nseq;
  int nsplit = 1;
  if (base < (lengthy ? 768 : 512)) {
    const int per = (int)(lengthy ? std::max<long>(1, G * base * 9 / 10240)
                                  : (G * base + 767) / 768);
    nsplit = (G + per - 1) / per;
  }
  torch::Tensor part;
  if (nsplit > 1)
    part = torch::empty({nsplit, 2, total_k, (long)Hk, (long)D},
                        lse.options());
  attn_bwd_dkv_kernel<D><<<blocks(base * nsplit), dim3(256), 0, stream>>>(
      (bf16_t*)dk.data_ptr(), (bf16_t*)dv.data_ptr(),
      nsplit > 1 ? part.data_ptr<float>() : nullptr,
      (const bf16_t*)q.data_ptr(), (const bf16_t*)k.data_ptr(),
      (const bf16_t*)v.data_ptr(), (const bf16_t*)dout.data_ptr(),
      lse.data_ptr<float>(), delta.data_ptr<float>(), cu_q.data_ptr<int>(),
      cu_k.data_ptr<int>(), t_seq.data_ptr<int>(), t_q0.data_ptr<int>(),
      nseq, (int)ntiles, nsplit, total_k, Hq, Hk, G, scale, causal ? 1 : 0,
      q.stride(0), k.stride(0), v.stride(0));
  if (nsplit > 1) {
    const long n = total_k * Hk * D;
    attn_bwd_sum_kernel<<<dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0,
                          stream>>>((bf16_t*)dk.data_ptr(),
                                    (bf16_t*)dv.data_ptr(),
                                    part.data_ptr<float>(), nsplit, n);
  }
  HIP_CHECK_KERNEL();
}

// t64_seq / t64_q0: the 64-row tiles of the packed rows (build_varlen_tiles);
// query and key rows share them, so both sides are cut alike.
void varlen_attention_backward_v3(
    torch::Tensor dq, torch::Tensor dk, torch::Tensor dv,  // bf16 (empty ok)
    torch::Tensor q, torch::Tensor k, torch::Tensor v,
    torch::Tensor out, torch::Tensor dout, torch::Tensor lse,
    torch::Tensor cu_seqlens_q, torch::Tensor cu_seqlens_k,
    torch::Tensor t64_seq, torch::Tensor t64_q0,
    double scale, bool causal) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16);
  auto packed = [](const torch::Tensor& t) {
    return t.stride(2) == 1 && t.stride(1) == t.size(2);
  };
  TORCH_CHECK(packed(q) && packed(k) && packed(v));
  TORCH_CHECK(out.is_contiguous() && dout.is_contiguous());
  TORCH_CHECK(out.dtype() == torch::kBFloat16 &&
              dout.dtype() == torch::kBFloat16);
  TORCH_CHECK(lse.is_contiguous() && lse.dtype() == torch::kFloat32);
  for (const auto* g : {&dq, &dk, &dv})
    TORCH_CHECK(g->dtype() == torch::kBFloat16 && g->is_contiguous());
  const int Hq = q.size(1), D = q.size(2), Hk = k.size(1);
  TORCH_CHECK(D == 128 || D == 64, "backward v3 supports head_dim 64/128");
  TORCH_CHECK(Hq % Hk == 0 && (long)Hq * D < AttnTile<64>::STORE_LD);
  if (t64_seq.size(0) == 0) return;
  (D == 128 ? launch_bwd<128> : launch_bwd<64>)(
      dq, dk, dv, rows_by16(q), rows_by16(k), rows_by16(v), out,
      rows_by16(dout), lse, cu_seqlens_q, cu_seqlens_k,
      t64_seq, t64_q0, (float)scale, causal);
}
