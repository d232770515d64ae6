// Fused sampling: temperature + top-k + top-p filter + categorical draw +
// sampled-token logprob capture.
//
// Reference capability: the engine-side sampling + per-token logprob kernels.
// Semantics:
//  * top-k threshold = k-th largest logit, found by radix select over the
//    monotone uint32 encoding of the logit (temperature doesn't change order,
//    so select on raw logits).
//  * top-p threshold found by the same walk, accumulating per-bin
//    sum(exp((x - m)/T)) mass instead of counts.
//  * the draw is Gumbel-argmax over the kept set: argmax(x/T + G_i), exact
//    categorical sampling in one streaming pass, counter-based RNG
//    (splitmix64 keyed by (seed, row, i)) so replay is deterministic.
//  * reported logprob is under the raw (unfiltered, T=1) softmax, matching
//    what rollout clients consume as output_token_logprobs.
//
// Split.  A row is cut into ``split`` pieces, one block each, so that a few
// rows fill the chip too (a block per row left half of it idle at 128 rows);
// the pieces meet in small per-row arrays.  Without a filter that is one pass,
// sums of the raw softmax and the draw together, and a merging launch.  With one:
// sums; the candidates of both thresholds, from which, where they are few, the
// row's last block has the token at once; else one pass per radix digit (11 bits,
// then the rest of a bf16 number's 16 or an fp32 number's 32), whose last block
// walks the bins, and the draw over the kept set, whose last block merges.  Short
// rows take the same steps in one launch, a block each.  (64 x 151936, T 0.7, k
// 50, p 0.9: 52.8 us with plans and a merge in launches of their own, eight in all,
// 24 now; top-p 0.95 alone 70 and 61; at a temperature of 0 33 and 17.)
//
// Only entries that can stand at a threshold go into a digit's bins (cut_of):
// with k at most the number of lane groups, the k-th largest of the groups'
// maxima is no more than the k-th largest entry; and entries that each have
// less than 0.99 (1 - p) / V of the mass have less than 1 - p together, so the
// nucleus ends above them.  (Total and bins add the same exp((x - m)/T), which
// is exact near m however large m/T is; should rounding leave the bins short
// of p all the same, the nucleus ends at the cut.)  All entries of 64 x 151936
// (0.7, 50, 0.9) in LDS atomics took 73 us a digit; half of 1 - p in place of 0.99
// took 11% longer (top-p 0.95 of 256 x 152064, 229 and 254 us in the eight launches
// of before, 157 now).
//
// What bounds it: vector instructions, most of them the generator's integer
// multiplies (two 64-bit products a number; a number's place in the sequence is
// the last one's plus a constant, kept from the compiler, which would multiply; of
// the second product the upper word alone).  The two logarithms of a number's noise
// are only taken where its 24 random bits can beat the best so far: z > best means
// u > exp(-exp(x/T - best)), one threshold per 16-byte word of logits from the
// word's largest, with a margin far above the rounding of either side.  The best so
// far is the block's: its waves raise a number in LDS, which only ever holds what
// some entry has, so that whoever is late reads less and nobody waits; and the
// first words, which know of none, take it from noise in seven instructions, less
// its error.  (128 x 128256 at temperature 1: 33.1 us with a product for the place
// and exchanges of a wave's lanes through LDS, 28.7 with each wave's own best, every
// number of its first word by the full logarithms, 25.8 so in blocks of four waves,
// 23.1 of sixteen; 256 x 32000, a block a row, 17.1 and 13.7.)
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "vocab_row.h"

DEV_INLINE uint32_t enc_f32(float x) {
  uint32_t b = __float_as_uint(x);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// The upper word of splitmix64(z) but for its lowest bit (the last step's z >> 31
// reaches no other)
DEV_INLINE uint32_t splitmix64_upper(uint64_t z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return (uint32_t)(z >> 32);
}

// Random bits of an entry, of which the upper 24 are used.  ``at``: the entry's
// place in the sequence, rng_at() of it or of another one plus the distance
constexpr uint64_t RNG_STEP = 0xd1342543de82ef95ull;
DEV_INLINE uint64_t rng_at(int i) {
  return (uint64_t)(int64_t)i * RNG_STEP + 0x2545f4914f6cdd1dull;
}
DEV_INLINE uint32_t rng_bits(uint64_t rowkey, uint64_t at) {
  return splitmix64_upper(rowkey ^ at);
}

// Gumbel noise of 24 bits: u = (bits + 1) / 2^24.  The largest bits stand
// for the numbers between 1 - 2^-24 and 1: -log u is 2^-25 in their middle (at
// u = 1 the noise would be infinite and the entry drawn whatever its logit,
// in one row of 130 at 128256 entries).
DEV_INLINE float gumbel(uint32_t bits) {
  const float u = ((float)(bits >> 8) + 1.0f) * (1.0f / 16777216.0f);
  return -__logf(fmaxf(-__logf(u), 0x1p-25f));
}

// The same noise in seven instructions for thirty.  Over all 2^24 inputs the two
// are at most 1.91e-6 apart, and at most 2.2e-7 of 1 + the noise.
DEV_INLINE float gumbel_about(uint32_t bits) {
  const float u = ((float)(bits >> 8) + 1.0f) * (1.0f / 16777216.0f);
  const float l = -0.6931471805599453f * __builtin_amdgcn_logf(u);
  return -0.6931471805599453f * __builtin_amdgcn_logf(fmaxf(l, 0x1p-25f));
}

constexpr int SNT = 256;              // threads of a block
constexpr int SNW = SNT / 64;
constexpr int DIGIT = 2048;           // bins of a radix pass
constexpr int TOPS = SNT / 16;        // maxima that a piece leaves

// A piece's share of a row: raw softmax sums relative to m, the same at the
// temperature, and the best entry of the draw (or the largest logit).
struct alignas(8) Share {
  float m, s, st;
  float best;
  int best_i;
  int pad;
};

DEV_INLINE bool better(float v, int i, float w, int j) {
  return v > w || (v == w && i < j);
}

// x or that of the lane that CTRL names, if larger (its own where none stands)
template <int CTRL, int ROWS>
DEV_INLINE float larger_from(float x) {
  const int own = __float_as_int(x);
  return fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(
                      own, own, CTRL, ROWS, 0xf, false)));
}
// the largest of the wave's numbers; all lanes take part
DEV_INLINE float wave_largest(float x) {
  x = larger_from<0x111, 0xf>(x);        // row_shr 1, 2, 4, 8
  x = larger_from<0x112, 0xf>(x);
  x = larger_from<0x114, 0xf>(x);
  x = larger_from<0x118, 0xf>(x);
  x = larger_from<0x142, 0xa>(x);        // row_bcast 15, 31
  x = larger_from<0x143, 0xc>(x);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

template <int CTRL, int ROWS>
DEV_INLINE float plus_from(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(
                 0, __float_as_int(x), CTRL, ROWS, 0xf, ROWS == 0xf));
}
DEV_INLINE float wave_sum(float x) {
  x = plus_from<0x111, 0xf>(x);
  x = plus_from<0x112, 0xf>(x);
  x = plus_from<0x114, 0xf>(x);
  x = plus_from<0x118, 0xf>(x);
  x = plus_from<0x142, 0xa>(x);
  x = plus_from<0x143, 0xc>(x);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}
template <int CTRL, int ROWS>
DEV_INLINE int smaller_from(int x) {
  return min(x, __builtin_amdgcn_update_dpp(x, x, CTRL, ROWS, 0xf, false));
}
DEV_INLINE int wave_smallest(int x) {
  x = smaller_from<0x111, 0xf>(x);
  x = smaller_from<0x112, 0xf>(x);
  x = smaller_from<0x114, 0xf>(x);
  x = smaller_from<0x118, 0xf>(x);
  x = smaller_from<0x142, 0xa>(x);
  x = smaller_from<0x143, 0xc>(x);
  return __builtin_amdgcn_readlane(x, 63);
}

// the wave's best, in every lane
DEV_INLINE void wave_best(float& v, int& i) {
  const float most = wave_largest(v);
  i = wave_smallest(v == most ? i : 0x7fffffff);
  v = most;
}

// running maximum and softmax sums of a thread
template <bool TEMP>
struct Sums {
  float m = -INFINITY, s = 0.f, st = 0.f;
  // what a sum relative to m counts relative to c, at most 2^127: finite, so
  // that an empty sum (m = -inf) stays 0 also at a negative temperature
  DEV_INLINE static float shift(float m, float c, float inv_temp) {
    return __expf(fminf((m - c) * inv_temp, 88.f));
  }
  // c: the largest of v
  template <int N>
  DEV_INLINE void add(const float (&v)[N], float c, float inv_temp) {
    if (c > m) {
      s *= __expf(m - c);              // 0 at the first numbers
      if (TEMP) st *= shift(m, c, inv_temp);
      m = c;
    }
    if (m == -INFINITY) {              // nothing but -inf and NaN so far
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (v[j] != v[j]) {
          s = v[j];
          if (TEMP) st = v[j];
        }
      return;
    }
#pragma unroll
    for (int j = 0; j < N; ++j) s += __expf(v[j] - m);
    if (!TEMP) return;
    // (-inf, also what stands in for entries outside the row, has no mass
    // at a negative or infinite temperature either)
    if (inv_temp > 0.f) {
#pragma unroll
      for (int j = 0; j < N; ++j) st += __expf((v[j] - m) * inv_temp);
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j)
        st += v[j] == -INFINITY ? 0.f : __expf((v[j] - m) * inv_temp);
    }
  }
  // the wave's, in every lane
  DEV_INLINE void wave(float inv_temp) {
    const float c = wave_largest(m);
    // (equal also where both are -inf: the sum is 0 or NaN then)
    const float own = m == c ? 1.f : __expf(m - c);
    s = wave_sum(s * own);
    if (TEMP) st = wave_sum(m == c ? st : st * shift(m, c, inv_temp));
    m = c;
  }
};

DEV_INLINE float dec_f32(uint32_t e) {
  return __uint_as_float(e & 0x80000000u ? e ^ 0x80000000u : ~e);
}

// The draw of a thread, pruned by the best that the block's waves know of: a number
// in LDS that they raise and read in passing.
struct Draw {
  float best = -INFINITY, wbest = -INFINITY;
  int best_i = 0;
  uint32_t* known;                     // encoding of the block's best so far

  DEV_INLINE explicit Draw(uint32_t* known_) : known(known_) {}
  // before the block's waves start (a barrier is between)
  DEV_INLINE static void start(uint32_t* known) {
    if (threadIdx.x == 0) *known = enc_f32(-INFINITY);
  }

  DEV_INLINE void raise(float z) {
    wbest = wave_largest(z);
    if ((threadIdx.x & 63) == 0) atomicMax(known, enc_f32(wbest));
  }

  // v: entries i0 .. of the row, c the largest; tau: encoding that an entry
  // must reach (0: all)
  template <int N>
  DEV_INLINE void add(const float (&v)[N], float c, int i0, int V,
                      uint64_t rowkey, float inv_temp, uint32_t tau) {
    if (tau != 0 && !__any(enc_f32(c) >= tau)) return;
    wbest = fmaxf(wbest, dec_f32(*(volatile uint32_t*)known));
    uint32_t bits[N];
    {
      uint64_t at = rng_at(i0), step = RNG_STEP;
      asm("" : "+s"(step));              // (else the sums become products)
#pragma unroll
      for (int j = 0; j < N; ++j) bits[j] = rng_bits(rowkey, at), at += step;
    }
    uint32_t most = bits[0];
#pragma unroll
    for (int j = 1; j < N; ++j) most = max(most, bits[j]);
    // bits below this lose whatever the logit (all may win at a temperature that
    // is not positive, where c is no bound)
    uint32_t least = 0;
    if (inv_temp > 0.f) {
      if (tau == 0 && __all(wbest == -INFINITY)) {
        // the first words: what some entry certainly has
        float z = -INFINITY;
#pragma unroll
        for (int j = 0; j < N; ++j)
          z = fmaxf(z, __fmaf_rn(v[j], inv_temp, gumbel_about(bits[j])));
        raise(z - (1e-4f + 1e-5f * fabsf(z)));
      }
      // (an entry whose z rounds to the best one's wins by a lower index, whichever
      // wave comes first: less twice the last place of the best)
      const float bound = __fmaf_rn(fminf(fabsf(wbest), 3.4e38f), -0x1p-22f, wbest);
      const float u = __expf(-__expf(__fmaf_rn(c, inv_temp, -bound)));
      least = (uint32_t)max((int)(u * (16777216.f * (1.f - 1e-5f))) - 2, 0) << 8;
    }
    if (!__any(most >= least)) return;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (bits[j] < least || (unsigned)(i0 + j) >= (unsigned)V ||
          (tau != 0 && enc_f32(v[j]) < tau))
        continue;
      const float z = __fmaf_rn(v[j], inv_temp, gumbel(bits[j]));
      if (better(z, i0 + j, best, best_i)) best = z, best_i = i0 + j;
    }
    raise(fmaxf(best, wbest));
  }
};

// sums of a whole row (every lane of the wave gets them, after wave()); split <= 64
template <bool TEMP>
DEV_INLINE Sums<TEMP> piece_sums(const Share* share, int split) {
  const int lane = threadIdx.x & 63;
  Sums<TEMP> a;
  if (lane < split)
    a.m = share[lane].m, a.s = share[lane].s, a.st = share[lane].st;
  return a;
}
template <bool TEMP>
DEV_INLINE Sums<TEMP> row_sums(const Share* share, int split, float inv_temp) {
  Sums<TEMP> a = piece_sums<TEMP>(share, split);
  a.wave(inv_temp);
  return a;
}

// ------------------------------------------------------- radix selection
// Bins of a digit of the encoding: [shift, shift + bits).  Per row and digit
// two arrays of DIGIT words: counts of the entries with top-k's prefix, mass
// of those with top-p's.
struct alignas(8) Plan {              // where a row's two selections stand
  float cut;                          // entries below it stand at neither
  float m, target;                    // largest entry; top-p: mass to reach
  uint32_t prefix_k, prefix_p;        // digits decided so far, left-aligned
  float cnt, mass;                    // count / mass above them
  uint32_t least, most;               // encodings of the cut (0: none) and m
  int by;                             // 1: top-k, 2: top-p

  DEV_INLINE Plan(float cut_, const Sums<true>& all, float p, bool by_k,
                  bool by_p)
      : cut(cut_), m(all.m), target(p * all.st), prefix_k(0), prefix_p(0),
        cnt(0.f), mass(0.f),
        // (-0 stands below +0 in the encoding)
        least(cut_ > -INFINITY ? enc_f32(cut_ == 0.f ? -0.f : cut_) : 0u),
        most(enc_f32(all.m)), by((by_k ? 1 : 0) + (by_p ? 2 : 0)) {}
  // encoding that a kept entry reaches: the higher threshold, but no less than
  // the cut (where rounding leaves the mass in the bins short of its goal the
  // walk ends at bin 0) and no more than the largest entry (with p = 0 it
  // stops at the topmost, empty bin)
  DEV_INLINE uint32_t threshold() const {
    return min(max(max(prefix_k, prefix_p), least), most);
  }
};

// Writes that blocks on other dies read in the same launch, and such reads: past
// this die's L2
template <typename U>
DEV_INLINE void write_through(U* to, U v) {
  __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
DEV_INLINE U read_through(const U* from) {
  return __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Walks the bins from the top until the running count reaches ``need`` (or
// the running mass ``target``); bin 0 if none does.  All threads of the block
// get the bin and the sum above it.  lds: the waves' sums, the first thread
// that reaches the goal, its bin and the sum above that, each in words of its
// own: a wave may still read the thread while that thread writes its bin.
template <bool MASS, int NT>
DEV_INLINE void find_bin(const uint32_t* bins, int n, float above, float goal,
                         float* lds, int& bin, float& before) {
  // thread t has bins [t*per, +per) counted from the top
  const int per = (n + NT - 1) / NT;     // at most DIGIT / NT
  constexpr int MOST = DIGIT / NT, NW = NT / 64;
  float val[MOST], own = 0.f;
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    const int at = threadIdx.x * per + i;
    val[i] = 0.f;
    if (i < per && at < n)
      val[i] = MASS ? __uint_as_float(bins[n - 1 - at]) : (float)bins[n - 1 - at];
  }
#pragma unroll
  for (int i = 0; i < MOST; ++i) own += val[i];
  float upto = own;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float o = __shfl_up(upto, off, 64);
    if (lane >= off) upto += o;
  }
  __syncthreads();
  if (lane == 63) lds[wid] = upto;
  int* found = reinterpret_cast<int*>(lds + NW);
  if (threadIdx.x == 0) *found = NT;
  __syncthreads();
  float base = above;
  for (int w = 0; w < wid; ++w) base += lds[w];
  if (base + upto >= goal) atomicMin(found, (int)threadIdx.x);
  __syncthreads();
  const int who = *found;
  if (who == NT) {                    // short of the goal: keep all bins
    bin = 0;
    before = 0.f;
    return;
  }
  if ((int)threadIdx.x == who) {
    float run = base + upto - own, at_run = run;
    int at = per - 1;                  // the last one, if rounding hides it
    bool done = false;
#pragma unroll
    for (int i = 0; i < MOST; ++i) {
      if (done || i >= per) continue;
      at_run = run;
      run += val[i];
      if (run >= goal) at = i, done = true;
    }
    run = at_run;
    lds[NW + 1] = run;
    found[2] = max(n - 1 - (who * per + at), 0);
  }
  __syncthreads();
  bin = found[2];
  before = lds[NW + 1];
}

DEV_INLINE int digit_shift(int d) { return d == 0 ? 21 : d == 1 ? 10 : 0; }
// digits of a type: bf16 numbers have 16 bits, 11 + 5; fp32 11 + 11 + 10
template <typename T>
DEV_INLINE int digit_low(int d) {     // lowest bit of digit d
  return sizeof(T) == 2 && d == 1 ? 16 : digit_shift(d);
}
template <typename T>
DEV_INLINE int digit_bins(int d) {
  return d == 0 ? DIGIT : sizeof(T) == 2 ? 32 : d == 1 ? DIGIT : 1024;
}

// Entries below this stand at neither threshold of their row (the top of this
// file).  tops: n maxima of 16 lanes each; lds: n floats.
template <int NT = SNT>
DEV_INLINE float cut_of(const float* tops, int n, bool by_k, bool by_p, int k,
                        float p, float inv_temp, const Sums<true>& all, int V,
                        float* lds) {
  float cut = -INFINITY;
  if (by_p && inv_temp > 0.f && p > 0.f)
    cut = all.m + __logf(0.99f * (1.f - p) * all.st / V) / inv_temp;
  if (!(cut > -INFINITY)) cut = -INFINITY;   // (NaN logits)
  if (!by_k || k > n) return cut;
  // waves' maxima where they are enough, else those of 16 lanes
  const int width = k <= n / 4 ? 4 : 1, m = n / width;
  __syncthreads();
  for (int i = threadIdx.x; i < m; i += NT) {
    float t = tops[i * width];
    for (int j = 1; j < width; ++j) t = fmaxf(t, tops[i * width + j]);
    lds[i] = t;
  }
  __syncthreads();
  __shared__ float kth;
  for (int i = threadIdx.x; i < m; i += NT) {
    const float t = lds[i];
    int rank = 0;
    for (int j = 0; j < m; ++j) {
      const float o = lds[j];
      rank += o > t || (o == t && j < i);
    }
    if (rank == k - 1) kth = t;
  }
  __syncthreads();
  return fmaxf(cut, kth);
}

// The same from a wave of a block of the passes, which has the maxima in registers
// (lane l's are 4 l .. 4 l + 3 of each 256, a wave's in turn; -inf past the last):
// the k-th largest is found bit by bit, the lanes counting those that are no smaller.
// Of bf16 numbers' encodings the lower half is all sign.
template <typename T, int J>
DEV_INLINE uint32_t kth_largest(const uint32_t (&e)[J], int k) {
  uint32_t found = 0;
  for (int bit = 31; bit >= (sizeof(T) == 2 ? 16 : 0); --bit) {
    const uint32_t at = found | 1u << bit;
    int n = 0;
#pragma unroll
    for (int j = 0; j < J; ++j) n += __popcll(__ballot(e[j] >= at));
    if (n >= k) found = at;
  }
  return sizeof(T) == 2 && !(found >> 31) ? found | 0xffff : found;
}
constexpr int MOST_TOPS = 64 * TOPS / 256;     // of 256 maxima, in 64 pieces
template <typename T, int C>
DEV_INLINE uint32_t kth_of_tops(const float (&tops)[MOST_TOPS][4], int n, int k) {
  const int lane = threadIdx.x & 63;
  if (k <= n / 4) {                    // waves' maxima, as above
    uint32_t e[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      float t = tops[c][0];
#pragma unroll
      for (int w = 1; w < 4; ++w) t = fmaxf(t, tops[c][w]);
      e[c] = c * 256 + lane * 4 < n ? enc_f32(t) : 0u;
    }
    return kth_largest<T>(e, k);
  }
  if (C == 1 && n <= 64) {             // one a lane
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float o = __shfl(tops[0][w], lane / 4, 64);
      if (lane % 4 == w) t = o;
    }
    const uint32_t e[1] = {lane < n ? enc_f32(t) : 0u};
    return kth_largest<T>(e, k);
  }
  uint32_t e[4 * C];
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int w = 0; w < 4; ++w)
      e[c * 4 + w] = c * 256 + lane * 4 < n ? enc_f32(tops[c][w]) : 0u;
  return kth_largest<T>(e, k);
}
template <typename T>
DEV_INLINE float wave_cut(const float (&tops)[MOST_TOPS][4], int n, bool by_k,
                          bool by_p, int k, float p, float inv_temp,
                          const Sums<true>& all, int V) {
  float cut = -INFINITY;
  if (by_p && inv_temp > 0.f && p > 0.f)
    cut = all.m + __logf(0.99f * (1.f - p) * all.st / V) / inv_temp;
  if (!(cut > -INFINITY)) cut = -INFINITY;   // (NaN logits)
  if (!by_k || k > n) return cut;
  const uint32_t e = n <= 256 ? kth_of_tops<T, 1>(tops, n, k)
                              : kth_of_tops<T, MOST_TOPS>(tops, n, k);
  return fmaxf(cut, __uint_as_float(e >> 31 ? e ^ 0x80000000u : ~e));
}

// What the passes over a filtered row tell each other, zeros at first: the
// entries at or above the cut so far, the blocks that are through with each
// pass, whether the row's token is written, and, if the list was too short, one
// more than the entries in it.
struct RowState {
  uint32_t listed, arrived[4], done, overfull, pad;
};
constexpr int LISTED = 1024;          // entries that a row's list holds
// Up to which they are counted, one a thread, and not binned: counting takes the
// square of their number (64 x 151936, top-p 0.95 at T 0.7, 500 candidates: 65 us
// counted, 38 binned; 58 without lists).
constexpr int COUNTED = SNT;

// Whether this block is the last of its row's to come here: what the others added
// with atomics or wrote through can then be read through.  Nobody waits for
// another block.  (Such writes have arrived when their wave's counter says so.
// Fences would write back and drop this die's whole L2, under the blocks that
// still read logits: 87 us for 12.)
DEV_INLINE bool last_of_row(uint32_t* arrived, int split) {
  __shared__ bool last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    last = atomicAdd(arrived, 1u) == (uint32_t)split - 1;
  __syncthreads();
  asm volatile("" ::: "memory");
  return last;
}

// A digit's bins decide (all threads of a block)
template <int NT, typename T>
DEV_INLINE void walk_bins(Plan& plan, const uint32_t* cnt, const float* mass,
                          int digit, int k, float* lds) {
  const int bins = digit_bins<T>(digit), low = digit_low<T>(digit);
  int bin;
  float before;
  if (plan.by & 1) {
    find_bin<false, NT>(cnt, bins, plan.cnt, (float)k, lds, bin, before);
    plan.prefix_k |= (uint32_t)bin << low, plan.cnt = before;
  }
  if (plan.by & 2) {
    find_bin<true, NT>(reinterpret_cast<const uint32_t*>(mass), bins, plan.mass,
                       plan.target, lds, bin, before);
    plan.prefix_p |= (uint32_t)bin << low, plan.mass = before;
  }
}

// The row's bins, to which the other blocks added, into LDS: whole lines, all on
// their way at once.  No load stands under a condition: its wait would stand there
// too, and with sixteen waits in turn for what comes past the L2 64 x 50257 fp32,
// top-p 0.8 at T 0.7, took 62 us (the three plan launches before it 61), 56 now.
template <typename T>
DEV_INLINE void read_bins(int digit, const uint32_t* h, uint32_t* cnt,
                          float* mass) {
  constexpr int PER = DIGIT / SNT;
  const int last = digit_bins<T>(digit) - 1;
  uint32_t c[PER], m[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int at = min(i * SNT + (int)threadIdx.x, last);
    c[i] = read_through(&h[at]);
    m[i] = read_through(&h[DIGIT + at]);
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    cnt[i * SNT + threadIdx.x] = c[i];
    mass[i * SNT + threadIdx.x] = __uint_as_float(m[i]);
  }
  __syncthreads();
}

// the block's best entry, in every wave
DEV_INLINE void block_best(float& best, int& best_i, Share* part) {
  wave_best(best, best_i);
  if ((threadIdx.x & 63) == 0)
    part[threadIdx.x >> 6].best = best, part[threadIdx.x >> 6].best_i = best_i;
  __syncthreads();
  best = part[threadIdx.x % SNW].best, best_i = part[threadIdx.x % SNW].best_i;
  wave_best(best, best_i);
}

// ------------------------------------------------------------- one pass
// MODE 0: sums and draw in one (no filter); 1: sums (and the largest logit)
// of a filtered row; 2: its draw.
//
// One thread's part of a pass over the groups [first, first + NT) of every
// ``stride``.  Every lane of a wave takes part in every round (the draw votes).
// Rounds of whole words only run without a look at the row's ends, the next
// word under way; the first, the last and the ones past them take the long form.
template <int MODE, int NT, typename T>
DEV_INLINE void walk(const VocabRow<T>& r, int first, int stride, bool greedy,
                     float inv_temp, uint64_t rowkey, uint32_t tau,
                     Sums<MODE == 1>& sums, Draw& d) {
  constexpr int VEC = VocabRow<T>::VEC;
  const int groups = r.groups();
  auto round = [&](const float (&v)[VEC], int i0) {
    float c = v[0];
#pragma unroll
    for (int j = 1; j < VEC; ++j) c = fmaxf(c, v[j]);
    if (MODE != 2) sums.add(v, c, inv_temp);
    if (MODE == 1 || greedy) {
      if (c > d.best) {
        d.best = c;
#pragma unroll
        for (int j = VEC - 1; j >= 0; --j)
          if (v[j] == c) d.best_i = i0 + j;
      }
    } else {
      d.add(v, c, i0, r.V, rowkey, inv_temp, tau);
    }
  };
  // groups [1, whole) are whole words
  const int whole = r.lead + (groups - 1) * VEC > r.V ? groups - 1 : groups;
  auto inside = [&](int g0) { return g0 > 0 && g0 + NT <= whole; };
  int g0 = first;
  while (g0 < groups) {
    if (inside(g0)) {
      typename VocabRow<T>::Word next = r.word(g0 + threadIdx.x);
      do {
        const typename VocabRow<T>::Word w = next;
        if (inside(g0 + stride)) next = r.word(g0 + stride + threadIdx.x);
        float v[VEC];
        r.numbers(w, v);
        round(v, r.first(g0 + threadIdx.x));
        g0 += stride;
      } while (inside(g0));
    } else {
      const int g = g0 + threadIdx.x;
      float v[VEC];
      if (g < groups) {
        r.load(g, v);
      } else {
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = -INFINITY;
      }
      round(v, r.first(g));
      g0 += stride;
    }
  }
}

DEV_INLINE RowState* row_state(uint32_t* hist, int hist_words, long row) {
  return reinterpret_cast<RowState*>(hist + (row + 1) * hist_words) - 1;
}

// the row's token from the pieces' shares (the first wave)
template <typename T>
DEV_INLINE void write_row(int64_t* out_tokens, float* out_logprobs,
                          const Share* share, const VocabRow<T>& r, long row,
                          int split) {
  const int lane = threadIdx.x;
  if (lane >= 64) return;
  const Sums<false> a = row_sums<false>(share, split, 1.f);
  float best = lane < split ? read_through(&share[lane].best) : -INFINITY;
  int best_i = lane < split ? read_through(&share[lane].best_i) : 0x7fffffff;
  wave_best(best, best_i);
  if (lane == 0) {
    out_tokens[row] = best_i;
    out_logprobs[row] = (float)r.x[best_i] - (a.m + __logf(a.s));
  }
}

template <typename T, int MODE, int NT = SNT>
__global__ __launch_bounds__(NT) void sample_pass_kernel(
    int64_t* __restrict__ out_tokens, float* __restrict__ out_logprobs,
    Share* __restrict__ share, float* __restrict__ tops,
    uint32_t* __restrict__ hist, int hist_words,
    const Plan* __restrict__ plans, const T* __restrict__ logits,
    const float* __restrict__ temperature, uint64_t seed,
    const long long* __restrict__ seed_ptr, int V, int split) {
  __shared__ Share part[(NT / 64)];
  const long row = blockIdx.x / split;
  const int piece = blockIdx.x % split;
  if (seed_ptr != nullptr) seed = (uint64_t)*seed_ptr;
  const VocabRow<T> r(logits + row * V, V);
  const float temp = temperature[row];
  const bool greedy = temp == 0.f;
  RowState* state = row_state(hist, hist_words, row);
  if (MODE == 2 && state->done) return;
  const float inv_temp = greedy ? 1.f : 1.0f / temp;
  const uint64_t rowkey = seed + (uint64_t)row * 0x9e3779b97f4a7c15ull;
  const uint32_t tau = MODE == 2 ? plans[row].threshold() : 0;
  if (MODE == 1) {                    // the bins and the state start at 0
    uint32_t* h = hist + row * hist_words;
    for (int i = piece * NT + threadIdx.x; i < hist_words; i += split * NT)
      h[i] = 0;
  }

  __shared__ uint32_t known;
  if (MODE != 1 && !greedy) {         // (who draws)
    Draw::start(&known);
    __syncthreads();
  }
  Sums<MODE == 1> sums;
  Draw d(&known);
  walk<MODE, NT>(r, piece * NT, split * NT, greedy, inv_temp, rowkey, tau, sums,
             d);
  if (MODE == 1) {                    // largest of each 16 lanes
    float t = d.best;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) t = fmaxf(t, __shfl_xor(t, off, 64));
    if (threadIdx.x % 16 == 0)
      tops[(row * split + piece) * TOPS + threadIdx.x / 16] = t;
  }
  if (MODE != 2) sums.wave(inv_temp);
  wave_best(d.best, d.best_i);
  if ((threadIdx.x & 63) == 0)
    part[threadIdx.x >> 6] = {sums.m, sums.s, sums.st, d.best, d.best_i, 0};
  __syncthreads();
  if (threadIdx.x < 64) {               // the waves' shares, each once
    const Share o = part[threadIdx.x % (NT / 64)];
    const bool one = threadIdx.x < (NT / 64);
    sums.m = o.m, sums.s = one ? o.s : 0.f, sums.st = one ? o.st : 0.f;
    if (MODE != 2) sums.wave(inv_temp);
    d.best = o.best, d.best_i = o.best_i;
    wave_best(d.best, d.best_i);
  }
  if (threadIdx.x == 0) {
    Share* out = share + row * split + piece;
    if (MODE != 2) out->m = sums.m, out->s = sums.s, out->st = sums.st;
    write_through(&out->best, d.best);
    write_through(&out->best_i, d.best_i);
  }
  if (MODE == 2 && last_of_row(&state->arrived[3], split))
    write_row(out_tokens, out_logprobs, share + row * split, r, row, split);
}

template <typename T>
__global__ __launch_bounds__(64) void sample_merge_kernel(
    int64_t* __restrict__ out_tokens, float* __restrict__ out_logprobs,
    const Share* __restrict__ share, const T* __restrict__ logits, int V,
    int split) {
  const long row = blockIdx.x;
  write_row(out_tokens, out_logprobs, share + row * split,
            VocabRow<T>(logits + row * V, V), row, split);
}

// an entry into the bins of a digit, if it shares the digits before it with a
// threshold
template <typename T>
DEV_INLINE void add_entry(float v, int digit, const Plan& plan, float inv_temp,
                          uint32_t* cnt, float* mass) {
  const uint32_t above = digit == 0 ? 0u
      : 0xFFFFFFFFu << digit_low<T>(digit - 1);
  const uint32_t e = enc_f32(v);
  const uint32_t bin = (e >> digit_low<T>(digit)) & (digit_bins<T>(digit) - 1);
  if ((plan.by & 1) && (e & above) == plan.prefix_k) atomicAdd(&cnt[bin], 1u);
  if ((plan.by & 2) && (e & above) == plan.prefix_p && v != -INFINITY)
    atomicAdd(&mass[bin], __expf((v - plan.m) * inv_temp));
}

// a thread's entries of the groups [first, ..) of every ``stride`` into the
// bins of a digit
template <typename T>
DEV_INLINE void fill_bins(const VocabRow<T>& r, int first, int stride,
                          int digit, const Plan& plan, float inv_temp,
                          uint32_t* cnt, float* mass) {
  constexpr int VEC = VocabRow<T>::VEC;
  const int groups = r.groups();
  for (int g = first + threadIdx.x; g < groups; g += stride) {
    float v[VEC];
    r.load(g, v);
    const int i0 = r.first(g);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      if (v[j] < plan.cut || (unsigned)(i0 + j) >= (unsigned)r.V) continue;
      add_entry<T>(v[j], digit, plan, inv_temp, cnt, mass);
    }
  }
}

// both selections by one block; ``fill(digit)`` adds the entries to its bins
template <int NT, typename T, typename F>
DEV_INLINE void select_alone(Plan& plan, int k, uint32_t* cnt, float* mass,
                             float* lds, F fill) {
  for (int digit = 0; digit < (sizeof(T) == 2 ? 2 : 3); ++digit) {
    const int bins = digit_bins<T>(digit);
    for (int i = threadIdx.x; i < bins; i += NT) cnt[i] = 0, mass[i] = 0.f;
    __syncthreads();
    fill(digit);
    __syncthreads();
    walk_bins<NT, T>(plan, cnt, mass, digit, k, lds);
    __syncthreads();                    // the bins were read
  }
}

// entries into the row's bins of a digit: ``fill`` adds them to the block's own
template <typename T, typename F>
DEV_INLINE void add_bins(int digit, uint32_t* cnt, float* mass, uint32_t* h,
                         F fill) {
  const int bins = digit_bins<T>(digit);
  for (int i = threadIdx.x; i < bins; i += SNT) cnt[i] = 0, mass[i] = 0.f;
  __syncthreads();
  fill();
  __syncthreads();
  float* hm = reinterpret_cast<float*>(h + DIGIT);
  for (int i = threadIdx.x; i < bins; i += SNT) {
    if (cnt[i]) atomicAdd(&h[i], cnt[i]);
    if (mass[i] != 0.f) atomicAdd(&hm[i], mass[i]);
  }
}

// The cut, and what stands at or above it: into a list if that is little, into the
// first digit's bins else.  The row's last block then has the thresholds and the
// token from the list (by counting, for each entry, what is no smaller), or the
// first digit of the thresholds.  Every block finds the same cut: a launch for it
// between the passes takes longer.
//
// How much it is, the maxima of the lanes' groups tell: of g groups, n entries in
// random order leave a share of exp(-n / g) without one.  If they are not in random
// order and the list is too short, the pieces whose entries it does not hold add
// them to the bins, the last block those that it does, and the row goes on like
// one without a list (64 x 151936, top-p 0.95 at T 0.7, 4000 candidates side by
// side: 66 us; 183 with one block for such a row's passes, 69 without lists).
// What bounds it: a chain of short waits.  So what can be read early is read at once:
// the maxima with the sums, the whole list with its length, the winner's logit with
// the list; and one wave of a block searches the cut, whose counts are scalar work
// that the sixteen waves of a CU would take turns at.  (64 x 151936, T 0.7, k 50, p
// 0.9, all launches: 26.7 us as it was, 25.3 read early, 24.9 with half of the bits of
// bf16 maxima, 24.1 with one wave; 128 rows 35.1 and 31.8, one of 128256 18.6 and
// 16.4, 32 x 128256 fp32, k 200, 53.6 and 46.  The list's logits asked for before the
// cut, or two bits of it a step: no gain, 25.5 for 24.9.)
template <typename T>
__global__ __launch_bounds__(SNT) void sample_select_kernel(
    int64_t* __restrict__ out_tokens, float* __restrict__ out_logprobs,
    Plan* __restrict__ plans, uint32_t* __restrict__ hist, int hist_words,
    float* __restrict__ list_v, int* __restrict__ list_i,
    const Share* __restrict__ share, const float* __restrict__ tops,
    const T* __restrict__ logits, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p,
    uint64_t seed, int V, int split) {
  constexpr int VEC = VocabRow<T>::VEC;
  __shared__ alignas(16) uint32_t cnt[DIGIT];
  __shared__ alignas(16) float mass[DIGIT];
  __shared__ float lds[SNW + 4];
  __shared__ Share part[SNW];
  __shared__ int found;
  __shared__ uint32_t base, thr[2];
  const long row = blockIdx.x / split;
  const int piece = blockIdx.x % split;
  const VocabRow<T> r(logits + row * V, V);
  const int k = top_k[row];
  const float temp = temperature[row], p = top_p[row];
  const bool by_k = temp != 0.f && k > 0 && k < V;
  const bool by_p = temp != 0.f && p < 1.0f;
  const float inv_temp = temp == 0.f ? 1.f : 1.0f / temp;
  uint32_t* h = hist + row * hist_words;
  RowState* state = row_state(hist, hist_words, row);
  share += row * split;
  list_v += row * LISTED, list_i += row * LISTED;
  // The maxima come with the pieces' sums, not once for the cut and once more for
  // the list's length: the block is a chain of such waits.
  // (behind them: a row at a temperature of 0 waits for the sums alone)
  Sums<true> all = piece_sums<true>(share, split);
  const int most = split * TOPS;
  float top[MOST_TOPS][4];
  const int top_at = (threadIdx.x & 63) * 4;            // (four lanes a piece)
  auto read_tops = [&](int c) {
    const int at = c * 256 + top_at;
#pragma unroll
    for (int w = 0; w < 4; ++w)
      top[c][w] = tops[row * most + (at < most ? at : 0) + w];
  };
  read_tops(0);
  if (most > 256) {
#pragma unroll
    for (int c = 1; c < MOST_TOPS; ++c) read_tops(c);
  } else {
#pragma unroll
    for (int c = 1; c < MOST_TOPS; ++c)
      top[c][0] = top[c][1] = top[c][2] = top[c][3] = -INFINITY;
  }
  all.wave(inv_temp);
  if (!by_k && !by_p) {
    if (piece != 0) return;
    if (threadIdx.x == 0) plans[row] = Plan(-INFINITY, all, p, false, false);
    if (temp == 0.f) {                  // the first pass found it
      write_row(out_tokens, out_logprobs, share, r, row, split);
      if (threadIdx.x == 0) state->done = 1;
    }
    return;
  }
  // (one wave looks: sixteen a CU would take turns at the same scalar counts)
  if (threadIdx.x < 64) {
#pragma unroll
    for (int i = 0; i < MOST_TOPS; ++i)
#pragma unroll
      for (int w = 0; w < 4; ++w)
        if (i * 256 + top_at >= most) top[i][w] = -INFINITY;
    const float c = wave_cut<T>(top, most, by_k, by_p, k, p, inv_temp, all, V);
    // (a list needs numbers that add up)
    bool list = c > -INFINITY && inv_temp > 0.f && fabsf(all.m) < INFINITY &&
                all.st < INFINITY;
    if (list) {
      int with = 0;
#pragma unroll
      for (int i = 0; i < MOST_TOPS; ++i) {
        if (i * 256 >= most) break;
#pragma unroll
        for (int w = 0; w < 4; ++w) with += __popcll(__ballot(top[i][w] >= c));
      }
      list = with <= most * (1.f - __expf(-0.7f * LISTED / most));
    }
    if (threadIdx.x == 0) lds[0] = c, found = list ? 0 : -1;
  }
  __syncthreads();
  const float cut = lds[0];
  const bool listing = found == 0;
  Plan plan(cut, all, p, by_k, by_p);
  bool to_bins = !listing;
  if (listing) {
    int* own_i = reinterpret_cast<int*>(cnt);
    float* own_v = mass;
    __syncthreads();                    // (found was read)
    const int groups = r.groups();
    for (int g = piece * SNT + threadIdx.x; g < groups; g += split * SNT) {
      if (*(volatile int*)&found > LISTED) break;
      float v[VEC];
      r.load(g, v);
      float c = v[0];
#pragma unroll
      for (int j = 1; j < VEC; ++j) c = fmaxf(c, v[j]);
      if (c < cut) continue;
      const int i0 = r.first(g);
#pragma unroll
      for (int j = 0; j < VEC; ++j)
        if (v[j] >= cut) {              // (-inf stands outside the row)
          const int at = atomicAdd(&found, 1);
          if (at < LISTED) own_v[at] = v[j], own_i[at] = i0 + j;
        }
    }
    __syncthreads();
    const int n = min(found, LISTED + 1);
    if (threadIdx.x == 0) {
      base = n ? atomicAdd(&state->listed, (uint32_t)n) : 0;
      // (only the first one past the end: what comes later starts behind it)
      if (base <= LISTED && base + n > LISTED)
        write_through(&state->overfull, base + 1);
    }
    __syncthreads();
    if (base + n <= LISTED) {
      for (int t = threadIdx.x; t < n; t += SNT) {
        write_through(&list_v[base + t], own_v[t]);
        write_through(&list_i[base + t], own_i[t]);
      }
    } else if (n <= LISTED) {           // all that it has are in its own list
      float v[LISTED / SNT];
#pragma unroll
      for (int i = 0; i < LISTED / SNT; ++i)
        v[i] = own_v[i * SNT + threadIdx.x];
      __syncthreads();                  // (the list is where the bins will be)
      add_bins<T>(0, cnt, mass, h, [&] {
#pragma unroll
        for (int i = 0; i < LISTED / SNT; ++i)
          if (i * SNT + (int)threadIdx.x < n)
            add_entry<T>(v[i], 0, plan, inv_temp, cnt, mass);
      });
    } else {
      to_bins = true;
    }
  }
  if (to_bins)
    add_bins<T>(0, cnt, mass, h, [&] {
      fill_bins(r, piece * SNT, split * SNT, 0, plan, inv_temp, cnt, mass);
    });
  if (!last_of_row(&state->arrived[0], split)) return;

  // this thread's entries of the list and how many there are, all on their way at
  // once
  float own[LISTED / SNT];
  int own_at[LISTED / SNT];
#pragma unroll
  for (int i = 0; i < LISTED / SNT; ++i) {
    own[i] = read_through(&list_v[i * SNT + threadIdx.x]);
    own_at[i] = read_through(&list_i[i * SNT + threadIdx.x]);
  }
  const int overfull = read_through(&state->overfull);
  const int listed = read_through(&state->listed);
  auto each = [&](int n, auto take) {
#pragma unroll
    for (int i = 0; i < LISTED / SNT; ++i)
      if (i * SNT + (int)threadIdx.x < n) take(own_at[i], own[i]);
  };
  if (!listing || overfull) {
    read_bins<T>(0, h, cnt, mass);
    if (overfull) {
      each(overfull - 1, [&](int, float v) {
        add_entry<T>(v, 0, plan, inv_temp, cnt, mass);
      });
      __syncthreads();
    }
    walk_bins<SNT, T>(plan, cnt, mass, 0, k, lds);
    if (threadIdx.x == 0) plans[row] = plan;
    return;
  }
  const uint64_t rowkey = seed + (uint64_t)row * 0x9e3779b97f4a7c15ull;
  if (listed > COUNTED) {
    select_alone<SNT, T>(plan, k, cnt, mass, lds, [&](int digit) {
      each(listed, [&](int, float v) {
        add_entry<T>(v, digit, plan, inv_temp, cnt, mass);
      });
    });
  } else {
    // (four at a time; what fills up is no larger than any and weighs nothing)
    const int t = threadIdx.x;
    const uint32_t e = t < listed ? enc_f32(own[0]) : 0u;
    cnt[t] = e;
    mass[t] = t < listed ? __expf((own[0] - all.m) * inv_temp) : 0.f;
    if (t == 0) thr[0] = thr[1] = 0;
    __syncthreads();
    if (t < listed) {
      int count = 0;
      float sum = 0.f;
      for (int j = 0; j < listed; j += 4) {
        const uint4 ej = *reinterpret_cast<const uint4*>(&cnt[j]);
        const float4 wj = *reinterpret_cast<const float4*>(&mass[j]);
        count += (ej.x >= e) + (ej.y >= e) + (ej.z >= e) + (ej.w >= e);
        sum += (ej.x >= e ? wj.x : 0.f) + (ej.y >= e ? wj.y : 0.f) +
               (ej.z >= e ? wj.z : 0.f) + (ej.w >= e ? wj.w : 0.f);
      }
      if (by_k && count >= k) atomicMax(&thr[0], e);
      if (by_p && sum >= plan.target) atomicMax(&thr[1], e);
    }
    __syncthreads();
    plan.prefix_k = thr[0], plan.prefix_p = thr[1];
  }
  const uint32_t tau = plan.threshold();
  float best = -INFINITY, best_v = 0.f;
  int best_i = 0;
  each(listed, [&](int i, float v) {
    if (enc_f32(v) < tau) return;
    const float z = __fmaf_rn(v, inv_temp, gumbel(rng_bits(rowkey, rng_at(i))));
    if (better(z, i, best, best_i)) best = z, best_i = i, best_v = v;
  });
  const float own_best = best;
  const int own_i = best_i;
  block_best(best, best_i, part);
  // the thread that has the entry has its logit too; without one the row is read
  const bool none = !(best > -INFINITY);
  if (none && threadIdx.x == 0) best_v = (float)r.x[best_i];
  if (none ? threadIdx.x == 0 : own_best == best && own_i == best_i) {
    out_tokens[row] = best_i;
    out_logprobs[row] = best_v - (all.m + __logf(all.s));
    state->done = 1;
  }
}

// the digits after the first, of rows without a list
template <typename T>
__global__ __launch_bounds__(SNT) void sample_digit_kernel(
    Plan* __restrict__ plans, uint32_t* __restrict__ hist, int hist_words,
    const T* __restrict__ logits, const float* __restrict__ temperature,
    const int* __restrict__ top_k, int digit, int V, int split) {
  __shared__ uint32_t cnt[DIGIT];
  __shared__ float mass[DIGIT];
  __shared__ float lds[SNW + 4];
  const long row = blockIdx.x / split;
  RowState* state = row_state(hist, hist_words, row);
  if (state->done) return;
  Plan plan = plans[row];
  if (plan.by == 0) return;
  uint32_t* h = hist + row * hist_words + digit * 2 * DIGIT;
  const VocabRow<T> r(logits + row * V, V);
  const int piece = blockIdx.x % split;
  const float inv_temp = 1.0f / temperature[row];
  add_bins<T>(digit, cnt, mass, h, [&] {
    fill_bins(r, piece * SNT, split * SNT, digit, plan, inv_temp, cnt, mass);
  });
  if (!last_of_row(&state->arrived[digit], split)) return;
  read_bins<T>(digit, h, cnt, mass);
  walk_bins<SNT, T>(plan, cnt, mass, digit, top_k[row], lds);
  if (threadIdx.x == 0) plans[row] = plan;
}

// ------------------------------------------------------------- short rows
// The same steps with one block per row, in one launch: of a short row the
// steps are shorter than the launches of the pieces and plans.
template <typename T, bool FILTER, int NT>
__global__ __launch_bounds__(NT) void sample_row_kernel(
    int64_t* __restrict__ out_tokens, float* __restrict__ out_logprobs,
    const T* __restrict__ logits, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p,
    uint64_t seed, const long long* __restrict__ seed_ptr, int V) {
  constexpr int NW = NT / 64, NTOPS = NT / 16;
  __shared__ Share part[NW];
  __shared__ float lds[NTOPS], tops[FILTER ? NTOPS : 1];
  __shared__ uint32_t cnt[FILTER ? DIGIT : 1];
  __shared__ float mass[FILTER ? DIGIT : 1];
  const long row = blockIdx.x;
  if (seed_ptr != nullptr) seed = (uint64_t)*seed_ptr;
  const VocabRow<T> r(logits + row * V, V);
  const float temp = temperature[row];
  const bool greedy = temp == 0.f;
  const float inv_temp = greedy ? 1.f : 1.0f / temp;
  const uint64_t rowkey = seed + (uint64_t)row * 0x9e3779b97f4a7c15ull;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;

  __shared__ uint32_t known;
  Draw::start(&known);
  if (!FILTER && !greedy) __syncthreads();   // (with a filter others are between)
  Sums<FILTER> sums;
  Draw d(&known);
  walk<FILTER ? 1 : 0, NT>(r, 0, NT, greedy, inv_temp, rowkey, 0u, sums, d);
  if (FILTER) {                       // largest of each 16 lanes
    float t = d.best;
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) t = fmaxf(t, __shfl_xor(t, off, 64));
    if (threadIdx.x % 16 == 0) tops[threadIdx.x / 16] = t;
  }
  sums.wave(inv_temp);
  wave_best(d.best, d.best_i);
  if (lane == 0) part[wid] = {sums.m, sums.s, sums.st, d.best, d.best_i, 0};
  __syncthreads();
  {                                   // of the whole row, in every thread
    const Share& o = part[lane % NW];
    sums.m = o.m;                       // (every wave's share once)
    sums.s = lane < NW ? o.s : 0.f, sums.st = lane < NW ? o.st : 0.f;
    sums.wave(inv_temp);
    d.best = o.best, d.best_i = o.best_i;
    wave_best(d.best, d.best_i);
  }
  if constexpr (FILTER) {
    if (!greedy) {
      const int k = top_k[row];
      const float p = top_p[row];
      const bool by_k = k > 0 && k < V, by_p = p < 1.0f;
      uint32_t tau = 0;
      if (by_k || by_p) {
        Plan plan(cut_of<NT>(tops, NTOPS, by_k, by_p, k, p, inv_temp, sums, V, lds),
                  sums, p, by_k, by_p);
        select_alone<NT, T>(plan, k, cnt, mass, lds, [&](int digit) {
          fill_bins(r, 0, NT, digit, plan, inv_temp, cnt, mass);
        });
        tau = plan.threshold();
      }
      Draw pick(&known);              // (the first walk did not raise it)
      Sums<false> none;
      walk<2, NT>(r, 0, NT, false, inv_temp, rowkey, tau, none, pick);
      wave_best(pick.best, pick.best_i);
      __syncthreads();                // the shares were read
      if (lane == 0) part[wid].best = pick.best, part[wid].best_i = pick.best_i;
      __syncthreads();
      d.best = part[lane % NW].best, d.best_i = part[lane % NW].best_i;
      wave_best(d.best, d.best_i);
    }
  }
  if (threadIdx.x == 0) {
    out_tokens[row] = d.best_i;
    out_logprobs[row] = (float)r.x[d.best_i] - (sums.m + __logf(sums.s));
  }
}

template <typename T>
static void launch_sample(torch::Tensor& out_tokens,
                          torch::Tensor& out_logprobs,
                          const torch::Tensor& logits,
                          const torch::Tensor& temperature,
                          const torch::Tensor& top_k,
                          const torch::Tensor& top_p, uint64_t seed,
                          const long long* seed_ptr, bool no_filter) {
  const long N = logits.size(0);
  const int V = logits.size(1);
  if (N == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  // Rows in one launch, a block each, while that is no longer than the pieces and
  // their passes.  Without a filter: with few rows up to 16384 numbers (64 x 16000
  // bf16 9.1 us, in pieces 10.0), with a block for most CUs up to 65536 (256 x 50257
  // 18.4 and 20.7).  With one: up to 32768.  Pieces are quicker from there down to
  // 24000 (fp32 9000) with both filters (64 x 24000 34.7 us, in pieces 20.1, 64 x
  // 16000 32.2 and 41.1; fp32 64 x 9000 37.7 and 21.3), but not with top-p 0.95 alone
  // (64 x 24000 35.3 and 39.3, 256 x 32000 41.8 and 56.8, fp32 54.4 and 81.9) nor at a
  // temperature of 0, where nothing is selected (6.9 and 16.6).  What stays dearer
  // than a block a row is the draw at a temperature of 0 without a filter from 16384
  // numbers on, 10.3 us for 6.8: the temperature is on the device, and at 1 the pieces
  // take no more.
  // A block of 1024 threads takes rows of more than one round of 256 words (64 x
  // 9000 both filters 30.5 us, with 256 threads 35.1; 64 x 32000 36.4 and 65.5); where
  // there are more rows than CUs, 256 threads take them up to ten rounds (512 x
  // 9000 39.7 us, with 1024 threads 59.9; 512 x 24000 65.7 and 65.4).
  auto rows = [&](auto kern, int threads) {
    kern<<<dim3((unsigned)N), dim3(threads), 0, stream>>>(
        out_tokens.data_ptr<int64_t>(), out_logprobs.data_ptr<float>(),
        (const T*)logits.data_ptr(), temperature.data_ptr<float>(),
        top_k.data_ptr<int>(), top_p.data_ptr<float>(), seed, seed_ptr, V);
    HIP_CHECK_KERNEL();
  };
  const long words = (V + VocabRow<T>::VEC - 1) / VocabRow<T>::VEC;
  const long most = !no_filter ? 32768 : N >= 192 ? 65536 : 16384;
  if (V <= most) {
    if (words <= (N > 256 ? 2560 : 256)) {
      no_filter ? rows(sample_row_kernel<T, false, 256>, 256)
                : rows(sample_row_kernel<T, true, 256>, 256);
    } else {
      no_filter ? rows(sample_row_kernel<T, false, 1024>, 1024)
                : rows(sample_row_kernel<T, true, 1024>, 1024);
    }
    return;
  }
  // Pieces of a row, 1024 threads a CU in all.  With a filter blocks of 256 (with 512,
  // 768, 1024, 1536 and 2048 of them 64 x 151936 with both filters takes 29.3, 27.9,
  // 27.6, 31.4, 36.9 us, with top-p 0.95 alone 69, 64, 64, 65, 77; 24 and 61 with 1024
  // since the candidates' kernel waits less), none under two rounds of 256 words.
  // Without one the largest blocks, whose waves share what they know, that fill 7/8
  // of the chip or of the 2048 threads that a CU holds and have three rounds in two
  // blocks (128 x 128256 in blocks of 256, 512 and 1024: 25.8, 24.5 and 23.1; 100 x
  // 128256 in 1100, 500 and 500: 24.9, 22.3, 22.1, but in 300 of 1024 31.5; 200 x
  // 128256 in 1200 of 256, 1000 of 512 and 200 of 1024 35.8, 33.3, 36.9; 100 x 50257
  // in 1100 of 256, 500 of 512, 500 of 1024 16.0, 14.5, 16).
  int nt = SNT, split = 0;
  if (no_filter) {
    const int most_blocks[][2] = {{1024, 256}, {1024, 512}, {512, 512},
                                  {512, 1024}, {256, 1024}};
    for (const auto& o : most_blocks) {
      const long each = o[1] / N;
      if (each < 1 || each > 64 || each * N * 8 < o[1] * 7L ||
          words * 2 < each * o[0] * 3L)
        continue;
      nt = o[0], split = (int)each;
      break;
    }
    if (split == 0 && N > 256) {
      nt = 512;
      split = (int)std::max<long>(
          1, std::min<long>((1024 + N - 1) / N, words / 1024));
    }
  }
  if (split == 0)
    split = (int)std::max<long>(
        1, std::min<long>({64, (1024 + N - 1) / N, words / (2 * SNT)}));
  const int digits = sizeof(T) == 2 ? 2 : 3;
  const int hist_words =
      no_filter ? 0 : digits * 2 * DIGIT + (int)sizeof(RowState) / 4;
  // per row: the pieces' shares and maxima, the plan, the bins and the state, the
  // list.  From the caching allocator: a block per call and stream, also while a
  // graph is captured
  const long share_words = (long)split * (sizeof(Share) / 4);
  const long row_words =
      no_filter ? share_words
                : share_words + split * TOPS + sizeof(Plan) / 4 + hist_words +
                      2 * LISTED;
  auto ws = torch::empty({N * row_words}, logits.options().dtype(torch::kInt32));
  int* w = ws.data_ptr<int>();
  Share* share = reinterpret_cast<Share*>(w);
  Plan* plans = reinterpret_cast<Plan*>(w + N * share_words);
  float* tops = reinterpret_cast<float*>(plans + N);
  uint32_t* hist = reinterpret_cast<uint32_t*>(tops + N * split * TOPS);
  float* list_v = reinterpret_cast<float*>(hist + N * hist_words);
  int* list_i = reinterpret_cast<int*>(list_v + N * LISTED);
  int64_t* tokens = out_tokens.data_ptr<int64_t>();
  float* logprobs = out_logprobs.data_ptr<float>();
  const T* x = (const T*)logits.data_ptr();
  const float* temp = temperature.data_ptr<float>();
  TORCH_CHECK(N * split < (1L << 31), "too many rows");
  const dim3 grid((unsigned)(N * split)), block(nt);
  const int* k = top_k.data_ptr<int>();
  auto pass = [&](auto kern) {
    kern<<<grid, block, 0, stream>>>(tokens, logprobs, share, tops, hist,
                                     hist_words, plans, x, temp, seed, seed_ptr,
                                     V, split);
  };
  if (no_filter) {
    if (nt == 1024) pass(sample_pass_kernel<T, 0, 1024>);
    else if (nt == 512) pass(sample_pass_kernel<T, 0, 512>);
    else pass(sample_pass_kernel<T, 0>);
    sample_merge_kernel<T><<<dim3(N), dim3(64), 0, stream>>>(
        tokens, logprobs, share, x, V, split);
  } else {
    pass(sample_pass_kernel<T, 1>);
    sample_select_kernel<T><<<grid, block, 0, stream>>>(
        tokens, logprobs, plans, hist, hist_words, list_v, list_i, share, tops,
        x, temp, k, top_p.data_ptr<float>(), seed, V, split);
    for (int d = 1; d < digits; ++d)
      sample_digit_kernel<T><<<grid, block, 0, stream>>>(
          plans, hist, hist_words, x, temp, k, d, V, split);
    pass(sample_pass_kernel<T, 2>);
  }
  HIP_CHECK_KERNEL();
}

void sample(torch::Tensor out_tokens, torch::Tensor out_logprobs,
            torch::Tensor logits, torch::Tensor temperature,
            torch::Tensor top_k, torch::Tensor top_p, int64_t seed,
            bool no_filter, torch::Tensor seed_dev /* optional (1,) i64 */) {
  TORCH_CHECK(logits.is_cuda() && logits.dim() == 2 && logits.is_contiguous());
  TORCH_CHECK(out_tokens.dtype() == torch::kInt64);
  TORCH_CHECK(out_logprobs.dtype() == torch::kFloat32);
  TORCH_CHECK(temperature.dtype() == torch::kFloat32);
  TORCH_CHECK(top_k.dtype() == torch::kInt32);
  TORCH_CHECK(top_p.dtype() == torch::kFloat32);
  // the device seed counts for unfiltered rows only
  const long long* sp = no_filter && seed_dev.defined() && seed_dev.numel() > 0
                            ? (const long long*)seed_dev.data_ptr<int64_t>()
                            : nullptr;
  if (logits.dtype() == torch::kBFloat16)
    launch_sample<bf16_t>(out_tokens, out_logprobs, logits, temperature, top_k,
                          top_p, (uint64_t)seed, sp, no_filter);
  else if (logits.dtype() == torch::kFloat32)
    launch_sample<float>(out_tokens, out_logprobs, logits, temperature, top_k,
                         top_p, (uint64_t)seed, sp, no_filter);
  else
    TORCH_CHECK(false, "sample: dtype must be bf16 or fp32");
}
