// Token selection on the device: greedy argmax, or the reference's processor
// chain temperature -> top-k -> top-p -> multinomial
// (tiny_llm/pipeline/pipeline.cpp:156-164) without sorting the vocabulary.
//
// What the chain computes, written for a row sorted by descending logit
// (tiny_llm/logit_processors/sort_processors.cpp:54-142, sample_processors.cpp:7-54,
// temperature_processor.hpp:12-19, argmax_processor.cpp:6-35):
//   x_i = logit_i * (1/T);  keep the k largest;  prob_i = exp(x_i - x_0) / Z over the kept ones;
//   keep the shortest prefix whose probability reaches p (at least one token);
//   renormalise and take the first token at which the running sum exceeds u in [0,1).
// All three cuts are "the first place in the sorted order where a running measure
// (a count, or probability mass) reaches a target".  That place is found by radix
// descent over the bits of the logit: four passes, each a 256-bin histogram of the
// measure over the keys that share the prefix found so far.  Ties (equal logits)
// are ordered by token id.  Mass is kept as 64-bit fixed point (2^-40 units) and
// added with integer atomics, so the result does not depend on the order in which
// threads arrive and a (seed, position) pair always gives the same token.
//
// Nearly every row needs none of the four passes over all of its elements: what the three cuts look at lies within a few
// hundred of the largest logits, whatever lies below.  One histogram over the distance from the row's maximum
// (`candidates`) finds a bin behind which nothing matters, and the elements ahead of it are gathered into LDS, at most one
// a thread.  Every cut is read off the ranks of a short list; a longer one (and a whole row of no more elements than
// threads) takes the descent over the threads' own elements.  The counts and masses are the same integers, so the token
// is the descent's token; a row whose first cut reaches beyond kMaxListed elements, or that is flat and has no top-k,
// takes the descent over all elements.
//
// One workgroup per row.  u comes from a counter-based generator keyed by the
// row's seed and the row's position counter.
#include "common.h"

namespace {

constexpr int S_THREADS = 1024;
constexpr int S_WAVES = S_THREADS / TL_WAVE;
constexpr double kFix = 1099511627776.0;  // 2^40

__device__ __forceinline__ uint32_t order_key(float x) {
  if (x != x) return 0u;  // NaN sorts last
  const uint32_t b = __float_as_uint(x);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
  const uint32_t b = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __uint_as_float(b);
}

__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Bins of 2^15 neighbouring keys below the row's largest: 256 an octave of logits, eight octaves.  A logit row's
// values share a handful of exponents, so bins of the key's leading byte (the descent's first pass) are hit by
// thousands of elements each and their LDS atomics queue up: that is what the descent's passes wait for.
constexpr int kDistShift = 15, kDistBins = 2048;
// Most elements of a list (one a thread), and most of which the ranks are formed, for which each looks at all of them.  8
// rows of 32,000: the 200 best and three cuts take 34 us by ranks; the 1,000 best and one cut 132 us by ranks, 32 by
// descents over the list and 110 by descents over the row.
constexpr int kMaxListed = S_THREADS, kMaxRanked = 256;
// Rows of up to this many logits are read once and stay in registers.
constexpr int kHeldVecs = 8, kHeldVocab = kHeldVecs * 4 * S_THREADS;

struct Shared {
  union {
    struct {
      unsigned long long hmass[256];
      unsigned int hcnt[256];
    };
    struct {
      unsigned long long dmass[kDistBins];
      unsigned int dcnt[kDistBins];
    };
    struct {
      unsigned long long lmass[kMaxListed];
      unsigned int lkey[kMaxListed];
      int lid[kMaxListed];
    };
  };
  unsigned int listed;
  unsigned long long red64[S_WAVES];
  unsigned int red32[S_WAVES];
  // result of one histogram scan
  unsigned int bin;
  unsigned long long above_mass;
  unsigned int above_cnt;
  unsigned long long bin_mass;
  unsigned int bin_cnt;
  int token;
};

struct Row {
  const float* logits;
  int vocab;
  float inv_t;
  float xmax;
};

__device__ __forceinline__ float scaled(const Row& r, int i) { return r.logits[i] * r.inv_t; }

__device__ __forceinline__ unsigned long long mass_of(const Row& r, float x) {
  return (unsigned long long)((double)expf(x - r.xmax) * kFix);
}

// Finds the key K* at which the running measure, taken over keys in descending
// order, first reaches `target` (>= 1).  by_mass selects the measure.  On return
// (in sh): above_mass / above_cnt = mass and count of keys > K*; bin_mass / bin_cnt
// = mass and count of keys == K*.  Returns K*.  `each` calls its argument with the key of every element of the calling
// thread and a function that gives its mass.
template <typename E>
__device__ uint32_t descend(const E& each, Shared& sh, bool by_mass, unsigned long long target) {
  uint32_t prefix = 0;
  unsigned long long above_mass = 0;
  unsigned int above_cnt = 0;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int b = threadIdx.x; b < 256; b += S_THREADS) {
      sh.hmass[b] = 0;
      sh.hcnt[b] = 0;
    }
    __syncthreads();
    each([&](uint32_t key, auto mass) {
      const bool match = (shift == 24) || ((key >> (shift + 8)) == (prefix >> (shift + 8)));
      if (match) {
        const int bin = (key >> shift) & 255;
        atomicAdd(&sh.hmass[bin], mass());
        atomicAdd(&sh.hcnt[bin], 1u);
      }
    });
    __syncthreads();
    if (threadIdx.x < TL_WAVE) {
      // lane L owns bins 255-4L .. 252-4L, i.e. the scan runs from the largest keys down
      const int lane = threadIdx.x;
      unsigned long long lm[4], tm = 0;
      unsigned int lc[4], tc = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lm[i] = sh.hmass[255 - 4 * lane - i];
        lc[i] = sh.hcnt[255 - 4 * lane - i];
        tm += lm[i];
        tc += lc[i];
      }
      unsigned long long im = tm;  // inclusive scan over lanes
      unsigned int ic = tc;
#pragma unroll
      for (int off = 1; off < TL_WAVE; off <<= 1) {
        const unsigned long long um = __shfl_up(im, off, TL_WAVE);
        const unsigned int uc = __shfl_up(ic, off, TL_WAVE);
        if (lane >= off) {
          im += um;
          ic += uc;
        }
      }
      unsigned long long run_m = above_mass + (im - tm);
      unsigned int run_c = above_cnt + (ic - tc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const unsigned long long before = by_mass ? run_m : (unsigned long long)run_c;
        const unsigned long long after = by_mass ? run_m + lm[i] : (unsigned long long)(run_c + lc[i]);
        if (before < target && after >= target) {
          sh.bin = 255 - 4 * lane - i;
          sh.above_mass = run_m;
          sh.above_cnt = run_c;
          sh.bin_mass = lm[i];
          sh.bin_cnt = lc[i];
        }
        run_m += lm[i];
        run_c += lc[i];
      }
    }
    __syncthreads();
    prefix |= (uint32_t)sh.bin << shift;
    above_mass = sh.above_mass;
    above_cnt = sh.above_cnt;
    __syncthreads();
  }
  return prefix;
}

// Token id of the n-th (1-based) element, in ascending id order, whose key equals `key`.
__device__ int nth_with_key(const Row& r, Shared& sh, uint32_t key, unsigned int n) {
  const int chunk = (r.vocab + S_THREADS - 1) / S_THREADS;
  const int begin = min(r.vocab, (int)threadIdx.x * chunk), end = min(r.vocab, begin + chunk);
  unsigned int cnt = 0;
  for (int i = begin; i < end; ++i) cnt += order_key(scaled(r, i)) == key;
  // exclusive scan of cnt over the workgroup: within the wave, then over wave totals
  const int lane = threadIdx.x % TL_WAVE, wave = threadIdx.x / TL_WAVE;
  unsigned int inc = cnt;
#pragma unroll
  for (int off = 1; off < TL_WAVE; off <<= 1) {
    const unsigned int up = __shfl_up(inc, off, TL_WAVE);
    if (lane >= off) inc += up;
  }
  if (lane == TL_WAVE - 1) sh.red32[wave] = inc;
  if (threadIdx.x == 0) sh.token = -1;
  __syncthreads();
  unsigned int base = 0;
  for (int wv = 0; wv < wave; ++wv) base += sh.red32[wv];
  const unsigned int before = base + inc - cnt;
  if (before < n && before + cnt >= n) {
    unsigned int seen = before;
    for (int i = begin; i < end; ++i)
      if (order_key(scaled(r, i)) == key && ++seen == n) {
        sh.token = i;
        break;
      }
  }
  __syncthreads();
  const int tok = sh.token;
  __syncthreads();
  return tok;
}

// The row's scaled logits with their ids, from registers (HELD) or from memory.
template <bool HELD, typename F>
__device__ __forceinline__ void for_row(const Row& r, const f32x4* held, F f) {
  if constexpr (HELD) {
#pragma unroll
    for (int u = 0; u < kHeldVecs; ++u) {
      const int i = (u * S_THREADS + (int)threadIdx.x) * 4;
      if (i < r.vocab) {
#pragma unroll
        for (int e = 0; e < 4; ++e) f(held[u][e] * r.inv_t, i + e);
      }
    }
  } else {
#pragma unroll 4
    for (int i = threadIdx.x; i < r.vocab; i += S_THREADS) f(scaled(r, i), i);
  }
}

// Sum over the workgroup; every thread gets it.
__device__ __forceinline__ unsigned long long sum64(Shared& sh, unsigned long long part) {
#pragma unroll
  for (int off = TL_WAVE / 2; off > 0; off >>= 1) part += __shfl_xor(part, off, TL_WAVE);
  __syncthreads();
  if (threadIdx.x % TL_WAVE == 0) sh.red64[threadIdx.x / TL_WAVE] = part;
  __syncthreads();
  unsigned long long z = 0;
  for (int wv = 0; wv < S_WAVES; ++wv) z += sh.red64[wv];
  return z;
}

// Gathers (key, id, mass) of a set of the row's largest elements that reaches `target` of the measure (counts, or mass)
// and holds every element of the smallest key in it.  Returns their number, or 0: beyond the bins or beyond the list.
// `kmin`: no smaller key is in the set.
template <bool HELD>
__device__ int candidates(const Row& r, Shared& sh, const f32x4* held, uint32_t kmax, bool by_mass,
                          unsigned long long target, uint32_t* kmin) {
  for (int b = threadIdx.x; b < kDistBins; b += S_THREADS) {
    sh.dmass[b] = 0;
    sh.dcnt[b] = 0;
  }
  if (threadIdx.x == 0) {
    sh.listed = 0;
    sh.bin = kDistBins;
  }
  __syncthreads();
  for_row<HELD>(r, held, [&](float x, int) {
    const uint32_t b = (kmax - order_key(x)) >> kDistShift;
    if (b < kDistBins) {
      atomicAdd(&sh.dcnt[b], 1u);
      if (by_mass) atomicAdd(&sh.dmass[b], mass_of(r, x));
    }
  });
  __syncthreads();
  // thread t owns bins 2t and 2t + 1: the first bin at which the running measure reaches the target
  const int lane = threadIdx.x % TL_WAVE, wave = threadIdx.x / TL_WAVE;
  const unsigned int c0 = sh.dcnt[2 * threadIdx.x], c1 = sh.dcnt[2 * threadIdx.x + 1];
  const unsigned long long m0 = by_mass ? sh.dmass[2 * threadIdx.x] : c0, m1 = by_mass ? sh.dmass[2 * threadIdx.x + 1] : c1;
  unsigned int ic = c0 + c1;
  unsigned long long im = m0 + m1;
#pragma unroll
  for (int off = 1; off < TL_WAVE; off <<= 1) {
    const unsigned int uc = __shfl_up(ic, off, TL_WAVE);
    const unsigned long long um = __shfl_up(im, off, TL_WAVE);
    if (lane >= off) {
      ic += uc;
      im += um;
    }
  }
  if (lane == TL_WAVE - 1) {
    sh.red32[wave] = ic;
    sh.red64[wave] = im;
  }
  __syncthreads();
  for (int wv = 0; wv < wave; ++wv) {
    ic += sh.red32[wv];
    im += sh.red64[wv];
  }
  if (im >= target && im - m1 - m0 < target) {          // they reach through bin 2t + 1
    const bool first = im - m1 >= target;
    sh.bin = 2 * threadIdx.x + (first ? 0 : 1);
    sh.bin_cnt = first ? ic - c1 : ic;
  }
  __syncthreads();
  const unsigned int last = sh.bin;
  const int n = last < kDistBins ? (int)sh.bin_cnt : 0;
  const uint32_t reach = ((last + 1) << kDistShift) - 1;      // how far below the maximum they go
  *kmin = n > 0 && reach < kmax ? kmax - reach : 0u;
  __syncthreads();                          // the list takes the histograms' place
  if (n <= 0 || n > kMaxListed) return 0;
  for_row<HELD>(r, held, [&](float x, int i) {
    const uint32_t key = order_key(x);
    if ((kmax - key) >> kDistShift <= last) {
      const unsigned int at = atomicAdd(&sh.listed, 1u);
      sh.lkey[at] = key;
      sh.lid[at] = i;
      sh.lmass[at] = mass_of(r, x);
    }
  });
  __syncthreads();
  return n;
}

// At most one element a thread.
struct Own {
  bool mine;
  uint32_t key;
  int id;
  unsigned long long mass;
};

// The whole chain (top-k, top-p, the draw) by descents over the elements of `each`.  Returns the drawn key, with in `nth`
// which of the `ties` elements that share it.
template <typename E>
__device__ uint32_t cut_and_draw(const E& each, Shared& sh, bool cut_k, int k, float p, double u, unsigned long long z,
                                 unsigned int* nth, unsigned int* ties) {
  uint32_t key = 0;
  for (int cut = cut_k ? 0 : 1; cut < 3; ++cut) {
    if (cut == 1 && !(p < 1.f)) continue;
    unsigned long long target = (unsigned long long)k;
    if (cut == 1) {             // the shortest prefix whose mass reaches p * z
      target = (unsigned long long)((double)fmaxf(p, 0.f) * (double)z);
      target = min(max(target, 1ull), z);
    } else if (cut == 2) {      // the first token at which the running mass exceeds u * z
      target = min((unsigned long long)(u * (double)z) + 1ull, z);
    }
    key = descend(each, sh, cut > 0, target);
    *ties = sh.bin_cnt;
    if (cut == 0) {             // mass of the k largest
      z = sh.above_mass + (unsigned long long)((unsigned int)k - sh.above_cnt) * (sh.bin_mass / sh.bin_cnt);
    } else {
      const unsigned long long w = max(sh.bin_mass / sh.bin_cnt, 1ull);
      const unsigned long long n = min(max((target - sh.above_mass + w - 1) / w, 1ull), (unsigned long long)sh.bin_cnt);
      z = sh.above_mass + n * w;
      *nth = (unsigned int)n;
    }
    __syncthreads();
  }
  return key;
}

// The same for a short list of which each thread below n has an element (key, id and mass of all of them are in LDS): every
// element's place is formed at once, how many and how much lies above it, how many share its key, how many of those
// come first.
__device__ void draw_by_rank(const Own& own, Shared& sh, int n, bool cut_k, int k, float p, double u, unsigned long long z,
                             int32_t* out) {
  unsigned int above = 0, ties = 0, earlier = 0;
  unsigned long long above_mass = 0;
  if (own.mine) {
#pragma unroll 4
    for (int j = 0; j < n; ++j) {
      const uint32_t kj = sh.lkey[j];
      const unsigned long long mj = sh.lmass[j];
      const int ij = sh.lid[j];
      above += kj > own.key;
      above_mass += kj > own.key ? mj : 0ull;
      ties += kj == own.key;
      earlier += kj == own.key && ij < own.id;
    }
  }
  const bool first = own.mine && earlier == 0;            // one element speaks for its key
  const unsigned long long w = max(own.mass, 1ull), through = above_mass + own.mass * ties;
  if (cut_k) {
    if (first && above < (unsigned int)k && above + ties >= (unsigned int)k)
      sh.above_mass = above_mass + (unsigned long long)((unsigned int)k - above) * own.mass;
    __syncthreads();
    z = sh.above_mass;
    __syncthreads();
  }
  unsigned long long target;
  if (p < 1.f) {
    target = (unsigned long long)((double)fmaxf(p, 0.f) * (double)z);
    target = min(max(target, 1ull), z);
    if (first && above_mass < target && through >= target) {
      const unsigned long long kept = min(max((target - above_mass + w - 1) / w, 1ull), (unsigned long long)ties);
      sh.above_mass = above_mass + kept * w;
    }
    __syncthreads();
    z = sh.above_mass;
    __syncthreads();
  }
  target = min((unsigned long long)(u * (double)z) + 1ull, z);
  if (own.mine && above_mass < target && through >= target) {
    const unsigned long long nth = min(max((target - above_mass + w - 1) / w, 1ull), (unsigned long long)ties);
    if (earlier + 1 == nth) *out = own.id;
  }
}

// The chain over the threads' own elements, n of them.  ORDERED: the ids ascend with the threads.
template <bool ORDERED>
__device__ void draw_own(const Own& own, Shared& sh, int n, bool cut_k, int k, float p, double u, unsigned long long z,
                         int32_t* out) {
  if (n <= kMaxRanked) return draw_by_rank(own, sh, n, cut_k, k, p, u, z, out);
  __syncthreads();                          // the descent's histograms take the list's place
  unsigned int nth = 0, ties = 0;
  const uint32_t key = cut_and_draw([&](auto f) { if (own.mine) f(own.key, [&] { return own.mass; }); }, sh, cut_k, k, p, u,
                                    z, &nth, &ties);
  const bool drawn = own.mine && own.key == key;
  if (ties == 1) {
    if (drawn) *out = own.id;
    return;
  }
  if constexpr (ORDERED) {
    const int lane = threadIdx.x % TL_WAVE, wave = threadIdx.x / TL_WAVE;
    const unsigned long long all = __ballot(drawn);
    if (lane == 0) sh.red32[wave] = __popcll(all);
    __syncthreads();
    unsigned int before = __popcll(all & ((1ull << lane) - 1));
    for (int wv = 0; wv < wave; ++wv) before += sh.red32[wv];
    if (drawn && before + 1 == nth) *out = own.id;
  } else {          // the nth in ascending order of the ids: the nth largest of their complements
    const uint32_t id = ~descend([&](auto f) { if (drawn) f(~(uint32_t)own.id, [] { return 0ull; }); }, sh, false, nth);
    if (threadIdx.x == 0) *out = (int32_t)id;
  }
}

// By way of a list of the row's largest elements; z is the row's mass where there is no top-k.  False: this row takes the
// descent over all of its elements from `kmin` on.
template <bool HELD>
__device__ bool draw_listed(const Row& r, Shared& sh, const f32x4* held, uint32_t kmax, bool cut_k, int k, float p, double u,
                            unsigned long long z, uint32_t* kmin, int32_t* out) {
  unsigned long long target;
  if (cut_k) {
    target = (unsigned long long)k;
  } else {
    target = p < 1.f ? min(max((unsigned long long)((double)fmaxf(p, 0.f) * (double)z), 1ull), z)
                     : min((unsigned long long)(u * (double)z) + 1ull, z);
  }
  const int n = candidates<HELD>(r, sh, held, kmax, !cut_k, target, kmin);
  if (n == 0) return false;
  Own own = {(int)threadIdx.x < n, 0u, 0, 0ull};
  if (own.mine) {
    own.key = sh.lkey[threadIdx.x];
    own.id = sh.lid[threadIdx.x];
    own.mass = sh.lmass[threadIdx.x];
  }
  draw_own<false>(own, sh, n, cut_k, k, p, u, z, out);
  return true;
}

// Over all of the row's elements, read again in every pass (registers for 32 of them a thread would spill).  None below
// `kmin` matters to any cut, and without them the passes' atomics meet less often, which pays for the search that did not
// end in a list.
__device__ void draw_from_all(const Row& r, Shared& sh, uint32_t kmin, bool cut_k, int k, float p, double u,
                              unsigned long long z, int32_t* out) {
  unsigned int nth = 0, ties = 0;
  const uint32_t key = cut_and_draw(
      [&](auto f) {
        for (int i = threadIdx.x; i < r.vocab; i += S_THREADS) {
          const float x = scaled(r, i);
          const uint32_t key = order_key(x);
          if (key >= kmin) f(key, [&] { return mass_of(r, x); });
        }
      },
      sh, cut_k, k, p, u, z, &nth, &ties);
  const int tok = nth_with_key(r, sh, key, nth);
  if (threadIdx.x == 0) *out = tok;
}

__global__ __launch_bounds__(S_THREADS) void sample_kernel(
    const float* __restrict__ logits, int64_t row_stride, int vocab, const float* __restrict__ temperature,
    const int32_t* __restrict__ top_k, const float* __restrict__ top_p, const int64_t* __restrict__ seeds,
    const int32_t* __restrict__ counters, int32_t* __restrict__ out) {
  __shared__ Shared sh;
  const int row = blockIdx.x;
  Row r;
  r.logits = logits + (int64_t)row * row_stride;
  r.vocab = vocab;
  const float temp = temperature ? temperature[row] : 0.f;
  const bool greedy = !(temp > 0.f);
  r.inv_t = greedy ? 1.f : 1.f / temp;
  r.xmax = 0.f;

  if (greedy) {
    // One pass: the largest (key, lowest index) pair.  The index is stored inverted in the low
    // half, so the maximum of the pairs is the first maximum of the row.
    unsigned long long best = 0;
    const bool vec = (vocab % 4 == 0) && (((uintptr_t)r.logits & 15) == 0);
    if (vec) {
      for (int i = threadIdx.x * 4; i < vocab; i += S_THREADS * 4) {
        const f32x4 x = *(const f32x4*)(r.logits + i);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          best = max(best, ((unsigned long long)order_key(x[e]) << 32) | (uint32_t)(0xffffffffu - (uint32_t)(i + e)));
      }
    } else {
      for (int i = threadIdx.x; i < vocab; i += S_THREADS)
        best = max(best, ((unsigned long long)order_key(r.logits[i]) << 32) | (uint32_t)(0xffffffffu - (uint32_t)i));
    }
#pragma unroll
    for (int off = TL_WAVE / 2; off > 0; off >>= 1) {
      const uint32_t hi = (uint32_t)__shfl_xor((int)(best >> 32), off, TL_WAVE);
      const uint32_t lo = (uint32_t)__shfl_xor((int)(best & 0xffffffffu), off, TL_WAVE);
      best = max(best, ((unsigned long long)hi << 32) | lo);
    }
    if (threadIdx.x % TL_WAVE == 0) sh.red64[threadIdx.x / TL_WAVE] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int wv = 0; wv < S_WAVES; ++wv) best = max(best, sh.red64[wv]);
      out[row] = (int32_t)(0xffffffffu - (uint32_t)(best & 0xffffffffu));
    }
    return;
  }

  // maximum key of the row
  uint32_t kmax = 0;
  const bool held_row = vocab <= kHeldVocab && vocab % 4 == 0 && (((uintptr_t)r.logits & 15) == 0);
  f32x4 held[kHeldVecs];
  if (held_row) {
#pragma unroll
    for (int v = 0; v < kHeldVecs; ++v) {
      const int i = (v * S_THREADS + (int)threadIdx.x) * 4;
      held[v] = i < vocab ? *(const f32x4*)(r.logits + i) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for_row<true>(r, held, [&](float x, int) { kmax = max(kmax, order_key(x)); });
  } else {
    for_row<false>(r, held, [&](float x, int) { kmax = max(kmax, order_key(x)); });
  }
#pragma unroll
  for (int off = TL_WAVE / 2; off > 0; off >>= 1) kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, off, TL_WAVE));
  if (threadIdx.x % TL_WAVE == 0) sh.red32[threadIdx.x / TL_WAVE] = kmax;
  __syncthreads();
  kmax = 0;
  for (int wv = 0; wv < S_WAVES; ++wv) kmax = max(kmax, sh.red32[wv]);
  __syncthreads();

  r.xmax = key_value(kmax);
  const uint64_t seed = seeds ? (uint64_t)seeds[row] : 0ull;
  const uint64_t ctr = counters ? (uint64_t)(uint32_t)counters[row] : 0ull;
  const uint64_t bits = splitmix64(splitmix64(seed) ^ (ctr * 0xD1B54A32D192ED03ull));
  const double u = (double)(bits >> 40) * (1.0 / 16777216.0);  // 24 bits, [0, 1)
  const int k = top_k ? top_k[row] : 0;
  const float p = top_p ? top_p[row] : 1.f;

  const bool cut_k = k > 0 && k < vocab;
  unsigned long long z = 0;                 // the mass that is left: of all elements, then of those ahead of each cut
  if (!cut_k) {
    unsigned long long part = 0;
    auto add = [&](float x, int) { part += mass_of(r, x); };
    if (held_row) for_row<true>(r, held, add);
    else for_row<false>(r, held, add);
    z = sum64(sh, part);
    __syncthreads();
  }

  int32_t* token = out + row;
  const bool finite = fabsf(r.xmax) < INFINITY;       // else there are no masses to rank
  if (finite && vocab <= S_THREADS) {       // an element a thread: no list to look for
    Own own = {(int)threadIdx.x < vocab, 0u, (int)threadIdx.x, 0ull};
    if (own.mine) {
      const float x = scaled(r, threadIdx.x);
      own.key = order_key(x);
      own.mass = mass_of(r, x);
      if (vocab <= kMaxRanked) {
        sh.lkey[threadIdx.x] = own.key;
        sh.lid[threadIdx.x] = own.id;
        sh.lmass[threadIdx.x] = own.mass;
      }
    }
    __syncthreads();
    return draw_own<true>(own, sh, vocab, cut_k, k, p, u, z, token);
  }

  // Rows of 32,000 logits with the default options (temperature 0.7, the 50 best, mass 0.95): 154 us for one row and 163
  // us for 64 by the descent, 20 us from the list; 128,256 logits 569 and 63 us.  Without a top-k the list is
  // tried where the first cut cannot lie far down, the likeliest token holding a 64th of the mass or more (70 -> 23 us);
  // behind a flat row's first pass (normal logits: a thousandth) the list would only be found too short (70 -> 85 us).
  // Where it is found too short all the same, what the search learned makes up for it (normal logits of spread 3, mass 0.9,
  // 64 rows: 128 us by descents alone, 110 so); a row whose largest logit is so near zero that the first cut lies beyond
  // the bins takes 3 to 5 % more.
  uint32_t kmin = 0;
  if (finite && (cut_k ? k <= kMaxListed : z < 64ull << 40)) {
    const bool done = held_row ? draw_listed<true>(r, sh, held, kmax, cut_k, k, p, u, z, &kmin, token)
                               : draw_listed<false>(r, sh, held, kmax, cut_k, k, p, u, z, &kmin, token);
    if (done) return;
  }
  draw_from_all(r, sh, kmin, cut_k, k, p, u, z, token);
}

}  // namespace

extern "C" {

// temperature[row] <= 0 (or a null pointer) selects greedy argmax for that row.
// top_k[row] <= 0 or >= vocab keeps every token; top_p[row] >= 1 keeps every token.
int tl_sample(const float* logits, int64_t row_stride, int n_rows, int vocab, const float* temperature,
              const int32_t* top_k, const float* top_p, const int64_t* seeds, const int32_t* counters,
              int32_t* out, hipStream_t stream) {
  if (n_rows <= 0) return TL_OK;
  if (vocab <= 0 || row_stride < vocab) return TL_ERR_ARG;
  hipLaunchKernelGGL(sample_kernel, dim3(n_rows), dim3(S_THREADS), 0, stream, logits, row_stride, vocab,
                     temperature, top_k, top_p, seeds, counters, out);
  return tl_launch_status();
}

}  // extern "C"
