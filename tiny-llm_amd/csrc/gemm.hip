// Linear layers: out[m, n] = sum_k a[m, k] * w[n, k] (+ residual[m, n]).
// Weights are [out, in] row-major as in the checkpoint, the contraction the
// reference's GEMM family computes (tiny_llm/ops/cuda/gemm.cu:86-100); the
// residual add that the reference runs as a separate kernel
// (tiny_llm/ops/cuda/arithmetic.cu:13) is folded into the epilogue.
//
//  * gemm_f32_ring_kernel (tiles of 32 to 128 rows and 64 or 128 columns), gemm_f32_kernel (any rows and inner size), and
//    gemm_f32_rows_kernel for few rows: true float32 on the matrix cores (v_mfma_f32_16x16x4_f32), no
//    reduced-precision mode.  All add in ONE order, so a row gives the same bits whether it is computed
//    alone or in a batch, by any of them.
//  * gemm_bf16_kernel: bf16 inputs on the matrix cores, float32 accumulation, 256 x 256, 256 x 128, 128 x 128 or 64 x 128 tiles
//    with k steps of 64: operands straight from memory into two to four buffers in LDS (v_mfma_f32_16x16x32_bf16), or through
//    registers into two (v_mfma_f32_32x32x16_bf16; tile_mode says where); optionally over a share of the inner size (split k).
//  * gemm_oneshot_bf16_kernel: the split product for few rows, operands streamed through a ring of
//    LDS slabs filled straight from memory; splitk_reduce_kernel adds the parts and applies the epilogue.
//  * gemm_skinny_bf16_kernel: the fewest rows (decode steps), weights streamed once into registers; up to 64 for inner sizes that
//    are no multiple of 64.
//  * gemm_stripe_bf16_kernel: 6 to 64 rows (stripe_plan says which), the inner size whole.
#include <type_traits>

#include "common.h"

namespace {

// ===================================================================== float32
// True float32 on the matrix cores: v_mfma_f32_16x16x4_f32 takes float32 operands and keeps float32
// sums (no reduced-precision mode).  The kernels below add the terms of an output element in ONE
// order, so that a row gives the same bits alone and in any batch, by any of them:
//   * k runs in blocks of 256, each block summed from zero, the block sums added in ascending order;
//   * inside a block, groups of 16 k in ascending order; a group is four matrix instructions, the
//     e-th of which takes k = 16 group + {0, 4, 8, 12} + e (a lane holds four consecutive k of its row,
//     one for each of the four instructions);
//   * operands beyond K are zero.
constexpr int F_KBLOCK = 256;     // the k block of the order of addition
constexpr int F_BK = 16, F_THREADS = 256;
constexpr int F_LD = F_BK + 4;    // LDS row stride in floats (80 bytes: 16-byte aligned rows)

// What a bfloat16 product may apply to its float32 sums before they are rounded (a run-time choice, the same for the whole
// launch; epilogue 2 of the entry points): the square of max(v, 0).
constexpr int kActNone = 0, kActRelu2 = 2, kActTanh = 5;      // tanh: products of a set only, rounded to bfloat16 as they are stored
__device__ __forceinline__ float act_value(float v, int act) {
  if (act == kActRelu2) {
    v = fmaxf(v, 0.f);
    v *= v;
  }
  return v;
}

// silu(g) * u of an interleaved gate|up pair of output columns, as the reference computes it
// (tiny_llm/ops/cuda/silu.cu:10, arithmetic.cu:13), from the float32 accumulators.
__device__ __forceinline__ float swiglu_pair(float g, float u) { return g / (1.f + expf(-g)) * u; }
// The same for the bfloat16 kernels, whose result is rounded to 8 bits anyway: hardware exp2 and
// reciprocal (about 1 ulp of float32 each) instead of the library's exp and a full division, which
// were a tenth of the gate/up product's time.
__device__ __forceinline__ float swiglu_pair_fast(float g, float u) {
  return g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.44269504088896341f * g)) * u;
}
// The gated units that the bfloat16 products' epilogues form of interleaved (gate, up) columns: SiLU, from the float32 sums; the
// clamped unit min(g, limit) sigmoid(alpha .) (clamp(u, -limit, limit) + shift) and gelu(g) u (tanh form), from sums rounded to
// bfloat16: the bits that clamped_glu_kernel and gelu_glu_kernel make of a product's stored result.  Without those kernels a
// layer of a decode step has a launch less, a prompt of 1,944 rows of 5,632 pairs 26 us (workload Lufazen 12.9 -> 12.6 ms).
constexpr int kGateSilu = 0, kGateClamped = 1, kGateGelu = 2;
struct Gate {
  int kind = kGateSilu;
  float limit = 0.f, alpha = 0.f, shift = 0.f;
};
// GATED: 1 SiLU, 2 one of the others (apart, so that SiLU products of few rows keep their registers: a decode step of them lost
// 0.8 % to a choice at run time)
template <int GATED>
__device__ __forceinline__ float gated_pair(float g, float u, const Gate& gate) {
  if constexpr (GATED == 1) return swiglu_pair_fast(g, u);
  g = (float)(bf16_t)g;
  u = (float)(bf16_t)u;
  if (gate.kind == kGateClamped) {
    g = fminf(g, gate.limit);
    u = fminf(fmaxf(u, -gate.limit), gate.limit);
    return g / (1.f + expf(-gate.alpha * g)) * (u + gate.shift);
  }
  return 0.5f * g * (1.f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
}
// Which gate an epilogue's number names (tl_linear_tile), and whether it names one
static inline bool is_gated(int epilogue) { return epilogue == 1 || epilogue == 3 || epilogue == 4; }
static inline Gate gate_of(int epilogue, float limit, float alpha, float shift) {
  return Gate{epilogue == 3 ? kGateClamped : epilogue == 4 ? kGateGelu : kGateSilu, limit, alpha, shift};
}

// 16 bytes a lane from a buffer straight into LDS, side by side from `dst` on (the same for the whole wave; the
// instruction takes its place from M0).  Written as an instruction block: given the builtin, the compiler waits for every
// load on its way ahead of each LDS read, whichever buffer it reads.  M0 is an operand, so the compiler writes it and knows
// that it is used; what it does not see is that the block holds a load, which needs a wait state behind that write: the
// s_nop.  Whoever reads the data waits for it first (tl_wait_loads, then a barrier).
typedef int tl_rsrc_words __attribute__((ext_vector_type(4)));
__device__ __forceinline__ unsigned int tl_lds_address(void* p) {
  return __builtin_amdgcn_readfirstlane((unsigned int)(uintptr_t)(__attribute__((address_space(3))) void*)p);
}
__device__ __forceinline__ void tl_load_to_lds(tl_rsrc_words buf, unsigned int at, int voffset, int soffset) {
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "{m0}"(at), "v"(voffset), "s"(buf), "s"(soffset)
               : "memory");
}
template <int LEFT>       // until at most LEFT of the wave's loads are still on their way
__device__ __forceinline__ void tl_wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory"); }

// Workgroups are handed to the eight XCDs in turn, each with an L2 of its own.  The index is remapped so that an XCD owns a
// contiguous run of tiles, and, `banded`, the tiles that it works on at a time make a block about as high as it is wide, which
// asks the fewest rows of both operands of its L2 (8192^3 with 256 x 256 tiles in columns of 32 927 us, in bands of four 786):
// bands of 4 to 7 rows of tiles, column by column, of which the last may be lower (as even as can be was no faster: 256 x 256
// tiles, 21 rows of them, 8,192 x 2,048 144.8 us and 145.8 even; 11 rows, 11,264 x 2,048 97.6 and 99.6).  Fewer than eight rows of tiles are one band, found by one division: three
// more took 0.1 to 0.25 us a launch.  128 x 128 and 64 x 128 tiles through registers stand in columns, whatever their number:
// two to four share a unit and short steps wait for each other, not for the L2 (2,102 rows, 3,712 x 128 in 128 x 128 tiles
// 8.94 us in bands, 8.63 so; 4,096 rows, 2,560 x 328 18.5 and 17.4; 2,047 rows, 4,096 x 192 with a residual 16.9 and 14.4).
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_tile(int block, int total) {
  const int per_xcd = (total + kXcds - 1) / kXcds;
  return (block % kXcds) * per_xcd + block / kXcds;
}
__host__ __device__ __forceinline__ void tile_place(int t, int tiles_m, int tiles_n, bool banded, int* tm, int* tn) {
  if (!banded || tiles_m < 8) {
    *tm = t % tiles_m;
    *tn = t / tiles_m;
    return;
  }
  const int bands = max(tiles_m / 4, 1), band_m = (tiles_m + bands - 1) / bands;
  const int band = t / (band_m * tiles_n), in_band = t - band * band_m * tiles_n, high = min(band_m, tiles_m - band * band_m);
  *tm = band * band_m + in_band % high;
  *tn = in_band / high;
}

// Four consecutive k of one row, zero beyond K; VEC: 16-byte aligned rows and K a multiple of 4.
template <bool VEC>
__device__ __forceinline__ f32x4 load_k4(const float* __restrict__ row, int k, int K) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if constexpr (VEC) {
    if (k < K) v = *(const f32x4*)(row + k);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (k + e < K) v[e] = row[k + e];
  }
  return v;
}

// The factor of a row's RMSNorm from the sum of its squares: ONE expression for every kernel that
// takes part in a float32 norm, so that they agree to the bit.
__device__ __forceinline__ float f32_norm_factor(float sumsq, int K, float eps) {
  return 1.f / sqrtf(sumsq / (float)K + eps);
}

// The norm in front of a float32 product for any number of rows, as two kernels: this one writes
// h = norm_w * x (float32) and a row's factor 1 / rms; the product then multiplies its sums by the
// factor (row_scale).  The squares of a row are added up in the order of gemm_f32_rows_kernel<NORM>:
// per k block of 256 four chains (chain q takes k = 16 g + 4 q + e for g = 0..15, e = 0..3, in that
// order, by fused multiply-adds from zero), the chains as (c0 + c1) + (c2 + c3), the blocks in
// ascending order.  So a row's result has the same bits whether the norm rode in the few-row product
// or went through here: a row's logits do not depend on how many rows its step had.
constexpr int FN_THREADS = 256;
template <bool VEC>
__global__ __launch_bounds__(FN_THREADS) void norm_prescale_f32_kernel(const float* __restrict__ x,
                                                                       const float* __restrict__ norm_w,
                                                                       const int32_t* __restrict__ rows,
                                                                       float* __restrict__ h,
                                                                       float* __restrict__ inv_rms, int K,
                                                                       int64_t lda, float eps) {
  extern __shared__ float chain_sums[];     // [k blocks][4]
  const int m = blockIdx.x;
  const float* row = x + (int64_t)(rows ? rows[m] : m) * lda;
  float* dst = h + (int64_t)m * K;
  const int nkb = (K + F_KBLOCK - 1) / F_KBLOCK;
  for (int c = threadIdx.x; c < nkb * 4; c += FN_THREADS) {
    const int kb = (c >> 2) * F_KBLOCK, q = c & 3;
    // all sixteen pieces of the chain are requested before the first is used: one round trip, not sixteen
    f32x4 v[16], nw[16];
#pragma unroll
    for (int g = 0; g < 16; ++g) {
      v[g] = load_k4<VEC>(row, kb + g * 16 + q * 4, K);
      nw[g] = load_k4<VEC>(norm_w, kb + g * 16 + q * 4, K);
    }
    float ss = 0.f;
#pragma unroll
    for (int g = 0; g < 16; ++g) {
      const int k = kb + g * 16 + q * 4;
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ss = __builtin_fmaf(v[g][e], v[g][e], ss);
        o[e] = v[g][e] * nw[g][e];
      }
      if constexpr (VEC) {
        if (k < K) *(f32x4*)(dst + k) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (k + e < K) dst[k + e] = o[e];
      }
    }
    chain_sums[c] = ss;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float total = 0.f;
    for (int b = 0; b < nkb; ++b)
      total += (chain_sums[4 * b] + chain_sums[4 * b + 1]) + (chain_sums[4 * b + 2] + chain_sums[4 * b + 3]);
    inv_rms[m] = f32_norm_factor(total, K, eps);
  }
}

// Tiles of 32 T rows x 32 T columns, four waves of 16 T x 16 T (T x T matrix tiles of 16 x 16), k in
// steps of 16 through double-buffered LDS.  T = 4 (128 x 128) where that gives the chip enough
// tiles, T = 2 (64 x 64) where it does not (a portion of 512 tokens times 2048 columns is 64 tiles
// of 128 x 128 for 256 compute units); the order in which an output element is added up is the
// same for every T.  The matrix instruction's rows are the output COLUMNS (weights are its first
// operand), so a lane ends up with four consecutive columns of one row.
template <bool SWIGLU, bool VEC, int T>
__global__ __launch_bounds__(F_THREADS) void gemm_f32_kernel(const float* __restrict__ a,
                                                             const float* __restrict__ w,
                                                             float* __restrict__ out,
                                                             const float* __restrict__ residual, int M,
                                                             int N, int K, int64_t lda, int64_t ldo,
                                                             const float* __restrict__ row_scale) {
  constexpr int BT = 32 * T;        // rows and columns of the workgroup's tile
  constexpr int PIECES = BT / 64;   // 16-byte pieces of each operand per thread and k step
  static_assert(T == 2 || T == 4, "tiles of 64 x 64 or 128 x 128");
  __shared__ __attribute__((aligned(16))) float As[2][BT * F_LD];
  __shared__ __attribute__((aligned(16))) float Ws[2][BT * F_LD];
  const int tid = threadIdx.x, lane = tid % TL_WAVE, wave = tid / TL_WAVE;
  const int wm = wave / 2, wn = wave % 2;
  const int m0 = blockIdx.y * BT, n0 = blockIdx.x * BT;
  const int l16 = lane % 16, kk = lane / 16;
  // staging: piece h of a thread is row (h * 256 + tid) / 4 of the tile, four k from 4 * (tid % 4)
  const int sr = tid / 4, sk = (tid % 4) * 4;
  const float *arow[PIECES], *wrow[PIECES];
#pragma unroll
  for (int h = 0; h < PIECES; ++h) {
    arow[h] = a + (int64_t)min(m0 + h * 64 + sr, M - 1) * lda;
    wrow[h] = w + (int64_t)min(n0 + h * 64 + sr, N - 1) * K;
  }
  f32x4 acc[T][T], tot[T][T];
#pragma unroll
  for (int nt = 0; nt < T; ++nt)
#pragma unroll
    for (int mt = 0; mt < T; ++mt) {
      acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
      tot[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  f32x4 ga[PIECES], gw[PIECES];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int h = 0; h < PIECES; ++h) {
      ga[h] = load_k4<VEC>(arow[h], k0 + sk, K);
      gw[h] = load_k4<VEC>(wrow[h], k0 + sk, K);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int h = 0; h < PIECES; ++h) {
      *(f32x4*)(&As[buf][(h * 64 + sr) * F_LD + sk]) = ga[h];
      *(f32x4*)(&Ws[buf][(h * 64 + sr) * F_LD + sk]) = gw[h];
    }
  };
  fetch(0);
  stage(0);
  __syncthreads();
  const int steps = (K + F_BK - 1) / F_BK;
  for (int s = 0; s < steps; ++s) {
    const int buf = s & 1;
    if (s + 1 < steps) fetch((s + 1) * F_BK);
    f32x4 wv[T], av[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      wv[t] = *(const f32x4*)(&Ws[buf][(wn * 16 * T + t * 16 + l16) * F_LD + kk * 4]);
      av[t] = *(const f32x4*)(&As[buf][(wm * 16 * T + t * 16 + l16) * F_LD + kk * 4]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int nt = 0; nt < T; ++nt)
#pragma unroll
        for (int mt = 0; mt < T; ++mt)
          acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[nt][e], av[mt][e], acc[nt][mt], 0, 0, 0);
    if (((s + 1) * F_BK) % F_KBLOCK == 0 || s + 1 == steps) {     // a block of the order of addition ends
#pragma unroll
      for (int nt = 0; nt < T; ++nt)
#pragma unroll
        for (int mt = 0; mt < T; ++mt) {
          tot[nt][mt] += acc[nt][mt];
          acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (s + 1 < steps) stage(buf ^ 1);
    __syncthreads();
  }
  // lane (l16, kk) of tile (nt, mt) holds row m = mt*16 + l16, columns n = nt*16 + 4 kk + r
#pragma unroll
  for (int mt = 0; mt < T; ++mt) {
    const int m = m0 + wm * 16 * T + mt * 16 + l16;
    if (m >= M) continue;
#pragma unroll
    for (int nt = 0; nt < T; ++nt) {
      const int n = n0 + wn * 16 * T + nt * 16 + kk * 4;
      f32x4 v = tot[nt][mt];
      if (row_scale) {      // the factor of a norm in front (norm_prescale_f32_kernel)
        const float f = row_scale[m];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] *= f;
      }
      if constexpr (SWIGLU) {   // columns (2j, 2j+1) = (gate_j, up_j); N is even
#pragma unroll
        for (int r = 0; r < 4; r += 2)
          if (n + r < N) out[(int64_t)m * ldo + (n + r) / 2] = swiglu_pair(v[r], v[r + 1]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) {
            const int64_t at = (int64_t)m * ldo + n + r;
            out[at] = residual ? v[r] + residual[at] : v[r];
          }
      }
    }
  }
}

// gemm_f32_ring_kernel: the same for rows of 16-byte pieces and an inner size that is a multiple of 32.  Four waves side by
// side, each with MT x NT matrix tiles (16 MT rows, 16 NT columns), so that a tile can be cut to make the chip's 256 units
// equally busy: 640 rows x 2,048 are 256 tiles of 80 x 64.  What bounds it are the matrix pipes (32 clocks an instruction, one
// wave a SIMD): operands go straight into LDS as a ring of R steps of 32 k, R - 2 of them on their way, the fragments of the
// next 16 k are read while these are multiplied, and there is one barrier a step, in the middle of its products.
// 640 rows, 2,048 x 2,048: 100 -> 54 us (100 TFLOP/s of 155 that a loop of these instructions reaches), 2,048 x 5,632
// 261 -> 138, 11,264 x 2,048 332 -> 240 (123); 333 rows, 1,000 x 2,080: 74 -> 27.  Tiles of 64 x 64, one barrier every 16 k,
// had a fragment's way from LDS and the barrier between any 16 instructions, and 320 of them kept 64 units twice as busy.
template <int MT, int NT>
struct F32Ring {
  static constexpr int BM = 16 * MT, BN = 64 * NT, BK = 32;
  static constexpr int GROUPS = (BM + BN) / 8;             // 8 rows of 128 bytes: what one load of a wave brings
  static constexpr int PW = (GROUPS + 3) / 4;              // loads of a wave a step
  static constexpr int BYTES = PW * 4 * 1024;              // of a step in LDS
  static constexpr int R = 80 * 1024 / BYTES < 4 ? 4 : 80 * 1024 / BYTES > 6 ? 6 : 80 * 1024 / BYTES;
};
template <bool SWIGLU, int MT, int NT>
__global__ __launch_bounds__(F_THREADS) void gemm_f32_ring_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                  float* __restrict__ out, const float* __restrict__ residual,
                                                                  int M, int N, int K, int64_t lda, int64_t ldo,
                                                                  const float* __restrict__ row_scale, int vec_out) {
  using S = F32Ring<MT, NT>;
  constexpr int BM = S::BM, BN = S::BN, R = S::R, PW = S::PW;
  extern __shared__ __attribute__((aligned(1024))) unsigned char f32_ring[];
  const int tid = threadIdx.x, lane = tid % TL_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / TL_WAVE);
  const int l16 = lane % 16, kk = lane / 16;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int t = xcd_tile(blockIdx.x, tiles_m * tiles_n);
  if (t >= tiles_m * tiles_n) return;                      // the grid is padded to a multiple of 8
  int tile_m, tile_n;
  tile_place(t, tiles_m, tiles_n, true, &tile_m, &tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  // Each buffer begins at the tile's first row and ends with the matrix: rows beyond it read as zeros.
  auto buffer_words = [](const float* first_row, int rows, int64_t ld, int K_) {
    const int64_t bytes = ((int64_t)(rows - 1) * ld + K_) * 4;
    const uint64_t at = (uint64_t)first_row;
    return tl_rsrc_words{(int)(uint32_t)at, (int)(uint32_t)(at >> 32) & 0xffff, (int)bytes, 0x00020000};
  };
  const tl_rsrc_words words_a = buffer_words(a + (int64_t)m0 * lda, min(M - m0, BM), lda, K);
  const tl_rsrc_words words_w = buffer_words(w + (int64_t)n0 * K, min(N - n0, BN), K, K);
  // Wave v brings groups v, v + 4, ... of a step: the activations' 2 MT, then the weights' 8 NT, then, where they do not share
  // out evenly, nothing into a place that nobody reads.  Row r holds the four k of piece c at place c ^ (r / 2 % 8).
  int off[PW];
#pragma unroll
  for (int j = 0; j < PW; ++j) {
    const int gi = wave + 4 * j, row = (gi < BM / 8 ? gi : gi - BM / 8) * 8 + lane / 8;
    const int64_t ld = gi < BM / 8 ? lda : (int64_t)K;
    off[j] = gi < S::GROUPS ? (int)((row * ld + ((lane % 8) ^ (row / 2 % 8)) * 4) * 4) : 0;
  }
  const unsigned int lds = tl_lds_address(f32_ring);
  const int steps = K / S::BK;
  auto fill = [&](int s) {                                 // steps behind the last read as zeros from a buffer of no bytes
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      const int gi = wave + 4 * j;
      tl_rsrc_words from = gi < BM / 8 ? words_a : words_w;
      from[2] = s < steps && gi < S::GROUPS ? from[2] : 0;
      tl_load_to_lds(from, lds + (s % R) * S::BYTES + gi * 1024, off[j], min(s, steps - 1) * S::BK * 4);
    }
  };
  f32x4 acc[NT][MT], tot[NT][MT], av[2][MT], wv[2][NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
      tot[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  auto read = [&](int s, int half) {                       // the fragments of 16 k
    const float* buf = (const float*)(f32_ring + (s % R) * S::BYTES) + ((half * 4 + kk) ^ (l16 / 2 % 8)) * 4 + l16 * 32;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wv[half][nt] = *(const f32x4*)(buf + (BM + (wave * NT + nt) * 16) * 32);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) av[half][mt] = *(const f32x4*)(buf + mt * 16 * 32);
  };
  auto multiply = [&](int half) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[half][nt][e], av[half][mt][e], acc[nt][mt], 0, 0, 0);
  };
  auto meet = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int s = 0; s < R - 1; ++s) fill(s);
  tl_wait_loads<(R - 2) * PW>();
  meet();
  read(0, 0);
  for (int s = 0; s < steps; ++s) {
    read(s, 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
    // step s + 1 has arrived; and step s - 1, whose fragments every wave has multiplied, can be written over
    tl_wait_loads<(R - 3) * PW>();
    meet();
    fill(s + R - 1);
    read(s + 1, 0);                                        // behind the last step: read, not used
    __builtin_amdgcn_sched_barrier(0);
    multiply(1);
    if ((s + 1) % (F_KBLOCK / S::BK) == 0 || s + 1 == steps) {      // a block of the order of addition ends
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          tot[nt][mt] += acc[nt][mt];
          acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  tl_wait_loads<0>();                                      // nothing may arrive in LDS that is no longer this workgroup's
  // lane (l16, kk) of tile (nt, mt) holds row m = mt*16 + l16, columns n = nt*16 + 4 kk + r
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + mt * 16 + l16;
    if (m >= M) continue;
    const float f = row_scale ? row_scale[m] : 1.f;        // the factor of a norm in front (norm_prescale_f32_kernel)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = n0 + (wave * NT + nt) * 16 + kk * 4;
      if (n >= N) continue;
      f32x4 v = tot[nt][mt];
      if (row_scale) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] *= f;
      }
      if constexpr (SWIGLU) {   // columns (2j, 2j+1) = (gate_j, up_j); N is even
#pragma unroll
        for (int r = 0; r < 4; r += 2)
          if (n + r < N) out[(int64_t)m * ldo + (n + r) / 2] = swiglu_pair(v[r], v[r + 1]);
      } else {
        const int64_t at = (int64_t)m * ldo + n;
        if (vec_out) {          // uniform: rows are whole, aligned pieces of four
          if (residual) {
            const f32x4 x = *(const f32x4*)(residual + at);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += x[r];
          }
          *(f32x4*)(out + at) = v;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < N) out[at + r] = residual ? v[r] + residual[at + r] : v[r];
        }
      }
    }
  }
}

template <bool SWIGLU, int MT, int NT>
static int launch_f32_ring(const float* a, const float* w, float* out, const float* residual, int M, int N, int K, int64_t lda,
                           int64_t ldo, const float* row_scale, int vec_out, hipStream_t stream) {
  using S = F32Ring<MT, NT>;
  static bool configured = false;
  if (!configured) {
    if (hipFuncSetAttribute((const void*)gemm_f32_ring_kernel<SWIGLU, MT, NT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            S::R * S::BYTES) != hipSuccess)
      return TL_ERR_LAUNCH;
    configured = true;
  }
  const int64_t total = (int64_t)((M + S::BM - 1) / S::BM) * ((N + S::BN - 1) / S::BN);
  const int64_t grid = (total + kXcds - 1) / kXcds * kXcds;
  if (grid > 0x7fffffff) return TL_ERR_ARG;
  hipLaunchKernelGGL((gemm_f32_ring_kernel<SWIGLU, MT, NT>), dim3((unsigned)grid), dim3(F_THREADS), S::R * S::BYTES, stream, a, w,
                     out, residual, M, N, K, lda, ldo, row_scale, vec_out);
  return TL_OK;
}

// The tile whose rounds over 256 units are shortest, and the smaller of equals: a wave's matrix tiles and half of one for a
// step's barrier (with two for it, as one round takes, large tiles came out ahead of small ones that share units: 640 x
// 11,264 x 2,048 287 us instead of 240, 128 rows 77 instead of 61; 2,048 rows 874 instead of 892).  Returns an estimate of
// the time: 0.107 us for each matrix tile and two more a step of
// 32 k, 6 us for launch, first loads and epilogue (640 rows: 2,048 x 5,632 138 us estimated, 138 measured; 11,264 x 2,048
// 252 and 240; 257 rows, 2,048 x 2,048: 40 and 37).
static double f32_ring_us(int M, int N, int K, int* mt, int* nt) {
  double best = 0., units = 0.;
  for (int n = 1; n <= 2; ++n)
    for (int m = 2; m <= 8; ++m) {
      const int64_t wgs = (int64_t)((M + 16 * m - 1) / (16 * m)) * ((N + 64 * n - 1) / (64 * n));
      const double rounds = (double)((wgs + 255) / 256), cost = rounds * (m * n + 0.5);
      if (best == 0. || cost < best) {
        best = cost;
        units = rounds * (m * n + 2);
        *mt = m;
        *nt = n;
      }
    }
  return 6.0 + units * 0.107 * (K / 32);
}

// Whether it takes this product: whole vectors, and rows of a tile addressed with 32-bit byte offsets from its first.
static bool f32_ring_ok(bool vec, int K, int64_t lda) {
  return vec && K % 32 == 0 && 128 * lda * 4 < 0x7fffffff && (int64_t)128 * K * 4 < 0x7fffffff;
}

template <bool SWIGLU>
static int launch_f32_ring_any(const float* a, const float* w, float* out, const float* residual, int M, int N, int K,
                               int64_t lda, int64_t ldo, const float* row_scale, hipStream_t stream) {
  const int vec_out = N % 4 == 0 && ldo % 4 == 0 && ((uintptr_t)out | (uintptr_t)residual) % 16 == 0;
  int mt = 2, nt = 1;
  f32_ring_us(M, N, K, &mt, &nt);
#define TL_RING(MT)                                                                                                         \
  case MT:                                                                                                                  \
    return nt == 1 ? launch_f32_ring<SWIGLU, MT, 1>(a, w, out, residual, M, N, K, lda, ldo, row_scale, vec_out, stream)      \
                   : launch_f32_ring<SWIGLU, MT, 2>(a, w, out, residual, M, N, K, lda, ldo, row_scale, vec_out, stream)
  switch (mt) {
    TL_RING(2);
    TL_RING(3);
    TL_RING(4);
    TL_RING(5);
    TL_RING(6);
    TL_RING(7);
    TL_RING(8);
  }
#undef TL_RING
  return TL_ERR_ARG;
}

// The same product for 17 to 64 rows (and up to 256 where the tiled kernel has too few tiles), and with a norm in front: the weights stream
// once, straight from memory into the matrix instruction's operand registers.  A workgroup owns 16 output columns (8 with a norm where
// 16 would leave compute units without work: the matrix tile's other 8 rows then repeat them and
// are dropped); its eight waves deal the k blocks of 256 out among themselves, a wave requests a
// whole block (16 KB) at once; the block sums meet in LDS and
// are added in ascending order: the order of gemm_f32_kernel, to the bit.  Rows come in tiles of
// 16.  (Up to 16 rows: gemm_f32_lines_kernel.)
constexpr int FR_WAVES = 8, FR_THREADS = FR_WAVES * TL_WAVE, FR_MAX_MT = 4;

//
// NORM: `a` is the float32 residual stream and the product is that of its RMSNorm,
// ((norm_w * a) @ w.T) / sqrt(mean(a^2) + eps): the rows are multiplied by the norm's weight as they
// are loaded, their squares are added up on the way (per k block and row in a fixed order, the
// blocks in ascending order, so a row's factor depends on nothing but the row), and the factor is
// applied to the block sums' total.  That saves the norm's kernel in front of the product.
//
// The norm's arguments come first and as a structure, so that no argument is preloaded into registers (kernels are compiled to
// find the leading plain ones there).  Preloaded, eighteen such products took 0.7 % more on average: 16 rows of 2,048 x 2,048
// 10.9 -> 11.1 us, 65 of 2,048 x 5,632 49.4 -> 50.5, 100 of 2,560 x 2,048 35.2 -> 35.8, though the main loop's registers are
// the same; only 4 to 12 rows of 2,560 x 2,048 took 2 % less (9.8 -> 9.6).
struct F32RowsNorm {
  const float* w;
  float eps;
};
template <bool SWIGLU, int COLS, bool NORM, bool WIDE>
__global__ __launch_bounds__(FR_THREADS) void gemm_f32_rows_kernel(const F32RowsNorm norm, const float* __restrict__ a,
                                                                   const float* __restrict__ w,
                                                                   float* __restrict__ out,
                                                                   const float* __restrict__ residual, int M,
                                                                   int N, int K, int64_t lda, int64_t ldo,
                                                                   const float* __restrict__ row_scale = nullptr,
                                                                   int tiles_wg = FR_MAX_MT) {
  const float* __restrict__ norm_w = norm.w;
  const float eps = norm.eps;
  // WIDE (more than 16 rows): blockIdx.y picks a group of `tiles_wg` row tiles, so that a product with
  // few column tiles still gives every compute unit a workgroup with whole matrix tiles (16 columns)
  // instead of half-used ones (8 columns); the activations of the next row tile are requested before
  // this one is multiplied, and the registers that takes are those of the next block's weights, which
  // are requested behind the block's last row tile instead.
  static_assert(NORM != WIDE, "the norm rides in the product of few row tiles");
  extern __shared__ float rows_smem[];      // [m tiles][k blocks][16 rows][COLS columns], NORM: + [m tiles][k blocks][16]
  const int nkb = (K + F_KBLOCK - 1) / F_KBLOCK;
  const int mt0 = WIDE ? blockIdx.y * tiles_wg : 0;                       // first row tile of this workgroup
  const int mts = WIDE ? min(tiles_wg, (M + 15) / 16 - mt0) : (M + 15) / 16;   // and how many it owns
  const int tid = threadIdx.x, lane = tid % TL_WAVE, wave = tid / TL_WAVE;
  const int l16 = lane % 16, kk = lane / 16;
  const int n0 = blockIdx.x * COLS;
  const float* wrow = w + (int64_t)min(n0 + l16 % COLS, N - 1) * K;
  // A k block that lies wholly inside K is loaded without a predicate per load (each would be a
  // branch of its own, and the waits around branches are placed for the worst case); only the last,
  // partial block of an inner size that is no multiple of 256 takes the predicated loads.  The loop
  // body exists once per case (this block whole or not, the next block whole or not).
  auto load16 = [&](auto whole, f32x4 (&dst)[16], const float* row, int k0) {
#pragma unroll
    for (int g = 0; g < 16; ++g) {
      if constexpr (decltype(whole)::value) dst[g] = *(const f32x4*)(row + k0 + g * 16 + kk * 4);
      else dst[g] = load_k4<true>(row, k0 + g * 16 + kk * 4, K);
    }
  };
  auto a_row = [&](int mt) { return a + (int64_t)min((mt0 + mt) * 16 + l16, M - 1) * lda; };
  f32x4 wv[16];
  if (wave < nkb) {
    if ((wave + 1) * F_KBLOCK <= K) load16(std::true_type{}, wv, wrow, wave * F_KBLOCK);
    else load16(std::false_type{}, wv, wrow, wave * F_KBLOCK);
  }
  float* ss_smem = rows_smem + mts * nkb * 16 * COLS;
  // one row tile of one k block: the block sum of 16 rows x COLS columns goes to LDS
  auto multiply = [&](f32x4 (&av)[16], int mt, int b) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < 16; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[g][e], av[g][e], acc, 0, 0, 0);
    // lane (l16, kk): row m = l16, columns 4 kk + r
    if (kk * 4 < COLS) *(f32x4*)(&rows_smem[((mt * nkb + b) * 16 + l16) * COLS + kk * 4]) = acc;
  };
  // NORM: the rows times the norm's weights, their squares added up on the way (one row tile of one k block)
  auto scale_rows = [&](auto whole, f32x4 (&av)[16], int mt, int b) {
    f32x4 nw[16];
    load16(whole, nw, norm_w, b * F_KBLOCK);      // 4 * K bytes, from the caches
    float ss = 0.f;
#pragma unroll
    for (int g = 0; g < 16; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ss = __builtin_fmaf(av[g][e], av[g][e], ss);
        av[g][e] *= nw[g][e];
      }
    // the four lanes of a row (one per k quarter): every lane gets (s0 + s1) + (s2 + s3)
    ss += __shfl_xor(ss, 16, TL_WAVE);
    ss += __shfl_xor(ss, 32, TL_WAVE);
    if (kk == 0) ss_smem[(mt * nkb + b) * 16 + l16] = ss;
  };
  constexpr int AHEAD = FR_WAVES * F_KBLOCK;        // from a wave's block to its next
  auto block = [&](auto whole, auto next_whole, int b) {
    const int kb = b * F_KBLOCK;
    // The next block's weights are requested once this block is done: the norm's weights, or the next row tile, have the registers.
    f32x4 av[16];
    load16(whole, av, a_row(0), kb);
    if constexpr (WIDE) {
      f32x4 av2[16];
      for (int mt = 0; mt < mts; mt += 2) {
        if (mt + 1 < mts) load16(whole, av2, a_row(mt + 1), kb);
        multiply(av, mt, b);
        if (mt + 1 < mts) {
          if (mt + 2 < mts) load16(whole, av, a_row(mt + 2), kb);
          multiply(av2, mt + 1, b);
        }
      }
      if (b + FR_WAVES < nkb) load16(next_whole, wv, wrow, kb + AHEAD);
    } else {
      for (int mt = 0; mt < mts; ++mt) {
        if (mt > 0) load16(whole, av, a_row(mt), kb);
        scale_rows(whole, av, mt, b);
        multiply(av, mt, b);
      }
      if (b + FR_WAVES < nkb) load16(next_whole, wv, wrow, kb + AHEAD);
    }
  };
  for (int b = wave; b < nkb; b += FR_WAVES) {
    const bool whole = (b + 1) * F_KBLOCK <= K, next_whole = (b + FR_WAVES + 1) * F_KBLOCK <= K;
    if (whole && next_whole) block(std::true_type{}, std::true_type{}, b);
    else if (whole) block(std::true_type{}, std::false_type{}, b);
    else block(std::false_type{}, std::false_type{}, b);
  }
  __syncthreads();
  for (int e = tid; e < mts * 16 * COLS; e += FR_THREADS) {
    const int mt = e / (16 * COLS), r = (e % (16 * COLS)) / COLS, c = e % COLS;
    float t = 0.f;
    for (int b = 0; b < nkb; ++b) t += rows_smem[((mt * nkb + b) * 16 + r) * COLS + c];
    if constexpr (NORM) {
      float q = 0.f;
      for (int b = 0; b < nkb; ++b) q += ss_smem[(mt * nkb + b) * 16 + r];
      t *= f32_norm_factor(q, K, eps);
    }
    const int m = (mt0 + mt) * 16 + r, n = n0 + c;
    if constexpr (!NORM) {
      if (row_scale && m < M) t *= row_scale[m];    // the factor of a norm in front (norm_prescale_f32_kernel)
    }
    if constexpr (SWIGLU) {   // columns (2j, 2j+1) = (gate_j, up_j); N and n0 are even
      const float u = __shfl_down(t, 1, TL_WAVE);
      if (m < M && n < N && (c & 1) == 0) out[(int64_t)m * ldo + n / 2] = swiglu_pair(t, u);
    } else {
      if (m < M && n < N) {
        const int64_t at = (int64_t)m * ldo + n;
        out[at] = residual ? t + residual[at] : t;
      }
    }
  }
}

// The same product for one tile of rows (decode steps of up to 16), by whole lines.  gemm_f32_rows_kernel loads in the matrix instruction's order, 64
// bytes of each of sixteen rows an instruction, at 37 GB/s a unit; a unit gets 105 from its L2 in whole lines.  Here a wave fetches runs
// of 512 bytes, half a k block of sixteen rows at a time, of activations and of each column tile, and turns them into
// operands through 8 KB of LDS of its own; the next half block is on its way meanwhile.  Same blocks, same groups, same order: the bits of gemm_f32_kernel.
// 8 rows, weights from memory: 2,560 x 2,048 10.7 -> 8.5 us, 2,048 x 2,048 8.1 -> 6.6, 11,264 x 2,048 gated 23.0 -> 21.4, 2,048 x 5,632 16.4 ->
// 13.0, 32,000 x 2,048 63.7 -> 58.2, 6,144 x 4,096 28.3 -> 22.6; 16 rows of 2,048 x 5,632 25.4 -> 16.5.
// NORM: the product is that of `a`'s RMSNorm, as described there.
//
// CT (one row tile only): a workgroup owns CT column tiles side by side.  The activations of a k block,
// which weigh as much as one tile's weights, are fetched once for all of them, and a wide product
// (gate and up, the output head) becomes one or two rounds of workgroups instead of three to eight.
// Each tile's next half block is requested as soon as this one has left its registers for LDS.  A tile's block sums are what they are
// with one tile a workgroup, bit for bit.
//
// PAIR (8 columns, at most 8 rows): the matrix tile of 16 x 16 then holds two k blocks at
// once.  Operand rows 0 to 7 are the 8 columns (and the 8 activation rows) at the k of one block, rows
// 8 to 15 the same columns and rows at the k of the next; the two diagonal 8 x 8 blocks of the result
// are the two block sums, each accumulated from zero in the order it has everywhere else, and the
// rest of the tile is dropped.  Without it the second half of the tile repeats the first: every load
// instruction then fetches half of what it could, and 8 columns are what bounds these products,
// since a workgroup is as fast as its loads.  A wave takes pairs of blocks instead of blocks.
constexpr int FL_HALF = F_KBLOCK / 2, FL_AREA = 16 * FL_HALF;      // k of a step; floats of a wave's area
constexpr int64_t FL_MAX_STRIDE = 1 << 24;                         // floats between rows: sixteen rows end below 2^30 bytes, and offsets below twice that
constexpr size_t FL_STAGE_BYTES = (size_t)FR_WAVES * FL_AREA * sizeof(float), FL_SUM_BYTES = 96 * 1024;      // together a unit's LDS
template <bool SWIGLU, int CT, bool PAIR, bool NORM>
__global__ __launch_bounds__(FR_THREADS) void gemm_f32_lines_kernel(const F32RowsNorm norm, const float* __restrict__ a, const float* __restrict__ w,
                                                                    float* __restrict__ out, const float* __restrict__ residual,
                                                                    int M, int N, int K, int64_t lda, int64_t ldo,
                                                                    const float* __restrict__ row_scale, int cw) {
  static_assert(CT == 1 || (!PAIR && !NORM), "pairs of k blocks and the norm: one column tile");
  constexpr int UNIT = PAIR ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) float lines_smem[];
  constexpr int ROWS = PAIR ? 8 : 16;
  const int nkb = (K + F_KBLOCK - 1) / F_KBLOCK, units = (nkb + UNIT - 1) / UNIT;
  const int col_bits = PAIR || (CT == 1 && cw <= 8) ? 3 : 4, cols = 1 << col_bits;      // columns of a tile that have sums
  float* sums = lines_smem + FR_WAVES * FL_AREA;            // [CT][k blocks][ROWS][cols], NORM: + [k blocks][ROWS]
  float* squares = sums + CT * nkb * ROWS * cols;
  const int tid = threadIdx.x, lane = tid % TL_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / TL_WAVE);
  const int l16 = lane % 16, kk = lane / 16, lr = lane / 32, lc = lane % 32;
  const int n0 = blockIdx.x * cw, stride_a = (int)lda;
  // Both operands as buffers: rows beyond the matrices, and steps beyond this wave's, read as zeros and fetch nothing.  All of an
  // offset is a lane's own (scalar offset 0): that is what the check of a buffer's end is documented for.
  auto rows_of = [&](const float* base, int stride, int rows) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, rows > 0 ? ((rows - 1) * stride + K) * 4 : 0, 0x00020000);
  };
  const auto buf_w = rows_of(w + (int64_t)n0 * K, K, min(cw, N - n0)), buf_a = rows_of(a, stride_a, M);
  const int mine = wave < units ? 2 * ((units - wave + FR_WAVES - 1) / FR_WAVES) : 0;      // half blocks (PAIR: of two blocks)
  auto first_k = [&](int s) { return ((wave + s / 2 * FR_WAVES) * UNIT * F_KBLOCK) + s % 2 * FL_HALF; };
  // load i of a step: 16 bytes of row 2 i + lane / 32 (PAIR: from row 8 on the rows 0 .. of the next k block), k 4 (lane % 32) ..
  constexpr int PLACES = PAIR ? 4 : 8, BEYOND = 0x40000000;      // bytes: beyond every buffer here
  int at_w[PLACES], at_a[PLACES];
#pragma unroll
  for (int i = 0; i < PLACES; ++i) {
    const int from = mine > 0 ? first_k(0) * 4 : BEYOND;
    at_w[i] = ((2 * i + lr) * K + lc * 4) * 4 + from;
    at_a[i] = ((2 * i + lr) * stride_a + lc * 4) * 4 + from;
  }
  auto advance = [&](int (&at)[PLACES], int s) {      // from step s to the next
    const int by = s + 1 >= mine ? BEYOND : (s % 2 == 0 ? FL_HALF : FR_WAVES * UNIT * F_KBLOCK - FL_HALF) * 4;
#pragma unroll
    for (int i = 0; i < PLACES; ++i) at[i] += by;
  };
  struct Step {
    f32x4 a[8], w[CT][8];
  };
  auto load_tile = [&](f32x4 (&v)[8], auto buf, const int (&at)[PLACES], int tile) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(buf, at[i % PLACES] + tile + i / PLACES * F_KBLOCK * 4, 0, 0));
  };
  float* own = lines_smem + wave * FL_AREA;
  // chunk c of row r stands at place c ^ r of its 32; what lies beyond K is zero
  auto put = [&](f32x4 (&v)[8], int k0) {
    if (k0 + (PAIR ? F_KBLOCK : 0) + FL_HALF > K)      // uniform
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const bool in = k0 + (PAIR && i >= 4 ? F_KBLOCK : 0) + lc * 4 < K;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] = in ? v[i][e] : 0.f;
      }
#pragma unroll
    for (int i = 0; i < 8; ++i) *(f32x4*)(own + (2 * i + lr) * FL_HALF + (lc ^ (2 * i + lr)) * 4) = v[i];
    wave_sync();
  };
  auto get = [&](f32x4 (&v)[8]) {
#pragma unroll
    for (int g = 0; g < 8; ++g) v[g] = *(const f32x4*)(own + l16 * FL_HALF + ((g * 4 + kk) ^ l16) * 4);
    wave_sync();
  };
  Step st;
  load_tile(st.a, buf_a, at_a, 0);      // in the order in which they are needed
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) load_tile(st.w[ct], buf_w, at_w, ct * 16 * K * 4);
  // NORM: the norm's weights of a step, as operands (4 K bytes, from the caches), requested a step ahead
  f32x4 nw[NORM ? 8 : 1];
  auto load_norm = [&](int s) {
    if constexpr (NORM)
#pragma unroll
      for (int g = 0; g < 8; ++g)
        nw[g] = load_k4<true>(norm.w, first_k(min(s, mine - 1)) + (PAIR && l16 >= 8 ? F_KBLOCK : 0) + g * 16 + kk * 4, K);
  };
  if (mine > 0) load_norm(0);
  f32x4 acc[CT];
  float ss = 0.f;
  for (int s = 0; s < mine; ++s) {
    const int k0 = first_k(s);
    if (s % 2 == 0) {
      ss = 0.f;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    f32x4 av[8];
    put(st.a, k0);
    advance(at_a, s);
    load_tile(st.a, buf_a, at_a, 0);
    get(av);
    if constexpr (NORM) {      // the rows times the norm's weights, their squares added up on the way
#pragma unroll
      for (int g = 0; g < 8; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ss = __builtin_fmaf(av[g][e], av[g][e], ss);
          av[g][e] *= nw[g][e];
        }
      load_norm(s + 1);
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      f32x4 wv[8];
      put(st.w[ct], k0);
      if (ct == 0) advance(at_w, s);
      load_tile(st.w[ct], buf_w, at_w, ct * 16 * K * 4);
      get(wv);
#pragma unroll
      for (int g = 0; g < 8; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[g][e], av[g][e], acc[ct], 0, 0, 0);
    }
    if (s % 2 == 1) {      // the block's sums: lane (l16, kk) has row l16, columns 4 kk + r
      const int b = (wave + s / 2 * FR_WAVES) * UNIT + (PAIR ? l16 / 8 : 0);
      if constexpr (NORM) {      // the four lanes of a row, one per k quarter: (s0 + s1) + (s2 + s3)
        ss += __shfl_xor(ss, 16, TL_WAVE);
        ss += __shfl_xor(ss, 32, TL_WAVE);
        if (kk == 0 && b < nkb) squares[b * ROWS + l16 % ROWS] = ss;
      }
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        if constexpr (PAIR) {     // rows 0..7 x columns 0..7: the first block; 8..15 x 8..15: the second
          if ((l16 < 8) == (kk < 2) && b < nkb) *(f32x4*)(&sums[(b * ROWS + l16 % 8) * 8 + (kk % 2) * 4]) = acc[ct];
        } else {
          if (kk * 4 < cols) *(f32x4*)(&sums[(((ct * nkb + b) * ROWS + l16) << col_bits) + kk * 4]) = acc[ct];
        }
      }
    }
  }
  __syncthreads();
  for (int e = tid; e < CT * ROWS * cols; e += FR_THREADS) {
    const int ct = e / ROWS >> col_bits, r = (e >> col_bits) % ROWS, c = e % cols;
    float t = 0.f;
    for (int b = 0; b < nkb; ++b) t += sums[(((ct * nkb + b) * ROWS + r) << col_bits) + c];
    const int n = n0 + ct * 16 + c;
    if constexpr (NORM) {
      float q = 0.f;
      for (int b = 0; b < nkb; ++b) q += squares[b * ROWS + r];
      t *= f32_norm_factor(q, K, norm.eps);
    } else if (row_scale && r < M) {
      t *= row_scale[r];      // the factor of a norm in front (norm_prescale_f32_kernel)
    }
    const bool there = r < M && n < N && ct * 16 + c < cw;
    if constexpr (SWIGLU) {   // columns (2j, 2j+1) = (gate_j, up_j); N and n0 are even
      const float u = __shfl_down(t, 1, TL_WAVE);
      if (there && (c & 1) == 0) out[(int64_t)r * ldo + n / 2] = swiglu_pair(t, u);
    } else if (there) {
      const int64_t at = (int64_t)r * ldo + n;
      out[at] = residual ? t + residual[at] : t;
    }
  }
}

// ==================================================================== bfloat16
// Tiles of BM x BN outputs, k in steps of 64, WM x WN wave64, each owning (BM/WM) x (BN/WN)
// outputs as 32x32x16 MFMA tiles, or as 16x16x32 (operands straight into LDS).  Operand tiles go global -> registers -> LDS; LDS is
// double-buffered so an iteration needs one barrier, and the global loads of the next k step are
// in flight while the current one is multiplied.  Or they go straight into LDS, three or four buffers in turn
// (tile_mode says where), and the loads of the next two or three k steps are in flight; the 256 x 256 tile's two
// buffers are replaced quarter by quarter (kPhased).
//
// Tile shapes: 256 x 256 (eight waves of 128 x 64), 256 x 128, 128 x 128 and 64 x 128.  The larger
// the tile, the fewer operand bytes and LDS reads per flop and the higher the rate on a full chip;
// small products take small tiles all the same, because 256 compute units want at least that many
// workgroups (launch_gemm_bf16_any estimates the time of each shape and takes the best).
constexpr int B_BK = 64;
constexpr int B_LD = B_BK + 8;  // LDS row stride in elements: 144 bytes, keeps 16-byte alignment

// What the epilogue of the tiled kernel does to a row besides the product: a factor per row
// (`row_scale`), or a norm handed from product to product as the few-row kernel does it (see
// SkinnyArgs).  The producer (float32 output, no SiLU-gate, N a multiple of 64, ldo of 4) also writes
// emit_operand[m, n] = bf16(emit_w[n] * out[m, n]) and, for every 64 columns, the sum of out^2 into
// emit_sumsq[m, n / 64] (rows of `emit_parts` parts).  The consumer takes such an operand as `a`
// and in_sumsq [rows, in_parts], and its row factor is 1 / sqrt(sum / in_width + in_eps).
struct TileNorm {
  const float* row_scale = nullptr;
  const void* emit_w = nullptr;
  int emit_w_is_f32 = 0;
  int act = kActNone;                 // bfloat16 output: applied before rounding
  bf16_t* emit_operand = nullptr;
  int64_t emit_ld = 0;                // row stride of the operand
  float* emit_sumsq = nullptr;
  int emit_parts = 0;
  const float* in_sumsq = nullptr;
  int in_parts = 0, in_width = 0;
  float in_eps = 0.f;
  // Rows in groups with weights of their own: every aligned run of `group_rows` rows (a multiple of every tile
  // height) multiplies the weight matrix tile_group[run] * group_stride elements behind `w`; a run whose entry is
  // negative holds no row and is skipped.
  int group_rows = 0;
  const int32_t* tile_group = nullptr;
  int64_t group_stride = 0;
  Gate gate;                          // a gated product's unit
  TileNorm() = default;
  TileNorm(const float* rs, int act_ = kActNone) : row_scale(rs), act(act_) {}
};

template <int BM, int BN, int WM, int WN>
struct GemmShape {
  static constexpr int THREADS = WM * WN * TL_WAVE;
  static constexpr int TM = BM / WM, TN = BN / WN;        // a wave's outputs
  static constexpr int AC = BM * (B_BK / 8) / THREADS, WC = BN * (B_BK / 8) / THREADS;
  // operand tiles in LDS: two, or, straight from memory, as many as make three in flight beside the one in use
  static constexpr int BUFS = BM + BN > 384 ? 2 : BM + BN > 256 ? 3 : 4;
  static constexpr size_t smem(bool direct) {
    return direct ? (size_t)BUFS * (BM + BN) * B_BK * sizeof(bf16_t) : (size_t)2 * (BM + BN) * B_LD * sizeof(bf16_t);
  }
  static constexpr size_t smem_all(bool direct) { return smem(direct) + BM * sizeof(float); }     // and a factor per row
  static_assert(TM % 32 == 0 && TN % 32 == 0 && AC >= 1 && WC >= 1, "tile does not divide");
};

// K must be a multiple of 8 (16-byte chunks of bf16 never straddle the end).
// How operand tiles get into LDS: through registers, zeros beyond the end of a row (kTail); through registers, the inner
// size a multiple of the k step (kWhole); likewise, but straight from memory (kDirect).
// Straight from memory in quarters, each replaced as soon as it has been read (kPhased: the 256 x 256 tile).
constexpr int kTail = 0, kWhole = 1, kDirect = 2, kPhased = 3;
// What is known of the residual where the epilogue is compiled (kNoResidual: none, or one of rows without whole vectors).
constexpr int kNoResidual = 0, kResidual = 1, kAnyForm = 2;
template <int BM, int BN, int WM, int WN, typename TO, int SWIGLU, int MODE>
__global__ __launch_bounds__(WM * WN * TL_WAVE) void gemm_bf16_kernel(const bf16_t* __restrict__ a,
                                                                      const bf16_t* __restrict__ w,
                                                                      TO* __restrict__ out,
                                                                      const float* __restrict__ residual,
                                                                      const TileNorm nm, int M, int N, int K,
                                                                      int64_t lda, int64_t ldo, int k_per_split) {
  using S = GemmShape<BM, BN, WM, WN>;
  constexpr int THREADS = S::THREADS;
  constexpr bool PHASED = MODE == kPhased, DIRECT = MODE == kDirect || PHASED;
  constexpr int LD = DIRECT ? B_BK : B_LD;              // row stride of a staged tile
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  constexpr int BUFS = DIRECT ? S::BUFS : 2;
  bf16_t* As = (bf16_t*)smem_raw;                       // [BUFS][BM][LD]
  bf16_t* Ws = As + BUFS * BM * LD;                     // [BUFS][BN][LD]
  const int tid = threadIdx.x, lane = tid % TL_WAVE, wave = tid / TL_WAVE;
  const int wm = wave / WN, wn = wave % WN;
  // k_per_split > 0 (a multiple of the k step): the inner size is split over workgroups, each
  // writing its float32 partial product [M, N] behind `out` (no epilogue); a second kernel adds
  // them up.  That is how products with few output tiles still fill the chip.
  const int splits = k_per_split > 0 ? (K + k_per_split - 1) / k_per_split : 1;
  const int tiles_m = (M + BM - 1) / BM, tiles = tiles_m * ((N + BN - 1) / BN), total = tiles * splits;
  const int t_all = xcd_tile(blockIdx.x, total);
  if (t_all >= total) return;                           // the grid is padded to a multiple of 8
  const int split = t_all / tiles, t = t_all % tiles;
  int tile_m, tile_n;
  tile_place(t, tiles_m, (N + BN - 1) / BN, DIRECT || BM == 256, &tile_m, &tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int kbase = split * k_per_split;
  const int kend = k_per_split > 0 ? min(K, kbase + k_per_split) : K;
  if (k_per_split > 0) out += (int64_t)split * M * ldo;
  if (nm.tile_group) {      // uniform: this tile's rows belong to one group, with weights of its own
    const int group = __builtin_amdgcn_readfirstlane(nm.tile_group[m0 / nm.group_rows]);
    if (group < 0) return;
    w += (int64_t)group * nm.group_stride;
  }

  // Straight from memory: 16 x 16 matrix tiles; through registers: 32 x 32.
  constexpr int MI = S::TM / 16, NJ = S::TN / 16, MI32 = S::TM / 32, NJ32 = S::TN / 32;
  f32x4 acc[DIRECT ? MI : 1][DIRECT ? NJ : 1];
  f32x16 acc32[DIRECT ? 1 : MI32][DIRECT ? 1 : NJ32];
  if constexpr (DIRECT) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  } else {
#pragma unroll
    for (int i = 0; i < MI32; ++i)
#pragma unroll
      for (int j = 0; j < NJ32; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc32[i][j][r] = 0.f;
  }

  // A norm handed over: the factors of this tile's rows are worked out once, here, where the loads
  // hide behind the main loop (16 threads share a row's parts out), and wait in LDS for the
  // epilogue; the barriers of the main loop lie in between.
  float* row_factor = (float*)(smem_raw + S::smem(DIRECT));      // [BM]
  if (nm.in_sumsq) {      // uniform
    for (int r = tid / 16; r < BM; r += THREADS / 16) {
      const int64_t at = (int64_t)min(m0 + r, M - 1) * nm.in_parts;
      float t = 0.f;
      for (int q = tid % 16; q < nm.in_parts; q += 16) t += nm.in_sumsq[at + q];
      t = group_sum<16>(t);
      if (tid % 16 == 0) row_factor[r] = 1.f / sqrtf(t / (float)nm.in_width + nm.in_eps);
    }
  }

  // One k step of both operand tiles is AC + WC 16-byte pieces per thread, fetched with buffer
  // loads: the address is the tile's first row (the buffer's base, per workgroup) + an offset per
  // piece that never changes + the k offset, which is one scalar for all lanes, so a k step costs
  // no address arithmetic; and the buffer ends with the matrix, so rows beyond it read as zero
  // without a branch.  (A piece beyond K within a row is zeroed when it is written to LDS.)
  constexpr int PIECES = S::AC + S::WC;
  bf16x8 stage[PIECES];
  const int prow = tid / 8;                                // this thread's row within a pass
  // and its k offset.  DIRECT: the wave's 64 pieces land in LDS side by side, 8 rows of 8, so a row cannot be padded;
  // piece c of row r holds the k of piece c ^ (r / 2 % 8) instead, and 16 rows at one k then touch every bank once
  // (conflicts are 0.7 % of the cycles LDS works, 1,944 rows, 2,048 x 5,632, and as many with padded rows: the epilogue's).
  const int pk = DIRECT ? ((tid % 8) ^ (prow / 2 % 8)) * 8 : (tid % 8) * 8;
  constexpr int PASS = THREADS / 8;                        // rows per pass
  auto tile_buffer = [](const bf16_t* first_row, int rows, int64_t ld, int K_) {
    const int64_t bytes = rows > 0 ? ((int64_t)(rows - 1) * ld + K_) * 2 : 0;
    return __builtin_amdgcn_make_buffer_rsrc((void*)first_row, 0, (int)(bytes < 0x7fffffff ? bytes : 0x7fffffff), 0x00020000);
  };
  auto buffer_words = [](const bf16_t* first_row, int rows, int64_t ld, int K_) {      // the same as four words
    const int64_t bytes = rows > 0 ? ((int64_t)(rows - 1) * ld + K_) * 2 : 0;
    const uint64_t at = (uint64_t)first_row;
    return tl_rsrc_words{(int)(uint32_t)at, (int)(uint32_t)(at >> 32) & 0xffff, (int)(bytes < 0x7fffffff ? bytes : 0x7fffffff),
                         0x00020000};
  };
  const __amdgpu_buffer_rsrc_t buf_a = tile_buffer(a + (int64_t)m0 * lda, min(M - m0, BM), lda, K);
  const __amdgpu_buffer_rsrc_t buf_w = tile_buffer(w + (int64_t)n0 * K, min(N - n0, BN), K, K);
  const tl_rsrc_words words_a = buffer_words(a + (int64_t)m0 * lda, min(M - m0, BM), lda, K);
  const tl_rsrc_words words_w = buffer_words(w + (int64_t)n0 * K, min(N - n0, BN), K, K);
  int piece_off[PIECES];                                   // bytes from the tile's first row
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const bool is_a = p < S::AC;
    const int r = (is_a ? p : p - S::AC) * PASS + prow;
    piece_off[p] = (int)(((int64_t)r * (is_a ? lda : (int64_t)K) + pk) * 2);
  }
  typedef int tl_i32x4 __attribute__((ext_vector_type(4)));
  auto gload1 = [&](int k0, int p) {
    const tl_i32x4 v = __builtin_bit_cast(
        tl_i32x4, __builtin_amdgcn_raw_buffer_load_b128(p < S::AC ? buf_a : buf_w, piece_off[p], k0 * 2, 0));
    stage[p] = __builtin_bit_cast(bf16x8, v);
  };
  auto lds_write1 = [&](int buf, int k0, int p) {
    const bool is_a = p < S::AC;
    const int r = (is_a ? p : p - S::AC) * PASS + prow;
    const bool ok = MODE != kTail || k0 + pk < K;
    bf16x8 z = {};
    bf16_t* dst = is_a ? As + (buf * BM + r) * LD + pk : Ws + (buf * BN + r) * LD + pk;
    *(bf16x8*)dst = ok ? stage[p] : z;
  };
  // DIRECT: piece p of the k step at k0, straight into a buffer.
  auto direct1 = [&](int buf, int k0, int p) {
    const bool is_a = p < S::AC;
    const int r = (is_a ? p : p - S::AC) * PASS + wave * 8;
    bf16_t* dst = is_a ? As + (buf * BM + r) * LD : Ws + (buf * BN + r) * LD;
    tl_load_to_lds(is_a ? words_a : words_w, tl_lds_address(dst), piece_off[p], k0 * 2);
  };
  // pieces [n * per, (n + 1) * per) of `total`, for spreading `total` operations over slots
  auto spread = [](int n, int total, int slots, auto&& op) {
    const int per = (total + slots - 1) / slots;
#pragma unroll
    for (int p = n * per; p < (n + 1) * per; ++p)
      if (p < total) op(p);
  };

  const int nk = (kend - kbase + B_BK - 1) / B_BK;
  if constexpr (PHASED) {
    static_assert(BM == 256 && BN == 256 && WM == 2 && WN == 4 && BUFS == 2, "quarters of the 256 x 256 tile");
    // With both operands through registers and one barrier a k step the matrix pipes were busy for 69 % of the time (8192^3;
    // the loads of two whole buffers straight into LDS are too late, 1,138 us where registers take 889); so, 723 us.  2,048
    // rows, 28,672 x 4,096: 428 -> 360 us (1.34 PFLOP/s); 4,096 x 14,336 260 -> 217, where half the units work and run at
    // 2.2 GHz; on a full chip the part clocks at 1.7 to 1.75 GHz, and power bounds it: instructions of 16 x 16 x 32 move
    // half the sums of those of 32 x 32 x 16 for the same products (781 -> 723 and 381 -> 360 us; the bits are the same).
    // A k step is four items of 128 rows, in the order in which they are read: a weight half, the first half of the
    // activations, the other weight half, the rest of the activations.  A half holds the rows that every wave needs for half
    // of its outputs: of the activations 64 of each 128, of the weights 32 of each 64.  Which weight half comes first
    // alternates from step to step, so that a phase of sixteen matrix instructions always has one new half to read.  Phase f
    // reads item f + 1 into registers, asks for item f + 7 and waits for item f + 2: five items, a step and a quarter of
    // work, stay on their way.  The waves of a SIMD take turns: while one multiplies, the other reads; between two barriers
    // each half of the workgroup does one of the two, the second half a turn behind.  Item f + 7 takes the place of item
    // f - 1: it was read in phase f - 2, and by the end of that phase's products, which both halves have behind them a
    // barrier before the first asks for item f + 7, its reads have been waited for.
    const unsigned int lds_wave = tl_lds_address(As + __builtin_amdgcn_readfirstlane(wave) * 8 * LD);
    int off[2][2][2];                                      // of a thread's two pieces of an item: [weights][half][piece]
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        off[0][h][q] = (int)(((int64_t)(q * 128 + h * 64 + prow) * lda + pk) * 2);
        off[1][h][q] = (int)(((int64_t)(q * 128 + prow / 32 * 64 + h * 32 + prow % 32) * K + pk) * 2);
      }
    // Half h of the operand's k step kt.  A step behind the last is asked for from a buffer of no bytes: it reads as zeros.
    auto fill = [&](int buf, bool weights, int h, int kt) {
      const unsigned int dst = lds_wave + ((weights ? BUFS * BM : 0) + (buf * 2 + h) * 128) * LD * 2;
      tl_rsrc_words from = weights ? words_w : words_a;
      from[2] = kt < nk ? from[2] : 0;
#pragma unroll
      for (int q = 0; q < 2; ++q)
        tl_load_to_lds(from, dst + q * 64 * LD * 2, off[weights][h][q], (kbase + min(kt, nk - 1) * B_BK) * 2);
    };
    bf16x8 fa[2][4], fw[2][2][2];                          // fragments of a half of the activations, of both weight halves
    const bf16_t* pa = As + (wm * 64 + lane % 16) * LD;
    const bf16_t* pw = Ws + (wn * 32 + lane % 16) * LD;
    const int key = lane % 16 / 2;
    auto read_a = [&](int buf, int h) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          fa[ks][i] = *(const bf16x8*)(pa + ((buf * 2 + h) * 128 + i * 16) * LD + ((ks * 4 + lane / 16) ^ key) * 8);
    };
    auto read_w = [&](int buf, int h) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          fw[h][ks][j] = *(const bf16x8*)(pw + ((buf * 2 + h) * 128 + j * 16) * LD + ((ks * 4 + lane / 16) ^ key) * 8);
    };
    auto meet = [&]() {
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    // Phase P of the k step kt, whose weight half F comes first.
    auto phase = [&](auto p_, auto first, int kt) {
      constexpr int P = decltype(p_)::value, F = decltype(first)::value;
      if constexpr (P == 0) read_a(F, 0);
      if constexpr (P == 1) read_w(F, F ^ 1);
      if constexpr (P == 2) read_a(F, 1);
      if constexpr (P == 3) read_w(F ^ 1, F ^ 1);
      if constexpr (P == 0) fill(F ^ 1, false, 1, kt + 1);
      else fill(F, P % 2 == 1, P == 1 ? F : P == 3 ? F ^ 1 : 0, kt + 2);
      tl_wait_loads<10>();
      meet();
      constexpr int A = P / 2, B = P == 0 || P == 3 ? F : F ^ 1;
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[A * 4 + i][B * 2 + j] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[B][ks][j], fa[ks][i], acc[A * 4 + i][B * 2 + j], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
      if constexpr (P == 3) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // what it read is used a phase later
      meet();
    };
    auto step = [&](auto first, int kt) {
      phase(std::integral_constant<int, 0>{}, first, kt);
      phase(std::integral_constant<int, 1>{}, first, kt);
      phase(std::integral_constant<int, 2>{}, first, kt);
      phase(std::integral_constant<int, 3>{}, first, kt);
    };
#pragma unroll
    for (int b = 0; b < 2; ++b) {                          // items 0 to 6
      fill(b, true, b, b);
      fill(b, false, 0, b);
      fill(b, true, b ^ 1, b);
      if (b == 0) fill(b, false, 1, b);
    }
    tl_wait_loads<10>();
    meet();
    read_w(0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    meet();
    if (wm == 1) meet();                                   // this half of the waves stays one turn behind
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
      step(std::integral_constant<int, 0>{}, kt);
      step(std::integral_constant<int, 1>{}, kt + 1);
    }
    // (a pair's second step of zeros cost 1 us a tile: 300 rows, 8,192 x 64 11.0 us, 9.9 so; 2,047 rows, 11,264 x 2,112 101.6, 99.7)
    if (kt < nk) step(std::integral_constant<int, 0>{}, kt);
    tl_wait_loads<0>();
    if (wm == 0) meet();
    meet();
  } else if constexpr (DIRECT) {
    // Two k32 steps a buffer, software-pipelined by hand, because all waves of a workgroup meet at the barrier of every k step:
    // while the MFMAs of one run, the fragments of the next are read; the second is multiplied behind the barrier, ahead of
    // which the wave has waited for its part of the next buffer, and asks for the pieces that replace this one.
    // (1,944 rows, 2,048 x 5,632, 128 x 128 tiles: 52.9 us with 32 x 32 x 16 instructions, 48.8 so; 2,048 rows, 4,096 x 14,336,
    // 256 x 128 tiles: 213 and 201.  Through registers the same takes 5 to 20 % more: LDS writes then stand right ahead of the
    // barrier, or the loads behind them come late.)
    // MFMA operands of one k32 step: NJ weight pieces, then MI activation pieces, in the order of use
    struct Frag {
      bf16x8 w[NJ], a[MI];
    };
    constexpr int FRAG = NJ + MI;
    const bf16_t* ra = As + (wm * S::TM + lane % 16) * LD;
    const bf16_t* rw = Ws + (wn * S::TN + lane % 16) * LD;
    auto lds_read1 = [&](Frag& f, int buf, int ks, int p) {
      const int at = ((ks * 4 + lane / 16) ^ (lane % 16 / 2)) * 8;         // this lane's place in a row
      if (p < NJ) f.w[p] = *(const bf16x8*)(rw + (buf * BN + p * 16) * LD + at);
      else f.a[p - NJ] = *(const bf16x8*)(ra + (buf * BM + (p - NJ) * 16) * LD + at);
    };
    // The MFMAs of one k32 step, with memory operations issued between them: slot(n) comes after the
    // n-th pair.  The result tile is transposed (rows = n, columns = m) so that a lane holds four
    // consecutive n of one output row and can store them as one vector.  The scheduling barriers
    // keep the compiler from gathering the memory operations back into one place.
    constexpr int SLOTS = MI * NJ / 2;
    auto group = [&](const Frag& f, auto&& slot) {
#pragma unroll
      for (int n = 0; n < SLOTS; ++n) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int i = n * 2 / NJ, j = n * 2 % NJ + h;
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[j], f.a[i], acc[i][j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        slot(n);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int p = 0; p < PIECES; ++p) direct1(0, kbase, p);
#pragma unroll
    for (int b = 1; b < BUFS; ++b)
      if (b < nk) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) direct1(b, kbase + b * B_BK, p);
      }
    if (nk >= BUFS) tl_wait_loads<(BUFS - 1) * PIECES>();
    else tl_wait_loads<0>();
    __syncthreads();
    Frag f0, f1;
#pragma unroll
    for (int p = 0; p < FRAG; ++p) lds_read1(f0, 0, 0, p);
    static_assert(SLOTS >= 2, "a wave owns at least two pairs of MFMA tiles");
    auto step = [&](auto has_next, auto has_next2, int kt) {
      constexpr bool NX = decltype(has_next)::value, NX2 = decltype(has_next2)::value;
      const int cur = kt % BUFS, nxt = (kt + 1) % BUFS, k2 = kbase + (kt + BUFS) * B_BK;
      group(f0, [&](int n) {
        if (n < SLOTS / 2) spread(n, FRAG, SLOTS / 2, [&](int p) { lds_read1(f1, cur, 1, p); });
      });
      if constexpr (NX) tl_wait_loads<NX2 ? (BUFS - 2) * PIECES : 0>();      // the next tile has arrived
      __syncthreads();
      group(f1, [&](int n) {
        if constexpr (NX) spread(n, FRAG, SLOTS, [&](int p) { lds_read1(f0, nxt, 0, p); });
        if constexpr (NX2) spread(n, PIECES, SLOTS, [&](int p) { direct1(cur, k2, p); });     // cur has been read
      });
    };
    int kt = 0;
    for (; kt + BUFS < nk; ++kt) step(std::true_type{}, std::true_type{}, kt);
    for (; kt + 1 < nk; ++kt) step(std::true_type{}, std::false_type{}, kt);
    step(std::false_type{}, std::false_type{}, kt);
  } else {
    // MFMA operands of one k16 step: NJ32 weight pieces, then MI32 activation pieces, in the order of use
    struct Frag {
      bf16x8 w[NJ32], a[MI32];
    };
    constexpr int FRAG = NJ32 + MI32;
    const bf16_t* ra = As + (wm * S::TM + lane % 32) * LD + (lane / 32) * 8;
    const bf16_t* rw = Ws + (wn * S::TN + lane % 32) * LD + (lane / 32) * 8;
    auto lds_read1 = [&](Frag& f, int buf, int ks, int p) {
      const int at = ks * 16;
      if (p < NJ32) f.w[p] = *(const bf16x8*)(rw + (buf * BN + p * 32) * LD + at);
      else f.a[p - NJ32] = *(const bf16x8*)(ra + (buf * BM + (p - NJ32) * 32) * LD + at);
    };
    // The MFMAs of one k16 step, with memory operations issued between them: slot(n) comes after the
    // n-th MFMA.  The result tile is transposed (rows = n, columns = m) so that a lane holds four
    // consecutive n of one output row and can store them as one vector.  The scheduling barriers
    // keep the compiler from gathering the memory operations back into one place.
    constexpr int SLOTS = MI32 * NJ32;
    auto group = [&](const Frag& f, auto&& slot) {
#pragma unroll
      for (int n = 0; n < SLOTS; ++n) {
        acc32[n / NJ32][n % NJ32] =
            __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[n % NJ32], f.a[n / NJ32], acc32[n / NJ32][n % NJ32], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        slot(n);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // The loop is software-pipelined by hand, because all waves of a workgroup meet at the barrier
    // of every k step and so cannot cover for each other: while the MFMAs of one k16 step run, the
    // fragments of the next are read; the tile of step kt + 1 (loaded into registers during step
    // kt - 1) is written to the other LDS buffer in the middle of step kt, and the loads of tile
    // kt + 2 are issued right after; the last k16 step of a tile is multiplied after the barrier,
    // while the first fragments of the next tile are on their way.
#pragma unroll
    for (int p = 0; p < PIECES; ++p) gload1(kbase, p);
#pragma unroll
    for (int p = 0; p < PIECES; ++p) lds_write1(0, kbase, p);
    if (nk > 1) {
#pragma unroll
      for (int p = 0; p < PIECES; ++p) gload1(kbase + B_BK, p);
    }
    __syncthreads();
    Frag f0, f1;
#pragma unroll
    for (int p = 0; p < FRAG; ++p) lds_read1(f0, 0, 0, p);
    static_assert(SLOTS >= 2, "a wave owns at least two MFMA tiles");
    constexpr int HALF = SLOTS / 2;
    auto step = [&](auto has_next, auto has_next2, int kt) {
      constexpr bool NX = decltype(has_next)::value, NX2 = decltype(has_next2)::value;
      const int cur = kt & 1, nxt = cur ^ 1, k1 = kbase + (kt + 1) * B_BK, k2 = kbase + (kt + 2) * B_BK;
      group(f0, [&](int n) { spread(n, FRAG, SLOTS, [&](int p) { lds_read1(f1, cur, 1, p); }); });
      group(f1, [&](int n) {
        spread(n, FRAG, SLOTS, [&](int p) { lds_read1(f0, cur, 2, p); });
        if constexpr (NX)
          if (n >= SLOTS - HALF) spread(n - (SLOTS - HALF), PIECES / 2, HALF, [&](int p) { lds_write1(nxt, k1, p); });
      });
      group(f0, [&](int n) {
        spread(n, FRAG, SLOTS, [&](int p) { lds_read1(f1, cur, 3, p); });
        if constexpr (NX)
          if (n < HALF) spread(n, PIECES - PIECES / 2, HALF, [&](int p) { lds_write1(nxt, k1, PIECES / 2 + p); });
        if constexpr (NX2)
          if (n >= SLOTS - HALF) spread(n - (SLOTS - HALF), PIECES, HALF, [&](int p) { gload1(k2, p); });
      });
      __syncthreads();
      group(f1, [&](int n) {
        if constexpr (NX) spread(n, FRAG, SLOTS, [&](int p) { lds_read1(f0, nxt, 0, p); });
      });
    };
    int kt = 0;
    for (; kt + 2 < nk; ++kt) step(std::true_type{}, std::true_type{}, kt);
    for (; kt + 1 < nk; ++kt) step(std::true_type{}, std::false_type{}, kt);
    step(std::false_type{}, std::false_type{}, kt);
  }

  // Epilogue.  A lane's accumulators hold four consecutive n of 16 rows (straight from memory) or 32, so stored from
  // there a row would go out in 16-byte pieces.  Each wave therefore passes its result, 32 rows x
  // 64 columns at a time, through an LDS area of its own (the operand tiles are no longer read:
  // the last fragments were fetched before the loop's last barrier) and reads it back row by
  // row: 16 lanes then cover 256 contiguous bytes of one row, and so do the residual reads.
  static_assert(S::TN == 64, "the epilogue stages 64 columns per wave");
  constexpr int E_LD = 68;                 // floats per staged row: 16-byte aligned, conflict-free
  static_assert((size_t)WM * WN * 32 * E_LD * sizeof(float) <= S::smem(DIRECT), "staging areas fit the tile buffers");
  float* cstage = (float*)smem_raw + wave * (32 * E_LD);
  const bool vec_ok = (N % 4 == 0) && (ldo % 4 == 0);
  // Where a unit holds one workgroup and registers cost no wave, what 32 rows need from LDS is read together, and the residual
  // of the next 32 rows is requested before these are stored: one 256 x 256 tile of 64 k takes its epilogue from 6.6 to 4.5 us,
  // with a residual from 9.2 to 6.0 (on a full chip from 31 to 15); 3,288 rows, 2,048 x 2,048 with a residual, 256 x 128
  // tiles: 41.3 -> 35.7 us.
  constexpr bool TOGETHER = DIRECT || BM + BN > 256, NEXT = TOGETHER && sizeof(TO) == 4 && SWIGLU == 0;
  f32x4 res_next[NEXT ? 8 : 1];
  auto request_residual = [&](int i) {
    const int m = m0 + wm * S::TM + i * 32 + lane / 16, n = n0 + wn * S::TN + (lane % 16) * 4;
    const float* from = residual + (int64_t)m * ldo + n;
#pragma unroll
    for (int c8 = 0; c8 < 8; ++c8)
      if (m + c8 * 4 < M && n < N) res_next[NEXT ? c8 : 0] = *(const f32x4*)(from + c8 * 4 * ldo);      // others are not stored
  };
  auto load_emit_w = [&](float* wn, int n) {
    if (nm.emit_w_is_f32) {
      const f32x4 w4 = *(const f32x4*)((const float*)nm.emit_w + n);
      wn[0] = w4[0]; wn[1] = w4[1]; wn[2] = w4[2]; wn[3] = w4[3];
    } else {
      const bf16x4 w4 = *(const bf16x4*)((const bf16_t*)nm.emit_w + n);
      wn[0] = (float)w4[0]; wn[1] = (float)w4[1]; wn[2] = (float)w4[2]; wn[3] = (float)w4[3];
    }
  };
  float emit_w[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (NEXT) {
    const int n = n0 + wn * S::TN + (lane % 16) * 4;
    if (residual && vec_ok) request_residual(0);
    if (nm.emit_operand && n < N) load_emit_w(emit_w, n);
  }
#pragma unroll
  for (int i = 0; i < MI32; ++i) {
    if constexpr (DIRECT) {
#pragma unroll
      for (int ii = 0; ii < 2; ++ii)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          *(f32x4*)(cstage + (ii * 16 + lane % 16) * E_LD + j * 16 + (lane / 16) * 4) = acc[i * 2 + ii][j];
    } else {
#pragma unroll
      for (int j = 0; j < NJ32; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16& c = acc32[i][j];
          *(f32x4*)(cstage + (lane % 32) * E_LD + j * 32 + q * 8 + (lane / 32) * 4) =
              f32x4{c[q * 4 + 0], c[q * 4 + 1], c[q * 4 + 2], c[q * 4 + 3]};
        }
    }
    wave_sync();
    auto leave = [&](auto form) {
      constexpr int FORM = decltype(form)::value;
      constexpr bool AHEAD = FORM != kNoResidual && sizeof(TO) == 4 && !NEXT;
      // whether this launch's are: see below
      const bool ahead = AHEAD && residual && vec_ok;
      f32x4 res[AHEAD ? 8 : 1];
      if (FORM == kResidual || ahead) {
        const int m = m0 + wm * S::TM + i * 32 + lane / 16, n = n0 + wn * S::TN + (lane % 16) * 4;
        const float* from = residual + (int64_t)m * ldo + n;
#pragma unroll
        for (int c8 = 0; c8 < 8; ++c8)
          if (m + c8 * 4 < M && n < N) res[c8] = *(const f32x4*)(from + c8 * 4 * ldo);      // others are not stored
      }
      f32x4 all[TOGETHER ? 8 : 1];
      float all_rs[TOGETHER ? 8 : 1];
      f32x4 res_now[NEXT ? 8 : 1];
      if constexpr (TOGETHER) {
        const int r0 = wm * S::TM + i * 32 + lane / 16;
#pragma unroll
        for (int c8 = 0; c8 < 8; ++c8) all[c8] = *(const f32x4*)(cstage + (c8 * 4 + lane / 16) * E_LD + (lane % 16) * 4);
        if (nm.in_sumsq) {
#pragma unroll
          for (int c8 = 0; c8 < 8; ++c8) all_rs[c8] = row_factor[r0 + c8 * 4];
        } else if (nm.row_scale) {
#pragma unroll
          for (int c8 = 0; c8 < 8; ++c8) all_rs[c8] = nm.row_scale[min(m0 + r0 + c8 * 4, M - 1)];
        } else {
#pragma unroll
          for (int c8 = 0; c8 < 8; ++c8) all_rs[c8] = 1.f;
        }
        // used here, so that no read is put off into the branch of its row
        asm volatile("" : "+v"(all[0]), "+v"(all[1]), "+v"(all[2]), "+v"(all[3]), "+v"(all[4]), "+v"(all[5]), "+v"(all[6]), "+v"(all[7]));
        asm volatile("" : "+v"(all_rs[0]), "+v"(all_rs[1]), "+v"(all_rs[2]), "+v"(all_rs[3]), "+v"(all_rs[4]), "+v"(all_rs[5]), "+v"(all_rs[6]), "+v"(all_rs[7]));
        if constexpr (NEXT) {
#pragma unroll
          for (int c8 = 0; c8 < 8; ++c8) res_now[c8] = res_next[c8];
          if (i + 1 < MI32 && residual && vec_ok) request_residual(i + 1);
        }
      }
#pragma unroll
      for (int c8 = 0; c8 < 8; ++c8) {
        const int c = c8 * TL_WAVE + lane;
        const int r = c / 16, col = (c % 16) * 4;
        const int m = m0 + wm * S::TM + i * 32 + r, n = n0 + wn * S::TN + col;
        if (m >= M || n >= N) continue;
        // the row's factor (1 / rms of a norm left out of the operand): given, or that of a norm handed over
        float rs = 1.f;
        f32x4 s4;
        if constexpr (TOGETHER) {
          rs = all_rs[c8];
          s4 = all[c8];
        } else {
          if (nm.in_sumsq) rs = row_factor[m - m0];
          else if (nm.row_scale) rs = nm.row_scale[m];
          s4 = *(const f32x4*)(cstage + r * E_LD + col);
        }
        float v[4] = {s4[0] * rs, s4[1] * rs, s4[2] * rs, s4[3] * rs};
        if constexpr (SWIGLU != 0) {   // (gate, up, gate, up) -> two outputs; N is even and n a multiple of 4
          const int64_t oz = (int64_t)m * ldo + n / 2;
          if (n + 2 < N) {
            typedef TO to2 __attribute__((ext_vector_type(2)));
            to2 sv = {from_f32<TO>(gated_pair<SWIGLU>(v[0], v[1], nm.gate)), from_f32<TO>(gated_pair<SWIGLU>(v[2], v[3], nm.gate))};
            if (ldo % 2 == 0) {
              *(to2*)(out + oz) = sv;
            } else {
              out[oz] = sv[0];
              out[oz + 1] = sv[1];
            }
          } else {
            out[oz] = from_f32<TO>(gated_pair<SWIGLU>(v[0], v[1], nm.gate));
          }
          continue;
        }
        const int64_t o = (int64_t)m * ldo + n;
        if (vec_ok) {  // n + 3 < N because n and N are both multiples of 4
          if (FORM == kResidual || (FORM == kAnyForm && residual)) {
            f32x4 rv;
            if constexpr (NEXT) rv = res_now[c8];
            else if (FORM == kResidual || ahead) rv = res[AHEAD ? c8 : 0];
            else rv = *(const f32x4*)(residual + o);
            v[0] += rv[0]; v[1] += rv[1]; v[2] += rv[2]; v[3] += rv[3];
          }
          if constexpr (sizeof(TO) == 4) {
            f32x4 sv = {v[0], v[1], v[2], v[3]};
            *(f32x4*)((float*)out + o) = sv;
            if constexpr (SWIGLU == 0) {
              if (nm.emit_operand) {      // uniform; N is a multiple of 64: the 16 lanes of a row are all here or none is
                float wn[4];
                if constexpr (TOGETHER) {
#pragma unroll
                  for (int e = 0; e < 4; ++e) wn[e] = emit_w[e];
                } else {
                  load_emit_w(wn, n);
                }
                bf16x4 ev = {(bf16_t)(wn[0] * v[0]), (bf16_t)(wn[1] * v[1]), (bf16_t)(wn[2] * v[2]), (bf16_t)(wn[3] * v[3])};
                *(bf16x4*)(nm.emit_operand + (int64_t)m * nm.emit_ld + n) = ev;
                const float sq = group_sum<16>((v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]));
                if (lane % 16 == 0) nm.emit_sumsq[(int64_t)m * nm.emit_parts + n / 64] = sq;
              }
            }
          } else {
            if (nm.act != kActNone) {     // uniform
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] = act_value(v[e], nm.act);
            }
            bf16x4 sv = {(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
            *(bf16x4*)((bf16_t*)out + o) = sv;
          }
        } else {
          for (int e = 0; e < 4 && n + e < N; ++e) {
            float x = v[e];
            if (residual) x += residual[o + e];
            if constexpr (sizeof(TO) == 2) x = act_value(x, nm.act);
            out[o + e] = from_f32<TO>(x);
          }
        }
      }
    };
    // A float32 result's residual is requested for all 32 rows together: out may be the residual, so the compiler asks for
    // a piece only when the one before is stored (4,096 rows, 640 x 512: 13.6 -> 12.0 us; 3,000 rows, 1,280 x 256: 12.2 ->
    // 10.6).  What follows concerns the tiles of up to 128 x 128 through registers; the others asked for it 32 rows ago
    // (NEXT).  The smallest tile, whose products are mostly launch, has the two forms apart: 65 to 4,096 rows, 520 x 264, take
    // 2 % more without a residual where one piece of code serves both, bfloat16 results 3 % (they come without one, and load it
    // piece by piece).  The 128 x 128 tile would lose waves by it: 108 registers where 84 let four a SIMD run.
    if constexpr (BM > 64 || sizeof(TO) != 4) leave(std::integral_constant<int, SWIGLU ? kNoResidual : kAnyForm>{});
    else if (!SWIGLU && residual && vec_ok) leave(std::integral_constant<int, kResidual>{});
    else leave(std::integral_constant<int, kNoResidual>{});
    // the area is written again for the next 32 rows
    wave_sync();
  }
}

template <int BM, int BN, int WM, int WN, typename TO, int SWIGLU, int MODE>
static int launch_gemm_bf16_mode(const bf16_t* a, const bf16_t* w, TO* out, const float* residual,
                                 const TileNorm& row_scale, int M, int N, int K, int64_t lda, int64_t ldo,
                                 int k_per_split, hipStream_t stream) {
  using S = GemmShape<BM, BN, WM, WN>;
  static bool configured = false;
  if (!configured) {
    if (hipFuncSetAttribute((const void*)gemm_bf16_kernel<BM, BN, WM, WN, TO, SWIGLU, MODE>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::smem_all(MODE >= kDirect)) != hipSuccess)
      return TL_ERR_LAUNCH;
    configured = true;
  }
  // a tile's rows are addressed with 32-bit byte offsets from its first row
  if ((int64_t)BM * lda * 2 >= 0x7fffffff || (int64_t)BN * K * 2 >= 0x7fffffff) return TL_ERR_ARG;
  if (row_scale.emit_operand && (SWIGLU != 0 || sizeof(TO) != 4 || N % 64 || ldo % 4 || k_per_split > 0)) return TL_ERR_ARG;
  if (row_scale.in_sumsq && k_per_split > 0) return TL_ERR_ARG;      // a split product has no epilogue of its own
  const int64_t splits = k_per_split > 0 ? (K + k_per_split - 1) / k_per_split : 1;
  const int64_t total = (int64_t)((N + BN - 1) / BN) * ((M + BM - 1) / BM) * splits;
  const int64_t grid = (total + kXcds - 1) / kXcds * kXcds;
  if (grid > 0x7fffffff) return TL_ERR_ARG;
  hipLaunchKernelGGL((gemm_bf16_kernel<BM, BN, WM, WN, TO, SWIGLU, MODE>), dim3((unsigned)grid), dim3(S::THREADS),
                     S::smem_all(MODE >= kDirect), stream, a, w, out, residual, row_scale, M, N, K, lda, ldo, k_per_split);
  static_assert(sizeof(TileNorm) <= 120, "passed by value");
  return TL_OK;
}

// How the operands of a tile reach LDS.  Straight from memory where the inner size is whole steps: always in the 256 x 256
// tile; in the 256 x 128 tile from four steps on (with fewer its buffers are not even filled; 2,047 rows, 4,096 x 4,096, weights
// from memory: 68.1 us through registers, 61.8 so; 4,096 x 256 11.3 and 10.5); in the 128 x 128 tile likewise, if each
// workgroup has a unit to itself, or each has 32 steps and more.  Its four buffers leave a unit room for one workgroup, where
// through registers two share it, cover for each other's first loads, and make a second round for a few more workgroups than
// units cheap (1,500 rows, 1,408 x 1,088 in two parts, 264 workgroups: 23.3 us through registers, 25.9 so; 300 rows, 2,048 x
// 2,048 in six 20.0 and 22.8).  532 products of up to 256 workgroups: 1.0 to 1.26x as fast so, median 1.09; 340 of more and 4
// to 16 steps: 0.74 to 1.16x, median 0.91; where the choice below takes this tile for more and the inner size is whole, 4 to 11
// steps 0.76 to 1.05x, 16 0.97 to 1.08, 32 and 64 1.03 to 1.13 (2,102 rows, 3,712 x 4,096 76.3 and 72.4 us).  Four waves of twice the outputs, which read less from LDS,
// lose with float32 results (1,944 rows, 2,048 x 5,632: 59.0; 3,288 rows: 88.2 -> 100.6).
static int tile_mode(int bm, int bn, int M, int N, int K, int k_per_split) {
  if (K % B_BK) return kTail;
  if (bm + bn == 512) return kPhased;
  const int64_t splits = k_per_split > 0 ? (K + k_per_split - 1) / k_per_split : 1;
  const int64_t wgs = (int64_t)((N + bn - 1) / bn) * ((M + bm - 1) / bm) * splits;
  const bool alone = wgs <= 256 || (splits == 1 && K >= 32 * B_BK);
  return K >= 4 * B_BK && (bm + bn == 384 || (bm + bn == 256 && alone)) ? kDirect : kWhole;
}

template <int BM, int BN, int WM, int WN, typename TO, int SWIGLU>
static int launch_gemm_bf16(const bf16_t* a, const bf16_t* w, TO* out, const float* residual, const TileNorm& row_scale,
                            int M, int N, int K, int64_t lda, int64_t ldo, int k_per_split, hipStream_t stream) {
#define TL_GEMM(MODE)                                                                                                  \
  launch_gemm_bf16_mode<BM, BN, WM, WN, TO, SWIGLU, MODE>(a, w, out, residual, row_scale, M, N, K, lda, ldo, k_per_split, \
                                                          stream)
  const int mode = tile_mode(BM, BN, M, N, K, k_per_split);
  if (mode == kTail) return TL_GEMM(kTail);
  if constexpr (BM + BN == 512) {
    return TL_GEMM(kPhased);
  } else {
    if constexpr (BM + BN >= 256)
      if (mode == kDirect) return TL_GEMM(kDirect);
    return TL_GEMM(kWhole);
  }
#undef TL_GEMM
}

// Which tile: the one with the smallest estimated time.  A compute unit works through
// ceil(workgroups / 256) tiles one after the other, each at the rate that its tile shape reaches
// on a full chip (measured, TFLOP/s: the larger the tile, the fewer operand bytes per flop).  With fewer than eight steps first
// loads and the epilogue (10 us a 256 x 256 tile, whose step takes 1) count for more than the loop, and large tiles are worth
// less: `few` (2,200 rows, 3,712 x 64: 9.8 us with the 64 x 128 tiles that `few` chooses, 12.5 with the 256 x 256 that `rate`
// would; 700 rows, 11,264 x 192 13.4 and 15.3; x 512 20.8 and 19.1; x 2,048 53.1 and 43.6).  40 products for which the two
// choose another tile, in three forms, time of `few`'s choice over that of `rate`'s: inner size 64 to 200 0.96 to 1.0, 256 to
// 456 1.0 to 1.03, 512 and 520 1.04 and 1.02, 1,000 to 1,096 1.06 to 1.08, 2,048 to 4,104 1.09 to 1.12; sizes that end within a
// step, whose tiles all go through registers, as the others.
struct TileChoice {
  int bm, bn;
  double few, rate;
};
static const TileChoice kTiles[4] = {{256, 256, 1060., 1400.}, {256, 128, 900., 1130.}, {128, 128, 760., 980.}, {64, 128, 640., 650.}};

static double tile_cost(int c, int M, int N, int K) {
  const int64_t wgs = (int64_t)((M + kTiles[c].bm - 1) / kTiles[c].bm) * ((N + kTiles[c].bn - 1) / kTiles[c].bn);
  const double rate = K >= 8 * B_BK ? kTiles[c].rate : kTiles[c].few;
  return (double)((wgs + 255) / 256) * kTiles[c].bm * kTiles[c].bn / rate;
}

static int best_tile(int M, int N, int K, double* cost) {
  int best = 0;
  double best_cost = 0.;
  for (int c = 0; c < 4; ++c) {
    const double t = tile_cost(c, M, N, K);
    if (c == 0 || t < best_cost) {
      best = c;
      best_cost = t;
    }
  }
  if (cost) *cost = best_cost;
  return best;
}

template <typename TO, int SWIGLU>
static int launch_gemm_bf16_tile(int c, const bf16_t* a, const bf16_t* w, TO* out, const float* residual,
                                 const TileNorm& row_scale, int M, int N, int K, int64_t lda, int64_t ldo,
                                 int k_per_split, hipStream_t stream) {
  switch (c) {
    case 0:
      return launch_gemm_bf16<256, 256, 2, 4, TO, SWIGLU>(a, w, out, residual, row_scale, M, N, K, lda, ldo, k_per_split,
                                                          stream);
    case 1:
      return launch_gemm_bf16<256, 128, 4, 2, TO, SWIGLU>(a, w, out, residual, row_scale, M, N, K, lda, ldo, k_per_split,
                                                          stream);
    case 2:
      return launch_gemm_bf16<128, 128, 4, 2, TO, SWIGLU>(a, w, out, residual, row_scale, M, N, K, lda, ldo, k_per_split,
                                                          stream);
    default:
      return launch_gemm_bf16<64, 128, 2, 2, TO, SWIGLU>(a, w, out, residual, row_scale, M, N, K, lda, ldo, k_per_split,
                                                         stream);
  }
}

// tile: 1..4 force a tile shape, 0 lets the sizes decide.  Then a wide product may be launched in
// two parts: as many columns as fill the chip in whole rounds of the largest tile, and the rest
// with whatever tile suits the rest; a single tile shape would leave the last round of
// workgroups mostly empty (2048 x 11264: 352 tiles of 256 x 256 on 256 compute units).
template <typename TO, int SWIGLU>
static int launch_gemm_bf16_any(const bf16_t* a, const bf16_t* w, TO* out, const float* residual,
                                const TileNorm& row_scale, int M, int N, int K, int64_t lda, int64_t ldo,
                                int tile, int k_per_split, hipStream_t stream) {
  if (tile >= 1 && tile <= 4)
    return launch_gemm_bf16_tile<TO, SWIGLU>(tile - 1, a, w, out, residual, row_scale, M, N, K, lda, ldo, k_per_split,
                                             stream);
  double whole_cost;
  const int whole = best_tile(M, N, K, &whole_cost);
  if (k_per_split == 0) {
    const int tiles_m = (M + 255) / 256;
    const int cols_per_round = 256 / tiles_m * 256;          // columns that one round of 256 x 256 tiles covers
    const int n_first = cols_per_round > 0 ? N / cols_per_round * cols_per_round : 0;
    if (n_first > 0 && n_first < N) {
      double rest_cost;
      const int rest = best_tile(M, N - n_first, K, &rest_cost);
      if (tile_cost(0, M, n_first, K) + rest_cost < whole_cost) {
        int rc = launch_gemm_bf16_tile<TO, SWIGLU>(0, a, w, out, residual, row_scale, M, n_first, K, lda, ldo, 0, stream);
        if (rc != TL_OK) return rc;
        const int64_t o_off = SWIGLU ? n_first / 2 : n_first;
        TileNorm rest_norm = row_scale;      // what it emits belongs to columns n_first on (a multiple of 256)
        if (rest_norm.emit_operand) {
          rest_norm.emit_w = rest_norm.emit_w_is_f32 ? (const void*)((const float*)rest_norm.emit_w + n_first)
                                                     : (const void*)((const bf16_t*)rest_norm.emit_w + n_first);
          rest_norm.emit_operand += n_first;
          rest_norm.emit_sumsq += n_first / 64;
        }
        return launch_gemm_bf16_tile<TO, SWIGLU>(rest, a, w + (int64_t)n_first * K, out + o_off,
                                                 residual ? residual + o_off : nullptr, rest_norm, M, N - n_first, K,
                                                 lda, ldo, 0, stream);
      }
    }
  }
  return launch_gemm_bf16_tile<TO, SWIGLU>(whole, a, w, out, residual, row_scale, M, N, K, lda, ldo, k_per_split, stream);
}

// ------------------------------------------- split k for few rows: everything in flight
// At most 64 rows, the inner size split over workgroups.  A workgroup's share of both operands (64
// rows of activations and 128 weight rows per 64 k) goes straight into LDS
// (global_load_lds_dwordx4: no registers in between), as a ring of six slabs of 64 k, so that five
// slabs (120 KB) are on their way while one is multiplied; a share of up to six slabs is requested
// at once and the kernel is one round trip to memory long.  The tiled kernel above keeps one k
// step of 64 in flight through registers, two or three straight into LDS, and pays a round trip for each so many.
// A slab in LDS: [A: 8 groups of 8 rows | W: 16 groups of 8 rows][8 rows x 128 bytes]; one load
// instruction of a wave fills one group (1 KB, lane i -> bytes 16 i); the 16-byte chunk c of row r
// stands at position c ^ (r % 8), so that the fragment reads of 32 rows do not collide.
// Result: float32 partial products [split, M, N] for splitk_reduce_kernel.  K must be a multiple of 64.
constexpr int O_BM = 64, O_BN = 128, O_WAVES = 8, O_THREADS = O_WAVES * TL_WAVE, O_SLAB_K = 64, O_RING = 6;
constexpr int O_GROUPS = (O_BM + O_BN) / 8, O_GROUP_BYTES = 8 * O_SLAB_K * 2, O_SLAB_BYTES = O_GROUPS * O_GROUP_BYTES;
typedef __attribute__((address_space(3))) void* tl_lds_ptr;
typedef const __attribute__((address_space(1))) void* tl_global_ptr;

// waits until at most 3 * later of this wave's loads are outstanding (three loads a slab)
__device__ __forceinline__ void oneshot_wait(int later) {
  switch (later) {
    case 0: __builtin_amdgcn_s_waitcnt(0x0F70); break;
    case 1: __builtin_amdgcn_s_waitcnt(0x0F73); break;
    case 2: __builtin_amdgcn_s_waitcnt(0x0F76); break;
    case 3: __builtin_amdgcn_s_waitcnt(0x0F79); break;
    default: __builtin_amdgcn_s_waitcnt(0x0F7C); break;       // 12
  }
}

__global__ __launch_bounds__(O_THREADS) void gemm_oneshot_bf16_kernel(const bf16_t* __restrict__ a,
                                                                      const bf16_t* __restrict__ w,
                                                                      float* __restrict__ partial, int M, int N, int K,
                                                                      int64_t lda, int slabs_per_split) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char oneshot_smem[];
  const int tid = threadIdx.x, lane = tid % TL_WAVE, wave = tid / TL_WAVE;
  const int n0 = blockIdx.x * O_BN, split = blockIdx.y, m0 = blockIdx.z * O_BM;
  const int nslabs = K / O_SLAB_K, s0 = split * slabs_per_split, s1 = min(nslabs, s0 + slabs_per_split);
  const int mine = s1 - s0;                       // at least one: the grid has no empty split
  // requests: of every slab wave v fills group v (8 activation rows) and groups 8 + v and 16 + v
  // (16 weight rows); a lane's three addresses move on by 64 k from slab to slab
  static_assert(O_BM / 8 == O_WAVES && O_BN / 8 == 2 * O_WAVES, "one activation group and two weight groups a wave");
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const int lrow = lane / 8, lchunk = (lane % 8) ^ lrow;
  const int64_t k_first = (int64_t)s0 * O_SLAB_K + lchunk * 8;
  const bf16_t* src[3] = {a + (int64_t)min(m0 + wv * 8 + lrow, M - 1) * lda + k_first,
                          w + (int64_t)min(n0 + wv * 8 + lrow, N - 1) * K + k_first,
                          w + (int64_t)min(n0 + (O_WAVES + wv) * 8 + lrow, N - 1) * K + k_first};
  auto request = [&](int sl) {                    // slab sl of this workgroup, into buffer sl % O_RING
    unsigned char* sb = oneshot_smem + (sl % O_RING) * O_SLAB_BYTES + wv * O_GROUP_BYTES;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      __builtin_amdgcn_global_load_lds((tl_global_ptr)src[j], (tl_lds_ptr)(sb + j * O_WAVES * O_GROUP_BYTES), 16, 0, 0);
      src[j] += O_SLAB_K;
    }
  };
  for (int sl = 0; sl < min(mine, O_RING - 1); ++sl) request(sl);
  // wave (wm, wn) owns rows wm*32.., columns wn*32..; result transposed (rows of the instruction are
  // output columns), so a lane ends up with four consecutive columns of one row
  const int wm = wave / 4, wn = wave % 4;
  const int r8 = lane % 8;
  const int lane_off = ((lane % 32) / 8) * O_GROUP_BYTES + r8 * 128;
  const int a_off = (wm * 32 / 8) * O_GROUP_BYTES + lane_off;
  const int w_off = (O_BM / 8 + wn * 32 / 8) * O_GROUP_BYTES + lane_off;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  for (int sl = 0; sl < mine; ++sl) {
    // slab sl has landed for this wave once only the slabs requested after it are outstanding;
    // after the barrier it has landed for everybody, and nobody reads slab sl - 1 any more, whose
    // buffer the next request takes
    // (a bare barrier: __syncthreads() would also wait for every outstanding load, the slabs still on
    // their way included; the counter above is the wait that is needed, and the fragment reads of
    // the previous slab were consumed by its matrix instructions before any wave gets here)
    oneshot_wait(min(mine - 1, sl + O_RING - 2) - sl);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (sl + O_RING - 1 < mine) request(sl + O_RING - 1);
    const unsigned char* sb = oneshot_smem + (sl % O_RING) * O_SLAB_BYTES;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int pos = ((2 * ks + lane / 32) ^ r8) * 16;
      const bf16x8 fa = *(const bf16x8*)(sb + a_off + pos);
      const bf16x8 fw = *(const bf16x8*)(sb + w_off + pos);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw, fa, acc, 0, 0, 0);
    }
  }
  float* out = partial + (int64_t)split * M * N;
  const int m = m0 + wm * 32 + lane % 32;
  if (m < M) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = n0 + wn * 32 + q * 8 + (lane / 32) * 4;
      if ((N % 4 == 0) && n + 3 < N) {
        *(f32x4*)(out + (int64_t)m * N + n) = f32x4{acc[q * 4 + 0], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) out[(int64_t)m * N + n + e] = acc[q * 4 + e];
      }
    }
  }
}

// Whether and how this kernel takes a product of 17 to 64 rows that is split at all (stripe_plan, which compares its time
// with this estimate, keeps most of them whole): slabs of 64 k per split (0: not this
// kernel).  The number of splits with the smallest estimated time: rounds of workgroups over the 256
// compute units, each as long as a workgroup takes to fetch its share (about 35 GB/s), and the second
// kernel's reading of the partial sums.
static double oneshot_us(int M, int N, int K, int per) {
  const int tiles = ((M + O_BM - 1) / O_BM) * ((N + O_BN - 1) / O_BN), splits = (K / O_SLAB_K + per - 1) / per;
  return (tiles * splits + 255) / 256 * (2.0 + per * (O_SLAB_BYTES / 35e3)) + 1.5 + splits * (double)M * N * 4 / 3e6;
}
static int oneshot_plan(int M, int N, int K, int* slabs_per_split) {
  *slabs_per_split = 0;
  if (M <= 16 || K % O_SLAB_K || K < 4 * O_SLAB_K) return 1;
  // measured on whole decode steps: small weight matrices with few rows are faster in the few-row
  // kernel (one launch); up to 32 rows for matrices of 6 M weights (3 % of a step at 32 rows; from
  // 36 rows on this kernel is 2 to 7 % of a step faster), up to 18 rows for 17 M weights (4096 x 4096:
  // from 22 rows on this kernel is 1 to 2 % of a step faster)
  const int64_t weights = (int64_t)N * K;
  const int tiles = ((M + O_BM - 1) / O_BM) * ((N + O_BN - 1) / O_BN), nslabs = K / O_SLAB_K;
  if (M <= O_BM && ((weights <= ((int64_t)6 << 20) && M <= 32) || (weights <= ((int64_t)17 << 20) && K <= 4096 && M <= 18) ||
                    (tiles > 128 && M <= 32)))
    return 1;
  int best = 1, best_per = 0;
  double best_t = 0.;
  for (int want = 2; want <= 16; ++want) {
    const int per = (nslabs + want - 1) / want;
    // measured on whole steps: shares of fewer than four slabs lose to fewer, longer ones
    if (per < (nslabs >= 8 ? 4 : 2)) break;
    const int splits = (nslabs + per - 1) / per;
    if (splits < 2) continue;
    const double t = oneshot_us(M, N, K, per);
    if (best == 1 || t < best_t) {
      best = splits;
      best_per = per;
      best_t = t;
    }
  }
  *slabs_per_split = best_per;
  return best;
}

// ------------------------------------------------------------ split k: the second kernel
// Adds up the partial products [splits, M, N] of a product whose inner size was split over
// workgroups and applies what the product's own epilogue would have: row factor (given, or from
// sums of squares handed over by the producer of the input), residual, SiLU-gate, output type; it
// can also prepare the next norm (operand and sums of squares per chunk of 1024 columns).  One
// workgroup per (row, chunk of 1024 columns), four consecutive columns per thread.
constexpr int R_THREADS = 256, R_CHUNK = R_THREADS * 4;

struct ReduceArgs {
  const float* partial;
  int splits, M, N;
  void* out;
  int64_t ldo;
  const float* residual;
  const float* row_scale;
  const float* in_sumsq;
  int in_parts, in_width;
  float in_eps;
  const void* emit_w;
  int emit_w_is_f32;
  bf16_t* emit_operand;
  float* emit_sumsq;
  int act = kActNone;       // bfloat16 output: applied before rounding
  Gate gate;                // a gated product's unit
};

template <typename TO, int SWIGLU>
__global__ __launch_bounds__(R_THREADS) void splitk_reduce_kernel(const ReduceArgs p) {
  __shared__ float red[R_THREADS / TL_WAVE];
  const int m = blockIdx.x, tid = threadIdx.x;
  const int n = blockIdx.y * R_CHUNK + tid * 4;
  const int N = p.N;
  // Everything that has to come from memory is requested before anything is used: the kernel is
  // a few dependent round trips long, and every one it saves counts.
  float t = 0.f;
  if (p.in_sumsq)
    for (int q = tid; q < p.in_parts; q += R_THREADS) t += p.in_sumsq[(int64_t)m * p.in_parts + q];
  float scale = p.row_scale ? p.row_scale[m] : 1.f;
  float res[4] = {0.f, 0.f, 0.f, 0.f}, wn[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (SWIGLU == 0) {
    for (int e = 0; e < 4 && n + e < N; ++e) {
      if (p.residual) res[e] = p.residual[(int64_t)m * p.ldo + n + e];
      if (p.emit_operand)
        wn[e] = p.emit_w_is_f32 ? ((const float*)p.emit_w)[n + e] : (float)((const bf16_t*)p.emit_w)[n + e];
    }
  }
  const bool vec = (N % 4 == 0);
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (n < N) {
    if (vec) {
      // eight splits at a time, their loads in flight together; added in the order of the splits
      for (int sp0 = 0; sp0 < p.splits; sp0 += 8) {
        f32x4 x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          x[u] = *(const f32x4*)(p.partial + ((int64_t)min(sp0 + u, p.splits - 1) * p.M + m) * N + n);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (sp0 + u < p.splits) {
            v[0] += x[u][0]; v[1] += x[u][1]; v[2] += x[u][2]; v[3] += x[u][3];
          }
        }
      }
    } else {
      for (int sp = 0; sp < p.splits; ++sp) {
        const float* src = p.partial + ((int64_t)sp * p.M + m) * N + n;
        for (int e = 0; e < 4 && n + e < N; ++e) v[e] += src[e];
      }
    }
  }
  if (p.in_sumsq) {      // uniform
    t = block_sum<R_THREADS / TL_WAVE>(t, red);
    scale = 1.f / sqrtf(t / (float)p.in_width + p.in_eps);
  }
  TO* out = (TO*)p.out;
  float sq = 0.f;
  if (n < N) {
    if constexpr (SWIGLU != 0) {   // (gate, up, gate, up) -> two outputs; N is even and n a multiple of 4
      out[(int64_t)m * p.ldo + n / 2] = from_f32<TO>(gated_pair<SWIGLU>(v[0] * scale, v[1] * scale, p.gate));
      if (n + 2 < N)
        out[(int64_t)m * p.ldo + n / 2 + 1] = from_f32<TO>(gated_pair<SWIGLU>(v[2] * scale, v[3] * scale, p.gate));
    } else {
      for (int e = 0; e < 4 && n + e < N; ++e) {
        float x = v[e] * scale + res[e];
        if constexpr (sizeof(TO) == 2) x = act_value(x, p.act);
        out[(int64_t)m * p.ldo + n + e] = from_f32<TO>(x);
        if (p.emit_operand) {
          p.emit_operand[(int64_t)m * N + n + e] = (bf16_t)(wn[e] * x);
          sq += x * x;
        }
      }
    }
  }
  if (p.emit_operand) {       // uniform
    sq = block_sum<R_THREADS / TL_WAVE>(sq, red);
    if (tid == 0) p.emit_sumsq[(int64_t)m * gridDim.y + blockIdx.y] = sq;
  }
}

// How a bfloat16 product of these sizes is best split: returns the number of splits (1: not at
// all) and sets the tile (as tl_linear_tile's) and the inner size per split.  Splitting pays when
// the output has too few tiles to fill 256 compute units and the rows are too many for the
// few-row kernel to stream the weights at full rate.  The number of parts is the order in which a result's float32 sums are
// added, and the sizes here are those of a step's rows: another number moves the logits of a batch (by 0.2 to 1 % of their norm
// where an estimate of the time chose fewer).
static int splitk_plan(int M, int N, int K, int* tile, int* k_per_split) {
  *tile = 0;
  *k_per_split = 0;
  // The ring kernel's sizes.  Up to 64 rows: it or the few-row kernel.  Beyond (tiles of 64 rows side by
  // side), measured: it beats the k-step loop up to 128 rows on matrices up to 4096 x 6144 and up to 256
  // rows on small ones; its one accumulator tile a wave is no match for the tiled kernel beyond that.
  const int64_t weights = (int64_t)N * K;
  const bool ring_rows = M <= O_BM || (M <= 128 && N <= 6144 && weights <= ((int64_t)26 << 20)) ||
                         (M <= 256 && weights <= ((int64_t)6 << 20));
  if (M > 16 && ring_rows && K % O_SLAB_K == 0 && K >= 4 * O_SLAB_K) {
    int slabs;
    const int one = oneshot_plan(M, N, K, &slabs);
    *tile = -1;
    *k_per_split = slabs * O_SLAB_K;
    return one;
  }
  if (M <= 16 || K < 8 * B_BK) return 1;
  const int bm = M <= 64 ? 64 : 128, bn = 128;
  const int64_t wgs = (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  if (wgs >= 160) return 1;
  if (M <= 64 && (int64_t)N * K < (int64_t)8 << 20) return 1;      // small weights: the few-row kernel is faster
  const int nk = (K + B_BK - 1) / B_BK;
  const int want = (int)((256 + wgs - 1) / wgs);
  int per = (nk + want - 1) / want;
  if (per < 4) per = 4;
  const int splits = (nk + per - 1) / per;
  if (splits < 2) return 1;
  *tile = M <= 64 ? 4 : 3;
  *k_per_split = per * B_BK;
  return splits;
}

// ============================================================ bfloat16, few rows
// Decode-shaped products (M <= 64): the weight matrix is streamed once and is the
// whole cost, and a step is a chain of such kernels, so the kernel is built around
// (a) many 16-byte loads in flight and (b) as few dependent memory round trips and
// as few launches as possible.  A workgroup of eight wave64 owns 16 output columns
// (16 weight rows; 32 or 64 when there are more than 16 activation rows); the waves split K in
// blocks of 128 and each accumulates a
// 16 x 16 tile per group of 16 activation rows and 16 columns with v_mfma_f32_16x16x32_bf16
// (weight rows as the A operand read straight from global memory, activations as
// the B operand).  Partial tiles meet in LDS and are added in a fixed order, so
// results are deterministic.
//
// Fused into it, to save launches: a prologue on the activations, either RMSNorm of
// the float32 residual stream (statistics recomputed by every workgroup: a few KB
// from L2) or SiLU-gate of a [M, 2K] gate|up matrix; an optional gather of input
// rows; and the residual add in the epilogue, whose operand is fetched before the
// main loop starts.
constexpr int S_WAVES = 8, S_THREADS = S_WAVES * TL_WAVE, S_COLS = 16, S_KBLK = 128;
enum { PRO_NONE = 0, PRO_NORM = 1 };

struct SkinnyArgs {
  const void* a;            // PRO_NONE: bf16 [M, K]; PRO_NORM: float [rows, K]
  const bf16_t* w;          // [N, K]
  void* out;                // [M, N]
  const float* residual;    // [M, N] or null
  const void* norm_w;       // PRO_NORM: [K], float or bf16
  const int32_t* rows;      // optional gather of input rows
  const float* row_scale;   // optional factor of each output row (a norm applied by an earlier kernel)
  float eps;
  int norm_w_is_f32;
  int M, N, K;
  int64_t lda, ldo;
  // A norm handed from producer to consumer.  The producer (float32 output, no SiLU-gate) also
  // writes emit_operand[m, n] = bf16(emit_w[n] * out[m, n]) and, per group of columns (one group
  // a workgroup: 16 columns, or 8), the sum of out^2 into emit_sumsq[m, group].  The consumer takes
  // such an operand as `a` and turns in_sumsq [rows, in_parts] into its row factor
  // 1 / sqrt(sum / in_width + in_eps).
  const void* emit_w = nullptr;
  int emit_w_is_f32 = 0;
  bf16_t* emit_operand = nullptr;
  float* emit_sumsq = nullptr;
  const float* in_sumsq = nullptr;
  int in_parts = 0, in_width = 0;
  float in_eps = 0.f;
  // The columns a workgroup owns, even, at most 16 a column tile (0: all of them).  Fewer make one
  // balanced round of workgroups out of a product whose column tiles do not divide by 256.
  int cols_wg = 0;
  int act = kActNone;       // bfloat16 output: applied before rounding
  Gate gate;                // a gated product's unit
};

// One 8-wide k chunk of an activation row, as loaded (Raw) and as an MFMA operand.  With the norm
// prologue the operand is w * x of the float32 residual stream (rounded to bfloat16) and `ss`
// collects x^2: the row's 1 / rms is a common factor of the whole dot product and is applied to
// the result instead, so nothing has to wait for the row statistics.  Loading and converting are
// separate steps so that the loads of the next k block can be in flight while this one is used.
template <int PRO>
struct SkinnyChunk;
template <>
struct SkinnyChunk<PRO_NONE> {
  bf16x8 v;
  __device__ __forceinline__ void load(const SkinnyArgs& p, int64_t off) { v = *(const bf16x8*)((const bf16_t*)p.a + off); }
};
template <>
struct SkinnyChunk<PRO_NORM> {
  f32x4 x0, x1;
  __device__ __forceinline__ void load(const SkinnyArgs& p, int64_t off) {
    const float* x = (const float*)p.a + off;
    x0 = *(const f32x4*)x;
    x1 = *(const f32x4*)(x + 4);
  }
};
// the norm weights of one k chunk, as floats
struct NormChunk {
  f32x4 w0, w1;
  __device__ __forceinline__ void load(const SkinnyArgs& p, int k) {
    if (p.norm_w_is_f32) {
      w0 = *(const f32x4*)((const float*)p.norm_w + k);
      w1 = *(const f32x4*)((const float*)p.norm_w + k + 4);
    } else {
      const bf16x8 w8 = *(const bf16x8*)((const bf16_t*)p.norm_w + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        w0[e] = (float)w8[e];
        w1[e] = (float)w8[4 + e];
      }
    }
  }
};
// `k_ok`: the chunk lies inside the row (it counts towards the sum of squares); the product itself
// is protected by zeroing the weight chunk instead.
__device__ __forceinline__ bf16x8 skinny_operand(const SkinnyChunk<PRO_NONE>& c, const NormChunk&, bool, float&) {
  return c.v;
}
__device__ __forceinline__ bf16x8 skinny_operand(const SkinnyChunk<PRO_NORM>& c, const NormChunk& nw, bool k_ok,
                                                 float& ss) {
  bf16x8 r;
  float q = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    r[e] = (bf16_t)(nw.w0[e] * c.x0[e]);
    r[4 + e] = (bf16_t)(nw.w1[e] * c.x1[e]);
    q += c.x0[e] * c.x0[e] + c.x1[e] * c.x1[e];
  }
  ss += k_ok ? q : 0.f;
  return r;
}

// DEEP: two register stages also with one tile, for long inner sizes, where a wave works through
// several stages and the chain of their memory round trips sets the kernel's duration.
//
// HALF (at most 8 activation rows, one tile, no prologue, no SiLU-gate): a workgroup owns 8 columns only, so that
// a matrix with few rows still gives every compute unit a workgroup; what a workgroup can have in
// flight, not the memory system, bounds these kernels.  The 16 x 16 MFMA tile is then used as two
// 8 x 8 tiles that split k: weight row i of the operand is column i % 8 at k offset (i / 8) * 32,
// activation column j is row j % 8 at k offset (j / 8) * 32, and the wanted products are the two
// diagonal blocks of the result, added in the epilogue.  One MFMA so covers 64 k, and a load
// instruction reads whole 128-byte lines of 8 weight rows.
template <int MT, int CT, bool DEEP, typename TO, int PRO, int SWIGLU, bool HALF>
__device__ __forceinline__ void skinny_product(const SkinnyArgs& p) {
  static_assert(!HALF || (MT == 1 && CT == 1 && PRO == PRO_NONE && SWIGLU != 1), "HALF: one plain tile");
  constexpr int COLS = HALF ? 8 : S_COLS;          // columns of a tile that are outputs
  constexpr int KW = HALF ? 64 : 32;               // k covered by one MFMA
  constexpr int KBLK = 4 * KW;                     // k covered by a block of four MFMAs
  extern __shared__ __attribute__((aligned(16))) unsigned char skinny_smem[];
  typedef float Tile[16][17];
  Tile* part = (Tile*)skinny_smem;                                  // [S_WAVES][MT * CT]
  float* ss_part = (float*)(part + S_WAVES * MT * CT);              // [S_WAVES][MT * 16]
  const int tid = threadIdx.x, lane = tid % TL_WAVE, wave = tid / TL_WAVE;
  const int M = p.M, N = p.N, K = p.K;
  const int cw = (!HALF && p.cols_wg > 0) ? p.cols_wg : COLS * CT;      // columns of this workgroup
  const int n0 = blockIdx.x * cw;
  const int r16 = lane % 16, g = lane / 16;
  const int rr = HALF ? r16 % 8 : r16;             // the weight row / activation row this lane feeds
  const int kh = HALF ? (r16 / 8) * 32 : 0;        // and its k offset inside an MFMA's range
  const bf16_t* wrow[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) wrow[ct] = p.w + (int64_t)min(n0 + min(ct * 16 + rr, cw - 1), N - 1) * K;

  // epilogue operands first: their latency hides behind the main loop
  constexpr int TILES = MT * CT;
  constexpr int EPT = (TILES * 256 + S_THREADS - 1) / S_THREADS;
  float res_v[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = tid + j * S_THREADS;
    const int tile = e / 256;
    const int m = HALF ? e / 8 : (tile / CT) * 16 + (e % 256) / 16;
    const int n = HALF ? n0 + e % 8 : n0 + (tile % CT) * 16 + e % 16;
    res_v[j] = (p.residual && e < (HALF ? 64 : TILES * 256) && m < M && n < N && n - n0 < cw) ? p.residual[(int64_t)m * p.ldo + n] : 0.f;
  }

  // input row of each activation row this lane feeds
  int64_t row_off[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 16 + rr;
    const int src = p.rows ? p.rows[min(m, M - 1)] : min(m, M - 1);
    row_off[mt] = (int64_t)src * p.lda;
  }

  // Row factors of a norm whose sums of squares arrive in parts: one wave per row, fixed order.
  // The first 256 parts of a row are requested here, ahead of everything else, and added up once
  // the first weights have been requested (see the main loop).
  float* scale_s = ss_part + S_WAVES * MT * 16;                      // [MT * 16]
  constexpr int RPW = MT * 16 / S_WAVES;                             // rows per wave
  constexpr int PRE = 4;                                             // parts requested ahead, in wavefuls
  float pre[RPW][PRE];
  if (p.in_sumsq) {
#pragma unroll
    for (int ri = 0; ri < RPW; ++ri) {
      const int m = min(wave + ri * S_WAVES, M - 1);
      const int64_t src = p.rows ? p.rows[m] : m;
      const bool row_there = wave + ri * S_WAVES < M;        // the same for the whole wave
#pragma unroll
      for (int h = 0; h < PRE; ++h) {
        const int q = lane + h * TL_WAVE;
        pre[ri][h] = 0.f;
        if (!row_there || h * TL_WAVE >= p.in_parts) continue;      // the same for the whole wave: nothing to ask for
        if (q < p.in_parts) pre[ri][h] = p.in_sumsq[src * p.in_parts + q];
      }
    }
  }
  auto row_factors = [&]() {
    if (!p.in_sumsq) return;
#pragma unroll
    for (int ri = 0; ri < RPW; ++ri) {
      const int r = wave + ri * S_WAVES;
      float t = (pre[ri][0] + pre[ri][1]) + (pre[ri][2] + pre[ri][3]);
      if (p.in_parts > PRE * TL_WAVE) {
        const int m = min(r, M - 1);
        const int64_t src = p.rows ? p.rows[m] : m;
        for (int q = lane + PRE * TL_WAVE; q < p.in_parts; q += TL_WAVE) t += p.in_sumsq[src * p.in_parts + q];
      }
      t = wave_sum(t);
      if (lane == 0) scale_s[r] = 1.f / sqrtf(t / (float)p.in_width + p.in_eps);
    }
  };

  // A stage is UN k blocks of 128 (all loads of a stage are issued together).  Where the
  // registers allow, two stages take turns, so the loads of the next stage are in flight while
  // this one is multiplied; with one tile the registers are better spent on a second resident
  // workgroup.  Loads are unconditional with the address clamped into the matrix: a predicated
  // load would become a branch and the stages could not overlap.  Rows beyond M or N only feed
  // outputs that are never written; a chunk beyond K is zeroed on the weight side when it is used.
  constexpr int UN = TILES == 1 ? 2 : 1;
  constexpr bool TWO_STAGES = DEEP || (TILES > 1 && MT + CT <= 5);
  struct Stage {
    bf16x8 fw[UN][CT][4];
    SkinnyChunk<PRO> fa[UN][MT][4];
    NormChunk nw[PRO == PRO_NORM ? UN : 1][PRO == PRO_NORM ? 4 : 1];
  };
  const int nblk = (K + KBLK - 1) / KBLK;
  auto load = [&](Stage& st, int blk) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      // MFMA i of the block covers k = i*32 .. i*32+31, lane group g its 8 k from g*8: one load
      // instruction then reads 64 contiguous bytes of each of the 16 weight rows
      if (u > 0 && blk + u * S_WAVES >= nblk) continue;      // the same for the whole wave: no such block
      const int kb = (blk + u * S_WAVES) * KBLK + kh + g * 8;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) st.fw[u][ct][i] = *(const bf16x8*)(wrow[ct] + min(kb + i * KW, K - 8));
    }
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      if (u > 0 && blk + u * S_WAVES >= nblk) continue;
      const int kb = (blk + u * S_WAVES) * KBLK + kh + g * 8;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = min(kb + i * KW, K - 8);
        if constexpr (PRO == PRO_NORM) st.nw[u][i].load(p, k);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) st.fa[u][mt][i].load(p, row_off[mt] + k);
      }
    }
  };
  f32x4 acc[MT][CT];
  float ss[MT];                            // this lane's share of sum x^2 of its rows (norm prologue)
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    ss[mt] = 0.f;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[mt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto multiply = [&](const Stage& st, int blk) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      if (u > 0 && blk + u * S_WAVES >= nblk) continue;      // nothing was loaded for it
      const int kb = (blk + u * S_WAVES) * KBLK + kh + g * 8;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool k_ok = kb + i * KW < K;
        bf16x8 z = {};
        bf16x8 fa[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          fa[mt] = skinny_operand(st.fa[u][mt][i], st.nw[PRO == PRO_NORM ? u : 0][PRO == PRO_NORM ? i : 0], k_ok,
                                  ss[mt]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const bf16x8 fw = k_ok ? st.fw[u][ct][i] : z;
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[mt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw, fa[mt], acc[mt][ct], 0, 0, 0);
        }
      }
    }
  };
  constexpr int STEP = S_WAVES * UN;
  // The row factors are worked out while the first weights are on their way: their operands were
  // requested before and arrive first, and the wave has nothing else to do until the weights come.
  if constexpr (TWO_STAGES) {
    Stage s0, s1;
    int blk = wave;
    if (blk < nblk) load(s0, blk);
    if (blk + STEP < nblk) load(s1, blk + STEP);
    row_factors();
    if (blk < nblk) {
      while (true) {
        const int b1 = blk + STEP;
        multiply(s0, blk);
        if (b1 >= nblk) break;
        const int b2 = b1 + STEP;
        if (b2 < nblk) load(s0, b2);
        multiply(s1, b1);
        if (b2 >= nblk) break;
        blk = b2;
        if (blk + STEP < nblk) load(s1, blk + STEP);
      }
    }
  } else {
    Stage s0;
    int blk = wave;
    if (blk < nblk) load(s0, blk);
    row_factors();
    while (blk < nblk) {
      multiply(s0, blk);
      blk += STEP;
      if (blk < nblk) load(s0, blk);
    }
  }
  // tile layout: lane holds rows (weight rows) g*4 + r, column (activation row) r16
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave * TILES + mt * CT + ct][g * 4 + r][r16] = acc[mt][ct][r];
  if constexpr (PRO == PRO_NORM) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float t = ss[mt];
      t = sum_over_rows(t);
      if (g == 0) ss_part[wave * (MT * 16) + mt * 16 + r16] = t;
    }
  }
  __syncthreads();
  TO* out = (TO*)p.out;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = tid + j * S_THREADS;
    if (e >= (HALF ? 64 : TILES * 256)) continue;       // whole waves: 256 elements are four waves
    const int tile = e / 256, m_local = HALF ? e / 8 : (e % 256) / 16, nn = HALF ? e % 8 : e % 16;
    const int m = (tile / CT) * 16 + m_local, n = n0 + (tile % CT) * 16 + nn;
    const bool valid = m < M && n < N && n - n0 < cw;
    float scale = 1.f;                    // the row factor left out of the operands
    if (p.row_scale) scale = p.row_scale[min(m, M - 1)];
    if (p.in_sumsq) scale = scale_s[(tile / CT) * 16 + m_local];
    if constexpr (PRO == PRO_NORM) {
      float t = 0.f;
#pragma unroll
      for (int wv = 0; wv < S_WAVES; ++wv) t += ss_part[wv * (MT * 16) + (tile / CT) * 16 + m_local];
      scale = 1.f / sqrtf(t / (float)K + p.eps);
    }
    if constexpr (SWIGLU != 0) {   // columns (2j, 2j+1) = (gate_j, up_j): even threads make one output of a pair
      if ((nn & 1) || !valid) continue;
      float gv = 0.f, uv = 0.f;
#pragma unroll
      for (int wv = 0; wv < S_WAVES; ++wv) {
        gv += part[wv * TILES + tile][nn][m_local];
        uv += part[wv * TILES + tile][nn + 1][m_local];
        if constexpr (HALF) {
          gv += part[wv * TILES + tile][nn + 8][m_local + 8];
          uv += part[wv * TILES + tile][nn + 9][m_local + 8];
        }
      }
      out[(int64_t)m * p.ldo + n / 2] = from_f32<TO>(gated_pair<SWIGLU>(gv * scale, uv * scale, p.gate));
    } else {
      float v = 0.f;
#pragma unroll
      for (int wv = 0; wv < S_WAVES; ++wv) {
        v += part[wv * TILES + tile][nn][m_local];
        if constexpr (HALF) v += part[wv * TILES + tile][nn + 8][m_local + 8];
      }
      v = v * scale + res_v[j];
      if constexpr (sizeof(TO) == 2) v = act_value(v, p.act);
      if (valid) out[(int64_t)m * p.ldo + n] = from_f32<TO>(v);
      if constexpr (sizeof(TO) == 4) {
        if (p.emit_operand) {             // uniform: the lanes of a row group stay together
          if (valid) {
            const float wn = p.emit_w_is_f32 ? ((const float*)p.emit_w)[n] : (float)((const bf16_t*)p.emit_w)[n];
            p.emit_operand[(int64_t)m * N + n] = (bf16_t)(wn * v);
          }
          float sq = valid ? v * v : 0.f;
          sq = group_sum<COLS>(sq);
          if (nn == 0 && m < M) {
            if (CT > 1 && cw != COLS * CT) {
              // a part per workgroup and column tile, empty ones (beyond N) included
              p.emit_sumsq[(int64_t)m * ((N + cw - 1) / cw * CT) + blockIdx.x * CT + tile % CT] = sq;
            } else if (n < N) {     // a column group that begins beyond N has no part of its own
              if (cw == COLS * CT) p.emit_sumsq[(int64_t)m * ((N + COLS - 1) / COLS) + (n0 / COLS + tile % CT)] = sq;
              else p.emit_sumsq[(int64_t)m * ((N + cw - 1) / cw) + blockIdx.x] = sq;
            }
          }
        }
      }
    }
  }
}

template <int MT, int CT, bool DEEP, typename TO, int PRO, int SWIGLU, bool HALF>
__global__ __launch_bounds__(S_THREADS) void gemm_skinny_bf16_kernel(const SkinnyArgs p) {
  skinny_product<MT, CT, DEEP, TO, PRO, SWIGLU, HALF>(p);
}

// Several products of few rows that do not wait for each other, each with operands of its own, as ONE launch:
// blockIdx.y names the product, a workgroup owns 16 of its columns.
constexpr int S_SET = 6;
struct SkinnySet {
  SkinnyArgs p[S_SET];
  int vec;                  // every result's rows and address take groups of four columns
};
__global__ __launch_bounds__(S_THREADS) void gemm_skinny_set_kernel(const SkinnySet set) {
  const SkinnyArgs& p = set.p[blockIdx.y];
  if ((int)blockIdx.x * S_COLS >= p.N) return;
  skinny_product<1, 1, false, float, PRO_NONE, 0, false>(p);
}

// Column tiles per workgroup: every workgroup reads all M activation rows, so with more rows it
// should own more columns, or the activations are read more often than the weights.
template <int MT, int CT, bool DEEP, typename TO, int PRO, int SWIGLU, bool HALF = false>
static int launch_skinny_deep(const SkinnyArgs& p, hipStream_t stream) {
  constexpr size_t smem = (size_t)S_WAVES * MT * CT * 16 * 17 * sizeof(float) + (size_t)(S_WAVES + 1) * MT * 16 * sizeof(float);
  static bool configured = false;
  if (!configured) {
    if (hipFuncSetAttribute((const void*)gemm_skinny_bf16_kernel<MT, CT, DEEP, TO, PRO, SWIGLU, HALF>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      return TL_ERR_LAUNCH;
    configured = true;
  }
  constexpr int cols = HALF ? 8 : S_COLS * CT;
  const int cw = (!HALF && p.cols_wg > 0) ? p.cols_wg : cols;
  dim3 g((p.N + cw - 1) / cw), b(S_THREADS);
  hipLaunchKernelGGL((gemm_skinny_bf16_kernel<MT, CT, DEEP, TO, PRO, SWIGLU, HALF>), g, b, smem, stream, p);
  return TL_OK;
}

// Columns a workgroup owns in the plain one-tile kernel: 16, or fewer (even) where that turns 129
// to 255 workgroups, which leave compute units idle, into one round of at most 256; 8 where 16
// would leave half of the compute units without a workgroup (whole decode steps of 9 to 16 rows
// with products of 2,048 columns: 3 % faster).
static int skinny_cols_wg(int N) {
  const int tiles = (N + S_COLS - 1) / S_COLS;
  if (tiles > 64 && tiles <= 128) return 8;
  if (tiles <= 128 || tiles >= 256) return S_COLS;
  const int cw = (N + 255) / 256;
  return cw + (cw & 1);
}

// Columns a workgroup owns with `ct` (2 to 4) column tiles: what makes exactly 256 workgroups, where
// that needs all `ct` tiles (0: all columns of the tiles).
static int skinny_cols_wg_tiles(int N, int ct) {
  const int cw = (N + 255) / 256 + ((N + 255) / 256 & 1);
  return cw > S_COLS * (ct - 1) && cw < S_COLS * ct ? cw : 0;
}

// 8 columns a workgroup: for at most 8 rows and an inner size that gives every wave at least
// one block of four MFMAs, where that still gives no more workgroups than there are compute
// units (measured: otherwise it is slower).  With the clamped and the gelu unit too, whose stored products took it: their bits, and
// 6 rows by 512 pairs of inner size 4,096 8.6 us in 16 columns, 6.3 so (stored, with the unit's own kernel, 7.8); 1,024 pairs 7.5 and
// 7.6 (9.3).  SiLU products keep the order of sums that they have always had.
static bool skinny_half(int M, int N, int K) { return M <= 8 && K >= 2048 && (N + 7) / 8 <= 256; }

template <int MT, int CT, typename TO, int PRO, int SWIGLU>
static int launch_skinny_tile(const SkinnyArgs& p, hipStream_t stream) {
  if constexpr (MT * CT == 1 && PRO == PRO_NONE && SWIGLU != 1) {
    if (skinny_half(p.M, p.N, p.K)) {
      if (p.K > 4096) return launch_skinny_deep<MT, CT, true, TO, PRO, SWIGLU, true>(p, stream);
      return launch_skinny_deep<MT, CT, false, TO, PRO, SWIGLU, true>(p, stream);
    }
  }
  if constexpr (CT == 1) {
    SkinnyArgs q = p;
    q.cols_wg = skinny_cols_wg(p.N);
    if constexpr (MT == 1 && PRO == PRO_NONE) {
      if (p.K > 4096) return launch_skinny_deep<MT, CT, true, TO, PRO, SWIGLU>(q, stream);
    }
    return launch_skinny_deep<MT, CT, false, TO, PRO, SWIGLU>(q, stream);
  }
  return launch_skinny_deep<MT, CT, false, TO, PRO, SWIGLU>(p, stream);
}

// More column tiles only while at least 256 workgroups remain: fewer cannot pull the weights
// through fast enough.
template <int MT, typename TO, int SWIGLU>
static int launch_skinny_rows(const SkinnyArgs& p, hipStream_t stream) {
  if (p.N >= 256 * 64) return launch_skinny_tile<MT, 4, TO, PRO_NONE, SWIGLU>(p, stream);
  if (p.N >= 256 * 32) return launch_skinny_tile<MT, 2, TO, PRO_NONE, SWIGLU>(p, stream);
  return launch_skinny_tile<MT, 1, TO, PRO_NONE, SWIGLU>(p, stream);
}

template <typename TO, int PRO, int SWIGLU>
static int launch_skinny(const SkinnyArgs& p, hipStream_t stream) {
  const int mt = (p.M + 15) / 16;
  if (mt == 1) {
    if constexpr (PRO == PRO_NONE) {
      // A workgroup fetches at a rate of its own, and every workgroup fetches all activation rows:
      // the product is fastest with ONE round of workgroups over the 256 compute units, each owning
      // as many column tiles as that takes (up to four).  (Also with few rows: timed alone, more
      // workgroups looked faster below 8 rows; whole decode steps are 1 % faster at 4 rows with
      // one round and equal at 1 and 2.)  Wider products run several rounds: one column tile below
      // 8 rows, two from 8 rows on, where the activation rows a workgroup fetches weigh as much as
      // its weights (whole decode steps at hidden 4096, intermediate 14336, vocabulary 128256:
      // 3 % faster at 8 rows and 9 % at 16 with two tiles, 2 to 6 % slower at 1 to 6; four tiles
      // are slower than two at 16 rows).
      const int ct = (p.N + 256 * S_COLS - 1) / (256 * S_COLS);
      if (ct >= 2 && ct <= 4) {
        // exactly 256 workgroups where the columns allow it: the last column tile of each is partly used
        // (whole decode steps: 0.3 % faster at hidden 2048, 0.7 to 1.4 % at hidden 4096, where q/k/v went
        // from 192 workgroups to 256)
        SkinnyArgs q = p;
        q.cols_wg = skinny_cols_wg_tiles(p.N, ct);
        if (ct == 2) return launch_skinny_tile<1, 2, TO, PRO, SWIGLU>(q, stream);
        if (ct == 3) return launch_skinny_tile<1, 3, TO, PRO, SWIGLU>(q, stream);
        return launch_skinny_tile<1, 4, TO, PRO, SWIGLU>(q, stream);
      }
      // (below 8 rows too where one tile would leave the last of the kernel's stages, 16 k blocks of 128
      // over the eight waves, half empty or emptier at a long inner size: inner size 5120 x 27,648
      // columns at 1 row, 52 us against 61)
      const int tail_blocks = ((p.K + S_KBLK - 1) / S_KBLK) % (2 * S_WAVES);
      const bool half_empty_stage = p.K > 4096 && tail_blocks >= 1 && tail_blocks <= S_WAVES;
      if (ct > 4 && (p.M >= 8 || half_empty_stage)) {
        // several rounds of two column tiles: as many columns a workgroup (17 to 32, even) as make whole
        // rounds of 256 workgroups (28,672 columns: 1,024 workgroups of 28 instead of 896 of 32, which
        // are four rounds as well)
        SkinnyArgs q = p;
        const int rounds = (p.N + 256 * 2 * S_COLS - 1) / (256 * 2 * S_COLS);
        const int cw = (p.N + rounds * 256 - 1) / (rounds * 256);
        q.cols_wg = cw + (cw & 1);
        // (a product that prepares a norm keeps whole tiles: its parts are counted per 16 columns)
        if (q.cols_wg <= S_COLS || q.cols_wg >= 2 * S_COLS || p.emit_operand) q.cols_wg = 0;
        return launch_skinny_tile<1, 2, TO, PRO, SWIGLU>(q, stream);
      }
    }
    return launch_skinny_tile<1, 1, TO, PRO, SWIGLU>(p, stream);
  }
  if constexpr (PRO == PRO_NONE) {       // the norm prologue exists for one row tile only
    if (mt == 2) return launch_skinny_rows<2, TO, SWIGLU>(p, stream);
    if (mt == 3) return launch_skinny_rows<3, TO, SWIGLU>(p, stream);
    return launch_skinny_rows<4, TO, SWIGLU>(p, stream);
  }
  return TL_ERR_ARG;
}

// ============================================================ bfloat16, 6 to 64 rows
// Bound by what a unit fetches: every workgroup needs its activation rows (64 of them are 256 KB at an inner size of 2,048, beside
// 180 KB of weights), and a unit gets about 105 GB/s from its L2 in loads that take whole lines of 128 bytes (138 alone), but 37
// in the matrix instructions' own order, 64 bytes of each of sixteen rows, in which gemm_skinny_bf16_kernel loads.  So a wave fetches
// whole lines, turns them into operands through an area of LDS of its own (no barrier in the loop), and owns every eighth block of the
// inner size, so that each row is fetched once by a workgroup; the waves' sums meet in LDS, in a fixed order.  The inner size stays whole: no second
// kernel and no partial sums through memory, as splitting it over workgroups takes.  Blocks of 128 k where their LDS allows (64 otherwise),
// one on its way: 64 rows of 2,048 by 11,264 pairs took 15.1 us so, 15.8 with two and 17.8 with three.  (Every workgroup beginning
// with another block, so that they do not all ask for the same lines at once, took 14.7, but then a sum's order goes by its column.)
// 64 rows, weights from memory, against the split product's two kernels: 2,560 x 2,048 10.9 -> 6.4 us, 2,048 x 2,048 10.0 ->
// 5.5, 11,264 x 2,048 gated 18.1 -> 15.1, 2,048 x 5,632 14.4 -> 11.9.
constexpr int T_MAX_INNER = 1 << 20;      // offsets within a workgroup's rows fit 31 bits

template <int MT, int CT, int TK>
struct Stripe {
  static constexpr int kRows = MT * 16, kLd = CT * 16 + 4;                     // kLd: floats between rows of partial sums
  static constexpr int kChunks = TK / 8, kRowsPerLoad = 64 / kChunks;          // 16-byte chunks of a row's share of a block
  static constexpr int kA = kRows / kRowsPerLoad, kW = CT * 16 / kRowsPerLoad; // load instructions of a block
  static constexpr int kWaveBytes = (kA + kW) * 1024;
  static constexpr int kGroups = kRows * CT * 4;                               // groups of four columns of a row
  static constexpr size_t kBody = (size_t)S_WAVES * (kWaveBytes > kRows * kLd * 4 ? kWaveBytes : kRows * kLd * 4);
  static constexpr size_t kSmem = kBody + (size_t)(kRows + kGroups) * sizeof(float);
};

// p.cols_wg: a multiple of 4, at most 16 CT.  vec: the results' rows and addresses take groups of four columns.  GATHER: the input's
// rows are p.rows' (through addresses of their own, as the input may be longer than a buffer's 31 bits).
// SET: one of several products in a launch, whose results may leave as the tanh of the sums.
template <int MT, int CT, int TK, int SUMS, typename TO, int SWIGLU, bool GATHER, bool SET>
__device__ __forceinline__ void stripe_product(const SkinnyArgs& p, int groups_n, int vec, int block_n, int block_m) {
  using S = Stripe<MT, CT, TK>;
  extern __shared__ __attribute__((aligned(16))) unsigned char stripe_smem[];
  float* part = (float*)stripe_smem;                      // [S_WAVES][kRows][kLd], once the blocks are done with
  float* scale_s = (float*)(stripe_smem + S::kBody);      // [kRows]
  float* sq_s = scale_s + S::kRows;                       // [kRows][CT * 4]
  const int tid = threadIdx.x, lane = tid % TL_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / TL_WAVE);
  const int M = p.M, N = p.N, K = p.K, cw = p.cols_wg;
  const int n0 = block_n * cw, m0 = block_m * S::kRows;
  if (n0 >= N) return;

  // A lane fetches chunk lc of row lr + kRowsPerLoad j.  Rows beyond the matrices and blocks beyond the inner size lie beyond the
  // buffers: they read as zero and fetch nothing.  All of an offset is a lane's own (scalar offset 0): that is what the check of a
  // buffer's end is documented for.
  const int lr = lane / S::kChunks, lc = lane % S::kChunks, lda = (int)p.lda;
  const auto buf_w = __builtin_amdgcn_make_buffer_rsrc((void*)(p.w + (int64_t)n0 * K), 0, min(cw, N - n0) * K * 2, 0x00020000);
  const auto buf_a = __builtin_amdgcn_make_buffer_rsrc((void*)((const bf16_t*)p.a + (int64_t)m0 * lda), 0,
                                                       ((min(S::kRows, M - m0) - 1) * lda + K) * 2, 0x00020000);
  const int at_a = lr * lda * 2 + lc * 16, at_w = lr * K * 2 + lc * 16;
  const int step_a = S::kRowsPerLoad * lda * 2, step_w = S::kRowsPerLoad * K * 2;
  const int nblk = K / TK, mine = (nblk - wave + S_WAVES - 1) / S_WAVES;
  const bf16_t* row_a[GATHER ? S::kA : 1];
  if constexpr (GATHER)
#pragma unroll
    for (int j = 0; j < S::kA; ++j)
      row_a[j] = (const bf16_t*)p.a + (int64_t)p.rows[min(m0 + j * S::kRowsPerLoad + lr, M - 1)] * p.lda + lc * 8;
  struct Block {
    bf16x8 a[S::kA], w[S::kW];
  };
  auto load = [&](Block& st, int i) {       // this wave's i-th block
    const int k = i < mine ? (wave + i * S_WAVES) * TK * 2 : 0x70000000;
#pragma unroll
    for (int j = 0; j < S::kW; ++j)
      st.w[j] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(buf_w, at_w + k + j * step_w, 0, 0));
#pragma unroll
    for (int j = 0; j < S::kA; ++j) {
      if constexpr (GATHER) st.a[j] = i < mine ? *(const bf16x8*)(row_a[j] + k / 2) : bf16x8{};
      else st.a[j] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(buf_a, at_a + k + j * step_a, 0, 0));
    }
  };
  // chunk c of row r stands at place c ^ (r % kSwizzle) of its row, so that the operands of eight rows do not collide
  constexpr int kSwizzle = S::kChunks < 16 ? S::kChunks : 16;
  const int r16 = lane % 16, g = lane / 16;
  unsigned char* own = stripe_smem + wave * S::kWaveBytes;
  auto place = [&](int j) { return own + j * 1024 + lr * TK * 2 + (lc ^ ((j * S::kRowsPerLoad + lr) % kSwizzle)) * 16; };
  // SUMS 2: sums of their own for every other step of 32 k, added at the end, half the roundings in a row (2,048 x 5,632 against
  // 64 bits: 1.61e-7 of the result with one, 1.20e-7 with two; split over workgroups, as such products were, 1.30e-7).
  f32x4 acc[SUMS][MT][CT];
#pragma unroll
  for (int h = 0; h < SUMS; ++h)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[h][mt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](Block& st, int next) {      // and requests the next block as soon as this one has left its registers
#pragma unroll
    for (int j = 0; j < S::kW; ++j) *(bf16x8*)place(S::kA + j) = st.w[j];
#pragma unroll
    for (int j = 0; j < S::kA; ++j) *(bf16x8*)place(j) = st.a[j];
    load(st, next);
    wave_sync();      // other lanes read them
#pragma unroll
    for (int i = 0; i < TK / 32; ++i) {
      const unsigned char* from = own + r16 * TK * 2 + ((i * 4 + g) ^ (r16 % kSwizzle)) * 16;
      bf16x8 fa[MT], fw[CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) fw[ct] = *(const bf16x8*)(from + S::kA * 1024 + ct * 32 * TK);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) fa[mt] = *(const bf16x8*)(from + mt * 32 * TK);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[i % SUMS][mt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[ct], fa[mt], acc[i % SUMS][mt][ct], 0, 0, 0);
    }
    wave_sync();      // the area is written again for the next block
  };
  // The parts of the rows' sums of squares are requested ahead of everything else, up to 256 of a row together, and added up once the
  // first block has been requested (behind it, and one request after the other: a decode step of 8 rows 3.4 % slower).
  constexpr int RPW = S::kRows / S_WAVES, PRE = 4;      // rows a wave, requests a row
  float pre[RPW][PRE];
  const float* row_sq[RPW];
  if (p.in_sumsq) {
#pragma unroll
    for (int ri = 0; ri < RPW; ++ri) {
      const int m = min(m0 + wave * RPW + ri, M - 1);
      row_sq[ri] = p.in_sumsq + (int64_t)(GATHER ? p.rows[m] : m) * p.in_parts;
#pragma unroll
      for (int h = 0; h < PRE; ++h) {
        pre[ri][h] = 0.f;
        if (h * TL_WAVE >= p.in_parts) continue;      // uniform
        if (lane + h * TL_WAVE < p.in_parts) pre[ri][h] = row_sq[ri][lane + h * TL_WAVE];
      }
    }
  }
  Block st;
  load(st, 0);

  // what the epilogue needs is requested behind the first block
  constexpr int EPT = (S::kGroups + S_THREADS - 1) / S_THREADS;
  f32x4 res_v[EPT], next_w[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    res_v[j] = next_w[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (SWIGLU == 0) {      // the residual is float32 whatever the results are
      const int e = tid + j * S_THREADS, c = e % (CT * 4) * 4, n = n0 + c;
      const int m = min(m0 + e / (CT * 4), M - 1);
      if (p.residual) {
        const float* r = p.residual + (int64_t)m * p.ldo;
        if (vec && n + 3 < N) res_v[j] = *(const f32x4*)(r + n);
        else
#pragma unroll
          for (int q = 0; q < 4; ++q) res_v[j][q] = r[min(n + q, N - 1)];
      }
      if constexpr (sizeof(TO) == 4)
        if (p.emit_operand)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            next_w[j][q] = p.emit_w_is_f32 ? ((const float*)p.emit_w)[min(n + q, N - 1)] : (float)((const bf16_t*)p.emit_w)[min(n + q, N - 1)];
    }
  }
  if (p.in_sumsq) {      // the rows' factors: one wave a row, in a fixed order
#pragma unroll
    for (int ri = 0; ri < RPW; ++ri) {
      float t = (pre[ri][0] + pre[ri][1]) + (pre[ri][2] + pre[ri][3]);
      for (int q = lane + PRE * TL_WAVE; q < p.in_parts; q += TL_WAVE) t += row_sq[ri][q];
      t = wave_sum(t);
      if (lane == 0) scale_s[wave * RPW + ri] = 1.f / sqrtf(t / (float)p.in_width + p.in_eps);
    }
  }

  for (int i = 0; i < mine; ++i) multiply(st, i + 1);

  // a lane holds columns 4 g .. 4 g + 3 of row r16 of every tile
  __syncthreads();
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      f32x4 v = acc[0][mt][ct];
      if constexpr (SUMS == 2) v += acc[1][mt][ct];
      *(f32x4*)(part + (wave * S::kRows + mt * 16 + r16) * S::kLd + ct * 16 + g * 4) = v;
    }
  __syncthreads();
  TO* out = (TO*)p.out;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = tid + j * S_THREADS;
    if (e >= S::kGroups) break;
    const int ml = e / (CT * 4), c = e % (CT * 4) * 4, m = m0 + ml, n = n0 + c;
    const int left = m < M ? min(4, min(cw - c, N - n)) : 0;      // columns of this group that are results
    f32x4 sum[S_WAVES];
#pragma unroll
    for (int wv = 0; wv < S_WAVES; ++wv) sum[wv] = *(const f32x4*)(part + (wv * S::kRows + ml) * S::kLd + c);
    // Blocks of 64 k that do not share out evenly leave more sums, and shorter ones, than blocks of 128: added one after the other they
    // were 3 to 7 % further from 64 bits at inner sizes of 704 to 832 (1,024 x 704 at 9 rows 7.65e-8 of the result in blocks of 128,
    // 8.0e-8 so), in pairs they are closer (7.05e-8)
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
    if (TK == 64 && nblk % S_WAVES != 0) {      // uniform
      v = ((sum[0] + sum[1]) + (sum[2] + sum[3])) + ((sum[4] + sum[5]) + (sum[6] + sum[7]));
    } else {
#pragma unroll
      for (int wv = 0; wv < S_WAVES; ++wv) v += sum[wv];
    }
    float scale = 1.f;
    if (p.row_scale) scale = p.row_scale[min(m, M - 1)];
    if (p.in_sumsq) scale = scale_s[ml];
    if constexpr (SWIGLU != 0) {      // two pairs (gate, up)
      const TO y0 = from_f32<TO>(gated_pair<SWIGLU>(v[0] * scale, v[1] * scale, p.gate));
      const TO y1 = from_f32<TO>(gated_pair<SWIGLU>(v[2] * scale, v[3] * scale, p.gate));
      TO* to = out + (int64_t)m * p.ldo + n / 2;
      if (left > 1) to[0] = y0;
      if (left > 3) to[1] = y1;
    } else {
      float sq = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = v[q] * scale + res_v[j][q];
        if constexpr (sizeof(TO) == 2) v[q] = act_value(v[q], p.act);
        if (q < left) sq += v[q] * v[q];
      }
      if constexpr (SET) {
        if (p.act == kActTanh) {      // uniform
          bf16_t* low = (bf16_t*)p.out + (int64_t)m * p.ldo + n;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (q < left) low[q] = (bf16_t)tanhf(v[q]);
          continue;
        }
      }
      TO* to = out + (int64_t)m * p.ldo + n;
      if (vec && left == 4) {
        if constexpr (sizeof(TO) == 4) *(f32x4*)to = v;
        else *(bf16x4*)to = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q < left) to[q] = from_f32<TO>(v[q]);
      }
      if constexpr (sizeof(TO) == 4) {
        if (p.emit_operand) {
          bf16_t* op = p.emit_operand + (int64_t)m * N + n;
          const f32x4 x = next_w[j] * v;
          if (vec && left == 4) *(bf16x4*)op = bf16x4{(bf16_t)x[0], (bf16_t)x[1], (bf16_t)x[2], (bf16_t)x[3]};
          else
#pragma unroll
            for (int q = 0; q < 4; ++q)
              if (q < left) op[q] = (bf16_t)x[q];
          sq_s[e] = sq;
        }
      }
    }
  }
  if constexpr (SWIGLU == 0 && sizeof(TO) == 4) {
    if (!p.emit_operand) return;      // uniform
    __syncthreads();
    if (tid < S::kRows && m0 + tid < M) {      // a part of a row's sum of squares per workgroup
      float t = 0.f;
#pragma unroll
      for (int c = 0; c < CT * 4; ++c) t += sq_s[tid * CT * 4 + c];
      p.emit_sumsq[(int64_t)(m0 + tid) * groups_n + block_n] = t;
    }
  }
}

template <int MT, int CT, int TK, int SUMS, typename TO, int SWIGLU, bool GATHER>
__global__ __launch_bounds__(S_THREADS) void gemm_stripe_bf16_kernel(const SkinnyArgs p, int groups_n, int vec) {
  stripe_product<MT, CT, TK, SUMS, TO, SWIGLU, GATHER, false>(p, groups_n, vec, blockIdx.x, blockIdx.y);
}

// Several products of up to 16 rows that do not wait for each other as ONE launch (SkinnySet): blockIdx.y names the product, a
// workgroup owns up to 16 CT of its columns.  Five products of a decode step's six rows (four of 2,048 columns and one of 64, inner size 2,048)
// take 21.8 us as launches of their own, 11.9 in gemm_skinny_set_kernel (16 columns, two rounds of workgroups) and 9.6 so (36 columns, one round).
// Of 40 sets at 1 to 16 rows (inner sizes of 256 to 4,096) it takes 0.52 to 1.0 times as long for all but a few: inner size 256, 1.0 to 1.05
// times 2.7 us, up to 6 rows of 1,024 + 256 + 256 columns 1.04 to 1.08 times 4.3, of five times 4,096 by 2,048 1.05 to 1.09 times 20.
template <int CT, int TK>
__global__ __launch_bounds__(S_THREADS) void gemm_stripe_set_kernel(const SkinnySet set) {
  stripe_product<1, CT, TK, 1, float, 0, false, true>(set.p[blockIdx.y], 0, set.vec, blockIdx.x, 0);
}
template <int CT, int TK>
static int launch_stripe_set(SkinnySet& set, int count, int most, int cols, hipStream_t stream) {
  constexpr size_t smem = Stripe<1, CT, TK>::kSmem;
  static bool configured = false;
  if (!configured) {
    if (hipFuncSetAttribute((const void*)gemm_stripe_set_kernel<CT, TK>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
      return TL_ERR_LAUNCH;
    configured = true;
  }
  for (int i = 0; i < count; ++i) set.p[i].cols_wg = cols;
  hipLaunchKernelGGL((gemm_stripe_set_kernel<CT, TK>), dim3((most + cols - 1) / cols, count), dim3(S_THREADS), smem, stream, set);
  return TL_OK;
}
// As few columns a workgroup (8 to 48, a multiple of 4) as make one round of the 256 units, else 16.
static int stripe_set_cols(const SkinnySet& set, int count) {
  for (int cols = 8; cols <= 48; cols += 4) {
    int64_t groups = 0;
    for (int i = 0; i < count; ++i) groups += (set.p[i].N + cols - 1) / cols;
    if (groups <= 256) return cols;
  }
  return S_COLS;
}

// Several groups of rows: those of one group of columns fall on one die and find its weights in the L2 (48 rows of 5,120 x 5,120,
// three groups of 86 32.3 us where they fell on different dies, 19.3 so).
static int stripe_grid_n(int groups_n, int groups_m) { return groups_m > 1 ? (groups_n + kXcds - 1) / kXcds * kXcds : groups_n; }

template <int MT, int CT, int TK, int SUMS, typename TO, int SWIGLU, bool GATHER>
static int launch_stripe_sums(const SkinnyArgs& p, hipStream_t stream) {
  const auto kernel = gemm_stripe_bf16_kernel<MT, CT, TK, SUMS, TO, SWIGLU, GATHER>;
  constexpr size_t smem = Stripe<MT, CT, TK>::kSmem;
  static bool configured = false;
  if (!configured) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) return TL_ERR_LAUNCH;
    configured = true;
  }
  const int vec = p.ldo % 4 == 0 && p.N % 4 == 0 && (uintptr_t)p.out % 16 == 0 && (uintptr_t)p.residual % 16 == 0 && (uintptr_t)p.emit_operand % 8 == 0;
  const int groups_n = (p.N + p.cols_wg - 1) / p.cols_wg, groups_m = (p.M + MT * 16 - 1) / (MT * 16);
  dim3 g(stripe_grid_n(groups_n, groups_m), groups_m), b(S_THREADS);
  hipLaunchKernelGGL(kernel, g, b, smem, stream, p, groups_n, vec);
  return TL_OK;
}

// Two sums beyond 2,048 k (up to there one is as close to 64 bits as what took such products before), where the registers allow.
template <int MT, int CT, int TK, typename TO, int SWIGLU, bool GATHER>
static int launch_stripe_blocks(const SkinnyArgs& p, hipStream_t stream) {
  if constexpr (MT * CT <= 4)
    if (p.K > 2048) return launch_stripe_sums<MT, CT, TK, 2, TO, SWIGLU, GATHER>(p, stream);
  return launch_stripe_sums<MT, CT, TK, 1, TO, SWIGLU, GATHER>(p, stream);
}

template <int MT, int CT, typename TO, int SWIGLU>
static int launch_stripe_tile(const SkinnyArgs& p, hipStream_t stream) {
  // (four tiles of a short inner size go by shorter blocks: 64 rows of 2,560 x 2,048 in 2 x 2 tiles 7.8 us and 7.3, 16 of 11,264 x
  // 2,048 in 1 x 3 12.4 and 11.6, but 17 of 6,144 x 4,096 in 1 x 3 13.2 and 14.1)
  const bool long_blocks = p.K % 128 == 0 && (MT + CT <= 3 || p.K > 2048);
  if constexpr (sizeof(TO) == 4) {      // the output head's
    if (p.rows) {
      if constexpr (MT + CT <= 4)
        if (long_blocks) return launch_stripe_blocks<MT, CT, 128, TO, SWIGLU, true>(p, stream);
      return launch_stripe_blocks<MT, CT, 64, TO, SWIGLU, true>(p, stream);
    }
  }
  if constexpr (MT + CT <= 4)
    if (long_blocks) return launch_stripe_blocks<MT, CT, 128, TO, SWIGLU, false>(p, stream);
  return launch_stripe_blocks<MT, CT, 64, TO, SWIGLU, false>(p, stream);
}

// How this kernel takes a product of 6 to 64 rows, as tiles of sixteen rows and of sixteen columns a workgroup and the columns that
// it owns of them (false: not it).  A workgroup's time goes by the rows that it fetches, of both operands, so the cheapest cut of the product has
// the smallest sum of both, times the rounds of workgroups that it makes over the 256 units.  Timed for fifteen matrices of 1,024 x 704 to
// 27,648 x 5,120 at 17, 32, 48 and 64 rows, every cut of each (1,270 in all): the one this picks is within 3 % of the fastest, 0.05 % on average.
//  * Beyond 16 rows the estimate (us) is compared with the split product's own (oneshot_us; 4 us for its second launch), which is the
//    faster way for long inner sizes and few columns: 64 rows of 14,336 by 4,096 37.4 us here and 29.9 split; 5,120 x 5,120 20.4 and 19.9.
//  * 6 to 8 rows: in one round, where the few-row kernel has no form of eight columns and a workgroup's columns are not just one
//    tile of a short inner size (8 rows: 2,560 x 2,048 5.2 -> 4.7, 11,264 x 2,048 12.1 -> 11.6, 6,144 x 4,096 13.1 -> 11.7, 4,096 x
//    14,336 28.9 -> 25.2, but 4,096 x 4,096 9.7 and 10.0, 2,048 x 2,048 4.6 both).  At 1 row the few-row kernel is the faster one.
//  * Up to 32 rows and 2,048 k: not where the few-row kernel is the faster one, see below.
struct StripePlan {
  int mt, ct, cols;
};

// Whether the few-row kernel is the faster one for up to 32 rows of a short inner size.  Both timed at 3,700 products of 6 to 64 rows, 128 to
// 151,936 columns and 64 to 16,384 k, weights from memory (us, whole lines and few-row kernel):
//  * 6 to 8 rows: one column tile a workgroup below 1,536 k (8 rows of 2,560: 512 k 1.09 times as long, 1,024 k 1.01, 1,536 k 0.96),
//    two up to 2,048 (4,097 to 8,192 columns: 1.15 at 128 k, 8,192 x 2,048 10.2 and 9.3, 0.96 at 2,560 k).
//  * 9 to 16 rows in one round of up to 8,192 columns: 256 and 384 k 1.02 to 1.12 times, and beyond 1,024 columns up to 640 k 0.98 to 1.10;
//    at 9 and 10 rows up to 768 k (1.02 to 1.08), beyond 4,096 columns up to 2,048 k (9 rows of 8,192 x 2,048 10.3 and 9.4).
//  * 9 to 16 rows in several rounds: two or four column tiles a workgroup (9 rows of 32,000 x 2,048 31.8 and 27.1, 16 rows 31.7 and 29.4; 40,960
//    columns, two tiles, 1.1 to 1.34 times), three up to 12 rows beyond 1,024 k (18,432 x 2,048 1.08 to 1.15 times); from 11 rows on only
//    where its stages of 1,024 k are full (16 rows of 28,672 x 1,536 22.0 and 23.2).
//  * 17 to 32 rows of 2,049 to 4,096 columns: up to 512 k (17 rows 1.03 to 1.16 times), beyond 24 rows 256 k (1.0 to 1.07).
// An odd multiple of 64 stays: the few-row kernel pads it, and its sums of such inner sizes are further from 64 bits.  So do longer inner sizes, some
// of which cost up to a tenth more so (9 rows of 28,672 x 4,096 50.3 and 44.0; 48 rows of 5,120 x 5,120 20.0 and 18.2 split): their sums
// are closer to 64 bits by a quarter and more (1.15e-7 and 1.74e-7 of the result for the latter).
static bool stripe_few_rows_pay(int M, int N, int K, const StripePlan& plan, bool several_rounds) {
  if (K > 2048 || (K % 128 && K != 64)) return false;
  if (M <= 8) return plan.ct == 1 ? K < 1536 : plan.ct == 2;
  if (K < 256) return false;
  if (M <= 16) {
    if (several_rounds) return (M <= 10 ? K >= 512 : K == 512 || K % 1024 == 0) && (plan.ct != 3 || (M <= 12 && K > 1024));
    if (N > 8192) return false;
    return K < 512 || (N > 1024 && (K <= 640 || (M <= 10 && K <= (N <= 4096 ? 768 : 2048))));
  }
  return M <= 32 && N > 2048 && N <= 4096 && K <= (M <= 24 ? 512 : 256);
}
static bool stripe_plan(int M, int N, int K, StripePlan* plan) {
  if (M < 6 || M > 64 || K % 64 || K > T_MAX_INNER) return false;
  const int tiles = (M + 15) / 16;
  int64_t least = 0, fewest = 0;      // (of equal cuts the one with the fewest rows: 17 rows of 6,144 x 4,096 13.2 us in 1 x 3 tiles, 15.0 in 2 x 2)
  for (int mt = 1; mt <= tiles; ++mt)
    for (int ct = 1; ct <= 4; ++ct) {
      const int groups_m = (tiles + mt - 1) / mt, groups_n = (N + 16 * ct - 1) / (16 * ct);
      const int64_t groups = (int64_t)groups_m * stripe_grid_n(groups_n, groups_m), cost = (groups + 255) / 256 * (mt + ct);
      if (least && cost >= least) continue;
      least = cost;
      fewest = groups;
      // one round of three or four column tiles, or of up to 16 rows: as many columns as make 256 workgroups, at least 8 (64 rows of
      // 5,120 x 5,120 20.6 -> 19.0 us, 16 rows of 2,048 x 5,632 10.3 -> 9.0)
      int even = (int)((N * (int64_t)groups_m + 255) / 256 + 3) / 4 * 4;
      if (tiles == 1 && even < 8) even = 8;
      const bool one_round = (int64_t)groups_m * stripe_grid_n((N + even - 1) / even, groups_m) <= 256;      // also as the grid is filled up
      *plan = {mt, ct, one_round && (ct >= 3 || tiles == 1) && even > 16 * (ct - 1) && even < 16 * ct ? even : 16 * ct};
    }
  if (stripe_few_rows_pay(M, N, K, *plan, fewest > 256)) return false;
  if (M <= 8) return fewest <= 256 && N > 2048 && (plan->cols != 16 || K > 4096);
  if (M <= 16) return true;
  int slabs;
  if (oneshot_plan(M, N, K, &slabs) < 2) return true;
  return 2.4 + least * (K * 32 * 1.23e-5) + (double)N * K * 2 * 0.66 / 5.75e6 <= oneshot_us(M, N, K, slabs) + 4.0;
}

template <int MT, typename TO, int SWIGLU>
static int launch_stripe_rows(const SkinnyArgs& p, int ct, hipStream_t stream) {
  if (ct == 1) return launch_stripe_tile<MT, 1, TO, SWIGLU>(p, stream);
  if (ct == 2) return launch_stripe_tile<MT, 2, TO, SWIGLU>(p, stream);
  if (ct == 3) return launch_stripe_tile<MT, 3, TO, SWIGLU>(p, stream);
  return launch_stripe_tile<MT, 4, TO, SWIGLU>(p, stream);
}

template <typename TO, int SWIGLU>
static int launch_stripe(const SkinnyArgs& args, const StripePlan& plan, hipStream_t stream) {
  SkinnyArgs p = args;
  p.cols_wg = plan.cols;
  if (plan.mt == 1) return launch_stripe_rows<1, TO, SWIGLU>(p, plan.ct, stream);
  if (plan.mt == 2) return launch_stripe_rows<2, TO, SWIGLU>(p, plan.ct, stream);
  if (plan.mt == 3) return launch_stripe_rows<3, TO, SWIGLU>(p, plan.ct, stream);
  return launch_stripe_rows<4, TO, SWIGLU>(p, plan.ct, stream);
}

template <int PRO>
static int launch_skinny_out(const SkinnyArgs& p, int out_dtype, bool swiglu, hipStream_t stream) {
  if constexpr (PRO == PRO_NONE) {
    StripePlan plan;
    if (!(p.rows && out_dtype != 0) && p.lda <= T_MAX_INNER && stripe_plan(p.M, p.N, p.K, &plan)) {
      if (out_dtype == 0 && !swiglu) return launch_stripe<float, 0>(p, plan, stream);
      if (out_dtype == 1 && !swiglu) return launch_stripe<bf16_t, 0>(p, plan, stream);
      if (out_dtype == 1 && p.gate.kind == kGateSilu) return launch_stripe<bf16_t, 1>(p, plan, stream);
      if (out_dtype == 1) return launch_stripe<bf16_t, 2>(p, plan, stream);
    }
  }
  if (out_dtype == 0 && !swiglu) return launch_skinny<float, PRO, 0>(p, stream);
  if (out_dtype == 1 && !swiglu) return launch_skinny<bf16_t, PRO, 0>(p, stream);
  if (out_dtype == 1 && p.gate.kind == kGateSilu) return launch_skinny<bf16_t, PRO, 1>(p, stream);
  if constexpr (PRO == PRO_NONE)
    if (out_dtype == 1) return launch_skinny<bf16_t, PRO, 2>(p, stream);
  return TL_ERR_ARG;
}

// Column tiles a workgroup of the float32 few-row kernel owns: one, or, with one row tile and more
// than 256 column tiles of 16, up to three (four would not leave the registers for a piece of weights
// ahead) while the block sums fit into LDS, and of them as many columns (*cols_wg, even; 0: all) as make
// whole rounds of 256 workgroups: 5,120 columns are one round of 20, 15,360 two rounds of 30, 28,672
// three rounds of 38, where whole tiles would leave the last round a quarter full.
static int f32_rows_col_tiles(int M, int N, int K, int cols, int* cols_wg = nullptr) {
  if (cols_wg) *cols_wg = 0;
  if (M > 16 || cols != 16) return 1;
  const int tiles = (N + 15) / 16, nkb = (K + F_KBLOCK - 1) / F_KBLOCK;
  if (tiles <= 256) return 1;
  for (int rounds = 1; rounds <= 1024; ++rounds) {
    int cw = (N + 256 * rounds - 1) / (256 * rounds);
    cw += cw & 1;
    const int ct = (cw + 15) / 16;
    if (ct > 3 || (size_t)nkb * 16 * 16 * ct * sizeof(float) > 96 * 1024) continue;
    if (cols_wg && cw < 16 * ct && ct > 1) *cols_wg = cw;
    return ct;
  }
  return 1;
}

template <bool SWIGLU, int CT, bool PAIR, bool NORM>
static int launch_f32_lines_form(const F32RowsNorm& norm, const float* a, const float* w, float* out, const float* residual, int M, int N, int K,
                                 int64_t lda, int64_t ldo, const float* row_scale, int cw, size_t sums, hipStream_t stream) {
  const auto kernel = gemm_f32_lines_kernel<SWIGLU, CT, PAIR, NORM>;
  static bool configured = false;
  if (!configured) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(FL_STAGE_BYTES + FL_SUM_BYTES)) != hipSuccess)
      return TL_ERR_LAUNCH;
    configured = true;
  }
  hipLaunchKernelGGL(kernel, dim3((N + cw - 1) / cw), dim3(FR_THREADS), FL_STAGE_BYTES + sums, stream, norm, a, w, out, residual, M, N, K, lda, ldo,
                     row_scale, cw);
  return TL_OK;
}

// Whether and how the float32 product of at most 16 rows goes by whole lines: 8 columns a workgroup where that still is one round of
// workgroups over the 256 compute units (pairs of k blocks up to 8 rows), else one to three column tiles (f32_rows_col_tiles), one of as many
// (even) as make whole rounds of 256 workgroups.  With a norm one column tile, and not for the shortest inner sizes, where a wave has one block and
// gemm_f32_rows_kernel asks for all of it at once (us, that kernel and this one, which takes two steps: 1 row of 256 x 256 4.3 and 6.2, 512 x 512 5.0
// and 6.0, 768 x 768 6.2 and 6.5, 16 rows 6.6 and 6.4; beyond 2,048 columns, which have no pairs of blocks, 1 row of 4,096 x 1,152 1.08 times as long, 1,536
// 1.03, 2,048 1.01).  951 such products are 4 % faster on average for it; inner sizes that end just behind a block of 256, as 772 and 1,028, still are up to 1.11
// times as long as in that kernel.
struct F32Lines {
  int ct, cw;
  bool pair;
  size_t sums;      // bytes of block sums
};
static bool f32_lines_plan(int M, int N, int K, int64_t lda, bool norm, F32Lines* p) {
  if (M > 16 || lda > FL_MAX_STRIDE || K > FL_MAX_STRIDE) return false;
  if (norm && (K <= 640 || (K <= 768 && M <= 12) || (M < 8 && N > 2048 && K > 1024 && K <= 1536))) return false;
  const int nkb = (K + F_KBLOCK - 1) / F_KBLOCK;
  const bool eight = (N + 7) / 8 <= 256;
  p->pair = eight && M <= 8;
  p->cw = 0;
  p->ct = eight || norm ? 1 : f32_rows_col_tiles(M, N, K, 16, &p->cw);
  if (p->cw == 0) {
    const int rounds = (N + 256 * 16 - 1) / (256 * 16), even = ((N + 256 * rounds - 1) / (256 * rounds) + 1) / 2 * 2;
    p->cw = eight ? 8 : p->ct == 1 ? even : 16 * p->ct;
  }
  // (eight columns have sums for eight: 9 to 16 rows of up to 2,048 columns and inner sizes of 24,577 to 49,152 fit so)
  p->sums = (size_t)nkb * (p->pair ? 8 * 8 : 16 * (p->cw <= 8 ? 8 : 16 * p->ct)) * sizeof(float) + (norm ? (size_t)nkb * 16 * sizeof(float) : 0);
  return p->sums <= FL_SUM_BYTES;
}

template <bool SWIGLU, bool NORM>
static int launch_f32_lines(const F32Lines& p, const F32RowsNorm& norm, const float* a, const float* w, float* out, const float* residual, int M, int N,
                            int K, int64_t lda, int64_t ldo, const float* row_scale, hipStream_t stream) {
#define TL_LINES(CT, PAIR, NRM) launch_f32_lines_form<SWIGLU, CT, PAIR, NRM>(norm, a, w, out, residual, M, N, K, lda, ldo, row_scale, p.cw, p.sums, stream)
  if (p.pair) return TL_LINES(1, true, NORM);
  if (p.ct == 2) return TL_LINES(2, false, false);
  if (p.ct == 3) return TL_LINES(3, false, false);
  return TL_LINES(1, false, NORM);
#undef TL_LINES
}

}  // namespace

extern "C" {

int tl_linear_whole(int M, int N, int K);

// Float32, at most 64 rows: out = rmsnorm(x; norm_w, eps) @ w.T, then the epilogue of tl_linear_tile
// (0: + residual, 1: SiLU-gate), the norm inside the product's kernel.  Returns TL_ERR_ARG for sizes
// that kernel does not take (tl_linear_norm_f32_ok says which).
int tl_linear_norm_f32_ok(int M, int N, int K, int64_t lda) {
  const int nkb = (K + F_KBLOCK - 1) / F_KBLOCK, mts = (M + 15) / 16;
  const int cols = (N + 7) / 8 <= 256 ? 8 : 16;
  const size_t smem = (size_t)mts * nkb * 16 * (cols + 1) * sizeof(float);
  return M > 0 && M <= 16 * FR_MAX_MT && K % 4 == 0 && lda % 4 == 0 && smem <= 96 * 1024;
}

// Column tiles the plain float32 few-row product gives a workgroup at these sizes.  More than one: the
// product is so wide that a norm in front of it is cheaper as a kernel of its own (tl_norm_prescale_f32)
// with its factors applied to this product's sums than inside tl_linear_norm_f32, which fetches a
// workgroup's activation rows once per column tile; the bits are the same either way.
int tl_linear_f32_col_tiles(int M, int N, int K) {
  return f32_rows_col_tiles(M, N, K, (N + 7) / 8 <= 256 ? 8 : 16);
}

// Whether the float32 product of these sizes, rows in whole vectors, is gemm_f32_lines_kernel's (norm: with the norm inside).
int tl_linear_f32_lines(int M, int N, int K, int64_t lda, int norm) {
  F32Lines lines;
  return M > 0 && N > 0 && K > 0 && K % 4 == 0 && lda % 4 == 0 && f32_lines_plan(M, N, K, lda, norm != 0, &lines) ? 1 : 0;
}

int tl_linear_norm_f32(const float* x, const float* norm_w, float eps, const float* w, float* out,
                       const float* residual, int M, int N, int K, int64_t lda, int64_t ldo, int epilogue,
                       hipStream_t stream) {
  const bool swiglu = epilogue == 1;
  if (!tl_linear_norm_f32_ok(M, N, K, lda) || N <= 0 || lda < K || ldo < (swiglu ? N / 2 : N) || epilogue < 0 ||
      epilogue > 1 || ((uintptr_t)x | (uintptr_t)w | (uintptr_t)norm_w) % 16 != 0)
    return TL_ERR_ARG;
  if (swiglu && ((N & 1) || residual)) return TL_ERR_ARG;
  const int nkb = (K + F_KBLOCK - 1) / F_KBLOCK, mts = (M + 15) / 16;
  const int cols = (N + 7) / 8 <= 256 ? 8 : 16;
  const size_t smem = (size_t)mts * nkb * 16 * (cols + 1) * sizeof(float);
  F32Lines lines;
  if (f32_lines_plan(M, N, K, lda, true, &lines)) {
    const F32RowsNorm norm{norm_w, eps};
    const int rc = swiglu ? launch_f32_lines<true, true>(lines, norm, x, w, out, residual, M, N, K, lda, ldo, nullptr, stream)
                          : launch_f32_lines<false, true>(lines, norm, x, w, out, residual, M, N, K, lda, ldo, nullptr, stream);
    return rc == TL_OK ? tl_launch_status() : rc;
  }
  static bool configured = false;
  if (!configured) {
    const void* kernels[4] = {(const void*)gemm_f32_rows_kernel<true, 16, true, false>, (const void*)gemm_f32_rows_kernel<false, 16, true, false>,
                              (const void*)gemm_f32_rows_kernel<true, 8, true, false>, (const void*)gemm_f32_rows_kernel<false, 8, true, false>};
    for (const void* k : kernels)
      if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024) != hipSuccess) return TL_ERR_LAUNCH;
    configured = true;
  }
  dim3 gr((N + cols - 1) / cols);
#define TL_F32_ROWS_NORM(SW, CO)                                                                                 \
  hipLaunchKernelGGL((gemm_f32_rows_kernel<SW, CO, true, false>), gr, dim3(FR_THREADS), smem, stream, F32RowsNorm{norm_w, eps}, x, w, out, \
                     residual, M, N, K, lda, ldo)
  if (swiglu && cols == 16) TL_F32_ROWS_NORM(true, 16);
  else if (swiglu) TL_F32_ROWS_NORM(true, 8);
  else if (cols == 16) TL_F32_ROWS_NORM(false, 16);
  else TL_F32_ROWS_NORM(false, 8);
#undef TL_F32_ROWS_NORM
  return tl_launch_status();
}

// Float32, any number of rows: h[m, :] = norm_w * x[rows[m] or m, :] and inv_rms[m] = 1 / rms of that
// row, for a product that takes inv_rms as its row_scale: together rmsnorm(x) @ w.T with the bits of
// tl_linear_norm_f32.  h is [n_rows, K] contiguous.
int tl_norm_prescale_f32(const float* x, const float* norm_w, const int32_t* rows, float* h, float* inv_rms,
                         int n_rows, int K, int64_t lda, float eps, hipStream_t stream) {
  if (n_rows <= 0) return TL_OK;
  if (K <= 0 || lda < K) return TL_ERR_ARG;
  const int nkb = (K + F_KBLOCK - 1) / F_KBLOCK;
  const size_t smem = (size_t)nkb * 4 * sizeof(float);
  if (smem > 48 * 1024) return TL_ERR_ARG;
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ((uintptr_t)x | (uintptr_t)norm_w | (uintptr_t)h) % 16 == 0;
  if (vec)
    hipLaunchKernelGGL(norm_prescale_f32_kernel<true>, dim3(n_rows), dim3(FN_THREADS), smem, stream, x, norm_w, rows, h,
                       inv_rms, K, lda, eps);
  else
    hipLaunchKernelGGL(norm_prescale_f32_kernel<false>, dim3(n_rows), dim3(FN_THREADS), smem, stream, x, norm_w, rows,
                       h, inv_rms, K, lda, eps);
  return tl_launch_status();
}

// out = a @ w.T, then an epilogue.  dtype: element type of a and w (0 float32, 1 bfloat16);
// out_dtype: of out.  lda: row stride of a in elements; ldo: row stride of out and residual.
// row_scale (optional): every row m of the product is multiplied by row_scale[m] before the epilogue.
// epilogue 0: (+ residual[m, n]), out is [M, N].
// epilogue 1: SiLU-gate of interleaved columns, out[m, j] = silu(c[m, 2j]) * c[m, 2j+1], out is
//             [M, N/2] of the input's type; N must be even; no residual.
// epilogue 2 (bfloat16 in and out): out[m, n] = max(c[m, n], 0)^2; no residual.
// epilogues 3 and 4 (bfloat16 in and out): as 1 with the clamped unit of limit, alpha and shift, and with gelu(gate) * up.
// tile (bfloat16, M > 64): 0 lets the size decide; 1..4 force 256x256, 256x128, 128x128, 64x128.
int tl_linear_tile(const void* a, const void* w, void* out, const float* residual, const float* row_scale, int M,
                   int N, int K, int64_t lda, int64_t ldo, int dtype, int out_dtype, int epilogue, int tile,
                   float limit, float alpha, float shift, hipStream_t stream) {
  if (M <= 0) return TL_OK;
  const bool swiglu = is_gated(epilogue);
  if (N <= 0 || K <= 0 || lda < K || ldo < (swiglu ? N / 2 : N) || epilogue < 0 || epilogue > 4 || (dtype == 0 && epilogue > 2) || tile < 0 ||
      tile > 4)
    return TL_ERR_ARG;
  if (swiglu && ((N & 1) || residual || out_dtype != dtype)) return TL_ERR_ARG;
  const int act = epilogue == 2 ? kActRelu2 : kActNone;
  if (act != kActNone && (dtype != 1 || out_dtype != 1 || residual)) return TL_ERR_ARG;
  if (dtype == 0) {
    if (out_dtype != 0) return TL_ERR_ARG;
    const bool vec = K % 4 == 0 && lda % 4 == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0;
    const int nkb = (K + F_KBLOCK - 1) / F_KBLOCK;
    const int mts = (M + 15) / 16;
    F32Lines lines;
    if (vec && f32_lines_plan(M, N, K, lda, false, &lines)) {
      const F32RowsNorm none{};
      const int rc = swiglu ? launch_f32_lines<true, false>(lines, none, (const float*)a, (const float*)w, (float*)out, residual, M, N, K, lda,
                                                            ldo, row_scale, stream)
                            : launch_f32_lines<false, false>(lines, none, (const float*)a, (const float*)w, (float*)out, residual, M, N, K, lda,
                                                             ldo, row_scale, stream);
      return rc == TL_OK ? tl_launch_status() : rc;
    }
    // 17 to 64 rows, up to 256 by the estimate below (and what the kernel above does not take): matrix tiles of 16 columns, and the row
    // tiles shared out over as many groups of workgroups (1, 2 or 4) as it takes to give every compute unit a
    // workgroup and to fit the block sums into LDS (more groups only while they stay within one round of 256 workgroups: a second, partly
    // filled round costs as much as a full one).
    int groups = 1;
    const int col_tiles = (N + 15) / 16;
    while (groups < mts && (col_tiles * groups * 2 <= 256 || (size_t)((mts + groups - 1) / groups) * nkb * 16 * 16 * sizeof(float) > 96 * 1024))
      groups *= 2;
    const int tiles_wg = (mts + groups - 1) / groups;
    const size_t rows_smem = (size_t)tiles_wg * nkb * 16 * 16 * sizeof(float);
    // Up to 64 rows the few-row kernel; up to 256 where it is estimated faster than the tiled kernel, whose few
    // tiles each walk the whole inner size (f32_ring_us; where rows are no whole vectors, measured at inner size 2048: 87 us a
    // round of up to 352 tiles of 64 x 64, 204 us a round of 128 x 128; the few-row kernel 0.66 us per row tile and million
    // weights: 100 rows of 2560 x 2048 35 us, estimated 32, against 33; 200 rows of 2048 x 5632 119 against 81).  The bits are
    // the same.
    bool few_rows = M <= 16 * FR_MAX_MT;
    if (!few_rows && M <= 256) {
      const int64_t big_t = ceil_div64(N, 128) * ceil_div64(M, 128), small_t = ceil_div64(N, 64) * ceil_div64(M, 64);
      const bool small_tiles = (double)ceil_div64(small_t, 256) / (4 * 0.6) < (double)ceil_div64(big_t, 256);
      int mt, nt;
      const double tiled_us = f32_ring_ok(vec, K, lda) ? f32_ring_us(M, N, K, &mt, &nt)
                              : (K / 2048.0) * (small_tiles ? 87.0 * (small_t > 352 ? small_t / 352.0 : 1.0)
                                                            : 204.0 * (double)ceil_div64(big_t, 256));
      // (a long inner size leaves LDS for the block sums of one or two row tiles a workgroup only, and the
      // weights are then fetched once per row tile: 14336 x 4096 at 256 rows 876 us against 657)
      const double per_tile = tiles_wg >= 4 ? 0.66 : (tiles_wg >= 2 ? 0.8 : 0.98);
      few_rows = per_tile * mts * ((double)N * K / 1e6) + 8.0 < tiled_us;
    }
    if (few_rows && vec && rows_smem <= 96 * 1024) {
      static bool configured = false;
      if (!configured) {
        const void* kernels[2] = {(const void*)gemm_f32_rows_kernel<true, 16, false, true>, (const void*)gemm_f32_rows_kernel<false, 16, false, true>};
        for (const void* k : kernels)
          if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024) != hipSuccess)
            return TL_ERR_LAUNCH;
        configured = true;
      }
      dim3 gr((N + 15) / 16, (mts + tiles_wg - 1) / tiles_wg);
#define TL_F32_ROWS(SW)                                                                                              \
  hipLaunchKernelGGL((gemm_f32_rows_kernel<SW, 16, false, true>), gr, dim3(FR_THREADS), rows_smem, stream, F32RowsNorm{}, (const float*)a, \
                     (const float*)w, (float*)out, residual, M, N, K, lda, ldo, row_scale, tiles_wg)
      if (swiglu) TL_F32_ROWS(true);
      else TL_F32_ROWS(false);
#undef TL_F32_ROWS
      return tl_launch_status();
    }
    if (f32_ring_ok(vec, K, lda)) {
      const int rc = swiglu ? launch_f32_ring_any<true>((const float*)a, (const float*)w, (float*)out, nullptr, M, N, K, lda, ldo,
                                                        row_scale, stream)
                            : launch_f32_ring_any<false>((const float*)a, (const float*)w, (float*)out, residual, M, N, K, lda,
                                                         ldo, row_scale, stream);
      return rc == TL_OK ? tl_launch_status() : rc;
    }
    // 128 x 128 tiles, or 64 x 64 where those take fewer rounds of workgroups over the 256 compute
    // units even at 0.6 of the larger tile's rate (it fetches twice the operand bytes per flop)
    const int64_t big = ceil_div64(N, 128) * ceil_div64(M, 128), small = ceil_div64(N, 64) * ceil_div64(M, 64);
    const bool use_small = (double)ceil_div64(small, 256) / (4 * 0.6) < (double)ceil_div64(big, 256);
    const int bt = use_small ? 64 : 128;
    dim3 g((N + bt - 1) / bt, (M + bt - 1) / bt);
#define TL_F32_TILED(SW, VE)                                                                                        \
  do {                                                                                                              \
    if (use_small)                                                                                                  \
      hipLaunchKernelGGL((gemm_f32_kernel<SW, VE, 2>), g, dim3(F_THREADS), 0, stream, (const float*)a,              \
                         (const float*)w, (float*)out, residual, M, N, K, lda, ldo, row_scale);                     \
    else                                                                                                            \
      hipLaunchKernelGGL((gemm_f32_kernel<SW, VE, 4>), g, dim3(F_THREADS), 0, stream, (const float*)a,              \
                         (const float*)w, (float*)out, residual, M, N, K, lda, ldo, row_scale);                     \
  } while (0)
    if (swiglu && vec) TL_F32_TILED(true, true);
    else if (swiglu) TL_F32_TILED(true, false);
    else if (vec) TL_F32_TILED(false, true);
    else TL_F32_TILED(false, false);
#undef TL_F32_TILED
  } else if (dtype == 1) {
    if (K % 8 || lda % 8) return TL_ERR_ARG;
    if (out_dtype != 0 && out_dtype != 1) return TL_ERR_ARG;
    if (M <= 64) {
      SkinnyArgs p{a, (const bf16_t*)w, out, residual, nullptr, nullptr, row_scale, 0.f, 0, M, N, K, lda, ldo};
      p.act = act;
      p.gate = gate_of(epilogue, limit, alpha, shift);
      const int rc = launch_skinny_out<PRO_NONE>(p, out_dtype, swiglu, stream);
      if (rc != TL_OK) return rc;
    } else {
      int rc;
      TileNorm gated(row_scale);
      gated.gate = gate_of(epilogue, limit, alpha, shift);
      if (swiglu && gated.gate.kind != kGateSilu)
        rc = launch_gemm_bf16_any<bf16_t, 2>((const bf16_t*)a, (const bf16_t*)w, (bf16_t*)out, residual, gated, M, N, K, lda, ldo,
                                             tile, 0, stream);
      else if (swiglu)
        rc = launch_gemm_bf16_any<bf16_t, 1>((const bf16_t*)a, (const bf16_t*)w, (bf16_t*)out, residual, gated,
                                                M, N, K, lda, ldo, tile, 0, stream);
      else if (out_dtype == 0)
        rc = launch_gemm_bf16_any<float, 0>((const bf16_t*)a, (const bf16_t*)w, (float*)out, residual, row_scale,
                                                M, N, K, lda, ldo, tile, 0, stream);
      else
        rc = launch_gemm_bf16_any<bf16_t, 0>((const bf16_t*)a, (const bf16_t*)w, (bf16_t*)out, residual,
                                                 TileNorm(row_scale, act), M, N, K, lda, ldo, tile, 0, stream);
      if (rc != TL_OK) return rc;
    }
  } else {
    return TL_ERR_ARG;
  }
  return tl_launch_status();
}

int tl_linear(const void* a, const void* w, void* out, const float* residual, const float* row_scale, int M,
              int N, int K, int64_t lda, int64_t ldo, int dtype, int out_dtype, int epilogue,
              hipStream_t stream) {
  if (epilogue == 3) return TL_ERR_ARG;      // its limit has no place here
  return tl_linear_tile(a, w, out, residual, row_scale, M, N, K, lda, ldo, dtype, out_dtype, epilogue, 0, 0.f, 0.f, 0.f, stream);
}

// Whether tl_linear_set may be told to leave a product's results as tanh in bfloat16 (inner sizes of whole 64).
int tl_linear_set_tanh(int K) { return K > 0 && K % 64 == 0 && K <= T_MAX_INNER; }

// `count` products of at most 16 rows, one inner size: out[i] (float32 [M, n[i]], rows ldo[i] apart) = a[i] @ w[i]^T,
// a[i] bfloat16 [M, K] with rows lda[i] apart, w[i] bfloat16 [n[i], K]; tanh[i] (where tl_linear_set_tanh says so): out[i] is bfloat16, the tanh of
// the sums.  The arrays are read here, before the launch.
int tl_linear_set(const void* const* a, const void* const* w, void* const* out, const int32_t* n, const int64_t* lda,
                  const int64_t* ldo, const int32_t* tanh, int count, int M, int K, hipStream_t stream) {
  if (count <= 0 || M <= 0) return TL_OK;
  if (count > S_SET || M > 16 || K <= 0 || K % 8) return TL_ERR_ARG;
  SkinnySet set{};
  int most = 0;
  bool whole = tl_linear_set_tanh(K), any_tanh = false;
  set.vec = 1;
  for (int i = 0; i < count; ++i) {
    if (n[i] <= 0 || lda[i] % 8 || lda[i] < K || ldo[i] < n[i] || !a[i] || !w[i] || !out[i]) return TL_ERR_ARG;
    set.p[i] = SkinnyArgs{a[i], (const bf16_t*)w[i], out[i], nullptr, nullptr, nullptr, nullptr, 0.f, 0, M, n[i], K, lda[i], ldo[i]};
    set.p[i].act = tanh[i] ? kActTanh : kActNone;
    any_tanh = any_tanh || tanh[i];
    whole = whole && lda[i] <= T_MAX_INNER;
    if (!tanh[i] && (ldo[i] % 4 || n[i] % 4 || (uintptr_t)out[i] % 16)) set.vec = 0;
    most = n[i] > most ? n[i] : most;
  }
  if (any_tanh && !whole) return TL_ERR_ARG;
  if (whole) {
    const int cols = stripe_set_cols(set, count);
    const int rc = cols > 32 ? launch_stripe_set<3, 64>(set, count, most, cols, stream)
                   : cols > 16 ? (K % 128 == 0 ? launch_stripe_set<2, 128>(set, count, most, cols, stream)
                                               : launch_stripe_set<2, 64>(set, count, most, cols, stream))
                   : K % 128 == 0 ? launch_stripe_set<1, 128>(set, count, most, cols, stream)
                                  : launch_stripe_set<1, 64>(set, count, most, cols, stream);
    return rc == TL_OK ? tl_launch_status() : rc;
  }
  const size_t smem = (size_t)S_WAVES * 16 * 17 * sizeof(float) + (size_t)(S_WAVES + 1) * 16 * sizeof(float);
  hipLaunchKernelGGL(gemm_skinny_set_kernel, dim3((most + S_COLS - 1) / S_COLS, count), dim3(S_THREADS), smem, stream, set);
  return tl_launch_status();
}

// The bfloat16 product that takes part in handing a norm from one product to the next (see
// SkinnyArgs and TileNorm): the few-row kernel up to 64 rows, the tiled kernel beyond (no row
// gather then; a producer needs N to be a multiple of 64).  Consumer side: in_sumsq [rows of a,
// in_parts] (a is then the operand a producer wrote; `rows` gathers rows of both).  Producer side
// (out_dtype 0, epilogue 0): emit_w [N] (element type emit_w_dtype), emit_operand bf16 [M, N],
// emit_sumsq float [M, tl_handoff_parts(M, N, K)].  Either side may be absent.
int tl_linear_handoff(const void* a, const void* w, void* out, const float* residual, const int32_t* rows,
                      const float* in_sumsq, int in_parts, float in_eps, int in_width, const void* emit_w,
                      int emit_w_dtype, void* emit_operand, float* emit_sumsq, int M, int N, int K, int64_t lda,
                      int64_t ldo, int out_dtype, int epilogue, hipStream_t stream) {
  if (M <= 0) return TL_OK;
  const bool swiglu = epilogue == 1;
  if (N <= 0 || K <= 0 || K % 8 || lda % 8 || lda < K || ldo < (swiglu ? N / 2 : N) || epilogue < 0 ||
      epilogue > 1 || (out_dtype != 0 && out_dtype != 1))
    return TL_ERR_ARG;
  if (swiglu && ((N & 1) || residual || out_dtype != 1)) return TL_ERR_ARG;
  if (in_sumsq && (in_parts <= 0 || in_width <= 0)) return TL_ERR_ARG;
  const bool emit = emit_operand != nullptr;
  if (emit && (!emit_w || !emit_sumsq || swiglu || out_dtype != 0 || (emit_w_dtype != 0 && emit_w_dtype != 1)))
    return TL_ERR_ARG;
  if (M > 64) {      // the tiled kernel
    if (rows || (emit && (N % 64 || ldo % 4))) return TL_ERR_ARG;
    TileNorm nm;
    if (emit) {
      nm.emit_w = emit_w;
      nm.emit_w_is_f32 = emit_w_dtype == 0 ? 1 : 0;
      nm.emit_operand = (bf16_t*)emit_operand;
      nm.emit_ld = N;
      nm.emit_sumsq = emit_sumsq;
      nm.emit_parts = N / 64;
    }
    if (in_sumsq) {
      nm.in_sumsq = in_sumsq;
      nm.in_parts = in_parts;
      nm.in_width = in_width;
      nm.in_eps = in_eps;
    }
    int rc;
    if (swiglu)
      rc = launch_gemm_bf16_any<bf16_t, 1>((const bf16_t*)a, (const bf16_t*)w, (bf16_t*)out, residual, nm, M, N, K,
                                              lda, ldo, 0, 0, stream);
    else if (out_dtype == 0)
      rc = launch_gemm_bf16_any<float, 0>((const bf16_t*)a, (const bf16_t*)w, (float*)out, residual, nm, M, N, K,
                                              lda, ldo, 0, 0, stream);
    else
      rc = launch_gemm_bf16_any<bf16_t, 0>((const bf16_t*)a, (const bf16_t*)w, (bf16_t*)out, residual, nm, M, N, K,
                                               lda, ldo, 0, 0, stream);
    if (rc != TL_OK) return rc;
    return tl_launch_status();
  }
  SkinnyArgs p{a, (const bf16_t*)w, out, residual, nullptr, rows, nullptr, 0.f, 0, M, N, K, lda, ldo};
  if (emit) {
    p.emit_w = emit_w;
    p.emit_w_is_f32 = emit_w_dtype == 0 ? 1 : 0;
    p.emit_operand = (bf16_t*)emit_operand;
    p.emit_sumsq = emit_sumsq;
    if (lda > T_MAX_INNER && tl_linear_whole(M, N, K)) return TL_ERR_ARG;      // its parts would not be tl_handoff_parts'
  }
  if (in_sumsq) {
    p.in_sumsq = in_sumsq;
    p.in_parts = in_parts;
    p.in_width = in_width;
    p.in_eps = in_eps;
  }
  const int rc = launch_skinny_out<PRO_NONE>(p, out_dtype, swiglu, stream);
  if (rc != TL_OK) return rc;
  return tl_launch_status();
}

// out = a @ w[g]^T by runs of rows: a bfloat16 [M, K] whose aligned runs of `group_rows` rows (256: a multiple of
// every tile height; M a multiple of it) each belong to one group g = tile_group[run] (negative: the run holds no
// row and nothing is computed or written for it); w bfloat16 [groups, N, K]; out [M, N] bfloat16 or float32.
// swiglu: the N columns are (gate_j, up_j) pairs and out [M, N / 2] (bfloat16) = silu(gate) * up.
int tl_linear_grouped(const void* a, const void* w, void* out, const int32_t* tile_group, int group_rows, int M, int N,
                      int K, int64_t lda, int64_t ldo, int out_dtype, int swiglu, hipStream_t stream) {
  if (M <= 0) return TL_OK;
  if (N <= 0 || K <= 0 || K % 8 || lda % 8 || lda < K || ldo < (swiglu ? N / 2 : N) || (out_dtype != 0 && out_dtype != 1) ||
      !tile_group || group_rows != 256 || M % group_rows || !a || !w || !out || (swiglu && (out_dtype != 1 || (N & 1))))
    return TL_ERR_ARG;
  TileNorm nm;
  nm.tile_group = tile_group;
  nm.group_rows = group_rows;
  nm.group_stride = (int64_t)N * K;
  int rc;
  if (swiglu)
    rc = launch_gemm_bf16_any<bf16_t, 1>((const bf16_t*)a, (const bf16_t*)w, (bf16_t*)out, nullptr, nm, M, N, K, lda,
                                            ldo, 0, 0, stream);
  else if (out_dtype == 0)
    rc = launch_gemm_bf16_any<float, 0>((const bf16_t*)a, (const bf16_t*)w, (float*)out, nullptr, nm, M, N, K, lda,
                                            ldo, 0, 0, stream);
  else
    rc = launch_gemm_bf16_any<bf16_t, 0>((const bf16_t*)a, (const bf16_t*)w, (bf16_t*)out, nullptr, nm, M, N, K, lda,
                                             ldo, 0, 0, stream);
  if (rc != TL_OK) return rc;
  return tl_launch_status();
}

// Whether a bfloat16 product of these sizes is gemm_stripe_bf16_kernel's (see stripe_plan): it is not split then.
int tl_linear_whole(int M, int N, int K) {
  StripePlan plan;
  return stripe_plan(M, N, K, &plan) ? 1 : 0;
}

// How many partial sums of squares per row tl_linear_handoff writes as a producer for these sizes: by whole lines one per workgroup,
// whose columns are stripe_plan's (any multiple of 4 from 8 to 64); other products of up to 64 rows one per workgroup and column
// tile (8 or 16 columns, or as many as make whole rounds); beyond 64 rows one per 64 columns.
int tl_handoff_parts(int M, int N, int K) {
  if (M > 64) return (N + 63) / 64;
  StripePlan plan;
  if (stripe_plan(M, N, K, &plan)) return (N + plan.cols - 1) / plan.cols;
  if (skinny_half(M, N, K)) return (N + 7) / 8;
  // one column tile a workgroup (see launch_skinny and launch_skinny_rows): a part per workgroup
  if (M <= 16 && N > 256 * S_COLS && N <= 4 * 256 * S_COLS) {       // two to four column tiles a workgroup
    const int ct = (N + 256 * S_COLS - 1) / (256 * S_COLS), cwt = skinny_cols_wg_tiles(N, ct);
    return cwt ? (N + cwt - 1) / cwt * ct : (N + S_COLS - 1) / S_COLS;
  }
  const bool one_tile = M <= 16 || N < 256 * 32;
  const int cw = one_tile ? skinny_cols_wg(N) : S_COLS;
  return (N + cw - 1) / cw;
}

// How the operands of a tile (1 to 4, as tl_linear_tile's) reach LDS at these sizes (see tile_mode): 0 and 1 through
// registers, 2 and 3 straight from memory.
int tl_tile_mode(int tile, int M, int N, int K, int k_per_split) {
  return tile >= 1 && tile <= 4 ? tile_mode(kTiles[tile - 1].bm, kTiles[tile - 1].bn, M, N, K, k_per_split) : -1;
}

// The tile (1 to 4) that a product of these sizes takes unless it is split or launched in two parts.
int tl_best_tile(int M, int N, int K) { return best_tile(M, N, K, nullptr) + 1; }

// Where tile t of tiles_m x tiles_n stands (see tile_place): place[0] its row of tiles, place[1] its column.
void tl_tile_place(int t, int tiles_m, int tiles_n, int banded, int* place) {
  tile_place(t, tiles_m, tiles_n, banded != 0, place, place + 1);
}

// See splitk_plan.  A caller that gets more than one split allocates a float32 workspace of
// splits * M * N elements and calls tl_linear_splitk with the same sizes.
int tl_splitk_plan(int M, int N, int K) {
  int tile, kps;
  return splitk_plan(M, N, K, &tile, &kps);
}

// The bfloat16 product with its inner size split over workgroups: partial products into
// `workspace` (float32 [splits, M, N], splits as tl_splitk_plan says), then one kernel that adds
// them up and applies the epilogue.  Arguments as tl_linear and tl_linear_handoff (no row gather);
// emit_sumsq is float [M, ceil(N / 1024)].
int tl_linear_splitk(const void* a, const void* w, void* out, const float* residual, const float* row_scale,
                     const float* in_sumsq, int in_parts, float in_eps, int in_width, const void* emit_w,
                     int emit_w_dtype, void* emit_operand, float* emit_sumsq, int M, int N, int K, int64_t lda,
                     int64_t ldo, int out_dtype, int epilogue, float limit, float alpha, float shift, float* workspace,
                     hipStream_t stream) {
  const bool swiglu = is_gated(epilogue);
  if (M <= 0 || N <= 0 || K <= 0 || K % 8 || lda % 8 || lda < K || ldo < (swiglu ? N / 2 : N) || epilogue < 0 ||
      epilogue > 4 || (out_dtype != 0 && out_dtype != 1) || !workspace)
    return TL_ERR_ARG;
  if (swiglu && ((N & 1) || residual || out_dtype != 1)) return TL_ERR_ARG;
  const int act = epilogue == 2 ? kActRelu2 : kActNone;
  if (act != kActNone && (out_dtype != 1 || residual)) return TL_ERR_ARG;
  if (in_sumsq && (in_parts <= 0 || in_width <= 0)) return TL_ERR_ARG;
  const bool emit = emit_operand != nullptr;
  if (emit && (!emit_w || !emit_sumsq || swiglu || out_dtype != 0 || (emit_w_dtype != 0 && emit_w_dtype != 1)))
    return TL_ERR_ARG;
  int tile, kps;
  const int splits = splitk_plan(M, N, K, &tile, &kps);
  if (splits < 2) return TL_ERR_ARG;
  int rc = TL_OK;
  if (tile < 0) {
    const int slabs = kps / O_SLAB_K;
    const size_t smem = (size_t)(slabs < O_RING ? slabs : O_RING) * O_SLAB_BYTES;
    static bool configured = false;
    if (!configured) {
      if (hipFuncSetAttribute((const void*)gemm_oneshot_bf16_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                              O_RING * O_SLAB_BYTES) != hipSuccess)
        return TL_ERR_LAUNCH;
      configured = true;
    }
    hipLaunchKernelGGL(gemm_oneshot_bf16_kernel, dim3((N + O_BN - 1) / O_BN, splits, (M + O_BM - 1) / O_BM), dim3(O_THREADS), smem, stream,
                       (const bf16_t*)a, (const bf16_t*)w, workspace, M, N, K, lda, slabs);
  } else {
    rc = launch_gemm_bf16_any<float, 0>((const bf16_t*)a, (const bf16_t*)w, workspace, nullptr, nullptr, M, N, K, lda,
                                            N, tile, kps, stream);
  }
  if (rc != TL_OK) return rc;
  ReduceArgs p{workspace, splits, M, N, out, ldo, residual, row_scale, in_sumsq, in_parts, in_width, in_eps, emit_w,
               emit_w_dtype == 0 ? 1 : 0, (bf16_t*)emit_operand, emit_sumsq, act, gate_of(epilogue, limit, alpha, shift)};
  if (M > 65535) return TL_ERR_ARG;
  dim3 g(M, (N + R_CHUNK - 1) / R_CHUNK), b(R_THREADS);
  if (swiglu && p.gate.kind != kGateSilu)
    hipLaunchKernelGGL((splitk_reduce_kernel<bf16_t, 2>), g, b, 0, stream, p);
  else if (swiglu)
    hipLaunchKernelGGL((splitk_reduce_kernel<bf16_t, 1>), g, b, 0, stream, p);
  else if (out_dtype == 0)
    hipLaunchKernelGGL((splitk_reduce_kernel<float, 0>), g, b, 0, stream, p);
  else
    hipLaunchKernelGGL((splitk_reduce_kernel<bf16_t, 0>), g, b, 0, stream, p);
  return tl_launch_status();
}

// Few-row (M <= 16) bfloat16 product whose input is the float32 residual stream: the rows of a
// (gathered through `rows` if given) are RMS-normalised with norm_w (float32 or bfloat16) and eps
// inside the kernel.  Epilogues as in tl_linear.
int tl_linear_norm(const void* a, const void* w, void* out, const float* residual, const void* norm_w,
                   const int32_t* rows, float eps, int norm_w_dtype, int M, int N, int K, int64_t lda,
                   int64_t ldo, int out_dtype, int epilogue, hipStream_t stream) {
  if (M <= 0) return TL_OK;
  const bool swiglu = epilogue == 1;
  if (M > 16 || N <= 0 || K <= 0 || K % 8 || lda % 8 || lda < K || ldo < (swiglu ? N / 2 : N) || !norm_w ||
      (norm_w_dtype != 0 && norm_w_dtype != 1) || epilogue < 0 || epilogue > 1)
    return TL_ERR_ARG;
  if (swiglu && ((N & 1) || residual)) return TL_ERR_ARG;
  SkinnyArgs p{a, (const bf16_t*)w, out, residual, norm_w, rows, nullptr, eps, norm_w_dtype == 0 ? 1 : 0, M, N, K, lda, ldo};
  const int rc = launch_skinny_out<PRO_NORM>(p, out_dtype, swiglu, stream);
  if (rc != TL_OK) return rc;
  return tl_launch_status();
}

}  // extern "C"
