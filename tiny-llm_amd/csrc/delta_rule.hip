// The gated delta rule with one decay per head and key channel (or one per head, laid out over the
// channels where the recurrence reads it), as a recurrence over a state
// S [dim, vdim] per request and head:
//     S <- diag(g_t) S;  u = beta_t (v_t - S^T k_t);  S <- S + k_t u^T;  o_t = S^T q_t
// and what surrounds it: short causal convolutions with SiLU on q, k and v (their last taps - 1
// inputs are state as well), unit vectors q and k, the decay g = exp(-exp(A_log) softplus(a + dt_bias)),
// and the per-head norm with its gate on the way out.  The state, and everything that enters the
// recurrence, is float32 in both precisions.
//
// Per request the state is ONE row of float32: [S of every head: heads x dim x vdim | the
// convolutions' last inputs: channels x (taps - 1), oldest first].
#include "common.h"

#include <type_traits>

namespace {

constexpr int kPrepThreads = 128;
constexpr int kPrepWaves = kPrepThreads / TL_WAVE;
constexpr int kMaxDim = 256;      // key channels a head may have

__device__ __forceinline__ float silu(float x) { return x / (1.f + expf(-x)); }
__device__ __forceinline__ float softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// Input m of channel c (column `col` of the projections) of the request whose tokens of this step
// start at row t0: m >= 0 is row t0 + m of this step, m < 0 reaches back into the saved inputs.
template <typename T>
__device__ __forceinline__ float conv_input(const T* __restrict__ p, int64_t p_stride, int t0, int m, int col,
                                            const float* __restrict__ saved, int taps) {
  return m >= 0 ? to_f32(p[(int64_t)(t0 + m) * p_stride + col]) : saved[(taps - 1) + m];
}

// Up to four taps (the usual sizes) are requested together; the sum runs from the oldest input to the
// current one either way.
template <typename T>
__device__ __forceinline__ float conv_silu(const T* __restrict__ p, int64_t p_stride, int t0, int n, int col,
                                           const float* __restrict__ saved, const float* __restrict__ w, int taps) {
  float acc = 0.f;
  if (taps <= 4) {
    float x[4], wt[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {       // tap j of the weights meets input n - (taps - 1) + j
      x[j] = j < taps ? conv_input(p, p_stride, t0, n - (taps - 1) + j, col, saved, taps) : 0.f;
      wt[j] = j < taps ? w[j] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = fmaf(wt[j], x[j], acc);
    return silu(acc);
  }
  for (int j = 0; j < taps; ++j) acc = fmaf(w[j], conv_input(p, p_stride, t0, n - (taps - 1) + j, col, saved, taps), acc);
  return silu(acc);
}

// One workgroup per (token, head).  Row t of `p` holds [q (kv_heads x dim) | k (kv_heads x dim) |
// v (heads x vdim)] from column conv_off on, and beta's pre-activation at column b_off + head;
// row t of `a` holds the decay's pre-activation at column head * dim + i, or, with a_per_head, one per
// head at column head (dt_bias is indexed likewise).
template <typename T>
__global__ __launch_bounds__(kPrepThreads) void delta_prepare_kernel(
    const T* __restrict__ p, int64_t p_stride, int conv_off, int b_off, const float* __restrict__ a, int64_t a_stride,
    const float* __restrict__ conv_w, const float* __restrict__ a_log, const float* __restrict__ dt_bias,
    const float* __restrict__ state, int64_t state_stride, int64_t saved_off, const int32_t* __restrict__ req_of_token,
    const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ state_slots, float* __restrict__ qn,
    float* __restrict__ kn, float* __restrict__ vc, float* __restrict__ beta, float* __restrict__ decay, int heads,
    int kv_heads, int dim, int vdim, int taps, float q_scale, int a_per_head) {
  __shared__ float qs[kMaxDim], ks[kMaxDim], red[kPrepWaves];
  const int t = blockIdx.x, h = blockIdx.y;
  const int r = req_of_token[t];
  const int t0 = cu_seqlens[r], t1 = cu_seqlens[r + 1];
  const int64_t base = (int64_t)t * heads + h;
  if (t < t0 || t >= t1) {            // a padding row of a captured step: finite stand-ins, never read
    for (int i = threadIdx.x; i < dim; i += kPrepThreads) qn[base * dim + i] = kn[base * dim + i] = decay[base * dim + i] = 0.f;
    for (int j = threadIdx.x; j < vdim; j += kPrepThreads) vc[base * vdim + j] = 0.f;
    if (threadIdx.x == 0) beta[base] = 0.f;
    return;
  }
  const int n = t - t0;
  const int kh = h / (heads / kv_heads);
  const float* saved = state + (int64_t)state_slots[r] * state_stride + saved_off;
  const int q_ch = kh * dim, k_ch = kv_heads * dim + kh * dim, v_ch = 2 * kv_heads * dim + h * vdim;
  float sq = 0.f, sk = 0.f;
  for (int i = threadIdx.x; i < dim; i += kPrepThreads) {
    const float q = conv_silu(p, p_stride, t0, n, conv_off + q_ch + i, saved + (int64_t)(q_ch + i) * (taps - 1),
                              conv_w + (int64_t)(q_ch + i) * taps, taps);
    const float k = conv_silu(p, p_stride, t0, n, conv_off + k_ch + i, saved + (int64_t)(k_ch + i) * (taps - 1),
                              conv_w + (int64_t)(k_ch + i) * taps, taps);
    qs[i] = q;
    ks[i] = k;
    sq += q * q;
    sk += k * k;
  }
  sq = block_sum<kPrepWaves>(sq, red);
  sk = block_sum<kPrepWaves>(sk, red);
  const float rq = q_scale / sqrtf(sq + 1e-6f), rk = 1.f / sqrtf(sk + 1e-6f);
  const float rate = expf(a_log[h]);
  for (int i = threadIdx.x; i < dim; i += kPrepThreads) {
    qn[base * dim + i] = qs[i] * rq;
    kn[base * dim + i] = ks[i] * rk;
    const int ai = a_per_head ? h : h * dim + i;
    const float pre = a[(int64_t)t * a_stride + ai] + dt_bias[ai];
    decay[base * dim + i] = expf(-rate * softplus(pre));
  }
  for (int j = threadIdx.x; j < vdim; j += kPrepThreads)
    vc[base * vdim + j] = conv_silu(p, p_stride, t0, n, conv_off + v_ch + j, saved + (int64_t)(v_ch + j) * (taps - 1),
                                    conv_w + (int64_t)(v_ch + j) * taps, taps);
  if (threadIdx.x == 0) beta[base] = 1.f / (1.f + expf(-to_f32(p[(int64_t)t * p_stride + b_off + h])));
}

// The convolutions' saved inputs after a step: the last taps - 1 of (what was saved, this step's
// inputs, each with its channel's bias added if the projections carry one).  One thread per (request, channel); it
// reads all it needs before it writes.
constexpr int kMaxTaps = 16;
template <typename T>
__global__ void conv_state_update_kernel(const T* __restrict__ p, int64_t p_stride, int conv_off, int channels,
                                         const float* __restrict__ bias, float* __restrict__ state,
                                         int64_t state_stride, int64_t saved_off,
                                         const int32_t* __restrict__ cu_seqlens,
                                         const int32_t* __restrict__ state_slots, int taps) {
  const int r = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int t0 = cu_seqlens[r], n = cu_seqlens[r + 1] - t0;
  if (c >= channels || n <= 0) return;
  float* saved = state + (int64_t)state_slots[r] * state_stride + saved_off + (int64_t)c * (taps - 1);
  float next[kMaxTaps];
  const float b = bias ? bias[c] : 0.f;
#pragma unroll
  for (int i = 0; i < kMaxTaps; ++i)
    if (i < taps - 1) {
      const int m = n - (taps - 1) + i;
      next[i] = conv_input(p, p_stride, t0, m, conv_off + c, saved, taps);
      if (m >= 0) next[i] += b;           // what is saved has it already
    }
#pragma unroll
  for (int i = 0; i < kMaxTaps; ++i)
    if (i < taps - 1) saved[i] = next[i];
}

// The recurrence.  A wave owns 8 value columns of one (request, head): lane (s, c) keeps rows
// [s * DS, (s + 1) * DS) of column c of S in registers (eight slices of the key channels side by side,
// 8 lanes each), so a token costs DS steps and two sums over the eight slices instead of `dim` steps.
// The wave walks the request's tokens of this step in order, kCh at a time: q, k, decay, v and beta of a
// chunk go through LDS, and the next chunk's are requested before this one is worked on.  The four waves
// of a workgroup (32 columns) share the staged chunk: q, k and decay are the same for every column.
constexpr int kCh = 16;           // tokens per staged chunk
constexpr int kCols = 8;          // value columns per wave
constexpr int kRecWaves = 4, kRecThreads = kRecWaves * TL_WAVE, kRecCols = kRecWaves * kCols;
constexpr int kSlices = TL_WAVE / kCols;
// x and y summed over the lanes c, c + 8, ..., c + 56, every lane gets both: after the step over 8 lanes the two travel
// together, x in the even and y in the odd rows of 16 lanes.
__device__ __forceinline__ void sum_over_slices(float& x, float& y) {
  x += dpp_f32<TL_DPP_ROR8>(x);
  y += dpp_f32<TL_DPP_ROR8>(y);
  const tl_u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  float a, b;
  pair32(__uint_as_float(r[0]) + __uint_as_float(r[1]), a, b);
  pair16(a + b, x, y);
}
// VEC: the head's channels are a multiple of four, and their rows begin on 16 bytes.
template <int DS, bool VEC>
__global__ __launch_bounds__(kRecThreads) void delta_recurrence_kernel(
    const float* __restrict__ qn, const float* __restrict__ kn, const float* __restrict__ vc,
    const float* __restrict__ beta, const float* __restrict__ decay, float* __restrict__ state, int64_t state_stride,
    const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ state_slots, float* __restrict__ out,
    int heads, int dim, int vdim) {
  constexpr int DP = kSlices * DS;                // key channels, padded
  constexpr int PER = (kCh * DP + kRecThreads - 1) / kRecThreads;    // floats of one staged array a thread moves per chunk
  constexpr int PERV = kCh * kRecCols / kRecThreads;
  __shared__ __attribute__((aligned(16))) float ks[kCh][DP], qs[kCh][DP], gs[kCh][DP];
  __shared__ float vs[kCh][kRecCols], bs[kCh], kqs[kCh];
  const int r = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wave = tid / TL_WAVE, lane = tid % TL_WAVE;
  const int s = lane / kCols, c = wave * kCols + lane % kCols;
  const int col = blockIdx.z * kRecCols + c;
  const int t0 = cu_seqlens[r], t1 = cu_seqlens[r + 1];
  if (t1 <= t0) return;                           // a padding request owns no state
  const bool live = col < vdim;
  float* S_mem = state + (int64_t)state_slots[r] * state_stride + (int64_t)h * dim * vdim + col;
  constexpr int V = VEC ? 4 : 1, PIECES = (PER + V - 1) / V;
  typedef float piece __attribute__((ext_vector_type(V)));
  piece rk[PIECES], rq[PIECES], rg[PIECES];
  float rv[PERV], rb = 0.f;
  // element e of a staged array: token e / DP of the chunk, channel e % DP (channels beyond dim: k = q = 0, g = 1)
  auto fetch = [&](int tc) {
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
      const int e = (j * kRecThreads + tid) * V, tt = e / DP, i = e % DP;
      const bool ok = e < kCh * DP && tc + tt < t1 && i < dim;
      const int64_t at = ((int64_t)(tc + tt) * heads + h) * dim + i;
      rk[j] = rq[j] = 0.f;
      rg[j] = 1.f;
      if (ok) {
        rk[j] = *(const piece*)(kn + at);
        rq[j] = *(const piece*)(qn + at);
        rg[j] = *(const piece*)(decay + at);
      }
    }
#pragma unroll
    for (int j = 0; j < PERV; ++j) {
      const int e = j * kRecThreads + tid, tt = e / kRecCols, cc = e % kRecCols;
      const int vcol = blockIdx.z * kRecCols + cc;
      rv[j] = (tc + tt < t1 && vcol < vdim) ? vc[((int64_t)(tc + tt) * heads + h) * vdim + vcol] : 0.f;
    }
    rb = (tid < kCh && tc + tid < t1) ? beta[(int64_t)(tc + tid) * heads + h] : 0.f;
  };
  // The state is requested behind the first chunk, which is staged (and its k . q formed) while the state is on its way: a
  // portion of a few tokens is little else.  32 requests of 32 heads and two tokens, 64 x 128, behind the state 18.9 us, so
  // 16.5.  With 32 rows a lane the two are more loads than a wave can tell apart (63), so that it would wait for all.
  float S[DS];
  if constexpr (DS == 32) {
#pragma unroll
    for (int i = 0; i < DS; ++i) S[i] = (live && s * DS + i < dim) ? S_mem[(int64_t)(s * DS + i) * vdim] : 0.f;
  }
  fetch(t0);
  if constexpr (DS < 32) {
#pragma unroll
    for (int i = 0; i < DS; ++i) S[i] = (live && s * DS + i < dim) ? S_mem[(int64_t)(s * DS + i) * vdim] : 0.f;
  }
  for (int tc = t0; tc < t1; tc += kCh) {
    __syncthreads();                              // the chunk before has been read
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
      const int e = (j * kRecThreads + tid) * V;
      if (e < kCh * DP) {
        *(piece*)(&ks[0][0] + e) = rk[j];
        *(piece*)(&qs[0][0] + e) = rq[j];
        *(piece*)(&gs[0][0] + e) = rg[j];
      }
    }
#pragma unroll
    for (int j = 0; j < PERV; ++j) (&vs[0][0])[j * kRecThreads + tid] = rv[j];
    if (tid < kCh) bs[tid] = rb;
    __syncthreads();
    if (tc + kCh < t1) fetch(tc + kCh);           // on its way while this chunk is worked on
    const int n = min(kCh, t1 - tc);
    // k . q of the chunk's tokens, sixteen threads a token (all sixteen: skipping those that are not there cost 801 tokens 3 %)
    {
      static_assert(kRecThreads == 16 * kCh, "sixteen threads a token");
      const int tt = tid / 16;
      float kq = 0.f;
#pragma unroll
      for (int i = 0; i < DP / 16; ++i) kq = fmaf(ks[tt][tid % 16 + i * 16], qs[tt][tid % 16 + i * 16], kq);
      kq = group_sum<16>(kq);
      if (tid % 16 == 0) kqs[tt] = kq;
    }
    __syncthreads();
    // With S' = diag(g) S:  o = (S' + k u^T)^T q = S'^T q + u (k . q).  Both sums over S' are
    // taken in ONE pass (in four independent parts) and meet in one round of exchanges between the
    // slices; the update of S hangs off it.  A token's operands are read from LDS while the token before
    // it is worked on (two register sets, the loop goes two tokens at a time).  What a token costs is what its
    // waves issue (two a SIMD): with k . q in every wave and the sums exchanged one by one 801 tokens (five shorter prompts
    // beside them) took 314 us, now 275.  16 slices of half the rows, 4 columns a wave, took 8 % less for them in an
    // earlier form, but 1.45 times as long for eight prompts of 13 tokens.
    auto load = [&](int tt, float* k, float* q, float* g, float& v, float& bt, float& kq) {
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        k[i] = ks[tt][s * DS + i];
        q[i] = qs[tt][s * DS + i];
        g[i] = gs[tt][s * DS + i];
      }
      v = vs[tt][c];
      bt = bs[tt];
      kq = kqs[tt];
    };
    auto step = [&](int tt, const float* k, const float* q, const float* g, float v, float bt, float kq) {
      float sk[4] = {0.f, 0.f, 0.f, 0.f}, sq[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        S[i] *= g[i];
        sk[i & 3] = fmaf(S[i], k[i], sk[i & 3]);
        sq[i & 3] = fmaf(S[i], q[i], sq[i & 3]);
      }
      float sk_all = (sk[0] + sk[1]) + (sk[2] + sk[3]), sq_all = (sq[0] + sq[1]) + (sq[2] + sq[3]);
      sum_over_slices(sk_all, sq_all);
      const float u = bt * (v - sk_all);
#pragma unroll
      for (int i = 0; i < DS; ++i) S[i] = fmaf(k[i], u, S[i]);
      if (s == 0 && live) out[((int64_t)(tc + tt) * heads + h) * vdim + col] = fmaf(u, kq, sq_all);
    };
    float ka[DS], qa2[DS], ga[DS], kb[DS], qb[DS], gb[DS], va, ba, vb, bb, da, db;
    load(0, ka, qa2, ga, va, ba, da);
    for (int tt = 0; tt < n; tt += 2) {
      load(min(tt + 1, kCh - 1), kb, qb, gb, vb, bb, db);
      step(tt, ka, qa2, ga, va, ba, da);
      load(min(tt + 2, kCh - 1), ka, qa2, ga, va, ba, da);
      if (tt + 1 < n) step(tt + 1, kb, qb, gb, vb, bb, db);
    }
  }
#pragma unroll
  for (int i = 0; i < DS; ++i)
    if (live && s * DS + i < dim) S_mem[(int64_t)(s * DS + i) * vdim] = S[i];
}

// The recurrence in chunks of 16 tokens, on the matrix cores.  With G_t the product of a chunk's decays up to token t and
// S_0 the state ahead of the chunk,
//     u_t = beta_t (v_t - S_0^T (G_t k_t) - sum_(s<t) A_ts u_s),     A_ts = sum_i k_t[i] k_s[i] (g_(s+1) .. g_t)[i]
//     o_t = S_0^T (G_t q_t) + sum_(s<=t) B_ts u_s,                   B_ts = sum_i q_t[i] k_s[i] (g_(s+1) .. g_t)[i]
//     S   = diag(G_16) S_0 + sum_s (g_(s+1) .. g_16 k_s) u_s^T
// A, B and the solution of the first line for u = U0 - W S_0 (W and U0 by forward substitution, row by row as the recurrence
// goes) do not depend on the state: delta_chunk_kernel makes them for all chunks at once.  What is left for
// delta_chunk_scan_kernel to do in order are three products of 16 x dim (x vdim columns) a chunk.  Products of decays are
// taken of the decays themselves (none exceeds one), never as quotients, so decays near zero lose nothing.  A number
// that is not finite reaches no token ahead of its own: B's zeros never meet it.
// 1,944 tokens of six requests, the longest 801, 16 heads of 128 x 128: convolutions and decays 98 us and the recurrence 311,
// now 52 and 74; one request of 2,047 tokens 103 and 700, now 50 and 102.  What bounds them: the first its convolutions' and
// decays' functions; the second a chain of 0.8 us a chunk, of which the matrix instructions take a half.  Error against 64
// bits (2-norm, 1,000 tokens of 8 heads, mean of 16 draws, in chunks and token by token): of the results with one decay a channel
// 1.40e-7 and 1.45e-7 (64 x 64 1.54e-7 and 1.58e-7), with one a head 1.42e-7 and 1.41e-7 (1.52e-7 and 1.51e-7), of the states
// 1.59e-7 and 1.85e-7 (1.49e-7 and 1.65e-7), 1.54e-7 and 1.70e-7 (1.44e-7 and 1.51e-7).
constexpr int kChunkMaxDim = 128;      // channels and value columns a head may have here: a thread each
constexpr int kChunkThreads = 256;
constexpr int kChunkTaps = 4;

// What a (chunk, head) leaves for the scan, in floats: W, Q, K [dp / 16][64][4], U0 [vp / 16][64][4], B [64][4], G [dp].  A lane's
// four numbers are what it holds of a matrix operand in four instructions of 16 x 16 x 4: of W and Q token l % 16, channels
// 4 (l / 16) + j of sixteen; of K channel l % 16 of sixteen, tokens 4 (l / 16) + j; of U0 column l % 16, of B row l % 16, likewise.
__host__ __device__ __forceinline__ int64_t chunk_floats(int dp, int vp) { return 3 * kCT * dp + kCT * vp + kCT * kCT + dp; }

// One workgroup per (chunk, head).  Thread i < DP convolves q's channel i, i + DP k's; the others than the first DP also a value
// column each.  The decays, the dearest functions here, are shared out so that both are equally busy.
template <typename T, int DP>
__global__ __launch_bounds__(kChunkThreads) void delta_chunk_kernel(
    const T* __restrict__ p, int64_t p_stride, int conv_off, int b_off, const float* __restrict__ a, int64_t a_stride,
    const float* __restrict__ conv_w, const float* __restrict__ a_log, const float* __restrict__ dt_bias,
    const float* __restrict__ state, int64_t state_stride, int64_t saved_off, const int32_t* __restrict__ cu_seqlens,
    const int32_t* __restrict__ state_slots, const int32_t* __restrict__ tile_req, const int32_t* __restrict__ tile_tok0,
    const int32_t* __restrict__ tile_ntok, float* __restrict__ items, int heads, int kv_heads, int dim, int vdim, int taps,
    float q_scale, int a_per_head) {
  constexpr int LD = DP + 4;
  __shared__ __attribute__((aligned(16))) float qs[kCT][LD], ks[kCT][LD], gs[kCT][LD];
  __shared__ __attribute__((aligned(16))) float As[kCT][kCT], Bs[kCT][kCT];      // A[s][t], B[t][s]
  __shared__ __attribute__((aligned(16))) float beta[kCT];
  const int tile = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int n = tile_ntok[tile];
  if (n <= 0) return;                    // a padding tile
  const int req = tile_req[tile], tok0 = tile_tok0[tile], t0 = cu_seqlens[req];
  const int kh = h / (heads / kv_heads), vp = (vdim + 31) / 32 * 32;
  const float* saved = state + (int64_t)state_slots[req] * state_stride + saved_off;
  float* item = items + ((int64_t)(chunk_place(t0, req) + (tok0 - t0) / kCT) * heads + h) * chunk_floats(DP, vp);
  // One channel's convolution and SiLU for the chunk's tokens, zero behind the last of them; inputs ahead of the request's
  // first token of this step come from its state.
  auto conv = [&](int ch, float* y) {
    constexpr int BACK = kChunkTaps - 1;
    const T* col = p + (int64_t)tok0 * p_stride + conv_off + ch;
    T in[kCT + BACK];
    float x[kCT + BACK], wt[kChunkTaps];
#pragma unroll
    for (int j = 0; j < kCT + BACK; ++j) in[j] = col[(int64_t)(j < BACK ? (tok0 > t0 ? j - BACK : 0) : min(j - BACK, n - 1)) * p_stride];
#pragma unroll
    for (int j = 0; j < kChunkTaps; ++j) wt[j] = j >= kChunkTaps - taps ? conv_w[(int64_t)ch * taps + j - (kChunkTaps - taps)] : 0.f;
#pragma unroll
    for (int j = 0; j < kCT + BACK; ++j) x[j] = to_f32(in[j]);
    if (tok0 == t0) {
      const float* sv = saved + (int64_t)ch * (taps - 1);
#pragma unroll
      for (int j = 0; j < BACK; ++j) x[j] = j >= kChunkTaps - taps ? sv[j - (kChunkTaps - taps)] : 0.f;
    }
#pragma unroll
    for (int t = 0; t < kCT; ++t) y[t] = 0.f;
#pragma unroll
    for (int j = 0; j < kChunkTaps; ++j)
      if (j >= kChunkTaps - taps) {       // uniform: an input that no tap meets may be anything
#pragma unroll
        for (int t = 0; t < kCT; ++t) y[t] = fmaf(wt[j], x[t + j], y[t]);
      }
#pragma unroll
    for (int t = 0; t < kCT; ++t) y[t] = t < n ? silu(y[t]) : 0.f;
  };
  float y[kCT];
  const bool channel = tid < DP;
  const int vcol = tid - DP, ch = tid % DP, lane = tid % TL_WAVE;
  if (tid < 2 * DP) {
    // the decays: tokens 0 to 10 for those who convolve once, the others for those who do it twice
    constexpr int SPLIT = 11;
    const float rate = expf(a_log[h]);
    float pre[SPLIT];
    if (!a_per_head) {
#pragma unroll
      for (int i = 0; i < SPLIT; ++i) {
        const int t = channel ? i : min(SPLIT + i, kCT - 1);
        pre[i] = a[(int64_t)(tok0 + min(t, n - 1)) * a_stride + h * dim + min(ch, dim - 1)];
      }
    } else {
      pre[0] = a[(int64_t)(tok0 + min(lane % kCT, n - 1)) * a_stride + h];
    }
    const float bias = dt_bias[a_per_head ? h : h * dim + min(ch, dim - 1)];
#pragma unroll
    for (int t = 0; t < kCT; ++t) y[t] = 0.f;
    if (ch < dim) conv((channel ? 0 : kv_heads * dim) + kh * dim + ch, y);
    float(*const to)[LD] = channel ? qs : ks;
#pragma unroll
    for (int t = 0; t < kCT; ++t) to[t][ch] = y[t];
    if (a_per_head) {                   // a token's decay is worked out by one lane
      const float g = lane < n ? expf(-rate * softplus(pre[0] + bias)) : 1.f;
#pragma unroll
      for (int i = 0; i < SPLIT; ++i) {
        const int t = channel ? i : SPLIT + i;
        const float gt = __uint_as_float(__builtin_amdgcn_ds_bpermute((t % kCT) * 4, __float_as_uint(g)));
        if (t < kCT) gs[t][ch] = ch < dim ? gt : 1.f;
      }
    } else {
#pragma unroll
      for (int i = 0; i < SPLIT; ++i) {
        const int t = channel ? i : SPLIT + i;
        if (i >= kCT - SPLIT && !channel) break;
        gs[t][ch] = t < n && ch < dim ? expf(-rate * softplus(pre[i] + bias)) : 1.f;
      }
    }
  }
  if (!channel) {
#pragma unroll
    for (int t = 0; t < kCT; ++t) y[t] = 0.f;
    if (vcol < vdim) conv(2 * kv_heads * dim + h * vdim + vcol, y);
  }
  if (tid < kCT)
    beta[tid] = tid < n ? 1.f / (1.f + expf(-to_f32(p[(int64_t)(tok0 + tid) * p_stride + b_off + h]))) : 0.f;
  __syncthreads();
  // Unit vectors, sixteen threads a token.
  const int l = tid % 16;
  {
    const int t = tid / 16;
    f32x4 q4[DP / 64], k4[DP / 64];
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int i = 0; i < DP / 64; ++i) {
      q4[i] = *(const f32x4*)&qs[t][i * 64 + l * 4];
      k4[i] = *(const f32x4*)&ks[t][i * 64 + l * 4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sq = fmaf(q4[i][e], q4[i][e], sq);
        sk = fmaf(k4[i][e], k4[i][e], sk);
      }
    }
    sq = group_sum<16>(sq);
    sk = group_sum<16>(sk);
    const float rq = q_scale / sqrtf(sq + 1e-6f), rk = 1.f / sqrtf(sk + 1e-6f);
#pragma unroll
    for (int i = 0; i < DP / 64; ++i) {
      *(f32x4*)&qs[t][i * 64 + l * 4] = q4[i] * rq;
      *(f32x4*)&ks[t][i * 64 + l * 4] = k4[i] * rk;
    }
  }
  __syncthreads();
  // Columns s of A and B, sixteen threads a column: k_s, decayed from token to token, with every later token's k and q.  A
  // wave's four columns begin at its first; which wave has the long ones changes from workgroup to workgroup.
  const int s_first = (tid / TL_WAVE + (int)blockIdx.x) % 4 * 4, s = s_first + tid % TL_WAVE / 16;
  float pa[kCT], pb[kCT];
  {
    f32x4 x[DP / 64];
#pragma unroll
    for (int i = 0; i < DP / 64; ++i) x[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < kCT; ++t) {
      pa[t] = pb[t] = 0.f;
      if (t >= s_first && t < n) {      // uniform
        float ak[4] = {0.f, 0.f, 0.f, 0.f}, bq[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < DP / 64; ++i) {
          const f32x4 g4 = *(const f32x4*)&gs[t][i * 64 + l * 4], k4 = *(const f32x4*)&ks[t][i * 64 + l * 4],
                      q4 = *(const f32x4*)&qs[t][i * 64 + l * 4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[i][e] = t == s ? k4[e] : x[i][e] * g4[e];      // ahead of token s it is zero
            ak[e] = fmaf(x[i][e], k4[e], ak[e]);
            bq[e] = fmaf(x[i][e], q4[e], bq[e]);
          }
        }
        pa[t] = (ak[0] + ak[1]) + (ak[2] + ak[3]);
        pb[t] = (bq[0] + bq[1]) + (bq[2] + bq[3]);
      }
    }
  }
  {
    const float at = scatter_sums(pa, l), bt = scatter_sums(pb, l);      // of token l
    As[s][l] = l > s ? at : 0.f;
    Bs[l][s] = l >= s ? bt : 0.f;
  }
  __syncthreads();
  // W and U0, a column a thread: beta_t times x_t - sum A_ts w_s, summed in 64 bits (2 us of 52; in 32 the error against 64
  // bits is 5 % above that of token by token, not below).
  f32x4 *W = (f32x4*)item, *Q = W + 4 * DP, *K = Q + 4 * DP, *U0 = K + 4 * DP, *Bm = U0 + 4 * vp;
  if (channel) {
    // The products of decays in 64 bits: with one decay a head all channels would share their rounding errors, which token by
    // token they do not.
    double g = 1.0;
#pragma unroll
    for (int t = 0; t < kCT; ++t) {
      g *= (double)gs[t][tid];
      y[t] = ks[t][tid] * (float)g;
      qs[t][tid] *= (float)g;
    }
    ((float*)(Bm + kCT * kCT / 4))[tid] = (float)g;
    g = 1.0;
    f32x4 k4;
#pragma unroll
    for (int t = kCT - 1; t >= 0; --t) {
      k4[t % 4] = ks[t][tid] * (float)g;
      g *= (double)gs[t][tid];
      if (t % 4 == 0) K[tid / 16 * 64 + t / 4 * 16 + tid % 16] = k4;
    }
  }
  double z[kCT];
#pragma unroll
  for (int t = 0; t < kCT; ++t) z[t] = (double)y[t];
#pragma unroll
  for (int s0 = 0; s0 < kCT; ++s0) {
    z[s0] *= (double)beta[s0];
    y[s0] = (float)z[s0];
#pragma unroll
    for (int j = (s0 + 1) / 4; j < kCT / 4; ++j) {
      const f32x4 a4 = *(const f32x4*)&As[s0][j * 4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (j * 4 + e > s0) z[j * 4 + e] = fma(-(double)a4[e], z[s0], z[j * 4 + e]);
    }
  }
  if (channel) {
#pragma unroll
    for (int t = 0; t < kCT; ++t) ks[t][tid] = y[t];
  } else if (vcol < vp) {
#pragma unroll
    for (int i = 0; i < kCT / 4; ++i)
      U0[vcol / 16 * 64 + i * 16 + vcol % 16] = f32x4{y[i * 4], y[i * 4 + 1], y[i * 4 + 2], y[i * 4 + 3]};
  }
  __syncthreads();
  for (int e = tid; e < 4 * DP; e += kChunkThreads) {
    const int row = e % 16, ch = e / 64 * 16 + e % 64 / 16 * 4;
    W[e] = *(const f32x4*)&ks[row][ch];
    Q[e] = *(const f32x4*)&qs[row][ch];
  }
  if (tid < kCT * kCT / 4) {
    const int row = tid % 16, j = tid / 16 * 4;
    Bm[tid] = *(const f32x4*)&Bs[row][j];
  }
}

// A workgroup owns 16 value columns of one (request, head).  Wave rg < 4 keeps rows [rg * 16 NT, (rg + 1) * 16 NT) of S, as
// results of matrix instructions, which are the second operand of the next ones as they are.  A chunk: its rows' part of
// W S_0, left in LDS for the other three; its part of Q S_0, half of it ahead of the barrier and half behind, which hides
// both ways through LDS; then u, of all four parts, and the update.  Wave 4 forms the outputs, a chunk later (by the waves in
// turn they cost a chunk 0.38 of 1.05 us).  One barrier a chunk, which does not wait for the operands on their way: they come
// straight into registers, AHEAD chunks ahead, and no load stands in a branch (the compiler would wait for all at its end).
// Sums run in chains of two instructions, and what a chunk adds to S is summed by itself, so that the results are as close
// to 64 bits as token by token.
constexpr int kScanThreads = 5 * TL_WAVE;
template <int NT, int AHEAD>
__global__ __launch_bounds__(kScanThreads, AHEAD == 1 ? 5 : 3) void delta_chunk_scan_kernel(
    const float* __restrict__ items, float* __restrict__ state, int64_t state_stride, const int32_t* __restrict__ cu_seqlens,
    const int32_t* __restrict__ state_slots, float* __restrict__ out, int heads, int dim, int vdim) {
  constexpr int DP = 64 * NT;
  __shared__ f32x4 us[3][4][TL_WAVE], os[2][4][TL_WAVE];      // parts of chunk c: [c % 3], [c % 2]
  const int r = blockIdx.z, h = blockIdx.x, tid = threadIdx.x, lane = tid % TL_WAVE;
  const int rg = __builtin_amdgcn_readfirstlane(tid / TL_WAVE), q = lane / 16, vt = blockIdx.y, col = vt * 16 + lane % 16;
  const int t0 = cu_seqlens[r], t1 = cu_seqlens[r + 1];
  if (t1 <= t0) return;                           // a padding request owns no state
  const int chunks = (t1 - t0 + kCT - 1) / kCT, vp = (vdim + 31) / 32 * 32;
  const int64_t size = chunk_floats(DP, vp), step = size * heads / 4;
  const bool live = col < vdim;
  const f32x4* item0 = (const f32x4*)(items + ((int64_t)chunk_place(t0, r) * heads + h) * size);
  auto meet = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto u_of = [&](int slot) { return -((us[slot][0][lane] + us[slot][1][lane]) + (us[slot][2][lane] + us[slot][3][lane])); };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  if (rg == 4) {
    const int row_bytes = heads * vdim * 4;
    const f32x4* b_at = item0 + 12 * DP + 4 * vp + lane;
    f32x4 b = b_at[0];
    meet();
    for (int c = 0; c < chunks; ++c) {
      meet();
      const f32x4 u = u_of(c % 3), o = (os[c % 2][0][lane] + os[c % 2][1][lane]) + (os[c % 2][2][lane] + os[c % 2][3][lane]);
      f32x4 U = u, y = zero, y2 = zero;             // transposed: four columns a lane
      const bool hidden = hides_not_finite(U);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        y = __builtin_amdgcn_mfma_f32_16x16x4f32(U[j], b[j], y, 0, 0, 0);
        y2 = __builtin_amdgcn_mfma_f32_16x16x4f32(U[j + 2], b[j + 2], y2, 0, 0, 0);
      }
      y = o + (y + y2);
      if (hidden) add_not_finite(y, u, b, lane);
      b = b_at[step * min(c + 1, chunks - 1)];
      // a buffer that ends with the request's last token of the chunk: what lies behind is not stored, without a branch
      const int n = min(kCT, t1 - t0 - c * kCT);
      const __amdgpu_buffer_rsrc_t rows =
          __builtin_amdgcn_make_buffer_rsrc(out + ((int64_t)(t0 + c * kCT) * heads + h) * vdim, 0, (n - 1) * row_bytes + vdim * 4, 0x00020000);
      const int at = lane % 16 * row_bytes + (vt * 16 + q * 4) * 4;
      if (vdim % 4 == 0) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(tl_u32x4, y), rows, vt * 16 + q * 4 < vdim ? at : -16, 0, 0);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[j]), rows, vt * 16 + q * 4 + j < vdim ? at + j * 4 : -4, 0, 0);
      }
    }
    return;
  }
  float* S_mem = state + (int64_t)state_slots[r] * state_stride + (int64_t)h * dim * vdim;
  f32x4 S[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)                    // clamped, so that all rows are requested together
#pragma unroll
    for (int e = 0; e < 4; ++e) S[i][e] = S_mem[(int64_t)min((rg * NT + i) * 16 + q * 4 + e, dim - 1) * vdim + min(col, vdim - 1)];
  struct Operands {
    f32x4 w[NT], q[NT], k[NT], g[NT], u0;
  };
  Operands op[AHEAD];
  // A chunk's numbers through a buffer of their own: one offset a lane for each kind, no address arithmetic in vector registers.
  const int w_at = (rg * NT * TL_WAVE + lane) * 16, g_at = (12 * DP + 4 * vp + TL_WAVE + rg * NT * 4 + q) * 16,
            u0_at = (12 * DP + vt * TL_WAVE + lane) * 16;
  auto request = [&](Operands& x, int c) {        // (behind the last chunk: that one again)
    const __amdgpu_buffer_rsrc_t from =
        __builtin_amdgcn_make_buffer_rsrc((void*)(item0 + step * min(c, chunks - 1)), 0, (int)size * 4, 0x00020000);
    auto load = [&](int at, int more) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, at, more, 0)); };
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      x.w[i] = load(w_at + i * 1024, 0);
      x.q[i] = load(w_at + i * 1024, 64 * DP);
      x.k[i] = load(w_at + i * 1024, 128 * DP);
      x.g[i] = load(g_at + i * 64, 0);
    }
    x.u0 = load(u0_at, 0);
  };
  request(op[0], 0);
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!live || (rg * NT + i) * 16 + q * 4 + e >= dim) S[i][e] = 0.f;
  };
  const float first_part = rg == 0 ? 1.f : 0.f;
  auto chunk = [&](Operands& x, int c, int slot, auto ask) {
    f32x4 y[NT][2], o[NT][2];
    // instruction j of 16 rows i
    auto part_u = [&](int i, int j) {
      y[i][j % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w[i][j], S[i][j], j < 2 ? zero : y[i][j % 2], 0, 0, 0);
    };
    auto part_o = [&](int i, int j) {             // transposed
      o[i][j % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[i][j], x.q[i][j], j < 2 ? zero : o[i][j % 2], 0, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < NT; ++i) part_u(i, j);
    if constexpr (NT == 2) {
#pragma unroll
      for (int j = 0; j < 4; ++j) part_o(0, j);
    } else {
      part_o(0, 0);
      part_o(0, 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    f32x4 u = y[0][0] + y[0][1];
    if constexpr (NT == 2) u += y[1][0] + y[1][1];
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = fmaf(-first_part, x.u0[e], u[e]);
    us[slot][rg][lane] = u;
    meet();
    const f32x4 p0 = us[slot][0][lane], p1 = us[slot][1][lane], p2 = us[slot][2][lane], p3 = us[slot][3][lane];
    if constexpr (NT == 2) {
#pragma unroll
      for (int j = 0; j < 4; ++j) part_o(1, j);
    } else {
      part_o(0, 2);
      part_o(0, 3);
    }
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 U = -((p0 + p1) + (p2 + p3));
    f32x4 add[NT], add2[NT];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        add[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[i][j], U[j], j == 0 ? zero : add[i], 0, 0, 0);
        add2[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[i][j + 2], U[j + 2], j == 0 ? zero : add2[i], 0, 0, 0);
      }
    f32x4 os_ = o[0][0] + o[0][1];
    if constexpr (NT == 2) os_ += o[1][0] + o[1][1];
    os[c % 2][rg][lane] = os_;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[i][e] = fmaf(x.g[i][e], S[i][e], add[i][e] + add2[i][e]);
    if constexpr (decltype(ask)::value) request(x, c + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
  };
  if (chunks == 1) {                              // a step's single tokens: nothing is asked for ahead
    clear();
    chunk(op[0], 0, 0, std::false_type{});
  } else {
#pragma unroll
    for (int d = 1; d < AHEAD; ++d) request(op[d], d);
    clear();
    int c = 0, slot = 0;
    auto next = [&]() { return slot = slot == 2 ? 0 : slot + 1; };
    for (; c + AHEAD <= chunks; c += AHEAD) {
#pragma unroll
      for (int d = 0; d < AHEAD; ++d) {
        chunk(op[d], c + d, slot, std::true_type{});
        next();
      }
    }
#pragma unroll
    for (int d = 0; d < AHEAD - 1; ++d)
      if (c + d < chunks) {                       // (the whole workgroup)
        chunk(op[d], c + d, slot, std::true_type{});
        next();
      }
  }
  meet();
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = (rg * NT + i) * 16 + q * 4 + e;
      if (live && row < dim) S_mem[(int64_t)row * vdim + col] = S[i][e];
    }
}

// z[t, h, :] = scale * w * o[t, h, :] / sqrt(mean(o[t, h, :]^2) + eps) * act(gate[t, h, :]); one wave per (t, h).
// w is shared by the heads (w_head_stride 0) or each head's own (w_head_stride = vdim); act is the sigmoid
// (gate_kind 0) or g * sigmoid(g) (gate_kind 1).
template <typename T>
__global__ __launch_bounds__(TL_WAVE) void head_norm_gate_kernel(const float* __restrict__ o,
                                                                 const float* __restrict__ w, int w_head_stride,
                                                                 const float* __restrict__ gate, int64_t gate_stride,
                                                                 T* __restrict__ z, int heads, int vdim, float eps,
                                                                 int gate_kind, float scale) {
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const float* src = o + ((int64_t)t * heads + h) * vdim;
  const float* wh = w + (int64_t)h * w_head_stride;
  float ss = 0.f;
  for (int j = lane; j < vdim; j += TL_WAVE) ss += src[j] * src[j];
  ss = wave_sum(ss);
  const float r = scale / sqrtf(ss / (float)vdim + eps);
  const float* gp = gate + (int64_t)t * gate_stride + (int64_t)h * vdim;
  T* dst = z + ((int64_t)t * heads + h) * vdim;
  for (int j = lane; j < vdim; j += TL_WAVE) {
    const float g = gp[j], sg = 1.f / (1.f + expf(-g));
    dst[j] = from_f32<T>(src[j] * r * wh[j] * (gate_kind ? g * sg : sg));
  }
}

// A decode step in one kernel: every request brings ONE token.  One workgroup per (request, head),
// a thread per value column: the convolutions, unit vectors, decay and beta of the token, the
// recurrence on the column in registers, and the head's norm and gate on the way out
// (z[t, h, :] = w * o / rms(o) * act(gate), act the sigmoid or, with gate_kind 1, g * sigmoid(g)).  The saved convolution inputs are brought up to date
// here when every head has q/k channels of its own (update_saved); else several workgroups read a
// channel's saved inputs and conv_state_update_kernel runs behind this kernel.
constexpr int kDecodeCols = 256;        // value columns the one-kernel decode step takes
constexpr int kDecodeThreads = 512;
// The inputs and weights of one channel's convolution for the token at row t (n = 0 in its step),
// oldest first; taps <= 4.
template <typename T>
__device__ __forceinline__ void load_taps(const T* __restrict__ p, int64_t p_stride, int t, int col,
                                          const float* __restrict__ saved, const float* __restrict__ w, int taps,
                                          float* x, float* wt) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    x[j] = j < taps ? conv_input(p, p_stride, t, j - (taps - 1), col, saved, taps) : 0.f;
    wt[j] = j < taps ? w[j] : 0.f;
  }
}
__device__ __forceinline__ float conv_of(const float* x, const float* wt) {
  float acc = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = fmaf(wt[j], x[j], acc);
  return silu(acc);
}
// after the token the saved inputs are the last taps - 1 of x
__device__ __forceinline__ void store_saved(float* __restrict__ saved, const float* x, int taps) {
#pragma unroll
  for (int j = 1; j < 4; ++j)
    if (j < taps) saved[j - 1] = x[j];
}

// State phase of the kernel: thread (sl, cq) keeps rows [sl * DS, (sl + 1) * DS) of the FOUR value columns
// 4 cq .. 4 cq + 3 of S in registers (16-byte loads and stores: a lane that moves four bytes at a time gets a
// fraction of what a compute unit can fetch), the slices' partial sums meet in LDS in a fixed order.  There are few
// (request, head) pairs as a rule, so a workgroup is as wide as it may be: 16 slices where four kept two waves busy for 32
// rows each, and a thread per channel of q, k and v: 16.9 -> 9.9 us for 6 requests of 16 heads of 128 x 128
// (tl_delta_decode says where it is narrower).
template <typename T, typename TZ, int DS>
__global__ __launch_bounds__(kDecodeThreads) void delta_decode_kernel(
    const T* __restrict__ p, int64_t p_stride, int conv_off, int b_off, const float* __restrict__ a, int64_t a_stride,
    int a_per_head, const float* __restrict__ gate, int64_t gate_stride, int gate_kind,
    const float* __restrict__ conv_w, const float* __restrict__ a_log, const float* __restrict__ dt_bias,
    const float* __restrict__ w_norm, float* __restrict__ state, int64_t state_stride, int64_t saved_off,
    const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ state_slots, TZ* __restrict__ z, int heads,
    int kv_heads, int dim, int vdim, int taps, float q_scale, float eps, int update_saved, int slices) {
  __shared__ float qkv[2 * kMaxDim + kDecodeCols], gs[kMaxDim], red[2][kDecodeThreads / TL_WAVE];
  __shared__ f32x4 part[2][16 * 32];                // [slice][column quad], for either round of sums
  const int r = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wave = tid / TL_WAVE, lane = tid % TL_WAVE;
  const int nw = blockDim.x / TL_WAVE;
  const int t = cu_seqlens[r];
  if (cu_seqlens[r + 1] - t != 1) return;         // a padding request owns no state
  const int kh = h / (heads / kv_heads);
  float* row = state + (int64_t)state_slots[r] * state_stride;
  float* saved = row + saved_off;
  const int quads = vdim / 4;
  const int cq = tid % quads, sl = tid / quads;     // state phase: column quad and slice of the key channels
  const bool owner = sl < slices;
  const int items = 2 * dim + vdim;                 // the head's channels: q, k and v
  // Everything the token needs is requested here, before the first value is used.
  float x[2][4], wt[2][4];
  float* sv[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {                     // at most two channels a thread
    const int e = min(tid + i * (int)blockDim.x, items - 1);
    const int ch = e < dim ? kh * dim + e : e < 2 * dim ? kv_heads * dim + kh * dim + e - dim : 2 * kv_heads * dim + h * vdim + e - 2 * dim;
    sv[i] = saved + (int64_t)ch * (taps - 1);
    if (i == 0 || (int)blockDim.x < items)
      load_taps(p, p_stride, t, conv_off + ch, sv[i], conv_w + (int64_t)ch * taps, taps, x[i], wt[i]);
  }
  const int i0 = min(tid, dim - 1);
  const int ai = a_per_head ? h : h * dim + i0;
  const float pre_a = a[(int64_t)t * a_stride + ai] + dt_bias[ai];
  const float pre_b = to_f32(p[(int64_t)t * p_stride + b_off + h]);
  const float rate = expf(a_log[h]);
  float pre_g[4] = {0.f, 0.f, 0.f, 0.f}, wn[4] = {0.f, 0.f, 0.f, 0.f};
  if (sl == 0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      pre_g[e] = gate[(int64_t)t * gate_stride + h * vdim + cq * 4 + e];
      wn[e] = w_norm[cq * 4 + e];
    }
  }
  float* S_mem = row + (int64_t)h * dim * vdim + cq * 4;
  f32x4 S[DS];
#pragma unroll
  for (int j = 0; j < DS; ++j) {
    const int i = sl * DS + j;
    S[j] = (owner && i < dim) ? *(const f32x4*)(S_mem + (int64_t)i * vdim) : f32x4{0.f, 0.f, 0.f, 0.f};
  }

  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int e = tid + i * (int)blockDim.x;
    if (e >= items) break;
    const float v = conv_of(x[i], wt[i]);
    qkv[e] = v;
    if (e < dim) sq += v * v;
    else if (e < 2 * dim) sk += v * v;
    if (update_saved) store_saved(sv[i], x[i], taps);   // no other head reads these channels: their only reader
  }
  if (tid < dim) gs[tid] = expf(-rate * softplus(pre_a));
  sq = wave_sum(sq);
  sk = wave_sum(sk);
  if (lane == 0) {
    red[0][wave] = sq;
    red[1][wave] = sk;
  }
  __syncthreads();
  sq = sk = 0.f;
  for (int i = 0; i < nw; ++i) {
    sq += red[0][i];
    sk += red[1][i];
  }
  const float rq = q_scale / sqrtf(sq + 1e-6f), rk = 1.f / sqrtf(sk + 1e-6f);
  const float beta = 1.f / (1.f + expf(-pre_b));
  const float *qs = qkv, *ks = qkv + dim, *vs = qkv + 2 * dim;
  auto total = [&](const f32x4* from) {
    f32x4 s = from[cq];
    for (int i = 1; i < slices; ++i) s += from[i * quads + cq];
    return s;
  };
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (owner) {
#pragma unroll
    for (int j = 0; j < DS; ++j) {
      const int i = sl * DS + j;
      if (i < dim) {
        const float g = gs[i], k = ks[i] * rk;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          S[j][e] *= g;
          acc[e] = fmaf(S[j][e], k, acc[e]);
        }
      }
    }
    part[0][sl * quads + cq] = acc;
  }
  __syncthreads();
  if (owner) {
    const f32x4 sum = total(part[0]);
    f32x4 u, o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = beta * (vs[cq * 4 + e] - sum[e]);
#pragma unroll
    for (int j = 0; j < DS; ++j) {
      const int i = sl * DS + j;
      if (i < dim) {
        const float k = ks[i] * rk, q = qs[i] * rq;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          S[j][e] = fmaf(k, u[e], S[j][e]);
          o[e] = fmaf(S[j][e], q, o[e]);
        }
        *(f32x4*)(S_mem + (int64_t)i * vdim) = S[j];
      }
    }
    part[1][sl * quads + cq] = o;
  }
  __syncthreads();
  if (wave > 0) return;                 // the head's columns are at most 64 quads: one wave's
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  if (lane < quads) o = total(part[1]);
  const float ss = wave_sum((o[0] * o[0] + o[1] * o[1]) + (o[2] * o[2] + o[3] * o[3]));
  if (lane < quads) {
    const float rn = 1.f / sqrtf(ss / (float)vdim + eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float sg = 1.f / (1.f + expf(-pre_g[e]));
      z[((int64_t)t * heads + h) * vdim + cq * 4 + e] = from_f32<TZ>(o[e] * rn * wn[e] * (gate_kind ? pre_g[e] * sg : sg));
    }
  }
}

}  // namespace

#define TL_DISPATCH_T(dtype, ...)                 \
  if ((dtype) == 0) { using T = float; __VA_ARGS__ } \
  else if ((dtype) == 1) { using T = bf16_t; __VA_ARGS__ } \
  else return TL_ERR_ARG;

extern "C" {

int tl_delta_prepare(const void* p, int64_t p_stride, int conv_off, int b_off, const float* a, int64_t a_stride,
                     const float* conv_w, const float* a_log, const float* dt_bias, const float* state,
                     int64_t state_stride, int64_t saved_off, const int32_t* req_of_token, const int32_t* cu_seqlens,
                     const int32_t* state_slots, float* qn, float* kn, float* vc, float* beta, float* decay,
                     int n_tokens, int heads, int kv_heads, int dim, int vdim, int taps, float q_scale, int a_per_head,
                     int dtype, hipStream_t stream) {
  if (n_tokens <= 0) return TL_OK;
  if (heads <= 0 || heads > 65535 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || dim > kMaxDim || vdim <= 0 ||
      taps < 1 || taps > kMaxTaps)
    return TL_ERR_ARG;
  dim3 g(n_tokens, heads), b(kPrepThreads);
  TL_DISPATCH_T(dtype, hipLaunchKernelGGL(delta_prepare_kernel<T>, g, b, 0, stream, (const T*)p, p_stride, conv_off,
                                          b_off, a, a_stride, conv_w, a_log, dt_bias, state, state_stride, saved_off,
                                          req_of_token, cu_seqlens, state_slots, qn, kn, vc, beta, decay, heads,
                                          kv_heads, dim, vdim, taps, q_scale, a_per_head);)
  return tl_launch_status();
}

int tl_conv_state_update(const void* p, int64_t p_stride, int conv_off, int channels, const float* bias, float* state,
                         int64_t state_stride, int64_t saved_off, const int32_t* cu_seqlens,
                         const int32_t* state_slots, int n_requests, int taps, int dtype, hipStream_t stream) {
  if (n_requests <= 0 || taps <= 1) return TL_OK;
  if (channels <= 0 || taps > kMaxTaps || n_requests > 65535) return TL_ERR_ARG;
  dim3 g((channels + 255) / 256, n_requests), b(256);
  TL_DISPATCH_T(dtype, hipLaunchKernelGGL(conv_state_update_kernel<T>, g, b, 0, stream, (const T*)p, p_stride,
                                          conv_off, channels, bias, state, state_stride, saved_off, cu_seqlens, state_slots,
                                          taps);)
  return tl_launch_status();
}

int tl_delta_recurrence(const float* qn, const float* kn, const float* vc, const float* beta, const float* decay,
                        float* state, int64_t state_stride, const int32_t* cu_seqlens, const int32_t* state_slots,
                        float* out, int n_requests, int heads, int dim, int vdim, hipStream_t stream) {
  if (n_requests <= 0) return TL_OK;
  if (heads <= 0 || heads > 65535 || dim <= 0 || dim > kMaxDim || vdim <= 0 || (vdim + kRecCols - 1) / kRecCols > 65535)
    return TL_ERR_ARG;
  dim3 g(n_requests, heads, (vdim + kRecCols - 1) / kRecCols), b(kRecThreads);
  const bool vec = dim % 4 == 0 && !(((uintptr_t)qn | (uintptr_t)kn | (uintptr_t)decay) & 15);
#define TL_REC(DS, VEC)                                                                                           \
  hipLaunchKernelGGL((delta_recurrence_kernel<DS, VEC>), g, b, 0, stream, qn, kn, vc, beta, decay, state, state_stride, \
                     cu_seqlens, state_slots, out, heads, dim, vdim)
  // Up to 32 channels a thread stages two elements at most; vectors leave half the threads without a piece and cost 13
  // registers, two waves a SIMD
  if (dim <= 16) TL_REC(2, false);
  else if (dim <= 32) TL_REC(4, false);
  else if (dim <= 64 && vec) TL_REC(8, true);
  else if (dim <= 64) TL_REC(8, false);
  else if (dim <= 128 && vec) TL_REC(16, true);
  else if (dim <= 128) TL_REC(16, false);
  else if (vec) TL_REC(32, true);
  else TL_REC(32, false);
#undef TL_REC
  return tl_launch_status();
}

// The whole of a step's recurrence in chunks: convolutions, unit vectors, decays, the recurrence over states in place.
// tile_*: every request's tokens cut into chunks of at most 16, request after request (ntok 0: padding).  items: float32
// [(n_tokens / 16 + n_requests + 1) * heads * tl_delta_chunk_floats(dim, vdim)].
int64_t tl_delta_chunk_floats(int dim, int vdim) { return chunk_floats(dim <= 64 ? 64 : 128, (vdim + 31) / 32 * 32); }

int tl_delta_chunks(const void* p, int64_t p_stride, int conv_off, int b_off, const float* a, int64_t a_stride,
                    const float* conv_w, const float* a_log, const float* dt_bias, float* state, int64_t state_stride,
                    int64_t saved_off, const int32_t* cu_seqlens, const int32_t* state_slots, const int32_t* tile_req,
                    const int32_t* tile_tok0, const int32_t* tile_ntok, float* items, float* out, int n_tiles, int n_requests,
                    int heads, int kv_heads, int dim, int vdim, int taps, float q_scale, int a_per_head, int dtype,
                    hipStream_t stream) {
  if (n_tiles <= 0 || n_requests <= 0) return TL_OK;
  if (heads <= 0 || heads > 65535 || n_requests > 65535 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || dim > kChunkMaxDim || vdim <= 0 ||
      vdim > kChunkMaxDim || taps < 1 || taps > kChunkTaps || ((uintptr_t)items & 15))
    return TL_ERR_ARG;
  dim3 g(n_tiles, heads), b(kChunkThreads), gs(heads, (vdim + 15) / 16, n_requests), bs(kScanThreads);
  // Heads first in the grid: the workgroups of the longest request are then spread over all XCDs (with requests first, eight
  // of them, it had one), those of a head share one.
  // Where every workgroup has a unit to itself only its own chain counts: operands two chunks ahead (one prompt of 2,047
  // tokens, 16 heads of 128 x 128: 101 us, 138 one chunk ahead).  Beyond, registers for a second set cost waves (six
  // prompts of 67 to 801: 108 us, 80 one ahead; 64 of 13: 83 and 59).
  const bool few = (int64_t)n_requests * heads * ((vdim + 15) / 16) <= 256;
#define TL_DELTA_CHUNK(DP)                                                                                               \
  {                                                                                                                      \
    TL_DISPATCH_T(dtype, hipLaunchKernelGGL((delta_chunk_kernel<T, DP>), g, b, 0, stream, (const T*)p, p_stride, conv_off, \
                                            b_off, a, a_stride, conv_w, a_log, dt_bias, state, state_stride, saved_off,  \
                                            cu_seqlens, state_slots, tile_req, tile_tok0, tile_ntok, items, heads,       \
                                            kv_heads, dim, vdim, taps, q_scale, a_per_head);)                            \
    if (few)                                                                                                             \
      hipLaunchKernelGGL((delta_chunk_scan_kernel<DP / 64, 2>), gs, bs, 0, stream, items, state, state_stride, cu_seqlens, \
                         state_slots, out, heads, dim, vdim);                                                            \
    else                                                                                                                 \
      hipLaunchKernelGGL((delta_chunk_scan_kernel<DP / 64, 1>), gs, bs, 0, stream, items, state, state_stride, cu_seqlens, \
                         state_slots, out, heads, dim, vdim);                                                            \
  }
  if (dim <= 64) TL_DELTA_CHUNK(64)
  else TL_DELTA_CHUNK(128)
#undef TL_DELTA_CHUNK
  return tl_launch_status();
}

// Row t of `a`: the decay's pre-activations (heads x dim, or heads with a_per_head); of `gate`: the gate's (heads x
// vdim); both float32.
int tl_delta_decode(const void* p, int64_t p_stride, int conv_off, int b_off, const float* a, int64_t a_stride,
                    int a_per_head, const float* gate, int64_t gate_stride, int gate_kind, const float* conv_w, const float* a_log, const float* dt_bias, const float* w_norm, float* state,
                    int64_t state_stride, int64_t saved_off, const int32_t* cu_seqlens, const int32_t* state_slots,
                    void* z, int n_requests, int heads, int kv_heads, int dim, int vdim, int taps, float q_scale,
                    float eps, int update_saved, int dtype, int z_dtype, hipStream_t stream) {
  if (n_requests <= 0) return TL_OK;
  if (heads <= 0 || heads > 65535 || kv_heads <= 0 || heads % kv_heads || dim <= 0 || dim > kMaxDim || vdim <= 0 ||
      vdim > kDecodeCols || vdim % 4 || state_stride % 4 || taps < 1 || taps > 4 ||
      (update_saved && heads != kv_heads) || gate_kind < 0 || gate_kind > 1 || !a || !gate)
    return TL_ERR_ARG;
  // A thread per column quad and slice.  16 slices of the key channels (8 beyond 128 columns); fewer where a slice would
  // have less than four of them (4 heads of 32 x 32: 6.8 us by 16, 6.5 by 8; of 8 x 8: 6.8 by 16, 6.1 by 4).  With 1,024
  // (request, head) pairs, four a unit, waves beyond the state's own are in the way: 8 slices, and two of the head's
  // channels a thread (64 requests of 16 heads of 128 x 64: 23.9 us by 16 slices and a channel a thread, 17.8 so; 128 x
  // 128: 28.8 and 24.8; 32 heads of 64 x 128, 32 and 64 requests: 0.76 and 0.84 of the time).
  const int quads = vdim / 4;
  const bool many = (int64_t)n_requests * heads >= 1024;
  int slices = dim <= 16 ? 4 : dim <= 32 || many ? 8 : 16;
  if (quads > 32 && slices > 8) slices = 8;
  const int items = 2 * dim + vdim;         // the head's channels: at most two a thread, and a thread a key channel
  int threads = quads * slices;
  const int least = many ? (dim > (items + 1) / 2 ? dim : (items + 1) / 2) : items;
  if (threads < least) threads = least;
  threads = threads > kDecodeThreads ? kDecodeThreads : (threads + TL_WAVE - 1) / TL_WAVE * TL_WAVE;
  const int ds = (dim + slices - 1) / slices;
  dim3 g(n_requests, heads), b(threads);
#define TL_DEC(TT, TZ, D)                                                                                          \
  hipLaunchKernelGGL((delta_decode_kernel<TT, TZ, D>), g, b, 0, stream, (const TT*)p, p_stride, conv_off, b_off, a, \
                     a_stride, a_per_head, gate, gate_stride, gate_kind, conv_w, a_log, dt_bias, w_norm, state,     \
                     state_stride, saved_off, cu_seqlens, state_slots, (TZ*)z, heads, kv_heads, dim, vdim, taps,    \
                     q_scale, eps, update_saved, slices)
#define TL_DEC_D(TT, TZ)             \
  if (ds <= 4) TL_DEC(TT, TZ, 4);    \
  else if (ds <= 8) TL_DEC(TT, TZ, 8); \
  else if (ds <= 16) TL_DEC(TT, TZ, 16); \
  else TL_DEC(TT, TZ, 32);
  // the projections' element type and the result's: float32 projections may feed a bfloat16 output product
  if (dtype == 0 && z_dtype == 0) { TL_DEC_D(float, float) }
  else if (dtype == 0 && z_dtype == 1) { TL_DEC_D(float, bf16_t) }
  else if (dtype == 1 && z_dtype == 1) { TL_DEC_D(bf16_t, bf16_t) }
  else return TL_ERR_ARG;
#undef TL_DEC_D
#undef TL_DEC
  return tl_launch_status();
}

int tl_head_norm_gate(const float* o, const float* w, int w_head_stride, const float* gate, int64_t gate_stride, void* z,
                      int n_tokens, int heads, int vdim, float eps, int gate_kind, float scale, int dtype,
                      hipStream_t stream) {
  if (n_tokens <= 0) return TL_OK;
  if (heads <= 0 || heads > 65535 || vdim <= 0 || (w_head_stride != 0 && w_head_stride != vdim) || gate_kind < 0 ||
      gate_kind > 1)
    return TL_ERR_ARG;
  dim3 g(n_tokens, heads), b(TL_WAVE);
  TL_DISPATCH_T(dtype, hipLaunchKernelGGL(head_norm_gate_kernel<T>, g, b, 0, stream, o, w, w_head_stride, gate,
                                          gate_stride, (T*)z, heads, vdim, eps, gate_kind, scale);)
  return tl_launch_status();
}

}  // extern "C"
