// Time mixing with a decaying matrix state per head (a linear recurrence whose decay is a vector per
// token, one factor per head and key channel, and whose current token gets a bonus):
//     o_t = (S + diag(u) k_t v_t^T)^T r_t,      S <- diag(w_t) S + k_t v_t^T,      w_t = exp(-exp(x_t + w0))
// and the token shift in front of its projections: each projection reads h_t + (h_(t-1) - h_t) * mu.
//
// Per request the state row holds S of every head and the last token's h, all float32.  Everything
// that enters the recurrence is float32 in both precisions (r, k, v and x are products' float32 results).
#include "common.h"

#include <type_traits>

namespace {

constexpr int kThreads = 256;

// out[m, t, c] = h[t, c] + (prev - h[t, c]) * mu[m, c]; prev is h[t - 1, c], or for the first token a request
// brings in this step what the state row keeps at prev_off (zero for a request's very first token).
template <typename T>
__global__ __launch_bounds__(kThreads) void shift_mix_kernel(const T* __restrict__ h, int64_t h_stride,
                                                             const float* __restrict__ state, int64_t state_stride,
                                                             int64_t prev_off, const int32_t* __restrict__ req_of_token,
                                                             const int32_t* __restrict__ cu,
                                                             const int32_t* __restrict__ slots,
                                                             const float* __restrict__ mu, T* __restrict__ out,
                                                             int64_t plane, int n_mix, int width, int save_single) {
  const int t = blockIdx.x;
  const int c = blockIdx.y * kThreads + threadIdx.x;
  if (c >= width) return;
  const int r = req_of_token[t];
  const float cur = to_f32(h[(int64_t)t * h_stride + c]);
  float prev;
  if (t == cu[r]) {
    float* saved = const_cast<float*>(state) + (int64_t)slots[r] * state_stride + prev_off + c;
    prev = *saved;
    // a request's only token of the step is also its last: this thread has read what the state kept and leaves
    // the token's h in its place (steps of single tokens then need no kernel of their own for that)
    if (save_single && cu[r + 1] == t + 1) *saved = cur;
  } else {
    prev = to_f32(h[(int64_t)(t - 1) * h_stride + c]);
  }
  const float d = prev - cur;
  for (int m = 0; m < n_mix; ++m)
    out[(int64_t)m * plane + (int64_t)t * width + c] = from_f32<T>(fmaf(d, mu[(int64_t)m * width + c], cur));
}

// The last token a request brings becomes the state's saved h.  A request without tokens keeps its state.
template <typename T>
__global__ __launch_bounds__(kThreads) void shift_save_kernel(const T* __restrict__ h, int64_t h_stride,
                                                              float* __restrict__ state, int64_t state_stride,
                                                              int64_t prev_off, const int32_t* __restrict__ cu,
                                                              const int32_t* __restrict__ slots, int width) {
  const int r = blockIdx.x;
  const int c = blockIdx.y * kThreads + threadIdx.x;
  const int t0 = cu[r], t1 = cu[r + 1];
  if (c >= width || t1 <= t0) return;
  state[(int64_t)slots[r] * state_stride + prev_off + c] = to_f32(h[(int64_t)(t1 - 1) * h_stride + c]);
}

// The recurrence.  A workgroup owns EC value columns of one (request, head) and walks the request's
// tokens of this step in order.  The key channels are cut into P slices of 4 (P a power of two, 4 P >= dim);
// thread (e, p) keeps S[4 p .. 4 p + 3, e] in registers, and the P lanes of a column are neighbours, so the sum
// over the channels ends with log2 P lane exchanges (moves inside a row of 16 lanes, then lane swaps).  The
// order of additions is the same whatever the step holds.  Per token a thread's chain is one multiply-add a
// state element; a head's columns are shared out over V / EC workgroups, so that one long prompt still fills
// many compute units.  r, k and the decays of 16 tokens at a time are staged in LDS, the next 16 requested
// before these are worked on.  In memory S lies as [head][s][e][p] (s the index within a slice): a wave's
// accesses to the state are contiguous.
constexpr int kSlice = 4;
constexpr int kChunk = 16;

template <int P>
__device__ __forceinline__ float sum_over_slices(float v) {
  if constexpr (P >= 2) v += dpp_f32<TL_DPP_XOR1>(v);
  if constexpr (P >= 4) v += dpp_f32<TL_DPP_XOR2>(v);
  if constexpr (P >= 8) v += dpp_f32<TL_DPP_HALF_MIRROR>(v);      // the quads of a half row hold one value each by now
  if constexpr (P >= 16) v += dpp_f32<TL_DPP_MIRROR>(v);
  if constexpr (P >= 32) {
    float a, b;
    pair16(v, a, b);
    v = a + b;
  }
  if constexpr (P >= 64) {
    float a, b;
    pair32(v, a, b);
    v = a + b;
  }
  return v;
}

template <int P>
__global__ __launch_bounds__(kThreads) void time_mix_recurrence_kernel(
    const float* __restrict__ x, int64_t x_stride, int r_off, int k_off, int v_off, int w_off,
    const float* __restrict__ w0, const float* __restrict__ u, float* __restrict__ state, int64_t state_stride,
    const int32_t* __restrict__ cu, const int32_t* __restrict__ slots, float* __restrict__ o, int heads, int dim, int vdim) {
  constexpr int EC = kThreads / P, Dp = kSlice * P;
  constexpr int NST = (kChunk * Dp + kThreads - 1) / kThreads, NV = (kChunk * EC + kThreads - 1) / kThreads;
  __shared__ __align__(16) float r_s[kChunk * Dp];
  __shared__ __align__(16) float k_s[kChunk * Dp];
  __shared__ __align__(16) float w_s[kChunk * Dp];
  __shared__ float v_s[kChunk * EC];
  const int req = blockIdx.z, head = blockIdx.y;
  const int t0 = cu[req], n = cu[req + 1] - t0;
  if (n <= 0) return;                     // a request without tokens touches no state
  const int tid = threadIdx.x, p = tid % P, el = tid / P;
  const int e = blockIdx.x * EC + el;
  const bool col = e < vdim;
  float* Sg = state + (int64_t)slots[req] * state_stride + (((int64_t)head * kSlice) * vdim + (col ? e : 0)) * P + p;
  const int64_t s_step = (int64_t)vdim * P;
  float S[kSlice], uu[kSlice];
#pragma unroll
  for (int s = 0; s < kSlice; ++s) {
    S[s] = col ? Sg[s * s_step] : 0.f;
    const int d = p * kSlice + s;
    uu[s] = d < dim ? u[head * dim + d] : 0.f;
  }
  // what this thread stages of a chunk: element i = tid + j * kThreads of [token][channel], token i / Dp
  float pr[NST], pk[NST], pw[NST], pv[NV];
  auto fetch = [&](int c0) {
    const int m = min(kChunk, n - c0);
#pragma unroll
    for (int j = 0; j < NST; ++j) {
      const int i = tid + j * kThreads, tt = i / Dp, d = i % Dp;
      pr[j] = pk[j] = 0.f;
      pw[j] = -INFINITY;                   // a channel beyond the head's: decay exp(-exp(-inf)) = 1, nothing added
      if (i < kChunk * Dp && tt < m && d < dim) {
        const float* row = x + (int64_t)(t0 + c0 + tt) * x_stride + head * dim + d;
        pr[j] = row[r_off];
        pk[j] = row[k_off];
        pw[j] = row[w_off] + w0[head * dim + d];
      }
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = tid + j * kThreads, tt = i / EC, ee = blockIdx.x * EC + i % EC;
      pv[j] = (i < kChunk * EC && tt < m && ee < vdim) ? x[(int64_t)(t0 + c0 + tt) * x_stride + v_off + head * vdim + ee] : 0.f;
    }
  };
  fetch(0);
  for (int c0 = 0; c0 < n; c0 += kChunk) {
    const int m = min(kChunk, n - c0);
    __syncthreads();                       // the chunk before is done with
#pragma unroll
    for (int j = 0; j < NST; ++j) {
      const int i = tid + j * kThreads;
      if (i < kChunk * Dp) {
        r_s[i] = pr[j];
        k_s[i] = pk[j];
        w_s[i] = expf(-expf(pw[j]));
      }
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = tid + j * kThreads;
      if (i < kChunk * EC) v_s[i] = pv[j];
    }
    __syncthreads();
    if (c0 + kChunk < n) fetch(c0 + kChunk);      // on its way while this chunk is worked on
    float* orow = o + (int64_t)(t0 + c0) * ((int64_t)heads * vdim) + head * vdim + e;
    auto token = [&](int tt) {
      const float vv = v_s[tt * EC + el];
      const f32x4 r4 = *(const f32x4*)(r_s + tt * Dp + p * kSlice), k4 = *(const f32x4*)(k_s + tt * Dp + p * kSlice),
                  w4 = *(const f32x4*)(w_s + tt * Dp + p * kSlice);
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < kSlice; ++j) {
        const float kv = k4[j] * vv;
        acc = fmaf(r4[j], fmaf(uu[j], kv, S[j]), acc);
        S[j] = fmaf(w4[j], S[j], kv);
      }
      acc = sum_over_slices<P>(acc);
      if (p == 0 && col) orow[(int64_t)tt * heads * vdim] = acc;
    };
    if (m == kChunk) {
#pragma unroll
      for (int tt = 0; tt < kChunk; ++tt) token(tt);
    } else {
      for (int tt = 0; tt < m; ++tt) token(tt);
    }
  }
  if (col) {
#pragma unroll
    for (int s = 0; s < kSlice; ++s) Sg[s * s_step] = S[s];
  }
}

// The recurrence in chunks of 16 tokens, on the matrix cores.  With P_t the product of a chunk's decays up to token t and S_0 the
// state ahead of the chunk,
//     o_t = S_0^T (P_(t-1) r_t) + sum_(s<=t) B_ts v_s,    B_ts = sum_i r_t[i] k_s[i] (w_(s+1) .. w_(t-1))[i],  B_tt = r_t . (u k_t)
//     S   = diag(P_16) S_0 + sum_s (w_(s+1) .. w_16 k_s) v_s^T
// B and the decayed r and k (Q and K) do not depend on the state: time_mix_chunk_kernel makes them for all chunks at once, and
// time_mix_scan_kernel walks a request's chunks.  Products of decays are taken of the decays themselves, never as quotients,
// along a chunk in 64 bits, and so are B's sums; all else is float32.  A number that is not finite reaches no token ahead of its
// own: B's zeros never meet it.
// 1,944 tokens of six requests, the longest 801, 32 heads of 64 x 64: 187 us token by token, now 36 and 29; one request of 2,047
// tokens 458, now 36 and 54; heads of 128 x 128, half as many, 280, now 38 and 51.  The first kernel is bound by its vector
// instructions, the second by a chain of 0.4 us a chunk.  Error against 64 bits (2-norm, 700 to 1,000 tokens): 9.1e-8, token
// by token 9.5e-8; 128 x 128 9.2e-8 and 1.01e-7 (with B in float32 1.02e-7 and 1.05e-7, 8 us less).
constexpr int kMaxChunkDim = 128;      // channels and value columns a head may have here

// What a (chunk, head) leaves, in floats: Q, K [dp / 16][64][4], V [vp / 16][64][4], B [64][4], P_16 [dp].  A lane's four numbers are
// what it holds of a matrix operand in four instructions of 16 x 16 x 4: of Q token l % 16, channels 4 (l / 16) + j of sixteen;
// of K channel l % 16, tokens 4 (l / 16) + j; of V column l % 16, of B row l % 16, likewise.
__host__ __device__ __forceinline__ int64_t mix_chunk_floats(int dp, int vp) { return 2 * kCT * dp + kCT * vp + kCT * kCT + dp; }

// One workgroup per (chunk, head): a thread a channel and a share of the tokens.
template <int DP>
__global__ __launch_bounds__(kThreads) void time_mix_chunk_kernel(
    const float* __restrict__ x, int64_t x_stride, int r_off, int k_off, int v_off, int w_off, const float* __restrict__ w0,
    const float* __restrict__ u, const int32_t* __restrict__ cu, const int32_t* __restrict__ tile_req,
    const int32_t* __restrict__ tile_tok0, const int32_t* __restrict__ tile_ntok, float* __restrict__ items, int heads, int dim,
    int vdim) {
  constexpr int LD = DP + 4, PER = kCT * DP / kThreads;      // tokens a thread loads of a channel
  __shared__ __align__(16) float rs[kCT][LD], ks[kCT][LD], ws[kCT][LD], Bs[kCT][kCT];
  const int tile = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int n = tile_ntok[tile];
  if (n <= 0) return;                    // a padding tile
  const int req = tile_req[tile], tok0 = tile_tok0[tile], t0 = cu[req], vp = (vdim + 15) / 16 * 16;
  float* item = items + ((int64_t)(chunk_place(t0, req) + (tok0 - t0) / kCT) * heads + h) * mix_chunk_floats(DP, vp);
  f32x4 *Q = (f32x4*)item, *K = Q + 4 * DP, *V = K + 4 * DP, *Bm = V + 4 * vp;
  {
    const int ch = tid % DP, first = tid / DP * PER, at = h * dim + min(ch, dim - 1);
    const float* row = x + (int64_t)tok0 * x_stride + at;
    float r[PER], k[PER], w[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const float* p = row + (int64_t)min(first + i, n - 1) * x_stride;
      r[i] = p[r_off];
      k[i] = p[k_off];
      w[i] = p[w_off];
    }
    const float bias = w0[at];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const bool ok = ch < dim && first + i < n;
      rs[first + i][ch] = ok ? r[i] : 0.f;
      ks[first + i][ch] = ok ? k[i] : 0.f;
      ws[first + i][ch] = ok ? expf(-expf(w[i] + bias)) : 1.f;
    }
  }
  for (int e = tid; e < 4 * vp; e += kThreads) {               // four tokens of a value column
    const int col = e % vp, t = e / vp * 4;
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = col < vdim && t + i < n ? x[(int64_t)(tok0 + min(t + i, n - 1)) * x_stride + v_off + h * vdim + min(col, vdim - 1)] : 0.f;
    V[col / 16 * 64 + t / 4 * 16 + col % 16] = v;
  }
  __syncthreads();
  // Column s of B, sixteen threads each: k_s, decayed from token to token, with every later token's r.  A wave's four columns
  // begin at its first; which wave has the long ones changes from workgroup to workgroup.
  const int l = tid % 16, s_first = (tid / TL_WAVE + (int)blockIdx.x) % 4 * 4, s = s_first + tid % TL_WAVE / 16;
  float pb[kCT];
  {
    double y[DP / 64][4];
    f32x4 u4[DP / 64];
#pragma unroll
    for (int i = 0; i < DP / 64; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[i][e] = 0.0;
#pragma unroll
      for (int e = 0; e < 4; ++e) u4[i][e] = u[h * dim + min(i * 64 + l * 4 + e, dim - 1)];      // (beyond it k is zero)
    }
#pragma unroll
    for (int t0 = 0; t0 < kCT; t0 += 4) {
#pragma unroll
      for (int t = t0; t < t0 + 4; ++t) pb[t] = 0.f;
      if (t0 < s_first) continue;       // uniform; four tokens in one piece, so that all their operands are on their way
#pragma unroll
      for (int t = t0; t < t0 + 4; ++t) {
        double b[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < DP / 64; ++i) {
          const int ch = i * 64 + l * 4;
          const f32x4 w4 = *(const f32x4*)&ws[t][ch], k4 = *(const f32x4*)&ks[t][ch], r4 = *(const f32x4*)&rs[t][ch];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            b[e] = fma((double)r4[e], t == s ? (double)u4[i][e] * (double)k4[e] : y[i][e], b[e]);
            y[i][e] = t == s ? (double)k4[e] : y[i][e] * (double)w4[e];        // ahead of token s it is zero
          }
        }
        pb[t] = (float)((b[0] + b[1]) + (b[2] + b[3]));
      }
    }
  }
  const float bt = scatter_sums(pb, l);          // of token l
  Bs[l][s] = l >= s ? bt : 0.f;
  __syncthreads();
  if (tid < DP) {
    double g = 1.0;
#pragma unroll
    for (int t = 0; t < kCT; ++t) {
      rs[t][tid] = (float)((double)rs[t][tid] * g);
      g *= (double)ws[t][tid];
    }
    ((float*)(Bm + kCT * kCT / 4))[tid] = (float)g;
  } else if (tid < 2 * DP) {
    const int ch = tid - DP;
    double g = 1.0;
    f32x4 k4;
#pragma unroll
    for (int t = kCT - 1; t >= 0; --t) {
      k4[t % 4] = (float)((double)ks[t][ch] * g);
      g *= (double)ws[t][ch];
      if (t % 4 == 0) K[ch / 16 * 64 + t / 4 * 16 + ch % 16] = k4;
    }
  }
  __syncthreads();
  for (int e = tid; e < 4 * DP; e += kThreads) Q[e] = *(const f32x4*)&rs[e % 16][e / 64 * 16 + e % 64 / 16 * 4];
  if (tid < kCT * kCT / 4) Bm[tid] = *(const f32x4*)&Bs[tid % 16][tid / 16 * 4];
}

// A workgroup owns sixteen value columns of one (request, head).  Wave rg < 4 keeps rows [rg * 16 NT, (rg + 1) * 16 NT) of S, as
// results of matrix instructions, which are an operand of the next ones as they are, and leaves its part of Q S_0 in LDS; wave
// 4 adds the parts and the chunk's own and stores, transposed: a lane has four neighbouring columns of a token.  One barrier
// a chunk, which does not wait for the operands on their way: they come straight into registers, AHEAD chunks ahead, and no
// load stands in a branch (the compiler would wait for all at its end).  All rows in one wave, without a barrier, took 110 us
// where this takes 35 (six prompts of 67 to 801 tokens, 32 heads of 64 x 64): too many registers for what is on its way.
constexpr int kScanThreads = 5 * TL_WAVE;
template <int NT, int AHEAD>
__global__ __launch_bounds__(kScanThreads) void time_mix_scan_kernel(
    const float* __restrict__ items, float* __restrict__ state, int64_t state_stride, const int32_t* __restrict__ cu,
    const int32_t* __restrict__ slots, float* __restrict__ out, int heads, int dim, int vdim) {
  constexpr int DP = 64 * NT, P = DP / kSlice;
  __shared__ f32x4 os[2][4][TL_WAVE];             // parts of chunk c: [c % 2]
  const int r = blockIdx.z, h = blockIdx.x, vt = blockIdx.y, lane = threadIdx.x % TL_WAVE, q = lane / 16;
  const int rg = __builtin_amdgcn_readfirstlane(threadIdx.x / TL_WAVE);
  const int t0 = cu[r], t1 = cu[r + 1];
  if (t1 <= t0) return;                           // a request without tokens touches no state
  const int chunks = (t1 - t0 + kCT - 1) / kCT, vp = (vdim + 15) / 16 * 16, col = vt * 16 + lane % 16;
  const int64_t size = mix_chunk_floats(DP, vp), step = size * heads;
  const float* item0 = items + ((int64_t)chunk_place(t0, r) * heads + h) * size;
  auto buffer = [&](int c) {                      // (behind the last chunk: that one again)
    return __builtin_amdgcn_make_buffer_rsrc((void*)(item0 + step * min(c, chunks - 1)), 0, (int)size * 4, 0x00020000);
  };
  auto load = [](const __amdgpu_buffer_rsrc_t from, int at, int more) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, at, more, 0));
  };
  auto meet = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  const int v_at = (8 * DP + vt * TL_WAVE + lane) * 16;
  if (rg == 4) {
    const int row_bytes = heads * vdim * 4, b_at = (8 * DP + 4 * vp + lane) * 16;
    const int to = lane % 16 * row_bytes + (vt * 16 + q * 4) * 4;
    struct Own {
      f32x4 v, b;
    };
    auto request = [&](Own& x, int c) {
      const __amdgpu_buffer_rsrc_t from = buffer(c);
      x.v = load(from, v_at, 0);
      x.b = load(from, b_at, 0);
    };
    // Two chunks ahead: with one, what is done here between a chunk's values and the next request is on the way of every chunk
    // (2,047 tokens of 32 heads of 64 x 64, both kernels: 110 us with the products alone there, 120 with the look for numbers
    // that are not finite as well, 87 so).
    Own op[2];
    request(op[0], 0);
    request(op[1], 1);
    auto chunk = [&](Own& x, int c) {
      f32x4 own[4], v = x.v;
      const bool hidden = hides_not_finite(v);
#pragma unroll
      for (int j = 0; j < 4; ++j) own[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j], x.b[j], zero, 0, 0, 0);
      request(x, c + 2);
      __builtin_amdgcn_sched_barrier(0);
      meet();
      f32x4 y = ((os[c % 2][0][lane] + os[c % 2][1][lane]) + (os[c % 2][2][lane] + os[c % 2][3][lane])) + ((own[0] + own[1]) + (own[2] + own[3]));
      if (hidden) {                               // v and b once more: to keep them would cost registers and copies in every chunk
        Own again;
        request(again, c);
        add_not_finite(y, again.v, again.b, lane);
      }
      // a buffer that ends with the request's last token of the chunk: what lies behind is not stored, without a branch
      const int n = min(kCT, t1 - t0 - c * kCT);
      const __amdgpu_buffer_rsrc_t rows =
          __builtin_amdgcn_make_buffer_rsrc(out + ((int64_t)(t0 + c * kCT) * heads + h) * vdim, 0, (n - 1) * row_bytes + vdim * 4, 0x00020000);
      if (vdim % 4 == 0) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(tl_u32x4, y), rows, vt * 16 + q * 4 < vdim ? to : -16, 0, 0);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[j]), rows, vt * 16 + q * 4 + j < vdim ? to + j * 4 : -4, 0, 0);
      }
    };
    int c = 0;
    for (; c + 2 <= chunks; c += 2) {
      chunk(op[0], c);
      chunk(op[1], c + 1);
    }
    if (c < chunks) chunk(op[0], c);
    return;
  }
  float* Sg = state + (int64_t)slots[r] * state_stride + ((int64_t)h * kSlice * vdim + min(col, vdim - 1)) * P + rg * NT * 4 + q;
  f32x4 S[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) S[i][e] = Sg[(int64_t)e * vdim * P + i * 4];
  struct Operands {
    f32x4 q[NT], k[NT], g[NT], v;
  };
  Operands op[AHEAD];
  const int at = (rg * NT * TL_WAVE + lane) * 16, g_at = (8 * DP + 4 * vp + TL_WAVE + rg * NT * 4 + q) * 16;
  auto request = [&](Operands& x, int c) {
    const __amdgpu_buffer_rsrc_t from = buffer(c);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      x.q[i] = load(from, at, i * 1024);
      x.k[i] = load(from, at, 64 * DP + i * 1024);
      x.g[i] = load(from, g_at, i * 64);
    }
    x.v = load(from, v_at, 0);
  };
  auto chunk = [&](Operands& x, int c, auto ask) {
    f32x4 o[NT][4], add[NT][2];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        o[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(S[i][j], x.q[i][j], zero, 0, 0, 0);
        add[i][j % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.k[i][j], x.v[j], j > 1 ? add[i][j % 2] : zero, 0, 0, 0);
      }
    f32x4 sum = (o[0][0] + o[0][1]) + (o[0][2] + o[0][3]);
    if constexpr (NT == 2) sum += (o[1][0] + o[1][1]) + (o[1][2] + o[1][3]);
    os[c % 2][rg][lane] = sum;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[i][e] = fmaf(x.g[i][e], S[i][e], add[i][0][e] + add[i][1][e]);
    if constexpr (decltype(ask)::value) request(x, c + AHEAD);
    meet();
  };
  request(op[0], 0);
  if (chunks == 1) {                              // a step's single tokens: nothing is asked for ahead
    chunk(op[0], 0, std::false_type{});
  } else {
#pragma unroll
    for (int d = 1; d < AHEAD; ++d) request(op[d], d);
    int c = 0;
    for (; c + AHEAD <= chunks; c += AHEAD) {
#pragma unroll
      for (int d = 0; d < AHEAD; ++d) chunk(op[d], c + d, std::true_type{});
    }
#pragma unroll
    for (int d = 0; d < AHEAD - 1; ++d)
      if (c + d < chunks) chunk(op[d], c + d, std::true_type{});      // (the whole workgroup)
  }
  if (col < vdim) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) Sg[(int64_t)e * vdim * P + i * 4] = S[i][e];
  }
}

// out[i] = tanh(in[i]) rounded to T (the middle of a low-rank projection).
template <typename T>
__global__ void tanh_kernel(const float* __restrict__ in, int64_t in_stride, T* __restrict__ out, int64_t total, int n) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= total) return;
  const int64_t t = i / n;
  out[i] = from_f32<T>(tanhf(in[t * in_stride + (i - t * n)]));
}

}  // namespace

extern "C" {

int tl_time_mix_slices(int dim) {
  int P = 1;
  while (P * kSlice < dim) P *= 2;
  return P;
}

// h: [n_tokens, width] of the engine's type; mu: float32 [n_mix, width]; out: [n_mix, n_tokens, width].
// save_single: a request that brings exactly one token also gets that token's h saved in its state row (requests
// with more tokens need tl_shift_save behind this kernel).
int tl_shift_mix(const void* h, int64_t h_stride, float* state, int64_t state_stride, int64_t prev_off,
                 const int32_t* req_of_token, const int32_t* cu, const int32_t* slots, const float* mu, void* out,
                 int n_tokens, int n_mix, int width, int save_single, int dtype, hipStream_t stream) {
  if (n_tokens <= 0) return TL_OK;
  if (width <= 0 || n_mix <= 0 || !h || !state || !req_of_token || !cu || !slots || !mu || !out) return TL_ERR_ARG;
  dim3 g(n_tokens, (width + kThreads - 1) / kThreads), b(kThreads);
  const int64_t plane = (int64_t)n_tokens * width;
  if (dtype == 0)
    hipLaunchKernelGGL(shift_mix_kernel<float>, g, b, 0, stream, (const float*)h, h_stride, state, state_stride, prev_off,
                       req_of_token, cu, slots, mu, (float*)out, plane, n_mix, width, save_single);
  else if (dtype == 1)
    hipLaunchKernelGGL(shift_mix_kernel<bf16_t>, g, b, 0, stream, (const bf16_t*)h, h_stride, state, state_stride,
                       prev_off, req_of_token, cu, slots, mu, (bf16_t*)out, plane, n_mix, width, save_single);
  else
    return TL_ERR_ARG;
  return tl_launch_status();
}

int tl_shift_save(const void* h, int64_t h_stride, float* state, int64_t state_stride, int64_t prev_off,
                  const int32_t* cu, const int32_t* slots, int n_requests, int width, int dtype, hipStream_t stream) {
  if (n_requests <= 0) return TL_OK;
  if (width <= 0 || !h || !state || !cu || !slots) return TL_ERR_ARG;
  dim3 g(n_requests, (width + kThreads - 1) / kThreads), b(kThreads);
  if (dtype == 0)
    hipLaunchKernelGGL(shift_save_kernel<float>, g, b, 0, stream, (const float*)h, h_stride, state, state_stride, prev_off,
                       cu, slots, width);
  else if (dtype == 1)
    hipLaunchKernelGGL(shift_save_kernel<bf16_t>, g, b, 0, stream, (const bf16_t*)h, h_stride, state, state_stride,
                       prev_off, cu, slots, width);
  else
    return TL_ERR_ARG;
  return tl_launch_status();
}

// x: float32 rows that hold r, k, the decay's pre-activation (heads * dim columns each, from r_off, k_off, w_off)
// and v (heads * vdim columns from v_off).  state rows: S as [heads][4][vdim][P] floats from column 0, P =
// tl_time_mix_slices(dim).  o: float32 [n_tokens, heads * vdim].
int tl_time_mix_recurrence(const float* x, int64_t x_stride, int r_off, int k_off, int v_off, int w_off, const float* w0,
                           const float* u, float* state, int64_t state_stride, const int32_t* cu, const int32_t* slots,
                           float* o, int n_requests, int heads, int dim, int vdim, hipStream_t stream) {
  if (n_requests <= 0) return TL_OK;
  if (heads <= 0 || heads > 65535 || n_requests > 65535 || dim <= 0 || dim > 256 || vdim <= 0 || !x || !w0 || !u ||
      !state || !cu || !slots || !o)
    return TL_ERR_ARG;
  const int P = tl_time_mix_slices(dim);
  if (state_stride < (int64_t)heads * kSlice * vdim * P) return TL_ERR_ARG;
  const int EC = kThreads / P;
  if ((vdim + EC - 1) / EC > 65535) return TL_ERR_ARG;
  dim3 g((vdim + EC - 1) / EC, heads, n_requests), b(kThreads);
#define TL_TIME_MIX(PP)                                                                                               \
  case PP:                                                                                                            \
    hipLaunchKernelGGL(time_mix_recurrence_kernel<PP>, g, b, 0, stream, x, x_stride, r_off, k_off, v_off, w_off, w0, u, \
                       state, state_stride, cu, slots, o, heads, dim, vdim);                                          \
    break;
  switch (P) {
    TL_TIME_MIX(1) TL_TIME_MIX(2) TL_TIME_MIX(4) TL_TIME_MIX(8) TL_TIME_MIX(16) TL_TIME_MIX(32) TL_TIME_MIX(64)
    default: return TL_ERR_ARG;
  }
#undef TL_TIME_MIX
  return tl_launch_status();
}

// The same in chunks (heads of at most 128 x 128).  tile_*: every request's tokens cut into chunks of at most 16, request after
// request (ntok 0: padding).  items: float32 [(n_tokens / 16 + n_requests + 1) * heads * tl_time_mix_chunk_floats(dim, vdim)].
int64_t tl_time_mix_chunk_floats(int dim, int vdim) { return mix_chunk_floats(dim <= 64 ? 64 : 128, (vdim + 15) / 16 * 16); }

int tl_time_mix_chunks(const float* x, int64_t x_stride, int r_off, int k_off, int v_off, int w_off, const float* w0,
                       const float* u, float* state, int64_t state_stride, const int32_t* cu, const int32_t* slots,
                       const int32_t* tile_req, const int32_t* tile_tok0, const int32_t* tile_ntok, float* items, float* o,
                       int n_tiles, int n_requests, int heads, int dim, int vdim, hipStream_t stream) {
  if (n_tiles <= 0 || n_requests <= 0) return TL_OK;
  if (heads <= 0 || heads > 65535 || n_requests > 65535 || dim <= 32 || dim > kMaxChunkDim || vdim <= 0 || vdim > kMaxChunkDim || !x || !w0 || !u ||
      !state || !cu || !slots || !tile_req || !tile_tok0 || !tile_ntok || !items || ((uintptr_t)items & 15) || !o)
    return TL_ERR_ARG;
  if (state_stride < (int64_t)heads * kSlice * vdim * tl_time_mix_slices(dim)) return TL_ERR_ARG;
  // heads first in the grid of the scan: the workgroups of the longest request are then spread over all XCDs (eight requests
  // of the lengths above, requests first: 103 us), those of a head share one
  dim3 g(n_tiles, heads), b(kThreads), gs(heads, (vdim + 15) / 16, n_requests), bs(kScanThreads);
#define TL_MIX_CHUNK(DP, AHEAD)                                                                                          \
  {                                                                                                                      \
    hipLaunchKernelGGL(time_mix_chunk_kernel<DP>, g, b, 0, stream, x, x_stride, r_off, k_off, v_off, w_off, w0, u, cu,   \
                       tile_req, tile_tok0, tile_ntok, items, heads, dim, vdim);                                         \
    hipLaunchKernelGGL((time_mix_scan_kernel<DP / 64, AHEAD>), gs, bs, 0, stream, items, state, state_stride, cu, slots, o, \
                       heads, dim, vdim);                                                                                \
  }
  if (dim <= 64) TL_MIX_CHUNK(64, 4)
  else TL_MIX_CHUNK(128, 2)
#undef TL_MIX_CHUNK
  return tl_launch_status();
}

// out[t, j] = tanh(in[t, j]) for j < n; in float32 with row stride in_stride, out [n_rows, n] of the engine's type.
int tl_tanh_rows(const float* in, int64_t in_stride, void* out, int n_rows, int n, int dtype, hipStream_t stream) {
  if (n_rows <= 0) return TL_OK;
  if (n <= 0 || in_stride < n || !in || !out) return TL_ERR_ARG;
  const int64_t total = (int64_t)n_rows * n;
  dim3 g((unsigned)ceil_div64(total, kThreads)), b(kThreads);
  if (dtype == 0)
    hipLaunchKernelGGL(tanh_kernel<float>, g, b, 0, stream, in, in_stride, (float*)out, total, n);
  else if (dtype == 1)
    hipLaunchKernelGGL(tanh_kernel<bf16_t>, g, b, 0, stream, in, in_stride, (bf16_t*)out, total, n);
  else
    return TL_ERR_ARG;
  return tl_launch_status();
}

}  // extern "C"
