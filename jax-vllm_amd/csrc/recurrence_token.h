// One token of a recurrent mixer, from its input product to its gated and normed result, a (request, head) a block.
//
//   delta:  q, k, v through the causal filter (and its state) and silu, q and k to unit length;  g = exp(-exp(A) softplus(raw +
//           bias)), w = sigmoid(raw):   S <- g S;  u = w (v - S^T k);  S <- S + k u^T;  o = S^T q
//   gated:  a = exp(log(sigmoid(W low + b)) / tau) per key channel:    S <- diag(a) S + k v^T;  o = S^T q
//   both:   out = o / rms(o) * norm * silu(gate) * out_scale           per head
//
// Bound by reading and writing the states, 2 x 16.8 MB for 16 requests of 16 heads of 128 x 128 (6 us at a copy's rate).  As
// launches of their own the filter, the gates, the unit norms, the update and the norm behind it took 34 us a layer there, most of
// it round trips: nothing of a token is larger than a block's registers.  So the block asks for its whole state first (8 pieces
// of 16 bytes a thread) and makes everything else while that is on its way:
// 11.6 us as profiled (delta; 34 before) and 10.1 (gated; 24.6 before, with the decays' product).
// Sizes: dim and vdim up to 128, vdim in fours (rows of the state in pieces of 16 bytes), a q/k head per head (each filter channel
// belongs to one block, which alone moves its state).
#pragma once
#include "recurrence_math.h"

#define TK_DIM 128
#define TK_THREADS 512
#define TK_PARTS 16           // rows of the state that the block's threads stand on; a thread has rows part + 16 i
#define TK_ROWS (TK_DIM / TK_PARTS)

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct TokenArgs {
  void* out;                  // [n][heads * vdim]
  const void* proj;           // rows of the input product, stride ld; columns of q, k, v and the gate
  long long ld;
  int q_at, k_at, v_at, gate_at;
  const float* norm;          // [vdim]
  float eps, out_scale, q_scale;
  float* state;               // [slots][heads][dim][vdim]
  const int* slot_ids;
  const int* cu_seqlens;
  int heads, dim, vdim;
  // delta
  int dt_at, w_at, taps;
  const float *conv_w, *dt_bias, *a_log;
  float* conv_state;          // [slots][taps - 1][channels]
  float unit_eps;
  // gated
  int low_at, rank, vec;
  const void* up;             // [heads * dim][rank]
  const float* up_bias;
  float inv_tau;
};

// What a launch of it takes, kept by the caller until another kernel's launch takes it along.
struct TokenLaunch {
  TokenArgs args;
  int delta, bytes, n_requests;      // bytes: of an element of proj
};
extern "C" int jv_token_launch(const TokenLaunch* held, void* stream);

// The block of request r and head h.
template <typename T, bool DELTA>
__device__ __forceinline__ void recurrence_token_block(const TokenArgs& a, int r, int h) {
  __shared__ __attribute__((aligned(16))) float qs[TK_DIM], ks[TK_DIM], vs[TK_DIM], ds[TK_DIM], gs[TK_DIM], head[8], squares[4];
  __shared__ f32x4 sums_u[8][32], sums_o[8][32];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t0 = a.cu_seqlens[r];
  if (a.cu_seqlens[r + 1] <= t0) return;
  const int slot = a.slot_ids[r], dim = a.dim, vdim = a.vdim;
  const int cq = tid & 31, part = tid >> 5;
  const bool live = 4 * cq < vdim;
  float* S = a.state + ((long long)slot * a.heads + h) * dim * vdim + (live ? 4 * cq : 0);
  f32x4 s[TK_ROWS];
#pragma unroll
  for (int i = 0; i < TK_ROWS; ++i) s[i] = *(const f32x4*)(S + (long long)min(part + i * TK_PARTS, dim - 1) * vdim);

  // threads 0..127 a channel of q each, then k, v, and what else a head has
  const T* row = (const T*)a.proj + (long long)t0 * a.ld;
  const int kind = tid >> 7, i0 = tid & 127, size = kind == 0 || kind == 1 ? dim : vdim, at = min(i0, size - 1);
  const bool mine = i0 < size;
  const int gate_kind = DELTA ? 3 : 2;
  float gate = 0.f, norm = 0.f;
  if (kind == gate_kind) {
    gate = to_f32(row[a.gate_at + h * vdim + at]);
    norm = a.norm[at];
  }
  if (kind < 3) {
    const int col = (kind == 0 ? a.q_at + h * dim : kind == 1 ? a.k_at + h * dim : a.v_at + h * vdim) + at;
    const float x = to_f32(row[col]);
    float y = x;
    if (DELTA) {
      const int c = (kind == 0 ? h * dim : kind == 1 ? (a.heads + h) * dim : 2 * a.heads * dim + h * vdim) + at;
      const int lags = a.taps - 1, channels = a.heads * (2 * dim + vdim);
      const float* w = a.conv_w + (long long)c * a.taps;
      float* st = a.conv_state + (long long)slot * lags * channels + c;
      const float* old = lags ? st : w;            // an address to read where there is no state
      float win[RC_MAX_LAGS], wl[RC_MAX_LAGS];     // row p of the state, the input of lag lags - p
#pragma unroll
      for (int p = 0; p < RC_MAX_LAGS; ++p) {
        const int q = max(min(p, lags - 1), 0);
        win[p] = old[(long long)q * channels * (lags ? 1 : 0)];
        wl[p] = w[q];
      }
      const float w0 = w[lags];
      float acc = 0.f;
#pragma unroll
      for (int p = 0; p < RC_MAX_LAGS; ++p) acc = p < lags ? fmaf(wl[p], win[p], acc) : acc;
      y = rc_silu(fmaf(w0, x, acc));
      if (mine) {
#pragma unroll
        for (int p = 0; p < RC_MAX_LAGS; ++p)
          if (p < lags) st[(long long)p * channels] = p + 1 < lags ? win[p + 1 < RC_MAX_LAGS ? p + 1 : p] : x;
      }
    } else if (kind == 0) {
      y *= a.q_scale;
    }
    y = mine ? y : 0.f;
    (kind == 0 ? qs : kind == 1 ? ks : vs)[i0] = y;
    if (DELTA && kind < 2) {
      const float ss = wave_sum(y * y);
      if (lane == 0) squares[wave] = ss;
    }
  } else if (DELTA) {
    const float dt = rc_softplus(to_f32(row[a.dt_at + h]) + a.dt_bias[h]);
    const float g = expf(-expf(a.a_log[h]) * dt), w = 1.f / (1.f + expf(-to_f32(row[a.w_at + h])));
    if (i0 == 0) { head[0] = g; head[1] = w; }
  } else {      // the decay of key channel i0
    const int c = h * dim + min(i0, dim - 1);
    const T* w = (const T*)a.up + (long long)c * a.rank;
    const T* low = row + a.low_at;
    float z = a.up_bias[c];
    if (a.vec) {
      constexpr int EP = 16 / (int)sizeof(T);
      typedef T tv __attribute__((ext_vector_type(EP)));
#pragma unroll 2
      for (int j = 0; j < a.rank; j += EP) {
        const tv wv = *(const tv*)(w + j);
#pragma unroll
        for (int e = 0; e < EP; ++e) z = fmaf(to_f32<T>(wv[e]), to_f32(low[j + e]), z);
      }
    } else {
      for (int j = 0; j < a.rank; ++j) z = fmaf(to_f32(w[j]), to_f32(low[j]), z);
    }
    ds[i0] = expf(-(fmaxf(-z, 0.f) + softplus_of_negative(fabsf(z))) * a.inv_tau);
  }
  if (kind == gate_kind) gs[i0] = mine ? rc_silu(gate) * norm : 0.f;
  __syncthreads();

  float q_by = 1.f, k_by = 1.f, g = 1.f;
  if (DELTA) {
    q_by = a.q_scale / sqrtf(squares[0] + squares[1] + a.unit_eps);
    k_by = 1.f / sqrtf(squares[2] + squares[3] + a.unit_eps);
    g = head[0];
  }
  f32x4 u = *(const f32x4*)(vs + 4 * cq);
  if (DELTA) {
    f32x4 pred = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < TK_ROWS; ++i) {
      const int d = part + i * TK_PARTS;
      const float kd = ks[d] * k_by;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[i][e] = live && d < dim ? s[i][e] * g : 0.f;
        pred[e] = fmaf(s[i][e], kd, pred[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) pred[e] += __shfl_xor(pred[e], 32, JV_WAVE);
    if (lane < 32) sums_u[wave][cq] = pred;
    __syncthreads();
    pred = sums_u[0][cq];
#pragma unroll
    for (int w = 1; w < 8; ++w)
#pragma unroll
      for (int e = 0; e < 4; ++e) pred[e] += sums_u[w][cq][e];
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = head[1] * (u[e] - pred[e]);
  }
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < TK_ROWS; ++i) {
    const int d = part + i * TK_PARTS;
    const bool in = live && d < dim;
    const float kd = ks[d] * k_by, qd = qs[d] * q_by, a_d = DELTA ? 1.f : ds[d];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[i][e] = !in ? 0.f : DELTA ? fmaf(kd, u[e], s[i][e]) : fmaf(a_d, s[i][e], kd * u[e]);
      o[e] = fmaf(s[i][e], qd, o[e]);
    }
    if (in) *(f32x4*)(S + (long long)d * vdim) = s[i];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] += __shfl_xor(o[e], 32, JV_WAVE);
  if (lane < 32) sums_o[wave][cq] = o;
  __syncthreads();
  if (wave > 0) return;
  float y[2] = {0.f, 0.f};                 // columns 2 lane and 2 lane + 1
#pragma unroll
  for (int w = 0; w < 8; ++w)
#pragma unroll
    for (int e = 0; e < 2; ++e) y[e] += ((const float*)sums_o[w])[2 * lane + e];
  const float inv = rsqrtf(wave_sum(fmaf(y[0], y[0], y[1] * y[1])) / (float)vdim + a.eps) * a.out_scale;
  T* out = (T*)a.out + ((long long)t0 * a.heads + h) * vdim;
#pragma unroll
  for (int e = 0; e < 2; ++e)
    if (2 * lane + e < vdim) out[2 * lane + e] = from_f32<T>(y[e] * gs[2 * lane + e] * inv);
}
