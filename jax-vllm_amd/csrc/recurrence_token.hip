// Launches of recurrence_token_block by themselves, and what one takes for a launch beside another kernel's blocks.
#include "recurrence_token.h"

template <typename T, bool DELTA>
__global__ void __launch_bounds__(TK_THREADS)
recurrence_token_kernel(TokenArgs a) { recurrence_token_block<T, DELTA>(a, blockIdx.x, blockIdx.y); }

// dim and vdim up to this, vdim in fours, the state on 16 bytes.
extern "C" int jv_recurrence_token_max_dim() { return TK_DIM; }
extern "C" int jv_recurrence_token_max_rank() { return 64; }

static bool token_sizes(const TokenArgs& a, int n_requests) {
  return a.dim >= 1 && a.dim <= TK_DIM && a.vdim >= 4 && a.vdim <= TK_DIM && a.vdim % 4 == 0 && a.heads >= 1 && a.heads <= 65535 &&
         (uintptr_t)a.state % 16 == 0 && n_requests >= 1;
}

extern "C" int jv_token_launch_bytes() { return (int)sizeof(TokenLaunch); }

template <typename T>
static int launch_token(const TokenLaunch& l, hipStream_t stream) {
  const dim3 grid(l.n_requests, l.args.heads);
  if (l.delta) hipLaunchKernelGGL((recurrence_token_kernel<T, true>), grid, dim3(TK_THREADS), 0, stream, l.args);
  else hipLaunchKernelGGL((recurrence_token_kernel<T, false>), grid, dim3(TK_THREADS), 0, stream, l.args);
  return JV_LAUNCH_CHECK();
}
extern "C" int jv_token_launch(const TokenLaunch* held, void* stream) {
  return held->bytes == 2 ? launch_token<bf16_t>(*held, (hipStream_t)stream) : launch_token<float>(*held, (hipStream_t)stream);
}
// hold null: now
static int launch_or_hold(const TokenLaunch& l, TokenLaunch* hold, void* stream) {
  if (!hold) return jv_token_launch(&l, stream);
  *hold = l;
  return 0;
}

#define DEFINE_TOKEN(SUF, T)                                                                                                     \
  extern "C" int jv_delta_token_##SUF(void* out, const void* proj, long long ld, int q_at, int gate_at, int dt_at, int w_at,     \
                                      int taps, const float* conv_w, float* conv_state, const float* dt_bias,                    \
                                      const float* a_log, float unit_eps, float q_scale, const float* norm, float eps,           \
                                      float out_scale, float* state, const int* slot_ids, const int* cu_seqlens,                 \
                                      int n_requests, int heads, int dim, int vdim, void* stream, TokenLaunch* hold) {           \
    if (n_requests <= 0 || heads <= 0) return 0;                                                                                 \
    TokenArgs a = {out, proj, ld, q_at, q_at + heads * dim, q_at + 2 * heads * dim, gate_at, norm, eps, out_scale, q_scale,      \
                   state, slot_ids, cu_seqlens, heads, dim, vdim};                                                               \
    a.dt_at = dt_at, a.w_at = w_at, a.taps = taps, a.conv_w = conv_w, a.dt_bias = dt_bias, a.a_log = a_log;                      \
    a.conv_state = conv_state, a.unit_eps = unit_eps;                                                                            \
    if (!token_sizes(a, n_requests) || taps < 1 || taps > RC_MAX_LAGS + 1) return (int)hipErrorInvalidValue;                     \
    return launch_or_hold(TokenLaunch{a, 1, (int)sizeof(T), n_requests}, hold, stream);                                          \
  }                                                                                                                              \
  extern "C" int jv_gated_linear_token_##SUF(void* out, const void* proj, long long ld, int q_at, int gate_at, int low_at,       \
                                             int rank, const void* up, const float* up_bias, float tau, float q_scale,           \
                                             const float* norm, float eps, float* state, const int* slot_ids,                    \
                                             const int* cu_seqlens, int n_requests, int heads, int dim, int vdim,                \
                                             void* stream, TokenLaunch* hold) {                                                  \
    if (n_requests <= 0 || heads <= 0) return 0;                                                                                 \
    TokenArgs a = {out, proj, ld, q_at, q_at + heads * dim, q_at + 2 * heads * dim, gate_at, norm, eps, 1.f, q_scale,            \
                   state, slot_ids, cu_seqlens, heads, dim, vdim};                                                               \
    a.low_at = low_at, a.rank = rank, a.up = up, a.up_bias = up_bias, a.inv_tau = 1.f / tau;                                     \
    a.vec = rank % (16 / (int)sizeof(T)) == 0 && (uintptr_t)up % 16 == 0;                                                        \
    if (!token_sizes(a, n_requests) || rank < 1 || rank > jv_recurrence_token_max_rank() || !(tau > 0.f))                        \
      return (int)hipErrorInvalidValue;                                                                                          \
    return launch_or_hold(TokenLaunch{a, 0, (int)sizeof(T), n_requests}, hold, stream);                                          \
  }
DEFINE_TOKEN(bf16, bf16_t)
DEFINE_TOKEN(f32, float)
