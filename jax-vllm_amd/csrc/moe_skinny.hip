// The two grouped products of routed experts for steps of few tokens (decode): every chosen expert has a row or a few,
// so the time is the reading of its weights.  bfloat16, float accumulation; the grouping they read has tiles of at most
// 16 rows of one expert.
//
// A block of 4 waves takes one tile of (token, choice) rows against 64 / WK rows of the expert's weight: WK waves share
// out the inner size of 16 rows of W (a long inner size gives every wave enough of it, a short one goes to one wave).  A
// wave streams its slice of W straight into MFMA operands (v_mfma_f32_16x16x32_bf16, A = 16 rows of W, B = the tile's
// rows of x: rows beyond the tile repeat its last one and cost no bytes), STEPS steps asked for while the ones before are
// multiplied.  W's addresses hang on the tile's expert alone, so its first loads are on their way while the chain
// offsets -> order -> rows of x is walked.  The waves' sums are added in LDS in their order: an output row is one fixed
// sum whatever else is in the step.
//   MS_GATED:  z[pos] = act(w g) * (w u), g = Wg[e] x[token], u = Wu[e] x[token]    (bf16)
//   MS_PLAIN:  z[pos] = act(w u), u = Wu[e] x[token]: experts without a gate        (bf16)
//   MS_DOWN:   y[kk][token] = (Wd[e] z[pos]) * w_out                                (float)
#include "common.h"

typedef __bf16 ms_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ms_f32x4 __attribute__((ext_vector_type(4)));

enum { MS_DOWN = 0, MS_GATED = 1, MS_PLAIN = 2 };
#define MS_ROWS 16
#define MS_STEPS 2      // measured at 2,048 x 768 and 4,096 x 1,536, 8 tokens: 74 MB in 18.6 us and 440 MB in 79 us; 4 steps 21 and 81

template <int MODE, int WK>
__global__ void __launch_bounds__(256)
moe_skinny_kernel(void* __restrict__ out, const bf16_t* __restrict__ a_rows, const bf16_t* __restrict__ W0,
                  const bf16_t* __restrict__ W1, const int* __restrict__ meta, const int* __restrict__ offsets,
                  const int* __restrict__ tile_expert, const int* __restrict__ tile_row0, const int* __restrict__ order,
                  const float* __restrict__ weights, int top, int n_tokens, int K, int N, JvAct act, int use_weight) {
  constexpr bool GATED = MODE == MS_GATED, BY_TOKEN = MODE != MS_DOWN;
  constexpr int STEPS = MS_STEPS, NB = 64 / WK;          // rows of W a block takes
  __shared__ float red[GATED ? 2 : 1][4][16][17];
  // neighbouring blocks take neighbouring rows of one expert: what is read at one time lies side by side (blocks of
  // different experts at the same rows would be a whole expert apart, and meet on the same memory channels)
  const int per_tile = (N + NB - 1) / NB, tile = blockIdx.x / per_tile;
  const int tiles = meta[0], e = tile_expert[tile], row0 = tile_row0[tile];
  if (tile >= tiles) return;                             // (the entries beyond the tiles hold anything)
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, lc = lane >> 4;
  const int n0 = (blockIdx.x - tile * per_tile) * NB, wn = n0 + wave / WK * 16;
  const long long wr = ((long long)e * N + min(wn + li, N - 1)) * K;
  const bf16_t* w0 = W0 + wr;
  const bf16_t* w1 = GATED ? W1 + wr : W0;
  const int steps = (K + 31) / 32, per_wave = (steps + WK - 1) / WK;
  const int s_lo = wave % WK * per_wave, s_hi = min(steps, s_lo + per_wave);
  const ms_bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  ms_f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
  ms_bf16x8 a0[2][STEPS], a1[2][GATED ? STEPS : 1], b[2][STEPS];
  auto column = [&](int s) { return min(min(s, s_hi - 1) * 32 + lc * 8, K - 8); };   // beyond the slice: its last columns again
  auto fetch_w = [&](int buf, int s0) {
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      a0[buf][u] = *(const ms_bf16x8*)(w0 + column(s0 + u));
      if (GATED) a1[buf][u] = *(const ms_bf16x8*)(w1 + column(s0 + u));
    }
  };
  const bool live = s_lo < s_hi && wn < N;
  if (live) fetch_w(0, s_lo);
  const int rows = min(MS_ROWS, offsets[e + 1] - row0);
  const int mine = row0 + min(li, rows - 1);
  const bf16_t* xr = a_rows + (BY_TOKEN ? (long long)(order[mine] / top) : (long long)mine) * K;
  auto fetch_x = [&](int buf, int s0) {
#pragma unroll
    for (int u = 0; u < STEPS; ++u) b[buf][u] = *(const ms_bf16x8*)(xr + column(s0 + u));
  };
  auto multiply = [&](int buf, int s0) {
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      const bool in = s0 + u < s_hi && (s0 + u) * 32 + lc * 8 < K;
      const ms_bf16x8 x = in ? b[buf][u] : zero;
      acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[buf][u], x, acc0, 0, 0, 0);
      if (GATED) acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[buf][u], x, acc1, 0, 0, 0);
    }
  };
  if (live) {
    fetch_x(0, s_lo);
    for (int s = s_lo; s < s_hi; s += 2 * STEPS) {
      fetch_w(1, s + STEPS);
      fetch_x(1, s + STEPS);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0, s);
      fetch_w(0, s + 2 * STEPS);
      fetch_x(0, s + 2 * STEPS);
      __builtin_amdgcn_sched_barrier(0);
      multiply(1, s + STEPS);
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    red[0][wave][lc * 4 + c][li] = acc0[c];
    if (GATED) red[GATED ? 1 : 0][wave][lc * 4 + c][li] = acc1[c];
  }
  __syncthreads();
  for (int i = tid; i < NB * 16; i += 256) {
    const int m = i / NB, nl = i - m * NB, n = n0 + nl;
    if (m >= rows || n >= N) continue;
    float y0 = 0.f, y1 = 0.f;                            // sums with W0 and, gated, with W1
#pragma unroll
    for (int ww = 0; ww < WK; ++ww) {
      y0 += red[0][nl / 16 * WK + ww][nl & 15][m];
      if (GATED) y1 += red[GATED ? 1 : 0][nl / 16 * WK + ww][nl & 15][m];
    }
    const int s = order[row0 + m];
    const float w = use_weight ? weights[s] : 1.f;
    if (MODE == MS_GATED) {
      ((bf16_t*)out)[(long long)(row0 + m) * N + n] = from_f32<bf16_t>(jv_gated(act, y0 * w, y1 * w));
    } else if (MODE == MS_PLAIN) {
      ((bf16_t*)out)[(long long)(row0 + m) * N + n] = from_f32<bf16_t>(jv_act(act.id, y0 * w));
    } else {
      const int token = s / top, kk = s - token * top;
      ((float*)out)[((long long)kk * n_tokens + token) * N + n] = y0 * w;
    }
  }
}

// The same where an expert's rows begin on 16 bytes and the inner size is a multiple of 64 up to 4,096: WK of a block's waves share
// out the inner size of 16 rows of W, the others take further 16 rows.  A wave asks for its rows of x (into registers, where they
// stay) and for its first chunks of W (whole lines, straight into a ring of its own in LDS) in one go and waits for no other wave
// before the parts meet; several blocks share a unit, so one's chain of addresses runs beside the others' streams: two of 64 KB, or four and more of
// half of that or less where their slices stay long enough (microseconds in graphs, cold weights, two of 64 KB / so: 16 tokens, 4 of 32 experts, 768 x 2,048
// 30.2 + 16.5 / 28.9 + 15.4, 512 x 2,048 27.1 + 13.9 / 25.8 + 12.6; 48 of 64 x 1,024, width 4,096, down 102.7 / 99.0; inner sizes of 4,096 as before: 152 / 152).
// Both products of a layer in a graph, cold weights, microseconds (the kernel above): 32 experts x 768, 4 chosen, width 2,048: 4
// tokens 28.2 (29.9), 16 56.3 (59.9), 48 62.7 (69.9); 32 x 512 of width 1,536: 1 token 10.7 (14.2), 8 31.1 (35.0); 64 x 1,024, 8 chosen, width
// 4,096: 16 tokens 252 (261), 48 288 (318), 5.5 TB/s.  Not better: one wave a row tile at inner sizes up to 512, 4 at 2,048.
#define MF_K 64            // columns of a chunk: a row of it is 128 bytes, 8 pieces of 16

// WAVES of a block, the KB of their rings; CW: the most chunks of a wave.
template <int MODE, int WAVES, int KB, int WK, int CW>
__global__ void __launch_bounds__(64 * WAVES)
moe_few_kernel(void* __restrict__ out, const bf16_t* __restrict__ a_rows, const bf16_t* __restrict__ W0,
               const bf16_t* __restrict__ W1, const int* __restrict__ meta, const int* __restrict__ offsets,
               const int* __restrict__ tile_expert, const int* __restrict__ tile_row0, const int* __restrict__ order,
               const float* __restrict__ weights, int top, int n_tokens, int K, int N, JvAct act, int use_weight) {
  constexpr bool GATED = MODE == MS_GATED, BY_TOKEN = MODE != MS_DOWN;
  constexpr int NT = WAVES / WK, NB = 16 * NT, MATS = GATED ? 2 : 1, L = 2 * MATS, CHUNK = 16 * MATS * MF_K;
  constexpr int FIT = KB * 1024 / (WAVES * CHUNK * 2), S = FIT < CW ? FIT : CW;
  __shared__ __attribute__((aligned(1024))) bf16_t bufs[WAVES][S * CHUNK];
  const int per_tile = (N + NB - 1) / NB, tile = blockIdx.x / per_tile;      // (neighbouring blocks: see the kernel above)
  const int tiles = meta[0], e = tile_expert[tile], row0 = tile_row0[tile];
  if (tile >= tiles) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, lq = lane >> 4;
  const int part = wave % WK, n0 = (blockIdx.x - tile * per_tile) * NB + wave / WK * 16;
  const int all = K / MF_K, first = all * part / WK, chunks = n0 < N ? all * (part + 1) / WK - first : 0;
  const bf16_t* src[L];      // an instruction brings 8 rows; piece c of row r lies at slot c ^ (r % 8); rows beyond the last repeat it
#pragma unroll
  for (int j = 0; j < L; ++j)
    src[j] = (j < 2 ? W0 : W1) + ((long long)e * N + min(n0 + (j & 1) * 8 + (lane >> 3), N - 1)) * K + first * MF_K + ((lane & 7) ^ (lane >> 3)) * 8;
  const unsigned lds0 = (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)bufs[wave];
  auto fetch = [&](int c, int slot) {
#pragma unroll
    for (int j = 0; j < L; ++j)
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src[j] + c * MF_K), "s"(lds0 + slot * (CHUNK * 2) + j * 1024) : "memory", "m0");
  };
#pragma unroll
  for (int c = 0; c < S; ++c)
    if (c < chunks) fetch(c, c);
  const int rows = min(MS_ROWS, offsets[e + 1] - row0), mine = row0 + min(li, rows - 1), s = order[mine], token = s / top;
  const float weight = use_weight ? weights[s] : 1.f;
  const bf16_t* xr = a_rows + (long long)(BY_TOKEN ? token : mine) * K + first * MF_K + lq * 8;
  ms_bf16x8 xf[CW][2];      // rows beyond the tile's are zeros: their lanes load nothing
#pragma unroll
  for (int c = 0; c < CW; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xf[c][h] = ms_bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
      if (li < rows && c < chunks) xf[c][h] = *(const ms_bf16x8*)(xr + c * MF_K + h * 32);
    }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int c = 0; c < CW; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(xf[c][h]));      // x is there: nothing below waits for it, and with it for W
  ms_f32x4 acc[MATS] = {};
#pragma unroll
  for (int c = 0; c < CW; ++c) {
    if (c >= chunks) break;
    if (c >= S) {      // chunk c was asked for with chunk c - S; S - 1 of those behind it may be on their way
      if (c + S - 1 < chunks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * L) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const bf16_t* b = bufs[wave] + c % S * CHUNK + li * MF_K;
    ms_bf16x8 wf[MATS][2];
#pragma unroll
    for (int t = 0; t < MATS; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) wf[t][h] = *(const ms_bf16x8*)(b + t * 16 * MF_K + (((h * 4 + lq) ^ li) & 7) * 8);
    if (c + S < chunks) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // read before the slot is filled again
      fetch(c + S, c % S);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < MATS; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][h], xf[c][h], acc[t], 0, 0, 0);
  }
  ms_f32x4* red = (ms_f32x4*)bufs;
  static_assert(MATS * 1024 <= S * CHUNK * 2, "the parts meet in the ring's place");
  __syncthreads();
#pragma unroll
  for (int t = 0; t < MATS; ++t) red[(t * WAVES + wave) * 64 + lane] = acc[t];
  __syncthreads();
  if (part) return;
  ms_f32x4 sum[MATS];
#pragma unroll
  for (int t = 0; t < MATS; ++t) {
    sum[t] = red[(t * WAVES + wave) * 64 + lane];
#pragma unroll
    for (int p = 1; p < WK; ++p) sum[t] += red[(t * WAVES + wave + p) * 64 + lane];
  }
  const int n = n0 + lq * 4;      // a lane holds outputs n .. n + 3 of row li; N is a multiple of 4
  if (li >= rows || n >= N) return;
  if (MODE == MS_DOWN) {
    float* y = (float*)out + ((long long)(s - token * top) * n_tokens + token) * N + n;
    *(ms_f32x4*)y = ms_f32x4{sum[0][0] * weight, sum[0][1] * weight, sum[0][2] * weight, sum[0][3] * weight};
  } else {
    typedef __bf16 ms_bf16x4 __attribute__((ext_vector_type(4)));
    ms_bf16x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = from_f32<bf16_t>(GATED ? jv_gated(act, sum[0][i] * weight, sum[MATS - 1][i] * weight) : jv_act(act.id, sum[0][i] * weight));
    *(ms_bf16x4*)((bf16_t*)out + (long long)(row0 + li) * N + n) = v;
  }
}

template <int MODE, int WAVES, int KB, int WK, int CW, typename... Args>
static int launch_moe_few(int max_tiles, int N, hipStream_t stream, Args... args) {
  const int nb = 16 * WAVES / WK;
  const long long blocks = (long long)max_tiles * ((N + nb - 1) / nb);
  if (blocks > 0x7fffffffll) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((moe_few_kernel<MODE, WAVES, KB, WK, CW>), dim3((unsigned)blocks), dim3(64 * WAVES), 0, stream, args...);
  return JV_LAUNCH_CHECK();
}

template <int MODE>
static int launch_moe_skinny(void* out, const void* a, const void* W0, const void* W1, const int* meta, const int* offsets,
                             const int* tile_expert, const int* tile_row0, const int* order, const float* weights,
                             int max_tiles, int top, int n_tokens, int K, int N, JvAct act, int use_weight, void* stream) {
  if (K < 8 || K % 8) return (int)hipErrorInvalidValue;
  if (K % MF_K == 0 && K <= 4096 && N % 4 == 0 && (((uintptr_t)out | (uintptr_t)a | (uintptr_t)W0 | (uintptr_t)W1) & 15) == 0) {
    auto go = [&](auto waves, auto kb, auto wk, auto cw) {
      return launch_moe_few<MODE, decltype(waves)::value, decltype(kb)::value, decltype(wk)::value, decltype(cw)::value>(
          max_tiles, N, (hipStream_t)stream, out, (const bf16_t*)a, (const bf16_t*)W0, (const bf16_t*)W1, meta, offsets, tile_expert,
          tile_row0, order, weights, top, n_tokens, K, N, act, use_weight);
    };
#define GO(WAVES, KB, WK, CW) \
  go(std::integral_constant<int, WAVES>{}, std::integral_constant<int, KB>{}, std::integral_constant<int, WK>{}, std::integral_constant<int, CW>{})
    if (K <= 512) return GO(4, 24, 2, 4);
    if (K <= 1024 && MODE == MS_GATED) return GO(8, 64, 4, 4);
    if (K <= 1024) return GO(4, 24, 2, 8);
    if (K <= 2048) return GO(8, 32, 8, 4);
    return GO(8, 64, 8, 8);
#undef GO
  }
  const int wk = K >= 2048 ? 4 : 2;
  auto kernel = wk == 4 ? moe_skinny_kernel<MODE, 4> : moe_skinny_kernel<MODE, 2>;
  const int nb = 64 / wk;
  const long long blocks = (long long)max_tiles * ((N + nb - 1) / nb);
  if (blocks > 0x7fffffffll) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, out, (const bf16_t*)a,
                     (const bf16_t*)W0, (const bf16_t*)W1, meta, offsets, tile_expert, tile_row0, order, weights, top,
                     n_tokens, K, N, act, use_weight);
  return JV_LAUNCH_CHECK();
}

extern "C" int jv_moe_skinny_rows() { return MS_ROWS; }

// gate/up: x [tokens, hidden], Wg, Wu [experts, ff, hidden] -> z [entries, ff] bf16 by position.  Wg null: experts
// without a gate, act one that stands alone.
extern "C" int jv_moe_gate_up_skinny_bf16(void* z, const void* x, const void* Wg, const void* Wu, const int* meta,
                                          const int* offsets, const int* tile_expert, const int* tile_row0,
                                          const int* order, const float* weights, int max_tiles, int top, int hidden,
                                          int ff, int act, float act_limit, float act_slope, int scale_input, void* stream) {
  if (max_tiles <= 0 || ff <= 0) return 0;
  if (!(Wg ? jv_act_known(act) : jv_plain_act_known(act))) return (int)hipErrorInvalidValue;
  if (Wg)
    return launch_moe_skinny<MS_GATED>(z, x, Wg, Wu, meta, offsets, tile_expert, tile_row0, order, weights, max_tiles, top,
                                       0, hidden, ff, JvAct{act, act_limit, act_slope}, scale_input, stream);
  return launch_moe_skinny<MS_PLAIN>(z, x, Wu, nullptr, meta, offsets, tile_expert, tile_row0, order, weights, max_tiles,
                                     top, 0, hidden, ff, JvAct{act, act_limit, act_slope}, scale_input, stream);
}

// down: z [entries, ff] by position, Wd [experts, hidden, ff] -> y [top, tokens, hidden] float
extern "C" int jv_moe_down_skinny_bf16(float* y, const void* z, const void* Wd, const int* meta, const int* offsets,
                                       const int* tile_expert, const int* tile_row0, const int* order,
                                       const float* weights, int max_tiles, int top, int n_tokens, int hidden, int ff,
                                       int scale_output, void* stream) {
  if (max_tiles <= 0 || hidden <= 0) return 0;
  return launch_moe_skinny<MS_DOWN>(y, z, Wd, nullptr, meta, offsets, tile_expert, tile_row0, order, weights, max_tiles,
                                    top, n_tokens, ff, hidden, JvAct{}, scale_output, stream);
}
