// y[M,N] = x[M,K] W[N,K]^T for 17 to 128 rows, bf16 in, float sums: the product of a decode step of many requests and of a
// short prompt, bound by the stream of W.
//
// A block takes all rows of x (TM = 32, 64 or 128) against TW rows of W, over its share of the inner size (gridDim.y blocks
// share it out, as float partial products that the reader adds in order).  Chunks of 64 columns of both go straight from
// memory into a ring in LDS that fills the compute unit (one block a unit, 4 to 8 chunks = 100 to 130 KB on their way
// without a register held for them); a wave multiplies one 32 x 32 tile, v_mfma_f32_32x32x16_bf16 with A = rows of W, B = rows
// of x.  N is cut so that every unit has one block: x is then read 256 times from the L2s, W once from memory.
//
// Blocks begin at different chunks and walk round (by their number on their XCD, which takes every eighth block): in
// lockstep all units would ask for the same 128-byte columns of rows that lie a power of two apart, which few channels
// hold (24,576 x 4,096 at 64 rows: 50.6 us in lockstep, 40.2 so).  In one form (rows of x, rows of W, shares) which
// chunk comes first depends on the columns of y alone, so a row's result does not depend on the other rows; the form is
// chosen by their number.
//
// Measured at 64 rows, microseconds (before; a plain read of W): 24,576 x 4,096 with its activation 40.2 (52.3; 33.6),
// 4,096 x 12,288 25.5 (32.8; 16.8), 4,096 x 4,096 11.6 (13.4; 5.6), 6,144 x 4,096 14.0 (17.6; 8.4); at 128 rows 46.9 (57.1),
// 33.8 (67.7), 14.5 (24.5), 17.7 (25.9); before: the library, blocks of 64 rows of W through registers (gemm_tile64), or
// blocks that stay with x in registers.
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define ST_K 64            // columns of a chunk: a row of it is 128 bytes, 8 pieces of 16
#define ST_LDS (155 * 1024)

// ST_PARTS: float partial products [gridDim.y][M][N]; ST_BF16: bf16 [M][N]; ST_PAIRS: rows of W alternate gate and up rows,
// act(gate) * up in bf16 [M][N / 2]
enum { ST_PARTS = 0, ST_BF16 = 1, ST_PAIRS = 2 };

// Rows of x whose norm's scale is still to be applied (add_parts_unscaled_kernel): row m of the result is multiplied by
// rsqrt(sum_j ssq[m * 16 + j] inv_width + eps), j < shares.
struct StScale {
  const float* ssq;
  int shares;
  float inv_width, eps;
};

constexpr int st_loads(int total, int waves) {      // loads of a wave: the fewest that share `total` out to whole waves
  int n = (total + waves - 1) / waves;
  while (total % n) ++n;
  return n;
}

template <int MODE, int TM, int TW, bool SCALED>
__global__ void __launch_bounds__(64 * (TM / 32) * (TW / 32))
gemm_stream_kernel(void* __restrict__ y, const bf16_t* __restrict__ x, const bf16_t* __restrict__ W, int M, int N, int K,
                   long long ldx, JvAct act, StScale scale) {
  constexpr int WN = TW / 32, WAVES = TM / 32 * WN, ROWS = TM + TW;
  constexpr int LPW = st_loads(ROWS / 8, WAVES), LOADERS = ROWS / 8 / LPW;
  constexpr int FIT = ST_LDS / (ROWS * ST_K * 2), BUFS = FIT < 9 ? FIT : 9;
  static_assert((BUFS - 2) * LPW <= 63, "what s_waitcnt counts to");
  __shared__ __attribute__((aligned(1024))) bf16_t bufs[BUFS * ROWS * ST_K];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * TW;
  const int all = K / ST_K, c0 = (int)((long long)all * blockIdx.y / gridDim.y), chunks = (int)((long long)all * (blockIdx.y + 1) / gridDim.y) - c0;
  const int rot = (int)((blockIdx.x >> 3) * 2 % chunks);
  // An instruction brings 8 rows, lane l row l / 8, and fills 1 KB in the order of the lanes; piece c of row r lies at slot
  // c ^ ((r / 2) % 8) of its row, so that 16 lanes reading one piece of 16 rows meet 16 slots.  Rows beyond the last repeat it.
  const bf16_t* src[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int r = (wave * LPW + j) * 8 + (lane >> 3);       // row of the buffer: rows of x, then rows of W
    const int piece = ((lane & 7) ^ (r >> 1)) & 7;
    const bf16_t* row = r < TM ? x + (long long)min(r, M - 1) * ldx : W + (long long)min(n0 + r - TM, N - 1) * K;
    src[j] = row + piece * 8 + (long long)c0 * ST_K;
  }
  auto fetch = [&](int c, int buf) {
    if (wave >= LOADERS) return;
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
      const bf16_t* from = src[j] + (c + rot < chunks ? c + rot : c + rot - chunks) * ST_K;
      const unsigned at = (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)(bufs + (buf * ROWS + (wave * LPW + j) * 8) * ST_K);
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "s"(at) : "memory", "m0");
    }
  };
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  const int wm = wave / WN, wn = wave - wm * WN, l32 = lane & 31, half = lane >> 5, swz = (l32 >> 1) & 7;
  // a lane's row of the result: its shares, eight in either half of the wave, asked for before everything else
  f32x4 sq[SCALED ? 2 : 1];
  if constexpr (SCALED) {
#pragma unroll
    for (int i = 0; i < 2; ++i) sq[i] = *(const f32x4*)(scale.ssq + (long long)min(wm * 32 + l32, M - 1) * 16 + half * 8 + i * 4);
  }
  for (int c = 0; c < BUFS - 1 && c < chunks; ++c) fetch(c, c);
  for (int c = 0, buf = 0; c < chunks; ++c, buf = buf + 1 == BUFS ? 0 : buf + 1) {
    // this wave's part of chunk c is there (loads arrive in order; those of the next BUFS - 2 chunks may be on their way)
    if (c + BUFS - 2 < chunks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((BUFS - 2) * LPW) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                            // and everybody's, and the buffer before is no longer read
    if (c + BUFS - 1 < chunks) fetch(c + BUFS - 1, buf == 0 ? BUFS - 1 : buf - 1);
    const bf16_t* xb = bufs + (buf * ROWS + wm * 32 + l32) * ST_K;
    const bf16_t* wb = bufs + (buf * ROWS + TM + wn * 32 + l32) * ST_K;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int at = ((ks * 2 + half) ^ swz) * 8;
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(wb + at), *(const bf16x8*)(xb + at), acc, 0, 0, 0);
    }
  }
  // a lane holds row l32 of the wave's rows of x, columns 8 q + 4 half + e of its rows of W
  const int m = wm * 32 + l32;
  if constexpr (SCALED) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) t += half * 8 + i * 4 + e < scale.shares ? sq[i][e] : 0.f;
    t += __shfl_xor(t, 32, 64);
    acc *= rsqrtf(t * scale.inv_width + scale.eps);
  }
  if (m >= M) return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int n = n0 + wn * 32 + q * 8 + half * 4;
    if (n >= N) continue;                       // N is a multiple of 4
    if (MODE == ST_PARTS) {
      *(f32x4*)((float*)y + ((long long)blockIdx.y * M + m) * N + n) = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    } else if (MODE == ST_BF16) {
      typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = from_f32<bf16_t>(acc[4 * q + e]);
      *(bf16x4*)((bf16_t*)y + (long long)m * N + n) = v;
    } else {
      typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
      bf16x2 v;
#pragma unroll
      for (int e = 0; e < 2; ++e) v[e] = from_f32<bf16_t>(jv_gated(act, acc[4 * q + 2 * e], acc[4 * q + 2 * e + 1]));
      *(bf16x2*)((bf16_t*)y + (long long)m * (N / 2) + n / 2) = v;
    }
  }
}

template <int MODE, int TM, int TW>
static int st_launch(void* y, const void* x, const void* W, int M, int N, int K, long long ldx, int ksplit, JvAct act, StScale scale, hipStream_t s) {
  const auto kernel = scale.ssq ? gemm_stream_kernel<MODE, TM, TW, true> : gemm_stream_kernel<MODE, TM, TW, false>;
  hipLaunchKernelGGL(kernel, dim3((N + TW - 1) / TW, ksplit), dim3(2 * TM / 32 * TW), 0, s, y, (const bf16_t*)x, (const bf16_t*)W, M, N, K, ldx, act, scale);
  return JV_LAUNCH_CHECK();
}
template <int MODE, int TM>
static int st_tw(int tw, void* y, const void* x, const void* W, int M, int N, int K, long long ldx, int ksplit, JvAct act, StScale scale, hipStream_t s) {
  switch (tw) {
    case 32: return st_launch<MODE, TM, 32>(y, x, W, M, N, K, ldx, ksplit, act, scale, s);
    case 64: return st_launch<MODE, TM, 64>(y, x, W, M, N, K, ldx, ksplit, act, scale, s);
    case 96: return st_launch<MODE, TM, 96>(y, x, W, M, N, K, ldx, ksplit, act, scale, s);
    case 128: return st_launch<MODE, TM, 128>(y, x, W, M, N, K, ldx, ksplit, act, scale, s);
  }
  return (int)hipErrorInvalidValue;
}
template <int MODE>
static int st_tm(int tm, int tw, void* y, const void* x, const void* W, int M, int N, int K, long long ldx, int ksplit, JvAct act, StScale scale, hipStream_t s) {
  switch (tm) {
    case 32: return st_tw<MODE, 32>(tw, y, x, W, M, N, K, ldx, ksplit, act, scale, s);
    case 64: return st_tw<MODE, 64>(tw, y, x, W, M, N, K, ldx, ksplit, act, scale, s);
    case 128: return st_tw<MODE, 128>(tw, y, x, W, M, N, K, ldx, ksplit, act, scale, s);
  }
  return (int)hipErrorInvalidValue;
}
// ssq (rows of 16 floats, `shares` of them) or null: the scale of the norm over `width` columns is applied to the rows.
// mode: ST_*; tm (32, 64, 128; at least M) and tw (32, 64, 96, 128): rows of x and of W of a block; ksplit > 1: ST_PARTS only.
extern "C" int jv_gemm_stream_bf16(void* y, const void* x, const void* W, int M, int N, int K, long long ldx, int mode, int gate_act,
                                   float act_limit, float act_slope, int tm, int tw, int ksplit, const float* ssq, int shares, int width,
                                   float eps, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (ssq && (shares < 1 || shares > 16 || width <= 0 || ((uintptr_t)ssq & 15))) return (int)hipErrorInvalidValue;
  if (M > tm || K < ST_K || K % ST_K || N % 4 || ldx % 8 || ksplit < 1 || ksplit > K / ST_K || (ksplit > 1 && mode != ST_PARTS) ||
      (((uintptr_t)x | (uintptr_t)W | (uintptr_t)y) & 15))
    return (int)hipErrorInvalidValue;
  if (mode == ST_PAIRS && !jv_act_known(gate_act)) return (int)hipErrorInvalidValue;
  const JvAct act{gate_act, act_limit, act_slope};
  const StScale scale{ssq, shares, ssq ? 1.f / (float)width : 0.f, eps};
  const hipStream_t s = (hipStream_t)stream;
  switch (mode) {
    case ST_PARTS: return st_tm<ST_PARTS>(tm, tw, y, x, W, M, N, K, ldx, ksplit, act, scale, s);
    case ST_BF16: return st_tm<ST_BF16>(tm, tw, y, x, W, M, N, K, ldx, ksplit, act, scale, s);
    case ST_PAIRS: return st_tm<ST_PAIRS>(tm, tw, y, x, W, M, N, K, ldx, ksplit, act, scale, s);
  }
  return (int)hipErrorInvalidValue;
}
