// y[M,N] = x[M,K] W[N,K]^T for up to 16 rows of x and matrices too small for blocks that stay (gemm_skinny.hip): bf16 in, float
// sums, bf16 or float out, or the activation of pairs of rows of W as an epilogue.
//
// Bound by the stream of W and what stands before it: a matrix of 25 MB is read in 4.6 us, and every round trip to memory that a
// block waits for in a row costs one more.  So a block takes TW rows of W against all rows of x and its 8 waves an eighth of the
// inner size each; a wave asks for its part of x (into registers, where it stays) and for the first S chunks of its part of W
// (straight into a ring of its own in LDS) in one go, and no wave waits for another before the parts meet at the end.  Two blocks
// with rings of up to 64 KB share a unit; up to 512 blocks are on the chip at once, and their units need not carry equal loads, for
// what they share is the memory.  TW follows from where more are a further round (few_tile, with the figures).  The parts are added
// in ascending order, so a row's result does not depend on the others.
//
// Microseconds in a graph, cold weights, at 1, 8 and 16 rows (before, x staged chunk by chunk in LDS for all waves of a block): 1,536 x 768 2.9, 3.2, 3.4 (4.6,
// 5.0, 6.2).  Given rows of longer inner sizes, and many of shorter ones, go through gemm_thin.hip, to the same bits (thin_slots has the figures of both): given
// rows are taken up to 1,024 columns here, two chunks a wave, rows that the blocks make up to 4,096.
#include "common.h"
#include "row_source.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { FEW_BF16 = 0, FEW_F32 = 1, FEW_PAIRS = 2 };

#define FEW_K 64           // columns of a chunk: a row of it is 128 bytes, 8 pieces of 16
#define FEW_WAVES 8

// CW: the most chunks of a wave.  SRC (row_source.h): the block makes its MR rows of x itself and scales them; K is then KX columns.
template <int MODE, int TW, int CW, int SRC = ROWS_GIVEN, int MR = 1, int KX = 64>
__global__ void __launch_bounds__(64 * FEW_WAVES)
gemm_few_kernel(void* __restrict__ y, const bf16_t* __restrict__ x, const bf16_t* __restrict__ W, int M, int N, int K, long long ldx, JvAct act,
                RowSource src_rows) {
  constexpr int NT = TW / 16, L = TW / 8, CHUNK = TW * FEW_K, S = 64 * 1024 / (FEW_WAVES * CHUNK * 2) < CW ? 64 * 1024 / (FEW_WAVES * CHUNK * 2) : CW;
  static_assert(NT * 1024 <= S * CHUNK * 2, "the parts meet in the ring's place");
  __shared__ __attribute__((aligned(1024))) bf16_t bufs[FEW_WAVES][S * CHUNK];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, lq = lane >> 4;
  // Two blocks a unit: two made rows of 4,096 columns fill what the ring leaves of half its LDS to the byte, so they have no gap between them
  // and their sums of squares wait in registers for the ring's place.  With 96 bytes more, one block a unit, 12,288 x 4,096 at two rows took 28.3 us
  // (rows given, and made by a launch before: 25.7).
  constexpr int XSTRIDE = MR * KX > 4096 ? KX : KX + 8;
  __shared__ __attribute__((aligned(16))) bf16_t xmade[SRC == ROWS_GIVEN ? 8 : MR * XSTRIDE];
  static_assert(sizeof(bufs) + (SRC == ROWS_GIVEN ? 0 : sizeof(xmade)) <= 80 * 1024, "");
  float made_sq[MR];
  RowMaker<SRC, MR, KX> maker;
  if constexpr (SRC != ROWS_GIVEN) {
    maker.ask(src_rows, 0, K);
    __builtin_amdgcn_sched_barrier(0);
  }
  const int n0 = blockIdx.x * TW, all = K / FEW_K;
  const int first = all * wave / FEW_WAVES, chunks = all * (wave + 1) / FEW_WAVES - first;
  // an instruction brings 8 rows, lane l row l / 8, and fills 1 KB in the order of the lanes; piece c of row r lies at slot
  // c ^ (r % 8) of its row.  Rows beyond the last repeat it.
  const bf16_t* src[L];
#pragma unroll
  for (int j = 0; j < L; ++j)
    src[j] = W + (long long)min(n0 + j * 8 + (lane >> 3), N - 1) * K + first * FEW_K + ((lane & 7) ^ (lane >> 3)) * 8;
  const unsigned lds0 = (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)bufs[wave];
  auto fetch = [&](int c, int slot) {
#pragma unroll
    for (int j = 0; j < L; ++j)
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src[j] + c * FEW_K), "s"(lds0 + slot * (CHUNK * 2) + j * 1024) : "memory", "m0");
  };
#pragma unroll
  for (int c = 0; c < S; ++c)
    if (c < chunks) fetch(c, c);
  // rows of x beyond the last are zeros: their lanes load nothing
  bf16x8 xf[CW][2];
  if constexpr (SRC == ROWS_GIVEN) {
    const bf16_t* xr = x + (long long)min(li, M - 1) * ldx + first * FEW_K + lq * 8;
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        xf[c][h] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
        if (li < M && c < chunks) xf[c][h] = *(const bf16x8*)(xr + c * FEW_K + h * 32);
      }
  } else {
    maker.give(src_rows, 0, K, blockIdx.x == 0, xmade, XSTRIDE, made_sq);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        xf[c][h] = c < chunks ? *(const bf16x8*)(xmade + min(li, MR - 1) * XSTRIDE + (first + c) * FEW_K + h * 32 + lq * 8) : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int c = 0; c < CW; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(xf[c][h]));      // x is there: nothing below waits for it, and with it for W
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < CW; ++c) {
    if (c >= chunks) break;
    if (c >= S) {      // chunk c was asked for with chunk c - S; S - 1 of those behind it may be on their way
      if (c + S - 1 < chunks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * L) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    const bf16_t* b = bufs[wave] + c % S * CHUNK + li * FEW_K;
    bf16x8 wf[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) wf[t][h] = *(const bf16x8*)(b + t * 16 * FEW_K + (((h * 4 + lq) ^ li) & 7) * 8);
    if (c + S < chunks) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // read before the slot is filled again
      fetch(c + S, c % S);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][h], xf[c][h], acc[t], 0, 0, 0);
  }
  __syncthreads();
  f32x4* red = (f32x4*)bufs;
#pragma unroll
  for (int t = 0; t < NT; ++t) red[(t * FEW_WAVES + wave) * 64 + lane] = acc[t];
  float* const row_sq = (float*)(red + NT * FEW_WAVES * 64);      // [MR][FEW_WAVES]
  if constexpr (SRC != ROWS_GIVEN) {
    static_assert(NT * FEW_WAVES * 1024 + MR * FEW_WAVES * 4 <= sizeof(bufs), "");
#pragma unroll
    for (int m = 0; m < MR; ++m)
      if (lane == 0) row_sq[m * FEW_WAVES + wave] = made_sq[m];
  }
  __syncthreads();
  if (wave >= NT) return;
  f32x4 sum = red[wave * FEW_WAVES * 64 + lane];
#pragma unroll
  for (int p = 1; p < FEW_WAVES; ++p) sum += red[(wave * FEW_WAVES + p) * 64 + lane];
  if (SRC == ROWS_RESIDUAL) {
    float sq = 0.f;
#pragma unroll
    for (int w = 0; w < FEW_WAVES; ++w) sq += row_sq[min(li, MR - 1) * FEW_WAVES + w];
    sum *= rsqrtf(sq * src_rows.inv_width + src_rows.eps);
  }
  const int m = li, n = n0 + wave * 16 + lq * 4;      // a lane holds y[m][n .. n + 3]; N is a multiple of 4
  if (m >= M || n >= N) return;
  if (MODE == FEW_F32) {
    *(f32x4*)((float*)y + (long long)m * N + n) = sum;
  } else if (MODE == FEW_BF16) {
    bf16x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = from_f32<bf16_t>(sum[e]);
    *(bf16x4*)((bf16_t*)y + (long long)m * N + n) = v;
  } else {
    bf16x2 v;
#pragma unroll
    for (int e = 0; e < 2; ++e) v[e] = from_f32<bf16_t>(jv_gated(act, sum[2 * e], sum[2 * e + 1]));
    *(bf16x2*)((bf16_t*)y + (long long)m * (N / 2) + n / 2) = v;
  }
}

template <int MODE, int TW>
static int few_launch(void* y, const void* x, const void* W, int M, int N, int K, long long ldx, JvAct act, hipStream_t s) {
  hipLaunchKernelGGL((gemm_few_kernel<MODE, TW, 2>), dim3((N + TW - 1) / TW), dim3(64 * FEW_WAVES), 0, s, y, (const bf16_t*)x, (const bf16_t*)W, M, N, K, ldx, act,
                     RowSource{});
  return JV_LAUNCH_CHECK();
}
// mode: FEW_*; tw (16, 32): rows of W of a block.
extern "C" int jv_gemm_few_bf16(void* y, const void* x, const void* W, int M, int N, int K, long long ldx, int mode, int gate_act,
                                float act_limit, float act_slope, int tw, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || K < FEW_K || K > 2 * FEW_WAVES * FEW_K || K % FEW_K || N % 4 || ldx % 8 || (((uintptr_t)x | (uintptr_t)W | (uintptr_t)y) & 15))
    return (int)hipErrorInvalidValue;
  if (mode == FEW_PAIRS && !jv_act_known(gate_act)) return (int)hipErrorInvalidValue;
  const JvAct act{gate_act, act_limit, act_slope};
  const hipStream_t s = (hipStream_t)stream;
  if (mode == FEW_BF16) return tw == 16 ? few_launch<FEW_BF16, 16>(y, x, W, M, N, K, ldx, act, s) : few_launch<FEW_BF16, 32>(y, x, W, M, N, K, ldx, act, s);
  if (mode == FEW_F32) return tw == 16 ? few_launch<FEW_F32, 16>(y, x, W, M, N, K, ldx, act, s) : few_launch<FEW_F32, 32>(y, x, W, M, N, K, ldx, act, s);
  if (mode == FEW_PAIRS) return tw == 16 ? few_launch<FEW_PAIRS, 16>(y, x, W, M, N, K, ldx, act, s) : few_launch<FEW_PAIRS, 32>(y, x, W, M, N, K, ldx, act, s);
  return (int)hipErrorInvalidValue;
}

// y = (norm of h + parts) W^T for one or two rows that the blocks make themselves: bf16 [M][N], or with gate_act [M][N / 2].  h_out takes h + parts.
template <int MODE, int TW, int KX>
static int few_made(void* y, const void* W, int M, int N, JvAct act, const RowSource& src, hipStream_t s) {
  constexpr int CW = (KX / FEW_K + FEW_WAVES - 1) / FEW_WAVES;
  if (M == 1)
    hipLaunchKernelGGL((gemm_few_kernel<MODE, TW, CW, ROWS_RESIDUAL, 1, KX>), dim3((N + TW - 1) / TW), dim3(64 * FEW_WAVES), 0, s, y, (const bf16_t*)W,
                       (const bf16_t*)W, M, N, KX, (long long)KX, act, src);
  else
    hipLaunchKernelGGL((gemm_few_kernel<MODE, TW, CW, ROWS_RESIDUAL, 2, KX>), dim3((N + TW - 1) / TW), dim3(64 * FEW_WAVES), 0, s, y, (const bf16_t*)W,
                       (const bf16_t*)W, M, N, KX, (long long)KX, act, src);
  return JV_LAUNCH_CHECK();
}
extern "C" int jv_gemm_few_residual_bf16(void* y, const float* h, float* h_out, const float* parts, int n_parts, long long part_stride, const float* weight,
                                         float eps, const void* W, int M, int N, int K, int gate_act, float act_limit, float act_slope, int tw, void* stream) {
  if (M < 1 || M > 2 || N <= 0 || N % 4 || n_parts < 0 || n_parts > 4 || (n_parts && !parts) || h == h_out || (gate_act && !jv_act_known(gate_act)) ||
      (((uintptr_t)W | (uintptr_t)y) & 15))
    return (int)hipErrorInvalidValue;
  RowSource src{};
  src.h = h; src.h_out = h_out; src.parts = parts; src.n_parts = n_parts; src.part_stride = part_stride; src.weight = weight;
  src.inv_width = 1.f / (float)K; src.eps = eps;
  const JvAct act{gate_act, act_limit, act_slope};
  const hipStream_t s = (hipStream_t)stream;
#define FEW_MADE(KX)                                                                                                                   \
  if (K == KX)                                                                                                                         \
    return gate_act ? (tw == 16 ? few_made<FEW_PAIRS, 16, KX>(y, W, M, N, act, src, s) : few_made<FEW_PAIRS, 32, KX>(y, W, M, N, act, src, s)) \
                    : (tw == 16 ? few_made<FEW_BF16, 16, KX>(y, W, M, N, act, src, s) : few_made<FEW_BF16, 32, KX>(y, W, M, N, act, src, s));
  FEW_MADE(1024) FEW_MADE(2048) FEW_MADE(4096)
#undef FEW_MADE
  return (int)hipErrorInvalidValue;
}
