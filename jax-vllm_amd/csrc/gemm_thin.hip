// y[M,N] = x[M,K] W[N,K]^T for up to 16 rows of x, a block of four waves to 16 rows of W: bf16 in, float sums.  Out: bf16, float, the
// activation of pairs of rows of W, or the residual stream itself with what the next norm's reader needs.
//
// Bound by the stream of W and by what stands before it.  Each wave takes a quarter of the inner size through a ring of its own in LDS, chunks
// of 64 columns of W's rows AND of x, in the order in which they are multiplied: nothing of x is held in registers, so a wave waits for its oldest
// chunk only, never for x, and the inner size is free.  Blocks are small (24 or 48 KB of LDS at up to 8 rows): three to six share a unit, and
// one begins while another ends.  Every row of x is read by every block, from the L2: half of W's bytes on top at 8 rows.  Slots of the ring: 4
// while every unit has one block at most and beyond 1,024 blocks, 2 between, where more blocks at once count for more (microseconds at 8 rows by 4 / 2
// slots, before: 4,096 x 4,096 8.0 / 8.4, 9.4; 2,048 x 2,048 4.6 / 4.9, 5.1; 6,144 x 2,048 with its activation 8.0 / 7.2, 8.2; 8,192 x 2,048
// 8.4 / 8.0, 9.6; 12,288 x 4,096 19.2 / 19.4, 22.7; 8 waves 4,096 x 4,096 8.8, two waves of 8 slots 9.0).  Every wave makes two sums, of an eighth of
// the inner size each, and the eighths are added in ascending order: the bits of gemm_few.hip, whatever the other rows, the slots and the tiles.
// A chunk of more than 8 rows of x is as large as one of 16 rows of W, so a block then takes 32 of them where that leaves no unit more (16 rows, one tile / two:
// 6,144 x 4,096 13.4 / 11.7, 8,192 x 2,048 9.5 / 8.6, 24,576 x 4,096 41.4 / 36.5).
//
// THIN_STREAM: the product joins the residual stream h in place (a block owns its columns of it), and the block leaves the new rows times the next
// norm's weight in bf16 and its share of every row's sum of squares; the scale is left to the product that reads them (SCALED: its epilogue, up to
// 256 shares a row, asked for before everything else).  Against float parts and a launch that adds them, microseconds at 1, 8 and 16
// rows: 4,096 x 4,096 7.7, 8.1, 8.8 (10.6, 11.0, 11.5), x 12,288 19.8, 20.6, 23.6 (22.3, 23.1, 24.3), 2,048 x 2,048 4.6, 4.8, 5.3 (6.2, 6.5, 6.9),
// x 3,072 5.2, 5.9, 6.9 (7.8, 8.4, 9.1).
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { THIN_BF16 = 0, THIN_F32 = 1, THIN_PAIRS = 2, THIN_STREAM = 3 };

#define THIN_K 64          // columns of a chunk: a row of it is 128 bytes, 8 pieces of 16
#define THIN_WAVES 4
#define THIN_SHARES 256    // of a row's sum of squares: floats of a row of ssq

struct ThinScale {         // rows of x come times their norm's weight; out row m is multiplied by rsqrt(sum_j ssq[m][j] inv_width + eps), j < shares
  const float* ssq;
  int shares;
  float inv_width, eps;
};
struct ThinStream {        // THIN_STREAM, beside h in y's place
  const float* weight;     // of the next norm, or null: the stream alone
  bf16_t* rows;
  float* ssq;
};

// XL: instructions (of 8 rows) that bring a chunk of x; S: slots of the ring; NT: tiles of 16 rows of W a block takes (THIN_STREAM: one).
template <int MODE, bool SCALED, int XL, int S, int NT>
__global__ void __launch_bounds__(64 * THIN_WAVES)
gemm_thin_kernel(void* __restrict__ y, const bf16_t* __restrict__ x, const bf16_t* __restrict__ W, int M, int N, int K, long long ldx, JvAct act,
                 ThinScale scale, ThinStream stream) {
  constexpr int WL = 2 * NT, L = WL + XL, CHUNK = L * 8 * THIN_K, PER = 16 / THIN_WAVES;
  static_assert(MODE != THIN_STREAM || NT == 1, "a share of a row is 16 columns");
  __shared__ __attribute__((aligned(1024))) bf16_t bufs[THIN_WAVES][S * CHUNK];
  __shared__ float sq_part[THIN_WAVES][16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, lq = lane >> 4;
  const int n0 = blockIdx.x * (16 * NT), all = K / THIN_K;
  const int first = all * wave / THIN_WAVES, chunks = all * (wave + 1) / THIN_WAVES - first, last = max(chunks - 1, 0);
  // an instruction brings 8 rows, lane l row l / 8, and fills 1 KB in the order of the lanes; piece c of row r lies at slot c ^ (r % 8) of
  // its row.  Rows beyond the last repeat it, chunks beyond a wave's last too (into slots that nobody reads).
  const int piece = first * THIN_K + ((lane & 7) ^ (lane >> 3)) * 8;
  const bf16_t* src[L];
#pragma unroll
  for (int j = 0; j < WL; ++j) src[j] = W + (long long)min(n0 + j * 8 + (lane >> 3), N - 1) * K + piece;
#pragma unroll
  for (int j = 0; j < XL; ++j) src[WL + j] = x + (long long)min(j * 8 + (lane >> 3), M - 1) * ldx + piece;
  const unsigned lds0 = (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)bufs[wave];
  auto fetch = [&](int c, int slot) {
#pragma unroll
    for (int j = 0; j < L; ++j)
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src[j] + c * THIN_K), "s"(lds0 + slot * (CHUNK * 2) + j * 1024) : "memory", "m0");
  };
  const int m = li, n = n0 + (NT > 1 ? wave * 16 : 0) + lq * 4;      // at the end a lane of wave t < NT holds y[m][n .. n + 3]; N is a multiple of 4
  const int mc = min(m, M - 1), nc = min(n, N - 4);
  // what the epilogue reads is asked for first, so that it costs no round trip of its own at the end
  f32x4 hv = {0.f, 0.f, 0.f, 0.f}, wv = {0.f, 0.f, 0.f, 0.f}, rq[SCALED ? PER : 1];
  if constexpr (MODE == THIN_STREAM) {
    hv = *(const f32x4*)((const float*)y + (long long)mc * N + nc);
    wv = *(const f32x4*)((stream.weight ? stream.weight : (const float*)y) + nc);
  }
  if constexpr (SCALED) {
#pragma unroll
    for (int i = 0; i < PER; ++i)
      rq[i] = *(const f32x4*)(scale.ssq + (long long)mc * THIN_SHARES + min((wave * PER + i) * 16 + lq * 4, scale.shares - 4));
  }
#pragma unroll
  for (int c = 0; c < S; ++c) fetch(min(c, last), c);
  const int second = all * (2 * wave + 1) / (2 * THIN_WAVES) - first;      // the chunk with which the wave's second eighth begins
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[NT], acc0[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = acc0[t] = zero;
  auto next_eighth = [&]() {
#pragma unroll
    for (int t = 0; t < NT; ++t) acc0[t] = acc[t], acc[t] = zero;
  };
  for (int c0 = 0; c0 < chunks; c0 += S) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (c0 + s >= chunks) break;
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * L) : "memory");      // the oldest chunk is there, S - 1 are on their way
      const bf16_t* b = bufs[wave] + s * CHUNK;
      bf16x8 wf[NT][2], xf[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int at = (((h * 4 + lq) ^ li) & 7) * 8;
#pragma unroll
        for (int t = 0; t < NT; ++t) wf[t][h] = *(const bf16x8*)(b + (t * 16 + li) * THIN_K + at);
        xf[h] = *(const bf16x8*)(b + (16 * NT + (XL == 1 ? li & 7 : li)) * THIN_K + at);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // read before the slot is filled again
      fetch(min(c0 + s + S, last), s);
      if (c0 + s == second) next_eighth();
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][h], xf[h], acc[t], 0, 0, 0);
    }
  }
  if (second >= chunks) next_eighth();
  if constexpr (SCALED) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) t += (wave * PER + i) * 16 + lq * 4 < scale.shares ? (rq[i][0] + rq[i][1]) + (rq[i][2] + rq[i][3]) : 0.f;
    t += __shfl_xor(t, 16, 64);
    t += __shfl_xor(t, 32, 64);
    if (lq == 0) sq_part[wave][li] = t;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // nothing of the ring is still being filled where the sums meet
  __syncthreads();
  f32x4* red = (f32x4*)bufs;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    red[(2 * wave * NT + t) * 64 + lane] = acc0[t];
    red[((2 * wave + 1) * NT + t) * 64 + lane] = acc[t];
  }
  __syncthreads();
  if (wave >= NT) return;
  f32x4 sum = red[wave * 64 + lane];
#pragma unroll
  for (int p = 1; p < 2 * THIN_WAVES; ++p) sum += red[(p * NT + wave) * 64 + lane];
  if constexpr (SCALED) {
    float t = 0.f;
#pragma unroll
    for (int p = 0; p < THIN_WAVES; ++p) t += sq_part[p][li];
    sum *= rsqrtf(t * scale.inv_width + scale.eps);
  }
  if constexpr (MODE == THIN_STREAM) {
    const f32x4 v = hv + sum;
    float sq = n < N ? (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]) : 0.f;
    sq += __shfl_xor(sq, 16, 64);
    sq += __shfl_xor(sq, 32, 64);
    if (m >= M) return;
    if (stream.weight && lq == 0) stream.ssq[(long long)m * THIN_SHARES + blockIdx.x] = sq;
    if (n >= N) return;
    *(f32x4*)((float*)y + (long long)m * N + n) = v;
    if (!stream.weight) return;
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = from_f32<bf16_t>(v[e] * wv[e]);
    *(bf16x4*)(stream.rows + (long long)m * N + n) = o;
    return;
  }
  if (m >= M || n >= N) return;
  if constexpr (MODE == THIN_F32) {
    *(f32x4*)((float*)y + (long long)m * N + n) = sum;
  } else if constexpr (MODE == THIN_BF16) {
    bf16x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = from_f32<bf16_t>(sum[e]);
    *(bf16x4*)((bf16_t*)y + (long long)m * N + n) = v;
  } else if constexpr (MODE == THIN_PAIRS) {
    bf16x2 v;
#pragma unroll
    for (int e = 0; e < 2; ++e) v[e] = from_f32<bf16_t>(jv_gated(act, sum[2 * e], sum[2 * e + 1]));
    *(bf16x2*)((bf16_t*)y + (long long)m * (N / 2) + n / 2) = v;
  }
}

template <int MODE, bool SCALED, int NT = 1>
static int thin_launch(void* y, const void* x, const void* W, int M, int N, int K, long long ldx, int slots, JvAct act, ThinScale scale, ThinStream stream,
                       hipStream_t st) {
#define THIN(XL, S)                                                                                                                      \
  hipLaunchKernelGGL((gemm_thin_kernel<MODE, SCALED, XL, S, NT>), dim3((N + 16 * NT - 1) / (16 * NT)), dim3(64 * THIN_WAVES), 0, st, y, (const bf16_t*)x, \
                     (const bf16_t*)W, M, N, K, ldx, act, scale, stream)
  if constexpr (NT == 2) {                     // two tiles: more than 8 rows, rings of two slots
    if (slots != 2 || M <= 8) return (int)hipErrorInvalidValue;
    THIN(2, 2);
  } else if (slots == 4) {
    if (M <= 8) THIN(1, 4); else THIN(2, 4);
  } else if constexpr (MODE != THIN_STREAM) {
    if (slots != 2) return (int)hipErrorInvalidValue;
    if (M <= 8) THIN(1, 2); else THIN(2, 2);
  } else
    return (int)hipErrorInvalidValue;
#undef THIN
  return JV_LAUNCH_CHECK();
}
static bool thin_sizes(const void* y, const void* x, const void* W, int M, int N, int K, long long ldx) {
  return M <= 16 && K >= THIN_K && K % THIN_K == 0 && N % 4 == 0 && ldx >= K && ldx % 8 == 0 && !(((uintptr_t)x | (uintptr_t)W | (uintptr_t)y) & 15);
}
// mode: THIN_BF16, THIN_F32 or THIN_PAIRS; slots (2, 4) of a wave's ring; tiles (1, 2; two for 9 rows and more, with two slots) of 16 rows of W of a block; ssq (rows of
// 256 floats, shares of them, a multiple of 4; float sums and activations only) or null.
extern "C" int jv_gemm_thin_bf16(void* y, const void* x, const void* W, int M, int N, int K, long long ldx, int mode, int gate_act, float act_limit,
                                 float act_slope, int slots, int tiles, const float* ssq, int shares, int width, float eps, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (!thin_sizes(y, x, W, M, N, K, ldx) || mode < THIN_BF16 || mode > THIN_PAIRS || (mode == THIN_PAIRS && !jv_act_known(gate_act)) || tiles < 1 || tiles > 2 ||
      (ssq && (mode == THIN_BF16 || shares < 4 || shares > THIN_SHARES || shares % 4 || width <= 0 || ((uintptr_t)ssq & 15))))
    return (int)hipErrorInvalidValue;
  const JvAct act{gate_act, act_limit, act_slope};
  const ThinScale scale{ssq, shares, 1.f / (float)width, eps};
  const hipStream_t st = (hipStream_t)stream;
#define THIN(MODE, SCALED)                                                                                              \
  return tiles == 2 ? thin_launch<MODE, SCALED, 2>(y, x, W, M, N, K, ldx, slots, act, scale, ThinStream{}, st)          \
                    : thin_launch<MODE, SCALED>(y, x, W, M, N, K, ldx, slots, act, scale, ThinStream{}, st)
  if (mode == THIN_F32) {
    if (ssq) { THIN(THIN_F32, true); }
    THIN(THIN_F32, false);
  }
  if (mode == THIN_PAIRS) {
    if (ssq) { THIN(THIN_PAIRS, true); }
    THIN(THIN_PAIRS, false);
  }
  THIN(THIN_BF16, false);
#undef THIN
}
// h += x W^T in place; with a weight rows = bf16(h * weight) and ssq[row * 256 + block] the blocks' shares of the rows' sums of squares.
extern "C" int jv_gemm_thin_stream_bf16(float* h, const void* x, const void* W, int M, int N, int K, long long ldx, const float* weight, void* rows,
                                        float* ssq, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (!thin_sizes(h, x, W, M, N, K, ldx) ||
      (weight && ((N + 15) / 16 > THIN_SHARES || !rows || !ssq || (((uintptr_t)weight | (uintptr_t)rows) & 15))))
    return (int)hipErrorInvalidValue;
  return thin_launch<THIN_STREAM, false>(h, x, W, M, N, K, ldx, 4, JvAct{}, ThinScale{}, ThinStream{weight, (bf16_t*)rows, ssq}, (hipStream_t)stream);
}
