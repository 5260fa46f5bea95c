// C[M,N] = A[M,K] * W[N,K]^T in 32 bits: float inputs that are kept whole, float sums, on the bf16 matrix unit.
//
// A float is the sum of three bf16 numbers (8 bits each: the nearest bf16, the nearest to what that leaves, the rest).  Of the
// nine products of two such sums the six largest are taken; the others are below 2^-26 of the whole.  The bf16 unit makes 13
// times the products of the 32-bit one, so six of its instructions take half the time of one of the 32-bit unit's.
//
// Order of the sums: steps of 32 columns; a step's six products are summed from the smallest on by themselves, from zero; the
// inner size is cut into two halves of whole steps, a half's steps are added in ascending order, then the halves.  That
// order depends on K alone, so a row's result depends neither on the other rows of the batch nor on the kernel that computes
// it.  Error against 64 bits over normal, positive and wide (e^3N) inputs, K 32 to 4,096: 0.4 to 0.8 of that of one 32-bit
// matrix product after another (relative 2-norm at 1,003 x 2,048 x 2,048 1.3e-7, before 2.9e-7).
//
// The third term of a small number would be below bf16's range (from 2^-110 on, down to 8 bits at 2^-126), so both operands are
// multiplied by 2^24 first, which changes no bit of a float, and the sums by 2^-48: the terms of every float, the smallest
// one among them, are then whole.  A sum that is not finite may come from the split (2^80 of the true sum, a value near the
// largest float, infinity less itself): it is made again from the numbers themselves.
//
// Microseconds in graphs with cold weights, as first built (tiles of 16, 32 and 64 rows) / now: 5 rows against 2,048 x 2,048 10.1 / 8.2, 6,144 x 2,048 14.7 /
// 13.9 (50 MB: the stream of W); 300 x 6,144 x 2,048 75 / 65; 1,003 x 6,144 x 2,048 153 / 144 with what the terms of A take; 2,048 x 24,576 x 4,096
// 2,250 / 1,954 = 211 TFLOP/s of 32-bit products, 1.27 PFLOP/s of the matrix unit's.  The scaling takes 1 to 5 % of it (24 sizes).
#include "common.h"
#include "f32_terms.h"

using namespace f32_terms;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));      // 16 bytes from any address of a float
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// The products of a step, (term of w, term of x), from the smallest on.
#define G32_PRODUCTS 6
__device__ constexpr int G32_W[G32_PRODUCTS] = {0, 1, 2, 0, 1, 0}, G32_X[G32_PRODUCTS] = {2, 1, 0, 1, 0, 0};
__device__ __forceinline__ f32x4 mfma(const u32x4& w, const u32x4& x, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), c, 0, 0, 0);
}
// The result of a sum of scaled products, or of the numbers themselves where that left the range of float.
__device__ __forceinline__ float settle(float sum, const float* a, const float* w, int K) {
  const bool held = __builtin_fabsf(sum) <= 3.402823466e38f;
  sum *= G32_UNSCALE;
  if (!held) {
    sum = 0.f;
    int k = 0;
    for (; k + 8 <= K && sum == sum; k += 8) {      // a NaN stays one
      float p[8], q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] = a[k + e], q[e] = w[k + e];
#pragma unroll
      for (int e = 0; e < 8; ++e) sum = fmaf(p[e], q[e], sum);
    }
    for (; k < K && sum == sum; ++k) sum = fmaf(a[k], w[k], sum);
  }
  return sum;
}
// Numbers n .. n + 3 of row m of C, settled; with an activation (ACT) the rows of W alternate gate and up rows and C is [M, N / 2].  Kernels without one
// do not hold its code: beside it the smallest products took 0.1 to 0.2 us more.
template <bool ACT>
__device__ __forceinline__ void leave(float* C, int m, int n, int N, const float (&v)[4], JvAct act) {
  if constexpr (ACT) {
#pragma unroll
    for (int e = 0; e < 4; e += 2)
      if (n + e < N) C[(long long)m * (N / 2) + (n + e) / 2] = jv_gated(act, v[e], v[e + 1]);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) C[(long long)m * N + n + e] = v[e];
  }
}
// The same from sums of scaled products.  `pieces`: N a multiple of 4, C begins on 16 bytes.  `keep` takes the activation's two results too.
template <bool ACT>
__device__ __forceinline__ void leave_sums(float* C, int m, int n, int M, int N, const f32x4& v, bool pieces, JvAct act, const float* A, const float* W, int K, int KA,
                                           float* keep = nullptr) {
  bool ok = pieces && n + 4 <= N;
#pragma unroll
  for (int e = 0; e < 4; ++e) ok = ok && __builtin_fabsf(v[e]) <= 3.402823466e38f;
  if (ok) {
    const f32x4 r = v * G32_UNSCALE;
    if constexpr (ACT) {
      const f32x2 z = {jv_gated(act, r[0], r[1]), jv_gated(act, r[2], r[3])};
      *(f32x2*)(C + (long long)m * (N / 2) + n / 2) = z;
      if (keep) *(f32x2*)keep = z;
    } else
      *(f32x4*)(C + (long long)m * N + n) = r;
  } else {
    float r[4];
    for (int e = 0; e < 4; ++e)
      if (n + e < N) r[e] = settle(v[e], A + (long long)m * KA, W + (long long)(n + e) * K, KA);
    leave<ACT>(C, m, n, N, r, act);
    if (ACT && keep) keep[0] = jv_gated(act, r[0], r[1]), keep[1] = jv_gated(act, r[2], r[3]);
  }
}
// 16 bytes a lane from base + off straight into LDS, 1 KB in the order of the lanes from `at` on.
__device__ __forceinline__ void lds_load(unsigned off, const void* base, unsigned at) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(at) : "memory", "m0");
}
__device__ __forceinline__ unsigned lds_address(const void* p) {
  return (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)p;
}

// Waits for the oldest of a wave's rounds of L loads on their way: `left` rounds to go, this one among them, at most S of them asked for.
template <int S, int L>
__device__ __forceinline__ void wait_oldest(int left) {
  if constexpr (S > 1) {
    if (left >= S) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * L) : "memory");
      return;
    }
    if constexpr (S > 2) return wait_oldest<S - 1, L>(left);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// ---------------------------------------------------------------------------- few rows
// A block takes TW rows of W by XR rows of A; its 8 waves share out the steps (waves 0 to 3 every fourth of the first half, 4 to
// 7 of the second), each through a ring of its own in LDS, straight from memory, S steps on their way, no wave waiting for
// another but once in R steps of each, when the steps' sums meet in LDS and are added in their order.
// DMA false: operands through registers, a round ahead, for rows that do not begin on 16 bytes.
template <int TW, int XR, int S, int R, bool DMA, bool ACT>
__global__ void __launch_bounds__(512)
gemm_f32_few_kernel(float* __restrict__ C, const float* __restrict__ A, const float* __restrict__ W, int M, int N, int K, JvAct act) {
  constexpr int ROWS = TW + XR, L = ROWS / 8, BUF = ROWS * G32_STEP, NT = TW / 16, MT = XR / 16, TILES = NT * MT;
  static_assert(TW % 16 == 0 && XR % 16 == 0 && TILES <= 4 && L * (S - 1) <= 63, "a wave adds a tile; what s_waitcnt counts to");
  __shared__ __attribute__((aligned(1024))) float bufs[DMA ? 8 * S * BUF : 4];
  __shared__ f32x4 met[2][2][4 * R][TILES][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wave >> 2, turn = wave & 3;
  const int li = lane & 15, lq = lane >> 4, n0 = blockIdx.x * TW, m0 = blockIdx.y * XR;
  const int total = (K + G32_STEP - 1) / G32_STEP, first = half ? (total + 1) / 2 : 0, steps = half ? total / 2 : (total + 1) / 2;
  // piece c of row r lies at slot c ^ (r % 8); a row's last step may have fewer pieces than 8: the last one again for those
  const int piece = ((lane & 7) ^ (lane >> 3)) * 16, beyond = max(piece + 16 - (K * 4 - (total - 1) * G32_STEP * 4), 0);
  unsigned off[L];
  const float* row[NT + MT];
  if constexpr (DMA) {
#pragma unroll
    for (int j = 0; j < L; ++j) {
      const int r = (j < TW / 8 ? j : j - TW / 8) * 8 + (lane >> 3);
      const int at = j < TW / 8 ? min(n0 + r, N - 1) - n0 : min(m0 + r, M - 1) - m0;      // rows behind the last one repeat it
      off[j] = (unsigned)at * (unsigned)(K * 4) + piece;
    }
  } else {
#pragma unroll
    for (int t = 0; t < NT; ++t) row[t] = W + (long long)min(n0 + t * 16 + li, N - 1) * K;
#pragma unroll
    for (int t = 0; t < MT; ++t) row[NT + t] = A + (long long)min(m0 + t * 16 + li, M - 1) * K;
  }
  const float* ws = W + (long long)n0 * K;
  const float* xs = A + (long long)m0 * K;
  float* ring = bufs + (DMA ? wave * S * BUF : 0);
  const unsigned lds0 = lds_address(ring);
  auto dma = [&](int i, int slot) {      // the wave's step i; behind the last one the last step of all again
    const int s = min(first + turn + 4 * i, total - 1), less = s == total - 1 ? beyond : 0;
#pragma unroll
    for (int j = 0; j < L; ++j) lds_load(off[j] - less, (j < TW / 8 ? ws : xs) + s * G32_STEP, lds0 + slot * (BUF * 4) + j * 1024);
  };
  const int wrow = li * G32_STEP, xrow = (TW + li) * G32_STEP;
  const int p0 = ((2 * lq) ^ (li & 7)) * 4, p1 = ((2 * lq + 1) ^ (li & 7)) * 4;
  // without the ring: a round's numbers, those beyond K zeros
  f32x4 ahead[DMA ? 1 : R][NT + MT][2];
  auto load_round = [&](int s0) {
#pragma unroll
    for (int r = 0; r < (DMA ? 0 : R); ++r) {
      const int k0 = (first + turn + s0 + 4 * r) * G32_STEP + lq * 8;
#pragma unroll
      for (int t = 0; t < NT + MT; ++t) {
        if (k0 + 8 <= K) {
          ahead[r][t][0] = *(const f32x4u*)(row[t] + k0), ahead[r][t][1] = *(const f32x4u*)(row[t] + k0 + 4);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) ahead[r][t][e / 4][e % 4] = k0 + e < K ? row[t][k0 + e] : 0.f;
        }
      }
    }
  };
  const int mine = (steps - turn + 3) / 4;      // this wave's steps
  if constexpr (DMA)
    for (int v = 0; v < S; ++v) v < mine ? dma(v, v) : (void)0;
  else load_round(0);
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  int slot = 0;
  const int longest = (total + 1) / 2;
  // A round of steps.  FULL: every wave has them all and asks for one more behind each, so nothing is looked at (conditions in every round took 2 to
  // 7 % of 4,096 columns and more: 64 x 2,048 x 8,192 46.9 us for 43.6; without any, loads behind the last step take 3 to 4 % of 256).
  auto round_of = [&](auto full, int s0, int round) {
    constexpr bool FULL = decltype(full)::value;
    f32x4 now[DMA ? 1 : R][NT + MT][2];
    if constexpr (!DMA) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < NT + MT; ++t) now[r][t][0] = ahead[r][t][0], now[r][t][1] = ahead[r][t][1];
      load_round(s0 + 4 * R);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      f32x4 raw[NT + MT][2];
      if constexpr (DMA) {
        const int i = s0 / 4 + r;
        if (!FULL && i >= mine) break;
        if constexpr (FULL) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * L) : "memory");
        else wait_oldest<S, L>(mine - i);
        const float* b = ring + slot * BUF;
#pragma unroll
        for (int t = 0; t < NT + MT; ++t) {
          const float* at = b + (t < NT ? wrow + t * 16 * G32_STEP : xrow + (t - NT) * 16 * G32_STEP);
          raw[t][0] = *(const f32x4*)(at + p0), raw[t][1] = *(const f32x4*)(at + p1);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // read before the slot is filled again
        if (FULL || i + S < mine) dma(i + S, slot);
        slot = slot + 1 == S ? 0 : slot + 1;
        const int k0 = (first + turn + 4 * i) * G32_STEP;
        if (!FULL && k0 + G32_STEP > K) {      // zeros of A beyond K: what W repeats there does not count
#pragma unroll
          for (int t = NT; t < NT + MT; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              if (k0 + lq * 8 + h * 4 >= K) raw[t][h] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      } else {
#pragma unroll
        for (int t = 0; t < NT + MT; ++t) raw[t][0] = now[r][t][0], raw[t][1] = now[r][t][1];
      }
      u32x4 wt[NT][3], xt[3];
#pragma unroll
      for (int a = 0; a < NT; ++a) split8(raw[a], wt[a]);
#pragma unroll
      for (int b = 0; b < MT; ++b) {
        split8(raw[NT + b], xt);
        f32x4 t[NT];
#pragma unroll
        for (int e = 0; e < G32_PRODUCTS; ++e)
#pragma unroll
          for (int a = 0; a < NT; ++a) t[a] = mfma(wt[a][G32_W[e]], xt[G32_X[e]], e ? t[a] : zero);
#pragma unroll
        for (int a = 0; a < NT; ++a) met[round][half][4 * r + turn][a * MT + b][lane] = t[a];
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();      // (the buffer of the round before the last was read before the last round's barrier)
    asm volatile("" ::: "memory");
    if (turn < TILES) {
      f32x4 part[4 * R];      // (behind the last step: what the buffer held, not added)
#pragma unroll
      for (int s = 0; s < 4 * R; ++s) part[s] = met[round][half][s][turn][lane];
#pragma unroll
      for (int s = 0; s < 4 * R; ++s)
        if (FULL || s0 + s < steps) sum += part[s];
    }
  };
  int s0 = 0, round = 0;
  if constexpr (DMA)
    for (const int least = total / 8; s0 / 4 + R - 1 + S < least; s0 += 4 * R, round ^= 1) round_of(std::true_type{}, s0, round);
  for (; s0 < longest; s0 += 4 * R, round ^= 1) round_of(std::false_type{}, s0, round);
  __syncthreads();
  if (half && turn < TILES) met[0][1][0][turn][lane] = sum;
  __syncthreads();
  if (half || turn >= TILES) return;
  sum += met[0][1][0][turn][lane];
  const int m = m0 + turn % MT * 16 + li, n = n0 + turn / MT * 16 + lq * 4;      // a lane holds C[m][n .. n + 3]
  if (m >= M) return;
  float r[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < N) r[e] = settle(sum[e], A + (long long)m * K, W + (long long)(n + e) * K, K);
  leave<ACT>(C, m, n, N, r, act);
}

// ---------------------------------------------------------------------------- up to 8 rows
// A block takes 8 G rows of W by 8 rows of A.  Steps go in pairs: lanes 0 to 7 of an operand hold the rows of one step, lanes 8 to 15 those of
// the next, and of the product the two quarters that belong together count.  So nothing is split or multiplied twice, as it would be for half
// a tile of 16.  The 8 waves share out the pairs (waves 0 to 3 every fourth of the first half of the steps, 4 to 7 of the second), each through
// a ring of its own, S pairs on their way; every step leaves its sums in LDS, and after C pairs of each wave they are added in their order.
// What bounds few rows is a wave's chain from wait to sum (0.8 us a step of each wave with 16 x 16 tiles, which meet every two steps), not the
// stream of W: hence smaller tiles on twice the units and one meeting for up to 64 pairs.  Straight into registers instead of the ring, a lane a
// row (32 lines an instruction): 9.0 for 8.4.  Microseconds in graphs with cold weights, 16 x 16 or 32 x 16 tiles / these (rows of W): 8 rows
// against 2,048 x 2,048 9.7 / 8.4 (8), 2,048 x 3,072 12.5 / 9.7 (8), 512 x 8,192 25.5 / 17.5 (8), 3,072 x 2,048 9.9 / 9.2 (16), 1,024 x 1,024 6.3 /
// 5.5 (8), 6,144 x 2,048 14.5 / 14.0 (24), 6,144 x 8,192 51 / 45 (24), 32,000 x 2,048 54.6 / 55.2 (16): wide ones stay with 32 x 16.
template <int G, int S, int C, bool ACT>
__global__ void __launch_bounds__(512)
gemm_f32_pairs_kernel(float* __restrict__ out, const float* __restrict__ A, const float* __restrict__ W, int M, int N, int K, JvAct act) {
  constexpr int L = 2 * (G + 1), BUF = L * 256;      // loads of a pair, each 8 rows of a step, 1 KB
  static_assert(G <= 4 && L * (S - 1) <= 63, "a wave adds what a block leaves; what s_waitcnt counts to");
  __shared__ __attribute__((aligned(1024))) float bufs[8 * S * BUF];
  __shared__ f32x4 met[2][8 * C][16 * G];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wave >> 2, turn = wave & 3;
  const int li = lane & 15, lq = lane >> 4, odd = li >> 3, n0 = blockIdx.x * 8 * G;
  const int total = (K + G32_STEP - 1) / G32_STEP, first = half ? (total + 1) / 2 : 0, steps = half ? total / 2 : (total + 1) / 2;
  const int longest = ((total + 1) / 2 + 7) / 8;      // pairs of the wave that has the most
  const int mine = ((steps + 1) / 2 - turn + 3) / 4;
  // piece c of row r lies at slot c ^ r; a row's last step may have fewer pieces than 8: the last one again for those
  const int piece = ((lane & 7) ^ (lane >> 3)) * 16, beyond = max(piece + 16 - (K * 4 - (total - 1) * G32_STEP * 4), 0);
  unsigned off[G + 1];
#pragma unroll
  for (int t = 0; t <= G; ++t) {      // rows behind the last one repeat it
    const int r = lane >> 3, at = t < G ? min(n0 + t * 8 + r, N - 1) - n0 : min(r, M - 1);
    off[t] = (unsigned)at * (unsigned)(K * 4) + piece;
  }
  const float* ws = W + (long long)n0 * K;
  float* ring = bufs + wave * S * BUF;
  const unsigned lds0 = lds_address(ring);
  auto dma = [&](int i, int slot) {      // the wave's pair i; behind the last step that one again
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      const int s = min(first + 2 * (turn + 4 * i) + o, total - 1), less = s == total - 1 ? beyond : 0;
#pragma unroll
      for (int t = 0; t <= G; ++t) lds_load(off[t] - less, (t < G ? ws : A) + s * G32_STEP, lds0 + slot * (BUF * 4) + (2 * t + o) * 1024);
    }
  };
  const int at0 = odd * 256 + (li & 7) * G32_STEP, p0 = at0 + ((2 * lq) ^ (li & 7)) * 4, p1 = at0 + ((2 * lq + 1) ^ (li & 7)) * 4;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int v = 0; v < S; ++v)
    if (v < mine) dma(v, v);
  f32x4 sum = zero;
  int slot = 0;
  for (int c0 = 0; c0 < longest; c0 += C) {
    const int stop = min(c0 + C, longest);
    for (int i = c0; i < stop; ++i) {
      if (i >= mine) break;
      wait_oldest<S, L>(mine - i);
      const float* b = ring + slot * BUF;
      f32x4 raw[G + 1][2];
#pragma unroll
      for (int t = 0; t <= G; ++t) raw[t][0] = *(const f32x4*)(b + t * 512 + p0), raw[t][1] = *(const f32x4*)(b + t * 512 + p1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // read before the slot is filled again
      if (i + S < mine) dma(i + S, slot);
      slot = slot + 1 == S ? 0 : slot + 1;
      const int s = 2 * (turn + 4 * i);
      if ((first + s + 2) * G32_STEP > K) {      // zeros of A beyond K: what W repeats there does not count
        const int k = (first + s + odd) * G32_STEP + lq * 8;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (k + h * 4 >= K) raw[G][h] = zero;
      }
      u32x4 wt[G][3], xt[3];
      split8(raw[G], xt);
#pragma unroll
      for (int g = 0; g < G; ++g) split8(raw[g], wt[g]);
      f32x4 t[G];
#pragma unroll
      for (int e = 0; e < G32_PRODUCTS; ++e)
#pragma unroll
        for (int g = 0; g < G; ++g) t[g] = mfma(wt[g][G32_W[e]], xt[G32_X[e]], e ? t[g] : zero);
      f32x4* to = &met[half][(i - c0) * 8 + 2 * turn + odd][(li & 7) * 2 + (lq & 1)];
#pragma unroll
      for (int g = 0; g < G; ++g)
        if ((lq >> 1) == odd) to[g * 16] = t[g];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (turn == 0 && lane < 16 * G) {
      const int count = min(8 * C, steps - 8 * c0);
      for (int s = 0; s < count; s += 8) {
        f32x4 part[8];      // (behind the last step: what the buffer held, not added)
#pragma unroll
        for (int u = 0; u < 8; ++u) part[u] = met[half][s + u][lane];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (s + u < count) sum += part[u];
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();      // read before the next sums are left there
    asm volatile("" ::: "memory");
  }
  if (half && turn == 0 && lane < 16 * G) met[1][0][lane] = sum;
  __syncthreads();
  if (wave || lane >= 16 * G) return;
  sum += met[1][0][lane];
  const int m = lane % 16 / 2, n = n0 + lane / 16 * 8 + lane % 2 * 4;      // a lane holds C[m][n .. n + 3]
  if (m >= M) return;
  float r[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < N) r[e] = settle(sum[e], A + (long long)m * K, W + (long long)(n + e) * K, K);
  leave<ACT>(out, m, n, N, r, act);
}

// ---------------------------------------------------------------------------- many rows
// The rows of A as their three terms, [M][steps][term][32]: made once for all the blocks that multiply a row.
__global__ void __launch_bounds__(256)
split_rows_kernel(unsigned* __restrict__ y, const float* __restrict__ A, int K, int steps) {
  const int k = (blockIdx.y * 256 + threadIdx.x) * 8;
  if (k >= steps * G32_STEP) return;
  const float* a = A + (long long)blockIdx.x * K + k;
  f32x4 v[2];
  if (k + 8 <= K && ((uintptr_t)a & 15) == 0) {
    v[0] = *(const f32x4*)a, v[1] = *(const f32x4*)(a + 4);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e / 4][e % 4] = k + e < K ? a[e] : 0.f;
  }
  u32x4 t[3];
  split8(v, t);
  u32x4* out = (u32x4*)y + ((long long)blockIdx.x * steps + k / G32_STEP) * 12 + k % G32_STEP / 8;
#pragma unroll
  for (int e = 0; e < 3; ++e) out[e * 4] = t[e];
}

// Tiles of TM (64) rows of A (as terms) by TW rows of W (as floats); two groups of 2 x 2 waves take a half of the steps each, through
// rings of S steps in LDS.  Bound by what a SIMD issues: a product of 16 cycles takes 8 of them, a vector instruction 2 to 4
// (measured), so a wave splits the next 16 rows of W (52 instructions) while it multiplies these with all its rows of A.
template <int TM, int TW, bool ACT>
__global__ void __launch_bounds__(512, 2)
gemm_f32_tile_kernel(float* __restrict__ C, const unsigned* __restrict__ X, const float* __restrict__ A, const float* __restrict__ W, int M, int N, int K, int KA, JvAct act) {
  constexpr int MT = TM / 32, NT = TW / 32, XL = TM * 3 / 64, WL = TW / 32, L = XL + WL;      // L: loads of a wave for a step
  constexpr int XBYTES = TM * 192, BYTES = XBYTES + TW * 128, FIT = 160 * 1024 / (2 * BYTES), S = FIT < 4 ? FIT : 4;
  static_assert(S >= 2 && XL * 64 == TM * 3 && (S - 1) * L <= 63, "");
  __shared__ __attribute__((aligned(1024))) char bufs[2 * S * BYTES];
  const int lane = threadIdx.x & 63, all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), group = all >> 2, wave = all & 3;
  // Blocks b, b + 8, ... run on one XCD: each takes one run of the tiles, rows of A fastest
  const int mtiles = (M + TM - 1) / TM, live = mtiles * ((N + TW - 1) / TW), per = (live + 7) / 8;
  const int u = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || u >= live) return;
  const int m0 = u % mtiles * TM, n0 = u / mtiles * TW;
  const int total = (K + G32_STEP - 1) / G32_STEP, turns = (total + 1) / 2, first = group * turns, steps = group ? total - turns : turns;
  // (a row's last step may have fewer pieces of W than 8: the last one again for those, against zeros of A)
  const int piece = ((lane & 7) ^ (lane >> 3)) * 16, beyond = max(piece + 16 - (K * 4 - (total - 1) * 128), 0);
  unsigned off[L];
#pragma unroll
  for (int j = 0; j < XL; ++j) {      // an instruction brings 16 rows of 64 bytes of one term; piece c of row r lies at slot c ^ (r / 2 % 4)
    const int q = wave * XL + j, e = q / (TM / 16), r = q % (TM / 16) * 16 + (lane >> 2);
    off[j] = (unsigned)(min(m0 + r, M - 1) - m0) * (unsigned)(total * 192) + e * 64 + (((lane & 3) ^ (r >> 1)) & 3) * 16;
  }
#pragma unroll
  for (int j = 0; j < WL; ++j) {      // 8 rows of 128 bytes; piece c of row r lies at slot c ^ (r % 8)
    const int r = (wave * WL + j) * 8 + (lane >> 3);
    off[XL + j] = (unsigned)(min(n0 + r, N - 1) - n0) * (unsigned)(K * 4) + piece;
  }
  const char* xs = (const char*)X + (long long)m0 * total * 192;
  const char* ws = (const char*)(W + (long long)n0 * K);
  const char* ring = bufs + group * (S * BYTES);
  const unsigned lds0 = lds_address(ring);
  auto dma = [&](int c, int slot) {
    const int at = min(first + c, total - 1), less = at == total - 1 ? beyond : 0;
#pragma unroll
    for (int j = 0; j < L; ++j)
      lds_load(j < XL ? off[j] : off[j] - less, j < XL ? xs + at * 192 : ws + at * 128,
               lds0 + slot * BYTES + (j < XL ? (wave * XL + j) * 1024 : XBYTES + (wave * WL + j - XL) * 1024));
  };
  const int wm = wave >> 1, wn = wave & 1, li = lane & 15, lq = lane >> 4;
  const int xat = (wm * MT * 16 + li) * 64 + ((lq ^ (li >> 1)) & 3) * 16;
  const int wrow = XBYTES + (wn * NT * 16 + li) * 128;
  const int p0 = wrow + ((2 * lq) ^ (li & 7)) * 16, p1 = wrow + ((2 * lq + 1) ^ (li & 7)) * 16;
  f32x4 tot[NT][MT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) tot[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 xt[3][MT], wt[2][3];
  auto read_x = [&](int e, int slot) {
#pragma unroll
    for (int b = 0; b < MT; ++b) xt[e][b] = *(const u32x4*)(ring + slot * BYTES + e * (TM * 64) + xat + b * 1024);
  };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int v = 0; v < S; ++v) dma(v, v);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 1) * L) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  {
    const f32x4 v[2] = {*(const f32x4*)(ring + p0), *(const f32x4*)(ring + p1)};
    split8(v, wt[0]);
#pragma unroll
    for (int e = 0; e < 3; ++e) read_x(e, 0);
  }
  // W's rows a of step c against all rows of A; the rows that come next are read at `at` and split meanwhile
  auto stage = [&](auto last, auto set, int a, int at, int next, bool real) {
    constexpr bool LAST = decltype(last)::value;
    constexpr int SET = decltype(set)::value, SLOTS = G32_PRODUCTS * MT;
    const f32x4 v[2] = {*(const f32x4*)(ring + at + p0), *(const f32x4*)(ring + at + p1)};
    f32x4 t[MT];
    int pairs = 0;
#pragma unroll
    for (int e = 0; e < G32_PRODUCTS; ++e) {
#pragma unroll
      for (int b = 0; b < MT; ++b) {
        t[b] = mfma(wt[SET][G32_W[e]], xt[G32_X[e]][b], e ? t[b] : zero);
        const int i = e * MT + b + 1 - MT;      // the first MT products cover the reads' way
#pragma unroll
        for (int p = 0; p < 4; ++p)
          if (i > 0 && p == pairs && p * (SLOTS - MT) < i * 4) {
            split_pair(v[p / 2][p % 2 * 2], v[p / 2][p % 2 * 2 + 1], p, wt[SET ^ 1]);
            // the split stays between these products
            asm volatile("" : "+v"(wt[SET ^ 1][0][p]), "+v"(wt[SET ^ 1][1][p]), "+v"(wt[SET ^ 1][2][p]));
            ++pairs;
          }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (LAST && e == 0) read_x(2, next);      // a term's last product is made: the next step's
      if (LAST && e == 3) read_x(1, next);
      if (LAST && e == 5) read_x(0, next);
    }
    if (real) {
#pragma unroll
      for (int b = 0; b < MT; ++b) tot[a][b] += t[b];
    }
  };
  using std::integral_constant;
  int slot = 0;
  auto step = [&](auto parity, int c) {
    constexpr int P = decltype(parity)::value;
    const int next = slot + 1 == S ? 0 : slot + 1;
    const bool real = c < steps;
#pragma unroll
    for (int a = 0; a + 1 < NT; ++a) {
      if ((P + a) & 1) stage(integral_constant<bool, false>{}, integral_constant<int, 1>{}, a, slot * BYTES + (a + 1) * 2048, next, real);
      else stage(integral_constant<bool, false>{}, integral_constant<int, 0>{}, a, slot * BYTES + (a + 1) * 2048, next, real);
    }
    // step c is in registers everywhere, step c + 1 is there
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * L) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    dma(c + S, slot);
    stage(integral_constant<bool, true>{}, integral_constant<int, (P + NT - 1) & 1>{}, NT - 1, next * BYTES, next, real);
    slot = next;
  };
  if constexpr (NT % 2 == 0) {
    for (int c = 0; c < turns; ++c) step(integral_constant<int, 0>{}, c);
  } else {
    for (int c = 0; c < turns; c += 2) {
      step(integral_constant<int, 0>{}, c);
      if (c + 1 < turns) step(integral_constant<int, 1>{}, c + 1);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  f32x4* meet = (f32x4*)bufs;
  static_assert(TM * TW * 4 <= 2 * S * BYTES, "");
  if (group) {
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int b = 0; b < MT; ++b) meet[((a * MT + b) * 4 + wave) * 64 + lane] = tot[a][b];
  }
  __syncthreads();
  if (group) return;
  const bool pieces = !(N & 3) && !((uintptr_t)C & 15);
#pragma unroll
  for (int b = 0; b < MT; ++b) {
    const int m = m0 + (wm * MT + b) * 16 + li;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      const int n = n0 + (wn * NT + a) * 16 + lq * 4;
      leave_sums<ACT>(C, m, n, M, N, tot[a][b] + meet[((a * MT + b) * 4 + wave) * 64 + lane], pieces, act, A, W, K, KA);
    }
  }
}

// The same for 128 rows of A by TW rows of W, with v_mfma_f32_32x32x16_bf16: two of them give the bits of one 16x16x32 (its 32 products
// are added in four groups of 8, in order; measured over 80,000 sums of four kinds of numbers) for the issue of half as many.  Two
// groups of 4 waves take a half of the steps each, a wave 32 rows of A against all TW of W.  A wave's rows of A are its own: their
// terms come straight into registers, one or two steps ahead, in pieces of 1 KB in the order of the lanes (split_fragments_kernel; 16 bytes from
// each of 64 rows an instruction cost a fifth more).  W is split once a group: a thread takes 4 numbers a row two or three steps
// ahead, splits them beside the products of a step and leaves the terms in a ring of 3 steps in LDS.
// Both groups' sums go through LDS to rows of C in whole lines: from the lanes that hold them 32 bytes of a row left at once, and one group's waves added and
// stored everything, 6 us a block longer (2,048 x 24,576 x 512 with those 381 us, 2,048 x 8,192 x 256 85).
// Against tiles of 128 rows by the 16x16x32 instruction, in which every wave split its W and which were bound by what a SIMD issues,
// microseconds with the split of A, before -> now: 1,003 x 6,144 x 2,048 153 -> 144, x 2,048 61 -> 57, 384 x 4,096 x 4,096 110 -> 86, 2,048 x 24,576 x
// 4,096 2,250 -> 1,954, x 512 345 -> 310, 2,048 x 8,192 x 256 74 -> 65; 128 rows of W 1.14 to 1.30 times as fast on average by inner size, 96 1.06 to
// 1.23, 64 1.08 to 1.26.  Behind only where few rows meet many short ones: 65 to 200 x 24,576 x 256 and 512 by 4 to 7 %.
template <int TW, bool ACT>
__global__ void __launch_bounds__(512, 2)
gemm_f32_rows_kernel(float* __restrict__ C, const unsigned* __restrict__ X, const float* __restrict__ A, const float* __restrict__ W, int M, int N, int K, int KA, JvAct act,
                     unsigned* __restrict__ terms, bool fragments) {
  constexpr int TM = 128, NT = TW / 32, TERMS = 3 * TW * 64, RING = 3;
  static_assert(2 * RING * TERMS <= 160 * 1024 && 2 * TM * (TW + 4) * 4 <= 2 * RING * TERMS, "");
  __shared__ __attribute__((aligned(1024))) char bufs[2 * RING * TERMS];
  const int lane = threadIdx.x & 63, all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), group = all >> 2, wave = all & 3;
  const int mtiles = (M + TM - 1) / TM, live = mtiles * ((N + TW - 1) / TW), per = (live + 7) / 8;
  const int u = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || u >= live) return;
  const int m0 = u % mtiles * TM, n0 = u / mtiles * TW;
  const int total = (K + G32_STEP - 1) / G32_STEP, turns = (total + 1) / 2, first = group * turns, steps = group ? total - turns : turns;
  const int li = lane & 31, lh = lane >> 5;
  const char* xrow = (const char*)X + (long long)min(m0 / 32 + wave, (M - 1) / 32) * total * 6144 + lane * 16;
  const int gt = threadIdx.x & 255, wr = gt >> 3, wp = gt & 7;
  const float* wrow[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) wrow[j] = W + (long long)min(n0 + j * 32 + wr, N - 1) * K;
  char* const ring = bufs + group * (RING * TERMS);
  // where this thread's pieces go: piece c (16 bytes) of row r of a term lies at slot c ^ (r / 2 % 4)
  const int put = wr * 64 + (((wp >> 1) ^ (wr >> 1)) & 3) * 16 + (wp & 1) * 8;
  const int get0 = li * 64 + ((lh ^ (li >> 1)) & 3) * 16, get1 = li * 64 + (((2 + lh) ^ (li >> 1)) & 3) * 16;
  constexpr int XS = TW > 96 ? 2 : 3, WS = TW > 64 ? 2 : 3;      // sets of registers for rows of A and of W on their way
  f32x4 raw[WS][NT];
  u32x4 xt[XS][3][2], wt[2][3][2];
  f32x16 tot[NT], t[2];
  auto load_w = [&](int c, f32x4 (&r)[NT]) {
    const int at = min(min(first + c, total - 1) * G32_STEP + wp * 4, K - 4);
#pragma unroll
    for (int j = 0; j < NT; ++j) r[j] = *(const f32x4*)(wrow[j] + at);
  };
  auto load_x = [&](int c, u32x4 (&x)[3][2]) {
    const char* at = xrow + (long long)min(first + c, total - 1) * 6144;
#pragma unroll
    for (int e = 2; e >= 0; --e)
#pragma unroll
      for (int b = 0; b < 2; ++b) x[e][b] = *(const u32x4*)(at + (e * 2 + b) * 1024);
  };
  auto put_w = [&](const f32x4& r, int j, char* slot) {
    u32x4 q[3];
    split_pair(r[0], r[1], 0, q);
    split_pair(r[2], r[3], 1, q);
#pragma unroll
    for (int e = 0; e < 3; ++e) *(u32x2*)(slot + e * (TW * 64) + j * 2048 + put) = u32x2{q[e][0], q[e][1]};
  };
  auto get_w = [&](int a, const char* slot, u32x4 (&w)[3][2]) {
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      w[e][0] = *(const u32x4*)(slot + e * (TW * 64) + a * 2048 + get0);
      w[e][1] = *(const u32x4*)(slot + e * (TW * 64) + a * 2048 + get1);
    }
  };
  auto meet_all = [&] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int e = 0; e < 16; ++e) tot[a][e] = 0.f;
#pragma unroll
  for (int e = 0; e < 16; ++e) t[0][e] = t[1][e] = 0.f;
  {
    f32x4 w0[NT], w1[NT];
    load_w(0, w0);
    load_w(1, w1);
#pragma unroll
    for (int i = 0; i + 1 < XS; ++i) load_x(i, xt[i]);
#pragma unroll
    for (int i = 0; i < WS; ++i) load_w(2 + i, raw[i]);
#pragma unroll
    for (int j = 0; j < NT; ++j) put_w(w0[j], j, ring);
#pragma unroll
    for (int j = 0; j < NT; ++j) put_w(w1[j], j, ring + TERMS);
  }
  meet_all();
  get_w(0, ring, wt[0]);
  int slot = 0;
  // Step c: its W lies in `slot`, that of c + 1 in the next; W of c + 2, in registers, is split into the one after, a piece of 4 numbers
  // beside the products of 32 rows.  A tile's products of a step join its total beside the next tile's.
  auto step = [&](auto phase, int c) {
    constexpr int PH = decltype(phase)::value;
    const int s1 = slot + 1 == RING ? 0 : slot + 1, s2 = s1 + 1 == RING ? 0 : s1 + 1;
    load_x(c + XS - 1, xt[(PH + XS - 1) % XS]);
    __builtin_amdgcn_sched_barrier(0);
    if (c < steps) {
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        const int cur = (PH * NT + a) & 1, before = (a + NT - 1) % NT;
        auto& w = wt[cur];
        if (a + 1 < NT) get_w(a + 1, ring + slot * TERMS, wt[cur ^ 1]);
        else get_w(0, ring + s1 * TERMS, wt[cur ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
        f32x16 q;
#pragma unroll
        for (int e = 0; e < 16; ++e) q[e] = 0.f;
#pragma unroll
        for (int e = 0; e < G32_PRODUCTS; ++e)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            q = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w[G32_W[e]][b]), __builtin_bit_cast(bf16x8, xt[PH % XS][G32_X[e]][b]), q, 0, 0, 0);
        put_w(raw[PH % WS][a], a, ring + s2 * TERMS);
        tot[before] += t[cur ^ 1];
        t[cur] = q;
#pragma unroll
        for (int i = 0; i < 12; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);      // a product, then four or five others
          __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      load_w(c + 2 + WS, raw[PH % WS]);
    }
    meet_all();
    slot = s1;
  };
  using std::integral_constant;
  for (int c = 0; c < turns; c += 6) {
    step(integral_constant<int, 0>{}, c);
    if (c + 1 < turns) step(integral_constant<int, 1>{}, c + 1);
    if (c + 2 < turns) step(integral_constant<int, 2>{}, c + 2);
    if (c + 3 < turns) step(integral_constant<int, 3>{}, c + 3);
    if (c + 4 < turns) step(integral_constant<int, 4>{}, c + 4);
    if (c + 5 < turns) step(integral_constant<int, 5>{}, c + 5);
  }
  if constexpr (NT % 2 == 0) tot[NT - 1] += t[1];
  else tot[NT - 1] += steps & 1 ? t[0] : t[1];
  __syncthreads();
  // both groups' sums meet in LDS and leave it in whole lines of a row
  constexpr int ROW = TW + 4, SIDE = TM * ROW;
  float* const meet = (float*)bufs;
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *(f32x4*)(meet + group * SIDE + (wave * 32 + li) * ROW + a * 32 + q * 8 + lh * 4) = f32x4{tot[a][q * 4], tot[a][q * 4 + 1], tot[a][q * 4 + 2], tot[a][q * 4 + 3]};
  __syncthreads();
  const bool pieces = !(N & 3) && !((uintptr_t)C & 15);
#pragma unroll 4
  for (int i = threadIdx.x; i < TM * TW / 4; i += 512) {
    const int r = i / (TW / 4), c = (i - r * (TW / 4)) * 4;
    if (m0 + r >= M || n0 + c >= N) continue;
    float* at = meet + r * ROW + c;
    leave_sums<ACT>(C, m0 + r, n0 + c, M, N, *(const f32x4*)at + *(const f32x4*)(at + SIDE), pieces, act, A, W, K, KA, ACT && terms ? at : nullptr);
  }
  if constexpr (ACT) {
    if (!terms) return;
    __syncthreads();
    // the results again, 8 a thread, as the terms of the next product's rows; lanes along the rows
    for (int i = threadIdx.x; i < TM * TW / 16; i += 512) {
      const int r = i % TM, c = i / TM * 16;
      if (m0 + r >= M || n0 + c >= N) continue;      // N is a multiple of 64
      f32x4 v[2];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x2 z = *(const f32x2*)(meet + r * ROW + c + j * 4);
        v[j / 2][j % 2 * 2] = z[0], v[j / 2][j % 2 * 2 + 1] = z[1];
      }
      leave_terms(terms, fragments, N / 64, m0 + r, (n0 + c) / 16, v);
    }
  }
}

// How C is made (jv_gemm_f32): 0, 1: few rows, 16 x 16 or 32 x 32, through registers; 2 to 4: few rows through the ring, 16 x 16, 32 x 16, 32 x 32
// (rows of W x rows of A), for up to 8 rows of A in pairs of steps with form 2 (8 rows of W while their blocks go to 256 units at once, else 16)
// and form 4 (24); 5 to 7 tiles of 128 rows of A by 128, 96, 64 of W, 8 to 10 of 64 rows by 96, 64, 32.
template <int TW, int XR, int S, int R, bool DMA>
static int few_launch(float* C, const float* A, const float* W, int M, int N, int K, JvAct act, hipStream_t s) {
  if ((M + XR - 1) / XR > 65535) return (int)hipErrorInvalidValue;
  const auto kernel = act.id ? gemm_f32_few_kernel<TW, XR, S, R, DMA, true> : gemm_f32_few_kernel<TW, XR, S, R, DMA, false>;
  hipLaunchKernelGGL(kernel, dim3((N + TW - 1) / TW, (M + XR - 1) / XR), dim3(512), 0, s, C, A, W, M, N, K, act);
  return JV_LAUNCH_CHECK();
}
template <int G, int S, int C>
static int pairs_launch(float* out, const float* A, const float* W, int M, int N, int K, JvAct act, hipStream_t s) {
  const auto kernel = act.id ? gemm_f32_pairs_kernel<G, S, C, true> : gemm_f32_pairs_kernel<G, S, C, false>;
  hipLaunchKernelGGL(kernel, dim3((N + 8 * G - 1) / (8 * G)), dim3(512), 0, s, out, A, W, M, N, K, act);
  return JV_LAUNCH_CHECK();
}
template <int TM, int TW>
static int tile_launch(float* C, const void* X, const float* A, const float* W, int M, int N, int K, int KA, JvAct act, hipStream_t s) {
  const long long live = ((long long)M + TM - 1) / TM * (((long long)N + TW - 1) / TW);
  if (live > 1 << 24) return (int)hipErrorInvalidValue;
  const auto kernel = act.id ? gemm_f32_tile_kernel<TM, TW, true> : gemm_f32_tile_kernel<TM, TW, false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((live + 7) / 8 * 8)), dim3(512), 0, s, C, (const unsigned*)X, A, W, M, N, K, KA, act);
  return JV_LAUNCH_CHECK();
}
// The same in the order in which gemm_f32_rows_kernel multiplies: [M / 32][steps][term][16 columns][8 columns][32 rows][8].
__global__ void __launch_bounds__(256)
split_fragments_kernel(unsigned* __restrict__ y, const float* __restrict__ A, int M, int K, int steps) {
  const int row = threadIdx.x >> 3, m = blockIdx.x * 32 + row;
  if (m >= M) return;
  // 64 columns a block; a grid has no more than 65,535 blocks of columns, the longest rows have 65,536
  for (int at = blockIdx.y; at < (steps + 1) / 2; at += gridDim.y) {
    const int k = (at * 8 + (threadIdx.x & 7)) * 8;
    if (k >= steps * G32_STEP) return;
    const float* a = A + (long long)m * K + k;
    f32x4 v[2];
    if (k + 8 <= K && ((uintptr_t)a & 15) == 0) {
      v[0] = *(const f32x4*)a, v[1] = *(const f32x4*)(a + 4);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e / 4][e % 4] = k + e < K ? a[e] : 0.f;
    }
    u32x4 t[3];
    split8(v, t);
    u32x4* out = (u32x4*)y + ((long long)blockIdx.x * steps + k / G32_STEP) * 384 + k % G32_STEP / 16 * 64 + k % 16 / 8 * 32 + row;
#pragma unroll
    for (int e = 0; e < 3; ++e) out[e * 128] = t[e];
  }
}
extern "C" int jv_split_fragments_f32(void* X, const float* A, int M, int KA, void* stream) {
  if (M <= 0 || KA <= 0) return 0;
  if ((uintptr_t)X & 15) return (int)hipErrorInvalidValue;
  const int steps = (KA + G32_STEP - 1) / G32_STEP;
  hipLaunchKernelGGL(split_fragments_kernel, dim3((M + 31) / 32, (steps + 1) / 2 < 65535 ? (steps + 1) / 2 : 65535), dim3(256), 0, (hipStream_t)stream, (unsigned*)X, A, M, KA, steps);
  return JV_LAUNCH_CHECK();
}
template <int TW>
static int rows_launch(float* C, const void* X, const float* A, const float* W, int M, int N, int K, int KA, JvAct act, void* terms, bool fragments, hipStream_t s) {
  const long long live = ((long long)M + 127) / 128 * (((long long)N + TW - 1) / TW);
  if (live > 1 << 24) return (int)hipErrorInvalidValue;
  const auto kernel = act.id ? gemm_f32_rows_kernel<TW, true> : gemm_f32_rows_kernel<TW, false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((live + 7) / 8 * 8)), dim3(512), 0, s, C, (const unsigned*)X, A, W, M, N, K, KA, act, (unsigned*)terms, fragments);
  return JV_LAUNCH_CHECK();
}
// Rows of A [M][KA] as terms (of 2^24 times A), [M][steps][3][32] bf16 with zeros behind KA; steps = ceil(KA / 32).
extern "C" int jv_split_rows_f32(void* X, const float* A, int M, int KA, void* stream) {
  if (M <= 0 || KA <= 0) return 0;
  if ((uintptr_t)X & 15) return (int)hipErrorInvalidValue;
  const int steps = (KA + G32_STEP - 1) / G32_STEP;
  if ((steps * G32_STEP + 2047) / 2048 > 65535) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(split_rows_kernel, dim3(M, (steps * G32_STEP + 2047) / 2048), dim3(256), 0, (hipStream_t)stream, (unsigned*)X, A, KA, steps);
  return JV_LAUNCH_CHECK();
}
// A [M][KA], W [N][K], C [M][N].  K = KA but for tiles, where W may have columns behind KA (finite; as many steps of 32 as KA has).
// X, for tiles: the rows of A by jv_split_fragments_f32 (forms 5 to 7) or jv_split_rows_f32 (from 8 on).
// gate_act (JV_ACT_*, not 0): the rows of W alternate gate and up rows and C is [M][N / 2], act(gate) * up; forms 5 to 7 then also leave it as terms
// (`terms` not null, N a multiple of 64), by rows or with `fragments` as jv_split_fragments_f32 would.
extern "C" int jv_gemm_f32(float* C, const float* A, const float* W, const void* X, int M, int N, int K, int KA, int form, int gate_act, float act_limit,
                           float act_slope, void* terms, int fragments, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  const bool pieces = !(K & 3) && !((uintptr_t)W & 15) && K > 0;
  if (K < 0 || KA > K || (KA + 31) / 32 != (K + 31) / 32) return (int)hipErrorInvalidValue;
  if (gate_act && (!jv_act_known(gate_act) || N % 2)) return (int)hipErrorInvalidValue;
  if (terms && (!gate_act || N % 64 || form < 5 || form > 7 || (((uintptr_t)terms | (uintptr_t)C) & 15))) return (int)hipErrorInvalidValue;
  if (form >= 5 ? !pieces || !X || ((uintptr_t)X & 15) || K > 1 << 22 : KA != K || (form >= 2 && (!pieces || ((uintptr_t)A & 15) || K > 1 << 24)))
    return (int)hipErrorInvalidValue;
  const JvAct act{gate_act, act_limit, act_slope};
  const hipStream_t s = (hipStream_t)stream;
  switch (form) {
    case 0: return few_launch<16, 16, 1, 2, false>(C, A, W, M, N, K, act, s);
    case 1: return few_launch<32, 32, 1, 1, false>(C, A, W, M, N, K, act, s);
    case 2:
      if (M > 8) return few_launch<16, 16, 2, 2, true>(C, A, W, M, N, K, act, s);
      return N <= 8 * 256 ? pairs_launch<1, 2, 8>(C, A, W, M, N, K, act, s) : pairs_launch<2, 1, 4>(C, A, W, M, N, K, act, s);
    case 3: return few_launch<32, 16, 1, 1, true>(C, A, W, M, N, K, act, s);
    case 4: return M > 8 ? few_launch<32, 32, 1, 1, true>(C, A, W, M, N, K, act, s) : pairs_launch<3, 1, 2>(C, A, W, M, N, K, act, s);
    case 5: return rows_launch<128>(C, X, A, W, M, N, K, KA, act, terms, fragments != 0, s);
    case 6: return rows_launch<96>(C, X, A, W, M, N, K, KA, act, terms, fragments != 0, s);
    case 7: return rows_launch<64>(C, X, A, W, M, N, K, KA, act, terms, fragments != 0, s);
    case 8: return tile_launch<64, 96>(C, X, A, W, M, N, K, KA, act, s);
    case 9: return tile_launch<64, 64>(C, X, A, W, M, N, K, KA, act, s);
    case 10: return tile_launch<64, 32>(C, X, A, W, M, N, K, KA, act, s);
  }
  return (int)hipErrorInvalidValue;
}
