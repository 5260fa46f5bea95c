// y[parts][M,N] = x[M,K] W[N,K]^T for 129 to 1,792 rows against a narrow W with a long inner size (the down and output products
// of prompts), bf16 in, float sums: `ksplit` blocks share out the inner size of a tile, as float partial products that the
// reader adds in order, because the tiles of y alone do not fill the chip.
//
// Bound by how soon a tile's operands arrive: alone, a unit's blocks draw 96 bytes a nanosecond from the L2s (69 if each chunk
// is awaited before the next is asked for), beside the matrix unit two thirds of that.  So a block (one a compute unit) keeps
// a ring of half chunks of 64 columns in LDS, straight from memory, with one and a half to three chunks on their way, and
// spreads the loads over its products: asked for in one go they stop the waves that would multiply (4,096 rows against
// 4,096 x 12,288, tiles of 256 x 256: 343 us with two whole buffers, 324 with the loads spread out, 305 with the ring of 5
// halves; 262 with no loads at all).  A wave reads its operands of the next 16 columns while it multiplies these; the barrier
// that hands a chunk over stands before the products of the last 16 columns, whose operands are in registers.
//
// Against 4,096 x 12,288, microseconds (the library's bf16 product): 160 rows 36.9 (77.7), 300 rows 48.3 (69.6), 512 rows 54.2
// (81.6), 1,024 rows 94.1 (116); against 4,096 x 4,096: 17.0 (27.5), 20.5 (26.0), 25.8 (30.0), 39.2 (42.7).  With the norm that adds the parts, against 4,096 x 12,288: 1,525 rows by tiles of 192 x 256 (96 x 128 a wave,
// one a SIMD) 140 (162); 5,120 x 17,408 185 at 1,152 rows (310).
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define SH_K 64            // columns of a chunk: a row of it is 128 bytes, 8 pieces of 16

// Tiles of TM rows of x and TW rows of W; WM x WN waves with whole 32 x 32 tiles each, v_mfma_f32_32x32x16_bf16 with A = rows of
// W, B = rows of x.  A unit of the ring is the first or the second half of the rows of x and of W, of one chunk: unit v lies in
// slot v % S.
template <int TM, int TW, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN, 1)
gemm_shares_kernel(float* __restrict__ y, const bf16_t* __restrict__ x, const bf16_t* __restrict__ W, int M, int N, int K, int ksplit) {
  constexpr int WAVES = WM * WN, MT = TM / WM / 32, NT = TW / WN / 32;
  constexpr int HALF = (TM + TW) / 2 * SH_K;                                        // elements of a unit
  constexpr int FIT = 160 * 1024 / (HALF * 2), S = FIT < 8 ? FIT : 8;
  constexpr int XL = TM / 2 / 8 / WAVES, WL = TW / 2 / 8 / WAVES, L = XL + WL;      // loads of a wave for a unit
  constexpr int NF = MT * NT, NR = MT + NT, RPI = (NR + NF - 1) / NF;
  static_assert(S >= 5 && XL >= 1 && WL >= 1 && WM % 2 == 0 && WN % 2 == 0, "two chunks and a unit; a wave's rows lie in one unit");
  static_assert((S - 3) * L <= 63, "what s_waitcnt counts to");
  __shared__ __attribute__((aligned(1024))) bf16_t bufs[S * HALF];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Blocks b, b + 8, ... run on one XCD: each takes one run of the tiles, rows of x fastest, and its blocks walk in step, so
  // that a row of x or W is read into that L2 once.
  const int mtiles = (M + TM - 1) / TM, tiles = mtiles * ((N + TW - 1) / TW), live = tiles * ksplit, per = (live + 7) / 8;
  const int u = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || u >= live) return;
  const int part = u / tiles, t = u - part * tiles;
  const int m0 = t % mtiles * TM, n0 = t / mtiles * TW;
  const int all = K / SH_K, c0 = (int)((long long)all * part / ksplit), chunks = (int)((long long)all * (part + 1) / ksplit) - c0;
  // An instruction brings 8 rows, lane l row l / 8, and fills 1 KB in the order of the lanes; piece c of row r lies at slot
  // c ^ ((r / 2) % 8) of its row, so that 16 lanes reading one piece of 16 rows meet 16 slots.  Rows beyond the last repeat it.
  unsigned off[2 * L];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < L; ++j) {
      const int r = (j < XL ? wave * XL + j : wave * WL + j - XL) * 8 + (lane >> 3);   // row of the half of x or of W
      const int piece = ((lane & 7) ^ (r >> 1)) & 7;
      const int row = j < XL ? min(m0 + h * (TM / 2) + r, M - 1) - m0 : min(n0 + h * (TW / 2) + r, N - 1) - n0;
      off[h * L + j] = (unsigned)row * (unsigned)(K * 2) + piece * 16;
    }
  const bf16_t* xs = x + (long long)m0 * K + (long long)c0 * SH_K;
  const bf16_t* ws = W + (long long)n0 * K + (long long)c0 * SH_K;
  const unsigned lds0 = (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)bufs;
  auto dma = [&](int j, int h, int c, int slot) {
    const bf16_t* base = (j < XL ? xs : ws) + c * SH_K;
    const unsigned at = lds0 + slot * (HALF * 2) + (j < XL ? (wave * XL + j) * 8 : TM / 2 + (wave * WL + j - XL) * 8) * 128;
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off[h * L + j]), "s"(base), "s"(at) : "memory", "m0");
  };
  auto wrap = [](int s) { return s >= S ? s - S : s; };
  f32x16 acc[NT][MT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
  const int wm = wave / WN, wn = wave - wm * WN, l32 = lane & 31, half = lane >> 5, swz = (l32 >> 1) & 7;
  const int xh = wm / (WM / 2), wh = wn / (WN / 2);
  const int xrow = ((wm % (WM / 2)) * MT * 32 + l32) * SH_K, wrow = (TM / 2 + (wn % (WN / 2)) * NT * 32 + l32) * SH_K;
  bf16x8 xf[2][MT], wf[2][NT];
  auto read = [&](int i, int set, int ks, int s0) {      // s0: slot of the chunk's first unit
    const int at = ((ks * 2 + half) ^ swz) * 8;
    if (i < NT) wf[set][i] = *(const bf16x8*)(bufs + wrap(s0 + wh) * HALF + wrow + at + i * 2048);
    else xf[set][i - NT] = *(const bf16x8*)(bufs + wrap(s0 + xh) * HALF + xrow + at + (i - NT) * 2048);
  };
  // Chunk c: its products, and the loads of units 2 c + S - 1 and 2 c + S, into the slots that units of chunks c - 1 and c left.
  // more: 2: unit 2 c + S exists; 1: chunk c + 1 exists; 0: the last.
  auto chunk = [&](auto more, int c, int s0) {
    constexpr int MORE = decltype(more)::value;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int set = ks & 1;
      if (ks == 3 && MORE > 0) {      // chunk c is in registers everywhere, c + 1 is there (S - 4 units behind it may be on their way)
        if (MORE > 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 4) * L) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      int rd = 0;
#pragma unroll
      for (int i = 0; i < NF; ++i) {
#pragma unroll
        for (int q = 0; q < RPI; ++q)
          if (rd < NR && (ks < 3 || MORE > 0)) { read(rd, set ^ 1, (ks + 1) & 3, ks < 3 ? s0 : wrap(s0 + 2)); ++rd; }
        if (MORE > 1) {
#pragma unroll
          for (int j = 0; j < L; ++j) {
            constexpr int U0 = S - 1, U1 = S;       // units counted from 2 c
            if (ks < 3 && j * 3 * NF / L == ks * NF + i) dma(j, U0 & 1, c + U0 / 2, wrap(s0 + U0));
            if (ks == 3 && j * NF / L == i) dma(j, U1 & 1, c + U1 / 2, s0);
          }
        }
        acc[i / MT][i % MT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[set][i / MT], xf[set][i % MT], acc[i / MT][i % MT], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (MORE == 1 && ks == 0 && 2 * c + S - 1 < 2 * chunks) {
#pragma unroll
        for (int j = 0; j < L; ++j) dma(j, (S - 1) & 1, c + (S - 1) / 2, wrap(s0 + S - 1));
      }
    }
  };
  for (int v = 0; v < S - 1; ++v)
    if (v < 2 * chunks) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if ((v & 1) == h) {
#pragma unroll
          for (int j = 0; j < L; ++j) dma(j, h, v >> 1, v);
        }
    }
  if (2 * chunks >= S - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 3) * L) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NR; ++i) read(i, 0, 0, 0);
  int c = 0, s0 = 0;
  for (; 2 * c + S < 2 * chunks; ++c, s0 = wrap(s0 + 2)) chunk(std::integral_constant<int, 2>{}, c, s0);
  for (; c + 1 < chunks; ++c, s0 = wrap(s0 + 2)) chunk(std::integral_constant<int, 1>{}, c, s0);
  chunk(std::integral_constant<int, 0>{}, c, s0);
#pragma unroll
  for (int b = 0; b < MT; ++b) {         // a lane holds row l32 of each of the wave's tiles of x, columns 8 q + 4 half + e of its tiles of W
    const int m = m0 + (wm * MT + b) * 32 + l32;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + (wn * NT + a) * 32 + q * 8 + half * 4;
        const f32x16 v = acc[a][b];
        if (n < N) *(f32x4*)(y + ((long long)part * M + m) * N + n) = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
      }
  }
}

template <int TM, int TW, int WM, int WN>
static int sh_launch(float* y, const void* x, const void* W, int M, int N, int K, int ksplit, hipStream_t s) {
  const long long live = (long long)((M + TM - 1) / TM) * ((N + TW - 1) / TW) * ksplit;
  if (live > 1 << 24) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((gemm_shares_kernel<TM, TW, WM, WN>), dim3((unsigned)((live + 7) / 8 * 8)), dim3(64 * WM * WN), 0, s, y,
                     (const bf16_t*)x, (const bf16_t*)W, M, N, K, ksplit);
  return JV_LAUNCH_CHECK();
}
// tm, tw: rows of x and of W of a tile, (128, 128), (256, 128), (192, 256) or (256, 256); y float [ksplit][M][N].
extern "C" int jv_gemm_shares_bf16(float* y, const void* x, const void* W, int M, int N, int K, int tm, int tw, int ksplit, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K < SH_K || K % SH_K || K > 1 << 20 || N % 4 || ksplit < 1 || ksplit > K / SH_K || (((uintptr_t)x | (uintptr_t)W | (uintptr_t)y) & 15))
    return (int)hipErrorInvalidValue;
  const hipStream_t s = (hipStream_t)stream;
  if (tm == 128 && tw == 128) return sh_launch<128, 128, 2, 2>(y, x, W, M, N, K, ksplit, s);
  if (tm == 256 && tw == 128) return sh_launch<256, 128, 2, 2>(y, x, W, M, N, K, ksplit, s);
  if (tm == 192 && tw == 256) return sh_launch<192, 256, 2, 2>(y, x, W, M, N, K, ksplit, s);
  if (tm == 256 && tw == 256) return sh_launch<256, 256, 2, 4>(y, x, W, M, N, K, ksplit, s);
  return (int)hipErrorInvalidValue;
}
