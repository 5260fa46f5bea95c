// C[M,N] = A[M,K] * W[N,K]^T in true 32-bit: float inputs, float products and sums on the matrix cores
// (v_mfma_f32_16x16x4_f32), no reduced-precision matrix mode.
//
// Order of the sums: the inner size is cut into 8 parts of equal length (a multiple of 16); a part is summed in
// ascending steps of 16 columns (inside a step columns j, j + 4, j + 8, j + 12 enter together), the parts' sums are added
// in ascending order.  That order depends on K alone, so a row's result depends neither on the other rows of the
// batch nor on the tile that computes it, and eight short chains err less than one long one.
//
// A block's 8 waves take one part of the inner size each, all for the same tile of (16 NT) rows of W by (16 MT) rows of
// A; operands go from global memory straight into the matrix unit's registers (a lane's 16 bytes are 4 columns of one row:
// four products), one stage of U steps ahead of their use; the parts meet in LDS once, at the end.  Nothing waits for
// another wave inside the loop, and a decode step's narrow products still have 8 waves a row tile pulling at W.
// A 16 x 16 x 4 product keeps its unit busy for 32 cycles, so at 4 x 4 tiles a wave needs 8 KB per 2,048 cycles and the
// kernel is bound by the matrix unit; at few rows it is bound by the stream of W.
#include "common.h"

typedef float g32_f4 __attribute__((ext_vector_type(4)));
typedef float g32_f4u __attribute__((ext_vector_type(4), aligned(4)));      // 16 bytes from any address of a float

#define G32_PARTS 8
#define G32_ROUND_TILES 8      // 16 x 16 tiles that meet in LDS at once: 64 KB

template <int NT, int MT, int U>
__global__ void __launch_bounds__(64 * G32_PARTS)
gemm_f32_kernel(float* __restrict__ C, const float* __restrict__ A, const float* __restrict__ W,
                int M, int N, int K, long long lda, long long ldw, long long ldc) {
  constexpr int TILES = NT * MT;
  constexpr int ROUND = TILES < G32_ROUND_TILES ? TILES : G32_ROUND_TILES;
  __shared__ g32_f4 red[ROUND][G32_PARTS][64];
  const int tid = threadIdx.x, part = tid >> 6, lane = tid & 63, li = lane & 15, lq = lane >> 4;
  const int n0 = blockIdx.x * (16 * NT), m0 = blockIdx.y * (16 * MT);
  const int len = ((K + G32_PARTS - 1) / G32_PARTS + 15) / 16 * 16;
  const int k_begin = part * len;
  const int k_end = k_begin + len < K ? k_begin + len : K;

  // rows behind the last one read the last one's numbers; their results are not stored
  const float* wrow[NT];
  const float* arow[MT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = n0 + t * 16 + li;
    wrow[t] = W + (long long)(n < N ? n : N - 1) * ldw + lq * 4;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = m0 + t * 16 + li;
    arow[t] = A + (long long)(m < M ? m : M - 1) * lda + lq * 4;
  }
  // a lane's 4 columns k + 4 lq .. + 3 of a step that may reach beyond K: zeros there, in both operands
  auto load4_tail = [&](const float* row, int k) -> g32_f4 {
    g32_f4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (k + lq * 4 + e < K) v[e] = row[k + e];
    return v;
  };

  g32_f4 acc[NT][MT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) acc[a][b] = g32_f4{0.f, 0.f, 0.f, 0.f};
  auto products = [&](const g32_f4* w, const g32_f4* x) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[a][j], x[b][j], acc[a][b], 0, 0, 0);
  };

  const int full = k_end > k_begin ? (k_end - k_begin) / 16 : 0;
  const int stages = full / U;
  if (stages > 0) {
    g32_f4 wc[U][NT], xc[U][MT], wn[U][NT], xn[U][MT];
    auto load_stage = [&](int s, g32_f4 (*w)[NT], g32_f4 (*x)[MT]) {
      const int k = k_begin + s * (16 * U);
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int t = 0; t < NT; ++t) w[u][t] = *(const g32_f4u*)(wrow[t] + k + u * 16);
#pragma unroll
        for (int t = 0; t < MT; ++t) x[u][t] = *(const g32_f4u*)(arow[t] + k + u * 16);
      }
    };
    load_stage(0, wc, xc);
    for (int s = 0; s < stages; ++s) {
      load_stage(s + 1 < stages ? s + 1 : s, wn, xn);      // never skipped: a conditional prefetch would be waited for at once
      __builtin_amdgcn_sched_barrier(0);                   // and not moved down to its use
#pragma unroll
      for (int u = 0; u < U; ++u) products(wc[u], xc[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int t = 0; t < NT; ++t) wc[u][t] = wn[u][t];
#pragma unroll
        for (int t = 0; t < MT; ++t) xc[u][t] = xn[u][t];
      }
    }
  }
  for (int k = k_begin + stages * (16 * U); k < k_end; k += 16) {
    g32_f4 w[NT], x[MT];
#pragma unroll
    for (int t = 0; t < NT; ++t) w[t] = load4_tail(wrow[t], k);
#pragma unroll
    for (int t = 0; t < MT; ++t) x[t] = load4_tail(arow[t], k);
    products(w, x);
  }

  // the parts meet, a round of 16 x 16 tiles at a time; a lane holds C[m0 + 16 b + li][n0 + 16 a + 4 lq .. + 3]
#pragma unroll
  for (int r0 = 0; r0 < TILES; r0 += ROUND) {
    if (r0 > 0) __syncthreads();
#pragma unroll
    for (int t = 0; t < ROUND; ++t) red[t][part][lane] = acc[(r0 + t) / MT][(r0 + t) % MT];
    __syncthreads();
    for (int t = part; t < ROUND; t += G32_PARTS) {
      g32_f4 sum = red[t][0][lane];
#pragma unroll
      for (int p = 1; p < G32_PARTS; ++p) sum += red[t][p][lane];
      const int m = m0 + (r0 + t) % MT * 16 + li, n = n0 + (r0 + t) / MT * 16 + lq * 4;
      if (m < M) {
        float* c = C + (long long)m * ldc + n;
        if (n + 4 <= N && (ldc & 3) == 0 && ((uintptr_t)C & 15) == 0) {
          *(g32_f4*)c = sum;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) c[e] = sum[e];
        }
      }
    }
  }
}

extern "C" int jv_gemm_f32(float* C, const float* A, const float* W, int M, int N, int K,
                           long long lda, long long ldw, long long ldc, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K < 0) return (int)hipErrorInvalidValue;
  // The tile: all give the same bits, so it is chosen by time alone.  `us` is what a round of 256 blocks (one a compute
  // unit) was measured to take at K = 2,048; time grows with the rounds, and with K for all alike.  So few rows take
  // small tiles until W fills the chip (5 rows: N = 3,072 11.1 us with 1 x 1 and 13.7 with 2 x 1; N = 32,000 73 and 58), many
  // rows the tile whose last round is fullest (1,003 rows: N = 3,072 122 us with 4 x 4 and 148 with 4 x 8; N = 2,048 84 and
  // 79 = 107 TFLOP/s; 2,048 rows, N = 24,576, K = 4,096: 4 x 8 3.39 ms = 122 TFLOP/s, 4 x 4 4.06).
  struct Tile { int nt, mt; float us; };
  static const Tile tiles[] = {{1, 1, 13.f}, {2, 1, 16.3f}, {1, 2, 16.2f}, {2, 2, 22.3f}, {1, 4, 23.f}, {2, 4, 30.f}, {4, 4, 42.f}, {4, 8, 75.f}};
  int best = 0;
  double least = 0;
  for (int i = 0; i < (int)(sizeof(tiles) / sizeof(tiles[0])); ++i) {
    const long long blocks = ((long long)N + 16 * tiles[i].nt - 1) / (16 * tiles[i].nt) * (((long long)M + 16 * tiles[i].mt - 1) / (16 * tiles[i].mt));
    const double t = (double)((blocks + 255) / 256) * tiles[i].us;
    if (((long long)M + 16 * tiles[i].mt - 1) / (16 * tiles[i].mt) > 65535) continue;
    if (least == 0 || t < least) best = i, least = t;
  }
  if (least == 0) return (int)hipErrorInvalidValue;
#define G32_LAUNCH(NT, MT, U)                                                                             \
  hipLaunchKernelGGL((gemm_f32_kernel<NT, MT, U>),                                                        \
                     dim3(((long long)N + 16 * NT - 1) / (16 * NT), ((long long)M + 16 * MT - 1) / (16 * MT)), \
                     dim3(64 * G32_PARTS), 0, (hipStream_t)stream, C, A, W, M, N, K, lda, ldw, ldc)
  switch (best) {
    case 0: G32_LAUNCH(1, 1, 8); break;
    case 1: G32_LAUNCH(2, 1, 4); break;
    case 2: G32_LAUNCH(1, 2, 4); break;
    case 3: G32_LAUNCH(2, 2, 4); break;
    case 4: G32_LAUNCH(1, 4, 2); break;
    case 5: G32_LAUNCH(2, 4, 2); break;
    case 6: G32_LAUNCH(4, 4, 1); break;
    default: G32_LAUNCH(4, 8, 1); break;
  }
#undef G32_LAUNCH
  return JV_LAUNCH_CHECK();
}
