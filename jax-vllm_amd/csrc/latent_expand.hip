// Prompts through latent attention with every head's keys and values written out (bf16).
//
// In the latent's own space a (query, key) pair costs a head 2 (rank + rot) products, whatever its size, because queries and
// results are as long as the cached vector; with k[h] = [U_k[h] c | k_rot] and v[h] = U_v[h] c written out once per token it costs
// 2 (dim + rot).  A decoded token would pay that for its whole context; a prompt that begins its request pays once per token, and
// then every pair is cheaper.  2,048 tokens of 16 heads of 64 + 32 over a vector of 224 + 32, a window of 1,024 keys: writing out 14 us,
// queries 3, attention 38, results 5; before, queries and results through the matrices 17, 5 and 11 and attention 77.
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define LX_TOKENS 64       // tokens of a tile, from a request's first one on: a page of what is written out
#define LX_STEPS 8         // steps of 32 of the inner size whose weights a wave has at a time

// Cached vectors e = [c (rank) | k_rot (rot)] of a tile's tokens, read from their slots of the cache's key pages, become keys
// [page][heads][slot][D] and transposed values [page][heads][D][slot] of D = dim + rot, values filled up with zeros; a tile is a page,
// tokens behind the request's last are zeros.  grid (tiles, heads); the tile's vectors lie in LDS (rows 16 bytes longer, so that 16 rows'
// pieces meet all banks), 16 rows of U_k or U_v at a time go from memory to a wave's operands (the first 16 while the tile is
// staged), v_mfma_f32_16x16x32_bf16.  For keys A = rows of U, for values A = tokens, so that a lane holds 4 numbers that lie side by
// side.
__global__ void __launch_bounds__(256)
latent_expand_kernel(bf16_t* __restrict__ k_out, bf16_t* __restrict__ v_out, const bf16_t* __restrict__ e_pages,
                     const int* __restrict__ slot_mapping, const int* __restrict__ tiles, const bf16_t* __restrict__ k_up,
                     const bf16_t* __restrict__ v_up, int heads, int dim, int rot, int vdim, int rank) {
  extern __shared__ __attribute__((aligned(16))) bf16_t es[];      // [LX_TOKENS][rank + rot + 8]
  const int tile = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lc = lane >> 4;
  const int row0 = tiles[2 * tile], rows = tiles[2 * tile + 1], E = rank + rot, es_row = E + 8, D = dim + rot, pieces = E / 8;
  const int k_tiles = dim / 16, all = k_tiles + vdim / 16;
  bf16x8 wf[LX_STEPS];
  auto weights = [&](int nt, int k0) {
    const bf16_t* w = nt < k_tiles ? k_up + ((long long)h * dim + nt * 16 + li) * rank : v_up + ((long long)h * vdim + (nt - k_tiles) * 16 + li) * rank;
#pragma unroll
    for (int u = 0; u < LX_STEPS; ++u) wf[u] = *(const bf16x8*)(w + min(k0 + u * 32, rank - 32) + lc * 8);
  };
  weights(min(wave, all - 1), 0);
  for (int i = tid; i < LX_TOKENS * pieces; i += 256) {
    const int r = i / pieces, c = (i - r * pieces) * 8;
    const long long slot = max(slot_mapping[row0 + min(r, rows - 1)], 0);
    bf16x8 v = *(const bf16x8*)(e_pages + slot * E + c);
    if (r >= rows)
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = (bf16_t)0.f;
    *(bf16x8*)(es + r * es_row + c) = v;
  }
  __syncthreads();
  bf16_t* keys = k_out + ((long long)tile * heads + h) * LX_TOKENS * D;
  bf16_t* values = v_out + ((long long)tile * heads + h) * LX_TOKENS * D;
  for (int nt = wave; nt < all; nt += 4) {
    const bool key = nt < k_tiles;
    const int n0 = (key ? nt : nt - k_tiles) * 16;
    f32x4 acc[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < rank; k0 += 32 * LX_STEPS) {
      if (k0 || nt != wave) weights(nt, k0);
#pragma unroll
      for (int u = 0; u < LX_STEPS; ++u) {
        if (k0 + u * 32 >= rank) break;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const bf16x8 xf = *(const bf16x8*)(es + (m * 16 + li) * es_row + k0 + u * 32 + lc * 8);
          acc[m] = key ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], xf, acc[m], 0, 0, 0)
                       : __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, wf[u], acc[m], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (bf16_t)acc[m][e];
      if (key) *(bf16x4*)(keys + (m * 16 + li) * D + n0 + 4 * lc) = v;
      else *(bf16x4*)(values + (n0 + li) * LX_TOKENS + m * 16 + 4 * lc) = v;
    }
  }
  for (int i = tid; i < LX_TOKENS * (rot / 8); i += 256) {
    const int r = i / (rot / 8), c = (i - r * (rot / 8)) * 8;
    *(bf16x8*)(keys + r * D + dim + c) = *(const bf16x8*)(es + r * es_row + rank + c);
  }
  const bf16x8 none = {};
  for (int i = tid; i < (D - vdim) * (LX_TOKENS / 8); i += 256) *(bf16x8*)(values + vdim * LX_TOKENS + i * 8) = none;
}

// q[t, h, dim :] turns in place, h heads of dim + rot columns a row; a thread a pair.
__global__ void __launch_bounds__(256)
latent_turn_queries_kernel(bf16_t* __restrict__ q, long long ldq, int heads, int dim, int rot, int rot_dims,
                           const float* __restrict__ cos_sin, int interleaved) {
  const long long t = blockIdx.x;
  const int half = rot_dims / 2;
  const float* cs = cos_sin + t * rot_dims;
  for (int i = threadIdx.x; i < heads * half; i += blockDim.x) {
    const int h = i / half, p = i - h * half;
    bf16_t* x = q + t * ldq + h * (long long)(dim + rot) + dim;
    bf16_t *a = x + (interleaved ? 2 * p : p), *b = x + (interleaved ? 2 * p + 1 : p + half);
    const float u = to_f32(*a), v = to_f32(*b), c = cs[p], s = cs[half + p];
    *a = from_f32<bf16_t>(u * c - v * s);
    *b = from_f32<bf16_t>(v * c + u * s);
  }
}

// o[t, h * vdim + i] = att[t, h * D + i] * (g ? sigmoid(g[t * ldg + h * gn + (gn > 1 ? i : 0)]) : 1); 8 columns a thread.
__global__ void __launch_bounds__(256)
latent_cut_heads_kernel(bf16_t* __restrict__ o, const bf16_t* __restrict__ att, long long n, int heads, int vdim, int D,
                        const bf16_t* __restrict__ g, long long ldg, int gn, int vec) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const int per = heads * vdim / 8;
  if (i >= n * per) return;
  const long long t = i / per;
  const int c = (int)(i - t * per) * 8, h = c / vdim, e0 = c - h * vdim;
  bf16x8 v = *(const bf16x8*)(att + (t * heads + h) * D + e0);
  if (g) {
    const bf16_t* gp = g + t * ldg + (gn > 1 ? c : h);
    bf16x8 gv;
    if (vec) gv = *(const bf16x8*)gp;
    else
#pragma unroll
      for (int e = 0; e < 8; ++e) gv[e] = gp[gn > 1 ? e : 0];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = from_f32<bf16_t>(to_f32(v[e]) / (1.f + expf(-to_f32(gv[e]))));
  }
  *(bf16x8*)(o + t * heads * vdim + c) = v;
}

extern "C" int jv_latent_expand_tokens() { return LX_TOKENS; }
extern "C" int jv_latent_expand_max_vector() { return 64 * 1024 / 2 / LX_TOKENS - 8; }

// tiles [n_tiles][2] = (first row of the step, tokens of the request from there, at most 64).
extern "C" int jv_latent_expand_bf16(void* k_out, void* v_out, const void* e_pages, const int* slot_mapping, const int* tiles,
                                     int n_tiles, const void* k_up, const void* v_up, int heads, int dim, int rot, int vdim,
                                     int rank, void* stream) {
  if (n_tiles <= 0 || heads <= 0) return 0;
  if (dim < 16 || dim % 16 || vdim < 16 || vdim % 16 || rot < 0 || rot % 8 || rank < 32 || rank % 32 || vdim > dim + rot || heads > 65535 ||
      rank + rot > jv_latent_expand_max_vector() ||
      (((uintptr_t)k_out | (uintptr_t)v_out | (uintptr_t)e_pages | (uintptr_t)k_up | (uintptr_t)v_up) & 15))
    return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(latent_expand_kernel, dim3(n_tiles, heads), dim3(256), LX_TOKENS * (rank + rot + 8) * sizeof(bf16_t),
                     (hipStream_t)stream, (bf16_t*)k_out, (bf16_t*)v_out, (const bf16_t*)e_pages, slot_mapping, tiles,
                     (const bf16_t*)k_up, (const bf16_t*)v_up, heads, dim, rot, vdim, rank);
  return JV_LAUNCH_CHECK();
}

extern "C" int jv_latent_turn_queries_bf16(void* q, long long ldq, int n, int heads, int dim, int rot, int rot_dims,
                                           const float* cos_sin, int interleaved, void* stream) {
  if (n <= 0 || heads <= 0 || rot_dims <= 0) return 0;
  if (rot_dims % 2 || rot_dims > rot || ldq < (long long)heads * (dim + rot)) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(latent_turn_queries_kernel, dim3(n), dim3(256), 0, (hipStream_t)stream, (bf16_t*)q, ldq, heads, dim, rot,
                     rot_dims, cos_sin, interleaved);
  return JV_LAUNCH_CHECK();
}

extern "C" int jv_latent_cut_heads_bf16(void* o, const void* att, long long n, int heads, int vdim, int D, const void* g,
                                        long long ldg, int gn, void* stream) {
  if (n <= 0 || heads <= 0) return 0;
  if (vdim < 8 || vdim % 8 || D % 8 || vdim > D || (((uintptr_t)o | (uintptr_t)att) & 15) ||
      (n * heads * vdim / 8 + 255) / 256 > 0x7fffffffll)
    return (int)hipErrorInvalidValue;
  const int vec = gn > 1 && ldg % 8 == 0 && (uintptr_t)g % 16 == 0;
  hipLaunchKernelGGL(latent_cut_heads_kernel, dim3((unsigned)((n * heads * vdim / 8 + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, (bf16_t*)o, (const bf16_t*)att, n, heads, vdim, D, (const bf16_t*)g, ldg, gn, vec);
  return JV_LAUNCH_CHECK();
}
