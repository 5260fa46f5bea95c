// Linear attention with a per-head decay ("lightning"): per head a matrix state in float,
//     S_t = decay_h * S_(t-1) + k_t v_t^T,      o_t = S_t^T q_t,
// with q, k, v = silu of projections (the activation is applied as they are loaded).  The state of a
// request lives in a row of `state` [slots + 1][heads][dim][vdim] between steps; a step reads it, runs
// its tokens, and writes it back.  Columns of S (one per element of v) never mix, so a block takes one
// (request, head, slice of columns): a thread keeps up to LT_ROWS rows of one column in registers.
//
// Two kernels with the same numbers in a different order of operations:
//  * token by token (decoded tokens, short portions): S is updated and read once per token;
//  * by chunks of LC tokens (prompt portions): within a chunk
//        o_i = decay^(i+1) (S^T q_i) + sum_{j<=i} decay^(i-j) (q_i . k_j) v_j
//        S  <- decay^n S + sum_j decay^(n-1-j) k_j v_j^T                      (n tokens in the chunk)
//    so the state is touched once per chunk, a chunk's tokens run side by side, and so do the chunks
//    (everything but the second line's chain).  Only non-negative powers of the decay occur.  Everything is float.
#include "common.h"

#define LT_ROWS 32

__device__ __forceinline__ float lt_silu(float z) { return z / (1.f + expf(-z)); }

// grid (requests, heads, column slices); block 256 = parts x cols threads, cols a power of two
template <typename T>
__global__ void __launch_bounds__(256)
lightning_steps_kernel(float* __restrict__ out, const T* __restrict__ proj, long long ld, int q_off, int k_off,
                       int v_off, float* __restrict__ state, const int* __restrict__ slot_ids,
                       const int* __restrict__ cu_seqlens, const float* __restrict__ decay, int heads, int dim,
                       int vdim, int cols) {
  extern __shared__ float lds[];          // 2 x (q[dim] | k[dim] | v[cols]) | partial sums [parts][cols]
  const int r = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * cols;
  const int parts = blockDim.x / cols;
  const int col = threadIdx.x % cols, part = threadIdx.x / cols;
  const int t0 = cu_seqlens[r], t1 = cu_seqlens[r + 1];
  if (t1 <= t0) return;
  const int stage = 2 * dim + cols;
  float* red = lds + 2 * stage;
  const float lam = decay[h];
  const bool live = c0 + col < vdim;
  float* S = state + (((long long)slot_ids[r] * heads + h) * dim) * vdim + c0 + col;
  float s[LT_ROWS];
#pragma unroll
  for (int i = 0; i < LT_ROWS; ++i) {
    const int d = part + i * parts;
    s[i] = (live && d < dim) ? S[(long long)d * vdim] : 0.f;
  }
  for (int t = t0; t < t1; ++t) {
    float* buf = lds + ((t - t0) & 1) * stage;
    const T* row = proj + (long long)t * ld;
    for (int d = threadIdx.x; d < dim; d += blockDim.x) {
      buf[d] = lt_silu(to_f32(row[q_off + h * dim + d]));
      buf[dim + d] = lt_silu(to_f32(row[k_off + h * dim + d]));
    }
    if (threadIdx.x < cols)
      buf[2 * dim + threadIdx.x] = (c0 + threadIdx.x < vdim) ? lt_silu(to_f32(row[v_off + h * vdim + c0 + threadIdx.x])) : 0.f;
    __syncthreads();
    const float v = buf[2 * dim + col];
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < LT_ROWS; ++i) {
      const int d = part + i * parts;
      if (d < dim) {
        s[i] = fmaf(lam, s[i], buf[dim + d] * v);
        acc = fmaf(s[i], buf[d], acc);
      }
    }
    red[part * cols + col] = acc;
    __syncthreads();
    if (part == 0 && live) {
      float o = 0.f;
      for (int p = 0; p < parts; ++p) o += red[p * cols + col];
      out[(long long)t * heads * vdim + h * vdim + c0 + col] = o;
    }
    // the next token fills the other stage; `red` is rewritten only after the barrier behind that fill
  }
#pragma unroll
  for (int i = 0; i < LT_ROWS; ++i) {
    const int d = part + i * parts;
    if (live && d < dim) S[(long long)d * vdim] = s[i];
  }
}

// ---------------------------------------------------------------- by chunks
// Three launches, so that the chunks of a long prompt run side by side and only the cheap part is serial:
//   chunk:  per (chunk, head)   U = sum_j decay^(n-1-j) k_j v_j^T                       -> scratch[chunk]
//   scan:   per (request, head) for its chunks in order: scratch[chunk] <- S (the state BEFORE the chunk),
//                               S <- decay^n S + U;  at the end state <- S
//   out:    per (chunk, head)   a[i][j] = decay^(i-j) q_i . k_j (j <= i);  out_i = decay^(i+1) S_before^T q_i + sum_j a[i][j] v_j
// The products are 32-bit on the matrix unit (v_mfma_f32_32x32x2_f32, lane l holds row or column l % 32 and inner index l / 32 of
// an operand); chunks of 64 tokens halve what the states of 32 cost in memory traffic, and two blocks of 80 KB share a unit, so that
// one's loads and activations (25 instructions each, as many cycles as the products) run beside the other's products.
// 2,048 tokens of 16 heads of 128 x 128, a layer, microseconds: chunk 35, scan 16,
// out 49 (chunks of 32 in float FMA: 96, 70 and 49 for the state's part alone).
#define LC 64        // tokens of a chunk
#define LV 128       // columns (elements of v) a block takes
#define LD 128       // the largest key size

typedef float lt_f16 __attribute__((ext_vector_type(16)));
typedef __bf16 lt_b4 __attribute__((ext_vector_type(4)));

// Four elements of a row, as floats; `pieces`: rows begin on 4 elements.
__device__ __forceinline__ float4 lt_load4(const bf16_t* p, bool pieces, int left) {
  if (pieces && left >= 4) {
    const lt_b4 v = *(const lt_b4*)p;
    return {(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
  }
  return {left > 0 ? (float)p[0] : 0.f, left > 1 ? (float)p[1] : 0.f, left > 2 ? (float)p[2] : 0.f, left > 3 ? (float)p[3] : 0.f};
}
__device__ __forceinline__ float4 lt_load4(const float* p, bool pieces, int left) {
  if (pieces && left >= 4) return *(const float4*)p;
  return {left > 0 ? p[0] : 0.f, left > 1 ? p[1] : 0.f, left > 2 ? p[2] : 0.f, left > 3 ? p[3] : 0.f};
}
__device__ __forceinline__ float4 lt_silu4(float4 z) { return {lt_silu(z.x), lt_silu(z.y), lt_silu(z.z), lt_silu(z.w)}; }
__device__ __forceinline__ lt_f16 lt_mfma(float a, float b, lt_f16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
// Thread t brings elements 4 (t % 32) .. + 3 of tokens t / 32 + 8 i, i < LC / 8: raw numbers, zeros behind the chunk or the row.
template <typename T>
__device__ __forceinline__ void lt_load_rows(float4 (&v)[LC / 8], const T* rows, long long ld, int n, int width, bool pieces) {
  const int c = (threadIdx.x & 31) * 4, j0 = threadIdx.x >> 5;
#pragma unroll
  for (int i = 0; i < LC / 8; ++i) {
    const int j = j0 + 8 * i;
    v[i] = j < n && c < width ? lt_load4(rows + j * ld + c, pieces, width - c) : float4{0.f, 0.f, 0.f, 0.f};
  }
}

// grid (chunks, heads, column slices of LV); work: chunk -> (request, first token)
template <typename T>
__global__ void __launch_bounds__(256)
lightning_chunk_kernel(float* __restrict__ scratch, const T* __restrict__ proj, long long ld, int k_off, int v_off,
                       const int* __restrict__ work, const int* __restrict__ cu_seqlens, const float* __restrict__ decay, int heads,
                       int dim, int vdim, bool k_pieces, bool v_pieces) {
  __shared__ __attribute__((aligned(16))) float ks[LC * LD], vs[LC * LV], pw[LC];
  const int ch = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * LV;
  const int r = work[2 * ch], b0 = work[2 * ch + 1];
  const int n = min(LC, cu_seqlens[r + 1] - b0), ncols = min(LV, vdim - c0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, half = lane >> 5;
  {
    float4 k[LC / 8], v[LC / 8];
    lt_load_rows(k, proj + (long long)b0 * ld + k_off + h * dim, ld, n, dim, k_pieces);
    lt_load_rows(v, proj + (long long)b0 * ld + v_off + h * vdim + c0, ld, n, ncols, v_pieces);
    if (threadIdx.x < LC) pw[threadIdx.x] = powf(decay[h], (float)threadIdx.x);
    __syncthreads();
    const int c = (threadIdx.x & 31) * 4, j0 = threadIdx.x >> 5;
#pragma unroll
    for (int i = 0; i < LC / 8; ++i) {
      const int j = j0 + 8 * i;
      const float w = j < n ? pw[n - 1 - j] : 0.f;
      const float4 kk = lt_silu4(k[i]);
      *(float4*)(ks + j * LD + c) = float4{w * kk.x, w * kk.y, w * kk.z, w * kk.w};
      *(float4*)(vs + j * LV + c) = lt_silu4(v[i]);
    }
  }
  __syncthreads();
  // wave w: rows 32 w .. of U against all columns
  if (wave * 32 >= dim) return;
  lt_f16 acc[LV / 32] = {};
  const int tiles = (ncols + 31) / 32;
  const float *kr = ks + half * LD + wave * 32 + l32, *vr = vs + half * LV + l32;
  float a[2][4], b[2][4][LV / 32];
  auto read = [&](int set, int j) {      // tokens behind the chunk are zeros
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int row = min(j + 2 * u, LC - 2);
      a[set][u] = kr[row * LD];
#pragma unroll
      for (int t = 0; t < LV / 32; ++t) b[set][u][t] = vr[row * LV + t * 32];
    }
  };
  auto products = [&](int set) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = 0; t < LV / 32; ++t)
        if (t < tiles) acc[t] = lt_mfma(a[set][u], b[set][u][t], acc[t]);
  };
  read(0, 0);
  for (int j = 0; j < n; j += 16) {
    read(1, j + 8);
    products(0);
    read(0, j + 16);
    products(1);
  }
  float* U = scratch + (((long long)ch * heads + h) * dim) * vdim + c0;
#pragma unroll
  for (int t = 0; t < LV / 32; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int d = wave * 32 + i / 4 * 8 + half * 4 + i % 4, c = t * 32 + l32;
      if (d < dim && c < ncols) U[(long long)d * vdim + c] = acc[t][i];
    }
}

// grid (requests, heads, slices of the dim x vdim elements); req_chunks [requests + 1]: first chunk of each request.
// Bound by memory: a thread asks for eight chunks' numbers before it stores the first.
__global__ void __launch_bounds__(256)
lightning_scan_kernel(float* __restrict__ scratch, float* __restrict__ state, const int* __restrict__ slot_ids,
                      const int* __restrict__ req_chunks, const int* __restrict__ work,
                      const int* __restrict__ cu_seqlens, const float* __restrict__ decay, int heads, int dim, int vdim) {
  const int r = blockIdx.x, h = blockIdx.y;
  const int first = req_chunks[r], last = req_chunks[r + 1];
  if (last <= first) return;
  const int e = blockIdx.z * 256 + threadIdx.x;
  if (e >= dim * vdim) return;
  const float lam = decay[h], whole = powf(lam, (float)LC), rest = powf(lam, (float)(cu_seqlens[r + 1] - work[2 * (last - 1) + 1]));
  float* S = state + ((long long)slot_ids[r] * heads + h) * dim * vdim + e;
  const long long step = (long long)heads * dim * vdim;
  float* U = scratch + (long long)first * step + (long long)h * dim * vdim + e;
  float s = *S;
  for (int ch = first; ch < last; ch += 8, U += 8 * step) {
    float u[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) u[i] = U[min(i, last - 1 - ch) * step];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (ch + i < last) {
        U[i * step] = s;
        s = fmaf(ch + i + 1 < last ? whole : rest, s, u[i]);
      }
  }
  *S = s;
}

// grid as the chunk kernel
template <typename T>
__global__ void __launch_bounds__(256, 2)
lightning_out_kernel(float* __restrict__ out, const float* __restrict__ scratch, const T* __restrict__ proj, long long ld, int q_off,
                     int k_off, int v_off, const int* __restrict__ work, const int* __restrict__ cu_seqlens,
                     const float* __restrict__ decay, int heads, int dim, int vdim, bool k_pieces, bool v_pieces) {
  // q and k: element d of row j at d ^ (j % 32), so that 32 rows' element d lies in 32 banks; v takes k's place
  __shared__ __attribute__((aligned(16))) float qs[LC * LD], kv[LC * LD], as[3][32 * 33], pw[LC + 1];
  static_assert(LV == LD, "v takes k's place");
  const int ch = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * LV;
  const int r = work[2 * ch], b0 = work[2 * ch + 1];
  const int n = min(LC, cu_seqlens[r + 1] - b0), ncols = min(LV, vdim - c0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, half = lane >> 5;
  const int c = (tid & 31) * 4, j0 = tid >> 5;
  const T* rows = proj + (long long)b0 * ld;
  if (tid <= LC) pw[tid] = powf(decay[h], (float)tid);
  float4 v[LC / 8];
  {
    float4 q[LC / 8], k[LC / 8];
    lt_load_rows(q, rows + q_off + h * dim, ld, n, dim, k_pieces);
    lt_load_rows(k, rows + k_off + h * dim, ld, n, dim, k_pieces);
    lt_load_rows(v, rows + v_off + h * vdim + c0, ld, n, ncols, v_pieces);
#pragma unroll
    for (int i = 0; i < LC / 8; ++i) {
      const int j = j0 + 8 * i;
      const float4 a = lt_silu4(q[i]), b = lt_silu4(k[i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int at = j * LD + ((c + e) ^ (j & 31));
        qs[at] = (&a.x)[e], kv[at] = (&b.x)[e];
      }
    }
  }
  __syncthreads();
  // scores: waves 0 to 2 the tiles (0, 0), (1, 0), (1, 1) of 32 x 32 tokens
  const int ti = wave == 0 ? 0 : 1, tj = wave == 2 ? 1 : 0;
  if (wave < 3 && ti * 32 < n) {
    lt_f16 acc = {};
    const float *qr = qs + (ti * 32 + l32) * LD, *kr = kv + (tj * 32 + l32) * LD;
    float a[2][8], b[2][8];      // operands of 8 products are read while the 8 before them are made
    auto read = [&](int set, int d) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int at = min(d + 2 * u + half, LD - 1) ^ l32;      // behind the key size: zeros
        a[set][u] = qr[at], b[set][u] = kr[at];
      }
    };
    read(0, 0);
    for (int d = 0; d < dim; d += 32) {
      read(1, d + 16);
#pragma unroll
      for (int u = 0; u < 8; ++u) acc = lt_mfma(a[0][u], b[0][u], acc);
      read(0, d + 32);
#pragma unroll
      for (int u = 0; u < 8; ++u) acc = lt_mfma(a[1][u], b[1][u], acc);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {      // a lane holds column l32
      const int row = i / 4 * 8 + half * 4 + i % 4, back = ti * 32 + row - tj * 32 - l32;
      as[wave][row * 33 + l32] = back >= 0 ? acc[i] * pw[back] : 0.f;
    }
  }
  __syncthreads();
  bool odd = false;      // a value that is not finite: tokens before it must not meet it, not even times zero
#pragma unroll
  for (int i = 0; i < LC / 8; ++i) {
    const float4 x = lt_silu4(v[i]);
    odd = odd || !(fabsf(x.x) + fabsf(x.y) + fabsf(x.z) + fabsf(x.w) < INFINITY);
    *(float4*)(kv + (j0 + 8 * i) * LV + c) = x;
  }
  // wave w: columns 32 w .. of all rows; first the state's part
  const float* P = scratch + (((long long)ch * heads + h) * dim) * vdim + c0;
  const int col = wave * 32 + l32;
  const bool live = wave * 32 < ncols, two = n > 32;
  lt_f16 o[2] = {};
  if (live) {
    const float* p = P + min(col, ncols - 1);
    constexpr int G = 8;      // steps of two rows of the state that are asked for at once
    float now[G], next[G];
#pragma unroll
    for (int g = 0; g < G; ++g) now[g] = p[(long long)min(2 * g + half, dim - 1) * vdim];
    for (int d = 0; d < dim; d += 2 * G) {
#pragma unroll
      for (int g = 0; g < G; ++g) next[g] = p[(long long)min(d + 2 * (G + g) + half, dim - 1) * vdim];
#pragma unroll
      for (int g = 0; g < G; ++g)
        if (d + 2 * g < dim) {
          const int at = (d + 2 * g + half) ^ l32;
          o[0] = lt_mfma(qs[l32 * LD + at], now[g], o[0]);
          if (two) o[1] = lt_mfma(qs[(32 + l32) * LD + at], now[g], o[1]);
        }
#pragma unroll
      for (int g = 0; g < G; ++g) now[g] = next[g];
    }
  }
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[b][i] *= pw[b * 32 + i / 4 * 8 + half * 4 + i % 4 + 1];
  odd = __syncthreads_or(odd);
  if (!live) return;
  if (odd) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = i / 4 * 8 + half * 4 + i % 4;
        for (int j = 0; j <= b * 32 + row; ++j) o[b][i] = fmaf(as[b + (j >> 5)][row * 33 + (j & 31)], kv[j * LV + col], o[b][i]);
      }
  }
#pragma unroll 4
  for (int j = 0; j < 32 && !odd; j += 2) {
    const float a = kv[(j + half) * LV + col], b = kv[(32 + j + half) * LV + col];
    o[0] = lt_mfma(as[0][l32 * 33 + j + half], a, o[0]);
    if (two) {
      o[1] = lt_mfma(as[1][l32 * 33 + j + half], a, o[1]);
      o[1] = lt_mfma(as[2][l32 * 33 + j + half], b, o[1]);
    }
  }
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = b * 32 + i / 4 * 8 + half * 4 + i % 4;
      if (row < n && col < ncols) out[((long long)(b0 + row) * heads + h) * vdim + c0 + col] = o[b][i];
    }
}

extern "C" int jv_lightning_chunk_tokens() { return LC; }
extern "C" int jv_lightning_max_dim(int chunks) { return chunks ? LD : LT_ROWS * 256; }

template <typename T>
static int lightning_by_chunks(float* out, const T* proj, long long ld, int q_off, int k_off, int v_off, float* state, const int* slot_ids,
                               const int* cu_seqlens, const float* decay, int n_requests, int heads, int dim, int vdim, int chunks,
                               const int* work, const int* req_chunks, float* scratch, hipStream_t s) {
  if (dim > LD || dim % 4 || !work || !req_chunks || !scratch) return (int)hipErrorInvalidValue;
  const int slices = (vdim + LV - 1) / LV;
  const bool rows = ld % 4 == 0 && (uintptr_t)proj % (4 * sizeof(T)) == 0;      // begin on four elements
  const bool k_pieces = rows && q_off % 4 == 0 && k_off % 4 == 0, v_pieces = rows && v_off % 4 == 0 && vdim % 4 == 0;
  hipLaunchKernelGGL(lightning_chunk_kernel<T>, dim3(chunks, heads, slices), dim3(256), 0, s, scratch, proj, ld, k_off, v_off, work,
                     cu_seqlens, decay, heads, dim, vdim, k_pieces, v_pieces);
  hipLaunchKernelGGL(lightning_scan_kernel, dim3(n_requests, heads, (dim * vdim + 255) / 256), dim3(256), 0, s, scratch, state, slot_ids,
                     req_chunks, work, cu_seqlens, decay, heads, dim, vdim);
  hipLaunchKernelGGL(lightning_out_kernel<T>, dim3(chunks, heads, slices), dim3(256), 0, s, out, scratch, proj, ld, q_off, k_off, v_off,
                     work, cu_seqlens, decay, heads, dim, vdim, k_pieces, v_pieces);
  return JV_LAUNCH_CHECK();
}

// chunks = 0: token by token.  chunks = number of chunks (> 0): by chunks, with work [chunks][2] = (request,
// first token) in the order of requests and tokens, req_chunks [requests + 1], and scratch of
// chunks * heads * dim * vdim floats.
#define DEFINE_LIGHTNING(SUF, T)                                                                               \
  extern "C" int jv_lightning_##SUF(float* out, const void* proj, long long ld, int q_off, int k_off,          \
                                    int v_off, float* state, const int* slot_ids, const int* cu_seqlens,       \
                                    const float* decay, int n_requests, int heads, int dim, int vdim,          \
                                    int chunks, const int* work, const int* req_chunks, float* scratch,        \
                                    void* stream) {                                                            \
    if (n_requests <= 0 || heads <= 0) return 0;                                                               \
    if (dim <= 0 || vdim <= 0 || heads > 65535) return (int)hipErrorInvalidValue;                              \
    hipStream_t s = (hipStream_t)stream;                                                                       \
    if (chunks > 0) {                                                                                          \
      return lightning_by_chunks<T>(out, (const T*)proj, ld, q_off, k_off, v_off, state, slot_ids, cu_seqlens, \
                                    decay, n_requests, heads, dim, vdim, chunks, work, req_chunks, scratch, s);  \
    }                                                                                                          \
    int cols = 64;                       /* the widest slice that keeps a thread's rows in registers */        \
    while (cols > 1 && (cols / 2 >= vdim || (long long)dim * cols > 256LL * LT_ROWS)) cols /= 2;               \
    if ((long long)dim * cols > 256LL * LT_ROWS) return (int)hipErrorInvalidValue;                             \
    const int parts = 256 / cols;                                                                              \
    const size_t shmem = (2 * (2 * dim + cols) + parts * cols) * sizeof(float);                                \
    hipLaunchKernelGGL(lightning_steps_kernel<T>, dim3(n_requests, heads, (vdim + cols - 1) / cols),           \
                       dim3(256), shmem, s, out, (const T*)proj, ld, q_off, k_off, v_off,                      \
                       state, slot_ids, cu_seqlens, decay, heads, dim, vdim, cols);                            \
    return JV_LAUNCH_CHECK();                                                                                  \
  }

DEFINE_LIGHTNING(bf16, bf16_t)
DEFINE_LIGHTNING(f32, float)
