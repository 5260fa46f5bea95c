// The writer of many tokens' v heads into transposed pages, shared by the attention-input kernels.
#pragma once
#include "common.h"

// The v heads of many tokens into their transposed pages [page][kv head][Dp][slot] (a head of D elements, a page
// head of Dp >= D: the pad is never written).  A token's v heads start `v_off` elements into its row of
// `row_stride` elements; `v_scale` multiplies the values, behind an optional bias (`bias`, of the v heads' columns) and an
// optional blend with the same token's values of another layer, (1 - mix) v + mix first (`first`: rows of `first_stride`
// elements that begin with those values).  Token by token
// every element would be a store of its own, 2 bytes every `page_size` elements; here a block takes
// 16 consecutive tokens of one kv head through LDS and writes, for every element of the head, 8
// tokens at once (16 bytes) wherever 8 consecutive tokens have 8 consecutive slots that start at a
// multiple of 8 (the usual case for a prompt), and element by element elsewhere.
template <typename T> struct alignas(16) Pack8 { T v[8]; };

// The tokens' slots come in beside their values: looked up one after another where they are needed they were a chain of up to 9 round
// trips (2,048 tokens of 8 heads of 128 5.5 us as profiled, 1,501 beside 24 that decode 8.9).
template <typename T>
struct VPages {
  const T* src;                // the first token's first v head
  long long row_stride;
  const int* slot_mapping;
  T* v_pages;
  int page_size, n_tokens, nkv, D, Dp;
  float v_scale;
  const float* bias;
  const T* first;
  long long first_stride;
  float mix;
};
// A block of 256 threads: tokens 16 at .. of kv head kvh; LDS for v_tile_bytes.
template <typename T>
__device__ __forceinline__ void v_pages_tile(const VPages<T>& p, int at, int kvh, unsigned char* lds) {
  constexpr int EP = 16 / (int)sizeof(T);          // elements of a 16-byte piece
  int* slots = (int*)lds;                          // [16], -1 behind the last token
  T* tile = (T*)(lds + 64);                        // [16][D + EP]
  const int LROW = p.D + EP, t0 = at * 16;
  if (threadIdx.x < 16) slots[threadIdx.x] = t0 + (int)threadIdx.x < p.n_tokens ? p.slot_mapping[t0 + threadIdx.x] : -1;
  const T* src = p.src + (long long)kvh * p.D;
  const int ppt = p.D / EP;
  for (int i = threadIdx.x; i < 16 * ppt; i += 256) {
    const int j = i / ppt, c = (i - j * ppt) * EP;
    if (t0 + j >= p.n_tokens) continue;
    typedef T tv __attribute__((ext_vector_type(EP)));
    tv v = *(const tv*)(src + (t0 + j) * p.row_stride + c);
    if (p.bias) {
      float b[EP];
      load_floats<EP>(p.bias + kvh * p.D + c, b);
#pragma unroll
      for (int e = 0; e < EP; ++e) v[e] = from_f32<T>(to_f32<T>(v[e]) + b[e]);
    }
    if (p.first) {
      const T* f = p.first + (t0 + j) * p.first_stride + (long long)kvh * p.D + c;
#pragma unroll
      for (int e = 0; e < EP; ++e) v[e] = from_f32<T>((1.f - p.mix) * to_f32<T>(v[e]) + p.mix * to_f32<T>(f[e]));
    }
    *(tv*)(tile + j * LROW + c) = v;
  }
  __syncthreads();
  for (int item = threadIdx.x; item < 2 * p.D; item += 256) {
    const int half = item / p.D, d = item - half * p.D;
    const int* s = slots + half * 8;
    const int s0 = s[0];
    bool run = s0 >= 0 && (s0 & 7) == 0;
#pragma unroll
    for (int j = 1; j < 8; ++j) run = run & (s[j] == s0 + j);
    const T* col = tile + (half * 8) * LROW + d;
    if (run) {
      const long long page = s0 / p.page_size;
      const int off = (int)(s0 - page * p.page_size);
      Pack8<T> v;
#pragma unroll
      for (int j = 0; j < 8; ++j) v.v[j] = p.v_scale == 1.f ? col[j * LROW] : from_f32<T>(to_f32(col[j * LROW]) * p.v_scale);
      *(Pack8<T>*)(p.v_pages + ((page * p.nkv + kvh) * p.Dp + d) * (long long)p.page_size + off) = v;
    } else {
      for (int j = 0; j < 8; ++j) {
        if (s[j] < 0) continue;
        const long long page = s[j] / p.page_size;
        const int off = (int)(s[j] - page * p.page_size);
        p.v_pages[((page * p.nkv + kvh) * p.Dp + d) * (long long)p.page_size + off] =
            p.v_scale == 1.f ? col[j * LROW] : from_f32<T>(to_f32(col[j * LROW]) * p.v_scale);
      }
    }
  }
}
template <typename T> static size_t v_tile_bytes(int D) { return 64 + (size_t)16 * (D + 16 / sizeof(T)) * sizeof(T); }

template <typename T>
__global__ void __launch_bounds__(256) v_pages_write_kernel(VPages<T> p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char v_tile_mem[];
  v_pages_tile<T>(p, blockIdx.x, blockIdx.y, v_tile_mem);
}

// Whether the v heads of a step go through v_pages_write_kernel: many tokens, and sizes that keep
// its 16-byte pieces aligned (the caller also checks the row stride and the v heads' offset where they are its own).
template <typename T>
static bool v_written_by_tile(const void* k_pages, int n_tokens, int page_size, int D) {
  return k_pages != nullptr && n_tokens >= 256 && page_size % 8 == 0 && D % (16 / (int)sizeof(T)) == 0;
}

template <typename T>
static int launch_v_pages_write(const void* qkv, long long row_stride, long long v_off, const int* slot_mapping,
                                void* v_pages, int page_size, int n_tokens, int nkv, int D, int Dp, float v_scale,
                                void* stream, const float* bias = nullptr, const void* first = nullptr,
                                long long first_stride = 0, float mix = 0.f) {
  if (nkv > 65535) return (int)hipErrorInvalidValue;
  const VPages<T> p{(const T*)qkv + v_off, row_stride, slot_mapping, (T*)v_pages, page_size, n_tokens, nkv, D, Dp, v_scale, bias,
                    (const T*)first, first_stride, mix};
  hipLaunchKernelGGL(v_pages_write_kernel<T>, dim3((n_tokens + 15) / 16, nkv), dim3(256), v_tile_bytes<T>(D), (hipStream_t)stream, p);
  return JV_LAUNCH_CHECK();
}

