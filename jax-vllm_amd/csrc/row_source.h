// Rows of x that a product of one or two rows makes for itself, in LDS, instead of reading what a launch before it left: the
// residual step with the norm's weight (the scale is left to whoever holds the whole row), or the splits of a decode attention.
//
// At one row such a launch (128 threads a share of the row, or a head) costs its start and two round trips, 2.3 to 3.2 us of a
// layer's 90 or 42, and what it leaves is read by every block of the product; the blocks read its inputs instead, beside their first
// rows of W.  Three rows or more would draw more from the L2s than the launch costs (4 parts of 4,096 floats a row and block).
#pragma once
#include "common.h"

struct RowSource {
  // ROWS_RESIDUAL: v = h + (parts[0] + parts[1] + ...), x = v * weight in bf16; one block of every range of columns leaves v in h_out
  // and, where a row's columns are shared out, the sum of its squares in ssq_out[row * 16 + range]
  const float* h;
  float* h_out;
  const float* parts;
  long long part_stride;
  int n_parts;                 // 0 to 4
  const float* weight;
  float* ssq_out;
  float inv_width, eps;
  // ROWS_SPLITS: x = the heads that attn_decode_merge_kernel would leave (the same order of sums)
  const float* part_acc;       // [row][head][split][head_dim]
  const float2* part_ml;       // [row][head][split] (max, sum)
  const float* sinks;
  int splits, heads, head_dim;
};
enum { ROWS_GIVEN = 0, ROWS_RESIDUAL = 1, ROWS_SPLITS = 2 };

typedef __bf16 row_bf16x4 __attribute__((ext_vector_type(4)));
typedef float row_f32x4 __attribute__((ext_vector_type(4)));

// KB columns from k0 on of MR rows (MR = 1 or 2, no more than there are), by the 512 threads of a block in pieces of 4 columns.  ask() only
// loads; give() leaves the rows in xs (row_stride elements apart) and, for ROWS_RESIDUAL, the wave's sums of squares in sq[row], in every lane.
template <int SRC, int MR, int KB> struct RowMaker {
  static constexpr int IT = (KB + 2047) / 2048;
  row_f32x4 v[MR][IT], e[MR][IT][4], w[IT];
  static __device__ __forceinline__ int column(int i) { return (int)threadIdx.x * 4 + i * 2048; }

  __device__ __forceinline__ void ask(const RowSource& s, int k0, int K) {
    if constexpr (SRC == ROWS_RESIDUAL) {
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        const int c = k0 + min(column(i), KB - 4);      // threads without columns of their own read the last ones again
        w[i] = *(const row_f32x4*)(s.weight + c);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
          v[m][i] = *(const row_f32x4*)(s.h + (long long)m * K + c);
#pragma unroll
          for (int q = 0; q < 4; ++q) {                 // parts that are not there are read as the first one, or as h, and not added
            const float* p = s.n_parts ? s.parts + (q < s.n_parts ? q : 0) * s.part_stride : s.h;
            e[m][i][q] = *(const row_f32x4*)(p + (long long)m * K + c);
          }
        }
      }
    }
  }
  __device__ __forceinline__ void give(const RowSource& s, int k0, int K, bool leave, bf16_t* xs, int row_stride, float (&sq)[MR]) {
    if constexpr (SRC == ROWS_RESIDUAL) {
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < IT; ++i) {
          const int c = column(i);
          if (s.n_parts) {
            row_f32x4 d = e[m][i][0];
#pragma unroll
            for (int q = 1; q < 4; ++q)
              if (q < s.n_parts) d += e[m][i][q];
            v[m][i] += d;
          }
          if (c < KB) {
            const row_f32x4 x = v[m][i];
            sum += x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3];
            row_bf16x4 b;
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = from_f32<bf16_t>(x[j] * w[i][j]);
            *(row_bf16x4*)(xs + m * row_stride + c) = b;
            if (leave) *(row_f32x4*)(s.h_out + (long long)m * K + k0 + c) = x;
          }
        }
        sq[m] = wave_sum(sum);
      }
    } else if constexpr (SRC == ROWS_SPLITS) {
#pragma unroll
      for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int i = 0; i < IT; ++i) {
          const int c = k0 + min(column(i), KB - 4), head = c / s.head_dim;
          const long long base = ((long long)m * s.heads + head) * s.splits;
          const float2* ml = s.part_ml + base;
          const float* pa = s.part_acc + base * s.head_dim + (c - head * s.head_dim);
          float mx = -INFINITY, den = 0.f;
          row_f32x4 num = {0.f, 0.f, 0.f, 0.f};
          for (int s0 = 0; s0 < s.splits; s0 += 8) {
            float2 l[8];
            row_f32x4 a[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              const int at = min(s0 + q, s.splits - 1);
              l[q] = ml[at];
              a[q] = *(const row_f32x4*)(pa + (long long)at * s.head_dim);
            }
            float bm = mx;
#pragma unroll
            for (int q = 0; q < 8; ++q) bm = fmaxf(bm, l[q].x);
            if (bm == -INFINITY) continue;
            const float keep = __builtin_amdgcn_exp2f(mx - bm);
            num *= keep;
            den *= keep;
            mx = bm;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              // an empty split may hold anything: it gets no weight and is not read into the sum
              const bool live = s0 + q < s.splits && l[q].x != -INFINITY;
              const float f = live ? __builtin_amdgcn_exp2f(l[q].x - mx) : 0.f;
#pragma unroll
              for (int j = 0; j < 4; ++j) num[j] += live ? a[q][j] * f : 0.f;
              den += live ? l[q].y * f : 0.f;
            }
          }
          if (s.sinks && mx != -INFINITY) den += __builtin_amdgcn_exp2f(s.sinks[head] * 1.4426950408889634f - mx);
          if (column(i) < KB) {
            row_bf16x4 b;
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = from_f32<bf16_t>(num[j] / den);
            *(row_bf16x4*)(xs + m * row_stride + column(i)) = b;
          }
        }
    }
  }
};
