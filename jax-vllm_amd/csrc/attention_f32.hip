// Paged causal attention of the 32-bit path on the matrix cores in true 32-bit (v_mfma_f32_16x16x4_f32: float operands,
// products and sums), head sizes 32, 64, 96, 128 and 256, page sizes that are multiples of 4.  Same cache layout and same
// meaning of window, cap, keep and sinks as attention_generic.hip, which serves every other shape.
//
// A block takes 16 rows of one request and one kv head (a row: a (query, q head of the group) pair); its 4 waves take the
// keys in turns of 16 and meet once, at the end; while there are fewer blocks than compute units, blocks share out a
// row group's keys as well and a second kernel adds their parts.  S^T = K Q^T: a lane's 16 bytes of a key are 4 of its
// elements, four products.  A lane of the result holds 4 consecutive keys of one row, which is what the second product
// O^T += V^T P^T wants of P, against 16 bytes of V^T (4 consecutive slots of one element): nothing goes through LDS between
// the two, and K and V go from their pages straight into operands.  The next tile's keys are asked for before this
// tile's products.
//
// Measured at 16 q heads over 4 kv heads of 128 (before: one wave a (token, head), float FMA): three prompts of 1,003 tokens in
// all 36.8 us (864), 100 tokens behind 1,000 27.7 with two blocks a row group and 38.4 with one, one token each of 5 requests
// of 205..615 keys 9.5 and 6.7 for the parts (118.5).
// Rows in twos (32 a wave, each key feeding twice the products) take too many registers for two waves a SIMD: 43.3 us and
// 62 us behind 1,000.  Prompts are bound by the matrix unit (a 16 x 16 x 4 product keeps it for 32 cycles) and the
// exponentials, few tokens by what a compute unit pulls from memory.
#include "common.h"

typedef float af_f4 __attribute__((ext_vector_type(4)));
typedef float af_f4u __attribute__((ext_vector_type(4), aligned(4)));

struct AttnF32Args {
  float* out;
  const float* q;
  long long q_row_stride;
  const float* k_pages;
  const float* v_pages;
  const int* block_tables;
  int table_stride;
  const int* cu_seqlens;
  const int* context_lens;
  const int* work;            // [n_work, 2]: request, first row
  int page_size, nq, nkv;
  float scale;
  int window;                 // 0: all keys, > 0: the last so many, < 0: the query's own block of -window positions
  const float* sinks;
  float cap;
  int keep;
  float* parts;               // [n_work * nkv][splits][16][D + 4]: sums, then (maximum, sum of weights)
};

__device__ __forceinline__ int af_first_key(int pos, int window) {
  if (window == 0) return 0;
  if (window < 0) return pos - pos % -window;
  return pos - window + 1 > 0 ? pos - window + 1 : 0;
}

#define AF_WAVES 4
#define AF_ROWS 16

template <int DT>
__global__ void __launch_bounds__(64 * AF_WAVES) attn_f32_kernel(AttnF32Args p) {
  constexpr int D = 16 * DT, LROW = D + 4;
  extern __shared__ __attribute__((aligned(16))) float af_lds[];     // [AF_WAVES][AF_ROWS][LROW] | [AF_WAVES][AF_ROWS][2]
  float* ml = af_lds + AF_WAVES * AF_ROWS * LROW;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lq = lane >> 4;
  const int item = blockIdx.x / p.nkv, kvh = blockIdx.x - item * p.nkv;
  const int r = p.work[2 * item], m0 = p.work[2 * item + 1];
  const int G = p.nq / p.nkv, ps = p.page_size;
  const int q_start = p.cu_seqlens[r], ctx = p.context_lens[r];
  const int M = (p.cu_seqlens[r + 1] - q_start) * G;
  const int* table = p.block_tables + (long long)r * p.table_stride;

  // this lane's row, its position and first key; rows behind the last one repeat it and are not stored
  const int row = m0 + li < M ? m0 + li : M - 1;
  const int pos = ctx + row / G;
  const int first = af_first_key(pos, p.window);
  af_f4 qf[DT];
  const float* qrow = p.q + (long long)(q_start + row / G) * p.q_row_stride + (long long)(kvh * G + row % G) * D + lq * 4;
#pragma unroll
  for (int d = 0; d < DT; ++d) qf[d] = *(const af_f4u*)(qrow + d * 16);

  // tiles of 16 keys: those of the kept first keys in front of the first row's first key, then from there to the last row
  const int last = ctx + ((m0 + AF_ROWS < M ? m0 + AF_ROWS : M) - 1) / G;      // the last key any row sees
  const int min_pos = ctx + m0 / G;
  const int full_from = af_first_key(last, p.window);         // from here to min_pos every row sees every key
  const int begin_tile = af_first_key(min_pos, p.window) / 16;
  const int kept_tiles = (p.keep + 15) / 16 < begin_tile ? (p.keep + 15) / 16 : begin_tile;
  const int tiles = kept_tiles + last / 16 - begin_tile + 1;
  auto tile_key = [&](int t) { return (t < kept_tiles ? t : begin_tile + t - kept_tiles) * 16; };

  af_f4 o[DT];
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = af_f4{0.f, 0.f, 0.f, 0.f};

  // a lane reads 16 bytes of key j0 + li and, of each of its value elements, the slots of keys j0 + 4 lq .. + 3; keys
  // behind the last one stand for the last one (their scores are masked, their values taken out)
  af_f4 kf[DT], kn[DT];
  long long v_at = 0, v_next = 0;
  auto load_keys = [&](int t, af_f4* k, long long& v_offset) {
    const int j0 = tile_key(t);
    const int kj = j0 + li < last ? j0 + li : last;
    const int vj = j0 + lq * 4 <= last ? j0 + lq * 4 : last & ~3;
    const long long kpage = table[kj / ps], vpage = table[vj / ps];
    const float* kr = p.k_pages + ((kpage * p.nkv + kvh) * ps + kj % ps) * (long long)D + lq * 4;
#pragma unroll
    for (int d = 0; d < DT; ++d) k[d] = *(const af_f4u*)(kr + d * 16);
    v_offset = ((vpage * p.nkv + kvh) * (long long)D + li) * ps + vj % ps;
  };
  const int step = AF_WAVES * gridDim.y, own = blockIdx.y * AF_WAVES + wave;
  if (own < tiles) load_keys(own, kf, v_at);
  for (int t = own; t < tiles; t += step) {
    const int j0 = tile_key(t);
    af_f4 vf[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d) vf[d] = *(const af_f4u*)(p.v_pages + v_at + (long long)d * 16 * ps);
    load_keys(t + step < tiles ? t + step : t, kn, v_next);       // never skipped: a conditional load would be waited for at once
    __builtin_amdgcn_sched_barrier(0);

    const bool whole = j0 >= full_from && j0 + 15 <= min_pos;     // every row sees every key of the tile
    bool careful = false;
    if (!whole) {
      // values behind the last key are nobody's; a value that is not finite must not reach rows that do not see its key
      bool odd = false;
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (j0 + lq * 4 + e > last) vf[d][e] = 0.f;
          odd |= !(fabsf(vf[d][e]) < INFINITY);
        }
      careful = __any(odd);
    }
    af_f4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[d][e], qf[d][e], s, 0, 0, 0);
    float top = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = j0 + lq * 4 + e;
      float x = s[e] * p.scale;
      if (p.cap > 0.f) x = p.cap * tanhf(x / p.cap);
      if (!whole && !(j <= pos && (j >= first || j < p.keep))) x = -INFINITY;
      s[e] = x;
      top = fmaxf(top, x);
    }
    top = fmaxf(top, __shfl_xor(top, 16));
    top = fmaxf(top, __shfl_xor(top, 32));
    const float m_new = fmaxf(m, top);
    const float ref = m_new == -INFINITY ? 0.f : m_new;            // no key of this row yet: everything is exp(-inf)
    const float alpha = expf(m - ref);
    af_f4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = expf(s[e] - ref);
    l = l * alpha + ((w[0] + w[1]) + (w[2] + w[3]));               // this lane's keys; the row's lanes meet at the end
    m = m_new;
#pragma unroll
    for (int d = 0; d < DT; ++d) o[d] *= alpha;
    if (!careful) {
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[d][e], w[e], o[d], 0, 0, 0);
    } else {
      for (int kk = 0; kk < 16; ++kk) {
        const int j = j0 + kk;
        const float wk = __shfl(kk % 4 == 0 ? w[0] : kk % 4 == 1 ? w[1] : kk % 4 == 2 ? w[2] : w[3], kk / 4 * 16 + li);
        if (!(j <= pos && (j >= first || j < p.keep))) continue;    // pos <= last: a key that is seen is the request's own
        const float* vr = p.v_pages + ((table[j / ps] * (long long)p.nkv + kvh) * D + lq * 4) * ps + j % ps;
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[d][e] += wk * vr[(long long)(d * 16 + e) * ps];
      }
    }
#pragma unroll
    for (int d = 0; d < DT; ++d) kf[d] = kn[d];
    v_at = v_next;
  }

  // the waves meet: a lane holds elements 16 d + 4 lq .. + 3 of its row
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  float* dst = af_lds + (wave * AF_ROWS + li) * LROW + lq * 4;
#pragma unroll
  for (int d = 0; d < DT; ++d) *(af_f4*)(dst + d * 16) = o[d];
  if (lq == 0) {
    ml[(wave * AF_ROWS + li) * 2] = m;
    ml[(wave * AF_ROWS + li) * 2 + 1] = l;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < AF_ROWS * (D / 4); i += 64 * AF_WAVES) {
    const int rr = i / (D / 4), d = (i - rr * (D / 4)) * 4;
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) top = fmaxf(top, ml[(w * AF_ROWS + rr) * 2]);
    const float ref = top == -INFINITY ? 0.f : top;
    af_f4 sum = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) {
      const float f = expf(ml[(w * AF_ROWS + rr) * 2] - ref);
      den += f * ml[(w * AF_ROWS + rr) * 2 + 1];
      sum += f * *(const af_f4*)(af_lds + (w * AF_ROWS + rr) * LROW + d);
    }
    if (gridDim.y > 1) {                                            // this block's part: sums relative to its own maximum
      float* part = p.parts + (((long long)blockIdx.x * gridDim.y + blockIdx.y) * AF_ROWS + rr) * (D + 4);
      *(af_f4*)(part + d) = sum;
      if (d == 0) *(af_f4*)(part + D) = af_f4{top, den, 0.f, 0.f};
    } else if (m0 + rr < M) {
      const int qi = (m0 + rr) / G, h = kvh * G + (m0 + rr) - qi * G;
      if (p.sinks) den += expf(p.sinks[h] - top);
      float* out = p.out + (long long)(q_start + qi) * p.nq * D + (long long)h * D + d;
#pragma unroll
      for (int e = 0; e < 4; ++e) out[e] = sum[e] / den;
    }
  }
}

// Adds the parts of the blocks that shared out a row group's keys, in their order: a block a (work item, kv head).
__global__ void __launch_bounds__(256) attn_f32_merge_kernel(AttnF32Args p, int splits, int D) {
  const int item = blockIdx.x / p.nkv, kvh = blockIdx.x - item * p.nkv;
  const int r = p.work[2 * item], m0 = p.work[2 * item + 1], G = p.nq / p.nkv;
  const int q_start = p.cu_seqlens[r], M = (p.cu_seqlens[r + 1] - q_start) * G;
  const int rows = M - m0 < AF_ROWS ? M - m0 : AF_ROWS;
  for (int i = threadIdx.x; i < rows * (D / 4); i += 256) {
    const int rr = i / (D / 4), d = (i - rr * (D / 4)) * 4;
    const float* part = p.parts + ((long long)blockIdx.x * splits * AF_ROWS + rr) * (D + 4);
    const long long stride = (long long)AF_ROWS * (D + 4);
    float top = -INFINITY;
    for (int s = 0; s < splits; ++s) top = fmaxf(top, part[s * stride + D]);
    const float ref = top == -INFINITY ? 0.f : top;
    af_f4 sum = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
    for (int s = 0; s < splits; ++s) {
      const float f = expf(part[s * stride + D] - ref);
      den += f * part[s * stride + D + 1];
      sum += f * *(const af_f4*)(part + s * stride + d);
    }
    const int qi = (m0 + rr) / G, h = kvh * G + (m0 + rr) - qi * G;
    if (p.sinks) den += expf(p.sinks[h] - top);
    float* out = p.out + (long long)(q_start + qi) * p.nq * D + (long long)h * D + d;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = sum[e] / den;
  }
}

template <int DT>
static int attn_f32_launch(const AttnF32Args& a, int n_work, int splits, hipStream_t stream) {
  constexpr size_t shmem = AF_WAVES * AF_ROWS * (16 * DT + 4 + 2) * sizeof(float);
  static_assert(shmem <= 160 * 1024, "the waves' results must fit a compute unit's LDS");
  if (shmem > 64 * 1024) {
    static bool raised = false;
    if (!raised) {
      const hipError_t e = hipFuncSetAttribute((const void*)attn_f32_kernel<DT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
      if (e != hipSuccess) return (int)e;
      raised = true;
    }
  }
  hipLaunchKernelGGL((attn_f32_kernel<DT>), dim3(n_work * a.nkv, splits), dim3(64 * AF_WAVES), shmem, stream, a);
  if (splits > 1)
    hipLaunchKernelGGL(attn_f32_merge_kernel, dim3(n_work * a.nkv), dim3(256), 0, stream, a, splits, 16 * DT);
  return JV_LAUNCH_CHECK();
}

extern "C" int jv_attn_f32_rows() { return AF_ROWS; }
extern "C" int jv_attn_f32_tile_keys() { return 16 * AF_WAVES; }      // keys that a block takes at once

// Floats of `parts` for `splits` > 1 blocks a row group.
extern "C" long long jv_attn_f32_part_floats(int n_work, int nkv, int splits, int D) {
  return splits > 1 ? (long long)n_work * nkv * splits * AF_ROWS * (D + 4) : 0;
}

extern "C" int jv_attn_f32(float* out, const float* q, long long q_row_stride, const float* k_pages, const float* v_pages,
                           const int* block_tables, int table_stride, const int* cu_seqlens, const int* context_lens,
                           const int* work, int n_work, int splits, float* parts, int page_size, int nq, int nkv, int D,
                           float scale, int window, const float* sinks, float cap, int keep, void* stream) {
  if (n_work <= 0) return 0;
  if (nkv <= 0 || nq % nkv != 0 || page_size <= 0 || page_size % 4 != 0 || keep < 0 || (long long)n_work * nkv > 0x7fffffffll ||
      splits < 1 || splits > 65535 || (splits > 1 && !parts))
    return (int)hipErrorInvalidValue;
  const AttnF32Args a = {out, q, q_row_stride, k_pages, v_pages, block_tables, table_stride, cu_seqlens, context_lens, work,
                         page_size, nq, nkv, scale, window, sinks, cap, keep, parts};
  const hipStream_t st = (hipStream_t)stream;
  switch (D) {
    case 32: return attn_f32_launch<2>(a, n_work, splits, st);
    case 64: return attn_f32_launch<4>(a, n_work, splits, st);
    case 96: return attn_f32_launch<6>(a, n_work, splits, st);
    case 128: return attn_f32_launch<8>(a, n_work, splits, st);
    case 256: return attn_f32_launch<16>(a, n_work, splits, st);
    default: return (int)hipErrorInvalidValue;
  }
}
