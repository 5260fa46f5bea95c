// Paged causal attention of the 32-bit path on the matrix cores in true 32-bit (v_mfma_f32_16x16x4_f32: float operands,
// products and sums), head sizes 32, 64, 96, 128 and 256, page sizes that are multiples of 4.  Same cache layout and same
// meaning of window, cap, keep and sinks as attention_generic.hip, which serves every other shape.
//
// A block takes 16 rows of one request and one kv head (a row: a (query, q head of the group) pair).  Keys are counted in tiles
// of 16 and ranges of 16 tiles from key 0; in a range wave w of the 4 takes tiles w, w + 4, ..., and a row's result is, for
// each wave, its ranges' sums added in ascending order, then the four waves'.  So the order depends on the query's position and
// what it sees alone: not on the other requests, the cut into portions or who makes the sums.  While there are fewer blocks than
// compute units, an item's blocks share out its ranges and a second kernel adds their parts, with the same operations.
// S^T = K Q^T: a lane's 16 bytes of a key are 4 of its elements, four products.  A lane of the result holds 4 consecutive
// keys of one row, which is what the second product O^T += V^T P^T wants of P, against 16 bytes of V^T (4 consecutive slots
// of one element): nothing goes through LDS between the two, and K and V go from their pages straight into operands.  The next
// tile's keys are asked for before this tile's products.
//
// Measured at 16 q heads over 4 kv heads of 128, microseconds (one wave a (token, head), float FMA): three prompts of 1,003 tokens
// in all 40 (864), 4,000 tokens 813, 100 tokens behind 1,000 32 with two blocks an item and 37 with one, one token each of 5
// requests of 205..615 keys 15.6 (118), of 16 of 1,000 keys 18.9 with 4 blocks an item and 35 with one.  Ranges of 8 tiles: 41, 822, 35, 13.0,
// 22.8; of 32: 39, 815, 29, 21.5, 23.5.  The order costs prompts 4 to 8 % beside one chain a wave (38, 757).
// Rows in twos (32 a wave, each key feeding twice the products) take too many registers for two waves a SIMD.  Prompts are bound
// by the matrix unit (a 16 x 16 x 4 product keeps it for 32 cycles) and the exponentials, few tokens by what a compute unit
// pulls from memory.
#include "common.h"
#include "f32_terms.h"

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
  float* parts;               // [n_work * nkv][part_ranges][AF_WAVES][16][D + 4]: sums, then (maximum, sum of weights)
  int part_ranges;
  unsigned* terms;            // null, or out's rows as terms too (f32_terms.h); one block an item only
  int fragments;
};

__device__ __forceinline__ int af_first_key(int pos, int window) {
  if (window == 0) return 0;
  if (window < 0) return pos - pos % -window;
  return pos - window + 1 > 0 ? pos - window + 1 : 0;
}

#define AF_WAVES 4
#define AF_ROWS 16
#define AF_RANGE 16      // tiles of 16 keys

// The tiles a work item walks: those of the kept first keys in front of the first row's first key, then from there to the
// last row's position.  Tiles and ranges are counted from key 0, whatever else is in the item.
struct AfWalk {
  int rows, last, min_pos, begin_tile, kept_tiles, kept_ranges, first_range, ranges;
  __device__ AfWalk(const AttnF32Args& p, int ctx, int M, int G, int m0) {
    rows = M - m0 < AF_ROWS ? M - m0 : AF_ROWS;
    last = ctx + (m0 + rows - 1) / G;                          // the last key any row sees
    min_pos = ctx + m0 / G;
    begin_tile = af_first_key(min_pos, p.window) / 16;
    kept_tiles = (p.keep + 15) / 16 < begin_tile ? (p.keep + 15) / 16 : begin_tile;
    first_range = begin_tile / AF_RANGE;
    kept_ranges = (kept_tiles + AF_RANGE - 1) / AF_RANGE;      // those that lie in front of first_range
    if (kept_ranges > first_range) kept_ranges = first_range;
    ranges = kept_ranges + last / (16 * AF_RANGE) - first_range + 1;
  }
  __device__ int first_tile(int i) const { return (i < kept_ranges ? i : first_range + i - kept_ranges) * AF_RANGE; }
  // whether the item's blocks share out its ranges; else (one is enough, or they have no room) the first takes all
  __device__ bool shared(const AttnF32Args& p, int blocks) const { return blocks > 1 && ranges > 1 && ranges <= p.part_ranges; }
};

// What follows is spelled out operation by operation: blocks that keep their sums and the kernel that adds parts must round alike.

// Adds a range's sums (relative to its own maximum) to those of the ranges before it: the factors.  A range in which a row sees
// nothing (maximum -inf, zeros) leaves the row's sums as they are, to the bit.
__device__ __forceinline__ void af_fold(float& top, float& den, float part_top, float part_den, float& a, float& b) {
  const float both = fmaxf(top, part_top), ref = both == -INFINITY ? 0.f : both;
  a = expf(top - ref), b = expf(part_top - ref);
  den = fmaf(b, part_den, a * den);
  top = both;
}
__device__ __forceinline__ void af_add(af_f4& sum, float a, float b, af_f4 part) {
#pragma unroll
  for (int e = 0; e < 4; ++e) sum[e] = fmaf(b, part[e], a * sum[e]);
}

// The waves' sums of one row: 4 elements of the result.
__device__ __forceinline__ af_f4 af_meet(const float* top, const float* den, const af_f4* sum, const float* sink) {
  float most = top[0];
#pragma unroll
  for (int w = 1; w < AF_WAVES; ++w) most = fmaxf(most, top[w]);
  const float ref = most == -INFINITY ? 0.f : most;
  af_f4 v = {0.f, 0.f, 0.f, 0.f};
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < AF_WAVES; ++w) {
    const float f = expf(top[w] - ref);
    total = fmaf(f, den[w], total);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = fmaf(f, sum[w][e], v[e]);
  }
  if (sink) total += expf(*sink - most);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = v[e] / total;
  return v;
}

template <int DT>
__global__ void __launch_bounds__(64 * AF_WAVES) __attribute__((amdgpu_waves_per_eu(DT <= 8 ? 2 : 1))) attn_f32_kernel(AttnF32Args p) {
  constexpr int D = 16 * DT, LROW = D + 4;
  extern __shared__ __attribute__((aligned(16))) float af_lds[];     // [AF_WAVES][AF_ROWS][LROW] | [AF_WAVES][AF_ROWS][2]
  float* ml = af_lds + AF_WAVES * AF_ROWS * LROW;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, lq = lane >> 4;
  const int item = blockIdx.x / p.nkv, kvh = blockIdx.x - item * p.nkv;
  const int r = p.work[2 * item], m0 = p.work[2 * item + 1];
  const int G = p.nq / p.nkv, ps = p.page_size;
  const int q_start = p.cu_seqlens[r], ctx = p.context_lens[r];
  const int M = (p.cu_seqlens[r + 1] - q_start) * G;
  const int* table = p.block_tables + (long long)r * p.table_stride;

  const AfWalk walk(p, ctx, M, G, m0);
  const bool shared = walk.shared(p, gridDim.y);
  if (!shared && blockIdx.y > 0) return;
  const int i_begin = shared ? (int)((long long)walk.ranges * blockIdx.y / gridDim.y) : 0;
  const int i_end = shared ? (int)((long long)walk.ranges * (blockIdx.y + 1) / gridDim.y) : walk.ranges;
  if (i_begin >= i_end) return;

  // this lane's row, its position and first key; rows behind the last one repeat it and are not stored
  const int row = m0 + li < M ? m0 + li : M - 1;
  const int pos = ctx + row / G;
  const int first = af_first_key(pos, p.window);
  af_f4 qf[DT];
  const float* qrow = p.q + (long long)(q_start + row / G) * p.q_row_stride + (long long)(kvh * G + row % G) * D + lq * 4;
#pragma unroll
  for (int d = 0; d < DT; ++d) qf[d] = *(const af_f4u*)(qrow + d * 16);

  const int last = walk.last, min_pos = walk.min_pos;
  const int full_from = af_first_key(last, p.window);         // from here to min_pos every row sees every key
  // this wave's tiles: every AF_WAVES-th of all; from t on, the first that the item walks
  auto walked = [&](int t) {
    return t >= walk.kept_tiles && t < walk.begin_tile ? walk.begin_tile + ((wave - walk.begin_tile) & (AF_WAVES - 1)) : t;
  };
  auto stop_of = [&](int i) { return min(walk.first_tile(i) + AF_RANGE - 1, last / 16); };
  const int stop_all = stop_of(i_end - 1);

  // a lane reads 16 bytes of key j0 + li and, of each of its value elements, the slots of keys j0 + 4 lq .. + 3; keys
  // behind the last one stand for the last one (their scores are masked, their values taken out)
  af_f4 kf[DT], kn[DT];
  long long v_at = 0, v_next = 0;
  auto load_keys = [&](int t, af_f4* k, long long& v_offset) {
    const int j0 = t * 16;
    const int kj = j0 + li < last ? j0 + li : last;
    const int vj = j0 + lq * 4 <= last ? j0 + lq * 4 : last & ~3;
    const long long kpage = table[kj / ps], vpage = table[vj / ps];
    const float* kr = p.k_pages + ((kpage * p.nkv + kvh) * ps + kj % ps) * (long long)D + lq * 4;
#pragma unroll
    for (int d = 0; d < DT; ++d) k[d] = *(const af_f4u*)(kr + d * 16);
    v_offset = ((vpage * p.nkv + kvh) * (long long)D + li) * ps + vj % ps;
  };
  // the sums of the wave's ranges so far
  af_f4 o_all[DT];
  float m_all = -INFINITY, l_all = 0.f;
#pragma unroll
  for (int d = 0; d < DT; ++d) o_all[d] = af_f4{0.f, 0.f, 0.f, 0.f};

  int t = walked(walk.first_tile(i_begin) + wave);
  if (t <= stop_all) load_keys(t, kf, v_at);
  for (int range = i_begin; range < i_end; ++range) {
    const int stop = stop_of(range);
    af_f4 o[DT];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int d = 0; d < DT; ++d) o[d] = af_f4{0.f, 0.f, 0.f, 0.f};
    while (t <= stop) {
      const int j0 = t * 16, t_next = walked(t + AF_WAVES);
      af_f4 vf[DT];
#pragma unroll
      for (int d = 0; d < DT; ++d) vf[d] = *(const af_f4u*)(p.v_pages + v_at + (long long)d * 16 * ps);
      load_keys(t_next <= stop_all ? t_next : t, kn, v_next);       // never skipped: a conditional load would be waited for at once
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
      t = t_next;
    }

    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (shared) {
      float* part = p.parts + ((((long long)blockIdx.x * p.part_ranges + range) * AF_WAVES + wave) * AF_ROWS + li) * LROW;
#pragma unroll
      for (int d = 0; d < DT; ++d) *(af_f4*)(part + d * 16 + lq * 4) = o[d];
      if (lq == 0) *(af_f4*)(part + D) = af_f4{m, l, 0.f, 0.f};
    } else {
      float a, b;
      af_fold(m_all, l_all, m, l, a, b);
#pragma unroll
      for (int d = 0; d < DT; ++d) af_add(o_all[d], a, b, o[d]);
    }
  }
  if (shared) return;

  // the waves meet: a lane holds elements 16 d + 4 lq .. + 3 of its row
  float* dst = af_lds + (wave * AF_ROWS + li) * LROW + lq * 4;
#pragma unroll
  for (int d = 0; d < DT; ++d) *(af_f4*)(dst + d * 16) = o_all[d];
  if (lq == 0) {
    ml[(wave * AF_ROWS + li) * 2] = m_all;
    ml[(wave * AF_ROWS + li) * 2 + 1] = l_all;
  }
  __syncthreads();
  auto result = [&](int rr, int d, int h) {
    float top[AF_WAVES], den[AF_WAVES];
    af_f4 sum[AF_WAVES];
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) {
      top[w] = ml[(w * AF_ROWS + rr) * 2], den[w] = ml[(w * AF_ROWS + rr) * 2 + 1];
      sum[w] = *(const af_f4*)(af_lds + (w * AF_ROWS + rr) * LROW + d);
    }
    return af_meet(top, den, sum, p.sinks ? p.sinks + h : nullptr);
  };
  if (p.terms) {      // 8 elements a thread
    for (int i = threadIdx.x; i < walk.rows * (D / 8); i += 64 * AF_WAVES) {
      const int rr = i / (D / 8), d = (i - rr * (D / 8)) * 8;
      const int qi = (m0 + rr) / G, h = kvh * G + (m0 + rr) - qi * G;
      const long long token = q_start + qi;
      const af_f4 v[2] = {result(rr, d, h), result(rr, d + 4, h)};
      af_f4* out = (af_f4*)(p.out + token * p.nq * D + (long long)h * D + d);
      out[0] = v[0], out[1] = v[1];
      f32_terms::leave_terms(p.terms, p.fragments != 0, p.nq * D / G32_STEP, token, (h * D + d) / 8, v);
    }
    return;
  }
  for (int i = threadIdx.x; i < walk.rows * (D / 4); i += 64 * AF_WAVES) {
    const int rr = i / (D / 4), d = (i - rr * (D / 4)) * 4;
    const int qi = (m0 + rr) / G, h = kvh * G + (m0 + rr) - qi * G;
    const af_f4 v = result(rr, d, h);
    float* out = p.out + (long long)(q_start + qi) * p.nq * D + (long long)h * D + d;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = v[e];
  }
}

// Adds the ranges of the items that blocks shared out, each wave's in their order, then the waves: a block takes 64 of an
// item's 4-element pieces, a wave of it the parts of one wave, asked for several ranges ahead.
__global__ void __launch_bounds__(64 * AF_WAVES) attn_f32_merge_kernel(AttnF32Args p, int blocks, int D) {
  __shared__ float tops[AF_WAVES][64], dens[AF_WAVES][64];
  __shared__ af_f4 sums[AF_WAVES][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int item = blockIdx.x / p.nkv, kvh = blockIdx.x - item * p.nkv;
  const int r = p.work[2 * item], m0 = p.work[2 * item + 1], G = p.nq / p.nkv;
  const int q_start = p.cu_seqlens[r], M = (p.cu_seqlens[r + 1] - q_start) * G;
  const AfWalk walk(p, p.context_lens[r], M, G, m0);
  const int i = blockIdx.y * 64 + lane, rr = i / (D / 4), d = (i - rr * (D / 4)) * 4;
  if (!walk.shared(p, blocks) || blockIdx.y * 64 >= walk.rows * (D / 4)) return;
  const long long stride = (long long)AF_WAVES * AF_ROWS * (D + 4);
  const float* part = p.parts + (long long)blockIdx.x * p.part_ranges * stride + (long long)(wave * AF_ROWS + (rr < walk.rows ? rr : 0)) * (D + 4);
  float top = -INFINITY, den = 0.f;
  af_f4 sum = {0.f, 0.f, 0.f, 0.f};
  constexpr int AHEAD = 8;
  for (int s = 0; s < walk.ranges; s += AHEAD) {
    float tp[AHEAD], dn[AHEAD];
    af_f4 v[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const float* from = part + (s + u < walk.ranges ? s + u : walk.ranges - 1) * stride;
      tp[u] = from[D], dn[u] = from[D + 1], v[u] = *(const af_f4*)(from + d);
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (s + u >= walk.ranges) break;
      float a, b;
      af_fold(top, den, tp[u], dn[u], a, b);
      af_add(sum, a, b, v[u]);
    }
  }
  tops[wave][lane] = top, dens[wave][lane] = den, sums[wave][lane] = sum;
  __syncthreads();
  if (wave > 0 || rr >= walk.rows) return;
  float t4[AF_WAVES], d4[AF_WAVES];
  af_f4 s4[AF_WAVES];
#pragma unroll
  for (int w = 0; w < AF_WAVES; ++w) t4[w] = tops[w][lane], d4[w] = dens[w][lane], s4[w] = sums[w][lane];
  const int qi = (m0 + rr) / G, h = kvh * G + (m0 + rr) - qi * G;
  const af_f4 v = af_meet(t4, d4, s4, p.sinks ? p.sinks + h : nullptr);
  float* out = p.out + (long long)(q_start + qi) * p.nq * D + (long long)h * D + d;
#pragma unroll
  for (int e = 0; e < 4; ++e) out[e] = v[e];
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
    hipLaunchKernelGGL(attn_f32_merge_kernel, dim3(n_work * a.nkv, AF_ROWS * 4 * DT / 64), dim3(64 * AF_WAVES), 0, stream, a, splits, 16 * DT);
  return JV_LAUNCH_CHECK();
}

extern "C" int jv_attn_f32_rows() { return AF_ROWS; }
extern "C" int jv_attn_f32_range_keys() { return 16 * AF_RANGE; }

// Floats of `parts` for items of up to `ranges` > 1 ranges.
extern "C" long long jv_attn_f32_part_floats(int n_work, int nkv, int ranges, int D) {
  return ranges > 1 ? (long long)n_work * nkv * ranges * AF_WAVES * AF_ROWS * (D + 4) : 0;
}

extern "C" int jv_attn_f32(float* out, const float* q, long long q_row_stride, const float* k_pages, const float* v_pages,
                           const int* block_tables, int table_stride, const int* cu_seqlens, const int* context_lens,
                           const int* work, int n_work, int splits, float* parts, int part_ranges, int page_size, int nq, int nkv, int D,
                           float scale, int window, const float* sinks, float cap, int keep, void* terms, int fragments, void* stream) {
  if (n_work <= 0) return 0;
  if (terms && (splits > 1 || (nq * D) % G32_STEP || (((uintptr_t)terms | (uintptr_t)out) & 15))) return (int)hipErrorInvalidValue;
  if (nkv <= 0 || nq % nkv != 0 || page_size <= 0 || page_size % 4 != 0 || keep < 0 || (long long)n_work * nkv > 0x7fffffffll ||
      splits < 1 || splits > 65535 || (splits > 1 && (!parts || part_ranges < 1)))
    return (int)hipErrorInvalidValue;
  const AttnF32Args a = {out, q, q_row_stride, k_pages, v_pages, block_tables, table_stride, cu_seqlens, context_lens, work,
                         page_size, nq, nkv, scale, window, sinks, cap, keep, parts, part_ranges, (unsigned*)terms, fragments};
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
