// The two grouped products of routed experts on the matrix cores (bfloat16, float accumulation); the
// grouping they read (tiles of 64, 128 or 192 rows of one expert each) is made by moe.hip.  And the router's logits.
//
// A block takes one tile of (token, choice) rows against TW rows of the expert's weight and walks the inner size in
// chunks of 64: the rows of x (gathered by token) and of W go straight from memory into LDS, chunks ahead of their use;
// v_mfma_f32_32x32x16_bf16 with A = 32 rows of x, B = 32 rows of W, a wave 64 (or 32) rows of x against 64 of W.
// Each output is a sum over the inner size in ascending steps of 16, whatever else is in the step.
//
// Bound by what a compute unit draws from its L2, 40..45 bytes a nanosecond as in every product of this kind here: a tile of
// 128 rows needs 1.5 bytes of operands where 256 x 256 would need 1, but an expert of a prompt has few rows, and half the
// tiles are not full.  2,048 tokens, gate/up + down, microseconds (before: one buffer through registers, 64 rows of W):
//   32 experts x 512, 4 chosen, width 2,048:    85 + 50   (96 + 76)
//   64 experts x 1,024, 8 chosen, width 4,096: 478 + 296  (570 + 439)
// What a block begins and ends with weighs as much as a third of its chunks (17 us at one chunk of 64, 0.95 us for each further): the weights of its
// rows are not waited for at the start, and its results leave through LDS in whole lines.  Before / so, tiles of 192 rows, 2,048 tokens:
// 32 x 512, 4 chosen, width 2,048 62.0 + 56.1 / 59.7 + 48.5; 64 x 1,024, 8 chosen, 4,096 tokens, width 4,096 660 + 413 / 634 + 399; tiles of 128, 32 x 768
// 98.4 + 67.3 / 91.7 + 65.6; of 64, 1,003 tokens 48.5 + 31.7 / 47.9 + 31.7.  Not better: the ring by 4 waves of 96 x 128 (0.81 us a
// chunk, but 24 us at one: 65.6 + 51.2; 398 + 256 for 432 + 251 at 64 x 1,024 and 2,048 tokens only).
// Not better: 128 rows of W and two blocks a unit 83 + 50, 495 + 300; a wave for 64 x 128 (one a SIMD: nothing overlaps its own
// reads) 134 + 71, 626 + 358; a register copy of row tiles to skip empty ones 87 + 56.
//   MM_GATED:  z[pos] = act(w g) * (w u), g = Wg[e] x[token], u = Wu[e] x[token]    (bf16)
//   MM_PLAIN:  z[pos] = act(w u), u = Wu[e] x[token]: experts without a gate        (bf16)
//   MM_DOWN:   y[kk][token] = (Wd[e] z[pos]) * w_out                                (float)
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

enum { MM_DOWN = 0, MM_GATED = 1, MM_PLAIN = 2 };

#define MM_K 64            // columns of a chunk: a row of it is 128 bytes, 8 pieces of 16

// What a lane reads for columns behind the inner size, of x and of W alike.
static __device__ __attribute__((aligned(16))) const unsigned mm_zeros[4] = {0, 0, 0, 0};

// TM: rows of a tile of the grouping, 64, 128 or 192; TW: rows of W of a block (gated: half of them of each matrix).
template <int MODE, int TM, int TW, int BUFS>
__global__ void __launch_bounds__(2 * TW, TW == 128 ? 2 : 1)
moe_mfma_kernel(void* __restrict__ out, const bf16_t* __restrict__ a_rows, const bf16_t* __restrict__ W0,
                const bf16_t* __restrict__ W1, const int* __restrict__ meta, const int* __restrict__ offsets,
                const int* __restrict__ tile_expert, const int* __restrict__ tile_row0, const int* __restrict__ order,
                const float* __restrict__ weights, int top, int n_tokens, int K, int N, JvAct act, int use_weight) {
  constexpr int MT = TM / 64;               // 32-row tiles of x of a wave
  constexpr bool GATED = MODE == MM_GATED, BY_TOKEN = MODE != MM_DOWN;
  constexpr int WAVES = TW / 32;                    // 2 along the rows of x, the others 64 rows of W each
  constexpr int NB = GATED ? TW / 2 : TW;           // output columns of a block
  constexpr int XI = TM / 8 / WAVES, WI = TW / 8 / WAVES;      // instructions a wave brings of a chunk, each 8 rows of 128 bytes
  constexpr int BUF = (TM + TW) * MM_K;             // elements of a buffer: rows of x, then rows of W
  constexpr bool RING = BUFS == 0;                  // units of half the rows of x and of W of a chunk in a ring of five
  constexpr int HALF = BUF / 2, SLOTS = 5;
  static_assert(!RING || (WAVES == 8 && MT == 3 && WI == 4), "how a wave's loads fall on the two units of a chunk");
  // Blocks b, b + 8, b + 16, ... run on one XCD (with an L2 of its own): each of the 8 takes one run of the (tile, rows of W)
  // pairs, rows of W fastest, so the rows of x of a tile and the weights of an expert are read into one L2 and used there.
  const int per_tile = (N + NB - 1) / NB;
  const int live = meta[0] * per_tile, chunk = (live + 7) / 8;
  const int pair = ((int)blockIdx.x & 7) * chunk + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= chunk || pair >= live) return;
  const int tile = pair / per_tile;
  __shared__ __attribute__((aligned(1024))) bf16_t bufs[RING ? SLOTS * HALF : BUFS * BUF];
  __shared__ int from[TM];                  // a row's row of x
  __shared__ long long to[TM];              // where its results go
  __shared__ float wts[TM];
  const int e = tile_expert[tile], row0 = tile_row0[tile];
  const int rows = min(TM, offsets[e + 1] - row0);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = (pair - tile * per_tile) * NB;
  float mine = 1.f;
  if (tid < TM) {                           // rows beyond the tile repeat its last row
    const int s = order[row0 + min(tid, rows - 1)];
    const int token = s / top;
    from[tid] = BY_TOKEN ? token : row0 + min(tid, rows - 1);
    to[tid] = (MODE == MM_DOWN ? (long long)(s - token * top) * n_tokens + token : (long long)(row0 + tid)) * N;
    if (use_weight) mine = weights[s];      // not waited for until the sums are there
  }
  __syncthreads();

  // Loads straight into LDS: an instruction brings 8 rows, lane l row l / 8, and fills 1 KB in the order of the lanes.  Piece
  // c of row r lies at slot c ^ ((r / 2) % 8) of its row, so that 16 lanes reading one piece of 16 rows meet 16 slots.
  const int lr = lane >> 3;
  const bf16_t* src[XI + WI];
  int col[2];                               // a lane's columns in a chunk, for rows 16 i + lr and 16 i + 8 + lr
#pragma unroll
  for (int h = 0; h < 2; ++h) col[h] = (((lane & 7) ^ ((lr + 8 * h) >> 1)) & 7) * 8;
  // In a ring, unit h of a chunk has rows h TM / 2 .. of x and h TW / 2 .. of W.  A wave brings 8 rows of x and 16 of W of each, and the 8
  // that are left over of x: of unit 0 by waves 0 to 3, of unit 1 by 4 to 7.  src: x of units 0, 1, left over; W two of unit 0, two of 1.
  auto first_row = [&](int i) {             // of instruction i of this wave, in x or in W
    if (!RING) return (i < XI ? wave * XI + i : wave * WI + i - XI) * 8;
    if (i < 2) return i * (TM / 2) + wave * 8;
    if (i == 2) return (wave >> 2) * (TM / 2) + 64 + (wave & 3) * 8;
    return ((i - XI) >> 1) * (TW / 2) + (wave * 2 + ((i - XI) & 1)) * 8;
  };
#pragma unroll
  for (int i = 0; i < XI; ++i) src[i] = a_rows + (long long)from[first_row(i) + lr] * K;
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = first_row(XI + i) + lr;
    // gated: rows 64 w .. + 31 of the block's W are gate rows 32 w .. + 31, the 32 behind them the same rows of up
    const int n = GATED ? n0 + (r >> 6) * 32 + (r & 31) : n0 + r;
    const bf16_t* w = GATED && (r & 32) ? W1 : W0;
    src[XI + i] = w + ((long long)e * N + min(n, N - 1)) * K;
  }
  auto fetch = [&](int k0, int buf) {
#pragma unroll
    for (int i = 0; i < XI + WI; ++i) {
      const int first = i < XI ? (wave * XI + i) * 8 : TM + (wave * WI + i - XI) * 8;      // the instruction's first row in the buffer
      const int k = k0 + col[(first >> 3) & 1];       // odd groups of 8 rows are the upper half of 16
      const bf16_t* piece = k < K ? src[i] + k : (const bf16_t*)mm_zeros;
      const unsigned at = (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)(bufs + buf * BUF + first * MM_K);
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(piece), "s"(at) : "memory", "m0");
    }
  };

  f32x16 acc[2][MT];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][mt][i] = 0.f;
  // wave (wm, wn): rows of x (TM / 2) wm .., rows of W 64 wn ..
  const int wm = wave & 1, wn = wave >> 1, l32 = lane & 31, half = lane >> 5, swz = (l32 >> 1) & 7;
  const int chunks = (K + MM_K - 1) / MM_K;
  if constexpr (RING) {
    auto load = [&](int i, int c, int slot) {       // instruction i, columns of chunk c, into the slot of its unit
      const int row = first_row(i), h = i < 2 ? i : i == 2 ? wave >> 2 : (i - XI) >> 1;
      const int in_unit = i < XI ? row - h * (TM / 2) : TM / 2 + row - h * (TW / 2), k = c * MM_K + col[(in_unit >> 3) & 1];
      const bf16_t* piece = k < K ? src[i] + k : (const bf16_t*)mm_zeros;
      const unsigned at = (unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)(bufs + slot * HALF + in_unit * MM_K);
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(piece), "s"(at) : "memory", "m0");
    };
    // load j of a wave's 4 (or 3: no left-over rows) of unit h
    auto unit = [&](int j, int h, int c, int slot) {
      if (j < 2) load(XI + 2 * h + j, c, slot);
      else if (j == 2) load(h, c, slot);
      else if ((wave >> 2) == h) load(2, c, slot);
    };
    auto wrap = [](int v) { return v >= SLOTS ? v - SLOTS : v; };
    bf16x8 xf[2][MT], wf[2][2];
    auto read = [&](int i, int set, int ks, int s0) {      // s0: slot of the chunk's first unit
      const int at = ((ks * 2 + half) ^ swz) * 8;
      if (i < 2) wf[set][i] = *(const bf16x8*)(bufs + wrap(s0 + (wn >> 1)) * HALF + (TM / 2 + (wn & 1) * 64 + i * 32 + l32) * MM_K + at);
      else xf[set][i - 2] = *(const bf16x8*)(bufs + wrap(s0 + wm) * HALF + ((i - 2) * 32 + l32) * MM_K + at);
    };
    // Chunk c: its products, the reads of the next 16 columns between them, and the loads of units 2 c + 4 and 2 c + 5 into the slots
    // that chunks c - 1 and c left.  more: 2: those units exist; 1: chunk c + 1 exists; 0: the last.
    auto chunk = [&](auto more, int c, int s0) {
      constexpr int MORE = decltype(more)::value;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int set = ks & 1;
        if (ks == 3 && MORE > 0) {      // chunk c is in registers everywhere, c + 1 is there; unit 2 c + 4 may be on its way
          if (MORE == 1) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
          else if (wave < 4) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
          else asm volatile("s_waitcnt vmcnt(3) lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) {
          if (i < MT + 2 && (ks < 3 || MORE > 0)) read(i, set ^ 1, (ks + 1) & 3, ks < 3 ? s0 : wrap(s0 + 2));
          if (MORE > 1 && ks < 3 && (ks * 6 + i) % 4 == 1 && (ks * 6 + i) / 4 < 4) unit((ks * 6 + i) / 4, 0, c + 2, wrap(s0 + 4));
          if (MORE > 1 && ks == 3 && i < 4) unit(i, 1, c + 2, s0);
          acc[i / MT][i % MT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[set][i % MT], wf[set][i / MT], acc[i / MT][i % MT], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    for (int c = 0; c < 2 && c < chunks; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) unit(j, h, c, 2 * c + h);
    if (chunks > 1) asm volatile("s_waitcnt vmcnt(7)" ::: "memory");      // of both units of a chunk a wave has 7
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT + 2; ++i) read(i, 0, 0, 0);
    int c = 0, s0 = 0;
    for (; c + 2 < chunks; ++c, s0 = wrap(s0 + 2)) chunk(std::integral_constant<int, 2>{}, c, s0);
    if (c + 1 < chunks) { chunk(std::integral_constant<int, 1>{}, c, s0); ++c, s0 = wrap(s0 + 2); }
    chunk(std::integral_constant<int, 0>{}, c, s0);
  } else {
  for (int c = 0; c < BUFS - 1 && c < chunks; ++c) fetch(c * MM_K, c);
  for (int c = 0, buf = 0; c < chunks; ++c, buf = buf + 1 == BUFS ? 0 : buf + 1) {
    // this wave's part of chunk c is there (loads arrive in order; those of the next BUFS - 2 chunks may be on their way)
    if (BUFS > 2 && c + BUFS - 2 < chunks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((BUFS - 2) * (XI + WI)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                                      // and everybody's, and the buffer before is no longer read
    if (c + BUFS - 1 < chunks) fetch((c + BUFS - 1) * MM_K, buf == 0 ? BUFS - 1 : buf - 1);
    const bf16_t* xb = bufs + buf * BUF + (wm * (TM / 2) + l32) * MM_K;
    const bf16_t* wb = bufs + buf * BUF + (TM + wn * 64 + l32) * MM_K;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int at = ((ks * 2 + half) ^ swz) * 8;
      bf16x8 xf[MT], wf[2];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xf[mt] = *(const bf16x8*)(xb + mt * 32 * MM_K + at);
#pragma unroll
      for (int a = 0; a < 2; ++a) wf[a] = *(const bf16x8*)(wb + a * 32 * MM_K + at);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[a][mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[mt], wf[a], acc[a][mt], 0, 0, 0);
    }
  }
  }
  // The sums go through LDS, 32 rows of both halves of x at a time, so that a thread leaves 4 neighbouring columns: the activation's code is
  // there once instead of once for every number a lane holds, and a row is written in whole lines.
  constexpr int ROW = TW + 4, THREADS = 2 * TW;      // floats of a row there: 4 rows further on lie half the banks further on
  static_assert(64 * ROW * 4 <= (RING ? SLOTS * HALF : BUFS * BUF) * 2, "");
  float* const stage = (float*)bufs;
  const bool fours = N % 4 == 0 && ((unsigned long long)out & 15) == 0;
  if (tid < TM) wts[tid] = mine;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    __syncthreads();
    // a lane holds column l32 of both tiles of W, rows 8 q + 4 half + i of a tile of x
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        stage[(wm * 32 + (i >> 2) * 8 + half * 4 + (i & 3)) * ROW + wn * 64 + a * 32 + l32] = acc[a][mt][i];
    __syncthreads();
#pragma unroll 1
    for (int q = tid; q < 64 * NB / 4; q += THREADS) {
      const int r = q / (NB / 4), o = (q - r * (NB / 4)) * 4, m = (r >> 5) * (TM / 2) + mt * 32 + (r & 31), n = n0 + o;
      if (m >= rows || n >= N) continue;
      const float w = wts[m];
      const long long at = to[m] + n;
      const f32x4 v = *(const f32x4*)(stage + r * ROW + (GATED ? (o >> 5) * 64 + (o & 31) : o)) * w;
      if constexpr (MODE == MM_DOWN) {
        if (fours) *(f32x4*)((float*)out + at) = v;
        else
          for (int k = 0; k < 4 && n + k < N; ++k) ((float*)out)[at + k] = v[k];
      } else {
        typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
        bf16x4 y;
        if constexpr (GATED) {
          const f32x4 u = *(const f32x4*)(stage + r * ROW + (o >> 5) * 64 + 32 + (o & 31)) * w;
#pragma unroll
          for (int k = 0; k < 4; ++k) y[k] = from_f32<bf16_t>(jv_gated(act, v[k], u[k]));
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k) y[k] = from_f32<bf16_t>(jv_act(act.id, v[k]));
        }
        if (fours) *(bf16x4*)((bf16_t*)out + at) = y;
        else
          for (int k = 0; k < 4 && n + k < N; ++k) ((bf16_t*)out)[at + k] = y[k];
      }
    }
  }
}

template <int MODE, int TM, int TW, int BUFS>
static int launch_moe_tiles(int max_tiles, hipStream_t stream, void* out, const bf16_t* a, const bf16_t* W0,
                            const bf16_t* W1, const int* meta, const int* offsets, const int* tile_expert,
                            const int* tile_row0, const int* order, const float* weights, int top, int n_tokens, int K,
                            int N, JvAct act, int use_weight) {
  const int nb = MODE == MM_GATED ? TW / 2 : TW;
  const long long pairs = (long long)max_tiles * ((N + nb - 1) / nb);
  if (pairs > 0x7ffffff0ll) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((moe_mfma_kernel<MODE, TM, TW, BUFS>), dim3((unsigned)(pairs + 7)), dim3(2 * TW), 0, stream, out, a, W0, W1,
                     meta, offsets, tile_expert, tile_row0, order, weights, top, n_tokens, K, N, act, use_weight);
  return JV_LAUNCH_CHECK();
}

// 128 rows against 256 of W by 8 waves with two chunks on their way; 192 rows, for groupings that fill the units with fewer tiles (32
// experts x 512, width 2,048, 256 rows each: 256 tiles instead of 320, gate/up 61 us, before 85), through a ring of five half chunks
// (three whole ones do not fit), whose loads are spread over the products: both products of 4,096 tokens, 8 of 64 x 1,024, width 4,096
// 1,038 us (1,136 with two whole buffers), width 2,048 547 (597), 2 of 8 x 4,096 605 (654), 4 of 32 x 512 at 2,500 tokens 108 (113);
// 64 rows against 128 by 4 waves, three blocks a compute unit with
// one chunk on its way each, or (`deep`) two blocks with two: where an expert gets so few rows that nearly all are one tile, the
// stream of the weights is what is waited for.  gate/up + down, cold weights, microseconds (deep / not): 64 experts x 1,024, width
// 4,096, 25 rows each 302 / 334, 8 x 4,096 at 40 rows 167 / 184, 16 x 2,048, width 1,024, at 25 56 / 64, 32 x 512, width 2,048, at
// 40 52 / 57; at 50 rows, with second tiles, 66 / 62.
template <int MODE, typename... Args>
static int launch_moe_mfma(int tile_rows, int deep, Args... args) {
  if (tile_rows == 192) return launch_moe_tiles<MODE, 192, 256, 0>(args...);
  if (tile_rows == 128) return launch_moe_tiles<MODE, 128, 256, 3>(args...);
  if (tile_rows == 64 && deep) return launch_moe_tiles<MODE, 64, 128, 3>(args...);
  if (tile_rows == 64) return launch_moe_tiles<MODE, 64, 128, 2>(args...);
  return (int)hipErrorInvalidValue;
}

// gate/up: x [tokens, hidden], Wg, Wu [experts, ff, hidden] -> z [entries, ff] bf16 by position; tile_rows (64,
// 128 or 192) is what the grouping was made with; deep: see launch_moe_mfma.  Wg null: experts without a gate, act one that stands alone.
extern "C" int jv_moe_gate_up_mfma_bf16(void* z, const void* x, const void* Wg, const void* Wu, const int* meta,
                                        const int* offsets, const int* tile_expert, const int* tile_row0,
                                        const int* order, const float* weights, int max_tiles, int top, int hidden,
                                        int ff, int act, float act_limit, float act_slope, int scale_input, int tile_rows, int deep, void* stream) {
  if (max_tiles <= 0 || ff <= 0) return 0;
  if (!(Wg ? jv_act_known(act) : jv_plain_act_known(act)) || hidden < 8 || hidden % 8 || (((uintptr_t)x | (uintptr_t)Wg | (uintptr_t)Wu) & 15))
    return (int)hipErrorInvalidValue;
  if (!Wg)
    return launch_moe_mfma<MM_PLAIN>(tile_rows, deep, max_tiles, (hipStream_t)stream, z,
                                     (const bf16_t*)x, (const bf16_t*)Wu, nullptr, meta, offsets, tile_expert, tile_row0,
                                     order, weights, top, 0, hidden, ff, JvAct{act, act_limit, act_slope}, scale_input);
  return launch_moe_mfma<MM_GATED>(tile_rows, deep, max_tiles, (hipStream_t)stream, z, (const bf16_t*)x,
                               (const bf16_t*)Wg, (const bf16_t*)Wu, meta, offsets, tile_expert, tile_row0, order,
                               weights, top, 0, hidden, ff, JvAct{act, act_limit, act_slope}, scale_input);
}

// down: z [entries, ff] by position, Wd [experts, hidden, ff] -> y [top, tokens, hidden] float
extern "C" int jv_moe_down_mfma_bf16(float* y, const void* z, const void* Wd, const int* meta, const int* offsets,
                                     const int* tile_expert, const int* tile_row0, const int* order,
                                     const float* weights, int max_tiles, int top, int n_tokens, int hidden, int ff,
                                     int scale_output, int tile_rows, int deep, void* stream) {
  if (max_tiles <= 0 || hidden <= 0) return 0;
  if (ff < 8 || ff % 8 || (((uintptr_t)z | (uintptr_t)Wd) & 15)) return (int)hipErrorInvalidValue;
  return launch_moe_mfma<MM_DOWN>(tile_rows, deep, max_tiles, (hipStream_t)stream, y,
                                (const bf16_t*)z, (const bf16_t*)Wd, nullptr, meta, offsets, tile_expert, tile_row0, order,
                                weights, top, n_tokens, ff, hidden, JvAct{}, scale_output);
}

// y [M, N] float = x [M, K] W[N, K]^T for bfloat16 x and W: the router's logits of a prompt's rows, few columns over a long
// inner size.  A block takes 16 rows of x against 16 NT rows of W; its 8 waves take an eighth of the inner size each, in
// steps of 32 columns straight from memory into operands, and meet in LDS: the parts are added in ascending order, so a row's
// logits do not depend on the batch.  Bound by its one round trip to memory: 2,048 rows x 32 x 2,048 7.9 us (25 as one
// column of the tiles above, 16 blocks of 32 chunks in a row).
template <int NT>
__global__ void __launch_bounds__(512)
gemm_rows_kernel(float* __restrict__ y, const bf16_t* __restrict__ x, const bf16_t* __restrict__ W, int M, int N, int K) {
  __shared__ f32x4 red[NT][8][64];
  const int part = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
  const int m0 = blockIdx.x * 16, n0 = blockIdx.y * (16 * NT);
  const int len = (K + 255) / 256 * 32, k_begin = part * len, k_end = min(K, k_begin + len);
  const bf16_t* xrow = x + (long long)min(m0 + li, M - 1) * K;
  const bf16_t* wrow[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wrow[t] = W + (long long)min(n0 + t * 16 + li, N - 1) * K;
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  constexpr int U = NT > 2 ? 2 : 4;               // steps whose loads are asked for together
  for (int k0 = k_begin; k0 < k_end; k0 += 32 * U) {
    bf16x8 xf[U], wf[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * 32 + lq * 8, at = min(k, K - 8);
      xf[u] = *(const bf16x8*)(xrow + at);
#pragma unroll
      for (int t = 0; t < NT; ++t) wf[u][t] = *(const bf16x8*)(wrow[t] + at);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool inside = k0 + u * 32 + lq * 8 < k_end;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(inside ? wf[u][t] : zero, inside ? xf[u] : zero, acc[t], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) red[t][part][lane] = acc[t];
  __syncthreads();
  if (part < NT) {
    f32x4 sum = red[part][0][lane];
#pragma unroll
    for (int p = 1; p < 8; ++p) sum += red[part][p][lane];
    const int m = m0 + li, n = n0 + part * 16 + lq * 4;      // a lane holds 4 columns of a row
    if (m < M)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (n + c < N) y[(long long)m * N + n + c] = sum[c];
  }
}

extern "C" int jv_gemm_rows_f32out_bf16(float* y, const void* x, const void* W, int M, int N, int K, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  const int nt = N <= 16 ? 1 : N <= 32 ? 2 : 4;
  const dim3 grid((M + 15) / 16, (N + 16 * nt - 1) / (16 * nt));
  if (K < 8 || K % 8 || grid.y > 65535) return (int)hipErrorInvalidValue;
  const bf16_t *xb = (const bf16_t*)x, *wb = (const bf16_t*)W;
  if (nt == 1) hipLaunchKernelGGL(gemm_rows_kernel<1>, grid, dim3(512), 0, (hipStream_t)stream, y, xb, wb, M, N, K);
  else if (nt == 2) hipLaunchKernelGGL(gemm_rows_kernel<2>, grid, dim3(512), 0, (hipStream_t)stream, y, xb, wb, M, N, K);
  else hipLaunchKernelGGL(gemm_rows_kernel<4>, grid, dim3(512), 0, (hipStream_t)stream, y, xb, wb, M, N, K);
  return JV_LAUNCH_CHECK();
}
