// The order in which a decode attention's blocks take their requests, where a compute unit gets blocks of more than one (`at_once`
// requests' blocks go to the units at once, in launch order; then each unit its next): by their numbers of keys, so that every unit
// has about as many in all.  Up to twice at_once requests: the units that get a second block begin with the shorter requests of the
// first lap, the longest of these followed by the shortest of all; beyond, laps of descending and ascending length in turn.
// Nothing that is computed depends on it.  One launch a step and kind of layer, 8 kv heads, half to one and a half of the keys,
// microseconds of a layer's attention as the requests come / so: 33 of 1,024 keys 40.3 / 34.3, 40 of 1,024 48.5 / 38.0, 48 of 1,000
// 50.3 / 43.4, 64 of 1,024 60.7 / 55.8, 64 of 2,000 108 / 100, 128 of 500 62.5 / 57.8, 64 of 200 18.1 / 18.2.  Ranked by every block of the
// attention itself: 4 us a layer at 64 requests, 15 at 128.
#include "common.h"

#define DO_MAX 1024

__global__ void __launch_bounds__(256)
decode_order_kernel(int* __restrict__ order, const int* __restrict__ context_lens, int n, int at_once, int window) {
  __shared__ __attribute__((aligned(16))) int keys[DO_MAX];
  for (int i = threadIdx.x; i < (n + 3) / 4 * 4; i += 256) {
    const int pos = i < n ? context_lens[i] : -1;
    keys[i] = window > 0 ? min(pos, window) : window < 0 && pos >= 0 ? pos % -window : pos;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += 256) {
    const int mine = keys[i];
    int rank = 0;                       // longer ones, and equal ones of lower number, are ahead
    for (int k = 0; k < n; k += 4) {
      const int4 other = *(const int4*)(keys + k);
      rank += (other.x > mine || (other.x == mine && k < i)) + (other.y > mine || (other.y == mine && k + 1 < i)) +
              (other.z > mine || (other.z == mine && k + 2 < i)) + (other.w > mine || (other.w == mine && k + 3 < i));
    }
    const int second = n - at_once;
    int slot = rank;
    if (n > 2 * at_once) {
      const int lap = rank / at_once, j = rank - lap * at_once, size = min(at_once, n - lap * at_once);
      slot = lap * at_once + (lap & 1 ? size - 1 - j : j);
    } else if (n > at_once) {
      slot = rank >= at_once ? at_once + n - 1 - rank : rank < at_once - second ? rank + second : rank - (at_once - second);
    }
    order[slot] = i;
  }
}

// order, context_lens: int [n], n <= 1,024; window as in the attention kernels (0: all keys, > 0: the last so many, < 0: blocks of -window).
extern "C" int jv_decode_order(int* order, const int* context_lens, int n, int at_once, int window, void* stream) {
  if (n <= 0) return 0;
  if (n > DO_MAX || at_once < 1) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(decode_order_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, order, context_lens, n, at_once, window);
  return JV_LAUNCH_CHECK();
}
