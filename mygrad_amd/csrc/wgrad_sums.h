// What the reductions of filter gradients on three bf16 parts share (wgrad_split.hip, few_wgrad.hip).
#pragma once

#include "conv_device.h"
#include "wgrad_split.h"

namespace mg {

// dw, of `terms` = C * wvol columns, from the sums of the single-precision kernel; all threads of blocks of 256.
__device__ __forceinline__ void reduce_single(const WgradSums &single, float *dw, int F, int C, int wvol) {
  for (int i = (int)blockIdx.x * 256 + (int)threadIdx.x; i < F * C * wvol; i += (int)gridDim.x * 256) {
    const int tap = i % wvol, c = i / wvol % C, f = i / wvol / C;
    // (the last group of 16 channels is moved back to end with the last channel, see WGroup; those of the one before it are that one's)
    const int moved = single.groups && c / 16 * 16 + 16 > C ? 16 - C % 16 : 0;
    const int column = single.groups ? (c / 16 * wvol + tap) * 16 + c % 16 + moved : c * wvol + tap;
    const float *const from = single.partial + (long long)f * single.ct + column;
    const long long stride = (long long)F * single.ct;
    const int per = (single.splits + single.runs - 1) / single.runs;
    // (seldom: not with sum_in_order()'s sixteen loads at a time, whose registers would halve the waves of the usual reduction beside it)
    float sum = 0.0f;
    for (int first = 0; first < single.splits; first += per) {
      const int last = min(first + per, single.splits);
      float run = from[first * stride];
#pragma unroll 8
      for (int k = first + 1; k < last; ++k) run += from[k * stride];
      sum = first == 0 ? run : sum + run;
    }
    dw[i] = sum;
  }
}

// The last block to have read words[0] leaves all words as they were.  (Counted by 32 lines of memory first: one counter for all takes 10 ns a block.)
__device__ __forceinline__ void leave_words(unsigned *words) {
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned lines = min(gridDim.x, 32u), line = blockIdx.x % lines;
    unsigned *const arrived = words + 32 * (1 + line);
    if (atomicAdd(arrived, 1u) + 1 == (gridDim.x - line + lines - 1) / lines) {
      *arrived = 0;
      if (atomicAdd(&words[1], 1u) + 1 == lines) words[0] = words[1] = 0;
    }
  }
}

}  // namespace mg
