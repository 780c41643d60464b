// Device-side helpers of the kernels that multiply in three bf16 parts (conv_split.hip, product_split.hip, wgrad_split.hip, few_split.hip,
// few_wgrad.hip).
#pragma once

#include "conv_device.h"

namespace mg {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr unsigned kOutside = 0x80000000u;  // a byte offset past the end of any tensor (each below 2 GiB): reads as zero

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ unsigned bits_of(float v) { return __builtin_bit_cast(unsigned, v); }
__device__ __forceinline__ float float_of(unsigned v) { return __builtin_bit_cast(float, v); }

// a = h[0] + m[0] + l[0] and b likewise, exactly.  Every part is rounded to nearest (the last one, of at most
// eight bits, needs none): x1 is at most 2^-8 of x and x2 2^-17, so what the six products leave out, x1 w2 + x2
// w1 + x2 w2, is at most 2^-24 of x w and has no sign of its own (with the first part cut off instead it was up
// to 2^-22).  A value that rounds to infinity leaves a NaN in its second part.  Eleven vector instructions for
// two values.  The low sixteen bits of `lost` are set where the last part has lost some (see the head of
// conv_split.hip).
__device__ __forceinline__ void split_pair(float a, float b, unsigned &h, unsigned &m, unsigned &l, unsigned &lost) {
  h = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a, b}), bf16x2));
  const float ra = a - float_of(h << 16), rb = b - float_of(h & 0xffff0000u);
  m = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{ra, rb}), bf16x2));
  const float qa = ra - float_of(m << 16), qb = rb - float_of(m & 0xffff0000u);
  l = __builtin_amdgcn_perm(bits_of(qb), bits_of(qa), 0x07060302u);
  lost |= bits_of(qa) | bits_of(qb);
}

// BYTES a lane from a buffer straight into LDS, the lanes' pieces one behind the other from byte `to` on.  Whoever reads it waits
// with landed() (__syncthreads() would do too; what must not come in between are waits for these loads in front of other LDS reads,
// and the compiler puts none there).
template <int BYTES>
__device__ __forceinline__ void to_lds(__amdgpu_buffer_rsrc_t buffer, unsigned lane_at, unsigned at, unsigned to) {
  typedef __attribute__((address_space(3))) void *LdsPointer;
  static_assert(BYTES == 4 || BYTES == 16, "a word or four a lane");
  if (BYTES == 16)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer, (LdsPointer)(unsigned long long)to, 16, (int)lane_at, (int)at, 0, 0);
  else
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer, (LdsPointer)(unsigned long long)to, 4, (int)lane_at, (int)at, 0, 0);
}

// Every load of this wave has landed, and its LDS reads are done; then all waves of the block are here.
__device__ __forceinline__ void landed() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The largest |value| so far (a NaN stays): one instruction for two values.
__device__ __forceinline__ void widen(float &widest, float a, float b) {
  widest = __builtin_elementwise_maximum(widest, __builtin_elementwise_maximum(__builtin_fabsf(a), __builtin_fabsf(b)));
}

// What a product can have lost where an operand of `lost` has low bits below the smallest number of bf16, 2^-133, is 2^-133 of the other operand; a
// sum of `terms` of them is as good as any where it is 2^24 times that.
__device__ __forceinline__ float least_sum(bool lost_a, float widest_a, bool lost_b, float widest_b, int terms) {
  return ((lost_a ? widest_b : 0.0f) + (lost_b ? widest_a : 0.0f)) * (float)terms * 0x1p-109f;
}

}  // namespace mg
