// Device-side helpers that the convolution kernels of several translation units share.
#pragma once

#include "conv_kernels.h"

namespace mg {

// Tables that every lane of a wavefront reads at the same index are addressed
// through the constant address space, which lets the compiler fetch them with
// scalar loads (one request per wavefront, no vector-memory wait) instead of 64
// identical vector loads.
#define MG_CONSTANT __attribute__((address_space(4)))
typedef int int4v __attribute__((ext_vector_type(4)));
static_assert(sizeof(TabEntry) == sizeof(int4v), "a table row is read as one 16-byte vector");
__device__ __forceinline__ const int4v MG_CONSTANT *as_constant(const TabEntry *p) {
  return (const int4v MG_CONSTANT *)(p);
}
__device__ __forceinline__ const int MG_CONSTANT *as_constant(const int *p) { return (const int MG_CONSTANT *)(p); }
__device__ __forceinline__ TabEntry table_row(const int4v MG_CONSTANT *tab, int i) {
  const int4v v = tab[i];
  return TabEntry{v.x, v.y, v.z, v.w};
}
// The wavefront-uniform value of x as a scalar register.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

typedef int int8v __attribute__((ext_vector_type(8)));
// A row of the phase table through the scalar data path (the index is wave-uniform).
__device__ __forceinline__ Phase load_phase(const Phase *phases, int i) {
  const int8v MG_CONSTANT *q = (const int8v MG_CONSTANT *)(phases + uniform(i));
  const int8v a = q[0], b = q[1], c = q[2];
  Phase ph;
  ph.J[0] = a[0], ph.J[1] = a[1], ph.J[2] = a[2];
  ph.o0[0] = a[3], ph.o0[1] = a[4], ph.o0[2] = a[5];
  ph.k_begin = a[6], ph.k_count = a[7];
  ph.blk_begin = b[0], ph.npos = b[1];
  ph.by_jvol = FastDiv{(unsigned)b[2], (unsigned)b[3], (unsigned)b[4], 0u};
  ph.by_j12 = FastDiv{(unsigned)b[6], (unsigned)b[7], (unsigned)c[0], 0u};
  ph.by_j2 = FastDiv{(unsigned)c[2], (unsigned)c[3], (unsigned)c[4], 0u};
  return ph;
}
__device__ __forceinline__ int phase_first_block(const Phase *phases, int i) {
  return ((const int MG_CONSTANT *)(phases + uniform(i)))[8];
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

// D(16x16) += A(16x4) * B(4x16) on one wavefront.  Lane l supplies A[l%16][l/16]
// and B[l/16][l%16].  Lane l receives four elements of column l%16 of D; their
// rows are row_of(l, r), r = 0..3, which differs between the two instructions.
template <typename T>
struct Mma;

template <>
struct Mma<float> {
  using Acc = f32x4;
  static __device__ __forceinline__ Acc run(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row_of(int lane, int r) { return 4 * (lane >> 4) + r; }
};

template <>
struct Mma<double> {
  using Acc = f64x4;
  static __device__ __forceinline__ Acc run(double a, double b, Acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row_of(int lane, int r) { return 4 * r + (lane >> 4); }
};

// ((p[0] + p[stride]) + p[2*stride]) + ... over `terms` terms: always this order, so
// the result does not change from run to run; sixteen loads are in flight at a time
// (the partial sums were written by other XCDs a moment ago: every load is a trip
// past this XCD's L2).
template <typename T>
__device__ __forceinline__ T sum_in_order(const T *__restrict__ p, long long stride, int terms) {
  constexpr int BATCH = 16;
  T s = p[0];
  int k = 1;
  for (; k + BATCH <= terms; k += BATCH) {
    T v[BATCH];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) v[u] = p[(long long)(k + u) * stride];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) s += v[u];
  }
  if (k < terms) {
    // the rest in one more batch: loads past the end repeat the last term and are not added
    T v[BATCH];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) v[u] = p[(long long)min(k + u, terms - 1) * stride];
#pragma unroll
    for (int u = 0; u < BATCH; ++u)
      if (k + u < terms) s += v[u];
  }
  return s;
}

}  // namespace mg
