// Large single-precision matrix products on three bf16 parts (product_split.hip): what the kernels and the
// entry points share.
#pragma once

#include "conv_kernels.h"

namespace mg {

// One operand of  dst(m, j) = sum over k of A(m, k) B(j, k)  where it lies.  Its rows (m or j) are `rows_in` at a
// time `row_stride` apart, `rows_out` from one such run to the next; the K axis likewise, counted in octets
// (eight consecutive k, the last octet of a run with fewer).  One of the two strides is 1.
struct ProductOperand {
  const float *base;
  int rows;          // in all
  FastDiv by_rows;   // rows_in
  long long rows_out, row_stride;
  int k_in;
  FastDiv by_octets;  // octets of a run of k_in
  long long k_out, k_stride;
};

struct ProductParams {
  ProductOperand a, b;
  int octets, steps;     // of the K axis: octets, K steps of 32
  int a_panels, b_panels;  // of 128 rows, as many as the tiles cover
  void *packed_a, *packed_b;  // [panel][step][part][octet of 4][row of 128][8] bf16
  unsigned *notes;       // [panel of a, then of b][step]: twice the largest |value|, plus one if an element has lost bits
  unsigned *redo;        // whether there is a marked tile, then the marks, a bit each
  int marks;             // words of redo
  int m_tiles, tiles;
  int full_tiles;        // computed by one block each: a multiple of the grid
  int share_blocks;      // blocks that share the K steps of the others, end to end; 0: there are none
  int share_steps, share_extra;  // of each block, and one more of the first share_extra
  float *partial;        // [2 slots of a sharing block][BM][BN]
  float *dst;            // row m, column j = (batch, n): batch * dst_batch + m * dst_mstride + n
  int M, columns;
  FastDiv by_n;
  long long dst_batch, dst_mstride;
};

constexpr int kProductPanel = 128;                      // rows
constexpr int kProductPanelBytes = kProductPanel * 32 * 6;  // of one K step

// Whether a product with `runs` runs of `run` terms to a sum is large enough to run there.
bool product_applies(long long M, long long columns, long long runs, long long run);

// mg_matmul, mg_matmul_da and mg_matmul_dx in float32; MG_ERR_UNSUPPORTED, and nothing done, where there is no memory
// for the parts.
int product_forward(long long batch, long long M, long long K, long long N, const void *a, const void *x, void *out);
int product_da(long long batch, long long M, long long K, long long N, const void *grad, const void *x, void *da);
int product_dx(long long batch, long long M, long long K, long long N, const void *grad, const void *a, void *dx);

}  // namespace mg
