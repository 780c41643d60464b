// Large single-precision filter gradients on three bf16 parts (wgrad_split.hip): what the kernels and the planner share.
#pragma once

#include "conv_kernels.h"

namespace mg {

struct WgradSplitParams {
  const float *x, *grad;
  float *partial;         // [split][tile][filter of the tile][frag * 16 + channel]
  float *dw;
  unsigned *words;        // whether the gradient has to be computed on the single-precision instruction; and counts of the blocks that have read that
  unsigned x_bytes, grad_bytes;  // each below 2 GiB
  int C, F, wvol, kpos;
  int X[3], G[3], S[3], D[3], P[3], W[3];
  // Eight segments make an octet of the contraction: a sample's planes of positions (one per position of axis 0), each in
  // 1 << seg_shift runs of seg_len columns, a multiple of four.
  int seg_shift, seg_len;
  FastDiv by_g0;
  // A walk: one octet of segments, one strip of 4 * quads columns, `stages` stages of `rows` rows each; along the columns, where
  // there is one row: one octet, a stage a strip.
  int octets, strips, stages;
  int rows, quads;        // rows * quads quads of positions to a stage, one for each of a tile's waves along K
  // A column tile's patch of x: a ring of depth + 2 groups of new_rows rows, row_locs locations (x_quads of four) to a row.
  int new_rows, depth, row_locs, x_quads;
  // Column tiles: 16 channels, one tap of axis 0, up to nine taps of axes 1 and 2 (of W[1] * W[2], in `chunks` chunks).
  int chunks, columns;
  int tiles, f_tiles;     // of a block: some column tiles by some filters
  int splits;
  long long total;        // stages of all walks
};

constexpr int kWgradSplitFrags = 9;  // taps of a tile at most
constexpr int kWgradSplitWords = 32 * 33;

// How the filter gradient runs there (waves along filters, column tiles and K, tasks of a wave; splits and the fields of the geometry),
// false where it does not.
struct WgradSplitPlan {
  int fw = 0, cw = 0, kw = 0, tasks = 0;
  bool along = false;
  double time = 0;  // modelled, us
  WgradSplitParams p{};
};

WgradSplitPlan plan_wgrad_split(int N, int C, int F, const int *X, const int *G, const int *W, const int *S, const int *D, const int *P, int cus);
size_t wgrad_split_scratch(const WgradSplitPlan &pl);

// The sums of the single-precision kernels, where the parts cannot hold a gradient: [split][F][ct], columns by tap groups of 16
// channels (see WGroup) or in dw's own order; nullptr: they are in dw.  They are added as that kernel's own reduction adds them: the
// splits in `runs` runs, in order, then the runs.
struct WgradSums {
  const float *partial;
  int splits, runs, ct;
  bool groups;
};

// Partial sums on the parts into `scratch`, and words[0] != 0 where they cannot be used; a single-precision kernel that does
// nothing otherwise is to come between this and the reduction, which leaves all words zero again, as they have to be to begin with.
int launch_wgrad_split(const WgradSplitPlan &pl, const void *grad, const void *x, void *scratch, unsigned *words, hipStream_t s);
int launch_wgrad_split_reduce(const WgradSplitPlan &pl, const WgradSums &single, void *dw, void *scratch, unsigned *words, hipStream_t s);

}  // namespace mg
