// Forward pass of single-precision layers with few terms to a sum (a first layer: one or three channels) on three bf16 parts
// (few_split.hip): what the kernel, the planner and the entry points share.
#pragma once

#include "conv_kernels.h"

namespace mg {

struct FewParams {
  const float *x, *w;
  float *dst;
  unsigned x_bytes;     // below 2 GiB
  int C, F, K, steps;   // K = C * taps terms to a sum, in steps of 32
  int X1, X2, G2, gvol; // (axis 0 is trivial)
  int S1, S2, D1, D2, P1, P2, W1, W2;
  // A tile's positions are consecutive in the plane of results: runs of the whole plane, or (along) of a row.
  int along, run_tiles; // tiles of a plane, or of a row
  int sample_tiles, items;  // tiles of a sample, of all samples
  // A tile's patch of x, [channel][row][column], zeros outside: patch_rows rows of `pitch` columns, the windows' first one behind `lead`
  // others, so that it begins on a multiple of four (-1: rows of up to 64 columns, as they come)
  int patch_rows, pitch, lead, patch;  // (patch: in all)
  int m_tiles;
  FastDiv by_sample, by_run, by_row, by_patch_rows, by_window, by_w2;
};

struct FewPlan {
  int tm = 0, tn = 0;  // a wave's results: 16 tm filters by 16 tn positions; 0: the layer does not run there
  int grid = 0;
  double time = 0;     // modelled, us
  FewParams p{};
};

constexpr int kFewLds = 160 * 1024;

// How tiles of `bm` filters by `positions` (along: of a row) lie; false: their patches are too large, or the layer is none that the kernels take.
// (LDS that they need beside the patches is not looked at.)
bool few_geometry(FewParams &p, int N, int C, int F, const int *X, const int *G, const int *W, const int *S, const int *D, const int *P, int bm, int positions, bool along);
// Loads that a tile's patch takes.
long long few_requests(const FewParams &p);

FewPlan plan_few_split(int N, int C, int F, const int *X, const int *G, const int *W, const int *S, const int *D, const int *P, int cus);
int launch_few_split(const FewPlan &pl, const void *x, const void *w, void *out, hipStream_t s);

}  // namespace mg
