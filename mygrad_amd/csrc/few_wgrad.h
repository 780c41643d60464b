// Filter gradient of single-precision layers with few terms to a filter on three bf16 parts (few_wgrad.hip): what the
// kernels, the planner and the entry points share.
#pragma once

#include "few_split.h"
#include "wgrad_split.h"

namespace mg {

struct FewGradParams {
  FewParams at;         // where a tile's positions and its patch of x lie
  const float *grad;
  unsigned grad_bytes;  // below 2 GiB
  float *partial;       // [split][F][K]
  unsigned *words;      // see WgradSplitParams
  int splits;
};

struct FewGradPlan {
  int tm = 0, tk = 0;   // a wave's results: 16 tm filters by 16 tk columns; 0: the gradient does not run there
  double time = 0;      // modelled, us
  FewGradParams p{};
};

FewGradPlan plan_few_wgrad(int N, int C, int F, const int *X, const int *G, const int *W, const int *S, const int *D, const int *P, int cus);
size_t few_wgrad_scratch(const FewGradPlan &pl);
// As launch_wgrad_split and launch_wgrad_split_reduce.
int launch_few_wgrad(const FewGradPlan &pl, const void *grad, const void *x, void *scratch, unsigned *words, hipStream_t s);
int launch_few_wgrad_reduce(const FewGradPlan &pl, const WgradSums &single, void *dw, void *scratch, unsigned *words, hipStream_t s);

}  // namespace mg
