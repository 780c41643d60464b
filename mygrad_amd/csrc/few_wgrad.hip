// Filter gradient of single-precision layers with few terms to a filter, such as a first layer's 3 x 7 x 7, on the bf16
// matrix instructions: see conv_split.hip for the arithmetic and its accuracy (two accumulators), few_split.hip for the patch.
//
// What bounds it: (64,3,225,225) * (64,3,7,7), stride 2, 15.4 GFLOP, takes 149 - 166 us, its reduction and the single-precision kernel that
// returns at once 10 (227 there, 68 TFLOP/s): 25 tiles a block of about 5.5 us each, of which the products are 1.8 at the
// instruction's rate; the modelled time puts 1.5 of the rest on the requests of the next tile.  Four bytes a request and lane it took 217, where
// this took 158.  The matrix pipes are 32 % busy, seven vector instructions to a product.
// (112,44,3493) * (237,44,3) 402 -> 302.  Error against 64 bits (2-norm), normal values: 2.4e-7 (single precision 1.0e-6).
//
// What the parts cannot represent (a sum that is not finite, or smaller than what lost bits of its operands can have been worth) sets a word, and the
// single-precision kernel behind computes the gradient (see wgrad_split.h).
#include "few_wgrad.h"
#include "few_device.h"
#include "internal.h"
#include "wgrad_sums.h"

#include <algorithm>
#include <cstdlib>

namespace mg {

namespace {

constexpr int kWaves = 8, kPositions = 128;

// A block sums 16 TM filters by 32 TK columns (terms of a filter) over its tiles of 128 positions: waves 2 along the columns by 4 along the
// positions, 32 of a tile each.  A tile's patch of x and its rows of grad go straight into LDS while the tile before is
// multiplied; a lane reads the eight values of its column (or filter) at eight positions and splits them in registers.
template <int TM, int TK>
__global__ void __launch_bounds__(64 * kWaves, 2) few_wgrad_kernel(const FewGradParams params) {
  constexpr int BM = 16 * TM, BK = 32 * TK, GRAD = BM * kPositions;
  const FewParams &p = params.at;
  // [2] rows of grad, 128 positions each; [2] bytes to each position in the patch; [2] patches.  At the end: sums of two waves along the positions
  extern __shared__ __attribute__((aligned(16))) float lds[];
  int *const position_at = reinterpret_cast<int *>(lds + 2 * GRAD);
  float *const patches = lds + 2 * GRAD + 2 * kPositions;
  const int lane = (int)threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4, wave = uniform((int)threadIdx.x >> 6), cw = wave & 1, kq = wave >> 1;
  const int grid = (int)gridDim.x, place = grid % 8 == 0 ? (int)(blockIdx.x & 7) * (grid / 8) + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
  const int m0 = place % p.m_tiles * BM, first_item = place / p.m_tiles;
  const unsigned lds_at = (unsigned)reinterpret_cast<unsigned long long>((__attribute__((address_space(3))) char *)lds);
  const unsigned patches_at = lds_at + (unsigned)(2 * GRAD + 2 * kPositions) * 4u;
  auto request = [&](int item, int buf) {
    const FewTile t = few_tile<kPositions>(p, item);
    for (int line = wave; line < p.C * p.patch_rows; line += kWaves) few_request_line(p, t, line, patches_at + (unsigned)(buf * p.patch) * 4u, lane);
    // Two filters' positions at a time, sixteen bytes a lane.  Piece s of row r holds positions 4 (s ^ r % 16) and on, so that sixteen rows' reads are
    // free of bank conflicts; what is loaded of the next row beyond the last position is masked where it is read.
    const __amdgpu_buffer_rsrc_t grad = buffer_of(params.grad, params.grad_bytes);
    const unsigned at = (unsigned)((t.n * p.F + m0) * p.gvol + t.q0) * 4u;
    for (int pair = wave; pair < BM / 2; pair += kWaves) {
      const int r = pair * 2 + lane / 32, q = ((lane & 31) ^ (r & 15)) * 4;
      const bool there = m0 + r < p.F && t.q0 + q < t.end;
      to_lds<16>(grad, there ? at + (unsigned)(r * p.gvol + q) * 4u : kOutside, 0, lds_at + (unsigned)(buf * GRAD + pair * 2 * kPositions) * 4u);
    }
    if ((int)threadIdx.x < kPositions) {
      const int q = min(t.q0 + (int)threadIdx.x, t.end - 1), row = (int)p.by_row.div((unsigned)q);
      position_at[buf * kPositions + (int)threadIdx.x] = ((row - t.row) * p.S1 * p.pitch + (q - row * p.G2 - t.col) * p.S2 + max(p.lead, 0)) * 4;
    }
  };
  int term_at[TK];  // bytes: of the lane's columns, in the patch (beyond the last one: the first one)
#pragma unroll
  for (int j = 0; j < TK; ++j) {
    const int k = (cw * TK + j) * 16 + l16;
    const int c = (int)p.by_window.div((unsigned)k), tap = k - c * (int)p.by_window.d, t1 = (int)p.by_w2.div((unsigned)tap), t2 = tap - t1 * p.W2;
    term_at[j] = k < p.K ? ((c * p.patch_rows + t1 * p.D1) * p.pitch + t2 * p.D2) * 4 : 0;
  }
  // Sums of the large product and of the five small ones; where two accumulators for every column do not fit 256 registers, small
  // ones of a tile, added one column later.
  constexpr bool OWN = TM * TK < 16;
  constexpr int LOWS = OWN ? TK : 2;
  f32x4 acc[TK][TM], low[LOWS][TM];
#pragma unroll
  for (int j = 0; j < TK; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i) acc[j][i] = low[j % LOWS][i] = f32x4{0, 0, 0, 0};
  unsigned lost = 0;
  float raw[8];
  auto split = [&](bf16x8(&into)[3]) {
    u32x4 parts[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      unsigned h, m, l;
      split_pair(raw[2 * e], raw[2 * e + 1], h, m, l, lost);
      parts[0][e] = h, parts[1][e] = m, parts[2][e] = l;
    }
#pragma unroll
    for (int part = 0; part < 3; ++part) into[part] = __builtin_bit_cast(bf16x8, parts[part]);
  };

  int item = first_item;
  if (item < p.items) {
    request(item, 0);
    landed();
  }
  for (int buf = 0; item < p.items; buf ^= 1) {
    const FewTile here = few_tile<kPositions>(p, item);
    const int live = here.end - here.q0 - kq * 32 - lk * 8;  // positions from this lane's first one on
    const bool whole = here.end - here.q0 == kPositions;
    item += params.splits;
    if (item < p.items) request(item, buf ^ 1);
    const char *const patch = reinterpret_cast<const char *>(patches + buf * p.patch);
    const float *const rows = lds + buf * GRAD + l16 * kPositions;
    const int piece0 = ((kq * 8 + lk * 2) ^ l16) * 4, piece1 = ((kq * 8 + lk * 2 + 1) ^ l16) * 4;
    int at[8];
    {
      const int4v *const from = reinterpret_cast<const int4v *>(position_at + buf * kPositions + kq * 32 + lk * 8);
      const int4v a = from[0], b = from[1];
#pragma unroll
      for (int e = 0; e < 4; ++e) at[e] = a[e], at[e + 4] = b[e];
    }
    bf16x8 g[TM][3], x[2][3];
    auto gather = [&](int j) {
#pragma unroll
      for (int e = 0; e < 8; ++e) raw[e] = *reinterpret_cast<const float *>(patch + (at[e] + term_at[j]));
    };
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const f32x4 a = *reinterpret_cast<const f32x4 *>(rows + i * 16 * kPositions + piece0), b = *reinterpret_cast<const f32x4 *>(rows + i * 16 * kPositions + piece1);
#pragma unroll
      for (int e = 0; e < 4; ++e) raw[e] = a[e], raw[e + 4] = b[e];
      if (!whole) {
#pragma unroll
        for (int e = 0; e < 8; ++e) raw[e] = e < live ? raw[e] : 0.0f;
      }
      split(g[i]);
    }
    gather(0);
    split(x[0]);
    if (TK > 1) gather(1);
#pragma unroll
    for (int j = 0; j < TK; ++j) {
      // smallest products first; beside the first half of them the next column's values are split
      constexpr int PX[6] = {2, 0, 1, 1, 0, 0}, PG[6] = {0, 2, 1, 0, 1, 0};
      __builtin_amdgcn_sched_barrier(0);
      if (j + 1 < TK) split(x[(j + 1) % 2]);
#pragma unroll
      for (int k = 0; k < 6; ++k) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          f32x4 &into = k < 5 ? low[j % LOWS][i] : acc[j][i];
          const f32x4 onto = !OWN && k == 0 ? f32x4{0, 0, 0, 0} : into;
          into = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j % 2][PX[k]], g[i][PG[k]], onto, 0, 0, 0);
        }
        if (!OWN && k == 3 && j > 0) {
#pragma unroll
          for (int i = 0; i < TM; ++i) acc[j - 1][i] += low[(j - 1) % 2][i];
        }
        if (k == 2) {
          if (j + 1 < TK) {
#pragma unroll
            for (int u = 0; u < 3 * TM; ++u) {
              __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);              // a product
              __builtin_amdgcn_sched_group_barrier(0x002, 48 / (3 * TM), 0);  // vector instructions
            }
          }
          __builtin_amdgcn_sched_barrier(0);
          if (j + 2 < TK) gather(j + 2);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if constexpr (!OWN) {
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[TK - 1][i] += low[(TK - 1) % 2][i];
    }
    landed();  // the next tile is there, and nobody reads this one any more
  }

  // ---- the sums of the waves along the positions, two and two; acc[j][i][q] is filter 16 i + l16, column 16 (cw TK + j) + 4 lk + q
  constexpr int SUMS = BK + 4;
#pragma unroll
  for (int j = 0; j < TK; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i)
      if (OWN) acc[j][i] += low[j % LOWS][i];
  // (behind what the block loads, and behind its sums)
  constexpr int ROWS = BM + BK;  // filters, then columns
  unsigned *const notes = reinterpret_cast<unsigned *>(lds + max(2 * (GRAD + kPositions + p.patch), 2 * BM * SUMS)), *const waves = notes + 2 * ROWS;
  const bool own_lost = __any((lost & 0xffffu) != 0);
  if (lane == 0) waves[wave] = own_lost;
  float *const sums = lds + l16 * SUMS + cw * TK * 16 + lk * 4;
#pragma unroll
  for (int round = 0; round < 2; ++round) {
    const int step = 1 << round;  // 1 into 0 and 3 into 2, then 2 into 0
    __syncthreads();
    if ((kq & (2 * step - 1)) == step) {
#pragma unroll
      for (int j = 0; j < TK; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) *reinterpret_cast<f32x4 *>(sums + (kq >> (round + 1)) * BM * SUMS + i * 16 * SUMS + j * 16) = acc[j][i];
    }
    __syncthreads();
    if ((kq & (2 * step - 1)) == 0) {
#pragma unroll
      for (int j = 0; j < TK; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[j][i] += *reinterpret_cast<const f32x4 *>(sums + (kq >> (round + 1)) * BM * SUMS + i * 16 * SUMS + j * 16);
    }
  }
  bool any = false;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) any |= waves[w] != 0;
  if (any) {  // seldom: a second look at the block's values, for the widest of every filter and column, and whether it has lost bits
    for (int r = (int)threadIdx.x; r < 2 * ROWS; r += 64 * kWaves) notes[r] = 0;
    float widest[TM + TK];
    unsigned low[TM + TK];
#pragma unroll
    for (int r = 0; r < TM + TK; ++r) widest[r] = 0.0f, low[r] = 0;
    auto look = [&](int r) {
      unsigned h, m, l;
#pragma unroll
      for (int e = 0; e < 8; e += 2) split_pair(raw[e], raw[e + 1], h, m, l, low[r]), widen(widest[r], raw[e], raw[e + 1]);
    };
    item = first_item;
    __syncthreads();  // the sums, which lie where the loads go, have been read
    request(item, 0);
    landed();
    for (int buf = 0; item < p.items; buf ^= 1) {
      const FewTile here = few_tile<kPositions>(p, item);
      const int from = kq * 32 + lk * 8, live = here.end - here.q0 - from;
      item += params.splits;
      if (item < p.items) request(item, buf ^ 1);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const float *const row = lds + buf * GRAD + (i * 16 + l16) * kPositions;
#pragma unroll
        for (int e = 0; e < 8; ++e) raw[e] = e < live ? row[(((from + e) / 4) ^ l16) * 4 + e % 4] : 0.0f;
        look(i);
      }
#pragma unroll
      for (int j = 0; j < TK; ++j) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          raw[e] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(patches + buf * p.patch) + (position_at[buf * kPositions + from + e] + term_at[j]));
        look(TM + j);
      }
      landed();
    }
#pragma unroll
    for (int r = 0; r < TM + TK; ++r) {
      const int row = (r < TM ? r : TM + cw * TK + r - TM) * 16 + l16;
      atomicMax(&notes[row], bits_of(widest[r]));
      if ((low[r] & 0xffffu) != 0) atomicOr(&notes[ROWS + row], 1u);
    }
    __syncthreads();
  }
  if (kq != 0) return;
  const int terms = ((p.items - first_item - 1) / params.splits + 1) * kPositions;
  bool odd = false;  // a sum is not finite, or smaller than what lost bits can have been worth
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + i * 16 + l16;
    if (m >= p.F) continue;
    float *const out = params.partial + ((long long)first_item * p.F + m) * p.K;
#pragma unroll
    for (int j = 0; j < TK; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = (cw * TK + j) * 16 + lk * 4 + q;
        if (k >= p.K) continue;
        out[k] = acc[j][i][q];
        odd |= !(__builtin_fabsf(acc[j][i][q]) < __builtin_inff());
        if (any) {
          const int f = i * 16 + l16, c = BM + k;
          odd |= !(__builtin_fabsf(acc[j][i][q]) >= least_sum(notes[ROWS + f] != 0, float_of(notes[f]), notes[ROWS + c] != 0, float_of(notes[c]), terms));
        }
      }
  }
  if (__any(odd) && lane == 0) atomicOr(&params.words[0], 1u);
}

// dw from the partial sums, in the order of the splits, four runs of them at a time (see wgrad_split_reduce_kernel).
__global__ void __launch_bounds__(256) few_wgrad_reduce_kernel(const FewGradParams params, float *dw, const WgradSums single) {
  __shared__ float runs[4][64];
  const FewParams &p = params.at;
  const int t = (int)threadIdx.x, q = t / 64, count = p.F * p.K, e = (int)blockIdx.x * 64 + t % 64;
  if (params.words[0] == 0) {
    const int per = (params.splits + 3) / 4, first = min(q * per, params.splits), last = min(first + per, params.splits);
    runs[q][t % 64] = e < count && first < last ? sum_in_order(params.partial + (long long)first * count + e, count, last - first) : 0.0f;
    __syncthreads();
    if (q == 0 && e < count) {
      float sum = runs[0][t];
#pragma unroll
      for (int r = 1; r < 4; ++r) sum += runs[r][t];
      dw[e] = sum;
    }
  } else if (single.partial != nullptr) {
    reduce_single(single, dw, p.F, p.C, p.K / p.C);
  }
  leave_words(params.words);
}

#define MG_FEW_GRADS(X) X(4, 1) X(4, 2) X(4, 3) X(4, 4) X(4, 5) X(2, 1) X(2, 2) X(2, 3) X(2, 4) X(2, 5)

size_t few_lds(const FewGradPlan &pl) {
  const size_t bm = 16 * pl.tm;
  return (std::max<size_t>(2 * (bm * kPositions + kPositions + pl.p.at.patch), 2 * bm * (32 * pl.tk + 4)) + 2 * (bm + 32 * pl.tk) + kWaves) * 4;
}

}  // namespace

// Modelled time in us: fitted to 85 timed layers, 9 in 10 within 6 % of it.
FewGradPlan plan_few_wgrad(int N, int C, int F, const int *X, const int *G, const int *W, const int *S, const int *D, const int *P, int cus) {
  FewGradPlan best;
  const long long K = (long long)C * W[1] * W[2];
  if (K > 160 || F > 4096) return best;
  for (const bool along : {false, true}) {
    FewGradPlan pl;
    pl.tm = F > 32 ? 4 : 2, pl.tk = (int)ceil_div(K, 32);
    FewParams &p = pl.p.at;
    if (!few_geometry(p, N, C, F, X, G, W, S, D, P, 16 * pl.tm, kPositions, along) || p.m_tiles > cus || few_lds(pl) > (size_t)kFewLds) continue;
    pl.p.splits = std::max(1, std::min(p.items, cus / p.m_tiles));
    const double rounds = (double)ceil_div(p.items, pl.p.splits), requests = (double)(few_requests(p) + 8 * pl.tm);
    pl.time = 19.1 + rounds * (0.785 + 0.161 * pl.tm * pl.tk + 0.0157 * requests) + 0.518e-6 * 8.0 * (double)pl.p.splits * F * (double)K;
    if (best.tm == 0 || pl.time < best.time) best = pl;
  }
  return best;
}

size_t few_wgrad_scratch(const FewGradPlan &pl) { return ((size_t)pl.p.splits * pl.p.at.F * pl.p.at.K * 4 + 255) & ~size_t(255); }

int launch_few_wgrad(const FewGradPlan &pl, const void *grad, const void *x, void *scratch, unsigned *words, hipStream_t s) {
  FewGradParams p = pl.p;
  const size_t samples = (size_t)(p.at.items / p.at.sample_tiles);
  p.at.x = static_cast<const float *>(x), p.at.x_bytes = (unsigned)(samples * p.at.C * p.at.X1 * p.at.X2 * 4);
  p.grad = static_cast<const float *>(grad), p.grad_bytes = (unsigned)(samples * p.at.F * p.at.gvol * 4);
  p.partial = static_cast<float *>(scratch), p.words = words;
  ScopedTiming timed(TAG_CONV_WGRAD);
#define MG_FEW_GRAD(TM, TK)                                                                                                              \
  if (pl.tm == TM && pl.tk == TK) {                                                                                                 \
    static const hipError_t allowed = hipFuncSetAttribute((const void *)few_wgrad_kernel<TM, TK>, hipFuncAttributeMaxDynamicSharedMemorySize, kFewLds); \
    MG_HIP(allowed);                                                                                                                \
    hipLaunchKernelGGL((few_wgrad_kernel<TM, TK>), dim3((unsigned)(p.splits * p.at.m_tiles)), dim3(64 * kWaves), few_lds(pl), s, p);      \
  }
  MG_FEW_GRADS(MG_FEW_GRAD)
#undef MG_FEW_GRAD
  MG_HIP(hipGetLastError());
  return MG_OK;
}

int launch_few_wgrad_reduce(const FewGradPlan &pl, const WgradSums &single, void *dw, void *scratch, unsigned *words, hipStream_t s) {
  FewGradParams p = pl.p;
  p.partial = static_cast<float *>(scratch), p.words = words;
  ScopedTiming timed(TAG_WGRAD_REDUCE);
  hipLaunchKernelGGL(few_wgrad_reduce_kernel, dim3((unsigned)ceil_div(p.at.F * p.at.K, 64)), dim3(256), 0, s, p, static_cast<float *>(dw), single);
  MG_HIP(hipGetLastError());
  return MG_OK;
}

}  // namespace mg
