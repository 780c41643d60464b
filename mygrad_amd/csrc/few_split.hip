// Forward pass of single-precision layers with few terms to a sum, such as a first layer's 3 x 7 x 7, on the bf16 matrix
// instructions: see conv_split.hip for the arithmetic and its accuracy (two accumulators).
//
// What bounds it: (64,3,225,225) * (64,3,7,7), stride 2, 15.4 GFLOP, takes 136 - 147 us (184 - 187 with one position per lane on the
// single-precision instruction); 100 - 110 of them without its loads and stores (92 GFLOP of parts and 8 % of dead terms, 46 us at
// the instruction's rate: eight waves to a unit, which all wait for a tile's patch, hide little of each other's latency), 69 with nothing
// but loads and stores (209 MB; loads of four bytes a lane, 141 us in all).  (48,4,123,123) * (84,4,5,5) 186 -> 157, (25,24,6716) * (178,24,5) 118 -> 82.
// Error against 64 bits (2-norm), normal values: 6.9e-8 (single precision 2.2e-7); at 27 terms 3.7e-8 (9.5e-8).
//
// What the parts cannot represent (an infinity, a NaN, an overflow, low bits below the smallest number of bf16): the wave that
// meets it computes its results again on the single-precision instruction, from the patch and the filters themselves; no other
// result's bits depend on it.
#include "few_device.h"
#include "internal.h"

#include <algorithm>
#include <cstdlib>

namespace mg {

namespace {

constexpr int kWaves = 8;

// A block keeps 16 TM filters, split, in LDS, and walks over tiles of 128 TN positions, 16 TN of them a wave.  The patch of x that a
// tile's windows touch goes into LDS as it is (two of them: the next tile's is loaded meanwhile); a lane reads the eight
// terms of its position one by one -- so that any window, stride and dilation leaves no dead terms but those up to a multiple of
// 32 -- and splits them in registers, once for all filters of the block.
template <int TM, int TN>
__global__ void __launch_bounds__(64 * kWaves, 2) few_split_kernel(const FewParams p) {
  constexpr int BM = 16 * TM, BN = 16 * TN * kWaves;
  // filters [step][part][octet of terms][row]; where a term lies in the patch, for one step more; two patches; of each filter the widest
  // value, and whether it has lost bits
  extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
  const int pieces = p.steps * 12 * BM, terms = p.steps * 32;
  int *const term_at = reinterpret_cast<int *>(lds + pieces);
  float *const patches = reinterpret_cast<float *>(term_at + terms + 32);
  unsigned *const notes = reinterpret_cast<unsigned *>(patches + 2 * p.patch);
  const int lane = (int)threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4, wave = uniform((int)threadIdx.x >> 6);
  // blocks are dealt to the eight XCDs in turn: an XCD's blocks take neighbouring tiles
  const int grid = (int)gridDim.x, place = grid % 8 == 0 ? (int)(blockIdx.x & 7) * (grid / 8) + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
  const int m0 = place % p.m_tiles * BM, stride = grid / p.m_tiles;

  const unsigned patches_at = (unsigned)reinterpret_cast<unsigned long long>((__attribute__((address_space(3))) char *)lds) + (unsigned)(pieces * 16 + (terms + 32) * 4);
  // the wave's share of a tile's patch: every eighth row of a channel, `count` of them from number `from` on
  const int lines = p.C * p.patch_rows, own_lines = (lines - wave + kWaves - 1) / kWaves;
  auto request = [&](const FewTile &t, int buf, int from, int count) {
    for (int own = from; own < min(from + count, own_lines); ++own) few_request_line(p, t, wave + own * kWaves, patches_at + (unsigned)(buf * p.patch) * 4u, lane);
  };
  int item = place / p.m_tiles;
  if (item >= p.items) return;
  request(few_tile<BN>(p, item), 0, 0, own_lines);

  // ---- the filters of the block, and where their terms lie
  if (threadIdx.x < 2 * BM) notes[threadIdx.x] = 0;
  for (int k = (int)threadIdx.x; k < terms + 32; k += 64 * kWaves) {
    const int c = (int)p.by_window.div((unsigned)k), tap = k - c * (int)p.by_window.d, t1 = (int)p.by_w2.div((unsigned)tap), t2 = tap - t1 * p.W2;
    term_at[k] = k < p.K ? ((c * p.patch_rows + t1 * p.D1) * p.pitch + t2 * p.D2) * 4 : 0;
  }
  __syncthreads();
  unsigned lost;
  for (int at = (int)threadIdx.x; at < p.steps * 4 * BM; at += 64 * kWaves) {
    const int m = at % BM, oct = at / BM;
    u32x4 parts[3];
    float widest = 0.0f;
    lost = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int k = oct * 8 + 2 * e + u;
        v[u] = m0 + m < p.F && k < p.K ? p.w[(long long)(m0 + m) * p.K + k] : 0.0f;
      }
      unsigned first, second, third;
      split_pair(v[0], v[1], first, second, third, lost);
      widen(widest, v[0], v[1]);
      parts[0][e] = first, parts[1][e] = second, parts[2][e] = third;
    }
    atomicMax(&notes[m], bits_of(widest));
    if ((lost & 0xffffu) != 0) atomicOr(&notes[BM + m], 1u);
#pragma unroll
    for (int part = 0; part < 3; ++part) lds[((oct / 4 * 3 + part) * 4 + oct % 4) * BM + m] = parts[part];
  }
  landed();
  const bool lossy = __any(notes[BM + lane % BM] != 0);  // some filter value has lost bits

  const u32x4 *const filters = lds + lk * BM + l16;
  const int4v *const mine_at = reinterpret_cast<const int4v *>(term_at) + lk * 2;
  for (int buf = 0; item < p.items; buf ^= 1) {
    const FewTile t = few_tile<BN>(p, item);
    const int end = t.end, first = t.q0 + wave * 16 * TN;
    const char *const patch = reinterpret_cast<const char *>(patches + buf * p.patch);
    item += stride;
    const FewTile ahead = few_tile<BN>(p, min(item, p.items - 1));
    const int per_step = item < p.items ? (own_lines + p.steps - 1) / p.steps : 0;

    int base[TN];  // bytes: of the lane's positions, in the patch (beyond the last one: that one's)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int q = min(first + j * 16 + l16, end - 1), row = (int)p.by_row.div((unsigned)q);
      base[j] = ((row - t.row) * p.S1 * p.pitch + (q - row * p.G2 - t.col) * p.S2 + max(p.lead, 0)) * 4;
    }
    f32x4 acc[TN][TM], low[TN][TM];  // sums of the large product and of the five small ones
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] = low[j][i] = f32x4{0, 0, 0, 0};
    bf16x8 w[TM][3], x[2][3];
    int at[2][8];  // of the terms of this step and of the next one
    float raw[8];
    auto read_filters = [&](int step, int part) {
#pragma unroll
      for (int i = 0; i < TM; ++i) w[i][part] = __builtin_bit_cast(bf16x8, filters[(step * 3 + part) * 4 * BM + i * 16]);
    };
    auto read_terms_at = [&](int step, int(&into)[8]) {
      const int4v a = mine_at[step * 8], b = mine_at[step * 8 + 1];
#pragma unroll
      for (int e = 0; e < 4; ++e) into[e] = a[e], into[e + 4] = b[e];
    };
    auto gather = [&](int j) {  // of position j of the step, j >= TN: of the next one
#pragma unroll
      for (int e = 0; e < 8; ++e) raw[e] = *reinterpret_cast<const float *>(patch + (base[j % TN] + at[j / TN][e]));
    };
    lost = 0;
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
    read_terms_at(0, at[0]);
    gather(0);
#pragma unroll
    for (int part = 0; part < 3; ++part) read_filters(0, part);
    split(x[0]);
    gather(1);
    for (int step = 0; step < p.steps; ++step) {
      const int next = min(step + 1, p.steps - 1);
      read_terms_at(step + 1, at[1]);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        // Smallest products first; each part of the filters makes room for the next step's as soon as it has been used.  Beside
        // the first half of the products the next position's terms are split, beside the other one those behind it are on
        // their way.
        constexpr int PX[6] = {0, 1, 0, 2, 1, 0}, PW[6] = {2, 1, 1, 0, 0, 0};
        __builtin_amdgcn_sched_barrier(0);
        split(x[(j + 1) % 2]);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            f32x4 &into = k < 5 ? low[j][i] : acc[j][i];
            into = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j % 2][PX[k]], w[i][PW[k]], into, 0, 0, 0);
          }
          if (k == 2) {
#pragma unroll
            for (int u = 0; u < 3 * TM; ++u) {
              __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product
              __builtin_amdgcn_sched_group_barrier(0x002, 48 / (3 * TM), 0);  // vector instructions
            }
            __builtin_amdgcn_sched_barrier(0);
            gather(j + 2);
            if (j == 0) request(ahead, buf ^ 1, step * per_step, per_step);  // (all at once they would hold the waves up)
            if (j + 1 == TN) read_filters(next, 2), read_filters(next, 1);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (j + 1 == TN) read_filters(next, 0);
      }
      if constexpr (TN % 2 != 0) {
#pragma unroll
        for (int part = 0; part < 3; ++part) x[0][part] = x[1][part];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) at[0][e] = at[1][e];
    }

    // ---- acc[j][i][q] is filter m0 + 16 i + l16 at position first + 16 j + 4 lk + q
    unsigned largest = 0;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        acc[j][i] += low[j][i];
#pragma unroll
        for (int q = 0; q < 4; ++q) largest = max(largest, bits_of(acc[j][i][q]) << 1);
      }
    // What the parts cannot hold: the wave's results again on the single-precision instruction.  Lost bits count where a result is not far above
    // what they can have been worth; the widest values of the wave's positions are looked up then.
    bool again = __any(largest >= 2u * (255u << 23));
    if (!again && (lossy || __any((lost & 0xffffu) != 0))) {
      bool below = false;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        float widest = 0.0f;
        unsigned low = 0;
        for (int step = 0; step < p.steps; ++step) {
          int terms[8];
          read_terms_at(step, terms);
#pragma unroll
          for (int e = 0; e < 8; ++e) raw[e] = *reinterpret_cast<const float *>(patch + (base[j] + terms[e]));
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            unsigned h, m, l;
            split_pair(raw[e], raw[e + 1], h, m, l, low);
            widen(widest, raw[e], raw[e + 1]);
          }
        }
#pragma unroll
        for (int d = 16; d < 64; d *= 2) {
          widest = fmaxf(widest, __shfl_xor(widest, d));
          low |= (unsigned)__shfl_xor((int)low, d);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float widest_x = __shfl(widest, lk * 4 + q);
          const bool lost_x = ((unsigned)__shfl((int)low, lk * 4 + q) & 0xffffu) != 0;
#pragma unroll
          for (int i = 0; i < TM; ++i)
            below |= !(__builtin_fabsf(acc[j][i][q]) >= least_sum(notes[BM + i * 16 + l16] != 0, float_of(notes[i * 16 + l16]), lost_x, widest_x, p.K));
        }
      }
      again = __any(below);
    }
    if (again) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[j][i] = f32x4{0, 0, 0, 0};
      for (int k0 = 0; k0 < p.K; k0 += 4) {
        const int k = k0 + lk;
        const bool real = k < p.K;
        float ws[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) ws[i] = real && m0 + i * 16 + l16 < p.F ? p.w[(long long)(m0 + i * 16 + l16) * p.K + k] : 0.0f;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const float xs = real ? *reinterpret_cast<const float *>(patch + (base[j] + term_at[k])) : 0.0f;
#pragma unroll
          for (int i = 0; i < TM; ++i) acc[j][i] = Mma<float>::run(xs, ws[i], acc[j][i]);
        }
      }
    }
    landed();  // the next patch is there, and nobody reads this one any more
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + i * 16 + l16;
      if (m >= p.F) continue;
      float *const out = p.dst + ((long long)t.n * p.F + m) * p.gvol;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        typedef float Quad __attribute__((ext_vector_type(4), aligned(4)));
        const int q = first + j * 16 + lk * 4;
        if (q + 4 <= end) {
          *reinterpret_cast<Quad *>(out + q) = acc[j][i];
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (q + u < end) out[q + u] = acc[j][i][u];
        }
      }
    }
  }
}

#define MG_FEW_SHAPES(X) X(4, 3) X(4, 2) X(2, 4) X(2, 2)

size_t few_lds(const FewPlan &pl) { return (size_t)pl.p.steps * 12 * 16 * pl.tm * 16 + (pl.p.steps + 1) * 32 * 4 + 2 * (size_t)pl.p.patch * 4 + 2 * 16 * pl.tm * 4; }

}  // namespace

// Tiles of BM filters by `positions`, and their patches of x.
bool few_geometry(FewParams &p, int N, int C, int F, const int *X, const int *G, const int *W, const int *S, const int *D, const int *P, int bm, int positions, bool along) {
  const long long K = (long long)C * W[1] * W[2], gvol = (long long)G[1] * G[2];
  if (X[0] != 1 || G[0] != 1 || W[0] != 1 || P[0] != 0 || gvol > 1 << 29 || N > 1 << 24) return false;
  p.C = C, p.F = F, p.K = (int)K, p.steps = (int)ceil_div(K, 32);
  p.X1 = X[1], p.X2 = X[2], p.G2 = G[2], p.gvol = (int)gvol;
  p.S1 = S[1], p.S2 = S[2], p.D1 = D[1], p.D2 = D[2], p.P1 = P[1], p.P2 = P[2], p.W1 = W[1], p.W2 = W[2];
  p.m_tiles = (int)ceil_div(F, bm), p.along = along, p.lead = -1;
  const long long rows = along ? 1 : std::min<long long>(G[1], ceil_div(positions - 1, G[2]) + 1), columns = along ? std::min(positions, G[2]) : G[2];
  const long long patch_rows = (rows - 1) * S[1] + (W[1] - 1ll) * D[1] + 1, needed = (columns - 1) * S[2] + (W[2] - 1ll) * D[2] + 1;
  long long pitch = needed;
  if (needed > 64) p.lead = (4 - P[2] % 4) % 4, pitch = ceil_div(p.lead + needed, 4) * 4;
  if (patch_rows > kFewLds || pitch > kFewLds || C * patch_rows * pitch * 8 > kFewLds) return false;
  p.patch_rows = (int)patch_rows, p.pitch = (int)pitch, p.patch = (int)ceil_div(C * patch_rows * pitch, 4) * 4;
  p.run_tiles = (int)ceil_div(along ? G[2] : gvol, positions), p.sample_tiles = p.run_tiles * (along ? G[1] : 1);
  if ((long long)N * p.sample_tiles > 1 << 30) return false;
  p.items = N * p.sample_tiles;
  p.by_sample = make_fastdiv((unsigned)p.sample_tiles), p.by_run = make_fastdiv((unsigned)p.run_tiles), p.by_row = make_fastdiv((unsigned)G[2]);
  p.by_patch_rows = make_fastdiv((unsigned)patch_rows), p.by_window = make_fastdiv((unsigned)(W[1] * W[2])), p.by_w2 = make_fastdiv((unsigned)W[2]);
  return true;
}

long long few_requests(const FewParams &p) { return (long long)p.C * p.patch_rows * (p.lead < 0 ? 1 : ceil_div(p.pitch, 256) + (p.X2 % 4 != 0)); }

// The shape and the walk with the least modelled time, in us: fitted to 160 timed (layer, shape), 9 in 10 within 9 % of it.
FewPlan plan_few_split(int N, int C, int F, const int *X, const int *G, const int *W, const int *S, const int *D, const int *P, int cus) {
  FewPlan best;
  if ((long long)C * W[1] * W[2] > 192) return best;
  int want = 0;
  if (const char *v = getenv("MYGRAD_HIP_FEW")) want = atoi(v);  // 10 tm + tn (tests)
#define MG_SHAPE(TM, TN) {TM, TN},
  constexpr int shapes[][2] = {MG_FEW_SHAPES(MG_SHAPE)};
#undef MG_SHAPE
  for (const auto &shape : shapes) {
    FewPlan pl;
    pl.tm = shape[0], pl.tn = shape[1];
    if (want > 10 ? want != 10 * pl.tm + pl.tn : (F > 32) != (pl.tm == 4)) continue;
    FewParams &p = pl.p;
    const int bn = 16 * pl.tn * kWaves;
    for (const bool along : {false, true}) {
      if (!few_geometry(p, N, C, F, X, G, W, S, D, P, 16 * pl.tm, bn, along) || p.m_tiles > cus || few_lds(pl) > (size_t)kFewLds) continue;
      const int per = std::max(1, std::min(p.items, cus / p.m_tiles));
      pl.grid = per * p.m_tiles;
      const double rounds = (double)ceil_div(p.items, per);
      const double requests = (double)few_requests(p);
      pl.time = 8.2 + 0.208 * p.steps + rounds * (0.895 + 0.162 * p.steps * pl.tn * pl.tm + 0.0155 * requests) + 0.137e-6 * 4.0 * (double)N * F * (double)p.gvol;
      if (best.tm == 0 || pl.time < best.time) best = pl;
    }
  }
  return best;
}

int launch_few_split(const FewPlan &pl, const void *x, const void *w, void *out, hipStream_t s) {
  FewParams p = pl.p;
  p.x = static_cast<const float *>(x), p.w = static_cast<const float *>(w), p.dst = static_cast<float *>(out);
  const long long samples = p.items / p.sample_tiles;
  p.x_bytes = (unsigned)(samples * p.C * p.X1 * p.X2 * 4);
  ScopedTiming timed(TAG_CONV_FWD);
#define MG_FEW(TM, TN)                                                                                                              \
  if (pl.tm == TM && pl.tn == TN) {                                                                                                 \
    static const hipError_t allowed = hipFuncSetAttribute((const void *)few_split_kernel<TM, TN>, hipFuncAttributeMaxDynamicSharedMemorySize, kFewLds); \
    MG_HIP(allowed);                                                                                                                \
    hipLaunchKernelGGL((few_split_kernel<TM, TN>), dim3((unsigned)pl.grid), dim3(64 * kWaves), few_lds(pl), s, p);                   \
  }
  MG_FEW_SHAPES(MG_FEW)
#undef MG_FEW
  MG_HIP(hipGetLastError());
  return MG_OK;
}

}  // namespace mg
