// Products of many small matrix pairs in one launch: out[p] = op(a[p]) @ op(b[p]), p < batch,
// where op transposes or not.  A pair of stacks whose matrices are too small to fill the device
// one pair at a time (np.matmul on two stacks, an einsum with a label that both operands and
// the result carry) is bound by launches, not arithmetic, when each pair gets a launch of the
// convolution kernels; here a wavefront makes one 16x16 tile of one product on the matrix cores,
// reading its operands where they lie (a transposed operand is a pair of swapped strides), so the
// whole stack is one grid.  Where it costs less (stack_time) it goes through a second kernel, where
// a block of four wavefronts makes a tile of one product from operands it has copied to
// LDS once (16 bytes per lane, coalesced) instead of every wavefront fetching its own rows and
// columns through L1.  Large pairs stay with the tiled convolution kernels.
#include "internal.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

namespace mg {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

// D(16x16) += A(16x4) * B(4x16) on one wavefront: lane l supplies A[l%16][l/16] and
// B[l/16][l%16] and receives four elements of column l%16 of D, in rows row_of(l, r).
template <typename T>
struct Tile;

template <>
struct Tile<float> {
  using Acc = f32x4;
  static __device__ __forceinline__ Acc run(float a, float b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row_of(int lane, int r) { return 4 * (lane >> 4) + r; }
};

template <>
struct Tile<double> {
  using Acc = f64x4;
  static __device__ __forceinline__ Acc run(double a, double b, Acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ int row_of(int lane, int r) { return 4 * r + (lane >> 4); }
};

struct BatchedParams {
  int M, K, N;
  int row_tiles, col_tiles;
  int pairs, dealt;                  // staged kernel: pairs, and whether they are dealt out to the XCDs in turn
  long long tiles;                   // batch * row_tiles * col_tiles
  long long a_pair, a_row, a_col;    // element strides of op(a): between pairs, along M, along K
  long long b_pair, b_row, b_col;    // of op(b): between pairs, along K, along N
};

// AV / BV: op(a) / op(b) is contiguous along K and K is a multiple of the 16-byte piece, so a
// lane reads a piece of VEC consecutive k at once.  The sum over k may run in any order as long
// as both operands use the same one: in a block of 4 * VEC values of k, the four lane groups
// (lane / 16 = q) take k = k0 + VEC * q + s at step s, which makes a lane's VEC steps one piece.
template <typename T, bool AV, bool BV>
__global__ void __launch_bounds__(256) batched_product_kernel(BatchedParams p, const T *__restrict__ a, const T *__restrict__ b,
                                                              T *__restrict__ out) {
  constexpr int VEC = 16 / sizeof(T);
  typedef T V __attribute__((ext_vector_type(VEC)));
  const int lane = threadIdx.x & 63;
  const long long tile = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);  // the same for a whole wavefront
  if (tile >= p.tiles) return;
  const int per_pair = p.row_tiles * p.col_tiles;
  const long long pair = tile / per_pair;
  const int within = (int)(tile - pair * per_pair);
  const int row0 = (within / p.col_tiles) * 16, col0 = (within % p.col_tiles) * 16;
  const int i = row0 + (lane & 15), j = col0 + (lane & 15), kk = lane >> 4;
  // rows and columns beyond the matrix supply zeros and are not stored
  const bool row_in = i < p.M, col_in = j < p.N;
  const T *pa = a + pair * p.a_pair + (row_in ? (long long)i * p.a_row : 0);
  const T *pb = b + pair * p.b_pair + (col_in ? (long long)j * p.b_col : 0);
  typename Tile<T>::Acc acc = {0, 0, 0, 0};
  const int whole = p.K & ~3;
  int done = 0;
  if constexpr (AV || BV) {
    const int blocked = p.K - p.K % (4 * VEC);
    for (; done < blocked; done += 4 * VEC) {
      const int k = done + VEC * kk;
      T av[VEC], bv[VEC];
      if constexpr (AV) {
        V v = {};
        if (row_in) v = *reinterpret_cast<const V *>(pa + k);
#pragma unroll
        for (int s = 0; s < VEC; ++s) av[s] = v[s];
      } else {
#pragma unroll
        for (int s = 0; s < VEC; ++s) av[s] = row_in ? pa[(long long)(k + s) * p.a_col] : T(0);
      }
      if constexpr (BV) {
        V v = {};
        if (col_in) v = *reinterpret_cast<const V *>(pb + k);
#pragma unroll
        for (int s = 0; s < VEC; ++s) bv[s] = v[s];
      } else {
#pragma unroll
        for (int s = 0; s < VEC; ++s) bv[s] = col_in ? pb[(long long)(k + s) * p.b_row] : T(0);
      }
#pragma unroll
      for (int s = 0; s < VEC; ++s) acc = Tile<T>::run(av[s], bv[s], acc);
    }
  }
  auto step = [&](int k0) {
    const int k = k0 + kk;
    const T av = row_in ? pa[(long long)k * p.a_col] : T(0);
    const T bv = col_in ? pb[(long long)k * p.b_row] : T(0);
    acc = Tile<T>::run(av, bv, acc);
  };
  if constexpr (AV || BV) {
    for (int k0 = done; k0 < whole; k0 += 4) step(k0);  // at most 4 * VEC - 1 values of k are left
  } else {
#pragma unroll 4
    for (int k0 = 0; k0 < whole; k0 += 4) step(k0);
  }
  if (whole < p.K) {  // the last one to three columns of op(a) / rows of op(b)
    const int k = whole + kk;
    const bool k_in = k < p.K;
    const T av = row_in && k_in ? pa[(long long)k * p.a_col] : T(0);
    const T bv = col_in && k_in ? pb[(long long)k * p.b_row] : T(0);
    acc = Tile<T>::run(av, bv, acc);
  }
  if (!col_in) return;
  T *po = out + pair * ((long long)p.M * p.N) + j;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = row0 + Tile<T>::row_of(lane, r);
    if (row < p.M) po[(long long)row * p.N] = acc[r];
  }
}


// ---- a tile of one product per block, operands staged in LDS -----------------------------------
// A block copies the pieces of op(a) and op(b) that its BM x BN tile needs, K chunk by K chunk, into
// LDS in the orientation they have in memory (a transposed operand is read differently, not stored
// differently), zeros beyond the matrices' edges, 16 bytes per lane whatever the row length (a
// global load of 16 bytes needs the alignment of an element only; the one piece of a row that the
// matrix's edge cuts goes element by element).  Each of the four wavefronts makes a 32 x 32 part.
//
// What bounds it: the trips of a chunk from memory to LDS to registers, not the matrix pipes, so
// the loads of the next chunk are issued before this one is multiplied, and the LDS reads are wide.
// Chunks of 128 bytes of k where there are many blocks (six or seven on a unit cover for one another:
// 794 x (86,117,322) 103 us, 117 with 256 bytes), of 64 values where there are few, whose trips
// follow one another (24 x (64,64,64) in double precision, forward: 6.4 -> 5.5 us).
// The sum over k may run in any order that both operands share: in a block of 4 * VEC values of k
// (VEC = 16 bytes) the lane groups (lane / 16 = q) take k = VEC * q + s at step s, so an operand
// that lies along k gives a lane VEC steps per LDS read; of one that lies along its rows or columns
// a lane takes two neighbours, the two MFMA fragments it feeds, per read.
template <typename T, bool TA, bool TB, int BM, int BN, int KC>
__global__ void __launch_bounds__(256) batched_staged_kernel(BatchedParams p, const T *__restrict__ a, const T *__restrict__ b,
                                                             T *__restrict__ out) {
  constexpr int VEC = 16 / sizeof(T);
  typedef T V __attribute__((ext_vector_type(VEC)));
  typedef T VU __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
  typedef T Pair __attribute__((ext_vector_type(2)));
  typedef T PairU __attribute__((ext_vector_type(2), aligned(sizeof(T))));
  static_assert((BM / 32) * (BN / 32) == 4, "four wavefronts of 32 x 32");
  // The stored pieces: rows x columns as in memory, rows 16-byte aligned in LDS.  Of pieces with k down
  // their rows the lane groups read rows VEC apart: 8 floats of padding put two groups' 32 banks
  // side by side.
  constexpr int AR = TA ? KC : BM, AC = TA ? BM : KC, LDA = AC + (TA ? 32 / (int)sizeof(T) : VEC);
  constexpr int BR = TB ? BN : KC, BC = TB ? KC : BN, LDB = BC + (TB ? VEC : 32 / (int)sizeof(T));
  constexpr int NA = AR * AC / VEC / 256, NB = BR * BC / VEC / 256;
  __shared__ __attribute__((aligned(16))) T As[AR * LDA];
  __shared__ __attribute__((aligned(16))) T Bs[BR * LDB];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, lk = lane >> 4;
  // Blocks are handed to the 8 XCDs round-robin, each with its own L2, in which the tiles of a pair
  // should meet: the pairs are dealt out to the XCDs in turn, so that all of them work on one
  // stretch of memory, or, with few pairs, an XCD takes one run of consecutive tiles, so that none
  // idles.  (Runs for 8192 pairs of 64^3: 76 -> 88 us, the XCDs' streams a power of two apart.)
  const int xcd = blockIdx.x % 8, nth = blockIdx.x / 8;
  const int per_pair = p.row_tiles * p.col_tiles;
  int pair, within;
  if (p.dealt) {
    pair = nth / per_pair * 8 + xcd;
    within = nth % per_pair;
    if (pair >= p.pairs) return;  // (the whole block)
  } else {
    const int per_xcd = gridDim.x / 8, extra = gridDim.x % 8;
    const int tile = xcd * per_xcd + min(xcd, extra) + nth;
    pair = tile / per_pair;
    within = tile - pair * per_pair;
  }
  const int row0 = (within / p.col_tiles) * BM, col0 = (within % p.col_tiles) * BN;
  const T *pa = a + (long long)pair * p.a_pair;
  const T *pb = b + (long long)pair * p.b_pair;

  // R x C elements of a stored matrix (`rows` x `cols`, row-major) from (r0, c0): through registers
  // into LDS; the loads of both operands are issued before either is parked, so that a chunk costs
  // one trip to memory, not two.  Loads are unconditional, from addresses clamped to the matrix (a
  // branch per piece is most of a short product's time); at its edges, a branch of the whole block,
  // pieces are put right before they are parked: the last one of a row was moved back to end with it.
  auto fetch = [&](auto rc, auto cc, const T *src, int rows, int cols, int r0, int c0, auto &reg) {
    constexpr int R = decltype(rc)::value, C = decltype(cc)::value, PIECES = C / VEC, PASS = 256 / PIECES;
    const int from = max(min(c0 + (tid % PIECES) * VEC, cols - VEC), 0);
#pragma unroll
    for (int i = 0; i < R / PASS; ++i) {
      const T *at = src + (long long)min(r0 + tid / PIECES + i * PASS, rows - 1) * cols + from;
      if (cols >= VEC) {
        reg[i] = *reinterpret_cast<const VU *>(at);
      } else {
#pragma unroll
        for (int s = 0; s < VEC; ++s) reg[i][s] = at[min(s, cols - 1)];
      }
    }
  };
  // (k: whether the rows, or else the columns, run along K.  What lies outside the matrix along M or N makes
  // results that are not stored, so only the columns of a row that is no whole pieces have to be put
  // back in place there; along K both operands are zero outside.)
  auto park = [&](auto rc, auto cc, auto k, int rows, int cols, int r0, int c0, T *dst, auto ld, auto &reg) {
    constexpr int R = decltype(rc)::value, C = decltype(cc)::value, PIECES = C / VEC, PASS = 256 / PIECES;
    constexpr bool K_ROWS = decltype(k)::value;
    const int c = c0 + (tid % PIECES) * VEC;
    if (c0 + C > cols && cols % VEC != 0) {
      const int moved = c - max(min(c, cols - VEC), 0);
#pragma unroll
      for (int i = 0; i < R / PASS; ++i) {
        V v = reg[i];
        if constexpr (VEC == 4)
          if (moved & 2) v = V{v[2], v[3], T(0), T(0)};
        if (moved & 1) {
#pragma unroll
          for (int s = 0; s + 1 < VEC; ++s) v[s] = v[s + 1];
        }
#pragma unroll
        for (int s = 0; s < VEC; ++s) reg[i][s] = K_ROWS || c + s < cols ? v[s] : T(0);
      }
    }
    if (K_ROWS ? r0 + R > rows : c0 + C > cols) {
#pragma unroll
      for (int i = 0; i < R / PASS; ++i)
        if (K_ROWS ? r0 + tid / PIECES + i * PASS >= rows : c >= cols) reg[i] = V{};
    }
#pragma unroll
    for (int i = 0; i < R / PASS; ++i)
      *reinterpret_cast<V *>(dst + (tid / PIECES + i * PASS) * decltype(ld)::value + (tid % PIECES) * VEC) = reg[i];
  };
  const std::integral_constant<int, AR> ar{};
  const std::integral_constant<int, AC> ac{};
  const std::integral_constant<int, BR> br{};
  const std::integral_constant<int, BC> bc{};
  V ra[NA], rb[NB];
  auto fetch_chunk = [&](int k0) {
    fetch(ar, ac, pa, TA ? p.K : p.M, TA ? p.M : p.K, TA ? k0 : row0, TA ? row0 : k0, ra);
    fetch(br, bc, pb, TB ? p.N : p.K, TB ? p.K : p.N, TB ? col0 : k0, TB ? k0 : col0, rb);
  };
  auto park_chunk = [&](int k0) {
    park(ar, ac, std::integral_constant<bool, TA>{}, TA ? p.K : p.M, TA ? p.M : p.K, TA ? k0 : row0, TA ? row0 : k0, As, std::integral_constant<int, LDA>{}, ra);
    park(br, bc, std::integral_constant<bool, !TB>{}, TB ? p.N : p.K, TB ? p.K : p.N, TB ? col0 : k0, TB ? k0 : col0, Bs, std::integral_constant<int, LDB>{}, rb);
  };

  constexpr int WAVES_N = BN / 32;
  const int wr = (wave / WAVES_N) * 32, wc = (wave % WAVES_N) * 32;
  const bool live = row0 + wr < p.M && col0 + wc < p.N;  // (the same for a whole wavefront)
  typename Tile<T>::Acc acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = typename Tile<T>::Acc{0, 0, 0, 0};

  fetch_chunk(0);
  for (int k0 = 0; k0 < p.K; k0 += KC) {
    if (k0 > 0) __syncthreads();  // everyone has finished with the previous chunk
    park_chunk(k0);
    __syncthreads();
    if (k0 + KC < p.K) fetch_chunk(k0 + KC);  // on its way while this chunk is multiplied
    constexpr int BLOCKS = KC / (4 * VEC);
    auto multiply = [&](int kb) {
      const int k = kb * (4 * VEC) + lk * VEC;
      T av[2][VEC], bv[2][VEC];
      // rows of the tile: fragment i's are wr + 16 i + l16, or (op(a) along its rows) wr + 2 l16 + i
      if constexpr (TA) {
#pragma unroll
        for (int s = 0; s < VEC; ++s) {
          const Pair two = *reinterpret_cast<const Pair *>(As + (k + s) * LDA + wr + 2 * l16);
          av[0][s] = two[0], av[1][s] = two[1];
        }
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const V v = *reinterpret_cast<const V *>(As + (wr + i * 16 + l16) * LDA + k);
#pragma unroll
          for (int s = 0; s < VEC; ++s) av[i][s] = v[s];
        }
      }
      // columns: fragment j's are wc + 2 l16 + j
      if constexpr (TB) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const V v = *reinterpret_cast<const V *>(Bs + (wc + 2 * l16 + j) * LDB + k);
#pragma unroll
          for (int s = 0; s < VEC; ++s) bv[j][s] = v[s];
        }
      } else {
#pragma unroll
        for (int s = 0; s < VEC; ++s) {
          const Pair two = *reinterpret_cast<const Pair *>(Bs + (k + s) * LDB + wc + 2 * l16);
          bv[0][s] = two[0], bv[1][s] = two[1];
        }
      }
#pragma unroll
      for (int s = 0; s < VEC; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = Tile<T>::run(av[i][s], bv[j][s], acc[i][j]);
    };
    const int blocks = live ? (min(KC, p.K - k0) + 4 * VEC - 1) / (4 * VEC) : 0;
    if (blocks == BLOCKS) {  // (unrolled: the next block's LDS reads under this one's products)
#pragma unroll
      for (int kb = 0; kb < BLOCKS; ++kb) multiply(kb);
    } else {
      for (int kb = 0; kb < blocks; ++kb) multiply(kb);
    }
  }

  const int col = col0 + wc + 2 * l16;
  if (!live || col >= p.N) return;
  T *po = out + pair * ((long long)p.M * p.N) + col;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = Tile<T>::row_of(lane, r);
      const int row = row0 + wr + (TA ? 2 * m + i : i * 16 + m);
      if (row >= p.M) continue;
      if (col + 1 < p.N) {
        PairU two;
        two[0] = acc[i][0][r], two[1] = acc[i][1][r];
        *reinterpret_cast<PairU *>(po + (long long)row * p.N) = two;
      } else {
        po[(long long)row * p.N] = acc[i][0][r];
      }
    }
}

// What a stack costs, in microseconds, on each kernel: the chain of a block's trips (`step` for one chunk of
// K, or for 4 values of k of the kernel that reads in place) or the work of the busiest unit (`work` for a
// block's trip), whichever is longer, on top of `base`.  Fitted to 6720 timed pairs of a product (960,
// 2 to 1000 pairs of 16 to 512 rows and columns, both precisions, forward, da and db) and a kernel.
// The one that costs least is 1.7 % slower than the best on average (9 % at the 95th percentile);
// staging every result larger than 32 x 32 in the tile of least area is 9 % slower, 64 x 64 tiles
// where they are half full 18 %.
struct StackRate {
  double step, work, base;
};
constexpr int kTileRows[3] = {32, 64, 128};  // x 128, 64, 32 columns
// [double precision][chunk of 64 values of k, or of 128 bytes][tile]
constexpr StackRate kStaged[2][2][3] = {{{{0.84, 0.74, 2.96}, {0.82, 0.76, 2.95}, {0.90, 0.74, 2.96}}, {{1.42, 1.50, 2.78}, {1.34, 1.40, 2.75}, {1.56, 1.53, 2.74}}},
                                        {{{0.81, 0.69, 2.94}, {0.76, 0.71, 2.87}, {0.92, 0.74, 2.86}}, {{0.06, 3.87, 1.89}, {0.07, 2.84, 2.67}, {0.06, 3.91, 1.95}}}};
// [double precision][forward; op(a) in 16-byte pieces; da; both in pieces; op(a) transposed]
constexpr StackRate kInPlace[2][5] = {{{0.172, 0.087, 2.39}, {0.054, 0.053, 2.76}, {0.129, 0.141, 2.19}, {0.002, 0.051, 2.88}, {0.131, 0.072, 2.61}},
                                      {{0.208, 0.125, 2.38}, {0.134, 0.096, 2.53}, {0.174, 0.167, 2.43}, {0.094, 0.106, 2.43}, {0.186, 0.108, 2.59}}};

double stack_time(const StackRate &r, double trips, double per_unit, double memory) {
  const double a = trips * r.step, b = trips * per_unit * r.work;
  return r.base + std::sqrt(std::sqrt(a * a * a * a + b * b * b * b + memory * memory * memory * memory));
}

template <typename T>
void launch_staged(const BatchedParams &p, int bm, bool deep, unsigned blocks, bool ta, bool tb, const void *a, const void *b, void *out, hipStream_t s) {
#define MG_STAGED_KC(TA, TB, BM, KC) \
  hipLaunchKernelGGL((batched_staged_kernel<T, TA, TB, BM, 4096 / BM, KC>), dim3(blocks), dim3(256), 0, s, p, (const T *)a, (const T *)b, (T *)out)
#define MG_STAGED(TA, TB, BM)                              \
  if (ta == TA && tb == TB && bm == BM) {                  \
    if (deep)                                              \
      MG_STAGED_KC(TA, TB, BM, 64);                        \
    else                                                   \
      MG_STAGED_KC(TA, TB, BM, 128 / (int)sizeof(T));      \
  }
#define MG_STAGED_BM(TA, TB) MG_STAGED(TA, TB, 64) MG_STAGED(TA, TB, 128) MG_STAGED(TA, TB, 32)
  MG_STAGED_BM(false, false)
  MG_STAGED_BM(false, true)
  MG_STAGED_BM(true, false)
  MG_STAGED_BM(true, true)
#undef MG_STAGED_BM
#undef MG_STAGED
#undef MG_STAGED_KC
}

}  // namespace
}  // namespace mg

using namespace mg;

extern "C" {

int mg_matmul_batched(int dtype, int64_t batch, int64_t M, int64_t K, int64_t N, int trans_a, int trans_b, const void *a, const void *b,
                      void *out) {
  std::lock_guard<std::recursive_mutex> guard(api_mutex());
  MG_REQUIRE_INIT();
  if (dtype != MG_F32 && dtype != MG_F64) return fail(MG_ERR_UNSUPPORTED, "mg_matmul_batched: dtype %d (only float32=0 / float64=1)", dtype);
  if (batch < 0 || M < 0 || K < 0 || N < 0)
    return fail(MG_ERR_BAD_ARG, "mg_matmul_batched: batch=%lld M=%lld K=%lld N=%lld", (long long)batch, (long long)M, (long long)K, (long long)N);
  if (batch == 0 || M == 0 || N == 0) return MG_OK;
  if (M >= (1 << 24) || K >= (1 << 24) || N >= (1 << 24) || batch >= (1ll << 31))
    return fail(MG_ERR_UNSUPPORTED, "mg_matmul_batched: an extent of 2^24 or more, or 2^31 pairs or more");
  if (!out || (K > 0 && (!a || !b))) return fail(MG_ERR_BAD_ARG, "null pointer in mg_matmul_batched");
  BatchedParams p{};
  p.M = (int)M, p.K = (int)K, p.N = (int)N;
  p.row_tiles = (int)ceil_div(M, 16);
  p.col_tiles = (int)ceil_div(N, 16);
  p.tiles = batch * p.row_tiles * p.col_tiles;
  if (ceil_div(p.tiles, 4) >= (1ll << 31)) return fail(MG_ERR_UNSUPPORTED, "mg_matmul_batched: 2^33 tiles of 16 x 16 results or more");
  p.a_pair = M * K, p.b_pair = K * N;
  p.a_row = trans_a ? 1 : K, p.a_col = trans_a ? M : 1;  // a[p] is stored (K, M) when transposed
  p.b_row = trans_b ? 1 : N, p.b_col = trans_b ? K : 1;  // b[p] is stored (N, K) when transposed
  hipStream_t s = runtime().stream;
  ScopedTiming timed(TAG_BATCHED_PRODUCT);
  // MYGRAD_HIP_BMM_STAGED=0 keeps every pair on the kernel that reads its operands in place.
  static const bool staged_on = [] {
    const char *flag = getenv("MYGRAD_HIP_BMM_STAGED");
    return !(flag && flag[0] == '0');
  }();
  // 16-byte pieces along K: the operand is contiguous there, K is a whole number of pieces (so
  // every row starts on one) and the stack itself is aligned
  const bool f64 = dtype == MG_F64;
  const int vec = f64 ? 2 : 4;
  const bool av = p.a_col == 1 && K % vec == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0;
  const bool bv = p.b_row == 1 && K % vec == 0 && reinterpret_cast<uintptr_t>(b) % 16 == 0;
  // Results of 16 rows or columns at most stay in place.  Of the others those whose 64 x 64 tiles are half
  // full leave it to an operand without pieces: what its strided reads cost depends on more than is fitted
  // here (16 x (197,64,197), db in double precision: 20.7 us in place, 14.1 staged, 11.9 expected).
  const double cus = runtime().props.multiProcessorCount;
  const double memory = (double)batch * (double)(M * K + K * N + M * N) * (f64 ? 8.0 : 4.0) / 6.0e6;
  int tile = -1, deep = 0;
  if (staged_on && K > 0 && M > 16 && N > 16) {
    const StackRate &in_place = kInPlace[f64][trans_a ? 4 : trans_b ? (av && bv ? 3 : 2) : av ? 1 : 0];
    double least = stack_time(in_place, (double)ceil_div(K, 4), std::ceil((double)ceil_div(p.tiles, 4) / cus), memory);
    const bool half_full = M >= 32 && N >= 32 && 2 * M * N >= ceil_div(M, 64) * ceil_div(N, 64) * 4096;
    if (half_full && !av && !bv) least = 1e30;
    for (int d = 0; d < 2; ++d)
      for (int t = 0; t < 3; ++t) {
        const double blocks = (double)batch * (double)ceil_div(M, kTileRows[t]) * (double)ceil_div(N, 4096 / kTileRows[t]);
        const double time = stack_time(kStaged[f64][d][t], (double)ceil_div(K, d ? 64 : 128 / (f64 ? 8 : 4)), std::max(blocks / cus, 1.0), memory);
        if (time < least) least = time, tile = t, deep = d;
      }
    // MYGRAD_HIP_BMM_TILE="rows,deep" (read at every call, for the tests of every tile): that one
    int rows = 0, chunk = 0;
    if (const char *v = getenv("MYGRAD_HIP_BMM_TILE"))
      if (sscanf(v, "%d,%d", &rows, &chunk) == 2)
        for (int t = 0; t < 3; ++t)
          if (kTileRows[t] == rows) tile = t, deep = chunk != 0;
  }
  static const char *const notes[3][2] = {{"batched: 32 x 128 tiles, short chunks", "batched: 32 x 128 tiles, deep chunks"},
                                          {"batched: 64 x 64 tiles, short chunks", "batched: 64 x 64 tiles, deep chunks"},
                                          {"batched: 128 x 32 tiles, short chunks", "batched: 128 x 32 tiles, deep chunks"}};
  note_plan(tile < 0 ? "batched: operands read in place" : notes[tile][deep]);
  const int bm = tile < 0 ? 64 : kTileRows[tile];
  const long long tiles = batch * ceil_div(M, bm) * ceil_div(N, 4096 / bm);
  // (dealing pairs out to the XCDs pays where each has many: with 100 pairs of five tiles some units get a
  // third block, 25 -> 37 us)
  p.dealt = batch >= 64 && tiles >= 8 * cus;
  // A launch has fewer than 2^32 threads along x, which is 2^24 - 1 blocks: a longer stack goes in runs of pairs.
  const long long most = (1ll << 24) - 1, per_pair = tile < 0 ? (long long)p.row_tiles * p.col_tiles : tiles / batch;
  long long at_once = (tile < 0 ? 4 * most : most) / per_pair;
  if (at_once < 1) return fail(MG_ERR_UNSUPPORTED, "mg_matmul_batched: a product of 2^24 tiles or more");
  if (at_once < 8) p.dealt = 0;
  if (p.dealt) at_once = at_once / 8 * 8;
  const size_t elem = f64 ? 8 : 4;
  for (long long first = 0; first < batch; first += at_once) {
    const long long count = std::min(at_once, batch - first);
    const void *pa = static_cast<const char *>(a) + first * p.a_pair * elem, *pb = static_cast<const char *>(b) + first * p.b_pair * elem;
    void *po = static_cast<char *>(out) + first * M * N * elem;
    p.pairs = (int)count;
    p.tiles = count * per_pair;
    if (tile >= 0) {
      p.row_tiles = (int)ceil_div(M, bm);
      p.col_tiles = (int)ceil_div(N, 4096 / bm);
      const unsigned blocks = (unsigned)(p.dealt ? ceil_div(count, 8) * 8 * per_pair : p.tiles);
      if (f64)
        launch_staged<double>(p, bm, deep != 0, blocks, trans_a != 0, trans_b != 0, pa, pb, po, s);
      else
        launch_staged<float>(p, bm, deep != 0, blocks, trans_a != 0, trans_b != 0, pa, pb, po, s);
      continue;
    }
    const dim3 grid((unsigned)ceil_div(p.tiles, 4)), block(256);
#define MG_BATCHED(T, AV, BV) \
  hipLaunchKernelGGL((batched_product_kernel<T, AV, BV>), grid, block, 0, s, p, (const T *)pa, (const T *)pb, (T *)po)
#define MG_BATCHED_T(T)                 \
  do {                                  \
    if (av && bv) MG_BATCHED(T, true, true);        \
    else if (av) MG_BATCHED(T, true, false);        \
    else if (bv) MG_BATCHED(T, false, true);        \
    else MG_BATCHED(T, false, false);               \
  } while (0)
    if (f64) MG_BATCHED_T(double); else MG_BATCHED_T(float);
#undef MG_BATCHED_T
#undef MG_BATCHED
  }
  MG_HIP(hipGetLastError());
  return MG_OK;
}

}  // extern "C"
