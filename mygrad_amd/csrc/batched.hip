// Products of many small matrix pairs in one launch: out[p] = op(a[p]) @ op(b[p]), p < batch,
// where op transposes or not.  A pair of stacks whose matrices are too small to fill the device
// one pair at a time (np.matmul on two stacks, an einsum with a label that both operands and
// the result carry) is bound by launches, not arithmetic, when each pair gets a launch of the
// convolution kernels; here a wavefront makes one 16x16 tile of one product on the matrix cores,
// reading its operands where they lie (a transposed operand is a pair of swapped strides), so the
// whole stack is one grid.  Results larger than 32 x 32 go through a second kernel, where a
// block of four wavefronts makes a tile of one product from operands it has copied to
// LDS once (16 bytes per lane, coalesced) instead of every wavefront fetching its own rows and
// columns through L1.  Large pairs stay with the tiled convolution kernels.
#include "internal.h"

#include <algorithm>
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
// the loads of the next chunk are issued before this one is multiplied, chunks are short (128 bytes
// of k: six or seven blocks on a unit cover for one another; 256 bytes: 794 x (86,117,322) 117 us
// instead of 103), and the LDS reads are wide.  Measured, single precision, forward / da / db: 96 x
// (197,64,197) 14.1 / 13.8 / 13.7 us (34 TFLOP/s; 19.9 / 17.3 / 20.4 with element loads and
// element LDS reads, which rows that are no whole pieces and every row took before), 794 x
// (86,117,322) 103 / 91 / 104 us (147 / 130 / 139), 8 x 512^3 29 / 28 / 30 us.
// The sum over k may run in any order that both operands share: in a block of 4 * VEC values of k
// (VEC = 16 bytes) the lane groups (lane / 16 = q) take k = VEC * q + s at step s, so an operand
// that lies along k gives a lane VEC steps per LDS read; of one that lies along its rows or columns
// a lane takes two neighbours, the two MFMA fragments it feeds, per read.
template <typename T, bool TA, bool TB, int BM, int BN>
__global__ void __launch_bounds__(256) batched_staged_kernel(BatchedParams p, const T *__restrict__ a, const T *__restrict__ b,
                                                             T *__restrict__ out) {
  constexpr int VEC = 16 / sizeof(T);
  typedef T V __attribute__((ext_vector_type(VEC)));
  typedef T VU __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
  typedef T Pair __attribute__((ext_vector_type(2)));
  typedef T PairU __attribute__((ext_vector_type(2), aligned(sizeof(T))));
  static_assert((BM / 32) * (BN / 32) == 4, "four wavefronts of 32 x 32");
  constexpr int KC = 128 / sizeof(T);  // depth of a chunk
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
  // (zeros outside the matrix) into LDS; the loads of both operands are issued before either is
  // parked, so that a chunk costs one trip to memory, not two
  auto fetch = [&](auto rc, auto cc, const T *src, int rows, int cols, int r0, int c0, auto &reg) {
    constexpr int R = decltype(rc)::value, C = decltype(cc)::value, PIECES = C / VEC, PASS = 256 / PIECES;
    const int c = c0 + (tid % PIECES) * VEC;
    const T *at = src + (long long)(r0 + tid / PIECES) * cols + c;
#pragma unroll
    for (int i = 0; i < R / PASS; ++i) {
      reg[i] = V{};
      if (r0 + tid / PIECES + i * PASS < rows) {
        const T *piece = at + (long long)(i * PASS) * cols;
        if (c + VEC <= cols) {
          reg[i] = *reinterpret_cast<const VU *>(piece);
        } else {
#pragma unroll
          for (int s = 0; s < VEC - 1; ++s)
            if (c + s < cols) reg[i][s] = piece[s];
        }
      }
    }
  };
  auto park = [&](auto rc, auto cc, T *dst, auto ld, const auto &reg) {
    constexpr int R = decltype(rc)::value, C = decltype(cc)::value, PIECES = C / VEC, PASS = 256 / PIECES;
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
    park(ar, ac, As, std::integral_constant<int, LDA>{}, ra);
    park(br, bc, Bs, std::integral_constant<int, LDB>{}, rb);
    __syncthreads();
    if (k0 + KC < p.K) fetch_chunk(k0 + KC);  // on its way while this chunk is multiplied
    const int blocks = live ? (min(KC, p.K - k0) + 4 * VEC - 1) / (4 * VEC) : 0;
    for (int kb = 0; kb < blocks; ++kb) {
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

// Rows of the tile: of 128 x 32, 64 x 64 and 32 x 128, all four wavefronts of 32 x 32, the one that covers
// M x N with the least area (the squarer one where they come out the same: it loads less).
inline int staged_rows(int64_t M, int64_t N) {
  int best = 64;
  int64_t least = ceil_div(M, 64) * ceil_div(N, 64);
  for (int bm : {128, 32})
    if (ceil_div(M, bm) * ceil_div(N, 4096 / bm) < least) best = bm, least = ceil_div(M, bm) * ceil_div(N, 4096 / bm);
  return best;
}

template <typename T>
void launch_staged(const BatchedParams &p, int bm, unsigned blocks, bool ta, bool tb, const void *a, const void *b, void *out, hipStream_t s) {
#define MG_STAGED(TA, TB, BM)                    \
  if (ta == TA && tb == TB && bm == BM)          \
    hipLaunchKernelGGL((batched_staged_kernel<T, TA, TB, BM, 4096 / BM>), dim3(blocks), dim3(256), 0, s, p, (const T *)a, (const T *)b, (T *)out);
#define MG_STAGED_BM(TA, TB) MG_STAGED(TA, TB, 64) MG_STAGED(TA, TB, 128) MG_STAGED(TA, TB, 32)
  MG_STAGED_BM(false, false)
  MG_STAGED_BM(false, true)
  MG_STAGED_BM(true, false)
  MG_STAGED_BM(true, true)
#undef MG_STAGED_BM
#undef MG_STAGED
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
  const int bm = staged_rows(M, N);
  p.dealt = batch >= 64;
  const long long blocks = (p.dealt ? ceil_div(batch, 8) * 8 : batch) * ceil_div(M, bm) * ceil_div(N, 4096 / bm);
  p.pairs = (int)batch;
  // A result of one wavefront's 32 x 32 or of 16 rows or columns stays with the kernel above (300 x
  // (20,100,20): 5.6 us there, 8.0 staged).  In double precision, whose 16x16x4 MFMA takes three
  // times as long, 32 x 32 parts that are less than 0.6 full lose too (64 x (300,400,18): 48 / 57 us;
  // 34 x (310,259,31): 31 / 21) unless 64 x 64 tiles are half full.
  const long long parts = ceil_div(M, 32) * ceil_div(N, 32) * 1024, t64 = ceil_div(M, 64) * ceil_div(N, 64) * 4096;
  const bool full = dtype == MG_F32 || 10 * M * N >= 6 * parts || (M >= 32 && N >= 32 && 2 * M * N >= t64);
  if (staged_on && K > 0 && M > 16 && N > 16 && (M > 32 || N > 32) && full && blocks < (1ll << 31)) {
    p.row_tiles = (int)ceil_div(M, bm);
    p.col_tiles = (int)ceil_div(N, 4096 / bm);
    if (dtype == MG_F32)
      launch_staged<float>(p, bm, (unsigned)blocks, trans_a != 0, trans_b != 0, a, b, out, s);
    else
      launch_staged<double>(p, bm, (unsigned)blocks, trans_a != 0, trans_b != 0, a, b, out, s);
    MG_HIP(hipGetLastError());
    return MG_OK;
  }
  const dim3 grid((unsigned)ceil_div(p.tiles, 4)), block(256);
  // 16-byte pieces along K: the operand is contiguous there, K is a whole number of pieces (so
  // every row starts on one) and the stack itself is aligned
  const int vec = dtype == MG_F32 ? 4 : 2;
  const bool av = p.a_col == 1 && K % vec == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0;
  const bool bv = p.b_row == 1 && K % vec == 0 && reinterpret_cast<uintptr_t>(b) % 16 == 0;
#define MG_BATCHED(T, AV, BV) \
  hipLaunchKernelGGL((batched_product_kernel<T, AV, BV>), grid, block, 0, s, p, (const T *)a, (const T *)b, (T *)out)
#define MG_BATCHED_T(T)                 \
  do {                                  \
    if (av && bv) MG_BATCHED(T, true, true);        \
    else if (av) MG_BATCHED(T, true, false);        \
    else if (bv) MG_BATCHED(T, false, true);        \
    else MG_BATCHED(T, false, false);               \
  } while (0)
  if (dtype == MG_F32) MG_BATCHED_T(float); else MG_BATCHED_T(double);
#undef MG_BATCHED_T
#undef MG_BATCHED
  MG_HIP(hipGetLastError());
  return MG_OK;
}

}  // extern "C"
