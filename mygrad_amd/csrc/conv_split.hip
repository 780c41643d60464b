// Gather-GEMM in single precision on the bf16 matrix instructions, for the forward pass and the
// data gradient of large problems.
//
// v_mfma_f32_16x16x4_f32 does 157 TFLOP/s at best on this device and shares its issue with the vector
// ALU (44 vector instructions next to 16 of them: 154 -> 110 TFLOP/s); v_mfma_f32_16x16x32_bf16 does
// 1800 - 2000 and does not.  A float is the sum of three bf16 numbers (8 + 8 + 8 bits of its significand;
// below 2^-110 see "what the split cannot represent"), x = x0 + x1 + x2, and
//   x * w = x0 w0 + (x0 w1 + x1 w0) + (x0 w2 + x1 w1 + x2 w0) + at most 2^-24 |x w|,
// six products, each exact in single precision: an effective peak of 300 - 330 TFLOP/s.
//
// Precision.  The large product and the five small ones have an accumulator each, added at the end.  An
// accumulator rounds once per 32 terms of a product, whatever the terms are, and loses some bits of what it
// adds; in one accumulator for all six that made sums of few terms less accurate than the single-precision
// instruction, which rounds only where a term is not zero.  Error against 64 bits (2-norm), (128,64,56,56) *
// (64,64,3,3), one accumulator / two / single precision:
//   normal values                    3.5e-7 / 1.4e-7 / 4.2e-7
//   behind a relu                    3.4e-7 / 1.2e-7 / 3.0e-7
//   one element in 100 not zero      9.8e-8 / 3.7e-8 / 4.9e-8
//   one product a sum                4.2e-8 / 2.6e-8 / 2.5e-8
// (In the last row what the six products leave out shows: no result is off by more than 2^-23 of itself, where
// one rounding is 2^-24.)  Two accumulators of 64 x 64 wave tiles do not fit 256 registers (70 - 85 of them
// spill: 186 us below become 246), those of 64 x 48 do but for a dozen values that no step needs.
//
// What bounds it: (128,64,56,56) * (64,64,3,3), 29.6 GFLOP, takes 178 - 194 us with its packing and the pass
// over marked tiles on most devices (single precision 232), 164 - 166 by itself, 180 TFLOP/s of the 300; 194 by
// itself on one where the filter gradient takes 280 us instead of 233.  Matrix pipes are busy 43 % of the
// cycles, LDS 38 % (64 x 48 and 48 x 64 waves: 21 reads of 16 bytes a lane for 72 matrix instructions; 32 x 64
// ones 18 for 48: 201 us for 186), the waves wait for 37 % of theirs: the turn between stages, where a block's
// waves wait for the patch to be split and parked; loads are hidden.  Smaller planes have smaller patches:
// (128,128,28,28) * (128,128,3,3), 29.6 GFLOP, 230 -> 161 us; (16,96,16001) * (48,96,9), 21.2 GFLOP, 172 -> 130.
//
// What the split cannot represent.  An infinite operand leaves Inf - Inf in its second part and makes every sum
// that it takes part in a NaN, as an infinite or NaN operand or an overflow makes it something not finite in
// any arithmetic.  And parts are multiples of 2^-133, the smallest number of bf16 (which the instruction takes
// as it is, like every product and sum below 2^-126): of an operand below 2^-110 bits may be lost, below 2^-134
// all of them.  K such losses times the largest value of the other operand are less than the last bit of a sum
// of K * 2^-109 times that value.  So where a block has a sum that is not finite, or has lost bits of an
// element or seen a filter value below 2^-109 and has a sum, zero included, below that bound, it marks its
// tile, and split_redo_kernel computes marked tiles again on the single-precision instruction.  The bits of
// other tiles do not depend on it, and few marked tiles cost little: the forward pass below 194 us as it is,
// 205 with one NaN, 252 with one sample in 20 of values about 1e-38, 811 where every tile is marked (single
// precision 232).  (The whole pass on the single-precision kernels, three launches that returned at once
// otherwise, took 381 for the first odd value and 9 more for none.)
#include "conv_device.h"
#include "conv_kernels.h"
#include "internal.h"
#include "split_device.h"

#include <algorithm>
#include <array>
#include <map>
#include <type_traits>

namespace mg {

namespace {

typedef int int16v __attribute__((ext_vector_type(16)));
static_assert(sizeof(KTile) == sizeof(int8v) && sizeof(SplitPhase) == sizeof(int16v), "table rows");

// What a block finds out about an item's operands and sums, bit by bit.
enum : unsigned { kNotFinite = 1, kLostElement = 2, kTinyFilter = 4, kLostSum = 8 };
constexpr unsigned short kTinyBits = 18 << 7;  // 2^-109 in bf16

// the element of dst at position ipos of the phase, row 0
__device__ __forceinline__ float *dst_of(const GemmParams &p, const Phase &ph, int ipos) {
  const int j12 = ph.J[1] * ph.J[2];
  const unsigned n = ph.by_jvol.div((unsigned)ipos);
  unsigned r = (unsigned)ipos - n * (unsigned)(ph.J[0] * j12);
  const int j0 = (int)ph.by_j12.div(r);
  r -= (unsigned)j0 * (unsigned)j12;
  const int j1 = (int)ph.by_j2.div(r);
  const int j2 = (int)r - j1 * ph.J[2];
  return static_cast<float *>(p.dst) + (long long)n * p.dst_nstride + (long long)(ph.o0[0] + j0 * p.oj[0]) * p.os[0] +
         (long long)(ph.o0[1] + j1 * p.oj[1]) * p.os[1] + (long long)(ph.o0[2] + j2 * p.oj[2]) * p.os[2];
}

// One tile is MW * WM rows (filters) by NW * 16 TN positions, a wave of the block for each WM x 16 TN of it.  The contraction
// runs in stages: 16 channels under the taps of one inner window (all taps, or those of the last axes where the
// others reach too far).  A stage's elements of src -- every row (position of src) that the tile's windows touch, 16
// channels of each -- are loaded and split once, parked in LDS, and serve all taps of the window from there: operand
// position n under tap t is row base(n) + offset(t), 16 bytes a lane.  (Split anew for every tap, as the waves
// gather them for the single-precision instruction, the vector ALU and the vector cache are the bound: 64 channels, 3x3, 56x56
// 180 us.)  A position without the tap (padding) reads a row of zeros.
//
// A K step is 32 deep: two taps, lanes 0 - 31 hold the first one's 16 channels, lanes 32 - 63 the second one's.  An
// odd last tap (ODD) makes a step of four products instead of six: lanes 0 - 31 and 32 - 63 hold different parts of the one tap, and
// nothing beside x0 w0.
//
// The positions are the rows of D, so that a lane holds four consecutive positions of one filter and stores them as a vector.  The filters,
// split and laid out in the order of the stages beforehand (split_pack_kernel), pass through LDS two steps ahead of their use.
// Blocks are persistent, as in tap_gemm_kernel.
template <int WM, int MW, int TN, int NW, int ROUNDS, bool ODD>
__global__ void __launch_bounds__(64 * MW * NW, WM == 16 ? 3 : 2) split_gemm_kernel(const GemmParams p) {
  constexpr int BM = WM * MW, WN = 16 * TN, BN = WN * NW, TM = WM / 16, THREADS = 64 * MW * NW;
  static_assert(WM % 16 == 0, "16 x 16 tiles");
  constexpr int PIECES = 12 * BM;  // of 16 bytes: a step's filters, [part][octet of K rows][row]
  constexpr int ALOADS = (PIECES + THREADS - 1) / THREADS;
  // [2][PIECES] filters, then the patch: [octet of channels][row][part], p.patch_rows + 1 rows, the last one
  // zeros; and three words (note)
  extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
  u32x4 *const patch = lds + 2 * PIECES;

  const int lane = threadIdx.x & 63;
  const int wave = uniform((threadIdx.x >> 6) % NW), wm0 = uniform((threadIdx.x >> 6) / NW) * WM;  // the wave's positions and rows
  const int l16 = lane & 15, lk = lane >> 4;
  const bool second = lk >= 2;  // this lane holds channels under the second tap of a step

  struct Item {
    int tile, pos0, m0, kt_begin, kt_end, slot;
    bool partial;
    Phase ph;
  };
  // of the item, this lane's: bits lost of the elements that it has split, the smallest |filter value| that it
  // has parked, less one (zeros aside)
  unsigned lost = 0;
  u16x2 tiniest = {0xffff, 0xffff};
  // The walk over items is tap_gemm_kernel's.  (Shared by the two in a struct it changes that kernel's allocation of
  // scalar registers: a 4096 x 4096 x 4096 product and its gradients 2931 -> 2943 us, where two runs differ by 0.3 %.)
  const bool shares = p.share_first != nullptr;
  const int share_begin = shares ? ((const int MG_CONSTANT *)p.share_first)[uniform((int)blockIdx.x)] : 0;
  const int share_end = shares ? ((const int MG_CONSTANT *)p.share_first)[uniform((int)blockIdx.x) + 1] : 0;
  const int item_end = shares ? p.full_tiles + share_end : p.items;
  const int chunk = p.xcd_chunk;
  const int place = chunk > 1 ? (((int)blockIdx.x >> 3) / chunk * 8 + ((int)blockIdx.x & 7)) * chunk + ((int)blockIdx.x >> 3) % chunk
                              : (int)blockIdx.x;
  const int item_first = (!shares || place < p.full_tiles) ? place : p.full_tiles + share_begin;
  auto next_item = [&](int item) -> int {
    if (!shares) return item + (int)gridDim.x;
    if (item >= p.full_tiles) return item + 1;
    return item + (int)gridDim.x < p.full_tiles ? item + (int)gridDim.x : p.full_tiles + share_begin;
  };
  auto locate = [&](int item, int &pi, Item &it) {  // pi: phase of the previous item of this cursor (tiles ascend)
    it.tile = item;
    it.slot = 0;
    it.partial = item >= p.full_tiles;
    int4v row = {0, 0, 0, 0};
    int piece = 0;
    if (it.partial) {
      if (shares) {
        row = ((const int4v MG_CONSTANT *)p.share_slices)[uniform(item - p.full_tiles)];
        it.tile = row[0];
        it.slot = row[3];
        it.partial = row[3] >= 0;
      } else {
        const int j = item - p.full_tiles;
        it.tile = p.full_tiles + j / p.tail_split;
        piece = j % p.tail_split;
        it.slot = j;
      }
    }
    const int pblk = it.tile / p.m_tiles;
    while (pi + 1 < p.nphases && pblk >= phase_first_block(p.phases, pi + 1)) ++pi;
    it.ph = load_phase(p.phases, pi);
    it.pos0 = (pblk - it.ph.blk_begin) * BN;
    it.m0 = (it.tile % p.m_tiles) * BM;
    it.kt_begin = 0;
    it.kt_end = it.ph.k_count;
    if (shares && item >= p.full_tiles) {
      it.kt_begin = row[1];
      it.kt_end = row[2];
    } else if (it.partial) {
      const int per = (it.ph.k_count + p.tail_split - 1) / p.tail_split;
      it.kt_begin = min(piece * per, it.ph.k_count);
      it.kt_end = min(it.kt_begin + per, it.ph.k_count);
    }
  };

  const __amdgpu_buffer_rsrc_t a_buf = buffer_of(p.A, p.a_bytes);
  const __amdgpu_buffer_rsrc_t src_buf = buffer_of(p.src, p.src_bytes);
  const __amdgpu_buffer_rsrc_t table_buf = buffer_of(p.positions, (unsigned)p.npos * 8u);  // (row, taps) of every position
  const unsigned piece_row = (unsigned)p.a_ld * 16u;  // bytes of one part of one octet of packed filters
  const unsigned c_step = (unsigned)p.src_cstride * 4u;
  const int octet_rows = p.patch_rows + 1;
  // what was found, the widest filter value, the widest element
  unsigned *const note = reinterpret_cast<unsigned *>(patch + 2 * octet_rows * 3);
  if (threadIdx.x < 6) patch[((int)threadIdx.x / 3 * octet_rows + p.patch_rows) * 3 + (int)threadIdx.x % 3] = u32x4{0, 0, 0, 0};
  int pi = 0;
  Item me;
  u32x4 raw[ROUNDS][4];  // elements on their way to the patch: [round][channel][row of four]
  bool ahead = false;    // those of the item's first stage were requested by the item before it
  // the patch being requested: its first row, its stage's row of the table, whether there is one
  int patch_row = 0;
  int8v patch_e = {0, 0, 0, 0, 0, 0, 0, 0};  // first half, channel offset, row offset, first tap, first channel, dead rows
  bool patch_real = false;
  auto first_of = [&](const Item &it) -> int { return ((const int MG_CONSTANT *)p.split_tiles)[uniform(it.pos0 / BN)]; };
  // A part of the patch's loads.  A thread takes four rows of four channels in each round; the rows begin on a
  // multiple of four and therefore lie in one sample (a sample's rows are numbered up to a multiple of four;
  // what is loaded for those beyond its last is of no use to anyone), and are loaded as one vector, whatever
  // its alignment: 16 bytes a lane take the vector cache 16 cycles, 4 bytes 8 - 11.
  const int quads = p.patch_rows / 4;
  auto quarter_of = [&](int idx) -> int { return (idx >= quads) + (idx >= 2 * quads) + (idx >= 3 * quads); };  // of the stage's channels
  auto request_part = [&](int k) {
    constexpr int CHANNELS = ROUNDS;  // a part is a round's four channels, a quarter or a half of them at a time
    const int round = k * ROUNDS / 4;
    if (round * THREADS >= p.patch_rows) return;
    const int idx = (int)threadIdx.x + round * THREADS, quarter = quarter_of(idx);
    const int row = ((patch_row + patch_e[2]) & ~3) + (idx - quarter * quads) * 4;
    const unsigned n = __umulhi((unsigned)max(row, 0), p.by_sample.mul) >> p.by_sample.shr;  // (more than one row to a sample)
    unsigned at = (n * (unsigned)p.src_nstride + (unsigned)(row - (int)n * p.sample_rows + patch_e[1] + quarter * 4 * p.src_cstride)) * 4u;
    at = ((idx < p.patch_rows) & (row >= 0) & ((int)n < p.samples) & patch_real) ? at : kOutside;
    const unsigned dead = (unsigned)patch_e[5] >> (quarter * 4);
#pragma unroll
    for (int u = 0; u < CHANNELS; ++u) {
      const int r = k * CHANNELS % 4 + u;
      const unsigned lane_at = at | ((dead << (31 - r)) & kOutside);
      raw[round][r] = __builtin_amdgcn_raw_buffer_load_b128(src_buf, (int)lane_at, (int)((unsigned)r * c_step), 0);
    }
  };
  auto park_patch = [&] {
#pragma unroll
    for (int round = 0; round < ROUNDS; ++round) {
      if (round * THREADS >= p.patch_rows) break;
      const int idx = (int)threadIdx.x + round * THREADS, quarter = quarter_of(idx);
      u32x2 *const out = reinterpret_cast<u32x2 *>(patch + (quarter / 2 * octet_rows + (idx - quarter * quads) * 4) * 3) + quarter % 2;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = float_of(raw[round][r][u]);
        unsigned parts[3][2];
        split_pair(v[0], v[1], parts[0][0], parts[1][0], parts[2][0], lost);
        split_pair(v[2], v[3], parts[0][1], parts[1][1], parts[2][1], lost);
        if (idx < p.patch_rows) {
#pragma unroll
          for (int part = 0; part < 3; ++part) out[(u * 3 + part) * 2] = u32x2{parts[part][0], parts[part][1]};
        }
      }
    }
  };
  for (int item = item_first; item < item_end; item = next_item(item)) {
    locate(item, pi, me);
    f32x4 acc[TN][TM], low[TN][TM];  // sums of x0 w0 and of the five small products
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] = low[j][i] = f32x4{0, 0, 0, 0};
    const int stages = me.kt_end - me.kt_begin;
    const int16v sp = ((const int16v MG_CONSTANT *)p.split_phases)[uniform(pi)];  // see SplitPhase
    const int window = sp[9];  // taps of the inner window
    const int inner = p.split_inner[sp[10] + min(lane, window - 1)];  // lane t: row offset of the window's tap t

    // ---- this lane's positions: their row in the patch and the taps they have (bit by bit; none beyond the
    // last position)
    const int first_row = first_of(me);
    int row_at[TN];
    unsigned taps[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      typedef int int2v __attribute__((ext_vector_type(2)));
      const int ipos = me.pos0 + wave * WN + j * 16 + l16;
      const int2v at = __builtin_bit_cast(int2v, __builtin_amdgcn_raw_buffer_load_b64(table_buf, (int)((unsigned)ipos * 8u), 0, 0));
      row_at[j] = at[0] - first_row;
      taps[j] = (unsigned)at[1];
    }
    unsigned a_at[ALOADS];
#pragma unroll
    for (int u = 0; u < ALOADS; ++u) {
      const int q = (int)threadIdx.x + THREADS * u;
      const int m = me.m0 + q % BM, oct = q / BM % 4, part = q / (4 * BM);
      a_at[u] = q < PIECES && m < p.a_ld ? (unsigned)(oct * 3 + part) * piece_row + (unsigned)m * 16u : kOutside;
    }

    // ---- filters: `half` counts taps of 16 channels in the order of the stages
    u32x4 areg[ALOADS];
    auto request_filters = [&](int half) {
      const unsigned at = (unsigned)half * 6u * piece_row;
#pragma unroll
      for (int u = 0; u < ALOADS; ++u) areg[u] = __builtin_amdgcn_raw_buffer_load_b128(a_buf, (int)(a_at[u] + at), 0, 0);
    };
    auto park_filters = [&](int buf) {
#pragma unroll
      for (int u = 0; u < ALOADS; ++u) {
        const int q = (int)threadIdx.x + THREADS * u;
        if (PIECES % THREADS == 0 || q < PIECES) lds[buf * PIECES + q] = areg[u];
      }
      static_assert(4 * BM <= THREADS, "first parts: the first piece of a thread");
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const u16x2 size = __builtin_bit_cast(u16x2, areg[0][e] & 0x7fff7fffu);
        tiniest = __builtin_elementwise_min(tiniest, (u16x2)(size - u16x2{1, 1}));
      }
    };
    bf16x8 w[TM][3];
    auto read_filters = [&](int buf, int i, bool single) {
      // (a single tap: parts 0 | 2 and 1 | 0 of its two octets)
      const u32x4 *mine = lds + buf * PIECES + (single ? lk & 1 : lk) * BM + wm0 + l16 + i * 16;
      if (single) {
        w[i][0] = __builtin_bit_cast(bf16x8, mine[(second ? 2 : 0) * 4 * BM]);
        w[i][1] = __builtin_bit_cast(bf16x8, mine[(second ? 0 : 1) * 4 * BM]);
      } else {
#pragma unroll
        for (int part = 0; part < 3; ++part) w[i][part] = __builtin_bit_cast(bf16x8, mine[part * 4 * BM]);
      }
    };

    // ---- the patch
    const int8v MG_CONSTANT *table = (const int8v MG_CONSTANT *)p.ktiles + (me.ph.k_begin + me.kt_begin);
    // what the steps of stage `stage` request: the next stage's patch, or the first one of the block's next item
    auto aim = [&](int stage) {
      patch_row = first_row;
      patch_real = stage + 1 < stages;
      if (patch_real) {
        patch_e = table[stage + 1];
      } else {
        const int then = next_item(item);
        if (then < item_end) {
          Item nx;
          int npi = pi;
          locate(then, npi, nx);
          if (nx.kt_begin < nx.kt_end) {
            patch_row = first_of(nx);
            patch_e = ((const int8v MG_CONSTANT *)p.ktiles)[uniform(nx.ph.k_begin + nx.kt_begin)];
            patch_real = true;
          }
        }
      }
    };
    int x_at[TN], x_next[TN];  // of the step under way and the one after it: 16-byte pieces from the start of the patch
    // tap0: number of the window's first tap; q: first tap of the step within it; lead: rows of the patch ahead
    // of the tile's first one
    auto place = [&](int tap0, int q, bool single, int lead) {
      const int off0 = __builtin_amdgcn_readlane(inner, q), off1 = __builtin_amdgcn_readlane(inner, single ? q : q + 1);
      const int off = (second ? off1 : off0) + lead;
      const unsigned tap = (unsigned)(tap0 + q + (!single && second ? 1 : 0));
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int keep = __builtin_amdgcn_sbfe((int)taps[j], tap, 1u);  // all ones where the position has the tap
        x_next[j] = (((row_at[j] + off - p.patch_rows) & keep) + p.patch_rows + (lk & 1) * octet_rows) * 3;
      }
    };
    auto enter_step = [&] {
#pragma unroll
      for (int j = 0; j < TN; ++j) x_at[j] = x_next[j];
    };
    auto read_position = [&](int j, bool single, bf16x8(&x)[3]) {
      const u32x4 *mine = patch + x_at[j];
      if (single) {  // parts 2 | 0, 1 | 1, 0 | nothing
        x[0] = __builtin_bit_cast(bf16x8, mine[second ? 0 : 2]);
        x[1] = __builtin_bit_cast(bf16x8, mine[1]);
        x[2] = __builtin_bit_cast(bf16x8, *(second ? patch + p.patch_rows * 3 : mine));
      } else {
#pragma unroll
        for (int part = 0; part < 3; ++part) x[part] = __builtin_bit_cast(bf16x8, mine[part]);
      }
    };

    // One K step (`step_no` of the item) whose operands' first position is in x[0] and whose filters are in w;
    // the next step starts at tap `q_next` of its window, `single_next`: it is a window's odd last tap.
    // `turn`: the stage ends here.
    bf16x8 x[2][3];
    int step_no = 0;
    auto step = [&](auto single_c, auto turn_c, auto single_next_c, int half_after, int tap0_next, int q_next, int lead_next,
                    int stage, int parts) {
      constexpr bool SINGLE = decltype(single_c)::value, TURN = decltype(turn_c)::value, NEXT = decltype(single_next_c)::value;
      // smallest first; x0 w0 alone into the sum of large products, for a sum of a few of those is exact
      constexpr int PRODUCTS = SINGLE ? 4 : 6;
      constexpr int PX[6] = {SINGLE ? 0 : 2, SINGLE ? 1 : 0, SINGLE ? 2 : 1, SINGLE ? 2 : 1, 0, 0}, PW[6] = {0, SINGLE ? 1 : 2, 1, 0, 1, 0};
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (j + 1 < TN) {
          read_position(j + 1, SINGLE, x[(j + 1) % 2]);
          if (j + 2 == TN) place(tap0_next, q_next, NEXT, lead_next);
        } else {
          park_filters((step_no + 1) & 1);
          __syncthreads();  // the next step's filters are there; nobody reads this one's patch any more
          // the patch's loads are spread over the steps (all at once they fill the vector cache's queue, and
          // every wave waits for memory there: 8000 cycles), ahead of the filters' so that parking those waits
          // for nothing younger
          if constexpr (!SINGLE) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if ((parts >> k) & 1) request_part(k);
          }
          request_filters(half_after);
          if constexpr (TURN) {
            if (stage + 1 < stages) park_patch();
          } else {
            enter_step();
            read_position(0, NEXT, x[TN % 2]);
          }
        }
#pragma unroll
        for (int i0 = 0; i0 < TM; i0 += 2) {
#pragma unroll
          for (int t = 0; t < PRODUCTS; ++t)
#pragma unroll
            for (int i = i0; i < TM && i < i0 + 2; ++i) {
              f32x4 &into = t + 1 < PRODUCTS ? low[j][i] : acc[j][i];
              into = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j % 2][PX[t]], w[i][PW[t]], into, 0, 0, 0);
            }
          if (j + 1 == TN) {
#pragma unroll
            for (int i = i0; i < TM && i < i0 + 2; ++i) read_filters((step_no + 1) & 1, i, NEXT);
          }
        }
        if (j + 1 < TN) __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (TURN) {
        __syncthreads();
        enter_step();
        read_position(0, NEXT, x[0]);
        if (stage + 1 < stages) aim(stage + 1);
      } else if constexpr (TN % 2 != 0) {
#pragma unroll
        for (int part = 0; part < 3; ++part) x[0][part] = x[1][part];
      }
      ++step_no;
    };
    if (stages > 0) {
      const std::true_type yes;
      const std::false_type no;
      const int half0 = table[0][0];
      __syncthreads();  // (the last item's operands and notes have been read)
      if (threadIdx.x < 3) note[threadIdx.x] = 0;
      lost = 0, tiniest = u16x2{0xffff, 0xffff};
      request_filters(half0);
      if (!ahead) {
        patch_row = first_row, patch_e = table[0], patch_real = true;
#pragma unroll
        for (int k = 0; k < 4; ++k) request_part(k);
      }
      park_patch();
      park_filters(0);
      request_filters(half0 + 2);
      aim(0);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < TM; ++i) read_filters(0, i, false);
      place(table[0][3], 0, false, (first_row + table[0][2]) & 3);
      enter_step();
      read_position(0, false, x[0]);
      for (int stage = 0; stage < stages; ++stage) {
        const int8v here = table[stage], there = table[min(stage + 1, stages - 1)];
        const int tap0 = here[3], tap0_next = there[3], lead = (first_row + here[2]) & 3, lead_next = (first_row + there[2]) & 3;
        const int half = half0 + stage * window;  // (stages follow each other in the packed filters)
        // the quarters of the next patch (bits) that pair s of `pairs` requests: all but the last pair share them
        const int pairs = window / 2, spread = max(pairs - 1, 1);
        auto parts_of = [&](int s) -> int {
          const int from = min(4, (4 * s + spread - 1) / spread), to = min(4, (4 * s + 4 + spread - 1) / spread);
          return (1 << to) - (1 << from);
        };
        if constexpr (ODD) {
          // window = 2 n + 1 >= 3: n pairs, then the single tap; filters are requested two steps ahead
          int q = 0;
          for (; q + 4 < window; q += 2) step(no, no, no, half + q + 4, tap0, q + 2, lead, stage, parts_of(q / 2));
          step(no, no, yes, half + window, tap0, q + 2, lead, stage, parts_of(q / 2));
          step(yes, yes, no, half + window + 2, tap0_next, 0, lead_next, stage, 0);
        } else {
          int q = 0;
          for (; q + 2 < window; q += 2) step(no, no, no, half + q + 4, tap0, q + 2, lead, stage, parts_of(q / 2));
          step(no, yes, no, half + window + 2, tap0_next, 0, lead_next, stage, parts_of(q / 2));
        }
      }
      ahead = patch_real;
    }

    // ---- epilogue: acc[j][i][q] is row m0 + wm0 + 16 i + l16 at position pos0 + 64 wave + 16 j + 4 lk + q
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[j][i] += low[j][i];
    const Phase &ph = me.ph;
    const int first = me.pos0 + wave * WN + lk * 4;
    if (stages > 0) {
      unsigned largest = 0;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) largest = max(largest, bits_of(acc[j][i][q]) << 1);
      const unsigned mine = (largest >= 2u * (255u << 23) ? kNotFinite : 0u) | ((lost & 0xffffu) != 0 ? kLostElement : 0u) |
                            ((int)threadIdx.x < 4 * BM && min(tiniest[0], tiniest[1]) < kTinyBits - 1 ? kTinyFilter : 0u);
      if (mine != 0) atomicOr(&note[0], mine);
      __syncthreads();
      unsigned found = (unsigned)uniform((int)note[0]);
      if ((found & (kLostElement | kTinyFilter)) != 0 && (found & kNotFinite) == 0) {
        // seldom: the largest value that meets one that has lost bits
        unsigned widest = 0;
        if ((found & kLostElement) != 0) {
          for (int at = (int)threadIdx.x; at < stages * window * 2 * BM; at += THREADS) {
            const int m = me.m0 + at % BM, octet = table[0][0] * 2 + at / BM;
            const unsigned from = m < p.a_ld ? (unsigned)(octet * 3) * piece_row + (unsigned)m * 16u : kOutside;
            const u32x4 firsts = __builtin_amdgcn_raw_buffer_load_b128(a_buf, (int)from, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) widest = max(widest, max((firsts[e] & 0x7fffu) << 16, firsts[e] & 0x7fff0000u));
          }
          atomicMax(&note[1], widest);
        }
        if ((found & kTinyFilter) != 0) {
          widest = 0;
          patch_row = first_row, patch_real = true;
          for (int stage = 0; stage < stages; ++stage) {
            patch_e = table[stage];
#pragma unroll
            for (int k = 0; k < 4; ++k) request_part(k);
#pragma unroll
            for (int round = 0; round < ROUNDS; ++round)
              if (round * THREADS < p.patch_rows) {
#pragma unroll
                for (int r = 0; r < 16; ++r) widest = max(widest, raw[round][r / 4][r % 4] & 0x7fffffffu);
              }
          }
          ahead = false;  // (the next item's first patch was there)
          atomicMax(&note[2], widest);
        }
        __syncthreads();
        const float bound = (float_of(note[1]) + float_of(note[2])) * (float)(stages * window * 16) * 0x1.02p-109f;  // (first parts are rounded)
        bool below = false;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              below |= me.m0 + wm0 + i * 16 + l16 < p.M && first + j * 16 + q < ph.npos && __builtin_fabsf(acc[j][i][q]) < bound;
        if (below) atomicOr(&note[0], (unsigned)kLostSum);
        __syncthreads();
        found = (unsigned)uniform((int)note[0]);
      }
      if ((found & (kNotFinite | kLostSum)) != 0 && threadIdx.x == 0) {
        p.redo[0] = 1;
        atomicOr(&p.redo[1 + me.tile / 32], 1u << (me.tile % 32));
      }
    }

    if (me.partial) {
      float *slot = static_cast<float *>(p.partial) + (long long)me.slot * (BM * BN) + wave * WN + lk * 4;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4 *>(slot + (wm0 + i * 16 + l16) * BN + j * 16) = acc[j][i];
      continue;
    }
    const int jvol = ph.J[0] * ph.J[1] * ph.J[2];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int four = first + j * 16;
      if (four >= ph.npos) continue;
      // four positions that are adjacent in dst leave as one vector, aligned or not (see GemmParams::run_store)
      bool together = p.vec_store;
      if (p.run_store && four + 4 <= ph.npos) {
        const unsigned n = ph.by_jvol.div((unsigned)four);
        together = (unsigned)four - n * (unsigned)jvol + 4u <= (unsigned)jvol;
      }
      if (together) {
        typedef float OutVec __attribute__((ext_vector_type(4), aligned(4)));
        float *out = dst_of(p, ph, four);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int m = me.m0 + wm0 + i * 16 + l16;
          if (m < p.M) *reinterpret_cast<OutVec *>(out + (long long)m * p.dst_mstride) = acc[j][i];
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (four + q >= ph.npos) continue;
          float *out = dst_of(p, ph, four + q);
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            const int m = me.m0 + wm0 + i * 16 + l16;
            if (m < p.M) out[(long long)m * p.dst_mstride] = acc[j][i][q];
          }
        }
      }
    }
  }
}

// The marked tiles (bm x bn, of one phase) of split_gemm_kernel again, on the single-precision instruction.
// Where few are marked a block takes up to 32 rows by 32 positions of one at a time, its waves a share of K
// each, which they add up in order: one marked tile is the work of twelve blocks.  Where many are, a wave takes
// 16 TM rows by 64 positions over the whole of K.  Elements are gathered one by one (a tap that a position does
// not have reads zero, as in the patch).  Filter values are the sums of their parts, which lie together as
// lanes want them, but for lanes that find one among theirs which the parts do not hold.  Seldom anything to
// do: 4.5 us behind every pass.  Not built for the last bit of speed: a step waits for its own loads (four
// parts of some 16 us a block is where the one way meets the other).
constexpr int kRedoWaves = 8, kRedoBlocks = 512;  // a power of two

template <int TM>
__global__ void __launch_bounds__(64 * kRedoWaves, 2) split_redo_kernel(const GemmParams p, int bm, int bn, int tiles) {
  const unsigned *const redo = p.redo;
  if (redo[0] == 0) return;
  constexpr int FEW = TM < 4 ? TM : 2;  // 16-row tiles of a block's part where few tiles are marked
  __shared__ f32x4 shares[kRedoWaves - 1][2 * FEW][64];
  const int lane = threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4, wave = uniform((int)threadIdx.x >> 6);
  const __amdgpu_buffer_rsrc_t a_buf = buffer_of(p.A, p.a_bytes);
  const __amdgpu_buffer_rsrc_t w_buf = buffer_of(p.split_w, p.split_w_bytes);
  const __amdgpu_buffer_rsrc_t src_buf = buffer_of(p.src, p.src_bytes);
  const __amdgpu_buffer_rsrc_t table_buf = buffer_of(p.positions, (unsigned)p.npos * 8u);
  const Phase ph = load_phase(p.phases, 0);
  const int16v sp = ((const int16v MG_CONSTANT *)p.split_phases)[0];
  const int window = sp[9], pairs = (window + 1) / 2;
  const unsigned piece_row = (unsigned)p.a_ld * 16u;
  const bool second = lk >= 2;  // as in split_gemm_kernel: this lane's are eight channels under the second tap of a step
  const int words = (tiles + 31) / 32;
  const int MG_CONSTANT *const inner = as_constant(p.split_inner) + sp[10];
  const int8v MG_CONSTANT *const table = (const int8v MG_CONSTANT *)p.ktiles + ph.k_begin;

  // part `part` of a tile: 16 ROWS rows by 16 COLS positions, by the block or (ALONE) by the wave
  auto compute = [&](auto rows_c, auto cols_c, auto alone_c, int tile, int part) {
    constexpr int ROWS = decltype(rows_c)::value, COLS = decltype(cols_c)::value;
    constexpr bool ALONE = decltype(alone_c)::value;
    const int across = bn / (16 * COLS);
    const int m0 = tile % p.m_tiles * bm + part / across * 16 * ROWS, pos0 = tile / p.m_tiles * bn + part % across * 16 * COLS;
    int row_at[COLS];
    unsigned taps[COLS];
#pragma unroll
    for (int j = 0; j < COLS; ++j) {
      typedef int int2v __attribute__((ext_vector_type(2)));
      const unsigned ipos = (unsigned)(pos0 + j * 16 + l16);
      const int2v at = __builtin_bit_cast(int2v, __builtin_amdgcn_raw_buffer_load_b64(table_buf, (int)(ipos * 8u), 0, 0));
      row_at[j] = at[0];
      taps[j] = (unsigned)at[1];
    }
    f32x4 acc[COLS][ROWS];
#pragma unroll
    for (int j = 0; j < COLS; ++j)
#pragma unroll
      for (int i = 0; i < ROWS; ++i) acc[j][i] = f32x4{0, 0, 0, 0};
    for (int step = ALONE ? 0 : wave; step < ph.k_count * pairs; step += ALONE ? 1 : kRedoWaves) {  // 16 channels under two taps
      const int8v here = table[step / pairs];  // see GemmParams
      const int q = step % pairs * 2 + (second ? 1 : 0), octet = lk & 1;
      const bool has_tap = q < window;
      const unsigned dead = (unsigned)here[5] >> (octet * 8);
      float xs[COLS][8];
#pragma unroll
      for (int j = 0; j < COLS; ++j) {
        const int row = row_at[j] + here[2] + inner[has_tap ? q : 0];
        const unsigned n = __umulhi((unsigned)max(row, 0), p.by_sample.mul) >> p.by_sample.shr;
        const unsigned at = (n * (unsigned)p.src_nstride + (unsigned)(row - (int)n * p.sample_rows + here[1] + octet * 8 * p.src_cstride)) * 4u;
        const unsigned from = has_tap && ((taps[j] >> (here[3] + q)) & 1u) != 0 ? at : kOutside;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const unsigned lane_at = from | ((dead << (31 - e)) & kOutside), channel_at = (unsigned)(e * p.src_cstride) * 4u;
          xs[j][e] = float_of(__builtin_amdgcn_raw_buffer_load_b32(src_buf, (int)lane_at, (int)channel_at, 0));
        }
      }
      float ws[ROWS][8];
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        const int m = m0 + i * 16 + l16;
        const unsigned at = has_tap && m < p.a_ld ? (unsigned)((here[0] + q) * 2 + octet) * 3u * piece_row + (unsigned)m * 16u : kOutside;
        u32x4 parts[3];
#pragma unroll
        for (int part = 0; part < 3; ++part) parts[part] = __builtin_amdgcn_raw_buffer_load_b128(a_buf, (int)at, (int)((unsigned)part * piece_row), 0);
        bool whole = true;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float v[3];
#pragma unroll
          for (int part = 0; part < 3; ++part) v[part] = float_of(e % 2 != 0 ? parts[part][e / 2] & 0xffff0000u : parts[part][e / 2] << 16);
          ws[i][e] = v[0] + (v[1] + v[2]);
          whole &= v[0] == 0.0f || (__builtin_fabsf(v[0]) >= 0x1p-109f && __builtin_fabsf(v[0]) < __builtin_inff());
        }
        if (!whole) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int c = here[4] + octet * 8 + e;
            const unsigned from = (unsigned)(m * p.split_w_mstride + c * p.split_w_cstride + here[3] + q) * 4u;
            ws[i][e] = float_of(__builtin_amdgcn_raw_buffer_load_b32(w_buf, (int)(from | ((dead << (31 - e)) & kOutside)), 0, 0));
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int i = 0; i < ROWS; ++i)
#pragma unroll
          for (int j = 0; j < COLS; ++j) acc[j][i] = Mma<float>::run(xs[j][e], ws[i][e], acc[j][i]);
    }
    if constexpr (!ALONE) {
      __syncthreads();  // (the shares of the part before have been read)
      if (wave > 0) {
#pragma unroll
        for (int j = 0; j < COLS; ++j)
#pragma unroll
          for (int i = 0; i < ROWS; ++i) shares[wave - 1][j * ROWS + i][lane] = acc[j][i];
      }
      __syncthreads();
      if (wave > 0) return;
#pragma unroll
      for (int j = 0; j < COLS; ++j)
#pragma unroll
        for (int i = 0; i < ROWS; ++i)
          for (int other = 0; other < kRedoWaves - 1; ++other) acc[j][i] += shares[other][j * ROWS + i][lane];
    }
#pragma unroll
    for (int j = 0; j < COLS; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ipos = pos0 + j * 16 + 4 * lk + q;
        if (ipos >= ph.npos) continue;
        float *const out = dst_of(p, ph, ipos);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
          const int m = m0 + i * 16 + l16;
          if (m < p.M) out[(long long)m * p.dst_mstride] = acc[j][i][q];
        }
      }
  };

  int count = 0;
  for (int first = 0; first < words; first += 64) {
    int mine = first + lane < words ? __popc(redo[1 + first + lane]) : 0;
    for (int step = 1; step < 64; step *= 2) mine += __shfl_xor(mine, step);
    count += mine;
  }
  const std::integral_constant<int, 2> two;
  const std::integral_constant<int, 4> four;
  const int few_parts = bn / 32 * (bm / (16 * FEW));
  if ((long long)count * few_parts <= 4 * kRedoBlocks) {
    // every wave finds the marked tiles in the same order, and the block's parts of them
    for (int first = 0; first < words; first += 64) {
      const unsigned mine = first + lane < words ? redo[1 + first + lane] : 0u;
      for (unsigned long long some = __ballot(mine != 0); some != 0; some &= some - 1) {
        const int from = __builtin_ctzll(some);
        for (unsigned word = (unsigned)__builtin_amdgcn_readlane((int)mine, from); word != 0; word &= word - 1) {
          const int tile = (first + from) * 32 + __builtin_ctz(word);
          for (int part = (int)((blockIdx.x - (unsigned)(tile * few_parts)) & (kRedoBlocks - 1)); part < few_parts; part += kRedoBlocks)
            compute(std::integral_constant<int, FEW>(), two, std::false_type(), tile, part);
        }
      }
    }
  } else {
    const int parts = bn / 64 * (bm / (16 * TM));
    for (int unit = (int)blockIdx.x * kRedoWaves + wave; unit < tiles * parts; unit += kRedoBlocks * kRedoWaves) {
      const int tile = unit / parts;
      if (((redo[1 + tile / 32] >> (tile % 32)) & 1u) != 0) compute(std::integral_constant<int, TM>(), four, std::true_type(), tile, unit % parts);
    }
  }
}

// The filters of split_gemm_kernel, in three parts: piece [octet of K rows][part][m] holds the eight bf16
// values of K rows 8 * octet .. + 7 of row m of the product, `ld` (a multiple of 16) pieces to a row.  Sixteen
// K rows are 16 channels from c0 on under one tap, named by halves[K row / 16] = (c0, tap): row m's value is
// w[m * m_stride + c * c_stride + tap], zero for c >= channels and m >= M.  A value that is not zero has a
// first part that is not, the smallest number of bf16 at least: that is how split_gemm_kernel knows of those
// that have lost bits.  Also clears the marks of tiles, `marks` words of them.
__global__ void __launch_bounds__(256) split_pack_kernel(const float *__restrict__ w, u32x4 *__restrict__ packed, const int2 *__restrict__ halves,
                                                         int count, unsigned *__restrict__ redo, int marks, int M, int channels, long long m_stride,
                                                         long long c_stride, int ld) {
  const unsigned block = blockIdx.y * gridDim.x + blockIdx.x, blocks = gridDim.x * gridDim.y;
  for (unsigned i = block * 256 + threadIdx.x; i < (unsigned)marks; i += blocks * 256) redo[i] = 0;
  const int oct = blockIdx.x * 16 + (int)(threadIdx.x >> 4), m = blockIdx.y * 16 + (int)(threadIdx.x & 15);
  if (oct >= 2 * count) return;
  const int2 h = halves[oct / 2];
  const int c0 = h.x + oct % 2 * 8;
  u32x4 parts[3];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = c0 + 2 * e + u;
      v[u] = m < M && c < channels ? w[(long long)m * m_stride + (long long)c * c_stride + h.y] : 0.0f;
    }
    unsigned first, second, third, lost = 0;
    split_pair(v[0], v[1], first, second, third, lost);
    if (v[0] != 0.0f && (first & 0x7fffu) == 0) first |= 1u;
    if (v[1] != 0.0f && (first & 0x7fff0000u) == 0) first |= 1u << 16;
    parts[0][e] = first, parts[1][e] = second, parts[2][e] = third;
  }
#pragma unroll
  for (int part = 0; part < 3; ++part) packed[((long long)oct * 3 + part) * ld + m] = parts[part];
}

// (row, taps) of every position: the row of src (sample * sample_rows + element of a channel's plane) that its
// window starts from, padding aside, and which taps have an element there, bit by bit.
__global__ void __launch_bounds__(256) split_positions_kernel(const SplitPositions p, int2 *__restrict__ out) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= p.npos) return;
  const int j12 = p.J[1] * p.J[2], n = idx / (p.J[0] * j12), r = idx - n * p.J[0] * j12;
  const int q0 = r / j12, q1 = r / p.J[2] % p.J[1], q2 = r % p.J[2];
  unsigned taps = 0;
  int t = 0;
  for (int a = 0; a < p.sp.count[0]; ++a)
    for (int b = 0; b < p.sp.count[1]; ++b)
      for (int c = 0; c < p.sp.count[2]; ++c, ++t) {
        const int i0 = q0 + p.sp.d[0] + a * p.sp.step[0], i1 = q1 + p.sp.d[1] + b * p.sp.step[1], i2 = q2 + p.sp.d[2] + c * p.sp.step[2];
        if ((unsigned)i0 < (unsigned)p.Q[0] && (unsigned)i1 < (unsigned)p.Q[1] && (unsigned)i2 < (unsigned)p.Q[2]) taps |= 1u << t;
      }
  out[idx] = int2{n * p.sample_rows + (q0 * p.Q[1] + q1) * p.Q[2] + q2, (int)taps};
}

// rows of a wave; waves along the rows of a tile; 16 positions of a wave; waves along the positions; rounds of
// a patch (the fewest that hold it)
#define MG_SPLIT_SHAPES(X) \
  X(32, 4, 4, 2, 1) X(64, 1, 3, 4, 2) X(32, 2, 4, 2, 1) X(32, 2, 4, 2, 2) X(48, 1, 4, 4, 2) X(32, 1, 4, 4, 2) X(16, 1, 4, 4, 2)

// Rows of a patch that a tile has room for: those of its threads' rounds, and two blocks share a unit's LDS
// (alone on it, a block's waves wait for their barriers: 256 filters, 3x3, stride 2, 27x27 161 us on patches of
// 540 rows, 134 on the other kernel).
constexpr int patch_limit(int bm, int threads, int rounds) {
  const int held = threads * rounds, room = (80 * 1024 / 16 - 24 * bm - 1) / 6 - 1;
  return held < room ? held : room;
}

size_t lds_bytes(int bm, int patch_rows) { return (size_t)(2 * 12 * bm + 2 * (patch_rows + 1) * 3 + 1) * 16; }

}  // namespace

int split_patch_limit(int bm, int bn) {
  int most = 0;
#define MG_LIMIT(WM, MW, TN, NW, ROUNDS) \
  if (bm == WM * MW && bn == 16 * TN * NW) most = std::max(most, patch_limit(bm, 64 * MW * NW, ROUNDS));
  MG_SPLIT_SHAPES(MG_LIMIT)
#undef MG_LIMIT
  return most;
}

int split_gemm_blocks_per_cu(int bm, int bn, int patch_rows) {
  static std::map<std::array<int, 3>, int> known;  // (behind the lock of the entry points)
  int &n = known[{bm, bn, patch_rows}];
  if (n > 0) return n;
#define MG_OCC(WM, MW, TN, NW, ROUNDS)                                                                                     \
  if (n == 0 && bm == WM * MW && bn == 16 * TN * NW && patch_rows <= patch_limit(bm, 64 * MW * NW, ROUNDS)) {              \
    const auto odd = split_gemm_kernel<WM, MW, TN, NW, ROUNDS, true>, even = split_gemm_kernel<WM, MW, TN, NW, ROUNDS, false>; \
    for (const auto kernel : {odd, even})                                                                                  \
      (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);             \
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, odd, 64 * MW * NW, lds_bytes(bm, patch_rows)) != hipSuccess) n = 0; \
  }
  MG_SPLIT_SHAPES(MG_OCC)
#undef MG_OCC
  if (n < 1) {
    (void)hipGetLastError();
    n = 1;
  }
  return n;
}

bool launch_split_gemm(const GemmParams &p, int bm, int bn, bool odd, unsigned grid, hipStream_t s) {
#define MG_LAUNCH(WM, MW, TN, NW, ROUNDS)                                                                                              \
  if (bm == WM * MW && bn == 16 * TN * NW && p.patch_rows <= patch_limit(bm, 64 * MW * NW, ROUNDS)) {                                  \
    const auto kernel = odd ? split_gemm_kernel<WM, MW, TN, NW, ROUNDS, true> : split_gemm_kernel<WM, MW, TN, NW, ROUNDS, false>;      \
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * MW * NW), lds_bytes(bm, p.patch_rows), s, p);                                     \
    return true;                                                                                                                       \
  }
  MG_SPLIT_SHAPES(MG_LAUNCH)
#undef MG_LAUNCH
  return false;
}

void launch_split_redo(const GemmParams &p, int bm, int bn, int tiles, hipStream_t s) {
  const auto kernel = bm % 64 == 0 ? split_redo_kernel<4>
                      : bm == 48   ? split_redo_kernel<3>
                      : bm == 32   ? split_redo_kernel<2>
                                   : split_redo_kernel<1>;
  hipLaunchKernelGGL(kernel, dim3(kRedoBlocks), dim3(64 * kRedoWaves), 0, s, p, bm, bn, tiles);
}

void launch_split_pack(const float *w, void *packed, const void *halves, int count, unsigned *redo, int marks, int M, int channels,
                       long long m_stride, long long c_stride, int ld, hipStream_t s) {
  hipLaunchKernelGGL(split_pack_kernel, dim3((unsigned)ceil_div(2 * count, 16), (unsigned)(ld / 16)), dim3(256), 0, s, w,
                     static_cast<u32x4 *>(packed), static_cast<const int2 *>(halves), count, redo, marks, M, channels, m_stride,
                     c_stride, ld);
}

void launch_split_positions(const SplitPositions &p, void *out, hipStream_t s) {
  hipLaunchKernelGGL(split_positions_kernel, dim3((unsigned)ceil_div(p.npos, 256)), dim3(256), 0, s, p, static_cast<int2 *>(out));
}

}  // namespace mg
