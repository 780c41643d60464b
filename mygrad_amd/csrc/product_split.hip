// Large matrix products in single precision on the bf16 matrix instructions, three parts of eight bits to a
// float and six products of parts to a product: see conv_split.hip for the arithmetic, its accuracy (two
// accumulators) and what parts cannot represent (marked tiles).
//
// With one tap nothing is used twice from a patch, so both operands are split in a pass of their own
// (product_pack_kernel), into the order in which the products want them: a panel of 128 rows by 32 k is 24 KiB that
// go into LDS as they lie, without a register or an address in between, and a wave's operands are its rows' pieces
// of 16 bytes side by side, free of bank conflicts in either orientation of the matrix.
//
// What bounds it: 4096 x 4096 x 4096, 137.4 GFLOP, takes 56 us for the packing (134 MB read, 202 MB written, 6.0
// TB/s), 495 - 513 by device for the products (825 GFLOP of parts, 1.61 - 1.67 PFLOP/s; 570 - 590 in the first passes from idle) and
// 5 for the pass behind them: 560 - 590, single precision 965 - 1000.  The matrix pipes are 80 % busy at 1.9 GHz, what the device's
// power allows beside them, LDS 20 %.
// Error against 64 bits (2-norm), normal values: 4.0e-7, single precision 1.15e-6; at 1024 terms 8.6e-8 and 2.9e-7, at 64
// 5.0e-8 and 1.05e-7.
#include "product_split.h"
#include "internal.h"
#include "split_device.h"

#include <algorithm>
#include <cstdlib>

namespace mg {

namespace {

// Eight consecutive k (octet `oct`) of row `row`, zeros outside the operand.
__device__ __forceinline__ void load_octet(const ProductOperand &o, int octets, int row, int oct, float (&v)[8]) {
  typedef float Quad __attribute__((ext_vector_type(4), aligned(4)));
  const int rb = (int)o.by_rows.div((unsigned)row), kb = (int)o.by_octets.div((unsigned)oct);
  const int k = (oct - kb * (int)o.by_octets.d) * 8;
  const float *from = o.base + rb * o.rows_out + (row - rb * (int)o.by_rows.d) * o.row_stride + kb * o.k_out + k * o.k_stride;
  const int count = row < o.rows && oct < octets ? min(o.k_in - k, 8) : 0;
  if (o.k_stride == 1 && count == 8) {
    const Quad first = *reinterpret_cast<const Quad *>(from), last = *reinterpret_cast<const Quad *>(from + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = first[e], v[e + 4] = last[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = e < count ? from[e * o.k_stride] : 0.0f;
  }
}

// A panel's K step, 128 rows by 32 k, in three parts: a block each.
__global__ void __launch_bounds__(256) product_pack_kernel(const ProductParams p) {
  const int step = (int)blockIdx.x, panel = (int)blockIdx.y, t = (int)threadIdx.x;
  if (blockIdx.y == 0)
    for (int i = step * 256 + t; i < p.marks; i += p.steps * 256) p.redo[i] = 0;
  const bool second = panel >= p.a_panels;
  const ProductOperand &o = second ? p.b : p.a;
  const int own = second ? panel - p.a_panels : panel;
  u32x4 *const out = static_cast<u32x4 *>(second ? p.packed_b : p.packed_a) + ((long long)own * p.steps + step) * (kProductPanelBytes / 16);
  const bool along = o.k_stride == 1;  // four lanes take the 128 bytes of a row, or 128 lanes a row of the transpose
  float v[2][8];
  int row[2], oct[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int idx = t + u * 256;
    row[u] = along ? idx >> 2 : idx & 127, oct[u] = along ? idx & 3 : idx >> 7;
    load_octet(o, p.octets, own * kProductPanel + row[u], step * 4 + oct[u], v[u]);
  }
  unsigned widest = 0, lost = 0;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    u32x4 parts[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      unsigned h, m, l;
      split_pair(v[u][2 * e], v[u][2 * e + 1], h, m, l, lost);
      parts[0][e] = h, parts[1][e] = m, parts[2][e] = l;
      widest = max(widest, max(bits_of(v[u][2 * e]) << 1, bits_of(v[u][2 * e + 1]) << 1));
    }
#pragma unroll
    for (int part = 0; part < 3; ++part) out[(part * 4 + oct[u]) * kProductPanel + row[u]] = parts[part];
  }
  __shared__ unsigned notes[4];
  unsigned note = widest | ((lost & 0xffffu) != 0 ? 1u : 0u);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const unsigned other = (unsigned)__shfl_xor((int)note, d);
    note = max(note & ~1u, other & ~1u) | ((note | other) & 1u);
  }
  if ((t & 63) == 0) notes[t >> 6] = note;
  __syncthreads();
  if (t == 0) {
    for (int w = 1; w < 4; ++w) note = max(note & ~1u, notes[w] & ~1u) | ((note | notes[w]) & 1u);
    p.notes[(long long)panel * p.steps + step] = note;
  }
}

// The tile'th tile: groups of four row tiles run along all columns, so that the 32 tiles of one XCD's blocks touch
// four row tiles and eight column tiles.
struct TilePlace {
  int m, n;
};
__device__ __forceinline__ TilePlace tile_place(int tile, int m_tiles, int n_tiles) {
  const int group = tile / (4 * n_tiles), within = tile - group * 4 * n_tiles, high = min(4, m_tiles - group * 4);
  return TilePlace{group * 4 + within % high, within / high};
}

// The K steps [begin, end) of all the tiles from full_tiles on, end to end, that sharing block b takes.
struct Share {
  int begin, end;
};
__device__ __forceinline__ Share share_of(const ProductParams &p, int b) {
  const int begin = b * p.share_steps + min(b, p.share_extra);
  return Share{begin, begin + p.share_steps + (b < p.share_extra ? 1 : 0)};
}

// Loads that a wave requests for the stage after next as soon as this one has been read; the others follow in the next stage.  (All at
// once they fill the vector cache's queue, and no wave gets to its products: 535 us at 4096 x 4096 x 4096, 490 so.)
constexpr int kEarly = 5;

template <int PM, int PN>
__global__ void __launch_bounds__(512, 2) product_gemm_kernel(const ProductParams p) {
  constexpr int BM = PM * kProductPanel, BN = PN * kProductPanel, STAGE = (PM + PN) * kProductPanelBytes;
  static_assert(PM * PN == 2, "eight waves of 64 x 64");
  extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
  unsigned *const note = reinterpret_cast<unsigned *>(lds + 2 * STAGE / 16);
  const int lane = (int)threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4, wave = uniform((int)threadIdx.x >> 6);
  const int wm = wave / (2 * PN) * 64, wn = wave % (2 * PN) * 64;
  const int n_tiles = p.tiles / p.m_tiles;
  const long long panel_bytes = (long long)p.steps * kProductPanelBytes;
  // blocks are dealt to the eight XCDs in turn: an XCD's blocks take consecutive tiles
  const int grid = (int)gridDim.x, place = grid % 8 == 0 ? (int)(blockIdx.x & 7) * (grid / 8) + (int)(blockIdx.x >> 3) : (int)blockIdx.x;

  struct Cursor {
    int index, tile, step, end, slot;
    bool live;
  };
  const int whole = p.full_tiles / grid;
  const Share share = place < p.share_blocks ? share_of(p, place) : Share{0, 0};
  auto enter = [&](Cursor &c) {
    c.slot = -1;
    if (c.index < whole) {
      c.tile = place + c.index * grid, c.step = 0, c.end = p.steps, c.live = true;
      return;
    }
    const int first = share.begin / p.steps, nth = c.index - whole, base = (first + nth) * p.steps;
    const int from = max(share.begin, base), to = min(share.end, base + p.steps);
    c.live = from < to;
    c.tile = p.full_tiles + first + nth, c.step = from - base, c.end = to - base;
    if (to - from < p.steps) c.slot = 2 * place + nth;
  };
  auto forward = [&](Cursor &c) {
    if (++c.step < c.end) return;
    ++c.index;
    enter(c);
  };

  __amdgpu_buffer_rsrc_t a_buf, b_buf;
  Cursor ahead{};  // of the stage that is requested next
  auto aim = [&](const Cursor &c) {
    const TilePlace at = tile_place(c.tile, p.m_tiles, n_tiles);
    a_buf = buffer_of(static_cast<const char *>(p.packed_a) + at.m * PM * panel_bytes, (unsigned)(PM * panel_bytes));
    b_buf = buffer_of(static_cast<const char *>(p.packed_b) + at.n * PN * panel_bytes, (unsigned)(PN * panel_bytes));
  };
  const unsigned lds_base = (unsigned)reinterpret_cast<unsigned long long>((__attribute__((address_space(3))) char *)lds);
  const unsigned lane_at = (unsigned)lane * 16;
  // A wave's loads of a stage, nine of 1 KiB: three pieces of each panel.
  constexpr int LOADS = 3 * (PM + PN);
  auto request = [&](int k, int stage) {
    const int panel = k / 3;
    const unsigned piece = (unsigned)(wave + k % 3 * 8) * 1024u;
    const unsigned at = (unsigned)(panel < PM ? panel : panel - PM) * (unsigned)panel_bytes + (unsigned)ahead.step * kProductPanelBytes + piece;
    to_lds<16>(panel < PM ? a_buf : b_buf, lane_at, at, lds_base + (unsigned)stage * STAGE + (unsigned)panel * kProductPanelBytes + piece);
  };
  auto step_ahead = [&] {
    if (!ahead.live) return;
    const int tile = ahead.tile;
    forward(ahead);
    if (!ahead.live) a_buf = b_buf = buffer_of(p.packed_a, 0);  // nothing more: zeros that nobody uses
    else if (ahead.tile != tile) aim(ahead);
  };
  enter(ahead);
  Cursor here = ahead;
  if (!here.live) return;
  aim(ahead);
#pragma unroll
  for (int k = 0; k < LOADS; ++k) request(k, 0);
  step_ahead();
  landed();
#pragma unroll
  for (int k = 0; k < kEarly; ++k) request(k, 1);

  bf16x8 w[4][3], x[2][3];
  const u32x4 *const rows = lds + (wm / kProductPanel) * (kProductPanelBytes / 16) + wm % kProductPanel + l16 + lk * kProductPanel;
  const u32x4 *const cols = lds + (PM + wn / kProductPanel) * (kProductPanelBytes / 16) + wn % kProductPanel + l16 + lk * kProductPanel;
  auto read_rows = [&](int stage, int part) {
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i][part] = __builtin_bit_cast(bf16x8, rows[stage * (STAGE / 16) + part * 4 * kProductPanel + i * 16]);
  };
  auto read_col = [&](int stage, int j, bf16x8(&into)[3]) {
#pragma unroll
    for (int part = 0; part < 3; ++part) into[part] = __builtin_bit_cast(bf16x8, cols[stage * (STAGE / 16) + part * 4 * kProductPanel + j * 16]);
  };
#pragma unroll
  for (int part = 0; part < 3; ++part) read_rows(0, part);
  read_col(0, 0, x[0]);

  int stage = 0;
  while (here.live) {
    f32x4 acc[4][4], low[4][4];  // [j][i]: sums of the large product and of the five small ones
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][i] = low[j][i] = f32x4{0, 0, 0, 0};
    const int first_step = here.step;
    for (int left = here.end - here.step; left > 0; --left) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j < 3) {
          read_col(stage, j + 1, x[(j + 1) % 2]);
        } else {
          landed();  // the next stage is there, and nobody reads this one any more
          step_ahead();
          read_col(stage ^ 1, 0, x[0]);
        }
        // The order of issue is the one written here (the scheduler's own puts reads right in front of their uses): a
        // position's operands are read 24 products ahead, the rows' parts again as soon as the last position is done with them.
        __builtin_amdgcn_sched_barrier(0);
        constexpr int PX[6] = {0, 1, 0, 2, 1, 0}, PW[6] = {2, 1, 1, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < 6; ++t) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            f32x4 &into = t < 5 ? low[j][i] : acc[j][i];
            into = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[j % 2][PX[t]], w[i][PW[t]], into, 0, 0, 0);
          }
          if (j == 3 && t < kEarly) request(t, stage);
          if (j == 0 && t + kEarly < LOADS) request(t + kEarly, stage ^ 1);
          if (j == 3 && (t == 0 || t == 2 || t == 5)) read_rows(stage ^ 1, PW[t]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      stage ^= 1;
    }

    // ---- acc[j][i][q] is row wm + 16 i + l16 at column wn + 16 j + 4 lk + q of the tile
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][i] += low[j][i];
    const TilePlace at = tile_place(here.tile, p.m_tiles, n_tiles);
    unsigned largest = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) largest = max(largest, bits_of(acc[j][i][q]) << 1);
    // the widest values of either operand and which of them have lost bits: bit 0
    unsigned a_note = 0, b_note = 0;
    for (int i = (int)threadIdx.x; i < (PM + PN) * p.steps; i += 512) {
      const int panel = i / p.steps, step = i - panel * p.steps;
      if (step < first_step || step >= here.end) continue;
      const unsigned found = p.notes[(long long)(panel < PM ? at.m * PM + panel : p.a_panels + at.n * PN + panel - PM) * p.steps + step];
      unsigned &into = panel < PM ? a_note : b_note;
      into = max(into & ~1u, found & ~1u) | ((into | found) & 1u);
    }
    __syncthreads();
    if (threadIdx.x < 4) note[threadIdx.x] = 0;
    __syncthreads();
    if (((a_note | b_note) & 1u) != 0) atomicOr(&note[0], (a_note & 1u) | (b_note & 1u) << 1);
    if (largest >= 2u * (255u << 23)) atomicOr(&note[0], 4u);
    __syncthreads();
    unsigned found = (unsigned)uniform((int)note[0]);
    if (found != 0) {  // seldom
      if ((found & 4u) == 0) {
        atomicMax(&note[1], a_note);
        atomicMax(&note[2], b_note);
        __syncthreads();
        const float bound = ((found & 2u ? float_of(note[1] >> 1) : 0.0f) + (found & 1u ? float_of(note[2] >> 1) : 0.0f)) * (float)(p.steps * 32) * 0x1p-109f;
        bool below = false;  // (sums beyond the results' edges are zeros that nobody stores)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              below |= at.m * BM + wm + i * 16 + l16 < p.M && at.n * BN + wn + j * 16 + lk * 4 + q < p.columns && !(__builtin_fabsf(acc[j][i][q]) >= bound);
        if (below) atomicOr(&note[0], 4u);
        __syncthreads();
        found = (unsigned)uniform((int)note[0]);
      }
      if ((found & 4u) != 0 && threadIdx.x == 0) {
        p.redo[0] = 1;
        atomicOr(&p.redo[1 + here.tile / 32], 1u << (here.tile % 32));
      }
    }
    if (here.slot >= 0) {
      float *const slot = p.partial + (long long)here.slot * (BM * BN) + (wm + l16) * BN + wn + lk * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4 *>(slot + i * 16 * BN + j * 16) = acc[j][i];
    } else {
      typedef float Quad __attribute__((ext_vector_type(4), aligned(4)));
      const int m0 = at.m * BM + wm + l16, n0 = at.n * BN + wn + lk * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int col = n0 + j * 16;
        const int batch = (int)p.by_n.div((unsigned)col), n = col - batch * (int)p.by_n.d;
        if (col + 4 <= p.columns && n + 4 <= (int)p.by_n.d) {
          float *const out = p.dst + batch * p.dst_batch + n;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (m0 + i * 16 < p.M) *reinterpret_cast<Quad *>(out + (m0 + i * 16) * p.dst_mstride) = acc[j][i];
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (col + q >= p.columns) continue;
            const int bq = (int)p.by_n.div((unsigned)(col + q));
            float *const out = p.dst + bq * p.dst_batch + (col + q - bq * (int)p.by_n.d);
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (m0 + i * 16 < p.M) out[(m0 + i * 16) * p.dst_mstride] = acc[j][i][q];
          }
        }
      }
    }
    here.step = here.end - 1;
    forward(here);
  }
  // (the zeros requested behind the last stage are on their way into LDS that the next block may have)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Behind the products: the partial sums of the tiles whose K steps were shared, added in the order of K (the first
// `fix_blocks` blocks, 1024 elements each), and marked tiles again on the single-precision instruction, from the operands
// themselves (the others: 64 x 64 of a tile at a time, a wave 32 x 32 of that; seldom anything to do).
constexpr int kProductRedoBlocks = 512, kFixBlocks = 2 * kProductPanel * kProductPanel / 1024;  // of a tile

template <int PM, int PN>
__global__ void __launch_bounds__(256) product_finish_kernel(const ProductParams p, int fix_blocks) {
  constexpr int BM = PM * kProductPanel, BN = PN * kProductPanel, LD = 65;
  const int n_tiles = p.tiles / p.m_tiles, t = (int)threadIdx.x;
  const bool any = p.redo[0] != 0;
  auto marked = [&](int tile) { return any && ((p.redo[1 + tile / 32] >> (tile % 32)) & 1u) != 0; };
  auto store = [&](int m, int col, float v) {
    if (m >= p.M || col >= p.columns) return;
    const int batch = (int)p.by_n.div((unsigned)col);
    p.dst[batch * p.dst_batch + m * p.dst_mstride + (col - batch * (int)p.by_n.d)] = v;
  };
  if ((int)blockIdx.x < fix_blocks) {
    const int rest = (int)blockIdx.x / kFixBlocks, idx = ((int)blockIdx.x % kFixBlocks * 256 + t) * 4;  // of the tile's elements
    if (marked(p.full_tiles + rest)) return;
    const int first = rest * p.steps, last = first + p.steps;
    int b = first / (p.share_steps + 1);
    while (share_of(p, b).end <= first) ++b;
    f32x4 sum = {0, 0, 0, 0};
    for (bool begun = false; b < p.share_blocks; ++b, begun = true) {
      const Share share = share_of(p, b);
      if (share.begin >= last) break;
      if (share.begin <= first && share.end >= last) return;  // one block had all of it
      const int nth = rest - share.begin / p.steps;
      const f32x4 part = *reinterpret_cast<const f32x4 *>(p.partial + (long long)(2 * b + nth) * (BM * BN) + idx);
      sum = begun ? sum + part : part;
    }
    const TilePlace at = tile_place(p.full_tiles + rest, p.m_tiles, n_tiles);
#pragma unroll
    for (int q = 0; q < 4; ++q) store(at.m * BM + idx / BN, at.n * BN + idx % BN + q, sum[q]);
    return;
  }
  if (!any) return;
  __shared__ float as[32 * LD], bs[32 * LD];
  const int lane = t & 63, l16 = lane & 15, lk = lane >> 4, wave = uniform(t >> 6);
  const int wm = wave / 2 * 32, wn = wave % 2 * 32, row = t & 63, oct = t >> 6;
  // the blocks take the marked tiles' eighths in turn (by the number of a tile, those of one column of tiles would meet in a few blocks)
  int word = 0, before = 0;  // of the marks; tiles marked in the words before it
  for (int turn = (int)blockIdx.x - fix_blocks;; turn += kProductRedoBlocks) {
    int skip = turn / 8 - before;
    while (word < p.marks - 1 && __popc(p.redo[1 + word]) <= skip) {
      const int here = __popc(p.redo[1 + word++]);
      before += here, skip -= here;
    }
    if (word >= p.marks - 1) break;
    unsigned marks = p.redo[1 + word];
    while (skip-- > 0) marks &= marks - 1;
    const int tile = word * 32 + __ffs(marks) - 1, sub = turn % 8;
    const TilePlace at = tile_place(tile, p.m_tiles, n_tiles);
    const int m0 = at.m * PM * kProductPanel + sub / (2 * PN) * 64, n0 = at.n * PN * kProductPanel + sub % (2 * PN) * 64;
    f32x4 acc[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[j][i] = f32x4{0, 0, 0, 0};
    float av[8], bv[8];
    load_octet(p.a, p.octets, m0 + row, oct, av);
    load_octet(p.b, p.octets, n0 + row, oct, bv);
    for (int step = 0; step < p.steps; ++step) {
      __syncthreads();
#pragma unroll
      for (int e = 0; e < 8; ++e) as[(oct * 8 + e) * LD + row] = av[e], bs[(oct * 8 + e) * LD + row] = bv[e];
      __syncthreads();
      if (step + 1 < p.steps) {
        load_octet(p.a, p.octets, m0 + row, (step + 1) * 4 + oct, av);
        load_octet(p.b, p.octets, n0 + row, (step + 1) * 4 + oct, bv);
      }
#pragma unroll
      for (int k = 0; k < 32; k += 4) {
        float w[2], x[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) w[i] = as[(k + lk) * LD + wm + i * 16 + l16], x[i] = bs[(k + lk) * LD + wn + i * 16 + l16];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[j][i] = Mma<float>::run(x[j], w[i], acc[j][i]);
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 2; ++i) store(m0 + wm + i * 16 + l16, n0 + wn + j * 16 + lk * 4 + q, acc[j][i][q]);
  }
}

constexpr size_t kProductLds = 2 * 3 * kProductPanelBytes + 16;

ProductOperand operand_of(const void *base, long long runs, long long rows_in, long long rows_out, long long row_stride, long long k_in,
                          long long k_out, long long k_stride) {
  return ProductOperand{static_cast<const float *>(base), (int)(runs * rows_in), make_fastdiv((unsigned)rows_in), rows_out, row_stride,
                        (int)k_in, make_fastdiv((unsigned)ceil_div(k_in, 8)), k_out, k_stride};
}

struct ProductPlan {
  bool tall = true;  // tiles of 256 rows by 128 columns, not 128 by 256
  long long m_tiles = 0, n_tiles = 0, full_tiles = 0;
  int share_blocks = 0;
  long long longest = 0;  // K steps of the busiest block
};

// The tile orientation with the shorter run.  Tiles beyond whole rounds are shared by all blocks, four K steps each or
// more (a share costs the traffic of a slot of partial sums).
ProductPlan plan_product(long long M, long long columns, long long steps) {
  const int cus = runtime().props.multiProcessorCount;
  ProductPlan best;
  for (const bool tall : {true, false}) {
    ProductPlan pl;
    pl.tall = tall;
    pl.m_tiles = ceil_div(M, tall ? 256 : 128), pl.n_tiles = ceil_div(columns, tall ? 128 : 256);
    const long long tiles = pl.m_tiles * pl.n_tiles, rest = tiles % cus;
    pl.full_tiles = tiles - rest;
    pl.longest = pl.full_tiles / cus * steps;
    if (rest > 0) {
      pl.share_blocks = (int)std::max<long long>(rest, std::min<long long>(cus, rest * steps / 4));
      pl.longest += ceil_div(rest * steps, pl.share_blocks);
    }
    if (best.m_tiles == 0 || pl.longest < best.longest) best = pl;
  }
  return best;
}

}  // namespace

// Where the parts are faster: by modelled time, in us, of both ways, fitted to 660 products and gradients of 3 - 160
// GFLOP (48 - 9000 rows, columns and terms, 9 in 10 within 13 % of the model for the parts and 20 % for the other).
// Packing an operand costs as much as 1000 - 2000 products of each of its values, so that extents of a few hundred
// beside large ones stay: (72,8611) (8611,3924) 4.9 GFLOP 136 us on parts, 72 without; (1411,3000) (3000,1411) 62 and
// 78; 4096 x 4096 x 4096 560 and 965.  With 8 % in favour of the single-precision kernels three of those it takes are slower, by
// 6 % at most; the others are faster by 1.37 in the mean.
// The parts pad each run of terms to octets, the single-precision kernels pad nothing, but load runs that are no multiple of four a value at
// a time.  Of 260 gradients of stacks of 1 - 17 columns times one matrix, 4 - 90 GFLOP, it takes 52, one of them 6 % slower on parts; all
// take 1.03 of the faster way's time in the mean, 1.11 on the single-precision kernels.  (1024,1024) (8192,1024,1), 17 GFLOP: 281 us there, 690 on parts.
// MYGRAD_HIP_SPLIT_MIN=flops takes the place of the rule (tests).
bool product_applies(long long M, long long columns, long long runs, long long run) {
  const char *least = getenv("MYGRAD_HIP_SPLIT_MIN");
  const long long octets = runs * ceil_div(run, 8);
  const double terms = (double)runs * (double)run, flops = 2.0 * (double)M * (double)columns * terms;
  if (flops < (least ? atof(least) : 4e9)) return false;
  const char *flag = getenv("MYGRAD_HIP_SPLIT");
  if (flag && flag[0] == '0') return false;
  if ((getenv("MYGRAD_HIP_TILE") || getenv("MYGRAD_HIP_WGRAD_TILE")) && !least) return false;  // a tile of the convolution kernels was asked for
  if (M > (1 << 30) || columns > (1 << 30) || octets > (1 << 17)) return false;
  if (ceil_div(M, kProductPanel) + ceil_div(columns, kProductPanel) > 65500) return false;  // (the packing's grid has a row for each)
  if (least) return true;
  const long long steps = ceil_div(octets, 4);
  const ProductPlan pl = plan_product(M, columns, steps);
  const double read = (double)(M + columns) * (double)octets * 32.0;
  const double packed = (double)(pl.m_tiles * (pl.tall ? 2 : 1) + pl.n_tiles * (pl.tall ? 1 : 2)) * (double)steps * kProductPanelBytes;
  const double parts = 27.0 + 0.218e-6 * (read + packed) + 2.08 * (double)pl.longest + 0.163e-6 * 4.0 * (double)M * (double)columns;
  const double narrow = runs > 1 && run % 4 != 0 ? 1.0 + std::min(0.7, 2.4 / (double)run) : 1.0;
  const double single = 22.0 + 8.28e-9 * flops * narrow + 0.108e-6 * 4.0 * (double)(M + columns) * terms;
  return parts < 0.92 * single && pl.m_tiles * pl.n_tiles < (1 << 24);
}

namespace {

int run_product(ProductParams &p, int tag, const char *name) {
  Runtime &rt = runtime();
  hipStream_t s = rt.stream;
  const int cus = rt.props.multiProcessorCount;
  p.steps = (int)ceil_div(p.octets, 4);
  const ProductPlan pl = plan_product(p.M, p.columns, p.steps);
  p.m_tiles = (int)pl.m_tiles, p.tiles = (int)(pl.m_tiles * pl.n_tiles);
  p.full_tiles = (int)pl.full_tiles, p.share_blocks = pl.share_blocks;
  if (p.share_blocks > 0) {
    const int all = (p.tiles - p.full_tiles) * p.steps;
    p.share_steps = all / p.share_blocks, p.share_extra = all % p.share_blocks;
  }
  p.a_panels = (int)pl.m_tiles * (pl.tall ? 2 : 1), p.b_panels = (int)pl.n_tiles * (pl.tall ? 1 : 2);
  const size_t panel_bytes = (size_t)p.steps * kProductPanelBytes;
  const size_t note_bytes = ((size_t)(p.a_panels + p.b_panels) * p.steps * 4 + 255) & ~size_t(255);
  p.marks = 1 + (int)ceil_div(p.tiles, 32);
  const size_t mark_bytes = ((size_t)p.marks * 4 + 255) & ~size_t(255);
  const size_t partial_bytes = (size_t)p.share_blocks * 2 * 2 * kProductPanel * kProductPanel * 4;
  void *scratch = nullptr;
  if (workspace_or_less((p.a_panels + p.b_panels) * panel_bytes + note_bytes + mark_bytes + partial_bytes, &scratch)) return MG_ERR_UNSUPPORTED;  // the kernels that need less stay
  char *at = static_cast<char *>(scratch);
  p.packed_a = at, at += p.a_panels * panel_bytes;
  p.packed_b = at, at += p.b_panels * panel_bytes;
  p.notes = reinterpret_cast<unsigned *>(at), at += note_bytes;
  p.redo = reinterpret_cast<unsigned *>(at), at += mark_bytes;
  p.partial = reinterpret_cast<float *>(at);
  static char note[160];  // (behind the lock of the entry points)
  snprintf(note, sizeof note, "%s: tile %dx%dx32, %d column tiles x %d row tiles, %d whole tiles, the rest shared by %d blocks, three bf16 parts", name,
           pl.tall ? 256 : 128, pl.tall ? 128 : 256, (int)pl.n_tiles, (int)pl.m_tiles, p.full_tiles, p.share_blocks);
  note_plan(note);
  {
    ScopedTiming timed(TAG_PACK_FILTERS);
    hipLaunchKernelGGL(product_pack_kernel, dim3((unsigned)p.steps, (unsigned)(p.a_panels + p.b_panels)), dim3(256), 0, s, p);
    MG_HIP(hipGetLastError());
  }
  ScopedTiming timed(tag);
  static const hipError_t allowed = [] {
    const hipError_t first = hipFuncSetAttribute((const void *)product_gemm_kernel<2, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kProductLds);
    return first != hipSuccess ? first : hipFuncSetAttribute((const void *)product_gemm_kernel<1, 2>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kProductLds);
  }();
  MG_HIP(allowed);
  const dim3 grid((unsigned)(p.full_tiles > 0 ? cus : p.share_blocks));
  const int fix_blocks = (p.tiles - p.full_tiles) * kFixBlocks;
#define MG_PRODUCT(PM, PN)                                                                \
  hipLaunchKernelGGL((product_gemm_kernel<PM, PN>), grid, dim3(512), kProductLds, s, p);   \
  hipLaunchKernelGGL((product_finish_kernel<PM, PN>), dim3((unsigned)(fix_blocks + kProductRedoBlocks)), dim3(256), 0, s, p, fix_blocks);
  if (pl.tall) {
    MG_PRODUCT(2, 1)
  } else {
    MG_PRODUCT(1, 2)
  }
#undef MG_PRODUCT
  MG_HIP(hipGetLastError());
  return MG_OK;
}

}  // namespace

int product_forward(long long batch, long long M, long long K, long long N, const void *a, const void *x, void *out) {
  ProductParams p{};
  p.a = operand_of(a, 1, M, 0, K, K, 0, 1);
  p.b = operand_of(x, batch, N, K * N, 1, K, 0, N);
  p.octets = (int)ceil_div(K, 8);
  p.dst = static_cast<float *>(out), p.M = (int)M, p.columns = (int)(batch * N), p.by_n = make_fastdiv((unsigned)N);
  p.dst_batch = M * N, p.dst_mstride = N;
  return run_product(p, TAG_CONV_FWD, "matmul");
}

int product_da(long long batch, long long M, long long K, long long N, const void *grad, const void *x, void *da) {
  ProductParams p{};
  p.a = operand_of(grad, 1, M, 0, N, N, M * N, 1);
  p.b = operand_of(x, 1, K, 0, N, N, K * N, 1);
  p.octets = (int)(batch * ceil_div(N, 8));
  p.dst = static_cast<float *>(da), p.M = (int)M, p.columns = (int)K, p.by_n = make_fastdiv((unsigned)K);
  p.dst_batch = 0, p.dst_mstride = K;
  return run_product(p, TAG_CONV_WGRAD, "matmul_da");
}

int product_dx(long long batch, long long M, long long K, long long N, const void *grad, const void *a, void *dx) {
  ProductParams p{};
  p.a = operand_of(a, 1, K, 0, 1, M, 0, K);
  p.b = operand_of(grad, batch, N, M * N, 1, M, 0, N);
  p.octets = (int)ceil_div(M, 8);
  p.dst = static_cast<float *>(dx), p.M = (int)K, p.columns = (int)(batch * N), p.by_n = make_fastdiv((unsigned)N);
  p.dst_batch = K * N, p.dst_mstride = N;
  return run_product(p, TAG_CONV_DGRAD, "matmul_dx");
}

}  // namespace mg
