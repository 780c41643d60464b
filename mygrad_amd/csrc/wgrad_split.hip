// Filter gradients of large problems in single precision on the bf16 matrix instructions: see conv_split.hip for the
// arithmetic, its accuracy (two accumulators) and what parts cannot represent.
#include "wgrad_split.h"
#include "internal.h"
#include "split_device.h"
#include "wgrad_sums.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <utility>

namespace mg {

namespace {

constexpr int kFrags = kWgradSplitFrags, kColumns = kFrags * 16;
constexpr int kSumStride = kColumns + 4;  // floats between the filters of a tile's sums in LDS
constexpr int kSums = 8 * 32 * kSumStride;  // floats of them: eight waves of 32 filters
constexpr int kMiddle = 4;  // taps of a stage ahead of which the second half of the waves parks
constexpr int kLoc = 48;                  // pieces of 16 bytes of 16 channels at one location: [part][channel]
constexpr int kDump = 3 * kLoc + 2 * 16 + 16;  // pieces behind the rings for what nobody reads

// f(0), f(1), ... with the counts as types: unrolled whatever its size
template <typename F, int... I>
__device__ __forceinline__ void unrolled(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
#define MG_INLINE __attribute__((always_inline))

// A column tile: 16 channels, a tap of axis 0, some taps of axes 1 and 2.
struct Columns {
  int cgroup, t0, tap, taps;
};
__device__ __forceinline__ Columns columns_of(const WgradSplitParams &p, int i) {
  const int chunk = i % p.chunks, rest = i / p.chunks;
  return Columns{rest / p.W[0], rest % p.W[0], chunk * kFrags, min(kFrags, p.W[1] * p.W[2] - chunk * kFrags)};
}

// What this wave wrote to LDS is there, and what it read is in registers; then all waves of the block are here.
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int FW, int CW, int KW, int TASKS, bool ALONG>
__global__ void __launch_bounds__(512, 2) wgrad_split_kernel(const WgradSplitParams p) {
  static_assert(FW * CW * KW == 8, "eight waves of 32 filters by a column tile");
  constexpr int FT = 32 * FW;
  constexpr int kOwnLow = TASKS == 1 ? kFrags : 4;  // taps whose small products have sums of their own
  extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
  constexpr int GRAD = KW * 4 * 2 * FW * kLoc;  // pieces of grad: [16 filters][position][part][filter]; then the column tiles' rings [row][location][part][channel]
  const int lane = (int)threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4, wave = uniform((int)threadIdx.x >> 6);
  const int fw = wave / (CW * KW), cw = wave / KW % CW, kq = wave % KW;
  const int grid = (int)gridDim.x, xcd = (int)(blockIdx.x & 7), place = xcd * (grid / 8) + min(xcd, grid % 8) + (int)(blockIdx.x >> 3);
  const int tile = place % p.tiles, split = place / p.tiles, f0 = tile % p.f_tiles * FT, first_columns = tile / p.f_tiles * CW;
  const int first_stage = (int)(p.total * split / p.splits), last_stage = (int)(p.total * (split + 1) / p.splits);
  const int row_pieces = p.row_locs * kLoc, group_pieces = p.new_rows * row_pieces, ring_pieces = (p.depth + 2) * group_pieces;

  // ---- What is loaded, split and parked for a tick: tasks of a wave, four locations (of a row of x, of a ring's next group) or
  // positions (of grad, of the next stage) of 16 channels or filters a lane group, of four of the eight segments a lane.
  constexpr int GTASKS = 8 / CW;
  const int xtasks = (p.new_rows * p.x_quads + 1) / 2;
  const int half = lk & 1;
  struct Task {
    bool is_x, active;
    int urow, ucol, t0, tap1;
    unsigned channel_at;  // bytes
    int put, put_group;   // pieces
  };
  Task tasks[TASKS];
  bool has[TASKS];
#pragma unroll
  for (int s = 0; s < TASKS; ++s) {
    Task &t = tasks[s];
    const int number = wave + 8 * s;
    has[s] = number < GTASKS + CW * xtasks;
    t.is_x = number >= GTASKS;
    if (t.is_x) {
      const int of = min((number - GTASKS) / xtasks, CW - 1), slot = (number - GTASKS - of * xtasks) * 2 + (lk >> 1);
      const Columns c = columns_of(p, min(first_columns + of, p.columns - 1));
      const int channel = c.cgroup * 16 + l16;
      t.urow = slot / p.x_quads, t.ucol = slot % p.x_quads * 4, t.t0 = c.t0, t.tap1 = c.tap / p.W[2];
      const bool room = t.urow < p.new_rows && has[s];
      t.active = room && channel < p.C && first_columns + of < p.columns;
      t.channel_at = (unsigned)channel * (unsigned)(p.X[0] * p.X[1] * p.X[2]) * 4u;
      t.put = GRAD + (room ? of * ring_pieces + t.urow * row_pieces + t.ucol * kLoc : CW * ring_pieces) + l16;
      t.put_group = room ? group_pieces : 0;
    } else {
      const int slot = number * 2 + (lk >> 1), filter = f0 + slot / KW * 16 + l16;
      t.urow = slot % KW / p.quads, t.ucol = slot % KW % p.quads * 4, t.t0 = 0, t.tap1 = 0;
      t.active = filter < p.F;
      t.channel_at = (unsigned)filter * (unsigned)(p.G[0] * p.G[1] * p.G[2]) * 4u;
      t.put = (slot / KW * 4 * KW + slot % KW * 4) * kLoc + l16;
      t.put_group = 0;
    }
  }

  // ---- Ticks: the walks of the block's stages one after the other, each with `depth` ticks ahead of its first stage that
  // only fill the rings.  Of the tick that is requested next: what is left of its walk, ticks that only fill, the stage that
  // begins the next walk.
  int ticks = 0;
  for (int stage = first_stage; stage < last_stage;) {
    const int in_walk = min(p.stages - stage % p.stages, last_stage - stage);
    ticks += in_walk + p.depth, stage += in_walk;
  }
  const int all_ticks = ticks;
  int to_request = ticks, left = 0, filling = 0, next_stage = first_stage, octet = 0, strip = 0;
  // Of the walk, segment by segment of the thread: byte offset in its first tick, and the place (row; ALONG: column) whose
  // distance from the walk's beginning decides whether four columns are there at all.
  unsigned walk_at[TASKS][4];
  int walk_row[TASKS], walk_col[TASKS][4];  // (walk_col: ALONG only)
  int moved[TASKS];                         // rows or columns from the walk's first tick on
  int whole[TASKS];                         // how far it is to four columns that are cut off by the end of their row; 0: the walk begins with some
  // first column of segment e of the thread, and the end of what is there
  auto columns_at = [&](const Task &t, int e, int &end) MG_INLINE -> int {
    const int seg = octet * 8 + half * 4 + e, begin = (seg & ((1 << p.seg_shift) - 1)) * p.seg_len;
    end = t.is_x ? p.X[2] : min(begin + p.seg_len, p.G[2]);
    const int col = begin + strip * p.quads * 4;
    return t.is_x ? col * p.S[2] + t.ucol - p.P[2] : col + t.ucol;
  };
  auto enter_walk = [&]() MG_INLINE {
    const int walk = next_stage / p.stages, stage = next_stage - walk * p.stages, in_walk = min(p.stages - stage, last_stage - next_stage);
    left = in_walk + p.depth, filling = p.depth, next_stage += in_walk;
    octet = ALONG ? walk : walk / p.strips, strip = ALONG ? stage : walk - octet * p.strips;
#pragma unroll
    for (int s = 0; s < TASKS; ++s) {
      const Task &t = tasks[s];
      const int extent1 = t.is_x ? p.X[1] : p.G[1], extent2 = t.is_x ? p.X[2] : p.G[2], row = ALONG ? 0 : stage;
      walk_row[s] = t.is_x ? t.urow + row * p.new_rows + t.tap1 * p.D[1] - p.P[1] : t.urow + (row - p.depth) * p.rows;
      moved[s] = 0;
      int room = 1 << 30;
      bool begins = false;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int end;
        const int col = columns_at(t, e, end), plane = (octet * 8 + half * 4 + e) >> p.seg_shift;
        const int n = (int)p.by_g0.div((unsigned)plane), g0 = plane - n * p.G[0];
        const int x0 = t.is_x ? g0 * p.S[0] + t.t0 * p.D[0] - p.P[0] : g0, extent0 = t.is_x ? p.X[0] : p.G[0];
        const bool there = t.active && (unsigned)x0 < (unsigned)extent0 && (!ALONG || (unsigned)walk_row[s] < (unsigned)extent1);
        const bool real = there && (ALONG || (col > -4 && col < end));
        // (four columns that begin ahead of their row are loaded from its first one on, and moved: see park)
        const int at = ((n * (t.is_x ? p.C : p.F) * extent0 + x0) * extent1 + walk_row[s]) * extent2 + (ALONG ? col : max(col, 0));
        walk_at[s][e] = real ? t.channel_at + (unsigned)at * 4u : kOutside;
        if constexpr (ALONG) walk_col[s][e] = there ? col + 3 + extent2 - end : 1 << 30;
        if (real) room = min(room, max(end - 3 - col, 0));
        begins |= real && col < 0;
      }
      for (int step = 1; step < 64; step *= 2) room = min(room, __shfl_xor(room, step));
      whole[s] = __any(begins) ? 0 : ALONG ? uniform(room) : uniform(room) > 0 ? 1 << 30 : 0;
    }
  };

  u32x4 raw[TASKS][4];
  // moves on to the next tick
  unsigned tick_bytes[TASKS], tick_limit[TASKS];
  auto advance = [&]() MG_INLINE {
    const bool walks = left == 0 && to_request > 0;
    if (walks) enter_walk();
#pragma unroll
    for (int s = 0; s < TASKS; ++s) {
      const Task &t = tasks[s];
      if (!walks) moved[s] += ALONG ? p.quads * 4 * (t.is_x ? p.S[2] : 1) : t.is_x ? p.new_rows : p.rows;
      const int extent1 = t.is_x ? p.X[1] : p.G[1], extent2 = t.is_x ? p.X[2] : p.G[2];
      // (there is nothing behind the last tick, and no grad ahead of a walk's first stage)
      const bool some = to_request > 0 && (t.is_x || filling <= 0);
      const int row = walk_row[s] + moved[s];
      tick_limit[s] = ALONG ? (some ? (unsigned)(extent2 + 3) : 0u) : (unsigned)row < (some ? (unsigned)extent1 : 0u) ? 0u : kOutside;
      tick_bytes[s] = (unsigned)moved[s] * (ALONG ? 4u : (unsigned)extent2 * 4u);
    }
    --left, --filling, --to_request;
  };
  // requests segment e of its four
  auto request = [&](int e) MG_INLINE {
#pragma unroll
    for (int s = 0; s < TASKS; ++s) {
      const Task &t = tasks[s];
      const __amdgpu_buffer_rsrc_t from = t.is_x ? buffer_of(p.x, p.x_bytes) : buffer_of(p.grad, p.grad_bytes);
      unsigned at = walk_at[s][e] + tick_bytes[s], outside = tick_limit[s];
      if constexpr (ALONG) {
        const int col = walk_col[s][e] + moved[s];
        outside = (unsigned)col < tick_limit[s] ? 0u : kOutside;
        // (in any tick of a walk that begins ahead of a row: with more padding than a tick has columns, a later one meets the row's first)
        if (whole[s] == 0) at += (unsigned)max(3 - col, 0) * 4u;
      }
      raw[s][e] = __builtin_amdgcn_raw_buffer_load_b128(from, (int)(at | outside), 0, 0);
    }
  };
  auto request_all = [&]() MG_INLINE {
#pragma unroll
    for (int e = 0; e < 4; ++e) request(e);
  };
  // what lies outside of a task's rows, among what was requested, is zero
  auto clear_outside = [&](int s) MG_INLINE {
    if ((ALONG ? moved[s] : 1) < whole[s]) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int end;
      const int col = columns_at(tasks[s], e, end) + (ALONG ? moved[s] : 0);
      u32x4 v = raw[s][e];
      v = col < 0 && (col & 1) != 0 ? u32x4{0, v[0], v[1], v[2]} : v;
      v = col < 0 && ((-col) & 2) != 0 ? u32x4{0, 0, v[0], v[1]} : v;
#pragma unroll
      for (int u = 0; u < 4; ++u) raw[s][e][u] = col + u < end ? v[u] : 0u;
    }
  };
  unsigned lost = 0;
  // splits and parks what was requested
  auto park = [&](int group) MG_INLINE {
#pragma unroll
    for (int s = 0; s < TASKS; ++s) {
      if (!has[s]) continue;
      const Task &t = tasks[s];
      clear_outside(s);
      u32x2 *const to = reinterpret_cast<u32x2 *>(lds + t.put + group * t.put_group) + half;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        u32x2 parts[3];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          unsigned h, m, l;
          split_pair(float_of(raw[s][2 * e][u]), float_of(raw[s][2 * e + 1][u]), h, m, l, lost);
          parts[0][e] = h, parts[1][e] = m, parts[2][e] = l;
        }
#pragma unroll
        for (int part = 0; part < 3; ++part) to[(u * kLoc + part * 16) * 2] = parts[part];
      }
    }
  };

  // ---- operands of a stage
  const Columns mine = columns_of(p, min(first_columns + cw, p.columns - 1));
  const int rr = kq / p.quads, cq = kq % p.quads;
  const u32x4 *const grads = lds + (fw * 2 * 4 * KW + kq * 4 + lk) * kLoc + l16;
  const u32x4 *const locs = lds + GRAD + cw * ring_pieces + (cq * 4 + lk) * p.S[2] * kLoc + l16;
  u32x4 g[2][3], x[4];  // (the first part of x, which is used last, in x[0] and x[3] in turn)
  auto read_grad = [&](int part) MG_INLINE {
#pragma unroll
    for (int i = 0; i < 2; ++i) g[i][part] = grads[i * 4 * KW * kLoc + part * 16];
  };
  // the tap whose operands are read: its column in the window, and its offset from the stage's first row (frags beyond the
  // tile's taps read what is there)
  const int tap_step = p.D[2] * kLoc, row_step = p.D[1] * row_pieces, first_col = mine.tap % p.W[2];
  int base = 0, tap_col = 0, tap_loc = 0;
  const u32x4 *from = locs;
  auto first_tap = [&](int group) MG_INLINE {  // of the stage whose last rows are in `group`
    int first = group - p.depth;
    first += first < 0 ? p.depth + 2 : 0;
    base = first * group_pieces + rr * p.S[1] * row_pieces;
    base -= base >= ring_pieces ? ring_pieces : 0;
    tap_col = first_col, tap_loc = first_col * tap_step;
    from = locs + base + tap_loc;
  };
  auto next_tap = [&]() MG_INLINE {
    const bool turn = tap_col + 1 == p.W[2];
    tap_col = turn ? 0 : tap_col + 1;
    tap_loc = turn ? 0 : tap_loc + tap_step;
    base += turn ? row_step : 0;
    base -= base >= ring_pieces ? ring_pieces : 0;
    from = locs + base + tap_loc;
  };
  auto read_x = [&](int part, int j) MG_INLINE { x[part == 0 && j % 2 != 0 ? 3 : part] = from[part * 16]; };

  // Sums of the large products; those of the five small ones, of the first kOwnLow taps over all stages and of the others
  // of a stage's, added one tap later (two accumulators for every tap do not fit 256 registers).
  f32x4 acc[kFrags][2], low[kOwnLow][2], small[2][2];
#pragma unroll
  for (int j = 0; j < kFrags; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      acc[j][i] = f32x4{0, 0, 0, 0};
      if (j < kOwnLow) low[j][i] = f32x4{0, 0, 0, 0};
    }

  if (ticks > 0) {
    // (what no tick has filled yet meets zeros of grad, and must not be a NaN)
    for (int i = (int)threadIdx.x; i < CW * ring_pieces; i += 512) lds[GRAD + i] = u32x4{0, 0, 0, 0};
    __syncthreads();
    advance();
    request_all();
    park(0);
    advance();
    request_all();
    meet();
    first_tap(0);
#pragma unroll
    for (int part = 0; part < 3; ++part) read_grad(part), read_x(part, 0);
    // Waves 0 - 3, one on each SIMD, split and park ahead of a stage's products, waves 4 - 7 in the middle of them: what one
    // wave of a SIMD does on the vector ALU then runs beside the other's products.
    int group = 1;  // of the rings, of the tick that is parked next
    for (; ticks > 0; --ticks) {
        unrolled(
            [&](auto tap) MG_INLINE {
              constexpr int j = decltype(tap)::value, LAST = kFrags - 1;
              if constexpr (j == 0) meet();  // everyone has read grad of this stage
              if constexpr (j == 0 || j == kMiddle) {
                if ((wave < 4) == (j == 0)) {
                  park(group);
                  advance();
                  request_all();
                }
              }
              if constexpr (j == LAST) {
                meet();  // the next stage is there
                first_tap(group);
              }
              // smallest first, nearly; the last tap's order frees first what the next stage uses first
              constexpr int order = j == LAST;
              constexpr int PX[2][6] = {{2, 1, 1, 0, 0, 0}, {0, 1, 2, 1, 0, 0}}, PG[2][6] = {{0, 1, 0, 2, 1, 0}, {0, 0, 0, 1, 1, 2}};
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int t = 0; t < 6; ++t) {
                const int px = PX[order][t], pg = PG[order][t];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                  f32x4 &into = px + pg == 0 ? acc[j][i] : j < kOwnLow ? low[j < kOwnLow ? j : 0][i] : small[j % 2][i];
                  const f32x4 onto = t == order && j >= kOwnLow ? f32x4{0, 0, 0, 0} : into;
                  into = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[px == 0 && j % 2 != 0 ? 3 : px]),
                                                                 __builtin_bit_cast(bf16x8, g[i][pg]), onto, 0, 0, 0);
                }
                if constexpr (j > kOwnLow) {
                  if (t == 2 || t == 3) acc[j - 1][t - 2] += small[(j - 1) % 2][t - 2];
                }
                if (j != LAST) {
                  if (t == 0) next_tap();
                  if (t == 0) read_x(0, j + 1), read_x(2, j + 1);
                  if (t == 2) read_x(1, j + 1);
                } else {
                  if (t == 2) read_grad(0), read_x(2, 0);
                  if (t == 3) read_x(1, 0);
                  if (t == 4) read_grad(1);
                  if (t == 5) read_grad(2), read_x(0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
              }
            },
            std::make_integer_sequence<int, kFrags>());
        if constexpr (kOwnLow < kFrags) {
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[kFrags - 1][i] += small[(kFrags - 1) % 2][i];
        }
        if (++group == p.depth + 2) group = 0;
    }
  }

  // ---- the sums of the waves along K, added in order: acc[j][i][q] is filter 32 fw + 16 i + l16, channel 4 lk + q of frag j
  __syncthreads();
  float *const sums = reinterpret_cast<float *>(lds);
#pragma unroll
  for (int j = 0; j < kFrags; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f32x4 sum = j < kOwnLow ? acc[j][i] + low[j < kOwnLow ? j : 0][i] : acc[j][i];
      *reinterpret_cast<f32x4 *>(sums + (((kq * CW + cw) * FT + fw * 32 + i * 16 + l16) * kSumStride + j * 16 + lk * 4)) = sum;
    }
  constexpr int ROWS = FT + CW * 16;  // filters, then channels
  unsigned *const notes = reinterpret_cast<unsigned *>(sums + kSums), *const waves = notes + 2 * ROWS;
  const bool own_lost = __any((lost & 0xffffu) != 0);
  if (lane == 0) waves[wave] = own_lost;
  __syncthreads();
  bool any = false;
#pragma unroll
  for (int w = 0; w < 8; ++w) any |= waves[w] != 0;
  // Seldom: a second look at the block's values, for the widest of every filter and channel, and whether it has lost bits.  (64 channels, 3 x 3, 56 x 56:
  // 166 us without a lost bit, 219 - 225 with one, 305 with some in every block, 390 - 410 where any sent the gradient to the
  // single-precision kernel.  With the widest values kept along the way all take 169, and the layers along one axis 3 % more.)
  if (any) {
    for (int i = (int)threadIdx.x; i < 2 * ROWS; i += 512) notes[i] = 0;
    float widest[TASKS];
    unsigned low[TASKS];
#pragma unroll
    for (int s = 0; s < TASKS; ++s) widest[s] = 0.0f, low[s] = 0;
    to_request = all_ticks, left = 0, next_stage = first_stage;
    while (to_request > 0) {
      advance();
      request_all();
#pragma unroll
      for (int s = 0; s < TASKS; ++s) {
        clear_outside(s);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int u = 0; u < 4; u += 2) {
            const float a = float_of(raw[s][e][u]), b = float_of(raw[s][e][u + 1]);
            unsigned h, m, l;
            split_pair(a, b, h, m, l, low[s]);
            widen(widest[s], a, b);
          }
      }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < TASKS; ++s) {
      if (!has[s]) continue;
      const int number = wave + 8 * s, row = tasks[s].is_x ? FT + min((number - GTASKS) / xtasks, CW - 1) * 16 + l16 : (number * 2 + (lk >> 1)) / KW * 16 + l16;
      atomicMax(&notes[row], bits_of(widest[s]));
      if ((low[s] & 0xffffu) != 0) atomicOr(&notes[ROWS + row], 1u);
    }
    __syncthreads();
  }
  float *const out = p.partial + (long long)(split * p.tiles + tile) * (CW * FT * kColumns);
  bool odd = false;  // a sum is not finite, or smaller than what lost bits can have been worth
  const int terms = (last_stage - first_stage) * (KW * 4 * 8);
  for (int e = (int)threadIdx.x; e < CW * FT * kColumns / 4; e += 512) {
    const int f = e / (kColumns / 4), c = e % (kColumns / 4) * 4;  // (f: column tile, filter)
    f32x4 sum = *reinterpret_cast<const f32x4 *>(sums + f * kSumStride + c);
#pragma unroll
    for (int k = 1; k < KW; ++k) sum += *reinterpret_cast<const f32x4 *>(sums + (k * CW * FT + f) * kSumStride + c);
    *reinterpret_cast<f32x4 *>(out + f * kColumns + c) = sum;
    const bool live = c / 16 < columns_of(p, first_columns + f / FT).taps;
#pragma unroll
    for (int q = 0; q < 4; ++q) odd |= !(__builtin_fabsf(sum[q]) < __builtin_inff()) && live;
    if (any && live) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int g = f % FT, x = FT + f / FT * 16 + c % 16 + q;
        odd |= !(__builtin_fabsf(sum[q]) >= least_sum(notes[ROWS + g] != 0, float_of(notes[g]), notes[ROWS + x] != 0, float_of(notes[x]), terms));
      }
    }
  }
  if (__any(odd) && lane == 0) atomicOr(&p.words[0], 1u);
}

// dw from the partial sums, in the order of the splits (four runs of them at a time): those of the parts, or of the
// single-precision kernel where they cannot be used.
template <int FW, int CW>
__global__ void __launch_bounds__(256) wgrad_split_reduce_kernel(const WgradSplitParams p, const WgradSums single) {
  constexpr int FT = 32 * FW, TILE = CW * FT * kColumns;
  __shared__ float runs[4][64];
  const int t = (int)threadIdx.x, q = t / 64, e = (int)blockIdx.x * 64 + t % 64;
  if (p.words[0] == 0) {
    const long long stride = (long long)p.tiles * TILE;
    const int per = (p.splits + 3) / 4, first = min(q * per, p.splits), last = min(first + per, p.splits);
    runs[q][t % 64] = first < last ? sum_in_order(p.partial + first * stride + e, stride, last - first) : 0.0f;
    __syncthreads();
    const int tile = e / TILE, within = e % TILE, columns = tile / p.f_tiles * CW + within / (FT * kColumns);
    if (q == 0 && columns < p.columns) {
      float sum = runs[0][t];
#pragma unroll
      for (int r = 1; r < 4; ++r) sum += runs[r][t];
      const Columns at = columns_of(p, columns);
      const int f = tile % p.f_tiles * FT + within / kColumns % FT, frag = e % kColumns / 16, c = at.cgroup * 16 + e % 16;
      if (f < p.F && c < p.C && frag < at.taps) p.dw[((long long)f * p.C + c) * p.wvol + at.t0 * p.W[1] * p.W[2] + at.tap + frag] = sum;
    }
  } else if (single.partial != nullptr) {
    reduce_single(single, p.dw, p.F, p.C, p.wvol);
  }
  leave_words(p.words);
}

// waves along filters, column tiles and K; tasks of a wave
#define MG_WGRAD_SHAPES(X) \
  X(2, 2, 2, 1, false) X(2, 2, 2, 2, false) X(1, 2, 4, 2, false) X(4, 2, 1, 2, false) X(1, 1, 8, 2, false) X(2, 2, 2, 1, true) X(1, 1, 8, 2, true) X(1, 2, 4, 2, true)
struct WgradShape {
  int fw, cw, kw, tasks;
  bool along;
};
#define MG_SHAPE(FW, CW, KW, TASKS, ALONG) {FW, CW, KW, TASKS, ALONG},
constexpr WgradShape kWgradShapes[] = {MG_WGRAD_SHAPES(MG_SHAPE)};
#undef MG_SHAPE

constexpr int kLds = 160 * 1024;

size_t lds_bytes(const WgradSplitPlan &pl) {
  const size_t rings = (size_t)pl.cw * (pl.p.depth + 2) * pl.p.new_rows * pl.p.row_locs * kLoc;
  return std::max<size_t>((pl.kw * 4 * 2 * pl.fw * kLoc + rings + kDump) * 16, (size_t)(kSums + 2 * (32 * pl.fw + 16 * pl.cw) + 8) * 4);
}

}  // namespace

// Every shape of the kernel and split of K that the problem fits, by modelled time, in us: fitted to 1700 timed (filter gradient,
// shape, quads) of 480 layers drawn over the range of sizes, 8 in 10 within 9 % of it; what it chooses is 0.5 % slower than the best
// in the mean.  A tick takes 2.1 - 3.3 us; one quad a row, of several to a stage, is left out: lines of memory are then touched by
// eight walks, up to twice the modelled time.  Where a stage is one quad (wide patches: strides), what it takes is the lines, 128 bytes each,
// that its sixteen bytes a row lie in, at 8 TB/s, where that is more: 9 in 10 of 77 layers within 14 % of it, two thirds more than modelled without
// ((128,64,55,55) * (128,64,3,3) stride 2: 104 us modelled, 152 measured, 139 on the single-precision kernel).
WgradSplitPlan plan_wgrad_split(int N, int C, int F, const int *X, const int *G, const int *W, const int *S, const int *D, const int *P, int cus) {
  WgradSplitPlan best;
  // MYGRAD_HIP_SPLIT_TILE="waves along filters,column tiles,quads of a row" (tests; part of the plan's key)
  int want[3] = {0, 0, 0};
  if (const char *v = getenv("MYGRAD_HIP_SPLIT_TILE")) sscanf(v, "%d,%d,%d", &want[0], &want[1], &want[2]);
  for (const WgradShape &shape : kWgradShapes)
    for (int quads = shape.kw; quads >= 1; quads /= 2) {
      if (want[0] != 0 ? shape.fw != want[0] || shape.cw != want[1] || quads != want[2] : quads == 1 && shape.kw > 1) continue;
      if (shape.along != (G[1] == 1) || (shape.along && quads != shape.kw)) continue;
      WgradSplitPlan pl;
      pl.fw = shape.fw, pl.cw = shape.cw, pl.kw = shape.kw, pl.tasks = shape.tasks, pl.along = shape.along;
      WgradSplitParams &p = pl.p;
      for (int k = 0; k < 3; ++k) p.X[k] = X[k], p.G[k] = G[k], p.W[k] = W[k], p.S[k] = S[k], p.D[k] = D[k], p.P[k] = P[k];
      p.C = C, p.F = F, p.wvol = W[0] * W[1] * W[2];
      p.kpos = N * G[0] * G[1] * G[2];
      const int planes = N * G[0], taps = W[1] * W[2];
      while ((planes << p.seg_shift) % 8 != 0) ++p.seg_shift;
      p.quads = quads, p.rows = pl.kw / quads;
      p.seg_len = (int)ceil_div(ceil_div(G[2], 1 << p.seg_shift), 4) * 4;
      p.by_g0 = make_fastdiv((unsigned)G[0]);
      p.octets = (planes << p.seg_shift) / 8;
      p.strips = (int)ceil_div(std::min(p.seg_len, G[2]), 4 * quads);
      p.stages = (int)ceil_div(G[1], p.rows);
      if (pl.along) p.stages = p.strips, p.strips = 1;
      p.chunks = (int)ceil_div(taps, kFrags);
      int tap_rows = 0;
      for (int c = 0; c < p.chunks; ++c) tap_rows = std::max(tap_rows, std::min(taps - 1, (c + 1) * kFrags - 1) / W[2] - c * kFrags / W[2] + 1);
      const long long live = (p.rows - 1ll) * S[1] + (tap_rows - 1ll) * D[1] + 1, locs = (4ll * quads - 1) * S[2] + (W[2] - 1ll) * D[2] + 1;
      if (live > 64 || locs > 64) continue;  // (far more than LDS holds)
      p.new_rows = pl.along ? (int)live : p.rows * S[1];
      p.depth = std::max(0, (int)ceil_div(live - p.new_rows, p.new_rows));
      p.row_locs = (int)ceil_div(locs, 4) * 4, p.x_quads = p.row_locs / 4;
      const int tasks = 8 / pl.cw + pl.cw * (int)ceil_div(p.new_rows * p.x_quads, 2);
      if (ceil_div(tasks, 8) != pl.tasks || lds_bytes(pl) > (size_t)kLds) continue;
      p.columns = (int)ceil_div(C, 16) * W[0] * p.chunks, p.f_tiles = (int)ceil_div(F, 32 * pl.fw);
      const long long tiles = ceil_div(p.columns, pl.cw) * p.f_tiles;
      p.tiles = (int)tiles;
      p.total = (long long)p.octets * p.strips * p.stages;
      if (p.total >= 1ll << 30 || tiles >= 1ll << 16) continue;
      double lines_time = 0;
      if (quads == 1) {
        const int planes_of = 8 >> std::min(p.seg_shift, 3), runs = 8 / planes_of;  // of an octet; of a row
        auto lines = [&](int run, int row) { return planes_of * std::min(runs * (1 + (run * 4 - 4) / 128.0), row * 4 / 128.0 + 1); };
        lines_time = 0.12e-6 * 128 * (double)p.total *
                     (F * lines(4, G[2]) + std::min(C, 16 * pl.cw) * (double)ceil_div(p.columns, pl.cw) * lines(4 * p.x_quads, X[2]) * p.new_rows * (1 + (double)p.depth / p.stages));
      }
      const long long most = std::min<long long>(p.total, std::max<long long>(1, 6 * cus / tiles));
      for (long long splits = 1; splits <= most; ++splits) {
        const double rounds = (double)ceil_div(splits * tiles, cus), stages = (double)ceil_div(p.total, splits);
        const double walks = p.total % (splits * p.stages) == 0 ? stages / p.stages : stages / p.stages + 1.0;
        const double tick = 1.19 + 0.121 * tasks + 0.065 * pl.cw * p.new_rows;
        const double traffic = (double)(splits * tiles) * (32 * pl.fw * pl.cw * kColumns) * 8e-6;  // of the partial sums, MB
        pl.time = 11.9 + rounds * (11.6 + 0.98 * walks) + std::max(lines_time, rounds * (stages + walks * p.depth) * tick) + 0.102 * traffic;
        p.splits = (int)splits;
        if (best.fw == 0 || pl.time < best.time) best = pl;
      }
    }
  return best;
}

size_t wgrad_split_scratch(const WgradSplitPlan &pl) {
  return ((size_t)pl.p.tiles * pl.p.splits * 32 * pl.fw * pl.cw * kColumns * 4 + 255) & ~size_t(255);
}

int launch_wgrad_split(const WgradSplitPlan &pl, const void *grad, const void *x, void *scratch, unsigned *words, hipStream_t s) {
  WgradSplitParams p = pl.p;
  p.grad = static_cast<const float *>(grad), p.x = static_cast<const float *>(x);
  const size_t samples = (size_t)p.kpos / ((size_t)p.G[0] * p.G[1] * p.G[2]);
  p.x_bytes = (unsigned)(samples * p.C * p.X[0] * p.X[1] * p.X[2] * 4), p.grad_bytes = (unsigned)((size_t)p.kpos * p.F * 4);
  p.words = words, p.partial = static_cast<float *>(scratch);
  ScopedTiming timed(TAG_CONV_WGRAD);
#define MG_WGRAD_SPLIT(FW, CW, KW, TASKS, ALONG)                                                                              \
  if (pl.fw == FW && pl.cw == CW && pl.tasks == TASKS && pl.along == ALONG) {                                                 \
    const auto kernel = wgrad_split_kernel<FW, CW, KW, TASKS, ALONG>;                                                         \
    static const hipError_t allowed = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLds); \
    MG_HIP(allowed);                                                                                                          \
    hipLaunchKernelGGL(kernel, dim3((unsigned)(p.tiles * p.splits)), dim3(512), lds_bytes(pl), s, p);                          \
  }
  MG_WGRAD_SHAPES(MG_WGRAD_SPLIT)
#undef MG_WGRAD_SPLIT
  MG_HIP(hipGetLastError());
  return MG_OK;
}

int launch_wgrad_split_reduce(const WgradSplitPlan &pl, const WgradSums &single, void *dw, void *scratch, unsigned *words, hipStream_t s) {
  WgradSplitParams p = pl.p;
  p.words = words, p.partial = static_cast<float *>(scratch), p.dw = static_cast<float *>(dw);
  ScopedTiming timed(TAG_WGRAD_REDUCE);
  const auto kernel = pl.fw == 4             ? wgrad_split_reduce_kernel<4, 2>
                      : pl.fw == 2           ? wgrad_split_reduce_kernel<2, 2>
                      : pl.cw == 2           ? wgrad_split_reduce_kernel<1, 2>
                                             : wgrad_split_reduce_kernel<1, 1>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(p.tiles * (32 * pl.fw * pl.cw) * kColumns / 64)), dim3(256), 0, s, p, single);
  MG_HIP(hipGetLastError());
  return MG_OK;
}

}  // namespace mg
