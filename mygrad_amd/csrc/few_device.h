// What the kernels of layers with few terms share (few_split.hip, few_wgrad.hip): tiles of positions and patches of x in LDS.
#pragma once

#include "few_split.h"
#include "split_device.h"

namespace mg {

// A tile: sample, first position, its row and (along) column, the end of its positions.
struct FewTile {
  int n, q0, row, col, end;
};
template <int POSITIONS>
__device__ __forceinline__ FewTile few_tile(const FewParams &p, int item) {
  const int n = (int)p.by_sample.div((unsigned)item), rest = item - n * p.sample_tiles;
  if (p.along) {
    const int row = (int)p.by_run.div((unsigned)rest), col = (rest - row * p.run_tiles) * POSITIONS;
    return FewTile{n, row * p.G2 + col, row, col, min(row * p.G2 + col + POSITIONS, (row + 1) * p.G2)};
  }
  const int q0 = rest * POSITIONS;
  return FewTile{n, q0, (int)p.by_row.div((unsigned)q0), 0, min(q0 + POSITIONS, p.gvol)};
}

// Row `line` (of channel line / patch_rows) of the tile's patch into LDS, from byte `patch` on: sixteen bytes a lane (requests are what the
// kernels wait for: 4 bytes a lane, four times as many, took the filter gradient of a 3 x 7 x 7 layer 217 us, 158 so on the same device), the four columns that
// the end of a row cuts by themselves.
__device__ __forceinline__ void few_request_line(const FewParams &p, const FewTile &t, int line, unsigned patch, int lane) {
  const int c = (int)p.by_patch_rows.div((unsigned)line), r = t.row * p.S1 - p.P1 + line - c * p.patch_rows;
  const int first = t.col * p.S2 - p.P2 - p.lead;  // a multiple of four, but for rows of up to 64 columns (lead -1)
  const bool there = (unsigned)r < (unsigned)p.X1;
  const __amdgpu_buffer_rsrc_t x = buffer_of(p.x, there ? p.x_bytes : 0u);
  const unsigned at = there ? (unsigned)(((t.n * p.C + c) * p.X1 + r) * p.X2) * 4u : 0u, to = patch + (unsigned)(line * p.pitch) * 4u;
  if (p.lead < 0) {  // a row that one request a word takes
    const int column = first - 1 + lane;
    if (lane < p.pitch) to_lds<4>(x, (unsigned)column < (unsigned)p.X2 ? (unsigned)column * 4u : kOutside, at, to);
    return;
  }
  const int cut = (p.X2 & ~3) - first;  // patch column of the cut four, if they are
  for (int q = 0; q < p.pitch; q += 256) {
    const int mine = q + lane * 4, column = first + mine;
    if (mine < p.pitch && (mine != cut || (p.X2 & 3) == 0))
      to_lds<16>(x, column >= 0 && column < p.X2 ? (unsigned)column * 4u : kOutside, at, to + (unsigned)q * 4u);
  }
  if ((p.X2 & 3) != 0 && cut >= 0 && cut < p.pitch) {
    if (lane < 4) to_lds<4>(x, lane < (p.X2 & 3) ? (unsigned)(first + cut + lane) * 4u : kOutside, at, to + (unsigned)cut * 4u);
  }
}

}  // namespace mg
