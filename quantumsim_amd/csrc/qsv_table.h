// PTM application for sizes the inline (<= 16 x 16) and the dense 64 x 64 /
// 256 x 256 kernels do not take: qutrit pairs 81 x 81, qutrit + qubit 36 x
// 36, rectangular reductions of such pairs, three qudits, ...
#pragma once

#include "qsv_geom.h"

namespace qsv {

// The targets in PTM axis order (the last one fastest): entry counts and
// element strides on each side.
struct TableGeo {
  int32_t k;
  int32_t din_t[QSV_MAX_TARGETS], dout_t[QSV_MAX_TARGETS];
  int64_t sin_t[QSV_MAX_TARGETS], sout_t[QSV_MAX_TARGETS];
};

// Offset of PTM index e on one side.
__host__ __device__ inline int64_t table_offset(int k, const int32_t* d, const int64_t* st,
                                                int e) {
  int64_t off = 0;
  for (int j = k - 1; j >= 0; --j) {
    off += int64_t(e % d[j]) * st[j];
    e /= d[j];
  }
  return off;
}

// PTM columns a workgroup holds in LDS at a time, and the most 16-row blocks
// of the output it computes.
constexpr int kTableCols = 96;
constexpr int kTableMaxRowBlocks = 6;

// 16-row blocks per workgroup for `dout` outputs: all of them up to 96, else
// equal shares of at most six blocks.
__host__ __device__ inline int table_row_blocks(int dout) {
  const int tiles = (dout + 15) / 16;
  const int shares = (tiles + kTableMaxRowBlocks - 1) / kTableMaxRowBlocks;
  return (tiles + shares - 1) / shares;
}

// LDS slot of PTM element (row r of the workgroup's rows, column kk of the
// chunk): MFMA A-fragment order, k-step major.
__host__ __device__ inline int table_slot(int mb, int r, int kk) {
  return ((kk >> 2) * mb + (r >> 4)) * 64 + (r & 15) + 16 * (kk & 3);
}

// y = P x over `batch` states (g.bs_in / g.bs_out elements apart), state b
// with the row-major device PTM ptm + b * pstride.
int launch_table(int dtype, const Geom& g, uint32_t n_orbits, const TableGeo& tg, const void* in,
                 void* out, const void* ptm, int64_t pstride, uint32_t batch, hipStream_t s);

}  // namespace qsv
