// Any PTM size on the matrix cores (see qsv_table.h): out = P in over the
// orbits, P of dout x din.
//
// A workgroup of eight waves holds up to 96 x 96 of the PTM in LDS in MFMA
// A-fragment order (padded with zeros to whole 16 x 4 fragments); a wave
// takes 16 NB orbits at a time, loads their entries straight from HBM as B
// fragments (lane (n, j) = (l % 16, l / 16): entry 4 s + j of orbit n) and
// writes the accumulators straight back.  Entry offsets are decoded from the
// targets' dims and strides into LDS, so no host table is needed and the
// launch can be captured.  PTMs of more than 96 columns stream through LDS
// in chunks (the waves of a workgroup then walk the tiles together); more
// than 96 rows are shared out over grid.z.
//
// Bound: an 81 x 81 PTM in float64 is 20 flop per byte (24 with the padding
// to 96 x 84), the card's ridge about 12-14: MFMA and HBM both matter.  The
// kernel this replaced kept 16 operands in registers, read the state six
// times for the 81 rows and used the vector units.  Measured in float64:
// 81 x 81 on 8 states of 6 qutrits (34 MB) 379 -> 37 us, 36 x 36 on 10
// qudits (9^6 4^4 entries, 1.1 GB) 1.5 ms -> 0.43 ms (5.1 TB/s).
#include "qsv_table.h"
#include "qsv_mfma.h"

#include <algorithm>

namespace qsv {

constexpr int kTableBlock = 512;

template <typename T, int MB, int NB>
__global__ void __launch_bounds__(kTableBlock)
    k_apply_table(const T* __restrict__ in, T* __restrict__ out, const Geom g,
                  const uint32_t n_orbits, const TableGeo tg, const T* __restrict__ ptm,
                  const int64_t pstride) {
  constexpr int KS = kTableCols / 4, U = 4, ROWS = 16 * MB;
  constexpr uint32_t COLS = 16 * NB;
  typedef typename Mfma<T>::acc Acc;
  __shared__ T As[KS * MB * 64];
  __shared__ int64_t so_in[kTableCols], so_out[ROWS];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, j = lane >> 4;
  const int row0 = blockIdx.z * ROWS;
  in += int64_t(blockIdx.y) * g.bs_in;
  out += int64_t(blockIdx.y) * g.bs_out;
  ptm += int64_t(blockIdx.y) * pstride;

  // columns [c0, c0 + 96) of this workgroup's rows, and their offsets
  auto stage = [&](int c0) {
    const int cols = min(kTableCols, (g.din - c0 + 4 * U - 1) / (4 * U) * (4 * U));
    for (int e = tid; e < ROWS * kTableCols; e += kTableBlock) {
      const int r = e / kTableCols, kk = e % kTableCols;
      if (kk >= cols) continue;
      const bool in_ptm = row0 + r < g.dout && c0 + kk < g.din;
      As[table_slot(MB, r, kk)] = in_ptm ? ptm[int64_t(row0 + r) * g.din + c0 + kk] : T(0);
    }
    for (int e = tid; e < kTableCols; e += kTableBlock)
      so_in[e] = c0 + e < g.din ? table_offset(tg.k, tg.din_t, tg.sin_t, c0 + e) : 0;
  };
  for (int r = tid; r < ROWS; r += kTableBlock)
    so_out[r] = row0 + r < g.dout ? table_offset(tg.k, tg.dout_t, tg.sout_t, row0 + r) : 0;
  stage(0);
  __syncthreads();

  Acc acc[MB][NB];
  const T* px[NB];
  int64_t bout[NB];
  uint32_t m[NB];
  auto start = [&](uint32_t tile) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      m[nb] = tile * COLS + 16 * nb + n;
      int64_t bin;
      // past the last orbit: a valid one is loaded, nothing is stored
      orbit_base(g, m[nb] < n_orbits ? m[nb] : n_orbits - 1, bin, bout[nb]);
      px[nb] = in + bin;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[mb][nb] = Acc(0);
    }
  };
  // the chunk's k-steps, U at a time: U entries per orbit are loaded, then
  // multiplied (entries past the PTM's columns are zeros, like the PTM's)
  auto contract = [&](int c0) {
    const int kn = min(kTableCols, g.din - c0);
    for (int s0 = 0; 4 * s0 < kn; s0 += U) {
      T b[NB][U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = 4 * (s0 + u) + j;
        const bool ok = k < kn;
        const int64_t off = so_in[ok ? k : 0];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const T v = px[nb][off];
          b[nb][u] = ok ? v : T(0);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (4 * (s0 + u) < kn) {
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) {
            const T a = As[((s0 + u) * MB + mb) * 64 + lane];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = Mfma<T>::op(a, b[nb][u], acc[mb][nb]);
          }
        }
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if (m[nb] >= n_orbits) continue;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * mb + (sizeof(T) == 8 ? j + 4 * r : 4 * j + r);
          if (row0 + row < g.dout) out[bout[nb] + so_out[row]] = acc[mb][nb][r];
        }
    }
  };

  const uint32_t tiles = (n_orbits + COLS - 1) / COLS;
  constexpr uint32_t W = kTableBlock / 64;
  if (g.din <= kTableCols) {
    for (uint32_t t = blockIdx.x * W + (tid >> 6); t < tiles; t += gridDim.x * W) {
      start(t);
      contract(0);
      store();
    }
    return;
  }
  // the trip count is the same for every wave of the workgroup; waves past
  // the last tile take part in the staging only
  for (uint32_t t0 = blockIdx.x * W; t0 < tiles; t0 += gridDim.x * W) {
    start(t0 + (tid >> 6));
    for (int c0 = 0; c0 < g.din; c0 += kTableCols) {
      __syncthreads();
      stage(c0);
      __syncthreads();
      contract(c0);
    }
    store();
  }
}

template <typename T, int MB, int NB>
static int launch(const Geom& g, uint32_t n_orbits, const TableGeo& tg, const void* in, void* out,
                  const void* ptm, int64_t pstride, uint32_t batch, hipStream_t s) {
  const auto kern = k_apply_table<T, MB, NB>;
  static const uint32_t cap = [&] {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
      cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, reinterpret_cast<const void*>(kern), kTableBlock, 0) != hipSuccess ||
        per_cu <= 0)
      per_cu = 1;
    (void)hipGetLastError();
    return uint32_t(per_cu) * uint32_t(cus);
  }();
  const uint32_t tiles = (n_orbits + 16 * NB - 1) / (16 * NB);
  const uint32_t want = (tiles + kTableBlock / 64 - 1) / (kTableBlock / 64);
  const uint32_t shares = (uint32_t(g.dout) + 16 * MB - 1) / (16 * MB);
  const uint32_t per = std::max<uint32_t>(1, cap / std::max<uint32_t>(1, batch * shares));
  hipLaunchKernelGGL(kern, dim3(std::min(want, per), batch, shares), dim3(kTableBlock), 0, s,
                     static_cast<const T*>(in), static_cast<T*>(out), g, n_orbits, tg,
                     static_cast<const T*>(ptm), pstride);
  QSV_CHECK_HIP(hipGetLastError());
  return QSV_OK;
}

// float32 lanes take two orbits 16 apart, so that a wave's row is 128 bytes
// in both types
template <typename T>
static int dispatch(const Geom& g, uint32_t n_orbits, const TableGeo& tg, const void* in,
                    void* out, const void* ptm, int64_t pstride, uint32_t batch, hipStream_t s) {
  constexpr int NB = sizeof(T) == 4 ? 2 : 1;
  switch (table_row_blocks(g.dout)) {
    case 1: return launch<T, 1, NB>(g, n_orbits, tg, in, out, ptm, pstride, batch, s);
    case 2: return launch<T, 2, NB>(g, n_orbits, tg, in, out, ptm, pstride, batch, s);
    case 3: return launch<T, 3, NB>(g, n_orbits, tg, in, out, ptm, pstride, batch, s);
    case 4: return launch<T, 4, NB>(g, n_orbits, tg, in, out, ptm, pstride, batch, s);
    case 5: return launch<T, 5, NB>(g, n_orbits, tg, in, out, ptm, pstride, batch, s);
    default: return launch<T, 6, NB>(g, n_orbits, tg, in, out, ptm, pstride, batch, s);
  }
}

int launch_table(int dtype, const Geom& g, uint32_t n_orbits, const TableGeo& tg, const void* in,
                 void* out, const void* ptm, int64_t pstride, uint32_t batch, hipStream_t s) {
  if (n_orbits == 0 || batch == 0) return QSV_OK;
  return dtype == QSV_F64
             ? dispatch<double>(g, n_orbits, tg, in, out, ptm, pstride, batch, s)
             : dispatch<float>(g, n_orbits, tg, in, out, ptm, pstride, batch, s);
}

}  // namespace qsv
