// Persistent kernels that run whole circuits: many qubit circuits of
// different widths and depths in one launch, the Pauli vector of each
// circuit resident in LDS (4^n entries: up to 7 qubits in float32 on
// gfx950's 160 KB of LDS per workgroup for the forward pass).
//
// A workgroup takes circuits from the circuit table (round robin over the
// grid) and, for each, runs its gates from the gate table:
//
//   forward:  S = |0..0><0..0|; per gate: save S to the trajectory (the
//             state before the gate, in the order the gate's lanes hold it)
//             and contract it in place; at the end write the float64
//             populations (the entries whose qubit digits are all |0><0| or
//             |1><1|).
//   adjoint:  Y = dL/dS (the population gradient scattered onto those
//             entries); per gate, last first: dL/dP[o][i] = sum over orbits of
//             Y[o] X[i], X the trajectory's state, on v_mfma_f64_16x16x4
//             (lane (c, k) supplies entry c of orbit k: four orbits per k-step
//             for 16 x 16 PTMs, sixteen for 4 x 4 ones packed as four 4 x 4
//             diagonal blocks; float64 products and sums, waves summed in a
//             fixed order), and Y <- P^T Y in place.
//
// A 16 x 16 PTM is applied to sixteen orbits at a time on the matrix cores
// (16x16x4, four k-steps in ascending order: the same chain of multiply-adds
// as one thread per orbit, bit for bit): lane (n, j) = (l % 16, l / 16) reads
// entries 4 s + j, s = 0..3, of orbit n and receives the results of the same
// four entries (float32 accumulators hold rows 4 j + r: the PTM's rows are
// permuted), so the contraction is in place and its operand, four PTM entries
// a lane, comes from memory one gate ahead.  A wave reads and writes the same
// 256-entry units in every phase of a gate, so a gate needs one barrier; the
// adjoint's X goes from memory straight into the lanes that multiply it.
//
// Bound, a 7-qubit circuit in float32, per gate: 2048 cycles of MFMA to apply a
// PTM, 4096 for its gradient (float64), 1024 and 1536 of LDS traffic, 64 KB of
// trajectory; measured about 6000 (forward) and 14000 (adjoint), the rest
// latency of the chain read - multiply - write - barrier with two waves a SIMD.
// 192 circuits of 4-7 qubits, 20-80 layers (the longest circuit's chain
// decides): forward 2.05 -> 0.80 ms, adjoint 6.2 -> 1.92 ms against one thread
// per orbit with the PTM broadcast from LDS and both states staged there.
//
// LDS holds the states XOR-swizzled (circ_swz): the entries of an orbit sit
// 4^q apart, and without the swizzle the sixteen entries the MFMA operand
// loads of one orbit touch would share an LDS bank.
//
// All qubits are in the general(2) basis (Pauli dimension 4: two bits per
// digit), qubit 0 most significant.  Gates act on 1 or 2 qubits with PTMs
// of 4 x 4 or 16 x 16, layout (out..., in...) in target order, as
// qsv_apply_ptm.  No counterpart in the reference (one circuit per
// PauliVector object there); the per-gate arithmetic is its apply_ptm
// (quantumsim/pauli_vectors/numpy.py:50-64).
#include "qsv_common.h"
#include "qsv_mfma.h"

#include <algorithm>
#include <vector>

namespace qsv {

// 512 threads (8 waves) per circuit: one workgroup per CU (a 7-qubit float32
// state and the adjoint's wave partials take 96 KB of LDS), so the
// waves of that one circuit are all the latency hiding there is.
constexpr int kCircBlock = 512;
constexpr int kCircWaves = kCircBlock / 64;
constexpr int kCircMaxQubits = 8;
// Largest state the adjoint's registers cover: 7 qubits in float32, 6 in
// float64.
template <typename T>
constexpr uint32_t kCircMaxEntries = sizeof(T) == 4 ? (1u << 14) : (1u << 12);

// Index of orbit m with zero 2-bit digits inserted at bit positions lo < hi
// (hi < 0: one target).
__host__ __device__ inline uint32_t circ_orbit_base(uint32_t m, int lo, int hi) {
  uint32_t t = ((m >> lo) << (lo + 2)) | (m & ((1u << lo) - 1u));
  if (hi >= 0) t = ((t >> hi) << (hi + 2)) | (t & ((1u << hi) - 1u));
  return t;
}

// Offset of PTM index i (target order: first target slowest) inside an orbit.
__host__ __device__ inline uint32_t circ_offset(int k, uint32_t i, int s0, int s1) {
  return k == 1 ? (i << s0) : (((i >> 2) << s0) | ((i & 3u) << s1));
}

// Pauli index of population j (qubit 0 = most significant bit of j): bit t
// of j becomes bit 2 t.
__host__ __device__ inline uint32_t circ_spread(uint32_t j) {
  uint32_t r = 0;
  for (int t = 0; t < 16; ++t) r |= ((j >> t) & 1u) << (2 * t);
  return r;
}

// LDS position of state entry a: the low 6 bits XORed with a hash of the
// higher ones (a bijection on [0, 4^n); entries below 64 stay in place).
__host__ __device__ inline uint32_t circ_swz(uint32_t a) {
  const uint32_t h = a >> 6;
  return a ^ ((h ^ (h >> 6) ^ (h >> 12)) & 63u);
}

struct GateGeom {
  int k, D, s0, s1, lo, hi;
  uint32_t n_orbits;
};

__host__ __device__ inline GateGeom circ_gate_geom(const qsv_gate& gd, int n) {
  GateGeom G;
  G.k = gd.k;
  G.D = gd.k == 1 ? 4 : 16;
  G.s0 = 2 * (n - 1 - gd.q0);
  G.s1 = gd.k == 2 ? 2 * (n - 1 - gd.q1) : 0;
  if (gd.k == 1) {
    G.lo = G.s0;
    G.hi = -1;
  } else {
    G.lo = G.s0 < G.s1 ? G.s0 : G.s1;
    G.hi = G.s0 < G.s1 ? G.s1 : G.s0;
  }
  G.n_orbits = (1u << (2 * n)) / uint32_t(G.D);
  return G;
}

// Order of the digits (2-bit positions, 0 innermost) that are not a two-qubit
// gate's targets, four bits each, lowest first: the first two are the sixteen
// orbits of a group, the others its index.  A bit b of an entry's index lands
// on bank bit b mod 6 (circ_swz), so the three digits of 64 lanes should differ
// mod 3: the targets' and the first (gradient), the second target's and the
// first two (apply).
struct CircOrder {
  uint32_t of[9][8][8];  // [n][first target's digit][second target's]
};
constexpr CircOrder circ_order_table() {
  CircOrder t{};
  for (int n = 2; n <= 8; ++n)
    for (int d0 = 0; d0 < n; ++d0)
      for (int d1 = 0; d1 < n; ++d1) {
        if (d0 == d1) continue;
        int order[8] = {}, used[8] = {}, c = 0;
        const int first = 1 << (d0 % 3) | 1 << (d1 % 3);  // classes the first avoids
        for (int pass = 0; pass < 2 && c == 0; ++pass)
          for (int d = 0; d < n && c == 0; ++d)
            if (d != d0 && d != d1 && !((pass ? 1 << (d1 % 3) : first) >> (d % 3) & 1)) {
              order[c++] = d;
              used[d] = 1;
            }
        for (int d = 0; d < n && c == 1; ++d)
          if (d != d0 && d != d1 && !used[d] && d % 3 != d1 % 3 && d % 3 != order[0] % 3) {
            order[c++] = d;
            used[d] = 1;
          }
        for (int d = 0; d < n; ++d)
          if (d != d0 && d != d1 && !used[d]) order[c++] = d;
        uint32_t packed = 0;
        for (int i = 0; i < c; ++i) packed |= uint32_t(order[i]) << (4 * i);
        t.of[n][d0][d1] = packed;
      }
  return t;
}
static __device__ const CircOrder kCircOrder = circ_order_table();
static constexpr CircOrder kCircOrderHost = circ_order_table();
__host__ __device__ inline uint32_t circ_order(const CircOrder& table, const qsv_gate& gd, int n) {
  return gd.k == 2 ? table.of[n][n - 1 - gd.q0][n - 1 - gd.q1] : 0;
}

// LDS part (before the swizzle) of orbit n of a group and of group gr, for a
// circuit of `digits` digits outside the targets in the order `order`.
__host__ __device__ inline uint32_t circ_lane_part(uint32_t order, int digits, uint32_t n) {
  uint32_t a = 0;
  if (digits > 0) a |= (n & 3u) << (2 * (order & 15u));
  if (digits > 1) a |= (n >> 2) << (2 * (order >> 4 & 15u));
  return a;
}
__host__ __device__ inline uint32_t circ_group_part(uint32_t order, int digits, uint32_t gr) {
  uint32_t a = 0;
  for (int i = 2; i < digits; ++i) a |= (gr >> (2 * (i - 2)) & 3u) << (2 * (order >> (4 * i) & 15u));
  return a;
}
// Orbits of a two-qubit gate that share a unit: 16, 4 or 1.
__host__ __device__ inline uint32_t circ_lanes(int digits) {
  return digits >= 2 ? 16u : (digits == 1 ? 4u : 1u);
}

// A wave's share of a gate: units u * 8 + w of 256 entries (64 orbits of a
// one-qubit gate, 16 of a two-qubit one; a state below 256 entries is one
// unit).  Every LDS address is the XOR of a part of the unit (uniform) and one of
// the lane:
//   apply:    v[s], s = 0..3: entry s of the lane's orbit, or entry 4 s + lj of
//             orbit ln of the unit; `writes` where the lane has an orbit
//   gradient: y[t], k-step t = 0..3: entry ln of orbit 4 t + lj, or entry ln % 4
//             of orbit 16 t + 4 lj + ln / 4; bit t of `has` where there is one
template <typename T>
struct CircGate {
  static constexpr int BITS = sizeof(T) == 4 ? 3 : 1;  // of u
  uint32_t own, bit[BITS], v[4], y[4];
  bool writes;
  uint32_t has;
  __host__ __device__ CircGate(const GateGeom& G, uint32_t order, int n, uint32_t w,
                               uint32_t lane) {
    const uint32_t ln = lane & 15, lj = lane >> 4;
    has = 0;
    if (G.k == 1) {
      writes = lane < G.n_orbits;
      const uint32_t b = circ_swz(circ_orbit_base(writes ? lane : 0, G.lo, -1));
#pragma unroll
      for (uint32_t s = 0; s < 4; ++s) {
        v[s] = b ^ circ_swz(s << G.s0);
        const uint32_t m = 16 * s + 4 * lj + (ln >> 2);
        has |= uint32_t(m < G.n_orbits) << s;
        y[s] = circ_swz(circ_orbit_base(m < G.n_orbits ? m : 0, G.lo, -1) | (ln & 3) << G.s0);
      }
      own = circ_swz(circ_orbit_base(64 * w, G.lo, -1));
#pragma unroll
      for (int i = 0; i < BITS; ++i)
        bit[i] = circ_swz(circ_orbit_base(64u * kCircWaves << i, G.lo, -1));
    } else {
      const int digits = n - 2;
      const uint32_t lanes = circ_lanes(digits);
      writes = ln < lanes;
      const uint32_t b = circ_swz(circ_lane_part(order, digits, writes ? ln : 0) | lj << G.s1);
#pragma unroll
      for (uint32_t s = 0; s < 4; ++s) {
        v[s] = b ^ circ_swz(s << G.s0);
        const uint32_t m = 4 * s + lj;
        has |= uint32_t(m < lanes) << s;
        y[s] = circ_swz(circ_lane_part(order, digits, m < lanes ? m : 0) |
                        circ_offset(2, ln, G.s0, G.s1));
      }
      own = circ_swz(circ_group_part(order, digits, w));
#pragma unroll
      for (int i = 0; i < BITS; ++i)
        bit[i] = circ_swz(circ_group_part(order, digits, uint32_t(kCircWaves) << i));
    }
  }
  __host__ __device__ uint32_t at(int u) const {
    uint32_t a = own;
#pragma unroll
    for (int i = 0; i < BITS; ++i) a ^= (u >> i & 1) ? bit[i] : 0;
    return a;
  }
};

// Positions inside a unit's 256 trajectory entries: the forward stores a lane's
// v[0..3] as one vector at circ_store; the adjoint reads what belongs to y[t] at
// circ_load.
__host__ __device__ inline uint32_t circ_store(int k, int n, uint32_t lane) {
  return 4 * (k == 1 ? lane : (lane >> 4) * circ_lanes(n - 2) + (lane & 15));
}
__host__ __device__ inline uint32_t circ_load(int k, int n, uint32_t lane, uint32_t t) {
  const uint32_t ln = lane & 15, lj = lane >> 4;
  return k == 1 ? 64 * t + lane : ((ln & 3) * circ_lanes(n - 2) + 4 * t + lj) * 4 + (ln >> 2);
}

// PTM row that MFMA row m stands for: accumulator slot r of lane group j then
// holds row 4 r + j.
template <typename T>
__host__ __device__ inline int circ_row(int m) {
  return sizeof(T) == 8 ? m : 4 * (m & 3) + (m >> 2);
}

// What a lane needs of one gate's PTM, fetched a gate ahead: its MFMA operand of
// a 16 x 16 PTM (TRANS: of P^T), entry lane % 16 of a 4 x 4 one in a[0].
template <typename T, bool TRANS>
__device__ inline void circ_frag(const T* __restrict__ P, int k, int lane, T (&a)[4]) {
  if (k == 1) {
    a[0] = P[lane & 15];
    return;
  }
  const int row = circ_row<T>(lane & 15), j = lane >> 4;
#pragma unroll
  for (int s = 0; s < 4; ++s) a[s] = TRANS ? P[(4 * s + j) * 16 + row] : P[row * 16 + 4 * s + j];
}

// Lane l's value in every lane.
template <typename T>
__device__ inline T circ_from_lane(T v, int l) {
  if constexpr (sizeof(T) == 4) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
  } else {
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane(int(b), l);
    const unsigned hi = __builtin_amdgcn_readlane(int(b >> 32), l);
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
  }
}

// A one-qubit gate on a lane's orbit of each of U units; a0: this lane's entry of
// the PTM.  TRANS: P^T.
template <typename T, bool TRANS, int U, typename A>
__device__ inline void circ_apply1(T a0, const A (&b)[U], A (&acc)[U]) {
  T p[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) p[e] = circ_from_lane(a0, e);
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      T sum = T(0);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum += (TRANS ? p[i * 4 + o] : p[o * 4 + i]) * b[u][i];
      acc[u][o] = sum;
    }
}

// Units a wave holds at most.
template <typename T>
constexpr int kCircUnits = kCircMaxEntries<T> / (256 * kCircWaves);
// Four trajectory entries, aligned as one is.
template <typename T>
struct CircT4 {
  typedef T t __attribute__((ext_vector_type(4), aligned(sizeof(T))));
};

template <typename T>
__global__ void __launch_bounds__(kCircBlock)
    k_circuits_fwd(const qsv_circuit* __restrict__ circs, int n_circ,
                   const qsv_gate* __restrict__ gates, const T* __restrict__ ptms,
                   T* __restrict__ traj, double* __restrict__ pops, int max_qubits) {
  extern __shared__ __align__(16) unsigned char qsv_circ_smem[];
  T* S = reinterpret_cast<T*>(qsv_circ_smem);
  typedef typename Mfma<T>::acc Acc;
  typedef typename CircT4<T>::t T4;
  constexpr int W = kCircWaves, UN = kCircUnits<T>, U = UN < 4 ? UN : 4;  // U units in flight
  const int tid = threadIdx.x, lane = tid & 63;
  const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int c = blockIdx.x; c < n_circ; c += gridDim.x) {
    const qsv_circuit cd = circs[c];
    const int n = cd.n, last = cd.n_gates - 1;
    const uint32_t N = 1u << (2 * n), units = N > 256 ? N >> 8 : 1;
    const qsv_gate* gt = gates + cd.gate0;
    T* tr = traj + cd.traj;
    for (uint32_t i = tid; i < N; i += kCircBlock) S[circ_swz(i)] = i == 0 ? T(1) : T(0);
    // lookahead: descriptors two gates, PTM entries and digit order one gate
    qsv_gate g1 = {}, g2 = {};
    T an[4] = {};
    uint32_t on = 0;
    if (last >= 0) {
      g1 = gt[0];
      g2 = gt[last < 1 ? last : 1];
      circ_frag<T, false>(ptms + g1.ptm, g1.k, lane, an);
      on = circ_order(kCircOrder, g1, n);
    }
    __syncthreads();
    for (int g = 0; g <= last; ++g, tr += N) {
      const GateGeom G = circ_gate_geom(g1, n);
      const CircGate<T> L(G, on, n, w, lane);
      T* const out = tr + circ_store(G.k, n, lane);
      T a[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) a[s] = an[s];
      g1 = g2;
      if (g < last) {
        circ_frag<T, false>(ptms + g1.ptm, g1.k, lane, an);
        on = circ_order(kCircOrder, g1, n);
      }
      g2 = gt[g + 2 < last ? g + 2 : last];
#pragma unroll
      for (int u0 = 0; u0 < UN; u0 += U) {
        if (u0 * W + w >= units) break;
        uint32_t at[U];
        Acc b[U], acc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          at[u] = L.at((u0 + u) * W + w < units ? u0 + u : u0);
#pragma unroll
          for (int s = 0; s < 4; ++s) b[u][s] = S[at[u] ^ L.v[s]];
          acc[u] = Acc(0);
        }
        if (G.k == 1) {
          circ_apply1<T, false, U>(a[0], b, acc);
        } else {
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int u = 0; u < U; ++u) acc[u] = Mfma<T>::op(a[s], b[u][s], acc[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (L.writes && (u0 + u) * W + w < units) {
            *reinterpret_cast<T4*>(out + ((u0 + u) * W + w) * 256) = T4(b[u]);
#pragma unroll
            for (int r = 0; r < 4; ++r) S[at[u] ^ L.v[r]] = acc[u][r];
          }
      }
      __syncthreads();
    }
    for (uint32_t j = tid; j < (1u << n); j += kCircBlock)
      pops[cd.pop + j] = double(S[circ_swz(circ_spread(j))]);
    __syncthreads();
  }
}

template <typename T>
__global__ void __launch_bounds__(kCircBlock)
    k_circuits_adj(const qsv_circuit* __restrict__ circs, int n_circ,
                   const qsv_gate* __restrict__ gates, const T* __restrict__ ptms,
                   const T* __restrict__ traj, const double* __restrict__ dpops,
                   double* __restrict__ dptms, int max_qubits) {
  extern __shared__ __align__(16) unsigned char qsv_circ_smem[];
  double* red = reinterpret_cast<double*>(qsv_circ_smem);  // [2][waves][64 lanes][4]
  T* Y = reinterpret_cast<T*>(red + 2 * kCircBlock * 4);
  typedef typename Mfma<T>::acc Acc;
  typedef typename Mfma<double>::acc AccD;
  constexpr int W = kCircWaves, UN = kCircUnits<T>;
  const int tid = threadIdx.x, lane = tid & 63;
  const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the states before the gates come straight into the lanes that multiply
  // them: a unit's four k-steps, each unit's registers loaded for the gate
  // before as soon as this gate has used them
  T x[UN][4];
  for (int ci = blockIdx.x; ci < n_circ; ci += gridDim.x) {
    const qsv_circuit cd = circs[ci];
    const int n = cd.n, last = cd.n_gates - 1;
    const uint32_t N = 1u << (2 * n), units = N > 256 ? N >> 8 : 1;
    const qsv_gate* gt = gates + cd.gate0;
    // lane offsets of the next gate's loads; where there is no entry, entry 0,
    // zeroed before use
    uint32_t vo[4];
    auto place = [&](int k) {
#pragma unroll
      for (uint32_t t = 0; t < 4; ++t) {
        vo[t] = circ_load(k, n, lane, t);
        if (vo[t] >= N) vo[t] = 0;
      }
    };
    auto fetch = [&](int u, const T* tr) {
      if (u * W + w < units) {
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) x[u][t] = (tr + (u * W + w) * 256)[vo[t]];
      }
    };
    for (uint32_t i = tid; i < N; i += kCircBlock) Y[i] = T(0);
    qsv_gate g1 = {}, g2 = {};
    T an[4] = {};
    uint32_t on = 0;
    const T* tr = traj + cd.traj + int64_t(last) * N;
    if (last >= 0) {
      g1 = gt[last];
      g2 = gt[last > 0 ? last - 1 : 0];
      circ_frag<T, true>(ptms + g1.ptm, g1.k, lane, an);
      on = circ_order(kCircOrder, g1, n);
      place(g1.k);
#pragma unroll
      for (int u = 0; u < UN; ++u) fetch(u, tr);
    }
    __syncthreads();
    for (uint32_t j = tid; j < (1u << n); j += kCircBlock)
      Y[circ_swz(circ_spread(j))] = T(dpops[cd.pop + j]);
    __syncthreads();
    for (int g = last; g >= 0; --g) {
      const GateGeom G = circ_gate_geom(g1, n);
      const CircGate<T> L(G, on, n, w, lane);
      const int64_t ptm = g1.ptm;
      T a[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) a[s] = an[s];
      g1 = g2;
      tr -= N;
      if (g > 0) {
        circ_frag<T, true>(ptms + g1.ptm, g1.k, lane, an);
        on = circ_order(kCircOrder, g1, n);
        place(g1.k);
      }
      g2 = gt[g > 2 ? g - 2 : 0];
      // dL/dP: A[row][k] = Y entry, B[k][col] = X entry, k = orbit (one qubit:
      // the sum of the four 4 x 4 diagonal blocks), then Y <- P^T Y on the
      // same unit, the next unit's reads before its writes
      AccD d = AccD(0);
      T y[2][4];
      Acc v[2];
      auto read = [&](int u) {
#pragma unroll
        for (int t = 0; t < 4; ++t) y[u & 1][t] = Y[L.at(u) ^ L.y[t]];
#pragma unroll
        for (int s = 0; s < 4; ++s) v[u & 1][s] = Y[L.at(u) ^ L.v[s]];
      };
      if (w < units) read(0);
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        if (u * W + w < units) {
          if (u + 1 < UN && (u + 1) * W + w < units) read(u + 1);
          if (u == 0 && N < 256) {  // lanes without an orbit
#pragma unroll
            for (int t = 0; t < 4; ++t)
              if (!(L.has >> t & 1)) y[0][t] = x[0][t] = T(0);
          }
          Acc acc[1] = {Acc(0)};
#pragma unroll
          for (int t = 0; t < 4; ++t)
            d = Mfma<double>::op(double(y[u & 1][t]), double(x[u][t]), d);
          if (g > 0) fetch(u, tr);
          if (G.k == 1) {
            const Acc b[1] = {v[u & 1]};
            circ_apply1<T, true, 1>(a[0], b, acc);
          } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) acc[0] = Mfma<T>::op(a[s], v[u & 1][s], acc[0]);
          }
          if (L.writes) {
#pragma unroll
            for (int r = 0; r < 4; ++r) Y[L.at(u) ^ L.v[r]] = acc[0][r];
          }
        }
      }
      double* part = red + (g & 1) * kCircBlock * 4;
#pragma unroll
      for (int r = 0; r < 4; ++r) part[(w * 64 + lane) * 4 + r] = d[r];
      __syncthreads();
      // entry (o, i): float64 accumulator layout, row = lane / 16 + 4 r,
      // column = lane % 16; the other half of red takes the next gate's
      if (tid < G.D * G.D) {
        double sum = 0.0;
        if (G.k == 2) {
          const int o = tid >> 4, i = tid & 15;
          const int src = (i + 16 * (o & 3)) * 4 + (o >> 2);
#pragma unroll
          for (int ww = 0; ww < W; ++ww) sum += part[ww * 256 + src];
        } else {
          const int o = tid >> 2, i = tid & 3;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int src = (4 * u + i + 16 * o) * 4 + u;  // row 4 u + o, column 4 u + i
#pragma unroll
            for (int ww = 0; ww < W; ++ww) sum += part[ww * 256 + src];
          }
        }
        dptms[ptm + tid] = sum;
      }
    }
    __syncthreads();
  }
}

static size_t circ_lds_bytes(int elem_bytes, int max_qubits, bool adjoint) {
  const size_t N = size_t(1) << (2 * max_qubits);
  if (!adjoint) return N * elem_bytes;
  return 2 * kCircBlock * 4 * 8 + N * elem_bytes;
}

static int lds_limit() {
  static int lim = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
      v = 65536;
    (void)hipGetLastError();
    return v;
  }();
  return lim;
}

template <typename T>
static uint32_t circ_grid(const void* kern, size_t lds, int n_circ) {
  int dev = 0, cus = 0, per = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    cus = 256;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, kCircBlock, lds) != hipSuccess ||
      per <= 0)
    per = 1;
  (void)hipGetLastError();
  const uint32_t cap = uint32_t(per) * uint32_t(cus);
  return std::min<uint32_t>(cap, uint32_t(n_circ));
}

}  // namespace qsv

using namespace qsv;

extern "C" int qsv_circuits_max_qubits(int dtype) {
  const int es = dtype_size(dtype);
  QSV_CHECK_ARG(es > 0, "unknown dtype %d", dtype);
  const uint32_t max_entries = es == 4 ? kCircMaxEntries<float> : kCircMaxEntries<double>;
  int best = 0;
  for (int n = 1; n <= kCircMaxQubits; ++n)
    if (circ_lds_bytes(es, n, true) <= size_t(lds_limit()) && (1u << (2 * n)) <= max_entries)
      best = n;
  return best;
}

extern "C" int64_t qsv_circuits_lds_bytes(int dtype, int max_qubits, int adjoint) {
  const int es = dtype_size(dtype);
  QSV_CHECK_ARG(es > 0, "unknown dtype %d", dtype);
  QSV_CHECK_ARG(max_qubits >= 1 && max_qubits <= kCircMaxQubits, "max_qubits %d outside [1, %d]",
                max_qubits, kCircMaxQubits);
  return int64_t(circ_lds_bytes(es, max_qubits, adjoint != 0));
}

template <typename T, typename K, typename... Args>
static int launch_circ(K kern, size_t lds, int n_circ, hipStream_t s, Args... args) {
  static size_t attr = 0;
  if (lds > 65536 && lds > attr) {
    QSV_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    attr = lds;
  }
  const uint32_t grid = circ_grid<T>(reinterpret_cast<const void*>(kern), lds, n_circ);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(kCircBlock), lds, s, args...);
  QSV_CHECK_HIP(hipGetLastError());
  return QSV_OK;
}

extern "C" int qsv_circuits_forward(int dtype, int n_circuits, const qsv_circuit* circs_dev,
                                    const qsv_gate* gates_dev, const void* ptms, void* traj,
                                    double* pops, int max_qubits, void* stream) {
  const int es = dtype_size(dtype);
  QSV_CHECK_ARG(es > 0, "unknown dtype %d", dtype);
  QSV_CHECK_ARG(n_circuits >= 0, "negative circuit count");
  if (n_circuits == 0) return QSV_OK;
  QSV_CHECK_ARG(circs_dev && gates_dev && ptms && traj && pops, "null pointer argument");
  QSV_CHECK_ARG(max_qubits >= 1 && max_qubits <= qsv_circuits_max_qubits(dtype),
                "max_qubits %d outside [1, %d] (LDS per workgroup)", max_qubits,
                qsv_circuits_max_qubits(dtype));
  const size_t lds = circ_lds_bytes(es, max_qubits, false);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == QSV_F64)
    return launch_circ<double>(k_circuits_fwd<double>, lds, n_circuits, s, circs_dev, n_circuits,
                               gates_dev, static_cast<const double*>(ptms),
                               static_cast<double*>(traj), pops, max_qubits);
  return launch_circ<float>(k_circuits_fwd<float>, lds, n_circuits, s, circs_dev, n_circuits,
                            gates_dev, static_cast<const float*>(ptms), static_cast<float*>(traj),
                            pops, max_qubits);
}

extern "C" int qsv_circuits_adjoint(int dtype, int n_circuits, const qsv_circuit* circs_dev,
                                    const qsv_gate* gates_dev, const void* ptms,
                                    const void* traj, const double* dpops, double* dptms,
                                    int max_qubits, void* stream) {
  const int es = dtype_size(dtype);
  QSV_CHECK_ARG(es > 0, "unknown dtype %d", dtype);
  QSV_CHECK_ARG(n_circuits >= 0, "negative circuit count");
  if (n_circuits == 0) return QSV_OK;
  QSV_CHECK_ARG(circs_dev && gates_dev && ptms && traj && dpops && dptms, "null pointer argument");
  QSV_CHECK_ARG(max_qubits >= 1 && max_qubits <= qsv_circuits_max_qubits(dtype),
                "max_qubits %d outside [1, %d] (LDS per workgroup)", max_qubits,
                qsv_circuits_max_qubits(dtype));
  const size_t lds = circ_lds_bytes(es, max_qubits, true);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == QSV_F64)
    return launch_circ<double>(k_circuits_adj<double>, lds, n_circuits, s, circs_dev, n_circuits,
                               gates_dev, static_cast<const double*>(ptms),
                               static_cast<const double*>(traj), dpops, dptms, max_qubits);
  return launch_circ<float>(k_circuits_adj<float>, lds, n_circuits, s, circs_dev, n_circuits,
                            gates_dev, static_cast<const float*>(ptms),
                            static_cast<const float*>(traj), dpops, dptms, max_qubits);
}

// The contraction of one gate on a host LDS image: the same waves, units and
// lanes, every entry read and written by one lane slot, every trajectory entry
// stored once (tr may be null).
static int emulate_apply(std::vector<double>& S, const double* P, bool trans, const GateGeom& G,
                         uint32_t order, int n, uint32_t N, double* tr, int c, int g) {
  std::vector<int> touched(N, 0), stored(N, 0);
  const uint32_t units = N > 256 ? N >> 8 : 1;
  // one orbit: entry i in slot i % 4 of lane[0] (one qubit), in slot i / 4 of
  // lane[i % 4] (two)
  auto contract = [&](uint32_t un, const uint32_t (&lane)[4]) {
    double xin[16];
    uint32_t at[16];
    for (int i = 0; i < G.D; ++i) {
      const uint32_t l = G.k == 1 ? lane[0] : lane[i & 3], slot = G.k == 1 ? i : i >> 2;
      const CircGate<float> L(G, order, n, un % kCircWaves, l);
      if (!L.writes) return int(QSV_OK);
      at[i] = L.at(un / kCircWaves) ^ L.v[slot];
      const uint32_t to = un * 256 + circ_store(G.k, n, l) + slot;
      QSV_CHECK_ARG(at[i] < N, "circuit %d gate %d: LDS index %u out of range", c, g, at[i]);
      QSV_CHECK_ARG(to < N && !stored[to]++, "circuit %d gate %d: trajectory entry %u", c, g, to);
      ++touched[at[i]];
      xin[i] = S[at[i]];
      if (tr) tr[to] = xin[i];
    }
    for (int o = 0; o < G.D; ++o) {
      double acc = 0.0;
      for (int i = 0; i < G.D; ++i) acc += (trans ? P[i * G.D + o] : P[o * G.D + i]) * xin[i];
      S[at[o]] = acc;
    }
    return int(QSV_OK);
  };
  for (uint32_t un = 0; un < units; ++un)
    for (uint32_t l = 0; l < (G.k == 1 ? 64 : 16); ++l) {
      const uint32_t lane[4] = {l, l + 16, l + 32, l + 48};
      if (const int rc = contract(un, lane)) return rc;
    }
  for (uint32_t a = 0; a < N; ++a)
    QSV_CHECK_ARG(touched[a] == 1, "circuit %d gate %d: entry %u in %d orbits", c, g, a,
                  touched[a]);
  return QSV_OK;
}

// Host replay of both kernels on host tables and arrays (float64), with
// every table entry, trajectory, population, PTM and LDS access checked.
extern "C" int qsv_emulate_circuits(int n_circuits, const qsv_circuit* circs,
                                    const qsv_gate* gates, int64_t n_gates_total,
                                    const double* ptms, int64_t ptm_elems, double* traj,
                                    int64_t traj_elems, double* pops, int64_t pop_elems,
                                    const double* dpops, double* dptms, int max_qubits) {
  QSV_CHECK_ARG(n_circuits >= 0 && circs && gates && ptms && traj && pops, "null argument");
  QSV_CHECK_ARG(max_qubits >= 1 && max_qubits <= kCircMaxQubits, "bad max_qubits");
  const uint32_t Nmax = 1u << (2 * max_qubits);
  std::vector<double> S(Nmax), Y(Nmax);
  {
    // every gate owns its PTM slot (the adjoint writes dL/dP there)
    std::vector<std::pair<int64_t, int64_t>> slots;
    for (int c = 0; c < n_circuits; ++c)
      for (int g = 0; g < circs[c].n_gates && circs[c].gate0 + g < n_gates_total; ++g) {
        const qsv_gate gd = gates[circs[c].gate0 + g];
        slots.push_back({gd.ptm, gd.ptm + (gd.k == 1 ? 16 : 256)});
      }
    std::sort(slots.begin(), slots.end());
    for (size_t i = 1; i < slots.size(); ++i)
      QSV_CHECK_ARG(slots[i].first >= slots[i - 1].second, "two gates share PTM elements");
  }
  for (int c = 0; c < n_circuits; ++c) {
    const qsv_circuit cd = circs[c];
    QSV_CHECK_ARG(cd.n >= 1 && cd.n <= max_qubits, "circuit %d: %d qubits", c, cd.n);
    QSV_CHECK_ARG(cd.n_gates >= 0 && cd.gate0 >= 0 && cd.gate0 + cd.n_gates <= n_gates_total,
                  "circuit %d: gate range out of the table", c);
    const uint32_t N = 1u << (2 * cd.n);
    {
      std::vector<char> seen(N, 0);
      for (uint32_t i = 0; i < N; ++i) {
        const uint32_t p = circ_swz(i);
        QSV_CHECK_ARG(p < N && !seen[p], "LDS swizzle not a bijection for %d qubits", cd.n);
        seen[p] = 1;
      }
    }
    QSV_CHECK_ARG(cd.traj >= 0 && cd.traj + int64_t(cd.n_gates) * N <= traj_elems,
                  "circuit %d: trajectory out of range", c);
    QSV_CHECK_ARG(cd.pop >= 0 && cd.pop + (int64_t(1) << cd.n) <= pop_elems,
                  "circuit %d: populations out of range", c);
    for (int g = 0; g < cd.n_gates; ++g) {
      const qsv_gate gd = gates[cd.gate0 + g];
      QSV_CHECK_ARG(gd.k == 1 || gd.k == 2, "circuit %d gate %d: k = %d", c, g, gd.k);
      QSV_CHECK_ARG(gd.q0 >= 0 && gd.q0 < cd.n && (gd.k == 1 || (gd.q1 >= 0 && gd.q1 < cd.n &&
                                                                  gd.q1 != gd.q0)),
                    "circuit %d gate %d: bad targets", c, g);
      const int D = gd.k == 1 ? 4 : 16;
      QSV_CHECK_ARG(gd.ptm >= 0 && gd.ptm + D * D <= ptm_elems, "circuit %d gate %d: PTM offset",
                    c, g);
    }
    // forward
    std::fill(S.begin(), S.end(), 0.0);
    S[circ_swz(0)] = 1.0;
    for (int g = 0; g < cd.n_gates; ++g) {
      const qsv_gate gd = gates[cd.gate0 + g];
      const GateGeom G = circ_gate_geom(gd, cd.n);
      const uint32_t order = circ_order(kCircOrderHost, gd, cd.n);
      if (const int rc = emulate_apply(S, ptms + gd.ptm, false, G, order, cd.n, N,
                                       traj + cd.traj + int64_t(g) * N, c, g))
        return rc;
    }
    for (uint32_t j = 0; j < (1u << cd.n); ++j) {
      const uint32_t a = circ_spread(j);
      QSV_CHECK_ARG(a < N, "population index out of range");
      pops[cd.pop + j] = S[circ_swz(a)];
    }
    if (!dpops) continue;
    QSV_CHECK_ARG(dptms != nullptr, "dptms missing");
    // adjoint
    std::fill(Y.begin(), Y.end(), 0.0);
    for (uint32_t j = 0; j < (1u << cd.n); ++j) Y[circ_swz(circ_spread(j))] = dpops[cd.pop + j];
    for (int g = cd.n_gates - 1; g >= 0; --g) {
      const qsv_gate gd = gates[cd.gate0 + g];
      const GateGeom G = circ_gate_geom(gd, cd.n);
      const uint32_t order = circ_order(kCircOrderHost, gd, cd.n);
      const double* tr = traj + cd.traj + int64_t(g) * N;
      // MFMA replay: waves, units, k-steps and lanes as in k_circuits_adj
      constexpr int W = kCircWaves;
      const uint32_t units = N > 256 ? N >> 8 : 1;
      std::vector<double> red(size_t(W) * 64 * 4, 0.0);
      std::vector<int> used(N, 0);
      for (uint32_t un = 0; un < units; ++un)
        for (uint32_t t = 0; t < 4; ++t) {
          const uint32_t w = un % W;
          double A[64], B[64];
          for (uint32_t lane = 0; lane < 64; ++lane) {
            const CircGate<float> L(G, order, cd.n, w, lane);
            A[lane] = B[lane] = 0.0;
            if (!(L.has >> t & 1)) continue;
            const uint32_t e = L.at(un / W) ^ L.y[t];
            const uint32_t from = un * 256 + circ_load(G.k, cd.n, lane, t);
            QSV_CHECK_ARG(e < N && from < N, "adjoint: index out of range");
            A[lane] = Y[e];
            B[lane] = tr[from];
            ++used[e];
          }
          for (int lane = 0; lane < 64; ++lane)
            for (int r = 0; r < 4; ++r) {
              const int row = (lane >> 4) + 4 * r, col = lane & 15;
              double d = 0.0;
              for (int q = 0; q < 4; ++q) d += A[row + 16 * q] * B[col + 16 * q];
              red[(w * 64 + lane) * 4 + r] += d;
            }
        }
      for (uint32_t e = 0; e < N; ++e)
        QSV_CHECK_ARG(used[e] == 1, "adjoint: entry %u used %d times", e, used[e]);
      for (int tid = 0; tid < G.D * G.D; ++tid) {
        double sum = 0.0;
        if (G.k == 2) {
          const int o = tid >> 4, i = tid & 15;
          const int src = (i + 16 * (o & 3)) * 4 + (o >> 2);
          for (int ww = 0; ww < W; ++ww) sum += red[ww * 256 + src];
        } else {
          const int o = tid >> 2, i = tid & 3;
          for (int u = 0; u < 4; ++u) {
            const int src = (4 * u + i + 16 * o) * 4 + u;
            for (int ww = 0; ww < W; ++ww) sum += red[ww * 256 + src];
          }
        }
        dptms[gd.ptm + tid] = sum;
      }
      if (const int rc = emulate_apply(Y, ptms + gd.ptm, true, G, order, cd.n, N, nullptr, c, g))
        return rc;
    }
  }
  return QSV_OK;
}
