// Qubit circuits applied several gates to a pass over the Pauli vector.
//
// Gate by gate, a circuit reads and writes the whole vector once per gate;
// fused into dense three-qubit blocks, once per two brickwork bonds, at 128
// flops per entry and block.  Here a pass takes a set of qubits (the window),
// and every workgroup keeps a tile of the vector -- all the window's digits
// of a few neighbouring orbits, 64 KB -- in LDS while it applies every gate
// that the order allows inside the window: on a brickwork circuit of 13-14
// qubits 6 to 7 two-qubit gates per pass over HBM, at 32 flops per entry and
// gate.  One-qubit gates are folded into the two-qubit ones on the host.
//
// A two-qubit gate is a 16 x 16 PTM on 16 orbits at a time, four MFMA k-steps
// (16x16x4).  Lane (n, j) = (l % 16, l / 16) holds entries (s, j), s = 0..3,
// of its orbit: digit j of one target, the four digits s of the other.  The
// accumulators come out at the same four places (row j + 4 r), so a gate works
// in place and waves meet once per gate.
//
// LDS addresses are linear over the index bits (slab_phys: the low bits XOR a
// hash of the rest), so an address is the XOR of a lane part, a group part and
// a digit part, which the host tabulates per gate; which index bits the sixteen
// orbits of a group stand for, and which target plays the part of j, it chooses
// so that the lanes that the LDS serves together fall on distinct banks (the
// conflict counter does not move with the number of gates).
//
// Float64 vectors only: float32 ones are fused into dense blocks instead, whose
// rounding their populations carry (fusion.apply_circuit).
//
// Measured (14 qubits, 2 GiB, window of five middle qubits): 0.72 ms with one
// gate (6.0 TB/s), 0.91 with four, 1.16 with six, 2.0 with twelve: up to three
// gates the pass costs its HBM traffic, then 0.13 ms a gate (66 TFLOP/s; a large
// float64 matrix product reaches 72).  Windows of far outer qubits alone, whose
// tile is made of 64-byte runs, take 0.1-0.25 ms more.  The ten-layer brickwork
// circuit in 10 passes: 14 ms, in 41 applications of dense blocks 34.8 (and 46
// with their composition on the host).  Tried without gain: workgroups that
// stay and prefetch the next tile into registers, waves that split the tile by
// untouched bits and meet only when those change, per-pass hashes, wave
// priorities (all within 5 %, the prefetch slower).
#include "qsv_geom.h"
#include "qsv_mfma.h"

#include <algorithm>
#include <array>
#include <math.h>
#include <string.h>
#include <memory>
#include <new>
#include <vector>

namespace qsv {

constexpr int kSlabBlock = 512;
constexpr int kSlabWaves = kSlabBlock / 64;
constexpr int kSlabTileBits = 13;  // 64 KB: two workgroups per CU
constexpr int kSlabMaxQubits = 16;
constexpr int kSlabMaxBlkBits = 2 * kSlabMaxQubits - kSlabTileBits;
constexpr int kSlabRunBytes = 64;  // least contiguous run of a tile in memory

// LDS position of tile entry a: the bits that select one of the 32 pairs of
// banks XOR a hash of the higher ones.  Linear, and a bijection on any
// power-of-two range.
__host__ __device__ inline uint32_t slab_phys(uint32_t a) {
  const uint32_t h = a >> 5;
  return a ^ ((h ^ (h >> 2) ^ (h << 1)) & 31u);
}

// A gate's record: the PTM in fragment order (a lane's four k-steps side by
// side) and the parts of its LDS positions.
struct alignas(64) SlabGate {
  double frag[64 * 4];
  uint32_t digit[4];
  uint32_t lane_bit[6];  // the parts of a lane's bits; with fewer than 16
  uint32_t lanes;        // orbits, only lanes below `lanes` (of 16) have one
  uint32_t reserved;
  uint32_t group[1 << (kSlabTileBits - 8)];
};

struct SlabGeom {
  int32_t tbits, n_gates, n_blk;
  int64_t tstr[kSlabTileBits];    // element stride of each tile bit
  int64_t bstr[kSlabMaxBlkBits];  // and of each bit of the tile's index (0 past n_blk)
};

// Tiles that share a 128-byte line are neighbours in the index; give them to
// workgroups of the same XCD (workgroups go round the eight XCDs).
__host__ __device__ inline uint32_t slab_tile_of(uint32_t bid, int n_blk) {
  return n_blk < 4 ? bid : (bid & ~15u) | ((bid & 7u) << 1) | ((bid >> 3) & 1u);
}

typedef VT<double, 2>::t SlabVec;
typedef VT<double, 4>::t SlabFrag;
constexpr int kSlabIters = 1 << (kSlabTileBits - 10);  // 16-byte vectors per thread
constexpr int kSlabGroups = (1 << (kSlabTileBits - 8)) / kSlabWaves;  // per wave, full tile

// One gate on NG of a wave's groups of orbits; lanes without an orbit (tiles
// under 16 orbits) read slot 0 and write nothing.
template <int NG>
__device__ __forceinline__ void slab_gate(double* S, const SlabGate* gd, const SlabFrag& f,
                                          uint32_t lane_part, bool on, int first_group) {
  typedef Mfma<double>::acc Acc;
  uint32_t a[NG];
  double b[NG][4];
  Acc acc[NG];
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    a[i] = lane_part ^ gd->group[first_group + i * kSlabWaves];
#pragma unroll
    for (int s = 0; s < 4; ++s) b[i][s] = S[a[i] ^ gd->digit[s]];
    acc[i] = Acc(0);
  }
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int i = 0; i < NG; ++i) acc[i] = Mfma<double>::op(f[s], b[i][s], acc[i]);
#pragma unroll
  for (int i = 0; i < NG; ++i)
    if (on) {
#pragma unroll
      for (int r = 0; r < 4; ++r) S[a[i] ^ gd->digit[r]] = acc[i][r];
    }
}

// FULL: the tile has kSlabTileBits and every wave the same number of groups.
// `in` and `out` are the same vector from a circuit's second pass on: a tile is
// read whole before any of it is written, and tiles are disjoint.
template <bool FULL, bool NT>
__global__ void __launch_bounds__(kSlabBlock)
    k_slab(const double* in, double* out, const SlabGeom g, const SlabGate* __restrict__ gates) {
  extern __shared__ __align__(16) unsigned char qsv_slab_smem[];
  double* S = reinterpret_cast<double*>(qsv_slab_smem);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t E = 1u << g.tbits;

  // vector `it` of this thread covers tile entries 2 (512 it + tid)
  const uint32_t tile = slab_tile_of(blockIdx.x, g.n_blk);
  int64_t base = 0;
#pragma unroll
  for (int b = 0; b < kSlabMaxBlkBits; ++b) base += (tile >> b) & 1 ? g.bstr[b] : 0;
#pragma unroll
  for (int b = 0; b < 9; ++b)
    if (FULL || 1 + b < g.tbits) base += (tid >> b) & 1 ? g.tstr[1 + b] : 0;
  auto at = [&](int it) {
    int64_t o = base;
#pragma unroll
    for (int b = 0; b < kSlabTileBits - 10; ++b) o += (it >> b) & 1 ? g.tstr[10 + b] : 0;
    return o;
  };
  auto mine = [&](int it) { return FULL || uint32_t(it * kSlabBlock + tid) * 2 < E; };
  SlabVec v[kSlabIters];
#pragma unroll
  for (int it = 0; it < kSlabIters; ++it)
    if (mine(it)) v[it] = gload<NT>(reinterpret_cast<const SlabVec*>(in + at(it)));
#pragma unroll
  for (int it = 0; it < kSlabIters; ++it)
    if (mine(it)) {
      const uint32_t p = slab_phys(uint32_t(it * kSlabBlock + tid) * 2);
      S[p] = v[it][0];
      S[p ^ 1] = v[it][1];
    }
  __syncthreads();

  uint32_t bit_mask[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) bit_mask[i] = 0u - (uint32_t(lane) >> i & 1u);
  // one gate of lookahead: its PTM fragment
  SlabFrag next = *reinterpret_cast<const SlabFrag*>(gates[0].frag + 4 * lane);
  const int groups = g.tbits > 8 ? 1 << (g.tbits - 8) : 1;
  for (int gi = 0; gi < g.n_gates; ++gi) {
    const SlabGate* gd = gates + gi;
    const SlabFrag f = next;
    if (gi + 1 < g.n_gates) next = *reinterpret_cast<const SlabFrag*>(gd[1].frag + 4 * lane);
    const bool on = FULL || uint32_t(lane & 15) < gd->lanes;
    uint32_t la = 0;
#pragma unroll
    for (int i = 0; i < 6; ++i) la ^= bit_mask[i] & gd->lane_bit[i];
    if (!on) la = 0;
    if constexpr (FULL) {
      slab_gate<kSlabGroups>(S, gd, f, la, true, w);
    } else {
      for (int g0 = w; g0 < groups; g0 += kSlabWaves) slab_gate<1>(S, gd, f, la, on, g0);
    }
    __syncthreads();
  }

#pragma unroll
  for (int it = 0; it < kSlabIters; ++it)
    if (mine(it)) {
      const uint32_t p = slab_phys(uint32_t(it * kSlabBlock + tid) * 2);
      SlabVec o;
      o[0] = S[p];
      o[1] = S[p ^ 1];
      gstore<NT>(reinterpret_cast<SlabVec*>(out + at(it)), o);
    }
}

// ------------------------------------------------------------- host side
typedef std::array<double, 16> M4;
typedef std::array<double, 256> M16;

// P of a two-qubit block with one-qubit PTMs applied before it: P (A x B)
static M16 after_pair(const M16& p, const M4& a, const M4& b) {
  M16 t, o;
  for (int r = 0; r < 16; ++r)
    for (int ka = 0; ka < 4; ++ka)
      for (int ib = 0; ib < 4; ++ib) {
        double s = 0;
        for (int kb = 0; kb < 4; ++kb) s += p[r * 16 + 4 * ka + kb] * b[kb * 4 + ib];
        t[r * 16 + 4 * ka + ib] = s;
      }
  for (int r = 0; r < 16; ++r)
    for (int ia = 0; ia < 4; ++ia)
      for (int ib = 0; ib < 4; ++ib) {
        double s = 0;
        for (int ka = 0; ka < 4; ++ka) s += t[r * 16 + 4 * ka + ib] * a[ka * 4 + ia];
        o[r * 16 + 4 * ia + ib] = s;
      }
  return o;
}

// (A x I) P or (I x B) P
static M16 before_one(const M16& p, const M4& u, bool first) {
  M16 o;
  for (int x = 0; x < 4; ++x)
    for (int y = 0; y < 4; ++y)
      for (int c = 0; c < 16; ++c) {
        double s = 0;
        for (int k = 0; k < 4; ++k)
          s += first ? u[x * 4 + k] * p[(4 * k + y) * 16 + c] : u[y * 4 + k] * p[(4 * x + k) * 16 + c];
        o[(4 * x + y) * 16 + c] = s;
      }
  return o;
}

template <typename M, int D>
static M product(const M& a, const M& b) {
  M o;
  for (int r = 0; r < D; ++r)
    for (int c = 0; c < D; ++c) {
      double s = 0;
      for (int k = 0; k < D; ++k) s += a[r * D + k] * b[k * D + c];
      o[r * D + c] = s;
    }
  return o;
}

struct SlabBlock2 {
  int a, b;  // qubits, in the order of the PTM's axes
  M16 m;
};

// The circuit as two-qubit blocks: a qubit's one-qubit gates go into the next
// block on it (what is left at the end into the last one), a gate on the same
// pair as the latest block of both its qubits into that block.
static std::vector<SlabBlock2> slab_blocks(int n, int n_gates, const int32_t* ks,
                                           const int32_t* targets, const double* ptms) {
  std::vector<SlabBlock2> out;
  std::vector<int> last(n, -1);
  std::vector<M4> pend(n);
  std::vector<char> has(n, 0);
  const M4 eye4 = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1};
  M16 eye16{};
  for (int i = 0; i < 16; ++i) eye16[17 * i] = 1;
  for (int g = 0; g < n_gates; ++g) {
    if (ks[g] == 1) {
      const int q = targets[2 * g];
      M4 p;
      std::copy(ptms, ptms + 16, p.begin());
      ptms += 16;
      pend[q] = has[q] ? product<M4, 4>(p, pend[q]) : p;
      has[q] = 1;
      continue;
    }
    const int a = targets[2 * g], b = targets[2 * g + 1];
    M16 p;
    std::copy(ptms, ptms + 256, p.begin());
    ptms += 256;
    if (has[a] || has[b]) p = after_pair(p, has[a] ? pend[a] : eye4, has[b] ? pend[b] : eye4);
    has[a] = has[b] = 0;
    if (last[a] >= 0 && last[a] == last[b]) {
      SlabBlock2& k = out[last[a]];
      if (k.a != a) {  // the other order of the same pair
        M16 t;
        for (int r = 0; r < 16; ++r)
          for (int c = 0; c < 16; ++c)
            t[r * 16 + c] = p[(4 * (r & 3) + (r >> 2)) * 16 + 4 * (c & 3) + (c >> 2)];
        p = t;
      }
      k.m = product<M16, 16>(p, k.m);
      continue;
    }
    last[a] = last[b] = int(out.size());
    out.push_back({a, b, p});
  }
  for (int q = 0; q < n; ++q) {
    if (!has[q]) continue;
    if (last[q] >= 0) {
      SlabBlock2& k = out[last[q]];
      k.m = before_one(k.m, pend[q], k.a == q);
      continue;
    }
    // never in a pair: with the next such qubit, or with any other
    int r = -1;
    for (int t = q + 1; t < n && r < 0; ++t)
      if (has[t] && last[t] < 0) r = t;
    const int other = r >= 0 ? r : (q > 0 ? q - 1 : 1);
    out.push_back({q, other, after_pair(eye16, pend[q], r >= 0 ? pend[r] : eye4)});
    if (r >= 0) has[r] = 0;
  }
  return out;
}

static int bits_of(uint64_t m) { return __builtin_popcountll(m); }

// The tile bits of a window: its qubits' bits and the lowest others.  0 if
// the window does not fit the tile or leaves the tile short of contiguous
// runs of kSlabRunBytes.
static uint64_t slab_tile_mask(int n, uint64_t window) {
  uint64_t m = 0;
  for (int q = 0; q < n; ++q)
    if (window >> q & 1) m |= uint64_t(3) << (2 * (n - 1 - q));
  int left = std::min(kSlabTileBits, 2 * n) - bits_of(m);
  if (left < 0) return 0;
  for (int b = 0; b < 2 * n && left > 0; ++b)
    if (!(m >> b & 1)) {
      m |= uint64_t(1) << b;
      --left;
    }
  int run = 0;
  while (m >> run & 1) ++run;
  return run == 2 * n || (int64_t(8) << run) >= kSlabRunBytes ? m : 0;
}

// Gates of `pend` (qubit masks, in order) that the order allows inside the
// window: how many, and which if `take`.
static int slab_closure(const std::vector<uint32_t>& pend, uint32_t window,
                        std::vector<int>* take) {
  uint32_t blocked = 0;
  int count = 0;
  for (size_t i = 0; i < pend.size(); ++i) {
    const uint32_t m = pend[i];
    if (!(m & blocked) && !(m & ~window)) {
      ++count;
      if (take) take->push_back(int(i));
    } else {
      blocked |= m;
      if (!(window & ~blocked)) break;
    }
  }
  return count;
}

// Window of the next pass: grown from every gate that can run now (alone and
// with the innermost qubit, whose windows may be one wider), by the qubit or
// ready gate that lets most gates run per qubit; the best window met.
static uint32_t slab_window(int n, const std::vector<uint32_t>& pend) {
  const uint32_t full = (1u << n) - 1;
  std::vector<uint32_t> ready;
  uint32_t blocked = 0;
  for (size_t i = 0; i < pend.size() && blocked != full; ++i) {
    if (!(pend[i] & blocked)) ready.push_back(pend[i]);
    blocked |= pend[i];
  }
  uint32_t best = 0;
  int best_count = 0;
  for (size_t seed = 0; seed < 2 * ready.size(); ++seed) {
    uint32_t win = ready[seed >> 1] | (seed & 1 ? 1u << (n - 1) : 0);
    for (;;) {
      if (slab_tile_mask(n, win)) {
        const int c = slab_closure(pend, win, nullptr);
        if (c > best_count) {
          best_count = c;
          best = win;
        }
      }
      uint32_t next = 0;
      int next_count = 0, next_bits = 1;
      auto consider = [&](uint32_t cand) {
        if (cand == win || 2 * bits_of(cand) > kSlabTileBits) return;
        const int c = slab_closure(pend, cand, nullptr), b = bits_of(cand);
        // more gates per qubit; among equals, a window with whole runs
        const int d = c * next_bits - next_count * b;
        if (!next || d > 0 ||
            (d == 0 && slab_tile_mask(n, cand) &&
             !slab_tile_mask(n, next))) {
          next = cand;
          next_count = c;
          next_bits = b;
        }
      };
      for (int q = 0; q < n; ++q) consider(win | 1u << q);
      // gates next in line outside the window
      uint32_t held = 0;
      for (size_t i = 0; i < pend.size() && held != full; ++i) {
        const uint32_t m = pend[i];
        if (!(m & held) && !(m & ~win)) continue;
        if (!(m & held)) consider(win | m);
        held |= m;
      }
      if (!next) break;
      win = next;
    }
  }
  return best;
}

struct SlabPass {
  SlabGeom g;
  int first;  // gate record
  bool full, run128;
};

struct SlabPlan {
  int n;
  int64_t extent;
  std::vector<SlabPass> passes;
  std::vector<SlabGate> gates;
};

static int gf2_rank(uint32_t* v, int n) {
  int r = 0;
  for (int i = 0; i < n; ++i) {
    if (!v[i]) continue;
    ++r;
    const uint32_t low = v[i] & (0u - v[i]);
    for (int k = i + 1; k < n; ++k)
      if (v[k] & low) v[k] ^= v[i];
  }
  return r;
}

// Bank ranks missing when a group's orbits are bits nb[0..4) and j is at pb: a
// read of 8 bytes a lane is conflict-free if the banks are independent over 16
// lanes (of 16 pairs of banks) and over 32 (of 32).
static int slab_conflicts(const int* nb, int pb) {
  uint32_t a[4], b[5];
  for (int i = 0; i < 5; ++i) {
    const uint32_t p = slab_phys(1u << (i < 4 ? nb[i] : pb));
    if (i < 4) a[i] = p & 15u;
    b[i] = p & 31u;
  }
  return 4 - gf2_rank(a, 4) + 5 - gf2_rank(b, 5);
}

// The record of a block on tile-bit positions p0, p1 (its first and second
// target's digits).
static void slab_record(const SlabBlock2& blk, int p0, int p1, int tbits, SlabGate& out) {
  // which target is the lane digit j, and which bits the sixteen orbits
  int best = 1 << 20, bits[kSlabTileBits], nb = 0, orbit[4];
  bool swap = false;
  for (int b = 0; b < tbits; ++b)
    if (b != p0 && b != p0 + 1 && b != p1 && b != p1 + 1) bits[nb++] = b;
  const int nl = std::min(nb, 4);
  std::copy(bits, bits + nl, orbit);
  for (int sw = 0; sw < 2 && nb > 4 && best > 0; ++sw)
    for (int m = 0; m < 1 << nb && best > 0; ++m) {
      if (bits_of(m) != 4) continue;
      int at[4], c = 0;
      for (int i = 0; i < nb; ++i)
        if (m >> i & 1) at[c++] = bits[i];
      const int cost = slab_conflicts(at, sw ? p0 : p1);
      if (cost < best) {
        best = cost;
        swap = sw != 0;
        std::copy(at, at + 4, orbit);
      }
    }
  const int ps = swap ? p1 : p0, pj = swap ? p0 : p1;
  uint32_t rest = (1u << tbits) - 1;
  rest &= ~(3u << p0 | 3u << p1);
  memset(&out, 0, sizeof(out));
  for (int i = 0; i < nl; ++i) {
    out.lane_bit[i] = slab_phys(1u << orbit[i]);
    rest &= ~(1u << orbit[i]);
  }
  for (int i = 0; i < 2; ++i) out.lane_bit[4 + i] = slab_phys(1u << (pj + i));
  out.lanes = 1u << nl;
  for (int l = 0; l < 64; ++l) {
    // fragment: A row m = l % 16, k-steps s, column (s, j)
    const int j = l >> 4, m = l & 15, rd = m >> 2, rj = m & 3;
    for (int s = 0; s < 4; ++s) {
      const int row = swap ? 4 * rj + rd : 4 * rd + rj;
      const int col = swap ? 4 * j + s : 4 * s + j;
      out.frag[4 * l + s] = blk.m[row * 16 + col];
    }
  }
  for (uint32_t gr = 0; gr < sizeof(out.group) / sizeof(out.group[0]); ++gr) {
    uint32_t r = gr;
    for (int b = 0; b < tbits; ++b)
      if (rest >> b & 1) {
        if (r & 1) out.group[gr] ^= slab_phys(1u << b);
        r >>= 1;
      }
  }
  for (uint32_t d = 0; d < 4; ++d) out.digit[d] = slab_phys(d << ps);
}

static int slab_compile(int n, const int64_t* strides, int64_t extent, int n_gates,
                        const int32_t* ks, const int32_t* targets, const double* ptms,
                        SlabPlan& plan) {
  plan.n = n;
  plan.extent = extent;
  const std::vector<SlabBlock2> blocks = slab_blocks(n, n_gates, ks, targets, ptms);
  std::vector<uint32_t> pend;
  std::vector<int> index;
  for (size_t i = 0; i < blocks.size(); ++i) {
    pend.push_back(1u << blocks[i].a | 1u << blocks[i].b);
    index.push_back(int(i));
  }
  int records = 0;
  while (!pend.empty()) {
    const uint32_t win = slab_window(n, pend);
    const uint64_t mask = win ? slab_tile_mask(n, win) : 0;
    QSV_CHECK_ARG(mask != 0, "internal: no window for a circuit pass");
    SlabPass ps;
    memset(&ps, 0, sizeof(ps));
    ps.first = records;
    int pos[2 * kSlabMaxQubits];
    for (int b = 0; b < 2 * n; ++b) {
      const int64_t st = strides[n - 1 - b / 2] << (b & 1);
      if (mask >> b & 1) {
        pos[b] = ps.g.tbits;
        ps.g.tstr[ps.g.tbits++] = st;
      } else {
        ps.g.bstr[ps.g.n_blk++] = st;
      }
    }
    ps.full = ps.g.tbits == kSlabTileBits;
    int run = 0;
    while (run < 2 * n && (mask >> run & 1)) ++run;
    ps.run128 = (int64_t(8) << run) >= 128;
    std::vector<int> take;
    ps.g.n_gates = slab_closure(pend, win, &take);
    for (int t : take) {
      const SlabBlock2& blk = blocks[index[t]];
      plan.gates.emplace_back();
      slab_record(blk, pos[2 * (n - 1 - blk.a)], pos[2 * (n - 1 - blk.b)], ps.g.tbits,
                  plan.gates.back());
      ++records;
    }
    plan.passes.push_back(ps);
    std::vector<uint32_t> np;
    std::vector<int> ni;
    size_t t = 0;
    for (size_t i = 0; i < pend.size(); ++i) {
      if (t < take.size() && take[t] == int(i)) {
        ++t;
        continue;
      }
      np.push_back(pend[i]);
      ni.push_back(index[i]);
    }
    pend.swap(np);
    index.swap(ni);
  }
  return QSV_OK;
}

// Greedy fusion into blocks of up to max_qudits qubits, the blocks and their
// order those of quantumsim_amd.fusion.fuse: a gate joins the largest subset
// of the open blocks it touches that fits (ties: the one of more gates), the
// others it touches close; at the end the open ones close, in the order in
// which their qubits were opened.
struct FusedBlock {
  uint32_t q;            // qubits
  std::vector<int> src;  // gates in application order
};

struct FusedBlocks {
  int n;
  std::vector<int32_t> ks, targets;
  std::vector<double> ptms;
  std::vector<int64_t> at;  // a gate's PTM in ptms
  std::vector<FusedBlock> blocks;
};

static void fuse_blocks(int max_qudits, FusedBlocks& f) {
  std::vector<FusedBlock> work;
  std::vector<int> open(f.n, -1), opened;  // opened: open qubits, oldest first
  auto close = [&](int b) {
    for (int q = 0; q < f.n; ++q)
      if (work[b].q >> q & 1) {
        open[q] = -1;
        opened.erase(std::find(opened.begin(), opened.end(), q));
      }
  };
  for (int g = 0; g < int(f.ks.size()); ++g) {
    uint32_t mine = 0;
    std::vector<int> touched;
    for (int t = 0; t < f.ks[g]; ++t) {
      const int q = f.targets[2 * g + t];
      mine |= 1u << q;
      if (open[q] >= 0 && std::find(touched.begin(), touched.end(), open[q]) == touched.end())
        touched.push_back(open[q]);
    }
    const int nt = int(touched.size());
    // subsets (bit t: touched[t]), the larger ones first
    static const int kSubsets[3][4] = {{0}, {1, 0}, {3, 1, 2, 0}};
    int best = 0, best_qubits = -1, best_gates = 0;
    for (int i = 0; i < 1 << nt; ++i) {
      const int sub = kSubsets[nt][i];
      uint32_t u = mine;
      int gates = 0;
      for (int t = 0; t < nt; ++t)
        if (sub >> t & 1) {
          u |= work[touched[t]].q;
          gates += int(work[touched[t]].src.size());
        }
      if (sub && bits_of(u) > max_qudits) continue;
      const int qubits = sub ? bits_of(u) : 0;
      if (qubits > best_qubits || (qubits == best_qubits && gates > best_gates)) {
        best = sub;
        best_qubits = qubits;
        best_gates = gates;
      }
    }
    FusedBlock nb{mine, {}};
    for (int t = 0; t < nt; ++t)
      if (!(best >> t & 1)) {
        f.blocks.push_back(work[touched[t]]);
        close(touched[t]);
      }
    for (int t = 0; t < nt; ++t)
      if (best >> t & 1) {
        const FusedBlock& k = work[touched[t]];
        nb.q |= k.q;
        nb.src.insert(nb.src.end(), k.src.begin(), k.src.end());
        close(touched[t]);
      }
    nb.src.push_back(g);
    for (int q = 0; q < f.n; ++q)
      if (nb.q >> q & 1) {
        open[q] = int(work.size());
        opened.push_back(q);
      }
    work.push_back(std::move(nb));
  }
  std::vector<char> out(work.size(), 0);
  for (int q : opened)
    if (!out[open[q]]) {
      out[open[q]] = 1;
      f.blocks.push_back(work[open[q]]);
    }
}

// M <- G M on a block's rows: G (d x d) on the row digits at bit positions
// p0 (and p1; -1 for a one-qubit gate), M of D columns.
static void apply_rows(const double* gate, int p0, int p1, int D, double* M, double* tmp) {
  const int d = p1 < 0 ? 4 : 16;
  auto row_of = [&](int base, int e) {
    return p1 < 0 ? base | e << p0 : base | (e >> 2) << p0 | (e & 3) << p1;
  };
  for (int base = 0; base < D; ++base) {
    if (base >> p0 & 3 || (p1 >= 0 && base >> p1 & 3)) continue;
    std::fill(tmp, tmp + size_t(d) * D, 0.0);
    for (int o = 0; o < d; ++o)
      for (int i = 0; i < d; ++i) {
        const double u = gate[o * d + i];
        if (u == 0.0) continue;
        const double* src = M + size_t(row_of(base, i)) * D;
        double* dst = tmp + size_t(o) * D;
        for (int c = 0; c < D; ++c) dst[c] += u * src[c];
      }
    for (int o = 0; o < d; ++o)
      std::copy(tmp + size_t(o) * D, tmp + size_t(o + 1) * D, M + size_t(row_of(base, o)) * D);
  }
}

// The dense PTM of block b over its qubits in ascending order: one-qubit gates
// are folded into the next two-qubit gate on their qubit.
static void compose_block(const FusedBlocks& f, const FusedBlock& b, double* M) {
  int pos[kSlabMaxQubits], k = bits_of(b.q), c = 0;
  for (int q = 0; q < f.n; ++q)
    if (b.q >> q & 1) pos[q] = 2 * (k - 1 - c++);
  const int D = 1 << (2 * k);
  std::fill(M, M + size_t(D) * D, 0.0);
  for (int i = 0; i < D; ++i) M[size_t(i) * (D + 1)] = 1.0;
  std::vector<double> tmp(size_t(16) * D);
  std::vector<M4> pend(f.n);
  uint32_t has = 0;
  bool fresh = true;  // M is still the identity
  const M4 eye = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1};
  for (int g : b.src) {
    const double* p = f.ptms.data() + f.at[g];
    const int q0 = f.targets[2 * g], q1 = f.targets[2 * g + 1];
    if (f.ks[g] == 1) {
      M4 u;
      std::copy(p, p + 16, u.begin());
      pend[q0] = has >> q0 & 1 ? product<M4, 4>(u, pend[q0]) : u;
      has |= 1u << q0;
      continue;
    }
    M16 u;
    std::copy(p, p + 256, u.begin());
    if (has & (1u << q0 | 1u << q1))
      u = after_pair(u, has >> q0 & 1 ? pend[q0] : eye, has >> q1 & 1 ? pend[q1] : eye);
    has &= ~(1u << q0 | 1u << q1);
    if (fresh) {  // the gate's entries, the other digits unchanged
      for (int r = 0; r < D; ++r) {
        if (!(r >> pos[q0] & 3) && !(r >> pos[q1] & 3))
          for (int o = 0; o < 16; ++o)
            for (int i = 0; i < 16; ++i)
              M[size_t(r | (o >> 2) << pos[q0] | (o & 3) << pos[q1]) * D +
                (r | (i >> 2) << pos[q0] | (i & 3) << pos[q1])] = u[o * 16 + i];
      }
      fresh = false;
    } else {
      apply_rows(u.data(), pos[q0], pos[q1], D, M, tmp.data());
    }
  }
  for (int q = 0; q < f.n; ++q)
    if (has >> q & 1) apply_rows(pend[q].data(), pos[q], -1, D, M, tmp.data());
}

static int slab_check_gates(int n, int n_gates, const int32_t* ks, const int32_t* targets) {
  QSV_CHECK_ARG(n >= 2 && n <= kSlabMaxQubits, "%d qubits outside [2, %d]", n, kSlabMaxQubits);
  QSV_CHECK_ARG(n_gates >= 0 && (n_gates == 0 || (ks && targets)), "null gate list");
  for (int g = 0; g < n_gates; ++g) {
    QSV_CHECK_ARG(ks[g] == 1 || ks[g] == 2, "gate %d acts on %d qubits", g, ks[g]);
    for (int t = 0; t < ks[g]; ++t)
      QSV_CHECK_ARG(targets[2 * g + t] >= 0 && targets[2 * g + t] < n,
                    "gate %d: qubit %d does not exist", g, targets[2 * g + t]);
    QSV_CHECK_ARG(ks[g] == 1 || targets[2 * g] != targets[2 * g + 1],
                  "gate %d: qubit listed twice", g);
  }
  return QSV_OK;
}

template <bool FULL>
static int launch_slab(const SlabPass& ps, bool nt, const double* in, double* out,
                       const SlabGate* gates, hipStream_t s) {
  const size_t lds = sizeof(double) << ps.g.tbits;
  const dim3 grid(1u << ps.g.n_blk);
  if (nt)
    hipLaunchKernelGGL((k_slab<FULL, true>), grid, dim3(kSlabBlock), lds, s, in, out, ps.g,
                       gates + ps.first);
  else
    hipLaunchKernelGGL((k_slab<FULL, false>), grid, dim3(kSlabBlock), lds, s, in, out, ps.g,
                       gates + ps.first);
  QSV_CHECK_HIP(hipGetLastError());
  return QSV_OK;
}

// Host replay of every pass: loads, LDS positions, gate groups and stores.
static int emulate_slab(const SlabPlan& plan, double* v) {
  constexpr int VEC = 2;
  for (const SlabPass& ps : plan.passes) {
    const SlabGeom& g = ps.g;
    const uint32_t E = 1u << g.tbits, tiles = 1u << g.n_blk;
    std::vector<char> seen(size_t(plan.extent), 0);
    std::vector<char> tile_seen(tiles, 0);
    for (uint32_t bid = 0; bid < tiles; ++bid) {
      const uint32_t tile = slab_tile_of(bid, g.n_blk);
      QSV_CHECK_ARG(tile < tiles && !tile_seen[tile], "slab: tile %u", tile);
      tile_seen[tile] = 1;
      int64_t base = 0;
      for (int b = 0; b < g.n_blk; ++b)
        if (tile >> b & 1) base += g.bstr[b];
      std::vector<double> S(E);
      std::vector<int64_t> addr(E);
      std::vector<char> lds(E, 0);
      for (uint32_t l = 0; l < E; ++l) {
        int64_t a = base;
        for (int b = 0; b < g.tbits; ++b)
          if (l >> b & 1) a += g.tstr[b];
        QSV_CHECK_ARG(a >= 0 && a < plan.extent && !seen[a], "slab: entry %lld", (long long)a);
        QSV_CHECK_ARG(l % VEC == 0 ? a % VEC == 0 : a == addr[l - 1] + 1, "slab: vector of %lld",
                      (long long)a);
        seen[a] = 1;
        addr[l] = a;
        const uint32_t p = slab_phys(l);
        QSV_CHECK_ARG(p < E && !lds[p], "slab: LDS position %u", p);
        lds[p] = 1;
        S[p] = v[a];
      }
      for (int gi = 0; gi < g.n_gates; ++gi) {
        const SlabGate& gd = plan.gates[ps.first + gi];
        const int groups = g.tbits > 8 ? 1 << (g.tbits - 8) : 1;
        auto lane_part = [&](int l) {
          uint32_t a = 0;
          for (int i = 0; i < 6; ++i) a ^= l >> i & 1 ? gd.lane_bit[i] : 0;
          return a;
        };
        std::vector<char> used(E, 0);
        for (int gr = 0; gr < groups; ++gr) {
          double b[64][4];
          for (int l = 0; l < 64; ++l)
            for (int s = 0; s < 4; ++s) {
              const bool on = uint32_t(l & 15) < gd.lanes;
              const uint32_t a = (on ? lane_part(l) : 0) ^ gd.group[gr] ^ gd.digit[s];
              QSV_CHECK_ARG(a < E, "slab: LDS read %u", a);
              b[l][s] = S[a];
              if (on) {
                QSV_CHECK_ARG(!used[a], "slab: LDS entry %u in two orbits", a);
                used[a] = 1;
              }
            }
          for (int l = 0; l < 64; ++l) {
            if (uint32_t(l & 15) >= gd.lanes) continue;
            const int n = l & 15, j = l >> 4;
            for (int r = 0; r < 4; ++r) {
              const int row = j + 4 * r;
              double acc = 0;
              for (int s = 0; s < 4; ++s)
                for (int jk = 0; jk < 4; ++jk)
                  acc += gd.frag[4 * (row + 16 * jk) + s] * b[n + 16 * jk][s];
              S[lane_part(l) ^ gd.group[gr] ^ gd.digit[r]] = acc;
            }
          }
        }
        for (uint32_t a = 0; a < E; ++a) QSV_CHECK_ARG(used[a], "slab: LDS entry %u left out", a);
      }
      for (uint32_t l = 0; l < E; ++l) v[addr[l]] = S[slab_phys(l)];
    }
    int64_t total = 0;
    for (char c : seen) total += c;
    QSV_CHECK_ARG(total == int64_t(1) << (2 * plan.n), "slab: %lld entries", (long long)total);
  }
  return QSV_OK;
}

}  // namespace qsv

using namespace qsv;

extern "C" int qsv_circuit_blocks_create(int n_qubits, int n_gates, const int32_t* ks,
                                         const int32_t* targets, const double* ptms,
                                         int max_qudits, void** blocks_out) {
  if (const int rc = slab_check_gates(n_qubits, n_gates, ks, targets)) return rc;
  QSV_CHECK_ARG(blocks_out && (ptms || n_gates == 0), "null pointer argument");
  try {
    std::unique_ptr<FusedBlocks> f(new FusedBlocks);
    f->n = n_qubits;
    f->ks.assign(ks, ks + n_gates);
    f->targets.assign(targets, targets + 2 * n_gates);
    int64_t size = 0;
    for (int g = 0; g < n_gates; ++g) {
      f->at.push_back(size);
      size += ks[g] == 1 ? 16 : 256;
    }
    f->ptms.assign(ptms, ptms + size);
    // x - x is 0 for finite x only: sixteen sums (every PTM is a multiple of that), no
    // branch an entry
    double odd[16] = {};
    for (int64_t i = 0; i < size; i += 16)
      for (int e = 0; e < 16; ++e) odd[e] += ptms[i + e] - ptms[i + e];
    if (std::any_of(odd, odd + 16, [](double x) { return x != 0.0; })) {
      set_error("PTM entries that are not finite");
      return QSV_ENOTSUP;
    }
    fuse_blocks(max_qudits, *f);
    *blocks_out = f.release();
    return QSV_OK;
  } catch (const std::bad_alloc&) {
    set_error("out of host memory");
    return QSV_EINVAL;
  }
}

extern "C" void qsv_circuit_blocks_destroy(void* blocks) {
  delete static_cast<FusedBlocks*>(blocks);
}

extern "C" int qsv_circuit_blocks_count(const void* blocks) {
  return int(static_cast<const FusedBlocks*>(blocks)->blocks.size());
}

// A pass pays for each of its two-qubit gates, a dense block once.  Milliseconds
// as measured: on 14 qubits (2 GB) a pass takes 0.37 and 0.145 a gate, at least 0.72
// (its traffic); a dense block 0.72, 0.75, 0.9 and 2.0 for one to four qubits; in
// proportion to the vector otherwise.  The host spends 4 us a gate on the passes,
// 10.5 a gate and 30 a block on the blocks.  So passes on brickwork (14 qubits, 60
// gates: 13.0 ms against 28.2) and on small vectors, blocks where many gates meet on
// few qubits (two triples of qubits, 200 gates: 2.9 ms against 31.2).
extern "C" int qsv_circuit_pays(const void* plan, const void* blocks) {
  const SlabPlan* p = static_cast<const SlabPlan*>(plan);
  const FusedBlocks* f = static_cast<const FusedBlocks*>(blocks);
  if (!p || !f) return 0;
  const double scale = ldexp(1.0, 2 * (p->n - 14)), gates = double(f->ks.size());
  const double np = double(p->passes.size()), ng = double(p->gates.size());
  const double passes = scale * std::max(0.72 * np, 0.37 * np + 0.145 * ng) + 0.004 * gates;
  const double once[4] = {0.72, 0.72, 0.75, 0.9};
  double dense = 0.0105 * gates;
  for (const FusedBlock& b : f->blocks) {
    const int k = bits_of(b.q);
    dense += scale * (k < 4 ? once[k] : ldexp(2.0, 2 * (k - 4))) + 0.03;
  }
  return passes <= dense;
}

extern "C" int qsv_circuit_block_qubits(const void* blocks, int index, int32_t* qubits) {
  const FusedBlocks* f = static_cast<const FusedBlocks*>(blocks);
  QSV_CHECK_ARG(f && qubits && index >= 0 && index < int(f->blocks.size()), "no block %d", index);
  int k = 0;
  for (int q = 0; q < f->n; ++q)
    if (f->blocks[index].q >> q & 1) qubits[k++] = q;
  return k;
}

extern "C" int qsv_circuit_block_ptm(const void* blocks, int index, double* ptm) {
  const FusedBlocks* f = static_cast<const FusedBlocks*>(blocks);
  QSV_CHECK_ARG(f && ptm && index >= 0 && index < int(f->blocks.size()), "no block %d", index);
  try {
    compose_block(*f, f->blocks[index], ptm);
    return QSV_OK;
  } catch (const std::bad_alloc&) {
    set_error("out of host memory");
    return QSV_EINVAL;
  }
}

extern "C" int qsv_circuit_create(int n_qubits, const int64_t* strides, int n_gates,
                                  const int32_t* ks, const int32_t* targets, const double* ptms,
                                  void** plan_out) {
  if (const int rc = slab_check_gates(n_qubits, n_gates, ks, targets)) return rc;
  QSV_CHECK_ARG(strides && plan_out && (ptms || n_gates == 0), "null pointer argument");
  int64_t acc = 1;
  for (int q = n_qubits - 1; q >= 0; --q) {
    QSV_CHECK_ARG(strides[q] >= acc && strides[q] < (int64_t(1) << 40),
                  "strides of axis %d overlap the axes below it", q);
    // runs of whole 16-byte vectors: the innermost axis has stride 1 and the lowest
    // bits nest without a gap
    if (strides[q] < 8 || q == n_qubits - 1 ? strides[q] != acc : strides[q] % 8 != 0) {
      set_error("circuit passes need axes that nest in aligned runs of 64 bytes");
      return QSV_ENOTSUP;
    }
    acc = strides[q] * 4;
  }
  try {
    std::unique_ptr<SlabPlan> p(new SlabPlan);
    const int rc = slab_compile(n_qubits, strides, acc, n_gates, ks, targets, ptms, *p);
    if (rc) return rc;
    *plan_out = p.release();
    return QSV_OK;
  } catch (const std::bad_alloc&) {
    set_error("out of host memory");
    return QSV_EINVAL;
  }
}

extern "C" void qsv_circuit_destroy(void* plan) { delete static_cast<SlabPlan*>(plan); }

extern "C" int qsv_circuit_passes(const void* plan) {
  return int(static_cast<const SlabPlan*>(plan)->passes.size());
}

extern "C" int64_t qsv_circuit_table_bytes(const void* plan) {
  const SlabPlan* p = static_cast<const SlabPlan*>(plan);
  return int64_t(p->gates.size() * sizeof(SlabGate));
}

extern "C" int qsv_circuit_table(const void* plan, void* host) {
  const SlabPlan* p = static_cast<const SlabPlan*>(plan);
  QSV_CHECK_ARG(p && host, "null pointer argument");
  if (!p->gates.empty()) memcpy(host, p->gates.data(), p->gates.size() * sizeof(SlabGate));
  return QSV_OK;
}

extern "C" int qsv_circuit_run(const void* plan, const void* in, void* out, const void* table_dev,
                               void* stream) {
  const SlabPlan* p = static_cast<const SlabPlan*>(plan);
  QSV_CHECK_ARG(p && in && out && (table_dev || p->passes.empty()), "null pointer argument");
  QSV_CHECK_ARG(reinterpret_cast<uintptr_t>(in) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(table_dev) % 16 == 0,
                "pointers must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const double* src = static_cast<const double*>(in);
  double* dst = static_cast<double*>(out);
  const SlabGate* gates = static_cast<const SlabGate*>(table_dev);
  const bool big = 2 * p->extent * 8 > nt_threshold_bytes();
  if (p->passes.empty() && in != out)  // no gates
    QSV_CHECK_HIP(hipMemcpyAsync(out, in, p->extent * 8, hipMemcpyDeviceToDevice, s));
  for (const SlabPass& ps : p->passes) {
    // nontemporal only on whole lines, as in the other kernels
    const bool nt = big && ps.run128;
    const int rc = ps.full ? launch_slab<true>(ps, nt, src, dst, gates, s)
                           : launch_slab<false>(ps, nt, src, dst, gates, s);
    if (rc) return rc;
    src = dst;  // later passes work in place
  }
  return QSV_OK;
}

// Replays the passes on the CPU (float64 arithmetic, in place on `v`, the
// plan's physical layout), checking every access.  Diagnostic only.
extern "C" int qsv_emulate_circuit(const void* plan, double* v) {
  const SlabPlan* p = static_cast<const SlabPlan*>(plan);
  QSV_CHECK_ARG(p && v, "null pointer argument");
  QSV_CHECK_ARG(p->extent <= (int64_t(1) << 24), "emulation is for small vectors");
  return emulate_slab(*p, v);
}
