// Trigonometric factors of RZ(b) RX(a) and damping PTMs of the layered circuits'
// parameters in one launch, and the parameters' gradients in one more.
//
// The PTM of a rotation is a product of nine factors f_j(b) f_i(a),
// f = (1, cos, sin), with a constant [9][16] matrix.  By tensor operations the
// factors, the damping (Kraus sets, two complex contractions, a product) and the
// backwards of both take about 160 launches of a few microseconds each for a few
// hundred kilobytes: four circuit widths spent 5 ms of host time a training step on
// them.  Here a thread makes one rotation's factors, or one entry of a damping
// PTM, and the backward contracts a rotation's sixteen PTM gradients, staged in
// LDS, with the terms.  192 circuits of 4-7 qubits, 20-80 layers: training step
// 9.0 -> 4.5 ms.  Bound by its launches below about a million angles.
//
// The forward rounds as the tensor operations do (products one by one, the two
// equal terms of a contraction by a fused multiply-add), so the damping PTMs and,
// through the same product, the rotations are the same bit for bit.
//
// Reference: quantumsim/operations/qubits.py:38-90, 182-214 (Kraus sets),
// quantumsim/algebra/algebra.py:11-30 (PTM of a Kraus set).
#include "qsv_common.h"

#include <math.h>

#include <algorithm>
#include <vector>

namespace qsv {

constexpr int kParamBlock = 256;

// Rotation r of [batch][layers][n] -> its angle pair in [batch][own][n], or -1
// where the layer is past the circuit's own (angles 0).
__host__ __device__ inline int64_t rot_angle(int64_t r, int layers, int own, int n) {
  const int64_t per = int64_t(layers) * n, b = r / per, in = r - b * per;
  return in < int64_t(own) * n ? b * own * n + in : -1;
}

// coef[3 j + i] = f_j(b) f_i(a), f = (1, cos, sin).
__host__ __device__ inline void rot_coef(double ca, double sa, double cb, double sb,
                                         double (&coef)[9]) {
  const double fa[3] = {1.0, ca, sa}, fb[3] = {1.0, cb, sb};
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 3; ++i) coef[3 * j + i] = fb[j] * fa[i];
}

// dL/d(a, b) from dL/dcoef.
__host__ __device__ inline void rot_grad(double ca, double sa, double cb, double sb,
                                         const double (&dc)[9], double& da, double& db) {
  const double fa[3] = {1.0, ca, sa}, fb[3] = {1.0, cb, sb};
  da = db = 0.0;
#pragma unroll
  for (int j = 0; j < 3; ++j) da += fb[j] * (ca * dc[3 * j + 2] - sa * dc[3 * j + 1]);
#pragma unroll
  for (int i = 0; i < 3; ++i) db += fa[i] * (cb * dc[6 + i] - sb * dc[3 + i]);
}

// Damping for a time t: gamma = 1 - e^(-t/T1), lambda = 1 - e^(-2 t/Tphi),
// 1/Tphi = 1/T2 - 1/(2 T1); operations rounded one by one.
struct DampRates {
  double g, lam, i1, i2;  // i1 = 1/T1, i2 = 1/T2
};
__host__ __device__ inline DampRates damp_rates(double t1, double t2, double t) {
#pragma clang fp contract(off)
  DampRates r;
  r.i1 = 1.0 / t1;
  r.i2 = 1.0 / t2;
  r.g = 1.0 - exp(r.i1 * -t);
  r.lam = 1.0 - exp((r.i2 - r.i1 * 0.5) * (-2.0 * t));
  return r;
}
// Entry e of the product PTM (general(2) basis: |0><0|, |1><1|, X, Y).  A rate
// outside [0, 1] has no Kraus operator: not a number, everywhere.
__host__ __device__ inline double damp_entry(const DampRates& r, int e) {
#pragma clang fp contract(off)
  if (!(r.g >= 0.0 && 1.0 - r.g >= 0.0 && r.lam >= 0.0 && 1.0 - r.lam >= 0.0)) return NAN;
  const double h = 0.70710678118654757;  // X entries of the basis
  const double sg = sqrt(1.0 - r.g), qg = sqrt(r.g), sl = sqrt(1.0 - r.lam), ql = sqrt(r.lam);
  const double xa = h * sg, xp = h * sl;
  const double axx = fma(h, xa, h * xa), pxx = fma(h, xp, h * xp);
  switch (e) {
    case 0: return 1.0;
    case 1: return qg * qg;
    case 5: return fma(ql, ql, sl * sl) * (sg * sg);
    case 10:
    case 15: return pxx * axx;
    default: return 0.0;
  }
}
// dL/d(T1, T2) from dL/dPTM: entries (0, 1) = gamma, (1, 1) = 1 - gamma, (2, 2) =
// (3, 3) = sqrt((1 - gamma)(1 - lambda)).
__host__ __device__ inline void damp_grad(const DampRates& r, double t, double d01, double d11,
                                          double dxy, double& dt1, double& dt2) {
  const double sg = sqrt(1.0 - r.g), sl = sqrt(1.0 - r.lam);
  const double dg = d01 - d11 - 0.5 * dxy * sl / sg;
  const double dl = -0.5 * dxy * sg / sl;
  const double eg = 1.0 - r.g, el = 1.0 - r.lam;
  dt1 = -dg * eg * t * r.i1 * r.i1 + dl * el * t * r.i1 * r.i1;
  dt2 = -2.0 * dl * el * t * r.i2 * r.i2;
}

// Workgroups [0, rot_blocks): factors; the others: 16 damping PTMs each.
__global__ void __launch_bounds__(kParamBlock)
    k_gate_params(const double* __restrict__ angles, int64_t n_rot, int layers, int own, int n,
                  double* __restrict__ coef, uint32_t rot_blocks, const double* __restrict__ t1,
                  const double* __restrict__ t2, int64_t n_damp, double t,
                  double* __restrict__ damp) {
  const int tid = threadIdx.x;
  if (blockIdx.x >= rot_blocks) {
    const int64_t q = int64_t(blockIdx.x - rot_blocks) * (kParamBlock / 16) + (tid >> 4);
    if (q < n_damp) damp[q * 16 + (tid & 15)] = damp_entry(damp_rates(t1[q], t2[q], t), tid & 15);
    return;
  }
  const int64_t r = int64_t(blockIdx.x) * kParamBlock + tid;
  if (r >= n_rot) return;
  const int64_t at = rot_angle(r, layers, own, n);
  const double a = at < 0 ? 0.0 : angles[2 * at], b = at < 0 ? 0.0 : angles[2 * at + 1];
  double c[9];
  rot_coef(cos(a), sin(a), cos(b), sin(b), c);
#pragma unroll
  for (int k = 0; k < 9; ++k) coef[r * 9 + k] = c[k];
}

// Over the circuits' own layers: a workgroup stages its 256 PTM
// gradients in LDS (rows of 17: bank conflict free by rotation), a thread
// contracts one with the terms.
__global__ void __launch_bounds__(kParamBlock)
    k_gate_params_bwd(const double* __restrict__ angles, const double* __restrict__ terms,
                    int64_t n_own, int layers, int own, int n, const double* __restrict__ drot,
                    double* __restrict__ dangles, uint32_t rot_blocks,
                    const double* __restrict__ t1, const double* __restrict__ t2, int64_t n_damp,
                    double t, const double* __restrict__ ddamp, double* __restrict__ dt1,
                    double* __restrict__ dt2) {
  __shared__ double dp[kParamBlock][17];
  __shared__ double m[144];
  const int tid = threadIdx.x, e = tid & 15;
  if (blockIdx.x >= rot_blocks) {
    const int64_t q = int64_t(blockIdx.x - rot_blocks) * kParamBlock + tid;
    if (q < n_damp) {
      const double* d = ddamp + q * 16;
      damp_grad(damp_rates(t1[q], t2[q], t), t, d[1], d[5], d[10] + d[15], dt1[q], dt2[q]);
    }
    return;
  }
  const int64_t r0 = int64_t(blockIdx.x) * kParamBlock;  // of the own rotations
  const int64_t per = int64_t(own) * n;
  for (int i = 0; i < 16; ++i) {
    const int r = i * 16 + (tid >> 4);
    if (r0 + r >= n_own) break;
    const int64_t b = (r0 + r) / per;
    dp[r][e] = drot[((r0 + r) + b * int64_t(layers - own) * n) * 16 + e];
  }
  if (tid < 144) m[tid] = terms[tid];
  __syncthreads();
  if (r0 + tid >= n_own) return;
  double dc[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    dc[k] = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) dc[k] += m[k * 16 + i] * dp[tid][i];
  }
  const double a = angles[2 * (r0 + tid)], b = angles[2 * (r0 + tid) + 1];
  double da, db;
  rot_grad(cos(a), sin(a), cos(b), sin(b), dc, da, db);
  dangles[2 * (r0 + tid)] = da;
  dangles[2 * (r0 + tid) + 1] = db;
}

static int check_params(int batch, int layers, int own, int n) {
  QSV_CHECK_ARG(batch >= 0 && n >= 1 && own >= 0 && layers >= own, "bad gate parameter shape");
  QSV_CHECK_ARG(int64_t(batch) * std::max(layers, 1) * n < (int64_t(1) << 31),
                "too many gate parameters");
  return QSV_OK;
}

}  // namespace qsv

using namespace qsv;

extern "C" int qsv_gate_params(int batch, int layers, int own, int n, const double* angles,
                               double* coef, const double* t1, const double* t2, double t,
                               double* damp, void* stream) {
  if (const int rc = check_params(batch, layers, own, n)) return rc;
  const int64_t n_rot = int64_t(batch) * layers * n, n_damp = int64_t(batch) * n;
  if (n_damp == 0) return QSV_OK;
  QSV_CHECK_ARG((angles || own == 0) && (coef || layers == 0) && t1 && t2 && damp,
                "null pointer argument");
  const uint32_t rb = ceil_div_u32(n_rot, kParamBlock);
  const uint32_t db = ceil_div_u32(n_damp, kParamBlock / 16);
  hipLaunchKernelGGL(k_gate_params, dim3(rb + db), dim3(kParamBlock), 0,
                     static_cast<hipStream_t>(stream), angles, n_rot, layers, own, n, coef, rb, t1,
                     t2, n_damp, t, damp);
  QSV_CHECK_HIP(hipGetLastError());
  return QSV_OK;
}

extern "C" int qsv_gate_params_backward(int batch, int layers, int own, int n, const double* angles,
                                        const double* terms, const double* drot,
                                        double* dangles, const double* t1, const double* t2,
                                        double t, const double* ddamp, double* dt1, double* dt2,
                                        void* stream) {
  if (const int rc = check_params(batch, layers, own, n)) return rc;
  const int64_t n_own = int64_t(batch) * own * n, n_damp = int64_t(batch) * n;
  if (n_damp == 0) return QSV_OK;
  QSV_CHECK_ARG((own == 0 || (angles && drot && dangles)) && terms && t1 && t2 && ddamp && dt1 &&
                    dt2, "null pointer argument");
  const uint32_t rb = ceil_div_u32(n_own, kParamBlock);
  const uint32_t db = ceil_div_u32(n_damp, kParamBlock);
  hipLaunchKernelGGL(k_gate_params_bwd, dim3(rb + db), dim3(kParamBlock), 0,
                     static_cast<hipStream_t>(stream), angles, terms, n_own, layers, own, n, drot,
                     dangles, rb, t1, t2, n_damp, t, ddamp, dt1, dt2);
  QSV_CHECK_HIP(hipGetLastError());
  return QSV_OK;
}

// Host replay: the same index maps and formulas on host arrays (drot may be
// null: forward only).
extern "C" int qsv_emulate_gate_params(int batch, int layers, int own, int n, const double* angles,
                                       const double* terms, double* coef, const double* t1,
                                       const double* t2, double t, double* damp,
                                       const double* drot, double* dangles, const double* ddamp,
                                       double* dt1, double* dt2) {
  if (const int rc = check_params(batch, layers, own, n)) return rc;
  const int64_t n_rot = int64_t(batch) * layers * n, n_own = int64_t(batch) * own * n;
  std::vector<int> used(n_own, 0);
  for (int64_t r = 0; r < n_rot; ++r) {
    const int64_t at = rot_angle(r, layers, own, n);
    QSV_CHECK_ARG(at < n_own, "angle %lld out of range", (long long)at);
    const double a = at < 0 ? 0.0 : angles[2 * at], b = at < 0 ? 0.0 : angles[2 * at + 1];
    double c[9];
    rot_coef(cos(a), sin(a), cos(b), sin(b), c);
    for (int k = 0; k < 9; ++k) coef[r * 9 + k] = c[k];
    if (at >= 0) ++used[at];
  }
  for (int64_t i = 0; i < n_own; ++i)
    QSV_CHECK_ARG(used[i] == 1, "angle %lld used %d times", (long long)i, used[i]);
  for (int64_t q = 0; q < int64_t(batch) * n; ++q) {
    const DampRates r = damp_rates(t1[q], t2[q], t);
    for (int e = 0; e < 16; ++e) damp[q * 16 + e] = damp_entry(r, e);
    if (drot) {
      const double* d = ddamp + q * 16;
      damp_grad(r, t, d[1], d[5], d[10] + d[15], dt1[q], dt2[q]);
    }
  }
  if (!drot) return QSV_OK;
  for (int64_t r = 0; r < n_own; ++r) {
    const int64_t from = r + r / (int64_t(own) * n) * int64_t(layers - own) * n;
    QSV_CHECK_ARG(from < n_rot && rot_angle(from, layers, own, n) == r, "rotation %lld",
                  (long long)r);
    double dc[9];
    for (int k = 0; k < 9; ++k) {
      dc[k] = 0.0;
      for (int i = 0; i < 16; ++i) dc[k] += terms[k * 16 + i] * drot[from * 16 + i];
    }
    const double a = angles[2 * r], b = angles[2 * r + 1];
    rot_grad(cos(a), sin(a), cos(b), sin(b), dc, dangles[2 * r], dangles[2 * r + 1]);
  }
  return QSV_OK;
}
