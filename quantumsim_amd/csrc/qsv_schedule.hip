// The launches of a batched gate schedule, issued from one call per segment.
//
// A batch of 8-11-qubit circuits makes about 1650 launches a training step, each
// of 10-50 us on the device; issued one library call at a time from the
// interpreter they cost 13 us each on the host (allocation, views, argument
// arrays), 28 of the step's 32 ms, with the device idle between them.  The same
// calls in the same order from here cost 4-5 us each.
//
// Host code only: the entries it calls check their own arguments; the stream,
// the buffers' sizes and the order of use are the caller's (one segment: `active`
// states, gates in application order).
#include "qsv_grad.h"

namespace qsv {

static const void* step_ptr(const void* base, int64_t elems, int es) {
  return static_cast<const char*>(base) + elems * es;
}

static int check_segment(int dtype, int n_pos, const qsv_sched_pos* pos, int active, int n_gates,
                         const int32_t* gates) {
  QSV_CHECK_ARG(dtype_size(dtype) > 0, "unknown dtype %d", dtype);
  QSV_CHECK_ARG(active >= 0 && active <= 65535 && n_gates >= 0 && n_pos >= 0,
                "bad schedule segment");
  QSV_CHECK_ARG(n_gates == 0 || (pos && gates), "null pointer argument");
  for (int g = 0; g < n_gates; ++g) {
    const int p = gates[2 * g], w = gates[2 * g + 1];
    QSV_CHECK_ARG(p >= 0 && p < n_pos && w >= 0 && w < pos[p].n_steps,
                  "gate %d: (%d, %d) outside the steps", g, p, w);
    QSV_CHECK_ARG(pos[p].k >= 1 && pos[p].k <= QSV_MAX_TARGETS, "position %d: %d targets", p,
                  pos[p].k);
  }
  return QSV_OK;
}

// The launches of one gate, each between two calls of the hook (if any).
struct Segment {
  int dtype, es, rank, active;
  const int64_t* dims;
  const qsv_sched_pos* pos;
  qsv_sched_hook hook;
  void* stream;

  template <typename F>
  int launch(int kind, int p, F f) const {
    if (hook) hook(0, kind, p, active);
    const int rc = f();
    if (hook && rc == QSV_OK) hook(1, kind, p, active);
    return rc;
  }
  void dout(int p, int32_t (&d)[QSV_MAX_TARGETS]) const {
    for (int j = 0; j < pos[p].k; ++j) {
      const int t = pos[p].targets[j];
      d[j] = t >= 0 && t < rank ? int32_t(dims[t]) : 0;
    }
  }
  int apply(int p, const void* x, void* y, const void* ptm) const {
    const qsv_sched_pos& P = pos[p];
    int32_t d[QSV_MAX_TARGETS];
    dout(p, d);
    return launch(QSV_SCHED_APPLY, p, [&] {
      return qsv_apply_ptm_batched_tiled(dtype, x, y, active, rank, dims, P.k, P.targets, d, ptm,
                                         P.state, P.has_apply ? &P.apply : nullptr, stream);
    });
  }
  // Gradients leave their partials behind one another in the workspace; the
  // sums of sixteen, or of what fits, are one launch.
  char* ws;
  int64_t ws_bytes, ws_used = 0;
  GradFinals finals = {};
  int sums() {
    ws_used = 0;
    const int rc = launch_grad_finals(dtype, finals, active, 0, static_cast<hipStream_t>(stream));
    finals.n = 0;
    return rc;
  }
  template <typename F>
  int gradient(int kind, int p, F f) {
    const int64_t most = pos[p].workspace;
    if (finals.n == kGradFinals || ws_used + most > ws_bytes)
      if (const int rc = sums()) return rc;
    return launch(kind, p, [&] {
      const int before = finals.n;
      const int rc = f(ws + ws_used, most < ws_bytes - ws_used ? most : ws_bytes - ws_used);
      if (rc || finals.n == before) return rc;  // no states: no partials
      const GradFinal& l = finals.it[finals.n - 1];
      ws_used += (int64_t(l.nb) * l.dd * active * 8 + 255) / 256 * 256;
      return hook ? sums() : int(QSV_OK);  // a counted launch has its sum with it
    });
  }
  int grad(int p, const void* x, const void* gy, void* gp) {
    const qsv_sched_pos& P = pos[p];
    int32_t d[QSV_MAX_TARGETS];
    dout(p, d);
    return gradient(QSV_SCHED_GRAD, p, [&](void* part, int64_t bytes) {
      return ptm_grad_partials(dtype, x, gy, active, rank, dims, P.k, P.targets, d, gp, part,
                               bytes, P.has_grad ? &P.grad : nullptr, finals, stream);
    });
  }
  int backward(int p, const void* x, const void* gy, void* gx, const void* ptm, void* gp) {
    const qsv_sched_pos& P = pos[p];
    return gradient(QSV_SCHED_BACKWARD, p, [&](void* part, int64_t bytes) {
      return batched_backward_partials(dtype, x, gy, gx, active, rank, dims, P.k, P.targets, ptm,
                                       P.state, gp, part, bytes, finals, stream);
    });
  }
};

}  // namespace qsv

using namespace qsv;

extern "C" int qsv_schedule_forward(int dtype, int rank, const int64_t* dims, int n_pos,
                                    const qsv_sched_pos* pos, int active, int n_gates,
                                    const int32_t* gates, const void* x, void* const* outs,
                                    qsv_sched_hook hook, void* stream) {
  if (const int rc = check_segment(dtype, n_pos, pos, active, n_gates, gates)) return rc;
  QSV_CHECK_ARG(dims && (n_gates == 0 || (x && outs)), "null pointer argument");
  const Segment S = {dtype, dtype_size(dtype), rank, active, dims, pos, hook, stream, nullptr, 0};
  for (int g = 0; g < n_gates; ++g) {
    const int p = gates[2 * g], w = gates[2 * g + 1];
    const int rc = S.apply(p, x, outs[g], step_ptr(pos[p].ptm, w * pos[p].step, S.es));
    if (rc) return rc;
    x = outs[g];
  }
  return QSV_OK;
}

extern "C" int qsv_schedule_backward(int dtype, int rank, const int64_t* dims, int n_pos,
                                     const qsv_sched_pos* pos, int active, int n_gates,
                                     const int32_t* gates, int every, const void* const* kept,
                                     void* const* between, void* const* bufs, int cur,
                                     void* workspace, int64_t workspace_bytes, int* cur_out, qsv_sched_hook hook,
                                     void* stream) {
  if (const int rc = check_segment(dtype, n_pos, pos, active, n_gates, gates)) return rc;
  QSV_CHECK_ARG(dims && bufs && cur_out && every >= 1 && (cur == 0 || cur == 1),
                "bad schedule arguments");
  QSV_CHECK_ARG(n_gates == 0 || (kept && bufs[0] && bufs[1]), "null pointer argument");
  Segment S = {dtype, dtype_size(dtype), rank, active, dims, pos, hook, stream,
               static_cast<char*>(workspace), workspace_bytes};
  auto al = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; };
  for (int c = (n_gates + every - 1) / every - 1; c >= 0; --c) {
    const int lo = c * every, hi = n_gates < lo + every ? n_gates : lo + every;
    // the states before gates lo + 1 .. hi - 1, again
    for (int g = lo; g + 1 < hi; ++g) {
      const int p = gates[2 * g], w = gates[2 * g + 1];
      const int rc = S.apply(p, g == lo ? kept[c] : between[g - lo - 1], between[g - lo],
                             step_ptr(pos[p].ptm, w * pos[p].step, S.es));
      if (rc) return rc;
    }
    for (int g = hi - 1; g >= lo; --g) {
      const int p = gates[2 * g], w = gates[2 * g + 1];
      const qsv_sched_pos& P = pos[p];
      const void* x = g == lo ? kept[c] : between[g - lo - 1];
      const void* gy = bufs[cur];
      void* gx = bufs[1 - cur];
      const int64_t at = w * P.step;
      void* gp = P.grad_ptm ? const_cast<void*>(step_ptr(P.grad_ptm, at, S.es)) : nullptr;
      int rc;
      if (gp && P.fused && al(x) && al(gy) && al(gx)) {
        rc = S.backward(p, x, gy, gx, step_ptr(P.ptm, at, S.es), gp);
      } else {
        QSV_CHECK_ARG(P.ptm_t, "position %d: no transposed PTMs", p);
        rc = gp ? S.grad(p, x, gy, gp) : QSV_OK;
        if (!rc) rc = S.apply(p, gy, gx, step_ptr(P.ptm_t, at, S.es));
      }
      if (rc) return rc;
      cur = 1 - cur;
    }
  }
  if (const int rc = S.sums()) return rc;
  *cur_out = cur;
  return QSV_OK;
}
