// PTM gradients whose final sums a caller launches itself, several at a time.
#pragma once

#include "qsv_common.h"

namespace qsv {

// The block partials of one gradient [batch][nb][dd] and where their sum goes.
struct GradFinal {
  const double* partial;
  void* out;
  int nb, dd;
};
constexpr int kGradFinals = 16;
struct GradFinals {
  int n;
  GradFinal it[kGradFinals];
};

// Final sums of up to kGradFinals gradients of `batch` states in one launch.
int launch_grad_finals(int dtype, const GradFinals& finals, int batch, int accumulate,
                       hipStream_t s);

// qsv_ptm_grad_tiled and qsv_apply_ptm_batched_backward without their final sum,
// which is appended to `finals`; the partials take nb * dd * batch doubles of
// `workspace`.
int ptm_grad_partials(int dtype, const void* x, const void* ybar, int batch, int rank,
                      const int64_t* dims, int k, const int32_t* targets,
                      const int32_t* dims_out_t, void* dptm, void* workspace,
                      int64_t workspace_bytes, const qsv_tile* tile, GradFinals& finals,
                      void* stream);
int batched_backward_partials(int dtype, const void* x, const void* ybar, void* xbar, int batch,
                              int rank, const int64_t* dims, int k, const int32_t* targets,
                              const void* ptm_dev, int64_t ptm_batch_stride, void* dptm,
                              void* workspace, int64_t workspace_bytes, GradFinals& finals,
                              void* stream);

}  // namespace qsv
