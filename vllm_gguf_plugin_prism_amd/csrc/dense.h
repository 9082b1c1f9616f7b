// The GEMM of the codebook formats on the matrix unit (dense_core.h), for the code that routes to it.
#pragma once
#include "gguf_common.h"

namespace gguf {

struct DenseCall {
  const void *W, *X;
  void* Y;
  int dtype, M, N, K;
  float* partial;
  LinearArgs la;
};

// Tiles of `mt` rows of X by 128 weight rows.  `whole` tiles get a workgroup each; the units of 256 values of the `shared`
// tiles behind them, one tile after the other, are dealt to `workers` workgroups in runs of `per`, which leave fp32
// partial tiles, two each at most.
struct DensePlan {
  int mt, whole, shared, workers, per;
  int64_t partial_bytes() const { return (int64_t)workers * 2 * mt * 128 * 4; }
};

int dense_iq4_xs(const DenseCall& c, const DensePlan& p, hipStream_t s);
int dense_iq4_nl(const DenseCall& c, const DensePlan& p, hipStream_t s);
int dense_iq2_xxs(const DenseCall& c, const DensePlan& p, hipStream_t s);
int dense_iq2_xs(const DenseCall& c, const DensePlan& p, hipStream_t s);
int dense_iq2_s(const DenseCall& c, const DensePlan& p, hipStream_t s);
int dense_iq3_xxs(const DenseCall& c, const DensePlan& p, hipStream_t s);
int dense_iq3_s(const DenseCall& c, const DensePlan& p, hipStream_t s);
int dense_iq1_s(const DenseCall& c, const DensePlan& p, hipStream_t s);
int dense_iq1_m(const DenseCall& c, const DensePlan& p, hipStream_t s);

}  // namespace gguf
