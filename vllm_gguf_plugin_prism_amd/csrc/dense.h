// The GEMM of the codebook formats on the matrix unit (dense_core.h), for the code that routes to it.
#pragma once
#include "tile_runs.h"

namespace gguf {

struct DenseCall {
  const void *W, *X;
  void* Y;
  int dtype, M, N, K;
  float* partial;
  LinearArgs la;
};

double dense_us(int M, int N, int K);   // about how long it takes

int dense_iq4_xs(const DenseCall& c, const TilePlan& p, hipStream_t s);
int dense_iq4_nl(const DenseCall& c, const TilePlan& p, hipStream_t s);
int dense_iq2_xxs(const DenseCall& c, const TilePlan& p, hipStream_t s);
int dense_iq2_xs(const DenseCall& c, const TilePlan& p, hipStream_t s);
int dense_iq2_s(const DenseCall& c, const TilePlan& p, hipStream_t s);
int dense_iq3_xxs(const DenseCall& c, const TilePlan& p, hipStream_t s);
int dense_iq3_s(const DenseCall& c, const TilePlan& p, hipStream_t s);
int dense_iq1_s(const DenseCall& c, const TilePlan& p, hipStream_t s);
int dense_iq1_m(const DenseCall& c, const TilePlan& p, hipStream_t s);

}  // namespace gguf
