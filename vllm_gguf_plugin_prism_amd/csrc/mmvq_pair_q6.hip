// Pairs of formats on one launch of the GEMV (mmvq_pair.h): Q4_K and Q5_K with Q6_K.
#include "mmvq_pair.h"

namespace gguf {
int mmvq_pair_q6(const TsShard& a, const TsShard& b, const void* x, int dtype, int K, int M, hipStream_t s) {
  if (a.type == T_Q4_K) return pair_fmt<FmtQ4_K, FmtQ6_K>(a, b, x, dtype, K, M, s);
  if (a.type == T_Q5_K) return pair_fmt<FmtQ5_K, FmtQ6_K>(a, b, x, dtype, K, M, s);
  return GGUF_NOT_TAKEN;
}
}  // namespace gguf
