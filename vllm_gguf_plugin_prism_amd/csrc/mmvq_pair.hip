// Pairs of formats on one launch of the GEMV (mmvq_pair.h): what the recipes mix that give one of a layer's tensors more bits.
#include "mmvq_pair.h"

namespace gguf {

int mmvq_pair_q6(const TsShard& a, const TsShard& b, const void* x, int dtype, int K, int M, hipStream_t s);

static int pair_any(const TsShard& a, const TsShard& b, const void* x, int dtype, int K, int M, hipStream_t s) {
  if (b.type == T_Q6_K) return mmvq_pair_q6(a, b, x, dtype, K, M, s);
  if (a.type == T_Q3_K && b.type == T_Q5_K) return pair_fmt<FmtQ3_K, FmtQ5_K>(a, b, x, dtype, K, M, s);
  if (a.type == T_IQ4_XS && b.type == T_Q5_K) return pair_fmt<FmtIQ4_XS, FmtQ5_K>(a, b, x, dtype, K, M, s);
  return GGUF_NOT_TAKEN;
}
int mmvq_pair(const TsShard& a, const TsShard& b, const void* x, int dtype, int K, int M, hipStream_t s) {
  const int rc = pair_any(a, b, x, dtype, K, M, s);
  return rc != GGUF_NOT_TAKEN ? rc : pair_any(b, a, x, dtype, K, M, s);
}

// Where the matrices are more than some tens of megabytes the launch saved is little beside them, and the larger one's own ways of
// fetching are the better ones (one row, 60 to 250 MB: two launches 0.93 to 1.4 times as long; K below 2048, 20 to 60 MB: 0.90 to 1.16).
bool mmvq_pair_takes(int type, int64_t N, int64_t w_pitch, int type2, int64_t N2, int64_t w_pitch2, int64_t K, int64_t M) {
  const auto is = [&](int t, int u) { return (type == t && type2 == u) || (type == u && type2 == t); };
  if (!is(T_Q4_K, T_Q6_K) && !is(T_Q5_K, T_Q6_K) && !is(T_Q3_K, T_Q5_K) && !is(T_IQ4_XS, T_Q5_K)) return false;
  if (M < 1 || M > 4 || K > 32768 || N > 0x7FFFFF0ll || N2 > 0x7FFFFF0ll || w_pitch > (int64_t)UINT32_MAX || w_pitch2 > (int64_t)UINT32_MAX) return false;
  const int64_t bytes = K / 256 * (N * block_bytes(type) + N2 * block_bytes(type2));
  return bytes <= (K < 2048 ? 20000000 : 60000000);
}

}  // namespace gguf
