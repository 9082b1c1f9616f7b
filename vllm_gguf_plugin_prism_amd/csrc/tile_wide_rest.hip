// Instances of the wide tile kernel (tile_wide_core.h) for dense products: Q2_K, Q3_K, Q4_1, Q5_1.
#include "tile_wide_core.h"

namespace gguf {
int wide_q2_k(const WideCall& c, hipStream_t s) { return wide_dense_run<WQ2_K>(c, s); }
int wide_q3_k(const WideCall& c, hipStream_t s) { return wide_dense_run<WQ3_K>(c, s); }
int wide_q4_1(const WideCall& c, hipStream_t s) { return wide_dense_run<WQ45_1<false>>(c, s); }
int wide_q5_1(const WideCall& c, hipStream_t s) { return wide_dense_run<WQ45_1<true>>(c, s); }
}  // namespace gguf
