// Instances of the codebook formats' GEMM (dense_core.h).
#include "dense_core.h"

namespace gguf {
int dense_iq3_s(const DenseCall& c, const TilePlan& p, hipStream_t s) { return dense_fmt<DIQ3_S>(c, p, s); }
int dense_iq1_s(const DenseCall& c, const TilePlan& p, hipStream_t s) { return dense_fmt<DIQ1_S>(c, p, s); }
int dense_iq1_m(const DenseCall& c, const TilePlan& p, hipStream_t s) { return dense_fmt<DIQ1_M>(c, p, s); }
}  // namespace gguf
