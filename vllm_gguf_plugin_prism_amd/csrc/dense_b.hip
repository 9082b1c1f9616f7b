// Instances of the codebook formats' GEMM (dense_core.h).
#include "dense_core.h"

namespace gguf {
int dense_iq2_xs(const DenseCall& c, const TilePlan& p, hipStream_t s) { return dense_fmt<DIQ2_XS>(c, p, s); }
int dense_iq2_s(const DenseCall& c, const TilePlan& p, hipStream_t s) { return dense_fmt<DIQ2_S>(c, p, s); }
int dense_iq3_xxs(const DenseCall& c, const TilePlan& p, hipStream_t s) { return dense_fmt<DIQ3_XXS>(c, p, s); }
}  // namespace gguf
