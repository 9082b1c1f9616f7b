// Instances of the codebook formats' GEMM (dense_core.h).
#include "dense_core.h"

namespace gguf {
int dense_iq4_xs(const DenseCall& c, const TilePlan& p, hipStream_t s) { return dense_fmt<DIQ4_XS>(c, p, s); }
int dense_iq4_nl(const DenseCall& c, const TilePlan& p, hipStream_t s) { return dense_fmt<DIQ4_NL>(c, p, s); }
int dense_iq2_xxs(const DenseCall& c, const TilePlan& p, hipStream_t s) { return dense_fmt<DIQ2_XXS>(c, p, s); }
}  // namespace gguf
