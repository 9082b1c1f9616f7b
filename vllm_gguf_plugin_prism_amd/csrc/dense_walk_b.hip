// Instances of the walking codebook GEMM (dense_walk_core.h).
#include "dense_walk_core.h"

namespace gguf {
int dwalk_iq2_xs(const DwalkCall& c, hipStream_t s) { return dwalk_run<DIQ2_XS>(c, s); }
int dwalk_iq2_s(const DwalkCall& c, hipStream_t s) { return dwalk_run<DIQ2_S>(c, s); }
int dwalk_iq3_xxs(const DwalkCall& c, hipStream_t s) { return dwalk_run<DIQ3_XXS>(c, s); }
}  // namespace gguf
