// Instances of the walking codebook GEMM (dense_walk_core.h).
#include "dense_walk_core.h"

namespace gguf {
int dwalk_iq4_xs(const DwalkCall& c, hipStream_t s) { return dwalk_run<DIQ4_XS>(c, s); }
int dwalk_iq4_nl(const DwalkCall& c, hipStream_t s) { return dwalk_run<DIQ4_NL>(c, s); }
int dwalk_iq2_xxs(const DwalkCall& c, hipStream_t s) { return dwalk_run<DIQ2_XXS>(c, s); }
}  // namespace gguf
