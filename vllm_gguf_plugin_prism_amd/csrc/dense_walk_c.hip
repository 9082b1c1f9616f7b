// Instances of the walking codebook GEMM (dense_walk_core.h).
#include "dense_walk_core.h"

namespace gguf {
int dwalk_iq3_s(const DwalkCall& c, hipStream_t s) { return dwalk_run<DIQ3_S>(c, s); }
int dwalk_iq1_s(const DwalkCall& c, hipStream_t s) { return dwalk_run<DIQ1_S>(c, s); }
int dwalk_iq1_m(const DwalkCall& c, hipStream_t s) { return dwalk_run<DIQ1_M>(c, s); }
}  // namespace gguf
