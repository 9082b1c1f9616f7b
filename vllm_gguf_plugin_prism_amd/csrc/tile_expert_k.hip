// Instances of the expert tile kernel (tile_expert_core.h): Q4_K, Q5_K.
#include "tile_expert_core.h"

namespace gguf {
int expert_q4_k(const ExpertCall& c, hipStream_t s) { return expert_run<KQ4_K<false>>(c, s); }
int expert_q5_k(const ExpertCall& c, hipStream_t s) { return expert_run<KQ5_K<false>>(c, s); }
}  // namespace gguf
