// Instances of the walking tile kernel (tile_walk_core.h): Q4_K.
#include "tile_walk_core.h"

namespace gguf {
int walk_q4_k(const WalkCall& c, hipStream_t s) { return walk_run_either<KQ4_K<false>, KQ4_K<true>>(c, s); }
}  // namespace gguf
