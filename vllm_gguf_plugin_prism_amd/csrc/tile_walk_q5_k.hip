// Instances of the walking tile kernel (tile_walk_core.h): Q5_K.
#include "tile_walk_core.h"

namespace gguf {
int walk_q5_k(const WalkCall& c, hipStream_t s) { return walk_run_either<KQ5_K<false>, KQ5_K<true>>(c, s); }
}  // namespace gguf
