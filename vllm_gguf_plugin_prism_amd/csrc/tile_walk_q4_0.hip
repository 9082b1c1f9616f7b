// Instances of the walking tile kernel (tile_walk_core.h): Q4_0.
#include "tile_walk_core.h"

namespace gguf {
int walk_q4_0(const WalkCall& c, hipStream_t s) { return walk_run_either<KQ4_0<false>, KQ4_0<true>>(c, s); }
}  // namespace gguf
