// Instances of the walking tile kernel (tile_walk_core.h): Q5_0.
#include "tile_walk_core.h"

namespace gguf {
int walk_q5_0(const WalkCall& c, hipStream_t s) { return walk_run_either<KQ5_0<false>, KQ5_0<true>>(c, s); }
}  // namespace gguf
