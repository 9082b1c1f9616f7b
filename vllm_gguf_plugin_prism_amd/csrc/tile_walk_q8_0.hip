// Instances of the walking tile kernel (tile_walk_core.h): Q8_0.
#include "tile_walk_core.h"

namespace gguf {
int walk_q8_0(const WalkCall& c, hipStream_t s) { return walk_run_either<KQ8_0<false>, KQ8_0<true>>(c, s); }
}  // namespace gguf
