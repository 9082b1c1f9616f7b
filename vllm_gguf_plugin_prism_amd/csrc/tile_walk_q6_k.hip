// Instances of the walking tile kernel (tile_walk_core.h): Q6_K.
#include "tile_walk_core.h"

namespace gguf {
int walk_q6_k(const WalkCall& c, hipStream_t s) { return walk_run<KQ6_K>(c, s); }
}  // namespace gguf
