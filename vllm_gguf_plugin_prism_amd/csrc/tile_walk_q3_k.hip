// Instances of the walking tile kernel (tile_walk_core.h): Q3_K.
#include "tile_walk_core.h"

namespace gguf {
int walk_q3_k(const WalkCall& c, hipStream_t s) { return walk_run<KQ3_K>(c, s); }
}  // namespace gguf
