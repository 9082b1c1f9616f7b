// Instances of the wide tile kernel (tile_wide_core.h): Q4_0.
#include "tile_wide_core.h"

namespace gguf {
int wide_q4_0(const WideCall& c, hipStream_t s) { return wide_run_either<WQ4_0T<false>, WQ4_0T<true>>(c, s); }
}  // namespace gguf
