// Instances of the wide tile kernel (tile_wide_core.h): Q4_0, Q8_0.
#include "tile_wide_core.h"

namespace gguf {
int wide_q4_0(const WideCall& c, hipStream_t s) { return wide_run_either<WQ4_0T<false>, WQ4_0T<true>>(c, s); }
int wide_q8_0(const WideCall& c, hipStream_t s) { return wide_run<WQ8_0>(c, s); }
}  // namespace gguf
