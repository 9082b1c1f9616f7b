// Instances of the wide tile kernel (tile_wide_core.h): Q5_K.
#include "tile_wide_core.h"

namespace gguf {
int wide_q5_k(const WideCall& c, hipStream_t s) { return wide_run_either<WQ5_KT<false>, WQ5_KT<true>>(c, s); }
}  // namespace gguf
