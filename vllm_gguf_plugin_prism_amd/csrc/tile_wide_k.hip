// Instances of the wide tile kernel (tile_wide_core.h): Q4_K, Q6_K.
#include "tile_wide_core.h"

namespace gguf {
int wide_q4_k(const WideCall& c, hipStream_t s) { return wide_run_either<WQ4_KT<false>, WQ4_KT<true>>(c, s); }
int wide_q6_k(const WideCall& c, hipStream_t s) { return wide_run<WQ6_K>(c, s); }
}  // namespace gguf
