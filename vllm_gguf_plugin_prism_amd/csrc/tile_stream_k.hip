// Instances of the streaming tile kernel (tile_stream_core.h): Q4_K, Q5_K, Q6_K.
#include "tile_stream_core.h"

namespace gguf {
int ts_q4_k(const TsCall& c, hipStream_t s) { return ts_run<TQ4_K>(c, s); }
int ts_q5_k(const TsCall& c, hipStream_t s) { return ts_run<TQ5_K>(c, s); }
int ts_q6_k(const TsCall& c, hipStream_t s) { return ts_run<TQ6_K>(c, s); }
}  // namespace gguf
