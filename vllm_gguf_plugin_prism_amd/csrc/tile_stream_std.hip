// Instances of the streaming tile kernel (tile_stream_core.h): Q4_0, Q8_0.
#include "tile_stream_core.h"

namespace gguf {
int ts_q4_0(const TsCall& c, hipStream_t s) { return ts_run<TQ4_0>(c, s); }
int ts_q8_0(const TsCall& c, hipStream_t s) { return ts_run<TQ8_0>(c, s); }
}  // namespace gguf
