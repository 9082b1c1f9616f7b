// Two matrices of a merged layer in one launch of the streaming tiles (tile_dealt_pair_kernel): the formats of the recipes that give
// one of the tensors more bits.
#include "tile_stream_core.h"

namespace gguf {
int ts_pair(int type, const TsCall& c, int type2, const TsCall& d, hipStream_t s) {
  if (type == T_Q4_K && type2 == T_Q6_K) return ts_dealt_pair<TQ4_K, TQ6_K>(c, d, s);
  if (type == T_Q5_K && type2 == T_Q6_K) return ts_dealt_pair<TQ5_K, TQ6_K>(c, d, s);
  if (type == T_Q3_K && type2 == T_Q5_K) return ts_dealt_pair<TQ3_K, TQ5_K>(c, d, s);
  if (type == T_IQ4_XS && type2 == T_Q5_K) return ts_dealt_pair<TIQ4_XS, TQ5_K>(c, d, s);
  return GGUF_NOT_TAKEN;
}
}  // namespace gguf
