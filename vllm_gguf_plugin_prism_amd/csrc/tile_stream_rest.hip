// Instances of the streaming tile kernel (tile_stream_core.h) for dense products: Q2_K, Q3_K, Q4_1, Q5_0, Q5_1, IQ4_NL, IQ4_XS.
#include "tile_stream_core.h"

namespace gguf {
int ts_q2_k(const TsCall& c, hipStream_t s) { return ts_dense_run<TQ2_K>(c, s); }
int ts_q3_k(const TsCall& c, hipStream_t s) { return ts_dense_run<TQ3_K>(c, s); }
int ts_q4_1(const TsCall& c, hipStream_t s) { return ts_dense_run<TQ45_1<false>>(c, s); }
int ts_q5_0(const TsCall& c, hipStream_t s) { return c.gemv ? ts_dense_run<TQ5_0<false>>(c, s) : ts_dense_run<TQ5_0<true>>(c, s); }
int ts_q5_1(const TsCall& c, hipStream_t s) { return ts_dense_run<TQ45_1<true>>(c, s); }
int ts_iq4_nl(const TsCall& c, hipStream_t s) { return ts_dense_run<TIQ4_NL>(c, s); }
int ts_iq4_xs(const TsCall& c, hipStream_t s) { return ts_dense_run<TIQ4_XS>(c, s); }
}  // namespace gguf
