// The expert tile kernel (tile_expert_core.h) by ggml type; instances of Q4_0, Q8_0.
#include "tile_expert_core.h"

namespace gguf {

int expert_q4_k(const ExpertCall& c, hipStream_t s);
int expert_q5_k(const ExpertCall& c, hipStream_t s);

int expert_any(int type, const ExpertCall& c, hipStream_t s) {
  switch (type) {
    case T_Q4_0: return expert_run<KQ4_0<false>>(c, s);
    case T_Q8_0: return expert_run<KQ8_0<false>>(c, s);
    case T_Q4_K: return expert_q4_k(c, s);
    case T_Q5_K: return expert_q5_k(c, s);
  }
  return GGUF_NOT_TAKEN;
}

}  // namespace gguf
