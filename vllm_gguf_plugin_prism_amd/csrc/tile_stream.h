// Calls of the streaming tile kernel (tile_stream_core.h), for the code that routes to it.
#pragma once
#include "mmq_formats.h"

namespace gguf {

constexpr int TS_NW = 8;       // waves per workgroup

// KS waves share a column group where the output has fewer groups than the chip has waves: rounds of workgroups x (the
// panels of a wave + a beginning and an end worth about five).
static inline int ts_ks(int np, double groups) {
  int best = 1;
  double best_cost = 1e30;
  for (int ks = 1; ks <= TS_NW; ks <<= 1) {
    const double wgs = ceil(groups * ks / TS_NW), cost = ((np + ks - 1) / ks + 5.0) * ceil(wgs / 256.0);
    if (cost < 0.97 * best_cost) { best_cost = cost; best = ks; }
  }
  return best;
}

// One call of the kernel, dense (moe.sorted_token_ids null) or per block of 16 RT slots.
struct TsCall {
  const void* W;
  const void* ws;              // q8_1 rows with permuted quants
  void* Y;
  int dtype, M, N, K, rt;      // rt: 16-row tiles of X per workgroup
  int64_t w_pitch, ldy;
  const void* bias;
  bool gemv_sums;              // offset term on d * sum(q) instead of the stored sums
  bool gemv;                   // the GEMV operator's arithmetic (Q5_0: see TQ5_0)
  bool dealt;                  // dense, up to 32 rows: a column group's panels dealt to the waves of a workgroup
  MoeArgs moe;
  int row_blocks;              // tiles of 16 rt rows (dense) or blocks of slots
  double live_blocks;          // how many of them hold pairs, estimated (dense: all)
  Gate16 gate;                 // rows != null: the gated epilogue
  int* finer_from;             // not null: nothing is launched, and this says from which row block on K is dealt to two waves each (ts_tail)
};

// tile_stream.hip: whether a call is taken -- a dense product of M rows, a layer with this many (token, expert) pairs, an
// expert GEMM on blocks of 16 slots by itself; how much faster than pair by pair a layer is (0: not taken)
bool ts_stream_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, bool gemv = false);   // without those that deal panels
bool ts_dense_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, bool gemv = false);   // gemv: in place of the GEMV
int ts_dense(int type, const void* W, const void* x, int dtype, void* workspace, void* Y, int64_t M, int N, int K, bool gemv, const LinearArgs& la, hipStream_t s);
// two products of the same rows of X, both with their panels dealt to the waves of a workgroup: the rows are quantized once
struct TsShard { const void* W; void* Y; int type; int64_t N; bool gemv; LinearArgs la; };
bool ts_two_takes(int type, int64_t N, int64_t w_pitch, bool gemv, int type2, int64_t N2, int64_t w_pitch2, bool gemv2, int64_t K, int64_t M);
int ts_two(const TsShard& a, const TsShard& b, const void* x, int dtype, void* workspace, int64_t M, int K, hipStream_t s);
// the same for up to four rows on the streaming GEMV (mmvq_pair.hip): whether a pair is taken; the call, or GGUF_NOT_TAKEN
bool mmvq_pair_takes(int type, int64_t N, int64_t w_pitch, int type2, int64_t N2, int64_t w_pitch2, int64_t K, int64_t M);
int mmvq_pair(const TsShard& a, const TsShard& b, const void* x, int dtype, int K, int M, hipStream_t s);
int ts_pair(int type, const TsCall& c, int type2, const TsCall& d, hipStream_t s);   // in one launch; GGUF_NOT_TAKEN for most types
bool ts_layer_takes(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t tokens, int64_t top_k, int64_t num_experts);
double ts_layer_gain(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t tokens, int64_t top_k, int64_t num_experts);
double ts_layer_us(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t pairs, int64_t num_experts);
double layer_live_mb(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t pairs, int64_t num_experts);
bool ts_moe_takes(int type, int64_t N, int64_t K, int64_t num_sorted, int64_t tokens, int64_t top_k);
int ts_any(int type, const TsCall& c, hipStream_t s);   // GGUF_NOT_TAKEN for other types
// the grouped contraction over blocks of 16 slots; gate.rows: with the gated epilogue (W is [experts][2 inner][K])
int ts_moe(const void* W, const void* ws, void* Y, int dtype, int type, int N, int K, int num_sorted, const MoeArgs& moe, hipStream_t s,
           const Gate16& gate = Gate16{});

}  // namespace gguf
