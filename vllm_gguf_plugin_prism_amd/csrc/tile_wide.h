// Calls of the wide tile kernel (tile_wide_core.h), for the code that routes to it.
#pragma once
#include "mmq_formats.h"
#include "q8_1_device.h"

namespace gguf {

// The quantized activations as the kernel takes them, a record per row and 128 values, [K / 128][rows][WIDE_REC], two for every
// 256 values of K that begin (zeros behind K): the quants as whole numbers in half precision, of four neighbours in the order 0, 2, 1, 3; four block scales and four block sums (halves,
// as which both are defined).  The length is an odd number of 16-byte pieces: the same piece of sixteen records lies in
// different banks.
static inline int64_t wide_rows_bytes(int64_t rows, int64_t K) { return (K + 255) / 256 * 2 * rows * WIDE_REC; }

struct WideCall {
  const void* W;
  const void* x;               // records
  int64_t x_rows;              // rows of the records
  void* Y;
  int dtype, M, N, K;          // M: rows of X (dense)
  int64_t w_pitch, ldy;
  const void* bias;
  MoeArgs moe;                 // sorted_token_ids null: dense
  int row_blocks, rt;          // tiles of 32 rt rows (dense) or blocks of 32 slots (rt 1)
  Gate16 gate;                 // rows != null: the gated epilogue; rows are records of x_rows(pairs) rows
  int ksplit;                  // workgroups that share a sum over K: then fp32 sums [ksplit][rows of Y][N] go to `partial`, and nothing to Y
  float* partial;
};

// Whether a layer runs here; the workspace that takes; the call
bool wide_layer_takes(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t tokens, int64_t top_k, int64_t num_experts);
int64_t wide_layer_workspace(int64_t tokens, int64_t top_k, int64_t H, int64_t I, int64_t N_out, int64_t num_experts, int elt);
int wide_layer(const void* X, int xdtype, void* workspace, const void* W13, int type13, const void* W2, int type2, const int32_t* topk_ids,
               const float* topk_w, void* out, int H, int I, int N_out, int top_k, int tokens, int act, int num_experts, hipStream_t s);   // mmq.hip
// A dense product: the plan (rt 0: it runs otherwise), the workspace to ask for, and the call
struct WidePlan { int rt, ksplit, passes; };
WidePlan wide_dense_plan(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes);
double wide_dense_us(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes);
int64_t wide_dense_room(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t others_bytes);
bool wide_dense_aligned(int type, const void* W);   // whether the weights begin where it can fetch them
int wide_dense(int type, const void* W, const void* x, int dtype, void* workspace, void* Y, int M, int N, int K, const WidePlan& p, const LinearArgs& la, hipStream_t s);
bool wide_aligned(int type, const void* W);   // whether the weights begin where the kernel can fetch them
int wide_any(int type, const WideCall& c, hipStream_t s);   // GGUF_NOT_TAKEN for what it does not serve
int wide_ksplit(double tiles, int K);   // into how many parts a product of this many tiles (estimated) cuts K
int quantize_wide(const void* x, int xdtype, void* records, int64_t M, int64_t K, hipStream_t s);   // q8_1.hip

}  // namespace gguf
