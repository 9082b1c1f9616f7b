// Calls of the expert tile kernel (tile_expert_core.h), for the code that routes to it.
#pragma once
#include "mmq_formats.h"
#include "q8_1_device.h"

namespace gguf {

// The quantized activations as the kernel takes them, a record per row and 128 values, [K / 128][rows][EXPERT_REC]: the quants, four block scales and
// four block sums (halves, as which both are defined).  The length is an odd number of 16-byte pieces: the same piece of sixteen records
// lies in different banks.
static inline int64_t expert_rows_bytes(int64_t rows, int64_t K) { return (K + 255) / 256 * 2 * rows * EXPERT_REC; }

struct ExpertCall {
  const void* W;
  const void* x;               // records
  int64_t x_rows;              // rows of the records
  void* Y;
  int dtype, N, K;
  MoeArgs moe;
  int row_blocks;              // blocks of 32 slots
  Gate16 gate;                 // rows != null: the gated epilogue; rows are records of x_rows(pairs) rows
  int ksplit;                  // workgroups that share a sum over K: then fp32 sums [ksplit][pairs][N] go to `partial`, and nothing to Y
  float* partial;
};

int expert_any(int type, const ExpertCall& c, hipStream_t s);   // GGUF_NOT_TAKEN for what it does not serve

}  // namespace gguf
