// The prefill GEMM of the super-block formats on the half-precision matrix unit (mmq_f_core.h), for the code that routes to it.
#pragma once
#include "tile_runs.h"

namespace gguf {

// The quantized activations as the kernel takes them: rows of quants as whole numbers in half precision, `pitch` apart;
// block scales [K / 32][rows]; block sums [K / 256][rows][8].  `rows` is M rounded up to the tallest tile: a tile's last
// rows may be anything, they are read and multiplied but not stored.
struct MmqfRows {
  _Float16* x;
  float* d;
  _Float16* s;
  int64_t pitch, rows;
};
MmqfRows mmqf_rows(void* at, int64_t M, int64_t K);
int64_t mmqf_rows_bytes(int64_t M, int64_t K);
int quantize_whole(const void* x, int xdtype, const MmqfRows& r, int64_t M, int64_t K, hipStream_t stream);   // q8_1.hip

struct MmqfCall {
  const void* W;
  MmqfRows x;
  void* Y;
  int dtype, M, N, K;
  float* partial;
  int64_t partial_bytes;
  LinearArgs la;
};

TilePlan mmqf_plan(int M, int N, int K, int64_t partial_bytes_available);

double mmqf_us(int type, int M, int N, int K, int64_t partial_bytes_available);
double mmq_int_us(int type, int M, int N, int K, int64_t partial_bytes_available);   // mmq_i.hip

// Whether a product with a workspace of this size is taken: it has room for the rows here, and is the faster one with what is
// left for partial tiles here and behind the int8 rows (int8_rows_bytes) there.
bool mmqf_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes, int64_t int8_rows_bytes);
int mmqf(int type, const MmqfCall& c, hipStream_t stream);

}  // namespace gguf
