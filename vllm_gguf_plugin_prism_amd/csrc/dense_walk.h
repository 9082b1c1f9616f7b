// Calls of the walking codebook GEMM (dense_walk_core.h), for the code that routes to it.
#pragma once
#include "dense.h"
#include "tile_walk.h"

namespace gguf {

// The activations as the kernel takes them, a record per 32 rows and 256 values, [rows / 32][K / 256][DWALK_REC], in the order in which a wave's lanes take them: of
// block b (32 values) values 8 t .. 8 t + 7 of half h of row r, 16 bytes, at 2048 b + 1024 t + 16 (32 h + r).  What lies behind K and behind the last row may
// be anything.
constexpr int DWALK_REC = 16384;
static inline int64_t dwalk_rows_bytes(int64_t M, int64_t K) { return (M + 31) / 32 * ((K + 255) / 256) * DWALK_REC; }

// Tiles of 32 rt rows, nw waves; direct: one tile of rows, loaded from X as it lies
struct DwalkPlan { int rt, nw; bool direct; };

struct DwalkCall {
  const void* W;
  const void* x;               // records; of a direct plan the rows as they lie
  void* Y;
  int dtype, M, N, K;
  DwalkPlan plan;
  LinearArgs la;
};

// Whether a product runs here with a workspace of this size, and how (rt 0: not); the workspace that takes; the call
DwalkPlan dwalk_plan(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes);
int64_t dwalk_workspace_bytes(int64_t M, int64_t K);
int dwalk_linear(int type, const void* W, const void* x, int dtype, void* workspace, void* Y, int M, int N, int K, const DwalkPlan& p, const LinearArgs& la, hipStream_t s);

}  // namespace gguf
