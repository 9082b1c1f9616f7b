// Calls of the walking tile kernel (tile_walk_core.h), for the code that routes to it.
#pragma once
#include "mmq_formats.h"
#include "q8_1_device.h"

namespace gguf {

// The quantized activations as the kernel takes them: a record per 32 rows and 256 values, [rows / 32][K / 256][WALK_REC], in the order in which a wave's
// lanes take them: the quants of block b (32 values), 16 bytes of row r's upper or lower half h at 1024 b + 16 (32 h + r), or, for weights with a scale
// per 16 values (`groups`), 8 bytes of half h of its group g at 1024 b + 512 g + 8 (32 h + r); eight block scales of row r,
// halves, at WALK_D_AT + 16 r, and as many block sums at WALK_S_AT + 16 r.  Zeros behind K; rows past the last one may be anything: they are read and
// multiplied but not stored, and no result of another row sees them.
constexpr int WALK_REC = 9216, WALK_D_AT = 8192, WALK_S_AT = 8704;
static inline int64_t walk_rows_bytes(int64_t M, int64_t K) { return (M + 31) / 32 * ((K + 255) / 256) * WALK_REC; }
int quantize_walk(const void* x, int xdtype, void* records, int64_t M, int64_t K, bool groups, hipStream_t stream);   // q8_1.hip

// Tiles of 32 rt rows, nw waves to a workgroup; rt 0: not taken
struct WalkPlan { int rt, nw; };

struct WalkCall {
  const void* W;
  const void* x;               // records
  void* Y;
  int dtype, M, N, K;
  WalkPlan plan;
  LinearArgs la;
};

// How the tiles of 32 rt rows by 32 columns are numbered: bands of `band` row blocks, as tall as their rows of X fit an XCD's L2 (4 MB) beside the weights
// on their way, the row blocks of a band one after the other for each group of columns; the last band has `last`.  ok: the kernel's quotients by
// reciprocal are exact (dividend times divisor stays below 2^32).
struct WalkBands { int tiles, band, band_tiles, last; bool ok; };
static inline WalkBands walk_bands(int rt, int64_t M, int64_t N, int64_t K, int rec = WALK_REC) {
  const int64_t cols = (N + 31) / 32, blocks = (M + 32 * rt - 1) / (32 * rt), fit = (3 << 20) / (rt * ((K + 255) / 256) * rec);
  const int64_t band = fit >= blocks ? blocks : fit > 1 ? fit : 1, tiles = cols * blocks;
  return {(int)tiles, (int)band, (int)(cols * band), (int)(blocks - (blocks - 1) / band * band), tiles <= 0x7FFFFFF && tiles * cols * band <= 0xFFFFFFFFll};
}

// Whether a product runs here with a workspace of this size, and how; the workspace that takes; the call
bool walk_may_take(int type, int64_t M);                    // (a workspace for a call that may be taken has room for its records)
WalkPlan walk_plan(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes, bool w_on16 = true);   // w_on16: W begins on 16 bytes
int walk_linear(int type, const void* W, const void* x, int dtype, void* workspace, void* Y, int M, int N, int K, const WalkPlan& p, const LinearArgs& la, hipStream_t s);

}  // namespace gguf
