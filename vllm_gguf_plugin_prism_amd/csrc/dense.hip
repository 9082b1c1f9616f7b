// Plans, dispatch and entry points of the codebook formats' GEMM (dense_core.h).
#include "dense.h"
#include "dense_api.h"
#include "dense_walk.h"
#include <algorithm>

namespace gguf {

static bool dense_type_ok(int type) { return block_elems(type) && type >= T_IQ2_XXS; }

// A plan for tiles of `mt` rows of X and about how many us it takes.  The tiles of the last, partly filled round are shared
// by all workgroups where that is shorter than a round of its own: a run, the reduction's launch, and the partial tiles'
// way through memory.
static TilePlan dense_plan_for(int mt, int M, int N, int K, double* cost) {
  const int units = (K + 255) / 256, slots = mt == 256 ? 256 : 512;
  // us per unit of a tile, measured where the chip is full (two workgroups per CU below 256 rows) and where a CU has one
  const double full = mt == 64 ? 4.6 : mt == 128 ? 6.4 : 5.5, alone = mt == 64 ? 3.3 : mt == 128 ? 3.8 : 5.5;
  const int64_t t = (int64_t)((M + mt - 1) / mt) * ((N + 127) / 128);
  const int rest = (int)(t % slots);
  const double whole = (double)(t / slots) * units * full;
  const TilePlan plain = {mt, (int)t, 0, 0, 1};
  *cost = whole + (rest == 0 ? 0.0 : units * (rest <= 256 ? alone : 0.85 * full));
  if (rest == 0) return plain;
  const int per = (int)(((int64_t)rest * units + slots - 1) / slots), workers = (rest * units + per - 1) / per;
  const TilePlan shared = {mt, (int)(t - rest), rest, workers, per};
  const double c = whole + per * (workers <= 256 ? alone : full) + 3.0 + 0.012 * mt / 64 * (workers + rest);
  if (c >= *cost) return plain;
  *cost = c;
  return shared;
}

// Rows of X per tile: what M rows are had for in the least time (`least`, us).
static TilePlan dense_plan(int M, int N, int K, double& least) {
  TilePlan best = {};
  least = 1e300;
  for (int mt = 64; mt <= 256; mt *= 2) {
    double c;
    const TilePlan p = dense_plan_for(mt, M, N, K, &c);
    if (c < least) {
      least = c;
      best = p;
    }
  }
  return best;
}

double dense_us(int M, int N, int K) {
  double us;
  (void)dense_plan(M, N, K, us);
  return us;
}

static int dense_any(int type, const DenseCall& c, const TilePlan& p, hipStream_t s) {
  switch (type) {
    case T_IQ2_XXS: return dense_iq2_xxs(c, p, s);
    case T_IQ2_XS: return dense_iq2_xs(c, p, s);
    case T_IQ3_XXS: return dense_iq3_xxs(c, p, s);
    case T_IQ1_S: return dense_iq1_s(c, p, s);
    case T_IQ4_NL: return dense_iq4_nl(c, p, s);
    case T_IQ3_S: return dense_iq3_s(c, p, s);
    case T_IQ2_S: return dense_iq2_s(c, p, s);
    case T_IQ4_XS: return dense_iq4_xs(c, p, s);
    case T_IQ1_M: return dense_iq1_m(c, p, s);
  }
  return GGUF_ERR_TYPE;
}

}  // namespace gguf

extern "C" int gguf_dense_linear_takes(int type, int xdtype, int64_t N, int64_t K, int64_t M) {
  using namespace gguf;
  if (!dense_type_ok(type) || (xdtype != GGUF_DTYPE_F16 && xdtype != GGUF_DTYPE_BF16)) return 0;
  if (M <= 0 || N <= 0 || K <= 0 || K % block_elems(type) || M > 0x7FFFFFF0LL || N > 0x7FFFFFF0LL || K > 0x7FFFFFF0LL) return 0;
  // (offsets inside X are 32-bit, the units of all tiles are counted in an int)
  if (2 * M * K > 0xFFFF0000LL || (M / 64 + 1) * (N / 128 + 1) * (K / 256 + 1) > 0x7FFFFFFFLL) return 0;
  // Where it is faster than a dense copy and a library product, which take about 28 us at least (host), else 12, 0.85 per
  // million weights and the product at 1.3 PFLOP/s.  Measured, what a call runs (this or dense_walk_core.h) / those, us in a graph, without the
  // host's time: IQ4_XS [5120,5120] 17 rows 13 / 34, 128 27 / 44, 256 34 / 62; [17408,5120] 128 rows IQ2_XXS 54 / 105, IQ4_XS 61 / 92, 384 118 / 129 and 126 / 115,
  // 512 IQ2_XXS 138 / 146; IQ1_M [2048,2048] 256 13 / 22.
  double us;
  (void)dense_plan((int)M, (int)N, (int)K, us);
  const double weights = (double)N * K * 1e-6, two = 12.0 + 0.85 * weights + 2.0 * M * weights / 1300.0;
  return us < 0.95 * (two > 28.0 ? two : 28.0);
}

extern "C" int64_t gguf_dense_linear_workspace_bytes(int64_t N, int64_t K, int64_t M) {
  if (M <= 0 || N <= 0 || K <= 0 || M > 0x7FFFFFF0LL || N > 0x7FFFFFF0LL || K > 0x7FFFFFF0LL) return 0;
  double us;
  return std::max(gguf::dense_plan((int)M, (int)N, (int)K, us).partial_bytes(), gguf::dwalk_workspace_bytes(M, K));
}

extern "C" int gguf_dense_linear_walk(int type, int64_t N, int64_t K, int64_t M, int64_t w_row_pitch_bytes, int64_t workspace_bytes) {
  using namespace gguf;
  if (!gguf_dense_linear_takes(type, GGUF_DTYPE_F16, N, K, M)) return 0;
  const DwalkPlan p = dwalk_plan(type, M, N, K, w_row_pitch_bytes, workspace_bytes);
  return 256 * p.direct + 16 * p.rt + p.nw;
}

extern "C" int gguf_dense_linear(const void* W, int64_t w_row_pitch_bytes, const void* x, int xdtype, void* workspace, void* Y,
                                 int64_t y_row_pitch, const void* bias, int type, int64_t N, int64_t K, int64_t M,
                                 int64_t workspace_bytes, void* stream) {
  using namespace gguf;
  if (!dense_type_ok(type)) return GGUF_ERR_TYPE;
  if (xdtype != GGUF_DTYPE_F16 && xdtype != GGUF_DTYPE_BF16) return GGUF_ERR_DTYPE;
  const int qk = block_elems(type);
  if (N < 0 || M < 0 || K <= 0 || N > 0x7FFFFFF0LL || M > 0x7FFFFFF0LL || K > 0x7FFFFFF0LL || K % qk || w_row_pitch_bytes < K / qk * block_bytes(type) || y_row_pitch < N) return GGUF_ERR_SHAPE;
  if (N == 0 || M == 0) return GGUF_OK;
  if (2 * M * K > 0xFFFF0000LL || (M / 64 + 1) * (N / 128 + 1) * (K / 256 + 1) > 0x7FFFFFFFLL) return GGUF_ERR_SHAPE;
  double us;
  const TilePlan p = dense_plan((int)M, (int)N, (int)K, us);
  if (!W || !x || !Y || (p.shared && !workspace)) return GGUF_ERR_NULL;
  if (((uintptr_t)W & 1) || (w_row_pitch_bytes & 1) || ((uintptr_t)x & 15)) return GGUF_ERR_SHAPE;
  LinearArgs la;
  la.w_pitch = w_row_pitch_bytes;
  la.ldy = y_row_pitch;
  la.bias = bias;
  if (p.shared && (workspace_bytes < p.partial_bytes() || ((uintptr_t)workspace & 15))) return GGUF_ERR_WORKSPACE;
  // some or some tens of rows: waves that walk on their own, those that want records where the workspace has room for them
  const DwalkPlan walk = dwalk_plan(type, M, N, K, w_row_pitch_bytes, workspace && !((uintptr_t)workspace & 15) ? workspace_bytes : 0);
  if (walk.rt) return dwalk_linear(type, W, x, xdtype, workspace, Y, (int)M, (int)N, (int)K, walk, la, (hipStream_t)stream);
  const DenseCall c = {W, x, Y, xdtype, (int)M, (int)N, (int)K, (float*)workspace, la};
  return dense_any(type, c, p, (hipStream_t)stream);
}
