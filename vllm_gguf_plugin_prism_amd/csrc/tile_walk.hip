// Which products the walking tile kernel (tile_walk_core.h) takes, by ggml type.
#include "tile_walk.h"
#include "mmq_f.h"
#include "tile_stream.h"
#include "tile_wide.h"
#include <algorithm>
#include <cmath>

namespace gguf {

int walk_q4_0(const WalkCall& c, hipStream_t s);
int walk_q5_0(const WalkCall& c, hipStream_t s);
int walk_q8_0(const WalkCall& c, hipStream_t s);
int walk_q4_k(const WalkCall& c, hipStream_t s);
int walk_q5_k(const WalkCall& c, hipStream_t s);
int walk_q6_k(const WalkCall& c, hipStream_t s);
int walk_q3_k(const WalkCall& c, hipStream_t s);

static int walk_any(int type, const WalkCall& c, hipStream_t s) {
  switch (type) {
    case T_Q4_0: return walk_q4_0(c, s);
    case T_Q5_0: return walk_q5_0(c, s);
    case T_Q8_0: return walk_q8_0(c, s);
    case T_Q4_K: return walk_q4_k(c, s);
    case T_Q5_K: return walk_q5_k(c, s);
    case T_Q6_K: return walk_q6_k(c, s);
    case T_Q3_K: return walk_q3_k(c, s);
  }
  return GGUF_NOT_TAKEN;
}

// About how long a product takes, us, quantizer included, with each of the plans: rounds of workgroups on the chip (two of four waves share a CU, one of
// eight has it for itself) with the panels that a wave walks, which take longer beside other workgroups; the weights, the rows of X, the result.
// Fitted to 12900 products of random sizes (33 .. 2048 rows, 512 .. 28672 columns, K 512 .. 18944), right to 8 %; the plan chosen by it takes 0.9 %
// longer than the best.  (panel 0: no such plan.  Q6_K's tiles of 128 rows have no registers left for the sums of a panel, and without those the result is
// less exact than the other kernels' (1.3e-7 of it against 0.9e-7).)  moved: formats in blocks of 32 whose rows begin anywhere, as K is no multiple of 256, take longer than that;
// of 670 such products of 20M weights and more 71 were more than 3 % slower here than by what ran before ([10544,16960] Q8_0 346 rows 256 / 242 us), with these factors 24.
// cut: the panels begin anywhere inside 16 bytes, by the address and pitch of W (walk_run_either).  Q8_0 then has no tiles of 96 or 128 rows, for which LDS has room for one workgroup
// per CU only ([13696,2304] 593 rows, padded, 135 us; by what runs otherwise 84), and where K is a multiple of 256, as in a padded merged tensor, takes that factor too (400 such products 1.22 times as fast as by what ran before, four of them more than 3 % slower, none by 8); the others are estimated well without it (Q4_0, Q5_0,
// Q4_K, Q5_K: 415 products, five more than 3 % slower, none by 9; with it they would leave 1.1 to 1.2 times).
struct WalkType { int type; double panel[6], weights[2], moved; };
struct WalkShape { int rt, nw; double base, part, alone, x, y; };
static const WalkType walk_types[] = {
      {T_Q4_0, {2.38, 2.29, 3.57, 3.38, 4.78, 6.23}, {0.0582, 0.105}, 1.05},
      {T_Q5_0, {2.56, 2.51, 3.47, 3.34, 4.37, 5.39}, {0.0763, 0.142}, 1.07},
      {T_Q8_0, {2.15, 2.09, 2.97, 2.8, 3.28, 4.18}, {0.11, 0.175}, 1.09},
      {T_Q4_K, {1.84, 1.68, 2.67, 2.48, 3.76, 4.95}, {0.0696, 0.117}, 1.0},
      {T_Q5_K, {1.86, 1.74, 2.87, 2.64, 3.96, 5.14}, {0.0766, 0.132}, 1.0},
      {T_Q6_K, {3.18, 2.94, 4.77, 4.47, 6.50, 0.0}, {0.094, 0.172}, 1.0},
      {T_Q3_K, {2.27, 2.13, 3.14, 2.87, 4.02, 5.05}, {0.062, 0.125}, 1.0},
};
static const WalkShape walk_shapes[] = {
      {1, 4, 5.07, 0.221, 0.612, 1.78, 1.5},
      {1, 8, 4.15, 1.2, 0.831, 2.33, 3.29e-12},
      {2, 4, 5.48, 0.295, 0.634, 1.65, 1.32},
      {2, 8, 3.97, 1.66, 0.889, 2.27, 1.44e-10},
      {3, 4, 5.46, 1.25, 0.641, 1.57, 0.642},
      {4, 4, 5.92, 1.07, 0.636, 1.39, 0.802},
};
static double walk_us(const WalkType& t, int shape, int M, int N, int K, bool cut) {
  const WalkShape& p = walk_shapes[shape];
  const double slots = p.nw == 8 ? 256.0 : 512.0;
  const int per = ((K + 255) / 256 + p.nw - 1) / p.nw;
  const double r = (double)((M + 32 * p.rt - 1) / (32 * p.rt)) * (double)((N + 31) / 32) / slots;
  const double last = p.nw == 8 ? 0.6 : 0.5, rounds = last * ceil(r) + (1.0 - last) * (r > 1.0 ? r : 1.0);   // (what a round in part costs: alone on a CU, eight waves wait longer)
  return (K % 256 != 0 || (t.type == T_Q8_0 && cut) ? t.moved : 1.0) * (p.base + (t.panel[shape] * per + p.part) * (p.alone + (1.0 - p.alone) * (r < 1.0 ? r : 1.0)) * rounds +
         1e-6 * (t.weights[p.nw == 8] * N * K + p.x * M * K + p.y * M * N));
}

// How long the kernels take that run otherwise, by their own estimates and what 12900 products took of those, by type (mmq_int_us is fitted to the
// K-quants).  The streaming tiles, which small matrices run on, have none: they take 1.14 (Q6_K) to 1.25 times as long (of 2691 products 15 were slower here by
// more than 3 %, eight of those among the 296 of K = 512, which are 1.16 times as fast).
static double walk_others_us(int type, int M, int N, int K, int64_t w_pitch, int64_t workspace_bytes) {
  if (ts_dense_takes(type, M, N, K, w_pitch)) return 1e30;
  const int64_t int8_rows = (M * q8_row_bytes(K) + 255) / 256 * 256;
  const double few = M <= 64 ? 0.9 : 1.0, factor = type == T_Q4_0 ? 0.87 * few : type == T_Q5_0 ? 0.79 * few : type == T_Q8_0 ? 0.785 * few :
                                                        type == T_Q6_K ? 1.02 : type == T_Q3_K ? 1.05 : 1.09;
  double us = factor * mmq_int_us(type, M, N, K, workspace_bytes > int8_rows ? workspace_bytes - int8_rows : 0);
  if (mmqf_takes(type, M, N, K, w_pitch, workspace_bytes, int8_rows)) us = std::min(us, mmqf_us(type, M, N, K, workspace_bytes - mmqf_rows_bytes(M, K)));
  return std::min(us, 1.06 * wide_dense_us(type, M, N, K, w_pitch, workspace_bytes));
}

bool walk_may_take(int type, int64_t M) {
  for (const WalkType& t : walk_types)
    if (t.type == type) return M > 32 && M <= 2048;
  return false;
}

// Where it is the faster one by these estimates, by 8 %: over the 12900 products of the fit 1.19 times as fast as what ran before on average (Q6_K 1.12, Q3_K 1.26), 44 of them more
// than 3 % slower (88 with 6 % and with half the last round counted for eight waves too).  Drawn after the fit, taken ones: 1500 of its ranges 1.23, 13 more than 3 % slower, the
// worst 0.87; 300 of longer rows (to 57344) or more columns (to 152064) 1.17, eight, 0.89.  us, before / now, quantizer included: [4096,4096] 64 rows Q4_K 16.1 / 10.8, Q8_0 19.4 / 12.6, 128 rows Q4_K 24.9 / 13.2;
// [14336,4096] Q8_0 77 rows 38.7 / 26.5; but short rows of many columns keep to the others: [25456,512] Q4_K 1501 rows 91 / 137.  (Past 2048 rows: not measured.)
WalkPlan walk_plan(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes, bool w_on16) {
  if (!walk_may_take(type, M) || K % block_elems(type) != 0) return {0, 0};
  const int64_t pitch = w_pitch ? w_pitch : K / block_elems(type) * block_bytes(type);
  // (offsets inside the matrix are 32-bit)
  if (N * pitch > 0xFFFF0000ll || walk_rows_bytes(M, K) > workspace_bytes) return {0, 0};
  const WalkType* t = walk_types;
  while (t->type != type) ++t;
  const bool cut = !w_on16 || pitch % 16 != 0;
  WalkPlan best = {0, 0};
  double least = 1e30;
  for (int i = 0; i < 6; ++i) {
    const WalkShape& p = walk_shapes[i];
    if (t->panel[i] == 0.0 || (type == T_Q8_0 && cut && p.rt > 2) || (p.rt > 1 && M <= 32 * (p.rt - 1)) || !walk_bands(p.rt, M, N, K).ok) continue;
    const double us = walk_us(*t, i, (int)M, (int)N, (int)K, cut);
    if (us < least) { least = us; best = {p.rt, p.nw}; }
  }
  return best.rt && least < 0.92 * walk_others_us(type, (int)M, (int)N, (int)K, pitch, workspace_bytes) ? best : WalkPlan{0, 0};
}

int walk_linear(int type, const void* W, const void* x, int dtype, void* workspace, void* Y, int M, int N, int K, const WalkPlan& p, const LinearArgs& la, hipStream_t s) {
  int rc = quantize_walk(x, dtype, workspace, M, K, type == T_Q6_K, s);
  if (rc != GGUF_OK) return rc;
  const WalkCall c = {W, workspace, Y, dtype, M, N, K, p, la};
  return taken(walk_any(type, c, s));
}

}  // namespace gguf
