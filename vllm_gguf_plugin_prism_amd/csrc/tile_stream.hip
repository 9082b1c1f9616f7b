// Which calls the streaming tile kernel (tile_stream_core.h) takes, by ggml type.
#include "tile_stream.h"

namespace gguf {

int ts_q4_0(const TsCall& c, hipStream_t s);
int ts_q8_0(const TsCall& c, hipStream_t s);
int ts_q4_k(const TsCall& c, hipStream_t s);
int ts_q5_k(const TsCall& c, hipStream_t s);
int ts_q6_k(const TsCall& c, hipStream_t s);

static bool ts_type_ok(int type) {
  switch (type) {
    case T_Q4_0: case T_Q8_0: case T_Q4_K: case T_Q5_K: case T_Q6_K: return true;
    default: return false;
  }
}

// offsets inside a matrix and inside the quantized rows are 32-bit
static bool ts_size_ok(int64_t rows_w, int64_t w_pitch, int64_t rows_x, int64_t K) {
  return rows_w * w_pitch <= 0xFFFF0000ll && rows_x * q8_row_bytes(K) <= 0xFFFF0000ll;
}

// About how long a product of K-quants takes on this kernel, quantizer included, us: rounds of workgroups on the chip, each
// a beginning and its waves' panels, the weights' and the activations' way.  The same for the kernels that run otherwise:
// the one that reads the packed blocks (rows16_direct_us), and up to eight rows and 8M weights the GEMV, whose time is the
// rows of X that every workgroup quantizes and the columns.  Fitted to 4900 calls of 256 .. 28672 columns, K 512 ..
// 18944 and 5 .. 32 rows of X; on 2250 others of random sizes right to 4 .. 5 % here, 4 % (two tiles of rows) and 8 .. 11 %
// (one) there, so that they lose 0.3 to 0.5 % against always taking the faster kernel.
struct TsCost { double base, round, panel, weights, k; };
static double ts_us(int type, int M, int N, int K) {
  static const TsCost cost[2][3] = {{{-0.4, 6.76, 0.50, 0.056, 0.50}, {-0.2, 6.70, 0.65, 0.062, 0.48}, {1.0, 5.58, 1.11, 0.071, 0.44}},      // Q4_K, Q5_K, Q6_K
                                    {{-4.1, 10.4, 0.99, 0.057, 0.73}, {-3.3, 9.7, 1.13, 0.061, 0.71}, {-4.1, 10.4, 1.80, 0.075, 0.68}}};   // two tiles of rows
  const TsCost& c = cost[M > 16][type - T_Q4_K];
  const int np = (K + 255) / 256, groups = (N + 15) / 16, ks = ts_ks(np, groups);
  const double rounds = ceil(ceil((double)groups * ks / TS_NW) / 256.0);
  return c.base + rounds * (c.round + c.panel * ((np + ks - 1) / ks)) + 1e-6 * c.weights * N * K + 1e-3 * c.k * K;
}
double rows16_direct_us(int type, int M, int N, int K);   // rows16_direct.hip
static double ts_others_us(int type, int M, int N, int K) {
  const bool small = (int64_t)N * K < (8 << 20);
  // (Q6_K's GEMV takes four rows: below 8M weights, too, it is the kernel of the packed blocks, but another line fits)
  if (type == T_Q6_K && M <= 16 && small) return 8.8 + 1e-3 * (0.70 * N + 0.48 * K);
  // (the GEMV's eight rows have no room in LDS from K = 16384 on)
  if (type == T_Q6_K || M > 8 || !small || K >= 16384) return rows16_direct_us(type, M, N, K);
  return (type == T_Q4_K ? 4.2 : 4.7) + 1e-3 * ((type == T_Q4_K ? 0.26 : 0.41) * N + 0.15 * (M + 0.5) * K) + 0.11e-6 * N * K;
}

// Where the kernel is the faster one.
bool ts_dense_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch) {
  if (M < 5 || M > 32 || !ts_type_ok(type) || !ts_size_ok(N, w_pitch, M, K)) return false;
  // [11008,4096] Q4_K 24 rows, this / the other kernel: 19.9 / 39.1, [5120,4096] 14.7 / 25.6, [28672,1024] 5 rows 10.3 / 19.9; but
  // [8192,3584] 12 rows 13.1 / 11.2, [1024,14336] 17.0 / 11.7, [4096,1024] 5 rows 7.6 / 5.7.
  if (type >= T_Q4_K && type <= T_Q6_K) return ts_us(type, (int)M, (int)N, (int)K) < ts_others_us(type, (int)M, (int)N, (int)K);
  // Q4_0, Q8_0, from the same sweeps (us, this / the other kernel: the GEMV up to 8 rows, the 16-row kernels above).
  // Few columns and a long K leave most CUs without a workgroup, as K is shared by the waves of one and not by several
  // ([512,14336] Q4_0 24 rows 26.1 / 17.7, [1024,14336] 12 rows 18.5 / 17.9; [2048,8192] 24 rows 18.1 / 19.2, Q8_0 16.9 / 22.1;
  // [2304,11264] Q4_0 17 rows 23.0 / 25.8).
  if (N <= 2048 && (M <= 16 ? K > 8192 : K > 4096 && K > (type == T_Q8_0 ? 8 : 4) * N)) return false;
  // The GEMV's waves hold all rows' sums: from seven rows on it falls behind where K is long ([4096,8192] Q4_0, 8 rows:
  // 15.2 / 18.5; [4096,4096] 10.9 / 10.7; Q8_0 16.4 / 17.7, 11.6 / 10.8).
  // (rows that do not begin on 16 bytes are cut out of two reads each: [19504,6016] Q8_0, 8 rows: 38.6 / 33.6,
  // [12240,18112] Q4_0, 16 rows: 59 / 50; [6544,18144] Q8_0 40.5 / 49.9)
  const bool aligned = w_pitch % 16 == 0;
  if (type == T_Q4_0 && !aligned && K >= 6000) return false;
  if (M <= 8) return M >= 7 && K >= (aligned ? 5120 : 12000);
  // Above: all, but for what the kernel that reads the packed Q4_0 blocks has done in one launch and a single round, K not
  // split and the columns no more than the CUs hold: [4096,4096] 16 rows 11.1 / 10.3, [2048,3072] 10.1 / 9.0; where it is two
  // launches, [2560,4096] 10.7 / 16.0, or two rounds, [5120,4096] 12.9 / 14.7, or the rows short, [4096,2048] 8.7 / 10.0, it falls behind.
  return !(type == T_Q4_0 && M <= 16 && K > 2048 && K <= 4096 && K % 256 == 0 && N <= 4096 && (K < 4096 || N > 3056));
}

bool ts_moe_takes(int type, int64_t N, int64_t K, int64_t num_sorted, int64_t tokens, int64_t top_k) {
  if (!ts_type_ok(type) || !ts_size_ok(N, K / block_elems(type) * block_bytes(type), tokens, K)) return false;
  // (the kernel's quotients by reciprocal: tile_stream_core.h, ts_launch_d)
  const int64_t blocks = num_sorted / 16, wgs = ((N + 15) / 16 + 1) * blocks;
  return wgs * blocks <= 0xFFFFFFFFll && tokens * top_k * top_k <= 0xFFFFFFFFll;
}

// Up to how many pairs per expert a layer runs on it.  Each block of 16 pairs walks its expert's weights again (from the
// L2, mostly), where the others' blocks take 32 or 64; what that costs depends on how much of the other kernel's time was
// decoding.  us per layer, this kernel / the others, at 16, 32, 48, 64 pairs per expert:
//   Q4_K 64 experts, top-8, H 2048, I 1024: 89 / 134, 115 / 197 (25), 146 / 226 (37), 199 / 300
//   Q4_K, Q6_K 8 experts, top-2, H 4096, I 3584: 114 / 145, 176 / 232, 180 / 231 (40)
//   Q6_K H 2048, I 1024: 144 / 195, 233 / 281, 303 / 344, 342 / 385 (56);  H 2560, I 1280: 157 / 171, 229 / 211, 234 / 314 (40)
//   Q4_0 H 4096, I 2048: 112 / 132, 167 / 185, 217 / 203;  128 experts, H 2048, I 768: 154 / 195, 221 / 239, 289 / 300
//   Q8_0 H 2048, I 1024: 136 / 167, 202 / 204, 258 / 250;  H 1024, I 1536: 80 / 83, 104 / 99
// (longer rows than 2048 leave a CU's LDS room for one workgroup instead of two).
bool ts_layer_takes(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t tokens, int64_t top_k, int64_t num_experts) {
  const int64_t pairs = tokens * top_k, sorted = pairs + num_experts * 15;
  if (H > 4096 || !ts_moe_takes(type13, 2 * I, H, sorted, tokens, top_k) || !ts_moe_takes(type2, N_out, I, sorted, pairs, 1)) return false;
  int64_t most = 40;
  if (type13 == T_Q8_0) most = I < 768 ? 0 : 20;   // (I 512: 59 / 57, 80 / 74)
  else if (type13 == T_Q6_K) most = H <= 2048 ? 60 : 40;
  else if (type13 != T_Q4_0 && H <= 2048) most = 128;
  return pairs <= most * num_experts;
}

int ts_any(int type, const TsCall& c, hipStream_t s) {
  switch (type) {
    case T_Q4_0: return ts_q4_0(c, s);
    case T_Q8_0: return ts_q8_0(c, s);
    case T_Q4_K: return ts_q4_k(c, s);
    case T_Q5_K: return ts_q5_k(c, s);
    case T_Q6_K: return ts_q6_k(c, s);
  }
  return GGUF_NOT_TAKEN;
}

int ts_moe(const void* W, const void* ws, void* Y, int dtype, int type, int N, int K, int num_sorted, const MoeArgs& moe, hipStream_t s,
           const Gate16& gate) {
  TsCall c = {};
  c.W = W;
  c.ws = ws;
  c.Y = Y;
  c.dtype = dtype;
  c.N = N;
  c.K = K;
  c.rt = 1;
  c.gemv_sums = moe.gemv_sums != 0;
  c.moe = moe;
  c.row_blocks = num_sorted / 16;
  c.live_blocks = moe_blocks_estimate(num_sorted, moe.num_pairs, 16);
  c.gate = gate;
  if (c.row_blocks == 0) return GGUF_OK;
  return ts_any(type, c, s);
}

}  // namespace gguf
