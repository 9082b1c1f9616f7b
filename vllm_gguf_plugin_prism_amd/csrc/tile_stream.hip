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

// Where the kernel is the faster one, from sweeps of N 512 .. 28672, K 1024 .. 14336 and 5 .. 32 rows of X.  (us with the
// quantizer's launch, this kernel / the other; the others are the GEMV up to 8 rows, the 16-row kernels above.)
bool ts_dense_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch) {
  if (M < 5 || M > 32 || !ts_type_ok(type) || !ts_size_ok(N, w_pitch, M, K)) return false;
  const int64_t weights = N * K;
  // Few columns and a long K leave most CUs without a workgroup (K is shared by the waves of one, not by several).
  if (N <= 2048 && K > (M <= 16 && (type == T_Q4_0 || type == T_Q8_0) ? 8192 : 4096)) return false;
  if (type == T_Q4_0 || type == T_Q8_0) {
    // The GEMV's waves hold all rows' sums: from seven rows on it falls behind where K is long ([4096,8192] Q4_0, 8 rows:
    // 14.7 / 17.5; [4096,4096] 11.0 / 10.3).
    // (rows that do not begin on 16 bytes are cut out of two reads each: [19504,6016] Q8_0, 8 rows: 38.6 / 33.6,
    // [12240,18112] Q4_0, 16 rows: 59 / 50; [6544,18144] Q8_0 40.5 / 49.9)
    const bool aligned = w_pitch % 16 == 0;
    if (type == T_Q4_0 && !aligned && K >= 6000) return false;
    if (M <= 8) return M >= 7 && K >= (aligned ? 5120 : 12000);
    // Above: all, but for the sizes at which the other kernel's column tiles are one even round of the chip
    // ([4096,4096] Q4_0, 16 rows: 11.3 / 10.4; [2048,4096] 10.8 / 12.3; [5120,4096] 12.6 / 14.2; [14336,4096] 18.0 / 21.8;
    // Q8_0 11.3 / 11.9, 10.2 / 14.1, 12.7 / 18.4, 18.5 / 25.4).
    return !(type == T_Q4_0 && M <= 16 && N <= 4096 && weights > 9000000 && weights < 20000000);
  }
  // K-quants: the kernel that reads the packed blocks reaches the same rate in the middle of the range and starts in 3 us less.
  // Short rows ([6144,2048] Q4_K 9.0 / 10.4, [12288,1024] 8.7 / 12.5, Q6_K 11.8 / 13.8, 11.7 / 21.5; Q4_K [4096,2560] 9.8 / 8.4)
  if (K <= 2048) return M >= 9 || type == T_Q6_K || N >= 6144;
  // Narrow outputs ([2048,4096] Q4_K 9.8 / 11.0, Q6_K 12.1 / 13.3; [2048,3072] 9.4 / 8.2)
  if (N <= 2048) return K > (type == T_Q6_K ? 3072 : 3584);
  // Q6_K, whose other kernel reads nine fields per block: all but the middle ([4096,4096] 11.9 / 10.8, [6144,4096] 14.6 / 14.4,
  // [14336,4096] 21.5 / 22.7 and at 32 rows 28.2 / 27.5, [19536,4096], which is 60 % of a round, 30.8 / 29.7; [8192,2560] 12.6 / 14.3, [28672,4096] 31.6 / 38.0, [12288,5120]
  // 24.5 / 34.6, [4096,14336] 23.8 / 27.2 and at 32 rows 32.8 / 46.8)
  if (type == T_Q6_K) return K >= 5120 || (N >= 24000 || (N >= 8192 && (K <= 3072 || (M <= 16 && N <= 16384))));
  if (N > 4096 && N < 6144) return false;                   // (a round of workgroups and a quarter: [5120,12288] Q4_K 21.7 / 21.0)
  // Two tiles of rows ([4096,8192] Q4_K, 32 rows: 18.3 / 20.6; [4096,14336] 26.9 / 35.2)
  if (M > 16 && N >= 4096 && K >= 8192) return true;
  // Large ones ([8192,8192] Q4_K 18.4 / 20.7, [28672,4096] 21.5 / 24.5, [28672,8192] 37.0 / 44.6; [16384,4096] 17.1 / 16.0)
  return weights >= 110000000 || (weights >= 58000000 && K >= 8192);
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
