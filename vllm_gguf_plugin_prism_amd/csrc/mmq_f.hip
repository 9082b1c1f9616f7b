// Plans and dispatch of the prefill GEMM on the half-precision matrix unit (mmq_f_core.h).
#include "mmq_f_core.h"

namespace gguf {

// About how long a product takes, us, quantizer included (as mmq_int_us, fitted to the same calls and right to about 8 %): a
// super-block of a tile, the beginning and the store of a round of tiles, the partial tiles' way through memory and how
// many of them are added one after the other, the rows of X, the result.
double mmqf_us(int type, int M, int N, int K, int64_t avail) {
  const TilePlan p = mmqf_plan(M, N, K, avail);
  const int nsb = K / 256, rounds = (p.whole + 255) / 256;
  const double sb = type == T_Q4_K ? 5.85 : type == T_Q5_K ? 6.2 : 7.2;
  double us = 6.5 + rounds * (nsb * sb + 8.6) + 1e-6 * M * (0.9 * K + 1.2 * N);
  if (p.shared > 0) us += p.per * sb + (type == T_Q6_K ? 3.8 : 2.2) + 0.036 * (p.workers + p.shared) + 0.23 * nsb / p.per;
  return us;
}

bool mmqf_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes, int64_t int8_rows_bytes) {
  if ((type != T_Q4_K && type != T_Q5_K && type != T_Q6_K) || M < 128 || M > 0x7FFFFFF0ll) return false;
  // (offsets inside the matrix and inside the rows of X are 32-bit)
  const int64_t rows = mmqf_rows_bytes(M, K);
  if (N * w_pitch > 0xFFFF0000ll || rows > 0xFFFF0000ll || workspace_bytes < rows) return false;
  if ((M / 256 + 1) * (N / 128 + 1) * (K / 256) > 0x7FFFFFFFll) return false;   // (super-blocks of all tiles are counted in an int)
  // Where it is the faster one by the two estimates.  Its tiles of 256 rows want rows, and a long K to be worth a beginning;
  // us, this / int8: [2560,1024] Q4_K 288 rows 42 / 21, [18944,1024] 384 rows 85 / 53, [8192,2560] Q6_K 512 rows 94 / 70;
  // [4096,14336] Q4_K 512 rows 107 / 148, [11008,14336] 160 rows 147 / 264, [28672,14336] 256 rows 335 / 547.  Over 5100 calls of
  // random sizes the estimates lose 0.7 % against always taking the faster engine.
  // (A start of 1.5 us for the int8 engine: where the two are close, on products of 20 to 30 us, this one is the likelier to be
  // slower than its estimate.)
  return mmqf_us(type, (int)M, (int)N, (int)K, workspace_bytes - rows) + 1.5 <
         mmq_int_us(type, (int)M, (int)N, (int)K, workspace_bytes > int8_rows_bytes ? workspace_bytes - int8_rows_bytes : 0);
}

// (a pitch that is not a multiple of 4096 bytes: see q8_half_pitch)
MmqfRows mmqf_rows(void* at, int64_t M, int64_t K) {
  const int64_t rows = (M + 255) / 256 * 256, pitch = q8_half_pitch(K);
  _Float16* const x = (_Float16*)at;
  float* const d = (float*)(x + rows * pitch);
  return {x, d, (_Float16*)(d + K / 32 * rows), pitch, rows};
}
int64_t mmqf_rows_bytes(int64_t M, int64_t K) {
  const int64_t rows = (M + 255) / 256 * 256;
  return rows * (2 * q8_half_pitch(K) + K / 32 * 4 + K / 256 * 16);
}

// 256 x 128 tiles, one workgroup per CU.  The tiles of the last, partly filled round are shared by all workgroups where
// that is shorter than a round of its own: a run, its second beginning, and the partial tiles' way through memory (a
// super-block of a tile takes about 6 us, writing and adding a partial tile 0.06).
TilePlan mmqf_plan(int M, int N, int K, int64_t avail) {
  const int slots = 256, nsb = K / 256;
  const int64_t t = (int64_t)((M + 255) / 256) * ((N + 127) / 128);
  const int rest = (int)(t % slots);
  const TilePlan plain = {256, (int)t, 0, 0, 1};
  if (rest == 0) return plain;
  const int per = (rest * nsb + slots - 1) / slots, workers = (rest * nsb + per - 1) / per;
  const TilePlan p = {256, (int)(t - rest), rest, workers, per};
  return per + 2.0 + 0.011 * (workers + rest) < nsb + 1.0 && p.partial_bytes() <= avail ? p : plain;
}

int mmqf(int type, const MmqfCall& c, hipStream_t s) {
  switch (type) {
    case T_Q4_K: return mmqf_fmt<FQ4_K>(c, s);
    case T_Q5_K: return mmqf_fmt<FQ5_K>(c, s);
    case T_Q6_K: return mmqf_fmt<FQ6_K>(c, s);
  }
  return GGUF_NOT_TAKEN;
}

}  // namespace gguf
