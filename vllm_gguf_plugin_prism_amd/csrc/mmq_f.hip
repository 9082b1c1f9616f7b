// Plans and dispatch of the prefill GEMM on the half-precision matrix unit (mmq_f_core.h).
#include "mmq_f_core.h"

namespace gguf {

bool mmqf_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch) {
  if (type != T_Q4_K && type != T_Q5_K && type != T_Q6_K) return false;
  // (offsets inside the matrix and inside the rows of X are 32-bit)
  if (N * w_pitch > 0xFFFF0000ll || mmqf_rows_bytes(M, K) > 0xFFFF0000ll) return false;
  if ((M / 256 + 1) * (N / 128 + 1) * (K / 256) > 0x7FFFFFFFll) return false;   // (super-blocks of all tiles are counted in an int)
  // Where it is faster than the int8 engine (us, this / int8).  Below 193 rows most of a tile would be padding; up to 320 the
  // single row of tiles wants an output that is neither narrow nor much wider than the chip ([18944,3584] Q4_K, 256 rows
  // 105 / 101, [1024,4096] 23.9 / 23.2, [4096,14336] 64 / 85, [14336,4096] 69 / 88).  Q6_K has two operands to multiply:
  // from 448 rows on, and not on narrow outputs ([14336,4096] 384 rows 145 / 127, 512 rows 147 / 158; [1024,4096] 1024 rows
  // 40 / 38).
  if (type == T_Q6_K) return M >= 448 && N >= 2048;
  return M >= 320 || (M > 192 && N >= 2048 && N <= 16384);
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
MmqfPlan mmqf_plan(int M, int N, int K, int64_t avail) {
  const int slots = 256, nsb = K / 256;
  const int64_t t = (int64_t)((M + 255) / 256) * ((N + 127) / 128);
  const int rest = (int)(t % slots);
  const MmqfPlan plain = {256, 128, (int)t, 0, 0, 1};
  if (rest == 0) return plain;
  const int per = (rest * nsb + slots - 1) / slots, workers = (rest * nsb + per - 1) / per;
  const MmqfPlan p = {256, 128, (int)(t - rest), rest, workers, per};
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
