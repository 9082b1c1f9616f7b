// Which calls the streaming tile kernel (tile_stream_core.h) takes, by ggml type.
#include "tile_stream.h"
#include "dense_api.h"

namespace gguf {

int ts_q4_0(const TsCall& c, hipStream_t s);
int ts_q8_0(const TsCall& c, hipStream_t s);
int ts_q4_k(const TsCall& c, hipStream_t s);
int ts_q5_k(const TsCall& c, hipStream_t s);
int ts_q6_k(const TsCall& c, hipStream_t s);
int ts_q2_k(const TsCall& c, hipStream_t s);
int ts_q3_k(const TsCall& c, hipStream_t s);
int ts_q4_1(const TsCall& c, hipStream_t s);
int ts_q5_0(const TsCall& c, hipStream_t s);
int ts_q5_1(const TsCall& c, hipStream_t s);
int ts_iq4_nl(const TsCall& c, hipStream_t s);
int ts_iq4_xs(const TsCall& c, hipStream_t s);
int ts_iq2_xxs(const TsCall& c, hipStream_t s);
int ts_iq2_xs(const TsCall& c, hipStream_t s);
int ts_iq2_s(const TsCall& c, hipStream_t s);
int ts_iq3_xxs(const TsCall& c, hipStream_t s);
int ts_iq3_s(const TsCall& c, hipStream_t s);

static bool ts_type_ok(int type) {
  switch (type) {
    case T_Q4_0: case T_Q8_0: case T_Q4_K: case T_Q5_K: case T_Q6_K: return true;
    default: return false;
  }
}

// the tile operator's types that there are streaming tiles for, and the GEMV operator's
static bool ts_tile_type_ok(int type) {
  switch (type) {
    case T_Q2_K: case T_Q3_K: case T_Q4_1: case T_Q5_0: case T_Q5_1: return true;
    default: return ts_type_ok(type);
  }
}
static bool ts_gemv_type_ok(int type) {
  switch (type) {
    case T_IQ2_XXS: case T_IQ2_XS: case T_IQ2_S: case T_IQ3_XXS: case T_IQ3_S: case T_IQ4_NL: case T_IQ4_XS: return true;
    default: return ts_tile_type_ok(type);
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

// Five to eight rows of the types whose GEMV is the other kernel: its time hardly depends on the type (13 % off over 2300 calls of
// 512 .. 28672 columns and K 512 .. 18944), this kernel's is as above, with `cut` per panel where rows do not begin on 16 bytes and
// fields are cut out of two reads (right to 3 .. 5 %).
static bool ts_passes_gemv(int type, int M, int N, int K, bool aligned) {
  struct Cost { int type; double base, round, panel, weights, k, cut; };
  static const Cost costs[] = {{T_Q4_0, -1.5, 8.2, 1.01, 0.009, 0.32, 0.085}, {T_Q4_1, 0.3, 6.4, 1.12, 0.022, 0.38, 0.072}, {T_Q5_0, -2.1, 8.9, 1.18, 0.014, 0.36, 0.076},
                               {T_Q5_1, 0.4, 6.4, 1.48, 0.028, 0.34, 0.075}, {T_Q8_0, -2.2, 9.0, 0.71, 0.051, 0.29, 0.078}, {T_IQ4_NL, 0.6, 6.1, 1.09, 0.026, 0.32, 0.071},
                               {T_IQ4_XS, -2.0, 8.5, 1.05, 0.015, 0.37, 0.0}};
  for (const Cost& c : costs) {
    if (c.type != type) continue;
    const int np = (K + 255) / 256, groups = (N + 15) / 16, ks = ts_ks(np, groups);
    const double rounds = ceil(ceil((double)groups * ks / TS_NW) / 256.0);
    const double us = c.base + rounds * (c.round + c.panel * ((np + ks - 1) / ks)) + 1e-6 * c.weights * N * K + 1e-3 * c.k * K + (aligned ? 0.0 : c.cut * np);
    return us < 0.93 * (4.1 + 1e-3 * (0.18 * N + (0.2 * M - 0.08) * K) + 1e-6 * (0.072 + 0.015 * M) * N * K);
  }
  return false;
}

// More than 32 rows: every 32 of them read the weights again, which is nothing while the matrix is small and the tiles are few; the
// kernels behind it share a sum over K between workgroups there, two launches more than this one.  How many M products of
// rows (in whole tiles of 32) and weights, from 3000 calls of 33 .. 500 rows and up to 20M weights: below these 1.2 to 1.4 times as fast
// on average (three in a hundred slower by more than 3 %), over all of them 1.08 (Q3_K) to 1.18 (Q8_0, Q5_0).
static double ts_most_work(int type) {
  switch (type) {
    case T_Q8_0: return 28;
    case T_Q4_0: return 24;
    case T_Q4_K: case T_Q5_K: case T_Q6_K: case T_Q5_0: return 20;   // (Q5_0 at 32: [4880,640] 259 rows 15.5 / 21.3)
    case T_Q4_1: return 16;
    case T_Q5_1: return 14;
    case T_Q2_K: case T_Q3_K: return 12;
  }
  return 0;
}

// Where the panels of a column group are dealt to the waves of a workgroup (tile_dealt_kernel) instead.  Against what runs otherwise (the
// streaming tiles, the kernel of the packed blocks, the staged 16-row tiles, the GEMV), over 23000 random products of 5 .. 32 rows, N 256 ..
// 57344, K 512 .. 18944, both operators: 1.21 times as fast over all; one in 140 is slower by more than 3 %, the worst by 22 %.  us, before
// / dealt: [4096,4096] 12 rows Q4_K 11.0 / 8.4, Q6_K 12.5 / 10.0, [4096,14336] 12 rows Q6_K 25.4 / 18.9, [2048,2048] Q4_K 8.5 / 6.7.
// What it has against it are short rows, where the sum of eight partial tiles and the activations' way to every workgroup weigh, panels that the eight
// waves cannot share evenly (K = 1280: five of them, 2304: one with two), and the sizes that suit the streaming tiles best: their workgroups fill
// more than 0.76 of a round with 779 .. 1024 column groups (a pair of waves each) and with 1557 .. 2048 (`full`, `round`).
static bool ts_dealt_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, bool gemv) {
  if (M < 5 || M > 32 || N > 0x7FFFFFF0ll || K > 0x7FFFFFF0ll) return false;
  const int64_t groups = (N + 15) / 16, np = (K + 255) / 256;
  const bool blocks32 = type == T_Q4_0 || type == T_Q4_1 || type == T_Q5_0 || type == T_Q5_1 || type == T_Q8_0 || type == T_IQ4_NL;
  const bool halves = type == T_Q4_1 || type == T_Q5_1, packed = type == T_Q4_K || type == T_Q5_K || type == T_Q6_K;
  const bool grids = type == T_IQ2_XXS || type == T_IQ2_XS || type == T_IQ2_S || type == T_IQ3_XXS || type == T_IQ3_S;
  const bool round = groups > 1556 && groups <= 2048, full = round || (groups > 778 && groups <= 1024), even = (np & 7) == 0 || (np & 7) == 7;
  // The tile operator's kernel of the packed blocks cuts a long K on few columns between workgroups ([832,15872] Q6_K 11 rows 13.9 / 17.0); the GEMV
  // operator, which has none, is 1.4 to 1.7 times as fast dealt.  (Not from shorter rows on, where that is as fast on average, [528,12800] Q5_K 29
  // rows 14.3 / 15.9 at worst: q, k and v of two formats share a launch only where each is dealt, [432,11008] Q6_K beside [256,11008] Q5_K 19 rows 39 / 17.)
  if (!gemv && packed && groups <= 56 && K > 13000) return false;
  // Two tiles of rows: workgroups of several groups (ts_dealt_groups); past two groups rows must be long enough for the sum at their end.  us, the
  // streaming tiles / dealt, 20 rows: [14336,1536] Q4_K 10.4 / 8.7, [28672,1536] 14.0 / 14.2, [18944,4096] 27.3 / 19.5, [65536,4096] 58.4 / 55.1;
  // full: [13800,1280] Q6_K 23 rows 12.8 / 14.6, [25772,2304] IQ4_XS 23.5 / 25.2, but [16384,2048] Q4_K 1.13 times as fast.
  if (M > 16) {
    if (type == T_Q2_K) return groups <= 256 || (K >= 4096 && groups <= 768);
    if (groups <= 512) return true;
    if (K < 1024 || (full && np <= 5)) return false;
    if (halves) return K >= 2 * groups - 512;
    // (blocks of 32 values and Q5_K: at most four groups; [17952,2560] Q8_0 29 rows 22.7 / 26.0, [14384,2304] 17.1 / 17.9, [27289,4864] 38.1 / 43.3)
    if (type == T_Q8_0) return round ? K > 8192 : K >= 4 * groups - (groups <= 1024 ? 2048 : 1800) && !(full && np > 8 && np <= 12);
    if (blocks32 || type == T_Q5_K) return round ? K >= (type == T_Q5_0 ? 4608 : 6144) : K >= 4 * groups - 2048;
    return K >= groups * 5 / 4 && !(round && np == 9);
  }
  if (!blocks32) {
    // Two panels per row are work for two waves of eight.
    if (groups > 256 * np && K < 12000) return false;
    // A round: the formats that decode least lose most, [25456,10496] Q4_K 9 rows 44.6 / 48.6, [28656,3840] Q5_K 15 rows 23.3 / 25.8, 0.9 to 1.0 of the speed; Q6_K
    // and IQ4_XS up to 4096 ([26704,2304] Q6_K 16 rows 22.0 / 23.3, but, even, [26896,2048] 10 rows 22.7 / 20.7), grids up to 2048, Q2_K, one group always, up to 12000.
    // Before and behind it the dealt kernel reads the activations once per two groups, or has the CUs that the others leave: [24000,4096] Q4_K
    // 1.05, [36000,4096] 1.18 times as fast, grids 1.3 to 1.6.
    if (type == T_Q2_K) return groups <= 1536 || K >= 12000;
    if (type == T_Q4_K && round) return K >= 12000;
    if (type == T_Q5_K && round) return K > (M <= 8 ? 4096 : 8192);
    if ((type == T_Q6_K || type == T_IQ4_XS) && round) return K > 4096 || even;
    if (type == T_Q4_K && groups > 1024) return K > 1536;   // [20224,1280] 15 rows 10.2 / 10.8
    // (IQ2_S, the most lookups in the registers of one group: [14400,1280] 11 rows 11.4 / 13.8, [14304,1792] 13.6 / 14.8, [30720,2560] 25.5 / 29.5;
    // up to eight rows the others are the GEMV: [10640,768] IQ2_XS 6 rows 10.1 / 8.5)
    if (type == T_IQ2_S && groups > 512 && M >= 9) return K > (round ? 3072 : full ? 2048 : 1536);
    if (grids && groups > 512 && M >= 9) return K > (round ? 2048 : 768) || (round && even);   // [10064,768] IQ2_XXS 13 rows 8.1 / 8.7
    // (IQ4_XS up to eight rows on the GEMV is one launch, [1760,768] 6 rows 4.8 / 5.2, but beside Q5_K 11 / 6)
    return true;
  }
  // (these decode more per panel, or keep two values per block and row: the beginning weighs less there)
  if ((type == T_Q8_0 || type == T_Q4_0) && round && M >= 9 && K < 8192) return false;   // [26720,4096] Q8_0 16 rows 28.1 / 31.0, [27664,4832] Q4_0 34.7 / 37.4
  if (type == T_Q4_0 && round && M <= 6 && K < 4096) return false;   // [26592,2816] 5 rows 19.6 / 21.5, but [27156,2560] 8 rows 27.9 / 21.5
  if (M >= 9) return groups <= 512 || K >= 4096 || (halves && K >= 2 * groups - 512);
  // the GEMV, one launch, is ahead on short rows, with Q5_0 and Q8_0 on small matrices ([480,2336] Q8_0 5 rows 5.4 / 6.9) and where rows that do not begin
  // on 16 bytes are cut out of two reads each ([1072,2272] Q5_1 5 rows 6.0 / 7.3; up to 14 % with longer ones of few columns)
  if (K < 2048 || (halves && groups > 512 && K < 4096)) return false;
  if (M <= 6 && w_pitch % 16 != 0 && K < 2560 && N * K <= 6000000 && type != T_IQ4_NL) return false;
  return N * K > 3000000 || (type != T_Q5_0 && type != T_Q8_0);
}

// Where tile_stream_kernel is the faster one of those that do not deal panels.
bool ts_stream_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, bool gemv) {
  if (M < 5 || (M > 512 && !gemv) || N > 0x7FFFFFF0ll || K > 0x7FFFFFF0ll || M > 0x7FFFFFF0ll || !ts_size_ok(N, w_pitch, M < 512 ? M : 512, K)) return false;
  if (M > 32 && !gemv) return 1e-6 * ((M + 31) / 32) * N * K < ts_most_work(type);
  const bool aligned = w_pitch % 16 == 0;
  switch (type) {
    // Against the staged 16-row kernels, or the GEMV: 1.2 to 1.7 times as fast at 5 rows, from 9 on Q2_K 1.9 to 2.4 times, Q3_K 1.3 to
    // 1.6 ([4096,4096], 12 rows: Q2_K 26.3 / 10.6 us, Q3_K 15.8 / 10.9).
    case T_Q2_K: case T_Q3_K: return true;
    // 1.6 to 2.1 times from 9 rows on ([14336,4096] Q4_1 12 rows 41.1 / 18.3)
    case T_Q4_1: case T_Q5_1: return M >= 9 || ts_passes_gemv(type, (int)M, (int)N, (int)K, aligned);
    // (the staged kernel's decoding is the least here: 1.2 times, but 0.85 at 64M weights and more whose rows begin anywhere, and where
    // a long K on few columns leaves most CUs without a workgroup: [736,6560] 20 rows 15.8 / 19.1)
    case T_Q5_0: return M >= 9 ? (aligned || N * K < (64 << 20)) && (N > 1280 || K <= 5120) : ts_passes_gemv(type, (int)M, (int)N, (int)K, aligned);
    // (more rows than the GEMV's are not multiplied in whole numbers) 1.6 times from 9 rows on, [4096,14336] IQ4_XS 16 rows 69.6 / 22.1
    // (and 1.5 to 2.1 times with the grids' two or three lookups per eight weights, [4096,14336] IQ2_XXS 16 rows 68.8 / 21.9; fewer rows:
    // 1.2 to 1.4 times where rows are long, 1.2 at 7 and 8 rows of 8M to 64M weights, where larger ones lose up to 18 %)
    case T_IQ2_XXS: case T_IQ2_XS: case T_IQ2_S: case T_IQ3_XXS: case T_IQ3_S:
      return gemv && (M >= 9 || (K >= 2 * N && N * K >= (16 << 20)) || (M >= 7 && N * K >= (8 << 20) && N * K < (64 << 20)));
    case T_IQ4_NL: case T_IQ4_XS: return gemv && (M >= 9 || ts_passes_gemv(type, (int)M, (int)N, (int)K, aligned));
  }
  if (!ts_type_ok(type)) return false;
  // The GEMV operator: its time grows with the rows ([4096,14336] 6 rows, GEMV / this: Q4_K 32.7 / 19.0, Q6_K 41.2 / 23.2).  Q4_K and Q5_K,
  // whose GEMV decodes little, stay there on small matrices ([2048,2048] 5 rows 6.5 / 7.9).
  if (gemv && M >= 9) return true;
  if (gemv && type >= T_Q4_K && type <= T_Q6_K) return type == T_Q6_K || N * K >= (8 << 20);
  if (gemv || (M <= 6 && type <= T_Q8_0)) return ts_passes_gemv(type, (int)M, (int)N, (int)K, aligned);
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
  if (type == T_Q4_0 && !aligned && K >= 6000) return false;
  if (M <= 8) return M >= 7 && K >= (aligned ? 5120 : 12000);
  // Above: all, but for what the kernel that reads the packed Q4_0 blocks has done in one launch and a single round, K not
  // split and the columns no more than the CUs hold: [4096,4096] 16 rows 11.1 / 10.3, [2048,3072] 10.1 / 9.0; where it is two
  // launches, [2560,4096] 10.7 / 16.0, or two rounds, [5120,4096] 12.9 / 14.7, or the rows short, [4096,2048] 8.7 / 10.0, it falls behind.
  return !(type == T_Q4_0 && M <= 16 && K > 2048 && K <= 4096 && K % 256 == 0 && N <= 4096 && (K < 4096 || N > 3056));
}

// Dense products on either kernel.
bool ts_dense_takes(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, bool gemv) {
  return ((gemv ? ts_gemv_type_ok(type) : ts_tile_type_ok(type)) && ts_dealt_takes(type, M, N, K, w_pitch, gemv) && ts_size_ok(N, w_pitch, M, K)) ||
         ts_stream_takes(type, M, N, K, w_pitch, gemv);
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

// How many times as long a layer with a few pairs per expert takes on the kernels that take pair by pair, by two estimates; 0 where
// it does not run here.  Pair by pair costs every pair's products with its expert's weights, and the weights of the
// experts that are hit once from memory; the tiles cost the experts' weights and decoding once, and rounds of workgroups.
// us, M weights, MB; fitted to 2000 layers of 8 .. 128 experts with 0.5 .. 4 pairs each and right to 13 and 12 %.  [gate|up] 128 x 1536 x 2048, Q4_K and Q6_K down, 24
// tokens of 8 pairs 109 us pair by pair, 79 here; 32 x 2048 x 1536 Q8_0 12 tokens of 4 pairs 36, 41.
double ts_layer_gain(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t tokens, int64_t top_k, int64_t num_experts) {
  if (num_experts <= 0 || num_experts > 256 || !ts_type_ok(type13) || !ts_type_ok(type2) || !ts_layer_takes(type13, type2, H, I, N_out, tokens, top_k, num_experts)) return 0.0;
  struct Cost { int type; double pair, tile; };
  static const Cost costs[] = {{T_Q4_0, 0.0685, 0.050}, {T_Q8_0, 0.0992, 0.042}, {T_Q4_K, 0.0768, 0.024}, {T_Q5_K, 0.105, 0.062}, {T_Q6_K, 0.136, 0.117}};
  const auto of = [&](int type) { int i = 0; while (costs[i].type != type) ++i; return costs[i]; };
  const Cost c13 = of(type13), c2 = of(type2);
  const double pairs = (double)(tokens * top_k), live = num_experts * (1.0 - exp(-pairs / num_experts)), w13 = 2e-6 * I * H, w2 = 1e-6 * N_out * I;
  const double mb = live * (w13 / block_elems(type13) * block_bytes(type13) + w2 / block_elems(type2) * block_bytes(type2));
  const double by_pair = 9.2 + pairs * (w13 * c13.pair + w2 * c2.pair) + 0.035 * mb;
  const double rounds13 = live * (I / 64.0) / 512.0, rounds2 = live * (N_out / 128.0) / 512.0;
  const double by_tile = 15.7 + live * (w13 * c13.tile + w2 * c2.tile) + 0.136 * mb + 0.65 * (rounds13 > 1.0 ? rounds13 : 1.0) * H / 256.0 +
                         0.236 * (rounds2 > 1.0 ? rounds2 : 1.0) * I / 256.0;
  return by_pair / by_tile;
}

// The weights of the experts that are hit, MB, estimated for pairs spread over the experts at random.
double layer_live_mb(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t pairs, int64_t num_experts) {
  const double bytes = (double)(2 * I) * (double)(H / block_elems(type13) * block_bytes(type13)) + (double)N_out * (double)(I / block_elems(type2) * block_bytes(type2));
  return 1e-6 * bytes * num_experts * (1.0 - exp(-(double)pairs / num_experts));
}

// About how long a layer takes here, us, for the choice between this kernel and the wide tiles (wide_layer_us, fitted to the same
// layers; right to 9 %): two workgroups share a CU's LDS up to rows of 2048 values (Q4_0, Q4_K) or 1024 (Q5_K, Q6_K), one
// pays for its beginning; from four rounds on they walk two column groups each.
double ts_layer_us(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t pairs, int64_t num_experts) {
  const double blocks = moe_blocks_estimate((int)(pairs + num_experts * 15), (int)pairs, 16);
  const auto product = [](int type, int64_t K, double wgs) {
    const double panel = type == T_Q4_0 ? 0.846 : type == T_Q8_0 ? 0.642 : type == T_Q4_K ? 0.627 : type == T_Q5_K ? 0.787 : 1.31;
    const bool two = K <= (type == T_Q4_0 || type == T_Q4_K ? 2048 : type == T_Q8_0 ? 0 : 1024);
    const double r = wgs / (two ? 512.0 : 256.0), passes = r >= 4.0 ? 2.0 : 1.0;
    return ((two ? 0.0 : 1.19 / passes) + panel * (double)(K / 256)) * (0.338 + 0.662 * (r < 1.0 ? r : 1.0)) * 0.5 * (ceil(r / passes) * passes + (r > 1.0 ? r : 1.0));
  };
  return 17.8 + product(type13, H, blocks * (double)((I + 63) / 64)) + product(type2, I, blocks * (double)((N_out + 127) / 128)) +
         0.111 * layer_live_mb(type13, type2, H, I, N_out, pairs, num_experts) + 8.9e-6 * (double)pairs * (double)(I + N_out);
}

int ts_any(int type, const TsCall& c, hipStream_t s) {
  switch (type) {
    case T_Q4_0: return ts_q4_0(c, s);
    case T_Q8_0: return ts_q8_0(c, s);
    case T_Q4_K: return ts_q4_k(c, s);
    case T_Q5_K: return ts_q5_k(c, s);
    case T_Q6_K: return ts_q6_k(c, s);
    case T_Q2_K: return ts_q2_k(c, s);
    case T_Q3_K: return ts_q3_k(c, s);
    case T_Q4_1: return ts_q4_1(c, s);
    case T_Q5_0: return ts_q5_0(c, s);
    case T_Q5_1: return ts_q5_1(c, s);
    case T_IQ4_NL: return ts_iq4_nl(c, s);
    case T_IQ4_XS: return ts_iq4_xs(c, s);
    case T_IQ2_XXS: return ts_iq2_xxs(c, s);
    case T_IQ2_XS: return ts_iq2_xs(c, s);
    case T_IQ2_S: return ts_iq2_s(c, s);
    case T_IQ3_XXS: return ts_iq3_xxs(c, s);
    case T_IQ3_S: return ts_iq3_s(c, s);
  }
  return GGUF_NOT_TAKEN;
}

static TsCall ts_dense_call(int type, const void* W, int dtype, int64_t M, int N, int K, bool gemv, const LinearArgs& la) {
  TsCall c = {};
  c.W = W; c.dtype = dtype; c.N = N; c.K = K;
  c.rt = M <= 16 ? 1 : 2;
  c.w_pitch = la.w_pitch; c.ldy = la.ldy; c.bias = la.bias;
  c.gemv = gemv;
  c.dealt = ts_dealt_takes(type, M, N, K, la.w_pitch ? la.w_pitch : (int64_t)K / block_elems(type) * block_bytes(type), gemv);
  c.gemv_sums = gemv && (type == T_Q4_K || type == T_Q5_K);   // (the others' offset is on the stored sums there too)
  return c;
}

bool ts_two_takes(int type, int64_t N, int64_t w_pitch, bool gemv, int type2, int64_t N2, int64_t w_pitch2, bool gemv2, int64_t K, int64_t M) {
  return ts_dense_takes(type, M, N, K, w_pitch, gemv) && ts_dense_takes(type2, M, N2, K, w_pitch2, gemv2) && ts_dealt_takes(type, M, N, K, w_pitch, gemv) &&
         ts_dealt_takes(type2, M, N2, K, w_pitch2, gemv2);
}

int ts_two(const TsShard& a, const TsShard& b, const void* x, int dtype, void* workspace, int64_t M, int K, hipStream_t s) {
  int rc = quantize_q8_1(x, dtype, workspace, M, K, s, 0, nullptr, true);
  if (rc != GGUF_OK) return rc;
  const TsShard* const shards[2] = {&a, &b};
  TsCall c[2];
  for (int i = 0; i < 2; ++i) {
    c[i] = ts_dense_call(shards[i]->type, shards[i]->W, dtype, M, (int)shards[i]->N, K, shards[i]->gemv, shards[i]->la);
    c[i].ws = workspace; c[i].Y = shards[i]->Y; c[i].M = (int)M;
    c[i].row_blocks = 1; c[i].live_blocks = 1;
  }
  // Rows quantized once, and one beginning instead of two where a kernel for both formats is there.  Against two calls, 800 random pairs of
  // 5 .. 32 rows, 256 .. 28672 columns, K 512 .. 18944: 1.65 times as fast in one launch (1.09 at the least), 1.17 in two (1.04 at the least).
  // q, k and v of 4096 + 1024 and 1024 columns, K 4096, 12 rows: 7.3 us less of a layer's 67.5.
  rc = ts_pair(a.type, c[0], b.type, c[1], s);
  if (rc == GGUF_NOT_TAKEN) rc = ts_pair(b.type, c[1], a.type, c[0], s);
  if (rc != GGUF_NOT_TAKEN) return rc;
  rc = taken(ts_any(a.type, c[0], s));
  return rc != GGUF_OK ? rc : taken(ts_any(b.type, c[1], s));
}

int ts_dense(int type, const void* W, const void* x, int dtype, void* workspace, void* Y, int64_t M, int N, int K, bool gemv, const LinearArgs& la, hipStream_t s) {
  int rc = quantize_q8_1(x, dtype, workspace, M, K, s, 0, nullptr, true);
  if (rc != GGUF_OK) return rc;
  TsCall c = ts_dense_call(type, W, dtype, M, N, K, gemv, la);
  constexpr int64_t STEP = 512;                             // rows per launch, 16 tiles: the kernel's quotients by reciprocal stay exact
  for (int64_t m = 0; m < M; m += STEP) {
    c.ws = (const char*)workspace + m * q8_row_bytes(K);
    c.Y = (char*)Y + m * (la.ldy ? la.ldy : N) * (dtype == GGUF_DTYPE_F32 ? 4 : 2);
    c.M = (int)(M - m < STEP ? M - m : STEP);
    c.row_blocks = (c.M + 16 * c.rt - 1) / (16 * c.rt);
    c.live_blocks = c.row_blocks;
    rc = ts_any(type, c, s);
    if (rc != GGUF_OK) return taken(rc);   // (part of Y may be written)
  }
  return GGUF_OK;
}

static TsCall ts_moe_call(const void* W, const void* ws, void* Y, int dtype, int N, int K, int num_sorted, const MoeArgs& moe, const Gate16& gate) {
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
  return c;
}

int ts_moe(const void* W, const void* ws, void* Y, int dtype, int type, int N, int K, int num_sorted, const MoeArgs& moe, hipStream_t s,
           const Gate16& gate) {
  const TsCall c = ts_moe_call(W, ws, Y, dtype, N, K, num_sorted, moe, gate);
  if (c.row_blocks == 0) return GGUF_OK;
  return taken(ts_any(type, c, s));
}

}  // namespace gguf

namespace gguf {
int mmvq_any(int type, const void* W, const void* x, void* q8_workspace, void* Y, int xdtype, int64_t N, int64_t K, int64_t M, hipStream_t s, const LinearArgs& la);
}  // namespace gguf

extern "C" int gguf_linear_dealt(int type, int64_t N, int64_t K, int64_t M, int64_t w_row_pitch_bytes, int gemv) {
  using namespace gguf;
  if (N <= 0 || K <= 0 || block_elems(type) == 0 || K % block_elems(type) || !ts_dense_takes(type, M, N, K, w_row_pitch_bytes, gemv != 0)) return 0;
  LinearArgs la;
  la.w_pitch = w_row_pitch_bytes;
  return ts_dense_call(type, nullptr, GGUF_DTYPE_F16, M, (int)N, (int)K, gemv != 0, la).dealt;
}

extern "C" int gguf_moe_mmq_layer_finer(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t top_k, int64_t tokens, int64_t num_experts, int product) {
  using namespace gguf;
  if (H <= 0 || I <= 0 || N_out <= 0 || top_k <= 0 || tokens <= 0 || num_experts <= 0 || product < 1 || product > 2) return -1;
  if (block_elems(type13) == 0 || block_elems(type2) == 0 || !ts_layer_takes(type13, type2, H, I, N_out, tokens, top_k, num_experts)) return -1;
  const int64_t pairs = tokens * top_k, sorted = (pairs + num_experts * 15) / 16 * 16;
  static const int32_t some[1] = {0};                       // (stands for the arrays that the call would have: nothing reads it)
  int from = -1;
  MoeArgs moe = {some, some, some, 0, product == 1 ? (int)top_k : 1, (int)pairs, 0};
  const int type = product == 1 ? type13 : type2;
  moe.expert_stride = (product == 1 ? 2 * I : N_out) * ((product == 1 ? H : I) / block_elems(type)) * block_bytes(type);
  const Gate16 gate = product == 1 ? Gate16{(char*)some, 0, (int)I, 0, 0} : Gate16{};
  TsCall c = ts_moe_call(nullptr, nullptr, nullptr, GGUF_DTYPE_F16, (int)(product == 1 ? 2 * I : N_out), (int)(product == 1 ? H : I), (int)sorted, moe, gate);
  c.finer_from = &from;
  return ts_any(type, c, nullptr) == GGUF_OK && from < c.row_blocks ? from : -1;
}

extern "C" int gguf_linear_two_takes(int type, int64_t N, int64_t w_row_pitch_bytes, int type2, int64_t N2, int64_t w_row_pitch_bytes2, int64_t K, int64_t M, int gemv) {
  if (M < 1 || M > 32 || N <= 0 || N2 <= 0 || K <= 0) return 0;
  if (M <= 4) return gemv == 3 && gguf::mmvq_pair_takes(type, N, w_row_pitch_bytes, type2, N2, w_row_pitch_bytes2, K, M);
  return gguf::ts_two_takes(type, N, w_row_pitch_bytes, gemv & 1, type2, N2, w_row_pitch_bytes2, gemv & 2, K, M);
}

extern "C" int gguf_linear_two(const void* W, int64_t w_row_pitch_bytes, int type, int64_t N, void* Y, const void* bias, const void* W2, int64_t w_row_pitch_bytes2, int type2,
                               int64_t N2, void* Y2, const void* bias2, const void* x, int xdtype, void* q8_workspace, int64_t y_row_pitch, int64_t K, int64_t M, int gemv,
                               void* stream) {
  using namespace gguf;
  const int qk = block_elems(type), qk2 = block_elems(type2);
  if (qk == 0 || qk2 == 0) return GGUF_ERR_TYPE;
  if (N <= 0 || N2 <= 0 || M < 1 || M > 32 || K <= 0 || K % qk || K % qk2 || N > 0x7FFFFFF0LL || N2 > 0x7FFFFFF0LL || K > 0x7FFFFFF0LL) return GGUF_ERR_SHAPE;
  if (w_row_pitch_bytes < K / qk * block_bytes(type) || w_row_pitch_bytes2 < K / qk2 * block_bytes(type2) || y_row_pitch < N || y_row_pitch < N2) return GGUF_ERR_SHAPE;
  if (xdtype < 0 || xdtype > 2) return GGUF_ERR_DTYPE;
  if (!W || !W2 || !x || !q8_workspace || !Y || !Y2) return GGUF_ERR_NULL;
  if (((uintptr_t)W & 1) || ((uintptr_t)W2 & 1) || (w_row_pitch_bytes & 1) || (w_row_pitch_bytes2 & 1) || !on16(q8_workspace)) return GGUF_ERR_SHAPE;
  if (!gguf_linear_two_takes(type, N, w_row_pitch_bytes, type2, N2, w_row_pitch_bytes2, K, M, gemv)) return GGUF_ERR_TYPE;
  TsShard a = {W, Y, type, N, (gemv & 1) != 0, LinearArgs()}, b = {W2, Y2, type2, N2, (gemv & 2) != 0, LinearArgs()};
  a.la.w_pitch = w_row_pitch_bytes; a.la.ldy = y_row_pitch; a.la.bias = bias;
  b.la.w_pitch = w_row_pitch_bytes2; b.la.ldy = y_row_pitch; b.la.bias = bias2;
  if (M > 4) return ts_two(a, b, x, xdtype, q8_workspace, M, (int)K, (hipStream_t)stream);
  int rc = mmvq_pair(a, b, x, xdtype, (int)K, (int)M, (hipStream_t)stream);
  if (rc != GGUF_NOT_TAKEN) return rc;
  rc = mmvq_any(type, W, x, q8_workspace, Y, xdtype, N, K, M, (hipStream_t)stream, a.la);
  return rc != GGUF_OK ? rc : mmvq_any(type2, W2, x, q8_workspace, Y2, xdtype, N2, K, M, (hipStream_t)stream, b.la);
}
