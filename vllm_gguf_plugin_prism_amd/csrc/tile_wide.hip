// Which calls the wide tile kernel (tile_wide_core.h) takes, by ggml type.
#include "tile_wide.h"
#include "mmq_f.h"
#include "tile_stream.h"

namespace gguf {

int wide_q4_0(const WideCall& c, hipStream_t s);
int wide_q4_k(const WideCall& c, hipStream_t s);
int wide_q5_k(const WideCall& c, hipStream_t s);
int wide_q6_k(const WideCall& c, hipStream_t s);
int wide_q2_k(const WideCall& c, hipStream_t s);
int wide_q3_k(const WideCall& c, hipStream_t s);
int wide_q4_1(const WideCall& c, hipStream_t s);
int wide_q5_1(const WideCall& c, hipStream_t s);

static bool wide_type_ok(int type) {
  switch (type) {
    case T_Q4_0: case T_Q8_0: case T_Q4_K: case T_Q5_K: case T_Q6_K: return true;
    default: return false;
  }
}

// (blocks of 144, 176, 18, 34 bytes: 256 values are whole 16-byte pieces, and rows of whole super-blocks begin where W does)
bool wide_aligned(int type, const void* W) { return type == T_Q6_K || on16(W); }

// offsets inside a matrix and inside the records of a row of super-blocks are 32-bit
static bool wide_size_ok(int type, int64_t N, int64_t K, int64_t x_rows) {
  return N * (K / block_elems(type) * block_bytes(type)) <= 0xFFFF0000ll && x_rows * WIDE_REC <= 0xFFFF0000ll;
}

// About how long a layer takes here, us (ts_layer_us is the streaming tiles' estimate): what its panels take, rounds of
// workgroups on the chip, whose panels take longer the more workgroups share a CU; the experts that are hit from memory; the
// rows of X, h and the result.  Fitted to 10000 layers of random sizes (H 1024 .. 4096, I 512 .. 8192, 8 .. 256 experts with 0.5 ..
// 128 pairs each), right to 8 % on as many others; the panels of the expert tiles' formats to 1200.
static double wide_layer_us(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t pairs, int64_t num_experts) {
  const auto panel = [](int type) { return type == T_Q4_0 ? 1.70 : type == T_Q8_0 ? 2.65 : type == T_Q4_K ? 1.61 : type == T_Q5_K ? 1.94 : 3.45; };
  const double blocks = moe_blocks_estimate((int)(pairs + num_experts * 31), (int)pairs, 32), tiles2 = blocks * (double)((N_out + 127) / 128);
  const int parts = wide_ksplit(tiles2, (int)I);
  const auto product = [](double us_panel, int64_t panels, double wgs) {
    const double r = wgs / 768.0;
    return us_panel * (double)panels * (0.438 + 0.562 * (r < 1.0 ? r : 1.0)) * 0.5 * (ceil(r) + (r > 1.0 ? r : 1.0));
  };
  return 19.2 + product(panel(type13), H / 256, blocks * (double)((I + 63) / 64)) + product(panel(type2), (I / 256 + parts - 1) / parts, tiles2 * parts) +
         0.0821 * layer_live_mb(type13, type2, H, I, N_out, pairs, num_experts) + 5.48e-6 * (double)pairs * (double)(I + N_out);
}

bool wide_layer_takes(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t tokens, int64_t top_k, int64_t num_experts) {
  const int64_t pairs = tokens * top_k;
  if (!wide_type_ok(type13) || !wide_type_ok(type2) || num_experts > 256 || H % 256 != 0 || I % 256 != 0 || !wide_size_ok(type13, 2 * I, H, tokens) || !wide_size_ok(type2, N_out, I, pairs)) return false;
  if (pairs * top_k > 0xFFFFFFFFll) return false;               // (the kernel's quotient by reciprocal)
  // Both sides of 2200 layers of random sizes were measured, 4 to 1500 pairs per expert, how many times as long the others take:
  //   * past what the streaming tiles take: 1.33 (Q8_0, 150 layers of 4 to 100 pairs per expert), 1.47 from 60 pairs on over all types and
  //     never below 1.05 there (Q8_0 1.23 to 1.36, also at 300 to 2500, 1.15 at least).  A second product of Q6_K behind Q8_0, on the wide tiles here and on blocks of 64 slots
  //     there, is up to 1.15 times as long here once it is long and its rows are many (277 layers of 200 to 2500 pairs per expert).  All of those that are more than
  //     1 % slower but one have 2 pairs I N_out > 240e9, below which these tiles are 1.15 times as fast on average (the one, H 3072, I 5888: 0.91 to 0.98); the line there loses 0.5 % against always taking
  //     the faster one, one at 640 pairs per expert 4.8 %;
  //   * Q8_0 past what they take (I below 768) with up to 16 pairs per expert, where the others have blocks of 16 slots and a panel there costs less while
  //     the workgroups are few, first of all the second product's (307 layers, H 256 .. 4096, I 256 or 512, 8 to 128 experts): from 180 blocks times (panels of a row of X + 1)
  //     on 1.17 (0.94 .. 1.65), below that 0.96 (0.89 .. 1.12); with the lighter panels of Q4_K, Q5_K from 60 on.  The line loses 0.5 % on average against
  //     always taking the faster one (without it 1.9 %); of 300 others 5 are more than 3 % slower than before the expert tiles (53).  Rows past 4096: 1.04 to 1.85 at any number of experts;
  //   * against the streaming tiles from 40 pairs per expert on: 1.3 to 1.6, hardly ever less than 1.05.
  // Below that a block of 32 slots is padding for the most part, and the one or the other is faster by the type, the rows'
  // length and how the workgroups fall into rounds: by the two estimates, which lose 0.5 % on average against always taking the faster one.
  if (type13 == T_Q8_0 && type2 == T_Q6_K && pairs > 256 * num_experts && 2.0 * (double)pairs * (double)I * (double)N_out > 240e9) return false;
  if (pairs > 40 * num_experts) return true;
  if (!ts_layer_takes(type13, type2, H, I, N_out, tokens, top_k, num_experts)) {
    if (type13 != T_Q8_0 || H > 4096 || I >= 768 || pairs > 16 * num_experts) return true;
    return moe_blocks_estimate((int)(pairs + num_experts * 15), (int)pairs, 16) * (double)(H / 256 + 1) >= (type2 == T_Q4_K || type2 == T_Q5_K ? 60.0 : 180.0);
  }
  return wide_layer_us(type13, type2, H, I, N_out, pairs, num_experts) < ts_layer_us(type13, type2, H, I, N_out, pairs, num_experts);
}

// A workgroup walks its panels one after the other, about 1.7 us each beside two others on the CU, which holds three: where the
// tiles are fewer than that, the panels of a tile are dealt to several, three panels each at least.
int wide_ksplit(double tiles, int K) {
  const int np = K / 256;
  int ks = 1;
  while (ks < 8 && tiles * ks < 500.0 && np >= 3 * 2 * ks) ks *= 2;
  return ks;
}

// Y = the sum of the parts of K in their order, rounded, plus the bias
template <typename T, int V>
__global__ __launch_bounds__(256) void wide_sum_kernel(const float* __restrict__ parts, int ksplit, int64_t stride, T* __restrict__ Y, int N, int64_t ldy,
                                                       const T* __restrict__ bias) {
  const int n = (blockIdx.x * 256 + threadIdx.x) * V;
  if (n >= N) return;
  const float* const p = parts + (int64_t)blockIdx.y * N + n;
  struct alignas(4 * V) Row { float v[V]; } v = *(const Row*)p;
#pragma unroll 4
  for (int z = 1; z < ksplit; ++z) {
    const Row r = *(const Row*)(p + z * stride);
#pragma unroll
    for (int e = 0; e < V; ++e) v.v[e] += r.v[e];
  }
  T* const y = Y + (int64_t)blockIdx.y * ldy + n;
#pragma unroll
  for (int e = 0; e < V; ++e) y[e] = finish<T>(v.v[e], bias, n + e);
}

int wide_any(int type, const WideCall& c, hipStream_t s) {
  switch (type) {
    case T_Q4_0: return wide_q4_0(c, s);
    case T_Q4_K: return wide_q4_k(c, s);
    case T_Q5_K: return wide_q5_k(c, s);
    case T_Q6_K: return wide_q6_k(c, s);
    case T_Q2_K: return wide_q2_k(c, s);
    case T_Q3_K: return wide_q3_k(c, s);
    case T_Q4_1: return wide_q4_1(c, s);
    case T_Q5_1: return wide_q5_1(c, s);
  }
  return GGUF_NOT_TAKEN;
}

static int64_t wide_records(int64_t M, int64_t K) { return (wide_rows_bytes(M, K) + 255) / 256 * 256; }

// rows of a pass
static int64_t wide_pass_rows(int64_t M, const WidePlan& p) { return p.passes == 1 ? M : (M + 64 * p.passes - 1) / (64 * p.passes) * 64; }

static int64_t wide_dense_workspace(int64_t M, int64_t N, int64_t K, const WidePlan& p) {
  M = wide_pass_rows(M, p);
  return wide_records(M, K) + (p.ksplit > 1 ? 4 * p.ksplit * M * N : 0);
}

// number of a type that dense products are taken of, else -1
static int wide_dense_type(int type) {
  static const int types[] = {T_Q4_0, T_Q4_K, T_Q5_K, T_Q6_K, T_Q2_K, T_Q3_K, T_Q4_1, T_Q5_1};
  for (int i = 0; i < 8; ++i)
    if (types[i] == type) return i;
  return -1;
}

// About how long a product takes, us, quantizer and the sum of the parts included: rounds of workgroups on the chip with their
// panels, which take longer the more workgroups share a CU; the weights, the rows of X, the parts of K.  Fitted to 4000 calls of
// random sizes (33 .. 700 rows, 512 .. 28672 columns, K 512 .. 18944, both heights of tiles, K cut into 1 .. 16); right to
// 6 .. 8 %, so that the plan chosen by it takes 1.5 .. 3 % longer than the best.
struct WideCost { double base, panel, weights, x, part, alone; };
static double wide_us(int type, int M, int N, int K, const WidePlan& p) {
  static const WideCost cost[8][2] = {{{7.8, 3.15, 0.028, 1.34, 1.36, 0.45}, {8.6, 3.87, 0.0, 1.29, 1.33, 0.63}},     // Q4_0
                                      {{7.2, 2.85, 0.009, 1.72, 1.44, 0.40}, {8.3, 3.08, 0.0, 1.73, 1.23, 0.54}},     // Q4_K
                                      {{7.4, 3.20, 0.014, 1.82, 1.38, 0.40}, {8.4, 3.27, 0.0, 1.50, 1.46, 0.57}},     // Q5_K
                                      {{7.3, 4.77, 0.019, 1.50, 1.43, 0.40}, {8.5, 4.80, 0.0, 1.71, 1.18, 0.54}},     // Q6_K
                                      {{7.9, 3.82, 0.026, 1.52, 1.16, 0.43}, {9.1, 4.37, 0.007, 1.36, 1.08, 0.58}},   // Q2_K
                                      {{8.3, 3.50, 0.021, 1.27, 1.01, 0.41}, {9.3, 3.64, 0.0, 1.20, 0.94, 0.56}},     // Q3_K
                                      {{8.6, 3.96, 0.026, 1.26, 1.11, 0.41}, {9.6, 5.04, 0.0, 1.13, 1.00, 0.58}},     // Q4_1
                                      {{7.7, 4.60, 0.015, 1.21, 1.08, 0.42}, {9.3, 5.51, 0.0, 1.22, 0.71, 0.56}}};    // Q5_1
  const WideCost& c = cost[wide_dense_type(type)][p.rt - 1];
  const double r = (double)((M + 32 * p.rt - 1) / (32 * p.rt)) * (double)((N + 127) / 128) * p.ksplit / (p.rt == 1 ? 768.0 : 512.0);
  const int np = (K + 255) / 256, per = (np + p.ksplit - 1) / p.ksplit;
  double us = c.base + c.panel * per * (c.alone + (1.0 - c.alone) * (r < 1.0 ? r : 1.0)) * 0.5 * (ceil(r) + (r > 1.0 ? r : 1.0)) + 1e-6 * (c.weights * N * K + c.x * M * K);
  if (p.ksplit > 1) us += 2.0 + 1e-6 * c.part * p.ksplit * M * N;
  return us;
}

static WidePlan wide_best(int type, int M, int N, int K, int64_t workspace_bytes, double& us) {
  static const int parts[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 16};
  WidePlan best = {0, 1, 1};
  us = 1e30;
  // (two passes over the rows where the workspace has room for half of them, of products that fill the chip several times)
  for (int passes = 1; passes <= (M >= 1024 ? 2 : 1); ++passes)
    for (int rt = 1; rt <= 2; ++rt)
      for (int ks : parts) {
        const WidePlan p = {rt, ks, passes};
        if ((ks > 1 && 3 * ks > (K + 255) / 256) || wide_dense_workspace(M, N, K, p) > workspace_bytes) continue;
        const int rows = (int)wide_pass_rows(M, p);
        const double t = passes == 1 ? wide_us(type, M, N, K, p) : wide_us(type, rows, N, K, p) + wide_us(type, M - rows, N, K, p);
        if (t < us) { us = t; best = p; }
      }
  return best;
}

static bool wide_dense_ok(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch) {
  const int t = wide_dense_type(type);
  if (t < 0 || K % (t >= 6 ? 32 : 256) != 0) return false;
  const int64_t pitch = w_pitch ? w_pitch : K / block_elems(type) * block_bytes(type);
  return M >= 33 && M <= (t >= 4 ? 8192 : 2048) && (t < 6 || pitch % 16 == 0) && N * pitch <= 0xFFFF0000ll && wide_size_ok(type, N, K, M);
}
bool wide_dense_aligned(int type, const void* W) { return (type != T_Q4_1 && type != T_Q5_1) || (uintptr_t)W % 16 == 0; }

// How long the unit takes that runs otherwise (mmq_int_us is fitted to Q4_K .. Q6_K and to types whose decoding is nothing: the
// others by a factor measured on 130 to 270 products each, of up to 64 and of more tiles of 128 by 128).
static double wide_others_us(int type, int M, int N, int K, int64_t workspace_bytes) {
  const int64_t int8_rows = (M * q8_row_bytes(K) + 255) / 256 * 256;
  static const double factor[8][2] = {{0.86, 0.86}, {1.0, 1.0}, {1.0, 1.0}, {1.0, 1.0}, {1.21, 1.32}, {1.0, 1.0}, {1.11, 1.23}, {1.11, 1.23}};
  const bool many = (int64_t)((M + 127) / 128) * ((N + 127) / 128) > 64;
  double us = mmq_int_us(type, M, N, K, workspace_bytes > int8_rows ? workspace_bytes - int8_rows : 0) * factor[wide_dense_type(type)][many];
  if (type >= T_Q4_K && M >= 128 && workspace_bytes >= mmqf_rows_bytes(M, K)) us = std::min(us, mmqf_us(type, M, N, K, workspace_bytes - mmqf_rows_bytes(M, K)) + 1.5);
  return us;
}

// By how much the estimate has to be the shorter one.  Over some 500 rows the types that it was fitted to at 33 .. 700 take 1.08 of
// it (440 products of 500 .. 2048 rows: on average 1.10 of the speed with this margin, four in a hundred slower by more than 4 %).
static double wide_margin(int type, int64_t M) { return M > 500 && wide_dense_type(type) < 4 ? 0.91 : 0.98; }

// Where it is the faster one by these estimates: [7968,2560] Q4_K 308 rows, others / this: 57 / 41 us, [11008,4096] 64 rows 29 / 19; but
// [14784,4352] Q6_K 398 rows 156 / 188.  Q2_K, Q3_K, Q4_1, Q5_1, which the int8 unit decodes at length, nearly always are:
// on average 1.47, 1.28, 1.26 and 1.21 times as fast, [4096,4096] Q2_K 2048 rows 271 / 176 us, Q4_1 256 rows 43 / 38.  (Q5_0, whole numbers to the int8 unit, would be
// as fast on average; Q8_0, whose operands need no scale on the int8 unit, is never more than a few per
// cent faster here, and up to 45 % slower.)
WidePlan wide_dense_plan(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes) {
  if (!wide_dense_ok(type, M, N, K, w_pitch)) return {0, 1, 1};
  double us;
  const WidePlan p = wide_best(type, (int)M, (int)N, (int)K, workspace_bytes, us);
  return p.rt && us < wide_margin(type, M) * wide_others_us(type, (int)M, (int)N, (int)K, workspace_bytes) ? p : WidePlan{0, 1, 1};
}

// How long a product that it takes is estimated to take here, else a time beyond any other's
double wide_dense_us(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes) {
  double us = 1e30;
  if (wide_dense_ok(type, M, N, K, w_pitch)) wide_best(type, (int)M, (int)N, (int)K, workspace_bytes, us);
  return us;
}

// The workspace that takes the call, given the size that the others would want: theirs where that costs less than a tenth.
int64_t wide_dense_room(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t others_bytes) {
  if (!wide_dense_ok(type, M, N, K, w_pitch)) return others_bytes;
  double us, us_there;
  const WidePlan p = wide_best(type, (int)M, (int)N, (int)K, INT64_MAX, us);
  wide_best(type, (int)M, (int)N, (int)K, others_bytes, us_there);
  if (us_there < 1.10 * us || us >= wide_margin(type, M) * wide_others_us(type, (int)M, (int)N, (int)K, others_bytes)) return others_bytes;
  return std::max(others_bytes, wide_dense_workspace(M, N, K, p));
}

static int wide_pass(int type, const void* W, const void* x, int dtype, void* workspace, void* Y, int M, int N, int K, const WidePlan& p, const LinearArgs& la, hipStream_t s) {
  int rc = quantize_wide(x, dtype, workspace, M, K, s);
  if (rc != GGUF_OK) return rc;
  WideCall c = {};
  c.W = W; c.x = workspace; c.x_rows = M; c.Y = Y; c.dtype = dtype; c.M = M; c.N = N; c.K = K;
  c.w_pitch = la.w_pitch; c.ldy = la.ldy; c.bias = la.bias;
  c.row_blocks = (M + 32 * p.rt - 1) / (32 * p.rt);
  c.rt = p.rt; c.ksplit = p.ksplit;
  c.partial = (float*)((char*)workspace + wide_records(M, K));
  rc = taken(wide_any(type, c, s));
  if (rc != GGUF_OK || p.ksplit == 1) return rc;
  const int64_t ldy = la.ldy ? la.ldy : N;
  const int V = N % 4 == 0 ? 4 : 1;
  const dim3 grid((unsigned)((N / V + 255) / 256), (unsigned)M);
  if (V == 4) {
    GGUF_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((wide_sum_kernel<scalar_t, 4>), grid, dim3(256), 0, s, c.partial, p.ksplit, (int64_t)M * N, (scalar_t*)Y, N, ldy, (const scalar_t*)la.bias));
  } else {
    GGUF_DISPATCH_DTYPE(dtype, hipLaunchKernelGGL((wide_sum_kernel<scalar_t, 1>), grid, dim3(256), 0, s, c.partial, p.ksplit, (int64_t)M * N, (scalar_t*)Y, N, ldy, (const scalar_t*)la.bias));
  }
  return launch_status();
}

int wide_dense(int type, const void* W, const void* x, int dtype, void* workspace, void* Y, int M, int N, int K, const WidePlan& p, const LinearArgs& la, hipStream_t s) {
  const int64_t elt = dtype == GGUF_DTYPE_F32 ? 4 : 2, ldy = la.ldy ? la.ldy : N;
  const int rows = (int)wide_pass_rows(M, p);
  for (int m = 0; m < M; m += rows) {
    const int rc = wide_pass(type, W, (const char*)x + elt * K * m, dtype, workspace, (char*)Y + elt * ldy * m, M - m < rows ? M - m : rows, N, K, p, la, s);
    if (rc != GGUF_OK) return rc;
  }
  return GGUF_OK;
}

}  // namespace gguf
