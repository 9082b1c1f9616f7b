// Which products the walking codebook GEMM (dense_walk_core.h) takes, and its activations.
#include "dense_walk.h"
#include <algorithm>
#include <cmath>

namespace gguf {

int dwalk_iq4_xs(const DwalkCall& c, hipStream_t s);
int dwalk_iq4_nl(const DwalkCall& c, hipStream_t s);
int dwalk_iq2_xxs(const DwalkCall& c, hipStream_t s);
int dwalk_iq2_xs(const DwalkCall& c, hipStream_t s);
int dwalk_iq2_s(const DwalkCall& c, hipStream_t s);
int dwalk_iq3_xxs(const DwalkCall& c, hipStream_t s);
int dwalk_iq3_s(const DwalkCall& c, hipStream_t s);
int dwalk_iq1_s(const DwalkCall& c, hipStream_t s);
int dwalk_iq1_m(const DwalkCall& c, hipStream_t s);

static int dwalk_any(int type, const DwalkCall& c, hipStream_t s) {
  switch (type) {
    case T_IQ4_XS: return dwalk_iq4_xs(c, s);
    case T_IQ4_NL: return dwalk_iq4_nl(c, s);
    case T_IQ2_XXS: return dwalk_iq2_xxs(c, s);
    case T_IQ2_XS: return dwalk_iq2_xs(c, s);
    case T_IQ2_S: return dwalk_iq2_s(c, s);
    case T_IQ3_XXS: return dwalk_iq3_xxs(c, s);
    case T_IQ3_S: return dwalk_iq3_s(c, s);
    case T_IQ1_S: return dwalk_iq1_s(c, s);
    case T_IQ1_M: return dwalk_iq1_m(c, s);
  }
  return GGUF_NOT_TAKEN;
}

// About how long a product takes, us, the reordering of the activations included, with each of the plans (tiles of 32 rt rows, nw waves): rounds of workgroups on the chip
// with the panels that a wave walks, which are the matrix instructions and the decoding and take longer beside other workgroups; the weights, the rows of X, the
// result.  Fitted to 9700 products of random sizes (17 .. 1024 rows, 512 .. 28672 columns, K 512 .. 18944) of the nine types, right to 8 %; the plan chosen by it takes
// 1.3 % longer than the best.  The direct ones, whose panels take longer with each row past 12 (the rows' lines of all waves no longer fit the first cache), to 4000 of 5 .. 32
// rows, right to 10 %: estimates 3 % high, so that the records are taken in doubt (with 31 rows of IQ1_S [25152,5120] 32 / 43 us).
struct DwalkType { int type; double decoding, weights[2], others; };
struct DwalkShape { int rt, nw; bool direct; double base, part, alone, x, y, products, decoding, lines; };
static const DwalkType dwalk_types[] = {
      {T_IQ2_XXS, 1.011, {0.103, 0.052}, 0.822},
      {T_IQ2_XS, 1.199, {0.084, 0.071}, 0.840},
      {T_IQ3_XXS, 1.650, {0.104, 0.088}, 0.903},
      {T_IQ1_S, 0.921, {0.071, 0.054}, 0.804},
      {T_IQ4_NL, 1.174, {0.082, 0.127}, 0.866},
      {T_IQ3_S, 1.502, {0.108, 0.090}, 0.929},
      {T_IQ2_S, 1.154, {0.083, 0.069}, 0.883},
      {T_IQ4_XS, 1.159, {0.078, 0.120}, 0.796},
      {T_IQ1_M, 1.042, {0.076, 0.057}, 0.824},
};
static const DwalkShape dwalk_shapes[] = {
      {1, 4, true, 3.87, 0.000, 0.841, 6.05, 0.0, 0.612, 1.108, 0.045},
      {1, 8, true, 2.99, 1.031, 1.179, 9.22, 0.0, 0.698, 1.167, 0.044},
      {1, 4, false, 5.15, 0.209, 0.747, 3.72, 0.789, 0.697, 1.397, 0.0},
      {1, 8, false, 4.86, 0.959, 1.015, 3.30, 0.546, 0.653, 1.566, 0.0},
      {2, 4, false, 5.81, 0.010, 0.680, 2.67, 1.253, 1.393, 1.208, 0.0},
      {2, 8, false, 4.21, 2.189, 0.865, 2.32, 0.898, 1.273, 1.737, 0.0},
      {3, 4, false, 5.51, 0.941, 0.600, 2.15, 1.297, 2.251, 1.129, 0.0},
      {4, 4, false, 5.37, 1.322, 0.605, 2.24, 0.895, 3.291, 0.900, 0.0},
      {4, 8, false, 4.32, 2.567, 0.879, 2.15, 1.118, 3.301, 1.270, 0.0},
};
static double dwalk_us(const DwalkType& t, const DwalkShape& p, int M, int N, int K) {
  // (of eight waves two share a SIMD: the panels of both, halved)
  const int np = (K + 255) / 256;
  const double per = p.nw == 8 ? 0.5 * ((np + 7) / 8 + (np + 3) / 8) : (np + 3) / 4;
  const double r = (double)((M + 32 * p.rt - 1) / (32 * p.rt)) * (double)((N + 31) / 32) / (p.nw == 8 ? 256.0 : 512.0);
  const double alone = r < 1.0 ? r : 1.0, lines = M > 12 ? p.lines * (M - 12) * alone : 0.0;
  const double us = p.base + ((p.products + t.decoding * p.decoding + lines) * per + p.part) * (p.alone + (1.0 - p.alone) * alone) * 0.5 * (ceil(r) + (r > 1.0 ? r : 1.0)) +
         1e-6 * (t.weights[p.nw == 8] * N * K + p.x * M * K + p.y * M * N);
  return p.direct ? 1.03 * us : us;
}
// How long dense_kernel takes: its own estimate, corrected by what the same products took (right to 8 %).
static double dwalk_others_us(const DwalkType& t, int M, int N, int K) {
  return t.others * dense_us(M, N, K) + 3.82 + 1e-6 * (0.036 * N * K + 0.697 * M * N + 1.557 * M * K);
}

static bool dwalk_rows_ok(int64_t M) { return M >= 5 && M <= 1024; }   // (others: not measured)
int64_t dwalk_workspace_bytes(int64_t M, int64_t K) { return dwalk_rows_ok(M) ? dwalk_rows_bytes(M, K) : 0; }

// Taken where these estimates put it below the others by more than they err: over products drawn after the fit, taken or not, 1.16 times as fast as dense_kernel alone on
// average (600 of 17 .. 700 rows, four of them more than 3 % slower, none by 7 %), of 5 .. 32 rows 1.35 times (500, none more than 3 % slower).  Rows of 10000 values and more keep to the others mostly: IQ3_S [4160,18688] 141 rows 69 / 88 us.
DwalkPlan dwalk_plan(int type, int64_t M, int64_t N, int64_t K, int64_t w_pitch, int64_t workspace_bytes) {
  DwalkPlan best = {0, 0, false};
  if (!dwalk_rows_ok(M) || N * w_pitch > 0xFFFF0000ll) return best;   // (offsets inside the matrix are 32-bit)
  for (const DwalkType& t : dwalk_types) {
    if (t.type != type) continue;
    const double others = dwalk_others_us(t, (int)M, (int)N, (int)K);
    double least = (others < 20.0 ? 0.92 : 0.88) * others;   // (the longer ones' estimates are off by more)
    for (const DwalkShape& p : dwalk_shapes) {
      if (p.direct ? M > 32 : dwalk_rows_bytes(M, K) > workspace_bytes) continue;
      if ((p.rt > 1 && M <= 32 * (p.rt - 1)) || !walk_bands(p.rt, M, N, K, DWALK_REC).ok) continue;
      const double us = dwalk_us(t, p, (int)M, (int)N, (int)K);
      if (us < least) { least = us; best = {p.rt, p.nw, p.direct}; }
    }
  }
  return best;
}

// A thread per eight values.  A workgroup has 32 rows of 64 values, eight threads to a row.
__global__ __launch_bounds__(256) void dwalk_rows_kernel(const uint4* __restrict__ x, char* __restrict__ records, int K, int np, int64_t M) {
  const int row = threadIdx.x >> 3, k = 64 * blockIdx.x + 8 * (threadIdx.x & 7), b = (k >> 5) & 7;
  const int64_t m = 32 * (int64_t)blockIdx.y + row;
  if (m >= M || k >= K) return;
  const uint4 v = x[(m * (int64_t)K + k) >> 3];
  *(uint4*)(records + ((int64_t)blockIdx.y * np + (k >> 8)) * DWALK_REC + 2048 * b + 1024 * ((k >> 3) & 1) + 16 * (2 * (k & 16) + row)) = v;
}

// (sizes and addresses checked by the caller)
int dwalk_linear(int type, const void* W, const void* x, int dtype, void* workspace, void* Y, int M, int N, int K, const DwalkPlan& p, const LinearArgs& la, hipStream_t s) {
  if (!p.direct)
    hipLaunchKernelGGL(dwalk_rows_kernel, dim3((unsigned)((K + 63) / 64), (unsigned)((M + 31) / 32)), dim3(256), 0, s, (const uint4*)x, (char*)workspace, K, (K + 255) / 256, (int64_t)M);
  const DwalkCall c = {W, p.direct ? x : workspace, Y, dtype, M, N, K, p, la};
  return taken(dwalk_any(type, c, s));
}

}  // namespace gguf
