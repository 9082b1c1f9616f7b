// GEMM of the codebook formats on unquantized activations: Y = X . dequant(W)^T in the dtype of X, fp16 or bf16.
//
// The reference has no integer kernel for these formats past a few rows of X and multiplies by the dequantized weights
// (quantization/linear.py:50-58).  As two steps that is a dense copy of W written and read again (52 MB for [5120,5120]
// beside 14 MB of packed weights) and a library GEMM that leaves most of the chip idle at a few hundred rows.  Here the
// weights of a tile are decoded once per step of K into LDS, rounded to X's dtype exactly as the dequantize kernels
// round them, so the matrix unit gets the same operands and only the order of the fp32 sum differs.
//
// Work split: tiles of M_T rows of X by 128 weight rows, eight waves, K in steps of 64 and in two buffers with one barrier
// per step.  The rows of X go straight to LDS from where the caller has them (16-byte pieces, the piece number xored with
// the row's, so that the operand reads meet all banks); a thread has sixteen neighbouring weights of a row per step, their
// packed bytes fetched a step ahead into registers.  M_T = 256: waves of 64 x 64, one workgroup per CU; 128 and 64: waves
// of 32 x 64 and 32 x 32 on half the registers, two workgroups per CU, one decoding while the other multiplies.
//
// Measured, us per call in a graph, this / a dense copy and a library product: IQ4_XS [5120,5120] 64 rows 22.5 / 36.5, [17408,5120] 128
// 61 / 92, 384 126 / 115; IQ2_XXS [17408,5120] 64 rows 40 / 97, 128 54 / 105, 256 83 / 127, 512 138 / 146.  (Some rows to some hundred of
// smaller matrices run dense_walk_core.h.)  What bounds it at many rows is the fetching of a step, about 1 us behind its request: 16 rows of packed bytes per load instruction
// cost the memory pipeline as much as the rows of X do, and neither is asked for more than a step ahead ([5120,5120], 2048
// rows: 168 us, without the packed bytes' fetch 124, without the decoding 114, matrix instructions and operand reads alone
// 93).  At few rows it is the decoding and the partial tiles.
#pragma once
#include "dense.h"
#include "dense_formats.h"

namespace gguf {

struct DenseArgs {
  TileRuns r;                                 // (the last unit of a row may be part of one)
  int K;
  int64_t w_pitch;
};

template <typename T> struct DenseType;
template <> struct DenseType<_Float16> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  typedef _Float16 v2 __attribute__((ext_vector_type(2)));
  template <class A> static __device__ __forceinline__ A mfma(v8 a, v8 b, A c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
template <> struct DenseType<bf16_t> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  typedef __bf16 v2 __attribute__((ext_vector_type(2)));
  template <class A> static __device__ __forceinline__ A mfma(v8 a, v8 b, A c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};

typedef float dense_f16v __attribute__((ext_vector_type(16)));

template <int J> struct DenseStep { static constexpr int value = J; };

template <int M_T> __host__ __device__ constexpr int dense_buffer_bytes() { return 128 * (M_T + 128); }
template <class F, int M_T> __host__ __device__ constexpr size_t dense_lds() {
  return 2 * (size_t)dense_buffer_bytes<M_T>() + F::TABLE * sizeof(typename F::Entry);
}

template <class F, int WM, int WN, int TM, int TN, int OCC, typename T>
__global__ __launch_bounds__(64 * WM * WN, 2 * OCC) void dense_kernel(const uint8_t* __restrict__ W, const char* __restrict__ X, T* __restrict__ Y,
                                                                      float* __restrict__ partial, const T* __restrict__ bias, DenseArgs a) {
  constexpr int M_T = 32 * WM * TM, N_T = 32 * WN * TN, BUF = dense_buffer_bytes<M_T>(), XI = M_T / 64;
  static_assert(WM * WN == 8 && N_T == 128, "eight waves, a thread per sixteen weights of a step");
  typedef DenseType<T> D;
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, lrow = lane & 31, lhalf = lane >> 5;
  typename F::Entry* const table = (typename F::Entry*)(smem + 2 * BUF);
  for (int i = tid; i < F::TABLE; i += 512) table[i] = F::entry(i);
  if (F::TABLE) __syncthreads();

  const TileWork work = tile_work(a.r);
  const int unit_end = work.end;
  int unit = work.first;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  for (int segment = 0; unit < unit_end; ++segment) {
    const int tile = unit / a.r.units, u0 = unit - tile * a.r.units, u1 = min(a.r.units, u0 + unit_end - unit);
    unit += u1 - u0;
    const int m_base = (tile % a.r.tiles_m) * M_T, n_base = (tile / a.r.tiles_m) * N_T;
    const int g0 = 4 * u0, g1 = min(4 * u1, (a.K + 63) >> 6), g_half = a.K & 63 ? a.K >> 6 : -1;   // g_half: a step of 32 values

    // ---- rows of X: a fetch puts its lanes' 16 bytes one behind the other, so the lane of slot l % 8 of a row asks for
    // the piece that belongs there.  Rows past M repeat the last one; the second half of a step of 32 repeats the first.
    const int x_piece = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7);
    uint32_t x_at[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) x_at[i] = (uint32_t)min(m_base + 8 * (wave + 8 * i) + (lane >> 3), a.r.M - 1) * (uint32_t)(2 * a.K) + 16 * x_piece;
    const auto fetch_x = [&](int g, int buf) {
#pragma unroll
      for (int i = 0; i < XI; ++i) {
        const uint32_t at = x_at[i] - (g == g_half && x_piece >= 4 ? 64u : 0u), to = lds0 + buf * BUF + 1024 * (wave + 8 * i);
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(at), "s"(X + 128 * (int64_t)g), "s"(to) : "memory");
      }
    };
    // ---- weights: sixteen values, part w_p of row w_n's step
    const int w_n = tid >> 2, w_p = tid & 3, h = w_p & 1, w_swz = (w_n >> 1) & 7;
    const uint8_t* const w_row = W + (int64_t)min(n_base + w_n, a.r.N - 1) * a.w_pitch;
    const auto fetch_raw = [&](int g) {
      const int ib = 2 * g + (g == g_half ? 0 : w_p >> 1);   // sub-block of 32 of the row
      if constexpr (F::QK == 256) return F::fetch(w_row + (uint32_t)(g >> 2) * F::BS, ib & 7, h);
      else return F::fetch(w_row + (uint32_t)ib * F::BS, 0, h);
    };
    const auto stash = [&](const typename F::Raw& raw, int j, int buf) {   // step j of its unit
      uint32_t v[4], s[2] = {0, 0}, o[8];
      const float d = F::decode(raw, table, 2 * j + (w_p >> 1), h, v, s);
      dense_operands<F, typename D::v2>(v, s, d, o);
      char* const row = smem + (buf * BUF + 128 * (M_T + w_n));
      *(uint4*)(row + 16 * ((2 * w_p) ^ w_swz)) = make_uint4(o[0], o[1], o[2], o[3]);
      *(uint4*)(row + 16 * ((2 * w_p + 1) ^ w_swz)) = make_uint4(o[4], o[5], o[6], o[7]);
    };

    dense_f16v acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int k = 0; k < TM; ++k)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][k][r] = 0.0f;
    const int swz = (lrow >> 1) & 7;                        // (tile bases are multiples of 16 rows)
    const int op0 = 128 * lrow + 16 * (lhalf ^ swz), x_op = 128 * 32 * TM * wm, w_op = 128 * (M_T + 32 * TN * wn);
    struct Operands { typename D::v8 x[TM], w[TN]; };
    const auto operands = [&](int buf, int t, Operands& o) {
      const char* const at = smem + (buf * BUF + (op0 ^ (32 * t)));
#pragma unroll
      for (int k = 0; k < TM; ++k) o.x[k] = *(const typename D::v8*)(at + x_op + 4096 * k);
#pragma unroll
      for (int i = 0; i < TN; ++i) o.w[i] = *(const typename D::v8*)(at + w_op + 4096 * i);
    };

    typename F::Raw raw[2];
    fetch_x(g0, 0);
    raw[0] = fetch_raw(g0);
    raw[1] = fetch_raw(min(g0 + 1, g1 - 1));
    stash(raw[0], 0, 0);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0), known to the compiler
    __syncthreads();
    // In step g the rows of X of g + 1 and the packed weights of g + 2 are asked for, the registers (step g + 1) are decoded
    // into the other buffer and step g is contracted, the one between the matrix instructions of the other.  Without
    // branches: what the last step of a run prepares is not used.
    const auto turn = [&](int u, auto step) {
      constexpr int J = decltype(step)::value, buf = J & 1;
      const int g = 4 * u + J;
      if (F::QK != 256 && J > 0 && g >= g1) return;
      const int gn = min(g + 1, g1 - 1);
      raw[J & 1] = fetch_raw(min(g + 2, g1 - 1));
      fetch_x(gn, buf ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      Operands o[2];
      operands(buf, 0, o[0]);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (F::QK != 256 && t == 2 && g == g_half) break;
        if (t < 3) operands(buf, t + 1, o[(t + 1) & 1]);
        if (t == 0) stash(raw[(J + 1) & 1], (J + 1) & 3, buf ^ 1);
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int k = 0; k < TM; ++k) acc[i][k] = D::mfma(o[t & 1].w[i], o[t & 1].x[k], acc[i][k]);
      }
      // the order of issue: operands one quarter ahead, a share of the decoding behind each matrix instruction
      __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t < 3) __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);
#pragma unroll
        for (int i = 0; i < TM * TN; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 28 / (TM * TN), 0);
        }
      }
      __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    };
    for (int u = u0; u < u1; ++u) {
      turn(u, DenseStep<0>());
      turn(u, DenseStep<1>());
      turn(u, DenseStep<2>());
      turn(u, DenseStep<3>());
    }

    // ---- store: lane = one row of X, 16 features per tile in runs of four
    float* const mine = u1 - u0 < a.r.units ? partial + (int64_t)(2 * work.worker + segment) * (M_T * N_T) : nullptr;
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int k = 0; k < TM; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const tile_f4v v = {acc[i][k][4 * q], acc[i][k][4 * q + 1], acc[i][k][4 * q + 2], acc[i][k][4 * q + 3]};
          if (mine) {   // in the order of the registers: [wave][tile][run][lane] of four
            *(tile_f4v*)(mine + (((wave * TN * TM + i * TM + k) * 4 + q) * 64 + lane) * 4) = v;
          } else {
            const int m = m_base + 32 * (TM * wm + k) + lrow, n = n_base + 32 * (TN * wn + i) + 8 * q + 4 * lhalf;
            tile_store(v, m, n, Y, bias, a.r);
          }
        }
  }
}

template <class F, int WM, int WN, int TM, int TN, int OCC, typename T>
static int dense_launch(const DenseCall& c, const TilePlan& p, hipStream_t stream) {
  constexpr int M_T = 32 * WM * TM;
  constexpr size_t lds = dense_lds<F, M_T>();
  static_assert(OCC * lds <= 160 * 1024, "tile does not fit in LDS");
  auto kern = dense_kernel<F, WM, WN, TM, TN, OCC, T>;
  static std::atomic<uint64_t> done{0};
  allow_large_lds(kern, lds, done);
  const int64_t ldy = c.la.ldy ? c.la.ldy : (int64_t)c.N;
  const DenseArgs a = {tile_runs<T>(p, c.M, c.N, (c.K + 255) / 256, c.Y, ldy), c.K, c.la.w_pitch ? c.la.w_pitch : (int64_t)(c.K / F::QK) * F::BS};
  hipLaunchKernelGGL(kern, dim3(p.whole + p.workers), dim3(512), lds, stream, (const uint8_t*)c.W, (const char*)c.X, (T*)c.Y, c.partial,
                     (const T*)c.la.bias, a);
  if (p.shared > 0)
    hipLaunchKernelGGL((tile_reduce_kernel<WM, WN, TM, TN, T>), dim3(p.shared, 8 * TM * TN), dim3(256), 0, stream, c.partial, (T*)c.Y,
                       (const T*)c.la.bias, a.r);
  return launch_status();
}

template <class F, typename T>
static int dense_typed(const DenseCall& c, const TilePlan& p, hipStream_t s) {
  switch (p.mt) {
    case 64: return dense_launch<F, 2, 4, 1, 1, 2, T>(c, p, s);
    case 128: return dense_launch<F, 4, 2, 1, 2, 2, T>(c, p, s);
    default: return dense_launch<F, 4, 2, 2, 2, 1, T>(c, p, s);
  }
}

template <class F>
static int dense_fmt(const DenseCall& c, const TilePlan& p, hipStream_t s) {
  return c.dtype == GGUF_DTYPE_F16 ? dense_typed<F, _Float16>(c, p, s) : dense_typed<F, bf16_t>(c, p, s);
}

}  // namespace gguf
