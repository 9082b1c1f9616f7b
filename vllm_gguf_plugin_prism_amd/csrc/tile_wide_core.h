// Products with some tens of rows of activations -- dense layers past the few rows of the streaming tiles, Q6_K in MoE layers whose
// experts see more than a few pairs each (the other formats: tile_expert_core.h) -- on 32 or 64 rows by 128 columns per workgroup.
//
// What bounds them is the work around the multiplications: weights decoded again for every 16 rows (tile_stream_core.h) or
// staged, decoded, for the workgroup behind a barrier per 128 values (mmq_i_core.h).  Here
//   * a wave decodes its own 32 weight rows, once for all of the tile's rows, from packed bytes that it fetched into its own
//     LDS ring (global_load_lds, a panel of 32 rows x 256 values ahead) straight into matrix operands;
//   * the operands are whole numbers in half precision with the integer scale of the super-block formats inside, exact as
//     in mmq_f_core.h: a block's sum leaves the matrix unit as a float and costs one multiply-add per result (by the row's
//     block scale, which a lane has in a register: a lane holds one row of X), and one per super-block;
//   * the rows of X come as records of 128 values, quants and scales together (tile_wide.h), 16-byte pieces that land in LDS one
//     behind the other, gathered row by row for the experts; two buffers and a barrier per 128 values;
//   * a workgroup is four waves, so that a CU holds two or three and one's beginning and end lie beside another's middle.
// Measured, us per call, before / now (quantizer, sorting and sums included; 4.83 TB/s is what a copy of 2 GiB reaches): Q4_K
// [7968,2560] 308 rows 57 / 41, [11008,4096] 64 rows 29 / 21; K-quants of 33 to 2048 rows take 0.77 (Q4_K), 0.79 (Q5_K), 0.92 (Q6_K) of
// the time on average, Q4_0 0.93.  A MoE layer of Q6_K, 64 experts, 181 us on tiles of 32 slots only, 175 with the tiles of 16 for blocks
// that are half empty.  (Tiles of 16 x 16 for everything: 0.84 to 1.0 times as fast.  Q6_K on the expert tiles: sixteen scales a
// super-block are 849 vector instructions a panel and registers that spill; slower.)
// What bounds it: no single thing.  With the fetches, the decoding, the operand reads or the multiply-adds left out in turn a
// layer's first product (64 rows a workgroup) is 9 to 14 % faster each; a matrix instruction beside eight multiply-adds takes a
// SIMD 44 cycles (2 waves) where it issues alone in 32.  A beginning and an end are 4 us of a workgroup's 15 to 30.
// Tried and slower: 256 columns on eight waves, one workgroup per CU (Q4_K 32 rows 88 against 70 us); a third buffer of records
// (no change); a grid that stays on the chip and walks runs of tiles with the next one's data under way (1.2 times as long:
// the runs end unevenly, and their state spills at three workgroups per CU).
// Arithmetic as in the other integer kernels (mmq.cuh:2-104, moe.cuh:5-129): exact block sums, scales in fp32.
#pragma once
#include "layer_seam.h"
#include "tile_wide.h"
#include "tile_wide_formats.h"

namespace gguf {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float wide_f4 __attribute__((ext_vector_type(4)));

constexpr int WIDE_NW = 4, WIDE_N = 32 * WIDE_NW;

struct WideArgs {
  int M, N, np, nkb;           // rows of X (dense); weight rows; panels and blocks per row (the last panel may have fewer than eight)
  int col_wgs;                 // workgroups side by side
  uint32_t w_pitch, x_plane;   // bytes between weight rows; between the records of neighbouring panels of a row of X
  uint32_t topk_inv;           // 2^32 / top_k rounded up
  int dtype, quads;            // GGUF_DTYPE_* of Y; rows of Y take stores of four values
  int64_t ldy;
  const void* bias;
  int ksplit;                  // workgroups that share a sum over K: fp32 sums [ksplit][rows of Y][ldy], without the bias
  int64_t split_stride;        // (values between them)
};

template <int N> __device__ __forceinline__ void wide_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// wave-uniform 16-byte-per-lane fetch into LDS: lane l's bytes land at m0 + 16 l
__device__ __forceinline__ void wide_fetch(uint32_t at, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(at), "s"(base), "s"(lds) : "memory");
}
// the same for lanes 0 .. 31 (all lanes are active before and after)
__device__ __forceinline__ void wide_fetch_half(uint32_t at, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(at), "s"(base), "s"(lds), "s"(0xFFFFFFFFull) : "memory");
}
// four bytes a lane
__device__ __forceinline__ void wide_fetch_words(uint32_t at, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(at), "s"(base), "s"(lds) : "memory");
}
template <typename T>
__device__ __forceinline__ void wide_store(const wide_f4& v, T* y, const T* bias, int n, int N, int quads) {
  if (quads && n + 3 < N) {
    struct alignas(4 * sizeof(T)) { T v[4]; } o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o.v[e] = finish<T>(v[e], bias, n + e);
    *(decltype(o)*)(y + n) = o;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) y[n + e] = finish<T>(v[e], bias, n + e);
  }
}
__device__ __forceinline__ void wide_store(const wide_f4& v, int64_t row, int n, void* Y, const WideArgs& a) {
  if (a.dtype == GGUF_DTYPE_F16) wide_store<_Float16>(v, (_Float16*)Y + row * a.ldy, (const _Float16*)a.bias, n, a.N, a.quads);
  else if (a.dtype == GGUF_DTYPE_BF16) wide_store<bf16_t>(v, (bf16_t*)Y + row * a.ldy, (const bf16_t*)a.bias, n, a.N, a.quads);
  else wide_store<float>(v, (float*)Y + row * a.ldy, (const float*)a.bias, n, a.N, a.quads);
}
__device__ __forceinline__ void wide_pin(float (&v)[16]) {   // the sixteen values are computed at this point
  asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
  asm volatile("" : "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]), "+v"(v[12]), "+v"(v[13]), "+v"(v[14]), "+v"(v[15]));
}

// LDS: two buffers of records | a panel per wave | a wave's scales for the lanes that hold results | the slots' pairs
template <class F> constexpr int wide_ppr() { return ((F::CUT ? F::PB + 29 : F::PB) / 16) | 1; }   // 16-byte pieces of a panel row (odd: banks)
template <int R> constexpr int wide_xbuf() { return (32 * R * (WIDE_REC / 16) + 63) / 64 * 1024; }
template <class F> constexpr int wide_scale_bytes() { return F::KIND == SUPER ? (F::OFF ? 256 : 128) : 1024; }
template <class F, int R> constexpr size_t wide_lds() {
  return 2 * wide_xbuf<R>() + (size_t)WIDE_NW * (512 * wide_ppr<F>() + wide_scale_bytes<F>() + 256) + 16;
}

// GATE: the first expert GEMM of a layer with its seam (Gate16): a wave's 32 weight rows are 16 features of the gate half and the
// same of the up half, so that a lane has both sums of eight features; two waves finish a q8_1 block of h together.
template <class F, int R, bool MOE, bool GATE>
__global__ __launch_bounds__(64 * WIDE_NW, R == 1 ? 3 : 2) void tile_wide_kernel(const uint8_t* __restrict__ W, const char* __restrict__ X, void* __restrict__ Y,
                                                                                 WideArgs a, MoeArgs moe, Gate16 gate) {
  constexpr int M_T = 32 * R, PPR = wide_ppr<F>(), SLOT = 512 * PPR, NI = (32 * PPR + 63) / 64;   // (the last fetch: lanes 0 .. 31)
  constexpr int XB = wide_xbuf<R>(), RING_AT = 2 * XB, SC_AT = RING_AT + WIDE_NW * SLOT, ID_AT = SC_AT + WIDE_NW * wide_scale_bytes<F>();
  constexpr int XP = WIDE_REC / 16, XI = (M_T * XP + 63) / 64, XW = (XI + WIDE_NW - 1) / WIDE_NW;   // pieces of a record; fetches of a buffer; a wave's, at most
  static_assert(wide_lds<F, R>() <= 80 * 1024, "two workgroups do not fit in LDS");
  static_assert(!GATE || MOE, "a gated product is a layer's");
  static_assert(!MOE || (R == 1 && F::KIND == SUPER && !F::OFF), "blocks of 32 slots; the small ones below have no offsets");
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lane = tid & 63, lrow = lane & 31, half = lane >> 5;
  // (a layer's instances count the lanes again before and behind their panels: what is formed from the number would go to scratch beside them)
  const auto lane_again = [&] {
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lane));
    lrow = lane & 31;
    half = lane >> 5;
  };

  // ---- which rows and columns.  Tiles are numbered along the columns of a row block, and the workgroups go to the XCDs in turn: with
  // a multiple of eight columns the blocks of an expert find its weights in one L2, and the blocks past the last live one, of
  // which nothing is done, are spread over all XCDs.  (Runs of 4 / 16 tiles to an XCD: +1 to 4 % / +3 to 6 %; whole blocks, 8
  // experts, 80 tokens: 109 us the layer against 81.)
  const int tile = (int)blockIdx.x;
  const int block = tile / a.col_wgs, col_wg = tile - block * a.col_wgs;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const int ids_at = ID_AT + wave * 256;
  if constexpr (MOE) {
    const int live = moe.num_tokens_post_padded[0], e = moe.expert_ids[block];
    if (block * M_T >= live || e < 0 || e > 255) return;    // (experts above 255: the reference's guard, moe.cuh:33)
    W += (int64_t)e * moe.expert_stride;
    wide_fetch_words(4 * min(lane, M_T - 1), moe.sorted_token_ids + block * M_T, lds0 + ids_at);
  }
  const int p0 = a.ksplit > 1 ? a.np * (int)blockIdx.y / a.ksplit : 0, p1 = a.ksplit > 1 ? a.np * ((int)blockIdx.y + 1) / a.ksplit : a.np;

  // ---- fetching weights: piece number -> (row of the panel, 16-byte piece of it)
  const int rows_all = GATE ? 2 * gate.inner : a.N;
  const int n0 = GATE ? 64 * col_wg + 16 * wave : WIDE_N * col_wg + 32 * wave;   // this wave's first weight row (feature)
  const auto row_of = [&](int r) { return GATE ? (r < 16 ? min(n0 + r, gate.inner - 1) : gate.inner + min(n0 + r - 16, gate.inner - 1)) : min(n0 + r, a.N - 1); };
  const uint32_t wmis = F::CUT ? (uint32_t)((uintptr_t)W & 15) : 0u;
  const uint8_t* const wbase = W - wmis;
  const uint32_t row_bytes = F::KIND == SUPER ? (uint32_t)(a.np * F::PB) : (uint32_t)(a.nkb * (F::PB / 8));
  const uint32_t last16 = ((uint32_t)(rows_all - 1) * a.w_pitch + wmis + row_bytes - 1) & ~15u;   // the last granule that holds bytes of W
  uint32_t w_at[NI], w_piece[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int q = min(64 * i + lane, 32 * PPR - 1), r = q / PPR;
    w_at[i] = (uint32_t)row_of(r) * a.w_pitch + wmis;
    w_piece[i] = 16 * (uint32_t)(q - r * PPR);
    if constexpr (MOE) asm volatile("" : "+v"(w_at[i]));    // (one value for both of the loops below: a second form of it would go to scratch)
  }
  const auto request = [&](int p) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const uint32_t v = min(((w_at[i] + (uint32_t)(p * F::PB)) & ~15u) + w_piece[i], last16);
      const uint32_t to = lds0 + RING_AT + wave * SLOT + 1024 * i;
      if (i < NI - 1) wide_fetch(v, wbase, to);
      else wide_fetch_half(v, wbase, to);   // (lanes past the panel's last piece stay out: their bytes would land in the next slot)
    }
  };
  request(p0);

  // ---- fetching records: a wave's fetches of a buffer, pieces 64 i .. of it for i = wave, wave + 4, ...
  uint32_t x_at[XW];
  if constexpr (MOE) wide_wait<NI>();                       // (the slots' pairs are here)
#pragma unroll
  for (int j = 0; j < XW; ++j) {
    const int q = min(64 * (wave + WIDE_NW * j) + lane, M_T * XP - 1), r = q / XP;
    int row;
    if constexpr (MOE) {
      const int id = *(const int*)(smem + ids_at + 4 * r);
      row = id < moe.num_pairs ? (moe.top_k == 1 ? id : (int)__umulhi((uint32_t)id, a.topk_inv)) : 0;   // row 0 stands in for padding
    } else {
      row = min(block * M_T + r, a.M - 1);
    }
    x_at[j] = (uint32_t)row * WIDE_REC + 16 * (uint32_t)(q - r * XP);
  }
  const auto fetch_x = [&](int ch) {                        // chunk ch: 128 values
    const char* const base = X + (uint64_t)(uint32_t)ch * a.x_plane;
#pragma unroll
    for (int j = 0; j < XW; ++j)
      if (wave + WIDE_NW * j < XI) wide_fetch(x_at[j], base, lds0 + (ch & 1) * XB + 1024 * (wave + WIDE_NW * j));
  };
  fetch_x(2 * p0);

  if constexpr (MOE) {
    // The pairs of a block come first, padding behind them: where the upper sixteen slots hold none, as in about every second expert's last block, tiles of
    // 16 x 16, half the matrix instructions and multiply-adds: a lane has one row of X and weight rows 16 i + 4 g + e.
    if ((__ballot(*(const int*)(smem + ids_at + 4 * lrow) < moe.num_pairs) >> 16 & 0xFFFFu) == 0) {
      lane_again();
      int c = lane & 15, g = lane >> 4;
      char* const scales = smem + SC_AT + wave * wide_scale_bytes<F>();
      const wide_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
      wide_f4 acc[2] = {zero, zero}, part[2];
      for (int p = p0; p < p1; ++p) {
        F w;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          if (hh == 1 && p + 1 < p1) wide_wait<NI>();       // (as below)
          else wide_wait<0>();
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          if (hh == 0 || p + 1 < p1) fetch_x(2 * p + hh + 1);
          if (hh == 0) {
            w.read(smem + RING_AT + wave * SLOT + lrow * (16 * PPR), F::CUT ? ((uint32_t)row_of(lrow) * a.w_pitch + wmis + (uint32_t)(p * F::PB)) & 15 : 0u, half);
            w.scale_to((float*)scales, lrow, half);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (p + 1 < p1) request(p + 1);
          }
          const char* const xrow = smem + hh * XB + c * WIDE_REC;
          const uint2 head = *(const uint2*)(xrow + WIDE_D_AT);
          float d8[4] = {half_bits(head.x & 0xFFFF), half_bits(head.x >> 16), half_bits(head.y & 0xFFFF), half_bits(head.y >> 16)};
          asm volatile("" : "+v"(d8[0]), "+v"(d8[1]), "+v"(d8[2]), "+v"(d8[3]));
          f16x8 xo[2], wo[2][F::PLANES];
          wide_f4 s[2][2];
          const auto load_x = [&](int b) { xo[b & 1] = *(const f16x8*)(xrow + 64 * b + 16 * g); };
          // Of the lane's two operands, eight values each of one of 32 rows, the second of lanes 0 .. 15 and 32 .. 47 and the first of the lanes behind them
          // change places: then either has 16 rows' 32 values.
          const auto decode = [&](int b) {
            f16x8 o[F::PLANES][2];
            w.operand(4 * hh + b, half, o);
#pragma unroll
            for (int pl = 0; pl < F::PLANES; ++pl) {
              typedef uint32_t Words __attribute__((ext_vector_type(4)));
              Words u = __builtin_bit_cast(Words, o[pl][0]), v = __builtin_bit_cast(Words, o[pl][1]);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const auto z = __builtin_amdgcn_permlane16_swap(u[e], v[e], false, false);
                u[e] = z[0];
                v[e] = z[1];
              }
              wo[0][pl] = __builtin_bit_cast(f16x8, u);
              wo[1][pl] = __builtin_bit_cast(f16x8, v);
            }
          };
          const auto scale = [&](int b, int i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) part[i][r] = hh == 0 && b == 0 ? s[b & 1][i][r] * d8[b] : __builtin_fmaf(s[b & 1][i][r], d8[b], part[i][r]);
            asm volatile("" : "+v"(part[i]));
          };
          load_x(0);
          load_x(1);
          decode(0);
#pragma unroll
          for (int b = 0; b < 4; ++b) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
              for (int pl = 0; pl < F::PLANES; ++pl) s[b & 1][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wo[i][pl], xo[b & 1], pl == 0 ? zero : s[b & 1][i], 0, 0, 0);
              __builtin_amdgcn_sched_barrier(0);
              if (b > 0) scale(b - 1, i);
              __builtin_amdgcn_sched_barrier(0);
            }
            if (b + 2 < 4) load_x(b + 2);
            if (b + 1 < 4) decode(b + 1);
          }
          scale(3, 0);
          scale(3, 1);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const wide_f4 d = *(const wide_f4*)(scales + 4 * (16 * i + 4 * g));
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][e] = __builtin_fmaf(part[i][e], d[e], acc[i][e]);
        }
      }
      lane_again();
      c = lane & 15;
      g = lane >> 4;
      const int pair = *(const int*)(smem + ids_at + 4 * c);
      if constexpr (GATE) {
        float h[4];                                         // features 4 g + e of the wave's sixteen
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = seam_gate(seam_rounded(acc[0][e], a.dtype), seam_rounded(acc[1][e], a.dtype), gate.act, a.dtype);
        __syncthreads();
        wide_f4* const all = (wide_f4*)smem;
        all[wave * 64 + lane] = (wide_f4){h[0], h[1], h[2], h[3]};
        __syncthreads();
        if (n0 >= gate.inner) return;
        const wide_f4 o = all[(wave ^ 1) * 64 + lane];
        float amax = 0.0f, t[4];                            // (the same butterfly: 16, 8, 4, 2, 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          amax = fmaxf(fmaxf(amax, fabsf(h[e])), fabsf(o[e]));
          t[e] = h[e] + o[e];
          t[e] += __shfl_xor(t[e], 32);
          t[e] += __shfl_xor(t[e], 16);
        }
        amax = fmaxf(amax, __shfl_xor(amax, 32));
        amax = fmaxf(amax, __shfl_xor(amax, 16));
        const float sum = (t[0] + t[2]) + (t[1] + t[3]), d = amax / 127.0f;
        float q[4];
        seam_quants(h, d, amax == 0.0f, q);
        if (pair < moe.num_pairs) {
          char* const rec = seam_h_record(gate, n0, pair, moe.num_pairs);
          const int blk = (n0 >> 5) & 3;
          seam_h_store(rec, gate, blk, (n0 & 16) + 4 * g, q);
          if (g == 0 && (n0 & 16) == 0) seam_h_scales(rec, gate, blk, d, sum);
        }
      } else {
        if (a.ksplit > 1) Y = (float*)Y + (int64_t)blockIdx.y * a.split_stride;
        if (pair < moe.num_pairs)
#pragma unroll
          for (int i = 0; i < 2; ++i) wide_store(acc[i], pair, n0 + 16 * i + 4 * g, Y, a);
      }
      return;
    }
  }

  float acc[R][16], part[R][16];
#pragma unroll
  for (int k = 0; k < R; ++k)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[k][r] = 0.0f;
  f32x16 zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.0f;
  char* const scales = smem + SC_AT + wave * wide_scale_bytes<F>();

  for (int p = p0; p < p1; ++p) {
    F w;
    uint2 sums[R][2];
    f32x16 off[R];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      // This chunk's records have landed, and with hh = 0 the panel; what was asked for behind them are the next panel's weights.
      // (Records asked for two chunks ahead: no faster.)
      if (hh == 1 && p + 1 < p1) wide_wait<NI>();
      else wide_wait<0>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // (and this wave has read the last of the chunk before)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (hh == 0 || p + 1 < p1) fetch_x(2 * p + hh + 1);
      if (hh == 0) {
        const char* const panel = smem + RING_AT + wave * SLOT + lrow * (16 * PPR);
        const uint32_t at = F::CUT ? ((uint32_t)row_of(lrow) * a.w_pitch + wmis + (uint32_t)(p * F::PB)) & 15 : 0u;
        w.read(panel, at, half);
        if (F::KIND != SUPER && a.nkb < 8 * (p + 1)) w.limit(a.nkb - 8 * p);
        w.scale_to((float*)scales, lrow, half);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the panel's place may be filled again
        if (p + 1 < p1) request(p + 1);
      }
      const char* const xrow = smem + hh * XB + lrow * WIDE_REC;
      float d8[R][4], s8[R][4];                             // (s8: FACTOR times the sums)
      uint2 dh[R], sh[R];                                   // the same as halves, and the sums
      f16x8 xo[2][2], wo[F::PLANES][2];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const uint4 v = *(const uint4*)(xrow + 32 * WIDE_REC * k + WIDE_D_AT);
        d8[k][0] = half_bits(v.x & 0xFFFF);
        d8[k][1] = half_bits(v.x >> 16);
        d8[k][2] = half_bits(v.y & 0xFFFF);
        d8[k][3] = half_bits(v.y >> 16);
        sums[k][hh] = sh[k] = make_uint2(v.z, v.w);
        dh[k] = make_uint2(v.x, v.y);
        // (as floats from here on: the compiler would have every multiply-add convert its scale, in a form that takes twice as long)
        asm volatile("" : "+v"(d8[k][0]), "+v"(d8[k][1]), "+v"(d8[k][2]), "+v"(d8[k][3]));
        if constexpr (F::FACTOR != 0.0f) {
          s8[k][0] = F::FACTOR * half_bits(v.z & 0xFFFF);
          s8[k][1] = F::FACTOR * half_bits(v.z >> 16);
          s8[k][2] = F::FACTOR * half_bits(v.w & 0xFFFF);
          s8[k][3] = F::FACTOR * half_bits(v.w >> 16);
          asm volatile("" : "+v"(s8[k][0]), "+v"(s8[k][1]), "+v"(s8[k][2]), "+v"(s8[k][3]));
        }
      }
      const auto load_x = [&](int u, f16x8 (&o)[2]) {       // unit u: block u / R of the chunk, rows 32 (u % R) ..
#pragma unroll
        for (int h = 0; h < 2; ++h) o[h] = *(const f16x8*)(xrow + 32 * WIDE_REC * (u % R) + 64 * (u / R) + 32 * half + 16 * h);
      };
      f32x16 s[2];
      constexpr int U = 4 * R, P = 2 * F::PLANES;
      const auto mfma = [&](int u, int piece) {
        f32x16& v = s[u & 1];
        v = __builtin_amdgcn_mfma_f32_32x32x16_f16(wo[piece >> 1][piece & 1], xo[u & 1][piece & 1], piece == 0 ? zero : v, 0, 0, 0);
      };
      load_x(0, xo[0]);
      load_x(1, xo[1]);
      w.operand(4 * hh, half, wo);
#pragma unroll
      for (int piece = 0; piece < P; ++piece) mfma(0, piece);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int b = 4 * hh + u / R, k = u % R;
        __builtin_amdgcn_sched_barrier(0);
        f16x8 xm, xn;                                       // the operands of unit u, whose place is taken now
        if constexpr (F::MIN16) { xm = xo[u & 1][0]; xn = xo[u & 1][1]; }
        if (u + 2 < U) load_x(u + 2, xo[u & 1]);
        if (u + 1 < U && (u + 1) % R == 0) w.operand(4 * hh + (u + 1) / R, half, wo);
        wide_f4 dw[4];
        uint2 wd[4], wm[4];
        f16x2 xd, xs;
        if constexpr (F::KIND == BLOCK)
#pragma unroll
          for (int q = 0; q < 4; ++q) dw[q] = *(const wide_f4*)(scales + 4 * (32 * b + 8 * q + 4 * half));
        if constexpr (F::KIND == HALVES) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            wd[q] = *(const uint2*)(scales + 2 * (32 * b + 8 * q + 4 * half));
            wm[q] = *(const uint2*)(scales + 512 + 2 * (32 * b + 8 * q + 4 * half));
          }
          const uint32_t twice = u / R & 1 ? 0x03020302u : 0x01000100u;
          xd = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0u, u / R < 2 ? dh[k].x : dh[k].y, twice));
          xs = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0u, u / R < 2 ? sh[k].x : sh[k].y, twice));
        }
        if constexpr (F::MIN16) {
          // d8 times the sum of the lane's sixteen quants (whole numbers up to 2032, exact as halves), a contraction over the
          // block's two groups in fp32
          f16x8 v = xm + xn;
          const f16x2 t = (f16x2){v[0], v[1]} + (f16x2){v[2], v[3]}, z = (f16x2){v[4], v[5]} + (f16x2){v[6], v[7]}, y = t + z;
          off[k] = __builtin_amdgcn_mfma_f32_32x32x2f32(w.min16(b), d8[k][b & 3] * (float)(y[0] + y[1]), b == 0 ? zero : off[k], 0, 0, 0);
        }
#pragma unroll
        for (int piece = 0; piece < P; ++piece) {
          if (u + 1 < U) mfma(u + 1, piece);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int r = 16 / P * piece; r < 16 / P * (piece + 1); ++r) {
            if constexpr (F::KIND == SUPER) {
              part[k][r] = b == 0 ? s[u & 1][r] * d8[k][b & 3] : __builtin_fmaf(s[u & 1][r], d8[k][b & 3], part[k][r]);
            } else if constexpr (F::KIND == BLOCK && F::FACTOR != 0.0f) {
              acc[k][r] = __builtin_fmaf(__builtin_fmaf(s[u & 1][r], d8[k][b & 3], s8[k][b & 3]), dw[r >> 2][r & 3], acc[k][r]);
            } else if constexpr (F::KIND == BLOCK) {
              acc[k][r] = __builtin_fmaf(s[u & 1][r] * dw[r >> 2][r & 3], d8[k][b & 3], acc[k][r]);
            } else {
              const uint32_t dp = r & 2 ? wd[r >> 2].y : wd[r >> 2].x, mp = r & 2 ? wm[r >> 2].y : wm[r >> 2].x;
              const f16x2 dd = __builtin_bit_cast(f16x2, dp) * xd, ms = __builtin_bit_cast(f16x2, mp) * xs;
              acc[k][r] += __builtin_fmaf(s[u & 1][r], (float)dd[r & 1], (float)ms[r & 1]);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (F::KIND == SUPER) wide_pin(part[k]);
        else wide_pin(acc[k]);
      }
    }
    // ---- the end of the panel: the offsets (a contraction over eight: the upper half of the lanes holds values 8 .. 15, zeros),
    // the super-block's scales
    uint4 mv = make_uint4(0, 0, 0, 0);
    if constexpr (F::OFF && !F::MIN16) {
      if (half == 0) mv = w.offsets();
    }
    if constexpr (F::KIND == SUPER)
#pragma unroll
    for (int k = 0; k < R; ++k) {
      if constexpr (F::OFF && !F::MIN16) {
        const uint4 sv = half ? make_uint4(0, 0, 0, 0) : make_uint4(sums[k][0].x, sums[k][0].y, sums[k][1].x, sums[k][1].y);
        off[k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, mv), __builtin_bit_cast(f16x8, sv), zero, 0, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        wide_f4 d, dm;
        d = *(const wide_f4*)(scales + 4 * (8 * q + 4 * half));
        if constexpr (F::OFF) dm = *(const wide_f4*)(scales + 128 + 4 * (8 * q + 4 * half));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float& v = acc[k][4 * q + e];
          v = __builtin_fmaf(part[k][4 * q + e], d[e], v);
          if constexpr (F::OFF) v = __builtin_fmaf(off[k][4 * q + e], dm[e], v);
        }
      }
    }
  }

  // ---- results: lane = one row of X, 16 weight rows in runs of four
  if constexpr (MOE) lane_again();
  if constexpr (GATE) {
    // h of eight features, 8 q + 4 half + e of the wave's sixteen: rows 0 .. 15 of the panel are the gate's sums, 16 .. 31 the up half's
    float h[R][8];
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float gv = seam_rounded(acc[k][i], a.dtype), uv = seam_rounded(acc[k][8 + i], a.dtype);
        h[k][i] = seam_gate(gv, uv, gate.act, a.dtype);
      }
    // The q8_1 block has 32 features: the other sixteen are the next wave's (the last one's).  amax and the sum as q8_1_quantize8
    // forms them, by a butterfly over 16 (the other wave), 8 (the lane's other run), 4 (the other half's lane), 2, 1.
    __syncthreads();                                        // (the values go over the records)
    wide_f4* const mine = (wide_f4*)smem + (wave * R * 2) * 64 + lane;
    const wide_f4* const other = (const wide_f4*)smem + ((wave ^ 1) * R * 2) * 64 + lane;
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
      for (int q = 0; q < 2; ++q) mine[(2 * k + q) * 64] = (wide_f4){h[k][4 * q], h[k][4 * q + 1], h[k][4 * q + 2], h[k][4 * q + 3]};
    __syncthreads();
    if (n0 >= gate.inner) return;
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const wide_f4 o0 = other[(2 * k) * 64], o1 = other[(2 * k + 1) * 64];
      float amax = 0.0f, t[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        amax = fmaxf(fmaxf(amax, fmaxf(fabsf(h[k][e]), fabsf(h[k][4 + e]))), fmaxf(fabsf(o0[e]), fabsf(o1[e])));
        t[e] = (h[k][e] + o0[e]) + (h[k][4 + e] + o1[e]);
        t[e] += __shfl_xor(t[e], 32);
      }
      amax = fmaxf(amax, __shfl_xor(amax, 32));
      const float sum = (t[0] + t[2]) + (t[1] + t[3]), d = amax / 127.0f;
      float q[8];
      seam_quants(h[k], d, amax == 0.0f, q);
      const int pair = *(const int*)(smem + ids_at + 4 * (32 * k + lrow));
      if (pair < moe.num_pairs) {
        char* const rec = seam_h_record(gate, n0, pair, moe.num_pairs);
        const int blk = (n0 >> 5) & 3;
#pragma unroll
        for (int i = 0; i < 2; ++i) seam_h_store(rec, gate, blk, (n0 & 16) + 8 * i + 4 * half, q + 4 * i);
        if (half == 0 && (n0 & 16) == 0) seam_h_scales(rec, gate, blk, d, sum);
      }
    }
    return;
  }
  if (a.ksplit > 1) Y = (float*)Y + (int64_t)blockIdx.y * a.split_stride;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    int64_t row = block * M_T + 32 * k + lrow;
    if constexpr (MOE) row = *(const int*)(smem + ids_at + 4 * (32 * k + lrow));
    const bool live = row < (MOE ? moe.num_pairs : a.M);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const wide_f4 v = {acc[k][4 * q], acc[k][4 * q + 1], acc[k][4 * q + 2], acc[k][4 * q + 3]};
      if (live) wide_store(v, row, n0 + 8 * q + 4 * half, Y, a);
    }
  }
}

template <class F, int R, bool MOE, bool GATE>
static int wide_launch(const WideCall& c, hipStream_t stream) {
  constexpr size_t lds = wide_lds<F, R>();
  const int qk = F::KIND == SUPER ? 256 : 32, bs = F::KIND == SUPER ? F::PB : F::PB / 8;
  const int64_t pitch = c.w_pitch ? c.w_pitch : (int64_t)(c.K / qk) * bs;
  if (!F::CUT && (pitch % 16 != 0 || (uintptr_t)c.W % 16 != 0 || (c.moe.sorted_token_ids && c.moe.expert_stride % 16 != 0))) return GGUF_NOT_TAKEN;
  auto kern = tile_wide_kernel<F, R, MOE, GATE>;
  static std::atomic<uint64_t> done{0};
  allow_large_lds(kern, lds, done);
  const int cols = GATE ? (c.gate.inner + 63) / 64 : (c.N + WIDE_N - 1) / WIDE_N, top_k = c.moe.top_k > 0 ? c.moe.top_k : 1;
  const bool split = c.ksplit > 1;
  const int dtype = split ? GGUF_DTYPE_F32 : c.dtype, elt = dtype == GGUF_DTYPE_F32 ? 4 : 2;
  const int64_t ldy = split || !c.ldy ? (int64_t)c.N : c.ldy, rows_y = c.moe.sorted_token_ids ? c.moe.num_pairs : c.M;
  void* const y = split ? (void*)c.partial : c.Y;
  const WideArgs a = {c.M, c.N, (c.K + 255) / 256, c.K / 32, cols, (uint32_t)pitch, (uint32_t)(c.x_rows * WIDE_REC), (uint32_t)((0x100000000ull + top_k - 1) / top_k),
                      dtype, ldy % 4 == 0 && (uintptr_t)y % (4 * elt) == 0, ldy, split ? nullptr : c.bias, split ? c.ksplit : 1, rows_y * ldy};
  hipLaunchKernelGGL(kern, dim3((unsigned)((int64_t)c.row_blocks * cols), (unsigned)a.ksplit), dim3(64 * WIDE_NW), lds, stream, (const uint8_t*)c.W, (const char*)c.x,
                     y, a, c.moe, c.gate);
  return launch_status();
}

template <class F>
static int wide_dense_run(const WideCall& c, hipStream_t s) {
  if (c.gate.rows || c.moe.sorted_token_ids || c.K % (F::KIND == SUPER ? 256 : 32) != 0) return GGUF_NOT_TAKEN;
  return c.rt == 1 ? wide_launch<F, 1, false, false>(c, s) : wide_launch<F, 2, false, false>(c, s);
}
// a layer's products (blocks of 32 slots)
template <class F>
static int wide_moe_run(const WideCall& c, hipStream_t s) {
  if (!c.moe.sorted_token_ids || c.K % 256 != 0 || c.rt != 1) return GGUF_NOT_TAKEN;
  return c.gate.rows ? wide_launch<F, 1, true, true>(c, s) : wide_launch<F, 1, true, false>(c, s);
}
template <class F>
static int wide_run(const WideCall& c, hipStream_t s) { return c.moe.sorted_token_ids ? wide_moe_run<F>(c, s) : wide_dense_run<F>(c, s); }
// a dense product whose rows do not begin on 16 bytes (a shard of a merged tensor as wide as its widest one): A the panels that do
template <class A, class F>
static int wide_run_either(const WideCall& c, hipStream_t s) {
  return (uintptr_t)c.W % 16 == 0 && c.w_pitch % 16 == 0 ? wide_dense_run<A>(c, s) : wide_dense_run<F>(c, s);
}

}  // namespace gguf
