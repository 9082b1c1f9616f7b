// Products with a few rows of activations (5 to 32; up to 512 of a small matrix), dense and per expert of an MoE layer, that run near the rate
// the packed weights stream in.
//
// What bounds such a product is the weight stream; what keeps a kernel from it is everything around it: decoded weights
// staged in LDS for the whole workgroup cost a barrier per step of K and line the waves up; operands read straight from
// the packed blocks need four matrix instructions per block with three quarters of the activations zeroed.  Here the
// waves of a workgroup walk their own weights on their own:
//   * A wave's unit of work is a panel: 16 weight rows x 256 values of K.  It fetches the panel's bytes as 16-byte
//     pieces, lane after lane, straight into its own LDS ring (global_load_lds; D panels in flight), reads its lanes'
//     fields from there, asks for another panel and multiplies: one v_mfma_i32_16x16x32_i8 per 32-value block and 16
//     rows of X.  No register holds bytes in flight and no barrier stands between panels.
//   * The activations of a chunk of K (up to 16 panels) lie in LDS for the eight waves, fetched the same way, a row's
//     1 KB per request; a chunk is fetched while the one before is multiplied where LDS has room for two.  (Operands
//     read from global memory instead cost the CU's memory pipeline 64 cycles per request -- 16 rows, 16 cache lines --
//     450 of them per panel, where the panel's bytes arrive in 250.)  The quantizer stores a row such that a lane's
//     operand of two blocks is one 16-byte read (q8_permuted).
//   * The offset term of Q4_0, Q4_K, Q5_K -- minus min times block sum, a contraction over blocks -- is two fp32 matrix
//     instructions per panel (v_mfma_f32_16x16x4_f32, fp32 inputs and sums) instead of a multiply-add per result and
//     block, and each lane decodes two of the eight mins instead of all of them.
//   * Block sums leave the matrix unit as floats (the accumulator starts at the bit pattern of 1.5 * 2^23), so the two
//     block scales are two multiply-adds per result.  About 150 vector instructions per 4096 Q4_K weights at 16 rows.
//   * Where the output has fewer column groups than the chip has waves, KS waves share a group and deal K panel by
//     panel; their partial tiles are added through LDS in the order of K (SPLIT).  Else a wave finishes its columns alone.
// Measured (us per call with the quantizer's launch, before -> now; 5.15 TB/s is what a copy of 1 GiB reaches): [28672,8192]
// Q4_K, 16 rows 45.7 -> 37.6 (3.5 TB/s with the quantizer's 3.5 us inside), 32 rows 73.7 -> 54.0; [6144,4096] Q8_0, 16 rows 18.8 -> 13.4;
// [12288,1024] Q6_K, 16 rows 21.5 -> 11.7.  MoE layers: Q4_0, 64 experts, top-8, 64 tokens 112 -> 76; Q4_K with Q6_K, 128
// experts, 300 tokens 262 -> 175.  What is left is the beginning of a workgroup (first chunk of activations, first
// panels: 4 to 6 us) and the vector instructions around the multiplications.
// Arithmetic as in the other integer kernels (mmq.cuh:2-104, vecdotq.cuh: exact int32 block sums, scales in fp32).
#pragma once
#include "mmq_i_core.h"
#include "q8_1_device.h"
#include "tile_stream.h"
#include "tile_stream_formats.h"
#include <type_traits>

namespace gguf {

struct TsArgs {
  int M, N, K, Kp;             // M: rows of X (dense)
  uint32_t w_pitch, ws_row_bytes;
  int np, ks_log2, ppr;        // panels per row; waves that share a column group; 16-byte pieces of LDS for a weight row's panel
  int pc_log2, nbuf;           // panels per chunk of activations in LDS, chunks in LDS
  int passes;                  // column groups a wave walks one after the other (more than one: all of K is one chunk)
  uint32_t ppr_inv, rb_inv, topk_inv;   // 2^32 / (ppr, the coarse row blocks, top_k) rounded up: the kernel starts without a division
  int coarse;                  // MoE: workgroups of the coarse row blocks; those behind them share a column group's K between two waves
  int coarse_blocks;           // (all blocks, where nothing is cut finer)
  uint32_t fine_inv;           // 2^32 / the other row blocks
  int plane, dtype;            // block sums for the offset term: 1 = stored sums, 2 = d * sum(q); GGUF_DTYPE_* of Y
  int64_t ldy;
  const void* bias;
};

// What the first requests are formed from comes as scalars in front as well (GGUF_GEOM, mmvq_core.h): the kernels take those fields from there.
#define GGUF_TS_HEAD uint32_t h_pitch, uint32_t h_ws_row, int h_m, int h_n, int h_k, uint32_t h_small, uint32_t h_ppr_inv
#define GGUF_TS_HEAD_ARGS(a)                                                                                                                                             \
  (a).w_pitch, (a).ws_row_bytes, (a).M, (a).N, (a).K,                                                                                                                     \
      (uint32_t)(a).ppr | (uint32_t)(a).ks_log2 << 8 | (uint32_t)(a).pc_log2 << 10 | (uint32_t)(a).nbuf << 13 | (uint32_t)(a).plane << 15 | (uint32_t)(a).passes << 17, (a).ppr_inv
__device__ __forceinline__ TsArgs ts_args(GGUF_TS_HEAD, TsArgs a) {
  a.w_pitch = h_pitch; a.ws_row_bytes = h_ws_row; a.M = h_m; a.N = h_n; a.K = h_k; a.ppr_inv = h_ppr_inv;
  a.Kp = (int)q8_kp(h_k); a.np = (h_k + 255) >> 8;
  a.ppr = h_small & 255; a.ks_log2 = h_small >> 8 & 3; a.pc_log2 = h_small >> 10 & 7; a.nbuf = h_small >> 13 & 3; a.plane = h_small >> 15 & 3; a.passes = h_small >> 17;
  return a;
}
#define GGUF_TS_ARGS(rest) ts_args(h_pitch, h_ws_row, h_m, h_n, h_k, h_small, h_ppr_inv, rest)

typedef uint32_t u32x4_s __attribute__((ext_vector_type(4)));
typedef _Float16 ts_h2 __attribute__((ext_vector_type(2)));

template <int N> __device__ __forceinline__ void ts_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// wave-uniform 16-byte-per-lane fetch into LDS: lane l's bytes land at m0 + 16 l
__device__ __forceinline__ void ts_fetch(uint32_t at, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(at), "s"(base), "s"(lds) : "memory");
}
// the same for the lanes in `mask` only (all lanes are active before and after)
__device__ __forceinline__ void ts_fetch_some(uint32_t at, const void* base, uint32_t lds, uint64_t mask) {
  asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(at), "s"(base), "s"(lds), "s"(mask) : "memory");
}
template <int ROR>
__device__ __forceinline__ float ts_ror(float v) {   // rotation inside a row of 16 lanes
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + ROR, 0xF, 0xF, true));
}
__device__ __forceinline__ float ts_rounded(float v, int dtype) {   // to the result's type and back
  return dtype == GGUF_DTYPE_F32 ? v : dtype == GGUF_DTYPE_F16 ? (float)(_Float16)v : bf16_to_f32(f32_to_bf16(v));
}
__device__ __forceinline__ void ts_store(void* Y, int64_t at, float v, const void* bias, int n, int dtype) {
  if (dtype == GGUF_DTYPE_F16) ((_Float16*)Y)[at] = finish<_Float16>(v, (const _Float16*)bias, n);
  else if (dtype == GGUF_DTYPE_BF16) ((bf16_t*)Y)[at] = finish<bf16_t>(v, (const bf16_t*)bias, n);
  else ((float*)Y)[at] = finish<float>(v, (const float*)bias, n);
}

// Where the scales of block b of a chunk begin, in floats: XR per block, and a gap of sixteen behind every four blocks so
// that threads that place four blocks each, one behind the other, meet different banks.  (Sums over whole fours of blocks.)
template <int XR> __host__ __device__ __forceinline__ constexpr int ts_scale_at(int b) { return b * XR + (b >> 2) * 16; }

// GATE: the first expert GEMM of a layer with its seam (Gate16): of four neighbouring column groups two are 32 features of
// the gate half and two the same features of the up half; the sums meet in LDS and the workgroup finishes the q8_1
// blocks of h from them.
// bytes of LDS that a format's tables take (F::TABLE, filled by F::tables, read through the member tab), 0 for most
template <class F, class = void> struct TsTable { static constexpr int value = 0; };
template <class F> struct TsTable<F, std::void_t<decltype(F::TABLE)>> { static constexpr int value = (F::TABLE + 15) / 16 * 16; };
// formats of which an MoE layer's last round of workgroups may be cut finer (ts_tail; the other two that layers have, Q6_K and Q8_0, gain nothing)
template <class F> constexpr bool ts_fine() { return std::is_same<F, TQ4_0>::value || std::is_same<F, TQ4_K>::value || std::is_same<F, TQ5_K>::value; }
template <class F> constexpr bool ts_sums() { return F::OFF == 1 || F::HALVES; }   // the activations' block sums are wanted

// A panel's products: sum += (without ADD sum =) what the lane's column of it has with the rows of X.  (Handing the panel's sums to every caller
// takes registers off the kernels that only add them, and 4 % off the speed of Q2_K, 1 % of Q4_K and Q5_K at two tiles of rows.)  xa: the
// lane's quants of the eight blocks; so: block sums g and 4 + g of row c; left: blocks of the panel inside the row; half0: all bits in the lanes that hold the first 16
// values of a block; d8_of, s8_of: block scales and sums of the lane's four result rows.
template <class F, int RT, bool ADD, class D8, class S8>
__device__ __forceinline__ void ts_multiply(F& w, const u32x4_s (&xa)[RT][4], const float (&so)[RT][2], int left, int g, uint32_t half0, D8 d8_of, S8 s8_of,
                                            f32x4 (&sum)[RT]) {
  constexpr bool OFFSET = F::OFF == 1;
  const v4i seed = {kSeedBits, kSeedBits, kSeedBits, kSeedBits};
  float dw[8 * (32 / F::G)];
  w.ready();
  uint32_t dm[8];
  if constexpr (F::HALVES) w.words(dm);
  else w.scales(dw);
  // (opaque to the compiler, which would keep both masked copies of all operands over the column groups and spill)
  uint32_t first = half0;
  asm volatile("" : "+v"(first));
  if (!F::KQ && left < 8) {
#pragma unroll
    for (int b = 0; b < 8; ++b) {                       // (bytes behind the row's end need not be a number)
      if constexpr (F::HALVES) dm[b] = b < left ? dm[b] : 0u;
      else dw[b] = b < left ? dw[b] : 0.0f;
    }
  }
  float m0 = 0.0f, m1 = 0.0f;
  if constexpr (OFFSET) {
    w.mins(g, m0, m1);
    if (!F::KQ && left < 8) { m0 = g < left ? m0 : 0.0f; m1 = 4 + g < left ? m1 : 0.0f; }
  }
  // A sum of the panel's own, added to the row's at its end: the partial sums stay small, and so does what they round off.  So too with the
  // offsets of four blocks, which cancel most of their products: they come between the second and the third (rel-L2 against 64 bits, Q4_K, 5 .. 32
  // rows, activations of one sign / normal: 10.2e-7 / 1.50e-7 with the offsets in front, now 5.8e-7 / 1.33e-7;
  // Q6_K 1.17e-7 with the sum carried on from panel to panel, now 0.95e-7).
  f32x4 part[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) part[rt] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    if (OFFSET && (b & 3) == 2) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) part[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(so[rt][b >> 2], b < 4 ? -m0 : -m1, part[rt], 0, 0, 0);
    }
    const uint2 q = w.codes(b, g);
    const long bv = (long)(((uint64_t)q.y << 32) | q.x);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const f32x4 d8 = d8_of(rt, b);
      const uint32_t alo = xa[rt][b >> 1][2 * (b & 1)], ahi = xa[rt][b >> 1][2 * (b & 1) + 1];
      if constexpr (F::HALVES) {
        const f32x4 s8 = s8_of(rt, b);
        const ts_h2 v = __builtin_bit_cast(ts_h2, dm[b]), dv = {v[0], v[0]}, mv = {v[1], v[1]};
        const v4i s = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(((uint64_t)ahi << 32) | alo), bv, seed, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; r += 2) {                // (d8 and s8 are halves in fp32)
          const ts_h2 dd = (ts_h2){(_Float16)d8[r], (_Float16)d8[r + 1]} * dv, ms = (ts_h2){(_Float16)s8[r], (_Float16)s8[r + 1]} * mv;
#pragma unroll
          for (int e = 0; e < 2; ++e) part[rt][r + e] += __builtin_fmaf(seeded_times(s[r + e], 1.0f, -kSeed), (float)dd[e], (float)ms[e]);
        }
      } else if constexpr (F::G == 32) {
        const float nsd = -kSeed * dw[b];
        const v4i s = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(((uint64_t)ahi << 32) | alo), bv, seed, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) part[rt][r] = __builtin_fmaf(seeded_times(s[r], dw[b], nsd), d8[r], part[rt][r]);
        if constexpr (F::OFF == 2) {
          const uint2 mq = w.min_codes(b);
          const float dmin = w.dmin();
          const v4i sm = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(((uint64_t)ahi << 32) | alo), (long)(((uint64_t)mq.y << 32) | mq.x), seed, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) part[rt][r] = __builtin_fmaf(seeded_times(sm[r], -dmin, kSeed * dmin), d8[r], part[rt][r]);
        }
      } else {
        // a scale per 16 values: the activations of either half of the block, the other half's lanes zeroed
        const long a0 = (long)(((uint64_t)(ahi & first) << 32) | (alo & first));
        const long a1 = (long)(((uint64_t)(ahi & ~first) << 32) | (alo & ~first));
        const float n0 = -kSeed * dw[2 * b], n1 = -kSeed * dw[2 * b + 1];
        const v4i s0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a0, bv, seed, 0, 0, 0);
        const v4i s1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a1, bv, seed, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          part[rt][r] = __builtin_fmaf(seeded_times(s0[r], dw[2 * b], n0), d8[r], part[rt][r]);
          part[rt][r] = __builtin_fmaf(seeded_times(s1[r], dw[2 * b + 1], n1), d8[r], part[rt][r]);
        }
      }
    }
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) sum[rt] = ADD ? sum[rt] + part[rt] : part[rt];
}

template <class F, int RT, bool GATE, bool SPLIT, int D, bool MOE>
__global__ __launch_bounds__(64 * TS_NW, RT == 1 && !SPLIT ? 4 : 2) void tile_stream_kernel(const uint8_t* __restrict__ W, const char* __restrict__ ws, GGUF_TS_HEAD,
                                                                                  int row_blocks, int total, void* __restrict__ Y, TsArgs rest, MoeArgs moe,
                                                                                  Gate16 gate) {
  const TsArgs a = GGUF_TS_ARGS(rest);
  static_assert(!GATE || (MOE && !SPLIT), "a gated product is a layer's and takes its column groups whole");
  static_assert(!MOE || RT == 1, "blocks of 16 slots");
  static_assert(D >= 2 && D <= 4, "one wait per number of panels requested behind the one at hand");
  constexpr int NW = TS_NW, XR = 16 * RT, XR_LOG2 = RT == 1 ? 4 : 5;
  constexpr bool SUMS = ts_sums<F>(), OFFSET = F::OFF == 1;
  constexpr int PPR_MIN = (F::PB + 15) / 16, PPR_MAX = (F::PB + 29) / 16;     // pieces of an aligned / of any panel row
  constexpr int NI = (16 * (PPR_MAX | 1) + 63) / 64, FULL = 16 * PPR_MIN / 64;      // fetch instructions; those with all lanes on
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;

  // ---- which rows, columns and panels
  // What the last round of workgroups has to do is cut finer (ts_tail): half as many column groups, two waves to each.
  constexpr bool FINER = MOE && !SPLIT && ts_fine<F>();
  const bool fine = FINER && (int)blockIdx.x >= a.coarse;
  int wg = fine ? blockIdx.x - a.coarse : blockIdx.x;
  const int rb = fine ? row_blocks - a.coarse_blocks : a.coarse_blocks;
  const int total8 = (fine ? total - a.coarse : a.coarse) & ~7;   // each of the 8 XCDs gets a contiguous run of workgroups
  if (wg < total8) wg = (wg & 7) * (total8 >> 3) + (wg >> 3);
  // (the blocks of one expert are neighbours: they share its weights)
  const int col_wg = rb == 1 ? wg : (int)__umulhi((uint32_t)wg, fine ? a.fine_inv : a.rb_inv), block = wg - col_wg * rb + (fine ? a.coarse_blocks : 0);
  if constexpr (MOE) {
    const int live = moe.num_tokens_post_padded[0], e = moe.expert_ids[block];
    if (block * XR >= live || e < 0 || e > 255) return;     // (experts above 255: the reference's guard, moe.cuh:33)
    W += (int64_t)e * moe.expert_stride;
  }
  const int ks_log2 = SPLIT ? a.ks_log2 : fine ? 1 : 0, KS = 1 << ks_log2, CS = NW >> ks_log2;
  const int ks = wave >> (3 - ks_log2), cs = wave & (CS - 1);
  const int passes = SPLIT || fine ? 1 : a.passes;
  const int groups = GATE ? gate.inner / 8 : (a.N + 15) / 16;   // (inner is a multiple of 32)
  const int group0 = (col_wg * CS + cs) * passes;           // the first of this wave's column groups

  // ---- LDS: [chunk buffers: quants [XR][pitch], scales and sums [blocks][XR]][fetch rings]; partial tiles over the chunks
  const int PC = 1 << a.pc_log2, pitch = 256 * PC + 16;
  const int xq_bytes = XR * pitch, xs_bytes = ts_scale_at<XR>(8 * PC) * 4 * (SUMS ? 2 : 1), buf_bytes = xq_bytes + xs_bytes;
  const int slot_bytes = 256 * a.ppr;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const int ring_off = a.nbuf * buf_bytes + wave * (D * slot_bytes);

  // ---- fetching weights: piece number -> (row of the panel, 16-byte piece of it)
  const int table_off = a.nbuf * buf_bytes + NW * (D * slot_bytes) + 16;   // (a last field's cut may touch the word behind the rings)
  const uint32_t wmis = (uint32_t)((uintptr_t)W & 15);
  const uint8_t* const wbase = W - wmis;
  const uint32_t row_bytes = (uint32_t)(F::KQ ? a.np * F::PB : (a.K >> 5) * (F::PB / 8));
  const int rows_all = GATE ? 2 * gate.inner : a.N;
  const uint32_t last16 = ((uint32_t)(rows_all - 1) * a.w_pitch + wmis + row_bytes - 1) & ~15u;   // the last granule that holds bytes of W
  uint32_t prow[NI], pc16[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int p = min(64 * i + lane, 16 * a.ppr - 1);
    const uint32_t r = __umulhi((uint32_t)p, a.ppr_inv);
    prow[i] = r * a.w_pitch;
    pc16[i] = (uint32_t)min(p - (int)r * a.ppr, PPR_MAX - 1) * 16;   // (the piece that only spaces rows: the last again)
  }
  // byte offset of the first row of a column group, and of the last row a group may touch
  const auto group_at = [&](int pass, uint32_t& last) -> uint32_t {
    const int grp = group0 + pass;
    if constexpr (GATE) {   // groups 4 u, 4 u + 1: features 32 u .. of the gate half; 4 u + 2, 4 u + 3: of the up half
      const int half = (grp >> 1) & 1;
      last = (uint32_t)((half + 1) * gate.inner - 1) * a.w_pitch;
      return (uint32_t)(half * gate.inner + 32 * (grp >> 2) + 16 * (grp & 1)) * a.w_pitch;
    } else {
      last = (uint32_t)(a.N - 1) * a.w_pitch;
      return (uint32_t)(16 * grp) * a.w_pitch;
    }
  };
  const auto request = [&](int pass, int p, int slot) {
    uint32_t last;
    const uint32_t at = group_at(pass, last), off = (uint32_t)(p * F::PB) + wmis;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const uint32_t row = min(at + prow[i], last);
      const uint32_t v = min(((row + off) & ~15u) + pc16[i], last16);
      const uint32_t to = lds0 + ring_off + slot * slot_bytes + 1024 * i;
      if (i < FULL) {
        ts_fetch(v, wbase, to);
      } else {   // (lanes past the panel's last piece stay out: their bytes would land in the next slot)
        const int on = 16 * a.ppr - 64 * i;
        ts_fetch_some(v, wbase, to, on >= 64 ? ~0ull : on <= 0 ? 0ull : (1ull << on) - 1);
      }
    }
  };
  // this wave's tasks, the panels of its column groups, and the next one to request
  const int my_passes = max(0, min(passes, groups - group0));
  const int np_mine = a.np > ks ? (a.np - ks + KS - 1) >> ks_log2 : 0;
  const int tasks = np_mine * my_passes;
  int rq_p = ks, rq_pass = 0, requested = 0;
  const auto request_next = [&](int slot) {
    if (requested >= tasks) return;
    request(rq_pass, rq_p, slot);
    ++requested;
    rq_p += KS;
    if (rq_p >= a.np) {
      rq_p = ks;
      ++rq_pass;
    }
  };

  // ---- fetching activations.  Lane l knows where row l % XR of the tile begins; quants go to LDS directly, one row's
  // 1 KB per request, scales and sums (four blocks of a row per thread) take a detour so that LDS holds them block-major.
  uint32_t row_at;
  int pair_at = 0;                                          // MoE: the pair behind slot lane % XR
  const int nb = a.Kp >> 5, nkb = a.K >> 5;
  const auto fetch_quants = [&](int ch, int buf) {
    const int parts_log2 = a.pc_log2 - 2;                   // KB of a row per chunk
    for (int q = wave; q < XR << parts_log2; q += NW) {
      const int row = q >> parts_log2, part = q & ((1 << parts_log2) - 1);
      const uint32_t base = __builtin_amdgcn_readlane(row_at, row);
      // (past the padded row's end: its last piece again)
      const uint32_t at = min((uint32_t)(256 * PC * ch + 1024 * part + 16 * lane), (uint32_t)a.Kp - 16);
      ts_fetch(base + at, ws, lds0 + buf * buf_bytes + row * pitch + 1024 * part);
    }
  };
  constexpr int NS = 2;                                     // (row, four blocks, plane) items per thread, at most
  u32x4_s sreg[NS];
  const int items = (XR * 2 * PC) * (SUMS ? 2 : 1);       // items, rows fastest
  const auto scales_at = [&](int ch, int i) -> uint32_t {
    const int it = tid + 64 * NW * i, row = it & (XR - 1), q = (it >> XR_LOG2) & (2 * PC - 1), plane = it >> (XR_LOG2 + 1 + a.pc_log2);
    return __shfl(row_at, row) + a.Kp + (plane ? 4 * a.plane * nb : 0) + min(16 * (uint32_t)(2 * PC * ch + q), 4 * (uint32_t)nb - 16);
  };
  const auto place_scales = [&](int ch, int buf) {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const int it = tid + 64 * NW * i, row = it & (XR - 1), q = (it >> XR_LOG2) & (2 * PC - 1), plane = it >> (XR_LOG2 + 1 + a.pc_log2);
      float* const to = (float*)(smem + buf * buf_bytes + xq_bytes) + plane * ts_scale_at<XR>(8 * PC) + row;
      if (it < items)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t bits = sreg[i][e];   // (a bit cast applied to the vector element itself reads element 0)
          to[ts_scale_at<XR>(4 * q) + e * XR] = 8 * PC * ch + 4 * q + e < nkb ? __uint_as_float(bits) : 0.0f;
        }
    }
  };
  // The first chunk's are asked for before the weights and must not wait for those, so the compiler cannot be the one that
  // waits, and a register of its own is nothing that a load in flight may own.  They land in LDS, the 64 items of a wave
  // one behind the other where the 64 items' transposed copy begins, and are spread out from there: the items of a wave
  // are all rows of neighbouring blocks, so nobody else has anything in that place, and a wave's reads come before its writes.
  const auto first_scales_lds = [&](int i) -> uint32_t {
    const int it = 64 * (wave + NW * i), q = (it >> XR_LOG2) & (2 * PC - 1), plane = it >> (XR_LOG2 + 1 + a.pc_log2);
    return (uint32_t)(xq_bytes + 4 * (plane * ts_scale_at<XR>(8 * PC) + ts_scale_at<XR>(4 * q)));
  };
  const auto fetch_first_scales = [&]() {
#pragma unroll
    for (int i = 0; i < NS; ++i)
      if (64 * (wave + NW * i) < items) ts_fetch(scales_at(0, i), ws, lds0 + first_scales_lds(i));
  };
  const auto place_first_scales = [&]() {
    f32x4 v[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i)
      if (64 * (wave + NW * i) < items) v[i] = *(const f32x4*)(smem + first_scales_lds(i) + 16 * lane);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const int it = tid + 64 * NW * i, row = it & (XR - 1), q = (it >> XR_LOG2) & (2 * PC - 1), plane = it >> (XR_LOG2 + 1 + a.pc_log2);
      float* const to = (float*)(smem + xq_bytes) + plane * ts_scale_at<XR>(8 * PC) + row;
      if (64 * (wave + NW * i) < items)
#pragma unroll
        for (int e = 0; e < 4; ++e) to[ts_scale_at<XR>(4 * q) + e * XR] = 4 * q + e < nkb ? v[i][e] : 0.0f;
    }
  };

  if constexpr (MOE) {
    // The weights do not wait for the routing: the pairs behind a block's slots come as scalar loads, which have a counter
    // of their own, and are waited for behind the first requests of weights without waiting for the weights.
    int slot_ids[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) slot_ids[r] = moe.sorted_token_ids[block * 16 + r];
#pragma unroll
    for (int d = 0; d < D; ++d) request_next(d);
    int id = slot_ids[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) id = c == r ? slot_ids[r] : id;
    pair_at = id;
    row_at = (id < moe.num_pairs ? (moe.top_k == 1 ? (uint32_t)id : __umulhi((uint32_t)id, a.topk_inv)) : 0u) * a.ws_row_bytes;   // row 0 stands in for padding
    fetch_first_scales();
    fetch_quants(0, 0);
    ts_wait<0>();
  } else {
    row_at = (uint32_t)min(block * XR + (lane & (XR - 1)), a.M - 1) * a.ws_row_bytes;
    fetch_first_scales();
    fetch_quants(0, 0);
#pragma unroll
    for (int d = 0; d < D; ++d) request_next(d);
    if (requested == D) ts_wait<D * NI>();
    else ts_wait<0>();
  }
  place_first_scales();
  if constexpr (TsTable<F>::value) F::tables(smem + table_off);
  __syncthreads();

  const uint32_t half0 = g < 2 ? ~0u : 0u;                  // lanes that hold the first 16 values of a block
  const auto store = [&](int m, int n, float v) {           // result row m of this workgroup's tile, feature n (all lanes together)
    const int row = MOE ? __shfl(pair_at, m) : block * XR + m;
    if (n < a.N && row < (MOE ? moe.num_pairs : a.M)) ts_store(Y, (int64_t)row * a.ldy + n, v, a.bias, n, a.dtype);
  };
  const int chunks = (a.np + PC - 1) >> a.pc_log2;
  int t = 0, slot = 0;                                      // tasks done, ring slot of the next
  // Where blocks may have K dealt to two waves, the others too add the even and the odd panels in two sums: a pair's result does not
  // depend on the block that it is in.
  f32x4 acc[RT], odd, kept[4];                              // kept (gated): the last four column groups' sums
  for (int pass = 0; pass < passes; ++pass) {
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  odd = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  const int pass_end = min(tasks, (pass + 1) * np_mine);
  int p = ks;
  for (int ch = 0; ch < chunks; ++ch) {
    const bool more = ch + 1 < chunks;
    const int buf = a.nbuf == 2 ? ch & 1 : 0;
    if constexpr (SPLIT) {
      if (more) {
        // (these loads are the compiler's to wait for, which will wait for every panel in flight along with them)
#pragma unroll
        for (int i = 0; i < NS; ++i) sreg[i] = *(const u32x4_s*)(ws + scales_at(ch + 1, i));
        if (a.nbuf == 2) fetch_quants(ch + 1, buf ^ 1);
      }
    }
    const char* const xq = smem + buf * buf_bytes;
    const float* const xd = (const float*)(xq + xq_bytes);
    for (; t < pass_end && p < (ch + 1) << a.pc_log2; p += KS) {
      const int pl = p - (ch << a.pc_log2);                 // panel of the chunk
      u32x4_s xa[RT][4];
      float so[RT][2];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) xa[rt][i] = *(const u32x4_s*)(xq + (16 * rt + c) * pitch + 256 * pl + 64 * i + 16 * g);
        if constexpr (OFFSET) {
          const float* const sums = xd + ts_scale_at<XR>(8 * PC) + ts_scale_at<XR>(8 * pl) + g * XR + 16 * rt + c;
          so[rt][0] = sums[0];
          so[rt][1] = sums[ts_scale_at<XR>(4)];
        }
      }
      const int left = nkb - 8 * p;                         // blocks of the panel inside the row
      // Loads return in order: the panel has landed once no more are outstanding than the panels behind it asked for.
      const int ahead = requested - t - 1;
      if (D > 3 && ahead >= 3) ts_wait<3 * NI>();
      else if (D > 2 && ahead >= 2) ts_wait<2 * NI>();
      else if (ahead >= 1) ts_wait<NI>();
      else ts_wait<0>();
      uint32_t last;
      const uint32_t w_at = min(group_at(pass, last) + c * a.w_pitch, last) + (uint32_t)(p * F::PB) + wmis;
      F w;
      if constexpr (TsTable<F>::value) w.tab = smem + table_off;
      w.read(smem + ring_off + slot * slot_bytes + c * (16 * a.ppr), F::PB % 16 == 0 && a.ppr == F::PB / 16 ? 0u : w_at & 15, g);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot may be filled again
      request_next(slot);
      ++t;
      slot = slot + 1 == D ? 0 : slot + 1;

      f32x4 part[RT];                                       // (FINER: of the panel alone)
      ts_multiply<F, RT, !FINER>(w, xa, so, left, g, half0, [&](int rt, int b) { return *(const f32x4*)(xd + ts_scale_at<XR>(8 * pl) + ts_scale_at<XR>(b) + 16 * rt + 4 * g); },
                         [&](int rt, int b) { return *(const f32x4*)(xd + ts_scale_at<XR>(8 * PC) + ts_scale_at<XR>(8 * pl) + ts_scale_at<XR>(b) + 16 * rt + 4 * g); }, FINER ? part : acc);
      if constexpr (FINER) {
        if (p & 1) odd += part[0];
        else acc[0] += part[0];
      }
    }
    // ---- the next chunk of activations
    if constexpr (SPLIT) {
      if (more) {
        if (a.nbuf == 1) {
          __syncthreads();                                  // every wave is done with this one
          fetch_quants(ch + 1, 0);
        }
        ts_wait<0>();
        place_scales(ch + 1, a.nbuf == 2 ? buf ^ 1 : 0);
        __syncthreads();
      }
    }
  }
  if constexpr (FINER) acc[0] += odd;                       // (a finer workgroup's waves have one of the two)
  if constexpr (GATE) {
#pragma unroll
    for (int i = 0; i < 3; ++i) kept[i] = kept[i + 1];
    kept[3] = acc[0];
  } else if constexpr (!SPLIT) {
    if (fine) {                                             // the two waves' sums, over the activations
      f32x4* const red = (f32x4*)smem;
      __syncthreads();
      if (ks) red[cs * 64 + lane] = acc[0];
      __syncthreads();
      if (ks) return;
      acc[0] += red[cs * 64 + lane];
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r) store(16 * rt + 4 * g + r, 16 * (group0 + pass) + c, acc[rt][r]);
  }
  }

  if constexpr (GATE) {
    // One (unit of 32 features, result register r) per wave and turn: a lane has slot 4 g + r of features 16 i + c, i = 0, 1:
    // sums rounded as the operator stores them, activated, and quantized as q8_1_quantize8 does -- amax and the sum over
    // the 32 features by the same butterfly (16 apart in the lane, then 8, 4, 2, 1 as rotations inside the row of 16 lanes,
    // whose partners agree at each step).
    // (the sums go over the activations, so that two workgroups still fit a CU's LDS)
    __syncthreads();
    float* const sums = (float*)smem;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i >= 4 - passes) *(f32x4*)(sums + ((wave * passes + i - (4 - passes)) * 64 + lane) * 4) = kept[i];
    __syncthreads();
    const int units = fine ? 1 : 2 * passes;                // of 32 features
    const float* const other = sums + 4 * 64 * 4;           // (fine: the sums of the second wave of each group)
    for (int it = wave; it < units * 4; it += NW) {
      const int u = it >> 2, r = it & 3, unit = units * col_wg + u;
      if (32 * unit >= gate.inner) break;
      const int pair = __shfl(pair_at, 4 * g + r);
      float h[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int at = ((4 * u + i) * 64 + lane) * 4 + r;
        const float gv = ts_rounded(fine ? sums[at] + other[at] : sums[at], a.dtype);
        const float uv = ts_rounded(fine ? sums[at + 512] + other[at + 512] : sums[at + 512], a.dtype);
        h[i] = a.dtype == GGUF_DTYPE_F32 ? gate1<float>(gv, uv, gate.act) : a.dtype == GGUF_DTYPE_F16 ? gate1<_Float16>(gv, uv, gate.act) : gate1<bf16_t>(gv, uv, gate.act);
      }
      float amax = fmaxf(fabsf(h[0]), fabsf(h[1])), sum = h[0] + h[1];
      amax = fmaxf(amax, ts_ror<8>(amax));
      sum += ts_ror<8>(sum);
      amax = fmaxf(amax, ts_ror<4>(amax));
      sum += ts_ror<4>(sum);
      amax = fmaxf(amax, ts_ror<2>(amax));
      sum += ts_ror<2>(sum);
      amax = fmaxf(amax, ts_ror<1>(amax));
      sum += ts_ror<1>(sum);
      const float d = amax / 127.0f, dd = amax == 0.0f ? 1.0f : d;
      int q[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) q[i] = (int)roundf(h[i] / dd);
      int isum = q[0] + q[1];
      isum += dpp_mov_i<0x128>(isum);
      isum += dpp_mov_i<0x124>(isum);
      isum += dpp_mov_i<0x122>(isum);
      isum += dpp_mov_i<0x121>(isum);
      if (pair < moe.num_pairs) {
        char* const row = gate.rows + (int64_t)pair * gate.row_bytes;
#pragma unroll
        for (int i = 0; i < 2; ++i) row[q8_permuted(32 * unit + 16 * i + (c & 8)) + (c & 7)] = (char)q[i];
        if (c == 0) {
          float* fd = (float*)(row + gate.kp);
          const int nbh = gate.kp >> 5;
          const float dh = (float)(_Float16)d;
          fd[unit] = dh;
          fd[nbh + unit] = (float)(_Float16)sum;
          fd[2 * nbh + unit] = dh * (float)isum;
        }
      }
    }
    return;
  }
  if constexpr (SPLIT) {
    // ---- the KS partial tiles of every column group, added in the order of K
    float* const red = (float*)smem;                        // [NW][RT][64] of four floats, over the activations
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) *(f32x4*)(red + ((wave * RT + rt) * 64 + lane) * 4) = acc[rt];
    __syncthreads();
    constexpr int per_cs = RT * 64;
    for (int i = tid; i < CS * per_cs; i += 64 * NW) {
      const int s = i / per_cs, rest = i - s * per_cs;      // column slice; (rt, lane) of its tiles
      f32x4 v = *(const f32x4*)(red + (s * per_cs + rest) * 4);
      for (int z = 1; z < KS; ++z) v += *(const f32x4*)(red + ((z * CS + s) * per_cs + rest) * 4);
      const int l = rest & 63, rt = rest >> 6;
#pragma unroll
      for (int r = 0; r < 4; ++r) store(16 * rt + 4 * (l >> 4) + r, 16 * (col_wg * CS + s) + (l & 15), v[r]);
    }
  }
}

// A column group per workgroup, its panels of K dealt to the eight waves: where the output has too few column groups for a wave
// each.  No two waves of a workgroup multiply the same activations then, so a wave fetches those of its panel beside the
// panel's weights, into a place of its own, and meets the others only for the sum: no chunk of activations that the workgroup
// waits for, loads, and waits for again (2.5 us each, seven of them at K = 14336).  A wave has one panel under way, asked for as soon
// as the one before is in registers, and sixteen waves share a CU: two panels a wave on eight waves were slower by a fifth, as
// were one workgroup of sixteen waves (a tenth) and of four.
// In LDS: the panel's bytes, block scales and sums of its sixteen rows of X (32 bytes each, 512 the plane), their quants, 256 bytes
// a row.  An operand is 16 bytes of each of sixteen rows, all in the same banks: piece j of row r lies in place j ^ r, which the
// fetch sees to (a lane asks for the piece that belongs where its bytes land).  Rows past X are fetched up to a multiple of four
// only: the rest of the place holds whatever it held, for rows of the result that are not stored.
// What bounds it is the weight stream, and beside it the activations' way to every workgroup (2.3 us of [4096,14336]'s 15) and the
// vector instructions of a panel (Q6_K 350: 5 us).  Without the quantizer's launch, us, streaming tiles / this, 12 rows: Q6_K [4096,14336]
// 22.1 / 15.1, [4096,4096] 9.6 / 7.1, [1024,4096] 8.5 / 5.9; Q4_K [4096,14336] 16.9 / 11.7, [11008,4096] 13.4 / 10.7, [2048,2048] 5.8 / 4.0; 24
// rows Q6_K [4096,14336] 29.5 / 25.0, [4096,4096] 11.5 / 8.9.
// CG: up to so many column groups of a workgroup (ts_dealt_groups), a panel of K after the other: the activations' operands and block scales stay
// in registers over the groups (the scales as the halves that they are), a group's panel is asked for while the one before is multiplied, and
// there is one beginning and one sum for all.  From two on the groups are walked by a loop that is not unrolled, which moves the partial tiles
// around by one each time: unrolled the compiler keeps more than there are registers.  (A ring of two weight panels per wave: 0.8 to 1.03 times
// the speed.)  Tried and slower: whole column groups one after the other,
// the activations fetched again for each (0.86 to 1.06 times the speed of a workgroup each).
template <int RT> __host__ __device__ constexpr int ts_dealt_place(int ppr) { return 256 * ppr + 1024 * RT + 4096 * RT; }
// where, behind the panel's bytes, piece 4 i + g of the quants of row 16 rt + c begins
template <int RT> __host__ __device__ constexpr int ts_dealt_quants(int rt, int i, int c, int g) { return 1024 * RT + 4096 * rt + 256 * c + 16 * ((4 * i + g) ^ c); }
template <int RT> constexpr bool ts_dealt_reads_inside() {
  for (int u = 0; u < 256 * RT; ++u)
    if (ts_dealt_quants<RT>(u >> 8, u & 3, (u >> 2) & 15, (u >> 6) & 3) + 16 > ts_dealt_place<RT>(0)) return false;
  return true;
}
static_assert(ts_dealt_reads_inside<1>() && ts_dealt_reads_inside<2>(), "a wave reads its own place only");
// (two workgroups of one tile of rows share a CU where its registers suffice)
template <class F, int RT> constexpr int ts_dealt_waves() { return RT == 1 && !F::HALVES && (F::KQ || F::OFF != 1) ? 4 : 2; }
template <class F, int RT, int CG>
__device__ __forceinline__ void tile_dealt_body(const uint8_t* __restrict__ W, const char* __restrict__ ws, void* __restrict__ Y, const TsArgs& a, int wg, int wgs) {
  constexpr int NW = TS_NW;
  constexpr bool SUMS = ts_sums<F>(), OFFSET = F::OFF == 1;
  constexpr int PPR_MIN = (F::PB + 15) / 16, PPR_MAX = (F::PB + 29) / 16;
  constexpr int NI = (16 * (PPR_MAX | 1) + 63) / 64, FULL = 16 * PPR_MIN / 64;
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int total8 = wgs & ~7;                              // each of the 8 XCDs gets a contiguous run of workgroups
  if (wg < total8) wg = (wg & 7) * (total8 >> 3) + (wg >> 3);
  const int ng = CG > 2 ? a.passes : CG;                    // column groups, the last of the last workgroup perhaps behind the matrix
  const int xn = (a.M + 3) >> 2;                            // fetches of quants per panel, four rows each
  const int w_bytes = 256 * a.ppr, place = ts_dealt_place<RT>(a.ppr);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const int mine = wave * place, table_off = NW * place + 16;   // (a last field's cut may touch the word behind its row)

  const uint32_t wmis = (uint32_t)((uintptr_t)W & 15);
  const uint8_t* const wbase = W - wmis;
  const uint32_t row_bytes = (uint32_t)(F::KQ ? a.np * F::PB : (a.K >> 5) * (F::PB / 8));
  const uint32_t last16 = ((uint32_t)(a.N - 1) * a.w_pitch + wmis + row_bytes - 1) & ~15u;   // the last granule that holds bytes of W
  uint32_t w_at[NI];                                        // the piece behind its row's beginning
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int p = min(64 * i + lane, 16 * a.ppr - 1);
    const uint32_t r = __umulhi((uint32_t)p, a.ppr_inv);
    w_at[i] = (uint32_t)min(16 * ng * wg + (int)r, a.N - 1) * a.w_pitch + wmis +
              (uint32_t)min(p - (int)r * a.ppr, PPR_MAX - 1) * 16;   // (the piece that only spaces rows: the last again)
  }
  const uint32_t step = 16 * a.w_pitch;                     // (a group behind the last column reads the last granule again)
  const auto request_w = [&](int p, int j) {
    const uint32_t to = lds0 + mine, off = (uint32_t)(p * F::PB) + (uint32_t)j * step;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const uint32_t v = min((w_at[i] + off) & ~15u, last16);
      if (i < FULL) {
        ts_fetch(v, wbase, to + 1024 * i);
      } else {   // (lanes past the panel's last piece stay out: their bytes would land behind it)
        const int on = 16 * a.ppr - 64 * i;
        ts_fetch_some(v, wbase, to + 1024 * i, on >= 64 ? ~0ull : on <= 0 ? 0ull : (1ull << on) - 1);
      }
    }
  };
  const auto request_x = [&](int p) {
    const uint32_t to = lds0 + mine + w_bytes;
    int l = lane;                                           // (opaque: computed every time, not kept in registers over the groups)
    if constexpr (CG > 1) asm volatile("" : "+v"(l));
    const int c = l & 15, g = l >> 4;
    uint32_t x_at[4 * RT], s_at[RT];
#pragma unroll
    for (int i = 0; i < 4 * RT; ++i) {
      const int row = 4 * i + g;
      x_at[i] = (uint32_t)min(row, a.M - 1) * a.ws_row_bytes + 16 * (uint32_t)(c ^ (row & 15));
    }
    // (a lane: half of a row's eight scales, in the upper half of the lanes of its sums)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      s_at[rt] = (uint32_t)min(16 * rt + ((l & 31) >> 1), a.M - 1) * a.ws_row_bytes + (uint32_t)a.Kp + 16 * (l & 1) + (SUMS && l >= 32 ? 4 * a.plane * (a.Kp >> 5) : 0);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) ts_fetch(s_at[rt] + 32 * (uint32_t)p, ws, to + 1024 * rt);
#pragma unroll
    for (int i = 0; i < 4 * RT; ++i)
      if (i < xn) ts_fetch(x_at[i] + 256 * (uint32_t)p, ws, to + 1024 * RT + 1024 * i);
  };
  if (wave < a.np) { request_w(wave, 0); request_x(wave); }
  if constexpr (TsTable<F>::value) {
    F::tables(smem + table_off);
    __syncthreads();
  }

  const uint32_t half0 = g < 2 ? ~0u : 0u;                  // lanes that hold the first 16 values of a block
  const int nkb = a.K >> 5;
  f32x4 acc[CG][RT];
#pragma unroll
  for (int j = 0; j < CG; ++j)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[j][rt] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  const char* const at = smem + mine;
  const char* const scales = at + w_bytes;
  const uint32_t w_lane = (uint32_t)min(16 * ng * wg + c, a.N - 1) * a.w_pitch + wmis;
  for (int p = wave; p < a.np; p += NW) {
    const int left = nkb - 8 * p;                           // blocks of the panel inside the row
    ts_wait<0>();
    u32x4_s xa[RT][4];
    float so[RT][2];
    // of rows 4 g + r, blocks 0 .. 7: the block scales, or, with HALVES, (scale, sum) as the halves that they are (behind a row's last
    // block lie the quantizer's zeros)
    float d8[RT][4][CG > 1 && !F::HALVES ? 1 : 8];
    uint32_t d8h[RT][4][4];                                  // CG > 1: as the halves that they are
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) xa[rt][i] = *(const u32x4_s*)(scales + ts_dealt_quants<RT>(rt, i, c, g));
      if constexpr (OFFSET) {
        so[rt][0] = *(const float*)(scales + 1024 * rt + 512 + 32 * c + 4 * g);
        so[rt][1] = *(const float*)(scales + 1024 * rt + 512 + 32 * c + 16 + 4 * g);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 v = *(const f32x4*)(scales + 1024 * rt + 32 * (4 * g + r) + 16 * h);
          f32x4 z = v;
          if constexpr (F::HALVES) z = *(const f32x4*)(scales + 1024 * rt + 512 + 32 * (4 * g + r) + 16 * h);
          if constexpr (CG > 1 && !F::HALVES) {
            d8h[rt][r][2 * h] = __builtin_bit_cast(uint32_t, (ts_h2){(_Float16)v[0], (_Float16)v[1]});
            d8h[rt][r][2 * h + 1] = __builtin_bit_cast(uint32_t, (ts_h2){(_Float16)v[2], (_Float16)v[3]});
          } else
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (F::HALVES) d8[rt][r][4 * h + e] = __builtin_bit_cast(float, (ts_h2){(_Float16)v[e], (_Float16)z[e]});
            else d8[rt][r][4 * h + e] = v[e];
          }
        }
    }
    const auto of = [&](int rt, int b, int half) {
      f32x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (F::HALVES) o[r] = (float)__builtin_bit_cast(ts_h2, d8[rt][r][b])[half];
        else if constexpr (CG > 1) o[r] = (float)__builtin_bit_cast(ts_h2, d8h[rt][r][b >> 1])[b & 1];
        else o[r] = d8[rt][r][b];
      }
      return o;
    };
#pragma unroll 1
    for (int j = 0; j < ng; ++j) {
      if (j > 0) ts_wait<0>();
      F w;                                                  // (read behind the activations: before them Q6_K spills, and loses a tenth)
      if constexpr (TsTable<F>::value) w.tab = smem + table_off;
      w.read(at + c * (16 * a.ppr), F::PB % 16 == 0 && a.ppr == F::PB / 16 ? 0u : (w_lane + (uint32_t)(p * F::PB) + (uint32_t)j * step) & 15, g);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // the place may be filled again
      if (j + 1 < ng) request_w(p, j + 1);
      else if (p + NW < a.np) { request_w(p + NW, 0); request_x(p + NW); }
      ts_multiply<F, RT, true>(w, xa, so, left, g, half0, [&](int rt, int b) { return of(rt, b, 0); }, [&](int rt, int b) { return of(rt, b, 1); }, acc[0]);
      if constexpr (CG > 1) {                               // (the next group's tile first: a tile by number would be in scratch)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          const f32x4 done = acc[0][rt];
#pragma unroll
          for (int i = 0; i < CG; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][rt][r] = i + 1 == ng || i + 1 == CG ? done[r] : acc[i + 1 < CG ? i + 1 : i][rt][r];
        }
      }
    }
  }

  // ---- the eight partial tiles, added in pairs, pairs of pairs and halves: each sum is rounded three times and not seven (Q5_K, activations of
  // one sign, 5 .. 32 rows, rel-L2 against 64 bits: one after the other 5.3e-8, the kernels that ran these products before 5.1e-8, so 4.5e-8)
  __syncthreads();
  float* const red = (float*)smem;                          // [NW][CG][RT][64] of four floats, over the panels
  constexpr int T = CG * RT;
#pragma unroll
  for (int j = 0; j < CG; ++j)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) *(f32x4*)(red + ((wave * T + j * RT + rt) * 64 + lane) * 4) = acc[j][rt];
  __syncthreads();
  for (int i = tid; i < 256 * RT * ng; i += 64 * NW) {
    const int n = i & 15, m = (i >> 4) % (16 * RT), j = i / (256 * RT), l = 16 * ((m >> 2) & 3) + n, t = j * RT + (m >> 4);   // result row m, feature n of group j
    float v[NW];
#pragma unroll
    for (int z = 0; z < NW; ++z) v[z] = red[((z * T + t) * 64 + l) * 4 + (m & 3)];
#pragma unroll
    for (int d = 1; d < NW; d *= 2)
#pragma unroll
      for (int z = 0; z < NW; z += 2 * d) v[z] += v[z + d];
    const int col = 16 * (ng * wg + j) + n;
    if (m < a.M && col < a.N) ts_store(Y, (int64_t)m * a.ldy + col, v[0], a.bias, col, a.dtype);
  }
}

template <class F, int RT, int CG>
__global__ __launch_bounds__(64 * TS_NW, (ts_dealt_waves<F, RT>())) void tile_dealt_kernel(const uint8_t* __restrict__ W, const char* __restrict__ ws, GGUF_TS_HEAD, int wgs, void* __restrict__ Y,
                                                                                                 TsArgs rest) {
  // (of many groups the scalars would go to scratch: from memory they are loaded where they are wanted)
  tile_dealt_body<F, RT, CG>(W, ws, Y, CG > 2 ? rest : GGUF_TS_ARGS(rest), blockIdx.x, wgs);
}

// The same for two matrices with the same rows of X, those of a merged layer whose recipe gives one of its tensors more bits: the
// workgroups of the second, often too few for the chip by themselves, run beside the first's, and a launch less.
template <class F, class G, int RT, int CG>
__global__ __launch_bounds__(64 * TS_NW, (ts_dealt_waves<F, RT>() < ts_dealt_waves<G, RT>() ? ts_dealt_waves<F, RT>() : ts_dealt_waves<G, RT>())) void tile_dealt_pair_kernel(
    const uint8_t* __restrict__ W, const char* __restrict__ ws, GGUF_TS_HEAD, int wgs, const uint8_t* __restrict__ V, void* __restrict__ Y, void* __restrict__ Z, TsArgs rest, TsArgs b) {
  if ((int)blockIdx.x < wgs) tile_dealt_body<F, RT, CG>(W, ws, Y, GGUF_TS_ARGS(rest), blockIdx.x, wgs);
  else tile_dealt_body<G, RT, CG>(V, ws, Z, b, blockIdx.x - wgs, gridDim.x - wgs);
}

static inline size_t ts_chunk_bytes(int rt, bool off, int pc) {
  return (size_t)16 * rt * (256 * pc + 16) + (size_t)(8 * pc * 16 * rt + 2 * pc * 16) * 4 * (off ? 2 : 1);
}

// From which row block on a product of an MoE layer is cut finer: the workgroups run in rounds of `slots`, and what is left for a last,
// partly filled one takes about as long as a full one, a beginning and an end worth about five panels and its waves' panels one
// behind the other, on a chip that is mostly idle.  There a workgroup takes four column groups instead of eight and deals K to two
// waves each, half the panels per wave, where that is one round with a fifth to spare (the number of blocks is an estimate, and
// one more than a round holds is a second one) and saves three panels at least.  (Blocks past the last full round that it
// expects are cut finer in any case.)  us per layer, before / now: 64 experts, top-8, Q4_0 [2048 -> 1024], 64 tokens 80.1 / 76.1; 8 experts, top-2,
// Q4_0 [1792 -> 3584], 43 tokens 58 / 52; 64 experts, top-6, Q4_K [2304 -> 1792], 10 tokens 88 / 82.  Over 200 random layers on streaming tiles
// Q4_K 3.3 %, Q4_0, Q5_K 1.5 %, none slower by more than 2; without the room and the margin as much, but one in fourteen slower, by up to 8 %.  Q6_K
// and Q8_0, whose weights are on their way at the rate that memory has with half the chip's waves, gain nothing (1.000, 1.003) and lose
// up to 7 % where one block more than estimated is there: not cut.
static inline int ts_tail(const TsCall& c, int np, int passes, int cols, int col_wgs, int slots) {
  const int cap = slots / col_wgs;                          // blocks per round
  if (np < 2 || cap == 0) return c.row_blocks;
  const int full = (int)(c.live_blocks / cap);
  const double rest = c.live_blocks - (double)full * cap;
  const bool finer = 1.2 * rest * ((cols + 3) / 4) <= slots && (np + 1) / 2 + 3 < passes * np;
  const int64_t from = (int64_t)(finer ? full : full + 1) * cap;
  return from < c.row_blocks ? (int)from : c.row_blocks;
}

template <class F, int RT, bool GATE, bool SPLIT, int D, bool MOE>
static int ts_launch_d(const TsCall& c, int ks, TsArgs a, size_t lds, hipStream_t stream) {
  auto kern = tile_stream_kernel<F, RT, GATE, SPLIT, D, MOE>;
  const int cols = GATE ? c.gate.inner / 8 : (c.N + 15) / 16, per_wg = TS_NW / ks * a.passes;
  const int col_wgs = (cols + per_wg - 1) / per_wg;
  a.coarse_blocks = SPLIT || !MOE || !ts_fine<F>() ? c.row_blocks : ts_tail(c, a.np, a.passes, cols, col_wgs, lds <= 80 * 1024 ? 512 : 256);
  if (c.finer_from) {
    *c.finer_from = a.coarse_blocks;
    return GGUF_OK;
  }
  const int64_t coarse = (int64_t)col_wgs * a.coarse_blocks, total = coarse + (int64_t)((cols + 3) / 4) * (c.row_blocks - a.coarse_blocks);
  if (total > 0x7FFFFFFFll) return GGUF_ERR_SHAPE;
  a.coarse = (int)coarse;
  a.rb_inv = (uint32_t)((0x100000000ull + a.coarse_blocks - 1) / (a.coarse_blocks > 0 ? a.coarse_blocks : 1));
  a.fine_inv = (uint32_t)((0x100000000ull + c.row_blocks - a.coarse_blocks - 1) / (c.row_blocks > a.coarse_blocks ? c.row_blocks - a.coarse_blocks : 1));
  // the quotients by reciprocal are exact while dividend times divisor stays below 2^32
  if (total * c.row_blocks > 0xFFFFFFFFll || (int64_t)c.moe.num_pairs * (c.moe.top_k > 0 ? c.moe.top_k : 1) > 0xFFFFFFFFll) return GGUF_ERR_SHAPE;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> done{0};
    allow_large_lds(kern, 160 * 1024, done);
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)total), dim3(64 * TS_NW), lds, stream, (const uint8_t*)c.W, (const char*)c.ws, GGUF_TS_HEAD_ARGS(a),
                     c.row_blocks, (int)total, c.Y, a, c.moe, c.gate);
  return launch_status();
}

// Column groups a wave walks one after the other, given the rounds of workgroups on the chip with one each.  A second
// group saves a beginning (4 to 6 us, as long as about six panels) but makes the last round longer: it pays from four
// rounds on (64 experts of Q4_0, 300 tokens: 168 -> 159 us the layer; 128 experts, 64 tokens, three rounds: 106 -> 113),
// and earlier where a group has only a few panels.
static inline int ts_passes(int np, double rounds) {
  int passes = rounds >= 4.0 ? 2 : 1;
  while (passes < 4 && np * passes < 6 && rounds >= 1.5 * passes) passes *= 2;
  return passes;
}

template <class F, int RT, bool GATE, bool SPLIT, bool MOE>
static int ts_launch(const TsCall& c, int ks, hipStream_t stream) {
  const int np = (c.K + 255) / 256, qk = F::KQ ? 256 : 32, bs = F::KQ ? F::PB : F::PB / 8;
  const int64_t pitch = c.w_pitch ? c.w_pitch : (int64_t)(c.K / qk) * bs;
  // pieces per row and panel: one more where a panel may begin inside one
  const bool aligned = F::PB % 16 == 0 && pitch % 16 == 0 && (uintptr_t)c.W % 16 == 0 && (!MOE || c.moe.expert_stride % 16 == 0);
  // (an odd number, so that the same field of 16 rows lies in different banks: [23376,1856] of Q4_0, 16 rows of X 23.2 -> 19.2 us)
  const int ppr = (aligned ? F::PB / 16 : (F::PB + 29) / 16) | 1, top_k = c.moe.top_k > 0 ? c.moe.top_k : 1;
  const auto bytes = [&](int pc, int nbuf, int d) { return nbuf * ts_chunk_bytes(RT, ts_sums<F>(), pc) + (size_t)TS_NW * d * 256 * ppr + 16 + TsTable<F>::value; };
  const size_t room = 160 * 1024;
  int pc_log2 = 2, nbuf = 1;
  while (pc_log2 < 4 && (1 << pc_log2) < np) ++pc_log2;
  if (!SPLIT) {
    if ((1 << pc_log2) < np || bytes(1 << pc_log2, 1, 2) > room) return GGUF_NOT_TAKEN;   // all of K in LDS
  } else if (np > 8 || bytes(1 << pc_log2, 1, 2) > room) {
    // two chunks, the second fetched while the first is multiplied, where that gives every wave of a split a panel
    pc_log2 = 3;
    while (pc_log2 > 2 && bytes(1 << pc_log2, 2, 2) > room) --pc_log2;
    nbuf = 2;
    if ((1 << pc_log2) < ks || bytes(1 << pc_log2, 2, 2) > room) {
      nbuf = 1;
      pc_log2 = 4;
      while (pc_log2 > 2 && bytes(1 << pc_log2, 1, 2) > room) --pc_log2;
    }
  }
  if ((1 << pc_log2) * 2 * 16 * RT * (ts_sums<F>() ? 2 : 1) > 2 * 64 * TS_NW) return GGUF_NOT_TAKEN;   // (two items of scales per thread)
  // (two workgroups per CU overlap their beginnings and ends, and have as many panels in flight between them)
  int d = RT == 1 && bytes(1 << pc_log2, nbuf, 2) <= room / 2 ? 2 : 4;
  while (d > 2 && bytes(1 << pc_log2, nbuf, d) > room) --d;
  size_t lds = bytes(1 << pc_log2, nbuf, d);                // (16 more: the cut of a last field may touch the word behind its row)
  if (SPLIT && lds < (size_t)TS_NW * RT * 1024) lds = (size_t)TS_NW * RT * 1024;
  if (lds > room) return GGUF_NOT_TAKEN;
  const int cols = GATE ? c.gate.inner / 8 : (c.N + 15) / 16;
  const int passes = SPLIT ? 1 : ts_passes(np, c.live_blocks * cols / TS_NW / (lds <= room / 2 ? 512.0 : 256.0));
  const TsArgs a = {c.M, c.N, c.K, (int)q8_kp(c.K), (uint32_t)pitch, (uint32_t)q8_row_bytes(c.K), np, 31 - __builtin_clz(ks), ppr, pc_log2, nbuf, passes,
                    (uint32_t)((0x100000000ull + ppr - 1) / ppr), 0, (uint32_t)((0x100000000ull + top_k - 1) / top_k), 0, 0, 0,
                    c.gemv_sums ? 2 : 1, c.dtype, c.ldy ? c.ldy : (int64_t)c.N, c.bias};
  switch (d) {
    case 4: return ts_launch_d<F, RT, GATE, SPLIT, 4, MOE>(c, ks, a, lds, stream);
    case 3: return ts_launch_d<F, RT, GATE, SPLIT, 3, MOE>(c, ks, a, lds, stream);
    default: return ts_launch_d<F, RT, GATE, SPLIT, 2, MOE>(c, ks, a, lds, stream);
  }
}

// How many column groups a workgroup takes.  Where one of them fills a CU (two tiles of rows, or formats that need the registers), as many as
// let one round do, up to what the registers hold: [11008,4096] Q4_K 20 rows, one to four groups 16.1 / 16.8 / 12.2 / 13.8 us, [28672,4096]
// 35.5 / 32.3 / 32.2 / 27.5, eight 25.9.  Where two share a CU, two groups between one and a half rounds and two, and past two and three
// quarters: [16384,4096] Q4_K 12 rows 14.3 / 12.6, but [10000,4096] 0.9 of the speed; of those formats whose two groups fit the registers (the
// others spill: Q6_K 0.9, IQ2_S 0.95 of the speed; IQ3_S spills three and gains 1.03 all the same).  (Q2_K, two products per block, spills, Q5_K at eight.)
template <class F, class = void> struct TsOneGroup { static constexpr bool value = false; };   // F::ONE_GROUP: registers for one group at four waves per SIMD
template <class F> struct TsOneGroup<F, std::void_t<decltype(F::ONE_GROUP)>> { static constexpr bool value = F::ONE_GROUP; };
template <class F, int RT> constexpr int ts_dealt_most() {
  if (F::OFF == 2) return 1;
  if (ts_dealt_waves<F, RT>() == 4) return F::KQ && !TsOneGroup<F>::value ? 2 : 1;
  return RT == 2 && F::KQ && !std::is_same<F, TQ5_K>::value ? 8 : 4;
}
template <class F, int RT>
static inline int ts_dealt_groups(int groups) {
  constexpr int MOST = ts_dealt_most<F, RT>();
  if (MOST <= 2) return MOST == 2 && ((groups > 768 && groups <= 1024) || groups > 1408) ? 2 : 1;
  const int rounds = (groups + 256 * MOST - 1) / (256 * MOST);
  return (groups + 256 * rounds - 1) / (256 * rounds);
}
// what the kernel is told of a product, and the LDS that it takes
template <class F, int RT>
static TsArgs ts_dealt_args(const TsCall& c, int ng, size_t& lds) {
  const int np = (c.K + 255) / 256, qk = F::KQ ? 256 : 32, bs = F::KQ ? F::PB : F::PB / 8;
  const int64_t pitch = c.w_pitch ? c.w_pitch : (int64_t)(c.K / qk) * bs;
  const bool aligned = F::PB % 16 == 0 && pitch % 16 == 0 && (uintptr_t)c.W % 16 == 0;
  const int ppr = (aligned ? F::PB / 16 : (F::PB + 29) / 16) | 1;   // (odd: banks)
  lds = (size_t)TS_NW * ts_dealt_place<RT>(ppr) + 16 + TsTable<F>::value;
  const int tiles = RT * (ng > 4 ? 8 : ng > 2 ? 4 : ng);    // (the sum's places are laid out for the most that an instance takes)
  if (lds < (size_t)TS_NW * tiles * 1024) lds = (size_t)TS_NW * tiles * 1024;
  return {c.M, c.N, c.K, (int)q8_kp(c.K), (uint32_t)pitch, (uint32_t)q8_row_bytes(c.K), np, 3, ppr, 0, 0, ng, (uint32_t)((0x100000000ull + ppr - 1) / ppr), 0, 0, 0, 0, 0,
          c.gemv_sums ? 2 : 1, c.dtype, c.ldy ? c.ldy : (int64_t)c.N, c.bias};
}
template <class F, int RT, int CG>
static int ts_dealt_launch_cg(const TsCall& c, int ng, hipStream_t stream) {
  size_t lds;
  const TsArgs a = ts_dealt_args<F, RT>(c, ng, lds);
  if (lds > 160 * 1024) return GGUF_NOT_TAKEN;
  auto kern = tile_dealt_kernel<F, RT, CG>;
  static std::atomic<uint64_t> done{0};
  if (lds > 64 * 1024) allow_large_lds(kern, 160 * 1024, done);
  const int wgs = (c.N + 16 * ng - 1) / (16 * ng);
  hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(64 * TS_NW), lds, stream, (const uint8_t*)c.W, (const char*)c.ws, GGUF_TS_HEAD_ARGS(a), wgs, c.Y, a);
  return launch_status();
}
template <class F, int RT>
static int ts_dealt_launch(const TsCall& c, hipStream_t stream) {
  if (c.M > 16 * RT || c.row_blocks != 1) return GGUF_NOT_TAKEN;
  constexpr int MOST = ts_dealt_most<F, RT>();
  const int ng = ts_dealt_groups<F, RT>((c.N + 15) / 16);
  if (ng == 1) return ts_dealt_launch_cg<F, RT, 1>(c, 1, stream);
  if constexpr (MOST >= 2) {
    if (ng == 2) return ts_dealt_launch_cg<F, RT, 2>(c, 2, stream);
  }
  if constexpr (MOST >= 4) {
    if (ng <= 4) return ts_dealt_launch_cg<F, RT, 4>(c, ng, stream);
  }
  if constexpr (MOST == 8) return ts_dealt_launch_cg<F, RT, 8>(c, ng, stream);
  return GGUF_NOT_TAKEN;
}
template <class F, class G, int RT, int CG>
static int ts_dealt_pair_launch(const TsCall& c, const TsCall& d, hipStream_t stream) {
  size_t lds, lds2;
  const TsArgs a = ts_dealt_args<F, RT>(c, CG, lds), b = ts_dealt_args<G, RT>(d, CG, lds2);
  if (lds < lds2) lds = lds2;
  if (lds > 160 * 1024) return GGUF_NOT_TAKEN;
  auto kern = tile_dealt_pair_kernel<F, G, RT, CG>;
  static std::atomic<uint64_t> done{0};
  if (lds > 64 * 1024) allow_large_lds(kern, 160 * 1024, done);
  const int wgs = (c.N + 16 * CG - 1) / (16 * CG);
  hipLaunchKernelGGL(kern, dim3((unsigned)wgs + (unsigned)((d.N + 16 * CG - 1) / (16 * CG))), dim3(64 * TS_NW), lds, stream, (const uint8_t*)c.W, (const char*)c.ws,
                     GGUF_TS_HEAD_ARGS(a), wgs, (const uint8_t*)d.W, c.Y, d.Y, a, b);
  return launch_status();
}
template <class F, class G, int RT>
static int ts_dealt_pair_rt(const TsCall& c, const TsCall& d, hipStream_t s) {
  if constexpr (RT == 2) {
    const int ng = ts_dealt_groups<F, RT>((c.N + 15) / 16 + (d.N + 15) / 16);
    if (ng > 2) return GGUF_NOT_TAKEN;                      // (each by itself: as many groups as suit it)
    if (ng == 2) return ts_dealt_pair_launch<F, G, RT, 2>(c, d, s);
  }
  return ts_dealt_pair_launch<F, G, RT, 1>(c, d, s);
}
template <class F, class G>
static int ts_dealt_pair(const TsCall& c, const TsCall& d, hipStream_t s) {
  return c.M <= 16 ? ts_dealt_pair_rt<F, G, 1>(c, d, s) : ts_dealt_pair_rt<F, G, 2>(c, d, s);
}

template <class F, int RT, bool MOE = false>
static int ts_run_rt(const TsCall& c, hipStream_t stream) {
  const int np = (c.K + 255) / 256;
  if constexpr (!MOE) {
    if (c.dealt) {
      const int rc = ts_dealt_launch<F, RT>(c, stream);
      if (rc != GGUF_NOT_TAKEN) return rc;
    }
  }
  const int ks = ts_ks(np, c.live_blocks * ((c.N + 15) / 16));
  if (ks == 1 && np <= 16) {
    const int rc = ts_launch<F, RT, false, false, MOE>(c, 1, stream);
    if (rc != GGUF_NOT_TAKEN) return rc;
  }
  return ts_launch<F, RT, false, true, MOE>(c, ks, stream);
}

template <class F>
static int ts_dense_run(const TsCall& c, hipStream_t stream) {
  if (c.moe.sorted_token_ids || c.gate.rows) return GGUF_NOT_TAKEN;
  return c.rt == 1 ? ts_run_rt<F, 1>(c, stream) : c.rt == 2 ? ts_run_rt<F, 2>(c, stream) : GGUF_NOT_TAKEN;
}

template <class F>
static int ts_run(const TsCall& c, hipStream_t stream) {
  if (!c.moe.sorted_token_ids) return ts_dense_run<F>(c, stream);
  if (c.rt != 1) return GGUF_NOT_TAKEN;
  return c.gate.rows ? ts_launch<F, 1, true, false, true>(c, 1, stream) : ts_run_rt<F, 1, true>(c, stream);
}

}  // namespace gguf
