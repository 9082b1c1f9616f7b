// The expert products of MoE layers whose experts see more than a few pairs each: Q4_0, Q8_0, Q4_K, Q5_K on the int8 matrix unit, 32
// slots by 128 columns per workgroup.  (Q6_K has sixteen scales a super-block: tile_wide_core.h.)
//
// What bounds it is vector issue: on a SIMD the matrix unit and everything else take turns for the most part, so that a panel costs the sum of its
// multiplications, its decoding and its multiply-adds.  Hence
//   * codes go to the matrix unit as the bytes they are (walk formats, tile_walk_formats.h), not as half-precision operands: a third of the decoding, and
//     one instruction for 32 values where two were needed;
//   * the unit's accumulators start as the bits of 1.5 * 2^23, so that what comes out IS a float (walk kernels' seed), and a
//     multiply-add by the row's block scale takes the seed off; the weights' scales come from LDS, four rows at a time;
//   * a wave fetches and decodes its own 32 weight rows, a panel of 256 values ahead (global_load_lds); records of X (tile_expert.h) are shared,
//     two buffers and a barrier per 128 values; three workgroups per CU;
//   * where the upper sixteen slots of a block hold no pair -- about every second expert's last block -- tiles of 16 x 16: half the matrix time
//     and half the multiply-adds, the same bits (a pair's result does not depend on how many share its block).
// Measured, us per layer, half-precision tiles / these: Q4_K 128 experts 300 tokens 137 / 121, Q5_K 178 / 156, Q4_0 64 experts 200 tokens 115 / 98, Q8_0 122 /
// 109, Q4_0 128 experts 120 tokens 119 / 99, Q4_K 8 experts 95 / 82; Q4_K with Q6_K, 128 experts, top-8,
// H 2048, I 768, 300 tokens 153 to 162 / 142 to 150 (floor 82); 300 layers of random sizes, 65 to 1500 tokens, by the rule of wide_layer_takes (tile_wide.hip): 1.106 on
// average, the slowest 0.994.
// Error against 64 bits over K 512 .. 8192 (rms, second product; normal / one-sign activations; half-precision tiles, then these, in 1e-8): Q4_0
// 13.6 / 8.0, 8.2 / 5.0; Q8_0 11.2 / 12.1, 7.9 / 8.1; Q4_K 9.9 / 18.4, 8.5 / 10.4; Q5_K 9.8 / 18.1, 8.8 / 10.6.
// Tried and slower: two sets of weight scales in registers, the next block's under way (120 to 133 us, 156 to 237: they spill).
// Arithmetic as in the other integer kernels (mmq.cuh:2-104, moe.cuh:5-129): exact block sums, scales in fp32.
#pragma once
#include "layer_seam.h"
#include "mmq_i_core.h"
#include "tile_expert.h"
#include "tile_walk_formats.h"
#include <type_traits>

namespace gguf {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float expert_f4 __attribute__((ext_vector_type(4)));

constexpr int EXPERT_NW = 4, EXPERT_N = 32 * EXPERT_NW, EXPERT_M = 32;

struct ExpertArgs {
  int N, np;                   // weight rows; panels of 256 values per row
  int col_wgs;                 // workgroups side by side
  uint32_t w_pitch, x_plane;   // bytes between weight rows; between the records of neighbouring panels of a row of X
  uint32_t topk_inv;           // 2^32 / top_k rounded up
  int dtype, quads;            // GGUF_DTYPE_* of Y; rows of Y take stores of four values
  int ksplit;                  // workgroups that share a sum over K: fp32 sums [ksplit][pairs][N]
  int64_t split_stride;        // (values between them)
};

template <int N> __device__ __forceinline__ void expert_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// wave-uniform 16-byte-per-lane fetch into LDS: lane l's bytes land at m0 + 16 l
__device__ __forceinline__ void expert_fetch(uint32_t at, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(at), "s"(base), "s"(lds) : "memory");
}
// the same for lanes 0 .. 31 (all lanes are active before and after)
__device__ __forceinline__ void expert_fetch_half(uint32_t at, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(at), "s"(base), "s"(lds), "s"(0xFFFFFFFFull) : "memory");
}
// four bytes a lane
__device__ __forceinline__ void expert_fetch_words(uint32_t at, const void* base, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(at), "s"(base), "s"(lds) : "memory");
}
template <typename T>
__device__ __forceinline__ void expert_store(const expert_f4& v, T* y, int n, int N, int quads) {
  if (quads && n + 3 < N) {
    struct alignas(4 * sizeof(T)) { T v[4]; } o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o.v[e] = from_f32<T>(v[e]);
    *(decltype(o)*)(y + n) = o;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) y[n + e] = from_f32<T>(v[e]);
  }
}
__device__ __forceinline__ void expert_store(const expert_f4& v, int64_t row, int n, void* Y, const ExpertArgs& a) {
  if (a.dtype == GGUF_DTYPE_F16) expert_store<_Float16>(v, (_Float16*)Y + row * a.N, n, a.N, a.quads);
  else if (a.dtype == GGUF_DTYPE_BF16) expert_store<bf16_t>(v, (bf16_t*)Y + row * a.N, n, a.N, a.quads);
  else expert_store<float>(v, (float*)Y + row * a.N, n, a.N, a.quads);
}
template <int N> __device__ __forceinline__ void expert_pin(float (&v)[N]) {   // the values are computed at this point
#pragma unroll
  for (int i = 0; i < N; i += 8)
    asm volatile("" : "+v"(v[i]), "+v"(v[i + 1]), "+v"(v[i + 2]), "+v"(v[i + 3]), "+v"(v[i + 4]), "+v"(v[i + 5]), "+v"(v[i + 6]), "+v"(v[i + 7]));
}

// LDS: two buffers of records | a panel per wave | a wave's scales for the lanes that hold results | the slots' pairs | a word per wave
template <class F> constexpr int expert_ppr() { return (F::PB / 16) | 1; }   // 16-byte pieces of a panel row (odd: banks)
constexpr int EXPERT_XBUF = (EXPERT_M * (EXPERT_REC / 16) + 63) / 64 * 1024;
template <class F> constexpr int expert_scales() { return 1024 + (F::OFF == MINS ? 128 : 0); }
template <class F> constexpr size_t expert_lds() {
  return 2 * EXPERT_XBUF + (size_t)EXPERT_NW * (512 * expert_ppr<F>() + expert_scales<F>() + 256) + 16 * EXPERT_NW + 16;
}

// GATE: the first expert GEMM of a layer with its seam (Gate16): a wave's 32 weight rows are 16 features of the gate half and the
// same of the up half, so that a lane has both sums of eight features; two waves finish a q8_1 block of h together.
template <class F, bool GATE>
__global__ __launch_bounds__(64 * EXPERT_NW, 3) void tile_expert_kernel(const uint8_t* __restrict__ W, const char* __restrict__ X, void* __restrict__ Y,
                                                                        ExpertArgs a, MoeArgs moe, Gate16 gate) {
  constexpr int PPR = expert_ppr<F>(), SLOT = 512 * PPR, NI = (32 * PPR + 63) / 64;   // (the last fetch: lanes 0 .. 31)
  constexpr int XB = EXPERT_XBUF, RING_AT = 2 * XB, SC_AT = RING_AT + EXPERT_NW * SLOT, ID_AT = SC_AT + EXPERT_NW * expert_scales<F>(), FLAG_AT = ID_AT + 256 * EXPERT_NW;
  constexpr int XP = EXPERT_REC / 16, XI = (EXPERT_M * XP + 63) / 64, XW = (XI + EXPERT_NW - 1) / EXPERT_NW;   // pieces of a record; fetches of a buffer; a wave's, at most
  static_assert(F::G == 32 && !F::WHOLE && !F::CUT && F::PB % 16 == 0, "a scale per block; panels are whole 16-byte pieces");
  static_assert(PPR % 2 == 1 && expert_lds<F>() <= 53 * 1024, "the last fetch of a panel is half a fetch; three workgroups fit in LDS");
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lrow = lane & 31, half = lane >> 5;                   // weights, and results of 32 rows of X
  int c = lane & 15, g = lane >> 4;                         // results of 16

  // ---- which rows and columns.  Tiles are numbered along the columns of a row block, and the workgroups go to the XCDs in turn: with
  // a multiple of eight columns the blocks of an expert find its weights in one L2, and the blocks past the last live one, of
  // which nothing is done, are spread over all XCDs.
  const int tile = (int)blockIdx.x;
  const int block = tile / a.col_wgs, col_wg = tile - block * a.col_wgs;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const int ids_at = ID_AT + wave * 256;
  const int live = moe.num_tokens_post_padded[0], e = moe.expert_ids[block];
  const int p0 = a.ksplit > 1 ? a.np * (int)blockIdx.y / a.ksplit : 0, p1 = a.ksplit > 1 ? a.np * ((int)blockIdx.y + 1) / a.ksplit : a.np;

  // ---- fetching weights: piece number -> (row of the panel, 16-byte piece of it)
  const int rows_all = GATE ? 2 * gate.inner : a.N;
  const int n0 = GATE ? 64 * col_wg + 16 * wave : EXPERT_N * col_wg + 32 * wave;   // this wave's first weight row (feature)
  const auto row_of = [&](int r) { return GATE ? (r < 16 ? min(n0 + r, gate.inner - 1) : gate.inner + min(n0 + r - 16, gate.inner - 1)) : min(n0 + r, a.N - 1); };
  const uint32_t last16 = ((uint32_t)(rows_all - 1) * a.w_pitch + (uint32_t)(a.np * F::PB) - 1) & ~15u;   // the last 16-byte piece of an expert's matrix
  const auto w_from = [&](int i, int of) {                  // where the bytes of fetch i begin
    const int q = min(64 * i + of, 32 * PPR - 1), r = q / PPR;
    return (uint32_t)row_of(r) * a.w_pitch + 16 * (uint32_t)(q - r * PPR);
  };
  uint32_t w_at[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) w_at[i] = w_from(i, lane);
  if (block * EXPERT_M >= live || e < 0 || e > 255) return; // (experts above 255: the reference's guard, moe.cuh:33)
  W += (int64_t)e * moe.expert_stride;
  expert_fetch_words(4 * min(lane, EXPERT_M - 1), moe.sorted_token_ids + block * EXPERT_M, lds0 + ids_at);
  const auto request = [&](int p, auto safe) {
    int of = lane;
    if (decltype(safe)::value) asm volatile("" : "+v"(of)); // (formed at each panel: the registers are short)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const uint32_t v = min((decltype(safe)::value ? w_from(i, of) : w_at[i]) + (uint32_t)(p * F::PB), last16);
      const uint32_t to = lds0 + RING_AT + wave * SLOT + 1024 * i;
      if (i < NI - 1) expert_fetch(v, W, to);
      else expert_fetch_half(v, W, to);   // (lanes past the panel's last piece stay out: their bytes would land in the next slot)
    }
  };
  request(p0, std::false_type());

  // ---- fetching records: a wave's fetches of a buffer, pieces 64 i .. of it for i = wave, wave + 4, ...
  uint32_t x_at[XW];
  expert_wait<NI>();                                        // (the slots' pairs are here)
#pragma unroll
  for (int j = 0; j < XW; ++j) {
    const int q = min(64 * (wave + EXPERT_NW * j) + lane, EXPERT_M * XP - 1), r = q / XP, id = *(const int*)(smem + ids_at + 4 * r);
    const int row = id < moe.num_pairs ? (moe.top_k == 1 ? id : (int)__umulhi((uint32_t)id, a.topk_inv)) : 0;   // row 0 stands in for padding
    x_at[j] = (uint32_t)row * EXPERT_REC + 16 * (uint32_t)(q - r * XP);
  }
  const auto fetch_x = [&](int ch) {                        // chunk ch: 128 values
    const char* const base = X + (uint64_t)(uint32_t)ch * a.x_plane;
#pragma unroll
    for (int j = 0; j < XW; ++j)
      if (wave + EXPERT_NW * j < XI) expert_fetch(x_at[j], base, lds0 + (ch & 1) * XB + 1024 * (wave + EXPERT_NW * j));
  };
  fetch_x(2 * p0);

  float acc[16];
  v16i seed;
#pragma unroll
  for (int r = 0; r < 16; ++r) seed[r] = kSeedBits;
  asm volatile("" : "+v"(seed));                            // (opaque: as constants they are moved into every result's registers)
  float* const scales = (float*)(smem + SC_AT + wave * expert_scales<F>());

  // A lane has one row of X and, of 32 rows, weight rows 8 q + 4 half + e (q = 0 .. 3), of 16 rows (SMALL) weight rows 16 i + 4 g + e (i = 0, 1).  SAFE: as
  // below, for activations whose block scale may be infinite.
  const auto walk = [&](auto safe, auto small) {
    constexpr bool SAFE = decltype(safe)::value, SMALL = decltype(small)::value;
    constexpr int Q = SMALL ? 2 : 4;                        // runs of four results
    const int xr = SMALL ? c : lrow, first = SMALL ? 4 * g : 4 * half;
    constexpr int RUN = SMALL ? 16 : 8;                     // weight rows between the runs
#pragma unroll
    for (int r = 0; r < 4 * Q; ++r) acc[r] = 0.0f;
    for (int p = p0; p < p1; ++p) {
      F w;
      uint2 sums[2];
      float part[4 * Q];
      typedef typename std::conditional<SMALL, long, v4i>::type Codes;
      typedef typename std::conditional<SMALL, v4i, v16i>::type Sums;
      typedef typename std::conditional<SMALL, expert_f4, f32x16>::type Offsets;
      Sums start;
#pragma unroll
      for (int r = 0; r < (SMALL ? 4 : 16); ++r) start[r] = seed[r];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        // This chunk's records have landed, and with hh = 0 the panel; what was asked for behind them are the next panel's weights.
        if (hh == 1 && p + 1 < p1) expert_wait<NI>();
        else expert_wait<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (and this wave has read the last of the chunk before)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (hh == 0 || p + 1 < p1) fetch_x(2 * p + hh + 1);
        if (hh == 0) {
          w.read(smem + RING_AT + wave * SLOT + lrow * (16 * PPR), 0u, half);
          w.scale_to(scales, lrow, half);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the panel's place may be filled again
          if (p + 1 < p1) request(p + 1, safe);
        }
        const char* const xrow = smem + hh * XB + xr * EXPERT_REC;
        const uint4 head = *(const uint4*)(xrow + EXPERT_D_AT);
        sums[hh] = make_uint2(head.z, head.w);
        Codes xo[2], wo[SMALL ? 2 : 1];
        Sums s[2][SMALL ? 2 : 1];
        expert_f4 dw[Q];
        const auto load_x = [&](int b) { xo[b & 1] = *(const Codes*)(xrow + 32 * b + (SMALL ? 8 * g : 16 * half)); };
        const auto load_dw = [&](int b) {
#pragma unroll
          for (int q = 0; q < Q; ++q) dw[q] = *(const expert_f4*)(scales + 32 * (4 * hh + b) + RUN * q + first);
        };
        const auto load_w = [&](int b) {
          const v4i o = w.codes(4 * hh + b, half);
          if constexpr (SMALL) {
            // Of the lane's sixteen values of one of 32 rows the second eight of lanes 0 .. 15 and 32 .. 47 change places with the first eight of the
            // lanes behind them: then the two halves are the values of 16 rows each.
            const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)o[0], (uint32_t)o[2], false, false), hi = __builtin_amdgcn_permlane16_swap((uint32_t)o[1], (uint32_t)o[3], false, false);
            const uint32_t l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
            wo[0] = (long)((uint64_t)h0 << 32 | l0);
            wo[1] = (long)((uint64_t)h1 << 32 | l1);
          } else {
            wo[0] = o;
          }
        };
        const auto mfma = [&](int b) {
          if constexpr (SMALL) {
#pragma unroll
            for (int i = 0; i < 2; ++i) s[b & 1][i] = __builtin_amdgcn_mfma_i32_16x16x32_i8(wo[i], xo[b & 1], start, 0, 0, 0);
          } else {
            s[b & 1][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wo[0], xo[b & 1], start, 0, 0, 0);
          }
        };
        // The offsets, a contraction over eight (of 32 rows the upper half of the lanes holds values 8 .. 15, zeros; of 16 lanes 16 i .. 16 i + 15
        // hold the mins of weight rows 16 i .., the others meet zeros).  Halfway: with activations of one sign the sum then runs from 0 up to half of the
        // products', to minus that, and back, and is rounded at half the size
        Offsets off[SMALL ? 2 : 1];
        if constexpr (F::OFF == MINS) if (hh == 1) {
          const uint4 none = make_uint4(0, 0, 0, 0), sv = make_uint4(sums[0].x, sums[0].y, sums[1].x, sums[1].y);
          const f16x8 mv = __builtin_bit_cast(f16x8, half ? none : w.offsets());
          Offsets zero;
#pragma unroll
          for (int r = 0; r < (SMALL ? 4 : 16); ++r) zero[r] = 0.0f;
          if constexpr (SMALL) {
#pragma unroll
            for (int i = 0; i < 2; ++i) off[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(mv, __builtin_bit_cast(f16x8, g == i ? sv : none), zero, 0, 0, 0);
          } else {
            off[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(mv, __builtin_bit_cast(f16x8, half ? none : sv), zero, 0, 0, 0);
          }
        }
        load_w(0);
        load_x(0);
        load_x(1);
        load_dw(0);
        mfma(0);
        if constexpr (F::OFF == MINS) if (hh == 1) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            const expert_f4 dm = *(const expert_f4*)(scales + 256 + RUN * q + first);
#pragma unroll
            for (int e = 0; e < 4; ++e) part[4 * q + e] = __builtin_fmaf(off[SMALL ? q : 0][SMALL ? e : 4 * q + e], dm[e], part[4 * q + e]);
          }
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          __builtin_amdgcn_sched_barrier(0);
          if (b + 2 < 4) load_x(b + 2);
          if (b + 1 < 4) load_w(b + 1);
          const uint32_t dp = b < 2 ? head.x : head.y;
          float d8 = half_bits(b & 1 ? dp >> 16 : dp & 0xFFFF);
          asm volatile("" : "+v"(d8));                      // (a float from here on: the compiler would have every multiply-add convert it, in a form that takes twice as long)
          const float nd = -kSeed * d8;
          float m8 = 0.0f;
          if constexpr (F::OFF == EIGHTS) {
            const uint32_t sp = b < 2 ? head.z : head.w;
            m8 = -8.0f * half_bits(b & 1 ? sp >> 16 : sp & 0xFFFF);
            asm volatile("" : "+v"(m8));
          }
          if (b + 1 < 4) mfma(b + 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int r = 0; r < 4 * Q; ++r) {
            const int of = SMALL ? s[b & 1][SMALL ? r >> 2 : 0][r & 3] : s[b & 1][0][SMALL ? 0 : r];
            const float bits = __builtin_bit_cast(float, of), w8 = dw[r >> 2][r & 3];
            float v = SAFE ? (bits - kSeed) * d8 : __builtin_fmaf(bits, d8, nd);   // d8 times the sum, rounded once
            if constexpr (SAFE && F::OFF == EIGHTS) asm("" : "+v"(v));   // (a product that is rounded: not half of a multiply-add)
            if constexpr (F::OFF == EIGHTS) v += m8;
            part[r] = hh == 0 && b == 0 ? v * w8 : __builtin_fmaf(v, w8, part[r]);
          }
          expert_pin(part);
          if (b + 1 < 4) load_dw(b + 1);
        }
      }
#pragma unroll
      for (int r = 0; r < 4 * Q; ++r) acc[r] += part[r];
    }
  };
  const auto run = [&](auto small) {
    constexpr bool SMALL = decltype(small)::value;
    walk(std::false_type(), small);
    // An activation past 8.3e6 has a block scale that a half does not hold: infinity, which the multiply-add takes from itself, so that none of the row's results is
    // a number (one of them tells).  Its product with the sum is an infinity, of a sum of 0 no number: where a row has none, the waves look through the records that they
    // fetch, and if a block scale is infinite, all four walk again with the seed taken off first (else it is an activation or a weight that is no number, and
    // stays that).  The rows beside it get the same bits.
    {
      const bool none = __any(__builtin_isnan(acc[0]) && *(const int*)(smem + ids_at + 4 * (SMALL ? c : lrow)) < moe.num_pairs);
      if (lane == 0) *(int*)(smem + FLAG_AT + 4 * wave) = none;
      __syncthreads();
      const auto flagged = [&] {
        const int4 flags = *(const int4*)(smem + FLAG_AT);
        return (flags.x | flags.y | flags.z | flags.w) != 0;
      };
      if (flagged()) {
        int l = tid & 63;
        asm volatile("" : "+v"(l));                           // (what is formed from it is formed again: kept beside the first walk, it would go to scratch)
        bool infinite = false;                                // (from the addresses of the fetches: nothing more is held over the walk)
        for (int ch = 2 * p0; ch < 2 * p1; ++ch)
#pragma unroll
          for (int j = 0; j < XW; ++j) {
            const int q = 64 * (wave + EXPERT_NW * j) + l;
            if (q >= EXPERT_M * XP || q % XP != EXPERT_D_AT / 16) continue;   // (the piece of a record that begins with its scales)
            const uint2 d = *(const uint2*)(X + (uint64_t)(uint32_t)ch * a.x_plane + x_at[j]);
            const auto inf = [](uint32_t two) { return (two & 0xFFFFu) == 0x7C00u || two >> 16 == 0x7C00u; };
            infinite |= inf(d.x) | inf(d.y);
          }
        infinite = __any(infinite);
        __syncthreads();                                      // (the first flags have been read)
        if (l == 0) *(int*)(smem + FLAG_AT + 4 * wave) = infinite;
        __syncthreads();
        lrow = l & 31; half = l >> 5; c = l & 15; g = l >> 4;
        if (flagged()) {
          request(p0, std::true_type());
          fetch_x(2 * p0);
          walk(std::true_type(), small);
        }
      }
    }

    // ---- results
    const int pair = *(const int*)(smem + ids_at + 4 * (SMALL ? c : lrow));
    if constexpr (GATE) {
      // h of eight features of the wave's sixteen, 8 q + 4 half + e, or of four, 4 g + e: weight rows 0 .. 15 are the gate's, 16 .. 31 the up half's
      constexpr int H = SMALL ? 4 : 8;
      float h[H];
  #pragma unroll
      for (int i = 0; i < H; ++i) {
        const float gv = seam_rounded(acc[i], a.dtype), uv = seam_rounded(acc[H + i], a.dtype);
        h[i] = seam_gate(gv, uv, gate.act, a.dtype);
      }
      // The q8_1 block has 32 features: the other sixteen are the next wave's (the last one's).  amax and the sum as q8_1_quantize8
      // forms them, by a butterfly over 16 (the other wave), 8, 4 (the lane's other run, other lanes), 2, 1.
      __syncthreads();                                        // (the values go over the records)
      expert_f4* const mine = (expert_f4*)smem + (wave * (H / 4)) * 64 + lane;
      const expert_f4* const other = (const expert_f4*)smem + ((wave ^ 1) * (H / 4)) * 64 + lane;
  #pragma unroll
      for (int q = 0; q < H / 4; ++q) mine[q * 64] = (expert_f4){h[4 * q], h[4 * q + 1], h[4 * q + 2], h[4 * q + 3]};
      __syncthreads();
      if (n0 >= gate.inner) return;
      expert_f4 o[H / 4];
      float amax = 0.0f, t[4];
  #pragma unroll
      for (int q = 0; q < H / 4; ++q) o[q] = other[q * 64];
  #pragma unroll
      for (int i = 0; i < 4; ++i) {
  #pragma unroll
        for (int q = 0; q < H / 4; ++q) amax = fmaxf(fmaxf(amax, fabsf(h[4 * q + i])), fabsf(o[q][i]));
        t[i] = h[i] + o[0][i];
        if constexpr (SMALL) t[i] += __shfl_xor(t[i], 32);
        else t[i] += h[4 + i] + o[1][i];
        t[i] += __shfl_xor(t[i], SMALL ? 16 : 32);
      }
      amax = fmaxf(amax, __shfl_xor(amax, 32));
      if constexpr (SMALL) amax = fmaxf(amax, __shfl_xor(amax, 16));
      const float sum = (t[0] + t[2]) + (t[1] + t[3]), d = amax / 127.0f;
      float q[H];
      seam_quants(h, d, amax == 0.0f, q);
      if (pair < moe.num_pairs) {
        char* const rec = seam_h_record(gate, n0, pair, moe.num_pairs);
        const int blk = (n0 >> 5) & 3, at = n0 & 16;
  #pragma unroll
        for (int i = 0; i < H / 4; ++i) seam_h_store(rec, gate, blk, at + (SMALL ? 4 * g : 8 * i + 4 * half), q + 4 * i);
        if ((SMALL ? g : half) == 0 && at == 0) seam_h_scales(rec, gate, blk, d, sum);
      }
    } else {
      if (a.ksplit > 1) Y = (float*)Y + (int64_t)blockIdx.y * a.split_stride;
      if (pair < moe.num_pairs)
  #pragma unroll
        for (int q = 0; q < (SMALL ? 2 : 4); ++q)
          expert_store((expert_f4){acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]}, pair, n0 + (SMALL ? 16 * q + 4 * g : 8 * q + 4 * half), Y, a);
    }
  };
  // (the pairs of a block come first, padding behind them)
  const bool upper = __ballot(*(const int*)(smem + ids_at + 4 * lrow) < moe.num_pairs) >> 16 & 0xFFFFu;
  if (upper) run(std::false_type());
  else run(std::true_type());
}

template <class F, bool GATE>
static int expert_launch(const ExpertCall& c, hipStream_t stream) {
  constexpr size_t lds = expert_lds<F>();
  const int qk = F::KQ ? 256 : 32, bs = F::KQ ? F::PB : F::PB / 8;
  const int64_t pitch = (int64_t)(c.K / qk) * bs;
  if (pitch % 16 != 0 || (uintptr_t)c.W % 16 != 0 || c.moe.expert_stride % 16 != 0) return GGUF_NOT_TAKEN;
  auto kern = tile_expert_kernel<F, GATE>;
  static std::atomic<uint64_t> done{0};
  allow_large_lds(kern, lds, done);
  const int cols = GATE ? (c.gate.inner + 63) / 64 : (c.N + EXPERT_N - 1) / EXPERT_N, top_k = c.moe.top_k > 0 ? c.moe.top_k : 1;
  const bool split = c.ksplit > 1;
  const int dtype = split ? GGUF_DTYPE_F32 : c.dtype, elt = dtype == GGUF_DTYPE_F32 ? 4 : 2;
  void* const y = split ? (void*)c.partial : c.Y;
  const ExpertArgs a = {c.N, c.K / 256, cols, (uint32_t)pitch, (uint32_t)(c.x_rows * EXPERT_REC), (uint32_t)((0x100000000ull + top_k - 1) / top_k),
                        dtype, c.N % 4 == 0 && (uintptr_t)y % (4 * elt) == 0, split ? c.ksplit : 1, (int64_t)c.moe.num_pairs * c.N};
  hipLaunchKernelGGL(kern, dim3((unsigned)((int64_t)c.row_blocks * cols), (unsigned)a.ksplit), dim3(64 * EXPERT_NW), lds, stream, (const uint8_t*)c.W, (const char*)c.x,
                     y, a, c.moe, c.gate);
  return launch_status();
}

template <class F>
static int expert_run(const ExpertCall& c, hipStream_t s) {
  if (!c.moe.sorted_token_ids || c.K % 256 != 0) return GGUF_NOT_TAKEN;
  return c.gate.rows ? expert_launch<F, true>(c, s) : expert_launch<F, false>(c, s);
}

}  // namespace gguf
