// Products of some tens to some hundred rows of activations on 32 columns per workgroup, whose waves walk K on their own.
//
// What such a product loses is waiting: tiles of 128 rows leave most CUs with one wave per SIMD, a barrier per step of K lines the waves up behind the
// slowest fetch (mmq_i_core.h: 2.2 us a step, tile_wide_core.h: a chunk of X lasts less than its successor takes to come), and K cut between
// workgroups costs a launch and a way through memory for the parts.  Here
//   * a workgroup is 32 weight rows by 32 R rows of X, and its NW waves deal K among them, a panel of 256 values each in turn; no barrier stands
//     before the sum of their tiles, which is formed in LDS and stored;
//   * the panel's packed bytes come straight to the wave's own place in LDS (global_load_lds), are taken into registers and give the place to the next
//     panel; where LDS has room for two, the panel after the next is on its way;
//   * X lies in memory in the order in which the matrix unit takes it (tile_walk.h), 1 KB per block of 32 values and 32 rows, a fetch whose lanes follow
//     one another: eight of these are on their way to a ring in the wave's place.  The L2 hands out 30 TB/s of such pieces (registers or LDS, 130 bytes per ns
//     and CU), so that nothing is shared between the waves of a workgroup;
//   * one v_mfma_i32_32x32x32_i8 per block; the sum leaves the matrix unit as a float (the accumulator starts at the bits of 1.5 * 2^23, which stay in
//     sixteen registers of their own: as constants the compiler moves them into every result, 1.3 times as long) and costs two multiply-adds per result:
//     a lane holds one row of X, whose block scale is a register, and sixteen weight rows, whose block scales come from LDS once per block for all
//     R tiles.  The mins of the super-block formats are a contraction over the eight blocks in half precision, exact.  Q6_K, with a scale per 16 values, takes two
//     v_mfma_i32_32x32x16_i8 per block and twice the multiply-adds; Q3_K has its integer scales in the operand, which is still eight bits, and one scale per panel.
// Four waves and two workgroups per CU, or eight waves where the output has few columns; R = 1 .. 4, as the rows fill them (walk_us).
// Measured, us per call with the quantizer, before / now: [4096,4096] 64 rows Q4_K 16.1 / 10.8, Q8_0 19.4 / 12.6, 128 rows Q4_K 24.9 / 13.2; Q8_0 [14336,4096] 77
// rows 38.7 / 26.5 (its weights take 12.4 from memory), Q6_K [4096,4096] 64 rows 20.4 / 13.6, Q3_K [14336,4096] 512 rows 128 / 98.  Over random products (33 .. 2048
// rows) of the formats with a scale per 32 values 1.17 to 1.22 times the speed, of Q6_K 1.12, of Q3_K 1.26 (walk_plan).
// What bounds it: at few rows the beginning and the end of a workgroup (7 us of [4096,4096]'s 8 beside the quantizer); at many the vector instructions and the
// traffic through LDS, which do not overlap as they might: a block of 32 x 32 x 32 takes a SIMD 100 ns, where its matrix instruction and 32 multiply-adds take
// 58, the fetches of X and of weights 13 each, the operand reads 9.
// Tried and no faster: block scales from lane to lane (row_newbcast) instead of through LDS; each workgroup touching a share of X first, so that all find it in the L2.
// Arithmetic as in the other integer kernels (mmq.cuh:2-104: exact int32 block sums, scales in fp32); rel-L2 against 64 bits over 40 random products per format, normal
// activations, the kernels before / this: Q8_0 9.8e-8 / 7.7e-8, Q5_0 9.7 / 7.7, Q4_0 13.2 / 7.7, Q4_K 14.4 / 11.6, Q5_K 9.3 / 8.1, Q6_K 9.9 / 8.8, Q3_K 8.1 / 7.5; of one sign Q8_0 10.0 / 7.8, Q5_0 7.0 / 5.3,
// Q4_0 46 / 31, Q4_K 117 / 85, Q5_K 5.8 / 4.7, Q6_K 9.9 / 8.9, Q3_K 8.2 / 7.7: with one and two tiles of rows (Q6_K: and three, Q3_K always) a panel has a sum of its own.
#pragma once
#include "mmq_i_core.h"
#include "q8_1_device.h"
#include "tile_walk.h"
#include "tile_walk_formats.h"
#include <type_traits>
#include <utility>

namespace gguf {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float walk_f4 __attribute__((ext_vector_type(4)));

struct WalkArgs {
  int M, N, np, nkb;           // rows of X, weight rows, panels and blocks per row (the last panel may have fewer than eight)
  int row_tiles;               // tiles of 32 rows of X
  int tiles, run;              // workgroups that have work, and of them an XCD's
  int band, band_tiles, last_band;   // row blocks that are walked together, all their tiles, and the row blocks of the last ones
  uint32_t band_inv, all_inv, last_inv;   // 2^32 / (band, band_tiles, last_band) rounded up
  uint32_t w_pitch;
  int dtype, quads;            // GGUF_DTYPE_* of Y; rows of Y take stores of four values
  int64_t ldy;
  const void* bias;
};

// What the first requests are formed from comes as scalars in front (GGUF_GEOM, mmvq_core.h), the rest behind.
struct WalkEnd { int dtype, quads; int64_t ldy; const void* bias; };
#define GGUF_WALK_HEAD int h_tiles, uint32_t h_bands, int h_n, uint32_t h_pitch, int h_nkb, int h_m, uint32_t h_band_inv, uint32_t h_all_inv, uint32_t h_last_inv
#define GGUF_WALK_ARGS                                                                                                                                                     \
  WalkArgs{h_m, h_n, (h_nkb + 7) >> 3, h_nkb, (h_m + 31) >> 5, h_tiles, (h_tiles + 7) >> 3, (int)(h_bands & 0xFFFF), (int)(h_bands & 0xFFFF) * ((h_n + 31) >> 5),            \
           (int)(h_bands >> 16), h_band_inv, h_all_inv, h_last_inv, h_pitch, end.dtype, end.quads, end.ldy, end.bias}
// (a band's rows of X fit in 3 MB: less than 2^16 row blocks)
static inline uint32_t walk_inverse(int d) { return (uint32_t)((0x100000000ull + d - 1) / d); }
#define GGUF_WALK_HEAD_ARGS(b, n, pitch, k, m) \
  (b).tiles, (uint32_t)(b).band | (uint32_t)(b).last << 16, n, pitch, (k) / 32, m, walk_inverse((b).band), walk_inverse((b).band_tiles), walk_inverse((b).last)

template <int N> __device__ __forceinline__ void walk_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// wave-uniform 16-byte-per-lane fetch into LDS: lane l's bytes land at lds + AT + 16 l.  (The sum is formed here, by a scalar instruction: as an operand the
// compiler may have formed it in a vector register, with the addresses that the lanes read from.)
template <int AT> __device__ __forceinline__ void walk_fetch(uint32_t at, const void* base, uint32_t lds) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(at), "s"(base), "s"(lds), "n"(AT) : "memory", "scc");
}
// the same for lanes 0 .. 31 (all lanes are active before and after)
template <int AT> __device__ __forceinline__ void walk_fetch_half(uint32_t at, const void* base, uint32_t lds) {
  asm volatile("s_add_u32 m0, %2, %4\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(at), "s"(base), "s"(lds), "s"(0xFFFFFFFFull), "n"(AT)
               : "memory", "scc");
}
template <typename T>
__device__ __forceinline__ void walk_store(const walk_f4& v, T* y, const T* bias, int n, int N, int quads) {
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

__device__ __forceinline__ void walk_pin(float (&v)[16]) {   // the sixteen values are computed at this point
  asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
  asm volatile("" : "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]), "+v"(v[12]), "+v"(v[13]), "+v"(v[14]), "+v"(v[15]));
}

// A wave's place in LDS: D panels | PD tiles of X | block scales and sums of a panel's rows of X | scales for the lanes that hold results
constexpr int WALK_PD = 8;
template <class F> constexpr int walk_ppr() { return ((F::CUT ? F::PB + 29 : F::PB) / 16) | 1; }   // 16-byte pieces of a panel row (odd: banks)
template <class F> constexpr int64_t walk_row_bytes(int64_t K) { return F::KQ ? K / 256 * F::PB : K / 32 * (F::PB / 8); }
template <class F> constexpr int walk_head() { return F::OFF ? 1024 : 512; }
template <class F> constexpr int walk_scales() { return (F::WHOLE ? 128 : F::G == 16 ? 2048 : 1024) + (F::OFF == MINS ? 128 : 0); }
template <class F, int R, int D> constexpr int walk_place() { return 512 * walk_ppr<F>() * D + 1024 * WALK_PD + walk_head<F>() * R + walk_scales<F>(); }
template <class F, int R, int NW, int D> constexpr size_t walk_lds() {
  return (size_t)NW * walk_place<F, R, D>() + 16 > (size_t)NW * R * 4096 ? (size_t)NW * walk_place<F, R, D>() + 16 : (size_t)NW * R * 4096;
}
template <class F, int R, int NW> constexpr int walk_slots() { return walk_lds<F, R, NW, 2>() <= NW * 20 * 1024 ? 2 : 1; }

template <int U> struct WalkUnit { static constexpr int value = U; };
template <class L, int... U> __device__ __forceinline__ void walk_units(const L& unit, std::integer_sequence<int, U...>) { (unit(WalkUnit<U>()), ...); }

template <class F, int R, int NW, int D>
__global__ __launch_bounds__(64 * NW, 2) void tile_walk_kernel(const uint8_t* __restrict__ W, const char* __restrict__ X, GGUF_WALK_HEAD, void* __restrict__ Y, WalkEnd end) {
  const WalkArgs a = GGUF_WALK_ARGS;
  constexpr int PPR = walk_ppr<F>(), SLOT = 512 * PPR, NI = (32 * PPR + 63) / 64, PD = WALK_PD, GS = 32 / F::G, U = 8 * R * GS;   // (the last fetch of a panel: lanes 0 .. 31)
  constexpr int HEAD = walk_head<F>(), XR_AT = SLOT * D, HD_AT = XR_AT + 1024 * PD, SC_AT = HD_AT + HEAD * R, PLACE = walk_place<F, R, D>();
  constexpr bool PART = R <= (F::G == 16 ? 3 : 2) || F::WHOLE;                             // a panel's sum of its own, where the registers hold it
  constexpr int NL = NI + R;                                // fetches of a panel and of the heads of a panel's rows of X
  static_assert(PD == 8 && 8 * R % PD == 0, "the ring's places are the same in every panel; the waits below count to eight");
  static_assert(PPR % 2 == 1 && walk_lds<F, R, NW, D>() <= 160 * 1024, "the last fetch of a panel is half a fetch; LDS");
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // ---- which rows and columns.  Each XCD has a run of tiles, as long as another's; the row blocks of a band follow one another, so that they find
  // their weights in the L2, and a band is as tall as its rows of X fit there.
  const int local = blockIdx.x >> 3, tile = (blockIdx.x & 7) * a.run + local;
  if (local >= a.run || tile >= a.tiles) return;
  const int bnd = a.band_tiles == 1 ? tile : (int)__umulhi((uint32_t)tile, a.all_inv), in = tile - bnd * a.band_tiles;
  const bool last = (bnd + 1) * a.band_tiles >= a.tiles;    // (whose row blocks may be fewer)
  const int rows = last ? a.last_band : a.band, col = rows == 1 ? in : (int)__umulhi((uint32_t)in, last ? a.last_inv : a.band_inv);
  const int rb = bnd * a.band + in - col * rows, n0 = 32 * col;
  char* const mine = smem + wave * PLACE;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * PLACE;

  // ---- weights: piece number -> (row of the panel, 16-byte piece of it)
  const uint32_t wmis = F::CUT ? (uint32_t)((uintptr_t)W & 15) : 0u;
  const uint8_t* const wbase = W - wmis;
  const uint32_t row_bytes = F::KQ ? (uint32_t)(a.np * F::PB) : (uint32_t)(a.nkb * (F::PB / 8));
  const uint32_t last16 = ((uint32_t)(a.N - 1) * a.w_pitch + wmis + row_bytes - 1) & ~15u;   // the last granule that holds bytes of W
  int lane = tid & 63, lrow = lane & 31, half = lane >> 5;
  const auto w_from = [&](int i, int of) {                  // where row and piece of fetch i begin
    const int q = min(64 * i + of, 32 * PPR - 1), r = q / PPR;
    return make_uint2((uint32_t)min(n0 + r, a.N - 1) * a.w_pitch + wmis, 16 * (uint32_t)(q - r * PPR));
  };
  uint2 w_at[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) w_at[i] = w_from(i, lane);
  const char* xt[R];
#pragma unroll
  for (int k = 0; k < R; ++k) xt[k] = X + (int64_t)min(rb * R + k, a.row_tiles - 1) * a.np * WALK_REC;
  const auto request_w = [&](int p, int slot, auto safe) {
    const uint32_t to = lds0 + slot * SLOT;
    int of = lane;
    if (decltype(safe)::value) asm volatile("" : "+v"(of));   // (formed at each panel: the registers are short)
    walk_units([&](auto at) {
      constexpr int i = decltype(at)::value;
      const uint2 from = decltype(safe)::value ? w_from(i, of) : w_at[i];
      const uint32_t v = min(((from.x + (uint32_t)(p * F::PB)) & ~15u) + from.y, last16);
      if constexpr (i < NI - 1) walk_fetch<1024 * i>(v, wbase, to);
      else walk_fetch_half<1024 * i>(v, wbase, to);
    }, std::make_integer_sequence<int, NI>());
  };
  const auto request_heads = [&](int p) {
    walk_units([&](auto at) {
      constexpr int k = decltype(at)::value;
      const char* const base = xt[k] + (int64_t)p * WALK_REC + WALK_D_AT;
      if constexpr (F::OFF) walk_fetch<HD_AT + 1024 * k>(16 * lane, base, lds0);
      else walk_fetch_half<HD_AT + 512 * k>(16 * lane, base, lds0);
    }, std::make_integer_sequence<int, R>());
  };
  const auto request_x = [&](int p, auto at) {              // tile x of a panel
    constexpr int x = decltype(at)::value;
    walk_fetch<XR_AT + 1024 * (x % PD)>(16 * lane, xt[x % R] + ((int64_t)p * WALK_REC + 1024 * (x / R)), lds0);
  };

  float acc[R][16];
  v16i seed;
#pragma unroll
  for (int k = 0; k < R; ++k)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[k][r] = 0.0f;
  float* const scales = (float*)(mine + SC_AT);

  // (SAFE: as below, for activations whose block scale may be infinite)
  const auto panel = [&](int p, int slot, auto any, auto safe) {
    constexpr bool MORE = decltype(any)::value, SAFE = decltype(safe)::value;   // MORE: another panel follows
    constexpr int DB = (F::CUT && R >= 3) || SAFE ? 1 : 2;  // block scales in registers, of this block and, where these suffice, of the next
    // This panel, asked for one (D = 2: two) panels ago, and its heads; behind them the tiles under way.
    if (D == 2 && p == wave && MORE) walk_wait<PD + NI>();
    else walk_wait<PD>();
    F w;
    const uint32_t at = F::CUT ? ((uint32_t)min(n0 + lrow, a.N - 1) * a.w_pitch + wmis + (uint32_t)(p * F::PB)) & 15 : 0u;
    w.read(mine + slot * SLOT + lrow * (16 * PPR), at, half);
    uint4 dh[R], sh[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      dh[k] = *(const uint4*)(mine + HD_AT + HEAD * k + 16 * lrow);
      if (F::OFF) sh[k] = *(const uint4*)(mine + HD_AT + HEAD * k + 512 + 16 * lrow);
    }
    if (!F::KQ && a.nkb < 8 * (p + 1)) w.limit(a.nkb - 8 * p);
    w.scale_to(scales, lrow, half);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // the panel's place may be filled again
    const bool refill = D == 1 ? MORE : MORE && p + 2 * NW < a.np;
    if constexpr (MORE) request_heads(p + NW);
    if (refill) request_w(p + D * NW, slot, safe);
    // A unit is a block's group of values and a tile of rows, in the order (block, group, tile).  Tile x of the panel (block x / R, rows x % R) takes the place of tile
    // x - PD as soon as the last unit of that has its operand.  Here unit u, which needs tile x, makes sure that it has landed, before unit `now` has asked for
    // its tile: behind it were asked for all tiles up to that one's and, if it was asked for before this panel began, what was asked for then.
    const auto ready = [&](auto at, auto before) {
      constexpr int u = decltype(at)::value, now = decltype(before)::value, x = u / (R * GS) * R + u % R;
      constexpr int asked = PD + now / (R * GS) * R + (now / R % GS == GS - 1 ? now % R : 0), behind = (MORE || asked < 8 * R ? asked : 8 * R) - 1 - x;
      if constexpr (u / R % GS != 0) return;                // (its first group's unit has made sure)
      else if constexpr (!MORE || x >= PD) walk_wait<behind>();
      else if (refill) walk_wait<behind + NL>();
      else walk_wait<behind + R>();
    };
    float part[PART ? R : 1][16];
    typedef typename std::conditional<GS == 2, long, v4i>::type Codes;
    Codes xo[2], wo;
    v16i s[2];
    walk_f4 dw[DB][4];
    const auto load_x = [&](int u) {
      const int x = u / (R * GS) * R + u % R, g = u / R % GS;
      xo[u & 1] = *(const Codes*)(mine + XR_AT + 1024 * (x % PD) + 512 * g + (GS == 2 ? 8 : 16) * lane);
    };
    const auto load_dw = [&](int i) {                       // scale i of the panel's rows
#pragma unroll
      for (int q = 0; q < 4; ++q) dw[i % DB][q] = *(const walk_f4*)(scales + 32 * i + 8 * q + 4 * half);
    };
    const auto load_w = [&](int i) {
      if constexpr (GS == 2) wo = w.codes(i >> 1, i & 1);
      else wo = w.codes(i, half);
    };
    const auto mfma = [&](int u) {
      if constexpr (GS == 2) s[u & 1] = __builtin_amdgcn_mfma_i32_32x32x16_i8(wo, xo[u & 1], seed, 0, 0, 0);
      else s[u & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wo, xo[u & 1], seed, 0, 0, 0);
    };
    load_w(0);
    ready(WalkUnit<0>(), WalkUnit<0>());
    load_x(0);
    ready(WalkUnit<1>(), WalkUnit<0>());
    load_x(1);
    if (!F::WHOLE) load_dw(0);
    mfma(0);
    const auto unit = [&](auto at) {
      constexpr int u = decltype(at)::value, i = u / R, b = i / GS, k = u % R, x = b * R + k;   // i: the scale of the panel
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (u + 2 < U) {
        ready(WalkUnit<u + 2>(), at);
        load_x(u + 2);
      }
      if (!F::WHOLE && DB == 2 && k == 0 && u + R < U) load_dw(i + 1);
      if constexpr (i % GS == GS - 1) {                               // (the unit's operand has been read: its matrix instruction has started)
        if constexpr (x + PD < 8 * R) request_x(p, WalkUnit<x + PD>());
        else if constexpr (MORE) request_x(p + NW, WalkUnit<x + PD - 8 * R>());
      }
      if (u + 1 < U && k == R - 1) load_w(i + 1);
      const uint32_t dp = b < 2 ? dh[k].x : b < 4 ? dh[k].y : b < 6 ? dh[k].z : dh[k].w;
      float d8 = half_bits(b & 1 ? dp >> 16 : dp & 0xFFFF);
      asm volatile("" : "+v"(d8));                          // (a float from here on: the compiler would have every multiply-add convert it, in a form that takes twice as long)
      const float nd = -kSeed * d8;
      float (&sum)[16] = PART ? part[PART ? k : 0] : acc[k];
      const bool over = SAFE && GS == 2 && d8 == __builtin_inff();
      float m8 = 0.0f;
      if constexpr (F::OFF == EIGHTS) {
        const uint32_t sp = b < 2 ? sh[k].x : b < 4 ? sh[k].y : b < 6 ? sh[k].z : sh[k].w;
        m8 = -8.0f * half_bits(b & 1 ? sp >> 16 : sp & 0xFFFF);
        asm volatile("" : "+v"(m8));
      }
      if (u + 1 < U) mfma(u + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float bits = __builtin_bit_cast(float, (int)s[u & 1][r]);
        float v = SAFE ? (bits - kSeed) * d8 : __builtin_fmaf(bits, d8, nd);   // d8 times the block's sum, rounded once
        if constexpr (SAFE && (F::OFF == EIGHTS || F::WHOLE)) asm("" : "+v"(v));   // (a product that is rounded: not half of a multiply-add)
        if constexpr (F::OFF == EIGHTS) v += m8;
        if constexpr (SAFE && GS == 2) {                    // (the scale is taken times the sum of both groups, formed in the panel's)
          static_assert(PART, "a panel has a sum of its own");
          const float w8 = dw[i % DB][r >> 2][r & 3];
          float group = (bits - kSeed) * w8;                // (rounded: the two are then equal and opposite where the exact ones are)
          asm volatile("" : "+v"(group));
          const float both = sum[r] + group, finite = i == 0 ? v * w8 : __builtin_fmaf(v, w8, sum[r]);
          if constexpr (i % GS == 0) sum[r] = over ? group : finite;
          else {
            acc[k][r] = over ? __builtin_fmaf(both, d8, acc[k][r]) : acc[k][r];
            sum[r] = over ? 0.0f : finite;
          }
        } else if constexpr (F::WHOLE) sum[r] = i == 0 ? v : sum[r] + v;
        else sum[r] = PART && i == 0 ? v * dw[i % DB][r >> 2][r & 3] : __builtin_fmaf(v, dw[i % DB][r >> 2][r & 3], sum[r]);
      }
      // The offsets, a contraction over eight (the upper half of the lanes holds values 8 .. 15, zeros), in the middle of the panel
      if constexpr (F::OFF == MINS) if constexpr (b == 3) {
        const uint4 none = make_uint4(0, 0, 0, 0), mv = half ? none : w.offsets(), sv = half ? none : sh[k];
        f32x16 zero;
#pragma unroll
        for (int r = 0; r < 16; ++r) zero[r] = 0.0f;
        const f32x16 off = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, mv), __builtin_bit_cast(f16x8, sv), zero, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const walk_f4 dm = *(const walk_f4*)(scales + 256 + 8 * q + 4 * half);
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[4 * q + e] = __builtin_fmaf(off[4 * q + e], dm[e], sum[4 * q + e]);
        }
      }
      if constexpr (PART && u + R >= U) {
        if (F::WHOLE && k == 0) load_dw(0);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[k][r] = F::WHOLE ? __builtin_fmaf(sum[r], dw[0][r >> 2][r & 3], acc[k][r]) : acc[k][r] + sum[r];
      }
      walk_pin(PART && u + R >= U ? acc[k] : sum);
      if (!F::WHOLE && DB == 1 && k == R - 1 && u + 1 < U) load_dw(i + 1);
    };
    walk_units(unit, std::make_integer_sequence<int, U>());
  };
  const auto walk = [&](auto safe) {
    if (wave >= a.np) return;
    request_w(wave, 0, safe);
    request_heads(wave);
    if (D == 2 && wave + NW < a.np) request_w(wave + NW, 1, safe);
    walk_units([&](auto x) { request_x(wave, x); }, std::make_integer_sequence<int, PD>());
#pragma unroll
    for (int r = 0; r < 16; ++r) seed[r] = kSeedBits;
    asm volatile("" : "+v"(seed));                          // (opaque: as constants they are moved into every result's registers)
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[k][r] = 0.0f;
    int p = wave, slot = 0;
    for (; p + NW < a.np; p += NW) {
      panel(p, slot, std::true_type(), safe);
      if (D == 2) slot ^= 1;
    }
    panel(p, slot, std::false_type(), safe);
  };
  walk(std::false_type());
  // An activation past 8.3e6 has a block scale that a half does not hold: infinity, which the multiply-add takes from itself, so that none of the row's results is a number (one of
  // them tells; rows past the last one may be anything).  Its product with the sum is an infinity, of a sum of 0 no number, as in the other kernels: a wave that finds such a
  // row walks again with the seed taken off first.  The rows beside it get the same bits.  (The test is 0.1 us of 11; a product with such a row takes 1.2 to 1.55 times as long.)
  bool none = false;
#pragma unroll
  for (int k = 0; k < R; ++k) none |= __builtin_isnan(acc[k][0]) && 32 * (rb * R + k) + lrow < a.M;
  if (__any(none)) {
    asm volatile("" : "+v"(lane));                          // (what is formed from it is formed again: kept beside the first walk, it would go to scratch)
    lrow = lane & 31;
    half = lane >> 5;
    bool infinite = false;                                  // (else it is an activation or a weight that is no number, and stays that)
    for (int p = wave; p < a.np; p += NW)
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const uint4 d = *(const uint4*)(xt[k] + ((int64_t)p * WALK_REC + WALK_D_AT) + 16 * lrow);
        const auto inf = [](uint32_t two) { return (two & 0xFFFFu) == 0x7C00u || two >> 16 == 0x7C00u; };
        infinite |= (inf(d.x) | inf(d.y) | inf(d.z) | inf(d.w)) && 32 * (rb * R + k) + lrow < a.M;
      }
    if (__any(infinite)) walk(std::true_type());
  }

  // ---- the waves' partial tiles, added in pairs
  __syncthreads();
  walk_f4* const red = (walk_f4*)smem;                      // [wave][tile][run of four and half][row ^ that]
#pragma unroll
  for (int k = 0; k < R; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q) red[((wave * R + k) * 8 + 2 * q + half) * 32 + (lrow ^ (2 * q + half))] = (walk_f4){acc[k][4 * q], acc[k][4 * q + 1], acc[k][4 * q + 2], acc[k][4 * q + 3]};
  __syncthreads();
  for (int i = 64 * wave + lane; i < R * 256; i += 64 * NW) {
    const int q = i & 7, row = (i >> 3) & 31, k = i >> 8, m = 32 * (rb * R + k) + row;
    walk_f4 v[NW];
#pragma unroll
    for (int z = 0; z < NW; ++z) v[z] = red[((z * R + k) * 8 + q) * 32 + (row ^ q)];
#pragma unroll
    for (int d = 1; d < NW; d *= 2)
#pragma unroll
      for (int z = 0; z < NW; z += 2 * d) v[z] += v[z + d];
    if (m < a.M) {
      if (a.dtype == GGUF_DTYPE_F16) walk_store<_Float16>(v[0], (_Float16*)Y + (int64_t)m * a.ldy, (const _Float16*)a.bias, n0 + 4 * q, a.N, a.quads);
      else if (a.dtype == GGUF_DTYPE_BF16) walk_store<bf16_t>(v[0], (bf16_t*)Y + (int64_t)m * a.ldy, (const bf16_t*)a.bias, n0 + 4 * q, a.N, a.quads);
      else walk_store<float>(v[0], (float*)Y + (int64_t)m * a.ldy, (const float*)a.bias, n0 + 4 * q, a.N, a.quads);
    }
  }
}

template <class F, int R, int NW>
static int walk_launch(const WalkCall& c, hipStream_t stream) {
  constexpr int D = walk_slots<F, R, NW>();
  constexpr size_t lds = walk_lds<F, R, NW, D>();
  const WalkBands bands = walk_bands(R, c.M, c.N, c.K);
  if (!bands.ok) return GGUF_NOT_TAKEN;
  auto kern = tile_walk_kernel<F, R, NW, D>;
  static std::atomic<uint64_t> done{0};
  allow_large_lds(kern, lds, done);
  const int64_t pitch = c.la.w_pitch ? c.la.w_pitch : walk_row_bytes<F>(c.K), ldy = c.la.ldy ? c.la.ldy : (int64_t)c.N;
  const int run = (bands.tiles + 7) / 8, elt = c.dtype == GGUF_DTYPE_F32 ? 4 : 2;
  const WalkEnd end = {c.dtype, ldy % 4 == 0 && (uintptr_t)c.Y % (4 * elt) == 0, ldy, c.la.bias};
  hipLaunchKernelGGL(kern, dim3((unsigned)(8 * run)), dim3(64 * NW), lds, stream, (const uint8_t*)c.W, (const char*)c.x,
                     GGUF_WALK_HEAD_ARGS(bands, c.N, (uint32_t)pitch, c.K, c.M), c.Y, end);
  return launch_status();
}

template <class F>
static int walk_run(const WalkCall& c, hipStream_t s) {
  switch (c.plan.rt * 16 + c.plan.nw) {
    case 1 * 16 + 4: return walk_launch<F, 1, 4>(c, s);
    case 1 * 16 + 8: return walk_launch<F, 1, 8>(c, s);
    case 2 * 16 + 4: return walk_launch<F, 2, 4>(c, s);
    case 2 * 16 + 8: return walk_launch<F, 2, 8>(c, s);
    case 3 * 16 + 4:
      if constexpr (F::TALL >= 3) return walk_launch<F, 3, 4>(c, s);   // (else there is no such plan)
      break;
    case 4 * 16 + 4:
      if constexpr (F::TALL >= 4) return walk_launch<F, 4, 4>(c, s);
  }
  return GGUF_NOT_TAKEN;
}
// A: the panels that begin on whole 16-byte pieces
template <class A, class F>
static int walk_run_either(const WalkCall& c, hipStream_t s) {
  const int64_t pitch = c.la.w_pitch ? c.la.w_pitch : walk_row_bytes<A>(c.K);
  return (uintptr_t)c.W % 16 == 0 && pitch % 16 == 0 ? walk_run<A>(c, s) : walk_run<F>(c, s);
}

}  // namespace gguf
