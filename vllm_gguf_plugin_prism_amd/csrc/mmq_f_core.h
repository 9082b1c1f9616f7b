// Prefill GEMM on the super-block formats: integer arithmetic on the half-precision matrix unit.
//
//   Y[m, n] = sum_sb  d[n, sb] * ( sum_b  d8[m, b] * S[m, n, b] )  ( - dmin[n, sb] * sum_b  mn[n, b] * s8[m, b] )
//   S[m, n, b] = sum over the 32 values of block b of  q8[m, k] * (sc[n, group of k] * q[n, k])         (exact)
//
// What bounds the contraction is the vector work per matrix result: a q8_1 block is 32 values deep and every result of a
// block has to be scaled before the next one is added.  With the weight's own scale in that factor (mmq_i_core.h: int8
// operands, d8 * d * sc per block) that is two or three multiply-adds per result and block, four where a weight scale
// covers 16 values: 41 to 90 ns per 32 x 32 x 32 block and SIMD at full rate, of which the matrix unit needs 14.  Here the
// integer scale sc goes into the weight operand.  sc * q is a whole number of at most 11 bits (Q4_K 63 * 15, Q5_K
// 63 * 31), which half precision holds exactly; so are the quants of X; and the block's sum stays below 2^24, so the fp32
// accumulator of v_mfma_f32_32x32x16_f16 (Q6_K 16x16x32) holds it exactly, too, and hands it over as a float.  One multiply-add per result
// and block is left (by d8, which is one register: a lane holds one row of X), and one per result and super-block for d:
// 34 ns per 32 x 32 x 32 block by that count at the full clock, 48 to 56 as measured (below).  Q6_K's products have 12 bits and a sign: two operands, the product rounded to half precision and what that
// leaves out, -1, 0 or 1 and hardly ever not 0: a matrix unit that multiplies zeros draws less, and the clock gives way less ([18944,3584] 512
// rows 150 us with the operands q * (sc & ~15) and q * (sc & 15), 144 so).
// The offset term is a contraction over the eight blocks of a super-block of exact halves (the mins are 6-bit whole
// numbers, the stored sums are halves): one more matrix instruction per super-block.
//
// Work split: workgroup tiles of 256 rows of X by 128 weight rows, eight waves of 64 x 64 (four accumulators of 32 x 32, Q6_K sixteen of
// 16 x 16, each twice: the super-block's sum and the total).  K in steps of 64: the rows of X (whole numbers in half precision,
// written by the quantizer) go straight to LDS (global_load_lds, 16-byte pieces, the piece number xored with the row's so
// that the operand reads meet all banks), the packed weights of the next step through registers, decoded once per
// workgroup.  Two buffers, one barrier per step.  Whole rounds of tiles have a workgroup per tile; the super-blocks of the
// tiles behind them are dealt in equal runs to all CUs (192 tiles on 256 CUs: 343 -> 288 us).
//
// Measured against the int8 engine, us per call with the quantizer: [4096,14336] 2100 rows Q4_K 615 -> 410, Q5_K 630 -> 415, 3000 rows Q4_K 834 -> 560; Q6_K
// [4096,14336] 1531 rows 485 -> 355, [18944,3584] 512 rows 199 -> 144, 1024 rows 369 -> 280.  (Up to 2048 rows Q4_K and Q5_K run tile_walk_core.h mostly: the figures of 1531
// rows below are those of this kernel, by which it was built.)
// What bounds it now is vector issue beside the matrix unit, at a clock that falls to about 2.0 GHz under this load: by
// counters ([4096,14336] Q4_K, 1531 rows) the vector ALU issues in 61 % of the SIMD cycles and the matrix unit is busy in
// 35 %, Q6_K ([18944,3584], 512 rows) 46 % and 38 %.  The matrix instructions, the multiply-adds and the operand reads of a step take about 0.45 us
// each; a step takes 1.2 us, a super-block, which is four steps and its end, 5.9 (Q6_K 7.2).  So what is left out counts, not
// what is hidden: with decoding in 30 instead of 50 vector instructions per wave and step (masks and the 1024s as one
// instruction, high nibbles left where they are), LDS addresses whose constants lie in the instructions (40 additions fewer per
// super-block) and the contraction in front of the other wave's decoding the same product takes 299 -> 287 us; Q6_K ([18944,3584], 512 rows) 169 -> 165, once
// the addresses of the store are formed behind the loop: held over it they put 7 registers of Q5_K and 11 to 14 of Q6_K into scratch (168).  The
// contraction alone, matrix instructions and multiply-adds in registers, takes a SIMD 48 to 56 ns per 32 x 32 x 32 block of one operand at any
// interleaving (one wave or two, bursts of one to four blocks): vector instructions hide behind matrix instructions only in part, and the clock falls as
// both get denser.  Of two operands it takes 82 to 86 ns on tiles of 32 x 32 and 71 on tiles of 16 x 16, whose results need half the registers
// on the way: Q6_K [18944,3584] 512 rows 156 -> 150 us, [4096,14336] 1531 rows 390 -> 374.  There a unit's matrix instructions are
// issued two units ahead of its multiply-adds (one ahead: 155 us, three: no change).  One operand is faster on tiles of 32 x 32: [4096,14336] Q4_K 2100 / 3000 rows 405 / 550 us,
// on tiles of 16 x 16 418 / 578, Q5_K 430 / 576 and 446 / 588; 80 random products of 1000 to 4096 rows 1.012 times as fast on average, 0.97 to 1.06,
// [4096,4096] 2500 rows 0.98.
// Tried and slower: four waves per workgroup and two workgroups per CU (decoding twice), the two waves of a SIMD decoding at
// different times, the fetches of X in front of the operand reads or spread over the step; the barrier in the middle of a step
// and the next step's operands behind it, so that no step begins with waiting (same bits, 299 -> 316 us, Q6_K 170 -> 190).
#pragma once
#include "mmq_formats.h"
#include "mmq_f.h"

namespace gguf {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2_m __attribute__((ext_vector_type(2)));

// Whole numbers x below 1024 as the halves 1024 + x: the bits `mask` of both halves of v (`magic`, 0x64006400, in a vector register,
// makes the two operations one instruction, which takes a single scalar operand); bytes 0 and 2, or 1 and 3, of v; the same
// byte of v twice.
__device__ __forceinline__ uint32_t in_register(uint32_t v) {
  uint32_t r;
  asm("v_mov_b32 %0, %1" : "=v"(r) : "s"(v));
  return r;
}
__device__ __forceinline__ f16x2 magic_bits(uint32_t v, uint32_t mask, uint32_t magic) { return __builtin_bit_cast(f16x2, (v & mask) | magic); }
template <int ODD> __device__ __forceinline__ f16x2 magic_bytes(uint32_t v) {
  return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, v, ODD ? 0x04030401u : 0x04020400u));
}
template <int AT> __device__ __forceinline__ f16x2 magic_twice(uint32_t v) {
  return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, v, 0x04000400u | AT << 16 | AT));
}
__device__ __forceinline__ uint32_t bits2(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x2 twice(_Float16 v) { return (f16x2){v, v}; }

// Packed formats.  A step is quarter j of a super-block: blocks 2 j and 2 j + 1.  A thread decodes part p of a row's step:
// values 8 p .. 8 p + 7 of both blocks, each as eight halves in the order of the rows of X (of four neighbours 0, 2, 1, 3).
//   Head     what it takes from the super-block's header, loaded once per super-block; Scales: the same, unpacked
//   PLANES   operands per weight;  OFF: the format has mins
struct FQ4_K {
  static constexpr int BS = 144, PLANES = 1, TILE = 32;
  static constexpr bool OFF = true;
  struct Head { uint4 h; };
  struct Scales { uint32_t s[2]; };
  struct Raw { uint2 q; };
  static __device__ __forceinline__ Head head(const uint8_t* sb) { return {ld<uint4>(sb)}; }
  static __device__ __forceinline__ Raw fetch(const uint8_t* sb, int j, int p) { return {ld<uint2>(sb + 16 + 32 * j + 8 * p)}; }
  static __device__ __forceinline__ Scales scales(const Head& hd) {
    return {{hd.h.y & 0x3F3F3F3Fu, (hd.h.w & 0x0F0F0F0Fu) | ((hd.h.y >> 2) & 0x30303030u)}};
  }
  static __device__ __forceinline__ float d(const Head& hd) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(hd.h.x & 0xFFFF)); }
  static __device__ __forceinline__ float dmin(const Head& hd) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(hd.h.x >> 16)); }
  static __device__ __forceinline__ uint4 mins(const Head& hd) {   // eight halves
    const uint32_t m[2] = {hd.h.z & 0x3F3F3F3Fu, ((hd.h.w >> 4) & 0x0F0F0F0Fu) | ((hd.h.z >> 2) & 0x30303030u)};
    const f16x2 k = twice((_Float16)1024.0f);
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = bits2(__builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, m[i >> 1], i & 1 ? 0x04030402u : 0x04010400u)) - k);
    return make_uint4(o[0], o[1], o[2], o[3]);
  }
  // 1024 + the scale of block 2 J + B, twice
  template <int J, int B> static __device__ __forceinline__ f16x2 scale(const Scales& sc) { return magic_twice<2 * (J & 1) + B>(sc.s[J >> 1]); }
  // (high nibbles stay where they are, sixteen times as large, and their scale is a sixteenth: all exact)
  template <int J> static __device__ __forceinline__ void decode(const Raw& r, const Scales& sc, int, uint4 (&lo)[1], uint4 (&hi)[1]) {
    const uint32_t magic = in_register(0x64006400u);
    const f16x2 s0 = scale<J, 0>(sc) - twice((_Float16)1024.0f);
    const f16x2 s1 = __builtin_elementwise_fma(scale<J, 1>(sc), twice((_Float16)0.0625f), twice((_Float16)-64.0f));
    const f16x2 k = twice((_Float16)-1024.0f), n0 = s0 * k, n1 = s1 * k;   // (exact: six bits times a power of two)
    uint32_t l[4], h[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t a = i ? r.q.y : r.q.x, b = a >> 8;
      l[2 * i] = bits2(__builtin_elementwise_fma(magic_bits(a, 0x000F000Fu, magic), s0, n0));
      l[2 * i + 1] = bits2(__builtin_elementwise_fma(magic_bits(b, 0x000F000Fu, magic), s0, n0));
      h[2 * i] = bits2(__builtin_elementwise_fma(magic_bits(a, 0x00F000F0u, magic), s1, n1));
      h[2 * i + 1] = bits2(__builtin_elementwise_fma(magic_bits(b, 0x00F000F0u, magic), s1, n1));
    }
    lo[0] = make_uint4(l[0], l[1], l[2], l[3]);
    hi[0] = make_uint4(h[0], h[1], h[2], h[3]);
  }
};

struct FQ5_K : FQ4_K {   // Q4_K with a fifth bit, bit b of qh[k] for block b
  static constexpr int BS = 176;
  struct Raw { uint2 q, h; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* sb, int j, int p) {
    return {ld<uint2>(sb + 48 + 32 * j + 8 * p), ld<uint2>(sb + 16 + 8 * p)};
  }
  template <int J> static __device__ __forceinline__ void decode(const Raw& r, const Scales& sc, int, uint4 (&lo)[1], uint4 (&hi)[1]) {
    const f16x2 k = twice((_Float16)-1024.0f), s0 = scale<J, 0>(sc) + k, s1 = scale<J, 1>(sc) + k, n0 = s0 * k, n1 = s1 * k;
    uint32_t l[4], h[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t a = i ? r.q.y : r.q.x, t = i ? r.h.y : r.h.x;
      const uint32_t a0 = (a & 0x0F0F0F0Fu) | (J < 2 ? (t << (4 - 2 * J)) & 0x10101010u : (t >> (2 * J - 4)) & 0x10101010u);
      const uint32_t a1 = ((a >> 4) & 0x0F0F0F0Fu) | (J < 2 ? (t << (3 - 2 * J)) & 0x10101010u : (t >> (2 * J - 3)) & 0x10101010u);
      l[2 * i] = bits2(__builtin_elementwise_fma(magic_bytes<0>(a0), s0, n0));
      l[2 * i + 1] = bits2(__builtin_elementwise_fma(magic_bytes<1>(a0), s0, n0));
      h[2 * i] = bits2(__builtin_elementwise_fma(magic_bytes<0>(a1), s1, n1));
      h[2 * i + 1] = bits2(__builtin_elementwise_fma(magic_bytes<1>(a1), s1, n1));
    }
    lo[0] = make_uint4(l[0], l[1], l[2], l[3]);
    hi[0] = make_uint4(h[0], h[1], h[2], h[3]);
  }
};

struct FQ6_K {
  static constexpr int BS = 210, PLANES = 2, TILE = 16;
  static constexpr bool OFF = false;
  struct Head { uint32_t d; };
  struct Scales {};
  struct Raw { uint2 l0, l1, h; uint32_t s; };   // s: the scales of the step's four groups
  static __device__ __forceinline__ Head head(const uint8_t* sb) { return {ld<uint16_t>(sb + 208)}; }
  static __device__ __forceinline__ Raw fetch(const uint8_t* sb, int j, int p) {
    const uint8_t* l = sb + 64 * (j >> 1) + 8 * p;
    return {ld<uint2>(l), ld<uint2>(l + 32), ld<uint2>(sb + 128 + 32 * (j >> 1) + 8 * p), ld<uint32_t>(sb + 192 + 4 * j)};
  }
  static __device__ __forceinline__ Scales scales(const Head&) { return {}; }
  static __device__ __forceinline__ float d(const Head& hd) { return (float)__builtin_bit_cast(_Float16, (uint16_t)hd.d); }
  static __device__ __forceinline__ float dmin(const Head&) { return 0.0f; }
  static __device__ __forceinline__ uint4 mins(const Head&) { return make_uint4(0, 0, 0, 0); }
  // four 6-bit codes -> (code - 32) * scale rounded to half precision, at most 12 bits, and what that leaves out, -1, 0 or 1
  static __device__ __forceinline__ void planes(uint32_t v, f16x2 s, uint32_t& h0, uint32_t& h1, uint32_t& l0, uint32_t& l1) {
    const f16x2 k = twice((_Float16)1056.0f);
    const f16x2 a = magic_bytes<0>(v) - k, b = magic_bytes<1>(v) - k, ha = a * s, hb = b * s;
    h0 = bits2(ha);
    h1 = bits2(hb);
    l0 = bits2(__builtin_elementwise_fma(a, s, -ha));
    l1 = bits2(__builtin_elementwise_fma(b, s, -hb));
  }
  template <int J> static __device__ __forceinline__ void decode(const Raw& r, const Scales&, int p, uint4 (&lo)[2], uint4 (&hi)[2]) {
    // scales of the values of this part: group p / 2 of blocks 2 j and 2 j + 1
    const uint32_t w = r.s >> (8 * (p >> 1));
    const f16x2 k = twice((_Float16)1152.0f);               // (the sign bit flipped: 1024 + 128 + scale)
    const f16x2 s0 = __builtin_bit_cast(f16x2, bits2(magic_twice<0>(w)) ^ 0x00800080u) - k, s1 = __builtin_bit_cast(f16x2, bits2(magic_twice<2>(w)) ^ 0x00800080u) - k;
    uint32_t a[2][4], b[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t q0 = i ? r.l0.y : r.l0.x, q1 = i ? r.l1.y : r.l1.x, t = i ? r.h.y : r.h.x;
      const uint32_t v0 = J & 1 ? ((q0 >> 4) & 0x0F0F0F0Fu) | (t & 0x30303030u) : (q0 & 0x0F0F0F0Fu) | ((t << 4) & 0x30303030u);
      const uint32_t v1 = J & 1 ? ((q1 >> 4) & 0x0F0F0F0Fu) | ((t >> 2) & 0x30303030u) : (q1 & 0x0F0F0F0Fu) | ((t << 2) & 0x30303030u);
      planes(v0, s0, a[0][2 * i], a[0][2 * i + 1], a[1][2 * i], a[1][2 * i + 1]);
      planes(v1, s1, b[0][2 * i], b[0][2 * i + 1], b[1][2 * i], b[1][2 * i + 1]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      lo[i] = make_uint4(a[i][0], a[i][1], a[i][2], a[i][3]);
      hi[i] = make_uint4(b[i][0], b[i][1], b[i][2], b[i][3]);
    }
  }
};

struct MmqfArgs {
  TileRuns r;                  // (units are super-blocks)
  int64_t w_pitch;
  uint32_t x_pitch, rows;      // bytes between the rows of X; rows of the planes
};

// The values are computed at this point.
__device__ __forceinline__ void pin(float (&v)[4]) { asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])); }
__device__ __forceinline__ void pin(float (&v)[16]) {
  asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
  asm volatile("" : "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]), "+v"(v[12]), "+v"(v[13]), "+v"(v[14]), "+v"(v[15]));
}

// eight waves of 64 x 64
constexpr int MMQF_WM = 4, MMQF_WN = 2, MMQF_MT = 64 * MMQF_WM, MMQF_NT = 64 * MMQF_WN;

template <class F>
__host__ __device__ constexpr int mmqf_buffer_bytes() { return 128 * (MMQF_MT + F::PLANES * MMQF_NT); }
// d8 [8][M_T], of two super-blocks; then of the one at hand, for its end: sums [M_T] of eight halves, d [N_T] and, with
// offsets, -dmin [N_T] and mins [N_T] of eight halves
template <class F>
__host__ __device__ constexpr size_t mmqf_lds() { return 2 * (size_t)(mmqf_buffer_bytes<F>() + 32 * MMQF_MT) + 16 * MMQF_MT + (F::OFF ? 24 : 4) * MMQF_NT; }

// v, opaque to the compiler: what is formed from it is formed where it stands, not kept in registers over the loop
__device__ __forceinline__ int afresh(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// LDS by byte numbers: what is constant in one goes into the instruction (from a pointer, a zero is added first).
template <typename V> using lds_ptr = __attribute__((address_space(3))) V*;
template <typename V> __device__ __forceinline__ V lds_get(uint32_t at) { return *(lds_ptr<const V>)(uintptr_t)at; }
template <typename V> __device__ __forceinline__ void lds_put(uint32_t at, V v) { *(lds_ptr<V>)(uintptr_t)at = v; }
typedef uint32_t u32x4_m __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4_m as_vector(const uint4& v) { return (u32x4_m){v.x, v.y, v.z, v.w}; }

template <int J> struct StepIndex { static constexpr int value = J; };

// Tiles of S x S, the format's choice: a block of 32 values is one instruction of 16 x 16 x 32 or two of 32 x 32 x 16.
template <int S> struct MmqfTile;
template <> struct MmqfTile<16> {
  typedef tile_f4v Sums;
  static constexpr int PIECES = 1, AHEAD = 2, SETS = 2;   // instructions a block; units asked for ahead; blocks of X in registers
  static __device__ __forceinline__ Sums mfma(f16x8 w, f16x8 x, Sums s) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(w, x, s, 0, 0, 0); }
};
template <> struct MmqfTile<32> {
  typedef f32x16 Sums;
  static constexpr int PIECES = 2, AHEAD = 1, SETS = 1;
  static __device__ __forceinline__ Sums mfma(f16x8 w, f16x8 x, Sums s) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(w, x, s, 0, 0, 0); }
};

template <class F, typename T, int S>
__global__ __launch_bounds__(64 * MMQF_WM * MMQF_WN, 2) void mmqf_kernel(const uint8_t* __restrict__ W, const char* __restrict__ X,
                                                               const char* __restrict__ XD, const char* __restrict__ XS,
                                                               T* __restrict__ Y, float* __restrict__ partial,
                                                               const T* __restrict__ bias, MmqfArgs a) {
  typedef MmqfTile<S> Tile;
  constexpr int WN = MMQF_WN, TM = 64 / S, TN = 64 / S, R = S * S / 64, NWV = MMQF_WM * WN, M_T = MMQF_MT, N_T = MMQF_NT;   // R: results of a tile in a lane
  constexpr int BUF = mmqf_buffer_bytes<F>(), PLANE_AT = 2 * BUF + 64 * M_T;
  constexpr int XI = M_T / 8 / NWV;                         // fetches of 8 rows of X per wave and step
  static_assert(4 * N_T == 64 * NWV && M_T == 256, "a thread per part of a row's step; a fetch per row of block scales");
  extern __shared__ __align__(128) char smem[];             // (rows of 128 bytes, whose pieces are told apart by xor with their addresses)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, lrow = lane & (S - 1), lgroup = lane / S;

  const TileWork work = tile_work(a.r);
  const int unit_end = work.end;
  int unit = work.first;
  for (int segment = 0; unit < unit_end; ++segment) {
  const int tile = unit / a.r.units, sb0 = unit - tile * a.r.units, sb1 = min(a.r.units, sb0 + unit_end - unit);
  unit += sb1 - sb0;
  const int m_base = (tile % a.r.tiles_m) * M_T, n_base = (tile / a.r.tiles_m) * N_T;

  // ---- staging plans
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  // (a fetch puts its lanes' 16 bytes one behind the other: the lane of slot l % 8 of a row asks for the piece that belongs there)
  const uint32_t x_at = (uint32_t)(8 * wave + (lane >> 3)) * a.x_pitch + 16 * ((lane & 7) ^ ((4 * wave + (lane >> 4)) & 7));
  const auto fetch_lds = [&](uint32_t at, const char* base, uint32_t to) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(at), "s"(base), "s"(to) : "memory");
  };
  const char* const x_tile = X + (int64_t)m_base * a.x_pitch;
  const auto fetch_x = [&](int g, int buf) {                // step g of the row (64 values, 128 bytes)
#pragma unroll
    for (int i = 0; i < XI; ++i)
      fetch_lds(x_at, x_tile + (128u * (uint32_t)g + (uint32_t)(8 * NWV * i) * a.x_pitch), lds0 + buf * BUF + 1024 * (wave + NWV * i));
  };
  // the planes of a super-block of the rows of X: d8 is 8 rows of M_T floats, the sums M_T rows of 16 bytes
  const auto fetch_d8 = [&](int sb, int pb) {
#pragma unroll
    for (int q = wave; q < 8; q += NWV)                     // (1 KB each, a block's)
      fetch_lds(16 * lane, XD + 4 * ((int64_t)(8 * sb + q) * a.rows + m_base), lds0 + 2 * BUF + 32 * M_T * pb + 1024 * q);
  };
  const auto fetch_sums = [&](int sb) {
#pragma unroll
    for (int q = wave; q < M_T / 64; q += NWV)
      fetch_lds(16 * lane, XS + 16 * ((int64_t)sb * a.rows + m_base + 64 * q), lds0 + PLANE_AT + 1024 * q);
  };
  // weights: a thread has one part of a row's step
  const int w_n = tid >> 2, part = tid & 3;
  // (its two places in a buffer are pieces p and 4 + p, xored like the operands' pieces)
  const auto w_place = [&](int id) { return lds0 + 128 * (M_T + (id >> 2)) + 16 * ((id & 3) ^ ((id >> 3) & 7)); };
  const uint32_t w_to = w_place(tid);                       // (two planes leave no register for it)
  const uint32_t w_row = (uint32_t)min(n_base + w_n, a.r.N - 1) * (uint32_t)a.w_pitch;   // (the matrix is below 4 GB: mmqf_takes)
  typename F::Head hd;
  typename F::Scales sc;
  typename F::Raw raw;
  const auto fetch_raw = [&](int g) { raw = F::fetch(W + (w_row + (uint32_t)(g >> 2) * F::BS), g & 3, part); };
  const auto fetch_head = [&](int sb) { hd = F::head(W + (w_row + (uint32_t)sb * F::BS)); };
  const auto stash_head = [&]() {
    const int id = afresh(tid), n = id >> 2;
    if ((id & 3) == 0) {
      const uint32_t at = lds0 + PLANE_AT + 16 * M_T + 4 * n;
      lds_put<float>(at, F::d(hd));
      if (F::OFF) {
        lds_put<float>(at + 4 * N_T, -F::dmin(hd));
        lds_put<u32x4_m>(at + 8 * N_T + 12 * n, as_vector(F::mins(hd)));
      }
    }
  };
  const auto stash = [&](auto step, int buf) {
    constexpr int J = decltype(step)::value;
    const uint32_t to = F::PLANES == 1 ? (uint32_t)afresh((int)w_to) : w_place(afresh(tid));
    uint4 lo[F::PLANES], hi[F::PLANES];
    F::template decode<J>(raw, sc, afresh(tid) & 3, lo, hi);
#pragma unroll
    for (int pl = 0; pl < F::PLANES; ++pl) {
      lds_put(to + (buf * BUF + 128 * N_T * pl), as_vector(lo[pl]));
      lds_put((to ^ 64) + (buf * BUF + 128 * N_T * pl), as_vector(hi[pl]));
    }
  };

  float acc[TN][TM][R], part_acc[TN][TM][R];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int k = 0; k < TM; ++k)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[i][k][r] = 0.0f;
  typename Tile::Sums zero;
#pragma unroll
  for (int r = 0; r < R; ++r) zero[r] = 0.0f;

  // ---- one step of K: 2 U units, a block and a pair of tiles each
  const int swz = (lrow >> 1) & 7;                          // (tile bases are multiples of 16 rows)
  // (the operands of block b, piece h are 64 b + 32 h away, by xor: rows are 128 bytes)
  const uint32_t op0 = 128 * lrow + 16 * (lgroup ^ swz), x_op = lds0 + 128 * 64 * wm, w_op = lds0 + 128 * (M_T + 64 * wn);
  constexpr int U = TM * TN, H = Tile::PIECES, P = H * F::PLANES, AHEAD = Tile::AHEAD, SETS = Tile::SETS;
  struct Operands { f16x8 x[SETS][TM][H], w[TN][F::PLANES][H]; };
  const auto load_x = [&](uint32_t at, int b, int k, Operands& o) {
#pragma unroll
    for (int h = 0; h < H; ++h) o.x[b % SETS][k][h] = lds_get<f16x8>((at ^ (64 * b + 32 * h)) + 128 * S * k);
  };
  const auto load_w = [&](uint32_t at, int b, int i, Operands& o) {
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int pl = 0; pl < F::PLANES; ++pl) o.w[i][pl][h] = lds_get<f16x8>((at ^ (64 * b + 32 * h)) + (128 * N_T * pl + 128 * S * i));
  };
  // The matrix instructions of unit v + AHEAD stand between the multiply-adds of unit v (each waits for the one before it), and an operand's
  // successor is read as soon as the last instruction that takes it has started.
  const auto load_first = [&](int buf, Operands& o) {
    const uint32_t xat = x_op + buf * BUF + afresh(op0), wat = w_op + buf * BUF + afresh(op0);
#pragma unroll
    for (int i = 0; i < TN; ++i) load_w(wat, 0, i, o);
#pragma unroll
    for (int k = 0; k < TM; ++k) load_x(xat, 0, k, o);
  };
  const auto contract = [&](auto step, int buf, int pb, Operands& o) {
    constexpr int J = decltype(step)::value;
    const uint32_t xd = lds0 + 2 * BUF + 32 * M_T * pb + 256 * wm + 4 * (afresh(lane) & (S - 1)), xat = x_op + buf * BUF + afresh(op0), wat = w_op + buf * BUF + afresh(op0);
    typename Tile::Sums s[2 * AHEAD];
    float d8[2][TM];
#pragma unroll
    for (int k = 0; k < TM; ++k) {
      d8[0][k] = lds_get<float>(xd + (8 * J * M_T + 4 * S * k));
      d8[1][k] = lds_get<float>(xd + (8 * J * M_T + 4 * M_T + 4 * S * k));
    }
    const auto mfma = [&](int v, int piece) {
      const int b = v / U, i = v % U / TM, k = v % TM, to = v % (2 * AHEAD);
      s[to] = Tile::mfma(o.w[i][piece / H][piece % H], o.x[b % SETS][k][piece % H], piece == 0 ? zero : s[to]);
    };
#pragma unroll
    for (int v = 0; v < AHEAD; ++v)
#pragma unroll
      for (int piece = 0; piece < P; ++piece) mfma(v, piece);
#pragma unroll
    for (int v = 0; v < 2 * U; ++v) {
      const int b = v / U, u = v % U, i = u / TM, k = u % TM, n = v + AHEAD, from = v % (2 * AHEAD);
#pragma unroll
      for (int piece = 0; piece < P; ++piece) {
        if (n < 2 * U) mfma(n, piece);
        if (piece == P - 1 && n < U) {
          if (n % TM == TM - 1) load_w(wat, 1, n / TM, o);
          if (n / TM == TN - SETS) load_x(xat, 1, n % TM, o);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = R / P * piece; r < R / P * (piece + 1); ++r)
          part_acc[i][k][r] = J == 0 && b == 0 ? s[from][r] * d8[b][k] : __builtin_fmaf(s[from][r], d8[b][k], part_acc[i][k][r]);
        __builtin_amdgcn_sched_barrier(0);
      }
      // (here and not later: the compiler would keep the products and scale them all at the end of the super-block)
      pin(part_acc[i][k]);
    }
  };
  // the end of a super-block
  const auto fold = [&]() {
    const int ln = afresh(lane), row = ln & (S - 1), group = ln / S;
    const uint32_t at = lds0 + PLANE_AT + 16 * M_T + 4 * (64 * wn + 4 * group);        // d of the lane's first result
    u32x4_m sv[TM];
    if constexpr (F::OFF)
#pragma unroll
      for (int k = 0; k < TM; ++k) {
        // (a contraction over eight: the other lanes hold the values behind them, zeros beside mins, which are finite)
        sv[k] = lds_get<u32x4_m>(lds0 + PLANE_AT + 16 * (64 * wm + row) + 16 * S * k);
        if (group) sv[k] = (u32x4_m){0, 0, 0, 0};
      }
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      typename Tile::Sums off[F::OFF ? TM : 1];
      tile_f4v d[R / 4], dm[R / 4];
      if constexpr (F::OFF) {
        const u32x4_m mv = lds_get<u32x4_m>(lds0 + PLANE_AT + 16 * M_T + 8 * N_T + 16 * (64 * wn + row) + 16 * S * i);
#pragma unroll
        for (int k = 0; k < TM; ++k) off[k] = Tile::mfma(__builtin_bit_cast(f16x8, mv), __builtin_bit_cast(f16x8, sv[k]), zero);
      }
#pragma unroll
      for (int q = 0; q < R / 4; ++q) {
        d[q] = lds_get<tile_f4v>(at + (4 * S * i + 32 * q));
        if (F::OFF) dm[q] = lds_get<tile_f4v>(at + (4 * N_T + 4 * S * i + 32 * q));
      }
#pragma unroll
      for (int k = 0; k < TM; ++k) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          acc[i][k][r] = __builtin_fmaf(part_acc[i][k][r], d[r >> 2][r & 3], acc[i][k][r]);
          if constexpr (F::OFF) acc[i][k][r] = __builtin_fmaf(off[k][r], dm[r >> 2][r & 3], acc[i][k][r]);
        }
        pin(acc[i][k]);
      }
    }
  };

  const int g1 = 4 * sb1;
  if (sb0 < sb1) {
    fetch_head(sb0);
    fetch_raw(4 * sb0);
    fetch_d8(sb0, 0);
    fetch_x(4 * sb0, 0);
    sc = F::scales(hd);
    stash(StepIndex<0>(), 0);
    fetch_raw(4 * sb0 + 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // In step g: the registers (step g + 1, loaded during g - 1) are decoded into the other buffer, the rows of X of
    // g + 1 are asked for, the packed weights of g + 2, and step g is contracted.
    for (int sb = sb0; sb < sb1; ++sb) {
      const int pb = (sb - sb0) & 1;
      const bool more = sb + 1 < sb1;
      const auto turn = [&](auto step) {
        constexpr int J = decltype(step)::value;
        const int g = 4 * sb + J;
        Operands o;
        load_first(J & 1, o);                               // (they arrive under the decoding)
        __builtin_amdgcn_sched_barrier(0);
        if (J == 1) stash_head();                           // (the end of the super-block before has been)
        if (J < 3 || more) {
          if (J == 3) sc = F::scales(hd);
          stash(StepIndex<(J + 1) & 3>(), (J + 1) & 1);
          fetch_x(g + 1, (J + 1) & 1);
          if (g + 2 < g1) fetch_raw(g + 2);
        }
        if (J == 1 && F::OFF) fetch_sums(sb);
        if (J == 2 && more) {
          fetch_d8(sb + 1, pb ^ 1);
          fetch_head(sb + 1);
        }
        __builtin_amdgcn_s_setprio(1);                      // (over the other wave's decoding)
        contract(step, J & 1, pb, o);
        __builtin_amdgcn_s_setprio(0);
        if (J == 3) fold();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
      };
      turn(StepIndex<0>());
      turn(StepIndex<1>());
      turn(StepIndex<2>());
      turn(StepIndex<3>());
    }
  }

  // ---- store: lane = one row of X, R features per tile in runs of four
  float* const mine = sb1 - sb0 < a.r.units ? partial + (int64_t)(2 * work.worker + segment) * (M_T * N_T) : nullptr;
  const int ln = afresh(lane), group = ln / S;              // (the places formed from it: not in scratch from before the first tile on)
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int k = 0; k < TM; ++k)
#pragma unroll
      for (int q = 0; q < R / 4; ++q) {
        const tile_f4v v = {acc[i][k][4 * q], acc[i][k][4 * q + 1], acc[i][k][4 * q + 2], acc[i][k][4 * q + 3]};
        if (mine) {   // in the order that tile_reduce_kernel adds: [wave][tile of 32 x 32][run][lane] of four
          const int of32 = wave * 4 + S * i / 32 * 2 + S * k / 32, run = S == 32 ? q : 2 * (i & 1) + (group >> 1), at = S == 32 ? ln : 32 * (group & 1) + 16 * (k & 1) + (ln & 15);
          *(tile_f4v*)(mine + ((of32 * 4 + run) * 64 + at) * 4) = v;
        } else {
          tile_store(v, m_base + 64 * wm + S * k + (ln & (S - 1)), n_base + 64 * wn + S * i + 8 * q + 4 * group, Y, bias, a.r);
        }
      }
  }
}

template <class F, typename T>
static int mmqf_typed(const MmqfCall& c, hipStream_t stream) {
  const TilePlan p = mmqf_plan(c.M, c.N, c.K, c.partial_bytes);
  constexpr size_t lds = mmqf_lds<F>();
  static_assert(lds <= 160 * 1024, "tile does not fit in LDS");
  auto kern = mmqf_kernel<F, T, F::TILE>;
  static std::atomic<uint64_t> done{0};
  allow_large_lds(kern, lds, done);
  const MmqfArgs a = {tile_runs<T>(p, c.M, c.N, c.K / 256, c.Y, c.la.ldy ? c.la.ldy : (int64_t)c.N),
                      c.la.w_pitch ? c.la.w_pitch : (int64_t)(c.K / 256) * F::BS, (uint32_t)(2 * c.x.pitch), (uint32_t)c.x.rows};
  hipLaunchKernelGGL(kern, dim3(p.whole + p.workers), dim3(64 * MMQF_WM * MMQF_WN), lds, stream, (const uint8_t*)c.W, (const char*)c.x.x,
                     (const char*)c.x.d, (const char*)c.x.s, (T*)c.Y, c.partial, (const T*)c.la.bias, a);
  if (p.shared > 0)
    hipLaunchKernelGGL((tile_reduce_kernel<MMQF_WM, MMQF_WN, 2, 2, T>), dim3(p.shared, MMQF_WM * MMQF_WN * 4), dim3(256),
                       0, stream, c.partial, (T*)c.Y, (const T*)c.la.bias, a.r);
  return launch_status();
}

template <class F>
static int mmqf_fmt(const MmqfCall& c, hipStream_t stream) {
  GGUF_DISPATCH_DTYPE(c.dtype, return (mmqf_typed<F, scalar_t>(c, stream)));
  return GGUF_ERR_DTYPE;
}

}  // namespace gguf
