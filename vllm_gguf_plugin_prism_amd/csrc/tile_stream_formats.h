// Packed formats as the streaming tile kernel (tile_stream_core.h) reads them: one *panel* is 256 values of K of one
// weight row, `PB` contiguous bytes that a wave has fetched into LDS.  A lane is (column c = lane % 16, k group
// g = lane / 16) of v_mfma_i32_16x16x32_i8 and supplies, of every 32-value block, the eight codes k = 8 g .. 8 g + 7
// of its column.  read() takes what the lane needs of a panel into registers (so that the LDS slot can be filled
// again), the other members decode from there.
//   G        values per weight scale: 32, or 16 (two scales per block)
//   OFF      0: no offset term; 1: minus mw(block) times a block sum of the activations (the plane is the caller's choice);
//            2: minus dmin() times the product of the block's quants with min_codes(), a matrix instruction of its own
//   HALVES   the block's sum takes half(d d8), and half(m s8) is added, the products rounded to half precision as the
//            reference's __hmul2 leaves them (vecdotq.cuh:71-93, 179-198); words() gives d and m of the eight blocks
//   ready()  work on the registers that no column's scale depends on, once per panel
//   KQ       the panel is one super-block; else it is eight 32-value blocks and a row may end inside it
#pragma once
#include "mmq_formats.h"

namespace gguf {

// Reads from LDS must lie on their own size: an 8-byte read at any other address takes 27 ns per instruction and CU, one
// lane after the other, against 1.8 ns (the compiler would emit it for a 2-byte-aligned type).  Blocks sit at even
// addresses, so a field of eight bytes is cut out of the two aligned 8-byte words it touches.  `at` counts bytes from
// `base`, which is 16-byte aligned.
__device__ __forceinline__ uint2 lds_cut8(const char* base, uint32_t at) {
  const uint2* const q = (const uint2*)(base + (at & ~7u));
  const uint2 lo = q[0], hi = q[1];
  const bool up = at & 4;
  const uint32_t x0 = up ? lo.y : lo.x, x1 = up ? hi.x : lo.y, x2 = up ? hi.y : hi.x, sh = (at & 2) * 8;
  return make_uint2(__builtin_amdgcn_alignbit(x1, x0, sh), __builtin_amdgcn_alignbit(x2, x1, sh));
}
__device__ __forceinline__ uint4 lds_cut16(const char* base, uint32_t at) {
  const uint2* const q = (const uint2*)(base + (at & ~7u));
  const uint2 a = q[0], b = q[1], c = q[2];
  const bool up = at & 4;
  const uint32_t x0 = up ? a.y : a.x, x1 = up ? b.x : a.y, x2 = up ? b.y : b.x, x3 = up ? c.x : b.y, x4 = up ? c.y : c.x, sh = (at & 2) * 8;
  return make_uint4(__builtin_amdgcn_alignbit(x1, x0, sh), __builtin_amdgcn_alignbit(x2, x1, sh), __builtin_amdgcn_alignbit(x3, x2, sh),
                    __builtin_amdgcn_alignbit(x4, x3, sh));
}
__device__ __forceinline__ uint32_t lds_h(const char* base, uint32_t at) { return *(const uint16_t*)(base + at); }
__device__ __forceinline__ float half_bits(uint32_t b) { return (float)__builtin_bit_cast(_Float16, (uint16_t)b); }

// Q4_K, Q5_K: 6-bit scales and mins of the eight sub-blocks out of the 12 packed bytes (dequantize.cuh:156-163), as
// bytes: blocks 0..3 in the low six bits of bytes 0..3 / 4..7, blocks 4..7 in the nibbles of bytes 8..11 and the top
// two bits of bytes 0..3 / 4..7.
struct KHead {
  uint4 h;
  __device__ __forceinline__ void scales(float (&dw)[8]) const {
    const float d = half_bits(h.x & 0xFFFF);
    const uint32_t s[2] = {h.y & 0x3F3F3F3Fu, (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u)};
#pragma unroll
    for (int b = 0; b < 8; ++b) dw[b] = d * (float)((s[b >> 2] >> (8 * (b & 3))) & 0xFF);
  }
  // the mins of blocks g and 4 + g
  __device__ __forceinline__ void mins(int g, float& m0, float& m1) const {
    const float dmin = half_bits(h.x >> 16);
    m0 = dmin * (float)(((h.z & 0x3F3F3F3Fu) >> (8 * g)) & 0xFF);
    m1 = dmin * (float)(((((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u)) >> (8 * g)) & 0xFF);
  }
};

struct TQ4_K {
  static constexpr int PB = 144, G = 32, OFF = 1;
  static constexpr bool KQ = true, HALVES = false;
  KHead hd;
  uint2 q[4];
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    if (at == 0) {                                          // (whole 16-byte pieces: the tensors that loaders produce)
      hd.h = *(const uint4*)p;
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = *(const uint2*)(p + 16 + 32 * i + 8 * g);
    } else {
      hd.h = lds_cut16(p, at);
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = lds_cut8(p, at + 16 + 32 * i + 8 * g);
    }
  }
  __device__ __forceinline__ void ready() {}
  __device__ __forceinline__ void scales(float (&dw)[8]) const { hd.scales(dw); }
  __device__ __forceinline__ void mins(int g, float& m0, float& m1) const { hd.mins(g, m0, m1); }
  __device__ __forceinline__ uint2 codes(int b, int) const {
    const int s = 4 * (b & 1);
    return make_uint2((q[b >> 1].x >> s) & 0x0F0F0F0Fu, (q[b >> 1].y >> s) & 0x0F0F0F0Fu);
  }
};

struct TQ5_K {
  static constexpr int PB = 176, G = 32, OFF = 1;
  static constexpr bool KQ = true, HALVES = false;
  KHead hd;
  uint2 qh, q[4];
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    if (at == 0) {
      hd.h = *(const uint4*)p;
      qh = *(const uint2*)(p + 16 + 8 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = *(const uint2*)(p + 48 + 32 * i + 8 * g);
    } else {
      hd.h = lds_cut16(p, at);
      qh = lds_cut8(p, at + 16 + 8 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = lds_cut8(p, at + 48 + 32 * i + 8 * g);
    }
  }
  __device__ __forceinline__ void ready() {}
  __device__ __forceinline__ void scales(float (&dw)[8]) const { hd.scales(dw); }
  __device__ __forceinline__ void mins(int g, float& m0, float& m1) const { hd.mins(g, m0, m1); }
  __device__ __forceinline__ uint2 codes(int b, int) const {
    const int s = 4 * (b & 1);
    return make_uint2(((q[b >> 1].x >> s) & 0x0F0F0F0Fu) | (((qh.x >> b) & 0x01010101u) << 4),
                      ((q[b >> 1].y >> s) & 0x0F0F0F0Fu) | (((qh.y >> b) & 0x01010101u) << 4));
  }
};

// Block b = 4 n + t: low nibbles (t < 2) or high ones of ql[64 n + 32 (t % 2) ..], bits 2 t of qh[32 n ..].  The code minus
// 32 is the six bits with the top one inverted, sign-extended; they are left in the top six bits of the byte (four
// times the value, still exact in int8), and the scale is a quarter.
struct TQ6_K {
  static constexpr int PB = 210, G = 16, OFF = 0;
  static constexpr bool KQ = true, HALVES = false, ONE_GROUP = true;
  uint2 ql[4], qh[2];
  uint4 sc;
  uint32_t d;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
#pragma unroll
    for (int i = 0; i < 4; ++i) ql[i] = lds_cut8(p, at + 32 * i + 8 * g);
#pragma unroll
    for (int n = 0; n < 2; ++n) qh[n] = lds_cut8(p, at + 128 + 32 * n + 8 * g);
    sc = lds_cut16(p, at + 192);
    d = lds_h(p, at + 208);
  }
  __device__ __forceinline__ void ready() {
#pragma unroll
    for (int n = 0; n < 2; ++n) { qh[n].x ^= 0xAAAAAAAAu; qh[n].y ^= 0xAAAAAAAAu; }   // the top bit of every two-bit field
  }
  __device__ __forceinline__ void scales(float (&dw)[16]) const {
    const float df = 0.25f * half_bits(d);
    const uint32_t s[4] = {sc.x, sc.y, sc.z, sc.w};
#pragma unroll
    for (int i = 0; i < 16; ++i) dw[i] = df * (float)(int8_t)((s[i >> 2] >> (8 * (i & 3))) & 0xFF);
  }
  static __device__ __forceinline__ uint32_t code4(uint32_t l, uint32_t h, int t) {
    return ((t < 2 ? l << 2 : l >> 2) & 0x3C3C3C3Cu) | ((h << (6 - 2 * t)) & 0xC0C0C0C0u);
  }
  __device__ __forceinline__ uint2 codes(int b, int) const {
    const int n = b >> 2, t = b & 3, i = 2 * n + (t & 1);
    return make_uint2(code4(ql[i].x, qh[n].x, t), code4(ql[i].y, qh[n].y, t));
  }
};

// Eight blocks of `BB` bytes, an fp16 scale in front of each.  A lane reads the scales of blocks g and 4 + g; lane swaps
// give it all eight (rows of 16 lanes g0 g1 g2 g3 -> g0 g1 g0 g1 and g2 g3 g2 g3, and once more).
template <int BB>
struct T32 {
  static constexpr int PB = 8 * BB, G = 32;
  static constexpr bool KQ = false, HALVES = false;
  uint32_t dg[2];
  uint2 q[8];
  __device__ __forceinline__ void ready() {}
  // the eight bytes from `at` + FIELD + `lane_at` of every block; with `at` zero the cuts are known to the compiler (the
  // blocks' bytes begin 2, 4, 6, 0, ... behind an 8-byte word)
  template <int FIELD>
  __device__ __forceinline__ void read_blocks(const char* p, uint32_t at, int g, uint32_t lane_at) {
    dg[0] = lds_h(p, at + BB * g);
    dg[1] = lds_h(p, at + BB * (4 + g));
    if (at == 0) {
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        constexpr int W = 8;
        const int first = BB * b + FIELD, cut = first % W;  // (lane_at is a multiple of 8)
        const uint2* const w = (const uint2*)(p + (first - cut) + lane_at);
        if (cut == 0) {
          q[b] = w[0];
        } else {
          const uint2 lo = w[0], hi = w[1];
          const uint32_t x0 = cut >= 4 ? lo.y : lo.x, x1 = cut >= 4 ? hi.x : lo.y, x2 = cut >= 4 ? hi.y : hi.x;
          q[b] = cut % 4 == 0 ? make_uint2(x0, x1) : make_uint2(__builtin_amdgcn_alignbit(x1, x0, 16), __builtin_amdgcn_alignbit(x2, x1, 16));
        }
      }
    } else {
#pragma unroll
      for (int b = 0; b < 8; ++b) q[b] = lds_cut8(p, at + BB * b + FIELD + lane_at);
    }
  }
  __device__ __forceinline__ void scales(float (&dw)[8]) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto half = __builtin_amdgcn_permlane32_swap(dg[i], dg[i], false, false);
      const auto d01 = __builtin_amdgcn_permlane16_swap(half[0], half[0], false, false);
      const auto d23 = __builtin_amdgcn_permlane16_swap(half[1], half[1], false, false);
      dw[4 * i] = half_bits(d01[0]);
      dw[4 * i + 1] = half_bits(d01[1]);
      dw[4 * i + 2] = half_bits(d23[0]);
      dw[4 * i + 3] = half_bits(d23[1]);
    }
  }
};

// values 0..15 of a block are the low nibbles of its 16 bytes, 16..31 the high ones; d (q - 8), the 8 on the block sum
struct TQ4_0 : T32<18> {
  static constexpr int OFF = 1;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) { read_blocks<2>(p, at, g, 8 * (g & 1)); }
  __device__ __forceinline__ void mins(int, float& m0, float& m1) const { m0 = 8.0f * half_bits(dg[0]); m1 = 8.0f * half_bits(dg[1]); }
  __device__ __forceinline__ uint2 codes(int b, int g) const {
    const int s = 4 * (g >> 1);
    return make_uint2((q[b].x >> s) & 0x0F0F0F0Fu, (q[b].y >> s) & 0x0F0F0F0Fu);
  }
};

struct TQ8_0 : T32<34> {
  static constexpr int OFF = 0;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) { read_blocks<2>(p, at, g, 8 * g); }
  __device__ __forceinline__ uint2 codes(int b, int) const { return q[b]; }
};

__device__ __forceinline__ uint32_t ts_word(const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// Block b = 4 n + t: bits 2 t of qs[32 n ..], bit b of hmask.  The code minus 4 is the three bits with the top one inverted,
// sign-extended; they are left in the top three bits of the byte (32 times the value), and the scale is a 32nd.
struct TQ3_K {
  static constexpr int PB = 110, G = 16, OFF = 0;
  static constexpr bool KQ = true, HALVES = false;
  uint2 q[2], hm;
  uint4 sc;                                                 // twelve bytes of scales, d
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    hm = lds_cut8(p, at + 8 * g);
#pragma unroll
    for (int n = 0; n < 2; ++n) q[n] = lds_cut8(p, at + 32 + 32 * n + 8 * g);
    sc = lds_cut16(p, at + 96);
  }
  __device__ __forceinline__ void ready() { hm.x = ~hm.x; hm.y = ~hm.y; }
  __device__ __forceinline__ void scales(float (&dw)[16]) const {
    const float df = 0.03125f * half_bits(sc.w & 0xFFFF);
    const uint32_t lo[4] = {sc.x & 0x0F0F0F0Fu, sc.y & 0x0F0F0F0Fu, (sc.x >> 4) & 0x0F0F0F0Fu, (sc.y >> 4) & 0x0F0F0F0Fu};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t s = lo[i >> 2] | (((sc.z >> (2 * (i >> 2))) & 0x03030303u) << 4);
      dw[i] = df * (float)((int)((s >> (8 * (i & 3))) & 0xFF) - 32);
    }
  }
  static __device__ __forceinline__ uint32_t code4(uint32_t l, uint32_t h, int b) {
    const int t = b & 3;
    return ((t < 3 ? l << (5 - 2 * t) : l >> 1) & 0x60606060u) | ((h << (7 - b)) & 0x80808080u);
  }
  __device__ __forceinline__ uint2 codes(int b, int) const { return make_uint2(code4(q[b >> 2].x, hm.x, b), code4(q[b >> 2].y, hm.y, b)); }
};

// Block b = 4 n + t: bits 2 t of qs[32 n ..]; a 4-bit scale and min per 16 values.  Code times scale is at most 45 and the min
// at most 15: both products are whole numbers of the matrix instruction, and d and dmin are on the block.
struct TQ2_K {
  static constexpr int PB = 84, G = 32, OFF = 2;
  static constexpr bool KQ = true, HALVES = false;
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  uint2 q[2];
  uint4 sc;                                                 // the lane's scales and mins: the even bytes
  uint32_t dm;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    const uint4 s = lds_cut16(p, at);
#pragma unroll
    for (int n = 0; n < 2; ++n) q[n] = lds_cut8(p, at + 16 + 32 * n + 8 * g);
    dm = lds_h(p, at + 80) | lds_h(p, at + 82) << 16;
    const int up = 8 * (g >> 1);
    sc = make_uint4(s.x >> up, s.y >> up, s.z >> up, s.w >> up);
  }
  __device__ __forceinline__ void ready() {}
  __device__ __forceinline__ void scales(float (&dw)[8]) const {
    const float df = half_bits(dm & 0xFFFF);
#pragma unroll
    for (int b = 0; b < 8; ++b) dw[b] = df;
  }
  __device__ __forceinline__ float dmin() const { return half_bits(dm >> 16); }
  __device__ __forceinline__ uint2 min_codes(int b) const {
    const uint32_t m = (ts_word(sc, b >> 1) >> (16 * (b & 1) + 4)) & 15u, v = __builtin_amdgcn_perm(m, m, 0u);
    return make_uint2(v, v);
  }
  __device__ __forceinline__ uint2 codes(int b, int) const {
    const uint16_t c = (uint16_t)((ts_word(sc, b >> 1) >> (16 * (b & 1))) & 15u);
    const auto times = [&](uint32_t v) {
      return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, (v >> (2 * (b & 3))) & 0x03030303u) * (u16x2){c, c});
    };
    return make_uint2(times(q[b >> 2].x), times(q[b >> 2].y));
  }
};

// The fifth bits of values 4 i .. 4 i + 3 of the lane's eight, in the top bits of four bytes (bits: of the eight).
__device__ __forceinline__ uint32_t ts_fifth_bits(uint32_t bits, int i) {
  return __umul24((i ? bits << 3 : bits << 7) & 0x780u, 0x204081u) & 0x80808080u;
}

// d (q - 16), values as in Q4_0 with a fifth bit.  SIGNED: the 16 is off the code, as the reference's tiles have it (the code
// in the top five bits of the byte, 8 times the value); else on the stored block sum, as its GEMV has it (vecdotq.cuh:98-125).
template <bool SIGNED>
struct TQ5_0 : T32<22> {
  static constexpr int OFF = SIGNED ? 0 : 1;
  uint32_t fifth[2];                                        // a byte per block
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    read_blocks<6>(p, at, g, 8 * (g & 1));
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint32_t f = *(const uint8_t*)(p + at + 22 * b + 2 + g);
      fifth[b >> 2] = b & 3 ? fifth[b >> 2] | f << (8 * (b & 3)) : f;
    }
  }
  __device__ __forceinline__ void ready() {
    if (SIGNED) { fifth[0] = ~fifth[0]; fifth[1] = ~fifth[1]; }
  }
  __device__ __forceinline__ void scales(float (&dw)[8]) const {
    T32<22>::scales(dw);
    if (SIGNED)
#pragma unroll
      for (int b = 0; b < 8; ++b) dw[b] *= 0.125f;
  }
  __device__ __forceinline__ void mins(int, float& m0, float& m1) const { m0 = 16.0f * half_bits(dg[0]); m1 = 16.0f * half_bits(dg[1]); }
  __device__ __forceinline__ uint2 codes(int b, int g) const {
    const int s = 4 * (g >> 1);
    const uint32_t f = fifth[b >> 2] >> (8 * (b & 3)), x = (q[b].x >> s) & 0x0F0F0F0Fu, y = (q[b].y >> s) & 0x0F0F0F0Fu;
    const uint32_t fx = ts_fifth_bits(f, 0), fy = ts_fifth_bits(f, 1);
    return SIGNED ? make_uint2(x << 3 | fx, y << 3 | fy) : make_uint2(x | fx >> 3, y | fy >> 3);
  }
};

// Q4_1, Q5_1: d q + m
template <bool FIFTH>
struct TQ45_1 : T32<FIFTH ? 24 : 20> {
  static constexpr int OFF = 0, BB = FIFTH ? 24 : 20;
  static constexpr bool HALVES = true;
  using T32<BB>::dg;
  using T32<BB>::q;
  uint32_t fifth[FIFTH ? 2 : 1];
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    this->template read_blocks<FIFTH ? 8 : 4>(p, at, g, 8 * (g & 1));
    dg[0] |= lds_h(p, at + BB * g + 2) << 16;
    dg[1] |= lds_h(p, at + BB * (4 + g) + 2) << 16;
    if constexpr (FIFTH)
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const uint32_t f = *(const uint8_t*)(p + at + 24 * b + 4 + g);
        fifth[b >> 2] = b & 3 ? fifth[b >> 2] | f << (8 * (b & 3)) : f;
      }
  }
  __device__ __forceinline__ void words(uint32_t (&dm)[8]) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto half = __builtin_amdgcn_permlane32_swap(dg[i], dg[i], false, false);
      const auto d01 = __builtin_amdgcn_permlane16_swap(half[0], half[0], false, false);
      const auto d23 = __builtin_amdgcn_permlane16_swap(half[1], half[1], false, false);
      dm[4 * i] = d01[0]; dm[4 * i + 1] = d01[1]; dm[4 * i + 2] = d23[0]; dm[4 * i + 3] = d23[1];
    }
  }
  __device__ __forceinline__ uint2 codes(int b, int g) const {
    const int s = 4 * (g >> 1);
    const uint32_t x = (q[b].x >> s) & 0x0F0F0F0Fu, y = (q[b].y >> s) & 0x0F0F0F0Fu;
    if constexpr (!FIFTH) return make_uint2(x, y);
    const uint32_t f = fifth[FIFTH ? b >> 2 : 0] >> (8 * (b & 3));
    return make_uint2(x | ts_fifth_bits(f, 0) >> 3, y | ts_fifth_bits(f, 1) >> 3);
  }
};

// the sixteen values of IQ4_NL and IQ4_XS by the nibbles at bit S of four bytes (vecdotq.cuh:1795-1815)
__device__ __forceinline__ uint32_t ts_iq4(uint32_t v) {
  const uint32_t at = v & 0x07070707u, lo = __builtin_amdgcn_perm(0xF6EADDCFu, 0xBFAD9881u, at), hi = __builtin_amdgcn_perm(0x71594535u, 0x26190D01u, at);
  return __builtin_amdgcn_perm(hi, lo, 0x03020100u | ((v >> 1) & 0x04040404u));
}
struct TIQ4_NL : T32<18> {
  static constexpr int OFF = 0;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) { read_blocks<2>(p, at, g, 8 * (g & 1)); }
  __device__ __forceinline__ uint2 codes(int b, int g) const {
    const int s = 4 * (g >> 1);
    return make_uint2(ts_iq4(q[b].x >> s), ts_iq4(q[b].y >> s));
  }
};
// d (6-bit scale - 32) per 32 values: d, the scales' top bits, their nibbles, the codes as in IQ4_NL
struct TIQ4_XS {
  static constexpr int PB = 136, G = 32, OFF = 0;
  static constexpr bool KQ = true, HALVES = false, ONE_GROUP = true;
  uint2 head, q[8];
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    if ((at & 7) == 0) {
      head = *(const uint2*)(p + at);
#pragma unroll
      for (int b = 0; b < 8; ++b) q[b] = *(const uint2*)(p + at + 8 + 16 * b + 8 * (g & 1));
    } else {
      head = lds_cut8(p, at);
#pragma unroll
      for (int b = 0; b < 8; ++b) q[b] = lds_cut8(p, at + 8 + 16 * b + 8 * (g & 1));
    }
  }
  __device__ __forceinline__ void ready() {}
  __device__ __forceinline__ void scales(float (&dw)[8]) const {
    const float d = half_bits(head.x & 0xFFFF);
#pragma unroll
    for (int b = 0; b < 8; ++b) dw[b] = d * (float)((int)(((head.y >> (4 * b)) & 15u) | ((head.x >> (16 + 2 * b)) & 3u) << 4) - 32);
  }
  __device__ __forceinline__ uint2 codes(int b, int g) const {
    const int s = 4 * (g >> 1);
    return make_uint2(ts_iq4(q[b].x >> s), ts_iq4(q[b].y >> s));
  }
};

}  // namespace gguf
