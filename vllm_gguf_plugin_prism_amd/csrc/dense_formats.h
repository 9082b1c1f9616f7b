// Codebook formats for the GEMM on the matrix unit (dense_core.h): sixteen neighbouring weights as bytes, their signs and one scale.
//
// Every weight of these formats is a scale of at most 16 significant bits times a whole number of at most eight (IQ1: an
// eighth of one), so the fp32 product is exact and rounding it once gives the value of the dequantize kernels.
//   Raw    what sixteen weights need of their block, in registers;  fetch(blk, ib, h): values 16 h .. 16 h + 15 of sub-block ib
//   Entry  an entry of the format's table in LDS (TABLE of them, 0: none);  entry(i) forms it from the 16-bit code word
//   decode the bytes, v[0] holding the first four: the whole numbers plus BIAS, or (BIAS 0) their magnitudes, negated where s[0] (values 0 .. 7, bits 0 .. 7; bits 8 .. 15
//          mean nothing, those behind are 0) and s[1] have a bit.  Returns the scale, of magnitudes 2^24 times it: a byte with a zero byte above it is the half 2^-24 times the
//          byte.
#pragma once
#include "gguf_common.h"
#include "grid_codes.h"
#include <type_traits>

namespace gguf {

__device__ __forceinline__ uint32_t parity8(uint32_t s7) { return s7 | (uint32_t)__builtin_popcount(s7) << 7; }   // the eighth sign makes them even

struct NoTable {
  static constexpr int TABLE = 0;
  typedef uint32_t Entry;
  static __device__ __forceinline__ Entry entry(int) { return 0; }
};
// eight bytes 8, 25, 43 out of 2-bit codes
__device__ __forceinline__ uint2 entry2(uint32_t code) {
  uint32_t b[2] = {0, 0};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t c = (code >> (2 * j)) & 3;
    b[j >> 2] |= (8 + 17 * c + (c >> 1)) << (8 * (j & 3));
  }
  return make_uint2(b[0], b[1]);
}

// the codes in bits 0 .. 3 of four bytes (bits 4 .. 7: anything) through the table of the non-linear 4-bit formats, plus 128
__device__ __forceinline__ uint32_t nonlinear4(uint32_t q) {
  constexpr uint32_t T0 = 0x3F2D1801u, T1 = 0x766A5D4Fu, T2 = 0xA6998D81u, T3 = 0xF1D9C5B5u;   // 1 24 ... 217 241
  const uint32_t sel = q & 0x07070707u, upper = ((q >> 3) & 0x01010101u) | 0x0C0C0C0Cu;
  const uint32_t lo = __builtin_amdgcn_perm(T1, T0, sel), hi = __builtin_amdgcn_perm(T3, T2, sel), m = __builtin_amdgcn_perm(0, 0, upper);   // (13: 0xFF, 12: 0)
  return (hi & m) | (lo & ~m);
}

struct DIQ4_XS : NoTable {
  static constexpr int BIAS = 128;
  static constexpr int BS = 136, QK = 256;
  struct Raw { uint2 hd; uint4 q; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int) { return {ld<uint2>(blk), ld<uint4>(blk + 8 + 16 * ib)}; }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry*, int ib, int h, uint32_t (&v)[4], uint32_t (&s)[2]) {
    const int ls = (int)(((r.hd.y >> (4 * ib)) & 15u) | (((r.hd.x >> (16 + 2 * ib)) & 3u) << 4));
    const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = nonlinear4(q[i] >> (4 * h));
    return (float)__builtin_bit_cast(_Float16, (uint16_t)r.hd.x) * (float)(ls - 32);
  }
};

struct DIQ4_NL : NoTable {
  static constexpr int BIAS = 128;
  static constexpr int BS = 18, QK = 32;
  struct Raw { uint16_t d; uint4 q; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int, int) { return {ld<uint16_t>(blk), ld<uint4>(blk + 2)}; }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry*, int, int h, uint32_t (&v)[4], uint32_t (&s)[2]) {
    const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = nonlinear4(q[i] >> (4 * h));
    return (float)__builtin_bit_cast(_Float16, r.d);
  }
};

struct DIQ2_XXS {
  static constexpr int BIAS = 0;
  static constexpr int BS = 66, QK = 256, TABLE = 256;
  typedef uint2 Entry;
  static __device__ __forceinline__ Entry entry(int i) { return entry2(k_iq2xxs_grid_codes[i]); }
  struct Raw { uint16_t d; uint2 q; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int) { return {ld<uint16_t>(blk), ld<uint2>(blk + 2 + 8 * ib)}; }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4], uint32_t (&s)[2]) {
    const uint32_t q = r.q.x >> (16 * h), s14 = r.q.y >> (14 * h);
    s[0] = parity8(s14 & 127u); s[1] = parity8((s14 >> 7) & 127u);
    const Entry a = t[q & 255u], b = t[(q >> 8) & 255u];
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)(r.q.y >> 28)) * (0.25f * 0x1p24f);
  }
};

struct DIQ2_XS {
  static constexpr int BIAS = 0;
  static constexpr int BS = 74, QK = 256, TABLE = 512;
  typedef uint2 Entry;
  static __device__ __forceinline__ Entry entry(int i) { return entry2(k_iq2xs_grid_codes[i]); }
  struct Raw { uint16_t d; uint32_t q; uint8_t sc; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int h) {
    return {ld<uint16_t>(blk), ld<uint32_t>(blk + 2 + 8 * ib + 4 * h), blk[66 + ib]};
  }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4], uint32_t (&s)[2]) {
    s[0] = parity8((r.q >> 9) & 127u); s[1] = parity8(r.q >> 25);
    const Entry a = t[r.q & 511u], b = t[(r.q >> 16) & 511u];
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)((r.sc >> (4 * h)) & 15)) * (0.25f * 0x1p24f);
  }
};

struct DIQ2_S {
  static constexpr int BIAS = 0;
  static constexpr int BS = 82, QK = 256, TABLE = 1024;
  typedef uint2 Entry;
  static __device__ __forceinline__ Entry entry(int i) { return entry2(k_iq2s_grid_codes[i]); }
  struct Raw { uint16_t d, q, s; uint8_t qh, sc; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int h) {
    return {ld<uint16_t>(blk), ld<uint16_t>(blk + 2 + 4 * ib + 2 * h), ld<uint16_t>(blk + 34 + 4 * ib + 2 * h), blk[66 + ib], blk[74 + ib]};
  }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4], uint32_t (&s)[2]) {
    const uint32_t qh = (uint32_t)r.qh >> (4 * h);   // two bits for each group of eight
    const Entry a = t[(r.q & 255u) | (qh & 3u) << 8], b = t[(r.q >> 8) | (qh & 12u) << 6];
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
    s[0] = r.s; s[1] = (uint32_t)r.s >> 8;
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)((r.sc >> (4 * h)) & 15)) * (0.25f * 0x1p24f);
  }
};

struct DIQ3_XXS {
  static constexpr int BIAS = 0;
  static constexpr int BS = 98, QK = 256, TABLE = 256;
  typedef uint32_t Entry;
  static __device__ __forceinline__ Entry entry(int i) {   // 4, 12, ..., 52, 62
    const uint32_t code = k_iq3xxs_grid_codes[i];
    uint32_t b = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t c = (code >> (3 * j)) & 7;
      b |= (4 + 8 * c + 2 * ((c + 1) >> 3)) << (8 * j);
    }
    return b;
  }
  struct Raw { uint16_t d; uint32_t q, aux; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int h) {
    return {ld<uint16_t>(blk), ld<uint32_t>(blk + 2 + 8 * ib + 4 * h), ld<uint32_t>(blk + 66 + 4 * ib)};
  }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4], uint32_t (&s)[2]) {
    const uint32_t s14 = r.aux >> (14 * h);
    s[0] = parity8(s14 & 127u); s[1] = parity8((s14 >> 7) & 127u);
    v[0] = t[r.q & 255u]; v[1] = t[(r.q >> 8) & 255u]; v[2] = t[(r.q >> 16) & 255u]; v[3] = t[r.q >> 24];
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)(r.aux >> 28)) * (0.5f * 0x1p24f);
  }
};

struct DIQ3_S {
  static constexpr int BIAS = 0;
  static constexpr int BS = 110, QK = 256, TABLE = 512;
  typedef uint32_t Entry;
  static __device__ __forceinline__ Entry entry(int i) {   // 4, 12, ..., 60
    const uint32_t code = k_iq3xs_grid_codes[i];
    uint32_t b = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) b |= (4 + 8 * ((code >> (3 * j)) & 7)) << (8 * j);
    return b;
  }
  struct Raw { uint16_t d; uint32_t q; uint16_t s; uint8_t qh, sc; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int h) {
    return {ld<uint16_t>(blk), ld<uint32_t>(blk + 2 + 8 * ib + 4 * h), ld<uint16_t>(blk + 74 + 4 * ib + 2 * h), blk[66 + ib], blk[106 + (ib >> 1)]};
  }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int ib, int h, uint32_t (&v)[4], uint32_t (&s)[2]) {
    const uint32_t qh = (uint32_t)r.qh >> (4 * h);   // one bit for each group of four
    v[0] = t[(r.q & 255u) | (qh & 1u) << 8]; v[1] = t[((r.q >> 8) & 255u) | (qh & 2u) << 7];
    v[2] = t[((r.q >> 16) & 255u) | (qh & 4u) << 6]; v[3] = t[(r.q >> 24) | (qh & 8u) << 5];
    s[0] = r.s; s[1] = (uint32_t)r.s >> 8;
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)((r.sc >> (4 * (ib & 1))) & 15)) * (0.5f * 0x1p24f);
  }
};

// The 1-bit formats: d (q - 1 -+ 1/8), q of {0, 1, 2}: an eighth of the whole number 8 q - 7 or 8 q - 9.
struct IQ1Table {
  static constexpr int TABLE = 2048, BIAS = 128;
  typedef uint2 Entry;                                      // 128 + 8 q, in the order of the values (the code word holds the even ones first)
  static __device__ __forceinline__ Entry entry(int i) {
    const uint32_t code = k_iq1s_grid_gpu_codes[i];
    uint32_t b[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < 8; ++j) b[j >> 2] |= (128 + 8 * ((code >> (4 * (j & 3) + 2 * (j >> 2))) & 3)) << (8 * (j & 3));
    return make_uint2(b[0], b[1]);
  }
  static __device__ __forceinline__ void group(Entry a, bool minus, uint32_t& v0, uint32_t& v1) {   // (no byte borrows)
    const uint32_t k = minus ? 0x09090909u : 0x07070707u;
    v0 = a.x - k;
    v1 = a.y - k;
  }
};

struct DIQ1_S : IQ1Table {
  static constexpr int BS = 50, QK = 256;
  struct Raw { uint16_t d, q, qh; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int h) {
    return {ld<uint16_t>(blk), ld<uint16_t>(blk + 2 + 4 * ib + 2 * h), ld<uint16_t>(blk + 34 + 2 * ib)};
  }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4], uint32_t (&s)[2]) {
    const uint32_t qh = r.qh, i3 = qh >> (6 * h);
    const bool minus = qh & 0x8000u;
    group(t[(r.q & 255u) | (i3 & 7u) << 8], minus, v[0], v[1]);
    group(t[(r.q >> 8) | (i3 & 0x38u) << 5], minus, v[2], v[3]);
    return (float)__builtin_bit_cast(_Float16, r.d) * (float)(2 * ((qh >> 12) & 7) + 1) * 0.125f;
  }
};

struct DIQ1_M : IQ1Table {
  static constexpr int BS = 56, QK = 256;
  struct Raw { uint2 s; uint16_t q; uint8_t qh; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int h) {
    return {ld<uint2>(blk + 48), ld<uint16_t>(blk + 4 * ib + 2 * h), blk[32 + 2 * ib + h]};
  }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int ib, int h, uint32_t (&v)[4], uint32_t (&s)[2]) {
    const uint32_t qh = r.qh;
    group(t[(r.q & 255u) | (qh & 7u) << 8], qh & 0x08u, v[0], v[1]);
    group(t[(r.q >> 8) | (qh & 0x70u) << 4], qh & 0x80u, v[2], v[3]);
    // the super-scale lies in the top nibbles of the four words of scales
    const uint32_t d = ((r.s.x >> 12) & 0xFu) | ((r.s.x >> 24) & 0xF0u) | ((r.s.y >> 4) & 0xF00u) | ((r.s.y >> 16) & 0xF000u);
    const int i16 = 2 * ib + h;
    const uint32_t w = i16 & 8 ? r.s.y : r.s.x;
    const uint32_t sc = (w >> (16 * ((i16 >> 2) & 1) + 3 * (i16 & 3))) & 7u;
    return (float)__builtin_bit_cast(_Float16, (uint16_t)d) * (float)(2 * sc + 1) * 0.125f;
  }
};

// Sixteen decoded weights rounded to 16 bits, two to a word.  Magnitudes go into halves of words, their signs beside them, and one multiply-add each takes them from there (in
// place of negated bytes, their conversion and the multiply-add: 460 random IQ2 and IQ3 products of 12 to 1500 rows: 1.03 times as fast where walked, else 1.01, the same results); bytes plus BIAS are converted (the other
// way: IQ4 0.99).
template <class F, typename V2> __device__ __forceinline__ void dense_operands(const uint32_t (&v)[4], const uint32_t (&s)[2], float d, uint32_t (&o)[8]) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  if constexpr (F::BIAS != 0) {
    const float c = -(float)F::BIAS * d;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t b = v[i >> 1] >> (16 * (i & 1));
      o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){__builtin_fmaf((float)(b & 255u), d, c), __builtin_fmaf((float)((b >> 8) & 255u), d, c)}, V2));
    }
  } else {
    uint32_t both[2];                                       // signs 2 i and 2 i + 1 sixteen bits apart
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      both[i] = s[i] << 15 | s[i];
      asm("" : "+v"(both[i]));                              // (else each use becomes a multiplication by its own constant)
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t w = __builtin_amdgcn_perm(0, v[i >> 1], i & 1 ? 0x0C030C02u : 0x0C010C00u) | ((both[i >> 2] << (15 - 2 * (i & 3))) & 0x80008000u);
      const h2 q = __builtin_bit_cast(h2, w);
      const float f0 = __builtin_fmaf((float)q.x, d, 0.0f), f1 = __builtin_fmaf((float)q.y, d, 0.0f);   // (multiply-adds: a product alone is not taken from halves)
      if constexpr (std::is_same_v<V2, h2>) o[i] = __builtin_bit_cast(uint32_t, (h2){(_Float16)f0, (_Float16)f1});
      else o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){f0, f1}, V2));
    }
  }
}

}  // namespace gguf
