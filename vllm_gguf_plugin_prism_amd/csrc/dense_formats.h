// Codebook formats for the GEMM on the matrix unit (dense_core.h): sixteen neighbouring weights as signed bytes and one scale.
//
// Every weight of these formats is a scale of at most 16 significant bits times a whole number of at most eight (IQ1: an
// eighth of one), so the fp32 product is exact and rounding it once gives the value of the dequantize kernels.
//   Raw    what sixteen weights need of their block, in registers;  fetch(blk, ib, h): values 16 h .. 16 h + 15 of sub-block ib
//   Entry  an entry of the format's table in LDS (TABLE of them, 0: none);  entry(i) forms it from the 16-bit code word
//   decode the bytes, v[0] holding the first four, and the scale
#pragma once
#include "gguf_common.h"
#include "grid_codes.h"

namespace gguf {

// bytes g of four magnitudes, negated where the low four bits of s are set
__device__ __forceinline__ uint32_t signed4(uint32_t g, uint32_t s) {
  const uint32_t m = ((s & 15u) * 0x204081u) & 0x01010101u;   // bit i -> bit 8 i
  return (g ^ ((m << 8) - m)) + m;
}
__device__ __forceinline__ uint32_t parity8(uint32_t s7) { return s7 | ((__builtin_popcount(s7) & 1) << 7); }   // the eighth sign makes them even

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

// four codes, one per byte, through the table of the non-linear 4-bit formats
__device__ __forceinline__ uint32_t nonlinear4(uint32_t idx) {
  constexpr uint32_t T0 = 0xBFAD9881u, T1 = 0xF6EADDCFu, T2 = 0x26190D01u, T3 = 0x71594535u;   // -127 -104 ... 89 113
  const uint32_t sel = idx & 0x07070707u, m8 = (idx >> 3) & 0x01010101u, m = (m8 << 8) - m8;
  const uint32_t lo = __builtin_amdgcn_perm(T1, T0, sel), hi = __builtin_amdgcn_perm(T3, T2, sel);
  return (hi & m) | (lo & ~m);
}

struct DIQ4_XS : NoTable {
  static constexpr int BS = 136, QK = 256;
  struct Raw { uint2 hd; uint4 q; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int) { return {ld<uint2>(blk), ld<uint4>(blk + 8 + 16 * ib)}; }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry*, int ib, int h, uint32_t (&v)[4]) {
    const int ls = (int)(((r.hd.y >> (4 * ib)) & 15u) | (((r.hd.x >> (16 + 2 * ib)) & 3u) << 4));
    const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = nonlinear4((q[i] >> (4 * h)) & 0x0F0F0F0Fu);
    return (float)__builtin_bit_cast(_Float16, (uint16_t)r.hd.x) * (float)(ls - 32);
  }
};

struct DIQ4_NL : NoTable {
  static constexpr int BS = 18, QK = 32;
  struct Raw { uint16_t d; uint4 q; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int, int) { return {ld<uint16_t>(blk), ld<uint4>(blk + 2)}; }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry*, int, int h, uint32_t (&v)[4]) {
    const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = nonlinear4((q[i] >> (4 * h)) & 0x0F0F0F0Fu);
    return (float)__builtin_bit_cast(_Float16, r.d);
  }
};

struct DIQ2_XXS {
  static constexpr int BS = 66, QK = 256, TABLE = 256;
  typedef uint2 Entry;
  static __device__ __forceinline__ Entry entry(int i) { return entry2(k_iq2xxs_grid_codes[i]); }
  struct Raw { uint16_t d; uint2 q; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int) { return {ld<uint16_t>(blk), ld<uint2>(blk + 2 + 8 * ib)}; }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4]) {
    const uint32_t q = r.q.x >> (16 * h), s = r.q.y >> (14 * h), s0 = parity8(s & 127u), s1 = parity8((s >> 7) & 127u);
    const Entry a = t[q & 255u], b = t[(q >> 8) & 255u];
    v[0] = signed4(a.x, s0); v[1] = signed4(a.y, s0 >> 4); v[2] = signed4(b.x, s1); v[3] = signed4(b.y, s1 >> 4);
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)(r.q.y >> 28)) * 0.25f;
  }
};

struct DIQ2_XS {
  static constexpr int BS = 74, QK = 256, TABLE = 512;
  typedef uint2 Entry;
  static __device__ __forceinline__ Entry entry(int i) { return entry2(k_iq2xs_grid_codes[i]); }
  struct Raw { uint16_t d; uint32_t q; uint8_t sc; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int h) {
    return {ld<uint16_t>(blk), ld<uint32_t>(blk + 2 + 8 * ib + 4 * h), blk[66 + ib]};
  }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4]) {
    const uint32_t s0 = parity8((r.q >> 9) & 127u), s1 = parity8(r.q >> 25);
    const Entry a = t[r.q & 511u], b = t[(r.q >> 16) & 511u];
    v[0] = signed4(a.x, s0); v[1] = signed4(a.y, s0 >> 4); v[2] = signed4(b.x, s1); v[3] = signed4(b.y, s1 >> 4);
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)((r.sc >> (4 * h)) & 15)) * 0.25f;
  }
};

struct DIQ2_S {
  static constexpr int BS = 82, QK = 256, TABLE = 1024;
  typedef uint2 Entry;
  static __device__ __forceinline__ Entry entry(int i) { return entry2(k_iq2s_grid_codes[i]); }
  struct Raw { uint16_t d, q, s; uint8_t qh, sc; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int h) {
    return {ld<uint16_t>(blk), ld<uint16_t>(blk + 2 + 4 * ib + 2 * h), ld<uint16_t>(blk + 34 + 4 * ib + 2 * h), blk[66 + ib], blk[74 + ib]};
  }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4]) {
    const uint32_t qh = (uint32_t)r.qh >> (4 * h), s = r.s;   // two bits for each group of eight
    const Entry a = t[(r.q & 255u) | (qh & 3u) << 8], b = t[(r.q >> 8) | (qh & 12u) << 6];
    v[0] = signed4(a.x, s); v[1] = signed4(a.y, s >> 4); v[2] = signed4(b.x, s >> 8); v[3] = signed4(b.y, s >> 12);
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)((r.sc >> (4 * h)) & 15)) * 0.25f;
  }
};

struct DIQ3_XXS {
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
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4]) {
    const uint32_t s = r.aux >> (14 * h), s0 = parity8(s & 127u), s1 = parity8((s >> 7) & 127u);
    v[0] = signed4(t[r.q & 255u], s0); v[1] = signed4(t[(r.q >> 8) & 255u], s0 >> 4);
    v[2] = signed4(t[(r.q >> 16) & 255u], s1); v[3] = signed4(t[r.q >> 24], s1 >> 4);
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)(r.aux >> 28)) * 0.5f;
  }
};

struct DIQ3_S {
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
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int ib, int h, uint32_t (&v)[4]) {
    const uint32_t qh = (uint32_t)r.qh >> (4 * h), s = r.s;   // one bit for each group of four
    v[0] = signed4(t[(r.q & 255u) | (qh & 1u) << 8], s); v[1] = signed4(t[((r.q >> 8) & 255u) | (qh & 2u) << 7], s >> 4);
    v[2] = signed4(t[((r.q >> 16) & 255u) | (qh & 4u) << 6], s >> 8); v[3] = signed4(t[(r.q >> 24) | (qh & 8u) << 5], s >> 12);
    return (float)__builtin_bit_cast(_Float16, r.d) * (0.5f + (float)((r.sc >> (4 * (ib & 1))) & 15)) * 0.5f;
  }
};

// The 1-bit formats: d (q - 1 -+ 1/8), q of {0, 1, 2}: an eighth of the whole number 8 q - 7 or 8 q - 9.
struct IQ1Table {
  static constexpr int TABLE = 2048;
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
    v0 = (a.x - k) ^ 0x80808080u;
    v1 = (a.y - k) ^ 0x80808080u;
  }
};

struct DIQ1_S : IQ1Table {
  static constexpr int BS = 50, QK = 256;
  struct Raw { uint16_t d, q, qh; };
  static __device__ __forceinline__ Raw fetch(const uint8_t* blk, int ib, int h) {
    return {ld<uint16_t>(blk), ld<uint16_t>(blk + 2 + 4 * ib + 2 * h), ld<uint16_t>(blk + 34 + 2 * ib)};
  }
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int, int h, uint32_t (&v)[4]) {
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
  static __device__ __forceinline__ float decode(const Raw& r, const Entry* t, int ib, int h, uint32_t (&v)[4]) {
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

}  // namespace gguf
