// Packed formats as the wide tile kernel (tile_wide_core.h) reads them: one *panel* is 256 values of K of one weight row, PB
// contiguous bytes that a wave has fetched into LDS.  A lane is (row = lane % 32, half = lane / 32) of v_mfma_f32_32x32x16_f16
// and supplies, of every block of 32 values, the sixteen k = 16 half .. 16 half + 15 of its row: two operands of eight
// halves, whole numbers, of four neighbours in the order 0, 2, 1, 3.
//   KIND     SUPER: super-blocks, the integer scale of a block (or of 16 values) is in the operand, d and -dmin on the sum of the
//            super-block; BLOCK: the block's scale is on every block's sum; HALVES: on every block's sum half(d * d8), and
//            half(m * s8) added, the products rounded to half precision as the reference's __hmul2 leaves them
//            (vecdotq.cuh:71-93, 179-198)
//   CUT      panels may begin anywhere, `at` bytes into a 16-byte piece (even); else all of them begin on one
//   PLANES   operands per weight;  OFF: an offset term, -dmin * sum over the blocks of offsets() * block sum;  FACTOR: one of BLOCK, d *
//            FACTOR * block sum, which joins the block's sum before d does (a sum of its own over the panel cancels against the product's in
//            fp32: activations of one sign, results 7.7e-7 from 64 bits instead of 1e-7)
//   MIN16    the offset is a min per 16 values, min16(), times d8 * the sum of those quants
//   read()   takes the lane's bytes into registers (so that the LDS slot can be filled again); scale_to() leaves scales for
//            the lanes that hold the results: [32] d, [32] -dmin; [8][32] block scales; [8][32] d, [8][32] m as halves
//   limit()  the panel has only so many blocks; what lies behind them need not be a number (formats of 32-value blocks)
#pragma once
#include "tile_stream_formats.h"

namespace gguf {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// Bytes 0 and 2 (or 1 and 3) of v, two whole numbers, as the halves 1024 + x: the bytes below 0x64.
template <int ODD> __device__ __forceinline__ f16x2 wide_bytes(uint32_t v) {
  return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, v, ODD ? 0x04030401u : 0x04020400u));
}
// The same for the bits of `mask` in the low byte of each half.  (The mask lies in a register, so that the two operations are one
// instruction, which takes a single scalar operand.)
__device__ __forceinline__ uint32_t in_vgpr(uint32_t v) {
  uint32_t r;
  asm("v_mov_b32 %0, %1" : "=v"(r) : "s"(v));
  return r;
}
__device__ __forceinline__ f16x2 wide_bits(uint32_t v, uint32_t mask) { return __builtin_bit_cast(f16x2, (v & mask) | 0x64006400u); }
__device__ __forceinline__ f16x2 both(float v) { return (f16x2){(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ f16x8 wide_operand(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
  return __builtin_bit_cast(f16x8, make_uint4(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, c),
                                              __builtin_bit_cast(uint32_t, d)));
}
__device__ __forceinline__ uint32_t word(const uint4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

enum WideKind { SUPER, BLOCK, HALVES };

template <bool C>
struct WQ4_KT {
  static constexpr int PB = 144, PLANES = 1, KIND = SUPER;
  static constexpr bool CUT = C, OFF = true, MIN16 = false;
  static constexpr float FACTOR = 0.0f;
  __device__ __forceinline__ void limit(int) {}
  uint4 h, q[4];
  uint32_t s[2];
  static __device__ __forceinline__ uint4 piece(const char* p, uint32_t at) { return C ? lds_cut16(p, at) : *(const uint4*)(p + at); }
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) {
    h = piece(p, at);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = piece(p, at + 16 + 32 * i + 16 * half);
  }
  __device__ __forceinline__ void scale_to(float* to, int row, int) {
    to[row] = half_bits(h.x & 0xFFFF);
    to[32 + row] = -half_bits(h.x >> 16);
    s[0] = h.y & 0x3F3F3F3Fu;
    s[1] = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
  }
  __device__ __forceinline__ uint4 offsets() const {   // the mins, eight halves
    const uint32_t m[2] = {h.z & 0x3F3F3F3Fu, ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u)};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, m[i >> 1], i & 1 ? 0x04030402u : 0x04010400u)) - both(1024.0f));
    return make_uint4(o[0], o[1], o[2], o[3]);
  }
  __device__ __forceinline__ f16x2 scale(int b) const {   // 1024 + the block's scale, twice
    const uint32_t at = b & 3;
    return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, s[b >> 2], 0x04000400u | at << 16 | at));
  }
  // (high nibbles stay where they are, sixteen times as large, and the scale is a sixteenth: all exact)
  __device__ __forceinline__ void operand(int b, int, f16x8 (&o)[1][2]) const {
    const bool high = b & 1;
    const f16x2 sc = high ? __builtin_elementwise_fma(scale(b), both(0.0625f), both(-64.0f)) : scale(b) - both(1024.0f);
    const f16x2 n = sc * both(-1024.0f);
    const uint32_t mask = in_vgpr(high ? 0x00F000F0u : 0x000F000Fu);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t x = word(q[b >> 1], 2 * i), y = word(q[b >> 1], 2 * i + 1);
      o[0][i] = wide_operand(__builtin_elementwise_fma(wide_bits(x, mask), sc, n), __builtin_elementwise_fma(wide_bits(x >> 8, mask), sc, n),
                             __builtin_elementwise_fma(wide_bits(y, mask), sc, n), __builtin_elementwise_fma(wide_bits(y >> 8, mask), sc, n));
    }
  }
};

template <bool C>
struct WQ5_KT : WQ4_KT<C> {   // Q4_K with a fifth bit, bit b of qh[k] for block b
  static constexpr int PB = 176;
  using WQ4_KT<C>::h;
  using WQ4_KT<C>::q;
  using WQ4_KT<C>::piece;
  uint4 qh;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) {
    h = piece(p, at);
    qh = piece(p, at + 16 + 16 * half);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = piece(p, at + 48 + 32 * i + 16 * half);
  }
  __device__ __forceinline__ void operand(int b, int, f16x8 (&o)[1][2]) const {
    const f16x2 sc = this->scale(b) - both(1024.0f), n = sc * both(-1024.0f);
    const auto codes = [&](int i) {
      const uint32_t a = word(q[b >> 1], i), t = word(qh, i);
      return ((b & 1 ? a >> 4 : a) & 0x0F0F0F0Fu) | ((b <= 4 ? t << (4 - b) : t >> (b - 4)) & 0x10101010u);
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t x = codes(2 * i), y = codes(2 * i + 1);
      o[0][i] = wide_operand(__builtin_elementwise_fma(wide_bytes<0>(x), sc, n), __builtin_elementwise_fma(wide_bytes<1>(x), sc, n),
                             __builtin_elementwise_fma(wide_bytes<0>(y), sc, n), __builtin_elementwise_fma(wide_bytes<1>(y), sc, n));
    }
  }
};

// Block b = 4 n + t: low nibbles (t < 2) or high ones of ql[64 n + 32 (t % 2) ..], bits 2 t of qh[32 n ..]; a scale per 16
// values, so one for a lane and block.  (code - 32) * scale has 12 bits and a sign: two operands, the product rounded to half precision and what that leaves out.
struct WQ6_K {
  static constexpr int PB = 210, PLANES = 2, KIND = SUPER;
  static constexpr bool CUT = true, OFF = false, MIN16 = false;
  static constexpr float FACTOR = 0.0f;
  __device__ __forceinline__ void limit(int) {}
  uint4 l[4], hi[2], sc;
  uint32_t d;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) {
#pragma unroll
    for (int i = 0; i < 4; ++i) l[i] = lds_cut16(p, at + 32 * i + 16 * half);
#pragma unroll
    for (int n = 0; n < 2; ++n) hi[n] = lds_cut16(p, at + 128 + 32 * n + 16 * half);
    sc = lds_cut16(p, at + 192);
    d = lds_h(p, at + 208);
  }
  __device__ __forceinline__ void scale_to(float* to, int row, int half) {
    to[row] = half_bits(d);
    const int up = 8 * half;                                // the lane's scales are the even bytes
    sc = make_uint4(sc.x >> up, sc.y >> up, sc.z >> up, sc.w >> up);
  }
  __device__ __forceinline__ void operand(int b, int, f16x8 (&o)[2][2]) const {
    const int n = b >> 2, t = b & 3;
    // 1024 + 128 + the scale, twice
    const uint32_t c = __builtin_bit_cast(uint32_t, __builtin_amdgcn_perm(0x64646464u, word(sc, b >> 1), b & 1 ? 0x04020402u : 0x04000400u));
    const f16x2 s = __builtin_bit_cast(f16x2, c ^ 0x00800080u) - both(1152.0f);
    const auto codes = [&](int i) {
      const uint32_t a = word(l[2 * n + (t & 1)], i), u = word(hi[n], i);
      return ((t < 2 ? a : a >> 4) & 0x0F0F0F0Fu) | ((t == 0 ? u << 4 : t == 1 ? u << 2 : t == 2 ? u : u >> 2) & 0x30303030u);
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t x = codes(2 * i), y = codes(2 * i + 1);
      const f16x2 k = both(1056.0f), x0 = wide_bytes<0>(x) - k, x1 = wide_bytes<1>(x) - k, y0 = wide_bytes<0>(y) - k, y1 = wide_bytes<1>(y) - k;
      // the products rounded to half precision, and what that leaves out: -1, 0 or 1
      const f16x2 px = x0 * s, qx = x1 * s, py = y0 * s, qy = y1 * s;
      o[0][i] = wide_operand(px, qx, py, qy);
      o[1][i] = wide_operand(__builtin_elementwise_fma(x0, s, -px), __builtin_elementwise_fma(x1, s, -qx), __builtin_elementwise_fma(y0, s, -py),
                             __builtin_elementwise_fma(y1, s, -qy));
    }
  }
};

// Codes of 3 bits less 4 times a signed 6-bit scale per 16 values: one operand.  Block b = 4 n + t: bits 2 t of qs[32 n ..], the
// third bit, of the other sign, bit b of hmask[k]; scale 2 b + half: four bits of the first eight bytes, two of the last four.
struct WQ3_K {
  static constexpr int PB = 110, PLANES = 1, KIND = SUPER;
  static constexpr bool CUT = true, OFF = false, MIN16 = false;
  static constexpr float FACTOR = 0.0f;
  uint4 q[2], hm, sc;
  uint32_t d;
  __device__ __forceinline__ void limit(int) {}
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) {
    hm = lds_cut16(p, at + 16 * half);
#pragma unroll
    for (int n = 0; n < 2; ++n) q[n] = lds_cut16(p, at + 32 + 32 * n + 16 * half);
    const uint2 lo = lds_cut8(p, at + 96), hi = lds_cut8(p, at + 102);   // (bytes 96 .. 103, 102 .. 109)
    sc = make_uint4(lo.x, lo.y, __builtin_amdgcn_alignbit(hi.y, hi.x, 16), 0);
    d = hi.y >> 16;
  }
  __device__ __forceinline__ void scale_to(float* to, int row, int half) {
    to[row] = half_bits(d);
    const int up = 8 * half;                                // the lane's scales are the even bytes
    sc = make_uint4(sc.x >> up, sc.y >> up, sc.z >> up, 0);
  }
  __device__ __forceinline__ void operand(int b, int, f16x8 (&o)[1][2]) const {
    const int n = b >> 2, t = b & 3;
    const uint32_t lo = ((t < 2 ? sc.x : sc.y) >> (16 * (t & 1) + 4 * n)) & 15u, hi = (sc.z >> (16 * (t & 1) + 4 * n + 2 * (t >> 1))) & 3u;
    const f16x2 s = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, lo | hi << 4, 0x04000400u)) - both(1056.0f), k = both(1028.0f);
    const auto codes = [&](int i) {
      const uint32_t a = word(q[n], i) >> (2 * t), m = word(hm, i);
      return (a & 0x03030303u) | ((b <= 2 ? m << (2 - b) : m >> (b - 2)) & 0x04040404u);
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t x = codes(2 * i), y = codes(2 * i + 1);
      o[0][i] = wide_operand((wide_bytes<0>(x) - k) * s, (wide_bytes<1>(x) - k) * s, (wide_bytes<0>(y) - k) * s, (wide_bytes<1>(y) - k) * s);
    }
  }
};

// Codes of 2 bits, a 4-bit scale and a 4-bit min per 16 values.  Block b = 4 n + t: bits 2 t of qs[32 n ..].
struct WQ2_K {
  static constexpr int PB = 84, PLANES = 1, KIND = SUPER;
  static constexpr bool CUT = true, OFF = true, MIN16 = true;
  static constexpr float FACTOR = 0.0f;
  uint4 q[2], sc;
  uint32_t dm;
  __device__ __forceinline__ void limit(int) {}
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) {
    sc = lds_cut16(p, at);
#pragma unroll
    for (int n = 0; n < 2; ++n) q[n] = lds_cut16(p, at + 16 + 32 * n + 16 * half);
    dm = lds_h(p, at + 80) | lds_h(p, at + 82) << 16;
  }
  __device__ __forceinline__ void scale_to(float* to, int row, int half) {
    to[row] = half_bits(dm & 0xFFFF);
    to[32 + row] = -half_bits(dm >> 16);
    const int up = 8 * half;                                // the lane's scales are the even bytes
    sc = make_uint4(sc.x >> up, sc.y >> up, sc.z >> up, sc.w >> up);
  }
  __device__ __forceinline__ float min16(int b) const { return (float)((word(sc, b >> 1) >> (16 * (b & 1) + 4)) & 15u); }
  __device__ __forceinline__ void operand(int b, int, f16x8 (&o)[1][2]) const {
    const int n = b >> 2, t = b & 3;
    const uint32_t c = (word(sc, b >> 1) >> (16 * (b & 1))) & 15u;
    const f16x2 s = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, c, 0x04000400u)) - both(1024.0f), z = s * both(-1024.0f);   // (exact)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t x = (word(q[n], 2 * i) >> (2 * t)) & 0x03030303u, y = (word(q[n], 2 * i + 1) >> (2 * t)) & 0x03030303u;
      o[0][i] = wide_operand(__builtin_elementwise_fma(wide_bytes<0>(x), s, z), __builtin_elementwise_fma(wide_bytes<1>(x), s, z),
                             __builtin_elementwise_fma(wide_bytes<0>(y), s, z), __builtin_elementwise_fma(wide_bytes<1>(y), s, z));
    }
  }
};

// Eight blocks of BB bytes, an fp16 scale in front of each.
template <int BB, bool C>
struct W32 {
  static constexpr int PB = 8 * BB, PLANES = 1, KIND = BLOCK;
  static constexpr bool CUT = C, OFF = false, MIN16 = false;
  static constexpr float FACTOR = 0.0f;
  __device__ __forceinline__ void limit(int left) {
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = 2 * i + 1 < left ? d[i] : 2 * i < left ? d[i] & 0xFFFFu : 0u;
  }
  uint4 q[8];
  uint32_t d[4];                                            // the eight scales, two in a word
  // sixteen bytes from 2 + lane_at of every block (lane_at a multiple of 16; the blocks' bytes begin 2, 4, 6, 0, ... behind an
  // 8-byte word)
  __device__ __forceinline__ void read_blocks(const char* p, uint32_t at, uint32_t lane_at) {
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (C) {
        q[b] = lds_cut16(p, at + BB * b + 2 + lane_at);
        continue;
      }
      const int first = BB * b + 2, cut = first % 8;
      const uint2* const w = (const uint2*)(p + (first - cut) + lane_at);
      const uint2 a = w[0], c = w[1];
      if (cut == 0) {
        q[b] = make_uint4(a.x, a.y, c.x, c.y);
      } else {
        const uint2 e = w[2];
        const uint32_t x0 = cut >= 4 ? a.y : a.x, x1 = cut >= 4 ? c.x : a.y, x2 = cut >= 4 ? c.y : c.x, x3 = cut >= 4 ? e.x : c.y, x4 = cut >= 4 ? e.y : e.x;
        q[b] = cut == 4 ? make_uint4(x0, x1, x2, x3)
                        : make_uint4(__builtin_amdgcn_alignbit(x1, x0, 16), __builtin_amdgcn_alignbit(x2, x1, 16), __builtin_amdgcn_alignbit(x3, x2, 16),
                                     __builtin_amdgcn_alignbit(x4, x3, 16));
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = lds_h(p, (C ? at : 0u) + BB * 2 * i) | lds_h(p, (C ? at : 0u) + BB * (2 * i + 1)) << 16;
  }
  __device__ __forceinline__ void scale_to(float* to, int row, int half) {
#pragma unroll
    for (int i = 0; i < 4; ++i) to[32 * (4 * half + i) + row] = half_bits(((half ? d[2 + (i >> 1)] : d[i >> 1]) >> (16 * (i & 1))) & 0xFFFF);
  }
};

// values 0..15 of a block are the low nibbles of its 16 bytes, 16..31 the high ones; d (q - 8), the 8 on the block sum
template <bool C>
struct WQ4_0T : W32<18, C> {
  static constexpr float FACTOR = -8.0f;
  using W32<18, C>::q;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int) { this->read_blocks(p, at, 0); }
  __device__ __forceinline__ void operand(int b, int half, f16x8 (&o)[1][2]) const {
    const uint32_t mask = half ? 0x00F000F0u : 0x000F000Fu;
    const f16x2 sc = both(half ? 0.0625f : 1.0f), n = both(half ? -64.0f : -1024.0f);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t x = word(q[b], 2 * i), y = word(q[b], 2 * i + 1);
      o[0][i] = wide_operand(__builtin_elementwise_fma(wide_bits(x, mask), sc, n), __builtin_elementwise_fma(wide_bits(x >> 8, mask), sc, n),
                             __builtin_elementwise_fma(wide_bits(y, mask), sc, n), __builtin_elementwise_fma(wide_bits(y >> 8, mask), sc, n));
    }
  }
};

// a block's fifth bits, of the lane's values 4 i .. 4 i + 3, as 16 in four bytes (bits: those of its sixteen values)
__device__ __forceinline__ uint32_t fifth_bits(uint32_t bits, int i) { return __umul24((i ? bits >> (4 * i - 4) : bits << 4) & 0xF0u, 0x204081u) & 0x10101010u; }

// Q4_1, Q5_1: d q + m
template <bool FIFTH>
struct WQ45_1 {
  static constexpr int BB = FIFTH ? 24 : 20, PB = 8 * BB, PLANES = 1, KIND = HALVES;
  static constexpr bool CUT = false, OFF = false, MIN16 = false;
  static constexpr float FACTOR = 0.0f;
  uint4 q[8];
  uint32_t dm[8], qh[FIFTH ? 4 : 1];
  __device__ __forceinline__ void limit(int left) {
#pragma unroll
    for (int b = 0; b < 8; ++b) dm[b] = b < left ? dm[b] : 0u;
  }
  __device__ __forceinline__ void read(const char* p, uint32_t, int half) {
    constexpr int N = BB / 4;
    uint32_t v[8 * N];
#pragma unroll
    for (int i = 0; i < 2 * N; ++i) {
      const uint4 x = ((const uint4*)p)[i];
      v[4 * i] = x.x; v[4 * i + 1] = x.y; v[4 * i + 2] = x.z; v[4 * i + 3] = x.w;
    }
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const int i = N * b;
      dm[b] = v[i];
      q[b] = make_uint4(v[i + N - 4], v[i + N - 3], v[i + N - 2], v[i + N - 1]);
      if constexpr (FIFTH) {
        const uint32_t five = (v[i + 1] >> (16 * half)) & 0xFFFFu;
        qh[b >> 1] = b & 1 ? qh[b >> 1] | five << 16 : five;
      }
    }
  }
  __device__ __forceinline__ void scale_to(float* to, int row, int half) {
    uint16_t* const h = (uint16_t*)to;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t v = half ? dm[4 + i] : dm[i];
      h[32 * (4 * half + i) + row] = (uint16_t)(v & 0xFFFF);
      h[256 + 32 * (4 * half + i) + row] = (uint16_t)(v >> 16);
    }
  }
  __device__ __forceinline__ void operand(int b, int half, f16x8 (&o)[1][2]) const {
    const f16x2 k = both(1024.0f);
    const auto codes = [&](int i) {
      const uint32_t v = (word(q[b], i) >> (4 * half)) & 0x0F0F0F0Fu;
      if constexpr (FIFTH) return v | fifth_bits(qh[b >> 1] >> (16 * (b & 1)), i);
      else return v;
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t x = codes(2 * i), y = codes(2 * i + 1);
      o[0][i] = wide_operand(wide_bytes<0>(x) - k, wide_bytes<1>(x) - k, wide_bytes<0>(y) - k, wide_bytes<1>(y) - k);
    }
  }
};

}  // namespace gguf
