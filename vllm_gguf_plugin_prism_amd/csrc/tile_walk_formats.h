// Packed formats as the walking tile kernel (tile_walk_core.h) reads them: a *panel* is 256 values of K of one weight row, PB
// contiguous bytes that a wave has fetched into LDS.  A lane is (row = lane % 32, half = lane / 32) of v_mfma_i32_32x32x32_i8 and
// supplies, of every block of 32 values, the sixteen codes k = 16 half .. 16 half + 15 of its row as signed bytes.
//   CUT      panels may begin anywhere, `at` bytes into a 16-byte piece (even); else all of them begin on one
//   KQ       the panel is one super-block; else it is eight 32-value blocks and a row may end inside it
//   OFF      MINS: -dmin * sum over the blocks of offsets() * block sum of X; EIGHTS: the block's scale on the products less 8 times the block sum
//   read()   takes the lane's bytes into registers (so that the LDS slot can be filled again); scale_to() leaves the scales for the lanes that
//            hold the results: [8][32] block scales ([16][32] with G = 16) and, of MINS, [32] -dmin
//   G        values per weight scale: 32, or 16 (v_mfma_i32_32x32x16_i8 twice per block: the lane's codes of a group are k = 8 half .. 8 half + 7 of it)
//   TALL     the most tiles of 32 rows that a workgroup has (walk_plan)
//   WHOLE    the integer scales are in the codes, and the panel has one scale per row: [32] scales
//   limit()  the panel has only so many blocks; what lies behind them need not be a number (formats of 32-value blocks)
#pragma once
#include "tile_wide_formats.h"

namespace gguf {

enum WalkOffset { NO_OFFSET, MINS, EIGHTS };

template <bool C>
struct KQ4_K : WQ4_KT<C> {
  static constexpr bool KQ = true, WHOLE = false;
  static constexpr int OFF = MINS, G = 32, TALL = 4;
  using WQ4_KT<C>::h;
  using WQ4_KT<C>::q;
  __device__ __forceinline__ void scale_to(float* to, int row, int half) const {
    const uint32_t mine = half ? (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u) : h.y & 0x3F3F3F3Fu;
    const float d = half_bits(h.x & 0xFFFF);
#pragma unroll
    for (int i = 0; i < 4; ++i) to[32 * (4 * half + i) + row] = d * (float)((mine >> (8 * i)) & 0xFF);
    to[256 + row] = -half_bits(h.x >> 16);
  }
  __device__ __forceinline__ v4i codes(int b, int) const {
    v4i o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (int)((word(q[b >> 1], i) >> (4 * (b & 1))) & 0x0F0F0F0Fu);
    return o;
  }
};

template <bool C>
struct KQ5_K : KQ4_K<C> {   // Q4_K with a fifth bit, bit b of qh[k] for block b
  static constexpr int PB = 176;
  using KQ4_K<C>::h;
  using KQ4_K<C>::q;
  uint4 qh;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) {
    h = this->piece(p, at);
    qh = this->piece(p, at + 16 + 16 * half);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = this->piece(p, at + 48 + 32 * i + 16 * half);
  }
  __device__ __forceinline__ v4i codes(int b, int) const {
    v4i o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t a = word(q[b >> 1], i), t = word(qh, i);
      o[i] = (int)(((b & 1 ? a >> 4 : a) & 0x0F0F0F0Fu) | ((b <= 4 ? t << (4 - b) : t >> (b - 4)) & 0x10101010u));
    }
    return o;
  }
};

template <bool C>
struct KQ8_0 : W32<34, C> {
  static constexpr bool KQ = false, WHOLE = false;
  static constexpr int OFF = NO_OFFSET, G = 32, TALL = C ? 2 : 4;
  using W32<34, C>::q;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) { this->read_blocks(p, at, 16 * half); }
  __device__ __forceinline__ v4i codes(int b, int) const { return (v4i){(int)q[b].x, (int)q[b].y, (int)q[b].z, (int)q[b].w}; }
};

// values 0..15 of a block are the low nibbles of its 16 bytes, 16..31 the high ones; d (q - 8), the 8 on the block sum
template <bool C>
struct KQ4_0 : W32<18, C> {
  static constexpr bool KQ = false, WHOLE = false;
  static constexpr int OFF = EIGHTS, G = 32, TALL = 4;
  using W32<18, C>::q;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int) { this->read_blocks(p, at, 0); }
  __device__ __forceinline__ v4i codes(int b, int half) const {
    v4i o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (int)((word(q[b], i) >> (4 * half)) & 0x0F0F0F0Fu);
    return o;
  }
};

// the same with a fifth bit, of value k bit k of the word in front of the nibbles; the 16 off the code
template <bool C>
struct KQ5_0 {
  static constexpr int PB = 176;
  static constexpr bool KQ = false, CUT = C, WHOLE = false;
  static constexpr int OFF = NO_OFFSET, G = 32, TALL = 4;
  uint4 q[8];
  uint32_t d[4], qh[4];
  __device__ __forceinline__ void limit(int left) {
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = 2 * i + 1 < left ? d[i] : 2 * i < left ? d[i] & 0xFFFFu : 0u;
  }
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) {
    if (!C) at = 0;
#pragma unroll
    for (int b = 0; b < 8; ++b) q[b] = lds_cut16(p, at + 22 * b + 6);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      d[i] = lds_h(p, at + 44 * i) | lds_h(p, at + 44 * i + 22) << 16;
      qh[i] = lds_h(p, at + 44 * i + 2 + 2 * half) | lds_h(p, at + 44 * i + 24 + 2 * half) << 16;
    }
  }
  __device__ __forceinline__ void scale_to(float* to, int row, int half) const {
#pragma unroll
    for (int i = 0; i < 4; ++i) to[32 * (4 * half + i) + row] = half_bits(((half ? d[2 + (i >> 1)] : d[i >> 1]) >> (16 * (i & 1))) & 0xFFFF);
  }
  __device__ __forceinline__ v4i codes(int b, int half) const {
    v4i o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t v = (word(q[b], i) >> (4 * half)) & 0x0F0F0F0Fu;
      // the bits inverted, 16 in four bytes; where one is set sixteen comes off, the upper nibble all ones
      const uint32_t t = fifth_bits(~qh[b >> 1] >> (16 * (b & 1)), i);
      o[i] = (int)(v | ((t << 4) - t));
    }
    return o;
  }
};

// Block b = 4 n + t: low nibbles (t < 2) or high ones of ql[64 n + 32 (t % 2) ..], bits 2 t of qh[32 n ..]; a scale per 16 values.  The code less 32 lies in
// the top six bits of the byte (four times the value), and the scale is a quarter.
struct KQ6_K {
  static constexpr int PB = 210, OFF = NO_OFFSET, G = 16, TALL = 3;
  static constexpr bool KQ = true, CUT = true, WHOLE = false;
  uint2 l[4][2], hi[2][2];                                  // of the lane's eight values of a block's lower and upper half
  uint2 sc;                                                 // the scales of half the blocks
  uint32_t d;
  __device__ __forceinline__ void limit(int) {}
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int g = 0; g < 2; ++g) l[i][g] = lds_cut8(p, at + 32 * i + 16 * g + 8 * half);
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        hi[n][g] = lds_cut8(p, at + 128 + 32 * n + 16 * g + 8 * half);
        hi[n][g].x ^= 0xAAAAAAAAu;                          // the top bit of every two-bit field
        hi[n][g].y ^= 0xAAAAAAAAu;
      }
    sc = lds_cut8(p, at + 192 + 8 * half);
    d = lds_h(p, at + 208);
  }
  __device__ __forceinline__ void scale_to(float* to, int row, int half) const {
    const float df = 0.25f * half_bits(d);
#pragma unroll
    for (int i = 0; i < 8; ++i) to[32 * (8 * half + i) + row] = df * (float)(int8_t)(((i < 4 ? sc.x : sc.y) >> (8 * (i & 3))) & 0xFF);
  }
  static __device__ __forceinline__ uint32_t code4(uint32_t a, uint32_t u, int t) {
    return ((t < 2 ? a << 2 : a >> 2) & 0x3C3C3C3Cu) | ((u << (6 - 2 * t)) & 0xC0C0C0C0u);
  }
  __device__ __forceinline__ long codes(int b, int g) const {
    const int n = b >> 2, t = b & 3;
    const uint2 a = l[2 * n + (t & 1)][g], u = hi[n][g];
    return (long)((uint64_t)code4(a.y, u.y, t) << 32 | code4(a.x, u.x, t));
  }
};

// Codes of 3 bits less 4 times a signed 6-bit scale per 16 values.  Of the other sign it is a whole number of eight bits, -128 .. 124, one of eight for a scale: a byte permute
// takes them from two registers.  Block b = 4 n + t: bits 2 t of qs[32 n ..], the third bit, of the other sign, bit b of hmask[k]; scale 2 b + half: four
// bits of the first eight bytes, two of the last four.
struct KQ3_K {
  static constexpr int PB = 110, OFF = NO_OFFSET, G = 32, TALL = 4;
  static constexpr bool KQ = true, CUT = true, WHOLE = true;
  uint4 q[2], hm;
  uint32_t sc[3], d;
  __device__ __forceinline__ void limit(int) {}
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) {
    hm = lds_cut16(p, at + 16 * half);
#pragma unroll
    for (int n = 0; n < 2; ++n) q[n] = lds_cut16(p, at + 32 + 32 * n + 16 * half);
    const uint2 lo = lds_cut8(p, at + 96), hi = lds_cut8(p, at + 102);   // (bytes 96 .. 103, 102 .. 109)
    const int up = 8 * half;                                // the lane's scales are the even bytes
    sc[0] = lo.x >> up;
    sc[1] = lo.y >> up;
    sc[2] = __builtin_amdgcn_alignbit(hi.y, hi.x, 16) >> up;
    d = hi.y >> 16;
  }
  __device__ __forceinline__ void scale_to(float* to, int row, int) const { to[row] = -half_bits(d); }
  __device__ __forceinline__ v4i codes(int b, int) const {
    const int n = b >> 2, t = b & 3;
    const uint32_t lo = ((t < 2 ? sc[0] : sc[1]) >> (16 * (t & 1) + 4 * n)) & 15u, hi = (sc[2] >> (16 * (t & 1) + 4 * n + 2 * (t >> 1))) & 3u;
    // the products with 4, 3, 2, 1 and 0, -1, -2, -3 (codes 0 .. 7), a byte each
    const int s = (int)(lo | hi << 4) - 32;
    const auto byte = [&](int f) { return (uint32_t)(f * s) & 0xFFu; };
    const uint32_t up = byte(4) | byte(3) << 8 | byte(2) << 16 | byte(1) << 24, down = byte(-1) << 8 | byte(-2) << 16 | byte(-3) << 24;
    v4i o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t a = word(q[n], i) >> (2 * t), m = word(hm, i);
      o[i] = (int)__builtin_amdgcn_perm(down, up, (a & 0x03030303u) | ((b <= 2 ? m << (2 - b) : m >> (b - 2)) & 0x04040404u));
    }
    return o;
  }
};

}  // namespace gguf
