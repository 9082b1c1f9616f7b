// Packed formats as the walking tile kernel (tile_walk_core.h) reads them: a *panel* is 256 values of K of one weight row, PB
// contiguous bytes that a wave has fetched into LDS.  A lane is (row = lane % 32, half = lane / 32) of v_mfma_i32_32x32x32_i8 and
// supplies, of every block of 32 values, the sixteen codes k = 16 half .. 16 half + 15 of its row as signed bytes.
//   CUT      panels may begin anywhere, `at` bytes into a 16-byte piece (even); else all of them begin on one
//   KQ       the panel is one super-block; else it is eight 32-value blocks and a row may end inside it
//   OFF      MINS: -dmin * sum over the blocks of offsets() * block sum of X; EIGHTS: the block's scale on the products less 8 times the block sum
//   read()   takes the lane's bytes into registers (so that the LDS slot can be filled again); scale_to() leaves the scales for the lanes that
//            hold the results: [8][32] block scales and, of MINS, [32] -dmin
//   limit()  the panel has only so many blocks; what lies behind them need not be a number (formats of 32-value blocks)
#pragma once
#include "tile_wide_formats.h"

namespace gguf {

enum WalkOffset { NO_OFFSET, MINS, EIGHTS };

template <bool C>
struct KQ4_K : WQ4_KT<C> {
  static constexpr bool KQ = true;
  static constexpr int OFF = MINS;
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
  static constexpr bool KQ = false;
  static constexpr int OFF = NO_OFFSET;
  using W32<34, C>::q;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int half) { this->read_blocks(p, at, 16 * half); }
  __device__ __forceinline__ v4i codes(int b, int) const { return (v4i){(int)q[b].x, (int)q[b].y, (int)q[b].z, (int)q[b].w}; }
};

// values 0..15 of a block are the low nibbles of its 16 bytes, 16..31 the high ones; d (q - 8), the 8 on the block sum
template <bool C>
struct KQ4_0 : W32<18, C> {
  static constexpr bool KQ = false;
  static constexpr int OFF = EIGHTS;
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
  static constexpr bool KQ = false, CUT = C;
  static constexpr int OFF = NO_OFFSET;
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

}  // namespace gguf
