// Packed formats as the streaming tile kernel (tile_stream_core.h) reads them: one *panel* is 256 values of K of one
// weight row, `PB` contiguous bytes that a wave has fetched into LDS.  A lane is (column c = lane % 16, k group
// g = lane / 16) of v_mfma_i32_16x16x32_i8 and supplies, of every 32-value block, the eight codes k = 8 g .. 8 g + 7
// of its column.  read() takes what the lane needs of a panel into registers (so that the LDS slot can be filled
// again), the other members decode from there.
//   G        values per weight scale: 32, or 16 (two scales per block)
//   OFF      0: no offset term; 1: minus mw(block) times a block sum of the activations (the plane is the caller's choice)
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
  static constexpr bool KQ = true;
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
  static constexpr bool KQ = true;
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
  static constexpr bool KQ = true;
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
  static constexpr bool KQ = false;
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

}  // namespace gguf
