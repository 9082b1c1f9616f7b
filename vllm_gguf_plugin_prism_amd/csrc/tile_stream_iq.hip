// Codebook formats on the streaming tile kernel (tile_stream_core.h), for the GEMV operator's rows: IQ2_XXS, IQ2_XS, IQ2_S, IQ3_XXS,
// IQ3_S.  A lane's eight codes of a block are one entry of the eight-value grids, or two of the four-value ones, and one sign
// byte: two or three reads from the GEMV kernels' tables, which lie behind the rings in LDS.
#include "tile_stream_core.h"
#include "mmvq_core.h"

namespace gguf {

// FMT: the GEMV's format, for its tables; a block's index (or both) and signs are kept in one register
template <class FMT, int SCALED>
struct TIQ {
  static constexpr int PB = FMT::BS, G = SCALED, OFF = 0, TABLE = FMT::TABLE_BYTES;
  static constexpr bool KQ = true, HALVES = false;
  const char* tab;
  uint32_t at8[8];                                          // the lane's index and signs of every block
  uint2 sc;
  uint32_t d;
  static __device__ __forceinline__ void tables(char* t) { FMT::init_tables(t); }
  __device__ __forceinline__ void ready() {}
  __device__ __forceinline__ uint32_t scale8(int b) const { return ((b < 4 ? sc.x : sc.y) >> (8 * (b & 3))) & 0xFF; }
};

__device__ __forceinline__ uint2 ts_signed(const uint2 mag, const char* signs, uint32_t s) {
  const uint2 m = ((const uint2*)signs)[s];
  return make_uint2(neg_bytes(mag.x, m.x), neg_bytes(mag.y, m.y));
}

struct TIQ2_XXS : TIQ<FmtIQ2_XXS, 32> {
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    d = lds_h(p, at);
    uint32_t s[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint2 v = lds_cut8(p, at + 2 + 8 * b);
      at8[b] = ((v.x >> (8 * g)) & 0xFF) | ((v.y >> (7 * g)) & 127) << 16;
      s[b] = v.y >> 28;
    }
    sc = make_uint2(s[0] | s[1] << 8 | s[2] << 16 | s[3] << 24, s[4] | s[5] << 8 | s[6] << 16 | s[7] << 24);
  }
  __device__ __forceinline__ void scales(float (&dw)[8]) const {
#pragma unroll
    for (int b = 0; b < 8; ++b) dw[b] = 0.25f * half_bits(d) * (0.5f + (float)scale8(b));
  }
  __device__ __forceinline__ uint2 codes(int b, int) const { return ts_signed(((const uint2*)tab)[at8[b] & 0xFFFF], tab + 256 * 8, at8[b] >> 16); }
};

// a scale per sixteen values: the nibbles of a block's byte
template <class FMT>
struct TIQ2 : TIQ<FMT, 16> {
  __device__ __forceinline__ void scales(float (&dw)[16]) const {
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint32_t s = this->scale8(b);
      dw[2 * b] = 0.25f * half_bits(this->d) * (0.5f + (float)(s & 15));
      dw[2 * b + 1] = 0.25f * half_bits(this->d) * (0.5f + (float)(s >> 4));
    }
  }
};
struct TIQ2_XS : TIQ2<FmtIQ2_XS> {
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    d = lds_h(p, at);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint32_t q = lds_h(p, at + 2 + 8 * b + 2 * g);
      at8[b] = (q & 511) | (q >> 9) << 16;
    }
    sc = lds_cut8(p, at + 66);
  }
  __device__ __forceinline__ uint2 codes(int b, int) const { return ts_signed(((const uint2*)tab)[at8[b] & 0xFFFF], tab + 512 * 8, at8[b] >> 16); }
};
struct TIQ2_S : TIQ2<FmtIQ2_S> {
  static constexpr bool ONE_GROUP = true;
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    d = lds_h(p, at);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint32_t q = *(const uint8_t*)(p + at + 2 + 4 * b + g), s = *(const uint8_t*)(p + at + 34 + 4 * b + g), h = *(const uint8_t*)(p + at + 66 + b);
      at8[b] = q | ((h << (8 - 2 * g)) & 0x300) | s << 16;
    }
    sc = lds_cut8(p, at + 74);
  }
  __device__ __forceinline__ uint2 codes(int b, int) const { return ts_signed(((const uint2*)tab)[at8[b] & 0xFFFF], tab + 1024 * 8, at8[b] >> 16); }
};

struct TIQ3_XXS : TIQ<FmtIQ3_XXS, 32> {
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    d = lds_h(p, at);
    uint32_t s[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint32_t aux = lds_h(p, at + 66 + 4 * b) | lds_h(p, at + 68 + 4 * b) << 16;
      at8[b] = lds_h(p, at + 2 + 8 * b + 2 * g) | ((aux >> (7 * g)) & 127) << 16;
      s[b] = aux >> 28;
    }
    sc = make_uint2(s[0] | s[1] << 8 | s[2] << 16 | s[3] << 24, s[4] | s[5] << 8 | s[6] << 16 | s[7] << 24);
  }
  __device__ __forceinline__ void scales(float (&dw)[8]) const {
#pragma unroll
    for (int b = 0; b < 8; ++b) dw[b] = 0.5f * half_bits(d) * (0.5f + (float)scale8(b));
  }
  __device__ __forceinline__ uint2 codes(int b, int) const {
    const uint32_t* const grid = (const uint32_t*)tab;
    return ts_signed(make_uint2(grid[at8[b] & 0xFF], grid[(at8[b] >> 8) & 0xFF]), tab + 256 * 4, at8[b] >> 16);
  }
};
struct TIQ3_S : TIQ<FmtIQ3_S, 32> {
  __device__ __forceinline__ void read(const char* p, uint32_t at, int g) {
    d = lds_h(p, at);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint32_t q = lds_h(p, at + 2 + 8 * b + 2 * g), h = *(const uint8_t*)(p + at + 66 + b), s = *(const uint8_t*)(p + at + 74 + 4 * b + g);
      // two indexes of nine bits, the signs
      at8[b] = (q & 0xFF) | ((h << (8 - 2 * g)) & 256) | ((q >> 8) | ((h << (7 - 2 * g)) & 256)) << 9 | s << 18;
    }
    sc.x = lds_h(p, at + 106) | lds_h(p, at + 108) << 16;
  }
  __device__ __forceinline__ void scales(float (&dw)[8]) const {
#pragma unroll
    for (int b = 0; b < 8; ++b) dw[b] = 0.5f * half_bits(d) * (0.5f + (float)((sc.x >> (4 * b)) & 15));
  }
  __device__ __forceinline__ uint2 codes(int b, int) const {
    const uint32_t* const grid = (const uint32_t*)tab;
    return ts_signed(make_uint2(grid[at8[b] & 511], grid[(at8[b] >> 9) & 511]), tab + 512 * 4, at8[b] >> 18);
  }
};

int ts_iq2_xxs(const TsCall& c, hipStream_t s) { return ts_dense_run<TIQ2_XXS>(c, s); }
int ts_iq2_xs(const TsCall& c, hipStream_t s) { return ts_dense_run<TIQ2_XS>(c, s); }
int ts_iq2_s(const TsCall& c, hipStream_t s) { return ts_dense_run<TIQ2_S>(c, s); }
int ts_iq3_xxs(const TsCall& c, hipStream_t s) { return ts_dense_run<TIQ3_XXS>(c, s); }
int ts_iq3_s(const TsCall& c, hipStream_t s) { return ts_dense_run<TIQ3_S>(c, s); }
}  // namespace gguf
