// How the GEMMs of dense_core.h and mmq_f_core.h hand out their tiles, and how partial tiles become results.
#pragma once
#include "gguf_common.h"

namespace gguf {

// Tiles of `mt` rows of X by 128 weight rows, K in units of 256 values.  `whole` tiles get a workgroup each; the units of the
// `shared` tiles behind them, one tile after the other, are dealt to `workers` workgroups in runs of `per` (at most a
// tile's), which leave fp32 partial tiles, two each at most.
struct TilePlan {
  int mt, whole, shared, workers, per;
  int64_t partial_bytes() const { return (int64_t)workers * 2 * mt * 128 * 4; }
};

struct TileRuns {
  int M, N, units;             // rows of X, weight rows, units per row
  int tiles_m, whole, shared, workers, per;
  int64_t ldy;
  int quads;                   // rows of Y take stores of four values
};

template <typename T>
static TileRuns tile_runs(const TilePlan& p, int M, int N, int units, const void* Y, int64_t ldy) {
  return {M, N, units, (M + p.mt - 1) / p.mt, p.whole, p.shared, p.workers, p.per, ldy, ldy % 4 == 0 && (uintptr_t)Y % (4 * sizeof(T)) == 0};
}

typedef float tile_f4v __attribute__((ext_vector_type(4)));

// The units of this workgroup, [first, end) counted over all tiles: whole tiles in runs per XCD, then equal runs of units
// of the shared tiles.  worker: its number among the workers, negative for a whole tile.
struct TileWork { int first, end, worker; };
__device__ __forceinline__ TileWork tile_work(const TileRuns& a) {
  int wg = blockIdx.x;
  const int whole8 = a.whole & ~7;
  if (wg < whole8) wg = (wg & 7) * (whole8 >> 3) + (wg >> 3);
  int sw = wg - a.whole;
  const int shared8 = a.workers & ~7;
  if (sw >= 0 && sw < shared8 && (a.whole & 7) == 0) sw = (sw & 7) * (shared8 >> 3) + (sw >> 3);
  const int unit = sw < 0 ? wg * a.units : a.whole * a.units + sw * a.per;
  return {unit, sw < 0 ? unit + a.units : min((a.whole + a.shared) * a.units, unit + a.per), sw};
}

// four neighbouring results of a row
template <typename T>
__device__ __forceinline__ void tile_store(tile_f4v v, int m, int n, T* Y, const T* bias, const TileRuns& a) {
  if (m >= a.M) return;
  T* const y = Y + (int64_t)m * a.ldy + n;
  if (a.quads && n + 3 < a.N) {
    struct alignas(4 * sizeof(T)) { T v[4]; } o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o.v[e] = finish<T>(v[e], bias, n + e);
    *(decltype(o)*)y = o;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < a.N) y[e] = finish<T>(v[e], bias, n + e);
  }
}

// Y tile = T(sum of its partial tiles) in the order of K; a workgroup per wave's share of a tile, a thread per run of four.
// WM x WN waves of TM x TN tiles of 32 x 32; a partial tile lies in the order of the registers, [wave][tile][run][lane] of four.
template <int WM, int WN, int TM, int TN, typename T>
__global__ __launch_bounds__(256) void tile_reduce_kernel(const float* __restrict__ partial, T* __restrict__ Y, const T* __restrict__ bias, TileRuns a) {
  constexpr int M_T = 32 * WM * TM, N_T = 32 * WN * TN;
  const int t = blockIdx.x, tile = a.whole + t, sub = blockIdx.y, q = threadIdx.x >> 6, lane = threadIdx.x & 63;   // sub: (wave, tile of the wave)
  const int wave = sub / (TN * TM), i = sub / TM % TN, k = sub % TM, wm = wave / WN, wn = wave % WN;
  const int m = (tile % a.tiles_m) * M_T + 32 * (TM * wm + k) + (lane & 31), n = (tile / a.tiles_m) * N_T + 32 * (TN * wn + i) + 8 * q + 4 * (lane >> 5);
  // the workers whose runs of units meet this tile; a worker's second partial tile is the tile it entered last
  const int first = t * a.units / a.per, last = ((t + 1) * a.units - 1) / a.per;
  if ((first == last && t * a.units == first * a.per && a.per == a.units) || m >= a.M) return;   // (stored whole, or padding)
  // (eight partial tiles asked for at a time: one after the other, sixteen of them take longer than the product did)
  tile_f4v v = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int w0 = first; w0 <= last; w0 += 8) {
    tile_f4v p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int w = min(w0 + i, last);
      p[i] = *(const tile_f4v*)(partial + (int64_t)(2 * w + t - w * a.per / a.units) * (M_T * N_T) + ((sub * 4 + q) * 64 + lane) * 4);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (w0 + i <= last) v += p[i];
  }
  tile_store(v, m, n, Y, bias, a);
}

}  // namespace gguf
