// The codebook GEMM (dense_core.h) for some tens of rows of activations: waves that walk K on their own, as in tile_walk_core.h.
//
// Tiles of 128 weight rows are too few of them there, so that K is cut into five to twelve parts: their tiles go through memory (26 MB at [5120,5120], 256 rows) and through a
// second launch, together a third of the time, and a step of 64 values waits for its fetches behind a barrier.  Here a workgroup is 32 weight rows by 32 R
// rows of X, its four or eight waves deal K among them by panels of 256 values, and the sum of their tiles is formed in LDS.
//   * A panel's packed bytes come straight to the wave's own place in LDS, the next one's while this one is decoded.
//   * A lane decodes sixteen values of one weight row, half of a block of 32, as dense_core.h does, rounded to X's type: two operands of v_mfma_f32_32x32x16.  The order of K
//     inside a block is the lanes': values 16 h .. of the block belong to half h.
//   * X is put into that order by a launch of its own (dwalk_rows_kernel: 2.3 us), so that an operand is 1 KB whose lanes follow one another, loaded straight to
//     registers, three blocks ahead (four tiles of rows: one, where the registers hold no more).
//   * DIRECT: one tile of rows, taken from X as it lies, without that launch: an instruction touches a line per row, which few enough rows allow (17 rows of [5120,5120] 11.0
//     instead of 12.6 us; 32 rows of [28672,4096] 42 instead of 33, 64 of [5120,5120] 22.5 instead of 15.7).
// Measured, us, before / now: IQ4_XS [14336,4096] 12 rows 27.6 / 17.5; [5120,5120] 17 rows 17.5 / 11.0, 128 rows 24.7 / 22, 256 rows 32.4 / 30.0 to 32.0 by machine; [4096,4096] 64 rows 19.2 / 11.6; [14336,4096] 64 rows 27.7 / 23; IQ2_XXS
// [4096,5120] 100 rows 25.8 / 15.9.  What bounds it: the decoding (60 to 75 vector instructions a block, again for every tile of rows) and the matrix instructions, which overlap
// little (tile_walk_core.h), and how the workgroups fill the chip.  Tried and no faster: seven blocks of X ahead.
// The operands are the ones of dense_kernel, in another order of the fp32 sum: 60 random products, rel-L2 of the half results against 64 bits 2.074e-4 both, results that are
// not the nearest half 0.08 % both; of 5 .. 32 rows 0.082 before and 0.074 % now, with activations of one sign 0.064 and 0.060 %.
#pragma once
#include "dense_core.h"
#include "dense_walk.h"
#include "tile_walk_core.h"

namespace gguf {

// 16-byte pieces that hold so many bytes wherever they begin (an odd number: banks)
constexpr int dwalk_ppr(int bytes) { return ((bytes + 29) / 16) | 1; }
template <class F> constexpr int dwalk_unit() { return F::QK == 256 ? F::BS : 8 * F::BS; }   // packed bytes of 256 values
// the format's table, two panels per wave; the waves' tiles in the end
template <class F, int R, int NW> constexpr size_t dwalk_lds() {
  const size_t table = F::TABLE * sizeof(typename F::Entry), place = (size_t)NW * 2 * 512 * dwalk_ppr(dwalk_unit<F>()) + 16;
  return table + (place > (size_t)NW * R * 4096 ? place : (size_t)NW * R * 4096);
}

template <class F, int R, int NW, bool DIRECT, typename T>
__global__ __launch_bounds__(64 * NW, 2) void dense_walk_kernel(const uint8_t* __restrict__ W, const char* __restrict__ X, GGUF_WALK_HEAD, T* __restrict__ Y, WalkEnd end) {
  const WalkArgs a = GGUF_WALK_ARGS;
  constexpr int UB = dwalk_unit<F>(), PPR = dwalk_ppr(UB), SLOT = 512 * PPR, NI = (32 * PPR + 63) / 64;   // (the last fetch of a panel: lanes 0 .. 31)
  typedef DenseType<T> D;
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, half = lane >> 5;
  // ---- which rows and columns: as tile_walk_kernel
  const int local = blockIdx.x >> 3, tile = (blockIdx.x & 7) * a.run + local;
  if (local >= a.run || tile >= a.tiles) return;
  const int bnd = a.band_tiles == 1 ? tile : (int)__umulhi((uint32_t)tile, a.all_inv), in = tile - bnd * a.band_tiles;
  const bool last = (bnd + 1) * a.band_tiles >= a.tiles;    // (whose row blocks may be fewer)
  const int rows = last ? a.last_band : a.band, col = rows == 1 ? in : (int)__umulhi((uint32_t)in, last ? a.last_inv : a.band_inv);
  const int rb = bnd * a.band + in - col * rows, n0 = 32 * col;
  typename F::Entry* const table = (typename F::Entry*)smem;
  constexpr int TABLE = F::TABLE * sizeof(typename F::Entry);
  char* const mine = smem + TABLE + wave * 2 * SLOT;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + TABLE + wave * 2 * SLOT;

  const uint32_t wmis = (uint32_t)((uintptr_t)W & 15);
  const uint8_t* const wbase = W - wmis;
  const uint32_t row_bytes = F::QK == 256 ? (uint32_t)(a.np * F::BS) : (uint32_t)(a.nkb * F::BS);
  const uint32_t last16 = ((uint32_t)(a.N - 1) * a.w_pitch + wmis + row_bytes - 1) & ~15u;   // the last granule that holds bytes of W
  uint32_t w_at[NI], w_piece[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int q = min(64 * i + lane, 32 * PPR - 1), r = q / PPR;
    w_at[i] = (uint32_t)min(n0 + r, a.N - 1) * a.w_pitch + wmis;
    w_piece[i] = 16 * (uint32_t)(q - r * PPR);
  }
  const auto request_w = [&](int p, int slot) {
    const uint32_t to = lds0 + slot * SLOT;
    walk_units([&](auto at) {
      constexpr int i = decltype(at)::value;
      const uint32_t v = min(((w_at[i] + (uint32_t)(p * UB)) & ~15u) + w_piece[i], last16);
      if constexpr (i < NI - 1) walk_fetch<1024 * i>(v, wbase, to);
      else walk_fetch_half<1024 * i>(v, wbase, to);
    }, std::make_integer_sequence<int, NI>());
  };
  const char* xt[R];
#pragma unroll
  for (int k = 0; k < R; ++k) xt[k] = DIRECT ? X : X + (int64_t)min(rb * R + k, a.row_tiles - 1) * a.np * DWALK_REC;
  const uint32_t x_lane = DIRECT ? (uint32_t)min(lrow, a.M - 1) * (uint32_t)(64 * a.nkb) + 32 * (uint32_t)half : 16 * (uint32_t)lane;
  typedef typename D::v8 v8;
  constexpr int XD = R >= 4 ? 2 : 4;                     // blocks of activations in registers
  v8 x[XD][R][2];
  const auto load_x = [&](int p, int b, v8 (&o)[R][2]) {
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
      for (int t = 0; t < 2; ++t) o[k][t] = *(const v8*)(xt[k] + ((int64_t)p * (DIRECT ? 512 : DWALK_REC) + (DIRECT ? 64 * b + 16 * t : 2048 * b + 1024 * t)) + x_lane);
  };

  dense_f16v acc[R], high;                               // DIRECT: the values 8 .. 15 of a half summed on their own (dense_kernel's parts of K are short: so are these chains)
#pragma unroll
  for (int k = 0; k < R; ++k)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[k][r] = high[r] = 0.0f;
  if (wave < a.np) {
    request_w(wave, 0);
#pragma unroll
    for (int b = 0; b < XD - 1; ++b)
      if (F::QK == 256 || b < a.nkb - 8 * wave) load_x(wave, b, x[b]);
  }
  for (int i = tid; i < F::TABLE; i += 64 * NW) table[i] = F::entry(i);
  if (F::TABLE) __syncthreads();
  walk_wait<0>();                                           // the first panel

  const uint32_t w_row = (uint32_t)min(n0 + lrow, a.N - 1) * a.w_pitch + wmis;
  int slot = 0;
  for (int p = wave; p < a.np; p += NW, slot ^= 1) {
    // (This panel was asked for in front of most of the activations of the one before; behind those come its own first blocks'.  Loads return in order.)
    walk_wait<2 * R * (XD - 1)>();
    const bool more = p + NW < a.np;
    if (more) request_w(p + NW, slot ^ 1);
    const uint8_t* const row = (const uint8_t*)mine + slot * SLOT + lrow * (16 * PPR) + ((w_row + (uint32_t)(p * UB)) & 15);
    const int blocks = F::QK == 256 ? 8 : min(8, a.nkb - 8 * p);
    typename F::Raw raw = F::fetch(row, 0, half);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (F::QK != 256 && b >= blocks) break;
      __builtin_amdgcn_sched_barrier(0);
      constexpr int A = XD - 1;
      if (b + A < 8) {
        if (F::QK == 256 || b + A < blocks) load_x(p, b + A, x[(b + A) % XD]);
      } else if (more) {                                    // (a panel with fewer blocks is the last)
        if (F::QK == 256 || b + A - 8 < a.nkb - 8 * (p + NW)) load_x(p + NW, b + A - 8, x[(b + A) % XD]);
      }
      const typename F::Raw now = raw;
      if (b < 7) raw = F::fetch(F::QK == 256 ? row : row + (b + 1) * F::BS, F::QK == 256 ? b + 1 : 0, half);
      uint32_t v[4], s[2] = {0, 0}, o[8];
      const float d = F::decode(now, table, b, half, v, s);
      dense_operands<F, typename D::v2>(v, s, d, o);
      const v8 w0 = __builtin_bit_cast(v8, make_uint4(o[0], o[1], o[2], o[3])), w1 = __builtin_bit_cast(v8, make_uint4(o[4], o[5], o[6], o[7]));
#pragma unroll
      for (int k = 0; k < R; ++k) acc[k] = D::mfma(w0, x[b % XD][k][0], acc[k]);
#pragma unroll
      for (int k = 0; k < R; ++k)
        if (DIRECT) high = D::mfma(w1, x[b % XD][k][1], high);
        else acc[k] = D::mfma(w1, x[b % XD][k][1], acc[k]);
    }
  }

  // ---- the waves' partial tiles, added in pairs
  if (DIRECT) acc[0] += high;
  __syncthreads();
  walk_f4* const red = (walk_f4*)(smem + TABLE);            // [wave][tile][run of four and half][row ^ that]
#pragma unroll
  for (int k = 0; k < R; ++k)
#pragma unroll
    for (int q = 0; q < 4; ++q) red[((wave * R + k) * 8 + 2 * q + half) * 32 + (lrow ^ (2 * q + half))] = (walk_f4){acc[k][4 * q], acc[k][4 * q + 1], acc[k][4 * q + 2], acc[k][4 * q + 3]};
  __syncthreads();
  for (int i = tid; i < R * 256; i += 64 * NW) {
    const int q = i & 7, r = (i >> 3) & 31, k = i >> 8, m = 32 * (rb * R + k) + r;
    walk_f4 v[NW];
#pragma unroll
    for (int z = 0; z < NW; ++z) v[z] = red[((z * R + k) * 8 + q) * 32 + (r ^ q)];
#pragma unroll
    for (int d = 1; d < NW; d *= 2)
#pragma unroll
      for (int z = 0; z < NW; z += 2 * d) v[z] += v[z + d];
    if (m < a.M) walk_store<T>(v[0], Y + (int64_t)m * a.ldy, (const T*)a.bias, n0 + 4 * q, a.N, a.quads);
  }
}

template <class F, int R, int NW, bool DIRECT, typename T>
static int dwalk_launch(const DwalkCall& c, hipStream_t stream) {
  constexpr size_t lds = dwalk_lds<F, R, NW>();
  const WalkBands tiles = walk_bands(R, c.M, c.N, c.K, DWALK_REC);
  if (!tiles.ok) return GGUF_NOT_TAKEN;
  auto kern = dense_walk_kernel<F, R, NW, DIRECT, T>;
  static std::atomic<uint64_t> done{0};
  allow_large_lds(kern, lds, done);
  const int64_t pitch = c.la.w_pitch ? c.la.w_pitch : (int64_t)(c.K / F::QK) * F::BS, ldy = c.la.ldy ? c.la.ldy : (int64_t)c.N;
  const int run = (tiles.tiles + 7) / 8;
  const WalkEnd end = {c.dtype, ldy % 4 == 0 && (uintptr_t)c.Y % (4 * sizeof(T)) == 0, ldy, c.la.bias};
  hipLaunchKernelGGL(kern, dim3((unsigned)(8 * run)), dim3(64 * NW), lds, stream, (const uint8_t*)c.W, (const char*)c.x,
                     GGUF_WALK_HEAD_ARGS(tiles, c.N, (uint32_t)pitch, c.K, c.M), (T*)c.Y, end);
  return launch_status();
}

template <class F, typename T>
static int dwalk_typed(const DwalkCall& c, hipStream_t s) {
  switch (c.plan.rt * 16 + c.plan.nw) {
    case 1 * 16 + 4: return c.plan.direct ? dwalk_launch<F, 1, 4, true, T>(c, s) : dwalk_launch<F, 1, 4, false, T>(c, s);
    case 1 * 16 + 8: return c.plan.direct ? dwalk_launch<F, 1, 8, true, T>(c, s) : dwalk_launch<F, 1, 8, false, T>(c, s);
    case 2 * 16 + 4: return dwalk_launch<F, 2, 4, false, T>(c, s);
    case 2 * 16 + 8: return dwalk_launch<F, 2, 8, false, T>(c, s);
    case 3 * 16 + 4: return dwalk_launch<F, 3, 4, false, T>(c, s);
    case 4 * 16 + 4: return dwalk_launch<F, 4, 4, false, T>(c, s);
    case 4 * 16 + 8: return dwalk_launch<F, 4, 8, false, T>(c, s);
  }
  return GGUF_NOT_TAKEN;
}
template <class F>
static int dwalk_run(const DwalkCall& c, hipStream_t s) { return c.dtype == GGUF_DTYPE_F16 ? dwalk_typed<F, _Float16>(c, s) : dwalk_typed<F, bf16_t>(c, s); }

}  // namespace gguf
