// Two matrices of a merged layer and up to four rows of activations in one launch of the streaming GEMV (mmvq_core.h).
//
// A launch for q and k and one for v are mostly beginning and end where the matrices are small: arguments, rows of X quantized by every
// workgroup, the first weights, 2.5 to 3 us before anything streams.  One grid of a workgroup per CU, shared out by the bytes, has them once, and
// the second matrix, often too small to fill the chip, streams beside the first.  Against two launches, 1600 random pairs
// of 1 .. 4 rows, 256 .. 28672 columns, K 512 .. 18944: 1.57 times as fast on average (1.9 below 2048 values of K, 1.2 at 60 MB), the worst 0.99;
// the projections of a 4096-wide Q4_K_M layer, one row: 38.6 us / 36.0.
// Each matrix's sums are those of a launch of its own: the parts of a row and their order follow from K alone.
#pragma once
#include "mmvq_core.h"
#include "tile_stream.h"

namespace gguf {

// Workgroups before `wgs` have rows of W, the others rows of V.  (Of the arguments the first 14 words are in registers, to pitch2: n2 and rows2 are loaded, and the
// workgroups of V wait for them before their first requests.)
template <class F, int DF, int SF, class G, int DG, int SG, int MT, int NW, typename T>
__global__ __launch_bounds__(64 * NW) void mmvq_pair_kernel(const uint8_t* __restrict__ W, const uint8_t* __restrict__ V, const T* __restrict__ X, int wgs, GGUF_GEOM,
                                                            uint32_t pitch2, int n2, int rows2, T* __restrict__ Y, T* __restrict__ Z, const T* __restrict__ bias,
                                                            const T* __restrict__ bias2, int64_t ldy) {
  if ((int)blockIdx.x < wgs) mmvq_stream_body<F, MT, NW, DF, T, false, MT <= 2, SF, false>(W, X, Y, bias, ldy, GGUF_GEOM_OF, ACT_NONE, blockIdx.x);
  else mmvq_stream_body<G, MT, NW, DG, T, false, MT <= 2, SG, false>(V, X, Z, bias2, ldy, StreamGeom{pitch2, n2, g_k, rows2, g_packed, g_g8_inv}, ACT_NONE, blockIdx.x - wgs);
}

template <class F, int MT, int NW, int D, int STAGED>
static size_t pair_lds(int K, int rows_per_wg) {
  const int nb = K / 32, S = (nb + 63) / 64;
  size_t lds = (size_t)MT * K + (size_t)MT * nb * 4 * (F::AUX != AUX_NONE ? 2 : 1) + F::TABLE_BYTES + (size_t)rows_per_wg * S * 16 * MT;
  if constexpr (STAGED == STAGED_DMA) lds += (size_t)NW * D * 1024 * SpanRegs<SpanOf<F>::value>::NR;
  else if constexpr (STAGED != 0) lds += (size_t)NW * 16 * SpanRegs<SpanOf<F>::value, STAGED == STAGED_ANY>::PIECES + SpanSlack<F>::value;
  return lds;
}

struct PairCall {
  const TsShard &a, &b;
  const void* x;
  int K, M, r1, r2;            // rows of the matrices per workgroup
  hipStream_t stream;
};

template <class F, int DF, int SF, class G, int DG, int SG, int MT, int NW, typename T>
static int pair_launch(const PairCall& c) {
  const size_t l1 = pair_lds<F, MT, NW, DF, SF>(c.K, c.r1), l2 = pair_lds<G, MT, NW, DG, SG>(c.K, c.r2), lds = l1 > l2 ? l1 : l2;
  if (lds > 160 * 1024) return GGUF_NOT_TAKEN;
  auto kern = mmvq_pair_kernel<F, DF, SF, G, DG, SG, MT, NW, T>;
  static std::atomic<uint64_t> done{0};
  if (lds > 64 * 1024) allow_large_lds(kern, 160 * 1024, done);
  const int wgs = ((int)c.a.N + c.r1 - 1) / c.r1, wgs2 = ((int)c.b.N + c.r2 - 1) / c.r2;
  const StreamGeom g1 = stream_geom((int)c.a.N, c.K, c.r1, c.a.la.w_pitch, c.M, NW), g2 = stream_geom((int)c.b.N, c.K, c.r2, c.b.la.w_pitch, c.M, NW);
  hipLaunchKernelGGL(kern, dim3(wgs + wgs2), dim3(64 * NW), lds, c.stream, (const uint8_t*)c.a.W, (const uint8_t*)c.b.W, (const T*)c.x, wgs, GGUF_GEOM_ARGS(g1),
                     g2.w_pitch, g2.N, g2.rows_per_wg, (T*)c.a.Y, (T*)c.b.Y, (const T*)c.a.la.bias, (const T*)c.b.la.bias, c.a.la.ldy);
  return launch_status();
}

template <class F, class G, typename T, int MT>
static int pair_rows(const TsShard& a, const TsShard& b, const void* x, int K, int M, hipStream_t s) {
  const int nb = K / 32, S = (nb + 63) / 64, cus = num_cus();
  if (S > MMVQ_NW) return GGUF_NOT_TAKEN;
  // one workgroup per CU, shared out by the bytes
  const double b1 = (double)a.N * (K / F::QK) * F::BS, b2 = (double)b.N * (K / G::QK) * G::BS;
  int wgs = (int)(cus * b1 / (b1 + b2) + 0.5);
  wgs = wgs < 1 ? 1 : wgs > cus - 1 ? cus - 1 : wgs;
  // (a wave has so many rows at least as it keeps in flight: less than two waves' stretches to a row are few bytes, one)
  const int least = nb < 64 ? 8 / S : MMVQ_DEPTH * (MMVQ_NW / S);
  const auto rows = [least](int64_t n, int w) { const int r = ((int)n + w - 1) / w; return r < least ? least : r; };
  const PairCall c = {a, b, x, K, M, rows(a.N, wgs), rows(b.N, cus - wgs), s};
  if (nb < 64) return pair_launch<F, 1, 0, G, 1, 0, MT, 8, T>(c);
  if constexpr (MT <= MMVQ_STAGED_MT) {
    if constexpr (DmaRing<F>::on && DmaRing<G>::on) {
      if (S <= 2 && nb % 64 == 0 && MT * K <= 32 * 64 * MMVQ_NW && span_aligned<F>(a.W, a.la.w_pitch, K) && span_aligned<G>(b.W, b.la.w_pitch, K)) {
        const int rc = pair_launch<F, MMVQ_DMA_DEPTH, STAGED_DMA, G, MMVQ_DMA_DEPTH, STAGED_DMA, MT, MMVQ_NW, T>(c);
        if (rc != GGUF_NOT_TAKEN) return rc;
      }
    }
    // rows that are not whole aligned stretches: fetched from any even address, or lane by lane
    return pair_launch<F, MMVQ_DEPTH, SpanAny<F>::value ? STAGED_ANY : 0, G, MMVQ_DEPTH, SpanAny<G>::value ? STAGED_ANY : 0, MT, MMVQ_NW, T>(c);
  }
  return pair_launch<F, MMVQ_DEPTH, 0, G, MMVQ_DEPTH, 0, MT, MMVQ_NW, T>(c);
}
template <class F, class G>
static int pair_fmt(const TsShard& a, const TsShard& b, const void* x, int dtype, int K, int M, hipStream_t s) {
  int rc = GGUF_ERR_DTYPE;
  GGUF_DISPATCH_DTYPE(dtype, rc = (M == 1 ? pair_rows<F, G, scalar_t, 1>(a, b, x, K, M, s) : M == 2 ? pair_rows<F, G, scalar_t, 2>(a, b, x, K, M, s)
                                                                                                  : pair_rows<F, G, scalar_t, 4>(a, b, x, K, M, s)));
  return rc;
}

}  // namespace gguf
