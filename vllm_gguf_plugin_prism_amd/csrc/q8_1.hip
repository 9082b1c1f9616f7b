// q8_1 activation quantizer for gfx950.
//
// Semantics follow the reference's quantize_q8_1 (csrc/gguf/gguf_kernel.cu:32-69):
// per 32 values, amax and sum are reduced by an xor butterfly over lane masks
// 16, 8, 4, 2, 1; d = amax / 127 in fp32; q = roundf(x / d) (0 when amax == 0);
// d and sum are stored rounded to half; columns [K, roundup(K, 512)) count as 0.
//
// Layout here: four lanes own one block, eight consecutive values each, so
// lane^2 / lane^1 are the butterfly partners for masks 16 / 8 (DPP quad
// permutes) and masks 4, 2, 1 are in-register.  The fp32 addition tree is
// therefore the same tree the reference evaluates.
#include "mmq_f.h"
#include "q8_1_device.h"
#include "tile_walk.h"

namespace gguf {

template <typename T>
__global__ __launch_bounds__(256) void quantize_q8_1_kernel(const T* __restrict__ x, char* __restrict__ ws, int K,
                                                           int Kp, int64_t row_bytes, int act,
                                                           _Float16* __restrict__ xh, bool permuted) {
  const int t = blockIdx.x * 256 + threadIdx.x;  // one thread per 8 values of the padded row
  if (t * 8 >= Kp) return;
  q8_1_quantize_thread<T>(x, ws, K, Kp, row_bytes, act, blockIdx.y, t, xh, permuted);
}

// The activations of mmq_f_core.h (MmqfRows): the quants as whole numbers in half precision, of four neighbours in the
// order 0, 2, 1, 3, the block scales [block][row], the block sums as halves [super-block][row][8].
template <typename T>
__global__ __launch_bounds__(256) void quantize_whole_kernel(const T* __restrict__ x, MmqfRows r, int K, int64_t m0) {
  const int t = blockIdx.x * 256 + threadIdx.x;  // one thread per 8 values
  if (t * 8 >= K) return;                        // (K is a multiple of 256: quads stay together)
  const int64_t m = m0 + blockIdx.y;
  float v[8];
  load8<T>(x + m * (int64_t)K + 8 * t, v);
  const Q8Quad q = q8_1_quantize8(v);
  union { _Float16 h[8]; uint4 v; } o;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    o.h[(i & 4) | ((i & 1) << 1) | ((i >> 1) & 1)] = (_Float16)(float)(int8_t)((i < 4 ? q.q.x >> (8 * i) : q.q.y >> (8 * (i - 4))) & 0xFF);
  *(uint4*)(r.x + m * r.pitch + 8 * t) = o.v;
  if ((t & 3) == 0) {
    const int b = t >> 2;
    r.d[(int64_t)b * r.rows + m] = q.d;
    r.s[((int64_t)(b >> 3) * r.rows + m) * 8 + (b & 7)] = (_Float16)q.s;
  }
}

int quantize_whole(const void* x, int xdtype, const MmqfRows& r, int64_t M, int64_t K, hipStream_t stream) {
  const int gx = (int)((K / 8 + 255) / 256);
  for (int64_t off = 0; off < M; off += 65535) {
    const int rows = (int)((M - off) < 65535 ? (M - off) : 65535);
    GGUF_DISPATCH_DTYPE(xdtype, hipLaunchKernelGGL(quantize_whole_kernel<scalar_t>, dim3(gx, rows), dim3(256), 0, stream, (const scalar_t*)x, r, (int)K, off));
  }
  return launch_status();
}

template <typename T>
__global__ __launch_bounds__(256) void quantize_wide_kernel(const T* __restrict__ x, char* __restrict__ records, int K, int64_t rows, int64_t m0) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t * 8 < (K + 255) / 256 * 256) wide_quantize_thread<T>(x, records, K, rows, m0 + blockIdx.y, t);   // (whole records: quads stay together)
}

int quantize_wide(const void* x, int xdtype, void* records, int64_t M, int64_t K, hipStream_t stream) {
  const int gx = (int)(((K + 255) / 256 * 32 + 255) / 256);
  for (int64_t off = 0; off < M; off += 65535) {
    const int rows = (int)((M - off) < 65535 ? (M - off) : 65535);
    GGUF_DISPATCH_DTYPE(xdtype, hipLaunchKernelGGL(quantize_wide_kernel<scalar_t>, dim3(gx, rows), dim3(256), 0, stream, (const scalar_t*)x, (char*)records, (int)K, M, off));
  }
  return launch_status();
}

// The records of tile_walk.h.  A workgroup has 32 rows of 64 values, eight threads to a row.
template <typename T>
__global__ __launch_bounds__(256) void quantize_walk_kernel(const T* __restrict__ x, char* __restrict__ records, int K, int np, int64_t M, bool groups) {
  const int row = threadIdx.x >> 3, k = 64 * blockIdx.x + 8 * (threadIdx.x & 7), b = (k >> 5) & 7;
  const int64_t m = 32 * (int64_t)blockIdx.y + row;
  if (m >= M) return;                            // (all eight threads of the row: quads stay together)
  float v[8] = {};
  if (k < K) load8<T>(x + m * (int64_t)K + k, v);   // (behind K: zeros)
  const Q8Quad q = q8_1_quantize8(v);
  char* const rec = records + ((int64_t)blockIdx.y * np + (k >> 8)) * WALK_REC;
  *(uint2*)(rec + 1024 * b + (groups ? 32 * (k & 16) + 8 * (4 * (k & 8) + row) : 16 * (2 * (k & 16) + row) + (k & 8))) = q.q;
  if ((threadIdx.x & 3) == 0) {
    *(_Float16*)(rec + WALK_D_AT + 16 * row + 2 * b) = (_Float16)q.d;
    *(_Float16*)(rec + WALK_S_AT + 16 * row + 2 * b) = (_Float16)q.s;
  }
}

int quantize_walk(const void* x, int xdtype, void* records, int64_t M, int64_t K, bool groups, hipStream_t stream) {
  const int np = (int)((K + 255) / 256);
  GGUF_DISPATCH_DTYPE(xdtype, hipLaunchKernelGGL(quantize_walk_kernel<scalar_t>, dim3(4 * np, (unsigned)((M + 31) / 32)), dim3(256), 0, stream, (const scalar_t*)x,
                                                 (char*)records, (int)K, np, M, groups));
  return launch_status();
}

__global__ void q8_1_unpack_kernel(const char* __restrict__ ws, int8_t* __restrict__ q, float* __restrict__ ds, int Kp,
                                   int64_t row_bytes) {
  const int64_t m = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= Kp) return;
  const char* row = ws + m * row_bytes;
  q[m * Kp + i] = ((const int8_t*)row)[i];
  if ((i & 31) == 0) {
    const float* fd = (const float*)(row + Kp);
    const int nb = Kp / 32, b = i >> 5;
    ds[(m * nb + b) * 2] = fd[b];
    ds[(m * nb + b) * 2 + 1] = fd[nb + b];
  }
}

int quantize_q8_1(const void* x, int xdtype, void* ws, int64_t M, int64_t K, hipStream_t stream, int act, void* half_plane, bool permuted) {
  if (M == 0) return GGUF_OK;
  const int Kp = (int)q8_kp(K);
  const int64_t rb = q8_row_bytes(K);
  const int gx = (Kp / 8 + 255) / 256;
  for (int64_t off = 0; off < M; off += 65535) {
    const int rows = (int)((M - off) < 65535 ? (M - off) : 65535);
    GGUF_DISPATCH_DTYPE(xdtype, hipLaunchKernelGGL(quantize_q8_1_kernel<scalar_t>, dim3(gx, rows), dim3(256), 0, stream,
                                                   (const scalar_t*)x + off * K * (act == ACT_NONE ? 1 : 2), (char*)ws + off * rb, (int)K, Kp, rb, act,
                                                   half_plane ? (_Float16*)half_plane + off * q8_half_pitch(K) : (_Float16*)nullptr, permuted));
  }
  return launch_status();
}

}  // namespace gguf

extern "C" int64_t gguf_q8_1_row_bytes(int64_t K) { return K <= 0 ? 0 : gguf::q8_row_bytes(K); }

extern "C" int gguf_quantize_q8_1(const void* x, int xdtype, void* ws, int64_t M, int64_t K, gguf_stream_t stream) {
  if (M < 0 || K <= 0 || K % 32 != 0) return GGUF_ERR_SHAPE;
  if (M > 0 && (!x || !ws)) return GGUF_ERR_NULL;
  if (xdtype < 0 || xdtype > 2) return GGUF_ERR_DTYPE;
  return gguf::quantize_q8_1(x, xdtype, ws, M, K, (hipStream_t)stream, gguf::ACT_NONE, nullptr);
}

extern "C" int gguf_q8_1_unpack(const void* ws, int8_t* q, float* ds, int64_t M, int64_t K, gguf_stream_t stream) {
  if (M < 0 || K <= 0 || K % 32 != 0) return GGUF_ERR_SHAPE;
  if (M == 0) return GGUF_OK;
  if (!ws || !q || !ds) return GGUF_ERR_NULL;
  const int Kp = (int)gguf::q8_kp(K);
  for (int64_t off = 0; off < M; off += 65535) {
    const int rows = (int)((M - off) < 65535 ? (M - off) : 65535);
    hipLaunchKernelGGL(gguf::q8_1_unpack_kernel, dim3((Kp + 255) / 256, rows), dim3(256), 0, (hipStream_t)stream,
                       (const char*)ws + off * gguf::q8_row_bytes(K), q + off * Kp, ds + off * (Kp / 32) * 2, Kp,
                       gguf::q8_row_bytes(K));
  }
  return gguf::launch_status();
}
