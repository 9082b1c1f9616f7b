/* Entry points that only this package's own layer calls use (torch_binding/gguf_calls.cpp, ops.py); include/gguf_hip.h is
 * the public ABI.
 *
 * The codebook formats (ids 16 and up) past a few rows of X, for one shard of a merged layer: Y = X . dequant(W)^T with
 * the weights rounded to X's dtype as gguf_dequantize rounds them and a 32-bit sum, the two steps of the reference's
 * fallback (quantization/linear.py:50-58) in one kernel.  Arguments as for gguf_mmq_linear; X and Y fp16 or bf16, X at a
 * 16-byte boundary, its rows dense.  gguf_dense_linear_takes: 1 for a call that it serves.  The workspace may be null
 * where gguf_dense_linear_workspace_bytes is 0; it needs no initialisation; with less than that the call is slower, with less than its partial tiles take GGUF_ERR_WORKSPACE.
 * gguf_dense_linear_walk: where a call with a workspace of this size, at a 16-byte boundary, runs dense_walk_kernel, 16 times the tiles of 32 rows that a workgroup has and its
 * waves, and 256 where it loads X as it lies, else 0.
 *
 * gguf_mmq_layer_workspace_bytes: the workspace with which gguf_mmq_linear on GGUF_MMQ_AUTO runs at full speed for weights
 * of this type, at a 16-byte boundary.  (gguf_mmq_workspace_bytes_engine does not know the type.)  gguf_mmq_layer_route: the
 * kernel that such a call with a workspace of this size runs where it is neither dealt nor walked: 1 the streaming tile kernel, 4 the wide tiles, 2 the
 * half-precision unit's, 0 another.  gguf_linear_dealt: 1 where they are, by tile_dealt_kernel, which comes before all of these (5 .. 32 rows;
 * gemv: of gguf_mmvq_linear), with rows in a workspace that begins on 16 bytes.
 * gguf_linear_walk: where a call of more than 32 rows with a workspace of this size runs tile_walk_kernel, which comes before them too, 16 times the tiles of
 * 32 rows that a workgroup has and its waves, else 0 (of weights that begin on 16 bytes: others of Q8_0 may run otherwise).
 * gguf_mmq_layer_unit: the kernel of gguf_mmq_layer_route, with 2 added to 1 (past 32 rows) and 4 where the half-precision unit would run a call that these decline.  gguf_moe_mmq_layer_wide: whether
 * gguf_moe_mmq_layer with the workspace it asks for, at addresses divisible by 16, runs on the expert and the wide tiles.
 * gguf_moe_mmq_layer_finer: the block of 16 slots from which on the first or second product (product) of a layer on the streaming tiles deals K to
 * two waves each; -1: none, or a layer that they do not take.
 *
 * gguf_mmvq_linear_whole: a call of gguf_mmvq_linear that needs no workspace, up to four rows which the GEMV quantizes by itself; taken = 0, and nothing is launched, for
 * another (more rows; rows too long for its LDS).
 *
 * gguf_linear_two: two products of the same x, up to 32 rows, as calls of gguf_mmvq_linear (gemv: bit 0 the first, bit 1 the second) or gguf_mmq_linear would run them
 * (the same results bit for bit), and for pairs of types that recipes mix in one launch: up to four rows of the GEMV, from five on behind the
 * quantizer's, which other pairs share too.  They are shards of a merged layer, columns of one result of this row pitch.  The workspace, M * gguf_q8_1_row_bytes(K), begins on 16 bytes.
 * gguf_linear_two_takes: 1 for a pair that it serves. */
#pragma once
#include <stdint.h>
#ifdef __cplusplus
extern "C" {
#endif
int gguf_dense_linear_takes(int type, int xdtype, int64_t N, int64_t K, int64_t M);
int64_t gguf_dense_linear_workspace_bytes(int64_t N, int64_t K, int64_t M);
int gguf_dense_linear_walk(int type, int64_t N, int64_t K, int64_t M, int64_t w_row_pitch_bytes, int64_t workspace_bytes);
int gguf_dense_linear(const void* W, int64_t w_row_pitch_bytes, const void* x, int xdtype, void* workspace, void* Y, int64_t y_row_pitch,
                      const void* bias, int type, int64_t N, int64_t K, int64_t M, int64_t workspace_bytes, void* stream);
int64_t gguf_mmq_layer_workspace_bytes(int type, int64_t N, int64_t K, int64_t M, int64_t w_row_pitch_bytes);
int gguf_moe_mmq_layer_finer(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t top_k, int64_t tokens, int64_t num_experts, int product);
int gguf_moe_mmq_layer_wide(int type13, int type2, int64_t H, int64_t I, int64_t N_out, int64_t top_k, int64_t tokens, int64_t num_experts);
int gguf_mmq_layer_unit(int type, int64_t N, int64_t K, int64_t M, int64_t w_row_pitch_bytes, int64_t workspace_bytes);
int gguf_mmvq_linear_whole(const void* W, int64_t w_row_pitch_bytes, const void* x, int xdtype, void* Y, int64_t y_row_pitch, const void* bias, int type, int64_t N, int64_t K,
                           int64_t M, void* stream, int* taken);
int gguf_linear_two_takes(int type, int64_t N, int64_t w_row_pitch_bytes, int type2, int64_t N2, int64_t w_row_pitch_bytes2, int64_t K, int64_t M, int gemv);
int gguf_linear_two(const void* W, int64_t w_row_pitch_bytes, int type, int64_t N, void* Y, const void* bias, const void* W2, int64_t w_row_pitch_bytes2, int type2,
                    int64_t N2, void* Y2, const void* bias2, const void* x, int xdtype, void* q8_workspace, int64_t y_row_pitch, int64_t K, int64_t M, int gemv, void* stream);
int gguf_linear_walk(int type, int64_t N, int64_t K, int64_t M, int64_t w_row_pitch_bytes, int64_t workspace_bytes);
int gguf_linear_dealt(int type, int64_t N, int64_t K, int64_t M, int64_t w_row_pitch_bytes, int gemv);
int gguf_mmq_layer_route(int type, int64_t N, int64_t K, int64_t M, int64_t w_row_pitch_bytes, int64_t workspace_bytes);
#ifdef __cplusplus
}
#endif
