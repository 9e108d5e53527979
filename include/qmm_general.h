/*
 * C ABI of the general quantized matmul (libqmm4.so): the formats and shapes that qmm4_affine_bf16
 * refuses and the reference hands to MLX's own op (src/mlx_tree_spec/packed_linear.py:56-57, 84-86).
 */
#ifndef MI355X_QMM_GENERAL_H
#define MI355X_QMM_GENERAL_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * y = x @ dequant(w)^T, bf16 [M, N], fp32 accumulation: 2-, 4- or 8-bit affine codes in groups of 32,
 * 64 or 128, any N, K % 64 == 0 and K % group_size == 0. The dequantized weights are those of
 * dequant4_affine_bf16. Meant for up to a few hundred rows (every 64 rows dequantize the weights
 * again).
 *   x: bf16 [M, K]; w: uint32 [N, K * bits / 32]; scales, biases: bf16 [N, K / group_size].
 *   x and w 16-byte aligned; x and w (each with 64 rows more) below 2 GiB. M == 0 or N == 0 is a
 *   no-op. Asynchronous on `hip_stream`; keeps no state and allocates nothing, so it may be captured.
 * Returns 0 or a negative QMM4_ERR_* code (qmm4.h), with the message in qmm4_last_error().
 */
int qmm_affine_general_bf16(const void* x, const uint32_t* w, const void* scales, const void* biases, void* y,
                            int64_t M, int64_t N, int64_t K, int group_size, int bits, void* hip_stream);

#ifdef __cplusplus
}
#endif

#endif /* MI355X_QMM_GENERAL_H */
