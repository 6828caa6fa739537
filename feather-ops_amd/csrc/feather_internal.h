// Entry points of libfeather_ops_gfx950.so that only this package's torch library calls (extension.cpp); the public C
// ABI is include/feather_ops.h.
#ifndef FEATHER_INTERNAL_H
#define FEATHER_INTERNAL_H

#include "feather_ops.h"

extern "C" {

/*
 * Gradients of y = (x @ W^T) * scale + bias for a frozen prepacked weight, enqueued on `stream`:
 *   grad_x[M, K] = (grad[M, N] * scale) @ W, grad_bias[N] = the column sums of grad.
 * No counterpart in the reference, which has no backward.
 *
 *   grad         [M, N] row-major, fp16 or (bf16 = true) bf16 bits; grad_x and grad_bias have the same type. Either
 *                may be null (not computed), not both.
 *   b_prepacked  the forward's [K_pad/16, N, 16] codes.
 *   scale        fp32, one value, or N (per_column, 16-byte aligned).
 *   tile, splits as launch_scaled_mm's and feather_scaled_mm_splitk's, for a matmul of M rows, K output columns and
 *                feather_linear_backward_depth(N, per_column) inputs; with bf16 gradients or per-column scales one of
 *                feather_ops/tiles.py GRAD_TILES. splits > 1 needs split_workspace, as feather_scaled_mm_splitk's
 *                (sized for that matmul); otherwise it is ignored.
 *   workspace    feather_linear_backward_workspace_bytes(...) bytes, 16-byte aligned, of any content.
 *
 * Sums are fp32: products of 16-bit gradients and fp8 codes are exact in them. A per-column scale is multiplied into the
 * gradient in fp32, and the matmul takes the product in three bf16 terms: all of it, but for what lies under 2^-133 times
 * the largest scale's code (fp16 gradients: where |gradient * scale| < 2^-110, far below what fp16 results hold). Requires N % 8 == 0, K % 16 == 0 and 16-byte aligned pointers;
 * returns false (nothing enqueued) otherwise, and for a tile or split count that feather_linear_backward_split_bytes
 * refuses, or a workspace that is too small.
 */
bool feather_linear_backward(const uint16_t* grad, const uint8_t* b_prepacked, const float* scale, uint16_t* grad_x,
                             uint16_t* grad_bias, int64_t M, int64_t N, int64_t K, bool per_column, bool use_fp8_e5m2,
                             bool bf16, int block_warps_m, int block_warps_n, int unroll_k, int repeat_m, int repeat_n,
                             bool prefetch, int splits, void* split_workspace, int64_t split_workspace_bytes,
                             void* workspace, int64_t workspace_bytes, hipStream_t stream);

/* Workspace bytes of feather_linear_backward (host only): -1 for sizes outside its contract, each buffer under 2 GiB. */
int64_t feather_linear_backward_workspace_bytes(int64_t M, int64_t N, int64_t K, bool per_column);

/* The inputs (contraction length) of feather_linear_backward's matmul: what its tile and splits are chosen for. */
int64_t feather_linear_backward_depth(int64_t N, bool per_column);

/*
 * Bytes of split_workspace that feather_linear_backward needs with this tile and split count (0 for splits = 1), for
 * gradients of either type; -1 where it refuses them. Host only: what a caller asks before it leaves another path.
 */
int64_t feather_linear_backward_split_bytes(int64_t M, int64_t N, int64_t K, bool per_column, int block_warps_m,
                                            int block_warps_n, int unroll_k, int repeat_m, int repeat_n, bool prefetch,
                                            int splits);

/*
 * w [N, K] row-major -> out [K_pad/16][N][16], zero-padded to K_pad = ceil(K / 128) * 128: the layout of
 * feather_prepack_b for a weight stored as a Linear stores it. Requires K % 16 == 0, 16-byte aligned pointers and
 * both buffers under 2 GiB; returns false (nothing enqueued) otherwise.
 */
bool feather_prepack_rows(const uint8_t* w, uint8_t* out, int64_t N, int64_t K, hipStream_t stream);

/*
 * The same for a weight to quantize (source 0: bf16, 1: fp16, 2: fp32): per row (scale holds N values) or per tensor
 * (one), scale = amax / the format's largest value, 1 where amax is zero or NaN, codes = w / scale rounded to nearest
 * even. amax: scratch of max(N, 1024) words, any content. Same contract; w's buffer under 2 GiB too.
 */
bool feather_quantize_rows(const void* w, int source, uint8_t* out, float* scale, uint32_t* amax, int64_t N, int64_t K,
                           bool use_fp8_e5m2, bool per_row, hipStream_t stream);

}  // extern "C"

#endif  // FEATHER_INTERNAL_H
