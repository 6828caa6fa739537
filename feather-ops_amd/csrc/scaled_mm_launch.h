// Host-side interface between the C ABI (scaled_mm_api.hip) and the per-dtype kernel instantiations
// (scaled_mm_launch.hip, compiled once per combination).
#pragma once

#include <hip/hip_runtime.h>

#include "scaled_mm_kernels.h"

namespace feather {

struct TileQuery {
    int warps_m;
    int warps_n;
    int unroll_k;
    int repeat_m;
    int repeat_n;
    bool prefetch;
};

#define FEATHER_COMBO_CAT_(e, a, o) launch_combo_##e##a##o
#define FEATHER_COMBO_FN(e, a, o) FEATHER_COMBO_CAT_(e, a, o)

// launch_combo_<e5m2><a_bf16><out_bf16>: false if the tile is not instantiated, else enqueues the kernel.
bool launch_combo_000(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_001(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_010(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_011(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_100(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_101(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_110(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_111(const TileQuery&, const Params&, hipStream_t);
// The gradient matmul's: bf16 MFMAs (FEATHER_A_BF16 = 2).
bool launch_combo_020(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_021(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_120(const TileQuery&, const Params&, hipStream_t);
bool launch_combo_121(const TileQuery&, const Params&, hipStream_t);

// grad_x [M, K] = operand [M, depth] @ b [depth/16, K, 16] * scale (one value; none: 1), the gradient matmul of
// linear_backward.hip: depth a multiple of 8 (streaming tiles: 16), the operand bf16 (operand_bf16) or fp16, the output bf16 or fp16 (fp16
// operands: fp16). `grad_matmul_split_bytes` says on the host what workspace the splits need, 256-byte aligned (0: none),
// or -1 where the tile or the splits do not fit.
int64_t grad_matmul_split_bytes(const TileQuery& tile, int64_t M, int64_t K, int64_t depth, bool operand_bf16,
                                int splits);
bool launch_grad_matmul(const TileQuery& tile, const uint16_t* operand, const uint8_t* b, const float* scale,
                        uint16_t* grad_x, int64_t M, int64_t K, int64_t depth, bool use_fp8_e5m2, bool operand_bf16,
                        bool out_bf16, int splits, void* split_workspace, hipStream_t stream);

}  // namespace feather
