"""Gradients of the fp8 linear layer on the gfx950 kernels (`csrc/linear_backward.hip`); not in the reference, which
has no backward.

`linear_backward` computes dX = (dY * scale) @ W and dbias = the column sums of dY for a frozen prepacked weight, as
fp32 arithmetic on the dequantized weight gives them, on the forward's MFMA kernels. The tile and split count are the
forward heuristic's for the same matmul with fp16 activations: M rows, K outputs, `depth` inputs.
"""

import functools

import torch

from . import _lib
from .scaled_mm import _auto_choice, _split_workspace

# Layers of fewer products than this keep torch's fp32 matmul: callers of such layers compare gradients with that product
# bit for bit, which another order of its sums does not give. Speed is not the reason: at 64 x 512 -> 512 forward and
# backward take 84 us a pass by the kernels against 117 by torch's operations, both bound by the host.
_MIN_PRODUCTS = 1 << 22


@functools.lru_cache(maxsize=4096)
def backward_plan(M: int, N: int, K: int, per_column: bool) -> tuple[tuple[int, ...], int, int, int] | None:
    """(tile, splits, split workspace bytes, workspace bytes) of a layer of N outputs and K inputs on M rows, or None
    where the layer stays with `composite`: small ones (_MIN_PRODUCTS), and what the library's own check refuses: buffers
    past 2 GiB, sizes outside the forward's contract."""
    if M * N * K < _MIN_PRODUCTS:
        return None
    lib = _lib.c_library()
    nbytes = lib.feather_linear_backward_workspace_bytes(M, N, K, per_column)
    if nbytes < 0:
        return None
    depth = lib.feather_linear_backward_depth(N, per_column)
    tile, splits, _ = _auto_choice(M, K, depth, torch.float16)
    split_bytes = lib.feather_linear_backward_split_bytes(M, N, K, per_column, *tile, splits)
    return (tile, splits, split_bytes, nbytes) if split_bytes >= 0 else None


def takes(grad: torch.Tensor, weight_fp8: torch.Tensor, weight_scale: torch.Tensor, k: int) -> bool:
    """Whether the kernels take these operands; the others go to `composite`."""
    return (grad.is_cuda and grad.dtype in (torch.float16, torch.bfloat16) and weight_scale.dtype == torch.float32
            and weight_fp8.dtype in (torch.float8_e5m2, torch.float8_e4m3fn) and grad.numel() > 0
            and backward_plan(grad.numel() // grad.shape[-1], grad.shape[-1], k, weight_scale.numel() > 1) is not None)


def composite(grad: torch.Tensor, weight_fp8: torch.Tensor, weight_scale: torch.Tensor,
              k: int) -> tuple[torch.Tensor, torch.Tensor]:
    """(dX, dbias) by torch's differentiable operations, in fp32 on the dequantized weight; neither is rounded."""
    chunks, n, _ = weight_fp8.shape
    w = weight_fp8.permute(0, 2, 1).reshape(chunks * 16, n)[:k].float() * weight_scale.float()  # [K, N]
    g = grad.reshape(-1, n).float()
    return g @ w.t(), g.sum(0)


@torch.library.custom_op("feather_ops::scaled_mm_linear_backward", mutates_args=())
def linear_backward(grad: torch.Tensor, weight_fp8: torch.Tensor, weight_scale: torch.Tensor, k: int, need_x: bool,
                    need_bias: bool) -> tuple[torch.Tensor, torch.Tensor]:
    """(dX [M, K], dbias [N]) in grad's dtype for `grad` [..., N]; one that is not needed comes back empty. An opaque op, so
    that a traced backward holds one node for it."""
    n = grad.shape[-1]
    g = grad.reshape(-1, n)
    m = g.shape[0]
    grad_x = grad.new_empty((m, k) if need_x else 0)
    grad_bias = grad.new_empty(n if need_bias else 0)
    if not takes(grad, weight_fp8, weight_scale, k):
        x, bias = composite(grad, weight_fp8, weight_scale, k)
        return x.to(grad.dtype) if need_x else grad_x, bias.to(grad.dtype) if need_bias else grad_bias
    if not g.is_contiguous() or g.data_ptr() % 16:
        g = g.clone(memory_format=torch.contiguous_format)  # the kernels read 16-byte-aligned rows
    per_column = weight_scale.numel() > 1
    if weight_scale.data_ptr() % 16 or not weight_scale.is_contiguous():
        weight_scale = weight_scale.clone(memory_format=torch.contiguous_format)
    tile, splits, split_bytes, nbytes = backward_plan(m, n, k, per_column)
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=g.device)
    split_workspace = _split_workspace(g.device, split_bytes) if need_x and splits > 1 else workspace[:0]
    torch.ops.feather_ops.linear_backward.default(
        g, weight_fp8, weight_scale, grad_x if need_x else None, grad_bias if need_bias else None, split_workspace,
        workspace, k, splits, *tile)
    return grad_x, grad_bias


@linear_backward.register_fake
def _(grad: torch.Tensor, weight_fp8: torch.Tensor, weight_scale: torch.Tensor, k: int, need_x: bool,
      need_bias: bool) -> tuple[torch.Tensor, torch.Tensor]:
    n = grad.shape[-1]
    rows = grad.numel() // n
    return grad.new_empty((rows, k) if need_x else (0,)), grad.new_empty((n,) if need_bias else (0,))
