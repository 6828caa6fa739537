"""The backward's host side on the CPU: every tile its picks can name is instantiated for bf16 operands, and operands the
kernels do not take go to torch's operations with the same result."""

import random

import pytest
import torch

from feather_ops import _lib
from feather_ops import linear_backward as lb
from feather_ops import prepack_transpose
from feather_ops.tiles import GRAD_TILES, SCALED_MM_TILES, split_workspace_bytes


def test_grad_tiles_cover_the_picks():
    rng = random.Random(0)
    assert set(GRAD_TILES) <= set(SCALED_MM_TILES)
    seen = set()
    for _ in range(6000):
        m = int(2 ** rng.uniform(0, 14))
        n = 8 * int(2 ** rng.uniform(0, 11.5))
        k = 16 * int(2 ** rng.uniform(0, 10.5))
        if rng.random() < 0.3:    # whole tiles of the wide kernel
            m, n, k = (-(-s // 256) * 256 for s in (m, n, k))
        for column in (False, True):
            plan = lb.backward_plan(m, n, k, column)
            if plan is None:
                continue
            tile, splits, split_bytes, nbytes = plan
            assert tile in GRAD_TILES, (m, n, k, tile)
            depth = 48 * -(-n // 16) if column else max(n, 16)
            assert splits == 1 or split_bytes == split_workspace_bytes(m, k, depth, tile, splits)
            assert nbytes >= -(-depth // 128) * 128 * k + (2 * m * depth if column else 0)
            seen.add(tile)
    assert seen == set(GRAD_TILES)


@pytest.mark.parametrize("m,n,k", [(512, 8, 4096), (4096, 8, 4096), (4112, 8, 3072), (64, 8, 16384), (512, 24, 4096)])
def test_plans_pass_the_librarys_check(m, n, k):
    """A router's or a gate's few outputs: one chunk of depth, the least any kernel takes."""
    lib = _lib.c_library()
    for column in (False, True):
        tile, splits, split_bytes, _ = lb.backward_plan(m, n, k, column)
        assert lib.feather_linear_backward_split_bytes(m, n, k, column, *tile, splits) == split_bytes >= 0
    assert lib.feather_linear_backward_split_bytes(m, n, k, False, 3, 3, 3, 3, 3, True, 1) == -1
    assert lib.feather_linear_backward_split_bytes(m, n, k, False, *tile, 99) == -1
    assert lib.feather_linear_backward_split_bytes(m, n + 4, k, False, *tile, 1) == -1


def test_only_small_layers_and_big_buffers_have_no_plan():
    rng = random.Random(1)
    for _ in range(4000):
        m, n, k = int(2 ** rng.uniform(0, 15)), 8 * int(2 ** rng.uniform(0, 11)), 16 * int(2 ** rng.uniform(0, 10))
        for column in (False, True):
            depth = 48 * -(-n // 16) if column else n + n % 16
            fits = max(2 * m * max(n, k, depth), -(-depth // 128) * 128 * k) < 1 << 31
            assert (lb.backward_plan(m, n, k, column) is not None) == (m * n * k >= 1 << 22 and fits), (m, n, k, column)


def test_plan_refuses_buffers_past_2_gib():
    assert lb.backward_plan(65536, 8192, 4096, True) is None      # the split gradient: 3.2 GB
    assert lb.backward_plan(65536, 8192, 4096, False) is not None


@pytest.mark.parametrize("column", [False, True])
def test_operands_off_the_gpu_take_torch(column):
    torch.manual_seed(0)
    wq = torch.randn(24, 48).to(torch.float8_e5m2)
    scale = torch.rand(24) + 0.5 if column else torch.tensor(0.5)
    grad = torch.randn(2, 5, 24).to(torch.bfloat16)
    x, bias = lb.linear_backward(grad, prepack_transpose(wq), scale, 48, True, True)
    w = wq.float() * (scale[:, None] if column else scale)
    want = grad.reshape(10, 24).float() @ w
    assert x.shape == (10, 48) and (x.float() - want).abs().max() <= 2.0**-8 * want.abs().max()
    assert torch.equal(bias, grad.reshape(10, 24).float().sum(0).to(torch.bfloat16))
    none_x, none_b = lb.linear_backward(grad, prepack_transpose(wq), scale, 48, False, False)
    assert none_x.numel() == none_b.numel() == 0


def test_small_layers_stay_out_of_the_op(monkeypatch):
    """A small layer's backward is torch's operations without the op's Python dispatch, rounded once."""
    import types

    from feather_ops.modules import _linear_backward

    def op(*args):
        raise AssertionError("the op")

    monkeypatch.setattr(lb, "linear_backward", op)
    torch.manual_seed(0)
    wq, scale, grad = torch.randn(24, 48).to(torch.float8_e5m2), torch.rand(24), torch.randn(10, 24).to(torch.bfloat16)
    ctx = types.SimpleNamespace(saved_tensors=(prepack_transpose(wq), scale), x_shape=(10, 48), x_dtype=torch.float16,
                                bias_dtype=torch.float32, needs_input_grad=(True, False, False, True))
    gx, _, _, gb = _linear_backward(ctx, grad)
    assert torch.equal(gx, (grad.float() @ (wq.float() * scale[:, None])).to(torch.float16))
    assert torch.equal(gb, grad.float().sum(0))


def test_tangents_of_gradients():
    """Forward mode over the backward (a Hessian-vector product): the gradient's tangent reaches both results."""
    import types

    from torch.autograd import forward_ad

    from feather_ops.modules import _linear_backward

    torch.manual_seed(0)
    packed, scale = prepack_transpose(torch.randn(24, 48).to(torch.float8_e5m2)), torch.rand(24)
    ctx = types.SimpleNamespace(saved_tensors=(packed, scale), x_shape=(2, 5, 48), x_dtype=torch.float16,
                                bias_dtype=torch.float16, needs_input_grad=(True, False, False, True))
    grad, tangent = torch.randn(2, 2, 5, 24).to(torch.float16)
    want = [x for x in _linear_backward(ctx, tangent) if x is not None]
    with forward_ad.dual_level():
        got = [x for x in _linear_backward(ctx, forward_ad.make_dual(grad, tangent)) if x is not None]
        got = [forward_ad.unpack_dual(x).tangent for x in got]
    assert len(got) == 2 and all(torch.equal(a, b) for a, b in zip(got, want))
