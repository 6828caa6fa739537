"""Shape propagation and make_fx over the auto path, with fake CUDA tensors on the CPU: each kind of launch (plain, split,
widened first, last rows apart) gives the output's shape and a program that runs alone, and leaves nothing behind."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx

import feather_ops
from feather_ops import scaled_mm as impl

FP16, BF16 = torch.float16, torch.bfloat16
SHAPES = [(0, 64, 128), (1, 1000, 2560), (77, 1000, 2560), (40, 5120, 12288), (4096, 12288, 3072), (4112, 4096, 12288)]


def _operands(m, n, k, dtype, device="cuda"):
    return (torch.empty((m, k), dtype=dtype, device=device),
            torch.empty((-(-k // 128) * 8, n, 16), dtype=torch.float8_e5m2, device=device),
            torch.empty((), device=device))


def test_shapes_cover_the_launches():
    kinds = set()
    for m, n, k in SHAPES:
        for dtype in (FP16, BF16):
            parts, widen, one_op = impl._auto_plan(m, n, k, dtype)
            kinds.add("parts" if len(parts) > 1 else "widened" if widen else "split" if parts[0][2] > 1 else "plain")
            assert (one_op is None) == (len(parts) == 1 and (widen or parts[0][2] > 1))
    assert kinds == {"plain", "split", "widened", "parts"}


@pytest.mark.parametrize("dtype", [FP16, BF16])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_shape_propagation(m, n, k, dtype):
    before = dict(impl._split_workspaces)
    with FakeTensorMode():
        a, b, scale = _operands(m, n, k, dtype)
        for out_dtype in (FP16, BF16):
            out = feather_ops.scaled_mm_hip(a, b, scale, None, out_dtype)
            assert out.shape == (m, n) and out.dtype == out_dtype and out.device == a.device and out.is_contiguous()
    assert impl._split_workspaces == before


@pytest.mark.parametrize("mode", ["fake", "symbolic"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_make_fx(m, n, k, mode):
    from torch.fx.experimental.symbolic_shapes import ShapeEnv

    with FakeTensorMode(shape_env=ShapeEnv()):
        operands = _operands(m, n, k, FP16)
    graph = make_fx(lambda a, b, s: feather_ops.scaled_mm_hip(a, b, s, None, FP16), tracing_mode=mode)(*operands).graph
    nodes = [node for node in graph.nodes if node.op != "placeholder"]
    assert not any(node.op == "get_attr" for node in nodes)
    for node in nodes:
        splits = {torch.ops.feather_ops.scaled_mm_splitk.default: (6, 5),
                  torch.ops.feather_ops.scaled_mm_parts_new.default: (9, 10)}.get(node.target)
        if splits is not None and node.args[splits[0]] > 1:
            assert node.args[splits[1]].target is torch.ops.aten.zeros.default   # its counters start at zero
    assert sum("feather_ops" in str(node.target) for node in nodes) == 1


def test_relabelled_linear_without_gradients():
    with FakeTensorMode():
        lin = torch.nn.Linear(2560, 1000, device="cuda", dtype=BF16).requires_grad_(False)
        feather_ops.to_scaled_mm_linear(lin)
        assert lin(torch.empty((2, 5, 2560), device="cuda", dtype=BF16)).shape == (2, 5, 1000)


def test_what_the_two_step_call_refuses():
    with pytest.raises(NotImplementedError, match="Meta"):
        feather_ops.scaled_mm_hip(*_operands(16, 1000, 2560, FP16, "meta"), None, FP16)
    before = dict(impl._split_workspaces)
    for m, n, k in SHAPES[:4] + SHAPES[5:]:
        with pytest.raises(NotImplementedError, match="CPU"):
            feather_ops.scaled_mm_hip(*_operands(m, n, k, FP16, "cpu"), None, FP16)
    assert impl._split_workspaces == before
    with FakeTensorMode():
        _, b, scale = _operands(16, 1000, 2560, FP16)
        with pytest.raises(RuntimeError, match="Batching rule not implemented"):
            torch.vmap(lambda a: feather_ops.scaled_mm_hip(a, b, scale, None, FP16))(
                torch.empty((3, 16, 2560), dtype=FP16, device="cuda"))
