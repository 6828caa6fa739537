"""The auto path's second launch for a few last rows: which shapes take it (CPU), and its outputs (GPU)."""

import random

import pytest
import torch

from feather_ops.scaled_mm import _TAIL_MAX_ROWS, _auto_choice, _auto_parts, _auto_plan, _launch_auto, _refined

FP16, BF16 = torch.float16, torch.bfloat16

# (m, n, k): one row, 16 and 64 of them past a whole round of wide tiles, of 256 x 192 ones, of 128 x 128 and 64 x 128
# ring tiles; a tail split along K; N off the tiles
SPLIT = [(4097, 5120, 2560), (4112, 4096, 4096), (4160, 4096, 4096), (4112, 3072, 3072), (1281, 5960, 5248),
         (1040, 4096, 12288), (2208, 3712, 2368)]


@pytest.mark.parametrize("dtype", [FP16, BF16])
@pytest.mark.parametrize("m,n,k", SPLIT)
def test_shapes_that_split(m, n, k, dtype):
    parts, widen = _auto_parts(m, n, k, dtype)
    assert len(parts) == 2 and widen == (dtype == BF16)
    assert parts[0] == (m - m % 128 if m % 256 > 64 else m - m % 256, *_auto_choice(parts[0][0], n, k, FP16)[:2])


def test_parts_cover_the_rows_once():
    rng = random.Random(0)
    split = 0
    for _ in range(20000):
        m, n, k = int(2 ** rng.uniform(0, 14)), 8 * int(2 ** rng.uniform(0, 11)), 16 * int(2 ** rng.uniform(0, 10))
        for dtype in (FP16, BF16):
            parts, widen = _auto_parts(m, n, k, dtype)
            assert sum(rows for rows, _, _ in parts) == m
            if len(parts) == 1:
                tile, splits, first = _auto_choice(m, n, k, dtype)
                assert widen == first
                assert parts[0][1:] == _refined(m, n, k, tile, splits, dtype == BF16 and not widen)
                continue
            split += 1
            (head, tile, splits), (tail, *tail_pick) = parts
            assert head % 128 == 0 and splits == 1 and 0 < tail <= _TAIL_MAX_ROWS and m >= 320 - 64
            assert (tile, splits) == _auto_choice(head, n, k, FP16)[:2]
            tile, splits, _ = _auto_choice(tail, n, k, FP16)
            assert tuple(tail_pick) == _refined(tail, n, k, tile, splits, False)
    assert split > 50
    for m in (1, 77, 256, 512, 4096, 4224, 4096 + 100):
        assert len(_auto_parts(m, 4096, 4096, FP16)[0]) == 1


@pytest.mark.parametrize("dtype", [FP16, BF16])
@pytest.mark.parametrize("m,n,k", [(320, 64, 0), (4112, 4096, 0), (300, 0, 64), (0, 64, 64), (4112, 4096, 8)])
def test_empty_sides_are_one_launch(m, n, k, dtype):
    """The op itself answers them: an empty result, or its refusal of K."""
    assert _auto_parts(m, n, k, dtype) == (((m, *_auto_choice(m, n, k, dtype)[:2]),), _auto_choice(m, n, k, dtype)[2])


@pytest.mark.parametrize("m,n,k", SPLIT + [(16, 1000, 2560), (77, 5120, 2560), (4096, 4096, 4096), (40, 5120, 12288)])
def test_traced_sizes(m, n, k):
    """torch.jit.trace passes sizes as tensors: the same plan, in plain numbers."""
    for dtype in (FP16, BF16):
        plan = _auto_plan(torch.tensor(m), torch.tensor(n), torch.tensor(k), dtype)
        assert repr(plan) == repr(_auto_plan(m, n, k, dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [SPLIT[1], SPLIT[5], (16, 1000, 2560)])
def test_jit_trace(m, n, k):
    import feather_ops

    a, b, scale, bias = _inputs(m, n, k, BF16, True)
    want = feather_ops.scaled_mm_hip(a, b, scale, bias, BF16)
    traced = torch.jit.trace(lambda x: feather_ops.scaled_mm_hip(x, b, scale, bias, BF16), (a,), check_trace=False)
    assert torch.equal(traced(a), want)


def _inputs(m, n, k, dtype, column):
    import feather_ops

    g = torch.Generator("cuda").manual_seed(m)
    a = torch.randn((m, k), generator=g, device="cuda").to(dtype)
    w = (torch.randn((n, k), generator=g, device="cuda") * 20).to(torch.float8_e4m3fn)
    scale = (torch.rand(n, generator=g, device="cuda") + 0.5) * 1e-3 if column else torch.tensor(1e-3, device="cuda")
    return a, feather_ops.prepack_transpose(w), scale, torch.randn(n, generator=g, device="cuda").to(dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [FP16, BF16])
@pytest.mark.parametrize("m,n,k", SPLIT)
def test_outputs(m, n, k, dtype):
    import feather_ops
    from gpu_helpers import check_against_oracle

    for column in (False, True):
        a, b, scale, bias = _inputs(m, n, k, dtype, column)
        out = feather_ops.scaled_mm_hip(a, b, scale, bias, dtype)
        rows = sorted({0, 1, 255, 256, m // 2, *range(m - m % 128 - 2, m)})
        check_against_oracle(out, a, b, scale, bias, rows=rows)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [FP16, BF16])
@pytest.mark.parametrize("m,n,k", SPLIT)
def test_one_op_and_the_launches_one_by_one_agree(m, n, k, dtype):
    """scaled_mm_parts_new against the ops that write into an output, which calls that autograd follows still take."""
    import feather_ops

    a, b, scale, bias = _inputs(m, n, k, dtype, True)
    for out_dtype in (FP16, BF16):
        add = bias.to(out_dtype)
        for s in (None, scale[0], scale):
            got = feather_ops.scaled_mm_hip(a, b, s, add, out_dtype)
            want = torch.empty_like(got)
            _launch_auto(a, b, s, add, want)
            assert got.is_contiguous() and torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.gpu
def test_other_streams():
    import feather_ops

    a, b, scale, bias = _inputs(*SPLIT[5], BF16, True)
    want = feather_ops.scaled_mm_hip(a, b, scale, bias, BF16)
    outs = []
    for _ in range(3):
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            outs.append(feather_ops.scaled_mm_hip(a, b, scale, bias, BF16))
        torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    assert all(torch.equal(out, want) for out in outs)


@pytest.mark.gpu
def test_graph_replays():
    import feather_ops

    m, n, k = SPLIT[5]      # the tail splits K: its workspace is part of the graph
    a, b, scale, bias = _inputs(m, n, k, BF16, True)
    inputs = [torch.randn_like(a) for _ in range(3)]
    want = [feather_ops.scaled_mm_hip(x, b, scale, bias, BF16) for x in inputs]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = feather_ops.scaled_mm_hip(a, b, scale, bias, BF16)
    for x, y in zip(inputs + inputs[:1], want + want[:1]):
        a.copy_(x)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), y.view(torch.int16))
        feather_ops.scaled_mm_hip(x, b, scale, bias, BF16)


@pytest.mark.gpu
def test_operands_that_require_grad():
    import feather_ops

    a, b, scale, bias = _inputs(1281, 5960, 5248, FP16, True)
    want = feather_ops.scaled_mm_hip(a, b, scale, bias, FP16)
    out = feather_ops.scaled_mm_hip(a.requires_grad_(), b, scale, bias, FP16)
    assert not out.requires_grad and torch.equal(out, want)


@pytest.mark.gpu
def test_refused_operands_are_refused_as_before():
    import feather_ops

    a, b, scale, bias = _inputs(4112, 4096, 4096, FP16, False)
    with pytest.raises(RuntimeError, match="stride"):
        feather_ops.scaled_mm_hip(torch.cat([a, a], dim=1)[:, :4096], b, scale, bias, FP16)
    with pytest.raises(RuntimeError, match="aligned"):
        feather_ops.scaled_mm_hip(torch.empty(a.numel() + 1, device="cuda", dtype=FP16)[1:].view_as(a), b, scale, bias, FP16)
    with pytest.raises(RuntimeError, match="bias"):
        feather_ops.scaled_mm_hip(a, b, scale, bias.to(BF16), FP16)
