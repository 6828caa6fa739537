"""The auto path's one-op launch: the bits of the two-step one, its refusals, and operands autograd follows."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fo():
    import feather_ops

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return feather_ops


def _operands(m, n, k, dtype):
    import feather_ops

    g = torch.Generator("cuda").manual_seed(0)
    w = (torch.randn((n, k), generator=g, device="cuda") * 20).to(torch.float8_e5m2)
    return (torch.randn((m, k), generator=g, device="cuda").to(dtype), feather_ops.prepack_transpose(w),
            torch.tensor(1e-3, device="cuda"))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1, 1000, 2560), (77, 5120, 2560), (16, 14336, 4096), (0, 1000, 2560)])
def test_same_bits_as_a_pinned_launch(fo, m, n, k, dtype):
    from feather_ops.scaled_mm import _auto_plan

    a, b, scale = _operands(m, n, k, dtype)
    parts, _, packed = _auto_plan(m, n, k, dtype)
    assert packed is not None
    for out_dtype in (torch.float16, torch.bfloat16):
        bias = torch.randn(n, device="cuda").to(out_dtype)
        for s in (None, scale, scale.expand(n).contiguous()):
            got = fo.scaled_mm_hip(a, b, s, bias, out_dtype)
            want = fo.scaled_mm_hip(a, b, s, bias, out_dtype, tile=parts[0][1])
            assert got.shape == (m, n) and got.dtype == out_dtype and got.is_contiguous()
            assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_refusals(fo):
    a, b, scale = _operands(4, 64, 128, torch.float16)
    for bad, match in [((a.float(), b, scale, None, torch.float16), "float16 or bfloat16"),
                       ((a[:, :120], b, scale, None, torch.float16), "divisible by 16"),
                       ((torch.cat([a, a], 1)[:, :128], b, scale, None, torch.float16), "stride"),
                       ((a, b.cpu(), scale, None, torch.float16), "CUDA"),
                       ((a, b, scale.double(), None, torch.float16), "float32"),
                       ((a, b, scale, torch.zeros(64, device="cuda"), torch.float16), "same dtype"),
                       ((a, b, scale, None, torch.float32), "float16 or bfloat16")]:
        with pytest.raises((RuntimeError, NotImplementedError), match=match):
            fo.scaled_mm_hip(*bad)


def test_operands_that_require_grad(fo):
    a, b, scale = _operands(4, 64, 128, torch.float16)
    want = fo.scaled_mm_hip(a, b, scale, None, torch.float16)
    for operands in ((a.clone().requires_grad_(), b, scale), (a, b, scale.clone().requires_grad_())):
        out = fo.scaled_mm_hip(*operands, None, torch.float16)
        assert not out.requires_grad and torch.equal(out, want)


def test_other_streams_and_inference_mode(fo):
    a, b, scale = _operands(4, 64, 128, torch.float16)
    want = fo.scaled_mm_hip(a, b, scale, None, torch.float16)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream), torch.inference_mode():
        out = fo.scaled_mm_hip(a, b, scale, None, torch.float16)
        assert out.is_inference()
    torch.cuda.current_stream().wait_stream(stream)
    assert torch.equal(out, want)
