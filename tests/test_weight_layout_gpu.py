"""Laying out and quantizing a weight stored [N, K]: the kernels' bytes and scales are those of torch's operations."""

import pytest
import torch

pytestmark = pytest.mark.gpu

FP8_MAX = {torch.float8_e5m2: 57344.0, torch.float8_e4m3fn: 448.0}


@pytest.fixture(scope="module")
def fo():
    import feather_ops

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return feather_ops


def _packed(w):
    n, k = w.shape
    w = torch.nn.functional.pad(w.view(torch.uint8), (0, -k % 128))
    return w.view(n, -1, 16).transpose(0, 1).contiguous()


def _quantized(w, fp8, per_channel):
    w = w.float()
    amax = w.abs().amax(dim=1) if per_channel else w.abs().max().reshape(1)
    scale = torch.where(amax > 0, amax / FP8_MAX[fp8], torch.ones_like(amax))
    return (w / (scale[:, None] if per_channel else scale)).to(fp8), scale if per_channel else scale.reshape(())


def _check_quantized(w, fp8, per_channel):
    from feather_ops.scaled_mm import quantize_and_pack

    codes, scale = quantize_and_pack(w, fp8, per_channel)
    want, want_scale = _quantized(w, fp8, per_channel)
    assert codes.dtype == fp8 and scale.shape == want_scale.shape
    assert torch.equal(scale.view(torch.int32), want_scale.view(torch.int32))
    assert torch.equal(codes.view(torch.uint8), _packed(want))


# (n, k): one unit; a tail of rows, of units, of both; whole tiles; a K with no pad; the sides of 2 MiB, where codes without
# a pad go from torch's copy to the kernel
SHAPES = [(1, 16), (33, 48), (264, 640), (1000, 2560), (32, 512), (40, 1040), (4096, 128), (4096, 512), (4104, 512)]


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("fp8", list(FP8_MAX))
def test_prepack_of_a_linear_weight(fo, n, k, fp8):
    torch.manual_seed(0)
    w = torch.randint(0, 256, (n, k), device="cuda", dtype=torch.uint8).view(fp8)
    assert torch.equal(fo.prepack_transpose(w).view(torch.uint8), _packed(w))
    assert torch.equal(fo.prepack_b_for_scaled_mm(w.t()).view(torch.uint8), _packed(w))
    storage = torch.empty(n * k + 1, device="cuda", dtype=torch.uint8)
    shifted = storage[1:].view(n, k).copy_(w.view(torch.uint8)).view(fp8)     # not 16-byte aligned: torch's copies
    assert torch.equal(fo.prepack_transpose(shifted).view(torch.uint8), _packed(w))
    assert torch.equal(fo.prepack_transpose(w[:, : k - 8]).view(torch.uint8), _packed(w[:, : k - 8].contiguous()))


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("fp8", list(FP8_MAX))
@pytest.mark.parametrize("per_channel", [False, True])
def test_quantize(fo, n, k, dtype, fp8, per_channel):
    torch.manual_seed(0)
    w = (torch.randn((n, k), device="cuda") * torch.rand((n, 1), device="cuda") * 0.1).to(dtype)
    if n > 8:
        w[5] = 0.0      # a row of zeros: scale 1
    _check_quantized(w, fp8, per_channel)


@pytest.mark.parametrize("fp8", list(FP8_MAX))
@pytest.mark.parametrize("per_channel", [False, True])
def test_quantize_every_bf16_value(fo, fp8, per_channel):
    """Every bf16 bit pattern in rows of 256: subnormals, infinities and NaN rows among them; and next to a row of
    ordinary values whose scale they then share, or do not."""
    bits = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(torch.bfloat16).reshape(256, 256)
    _check_quantized(bits, fp8, per_channel)
    finite = torch.where(bits.isfinite(), bits, torch.zeros_like(bits))
    _check_quantized(finite, fp8, per_channel)
    _check_quantized(finite * 2.0**-100, fp8, per_channel)


@pytest.mark.parametrize("fp8", list(FP8_MAX))
def test_quantize_ties_and_ends(fo, fp8):
    """fp32 weights whose quotients lie on, and one unit beside, the points where rounding changes, for scales of any
    mantissa: the quotient's own rounding decides there."""
    codes = torch.arange(256, device="cuda", dtype=torch.int32).to(torch.uint8).view(fp8).float()
    codes = codes[codes.isfinite()].sort().values
    middle = ((codes[1:] + codes[:-1]) / 2).clamp(-FP8_MAX[fp8], FP8_MAX[fp8])
    torch.manual_seed(1)
    scale = torch.rand(512, 1, device="cuda") * 2.0 ** torch.randint(-20, 20, (512, 1), device="cuda")
    w = middle[None] * scale
    bits = w.view(torch.int32)
    w = torch.cat([w, (bits + 1).view(torch.float32), (bits - 1).view(torch.float32)], dim=1)
    w = torch.nn.functional.pad(w, (0, -w.shape[1] % 16))
    w[:, -1] = FP8_MAX[fp8] * scale[:, 0]
    _check_quantized(w.nan_to_num(0.0), fp8, True)
    _check_quantized(torch.randn(2048, 2048, device="cuda").exp(), fp8, True)
    _check_quantized(torch.randn(512, 512, device="cuda") * 1e-30, fp8, False)


def test_relabelled_linear_uses_the_same_bytes(fo):
    torch.manual_seed(0)
    lin = torch.nn.Linear(640, 264, device="cuda", dtype=torch.bfloat16)
    want, scale = _quantized(lin.weight.detach(), torch.float8_e4m3fn, True)
    fo.to_scaled_mm_linear(lin, torch.float8_e4m3fn, per_channel=True)
    assert torch.equal(lin.weight_fp8.view(torch.uint8), _packed(want)) and torch.equal(lin.weight_scale, scale)
    assert "weight_fp8" not in lin.state_dict()
