"""Gradients of the fp8 linear layer on the GPU against fp64 on the dequantized weight, over the tiles, tails, formats and
scales the kernels take, and the calls that stay with torch's operations (double backward, batched gradients).

Bound of an element: half a unit of the output type, plus the fp32 sum's rounding, at most depth * 2^-24 of the sum of
the absolute products (every product is exact in fp32 up to the scale's own rounding, one more 2^-24 each)."""

import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu

FP16, BF16, E5M2, E4M3 = torch.float16, torch.bfloat16, torch.float8_e5m2, torch.float8_e4m3fn


@pytest.fixture(scope="module")
def lb():
    from feather_ops import linear_backward

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return linear_backward


@pytest.fixture
def every_size(lb, monkeypatch):
    monkeypatch.setattr(lb, "_MIN_PRODUCTS", 0)
    lb.backward_plan.cache_clear()
    yield
    lb.backward_plan.cache_clear()


def _operands(m, n, k, dtype, fp8, column, size=1e-2, seed=0):
    from feather_ops import prepack_transpose

    g = torch.Generator("cuda").manual_seed(seed)
    w = torch.randn((n, k), generator=g, device="cuda") * k**-0.5
    scale = (w.abs().amax(1) if column else w.abs().max()) / {E5M2: 57344.0, E4M3: 448.0}[fp8]
    wq = (w / (scale[:, None] if column else scale)).to(fp8)
    grad = (torch.randn((m, n), generator=g, device="cuda") * size).to(dtype)
    return grad, wq, scale


def _check(lb, grad, wq, scale, lost=0.0):
    from feather_ops import prepack_transpose

    n, k = wq.shape
    x, bias = lb.linear_backward(grad, prepack_transpose(wq), scale, k, True, True)
    assert x.dtype == bias.dtype == grad.dtype
    w = wq.double() * (scale.double()[:, None] if scale.dim() else scale.double())
    half, least = (2.0**-8, 2.0**-134) if grad.dtype == BF16 else (2.0**-11, 2.0**-25)
    for got, want, terms, depth in ((x, grad.double() @ w, grad.double().abs() @ w.abs(), 3 * n),
                                    (bias, grad.double().sum(0), grad.double().abs().sum(0), grad.shape[0])):
        bound = half * want.abs() + least + (depth + 2) * 2.0**-24 * terms + (lost if got is x else 0.0)
        assert ((got.double() - want).abs() <= bound).all()


# (m, n, k): a row; a depth of one and a half chunks; tails in every axis; N % 16 = 8 on the ring, wide and streaming
# kernels; each kernel's split launch; the wide tiles whole and ragged; 8 outputs on the ring kernel's tiles.
SHAPES = [(1, 1000, 1024), (3, 24, 32), (512, 8, 4096), (4096, 8, 4096), (77, 1000, 2560), (1000, 5120, 2560),
          (300, 1000, 1008), (513, 2568, 1040), (257, 4096, 4096), (20, 16384, 1024), (40, 5120, 12288),
          (4096, 3080, 3072), (4096, 4096, 4096), (1040, 6144, 1536)]


@pytest.mark.parametrize("column", [False, True])
@pytest.mark.parametrize("dtype,fp8", [(FP16, E5M2), (FP16, E4M3), (BF16, E5M2), (BF16, E4M3)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gradients(lb, every_size, m, n, k, dtype, fp8, column):
    _check(lb, *_operands(m, n, k, dtype, fp8, column))


@pytest.mark.parametrize("column", [False, True])
def test_fp16_subnormal_gradients(lb, every_size, column):
    """Unscaled fp16 gradients are often subnormal (below 6e-5)."""
    _check(lb, *_operands(200, 1024, 1024, FP16, E5M2, column, size=2e-6))


@pytest.mark.parametrize("factor", [2.0**-90, -1.0, 0.0, 2.0**60])
@pytest.mark.parametrize("column", [False, True])
def test_scales_of_any_size_and_sign(lb, every_size, column, factor):
    grad, wq, scale = _operands(70, 264, 272, BF16, E4M3, column)
    _check(lb, grad, wq, scale * factor)


@pytest.mark.parametrize("size", [1e-30, 1e-33, 1e-35, 1e-36, 1e-37])
@pytest.mark.parametrize("fp8", [E5M2, E4M3])
@pytest.mark.parametrize("column", [False, True])
def test_bf16_gradients_near_the_least_value(lb, every_size, column, fp8, size):
    """bf16's least normal value is 1.2e-38. At 1e-37 with per-column scales the gradient's last term ends at bf16's least
    step, 2^-133, which meets the codes over the power of two of the scales."""
    grad, wq, scale = _operands(70, 264, 272, BF16, fp8, column, size=size)
    lost = 0.0
    if column and size < 1e-36:
        lost = 2.0**-133 * wq.double().abs().sum(0) * 2.0**(scale.max().log2().floor() + 1).double()
    _check(lb, grad, wq, scale, lost)


@pytest.mark.parametrize("size", [1e-2, 1e-33, 2.0**120])
def test_scales_far_apart(lb, every_size, size):
    """One power of two serves all the columns of a layer, and the largest decides it."""
    grad, wq, scale = _operands(70, 264, 272, BF16, E5M2, True, size=size)
    powers = torch.arange(264, device="cuda") % 33 - 32
    _check(lb, grad, wq, scale * 2.0**powers)


def test_bf16_gradients_near_the_largest_value(lb, every_size):
    """The scale's power of two is in the weight: the sums do not overflow where the result does not."""
    grad, wq, scale = _operands(70, 264, 272, BF16, E5M2, False)
    _check(lb, grad.sign() * 2.0**120, wq, scale)


@pytest.mark.parametrize("column", [False, True])
@pytest.mark.parametrize("fp8", [E5M2, E4M3])
def test_infinities_and_nan(lb, every_size, fp8, column):
    from feather_ops import prepack_transpose

    grad, wq, scale = _operands(70, 264, 272, BF16, fp8, column)
    grad[3, 5], grad[9, 7], grad[20, 11] = float("inf"), float("-inf"), float("nan")
    bits = wq.view(torch.uint8)
    bits[13, 40] = 0x7F       # NaN in both formats
    if fp8 == E5M2:
        bits[17, 50] = 0xFC   # -inf
    packed = prepack_transpose(wq)
    x, bias = lb.linear_backward(grad, packed, scale, 272, True, True)
    want_x, want_bias = lb.composite(grad, packed, scale, 272)
    for got, want in ((x, want_x.to(BF16)), (bias, want_bias.to(BF16))):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        assert torch.equal(got[got.isinf()], want[want.isinf()])


@pytest.mark.parametrize("fp8", [E5M2, E4M3])
@pytest.mark.parametrize("dtype,power", [(FP16, 12), (BF16, 12), (BF16, -20)])
@pytest.mark.parametrize("m,n,k", [(70, 264, 272), (300, 1000, 1008), (1000, 1024, 512), (1040, 6144, 1536)])
def test_results_of_the_last_term_alone(lb, every_size, m, n, k, dtype, power, fp8):
    """Columns in pairs of opposite gradients and equal codes, whose scales differ in the 8 lowest bits: the first two of the
    gradient's three terms cancel. Gradients are +-1, codes of 3 significant bits and scales of one binade, so every sum
    is exact in fp32 (the first term's in steps of 2^-9 under 2^15, the last's of 2^-25) and only the result is rounded."""
    from feather_ops import prepack_transpose

    g = torch.Generator("cuda").manual_seed(0)
    sign = torch.randint(0, 2, (m, n // 2), generator=g, device="cuda") * 2 - 1
    grad = torch.stack([sign, -sign], 2).view(m, n).to(dtype)
    codes = torch.randint(4, 8, (n // 2, k), generator=g, device="cuda") * 0.25
    codes = codes * (torch.randint(0, 2, codes.shape, generator=g, device="cuda") * 2 - 1)
    wq = codes.repeat_interleave(2, 0).to(fp8)
    assert torch.equal(wq.float(), codes.repeat_interleave(2, 0))
    bits = torch.randint(0, 1 << 15, (n // 2,), generator=g, device="cuda").repeat_interleave(2) << 8
    low = torch.randint(0, 1 << 8, (n,), generator=g, device="cuda")
    scale, without = (((bits + x).double() * 2.0**-23 + 1.0) * 2.0**power for x in (low, torch.zeros_like(low)))
    x, _ = lb.linear_backward(grad, prepack_transpose(wq), scale.float(), k, True, False)
    want, two_terms = ((grad.double() * s) @ wq.double() for s in (scale, without))
    half, least = (2.0**-8, 2.0**-134) if dtype == BF16 else (2.0**-11, 2.0**-25)
    assert two_terms.abs().max() == 0.0 and want.abs().max() > 2.0**(power - 14)
    assert ((x.double() - want).abs() <= half * want.abs() + least).all()


def _layer(dtype=BF16, k=1024, n=4104, column=True):
    import feather_ops

    torch.manual_seed(0)
    lin = nn.Linear(k, n, device="cuda", dtype=dtype)
    feather_ops.to_scaled_mm_linear(lin, E4M3, column)
    return lin, torch.randn((2, 33, k), device="cuda").to(dtype).requires_grad_()


def test_expanded_and_strided_gradients(lb):
    lin, x = _layer()
    y = lin(x)
    (gx, gb) = torch.autograd.grad(y.sum(), (x, lin.bias), retain_graph=True)   # a gradient of stride 0
    (wx, wb) = torch.autograd.grad(y, (x, lin.bias), torch.ones_like(y), retain_graph=True)
    assert torch.equal(gx, wx) and torch.equal(gb, wb)
    g = torch.randn((y.shape[-1], 33, 2), device="cuda").to(y.dtype).permute(2, 1, 0)
    assert torch.equal(torch.autograd.grad(y, x, g, retain_graph=True)[0],
                       torch.autograd.grad(y, x, g.contiguous(), retain_graph=True)[0])


def test_double_backward_and_batched_gradients(lb):
    """Both take torch's operations, which have rules for them; the results agree with the kernels' to rounding."""
    lin, x = _layer()
    y = lin(x)
    g = torch.randn_like(y).requires_grad_()
    plain = torch.autograd.grad(y, x, g.detach(), retain_graph=True)[0].float()
    (gx,) = torch.autograd.grad(y, x, g, create_graph=True)
    assert (gx.float() - plain).norm() < 1e-3 * plain.norm()
    v = torch.randn_like(gx)
    (gg,) = torch.autograd.grad(gx, g, v, retain_graph=True)      # d(gx . v) / dg = the layer on v without its bias
    want = lin(v.detach()).float() - lin.bias.float()
    assert (gg.float() - want).norm() < 2e-2 * want.norm()
    (batched,) = torch.autograd.grad(y, x, torch.stack([g.detach(), 2 * g.detach()]), is_grads_batched=True)
    assert (batched[0].float() - plain).norm() < 1e-3 * plain.norm()


def test_compiled_training_step(lb):
    lin, x = _layer()
    model = nn.Sequential(lin, nn.GELU())
    g = torch.randn((2, 33, lin.out_features), device="cuda").to(x.dtype)
    want = torch.autograd.grad(lin(x), (x, lin.bias), g)
    got = torch.autograd.grad(torch.compile(lin, fullgraph=True)(x), (x, lin.bias), g)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert torch.autograd.grad(model(x).sum(), x)[0].isfinite().all()


def test_only_what_is_asked_for(lb):
    lin, x = _layer()
    y = lin(x.detach())
    (gb,) = torch.autograd.grad(y.sum(), lin.bias)
    lin.bias.requires_grad_(False)
    y = lin(x)
    (gx,) = torch.autograd.grad(y.sum(), x)
    assert gb.isfinite().all() and gx.isfinite().all()
