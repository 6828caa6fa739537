"""The streaming kernel past 16 rows: its tile order."""

import pytest
import torch

FP16, BF16 = torch.float16, torch.bfloat16


def _check(m, n, k, tile, dtype, splits=1):
    import feather_ops
    from gpu_helpers import check_against_oracle

    g = torch.Generator("cuda").manual_seed(m * n + k)
    a = torch.randn((m, k), generator=g, device="cuda").to(dtype)
    b = feather_ops.prepack_transpose((torch.randn((n, k), generator=g, device="cuda") * 20).to(torch.float8_e5m2))
    scale, bias = torch.tensor(1e-3, device="cuda"), torch.randn(n, generator=g, device="cuda").to(dtype)
    out = feather_ops.scaled_mm_hip(a, b, scale, bias, dtype, tile=tile, splits=splits)
    check_against_oracle(out, a, b, scale, bias)


@pytest.mark.gpu
@pytest.mark.parametrize("columns", [1, 7, 8, 9, 12, 20, 24])
@pytest.mark.parametrize("rows", [1, 2, 3, 13])
def test_every_tile_is_computed_once(rows, columns):
    """Rows and columns of tiles around the orders' boundaries (8 XCDs; runs of unequal length), the last ones partial."""
    _check(16 * rows - 3, 64 * columns - 8, 272, (4, 1, 4, 1, 4, 0), FP16)
    _check(16 * rows - 3, 64 * columns - 8, 1040, (4, 1, 4, 1, 4, 0), BF16, splits=2)
