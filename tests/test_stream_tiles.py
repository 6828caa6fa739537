"""The streaming kernel past 16 rows: its tile order, its taller tiles, and the rule that picks them."""

import random

import pytest
import torch

from feather_ops.scaled_mm import _STREAM_REFINED, _STREAM_TIME, _auto_choice, _refined, _stream_time
from feather_ops.tiles import SCALED_MM_TILES, split_workspace_bytes

FP16, BF16 = torch.float16, torch.bfloat16


def test_rule_stays_in_its_range():
    assert set(_STREAM_TIME) <= set(SCALED_MM_TILES) and all(t[5] == 0 for t in _STREAM_TIME)
    rng = random.Random(0)
    changed = set()
    for _ in range(6000):
        m, n, k = int(2 ** rng.uniform(0, 11)), 8 * int(2 ** rng.uniform(4, 11)), 16 * int(2 ** rng.uniform(3, 10))
        for dtype in (FP16, BF16):
            tile, splits, widen = _auto_choice(m, n, k, dtype)
            got, got_splits = _refined(m, n, k, tile, splits, dtype == BF16 and not widen)
            if (got, got_splits) == (tile, splits):
                continue
            changed.add((got, got_splits > 1))
            assert got in _STREAM_REFINED and tile[5] == 0
            assert 16 < m <= 704 and min(n, k) >= 512
            if got_splits > 1:
                assert m <= 32 and 0 < split_workspace_bytes(m, n, k, got, got_splits) < 64 << 20
                assert k // got_splits >= 3072 and 200 <= -(-n // 64) * got_splits <= 256
            else:
                assert splits == 1
                assert _stream_time(m, n, k, got, dtype == BF16) < _stream_time(m, n, k, tile, dtype == BF16)
    assert len(changed) >= 7 and any(split for _, split in changed)


NEW = [(4, 1, 4, 2, 2, 0), (4, 1, 4, 2, 4, 0), (8, 1, 4, 2, 4, 0), (4, 1, 4, 3, 4, 0), (4, 1, 4, 4, 4, 0)]


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


@pytest.mark.gpu
@pytest.mark.parametrize("columns", [2, 3, 5, 8])
@pytest.mark.parametrize("rows", [2, 9, 16, 27, 42])
def test_every_tile_of_a_tall_problem_is_computed_once(rows, columns):
    """Both sides of N = 4/3 M, where the runs turn from columns to rows; rows not a multiple of the 8 XCDs."""
    _check(16 * rows - 3, 64 * columns - 8, 272, (4, 1, 4, 1, 4, 0), FP16)
    _check(16 * rows, 64 * columns, 1040, (4, 1, 4, 1, 4, 0), BF16, splits=2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [FP16, BF16])
@pytest.mark.parametrize("tile", NEW + [(2, 2, 4, 4, 2, 0), (8, 1, 8, 1, 4, 0)])
def test_tall_tiles(tile, dtype):
    """Tails in every axis, K shorter than one round of the K slices and past two (the join lies over the activations)."""
    bm = 16 * tile[3]
    for m in (1, bm - 1, bm + 1, 3 * bm):
        for k in (16, 64 * tile[0] - 16, 128 * tile[0] + 48):
            _check(m, 200, k, tile, dtype)
    _check(2 * bm + 5, 136, 2064, tile, dtype, splits=3)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [FP16, BF16])
@pytest.mark.parametrize("m,n,k", [(77, 5120, 2560), (128, 3072, 3072), (300, 3072, 2560), (17, 4104, 528), (250, 2760, 1104),
                                   (25, 4736, 9216), (32, 5640, 12160)])
def test_auto_path(m, n, k, dtype):
    import feather_ops
    from gpu_helpers import check_against_oracle

    g = torch.Generator("cuda").manual_seed(0)
    a = torch.randn((m, k), generator=g, device="cuda").to(dtype)
    b = feather_ops.prepack_transpose((torch.randn((n, k), generator=g, device="cuda") * 20).to(torch.float8_e4m3fn))
    scale = torch.rand(n, generator=g, device="cuda") * 1e-3
    check_against_oracle(feather_ops.scaled_mm_hip(a, b, scale, None, dtype), a, b, scale, None)
