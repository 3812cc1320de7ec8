"""Gated units of few rows: blocks of 32, 40, 48, 64, 80 and 96 features (the last tile of 40 is half a tile), rows of X on both sides of
what is loaded of them (8, 16, 32), against float64; a row's result is the same bits whatever rows share the step."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 33, 65, 97, 129, 256])
@pytest.mark.parametrize("inter,k", [(8192, 200), (10239, 64), (12280, 136), (16384, 72), (20473, 64), (22000, 128)])
def test_features_of_a_block(m, inter, k):
    from pyre_amd.hip import ops

    g = torch.Generator(device=DEV).manual_seed(inter + m)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn(2 * inter, k, generator=g, device=DEV) * 0.1).bfloat16()
    out = torch.full((m, inter), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.gemm_mid_silu_bf16(x, w, out, m)
    gu = x.double() @ w.double().T
    want = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    # float32 sums (k 2^-24 of sums of size 1) and one rounding to 16 bits
    assert bool(((out.double() - want).abs() <= 2 ** -8 * want.abs() + 1e-5).all())
    rows = sorted({0, m // 2, m - 1})
    few = torch.full((len(rows), inter), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.gemm_mid_silu_bf16(x[rows].contiguous(), w, few, len(rows))
    assert torch.equal(few, out[rows])


@pytest.mark.parametrize("inter,m", [(20473, 66), (20473, 80), (20473, 96), (24571, 96), (27643, 25), (27643, 31), (27643, 32), (27643, 64)])
def test_few_rows_of_many_features(inter, m):
    """80 features against the 96 rows of X that are loaded, and 128."""
    test_features_of_a_block(m, inter, 136)
