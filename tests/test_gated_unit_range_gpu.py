"""The gated unit in the epilogues of the 16-bit gate/up products, over the gates whose exponential float32 holds."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("product,m", [("skinny", 5), ("mid", 5), ("mid", 130), ("tile", 70), ("tile", 300)])
@pytest.mark.parametrize("unit", [None, (0.0, 0.5, 1.0), (0.0, 1.0, 0.0, 0.125)])
def test_gates_of_all_sizes(product, m, unit):
    """A feature's gate is one weight, its up value 2^40: what a very negative gate leaves of it is an ordinary number, also where
    1 + exp(-slope gate) is beyond 2^126 and its reciprocal no longer a normal one."""
    from pyre_amd.hip import ops

    k, inter = 512, 512
    slope, shift, cubic = (1.0, 0.0, 0.0) if unit is None else (unit[1], unit[2], unit[3] if len(unit) > 3 else 0.0)
    z = torch.cat([torch.linspace(-88.5, -80.0, 200, dtype=torch.float64), torch.linspace(-80.0, 90.0, inter - 200, dtype=torch.float64)])
    # the gate whose argument of the exponential is z, rounded towards zero to bfloat16
    gate = z / slope
    if cubic:
        for _ in range(200):
            gate = gate - (gate + cubic * gate ** 3 - z / slope) / (1 + 3 * cubic * gate ** 2)
    gate = (gate * (1 - 2.0 ** -8)).to(torch.bfloat16)
    w = torch.zeros(2 * inter, k, dtype=torch.bfloat16)
    w[:inter, 7], w[inter:, 7] = gate, 2.0 ** 40
    x = torch.zeros(m, k, dtype=torch.bfloat16)
    x[:, 7] = 1.0
    w, x = w.to(DEV), x.to(DEV)
    out = torch.full((m, inter), float("nan"), device=DEV, dtype=torch.bfloat16)
    {"skinny": ops.gemm_skinny_silu_bf16, "mid": ops.gemm_mid_silu_bf16, "tile": ops.gemm_tile_glu_bf16}[product](x, w, out, m, unit)
    g = gate.double()
    want = g * torch.sigmoid(slope * (g + cubic * g ** 3)) * (2.0 ** 40 + shift)
    # half a unit of bfloat16's 8 bits; the exponential's argument, up to 128, is rounded a few times to 2^-24 of it
    assert bool(((out.cpu().double() - want).abs() <= want.abs() * (2.0 ** -8 + 2.0 ** -13)).all())
