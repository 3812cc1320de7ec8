"""The walk of gated linear attention in chunks, whose prompts are cut into segments that are walked at the same time: against
the recurrence in float64, token by token."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("heads,dk,dv", [(3, 128, 128), (5, 40, 24), (1, 17, 250), (2, 200, 16), (1, 12, 100), (2, 256, 36)])
@pytest.mark.parametrize("lengths", [[1, 700, 3], [64], [65], [80, 81, 79, 1, 1], [1300], [129, 5, 512]])
def test_segments(heads, dk, dv, lengths):
    from pyre_amd.hip import ops

    n, hk, hv = sum(lengths), heads * dk, heads * dv
    g = torch.Generator().manual_seed(n + dk)
    x = torch.randn(n, 3 * hk + 2 * hv, generator=g)
    # decays from one that forgets at once to one that keeps all
    x[:, 2 * hk:3 * hk] = -torch.rand(n, hk, generator=g) ** 4 * torch.logspace(-4, 1.2, hk)[torch.randperm(hk, generator=g)]
    slots = torch.randperm(len(lengths) + 2, generator=g)[:len(lengths)]
    state = torch.randn(len(lengths) + 2, heads, dk, dv, generator=g)
    starts = [0]
    for m in lengths:
        starts.append(starts[-1] + m)
    out = torch.full((n, hv), float("nan"), device=DEV)
    after = state.to(DEV)
    scratch = torch.full((ops.gla_chunks_scratch(n, len(lengths), heads, dk, dv),), float("nan"), device=DEV)
    ops.gla_scan(x.to(DEV), after, out, torch.tensor(starts, dtype=torch.int32, device=DEV),
                 torch.tensor(slots.tolist(), dtype=torch.int32, device=DEV), len(lengths), heads, dk, dv, dk ** -0.5, scratch, max(lengths))
    q, k, ld, v = (x[:, a:b].double().view(n, heads, -1) for a, b in ((0, hk), (hk, 2 * hk), (2 * hk, 3 * hk), (3 * hk, 3 * hk + hv)))
    want, wanted_state = torch.empty(n, heads, dv, dtype=torch.float64), state.double().clone()
    for s, m in enumerate(lengths):
        S = wanted_state[slots[s]]
        for t in range(starts[s], starts[s] + m):
            S = torch.exp(ld[t])[:, :, None] * S + k[t][:, :, None] * v[t][:, None, :]
            want[t] = torch.einsum("hdv,hd->hv", S, q[t]) * dk ** -0.5
        wanted_state[slots[s]] = S
    # sums of up to `reach` tokens of products of values around one, in float32; the exponents of a chunk are sums of sixteen logarithms
    for got, ref in ((out.cpu().double().view(n, heads, dv), want), (after.cpu().double(), wanted_state)):
        assert bool(torch.isfinite(got).all())
        assert float((got - ref).abs().max() / ref.pow(2).mean().sqrt()) <= 1e-4
        assert float((got - ref).norm() / ref.norm()) <= 4e-6


@pytest.mark.parametrize("heads,dk,dv", [(14, 128, 128), (3, 40, 24), (2, 256, 36), (1, 17, 250)])
@pytest.mark.parametrize("lengths", [[300, 1777], [700, 1, 65, 64, 1, 2, 700, 130], [1] * 70 + [513] + [40] * 70])
def test_a_request_has_the_same_bits_alone_and_among_others(heads, dk, dv, lengths):
    """Outputs and states of every request of a step, among them more than a wave has lanes, beside each by itself."""
    from pyre_amd.hip import ops

    n, hk, hv = sum(lengths), heads * dk, heads * dv
    g = torch.Generator().manual_seed(n + dk)
    x = torch.randn(n, 3 * hk + 2 * hv, generator=g)
    x[:, 2 * hk:3 * hk] = -torch.rand(n, hk, generator=g) ** 4 * torch.logspace(-4, 1.2, hk)
    x = x.to(DEV)
    state = torch.randn(len(lengths), heads, dk, dv, generator=g).to(DEV)

    def walk(first, lens, states):
        starts = [0]
        for m in lens:
            starts.append(starts[-1] + m)
        out = torch.full((starts[-1], hv), float("nan"), device=DEV)
        after = states.clone()
        scratch = torch.full((ops.gla_chunks_scratch(starts[-1], len(lens), heads, dk, dv),), float("nan"), device=DEV)
        ops.gla_scan(x[first:first + starts[-1]].contiguous(), after, out, torch.tensor(starts, dtype=torch.int32, device=DEV),
                     torch.arange(len(lens), dtype=torch.int32, device=DEV), len(lens), heads, dk, dv, dk ** -0.5, scratch, max(lens))
        return out, after

    out, after = walk(0, lengths, state)
    at = 0
    for s, m in enumerate(lengths):
        if m > 1 or s < 2:
            alone, state_alone = walk(at, [m], state[s:s + 1])
            assert torch.equal(alone, out[at:at + m]), s
            assert torch.equal(state_alone[0], after[s]), s
        at += m
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(after).all())
