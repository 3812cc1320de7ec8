"""Attention over compressed rows by row tiles that waves share: scores that rise from chunk to chunk, and values near the end of the
range under them."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
#: what a chunk's scores are around, in turn: small and large rises, falls, repeats
LEVELS = (0.0, 5.0, 14.0, -90.0, 12.0, 17.0, 400.0, 399.0, 404.0, 900.0, 0.0)


@pytest.mark.parametrize("heads,rank,rot,window", [(12, 512, 64, 0), (3, 512, 64, 100), (5, 256, 128, 0), (1, 200, 30, 70), (2, 512, 128, 0)])
def test_scores_that_rise_from_chunk_to_chunk(heads, rank, rot, window):
    from pyre_amd.hip import ops

    page, length, dk = 16, 340, rank + rot
    g = torch.Generator().manual_seed(heads * rank + window)
    level = torch.tensor([LEVELS[(t // 32) % len(LEVELS)] for t in range(length)])
    # the last element carries the level: every third head sees it the other way round, every fifth not at all
    q, rows = torch.randn(length, heads, dk, generator=g), torch.randn(length, dk, generator=g)
    sign = torch.tensor([0.0 if h % 5 == 4 else -1.0 if h % 3 == 2 else 1.0 for h in range(heads)])
    scale = 1.0 / dk ** 0.5
    q[:, :, -1], rows[:, -1] = sign, level / scale
    q, rows = q.to(torch.bfloat16), rows.to(torch.bfloat16)
    n_pages = -(-length // page)
    order = torch.randperm(n_pages, generator=g)
    pool = torch.full((n_pages, 1, page, dk), float("nan"), dtype=torch.bfloat16)
    for t in range(length):
        pool[order[t // page], 0, t % page] = rows[t]
    i, j = torch.arange(length)[:, None], torch.arange(length)[None]
    seen = (j <= i) & ((i - j < window) if window else torch.ones(1, dtype=torch.bool))
    s = torch.stack([(q[:, h].double() @ rows.double().T * scale).masked_fill(~seen, float("-inf")) for h in range(heads)])
    want = torch.stack([torch.softmax(x, 1) @ rows.double()[:, :rank] for x in s], 1)
    tiles = [(t, min(32, length - t)) for t in range(0, length, 32)]
    tiles[2:3] = [(64, 5), (69, 1), (70, 26)]
    pos, seq = torch.arange(length, dtype=torch.int32, device=DEV), torch.zeros(length, dtype=torch.int32, device=DEV)
    outs = []
    for sink in (None, torch.full((heads,), 50.0, device=DEV)):
        out = torch.full((length, heads, rank), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops.latent_attn_tile(q.to(DEV), pool.to(DEV), out, torch.tensor(tiles, dtype=torch.int32, device=DEV), len(tiles), pos, seq,
                             order.int()[None].to(DEV), heads, rank, dk, page, scale, window, sink)
        outs.append(out.cpu().double())
    # the output's 16 bits (2^-9 of a value), and scores of up to 1,000 whose float32 sums move a weight by 1,000 * 2^-22
    bound = 3e-3 * float(want.abs().max())
    assert float((outs[0] - want).abs().max()) < bound
    share = torch.stack([torch.exp(torch.logsumexp(x, 1) - torch.logaddexp(torch.logsumexp(x, 1), torch.tensor(50.0, dtype=torch.float64)))
                         for x in s], 1)
    assert float((outs[1] - want * share[:, :, None]).abs().max()) < bound


@pytest.mark.parametrize("heads,rank,rot", [(3, 512, 64), (2, 256, 128)])
def test_values_near_the_end_of_the_range(heads, rank, rot):
    """Scores that rise by 6 from chunk to chunk (8.7 in base two) over values of 2^118: no weight is above 1, so 340 keys stay below
    2^127. The output is an average of the values, whatever the weights."""
    from pyre_amd.hip import ops

    page, length, dk = 16, 340, rank + rot
    scale = 1.0 / dk ** 0.5
    rows, q = torch.full((length, dk), 2.0 ** 118), torch.zeros(length, heads, dk)
    rows[:, -1], q[:, :, -1] = torch.tensor([6.0 * (t // 32) for t in range(length)]) / scale, 1.0
    n_pages = -(-length // page)
    pool = torch.zeros(n_pages * page, dk)
    pool[:length] = rows
    tiles = torch.tensor([(t, min(32, length - t)) for t in range(0, length, 32)], dtype=torch.int32, device=DEV)
    pos, seq = torch.arange(length, dtype=torch.int32, device=DEV), torch.zeros(length, dtype=torch.int32, device=DEV)
    out = torch.full((length, heads, rank), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.latent_attn_tile(q.to(DEV).bfloat16(), pool.to(DEV).bfloat16().view(n_pages, 1, page, dk), out, tiles, tiles.shape[0], pos, seq,
                         torch.arange(n_pages, dtype=torch.int32, device=DEV)[None], heads, rank, dk, page, scale, 0, None)
    # 2^-9 of the result's own 16 bits, and the sums' roundings far below that
    assert float((out.double() / 2.0 ** 118 - 1).abs().max()) <= 2.0 ** -8
