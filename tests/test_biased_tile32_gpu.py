"""Attention with biases, caps, windows and gates over prompt portions in float32: blocks of sixteen tokens and two heads whose
keys are dealt to several waves, against float64."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("nq,nkv,dk,dv,page,window,keep,chunk,cap,far,sink_on,gate_dim", [
    (5, 1, 128, 128, 16, 0, 0, 0, 50.0, 700, False, 1), (6, 2, 64, 40, 16, 100, 5, 0, 20.0, 33, True, 0), (3, 3, 24, 64, 12, 300, 40, 0, 0.0, 0, False, 2),
    (4, 2, 96, 256, 16, 0, 0, 96, 0.0, 200, True, 2), (7, 1, 32, 16, 8, 1, 130, 0, 3.0, 90, False, 1), (2, 1, 128, 200, 16, 40, 0, 0, 0.0, 0, True, 0),
    (2, 2, 128, 128, 16, 64, 4, 0, 9.0, 40000, False, 1)])
def test_against_64_bits_however_tokens_are_cut(nq, nkv, dk, dv, page, window, keep, chunk, cap, far, sink_on, gate_dim):
    """Two requests, one that goes on behind earlier keys; what lies behind a request's last key and in pages of nobody is not a
    number; the same bits whatever the tiles; biases that do not fit into a compute unit's memory."""
    from pyre_amd.hip import ops

    g = torch.Generator().manual_seed(nq * dk + window)
    lens, first = (450, 190), (0, 111)
    rows = [(r, t) for r in (0, 1) for t in range(first[r], lens[r])]
    n = len(rows)
    ks, vs = [torch.randn(m, nkv, dk, generator=g) for m in lens], [torch.randn(m, nkv, dv, generator=g) for m in lens]
    q = torch.randn(n, nq, dk, generator=g)
    pages = [-(-m // page) for m in lens]
    order = torch.randperm(sum(pages) + 3, generator=g)
    kc, vc = (torch.full((sum(pages) + 3, nkv, page, d), float("nan")) for d in (dk, dv))
    table = torch.full((2, pages[0]), -1, dtype=torch.int32)
    for r in (0, 1):
        table[r, :pages[r]] = order[r * pages[0]:r * pages[0] + pages[r]].int()
        for t in range(lens[r]):
            kc[table[r, t // page], :, t % page], vc[table[r, t // page], :, t % page] = ks[r][t], vs[r][t]
    sink = torch.randn(nq, generator=g) + 2 if sink_on else None
    bias = torch.randn(nq, far + 1, generator=g) if far else None
    gate = torch.rand(n, nq * (dv if gate_dim == 2 else 1), generator=g) if gate_dim else None
    scale = 2.0 / dk ** 0.5
    want, at = torch.zeros(n, nq, dv, dtype=torch.float64), 0
    for r in (0, 1):
        i, j = torch.arange(first[r], lens[r])[:, None], torch.arange(lens[r])[None]
        seen = (j <= i) & (((i - j < window) | (j < keep)) if window else torch.ones(1, dtype=torch.bool))
        if chunk:
            seen = seen & (i // chunk == j // chunk)
        m = lens[r] - first[r]
        for head in range(nq):
            x = q[at:at + m, head].double() @ ks[r][:, head // (nq // nkv)].double().T * scale
            x = cap * torch.tanh(x / cap) if cap else x
            if bias is not None:
                x = x + bias[head].double()[(i - j).clamp(0, far)]
            x = x.masked_fill(~seen, -math.inf)
            if sink_on:
                x = torch.cat([x, sink[head].double().expand(m, 1)], 1)
            want[at:at + m, head] = torch.softmax(x, -1)[:, :lens[r]] @ vs[r][:, head // (nq // nkv)].double()
        at += m
    if gate is not None:
        want = want * gate.double().view(n, nq, -1)
    want = (want * 0.5).reshape(n, -1)
    d = lambda t: None if t is None else t.contiguous().to(DEV)  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    outs = []
    for width in (32, 16, 7):
        tiles = [(t, min(width, end - t)) for begin, end in ((0, 450), (450, n)) for t in range(begin, end, width)] + [(0, 0)]
        out = torch.zeros(n, nq * dv + 3, device=DEV)
        ops.attn_biased_tile(d(q.view(n, -1)), out, d(kc), d(vc), d(gate), 0.5, i32(tiles), len(tiles), i32([t for _, t in rows]),
                             i32([r for r, _ in rows]), d(table), nq, nkv, dk, dv, page, scale, cap, d(bias), far, window, keep, chunk,
                             sink=d(sink), gate_dim=dv if gate_dim == 2 else 1)
        got = out[:, :nq * dv].cpu().double()
        # float32 sums of up to 450 weighted values of around one, scores of up to ten: a few 1e-6
        assert bool(((got - want).abs() <= 2e-5).all()), (width, float((got - want).abs().max()))
        assert not bool(out[:, nq * dv:].any())
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("nq,nkv,dk,dv,page,window,keep,chunk,far", [
    (5, 1, 128, 128, 16, 0, 0, 0, 300), (6, 2, 64, 40, 16, 60, 40, 0, 33), (3, 3, 24, 64, 12, 100, 70, 0, 0), (4, 2, 96, 128, 16, 0, 0, 96, 40000),
    (7, 1, 32, 16, 8, 1, 130, 0, 0), (8, 1, 64, 64, 16, 33, 1, 0, 64), (2, 1, 128, 200, 16, 40, 0, 0, 0)])
def test_portions_of_many_tiles_have_the_bits_of_one_alone(nq, nkv, dk, dv, page, window, keep, chunk, far):
    """Tiles that fill the chip run in blocks of whole tiles whose waves have two parts of the keys each, few tiles in blocks of sixteen
    tokens and a wave for every part: first and last chunks of every part, kept tokens and windows that begin in any of them, halves
    of tiles that are not there."""
    from pyre_amd.hip import ops

    cases = [(0, 1), (0, 17), (0, 32), (31, 2), (32, 16), (33, 31), (64, 5), (95, 33), (127, 20), (128, 1), (129, 48), (250, 40)]
    repeat, pages = 90, -(-290 // page)
    rnd = lambda *shape, seed: torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)  # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    kc, vc = rnd(len(cases) * pages, nkv, page, dk, seed=1), rnd(len(cases) * pages, nkv, page, dv, seed=2)
    table = torch.randperm(len(cases) * pages, generator=torch.Generator().manual_seed(3)).view(len(cases), pages).int().to(DEV)
    bias = rnd(nq, far + 1, seed=4) if far else None

    def run(which):
        pos, seq, tiles, n = [], [], [], 0
        for r in which:
            first, count = cases[r]
            tiles += [(n + t, min(32, count - t)) for t in range(0, count, 32)]
            pos += range(first, first + count)
            seq += [r] * count
            n += count
        q = torch.cat([rnd(cases[r][1], nq * dk, seed=10 + r) for r in which])
        out = torch.full((n, nq * dv), float("nan"), device=DEV)
        ops.attn_biased_tile(q, out, kc, vc, None, 0.5, i32(tiles), len(tiles), i32(pos), i32(seq), table, nq, nkv, dk, dv, page, dk ** -0.5, 30.0,
                             bias, far, window, keep, chunk)
        return out

    alone = torch.cat([run([r]) for r in range(len(cases))])
    assert not bool(alone.isnan().any())
    assert torch.equal(run(list(range(len(cases))) * repeat), alone.repeat(repeat, 1))
