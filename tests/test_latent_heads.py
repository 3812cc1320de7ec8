"""Prompt portions over keys and values that are made of compressed rows: which portions go that way and how they are cut,
the product over paged rows and the attention kernel alone against float64, and both ways beside each other in an engine."""

from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from pyre_amd.parts import latent_attention as L

DEV = "cuda:0"


def spec_of(window, rank=512, heads=2):
    return SimpleNamespace(window=window, rank=rank, rot_dim=64, key_dim=128, value_dim=128, num_heads=heads)


def batch_of(portions):
    """(start, tokens) of every request, as the engine lays them out."""
    counts = [n for _, n in portions]
    q_start = np.cumsum([0] + counts).astype(np.int32)
    seq = np.repeat(np.arange(len(counts), dtype=np.int32), counts)
    positions = np.concatenate([np.arange(a, a + n) for a, n in portions]).astype(np.int32)
    hb = SimpleNamespace(q_start=q_start, seq_of_token=seq, positions=positions, arrays={})
    from pyre_amd.parts.attention import _prefill_tiles

    hb.arrays["attention.prefill_tiles"] = _prefill_tiles(hb)
    return hb


def test_pairs_of_a_portion():
    for start, n, window in [(0, 1, 0), (0, 5, 3), (7, 4, 3), (2, 9, 5), (5, 3, 9), (3, 6, 9), (4, 2, 0), (0, 8, 8), (8, 8, 8), (0, 9, 8)]:
        want = sum(min(p + 1, window) if window else p + 1 for p in range(start, start + n))
        assert L.portion_pairs(start, n, window) == want


@pytest.mark.parametrize("window", [0, 1, 50, 1024])
def test_the_plan_covers_every_portion_once_and_fits_its_capacity(window):
    spec = spec_of(window)
    portions = [(0, 300), (0, 1), (40, 65), (5000, 9), (3, 64), (1000, 1), (900, 130), (0, 2), (30000, 700)]
    hb = batch_of(portions)
    tiles, groups = L.plan_tiles(hb, spec), L.plan_groups(hb, spec)
    made = {s for s, (a, n) in enumerate(portions) if n > 1 and L.makes_heads(a, n, spec)}
    assert made == set(tiles[:, 3].tolist()) == set(groups[:, 0].tolist()) and 0 in made
    assert window not in (0, 1024) or 3 not in made  # nine tokens behind many keys
    tokens = np.concatenate([np.arange(t, t + n) for t, n in tiles[:, :2]])
    assert sorted(tokens) == [t for t in range(len(hb.seq_of_token)) if hb.seq_of_token[t] in made]
    position = {}  # (request, position) -> row
    for g, (s, p, last) in enumerate(groups):
        for i in range(L.GROUP):
            position.setdefault((s, min(p + i, last)), L.GROUP * g + i)
    for t0, n, pos, s, base in tiles:
        assert hb.positions[t0] == pos and hb.seq_of_token[t0] == s and n <= 64
        for p in range(max(0, pos - window + 1) if window else 0, pos + n):
            assert position[(s, p)] == base + p
    n_cap, s_cap = len(hb.seq_of_token), len(portions)
    assert groups.size <= 3 * (L.MOST_KEYS * n_cap // L.GROUP + 2 * s_cap) and tiles.size <= 5 * (n_cap // 64 + s_cap)
    assert plan_sums(L.plan_rounds(hb, spec)) == (len(groups), len(tiles))


def plan_sums(rounds):
    return tuple(int(x) for x in rounds.sum(axis=0))


def test_a_step_with_more_keys_than_are_made_at_a_time_makes_them_in_rounds(monkeypatch):
    spec = spec_of(100)
    portions = [(0, 300), (40, 65), (5000, 90), (0, 31), (900, 130)]
    monkeypatch.setattr(L, "MADE_BYTES", 352 * spec.num_heads * 512)  # 352 rows
    hb = batch_of(portions)
    rounds, tiles, groups = L.plan_rounds(hb, spec), L.plan_tiles(hb, spec), L.plan_groups(hb, spec)
    assert rounds[:, 0].tolist() == [10, 11, 8] and plan_sums(rounds) == (len(groups), len(tiles))
    at = 0
    for turn, (g, t) in enumerate(rounds):
        assert 32 * g <= 352 and sorted(set(tiles[at:at + t, 3])) == [[0], [1, 2, 3], [4]][turn]
        for t0, n, pos, s, base in tiles[at:at + t]:
            lo = max(0, portions[s][0] - 99)
            assert 0 <= base + lo and base + pos + n <= 32 * g  # rows of its own round
        at += t
    monkeypatch.setattr(L, "MADE_BYTES", 319 * spec.num_heads * 512)
    assert 0 not in L.plan_tiles(hb, spec)[:, 3]  # a portion with more than fit runs over the rows


@pytest.mark.parametrize("rank,heads,window,start,n,made", [
    (512, 12, 1024, 0, 16, True), (512, 12, 1024, 2048, 952, True), (512, 12, 1024, 1000, 64, True), (512, 28, 0, 8000, 1000, True),
    (512, 64, 1024, 1000, 128, True), (256, 28, 0, 8000, 256, True), (256, 12, 0, 1000, 128, True), (192, 4, 0, 0, 700, True),
    (512, 64, 1024, 1000, 32, False), (512, 64, 1024, 1000, 64, False), (512, 64, 0, 3000, 64, False), (256, 64, 0, 1000, 64, False),
    (256, 64, 0, 8000, 128, False), (256, 28, 0, 8000, 128, False), (192, 28, 0, 8000, 128, False), (256, 128, 1024, 1000, 64, False)])
def test_the_way_that_is_faster_where_portions_fill_the_chip(rank, heads, window, start, n, made):
    """Both ways measured, sixteen portions in a step: :func:`makes_heads` has the times."""
    assert L.makes_heads(start, n, spec_of(window, rank, heads)) == made


def test_a_portion_goes_its_way_whatever_runs_beside_it():
    spec = spec_of(1024)
    alone = L.plan_tiles(batch_of([(700, 90)]), spec)
    beside = L.plan_tiles(batch_of([(0, 33), (700, 90), (9, 1)]), spec)
    assert len(alone) and (beside[:, 3] == 1).sum() == len(alone)


def paged(rows, page, order, spare):
    pool = torch.full((len(order) + spare, 1, page, rows.shape[1]), float("nan"), dtype=rows.dtype)
    for t in range(rows.shape[0]):
        pool[order[t // page], 0, t % page] = rows[t]
    return pool


@pytest.mark.gpu
@pytest.mark.parametrize("heads,rank,window,page,start,n", [(1, 64, 0, 16, 0, 1), (3, 128, 40, 16, 0, 200), (2, 512, 0, 8, 0, 129),
                                                            (2, 192, 70, 5, 333, 150), (1, 64, 1, 16, 63, 66), (5, 64, 64, 32, 64, 64), (1, 64, 0, 1, 3950, 140),
                                                            (2, 256, 1024, 16, 1000, 321), (12, 512, 1024, 16, 0, 700), (11, 64, 0, 16, 10, 260)])
def test_made_keys_and_values_and_attention_over_them(heads, rank, window, page, start, n):
    """Pages in no order, NaN where no key lies; tiles that are not full. The product to its output's rounding; the attention
    against float64 on the keys and values as stored: scores, weights and sums are float32, the output is rounded once, 2^-9 of it."""
    from pyre_amd.hip import ops

    g = torch.Generator().manual_seed(heads * rank + n)
    kd, rot, vd, length = 128, 64, 128, start + n
    rows = torch.randn(length, rank + rot, generator=g).bfloat16()
    w = (torch.randn(heads * (kd + vd), rank, generator=g) / rank ** 0.5).bfloat16()
    q = torch.randn(n, heads, kd, generator=g).bfloat16()
    wide = torch.randn(n, heads, rank + rot, generator=g).bfloat16()
    gate, sink = torch.rand(n, heads * vd, generator=g), torch.randn(heads, generator=g) + 1.0
    n_pages = -(-length // page)
    order = torch.randperm(n_pages + 3, generator=g)[:n_pages]
    pool = paged(rows, page, order, 3).to(DEV)
    table = torch.full((2, n_pages + 2), -1, dtype=torch.int32)
    table[1, :n_pages] = order.int()
    lo = max(0, start - window + 1) if window else 0
    table[1, :lo // page] = -1  # released: the window has passed them
    table = table.to(DEV)

    groups = torch.tensor([(1, p, length - 1) for p in range(lo, length, 32)], dtype=torch.int32, device=DEV)
    kv = torch.full((heads, 32 * len(groups), kd + vd), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.gemm_tile_paged(pool, groups, len(groups), table, w.to(DEV), kv)
    made = kv.cpu().double()[:, :length - lo]
    want = (rows[lo:, :rank].double() @ w.double().T).view(-1, heads, kd + vd).transpose(0, 1)
    assert float((made - want).abs().max()) < 2 ** -8 * float(want.abs().max())

    cuts = sorted({0, min(n, 37), *range(64, n, 64)} - {n})
    tiles = [(t, b - t, start + t, 1, -lo) for t, b in zip(cuts, cuts[1:] + [n])]
    tiles_t = torch.tensor(tiles, dtype=torch.int32, device=DEV)
    k = torch.cat([made[:, :, :kd].transpose(0, 1),
                   rows[lo:, None, rank:].double().expand(-1, heads, -1)], 2)
    v = made[:, :, kd:].transpose(0, 1)
    scale = 1.5 / (kd + rot) ** 0.5
    s = torch.einsum("ihd,jhd->hij", torch.cat([q, wide[:, :, rank:]], 2).double(), k) * scale
    i, j = torch.arange(start, length)[:, None], torch.arange(lo, length)[None]
    s = s.masked_fill(~((j <= i) & ((i - j < window) if window else torch.ones(1, dtype=torch.bool))), float("-inf"))
    for with_sink, with_gate in ((False, False), (True, True)):
        a = torch.softmax(torch.cat([s, sink.double()[:, None, None].expand(heads, n, 1)], 2), 2)[:, :, :-1] if with_sink else torch.softmax(s, 2)
        ref = torch.einsum("hij,jhd->ihd", a, v)
        if with_gate:
            ref = ref * gate.double().view(n, heads, vd)
        out = torch.full((n, heads, vd), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.latent_heads(q.to(DEV), wide.to(DEV)[:, :, rank:], kv, pool, out, tiles_t, len(tiles), table, scale, window,
                         sink.to(DEV) if with_sink else None, gate.to(DEV) if with_gate else None)
        assert float((out.cpu().double() - ref).abs().max()) < 2 ** -8 * float(ref.abs().max())


@pytest.mark.gpu
def test_refusals():
    from pyre_amd.hip import ops
    from pyre_amd.hip.lib import KernelError

    z = lambda *s, dt=torch.bfloat16: torch.zeros(s, dtype=dt, device=DEV)  # noqa: E731
    table, tiles = z(1, 4, dt=torch.int32), z(1, 5, dt=torch.int32)
    with pytest.raises(KernelError):  # head sizes without a form
        ops.latent_heads(z(2, 1, 64), z(2, 1, 64), z(1, 32, 192), z(4, 1, 16, 128), z(2, 1, 128), tiles, 1, table, 1.0)
    with pytest.raises(KernelError):  # k that is no multiple of 64
        ops.gemm_tile_paged(z(4, 1, 16, 104), z(1, 3, dt=torch.int32), 1, table, z(64, 96), z(1, 32, 64))
    with pytest.raises(KernelError):  # too few rows for the groups
        ops.gemm_tile_paged(z(4, 1, 16, 128), z(2, 3, dt=torch.int32), 2, table, z(64, 64), z(1, 32, 64))


@pytest.fixture
def runs(monkeypatch):
    """What the engine's layers launch: (kernel, tiles) of every call over made keys and values and over the rows."""
    from pyre_amd.hip import ops

    seen = []
    for name, at in (("latent_heads", 6), ("latent_attn_tile", 4)):
        def counted(*args, name=name, at=at, real=getattr(ops, name)):
            seen.append((name, args[at]))
            return real(*args)

        monkeypatch.setattr(ops, name, counted)
    return seen


def both_ways(tmp_path, steps_of):
    import plain_rukosun as P
    import rukosun_models as M
    from test_rukosun_gpu import TOL, engine_of, write_model
    from helpers import first_bad, random_ids, replay

    raw = M.model(61, 64, [M.layer(M.mixer(2, 128, 64, 128, 256, 0.1, window=90, q_rank=24), 40),
                           M.layer(M.mixer(3, 128, 64, 128, 192, 0.1))], streams=2, places=600)
    _, cfg, w = write_model(tmp_path, raw, 5)
    reqs = {r: random_ids(61, n, seed=n) for r, n in (("a", 230), ("b", 67), ("c", 33))}
    want = {r: P.forward(w, cfg, ids).float() for r, ids in reqs.items()}
    eng = engine_of(tmp_path, "bfloat16")
    for steps in steps_of(reqs):
        bad, worst = first_bad(replay(eng, steps), want, TOL["bfloat16"])
        assert bad is None, bad


@pytest.mark.gpu
def test_both_ways_in_an_engine(tmp_path, runs):
    """Layers whose sizes the kernels take, whole prompts, portions (short ones behind many keys run over the rows themselves), single
    tokens and a mixture of all in a step, against the plain implementation."""
    from test_rukosun_gpu import in_portions, one_by_one, whole

    def steps_of(reqs):
        a, b, c = (reqs[r] for r in "abc")
        mixture = [([("a", a[:150], [0, 149]), ("b", b[:66], [65])], []),
                   ([("b", b[66:], [0]), ("a", a[150:155], [0, 4]), ("c", c, list(range(33)))], ["b", "c"]),
                   ([("a", a[155:], list(range(75)))], ["a"])]
        for steps, launched in ((whole(reqs), {"latent_heads"}), (in_portions(reqs, [100, 3, 70]), {"latent_heads", "latent_attn_tile"}),
                                (one_by_one({"b": b}, 4), {"latent_heads"}), (mixture, {"latent_heads", "latent_attn_tile"})):
            runs.clear()
            yield steps
            assert {name for name, tiles in runs if tiles} == launched

    both_ways(tmp_path, steps_of)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,tiles", [(256, [6, 1, 4, 3]), (128, [3, 2, 1])])
def test_keys_that_are_made_in_rounds(tmp_path, runs, monkeypatch, rows, tiles):
    """A step of three prompts whose keys and values do not fit together (two rounds in each of the two layers), or for the longest
    not even alone (which then runs over the rows; one round and two): each round's groups and tiles, in the scratch of the one before."""
    monkeypatch.setattr(L, "MADE_BYTES", rows * 3 * 512)

    def steps_of(reqs):
        yield [([(r, ids, list(range(len(ids)))) for r, ids in reqs.items()], list(reqs))]
        assert [t for name, t in runs if name == "latent_heads"] == tiles
        assert [t for name, t in runs if name == "latent_attn_tile"] == ([] if len(tiles) == 4 else [8, 8])

    both_ways(tmp_path, steps_of)


@pytest.mark.gpu
def test_a_cache_beyond_the_products_reach_is_read_row_by_row(tmp_path, runs, monkeypatch):
    from test_rukosun_gpu import whole

    monkeypatch.setattr(L, "PRODUCT_ELEMENTS", 0)
    both_ways(tmp_path, lambda reqs: [whole(reqs)])
    assert {name for name, _ in runs} == {"latent_attn_tile"}
