"""The product of many rows in tiles (`gemm_tile.hip`) against the product of the same 16-bit values in float64: at the edges
of its tiles, with every number of parts of k, with rows apart from each other, and in an engine's step against the library's
products."""

from __future__ import annotations

import functools
import math
import random

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def rnd(*shape, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).to(DEV)


#: float32 sums of k products of values around one: a rounding of 2^-24 of the running sum for every addition, the sums
#: growing as the root of k, k roundings at random: 2^-24 sqrt(k) of the result's size; eight times that for the largest
def bound(k: int) -> float:
    return 8.0 * 2.0 ** -24 * k ** 0.5


@pytest.mark.parametrize("n,k", [(16, 64), (144, 128), (272, 448), (1536, 192), (2064, 1536)])
@pytest.mark.parametrize("m", [1, 65, 128, 129, 255, 257, 600])
def test_sums(m, n, k):
    from pyre_amd.hip import ops

    assert ops.gemm_tile_supports(m, n, k, k, k)
    x, w = rnd(m, k, seed=m), rnd(n, k, seed=n)
    want = x.double() @ w.double().T
    for parts in sorted({1, ops.gemm_tile_parts(m, n, k), *([2, 6] if k == 1536 else [])}):
        out = torch.full((parts, m, n), float("nan"), device=DEV)
        ops.gemm_tile_bf16(x, w, out, m, parts)
        assert float((out.double().sum(0) - want).abs().max()) <= bound(k) * float(want.std()) * 4, parts


@pytest.mark.parametrize("m,n,k,rows", [(3000, 3584, 1536, 256), (2048, 5552, 512, 256), (500, 2064, 1024, 128), (260, 4608, 640, 128),
                                        (70, 4624, 1024, 64)])
def test_larger_sums(m, n, k, rows):
    """Sizes of about one round, and a row more than whole tiles."""
    from pyre_amd.hip import ops

    for mm in (m, m // rows * rows + 1):
        x, w = rnd(mm, k + 24, seed=1)[:, 8:k + 8], rnd(n, k + 8, seed=2)[:, :k]   # rows 48 and 16 bytes apart
        parts = ops.gemm_tile_parts(mm, n, k)
        out = torch.full((parts, mm, n), float("nan"), device=DEV)
        ops.gemm_tile_bf16(x, w, out, mm, parts)
        want = x.double() @ w.double().T
        assert float((out.double().sum(0) - want).abs().max()) <= bound(k) * float(want.std()) * 4


#: the forms of the kernel: rows of x and of w of a tile, and the stages of 64 k that its ring holds
SUMS = {(256, 256): 2, (256, 192): 2, (128, 192): 3, (128, 128): 4, (64, 128): 5}
UNITS = {(256, 256): 2, (192, 256): 2, (192, 192): 2, (128, 256): 2, (96, 256): 2, (96, 192): 3}
CASES = ("whole tiles", "a row more", "columns past the end", "fewer stages than slots", "an edge before a whole tile")


def walks_from_an_edge(m, n, parts, bm, bn, units):
    """Whether some block takes a whole tile after one that ends past the matrix (the kernel's order of tiles)."""
    mt, nt = -(-m // bm), -(-n // bn)
    tiles, blocks = mt * nt * parts, min(units, mt * nt * parts)

    def whole(t):
        t %= mt * nt
        first = t // (8 * nt) * 8
        t, gm = t - first * nt, min(8, mt - first)
        return (first + t % gm + 1) * bm <= m and (t // gm + 1) * bn <= n

    for die in range(min(8, blocks)):
        begin = die * (tiles // 8) + min(die, tiles % 8)
        end, step = begin + tiles // 8 + (die < tiles % 8), (blocks - die + 7) // 8
        if any(not whole(t) and whole(t + step) for t in range(begin, end - step)):
            return True
    return False


@functools.lru_cache(maxsize=None)
def sizes_of_every_form(gated: bool):
    """For every form and case the smallest size of many that the planner gives to it: {(tile, case): (m, n, k)}, in one launch;
    {("first" or "rest", tile): (m, n, k)} of those that it cuts."""
    from pyre_amd.hip import ops

    forms, units = UNITS if gated else SUMS, ops.compute_units()
    rng, found = random.Random(5), {}

    def note(key, size):
        if key not in found or math.prod(size) < math.prod(found[key]):
            found[key] = size

    for i in range(40000):
        bm, bn = list(forms)[i % len(forms)]
        m, n, k = rng.randint(1, 3000), 16 * rng.randint(1, 1600), 64 * rng.choice([1, 2, 3, 4, 5, 7, 16, 24, 40])
        if i % 3 == 1:
            m, n = -(-m // bm) * bm, -(-n // bn) * bn
        elif i % 3 == 2:
            m = m // bm * bm + 1
        if m * n > 4e7:
            continue
        tile, cut, _, rest = ops.gemm_tile_choice(m, n, k, gated)
        if cut:
            note(("first", tile), (m, n, k))
            note(("rest", rest), (m, n, k))
            continue
        parts = 1 if gated else ops.gemm_tile_parts(m, n, k)
        per = -(-(-(-k // parts)) // 64)
        is_so = (m % tile[0] == 0 and n % tile[1] == 0, m % tile[0] == 1, n % tile[1] != 0, per < forms[tile],
                 m % tile[0] and n % tile[1] and walks_from_an_edge(m, n, parts, *tile, units))
        for case, so in zip(CASES, is_so):
            if so:
                note((tile, case), (m, n, k))
    return found


def check_product(m, n, k, gated, tile, rest=None):
    """A product whose rows lie 16 and 48 bytes further apart than they are long, made by the tiles that are named."""
    from pyre_amd.hip import ops

    says, cut, _, then = ops.gemm_tile_choice(m, n, k, gated)
    assert (says == tile or tile is None) and (bool(cut), then) == ((False, (0, 0)) if rest is None else (True, rest))
    x, w = rnd(m, k + 24, seed=1)[:, 8:k + 8], rnd(n, k + 8, seed=2, scale=0.2 if gated else 1.0)[:, :k]
    want = x.double() @ w.double().T
    if gated:
        out = torch.full((m, n // 2), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops.gemm_tile_glu_bf16(x, w, out, m)
        want = torch.nn.functional.silu(want[:, :n // 2]) * want[:, n // 2:]
        # half a unit of the 8 bits that bfloat16 keeps, and the sums' rounding through factors that grow with the sums
        assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + 64 * bound(k)).all())
    else:
        parts = ops.gemm_tile_parts(m, n, k)
        out = torch.full((parts, m, n), float("nan"), device=DEV)
        ops.gemm_tile_bf16(x, w, out, m, parts)
        assert float((out.double().sum(0) - want).abs().max()) <= bound(k) * max(1.0, k ** 0.5) * 4


#: what the planner gives to no form: its smallest tiles of gated units are for products of one round
NEVER = {(True, (96, 192), CASES[4])}


@pytest.mark.parametrize("gated,tile,case", sorted(NEVER))
def test_what_no_form_is_given(gated, tile, case):
    """What the next test leaves out is not there to be taken: with other costs of the tiles it has to be looked at again."""
    assert (tile, case) not in sizes_of_every_form(gated)


@pytest.mark.parametrize("gated,tile,case", [(g, t, c) for g, forms in ((False, SUMS), (True, UNITS)) for t in forms for c in CASES
                                             if (g, t, c) not in NEVER])
def test_every_form(gated, tile, case):
    """Every form of the kernel at the edges of its tiles, rounds and ring, at sizes that the planner gives to it."""
    check_product(*sizes_of_every_form(gated)[tile, case], gated, tile)


@pytest.mark.parametrize("gated,tile", [(False, (256, 192)), (False, (128, 192)), (False, (128, 128)), (False, (64, 128)),
                                        (True, (256, 256)), (True, (192, 256)), (True, (192, 192)),
                                        (True, (128, 256)), (True, (96, 256)), (True, (96, 192))])
def test_every_form_behind_a_cut(gated, tile):
    size = sizes_of_every_form(gated)["rest", tile]
    check_product(*size, gated, None, tile)


@pytest.mark.parametrize("m,n,k", [(2100, 25616, 64), (2300, 24576, 128), (1800, 25600, 192), (3000, 16400, 320)])
@pytest.mark.parametrize("gated", [False, True])
def test_blocks_that_walk_short_tiles(m, n, k, gated):
    """Several tiles of one to five stages a block, in rings of two slots (k = 64 and 128: no more stages than those): what is asked for
    ahead is the next tiles'."""
    from pyre_amd.hip import ops

    (rows, cols), _, _, _ = ops.gemm_tile_choice(m, n, k, gated, 1)
    assert (UNITS if gated else SUMS)[rows, cols] == 2 and m // rows * (n // cols) > ops.compute_units()

    x, w = rnd(m, k, seed=8), rnd(n, k, seed=9, scale=0.2)
    want = x.double() @ w.double().T
    if gated:
        out = torch.full((m, n // 2), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops.gemm_tile_glu_bf16(x, w, out, m)
        want = torch.nn.functional.silu(want[:, :n // 2]) * want[:, n // 2:]
        # half a unit of the 8 bits that bfloat16 keeps, and the sums' rounding through factors that grow with the sums
        assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + 64 * bound(k)).all())
    else:
        out = torch.full((1, m, n), float("nan"), device=DEV)
        ops.gemm_tile_bf16(x, w, out, m, 1)
        assert float((out[0].double() - want).abs().max()) <= bound(k) * float(want.std()) * 4


@pytest.mark.parametrize("tile,m,n,k", [((128, 192), 641, 21808, 64), ((128, 192), 769, 18704, 128), ((128, 192), 769, 19088, 192),
                                        ((128, 128), 129, 24912, 64), ((128, 128), 257, 16848, 128), ((128, 128), 257, 16592, 192),
                                        ((128, 128), 257, 16496, 256), ((64, 128), 267, 11392, 64), ((64, 128), 170, 18608, 128),
                                        ((64, 128), 190, 17808, 192), ((64, 128), 192, 18560, 256), ((64, 128), 192, 20720, 320)])
def test_blocks_that_walk_short_tiles_in_longer_rings(tile, m, n, k):
    """Several tiles a block, of no more stages than its ring of three to five slots has: the tiles behind the next one are asked for already, and
    stores of several tiles stand among the loads that are counted, or (at an edge) do not."""
    from pyre_amd.hip import ops

    says, cut, _, _ = ops.gemm_tile_choice(m, n, k, False, 1)
    assert says == tile and not cut and k // 64 <= SUMS[tile] and -(-m // tile[0]) * -(-n // tile[1]) > ops.compute_units()
    x, w = rnd(m, k + 24, seed=1)[:, 8:k + 8], rnd(n, k + 8, seed=2)[:, :k]
    want = x.double() @ w.double().T
    for _ in range(3):
        out = torch.full((1, m, n), float("nan"), device=DEV)
        ops.gemm_tile_bf16(x, w, out, m, 1)
        assert float((out[0].double() - want).abs().max()) <= bound(k) * max(1.0, k ** 0.5) * 4


@pytest.mark.parametrize("unit", [None, (7.0, 1.702, 1.0), (0.0, float("inf"), 0.0, 0.0)])
@pytest.mark.parametrize("m,inter,k", [(1, 8, 64), (70, 8960, 128), (130, 18944, 64), (200, 18936, 64), (257, 136, 256), (300, 8960, 64),
                                       (520, 18944, 64), (1100, 1000, 128), (2049, 8968, 64)])
def test_gated_units(m, inter, k, unit):
    from pyre_amd.hip import ops

    x, w = rnd(m, k, seed=3), rnd(2 * inter, k, seed=4, scale=0.2)
    out = torch.full((m, inter), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.gemm_tile_glu_bf16(x, w, out, m, unit)
    gate, up = (x.double() @ w.double().T).split(inter, 1)
    if unit is None:
        want = torch.nn.functional.silu(gate) * up
    elif unit[1] == float("inf"):
        want = gate.clamp(min=0) * up
    else:
        gate, up = gate.clamp(max=unit[0]), up.clamp(-unit[0], unit[0])
        want = gate * torch.sigmoid(unit[1] * gate) * (up + unit[2])
    # half a unit of the 8 bits that bfloat16 keeps, and the sums' rounding through factors of up to 16
    assert bool(((out.double() - want).abs() <= want.abs() * 2.0 ** -8 + 64 * bound(k)).all())


def test_not_numbers_and_infinities_stay_in_their_rows():
    from pyre_amd.hip import ops

    x, w = rnd(300, 128, seed=5), rnd(512, 128, seed=6)
    x[7, 3], x[299, 127] = float("nan"), float("inf")
    out = torch.zeros(1, 300, 512, device=DEV)
    ops.gemm_tile_bf16(x, w, out, 300, 1)
    clean = torch.ones(300, dtype=torch.bool, device=DEV)
    clean[7] = clean[299] = False
    assert bool(torch.isnan(out[0, 7]).all()) and not bool(torch.isfinite(out[0, 299]).any())
    assert bool(torch.isfinite(out[0, clean]).all())


def test_what_it_refuses():
    from pyre_amd.hip import ops
    from pyre_amd.hip.lib import KernelError

    assert not ops.gemm_tile_supports(100, 24, 64, 64, 64) and not ops.gemm_tile_supports(100, 32, 96, 96, 96)
    assert not ops.gemm_tile_supports(100, 32, 64, 60, 64) and not ops.gemm_tile_supports(1 << 20, 32, 4096, 4096, 4096)
    x, w = rnd(100, 96), rnd(32, 96)
    with pytest.raises(KernelError):
        ops.gemm_tile_bf16(x, w, torch.empty(1, 100, 32, device=DEV), 100, 1)
    x, w = rnd(100, 128), rnd(32, 128)
    with pytest.raises(KernelError):
        ops.gemm_tile_bf16(x, w, torch.empty(3, 100, 32, device=DEV), 100, 3)     # parts of less than 256 k
    with pytest.raises(KernelError):
        ops.gemm_tile_bf16(x[:, 1:65], w[:, :64], torch.empty(1, 100, 32, device=DEV), 100, 1)


@pytest.mark.parametrize("n", [65, 300])
def test_a_step_against_the_librarys_products(n):
    """The whole prompt of a small model through both: 16-bit activations, three layers."""
    from pyre_amd.config import EngineConfig, preset
    from pyre_amd.engine.batch import Entry
    from pyre_amd.engine.engine import Engine
    from pyre_amd.weights import model_tensor_specs, random_state

    cfg = preset("tiny-a", hidden_size=128, head_dim=32, intermediate_size=320, num_hidden_layers=3)
    state = random_state(model_tensor_specs(cfg), 3, 0.08, 0.1, torch.bfloat16, device=DEV)
    eng = Engine.from_state(cfg, state, EngineConfig(max_cached_tokens=1024, max_num_batched_tokens=512, max_model_len=512))
    ids = [(7 * i + 3) % 512 for i in range(n)]
    rows = []
    for tile in (True, False):
        eng.runtime.options["tile_gemm"] = tile
        eng.runtime.options["mid_gemm"] = False
        rows.append(eng.step([Entry("a", ids, list(range(n)))]).clone())
        eng.finish("a")
    scale = rows[1].abs().amax(1)
    assert float(((rows[0] - rows[1]).abs().amax(1) / scale).max()) <= 2e-2


@pytest.mark.parametrize("m,n,k,gated,by_rows", [(1777, 37904, 1024, True, False), (2101, 17936, 1536, True, False),
                                                 (5501, 3600, 2048, True, True), (2101, 9040, 2048, False, False),
                                                 (4501, 3600, 2048, False, False), (7501, 2064, 2048, False, True)])
def test_a_last_round_in_smaller_tiles(m, n, k, gated, by_rows):
    """Products cut in two launches, along the rows of either operand: every element is the product of its own rows."""
    from pyre_amd.hip import ops

    _, cut, rows, rest = ops.gemm_tile_choice(m, n, k, gated)
    assert cut and rows == by_rows
    check_product(m, n, k, gated, None, rest)


def test_a_step_with_weights_that_are_views():
    """Weights that do not lie on 16 bytes: the step's products go to the library and give what they give there."""
    from pyre_amd.config import EngineConfig, preset
    from pyre_amd.engine.batch import Entry
    from pyre_amd.engine.engine import Engine
    from pyre_amd.weights import model_tensor_specs, random_state

    cfg = preset("tiny-a", hidden_size=128, head_dim=32, intermediate_size=320, num_hidden_layers=2)
    ids = [(7 * i + 3) % 512 for i in range(300)]
    rows = []
    for shift in (0, 4):
        state = random_state(model_tensor_specs(cfg), 3, 0.08, 0.1, torch.bfloat16, device=DEV)
        for name, t in state.items():
            if name.endswith(("o_proj.weight", "down_proj.weight")):
                state[name] = torch.cat([t.new_zeros(shift), t.flatten()])[shift:].view(t.shape)
                assert state[name].data_ptr() % 16 == 2 * shift
        eng = Engine.from_state(cfg, state, EngineConfig(max_cached_tokens=1024, max_num_batched_tokens=512, max_model_len=512))
        rows.append(eng.step([Entry("a", ids, list(range(300)))]).clone())
    assert float(((rows[0] - rows[1]).abs().amax(1) / rows[1].abs().amax(1)).max()) <= 2e-2


@pytest.mark.parametrize("m,view", [(64, False), (65, False), (190, False), (257, False), (190, True)])
def test_logits_of_many_rows_without_the_library(m, view, monkeypatch):
    """The head's float32 results in place, on both sides of the rows that the weight-streaming kernel takes; weights that do
    not lie on 16 bytes are the library's."""
    from types import SimpleNamespace

    from pyre_amd.hip import ops
    from pyre_amd.parts import fast

    n, k = 20016, 192
    x, w = rnd(m + 3, k, seed=1), rnd(n * k + 8, seed=2)
    weight = w[4:n * k + 4].view(n, k) if view else w[:n * k].view(n, k)
    lin = SimpleNamespace(in_features=k, out_features=n, weight=weight, bias=None, role="head")
    rt = SimpleNamespace(dtype=torch.bfloat16, options={}, compute_units=ops.compute_units())
    called, mm = [], torch.mm
    monkeypatch.setattr(torch, "mm", lambda *a, **b: (called.append(1), mm(*a, **b))[1])
    out = torch.full((m, n), float("nan"), device=DEV)
    p = fast.linear(lin, SimpleNamespace(runtime=rt), x, m, out)
    assert bool(called) == view
    want = x[:m].double() @ weight.double().T
    assert float((p.data[0].double() - want).abs().max()) <= bound(k) * float(want.std()) * 4


@pytest.mark.parametrize("n,k", [(1536, 1536), (2048, 1536), (4608, 3584), (3072, 4608), (1024, 1024), (48, 768)])
def test_few_rows_in_tiles_agree_with_their_captured_size(n, k):
    """From 129 rows on: a row of an eager step has the bits that it has in the padded one, and the sums are right."""
    from types import SimpleNamespace

    from pyre_amd.hip import ops
    from pyre_amd.parts import fast

    weight, x = rnd(n, k, seed=2), rnd(256, k, seed=1)
    want = x.double() @ weight.double().T
    buffers = {}
    workspace = SimpleNamespace(get=lambda name, shape, dtype: buffers.setdefault((name, shape), torch.full(shape, float("nan"), dtype=dtype, device=DEV)))
    rt = SimpleNamespace(dtype=torch.bfloat16, options={}, compute_units=ops.compute_units(), workspace=workspace)
    lin = SimpleNamespace(in_features=k, out_features=n, weight=weight, bias=None, role="attn.out", whole=False, partials_name="p")
    for captured, eager in ((128, 100), (192, 129), (192, 150), (256, 193), (256, 255)):
        got = [fast.linear(lin, SimpleNamespace(runtime=rt), x[:m], m, None).data.clone() for m in (captured, eager)]
        assert got[0].shape[0] == got[1].shape[0] and torch.equal(got[0][:, :eager], got[1])
        assert fast.few_tiles(captured, n, k) == (0 if captured == 128 else got[0].shape[0])
        assert float((got[0].double().sum(0) - want[:captured]).abs().max()) <= bound(k) * float(want.std()) * 4


@pytest.mark.parametrize("n,k", [(2048, 4096), (8000, 8192), (16000, 5120), (32000, 2048), (64000, 1024), (100352, 2560)])
def test_the_librarys_logits_in_a_graph(n, k):
    """The heads of fewer features are the library's product, in captured steps (up to 256 rows) too: every replay has the bits of the eager
    product of the rows that are there by then, with eager work on the same memory and synchronizations between the replays."""
    from types import SimpleNamespace

    from pyre_amd.hip import ops
    from pyre_amd.parts import fast

    weight = rnd(n, k, seed=2, scale=0.02)
    lin = SimpleNamespace(in_features=k, out_features=n, weight=weight, bias=None, role="head")
    ctx = SimpleNamespace(runtime=SimpleNamespace(dtype=torch.bfloat16, options={}, compute_units=ops.compute_units()))
    for m in (96, 128, 192, 256):
        assert not fast.head_in_tiles(m, n, k)
        x, out, eager = rnd(m, k, seed=m), torch.empty(m, n, device=DEV), torch.empty(m, n, device=DEV)
        fast.linear(lin, ctx, x, m, out)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            fast.linear(lin, ctx, x, m, out)
        for i in range(5):
            x.copy_(rnd(m, k, seed=1000 + i))
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            fast.linear(lin, ctx, x, m, eager)
            want = x.double() @ weight.double().T if i == 4 else None
            assert torch.equal(out, eager)
        assert float((out.double() - want).abs().max()) <= bound(k) * float(want.std()) * 4
