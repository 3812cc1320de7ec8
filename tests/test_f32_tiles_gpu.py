"""The 32-bit path's products of more than 32 rows in tiles and its prompts' attention with pieces of 16 bytes: at the edges
of their tiles, slots and pages."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


@pytest.mark.parametrize("n,k,ks", [(48, 16, 1), (130, 1520, 2), (200, 80, 1), (1536, 1104, 3), (4608, 48, 1)])
def test_products_at_every_row_count_have_the_bits_of_one_row(n, k, ks):
    """Parts of k that end with half a slot among them (1520 / 2 = 760 -> 768 + 752; 1104 / 3 = 368)."""
    from pyre_amd.hip import ops

    m = 600
    a, w = rnd(m, k, seed=1), rnd(n, k, seed=2)
    one = torch.empty(ks, 16, n, device=DEV)
    want = torch.empty(ks, m, n, device=DEV)
    for r in range(0, m, 16):                                  # the kernel that streams the weights
        rows = min(16, m - r)
        part = one[:, :rows].contiguous() if rows < 16 else one
        ops.gemm_f32(a[r:r + rows], w, None, part if ks > 1 else part[0], rows, ks)
        want[:, r:r + rows] = part
    exact = a.double() @ w.double().T
    # k additions of products of values around one, each rounded to 2^-24 of a sum that grows as the root of k
    assert float((want.double().sum(0) - exact).abs().max()) <= 8 * 2.0 ** -24 * k ** 0.5 * float(exact.std()) * 4
    for rows in (17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 129, 200, 400, 600):
        out = torch.full((ks, rows, n), float("nan"), device=DEV)
        ops.gemm_f32(a[:rows], w, None, out if ks > 1 else out[0], rows, ks)
        assert torch.equal(out, want[:, :rows]), rows


@pytest.mark.parametrize("hd,page,window", [(128, 16, 0), (128, 32, 40), (64, 8, 0), (36, 4, 50), (96, 12, 33), (256, 16, 0), (20, 16, 7),
                                            (30, 16, 0), (64, 6, 0)])
def test_attention_of_prompts(hd, page, window):
    """Against float64; what lies behind a step's last key in its page is not a number."""
    from pyre_amd.hip import ops

    nq, nkv, T = 6, 2, 77
    pages = -(-T // page) + 2
    k, v = rnd(T, nkv, hd, seed=1), rnd(T, nkv, hd, seed=2)
    q = rnd(T, nq, hd, seed=3)
    kc = torch.full((pages, nkv, page, hd), float("nan"), device=DEV)
    vc = torch.full((pages, nkv, hd, page), float("nan"), device=DEV)
    order = torch.randperm(pages, generator=torch.Generator().manual_seed(4)).tolist()
    for t in range(T):
        kc[order[t // page], :, t % page] = k[t]
        vc[order[t // page], :, :, t % page] = v[t]
    table = torch.tensor([order], dtype=torch.int32, device=DEV)
    first = 5                                                  # the step brings tokens 5 .. 76
    n = T - first
    pos = torch.arange(first, T, dtype=torch.int32, device=DEV)
    seq = torch.zeros(n, dtype=torch.int32, device=DEV)
    tiles = torch.tensor([[t, min(32, n - t)] for t in range(0, n, 32)], dtype=torch.int32, device=DEV)
    out = torch.full((n, nq, hd), float("nan"), device=DEV)
    ops.attn_prefill_f32(q[first:].contiguous(), out, kc, vc, tiles, len(tiles), pos, seq, table, nq, nkv, hd, page, hd ** -0.5, window)
    i, j = torch.arange(first, T, device=DEV)[:, None], torch.arange(T, device=DEV)[None]
    hidden = (j > i) | ((i - j >= window) if window else torch.zeros_like(j > i))
    for h in range(nq):
        s = (q[first:, h].double() @ k[:, h // 3].double().T * hd ** -0.5).masked_fill(hidden, float("-inf"))
        want = torch.softmax(s, 1) @ v[:, h // 3].double()
        assert float((out[:, h].double() - want).abs().max()) <= 2e-5


@pytest.mark.parametrize("first,n", [(0, 1), (0, 15), (0, 16), (0, 17), (31, 1), (96, 33), (127, 2), (128, 16), (120, 49), (300, 31)])
@pytest.mark.parametrize("nq,nkv,hd,page,window", [(5, 1, 128, 16, 0), (6, 2, 128, 16, 40), (3, 3, 160, 8, 0), (4, 2, 256, 16, 70),
                                                   (3, 1, 30, 16, 40)])
def test_prompts_at_the_edges_of_tokens_and_rounds(first, n, nq, nkv, hd, page, window):
    """Blocks of sixteen tokens and rounds of two or four chunks of keys, one head and two to a block; pages that lie wholly
    behind the window are gone from the table, and what they held is not a number."""
    from pyre_amd.hip import ops

    T = first + n
    pages = -(-T // page)
    k, v, q = rnd(T, nkv, hd, seed=1), rnd(T, nkv, hd, seed=2), rnd(n, nq, hd, seed=3)
    kc = torch.full((pages, nkv, page, hd), float("nan"), device=DEV)
    vc = torch.full((pages, nkv, hd, page), float("nan"), device=DEV)
    for t in range(T):
        kc[t // page, :, t % page] = k[t]
        vc[t // page, :, :, t % page] = v[t]
    table = torch.arange(pages, dtype=torch.int32, device=DEV)[None].clone()
    out_of_sight = (max(0, first - window + 1) // 32 * 32) // page if window else 0
    table[0, :out_of_sight] = -1
    kc[:out_of_sight], vc[:out_of_sight] = float("nan"), float("nan")
    pos, seq = torch.arange(first, T, dtype=torch.int32, device=DEV), torch.zeros(n, dtype=torch.int32, device=DEV)
    tiles = torch.tensor([[t, min(32, n - t)] for t in range(0, n, 32)], dtype=torch.int32, device=DEV)
    out = torch.full((n, nq, hd), float("nan"), device=DEV)
    ops.attn_prefill_f32(q, out, kc, vc, tiles, len(tiles), pos, seq, table, nq, nkv, hd, page, hd ** -0.5, window)
    i, j = torch.arange(first, T, device=DEV)[:, None], torch.arange(T, device=DEV)[None]
    hidden = (j > i) | ((i - j >= window) if window else torch.zeros_like(j > i))
    for h in range(nq):
        s = (q[:, h].double() @ k[:, h * nkv // nq].double().T * hd ** -0.5).masked_fill(hidden, float("-inf"))
        want = torch.softmax(s, 1) @ v[:, h * nkv // nq].double()
        assert float((out[:, h].double() - want).abs().max()) <= 2e-5


@pytest.mark.parametrize("hd,page", [(64, 16), (128, 8), (36, 4), (30, 16), (64, 6)])
def test_keys_without_a_page_are_not_seen(hd, page):
    """An entry of -1 in the block table, and a table that ends before the step's keys do: in both forms, as in the kernels of
    the other attentions."""
    from pyre_amd.hip import ops

    nq, nkv, T = 4, 2, 70
    pages = -(-T // page)
    k, v, q = rnd(T, nkv, hd, seed=1), rnd(T, nkv, hd, seed=2), rnd(T, nq, hd, seed=3)
    kc, vc = torch.zeros(pages, nkv, page, hd, device=DEV), torch.zeros(pages, nkv, hd, page, device=DEV)
    for t in range(T):
        kc[t // page, :, t % page] = k[t]
        vc[t // page, :, :, t % page] = v[t]
    pos, seq = torch.arange(T, dtype=torch.int32, device=DEV), torch.zeros(T, dtype=torch.int32, device=DEV)
    tiles = torch.tensor([[t, min(32, T - t)] for t in range(0, T, 32)], dtype=torch.int32, device=DEV)
    i, j = torch.arange(T, device=DEV)[:, None], torch.arange(T, device=DEV)[None]
    for gone, width in ((2, pages), (pages - 1, pages), (None, pages - 1)):
        table = torch.arange(width, dtype=torch.int32, device=DEV)[None].clone()
        if gone is not None:
            table[0, gone] = -1
        lost = (j // page == gone) if gone is not None else (j // page >= width)
        out = torch.full((T, nq, hd), float("nan"), device=DEV)
        ops.attn_prefill_f32(q, out, kc, vc, tiles, len(tiles), pos, seq, table.contiguous(), nq, nkv, hd, page, hd ** -0.5, 0)
        for h in range(nq):
            s = (q[:, h].double() @ k[:, h // 2].double().T * hd ** -0.5).masked_fill((j > i) | lost, float("-inf"))
            want = torch.softmax(s, 1) @ v[:, h // 2].double()
            assert float((out[:, h].double() - want).abs().max()) <= 2e-5, (gone, width)


@pytest.mark.parametrize("n,k,ks", [(130, 1520, 2), (1536, 1104, 3), (200, 8960, 16), (48, 80, 3), (300, 640, 40)])
def test_parts_added_where_they_are_made(n, k, ks):
    """The same bits as the parts added up in their order (parts that end with half a slot, a last part shorter than the
    others)."""
    from pyre_amd.hip import ops

    for m in (17, 40, 65, 100, 200, 520):
        a, w = rnd(m, k, seed=m), rnd(n, k, seed=n)
        parts = torch.empty(ks, m, n, device=DEV)
        ops.gemm_f32(a, w, None, parts, m, ks)
        want = parts[0].clone()
        for p in parts[1:]:
            want += p
        out = torch.full((m, n), float("nan"), device=DEV)
        ops.gemm_f32_whole(a, w, out, m, ks)
        assert torch.equal(out, want), m


@pytest.mark.parametrize("n,k,ks,off", [(48, 20, 1, 0), (130, 1524, 2, 0), (200, 8, 1, 0), (130, 1529, 2, 1), (77, 23, 1, 3), (70, 9, 1, 1),
                                        (1536, 1110, 3, 2), (200, 1104, 3, 1), (130, 272, 1, 0), (65, 9, 1, 0), (33, 15, 1, 1),
                                        (4608, 60, 1, 1), (9000, 45, 1, 0)])
def test_k_that_ends_within_a_step_and_rows_that_start_anywhere(n, k, ks, off):
    """The bits of the same product with zeros behind k, up to whole steps, and with rows on 16 bytes. What lies behind the rows and
    before them is not a number."""
    from pyre_amd.hip import ops

    m, whole = 600, -(-k // 16) * 16
    assert ops.f32_part(k, ks) == ops.f32_part(whole, ks)
    a, w = rnd(m, k, seed=1), rnd(n, k, seed=2)

    def laid(x, step):
        rows = torch.full((x.shape[0], off + k + step), float("nan"), device=DEV)
        rows[:, off:off + k] = x
        return rows[:, off:off + k]

    pad = torch.nn.functional.pad
    for rows in (1, 31, 32, 33, 64, 65, 129, 400, 600):
        want, out = torch.empty(ks, rows, n, device=DEV), torch.full((ks, rows, n), float("nan"), device=DEV)
        ops.gemm_f32(pad(a[:rows], (0, whole - k)), pad(w, (0, whole - k)), None, want if ks > 1 else want[0], rows, ks)
        ops.gemm_f32(laid(a[:rows], 0), laid(w, 3 if off else 0), None, out if ks > 1 else out[0], rows, ks)
        assert torch.equal(out, want), rows


@pytest.mark.parametrize("nq,nkv,hd,page,window", [(12, 2, 128, 16, 0), (7, 1, 64, 16, 40), (5, 5, 32, 8, 0), (6, 2, 96, 16, 70), (9, 3, 250, 16, 0),
                                                   (4, 2, 192, 12, 33), (3, 1, 128, 3, 0), (8, 1, 256, 16, 0)])
def test_prompts_of_many_tiles_have_the_bits_of_one_alone(nq, nkv, hd, page, window):
    """Tiles that fill the chip run in blocks of whole tiles whose waves have two parts of the keys each, few tiles in blocks of
    sixteen tokens and a wave for every part: first and last chunks of every part, halves of tiles that are not there."""
    from pyre_amd.hip import ops

    cases = [(0, 1), (0, 17), (0, 32), (31, 2), (32, 16), (33, 31), (64, 5), (95, 33), (127, 20), (128, 1), (129, 48), (250, 40)]
    repeat = 90
    pages = -(-290 // page)
    kc, vc = rnd(len(cases) * pages, nkv, page, hd, seed=1), rnd(len(cases) * pages, nkv, hd, page, seed=2)
    table = torch.randperm(len(cases) * pages, generator=torch.Generator().manual_seed(3)).view(len(cases), pages).int().to(DEV)

    def run(which):
        pos, seq, tiles, n = [], [], [], 0
        for r in which:
            first, count = cases[r]
            tiles += [(n + t, min(32, count - t)) for t in range(0, count, 32)]
            pos += range(first, first + count)
            seq += [r] * count
            n += count
        i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
        q = torch.cat([rnd(cases[r][1], nq, hd, seed=10 + r) for r in which])
        out = torch.full((n, nq, hd), float("nan"), device=DEV)
        ops.attn_prefill_f32(q, out, kc, vc, i32(tiles), len(tiles), i32(pos), i32(seq), table, nq, nkv, hd, page, hd ** -0.5, window)
        return out

    alone = torch.cat([run([r]) for r in range(len(cases))])
    assert not bool(alone.isnan().any())
    assert torch.equal(run(list(range(len(cases))) * repeat), alone.repeat(repeat, 1, 1))
