"""The 32-bit path's products, made of bfloat16 pieces: how far they are from 64 bits, and numbers whose pieces no bfloat16 holds."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
#: few rows, the smallest tiles (the others below); with k in one part and in several, with rows that start on 16 bytes and that do not
FORMS = [(m, n, k, ks, off) for m in (1, 32, 33, 300) for n, k, ks in ((33, 48, 1), (1537, 1040, 1), (200, 1536, 3)) for off in (0, 1)]


def operands(m, n, k, off, scale=1.0):
    g = torch.Generator().manual_seed(m + n + k)
    a = torch.zeros(m, k + 4, device=DEV)
    a[:, off:off + k] = torch.randn(m, k, generator=g).to(DEV) * scale
    return a[:, off:off + k], (torch.randn(n, k, generator=g) * 0.02).to(DEV)


@pytest.mark.parametrize("m,n,k,ks,off", FORMS)
def test_no_further_from_64_bits_than_a_chain_of_fused_multiply_adds(m, n, k, ks, off):
    from pyre_amd.hip import ops

    a, w = operands(m, n, k, off, scale=3.0)
    out, chain = torch.full((ks, m, n), float("nan"), device=DEV), torch.empty(m, n, device=DEV)
    ops.gemm_f32(a, w, None, out if ks > 1 else out[0], m, ks)
    ops.gemm_generic(a, w, None, chain, m)
    want = a.double() @ w.double().T
    err, err_chain = ((x.double() - want).square().mean().sqrt() for x in (out.sum(0), chain))
    # what is left out of a product is at most 2^-24 of it and in root mean square below 2^-26, the chain's own roundings are 2^-25 of
    # the sum each; a few dozen elements (one row) scatter by some ten per cent, and a sum of 48 has few roundings of either kind
    assert float(err) <= 1.1 * float(err_chain) + 2.0 ** -26 * float(want.square().mean().sqrt())


@pytest.mark.parametrize("m,n,k,ks,off", FORMS)
def test_infinities_and_the_largest_numbers(m, n, k, ks, off):
    """As float32 arithmetic has them: a row with an infinity, one with a NaN, one with the largest number (whose upper piece
    would round to infinity) times weights that keep its products finite."""
    from pyre_amd.hip import ops

    a, w = operands(m, n, k, off)
    big = torch.finfo(torch.float32).max
    for value, row in ((float("inf"), 0), (float("nan"), m // 2), (-float("inf"), m - 1), (big, m - 1)):
        b = a.clone() if off == 0 else torch.nn.functional.pad(a, (off, 0))[:, off:]
        b[row, k // 2] = value
        out = torch.full((ks, m, n), float("nan"), device=DEV)
        ops.gemm_f32(b, w, None, out if ks > 1 else out[0], m, ks)
        got, want = out.double().sum(0), b.double() @ w.double().T
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf()), (value, row)
        fine = want.isfinite()
        assert torch.equal(got[~fine & ~want.isnan()], want[~fine & ~want.isnan()])
        # roundings of 2^-24 of the largest partial sum: the row's scale is that of its largest product
        scale = (b.double().abs() @ w.double().abs().T)[fine]
        assert bool(((got - want)[fine].abs() <= 2.0 ** -22 * scale + 1e-30).all()), (value, row)


@pytest.mark.parametrize("m,n,k,ks,off", FORMS)
@pytest.mark.parametrize("low,high", [(-108, 100), (-113, 60), (-118, 100), (-126, 110), (-140, 100), (-70, -70), (45, 50)])
def test_small_and_large_operands(m, n, k, ks, off, low, high):
    """Small activations times large weights and the other way round, subnormal numbers among them; sums that are small themselves;
    sums that leave the range of the scaled pieces (2^80) and not that of a float32."""
    from pyre_amd.hip import ops

    a, w = operands(m, n, k, off)
    w = w * 50.0
    for ea, ew in ((low, high), (high, low)):
        x, y = torch.ldexp(a.double(), torch.tensor(float(ea), device=DEV)).float(), torch.ldexp(w.double(), torch.tensor(float(ew), device=DEV)).float()
        if off:
            x = torch.nn.functional.pad(x, (off, 0))[:, off:]
        out, chain = torch.full((ks, m, n), float("nan"), device=DEV), torch.empty(m, n, device=DEV)
        ops.gemm_f32(x, y, None, out if ks > 1 else out[0], m, ks)
        ops.gemm_generic(x, y, None, chain, m)
        want = x.double() @ y.double().T
        err, err_chain, rms = (float(v.square().mean().sqrt()) for v in (out.double().sum(0) - want, chain.double() - want, want))
        # what is left out of a product is at most 2^-24 of it, what a result below 2^-126 cannot hold at most 2^-149 for each part
        assert err <= 1.1 * err_chain + 2.0 ** -24 * rms + ks * 2.0 ** -149, (ea, ew)


@pytest.mark.parametrize("m,n,k", [(20, 17920, 1536), (300, 4608, 3584)])
def test_a_row_that_is_not_finite_does_not_hold_up_the_others(m, n, k):
    """Its elements are made again on a slower instruction: a few times the step's time (2 to 3 measured), not a hundred times."""
    from pyre_amd.hip import ops

    a, w = operands(m, n, k, 0)
    out = torch.empty(m, n, device=DEV)

    def least_time(x):
        times = []
        for _ in range(6):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            ops.gemm_f32(x, w, None, out, m)
            end.record()
            torch.cuda.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    fine = least_time(a)
    for value in (float("nan"), float("inf"), 3e38):
        b = a.clone()
        b[m // 2, 5] = value
        assert least_time(b) < 12 * fine, value


#: sums of all parts in tiles of each size (rows x columns)
WHOLES = [(100, 1536, 1104, 3, (64, 64)), (300, 6000, 560, 2, (64, 128)), (300, 8960, 560, 2, (128, 128))]


@pytest.mark.parametrize("m,n,k,ks,tile", WHOLES)
def test_numbers_beyond_the_pieces_have_the_bits_of_parts_added_in_order(m, n, k, ks, tile):
    """Numbers from 2^104 on, the largest, infinities and not-a-numbers, in rows of several row tiles and in one part of k or in all:
    whether a block adds the parts up itself or their consumer does."""
    from pyre_amd.hip import ops
    from pyre_amd.hip.lib import lib

    assert lib().pyre_gemm_f32_tile_choice(m, n, k, 1) == 1000 * tile[0] + tile[1]
    a, w = operands(m, n, k, 0)
    w[:, 5] *= 1e-31  # under a number of 1e32 its products are as large as the others', whose parts the element keeps
    for row, value, places in ((0, 3e38, (3,)), (33, 1e32, (5,)), (65, -3e32, (5,)), (m - 1, -3e38, (k - 2,)), (40, float("inf"), (k // 2,)),
                               (70, float("nan"), (1,)), (m - 2, 2e35, range(0, k, 7)), (m // 2, 1e30, (2, k // 2))):
        a[row, list(places)] = value
    w[n - 1, 4], w[n // 2, k - 3] = 1e33, -2e31
    parts, whole = torch.empty(ks, m, n, device=DEV), torch.full((m, n), float("nan"), device=DEV)
    ops.gemm_f32(a, w, None, parts, m, ks)
    ops.gemm_f32_whole(a, w, whole, m, ks)
    want = parts[0].clone()
    for p in parts[1:]:
        want += p
    assert torch.equal(whole.isnan(), want.isnan()) and torch.equal(whole.nan_to_num(), want.nan_to_num())
    exact = a.double() @ w.double().T
    fine, scale = exact.abs() < 1e38, a.double().abs() @ w.double().abs().T
    assert bool(((want.double() - exact)[fine].abs() <= 2.0 ** -21 * scale[fine]).all())
    rows = torch.tensor([0, 33, 40, 65, 70, m // 2, m - 1], device=DEV)  # in a step of few rows
    few = torch.empty(ks, len(rows), n, device=DEV)
    ops.gemm_f32(a[rows].contiguous(), w, None, few, len(rows), ks)
    assert torch.equal(few.nan_to_num(), parts[:, rows].nan_to_num())


@pytest.mark.parametrize("kind", ["random", "positive", "repeated", "one pair"])
@pytest.mark.parametrize("k,ks", [(1, 1), (2, 1), (3, 1), (4, 1), (7, 1), (8, 1), (16, 1), (20, 1), (128, 1), (1536, 1), (8960, 14), (4224, 2), (9216, 2)])
def test_sums_of_any_length_and_of_one_sign(kind, k, ks):
    """From one product to parts of 4,608 (the 32B shape's way down), whose chains are the longest: no further from 64 bits than a chain
    of fused multiply-adds. ``repeated``: an element's products are all the same, so that its roundings all go one way."""
    from pyre_amd.hip import ops

    g = torch.Generator().manual_seed(k)
    for m in (4, 40, 300):
        n = 256
        if kind == "random":
            a, w = torch.randn(m, k, generator=g).to(DEV), torch.randn(n, k, generator=g).to(DEV)
        elif kind == "positive":
            a, w = torch.rand(m, k, generator=g).to(DEV) + 0.01, torch.rand(n, k, generator=g).to(DEV) + 0.01
        elif kind == "repeated":
            a, w = ((1 + torch.rand(x, 1, generator=g)).to(DEV).expand(x, k).contiguous() for x in (m, n))
        else:  # the numbers whose left-out products are largest: 2^-24.0 of each
            a, w = (torch.full((x, k), 1.0038986206054688, device=DEV) for x in (m, n))
        out, chain = torch.empty(ks, m, n, device=DEV), torch.empty(m, n, device=DEV)
        ops.gemm_f32(a, w, None, out if ks > 1 else out[0], m, ks)
        part = ops.f32_part(k, ks)
        for p in range(ks):
            x, y = a[:, p * part:(p + 1) * part].contiguous(), w[:, p * part:(p + 1) * part].contiguous()
            ops.gemm_generic(x, y, None, chain, m)
            want = x.double() @ y.double().T
            err, err_chain, rms = (float(v.square().mean().sqrt()) for v in (out[p].double() - want, chain.double() - want, want))
            # one pair has one error of either kind, its sums' roundings being all alike: those of 16 k are six, each of 2^-24
            bound = 1.1 * err_chain if kind != "one pair" else 2.0 ** -24 * (1 + 6 * -(-part // 16) / 2) * rms
            assert err <= bound, (m, p)
            assert k >= 8 or torch.equal(out[p], chain)  # the float32 instruction: the same fused multiply-adds


@pytest.mark.parametrize("m,n,tile", [(100, 1500, (64, 64)), (290, 6000, (64, 128)), (290, 8960, (128, 128))])
@pytest.mark.parametrize("k,off", [(160, 0), (157, 0), (157, 3)])
def test_every_size_of_tiles(m, n, tile, k, off):
    """The distance from 64 bits, and numbers that are not finite or beyond the pieces in the second of a wave's row tiles and column
    tiles, alone and with a whole row, which leave all other elements as they are."""
    from pyre_amd.hip import ops
    from pyre_amd.hip.lib import lib

    assert lib().pyre_gemm_f32_tile_choice(m, n, k, 1) == 1000 * tile[0] + tile[1]
    a, w = operands(m, n, k, off)
    if off:
        w = torch.nn.functional.pad(w, (off, 0))[:, off:]
    out, chain = torch.full((m, n), float("nan"), device=DEV), torch.empty(m, n, device=DEV)
    ops.gemm_f32(a, w, None, out, m)
    ops.gemm_generic(a, w, None, chain, m)
    exact = a.double() @ w.double().T
    assert float((out.double() - exact).square().mean()) <= 1.1 ** 2 * float((chain.double() - exact).square().mean())
    b, v = a.clone() if off == 0 else torch.nn.functional.pad(a, (off, 0))[:, off:], w.clone()
    rows, cols = (33, 97, m - 1), (32, 40, 95, 127, 161, n - 1)
    b[33, 7], b[97, k - 1], b[m - 1, 0] = float("inf"), 2e38, float("nan")
    for i, col in enumerate(cols):
        v[col, (3 * i) % k] = (float("-inf"), 1e35, float("nan"))[i % 3]
    if off:
        v = torch.nn.functional.pad(v, (off, 0))[:, off:]
    got = torch.full((m, n), float("nan"), device=DEV)
    ops.gemm_f32(b, v, None, got, m)
    want = b.double() @ v.double().T
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.abs() > torch.finfo(torch.float32).max)
    fine = want.isfinite() & (want.abs() < 1e38)
    scale = b.double().abs() @ v.double().abs().T
    assert bool(((got.double() - want)[fine].abs() <= 2.0 ** -21 * scale[fine]).all())
    same = torch.ones(m, n, dtype=torch.bool, device=DEV)
    same[list(rows)], same[:, list(cols)] = False, False
    assert torch.equal(got[same], out[same])


@pytest.mark.parametrize("m,n,k,ks", [(129, 32768, 160, 1), (192, 32768, 157, 1), (566, 2048, 1536, 8), (400, 1500, 8960, 14), (260, 20000, 160, 2)])
def test_last_rows_in_smaller_tiles(m, n, k, ks):
    """Tiles of 128 rows with tiles of 64 behind them in one launch: the bits of a product of the last rows alone, bias, rows and columns past
    the end, a part's end within a step, and numbers that are not finite in either kind of tile; one launch for all parts in tiles of one size."""
    from pyre_amd.hip import ops
    from pyre_amd.hip.lib import lib

    assert lib().pyre_gemm_f32_tile_mixed(m, n, k, ks) == 1
    a, w = operands(m, n, k, 0)
    bias = torch.randn(n, generator=torch.Generator().manual_seed(1)).to(DEV)
    a[1, 3], a[m - 1, 2] = float("inf"), 1e33
    shape = (ks, m, n) if ks > 1 else (m, n)
    out = torch.full(shape, float("nan"), device=DEV)
    ops.gemm_f32(a, w, bias, out, m, ks)
    for rows in (torch.arange(0, 100), torch.arange(m - 100, m)):
        assert lib().pyre_gemm_f32_tile_mixed(100, n, k, ks) == 0
        want = torch.empty(shape[:-2] + (100, n), device=DEV)
        ops.gemm_f32(a[rows.to(DEV)].contiguous(), w, bias, want, 100, ks)
        assert torch.equal(out[..., rows.to(DEV), :].nan_to_num(), want.nan_to_num())
    exact = a.double() @ w.double().T + bias.double()
    got = (out.double().sum(0) if ks > 1 else out.double())
    fine = torch.ones(m, dtype=torch.bool, device=DEV)
    fine[[1, m - 1]] = False
    scale = a.double().abs() @ w.double().abs().T + bias.double().abs()
    assert bool(((got - exact)[fine].abs() <= 2.0 ** -21 * scale[fine]).all())
    if k % 16 == 0 and ks > 1:
        plain, whole = torch.empty(shape, device=DEV), torch.empty(m, n, device=DEV)
        ops.gemm_f32(a, w, None, plain, m, ks)
        ops.gemm_f32_whole(a, w, whole, m, ks)
        total = plain[0].clone()
        for p in plain[1:]:
            total += p
        assert torch.equal(whole.nan_to_num(), total.nan_to_num())


@pytest.mark.parametrize("m,n,k,ks", [(129, 32768, 160, 2), (192, 32700, 320, 3), (2049, 2048, 1536, 8), (2112, 2048, 1536, 8), (2305, 3584, 3584, 9)])
def test_last_rows_in_smaller_tiles_with_all_parts_added(m, n, k, ks):
    """The same tiles where a block adds all parts of k up itself: the bits of the parts added in their order, in the rows of the large
    tiles and of the small ones, whole rows and columns past the end, numbers that are not finite or beyond the pieces in both."""
    from pyre_amd.hip import ops
    from pyre_amd.hip.lib import lib

    assert lib().pyre_gemm_f32_tile_choice(m, n, k, 1) == 192128 and lib().pyre_gemm_f32_tile_mixed(m, n, k, 1) == 1
    a, w = operands(m, n, k, 0)
    behind = m // 128 * 128  # the first row of a small tile
    for row, value, places in ((3, float("inf"), (k // 2,)), (40, 2e35, range(0, k, 7)), (100, float("nan"), (1,)), (behind - 1, 3e38, (3,)),
                               (behind, -3e38, (k - 2,)), (m - 1, 1e30, (2, k // 2))):
        a[row, list(places)] = value
    if m - behind > 60:
        a[behind + 33, 5], a[behind + 40, k - 1] = float("-inf"), float("nan")
    w[n - 1, 4], w[n // 2, k - 3] = 1e33, -2e31
    parts, whole = torch.full((ks, m, n), float("nan"), device=DEV), torch.full((m, n), float("nan"), device=DEV)
    ops.gemm_f32(a, w, None, parts, m, ks)
    ops.gemm_f32_whole(a, w, whole, m, ks)
    want = parts[0].clone()
    for p in parts[1:]:
        want += p
    assert torch.equal(whole.isnan(), want.isnan()) and torch.equal(whole.nan_to_num(), want.nan_to_num())
    rows = torch.tensor(sorted({0, 3, 40, 100, behind - 2, behind - 1, behind, m - 1, *range(m - 70, m)}), device=DEV)  # in tiles of one size
    assert lib().pyre_gemm_f32_tile_choice(len(rows), n, k, ks) != 192128
    few = torch.empty(ks, len(rows), n, device=DEV)
    ops.gemm_f32(a[rows].contiguous(), w, None, few, len(rows), ks)
    assert torch.equal(few.nan_to_num(), parts[:, rows].nan_to_num())
    exact = a[rows].double() @ w.double().T
    fine, scale = exact.abs() < 1e38, a[rows].double().abs() @ w.double().abs().T
    assert bool(((whole[rows].double() - exact)[fine].abs() <= 2.0 ** -21 * scale[fine]).all())
