"""Into how many parts of k the 32-bit path splits its products: a rule on sizes, held against the kernels' conditions."""

from __future__ import annotations

import pytest

from pyre_amd.hip import ops


@pytest.mark.parametrize("units", [1, 64, 80, 120, 228, 256, 304])
def test_no_part_is_empty(units):
    """The kernels refuse a split that leaves a part without k: every k up to 20,000, weights from one block of output columns
    to more than the compute units."""
    for n_out in (1, 128, 129, 512, 1536, 2304, 2305, 4608, 8960, 17920, 40000, 152064):
        for k in range(1, 20001):
            ks = ops.gemm_f32_ksplit(n_out, k, units)
            assert 1 <= ks <= ops.F32_KSPLIT_MAX and (ks == 1 or k // ks >= ops.F32_KSPLIT_MIN_K), (n_out, k)
            assert (ks - 1) * ops.f32_part(k, ks) < k, (n_out, k)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [2688, 2689, 2692, 2700, 2704, 2705])
def test_the_kernels_take_the_split(k):
    """Around the sizes where fourteen parts of 208 are as long as k or longer: steps of few and of many rows against float64."""
    import torch

    g = torch.Generator().manual_seed(k)
    w = torch.randn(130, k, generator=g).cuda()
    ks = ops.gemm_f32_ksplit(130, k)
    for m in (1, 20, 300):
        a = torch.randn(m, k, generator=g).cuda()
        out = torch.full((ks, m, 130), float("nan"), device="cuda:0")
        ops.gemm_f32(a, w, None, out if ks > 1 else out[0], m, ks)
        want = a.double() @ w.double().T
        # sums of k products of values around one: a rounding of 2^-24 of a sum that grows as the root of k for each
        bound = 8 * 2.0 ** -24 * k ** 0.5 * k ** 0.5 * 4
        assert float((out.double().sum(0) - want).abs().max()) <= bound
        if k % 16 == 0 and m > 16 and ks > 1:
            whole = torch.full((m, 130), float("nan"), device="cuda:0")
            ops.gemm_f32_whole(a, w, whole, m, ks)
            assert float((whole.double() - want).abs().max()) <= bound
