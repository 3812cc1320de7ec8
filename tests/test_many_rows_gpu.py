"""Row kernels of steps of many rows, whose loads and stores go past the caches: bit for bit what the same rows give in smaller steps."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def rnd(*shape, seed=0, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV).to(dtype)


def parts(data, a, b, **more):
    from pyre_amd.hip.ops import Partials

    return Partials(data[:, a:b].contiguous(), **more)


def in_steps(run, n, step):
    """``run(a, b)`` on all rows at once and on steps of ``step`` rows (more than 128, whose rows are dealt to threads alike)."""
    whole = run(0, n)
    cut = [run(a, min(n, a + step)) for a in range(0, n, step)]
    for i, w in enumerate(whole):
        assert torch.isfinite(w.float()).all()
        assert torch.equal(w, torch.cat([c[i] for c in cut])), i


@pytest.mark.parametrize("hidden,n,parts_of_k,dtype", [(3584, 1171, 2, torch.float32), (3584, 1350, 1, torch.float32), (1540, 2731, 3, torch.bfloat16)])
def test_norms_with_pending_terms(hidden, n, parts_of_k, dtype):
    from pyre_amd.hip import ops

    assert n * hidden >= 1 << 22 > 400 * hidden
    resid, data, more = rnd(n, hidden, seed=1), rnd(parts_of_k, n, hidden, seed=2, dtype=dtype), rnd(parts_of_k, n, hidden, seed=3, dtype=dtype)
    gain, own = rnd(hidden, seed=4, dtype=torch.bfloat16), rnd(hidden, seed=5, dtype=torch.bfloat16)

    def layer(a, b, post):
        r, out = resid[a:b].clone(), torch.full((b - a, hidden), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops.add_layernorm(r, parts(data, a, b, post=post), gain, 1e-6, out)
        return r, out

    def terms(a, b):
        r, out = resid[a:b].clone(), torch.full((b - a, hidden), float("nan"), device=DEV, dtype=torch.bfloat16)
        post = ops.PostNorm(own, 1e-6, kind="rms")
        second = parts(more, a, b, post=post, scale=0.5)
        ops.add_rms_terms(r, parts(data, a, b, post=post, more=second, outer=ops.PostNorm(own, 1e-6, kind="rms")), gain, 1e-6, out)
        return r, out

    in_steps(lambda a, b: layer(a, b, None), n, 400)
    in_steps(lambda a, b: layer(a, b, ops.PostNorm(own, 1e-5)), n, 400)
    in_steps(terms, n, 400)
    # and what it is: the residual is the sum, the output its norm (rounded to 16 bits, of sums in float32)
    r, out = layer(0, n, None)
    want = resid.double() + data.double().sum(0)
    assert float((r.double() - want).abs().max()) <= 2.0 ** -21 * float(want.abs().max())
    normed = torch.nn.functional.layer_norm(want, (hidden,), gain.double(), None, 1e-6)
    assert float((out.double() - normed).abs().max()) <= 2.0 ** -8 * float(normed.abs().max())


@pytest.mark.parametrize("streams,hidden,n", [(2, 1536, 1400), (4, 1028, 1150), (2, 4096, 600)])
def test_streams(streams, hidden, n):
    from pyre_amd.hip import ops

    assert n * hidden * streams >= 1 << 22 > 200 * hidden * streams
    x, data = rnd(n, streams * hidden, seed=1), rnd(2, n, hidden, seed=2)
    mix, out_w, in_w, gain = rnd(streams, streams, seed=3), rnd(streams, seed=4), rnd(streams, seed=5), rnd(hidden, seed=6)

    def run(a, b):
        dst, out = torch.empty(b - a, streams * hidden, device=DEV), torch.full((b - a, hidden), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops.stream_norm(x[a:b].clone(), dst, streams, parts(data, a, b), mix, out_w, in_w, gain, None, 1e-6, out)
        return dst, out

    in_steps(run, n, 200)


@pytest.mark.parametrize("width,n,parts_of_k", [(8960, 470, 1), (12000, 360, 3), (18944, 230, 2)])
def test_poly_norm(width, n, parts_of_k):
    from pyre_amd.hip import ops

    assert n * width >= 1 << 22 > 150 * width
    data, abce = rnd(parts_of_k, n, width, seed=1), torch.tensor([0.5, -0.3, 0.2, 0.1], device=DEV)

    def run(a, b):
        out = torch.full((b - a, width), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops.poly_norm(parts(data, a, b), abce, 1e-6, out, b - a)
        return (out,)

    in_steps(run, n, 150)


@pytest.mark.parametrize("hidden,n,dtype", [(4100, 200, torch.bfloat16), (5120, 400, torch.float32), (8192, 600, torch.bfloat16), (16384, 130, torch.float32)])
def test_wide_rows(hidden, n, dtype):
    """More than 4,096 columns, whose residual is read behind the term's norm, against float64."""
    from pyre_amd.hip import ops

    resid, data, more = rnd(n, hidden, seed=1), rnd(2, n, hidden, seed=2, dtype=dtype), rnd(2, n, hidden, seed=3, dtype=dtype)
    gain, own = rnd(hidden, seed=4, dtype=torch.bfloat16), rnd(hidden, seed=5, dtype=torch.bfloat16)

    def norm(x, kind):
        x = x - x.mean(1, keepdim=True) if kind == "layer" else x
        return x / (x.square().mean(1, keepdim=True) + 1e-6).sqrt()

    r, out = resid.clone(), torch.full((n, hidden), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.add_layernorm(r, ops.Partials(data, post=ops.PostNorm(own, 1e-6)), gain, 1e-6, out)
    want = resid.double() + norm(data.double().sum(0), "layer") * own.double()
    checks = [(r, out, want, norm(want, "layer") * gain.double())]
    r, out, post = resid.clone(), torch.full_like(out, float("nan")), ops.PostNorm(own, 1e-6, kind="rms")
    ops.add_rms_terms(r, ops.Partials(data, post=post, more=ops.Partials(more, post=post, scale=0.5), outer=post), gain, 1e-6, out)
    both = norm(data.double().sum(0), "rms") * own.double() + 0.5 * norm(more.double().sum(0), "rms") * own.double()
    want = resid.double() + norm(both, "rms") * own.double()
    checks.append((r, out, want, norm(want, "rms") * gain.double()))
    for r, out, want, normed in checks:
        # float32 sums of some ten thousand values around one, and the output's 16 bits
        assert float((r.double() - want).abs().max()) <= 2.0 ** -19 * float(want.abs().max())
        assert float((out.double() - normed).abs().max()) <= 2.0 ** -8 * float(normed.abs().max())
