"""The decode attention that finishes the q/k/v product itself, whose own key and value do not come from the cache: with the
token at every place of a chunk, in pages of one chunk's half, of one and of two chunks, against the kernels apart."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from test_kernels_gpu import DEV, decode_attention, i32, paged_case, rnd, work_on_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("page,window", [(16, 0), (32, 0), (64, 9), (48, 0)])
@pytest.mark.parametrize("nq,nkv,hd", [(12, 2, 128), (3, 1, 64)])
def test_every_place_of_a_chunk(nq, nkv, hd, page, window):
    from pyre_amd.hip import ops
    from pyre_amd.hip.ops import Partials
    from pyre_amd.parts.attention_work import decode_alone, decode_capacity, decode_items, decode_work
    from pyre_amd.parts.rotary import rotary_tables

    ctx = [*range(1, 67), 385, 400, 417, 1000]
    _, kc, vc, table, pos, seq_of, _, _ = paged_case(ctx, [1] * len(ctx), nq, nkv, hd, page, torch.bfloat16, seed=3)
    n, scale, tab = len(ctx), hd ** -0.5, table.cpu()
    slots = [int(tab[s, (c - 1) // page]) * page + (c - 1) % page for s, c in enumerate(ctx)]
    for s, c in enumerate(ctx):
        last = int(tab[s, (c - 1) // page])
        kc[last, :, (c - 1) % page:, :] = float("nan")
        vc[last, :, :, (c - 1) % page:] = float("nan")
    parts = Partials(rnd(2, n, (nq + 2 * nkv) * hd, seed=5, scale=0.7), rnd((nq + 2 * nkv) * hd, seed=6))
    cos, sin = (t.to(DEV).contiguous() for t in rotary_tables(hd, 1e4, max(ctx) + 1))
    k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    q = torch.empty(n, nq * hd, device=DEV, dtype=torch.bfloat16)
    ops.rope_kv_write(parts, q, k1, v1, cos, sin, hd, pos, i32(slots), n, nq, nkv, hd, page)
    want = torch.empty(n, nq, hd, device=DEV, dtype=torch.bfloat16)
    decode_attention(ops, q.view(n, nq, hd), want, k1, v1, list(range(n)), pos, seq_of, table, nq, nkv, hd, page, scale, window)
    work = decode_work(np.arange(n, dtype=np.int32), pos.cpu().numpy(), n, window, nq, nkv)
    cap, items = max(decode_capacity(n, nq, nkv), int(work[0, 0])), decode_items(nq, nkv)
    got = torch.full((n, nq, hd), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.attn_decode_work_rope_bf16(parts, cos, sin, i32(slots), got, k2, v2, True, work_on_device(work, cap, pos, seq_of), cap, pos, seq_of,
                                   table, torch.empty(cap * items * 16 * hd, device=DEV), torch.empty(cap * items * 32, device=DEV),
                                   torch.zeros(cap * items, dtype=torch.int32, device=DEV), decode_alone(n, nq, nkv), nq, nkv, hd, page,
                                   scale, window)
    assert torch.isfinite(got.float()).all() and torch.equal(got, want)
    assert torch.equal(k1.view(torch.int16), k2.view(torch.int16)) and torch.equal(v1.view(torch.int16), v2.view(torch.int16))
