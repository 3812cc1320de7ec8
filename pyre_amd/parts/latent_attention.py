"""Softmax attention over one compressed row per token, from which every head's keys and values are made."""

from __future__ import annotations

import numpy as np
import torch

from pyre_amd.hip import ops
from pyre_amd.parts.attention import STEP_ARRAYS
from pyre_amd.parts.base import (LatentAttentionSpec, Mixer, PagedCacheSpec, PagedTensorSpec, StepArraySpec, TensorSpec,
                                 make_part, take)
from pyre_amd.parts.linear import Linear

#: rows of a request that keys and values are made of at a time (the product's groups)
GROUP = 32
#: keys of a portion, in multiples of its tokens, up to which keys and values are made of all of them (bounds the step's list of them)
MOST_KEYS = 64
#: keys and values that are made at a time: a portion with more of them runs over the rows, a step with more makes them in rounds
MADE_BYTES = 256 << 20
#: elements of a layer's cached rows from which on every portion runs over the rows: a product's operand lies within 4 GiB
PRODUCT_ELEMENTS = 1 << 31


def portion_pairs(start: int, n: int, window: int) -> int:
    """Pairs of a query and a key that it sees, of n tokens from position ``start`` on."""
    if not window or start + n <= window:
        return n * start + n * (n + 1) // 2
    short = max(0, window - start)  # tokens that see less than a window
    return short * start + short * (short + 1) // 2 + (n - short) * window


def seen_keys(start: int, n: int, window: int) -> int:
    return min(start + n, n + window - 1) if window else start + n


def made_rows(start: int, n: int, window: int) -> int:
    """Rows that the keys of a portion are made into: all that it sees, in whole groups."""
    return -(-seen_keys(start, n, window) // GROUP) * GROUP


def makes_heads(start: int, n: int, spec: LatentAttentionSpec) -> bool:
    """Whether a portion's attention runs over keys and values made of the compressed rows that it sees, or over the rows
    themselves. Decided by a portion's own sizes, so that its result does not depend on what runs beside it.

    Half multiply-adds of the attention kernels, which take 2.7e-9 us each of a full chip (a weight is three pieces). Over the rows a pair
    of a query and a key costs row + 3 rank of them where made ones cost key + 3 value elements, and a token and head is carried into the
    rows' space and out of it, rank x (key + value elements) at 4.5 times the price. To make a key costs rank / 2 a key or value element, and
    280 more since it is written and read. Few heads do not fill the chip even with several portions: a key is then less.

    Over the rows and over made keys and values, us a layer with what goes with each (heads of 128 + 64 and 128), one portion and sixteen in
    a step. Rows of 512 + 64, a window of 1,024: 12 heads, 64 tokens behind 1,000 105 and 48, 132 and 106, 128 tokens 114 and 52, 235 and 124;
    28 heads, 60 tokens behind 2,048 107 and 56, 238 and 213; 64 heads, 64 tokens behind 1,000 115 and 68 but 455 and 501, 32 tokens 108 and
    69 but 243 and 454, 128 tokens 116 and 70, 902 and 629. Without a window, 64 behind 3,000 of 64 heads 268 and 141 but 1,066 and 1,481. Rows
    of 256 + 64: 64 heads, 64 tokens behind 1,000 254 and 391 sixteen times, 28 heads 128 tokens behind 8,000 1,340 and 2,381, 256 tokens
    2,732 and 2,487. A whole prompt pays for no key twice: 12 heads, the first 2,048 tokens 183 and 55, the first 512 70 and 31, the first 16 31
    and 24. Of 1,392 portions, one and sixteen at a time, the line leaves 14 of those that make them more than 3 % slower for it, none of them alone
    in its step (12 heads, sixteen times 64 tokens behind 3,000, 288 and 362; else by 12 % at most)."""
    rows = made_rows(start, n, spec.window)
    elements = spec.key_dim + spec.value_dim
    if rows > MOST_KEYS * n + GROUP or rows * spec.num_heads * elements * 2 > MADE_BYTES:
        return False
    a_pair = 4 * spec.rank - spec.key_dim - 3 * spec.value_dim
    pairs, tokens = portion_pairs(start, n, spec.window) * a_pair, n * spec.rank * elements
    keys = seen_keys(start, n, spec.window) * elements * (560 + spec.rank)
    return 64 * (2 * pairs + 9 * tokens) > min(64, spec.num_heads + 32) * keys


def made_portions(hb, spec: LatentAttentionSpec):
    """The portions that :func:`makes_heads`: round, request, first token, tokens, position, first key, the row that it is made into."""
    counts = hb.q_start[1:] - hb.q_start[:-1]
    most = MADE_BYTES // (spec.num_heads * (spec.key_dim + spec.value_dim) * 2)
    rows = turn = 0
    for s in np.nonzero(counts != 1)[0]:
        t0, n = int(hb.q_start[s]), int(counts[s])
        start = int(hb.positions[t0])
        if makes_heads(start, n, spec):
            more = made_rows(start, n, spec.window)
            if rows + more > most:
                rows, turn = 0, turn + 1
            yield turn, int(s), t0, n, start, max(0, start - spec.window + 1) if spec.window else 0, rows
            rows += more


def plan_groups(hb, spec: LatentAttentionSpec) -> np.ndarray:
    """[G, 3], see :func:`~pyre_amd.hip.ops.gemm_tile_paged`, round by round."""
    out = [(s, p, start + n - 1) for _, s, _, n, start, lo, _ in made_portions(hb, spec) for p in range(lo, start + n, GROUP)]
    return np.asarray(out, dtype=np.int32).reshape(-1, 3)


def plan_tiles(hb, spec: LatentAttentionSpec) -> np.ndarray:
    """[T, 5], see :func:`~pyre_amd.hip.ops.latent_heads`, round by round, those that see the most keys first."""
    size = ops.LATENT_HEADS_TOKENS
    out = [(turn, t0 + k, min(size, n - k), start + k, s, row - lo) for turn, s, t0, n, start, lo, row in made_portions(hb, spec)
           for k in range(0, n, size)]
    out.sort(key=lambda t: (t[0], -(t[3] + t[2])))
    return np.asarray([t[1:] for t in out], dtype=np.int32).reshape(-1, 5)


def plan_rounds(hb, spec: LatentAttentionSpec) -> np.ndarray:
    """[R, 2]: groups and tiles of every round."""
    out: list[list[int]] = []
    for turn, _, _, n, start, _, _ in made_portions(hb, spec):
        if turn == len(out):
            out.append([0, 0])
        out[turn][0] += made_rows(start, n, spec.window) // GROUP
        out[turn][1] += -(-n // ops.LATENT_HEADS_TOKENS)
    return np.asarray(out, dtype=np.int32).reshape(-1, 2)


class LatentAttention(Mixer):
    """c = rms_norm(Wdkv h) gain; head i: k = Wuk_i c, v = Wuv_i c, out_i = softmax(q_i k^T scale) v; with a turned part
    r that all heads share, k = [Wuk_i c | r] and q_i = [unturned | turned].

    Only [c | r] is kept. 16-bit prompt portions make every head's keys and values of the rows that they see, in scratch memory
    (:func:`makes_heads`). Elsewhere neither is ever made: q_i . (Wuk_i c) = (Wuk_i^T q_i) . c, so a head's query is carried into the compressed row's space (a product per head), the attention kernels run with the kept
    rows as the one shared key head and their first part as the value head, and the weighted sum of rows is carried out
    again, Wuv_i (sum_j a_j c_j), the output's gate applied on the way. Queries (or the compressed row that they are
    made of), the kept row and the gate are one input product. A layer without a row of its own (``own_latent`` False)
    reads the pages that another layer of the same sizes wrote."""

    def __init__(self, spec: LatentAttentionSpec):
        row = spec.rank + spec.rot_dim
        if not (0 < spec.rank <= ops.LATENT_MAX_RANK) or row > ops.LATENT_MAX_ROW:
            raise ValueError(f"latent attention: a row of {spec.rank} + {spec.rot_dim} elements is outside 1..{ops.LATENT_MAX_RANK} "
                             f"(1..{ops.LATENT_MAX_ROW} with its turned part), the sizes that the attention kernels take")
        if min(spec.key_dim, spec.value_dim, spec.num_heads) <= 0 or min(spec.rot_dim, spec.q_rank, spec.window) < 0:
            raise ValueError("latent attention: bad head sizes")
        if spec.rot_dim:
            if spec.position is None or spec.position.kind != "rotary" or spec.position.pairing not in ("halves", "neighbours"):
                raise ValueError("latent attention: a turned part needs a rotary position encoding")
            if spec.position.head_dim != spec.rot_dim or spec.position.rotary_dim not in (None, spec.rot_dim):
                raise ValueError(f"latent attention: its turned part of {spec.rot_dim} elements is turned whole")
        self.spec = spec
        self.row = row
        self.position = make_part("position", spec.position) if spec.rot_dim else None
        self.q_dim = spec.num_heads * (spec.key_dim + spec.rot_dim)
        self.o_dim = spec.num_heads * spec.value_dim
        first = spec.q_rank or self.q_dim
        self.row_col = first
        self.gate_col = first + (row if spec.own_latent else 0)
        self.inp = Linear(spec.hidden_size, self.gate_col + (self.o_dim if spec.gated else 0), "lattn.in")
        self.q_up = Linear(spec.q_rank, self.q_dim, "lattn.q_up") if spec.q_rank else None
        self.out = Linear(self.o_dim, spec.hidden_size, "lattn.out")
        self.gain = self.q_gain = self.key_up = self.value_up = self.heads_up = self.sink = None
        self.plan_name = f"latent.{spec.num_heads}.{spec.window}.{spec.rank}.{spec.rot_dim}.{spec.key_dim}.{spec.value_dim}"

    def cache_spec(self):
        return PagedCacheSpec((PagedTensorSpec("c", (1, self.row), token_axis=1),), self.spec.window)

    def step_arrays(self):
        if self.heads_up is None:
            return list(STEP_ARRAYS)
        plan, spec = self.plan_name, self.spec

        def row_tiles(hb):  # the tiles of the other portions
            tiles = hb.arrays["attention.prefill_tiles"]
            made = np.zeros(hb.n_seqs, dtype=bool)
            made[hb.arrays[f"{plan}.tiles"][:, 3]] = True
            return tiles[~made[hb.seq_of_token[tiles[:, 0]]]]

        def plain_tokens(hb):  # the range of tokens in which those lie whose attention runs over the rows themselves
            singles, rows = hb.arrays["attention.decode_tokens"], hb.arrays[f"{plan}.row_tiles"]
            if not len(hb.arrays[f"{plan}.tiles"]) or not (len(singles) or len(rows)):
                return np.zeros(2, dtype=np.int32)
            first = [int(x.min()) for x in (singles, rows[:, 0]) if len(x)]
            last = [int(x.max()) + 1 for x in (singles, rows.sum(axis=1) - 1) if len(x)]
            return np.asarray([min(first), max(last)], dtype=np.int32)

        return [*STEP_ARRAYS,
                StepArraySpec(f"{plan}.groups", lambda n_cap, s_cap: 3 * (MOST_KEYS * n_cap // GROUP + 2 * s_cap), lambda hb: plan_groups(hb, spec)),
                StepArraySpec(f"{plan}.tiles", lambda n_cap, s_cap: 5 * (n_cap // ops.LATENT_HEADS_TOKENS + s_cap),
                              lambda hb: plan_tiles(hb, spec)),
                StepArraySpec(f"{plan}.rounds", lambda n_cap, s_cap: 2 * s_cap, lambda hb: plan_rounds(hb, spec)),
                StepArraySpec(f"{plan}.row_tiles", STEP_ARRAYS[1].capacity, row_tiles),
                StepArraySpec(f"{plan}.plain", lambda n_cap, s_cap: 2, plain_tokens)]  # once a step, not in every layer

    def linears(self) -> list:
        return [lin for lin in (self.inp, self.q_up, self.out) if lin is not None]

    def tensor_specs(self) -> list[TensorSpec]:
        s, p = self.spec, self.spec.prefix
        if s.q_rank:
            specs = [TensorSpec(f"{p}.dq", (s.q_rank, s.hidden_size)), TensorSpec(f"{p}.dq.norm", (s.q_rank,), init="gain"),
                     TensorSpec(f"{p}.uq", (self.q_dim, s.q_rank))]
        else:
            specs = [TensorSpec(f"{p}.q", (self.q_dim, s.hidden_size))]
        if s.own_latent:
            specs += [TensorSpec(f"{p}.dkv", (self.row, s.hidden_size)), TensorSpec(f"{p}.dkv.norm", (s.rank,), init="gain")]
        if s.sink:
            specs.append(TensorSpec(f"{p}.sink", (s.num_heads,)))
        if s.gated:
            specs.append(TensorSpec(f"{p}.g", (self.o_dim, s.hidden_size)))
        # random weights: the way up from the compressed row drawn wider, so that keys have the scale of queries
        return specs + [TensorSpec(f"{p}.uk", (s.num_heads * s.key_dim, s.rank), init="normal:0.1"),
                        TensorSpec(f"{p}.uv", (self.o_dim, s.rank), init="normal:0.1"),
                        TensorSpec(f"{p}.o", (s.hidden_size, self.o_dim))]

    def bind(self, tensors, runtime) -> None:
        s, p = self.spec, self.spec.prefix
        parts = [take(tensors, f"{p}.dq" if s.q_rank else f"{p}.q")]
        if s.own_latent:
            parts.append(take(tensors, f"{p}.dkv"))
            self.gain = take(tensors, f"{p}.dkv.norm").float().contiguous()
        if s.gated:
            parts.append(take(tensors, f"{p}.g"))
        w = torch.cat(parts, dim=0) if len(parts) > 1 else parts[0]
        del parts
        self.inp.set(w)
        if s.q_rank:
            self.q_gain = take(tensors, f"{p}.dq.norm").float().contiguous()
            self.q_up.set(take(tensors, f"{p}.uq"))
        if s.sink:
            self.sink = take(tensors, f"{p}.sink").float().contiguous()
        self.out.set(take(tensors, f"{p}.o"))
        # per head [outputs, inputs] both ways: [rank, key_dim] carries a query in, [value_dim, rank] a sum out
        uk, uv = take(tensors, f"{p}.uk"), take(tensors, f"{p}.uv")
        self.key_up = uk.view(s.num_heads, s.key_dim, s.rank).transpose(1, 2).contiguous()
        if uk.dtype == torch.bfloat16 and self._can_make_heads():
            both = [t.view(s.num_heads, -1, s.rank) for t in (uk, uv)]
            self.heads_up = torch.cat(both, dim=1).view(-1, s.rank)  # a head's key, then its value, of a row
        self.value_up = uv.view(s.num_heads, s.value_dim, s.rank).contiguous()

    def _can_make_heads(self) -> bool:
        """Sizes that the kernels over made keys and values take."""
        s = self.spec
        return (ops.latent_heads_supports(s.key_dim, s.rot_dim, s.value_dim) and s.rank % 64 == 0 and self.row % 8 == 0)

    def forward(self, ctx, h, cache):
        s, n, ws = self.spec, ctx.n_tokens, ctx.workspace
        heads, rows = s.num_heads, cache["c"]
        q = ws.get("lattn.q", (n, heads, s.key_dim), ctx.dtype)
        wide = ws.get("lattn.q_in", (n, heads, self.row), ctx.dtype)
        turn = {}
        if s.rot_dim:
            cos, sin, _ = self.position.rotary(ctx.runtime)
            turn = dict(cos=cos, sin=sin, neighbours=s.position.pairing == "neighbours", positions=ctx.positions)
        proj = self.inp.forward(ctx, h, n)
        row = (self.row_col, self.gain, rows, cache.slots) if cache.writes and s.own_latent else None
        gate = ws.get("lattn.gate", (n, self.o_dim), torch.float32) if s.gated else None
        latent = dict(row=row, gate=(self.gate_col, self.o_dim, gate) if s.gated else None, eps=s.norm_eps, **turn)
        if s.q_rank:
            cq = ws.get("lattn.cq", (n, s.q_rank), ctx.dtype)
            ops.latent_rows(proj, n, s.rank, s.rot_dim, ctx.dtype, normed_queries=(0, s.q_rank, self.q_gain, cq), **latent)
            ops.latent_rows(self.q_up.forward(ctx, cq, n), n, s.rank, s.rot_dim, ctx.dtype,
                            queries=(0, heads, s.key_dim, q, wide), **turn)
        else:
            ops.latent_rows(proj, n, s.rank, s.rot_dim, ctx.dtype, queries=(0, heads, s.key_dim, q, wide), **latent)
        o = ws.get("lattn.o", (n, heads, s.value_dim), ctx.dtype)
        made = 0
        if self.heads_up is not None and rows.numel() < PRODUCT_ELEMENTS:
            made = len(ctx.host.arrays[f"{self.plan_name}.tiles"])
        a, b = ctx.host.arrays[f"{self.plan_name}.plain"].tolist() if made else (0, n)
        if b > a:
            ops.head_matmul(q[a:b], self.key_up, wide[a:b], b - a)
            o_in = ws.get("lattn.o_in", (n, heads, s.rank), ctx.dtype)
            self._attend(ctx, wide, rows, o_in, cache, f"{self.plan_name}.row_tiles" if made else "attention.prefill_tiles")
            # (whatever lies between a and b besides is written again below)
            ops.head_matmul(o_in[a:b], self.value_up, o[a:b], b - a, None if gate is None else gate[a:b])
        if made:
            self._attend_made(ctx, q, wide[:, :, s.rank:], rows, o, cache, gate)
        return self.out.forward(ctx, o.view(n, self.o_dim), n)

    def _attend_made(self, ctx, q, turned, rows, out, cache, gate) -> None:
        s, g0, t0 = self.spec, 0, 0
        groups, tiles = ctx.arrays[f"{self.plan_name}.groups"], ctx.arrays[f"{self.plan_name}.tiles"]
        for g, t in ctx.host.arrays[f"{self.plan_name}.rounds"].tolist():
            kv = ctx.workspace.get("lattn.kv", (s.num_heads, GROUP * g, s.key_dim + s.value_dim), ctx.dtype)
            ops.gemm_tile_paged(rows, groups[3 * g0:], g, cache.table, self.heads_up, kv)
            ops.latent_heads(q, turned, kv, rows, out, tiles[5 * t0:], t, cache.table, s.scale, s.window, self.sink, gate)
            g0, t0 = g0 + g, t0 + t

    def _attend(self, ctx, q, rows, out, cache, tile_list: str) -> None:
        s = self.spec
        step = (ctx.positions, ctx.seq_of_token, cache.table, s.num_heads, s.rank, self.row, cache.page_size, s.scale, s.window,
                self.sink)
        tiles = ctx.host.arrays[tile_list]
        singles = ctx.host.arrays["attention.decode_tokens"]
        if len(tiles):
            ops.latent_attn_tile(q, rows, out, ctx.arrays[tile_list], len(tiles), *step)
        if len(singles):
            spans = ops.latent_attn_spans(cache.table.shape[1], cache.page_size, s.window)
            scratch = None
            if spans > 1:
                scratch = ctx.workspace.get("lattn.spans", (len(singles) * s.num_heads * spans * (s.rank + 2),), torch.float32)
            ops.latent_attn_single(q, rows, out, ctx.arrays["attention.decode_tokens"], len(singles), *step, scratch=scratch)
