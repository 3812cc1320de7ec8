"""Choice of the faster kernels of the 16-bit path.

Each function returns None / False when its fast path does not take the case
(element type, sizes, alignment); the caller then runs the general kernel.
Nothing here changes what is computed, only by which kernel. Sizes that no kernel
of this framework takes go to the vendor's BLAS through ``torch.mm``, as the
reference's products do (`pyre/model.py:84-87` are ``nn.Linear``), and so do the
logits of many rows where that is ahead (:func:`head_in_tiles`); the true 32-bit
path never comes here.
"""

from __future__ import annotations

from functools import lru_cache

import torch

from pyre_amd.hip import ops
from pyre_amd.hip.ops import DEFAULT_UNITS, Partials
from pyre_amd.parts import attention_work as plan

#: most rows the weight-streaming MFMA kernel takes; above, 16-bit products go to the kernel that keeps
#: up to 256 rows in a block where it pays and else to the one that takes tiles of rows and columns
SKINNY_MAX_ROWS = 64
#: the most partial sums of a weight-streaming product
SKINNY_MAX_KSPLIT = 12
#: up to this many rows the gate/up product and the SiLU-gate can be one weight-streaming kernel
#: (shapes whose features one round of the other kernel's blocks does not hold: the 32B shape's
#: at up to 24 rows)
FUSED_SILU_MAX_ROWS = 64
#: most rows of the kernel between the two, which keeps a step's rows against 64 rows of the weights
MID_MAX_ROWS = 256
MID_MAX_KSPLIT = 12
#: fewest rows at which that kernel takes the gate/up product with the SiLU-gate
MID_SILU_MIN_ROWS = 1
#: fewest rows at which its form with 128 rows of the weights a block takes a narrow product
#: (just above a size at which decode steps are captured, so that an eager step and its replay agree)
MID_WIDE_MIN_ROWS = 25


#: what the weight-streaming products reach while they stream, measured on the 7B shapes on an
#: MI355X, in bytes per microsecond over the whole chip; the time of one run of 128 k of a block
#: and of one more addend in the consumer, in microseconds
STREAM_BYTES_PER_US, STREAM_RUN_US, STREAM_PART_US = 6.5e6, 0.9, 0.1


def skinny_ksplit(m: int, n_out: int, k: int, units: int = DEFAULT_UNITS) -> int:
    """Into how many parts of k to split a weight-streaming product. A block (64 rows of the
    weights, 128 of wide ones) walks its part of k in dependent runs of 128, about 0.9 us
    each, and the blocks of a compute unit share its time: the product takes as long as the
    longest walk or as the unit with the most blocks needs for its bytes (6.5 TB/s over the
    ``units`` compute units), whichever is more; every part costs its consumer
    one more addend. The split with the least of that is chosen, at least four runs a part."""
    run_us, bytes_per_us, part_us = STREAM_RUN_US, STREAM_BYTES_PER_US, STREAM_PART_US
    tiles = -(-n_out // 16)
    row_blocks = -(-n_out // (128 if tiles >= 2048 else 64))
    runs = -(-k // 128)
    stream_us = 2.0 * n_out * k / bytes_per_us
    best, best_cost = 1, None
    for ks in range(1, SKINNY_MAX_KSPLIT + 1):
        per = -(-runs // ks)
        if ks > 1 and per < 4:
            break
        if -(-runs // per) != ks:
            continue  # would leave parts empty
        blocks = row_blocks * ks
        busiest = -(-blocks // units)
        cost = max(per * run_us, stream_us * busiest * units / blocks) + part_us * ks
        if best_cost is None or cost < best_cost - 1e-9:
            best, best_cost = ks, cost
    return best


def mid_ksplit(n_out: int, k: int, block_rows: int = 64, units: int = DEFAULT_UNITS) -> int:
    """Into how many parts of k the kernel that keeps a step's rows in a block (up to 256) splits a
    product, or 0 if it is not the one to take. A block has 64 rows of the weights; the kernel is at its best when the blocks
    of all parts fill the ``units`` compute units in one round, and beats the BLAS library where that
    takes at least two parts of 384 k or more (shorter parts gain nothing and cost the consumer
    another addend; measured on the 1.5B, 7B and 32B shapes: q/k/v, the
    attention output and the feed-forward's way down take 9 to 20 us where the library takes 19
    to 31, and 60 against 100 at 7B's way down; a product too wide for that, gate/up without the gate in its
    epilogue, is not this kernel's)."""
    blocks = -(-n_out // block_rows)
    ks = min(units // blocks, k // 384, MID_MAX_KSPLIT)
    while ks > 1 and (ks - 1) * (-(-(-(-k // ks)) // 64) * 64) >= k:
        ks -= 1  # would leave a part empty
    return ks if ks >= 2 else 0


#: products whose library result is kept in float32 instead of being rounded to 16 bits:
#: q/k/v (rotated and rounded once afterwards) and the attention output projection (added
#: to the float32 residual). Measured on the tiny test models this halves the 16-bit
#: path's distance from an exact run; it costs about 2 % of a 2,048-token prefill.
# The same holds for a sandwich layer's products whose results are normed before anything else rounds them:
# the shared input and output products of mixers side by side (and of each alone), and the way down of the
# gated unit with clipped inputs (measured on a four-layer model of 512 columns: whole prompts 0.059 -> the
# 0.026 of short portions, whose products hand on float32 partial sums anyway).
LIBRARY_F32_ROLES = frozenset({"attn.qkv", "attn.out", "mix.in", "mix.out", "cattn.in", "cattn.out", "gla.in", "gla.out",
                               "glu.down", "tattn.qk", "tattn.out", "lattn.in", "lattn.out", "geglu.down", "moe.router",
                               "moe.down", "mix.out0", "mix.out1", "sattn.in", "sattn.out", "ret.in", "ret.out",
                               "relu2.down", "gmoe.router", "gmoe.down", "wattn.in", "wattn.out", "gdr.in", "gdr.out",
                               "stmoe.router", "stmoe.down", "side.gate", "side.proj", "lattn.q_up", "poly.up",
                               "poly.down", "light.in", "light.out", "ssm.in", "ssm.out", "ssm.x", "ssm.dt", "reglu.down",
                               "pass.start", "pass.stream"})


#: products of many rows that are handed on in 16 bits, where the library takes them (the products of tiles hand on
#: float32 sums like those of few rows): activations that the next kernel reads once and rounds anyway
TILE_ROLES = LIBRARY_F32_ROLES | {"ffn.down"}


def takes_tiles(rt, lin, n: int, x=None) -> bool:
    """Whether a 16-bit product of ``n`` rows goes to the kernel of tiles of up to 256 x 256 (`gemm_tile.hip`): all of more
    rows than the weight-streaming kernel takes whose sizes it supports and whose operands lie on 16 bytes (``x`` None: rows like a
    workspace's; a weight that its owner hands over may be a view). Against the BLAS library's products (us here and there, the
    gated unit with them, launches one behind the other): the 7B shape's q/k/v 26 and 35 at 566 rows, 64 and 68 at 2,048, 113 and 122
    at 4,096, 204 and 212 at 8,192; its attention output 27 and 28, 50 and 53, 86 and 90, 160 and 169; its gate/up 159 and 185, 413 and
    553, 790 and 872, 1,528 and 1,778; its way down 89 and 143, 214 and 350, 396 and 670, 781 and 1,214. The 1.5B shape's q/k/v 12 and 21,
    20 and 23, 34 and 32, 47 and 54; its gate/up 32 and 46, 97 and 138, 183 and 215, 346 and 428; its way down 23 and 39, 50 and 66, 85 and
    99, 159 and 168. The 32B shape's gate/up 295 and 317, 831 and 1,068, 1,608 and 1,939, 3,139 and 3,586; its way down 163 and 252, 437 and
    450, 849 and 896, 1,650 and 2,241. A consumer's reading of more parts than one, up to six at 566 rows, comes to it (0.2 us a megabyte)."""
    if not rt.options.get("tile_gemm", True) or n <= SKINNY_MAX_ROWS or lin.weight.data_ptr() % 16 or (x is not None and x.data_ptr() % 16):
        return False
    return ops.gemm_tile_supports(n, lin.out_features, lin.in_features, lin.in_features if x is None else x.stride(0), lin.weight.stride(0))


#: rows from which, and the k and the weights' elements up to which, a product of few rows is ahead in tiles
FEW_TILES_MIN_ROWS, FEW_TILES_MAX_K, FEW_TILES_MAX_WEIGHTS = 129, 4608, 17 << 20


def few_tiles(n: int, n_out: int, k: int) -> int:
    """In how many parts of k the kernel of tiles makes a product of so few rows that a block could keep them all, where it is ahead of the
    one that does so, else 0. From 129 rows on what a block takes from L2 (all rows again for every 64 or 128 rows of
    W) bounds that kernel, and tiles of 64 x 128 fill the chip with fewer parts for the consumer to read. In a graph, weights from memory, the norm that
    reads the parts with it, us there and here at 129, 192 and 256 rows: the 1.5B shape's q/k/v 12.1 and 11.1, 13.3 and 12.3, 15.7 and 13.0, its
    attention output 11.3 and 10.2, 12.7 and 11.2, 14.8 and 12.4; the 7B shape's q/k/v (7 parts, and 2 or 3) 22.9 and 19.0, 24.0 and 20.8, 26.6 and 22.5
    (the products alone 15.4 and 14.9, 15.9 and 16.3, 19.0 and 17.0), its attention output (8 parts, and 3 or 4) 20.9 and 17.1, 22.6 and 18.1, 24.6 and
    20.5; 3,072 x 4,608 22.0 and 18.1, 23.4 and 19.6, 24.9 and 21.6; 1,024 x 4,608 13.0 and 11.7, 15.0 and 12.7, 17.5 and 13.8; 4,096 x 4,096 23.1 and 19.4, 23.2
    and 21.6, 26.6 and 21.6; 8,192 x 2,048 22.4 and 20.8, 23.9 and 22.5, 27.9 and 22.9, the least that is gained within these limits. At 128 rows they
    are about alike. Beyond the limits the products alone (1.5B way down 13.1 and 14.7, 14.7 and 15.9, 17.4 and 17.0; 7B 41.7 and 45.4, 42.5
    and 50.0, 50.3 and 51.1; the 32B shape's attention output 20.0 and 22.4, 21.8 and 24.3, 25.8 and 24.8) leave less to gain; 4,608 x 4,096 is ahead by 3 to 14 %
    with its consumer. The parts are those of the next multiple of 64 rows, at which such decode steps are captured."""
    if not FEW_TILES_MIN_ROWS <= n <= MID_MAX_ROWS or k > FEW_TILES_MAX_K or n_out * k > FEW_TILES_MAX_WEIGHTS:
        return 0
    return ops.gemm_tile_parts(-(-n // 64) * 64, n_out, k)


#: features of a head from which its product of many rows is made in tiles, and the k up to which one of any size is
HEAD_TILES_MIN_FEATURES, HEAD_TILES_MAX_SHORT_K = 120_000, 512
#: whole rows of tiles of 256 -> the k up to which the head's product is made in tiles where up to 64 rows stand behind them
HEAD_TILES_MAX_K_BEHIND = {1: 5120, 2: 2048}


def head_in_tiles(n: int, n_out: int, k: int) -> bool:
    """Whether the logits of ``n`` rows, more than the weight-streaming kernel takes, are made in tiles rather than by the library's product. k is
    not split (the results go to their place), so a head of fewer features than about two rounds of tiles leaves a round
    nearly empty here and there, and up to 64 rows behind whole rows of tiles of 256 cost a row of tiles of their own, the more the longer k.
    Us in tiles and by the library: 151,936 x 1,536 111 and 128 at 65 rows, 142 and 152 at 190, 153 and 164 at 256, 179 and 197 at 257, 228 and
    278 at 512, 282 and 304 at 513, 1,065 and 1,157 at 2,400; 152,064 x 3,584 219 and 231, 269 and 294, 289 and 322, 399 and 433, 459 and 554, but 609
    and 588 at 513, 619 and 606 at 566 (from 577 rows on 620 and 694), 2,111 and 2,199 at 2,400; 152,064 x 5,120 866 and 816 at 513, 872 and 840 at 566;
    151,936 x 8,192 941 and 866 at 257. 32,000 x 2,048 33 and 26 at 129, 48 and 37 at 257, though 55 and 57 at 512; 64,000 x 4,096 behind by 15 % at
    257 and at 513, 100,352 x 4,096 by 11 % at 257, 128,256 x 4,096 ahead by 10 % there. With k of up to 512, where the results bound both,
    ahead but for a few sizes that are alike, 3 % behind at worst (32,000 features: 0.47 of the library's time at 65 rows, 0.9 at 512)."""
    if k <= HEAD_TILES_MAX_SHORT_K:
        return True
    whole, behind = divmod(n, 256)
    return n_out >= HEAD_TILES_MIN_FEATURES and not (1 <= behind <= 64 and k > HEAD_TILES_MAX_K_BEHIND.get(whole, k))


def library_takes(lin, rt, n: int) -> bool:
    """Whether the 16-bit product of ``n`` rows (more than the weight-streaming kernel's) and this weight is left to the BLAS
    library once no kernel for few rows takes it."""
    by_tiles = lin.role in TILE_ROLES or (lin.role == "ffn.gate_up" and lin.bias is None)
    return not (by_tiles and takes_tiles(rt, lin, n))


def _is_bf16(ctx, lin, x) -> bool:
    return (ctx.runtime.dtype == torch.bfloat16 and lin.weight.dtype == torch.bfloat16
            and x.dtype == torch.bfloat16)


def narrow_kernel(n: int, n_out: int, k: int, options: dict | None = None,
                  units: int = DEFAULT_UNITS) -> tuple[str, int, bool]:
    """Which of our kernels takes a 16-bit product of ``n`` rows whose result is handed on as partial
    sums: ("stream", parts of k, False) for the weight-streaming kernel, ("block", parts, wide) for the
    kernel that keeps the step's rows in a block (``wide``: 128 rows of the weights a block instead
    of 64), ("", 0, False) for neither (the kernel of tiles then, or the BLAS library). From 129 rows on products of short k that it
    answers "block" for are made in tiles after all (:func:`few_tiles`). A function of the sizes (and of the
    device's compute units, which an engine reads once) alone; the
    thresholds in rows lie just above sizes at which decode steps are captured, so that an eager step
    and its replay at the padded size agree."""
    if not options:
        return _narrow_kernel(n, n_out, k, units, True, MID_WIDE_MIN_ROWS, True, True)
    opt = options
    return _narrow_kernel(n, n_out, k, units, opt.get("mid_gemm", True), opt.get("mid_wide_min_rows", MID_WIDE_MIN_ROWS),
                          opt.get("skinny_gemm", True), opt.get("mid_small", True))


@lru_cache(maxsize=4096)
def _narrow_kernel(n: int, n_out: int, k: int, units: int, block, wide_min_rows: int, stream, small) -> tuple[str, int, bool]:
    """The rule itself, kept by its sizes: three products a layer ask for it, and the splits that it weighs take longer than a launch."""
    if block and wide_min_rows <= n <= MID_MAX_ROWS:
        # With 128 rows of the weights a block, where such blocks fill three quarters of the chip at
        # least: a block's bytes are the step's rows of X and its rows of W, over its part of k, and
        # with as many of the one as of the other they are fewest (at few rows of X a stage, and the
        # barrier that goes with it, carries twice the bytes). From 25 rows on the weight-streaming
        # kernel slows down (64 activations come from L2 once per 128 rows of weights, and four
        # times the LDS reads and MFMAs sit between a run's arrival and the next run's request),
        # this one does not. Measured in steps of the 7B shape against the weight-streaming kernel:
        # 4.43 against 4.47 ms at 32 requests, 5.20 against 5.29 at 48, 5.74 against 5.88 at 64 (at 8
        # and 16: 3.46 against 3.44, 3.79 against 3.77); of the 32B shape 35.5 against 36.2 at 64.
        # Against 64 rows of the weights a block: 7.78 against 7.94 ms at 96 requests, 8.86 against
        # 8.90 at 128, and where every product was made by this kernel 12.56 against 12.63 at 192, 15.25 against 15.34 at 256.
        ks = mid_ksplit(n_out, k, 128, units)
        if ks and 4 * -(-n_out // 128) * ks >= 3 * units:
            return "block", ks, True
    if n <= SKINNY_MAX_ROWS and stream:
        ks = skinny_ksplit(n, n_out, k, units)
        if block and small and -(-n_out // 64) * ks < units and mid_ksplit(n_out, k, 64, units):
            # A product so small that the weight-streaming kernel's blocks do not fill the compute
            # units (the 1.5B shape's: 96, 72 and 240 blocks) is latency all the way, and the other
            # kernel, whose loads go straight into a ring in LDS, starts sooner: 1.7 % of a step of
            # 8 requests of that shape, 3 % at 32, 4 % at 64. Where the blocks fill the chip (7B:
            # 504) it is 3 % slower at 8 rows.
            return "block", mid_ksplit(n_out, k, 64, units), False
        return "stream", ks, False
    if n <= MID_MAX_ROWS and block:
        ks = mid_ksplit(n_out, k, 64, units)
        if not ks and int(block) == 2:  # tests: also where it does not pay, as with a tiny model
            ks = 2 if k > 64 else 1
        if ks:
            return "block", ks, False
    return "", 0, False


def linear(lin, ctx, x, n, out):
    rt = ctx.runtime
    if not _is_bf16(ctx, lin, x):
        return None
    k, n_out, weight = lin.in_features, lin.out_features, lin.weight
    ldx, ldw = x.stride(0), weight.stride(0)
    library = rt.options.get("library_gemm", True)

    def streams() -> bool:
        return rt.options.get("skinny_gemm", True) and ops.gemm_skinny_supports(min(n, SKINNY_MAX_ROWS), n_out, k, ldx, ldw)

    if out is not None:
        # float32 results wanted in place (the head's logits): of more rows than a block of the weight-streaming kernel keeps (a large
        # decode step, every row of a portion) in tiles, whole, where those are ahead of the library's product.
        if ((not library or head_in_tiles(n, n_out, k)) and takes_tiles(rt, lin, n, x) and out.is_contiguous()
                and out.data_ptr() % 16 == 0):
            ops.gemm_tile_bf16(x, weight, out, n, 1)
        elif (n <= SKINNY_MAX_ROWS or not library) and streams():  # no split, 64 rows at a time
            for r0 in range(0, n, SKINNY_MAX_ROWS):
                rows = min(SKINNY_MAX_ROWS, n - r0)
                ops.gemm_skinny_bf16(x[r0:r0 + rows], lin.weight, out[r0:r0 + rows], rows, 1)
        elif library:  # one pass over the weights
            torch.mm(x if n == x.shape[0] else x[:n], lin.weight.t(), out_dtype=torch.float32, out=out)
        else:
            return None
        return Partials(out.view(1, n, n_out), lin.bias)
    kernel, ks, wide = narrow_kernel(n, n_out, k, rt.options, rt.compute_units)
    if kernel == "stream" and not streams():
        kernel = ""
    if kernel == "block" and not ops.gemm_mid_supports(n, n_out, k, ldx, ldw):
        kernel, ks = ("stream", skinny_ksplit(n, n_out, k, rt.compute_units)) if n <= SKINNY_MAX_ROWS and streams() else ("", 0)
    parts = 0
    if (kernel == "block" and n >= FEW_TILES_MIN_ROWS and rt.options.get("mid_gemm", True) != 2 and lin.role in TILE_ROLES
            and not lin.whole and takes_tiles(rt, lin, n, x)):
        parts = few_tiles(n, n_out, k)
    if kernel and not parts:
        buf = rt.workspace.get(lin.partials_name, (ks, n, n_out), torch.float32)
        if kernel == "stream":
            ops.gemm_skinny_bf16(x, weight, buf, n, ks)
        else:
            ops.gemm_mid_bf16(x, weight, buf, n, ks, wide=wide)
        return Partials(buf, lin.bias)
    if lin.role in TILE_ROLES and takes_tiles(rt, lin, n, x):
        parts = parts or (1 if lin.whole else ops.gemm_tile_parts(n, n_out, k))
        buf = rt.workspace.get(lin.partials_name, (parts, n, n_out), torch.float32)
        ops.gemm_tile_bf16(x, lin.weight, buf, n, parts)
        return Partials(buf, lin.bias)
    if not library:
        return None
    if lin.role in rt.options.get("library_f32_roles", LIBRARY_F32_ROLES):
        buf = ctx.workspace.get(f"linear32.{lin.role}", (n, n_out), torch.float32)
        torch.mm(x if n == x.shape[0] else x[:n], lin.weight.t(), out_dtype=torch.float32, out=buf)
    else:
        buf = ctx.workspace.get(f"linear16.{lin.role}", (n, n_out), torch.bfloat16)
        torch.mm(x if n == x.shape[0] else x[:n], lin.weight.t(), out=buf)
    return Partials(buf.view(1, n, n_out), lin.bias)


def gate_up_silu(lin, ctx, x, n, act, unit=None) -> bool:
    """silu(x gate^T) * (x up^T) in one kernel (``unit`` = (limit, slope, shift): the gated unit
    g sigmoid(slope g) (u + shift) with clipped inputs instead, in the same epilogues): the kernel that keeps all rows in a block for up to
    256 rows where one round of blocks holds the features, else the kernel of tiles for many rows and the weight-streaming
    kernel for a decode step's few."""
    if not _is_bf16(ctx, lin, x) or lin.bias is not None:
        return False
    if ctx.runtime.options.get("mid_silu_min_rows", MID_SILU_MIN_ROWS) <= n <= MID_MAX_ROWS:
        # blocks of 64 features (96 where that is what it takes, up to 128 rows) against all rows,
        # where one round of blocks holds them (or fewer features, so that the blocks fill the chip). Measured on the 1.5B shape:
        # 17 to 19 us against the library's product and the SiLU-gate kernel's 29 at 65 to 128 rows, 23 against 30 at 192, 25 at 256;
        # on the 7B shape 58 against 66 at 128, and at 256 rows, as on the 32B shape, two rounds of
        # blocks: those go to the kernel of tiles. With blocks of 32 and 64 rows of X for steps that
        # small it is ahead of the weight-streaming kernel at every size: on the 7B shape 3.20
        # against 3.23 ms a step at one request, 3.44 against 3.49 at 8, 3.77 against 3.87 at 16,
        # 4.46 against 4.56 at 32, 5.87 against 6.13 at 64; on the 1.5B shape by 1 to 4 %.
        mid = ctx.runtime.options.get("mid_gemm", True)
        fits = mid and ops.gemm_mid_supports(n, lin.out_features, lin.in_features, x.stride(0), lin.weight.stride(0))
        if fits and (ops.gemm_mid_silu_blocks(n, lin.out_features) <= ctx.runtime.compute_units or int(mid) == 2):
            ops.gemm_mid_silu_bf16(x, lin.weight, act, n, unit)
            return True
    if takes_tiles(ctx.runtime, lin, n, x):
        ops.gemm_tile_glu_bf16(x, lin.weight, act, n, unit)
        return True
    if n > FUSED_SILU_MAX_ROWS or not ctx.runtime.options.get("skinny_gemm", True):
        return False
    if not ops.gemm_skinny_supports(n, lin.out_features, lin.in_features, x.stride(0), lin.weight.stride(0)):
        return False
    ops.gemm_skinny_silu_bf16(x, lin.weight, act, n, unit)
    return True


#: rows of the prompt-portion kernel's work list that one launch takes (the grid's second dimension)
PREFILL_MAX_LAUNCH = 65535


def rope_in_attention(mixer, ctx, qkv, cache, rotary_dim: int) -> bool:
    """Whether the step's attention kernel can finish the q/k/v product itself (sum of the partial
    sums, bias, rotation, the cache write): a step of single tokens only, on the 16-bit path's decode
    kernel, full-head rotation, heads of up to 128 elements. The kernel between product and attention
    is then left out; the bits are the same. A function of the step's shape and the model's sizes."""
    s = mixer.spec
    hb = ctx.host
    if ctx.dtype != torch.bfloat16 or cache["k"].dtype != torch.bfloat16 or qkv.data.dtype != torch.float32:
        return False
    if not ctx.runtime.options.get("mfma_attention", True) or not ctx.runtime.options.get("rope_in_attention", True):
        return False
    if rotary_dim != s.head_dim or len(hb.arrays["attention.prefill_tiles"]) or \
            len(hb.arrays["attention.decode_tokens"]) != ctx.n_tokens:
        return False
    return ops.attn_decode_work_rope_supports(s.head_dim, cache.page_size, s.num_heads, s.num_kv_heads, qkv.stride)


def attention(mixer, ctx, q, o, cache, rope=None) -> bool:
    """``rope``: (the q/k/v product's partial sums, cos, sin) when :func:`rope_in_attention` said that
    the decode kernel finishes the product; ``q`` is then not read."""
    s = mixer.spec
    k_pages, v_pages = cache["k"], cache["v"]
    if ctx.dtype != torch.bfloat16 or k_pages.dtype != torch.bfloat16:
        return False
    if not ctx.runtime.options.get("mfma_attention", True):
        return False
    if not ops.attn_mfma_supports(s.head_dim, cache.page_size, s.num_heads, s.num_kv_heads):
        return False
    hb = ctx.host
    dec, tiles = hb.arrays["attention.decode_tokens"], hb.arrays["attention.prefill_tiles"]
    n_dec, n_tiles = len(dec), len(tiles)
    if n_dec:
        # The launch's size follows from the step's rounded sizes and the list from the rounded
        # number of requests, so that a step gives bit for bit the same result whether it runs
        # eagerly or as a replayed graph at those sizes.
        rows, _ = hb.decode_shape()
        units = mixer.units
        capacity = plan.decode_capacity(rows, s.num_heads, s.num_kv_heads, units)
        listed_blocks = int(hb.arrays[mixer.decode_work_name].reshape(-1)[0])
        if listed_blocks > capacity:  # the kernel would leave the rest of the list undone, silently
            raise RuntimeError(f"the decode attention's work list has {listed_blocks} blocks, its launch {capacity}")
        items = plan.decode_items(s.num_heads, s.num_kv_heads)
        acc = ctx.workspace.get("attn.part_acc", (capacity, items, 16, s.head_dim), torch.float32)
        ml = ctx.workspace.get("attn.part_ml", (capacity, items, 16, 2), torch.float32)
        counters = ctx.workspace.get("attn.counters", (capacity, items), torch.int32, zeroed=True)
        alone = plan.decode_alone(rows, s.num_heads, s.num_kv_heads, units)
        if rope is not None:
            qkv, cos, sin = rope
            ops.attn_decode_work_rope_bf16(qkv, cos, sin, cache.slots, o, k_pages, v_pages, cache.writes,
                                           ctx.arrays[mixer.decode_work_name], capacity, ctx.positions,
                                           ctx.seq_of_token, cache.table, acc, ml, counters, alone, s.num_heads,
                                           s.num_kv_heads, s.head_dim, cache.page_size, mixer.scale, cache.window)
        else:
            ops.attn_decode_work_bf16(q, o, k_pages, v_pages, ctx.arrays[mixer.decode_work_name], capacity,
                                      ctx.positions, ctx.seq_of_token, cache.table, acc, ml, counters, alone,
                                      s.num_heads, s.num_kv_heads, s.head_dim, cache.page_size, mixer.scale,
                                      cache.window)
    if n_tiles and s.head_dim <= 128:
        work = hb.arrays[mixer.prefill_work_name]
        n_slots = plan.prefill_slots(work)
        if 8 * len(work) > ctx.arrays[mixer.prefill_work_name].numel():
            raise RuntimeError(f"the prompt attention's work list has {len(work)} blocks, its step array holds "
                               f"{ctx.arrays[mixer.prefill_work_name].numel() // 8}")
        per_slot = plan.prefill_items(s.num_heads, s.num_kv_heads) * ops.attn_prefill_waves(s.num_heads, s.num_kv_heads)
        partials = counters = None
        if n_slots:
            partials = ctx.workspace.get("attn.prefill_partials", (n_slots, per_slot, s.head_dim // 32 * 1024 + 128),
                                         torch.float32)
            counters = ctx.workspace.get("attn.prefill_counters", (n_slots, per_slot), torch.int32, zeroed=True)
        listed = ctx.arrays[mixer.prefill_work_name]
        for at in range(0, len(work), PREFILL_MAX_LAUNCH):  # a launch takes 65,535 rows of the list
            count = min(PREFILL_MAX_LAUNCH, len(work) - at)
            ops.attn_prefill_work_bf16(q, o, k_pages, v_pages, listed[8 * at:], count, partials, counters, n_slots,
                                       ctx.positions, ctx.seq_of_token, cache.table, s.num_heads, s.num_kv_heads,
                                       s.head_dim, cache.page_size, mixer.scale, cache.window)
    elif n_tiles:
        ops.attn_prefill_bf16(q, o, k_pages, v_pages, ctx.arrays["attention.prefill_tiles"], n_tiles, ctx.positions,
                              ctx.seq_of_token, cache.table, s.num_heads, s.num_kv_heads, s.head_dim,
                              cache.page_size, mixer.scale, cache.window)
    return True
