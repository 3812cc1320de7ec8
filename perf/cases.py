"""What a user of this framework has it do, as cases to be measured: steps of a serving engine.

A case is one kind of step on one model:

* ``decode``: every running request gets one more token (one call of ``Engine.step``). The requests
  grow by a token a pass, as they do in a server.
* ``prompt``: prompts from their first token to the logits of their last one (or of every one, as for
  scoring a text), in steps of at most ``portion`` tokens, then freed.
* ``mixed``: a step of continuous batching, with portions of some prompts beside one token of every
  running request.

``context`` is the length of a request (before the pass for ``decode``), ``ragged`` spreads the lengths
from a sixteenth of it up to it. Models are the repository's own: the Qwen2.5 shapes, and three further
designs at the same layer sizes with four layers (those whose feed-forwards are dense: the result of a
mixture jumps where two experts nearly tie, which no tolerance describes). The Qwen2.5 shapes run with 14
and 8 of their 28 layers: sixteen-bit rounding grows with the depth, and the values are to be compared.
Weights are random, N(0, 0.02), token ids uniform. Next tokens are given and not chosen, since the greedy
choice among nearly equal logits of a random model is a matter of rounding.
"""

import math
import random

import torch

from pyre_amd.config import EngineConfig, preset
from pyre_amd.engine.batch import Entry
from pyre_amd.engine.engine import Engine
from pyre_amd.registry import config_from_dict
from pyre_amd.weights import model_tensor_specs

DEVICE = "cuda:0"
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
F64 = torch.float64
WARM = 2        # passes that prepare() makes: a server has run this kind of step before
FILL = 2048     # tokens a step while caches are filled
ROOM = 4096     # tokens that a request of a decode case may grow by (fewer where many run)
FEEDS = 64      # different next tokens of a request

SIZES = {
    "1.5b": dict(width=1536, ff=8960, heads=12, kv_heads=2, head=128, vocab=151936),
    "7b": dict(width=3584, ff=18944, heads=28, kv_heads=4, head=128, vocab=152064),
}
LAYERS = {"qwen2.5-1.5b": 14, "qwen2.5-7b": 8}
DESIGNS = ("mafurax", "rukosun", "pinozen")


def case(name, kind, model, requests, context, **more):
    c = {"kind": kind, "model": model, "dtype": "bfloat16", "requests": requests, "context": context, "ragged": False,
         "portion": 2048, "prompts": 0, "all_logits": False}
    c.update(more)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one user talking to a small model: launches and latency
        case("qwen_1p5b_decode_1", "decode", "qwen2.5-1.5b", 1, 301),
        # the headline: eight requests with 4,096 tokens behind them
        case("qwen_7b_decode_8", "decode", "qwen2.5-7b", 8, 4096),
        # a full server: many requests of all lengths
        case("qwen_1p5b_decode_190_ragged", "decode", "qwen2.5-1.5b", 190, 1501, ragged=True),
        # a question of ordinary length: the time to its first token
        case("qwen_1p5b_prompt_99", "prompt", "qwen2.5-1.5b", 1, 99),
        # a long question or a page of text
        case("qwen_7b_prompt_2048", "prompt", "qwen2.5-7b", 1, 2048),
        # a document, in portions
        case("qwen_7b_prompt_12001", "prompt", "qwen2.5-7b", 1, 12001),
        # continuous batching: portions of four prompts beside 61 running requests
        case("qwen_1p5b_mixed_61", "mixed", "qwen2.5-1.5b", 61, 1100, ragged=True, prompts=4, portion=512),
        # scoring: the logits of every token of a few texts, in the true 32-bit mode
        case("qwen_1p5b_score_3_float32", "prompt", "qwen2.5-1.5b", 3, 333, ragged=True, all_logits=True, dtype="float32"),
        # decoding in the true 32-bit mode
        case("qwen_1p5b_decode_20_float32", "decode", "qwen2.5-1.5b", 20, 777, dtype="float32"),
        # the other designs: attention with biases beside gated linear attention, a prompt
        case("mafurax_7b_prompt_1777", "prompt", "mafurax-7b", 1, 1777),
        # latent attention and two residual streams, a prompt
        case("rukosun_1p5b_prompt_3000", "prompt", "rukosun-1.5b", 1, 3000),
        # attention over everything before beside a selective scan, a batch of running requests
        case("pinozen_7b_decode_30", "decode", "pinozen-7b", 30, 2050, ragged=True),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice(["qwen2.5-1.5b", "qwen2.5-1.5b", "qwen2.5-7b"] * 2 + [f"{d}-{s}" for d in DESIGNS for s in ("1.5b", "7b")])
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed"])
    dtype = "float32" if rng.random() < 0.15 else "bfloat16"
    large = model.endswith("7b")
    if kind == "decode":
        most = 32768 if dtype == "bfloat16" else 8192  # tokens in the caches
        requests = spread(1, 256)
        return case(None, kind, model, requests, spread(min(64, most // requests // 2), most // requests), ragged=rng.random() < 0.5, dtype=dtype)
    if kind == "mixed":
        return case(None, kind, model, spread(4, 120), spread(100, 1500), ragged=True, prompts=rng.randint(1, 4),
                    portion=rng.choice([200, 333, 512]) if dtype == "bfloat16" else 150, dtype=dtype)
    if rng.random() < 0.25:
        return case(None, kind, model, spread(1, 8), spread(16, 300), ragged=True, all_logits=True, dtype=dtype)
    most = (8000 if large else 12000) if dtype == "bfloat16" else 600
    return case(None, kind, model, 1, spread(16, most), portion=rng.choice([512, 1000, 2048]), dtype=dtype)


# ---------------------------------------------------------------------- what a case consists of


def lengths(c):
    n, most = c["requests"], c["context"]
    return [max(1, round(most * 16.0 ** -((i * 0.6180339887) % 1.0))) if c["ragged"] else most for i in range(n)]


def prompt_length(c):
    """Tokens of a prompt that rides beside running requests: four portions, the last not quite full."""
    return 4 * c["portion"] - c["portion"] // 4 - 3


def config_dict(model):
    """The configuration of a design at the layer sizes of a Qwen2.5 shape, as its ``config.json`` has it."""
    design, size = model.rsplit("-", 1)
    s, layers = SIZES[size], 4
    half, half_kv = s["heads"] // 2, max(1, s["kv_heads"] // 2)
    dense = {"kind": "dense", "ff": s["ff"]}
    common = {"vocab": s["vocab"], "width": s["width"], "norm": {"eps": 1e-6}}
    if design == "mafurax":
        left = {"heads": half, "kv_heads": half_kv, "dim": s["head"], "vdim": s["head"], "scale": s["head"] ** -0.5, "softcap": 50.0,
                "bias_max": 1024, "bias_rows": 32, "mask": {"size": 1024, "keep_first": 4}}
        right = {"heads": half, "dim": s["head"], "vdim": s["head"], "tau": 8.0, "rank": 32}
        layer = {"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 1.0, "right_scale": 1.0},
                 "mlp": dict(dense, limit=7.0)}
        return dict(common, architecture="Mafurax", layers=[layer] * layers, logit_scale=1.0)
    if design == "rukosun":
        row = {"heads": s["heads"], "dim": s["head"], "rot_dim": s["head"] // 2, "vdim": s["head"], "kv_rank": 4 * s["head"],
               "scale": (1.5 * s["head"]) ** -0.5, "mask": {"size": 1024}, "rot": {"base": 1e4, "dims": s["head"] // 2}}
        return dict(common, architecture="Rukosun", streams=2, max_positions=32768,
                    embedding={"bigram": {"buckets": 65521, "mul_prev": 1000003, "mul_cur": 31}},
                    layers=[{"type": "latent_attention" if i % 2 else "latent_attention_2", "mlp": dense,
                             "mixer": dict(row, q_rank=3 * s["width"] // 8) if i % 2 else row} for i in range(layers)])
    left = {"heads": half, "kv_heads": half_kv, "dim": s["head"], "vdim": s["head"], "scale": s["head"] ** -0.5, "softcap": 50.0, "conv": 4,
            "rot": {"base": 2.5e5, "dims": s["head"] // 2, "scaling": {"factor": 4.0, "low": 1.0, "high": 4.0, "original": 1024}}}
    right = {"inner": s["width"], "state": 16, "dt_rank": s["width"] // 16, "conv": 4}
    light = {"heads": s["heads"], "dim": s["head"], "vdim": s["head"],
             "decay": [0.9 + 0.0999 * i / (s["heads"] - 1) for i in range(s["heads"])]}
    return dict(common, architecture="Pinozen", embedding={"scale": 1.0}, logit_scale=1.0, max_positions=32768,
                layers=[{"type": "lightning", "mixer": light, "mlp": dense} if i % 4 == 2 else
                        {"type": "parallel", "mixer": {"left": left, "right": right}, "mlp": dense} for i in range(layers)],
                loop={"start": 1, "stop": layers, "times": 1})


def config_of(c):
    if c["model"] in LAYERS:
        return preset(c["model"], num_hidden_layers=LAYERS[c["model"]])
    return config_from_dict(config_dict(c["model"]))


def vocabulary(c):
    return SIZES["7b" if c["model"].endswith("7b") else "1.5b"]["vocab"]


def weights_of(c, seed):
    """Random tensors under the model's names, drawn on the device."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    out = {}
    for spec in model_tensor_specs(config_of(c)):
        if spec.alias_of is not None or spec.optional:
            continue
        shape = spec.random_shape if spec.random_shape is not None else spec.shape
        if spec.init == "gain":
            t = torch.randn(shape, generator=gen, device=DEVICE).mul_(0.1).add_(1.0)
        elif spec.init == "zeros":
            t = torch.randn(shape, generator=gen, device=DEVICE).mul_(0.02)
        else:
            t = torch.randn(shape, generator=gen, device=DEVICE).mul_(float(spec.init.split(":")[1]) if ":" in spec.init else 0.02)
        out[spec.name] = t.to(DTYPES[c["dtype"]])
    return out


class Tokens:
    """The token ids of a case: of every request before the measured passes, of the passes, of the prompts beside them."""

    def __init__(self, c, seed):
        rng, v = random.Random(seed), vocabulary(c)
        self.past = [[rng.randrange(v) for _ in range(n)] for n in lengths(c)]
        self.feeds = [[rng.randrange(v) for _ in range(FEEDS)] for _ in range(c["requests"])]
        self.prompts = [[rng.randrange(v) for _ in range(prompt_length(c))] for _ in range(c["prompts"])]


class Serving:
    """An engine in the middle of its work, and what its caller keeps of the requests."""

    def __init__(self, c, seed):
        self.case, self.tokens, self.passes = c, Tokens(c, seed), 0
        longest, n = max(lengths(c)), c["requests"]
        self.room = (ROOM if n <= 64 else ROOM // 4) if c["kind"] != "prompt" else 0
        cached = sum(-(-(x + self.room) // 16) * 16 for x in lengths(c)) + c["prompts"] * (prompt_length(c) + 16)
        step = max(c["portion"], FILL) + n if c["kind"] != "mixed" else max(FILL, c["prompts"] * c["portion"]) + n
        ec = EngineConfig(dtype=c["dtype"], device=DEVICE, page_size=16, max_num_seqs=n + c["prompts"], max_cached_tokens=cached + 1024,
                          max_model_len=max(longest + self.room, prompt_length(c)) + 16, max_num_batched_tokens=step,
                          prefill_chunk=c["portion"])
        self.engine = Engine.from_state(config_of(c), weights_of(c, seed), ec, consume=True)
        if c["kind"] != "prompt":
            self.fill()
        if c["kind"] == "mixed":  # every prompt one portion further than the one before
            for j, p in enumerate(self.tokens.prompts):
                for k in range(j % 4):
                    self.engine.step([Entry(("prompt", j), p[k * c["portion"]:(k + 1) * c["portion"]], [])])

    def fill(self):
        self.grown = 0
        self.feed_prompts(self.tokens.past, FILL, [[] for _ in self.tokens.past])

    def feed_prompts(self, prompts, portion, want):
        """Prompts one after the other, in steps of at most ``portion`` tokens; the logits asked for."""
        out, entries, used = [], [], 0
        for i, p in enumerate(prompts):
            at = 0
            while at < len(p):
                n = min(len(p) - at, portion - used)
                entries.append(Entry(i, p[at:at + n], [w - at for w in want[i] if at <= w < at + n]))
                at, used = at + n, used + n
                if used == portion or (i + 1 == len(prompts) and at == len(p)):
                    logits = self.engine.step(entries)
                    if logits is not None:
                        out.append(logits)
                    entries, used = [], 0
        return out

    def singles(self):
        """One more token of every running request."""
        if self.grown == self.room:  # as long as they may become: others take their places
            for i in range(self.case["requests"]):
                self.engine.finish(i)
            self.fill()
        self.grown += 1
        return [Entry(i, [f[self.passes % FEEDS]], [0]) for i, f in enumerate(self.tokens.feeds)]

    def prompt(self):
        past = self.tokens.past
        out = self.feed_prompts(past, self.case["portion"], [range(len(p)) if self.case["all_logits"] else [len(p) - 1] for p in past])
        for i in range(len(past)):
            self.engine.finish(i)
        return out

    def decode(self):
        return self.engine.step(self.singles())

    def mixed(self):
        entries, size, done = self.singles(), self.case["portion"], []
        for j, p in enumerate(self.tokens.prompts):
            k = (self.passes + j) % 4
            part = p[k * size:(k + 1) * size]
            entries.append(Entry(("prompt", j), part, [len(part) - 1] if k == 3 else []))
            if k == 3:
                done.append(("prompt", j))
        out = self.engine.step(entries)
        for rid in done:
            self.engine.finish(rid)
        return out


def prepare(c, seed):
    state = Serving(c, seed)
    for _ in range(WARM):
        run(state)
    return state


def run(state):
    out = getattr(state, state.case["kind"])()
    state.passes += 1
    return out


# ---------------------------------------------------------------------- what a pass cannot do without


def work(c):
    cfg_tensors = [s for s in model_tensor_specs(config_of(c)) if not s.optional and s.alias_of is None]
    size = 2 if c["dtype"] == "bfloat16" else 4
    table = ("embed", "model.embed_tokens.weight", "bigram", "pos", "head", "lm_head.weight")
    layers = sum(math.prod(s.random_shape or s.shape) for s in cfg_tensors if s.name not in table)
    sz = SIZES["7b" if c["model"].endswith("7b") else "1.5b"]
    design = c["model"].rsplit("-", 1)[0]
    head = sz["vocab"] * sz["width"]
    hd, n_layers = sz["head"], LAYERS.get(c["model"], 4)
    # a token's kept elements, and multiply-adds for a key that it sees, over all layers
    kept, per_key, window = {"qwen2.5": (2 * sz["kv_heads"] * hd * n_layers, 2 * sz["heads"] * hd * n_layers, 0),
                             "mafurax": (2 * max(1, sz["kv_heads"] // 2) * hd * 4, 2 * (sz["heads"] // 2) * hd * 4, 1024),
                             "rukosun": (4.5 * hd * 4, 2.5 * sz["heads"] * hd * 4, 1024),
                             "pinozen": (2 * max(1, sz["kv_heads"] // 2) * hd * 3, 2 * (sz["heads"] // 2) * hd * 3, 0)}[design]
    # float32 numbers of a request's recurrent state, read and written once a step
    state = {"mafurax": (sz["heads"] // 2) * hd * hd * 4, "pinozen": sz["heads"] * hd * hd + 3 * sz["width"] * 16}.get(design, 0)

    def seen(start, n):  # keys that n tokens from position ``start`` on see, and keys that are read for them
        total = sum(min(p + 1, window) if window else p + 1 for p in range(start, start + n))
        return total, min(start + n, n + window) if window else start + n

    spans, steps, rows = [], 1, 0  # (start, tokens) of every request in a pass, steps, rows of logits
    if c["kind"] == "prompt":
        spans = [(0, n) for n in lengths(c)]
        steps = -(-sum(lengths(c)) // c["portion"])
        rows = sum(lengths(c)) if c["all_logits"] else c["requests"]
    else:
        spans = [(n, 1) for n in lengths(c)]
        rows = c["requests"]
        for j in range(c["prompts"]):
            spans.append((j % 4 * c["portion"], c["portion"]))
    tokens = sum(n for _, n in spans)
    keys = [seen(a, n) for a, n in spans]
    flops = 2.0 * tokens * layers + 2.0 * rows * head + 2.0 * per_key * sum(k for k, _ in keys) + 4.0 * state * tokens
    moved = size * (steps * layers + head + tokens * sz["width"] + kept * sum(k for _, k in keys) + kept * tokens)
    return {"bytes": moved + 4.0 * rows * sz["vocab"] + 8.0 * state * len(spans), "flops": flops}


def tolerance(c):
    """Measured between two ways of the same framework (a prompt whole, in two halves, or with its last token alone): 0.016 to
    0.018 (largest 0.08) with 14 layers of the 1.5B and 8 of the 7B shape, 0.004 to 0.009 with four layers of a design, in
    bfloat16; against 64 bits 0.017 to 0.022, and 5e-6 in float32."""
    return {"rel": 2e-5, "max": 2e-4} if c["dtype"] == "float32" else {"rel": 0.03, "max": 0.3}


# ---------------------------------------------------------------------- the same in 64 bits


def exact(c, seed):
    t = Tokens(c, seed)
    if c["kind"] == "prompt":
        seqs = t.past
        want = [list(range(len(s))) if c["all_logits"] else [len(s) - 1] for s in seqs]
    else:
        seqs = [s + f[:WARM + 1] for s, f in zip(t.past, t.feeds)]
        want = [[len(s) - 1] for s in seqs]
        for j, p in enumerate(t.prompts):
            if (WARM + j) % 4 == 3:
                seqs.append(p)
                want.append([len(p) - 1])
    rows = Plain(c, weights_of(c, seed), seqs).logits(want)
    if c["kind"] != "prompt":
        return rows
    # a prompt's logits come step by step, as the portions end
    out, used, at = [], 0, 0
    ends = [sum(len(s) for s in seqs[:i]) + w for i, s in enumerate(seqs) for w in want[i]]
    while used < sum(len(s) for s in seqs):
        used += c["portion"]
        n = sum(1 for e in ends[at:] if e < used)
        if n:
            out.append(rows[at:at + n])
        at += n
    return out


def rms(x, gain=None, eps=1e-6):
    x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return x if gain is None else x * gain


def centred(x, gain, bias=None, eps=1e-6):
    x = rms(x - x.mean(-1, keepdim=True), gain, eps)
    return x if bias is None else x + bias


def turn(x, angles, neighbours):
    """x [T, heads, d]: the first 2 * angles.shape[1] elements of every head turned, in neighbouring pairs or half against half."""
    n = angles.shape[1]
    cos, sin = angles.cos()[:, None], angles.sin()[:, None]
    u, v = (x[..., 0:2 * n:2], x[..., 1:2 * n:2]) if neighbours else (x[..., :n], x[..., n:2 * n])
    a, b = u * cos - v * sin, v * cos + u * sin
    turned = torch.stack([a, b], -1).flatten(-2) if neighbours else torch.cat([a, b], -1)
    return torch.cat([turned, x[..., 2 * n:]], -1)


def softmax_attention(q, k, v, scale, window=0, keep=0, cap=0.0, bias=None, sink=None):
    """q [T, H, d], k and v [T, G, ...]: causal, over the last ``window`` keys and the first ``keep``; scores capped, then a
    number by distance added (``bias`` [H, T]); ``sink`` [H] joins the denominator."""
    n, heads, groups = q.shape[0], q.shape[1], k.shape[1]
    k, v = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    out = []
    for a in range(0, n, 512):
        b = min(n, a + 512)
        s = torch.matmul(q[a:b].transpose(0, 1).reshape(groups, -1, q.shape[2]), k[:, :, :b]).view(heads, b - a, b) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        i, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(b, device=q.device)[None]
        if bias is not None:
            s = s + bias[:, (i - j).clamp_min(0)]
        hidden = j > i
        if window:
            hidden |= (i - j >= window) & (j >= keep)
        s = s.masked_fill(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[:, None, None].expand(heads, b - a, 1)], -1)
        p = torch.softmax(s, -1)[..., :b].reshape(groups, -1, b)
        out.append(torch.matmul(p, v[:, :b]).view(heads, b - a, -1).transpose(0, 1))
    return torch.cat(out)


class Plain:
    """Whole sequences in 64 bits, without a cache: the sequences' rows one behind the other."""

    def __init__(self, c, tensors, seqs):
        self.c, self.t = c, tensors
        self.design = c["model"].rsplit("-", 1)[0]
        self.sz = SIZES["7b" if c["model"].endswith("7b") else "1.5b"]
        self.cfg = None if self.design == "qwen2.5" else config_dict(c["model"])
        self.ids = torch.tensor([t for s in seqs for t in s], device=DEVICE)
        ends = [0]
        for s in seqs:
            ends.append(ends[-1] + len(s))
        self.spans = list(zip(ends, ends[1:]))
        self.pos = torch.cat([torch.arange(b - a, device=DEVICE) for a, b in self.spans])

    def w(self, name):
        return self.t[name].to(F64)

    def lin(self, x, name):
        return x @ self.w(name).T

    def each(self, f, *rows):
        """``f`` on every sequence's rows."""
        return torch.cat([f(*(r[a:b] for r in rows)) for a, b in self.spans])

    def padded(self, x):
        out = x.new_zeros(len(self.spans), max(b - a for a, b in self.spans), *x.shape[1:])
        for i, (a, b) in enumerate(self.spans):
            out[i, :b - a] = x[a:b]
        return out

    def flat(self, x):
        return torch.cat([x[i, :b - a] for i, (a, b) in enumerate(self.spans)])

    def recurrence(self, decay, k, v, q):
        """S <- decay S + k v^T, read by q, a matrix for every sequence and head: rows [N, H, d]."""
        decay, k, v, q = (self.padded(x) for x in (decay, k, v, q))
        state = k.new_zeros(k.shape[0], k.shape[2], k.shape[3], v.shape[3])
        out = torch.empty_like(v)
        for t in range(k.shape[1]):
            state.mul_(decay[:, t, :, :, None]).addcmul_(k[:, t, :, :, None], v[:, t, :, None, :])
            out[:, t] = torch.matmul(q[:, t, :, None, :], state)[:, :, 0]
        return self.flat(out)

    def feed_forward(self, h, f, names, down):
        """In runs of rows: the inner width is large."""
        ws, wd = [self.w(n) for n in names], self.w(down)
        return torch.cat([f(*(x @ w.T for w in ws)) @ wd.T for x in h.split(8192)])

    def conv(self, x, taps):
        def one(u):
            n = taps.shape[1]
            p = torch.cat([u.new_zeros(n - 1, u.shape[1]), u])
            return sum(taps[:, j] * p[j:j + u.shape[0]] for j in range(n))

        return self.each(one, x)

    def logits(self, want):
        x = getattr(self, {"qwen2.5": "qwen"}.get(self.design, self.design))()
        rows = torch.tensor([a + i for (a, _), w in zip(self.spans, want) for i in w], device=DEVICE)
        head = next(n for n in ("lm_head.weight", "head", "model.embed_tokens.weight", "embed") if n in self.t)
        return self.lin(self.last_norm(x[rows]), head)

    # the Qwen2.5 shapes

    def qwen(self):
        s = self.sz
        self.last_norm = lambda x: rms(x, self.w("model.norm.weight"))  # noqa: E731
        # the angles are float32 numbers by the architecture's definition
        angles = (self.pos.float()[:, None] * (1.0 / (1e6 ** (torch.arange(0, 128, 2, dtype=torch.float32) / 128))).to(DEVICE)).to(F64)
        x = self.t["model.embed_tokens.weight"][self.ids].to(F64)
        for i in range(LAYERS[self.c["model"]]):
            p = f"model.layers.{i}."
            h = rms(x, self.w(p + "input_layernorm.weight"))
            q, k, v = ((self.lin(h, f"{p}self_attn.{n}_proj.weight") + self.w(f"{p}self_attn.{n}_proj.bias")).view(len(h), -1, s["head"]) for n in "qkv")
            o = self.each(lambda q, k, v: softmax_attention(q, k, v, 128 ** -0.5), turn(q, angles, False), turn(k, angles, False), v)
            x = x + self.lin(o.flatten(1), p + "self_attn.o_proj.weight")
            h = rms(x, self.w(p + "post_attention_layernorm.weight"))
            x = x + self.feed_forward(h, lambda g, u: torch.nn.functional.silu(g) * u, [p + "mlp.gate_proj.weight", p + "mlp.up_proj.weight"],
                                      p + "mlp.down_proj.weight")
        return x

    # attention with biases by distance beside gated linear attention, norms around every sublayer

    def mafurax(self):
        self.last_norm = lambda x: centred(x, self.w("final.norm"))  # noqa: E731
        x = self.t["embed"][self.ids].to(F64)
        for i, layer in enumerate(self.cfg["layers"]):
            a, r, p = layer["mixer"]["left"], layer["mixer"]["right"], f"l{i}."
            h = centred(x, self.w(p + "norm1"))
            q, k, v = (self.lin(h, f"{p}mix.left.{n}").view(len(h), -1, a["dim"]) for n in "qkv")
            rel = self.w(p + "mix.left.rel")
            half, rows = rel.shape[0] // 2, rel.shape[0]
            row = [n if n < half else min(rows - 1, half + math.floor(math.log(n / half) / math.log(a["bias_max"] / half) * (rows - half)))
                   for n in range(int(self.pos.max()) + 1)]
            bias = rel[torch.tensor(row, device=DEVICE)].T.contiguous()
            o = self.each(lambda q, k, v: softmax_attention(q, k, v, a["scale"], 1024, 4, 50.0, bias), rms(q), rms(k), v)
            left = self.lin((o * torch.sigmoid(self.lin(h, p + "mix.left.g"))[:, :, None]).flatten(1), p + "mix.left.o")
            q, k, v = (self.lin(h, f"{p}mix.right.{n}").view(len(h), -1, r["dim"]) for n in "qkv")
            z = self.lin(self.lin(h, p + "mix.right.a1"), p + "mix.right.a2") + self.w(p + "mix.right.a2.b")
            decay = (torch.nn.functional.logsigmoid(z) / r["tau"]).exp().view(q.shape)
            o = rms(self.recurrence(decay, k, v, q * r["dim"] ** -0.5), self.w(p + "mix.right.norm"))
            right = self.lin(o.flatten(1) * torch.nn.functional.silu(self.lin(h, p + "mix.right.g")), p + "mix.right.o")
            x = x + centred(left + right, self.w(p + "norm1b")) * self.w(p + "ls1")
            lim = layer["mlp"]["limit"]
            y = self.feed_forward(centred(x, self.w(p + "norm2")), lambda g, u: g.clamp(max=lim) * torch.sigmoid(1.702 * g.clamp(max=lim)) * (u.clamp(-lim, lim) + 1),
                                  [p + "mlp.gate", p + "mlp.up"], p + "mlp.down")
            x = x + centred(y, self.w(p + "norm2b")) * self.w(p + "ls2")
        return x

    # latent attention of two kinds, two residual streams, a polynomial activation

    def rukosun(self):
        self.last_norm = lambda x: centred(x, self.w("final.norm"), self.w("final.norm.b"))  # noqa: E731
        b = self.cfg["embedding"]["bigram"]
        before = torch.cat([self.ids[:1], self.ids[:-1]])
        pair = torch.where(self.pos == 0, b["buckets"], (before * b["mul_prev"] + self.ids * b["mul_cur"]) % b["buckets"])
        row = self.t["embed"][self.ids].to(F64) + self.t["bigram"][pair].to(F64) + self.t["pos"][self.pos].to(F64)
        streams = row[None].repeat(2, 1, 1)

        def through(p, streams, f):
            y = f(torch.einsum("s,stw->tw", self.w(p + "in"), streams))
            return torch.einsum("sr,stw->rtw", self.w(p + "mix"), streams) + self.w(p + "out")[:, None, None] * y

        def poly(z, c):
            return c[0] * rms(z) + c[1] * rms(z ** 2) + c[2] * rms(z ** 3) + c[3]

        for i, layer in enumerate(self.cfg["layers"]):
            m, p, first = layer["mixer"], f"l{i}.", layer["type"] == "latent_attention"
            angles = self.pos.to(F64)[:, None] * m["rot"]["base"] ** (-torch.arange(0, m["rot_dim"], 2, device=DEVICE, dtype=F64) / m["rot_dim"])

            def mixer(u):
                h = centred(u, self.w(p + "norm1"), self.w(p + "norm1.b"))
                q = self.lin(rms(self.lin(h, p + "mix.dq"), self.w(p + "mix.dq.norm")), p + "mix.uq") if first else self.lin(h, p + "mix.q")
                q = q.view(len(h), m["heads"], -1)
                both = self.lin(h, p + "mix.dkv")
                kept = rms(both[:, :m["kv_rank"]], self.w(p + "mix.dkv.norm"))
                shared = turn(both[:, None, m["kv_rank"]:], angles, first).expand(-1, m["heads"], -1)
                k = torch.cat([self.lin(kept, p + "mix.uk").view(len(h), m["heads"], -1), shared], -1)
                v = self.lin(kept, p + "mix.uv").view(len(h), m["heads"], -1)
                q = torch.cat([q[..., :m["dim"]], turn(q[..., m["dim"]:], angles, first)], -1)
                sink = self.w(p + "mix.sink") if first else None
                o = self.each(lambda q, k, v: softmax_attention(q, k, v, m["scale"], 1024, sink=sink), q, k, v).flatten(1)
                return self.lin(o * torch.sigmoid(self.lin(h, p + "mix.g")) if first else o, p + "mix.o")

            streams = through(p + "hc1.", streams, mixer)
            streams = through(p + "hc2.", streams, lambda u: self.feed_forward(
                centred(u, self.w(p + "norm2"), self.w(p + "norm2.b")), lambda z: poly(z, self.w(p + "mlp.act")), [p + "mlp.up"], p + "mlp.down"))
        return streams.sum(0)

    # attention behind a short convolution beside a selective scan, lightning attention

    def pinozen(self):
        self.last_norm = lambda x: rms(x, self.w("final.norm"))  # noqa: E731
        x = start = self.t["embed"][self.ids].to(F64) + self.t["pos"][self.pos].to(F64)
        for i, layer in enumerate(self.cfg["layers"]):
            p = f"l{i}."
            if i == self.cfg["loop"]["start"]:
                x = self.lin(torch.cat([x, start], 1), "loop.in")
            h = rms(x, self.w(p + "norm1"))
            x = x + (self.lightning if layer["type"] == "lightning" else self.two_branches)(h, p + "mix.", layer["mixer"])
            x = x + self.feed_forward(rms(x, self.w(p + "norm2")), lambda g, u: torch.relu(g) * u, [p + "mlp.gate", p + "mlp.up"], p + "mlp.down")
        return x

    def lightning(self, h, p, m):
        q, k, v = (torch.nn.functional.silu(self.lin(h, p + n)).view(len(h), m["heads"], -1) for n in "qkv")
        decay = torch.tensor(m["decay"], dtype=F64, device=DEVICE)[None, :, None].expand(q.shape)
        o = rms(self.recurrence(decay, k, v, q).flatten(1), self.w(p + "norm"))
        return self.lin(o * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def two_branches(self, h, p, m):
        a, r = m["left"], m["right"]
        q, k, v = (self.conv(self.lin(h, f"{p}left.{n}"), self.w(f"{p}left.{n}.conv")).view(len(h), -1, a["dim"]) for n in "qkv")
        rot = a["rot"]["scaling"]
        freq = a["rot"]["base"] ** (-torch.arange(0, a["rot"]["dims"], 2, device=DEVICE, dtype=F64) / a["rot"]["dims"])
        mix = ((rot["original"] * freq / (2 * math.pi) - rot["low"]) / (rot["high"] - rot["low"])).clamp(0, 1)
        angles = self.pos.to(F64)[:, None] * ((1 - mix) * freq / rot["factor"] + mix * freq)
        sink = self.w(p + "left.sink")
        o = self.each(lambda q, k, v: softmax_attention(q, k, v, a["scale"], cap=a["softcap"], sink=sink), turn(q, angles, True), turn(k, angles, True), v)
        left = self.lin(o.flatten(1), p + "left.o")
        x, z = self.lin(h, p + "right.in").split(r["inner"], 1)
        x = torch.nn.functional.silu(self.conv(x, self.w(p + "right.conv")) + self.w(p + "right.conv.b"))
        low, b, c = self.lin(x, p + "right.x").split([r["dt_rank"], r["state"], r["state"]], 1)
        dt = torch.nn.functional.softplus(self.lin(low, p + "right.dt") + self.w(p + "right.dt.b"), threshold=1e9)
        pace = -self.w(p + "right.A_log").exp()
        dts, xs, bs, cs = (self.padded(u) for u in (dt, x, b, c))
        state, y = dts.new_zeros(dts.shape[0], r["inner"], r["state"]), torch.empty_like(xs)
        for t in range(dts.shape[1]):
            state.mul_((dts[:, t, :, None] * pace).exp_()).addcmul_((dts[:, t] * xs[:, t])[:, :, None], bs[:, t, None, :])
            y[:, t] = torch.matmul(state, cs[:, t, :, None])[:, :, 0]
        y = self.flat(y) + self.w(p + "right.D") * x
        right = self.lin(y * torch.nn.functional.silu(z), p + "right.o")
        return 0.5 * (rms(left, self.w(p + "left.out")) + rms(right, self.w(p + "right.out")))
