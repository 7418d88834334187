"""The measured cases: what a user of the compiler has it run, from one short
sentence through one layer to a batch of long ones.

Every case is a plain PyTorch module compiled with ``mlc.compile`` and called.
A case names

* ``kind``: which module (a whole BERT-base encoder; one encoder or decoder
  layer; an MLP block; the vocabulary head; the embedding sum and its norm; a
  softmax over the vocabulary),
* its sizes (``batch``, ``seq``, ``width``, ``heads``, ``ffn``, ``vocab``), the
  configurations this repository measures and tests (BERT-base and GPT-2
  small: width 768, 12 heads, FFN 3072; the small suite models: width 512, 8
  heads, FFN 2048),
* ``dtype`` of weights and activations, and
* ``variants``: ``"none"`` is ``Config()``, the reference's schedule; ``"all"``
  turns the four opt-in schedule changes on.
"""

from __future__ import annotations

import math
import pathlib
import sys

import torch
import torch.nn as nn
import torch.nn.functional as F

_PACKAGE = str(pathlib.Path.cwd() / "mlc-compiler_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
SIZES = {768: (12, 3072), 512: (8, 2048)}
LAYERS = 12
#: what a masked score is offset by, as the models this repository measures do
#: it: in 16 bits it becomes -inf
MASKED = torch.finfo(torch.float32).min


def _case(name, kind, batch, seq, width=768, vocab=0, dtype="fp16", variants="none"):
    heads, ffn = SIZES[width]
    return {"name": name, "kind": kind, "batch": batch, "seq": seq, "width": width,
            "heads": heads, "ffn": ffn, "vocab": vocab, "dtype": dtype, "variants": variants}


def listed():
    return [
        # a short sentence through one layer of a small model: launches and latency
        _case("encoder-small-b1-s16", "encoder", 1, 16, width=512, variants="all"),
        # one BERT-base layer for a single request, on the reference schedule
        _case("encoder-b1-s128", "encoder", 1, 128),
        # a batch padded to an odd length, bf16: no size is a multiple of a tile
        _case("encoder-b6-s197-bf16", "encoder", 6, 197, dtype="bf16"),
        # one BERT-base layer at the serving batch, every schedule variant on
        _case("encoder-b32-s128-all", "encoder", 32, 128, variants="all"),
        # one GPT-2 block over a single short prompt, every schedule variant on
        _case("decoder-b1-s128-all", "decoder", 1, 128, variants="all"),
        # one GPT-2 block over a batch of long prompts: the largest work
        _case("decoder-b32-s512-all", "decoder", 32, 512, variants="all"),
        # the same block in bf16 over a few full-context prompts, all variants
        _case("decoder-b2-s1024-bf16-all", "decoder", 2, 1024, dtype="bf16", variants="all"),
        # the FFN block in full precision for one request
        _case("mlp-b1-s128-fp32", "mlp", 1, 128, dtype="fp32"),
        # final norm and GPT-2's 50257-wide vocabulary head: scoring one prompt
        _case("head-b1-s128", "head", 1, 128, vocab=50257),
        # probabilities over that vocabulary for a batch of positions (long rows)
        _case("softmax-b4-s128", "softmax", 4, 128, vocab=50257),
        # three embedding gathers, their sum and its norm for a serving batch
        _case("embed-b32-s128", "embed", 32, 128, vocab=30522),
        # the whole of BERT-base for a single request: the headline call
        _case("bert-b1-s128", "bert", 1, 128, vocab=30522),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c) -> float:
    """Seconds, roughly, at rates every path reaches: only to bound a draw."""
    w = work(c)
    size = DTYPES[c["dtype"]].itemsize
    scores = 6 * size * c["batch"] * c["heads"] * c["seq"] ** 2
    acts = 12 * size * c["batch"] * c["seq"] * (c["width"] + c["ffn"])
    layers = {"bert": LAYERS, "encoder": 1, "decoder": 1}.get(c["kind"], 0)
    rate = 6e13 if c["dtype"] == "fp32" else 4e14
    return w["flops"] / rate + (w["bytes"] + layers * (scores + acts)) / 3e12


def draw(rng):
    limit = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("encoder", "encoder", "decoder", "decoder", "mlp", "head",
                           "softmax", "embed"))
        width = rng.choice((768, 768, 512))
        batch = _log_int(rng, 1, 32)
        seq = _log_int(rng, 16, 1024 if kind in ("decoder", "head", "softmax") else 512)
        if rng.random() < 0.5:  # the lengths a padded batch usually has
            seq = max(16, seq // 32 * 32)
        vocab = {"head": rng.choice((8192, 50257)), "softmax": rng.choice((8192, 30522, 50257)),
                 "embed": rng.choice((8192, 30522))}.get(kind, 0)
        dtype = rng.choice(("fp16", "fp16", "bf16", "fp32"))
        variants = rng.choice(("none", "all"))
        if dtype == "bf16":  # one sequence alone: its attention products read strided views,
            batch = max(2, batch)  # which torch's bf16 batched product does not take safely
        c = _case("", kind, batch, seq, width, vocab, dtype, variants)
        del c["name"]
        if _cost(c) <= limit:
            return c


# ---------------------------------------------------------------------------
# the modules
# ---------------------------------------------------------------------------

class Attention(nn.Module):
    def __init__(self, width, heads, fused):
        super().__init__()
        self.heads, self.fused = heads, fused
        if fused:
            self.qkv = nn.Linear(width, 3 * width)
        else:
            self.q, self.k, self.v = (nn.Linear(width, width) for _ in range(3))
        self.proj = nn.Linear(width, width)

    def forward(self, x, mask):
        b, n, w = x.shape
        if self.fused:
            q, k, v = self.qkv(x).chunk(3, dim=-1)
        else:
            q, k, v = self.q(x), self.k(x), self.v(x)
        q, k, v = (t.view(b, n, self.heads, w // self.heads).transpose(1, 2) for t in (q, k, v))
        scores = q @ k.transpose(-2, -1) / (w // self.heads) ** 0.5 + mask
        ctx = scores.softmax(dim=-1) @ v
        return self.proj(ctx.transpose(1, 2).reshape(b, n, w))


class Encoder(nn.Module):
    """Post-norm layer (BERT)."""

    def __init__(self, width, heads, ffn):
        super().__init__()
        self.attn = Attention(width, heads, fused=False)
        self.norm1 = nn.LayerNorm(width, eps=1e-12)
        self.up, self.down = nn.Linear(width, ffn), nn.Linear(ffn, width)
        self.norm2 = nn.LayerNorm(width, eps=1e-12)

    def forward(self, x, mask):
        x = self.norm1(x + self.attn(x, mask))
        return self.norm2(x + self.down(F.gelu(self.up(x))))


class Decoder(nn.Module):
    """Pre-norm block (GPT-2)."""

    def __init__(self, width, heads, ffn):
        super().__init__()
        self.norm1 = nn.LayerNorm(width, eps=1e-5)
        self.attn = Attention(width, heads, fused=True)
        self.norm2 = nn.LayerNorm(width, eps=1e-5)
        self.up, self.down = nn.Linear(width, ffn), nn.Linear(ffn, width)

    def forward(self, x, mask):
        x = x + self.attn(self.norm1(x), mask)
        return x + self.down(F.gelu(self.up(self.norm2(x))))


class Mlp(nn.Module):
    def __init__(self, width, ffn):
        super().__init__()
        self.norm = nn.LayerNorm(width, eps=1e-12)
        self.up, self.down = nn.Linear(width, ffn), nn.Linear(ffn, width)

    def forward(self, x, r):
        return self.down(F.gelu(self.up(self.norm(x + r)), approximate="tanh"))


class Head(nn.Module):
    def __init__(self, width, vocab):
        super().__init__()
        self.norm = nn.LayerNorm(width, eps=1e-5)
        self.out = nn.Linear(width, vocab, bias=False)

    def forward(self, x):
        return self.out(self.norm(x))


class Probabilities(nn.Module):
    """Softmax over the vocabulary at a temperature."""

    def forward(self, logits):
        return torch.softmax(logits / 0.8, dim=-1)


class Embed(nn.Module):
    def __init__(self, vocab, width):
        super().__init__()
        self.tokens = nn.Embedding(vocab, width)
        self.places = nn.Embedding(512, width)
        self.segments = nn.Embedding(2, width)
        self.norm = nn.LayerNorm(width, eps=1e-12)
        self.register_buffer("place_ids", torch.arange(512), persistent=False)

    def forward(self, ids, segment_ids):
        places = self.places(self.place_ids[:ids.shape[1]])
        return self.norm(self.tokens(ids) + places + self.segments(segment_ids))


class Bert(nn.Module):
    def __init__(self, vocab, width, heads, ffn):
        super().__init__()
        self.embed = Embed(vocab, width)
        self.layers = nn.ModuleList(Encoder(width, heads, ffn) for _ in range(LAYERS))
        self.pool = nn.Linear(width, width)

    def forward(self, ids, segment_ids, attention_mask):
        mask = (1.0 - attention_mask[:, None, None, :]) * MASKED
        x = self.embed(ids, segment_ids)
        for layer in self.layers:
            x = layer(x, mask)
        return torch.tanh(self.pool(x[:, 0]))


def _module(c):
    w, h, f, v = c["width"], c["heads"], c["ffn"], c["vocab"]
    return {"encoder": lambda: Encoder(w, h, f), "decoder": lambda: Decoder(w, h, f),
            "mlp": lambda: Mlp(w, f), "head": lambda: Head(w, v), "softmax": Probabilities,
            "embed": lambda: Embed(v, w), "bert": lambda: Bert(v, w, h, f)}[c["kind"]]()


def _padding(c, gen, masked=None):
    """[B, T] ones with a padded tail of zeros on every row but the first, or
    as the offset of a masked score."""
    b, t = c["batch"], c["seq"]
    keep = torch.randint((t + 1) // 2, t + 1, (b,), generator=gen, device="cuda")
    keep[0] = t
    kept = torch.arange(t, device="cuda") < keep[:, None]
    if masked is not None:
        return torch.zeros(b, t, device="cuda").masked_fill(~kept, masked).to(DTYPES[c["dtype"]])
    return kept.to(DTYPES[c["dtype"]])


def _build(c, seed):
    """(module, inputs) on the GPU, made from the seed alone."""
    gen = torch.Generator("cuda").manual_seed(seed)
    dtype = DTYPES[c["dtype"]]
    with torch.device("meta"):
        module = _module(c)
    module = module.to_empty(device="cuda").to(dtype).eval()
    with torch.no_grad():
        for m in module.modules():
            if isinstance(m, nn.LayerNorm):
                m.weight.normal_(1.0, 0.02, generator=gen)
                m.bias.normal_(0.0, 0.02, generator=gen)
            elif isinstance(m, (nn.Linear, nn.Embedding)):
                m.weight.normal_(0.0, 0.02, generator=gen)
                if getattr(m, "bias", None) is not None:
                    m.bias.normal_(0.0, 0.02, generator=gen)
            if isinstance(m, Embed):
                m.place_ids = torch.arange(512, device="cuda")
    b, t = c["batch"], c["seq"]

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=dtype)

    def whole(high):
        return torch.randint(0, high, (b, t), generator=gen, device="cuda")

    kind = c["kind"]
    if kind == "encoder":  # an additive padding mask
        inputs = (normal(b, t, c["width"]), _padding(c, gen, MASKED)[:, None, None, :])
    elif kind == "decoder":  # an additive causal mask
        future = torch.ones(t, t, device="cuda").triu(1) > 0
        mask = torch.zeros(t, t, device="cuda").masked_fill(future, MASKED).to(dtype)[None, None]
        inputs = (normal(b, t, c["width"]), mask)
    elif kind == "mlp":
        inputs = (normal(b, t, c["width"]), normal(b, t, c["width"]))
    elif kind == "head":
        inputs = (normal(b, t, c["width"]),)
    elif kind == "softmax":
        inputs = (normal(b, t, c["vocab"]) * 3,)
    elif kind == "embed":
        inputs = (whole(c["vocab"]), whole(2))
    else:
        inputs = (whole(c["vocab"]), whole(2), _padding(c, gen))
    return module, inputs


def prepare(case, seed):
    import mlc
    from mlc.config import Config

    module, inputs = _build(case, seed)
    on = case["variants"] == "all"
    cfg = Config(merge_parallel_gemms=on, gemm_epilogue=on, layout_selection=on,
                 fused_attention=on)
    with torch.no_grad():
        return {"compiled": mlc.compile(module, inputs, cfg), "inputs": inputs}


def run(state):
    return state["compiled"](*state["inputs"])


def work(case):
    b, t, w, f, v = (case[k] for k in ("batch", "seq", "width", "ffn", "vocab"))
    size = DTYPES[case["dtype"]].itemsize
    n = b * t
    kind = case["kind"]
    layer_weights = 4 * w * w + 2 * w * f
    layer_flops = 2 * n * layer_weights + 4 * n * t * w
    io = 2 * n * w
    if kind == "encoder":
        return {"bytes": size * (io + layer_weights + b * t), "flops": layer_flops}
    if kind == "decoder":
        return {"bytes": size * (io + layer_weights + t * t), "flops": layer_flops}
    if kind == "mlp":
        return {"bytes": size * (3 * n * w + 2 * w * f), "flops": 4 * n * w * f}
    if kind == "head":
        return {"bytes": size * (n * w + w * v + n * v), "flops": 2 * n * w * v}
    if kind == "softmax":
        return {"bytes": size * 2 * n * v, "flops": 5 * n * v}
    if kind == "embed":  # ids, the rows gathered from each table, the result
        return {"bytes": 16 * n + size * w * (min(n, v) + t + 2 + n), "flops": 10 * n * w}
    return {"bytes": 16 * n + size * (n + w * (min(n, v) + t + 2) + LAYERS * layer_weights
                                      + w * w + b * w),
            "flops": LAYERS * layer_flops + 2 * b * w * w}


#: about four times the distance from float64 measured on one MI355X: single
#: layers 2.1e-4 to 4.9e-4 (fp16), 1.6e-3 to 2.6e-3 (bf16), 2e-7 to 1.2e-6
#: (fp32); the twelve layers of the whole encoder 1.2e-3 (fp16)
TOLERANCE = {"fp16": 2e-3, "bf16": 1e-2, "fp32": 1e-5}


def tolerance(case):
    return {"rel": 5e-3 if case["kind"] == "bert" else TOLERANCE[case["dtype"]]}


def exact(case, seed):
    """The same module in float64 over the same values."""
    module, inputs = _build(case, seed)
    with torch.no_grad():
        module = module.double()
        return module(*(x.double() if x.is_floating_point() else x for x in inputs))
