"""Products that absorb the pointwise kernels after them
(``Config.gemm_epilogue``): which groups form, that a tile's coordinates give
every operand the element its own index map names, and the results."""

import re

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

import mlc
from mlc.api import build_pipeline
from mlc.codegen.hip_gemm import emit_group
from mlc.config import Config
from mlc.ir.capture import capture
from mlc.kernels import ExternKernel
from mlc.passes.memory_planning import plan_memory
from mlc.runtime.native import STATIC_SLAB_BYTES
from oracle import compile_reference
from workload_cache import graph_of

ALL = Config(cuda_graphs=False, merge_parallel_gemms=True, gemm_epilogue=True,
             layout_selection=True, fused_attention=True)


class Mlp(nn.Module):
    def __init__(self, w=64, f=192):
        super().__init__()
        self.up, self.down = nn.Linear(w, f), nn.Linear(f, w)

    def forward(self, x):
        return x + self.down(F.gelu(self.up(x))) * 0.5


class Block(Mlp):
    """The residual is alive beside the product, as in a GPT-2 block."""

    def forward(self, x):
        h = torch.tanh(x)
        return h + self.down(F.gelu(self.up(F.layer_norm(h, h.shape[-1:]))))


class FanOut(nn.Module):
    """Two outputs as wide as the product, from an input four times that."""

    def __init__(self):
        super().__init__()
        self.up = nn.Linear(1024, 256, bias=False)

    def forward(self, x):
        y = self.up(torch.tanh(x))
        a, b = torch.relu(y), torch.sigmoid(y)
        return torch.cat([a.sum(-1), b.sum(-1)])


class Heads(nn.Module):
    """q, k and v re-laid out per head, V transposed by the attention."""

    def __init__(self, w=128, h=2):
        super().__init__()
        self.h, self.qkv = h, nn.Linear(w, 3 * w)

    def forward(self, x):
        b, n, w = x.shape
        q, k, v = (t.view(b, n, self.h, w // self.h).transpose(1, 2)
                   for t in self.qkv(x).chunk(3, -1))
        return ((q @ k.transpose(-2, -1)) / 8.0).softmax(-1) @ v


class RowScale(nn.Module):
    """An operand that moves with the row alone, and a sliced (pitched) one."""

    def __init__(self):
        super().__init__()
        self.w = nn.Parameter(torch.randn(128, 64) * 0.1)

    def forward(self, x, scale, wide):
        return torch.mm(x, self.w.t()) * scale + wide[:, 4:132]


class Transposed(nn.Module):
    """The product read column by column."""

    def __init__(self):
        super().__init__()
        self.w = nn.Parameter(torch.randn(96, 64) * 0.1)

    def forward(self, x):
        y = torch.mm(x, self.w.t())
        return (y.t() + 1.0).contiguous()


class TwiceRead(nn.Module):
    """A second reader that is not pointwise: no group."""

    def __init__(self):
        super().__init__()
        self.w = nn.Parameter(torch.randn(96, 64) * 0.1)

    def forward(self, x):
        y = torch.mm(x, self.w.t())
        return torch.relu(y) * 2.0, y.sum(-1)


class HeadSize(nn.Module):
    """A product re-laid out per head; ``act``: with a bias and ReLU on the way."""

    def __init__(self, heads, size, act):
        super().__init__()
        self.heads, self.size, self.act = heads, size, act
        self.lin = nn.Linear(64, heads * size, bias=act)

    def forward(self, x):
        y = self.lin(x)
        y = torch.relu(y) if self.act else y
        return y.view(*x.shape[:2], self.heads, self.size).transpose(1, 2).contiguous()


HEAD_SIZES = [(2, 6), (4, 2), (2, 10), (4, 7), (2, 8), (4, 16)]


def cases(dtype=torch.float16):
    def r(*s):
        return torch.randn(*s).to(dtype)

    torch.manual_seed(0)
    return [("mlp", Mlp(), (r(37, 64),), 2), ("mlp b2", Mlp(), (r(2, 16, 64),), 2),
            ("heads", Heads(), (r(2, 32, 128),), 1), ("row scale", RowScale(), (r(33, 64), r(33, 1), r(33, 140)), 1),
            ("transposed", Transposed(), (r(40, 64),), None), ("twice", TwiceRead(), (r(40, 64),), 0)]


def _schedule(model, args, cfg=ALL):
    return build_pipeline(capture(model.to(args[0].dtype), args), cfg)


@pytest.mark.parametrize("at", range(6))
def test_groups_and_their_addresses(at):
    name, model, args, groups = cases()[at]
    sched = _schedule(model, args)
    if groups is not None:
        assert len(sched.merged) == groups, sched
    for i, (end, parts) in sched.merged.items():
        y = sched.kernels[i].outputs[0]
        M, N = y.shape
        assert isinstance(sched.kernels[i], ExternKernel) and end == i + len(parts)
        for part in parts:
            k = part.kernel
            own = next(a for a, read in zip(k.inputs, part.reads) if read is None)
            for idx in range(k.numel):
                m, n = divmod(own.index.evaluate(idx=idx), N)
                assert part.lo <= n < part.hi
                place = sum(m // p % s * t for s, p, t in part.m_terms) + \
                    sum((n - part.lo) // p % s * t for s, p, t in part.n_terms)
                assert place == idx, name
                for a, read in zip(k.inputs, part.reads):
                    if read is not None:
                        assert a.index.evaluate(idx=idx) == \
                            read.base + read.row * m + read.col * (n - part.lo), name


@pytest.mark.parametrize("model,args", [(c[1], c[2]) for c in cases()[:4]]
                         + [(Block(), (torch.zeros(40, 64, dtype=torch.float16),))])
def test_a_group_takes_no_more_memory_than_its_kernels(model, args):
    """One launch never stores the product: it has no place in the arena."""
    sched = _schedule(model, args)
    products = [sched.kernels[i].outputs[0].buffer.name for i in sched.merged]
    assert products and not set(products) & set(sched.plan.offsets)
    merged = sched.arena_bytes
    sched.merged = {}
    assert merged <= plan_memory(sched.graph, sched, ALL).arena_bytes
    assert not _schedule(model, args, ALL.replace(memory_planning=False)).merged


@pytest.mark.parametrize("cfg,most", [(Config(gemm_epilogue=True), 0), (ALL, 0),
                                      (ALL.replace(fused_attention=False), 12)])
def test_a_launch_does_not_write_where_the_one_before_it_read(cfg, most):
    """BERT-base b32: within the memory that the kernels one by one need, what
    a launch read is left alone for one more launch. Without fused attention
    that memory has no such place for one buffer of a layer."""
    sched = build_pipeline(graph_of("C4"), cfg)
    offsets, ranges = sched.plan.offsets, sched.plan.live_ranges.values()
    end = {j: last for i, (last, _) in sched.merged.items() for j in range(i, last + 1)}

    def share(a, b):
        x, y = offsets[a.buffer.name], offsets[b.buffer.name]
        return x < y + b.size and y < x + a.size

    at_once = [(a.buffer.name, b.buffer.name) for a in ranges for b in ranges
               if a.end < b.start <= end.get(a.end + 1, a.end + 1) and share(a, b)]
    assert len(at_once) <= most, at_once
    arena, sched.merged = sched.arena_bytes, {}
    assert arena <= plan_memory(sched.graph, sched, cfg).arena_bytes


def test_the_static_arena_holds_what_it_held():
    """64 MiB hold the kernels one by one (60 MiB) and not the group (72)."""
    cfg = ALL.replace(static_arena=True, reduction_fusion=False)
    args = (torch.empty(24 * 1024, 1024, dtype=torch.float16, device="meta"),)
    with torch.device("meta"):
        model = FanOut()
    assert _schedule(model, args, cfg.replace(static_arena=False)).arena_bytes > STATIC_SLAB_BYTES
    sched = _schedule(model, args, cfg)
    assert not sched.merged and sched.arena_bytes <= STATIC_SLAB_BYTES


@pytest.mark.parametrize("at", range(5))
def test_a_group_whose_kernels_run_one_by_one(at):
    """A runner without one-launch groups, and the bindings that timing uses."""
    _, model, args, _ = cases(torch.float32)[at]
    got, want = (compile_reference(model.float(), args, c)
                 for c in (ALL, ALL.replace(gemm_epilogue=False)))
    assert torch.equal(got(*args), want(*args))
    assert len(got._plan) == len(got.schedule.kernels) and None not in got._plan


def _stored_at(text, part, i, m, n, along_m):
    """Where the emitted source stores the four elements it holds at (m, n):
    columns n to n + 3 of row m (rows m to m + 3 of column n)."""
    def at(expr, **names):
        return eval(re.sub(r"(\d)u\b", r"\1", expr).replace("/", "//"), {}, names)

    q = n - part.lo
    body = text.split("auto store_t =")[1] if along_m else text.split("auto store_t =")[0]
    start = re.search(rf"\* w = o{i} \+ (.*);\n", body)
    store = body[start.end() if start else 0:]
    if start and "store_pack<4>(w, o)" in store.split("    }\n")[0]:
        first = at(start[1], row=m, q=q)
        assert first % 4 == 0  # a pack is one aligned access
        return [first + j for j in range(4)]
    if start:
        step = int(re.search(r"st\(w \+ j \* (\d+), o\[j\]\)", store)[1])
        return [at(start[1], row=m, q=q) + j * step for j in range(4)]
    each = re.search(rf"mlc::st\(o{i} \+ (.*), o\[j\]\);", body)[1]
    return [at(each, row=m, q=q, j=j) for j in range(4)]


@pytest.mark.parametrize("act", [False, True])
@pytest.mark.parametrize("heads,size", HEAD_SIZES)
def test_every_element_is_stored_at_its_own_place(heads, size, act):
    """The four-wide store as emitted, for heads that a group of four columns
    ends inside of: each element of the output written once, by its owner."""
    sched = _schedule(HeadSize(heads, size, act), (torch.zeros(2, 8, 64, dtype=torch.float16),))
    (i, (_, parts)), = sched.merged.items()
    y, (part,) = sched.kernels[i].outputs[0], parts
    text, _ = emit_group(sched.kernels[i], parts)
    own = next(a for a, read in zip(part.kernel.inputs, part.reads) if read is None)
    place = {own.index.evaluate(idx=idx): idx for idx in range(part.kernel.numel)}
    for m in range(y.shape[0]):
        for n in range(part.lo, part.hi, 4):
            assert _stored_at(text, part, 0, m, n, False) == \
                [place[m * y.shape[1] + n + j] for j in range(4)], (m, n)


def test_a_group_keeps_its_buffers_alive_throughout():
    """The down projection's residual and input outlive the group's output's
    first write: no two of them share arena bytes."""
    sched = _schedule(*cases()[1][1:3])
    plan = sched.plan
    for i, (end, parts) in sched.merged.items():
        names = {v.buffer.name for k in sched.kernels[i:end + 1] for v in (*k.reads(), *k.writes())}
        spans = sorted((plan.offsets[n], plan.offsets[n] + plan.live_ranges[n].size)
                       for n in names if n in plan.offsets)
        assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("at", range(5))
def test_results(at, dtype):
    """Against float64 of the same values: a few roundings of the storage type
    over sums of at most 192 products."""
    name, model, args, _ = cases(dtype)[at]
    model = model.to(dtype)
    want = model.double()(*(a.double() for a in args))
    model = model.to(dtype).cuda()
    compiled = mlc.compile(model, tuple(a.cuda() for a in args), ALL)
    got = compiled(*(a.cuda() for a in args))
    torch.cuda.synchronize()
    runs = [kind for kind, _ in compiled._runs]
    if name not in ("twice", "transposed"):
        assert len(compiled.schedule.merged) >= 1 and "extern" not in runs
    ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
    err = (got.double().cpu() - want).abs().max() / want.abs().max()
    assert err <= 4 * ulp, (name, err)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,size", HEAD_SIZES)
def test_results_by_head_size(heads, size):
    """Against float64: two roundings to fp16 (product, then bias and ReLU)
    over sums of 64 products; a misplaced element is off by its own size."""
    torch.manual_seed(0)
    model, x = HeadSize(heads, size, True).half(), torch.randn(2, 33, 64).half()
    want = model.double()(x.double())
    x, model = x.cuda(), model.half().cuda()
    compiled = mlc.compile(model, (x,), ALL)
    assert compiled.schedule.merged
    assert (compiled(x).double().cpu() - want).abs().max() <= 2.0 ** -9 * want.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,n,w,h", [(3, 100, 512, 8), (6, 200, 768, 12), (8, 96, 768, 12)])
def test_merged_projections_with_one_stored_by_columns(b, n, w, h, dtype):
    """q, k and v out of one launch, one of them transposed by the attention
    (``store`` and ``store_t`` in one kernel), rows past the last whole tile."""
    torch.manual_seed(0)
    model, x = Heads(w, h).to(dtype), torch.randn(b, n, w).to(dtype)
    want = model.double()(x.double())
    x, model = x.cuda(), model.to(dtype).cuda()
    compiled = mlc.compile(model, (x,), ALL)
    (i, (_, parts)), = compiled.schedule.merged.items()
    assert "auto store_t =" in emit_group(compiled.schedule.kernels[i], parts)[0]
    ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
    err = (compiled(x).double().cpu() - want).abs().max() / want.abs().max()
    assert err <= 4 * ulp, err


@pytest.mark.gpu
def test_a_replayed_graph_gives_the_uncaptured_result():
    name, model, args, _ = cases()[2]
    model, args = model.half().cuda(), tuple(a.cuda() for a in args)
    want = mlc.compile(model, args, ALL)(*args).clone()
    compiled = mlc.compile(model, args, ALL.replace(cuda_graphs=True))
    for _ in range(3):
        assert torch.equal(compiled(*args), want)
        torch.cuda.synchronize()
        torch.zeros(1 << 16, device="cuda").add_(1)
