"""Native matrix products in the place of library GEMMs: which calls take
which form, and both forms at the edges of their tiles, strides and types."""

import pytest
import torch

import mlc
from mlc.api import build_pipeline
from mlc.codegen import hip_gemm
from mlc.codegen.hip_backend import PRELUDE, emit_kernel
from mlc.codegen.hip_gemm import (LDS_BYTES, MERGED_FLOPS, TILED_FLOPS, TILES, choose_tile, emit_product,
                                  plan_product)
from mlc.config import Config
from mlc.ir.capture import capture
from mlc.kernels import ExternKernel
from mlc.runtime import native
from mlc.runtime.executor import ProductCall

CFG = Config(cuda_graphs=False, gemm_epilogue=True)
HALF_ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 0.0}


class Linear(torch.nn.Module):
    def forward(self, x, w):
        return torch.mm(x, w.t())


class Biased(torch.nn.Module):
    def forward(self, x, w, bias):
        return torch.mm(x, w.t()) + bias


class Batched(torch.nn.Module):
    def __init__(self, a_order, b_order):
        super().__init__()
        self.a_order, self.b_order = a_order, b_order

    def forward(self, a, b):
        return torch.bmm(a.permute(self.a_order), b.permute(self.b_order))


def _plans(model, args):
    sched = build_pipeline(capture(model, args), CFG)
    return [plan_product(k) for k in sched.kernels if isinstance(k, ExternKernel)]


def _form(model, *args):
    plan, = _plans(model, args)
    return None if plan is None else plan.form[0]


def test_which_calls_run_natively():
    def half(*s):
        return torch.zeros(*s, dtype=torch.float16)

    assert _form(Linear(), half(128, 768), half(768, 768)) == "tiled"
    assert _form(Linear(), half(1, 64), half(48, 64)) == "tiled"
    assert _form(Linear(), half(16384, 768), half(2304, 768)) == "tiled"
    assert _form(Linear(), half(16384, 768), half(3072, 768)) is None      # past the flops line
    assert _form(Linear(), half(16384, 3072), half(768, 3072)) is None     # with long sums
    # a vocabulary head: few rows, or whole tiles of them
    for rows, native in ((16, True), (64, False), (128, True), (333, False), (512, True)):
        assert _form(Linear(), half(rows, 768), half(50257, 768)) == ("tiled" if native else None)
    assert _form(Linear(), torch.zeros(128, 768), torch.zeros(50257, 768)) is None
    assert _form(Linear(), half(128, 100), half(96, 100)) is None          # k not in whole pieces
    assert _form(Linear(), torch.zeros(64, 64, dtype=torch.float64),
                 torch.zeros(64, 64, dtype=torch.float64)) is None
    heads = half(12, 128, 64)
    assert _form(Batched((0, 1, 2), (0, 2, 1)), heads, heads) == "tiled"
    assert _form(Batched((0, 1, 2), (0, 1, 2)), half(12, 128, 128), heads) == "staged"
    assert _form(Batched((0, 1, 2), (0, 1, 2)), half(6, 197, 197), half(6, 197, 64)) == "staged"
    assert _form(Batched((0, 1, 2), (0, 1, 2)), half(64, 1024, 1024), half(64, 1024, 64)) is None


@pytest.mark.parametrize("size", [2, 4])
def test_every_tile_splits_its_product(size):
    """The tile chosen for any size divides among its waves and its k-splits
    and fits LDS (the template's own static conditions)."""
    for M in (1, 2, 15, 16, 17, 33, 64, 100, 128, 197, 300, 512, 1182, 2048, 4096, 20480):
        for N in (1, 16, 48, 64, 197, 512, 768, 2304, 3072, 4096):
            for K in (128 // size * n for n in (1, 2, 3, 5, 7, 8, 12, 48)):
                for batches in (1, 12, 64, 256):
                    if 2.0 * batches * M * N * K > max(TILED_FLOPS[size], MERGED_FLOPS):
                        continue
                    tile, pieces = choose_tile(M, N, K, batches, size), K * size // 128
                    if tile is None:  # few fp32 rows need a k-split of 4
                        assert size == 4 and M <= 128 and pieces % 4
                        continue
                    TM, TN, WM, WN, WK, stages = tile
                    assert pieces % WK == 0 and (TM + TN) % (8 * WM * WN) == 0
                    assert TM % (16 * WM) == 0 and TN % (16 * WN) == 0 and WM * WN * WK <= 16
                    ring = min(stages, pieces // WK) * WK * (TM + TN) * 128
                    assert 2 <= stages <= 4 and ring <= 160 * 1024
                    epilogue = WK * TM * (TN + 4) * 4 if WK > 1 else \
                        max(WM * 16 * (TN + 4 * WN) * 4, WM * TN * 20 * size)
                    assert epilogue <= 160 * 1024


def test_launches_stay_below_two_to_the_32_threads():
    """HIP's limit for a launch: a batch past it stays with the library, as a
    reduction over so many resident rows stays with the chunk loop."""
    def scores(batch):
        return _form(Batched((0, 1, 2), (0, 1, 2)), torch.empty(batch, 2, 3, dtype=torch.float16, device="meta"),
                     torch.empty(batch, 3, 2, dtype=torch.float16, device="meta"))

    assert scores((1 << 24) - 8) == "staged" and scores(1 << 24) is None

    class Long(torch.nn.Module):
        def forward(self, x):
            return x.sum(-1)

    def resident(rows):
        x = torch.empty(rows, 40000, dtype=torch.float16, device="meta")
        k, = build_pipeline(capture(Long(), (x,)), CFG).kernels
        return emit_kernel(k, CFG)[1].meta["resident"]

    assert resident((1 << 22) - 1) and not resident(1 << 22)


def _largest(size):
    """Products up to the operations line, by tile, that take a tile of 64 x 64
    or more over one piece of k: the ring is at its smallest."""
    K, found = 128 // size, {}
    for M in (33, 100, 300, 512, 2048, 4096, 20480):
        for N in (48, 197, 512, 768, 3072, 4096):
            for batches in (1, 64):
                tile = choose_tile(M, N, K, batches, size)
                if 2.0 * batches * M * N * K <= TILED_FLOPS[size] and tile[0] * tile[1] >= 64 * 64:
                    found.setdefault(tile, (batches, M, N, K))
    return found


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_the_large_tiles_compile_over_one_piece_of_k(dtype):
    """The template's conditions on the tile that is chosen, by the compiler:
    with one stage the epilogue's buffers are more of LDS than the ring is."""
    bodies = []
    found = _largest(dtype.itemsize)
    assert any(t[:2] == (256, 256) for t in found)
    for tile, (B, M, N, K) in found.items():
        model, args = Batched((0, 1, 2), (0, 2, 1)), (torch.empty(B, M, K, dtype=dtype, device="meta"),
                                                      torch.empty(B, N, K, dtype=dtype, device="meta"))
        sched = build_pipeline(capture(model, args), CFG)
        body, spec = emit_product(next(k for k in sched.kernels if isinstance(k, ExternKernel)))
        assert spec.meta["form"] == ("tiled", *tile)
        bodies.append(body.replace("KERNEL(", f"product{len(bodies)}(", 1))
    native.compile_code_object("\n\n".join([PRELUDE, '#include "mlc_gemm.h"', *bodies]) + "\n")


def _check(model, args, want, magnitude, K):
    """Within half an ulp of the storage type plus the bound of an fp32 sum of
    K terms in any order, K 2^-24 sum |a b|."""
    compiled = mlc.compile(model, args, CFG)
    got = compiled(*args)
    torch.cuda.synchronize()
    calls = [p for kind, p in compiled._plan if kind == "extern"]
    assert calls and all(isinstance(c, ProductCall) for c in calls)
    got = got.double().cpu()
    assert torch.isfinite(got).all()
    bound = HALF_ULP[args[0].dtype] * want.abs() + (K + 2) * 2.0 ** -24 * magnitude + 2.0 ** -25
    assert ((got - want).abs() <= bound).all(), ((got - want).abs() / bound).max()


def _inside(rows, cols, pad, dtype):
    """A [rows, cols] view with NaN all around it: nothing outside may count."""
    whole = torch.full((rows + 2, cols + 2 * pad), float("nan"))
    whole[1:-1, pad:pad + cols] = torch.randn(rows, cols)
    return whole.to(dtype).cuda()[1:-1, pad:pad + cols]


DTYPES = [torch.float16, torch.bfloat16, torch.float32]


class Inner(torch.nn.Module):
    """The same over views cut out of wider buffers inside the program."""

    def forward(self, x, w):
        return torch.mm(x[1:-1, 8:-8], w[1:-1, 8:-8].t())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(1, 16, 64), (17, 50, 320), (128, 768, 3072), (130, 2304, 768),
                                   (525, 512, 512), (600, 770, 192)])
def test_tiled(shape, dtype):
    M, N, K = shape
    torch.manual_seed(0)
    x, w = _inside(M, K, 8, dtype)._base, _inside(N, K, 8, dtype)._base
    a, b = x[1:-1, 8:-8].double().cpu(), w[1:-1, 8:-8].double().cpu()
    _check(Inner(), (x, w), a @ b.t(), a.abs() @ b.abs().t(), K)


class EveryTile(torch.nn.Module):
    """A product of its own number of rows for each tile, alone and re-laid out
    per head, the middle third of its columns transposed (the column store)."""

    def __init__(self, K):
        super().__init__()
        self.plain = torch.nn.Parameter(torch.randn(525, K))
        self.heads = torch.nn.Parameter(torch.randn(2304, K))

    def forward(self, x):
        out = []
        for i in range(len(TILES)):
            rows = x[:312 + 16 * i]
            out.append(torch.mm(rows, self.plain.t()))
            q, k, v = (t.view(2, -1, 12, 64).transpose(1, 2)
                       for t in torch.mm(rows, self.heads.t()).chunk(3, -1))
            out += [q.contiguous(), k.transpose(-2, -1).contiguous(), v.contiguous()]
        return tuple(out)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,pieces", [(torch.float16, 5), (torch.float16, 1), (torch.bfloat16, 3),
                                          (torch.float32, 5), (torch.float32, 1)])
def test_every_tile_at_ragged_sizes(dtype, pieces, monkeypatch):
    """Every entry of TILES, whatever size would choose it: rows and columns
    past its last whole tile (312 to 536 rows, 525 columns), k shorter and
    longer than the ring, stores along rows and along columns."""
    size, K = dtype.itemsize, 128 // dtype.itemsize * pieces

    def forced(M, N, K, batches, size, math=False):
        TM, TN, WM, WN, splits = TILES[(M - 312) // 16]
        WK = max((n for n in splits if pieces % n == 0), default=None)
        if WK is None:
            return choose_tile(M, N, K, batches, size, math)
        stages = next(n for n in (4, 3, 2)
                      if min(n, pieces // WK) * WK * (TM + TN) * 128 <= LDS_BYTES)
        return TM, TN, WM, WN, WK, min(stages, max(2, pieces // WK))

    monkeypatch.setattr(hip_gemm, "choose_tile", forced)
    torch.manual_seed(0)
    model = EveryTile(K).to(dtype).cuda()
    x = torch.randn(536, K, device="cuda", dtype=dtype)
    compiled = mlc.compile(model, (x,), CFG.replace(layout_selection=True))
    specs = {**compiled._module.product_table, **compiled._module.group_table}
    assert len(compiled.schedule.merged) == len(TILES) and len(specs) == 2 * len(TILES)
    got = compiled(x)
    x, plain, heads = (t.double() for t in (x, model.plain, model.heads))
    for i in range(len(TILES)):
        rows = x[:312 + 16 * i]
        q, k, v = (t.reshape(2, -1, 12, 64).transpose(1, 2) for t in (rows @ heads.t()).chunk(3, -1))
        wide = [t.reshape(2, -1, 12, 64).transpose(1, 2)
                for t in (rows.abs() @ heads.abs().t()).chunk(3, -1)]
        want = [rows @ plain.t(), q, k.transpose(-2, -1), v]
        sums = [rows.abs() @ plain.abs().t(), wide[0], wide[1].transpose(-2, -1), wide[2]]
        for g, w, m in zip(got[4 * i:4 * i + 4], want, sums):
            bound = HALF_ULP[dtype] * w.abs() + (K + 2) * 2.0 ** -24 * m + 2.0 ** -25
            assert ((g.double() - w).abs() <= bound).all(), (TILES[i], ((g.double() - w).abs() / bound).max())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
def test_bias_is_added_before_the_rounding(dtype):
    torch.manual_seed(0)
    x, w, bias = (torch.randn(*s).to(dtype).cuda() for s in ((70, 256), (100, 256), (100,)))
    a, b = x.double().cpu(), w.double().cpu()
    want = a @ b.t() + bias.double().cpu()
    _check(Biased(), (x, w, bias), want, a.abs() @ b.abs().t() + want.abs(), 256)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("orders", [((0, 1, 2), (0, 1, 2)), ((0, 1, 2), (0, 2, 1)),
                                    ((0, 2, 1), (0, 1, 2)), ((1, 0, 2), (1, 2, 0)),
                                    ((2, 0, 1), (1, 0, 2))])
@pytest.mark.parametrize("shape", [(5, 17, 64, 33), (2, 65, 197, 128), (1, 1, 1, 1)])
def test_batched_in_every_order(shape, orders, dtype):
    B, M, N, K = shape
    torch.manual_seed(0)
    args = []
    for order, full in zip(orders, ((B, M, K), (B, K, N))):
        stored = [0, 0, 0]
        for at, axis in enumerate(order):
            stored[axis] = full[at]
        args.append(torch.randn(*stored).to(dtype).cuda())
    a, b = (t.double().cpu().permute(o) for t, o in zip(args, orders))
    _check(Batched(*orders), tuple(args), a @ b, a.abs() @ b.abs(), K)


class Stack(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = torch.nn.Parameter(weight)

    def forward(self, x):
        return torch.relu(torch.mm(x, self.weight.t())) * 2.0


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", [Config(), CFG, CFG.replace(cuda_graphs=True),
                                 CFG.replace(memory_planning=False)])
def test_a_weight_off_16_bytes_goes_to_the_library(cfg):
    torch.manual_seed(0)
    flat = torch.randn(96 * 64 + 1, device="cuda", dtype=torch.float16)
    model = Stack(flat[1:].view(96, 64))
    x = torch.randn(37, 64, device="cuda", dtype=torch.float16)
    want = torch.relu(x.double() @ model.weight.double().t()) * 2.0
    compiled = mlc.compile(model, (x,), cfg)
    for _ in range(3):
        got = compiled(x)
        assert (got.double() - want).abs().max() <= 2.0 ** -10 * want.abs().max()
        torch.cuda.synchronize()


@pytest.mark.gpu
def test_launch_floor_counts_native_products():
    """The graph decomposition takes a native product as a product, in every graph."""
    from mlc.bench.launch_floor import decompose_compiled

    torch.manual_seed(0)
    lin = torch.nn.Linear(128, 128).half().cuda()
    x = torch.randn(128, 128, device="cuda", dtype=torch.float16)
    compiled = mlc.compile(torch.nn.Sequential(lin, torch.nn.ReLU()), (x,))
    d = decompose_compiled(compiled, (x,), replays=2, shapes=False, log=lambda line: None)
    assert compiled._module.product_table and d["library"] >= 1 and d["generated"] >= 1
    # a product that runs the ReLU in its epilogue is one node, as in a pass
    compiled = mlc.compile(torch.nn.Sequential(lin, torch.nn.ReLU()), (x,), Config(gemm_epilogue=True))
    d = decompose_compiled(compiled, (x,), replays=2, shapes=False, log=lambda line: None)
    nodes = {label: n for label, n, _, _ in d["results"]}
    assert (d["library"], d["generated"], nodes["forward (every node real)"]) == (1, 0, 1)
