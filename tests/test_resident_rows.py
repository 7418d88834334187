"""Streamed rows that stay in one workgroup's registers: the packs at a row's
ends, rows that start off the 16-byte grid, and the sizes where the layout
changes."""

import pytest
import torch

import mlc
from mlc.api import build_pipeline
from mlc.codegen.hip_backend import build_module
from mlc.config import Config
from mlc.ir.capture import capture
from oracle import compile_reference

CFG = Config(cuda_graphs=False)


class Softmax(torch.nn.Module):
    def forward(self, x):
        return torch.softmax(x / 0.8, dim=-1)


class Norm(torch.nn.Module):
    """Two column operands, two reductions, a row output."""

    def forward(self, x, y):
        s = x + y
        return (s - s.mean(-1, keepdim=True)) / 2.0, s.amax(-1)


def _spec(model, args):
    sched = build_pipeline(capture(model, args), CFG)
    specs = build_module(sched, CFG).launches.values()
    return [s.meta for s in specs if s.meta["kind"] == "reduction"]


@pytest.mark.parametrize("cols,dtype,resident", [
    (16384, torch.float16, None),    # held by the persistent form
    (16385, torch.float16, True), (16392, torch.bfloat16, True), (50257, torch.float16, True),
    (65528, torch.float16, True), (65536, torch.float16, True),
    (65529, torch.float16, False),   # an odd row of 8 packs and one more
    (65537, torch.float16, False), (65536, torch.float32, True), (65537, torch.float32, False)])
def test_which_rows_stay_resident(cols, dtype, resident):
    meta, = _spec(Softmax(), (torch.zeros(2, cols, dtype=dtype),))
    assert meta["mode"] == ("persistent" if resident is None else "streamed")
    assert meta["resident"] == (resident is not False)


def test_operands_off_the_grid_by_different_amounts_are_streamed():
    class Add(torch.nn.Module):
        def forward(self, x, y):
            return (x + y).softmax(-1)

    x = torch.zeros(3, 20001, dtype=torch.float16)
    meta, = _spec(Add(), (x, x[0]))  # y does not move with the row
    assert meta["mode"] == "streamed" and not meta["resident"]


SHAPES = [(3, 16385), (9, 16391), (2, 16392), (5, 50257), (1, 65528), (4, 65521)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", SHAPES)
def test_softmax(shape, dtype):
    """Against float64: a probability is rounded once to its storage type
    (half an ulp: 2^-11, 2^-8) after fp32 work (2e-6 covers the exponent's
    rounding and the sum); fp16's subnormal spacing is 2^-24."""
    torch.manual_seed(0)
    x = (torch.randn(*shape) * 3).to(dtype)
    x[0, : shape[1] // 2] = float("-inf")
    got = mlc.compile(Softmax(), (x.cuda(),), CFG)(x.cuda()).double().cpu()
    want = torch.softmax(x.double() / 0.8, dim=-1)
    rel = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2e-6}[dtype] + 2e-6
    tiny = 2.0 ** -25 if dtype == torch.float16 else 1e-37
    assert ((got - want).abs() <= rel * want + tiny).all()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES[:4])
def test_two_operands_and_a_row_output(shape):
    torch.manual_seed(0)
    x, y = torch.randn(*shape).half(), torch.randn(*shape).half()
    if shape[1] > 32768:  # two operands: past the register limit, streamed
        assert not _spec(Norm(), (x, y))[0]["resident"]
    want = compile_reference(Norm(), (x, y), CFG)(x, y)
    got = mlc.compile(Norm(), (x.cuda(), y.cuda()), CFG)(x.cuda(), y.cuda())
    for g, w in zip(got, want):
        # one fp16 ulp of the largest value: the mean's sum order differs
        assert (g.cpu().float() - w.float()).abs().max() <= 2.0 ** -10 * w.float().abs().max()
    assert torch.equal(got[1].cpu(), want[1])
