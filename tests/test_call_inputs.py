"""What a call does with the caller's inputs before its kernels run, on the
CPU: the executor's own code with a stand-in for the native launches."""

import ctypes
from types import SimpleNamespace

import pytest
import torch
import torch.nn as nn

from mlc.api import build_pipeline
from mlc.codegen.hip_backend import build_products
from mlc.config import Config
from mlc.ir.capture import capture
from mlc.runtime.executor import CompiledModel
from mlc.runtime.hip_runtime import HipRuntime
from oracle import TorchReferenceRunner

CFG = Config(cuda_graphs=False)
STREAM = SimpleNamespace(cuda_stream=0)


class _Replaying(TorchReferenceRunner):
    """The copies of ``graph_call`` have no order among them: run here in the
    given one or the other way round."""

    MAX_COPIES = 8

    def __init__(self, backwards=False):
        self.backwards, self.copies = backwards, []

    def graph_call(self, copies, stream):
        self.copies = copies
        for dst, src, nbytes in copies[::-1] if self.backwards else copies:
            assert dst and src
            ctypes.memmove(dst, src, nbytes)


def _compile(model, args, runner):
    graph = capture(model, args)
    compiled = CompiledModel(graph, build_pipeline(graph, CFG), CFG, torch.device("cpu"),
                             runner=runner)
    compiled(*args)  # the buffers exist
    return compiled


class Shift(nn.Module):
    """Hands its second input back."""

    def forward(self, a, b):
        return b, a + b


@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("backwards", [False, True])
@pytest.mark.parametrize("at", [0, 1])
def test_a_returned_input_fed_to_another_place(at, backwards, strided):
    """An output that is a view of an input's own buffer is read before any
    input is written, whichever copy runs first."""
    torch.manual_seed(0)
    a, b, c = (torch.randn(6, 8) for _ in range(3))
    compiled = _compile(Shift(), (a, b), _Replaying(backwards))
    shown = compiled(a, b)[0]
    assert torch.equal(shown, b)
    fresh = torch.stack([c, c], -1)[..., 0] if strided else c
    compiled._replay((shown, fresh) if at == 0 else (fresh, shown), STREAM)
    got = [t.view(6, 8) for t in compiled._buffers.inputs]
    want = [b, c] if at == 0 else [c, b]
    assert all(torch.equal(g, w) for g, w in zip(got, want))


class _Apart(TorchReferenceRunner):
    """A runtime that cannot run any group as one launch."""

    def bind_group(self, k, buffers):
        return None


def _linear():
    model = nn.Sequential(nn.Linear(64, 64), nn.ReLU())
    args = (torch.randn(32, 64),)
    graph = capture(model, args)
    return model, args, graph, build_pipeline(graph, CFG.replace(gemm_epilogue=True))


def test_a_group_that_cannot_be_bound_runs_its_kernels():
    model, args, graph, sched = _linear()
    assert sched.merged
    compiled = CompiledModel(graph, sched, CFG, torch.device("cpu"), runner=_Apart())
    torch.testing.assert_close(compiled(*args), model(*args))


def test_a_product_off_16_bytes_is_the_librarys():
    """A weight at an odd place in flat storage, an input view in the unplanned
    mode: the native kernels' loads need 16-byte aligned buffers, the library's
    do not."""
    _, _, _, sched = _linear()
    module, groups = build_products(sched)
    at = {v.buffer.name: 4096 * (i + 1) for i, v in enumerate(
        {v.buffer.name: v for k in sched.kernels for v in (*k.reads(), *k.writes())}.values())}
    buffers = {v.buffer.name: SimpleNamespace(
        device=torch.device("cuda"), dtype=v.buffer.dtype, numel=lambda n=v.buffer.numel: n,
        data_ptr=lambda n=v.buffer.name: at[n])
        for k in sched.kernels for v in (*k.reads(), *k.writes())}
    rt = object.__new__(HipRuntime)
    rt._plans, rt.lib = [], None
    rt.product_table, rt.group_table = groups, groups  # the same operands either way
    rt.functions = {spec.symbol: 1 for spec in groups.values()}
    k = sched.kernels[min(sched.merged)]
    assert rt.bind_product(k, buffers) is not None and rt.bind_group(k, buffers) is not None
    at[k.node.args[1].buffer.name] += 2
    assert rt.bind_product(k, buffers) is None and rt.bind_group(k, buffers) is None


class Add(nn.Module):
    def forward(self, a, b):
        return a + b


def test_a_zero_tensor_has_no_memory_to_read():
    """torch's efficient zero tensors have a null address: they go through
    torch's own copy, on both ways in."""
    a = torch.randn(6, 8)
    compiled = _compile(Add(), (a, a), _Replaying())
    compiled._buffers.inputs[1].fill_(7.0)
    zero = torch._efficientzerotensor(6, 8)
    assert zero.data_ptr() == 0
    compiled._replay((a, zero), STREAM)
    assert torch.equal(compiled._buffers.inputs[1], torch.zeros(48))
    assert compiled._in_place((a, a)) == [a.data_ptr()] * 2
    assert compiled._in_place((a, zero)) is None


def test_the_seams_methods_for_invalid_inputs():
    for name in ("fetch_errors", "pending_error", "clear_errors", "check_errors"):
        assert callable(getattr(HipRuntime, name))
    assert object.__new__(HipRuntime).fetch_errors(0) is None  # nothing to enqueue


@pytest.mark.parametrize("launches,rows,asked,direct", [
    (1, 6, False, True), (8, 6, False, True), (9, 6, False, False), (9, 1 << 20, True, True),
    (32, 1 << 20, True, True), (33, 1 << 20, False, False)])
def test_the_device_estimate_is_made_only_where_it_decides(launches, rows, asked, direct, monkeypatch):
    """A first pass pays for it on the host: eight native launches are made
    one by one whatever it says, more than 32 never are, and nine not where
    the buffers themselves are too small to keep the device busy."""
    a = torch.zeros(rows, 8)
    compiled = _compile(Add(), (a, a + 1), _Replaying())
    asked_for = []
    monkeypatch.setattr(CompiledModel, "_device_estimate",
                        staticmethod(lambda work: asked_for.append(len(work)) or 1e9))
    compiled._launches = compiled._launches * launches
    assert compiled._launch_directly() == direct
    assert asked_for == [launches] * asked
