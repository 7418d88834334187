"""Short schedules launched kernel by kernel on the caller's own inputs: when
that is allowed, and that every kind of input gives what a copied one gives."""

import pytest
import torch
import torch.nn as nn

import mlc
from mlc.config import Config

pytestmark = pytest.mark.gpu


class Chain(nn.Module):
    """Two kernels: the second input is read after the first output exists."""

    def forward(self, x, y):
        return (x * 2.0 + 1.0).softmax(-1) - y, y.sum(-1)


class Identity(nn.Module):
    def forward(self, x):
        return x, x + 1.0


class LibraryFirst(nn.Module):
    """A product left to the library reads the input."""

    def __init__(self):
        super().__init__()
        self.w = nn.Parameter(torch.randn(48, 100) * 0.1)

    def forward(self, x):
        return torch.relu(torch.mm(x, self.w.t()) + 1.0)


def _args(dtype=torch.float32):
    torch.manual_seed(0)
    return torch.randn(64, 96).cuda().to(dtype), torch.randn(64, 96).cuda().to(dtype)


def _same(got, want):
    return all(torch.equal(g, w) for g, w in zip(got, want))


def test_every_kind_of_input():
    x, y = _args()
    compiled = mlc.compile(Chain(), (x, y))
    want = [t.clone() for t in mlc.compile(Chain(), (x, y), Config(cuda_graphs=False))(x, y)]
    assert _same(compiled(x, y), want) and compiled._direct and not compiled._captured
    wide = torch.empty(64, 200, device="cuda")
    wide[:, 3:99] = x
    odd = torch.empty(64 * 96 + 1, device="cuda")
    odd[1:] = x.reshape(-1)
    kinds = {"strided": wide[:, 3:99], "transposed": x.t().contiguous().t(), "host": x.cpu(),
             "pinned": x.cpu().pin_memory(), "double": x.double(), "misaligned": odd[1:].view(64, 96),
             "parameter": nn.Parameter(x), "another buffer": x.clone()}
    for name, t in kinds.items():
        assert _same(compiled(t, y), want), name
        assert _same(compiled(x, y), want), name


def test_a_kernel_of_many_operands():
    """One launch of more than 128 pointers (1 KiB of arguments)."""
    class Sum(nn.Module):
        def forward(self, *xs):
            return sum(xs[1:], xs[0] * 2.0)

    torch.manual_seed(0)
    xs = tuple(torch.randn(8, 64, device="cuda") for _ in range(150))
    compiled = mlc.compile(Sum(), xs)
    want = mlc.compile(Sum(), xs, Config(cuda_graphs=False))(*xs).clone()
    assert torch.equal(compiled(*xs), want) and compiled._direct
    odd = torch.empty(8 * 64 + 1, device="cuda")
    odd[1:] = xs[7].reshape(-1)
    assert torch.equal(compiled(*xs[:7], odd[1:].view(8, 64), *xs[8:]), want)


def test_an_output_fed_back_is_copied_first():
    x, y = _args()
    compiled = mlc.compile(Chain(), (x, y))
    plain = mlc.compile(Chain(), (x, y), Config(cuda_graphs=False))
    first = compiled(x, y)[0]
    kept = first.clone()
    want = [t.clone() for t in plain(kept, kept)]
    assert _same(compiled(first, first), want)


def test_the_input_may_change_after_the_call():
    x, y = _args()
    compiled = mlc.compile(Chain(), (x, y))
    want = [t.clone() for t in compiled(x, y)]
    z = x.clone()
    got = compiled(z, y)
    z.fill_(7.0)  # same stream: after the pass
    assert _same(got, want)


def test_another_stream_and_device_order():
    x, y = _args()
    compiled = mlc.compile(Chain(), (x, y))
    want = [t.clone() for t in compiled(x, y)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = [t.clone() for t in compiled(x, y)]
    side.synchronize()
    assert _same(got, want)


def test_an_input_of_another_stream_may_be_dropped():
    x, y = _args()
    compiled = mlc.compile(Chain(), (x, y))
    want = [t.clone() for t in compiled(x, y)]
    z = x.clone()
    at = z.data_ptr()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(2_000_000)  # the pass is still to come when z goes
        got = compiled(z, y)
    del z
    fresh = torch.full_like(x, 7.0)
    assert fresh.data_ptr() != at
    side.synchronize()
    assert _same(got, want)


def test_when_a_graph_is_kept():
    x, _ = _args()
    identity = mlc.compile(Identity(), (x,))
    assert torch.equal(identity(x)[0], x) and not identity._direct
    x = torch.randn(16, 100, device="cuda", dtype=torch.float16)
    model = LibraryFirst().half().cuda()
    lib = mlc.compile(model, (x,))
    got = lib(x)
    assert not lib._direct and lib._captured
    want = torch.relu((x.double() @ model.w.double().t()).half().double() + 1.0)
    assert (got.double() - want).abs().max() <= 2e-3 * want.abs().max()
    # the graph's inputs: several in one launch, odd sizes, host tensors
    for t in (x.clone(), x.cpu(), x.float(), x.t().contiguous().t()):
        assert torch.equal(lib(t), got)


def test_ids_are_checked_without_a_copy_back():
    class Gather(nn.Module):
        def __init__(self):
            super().__init__()
            self.e = nn.Embedding(10, 64)

        def forward(self, ids):
            return self.e(ids) * 2.0

    ids = torch.randint(0, 10, (4, 7), device="cuda")
    compiled = mlc.compile(Gather().cuda(), (ids,))
    want = compiled(ids).clone()
    assert compiled._direct
    bad = ids.clone()
    bad[1, 2] = 10
    compiled(bad)
    torch.cuda.synchronize()
    with pytest.raises(Exception, match="outside its table"):
        compiled(ids)
    assert torch.equal(compiled(ids), want)
