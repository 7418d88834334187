"""Algorithmic HBM bytes of a generated kernel, the unit the bandwidth
roofline is priced in.

    bytes(k) = sum over distinct (buffer, index map) inputs of
                   (distinct elements addressed) * itemsize
             + sum over outputs of (elements written) * itemsize

An index map's distinct elements are the product of the sizes of its
canonical terms (stride-0 dims are already dropped, so a broadcast operand
counts once). This equals the reference cost model's traffic
(``mlc/passes/cost.py:44-59``) when no operand is broadcast-expanded. A fused
attention kernel is priced the same way: q, k, v and the reduction's other
operands read once, the output written once (the scores and probabilities it
keeps on chip are not HBM traffic).
"""

from __future__ import annotations

from ..codegen.index import IndexMap
from ..kernels import AttentionKernel, ExternKernel, PointwiseKernel, ReductionKernel

#: MI355X published peak HBM3E bandwidth, GB/s
HBM_PEAK_GBS = 8000.0


def distinct_elements(imap: IndexMap) -> int:
    n = 1
    for axis in imap.axes:
        for size, _, _ in axis.terms:
            n *= size
    return n


def _moved(kernels, unstored: str | None = None) -> int:
    """Bytes of every distinct operand view and every output of ``kernels``
    but the buffer ``unstored``. Views are compared only where a buffer comes
    up again: a first pass prices its launches so on the host."""
    total, seen = 0, {}
    for k in kernels:
        if isinstance(k, ExternKernel):
            reads = [(v.buffer.name, v.layout, v.numel * v.dtype.itemsize) for v in k.inputs]
            writes = [(v.buffer.name, v.numel * v.dtype.itemsize) for v in k.outputs]
        else:
            reads = [(a.value.buffer.name, a.index, distinct_elements(a.index) * a.dtype.itemsize)
                     for a in k.inputs]
            writes = [(a.value.buffer.name, distinct_elements(a.index) * a.dtype.itemsize)
                      for a in k.outputs]
        for name, view, nbytes in reads:
            views = seen.setdefault(name, [])
            if name != unstored and view not in views:
                views.append(view)
                total += nbytes
        total += sum(nbytes for name, nbytes in writes if name != unstored)
    return total


def algorithmic_bytes(k) -> int:
    if isinstance(k, ExternKernel):
        if k.node.op == "aten.embedding.default":
            out = k.outputs[0]
            ids = k.node.args[1]
            return 2 * out.numel * out.dtype.itemsize + ids.numel * ids.dtype.itemsize
        raise TypeError(f"no byte model for extern {k.node.op}")
    if not isinstance(k, (PointwiseKernel, ReductionKernel, AttentionKernel)):
        raise TypeError(type(k).__name__)
    return _moved([k])


def extern_bytes(k: ExternKernel) -> int:
    """Algorithmic bytes of a library call: every distinct operand view read
    once (a GEMM's weights included) plus every output written once."""
    return _moved([k])


def launch_bytes(kernels) -> int:
    """Algorithmic bytes of one launch: a kernel's, or those of a product and
    the pointwise kernels after it as one, which never stores the product and
    reads what several of them read once."""
    first = kernels[0]
    if len(kernels) == 1:
        gather = isinstance(first, ExternKernel) and first.node.op == "aten.embedding.default"
        return algorithmic_bytes(first) if gather or not isinstance(first, ExternKernel) \
            else extern_bytes(first)
    return _moved(kernels, first.outputs[0].buffer.name)


def forward_bytes(schedule) -> int:
    """Algorithmic bytes of one whole forward: every kernel, generated or
    library, at its algorithmic traffic. Divided by the HBM peak it is the
    bytes-moved floor of the forward's latency."""
    return sum(launch_bytes([k]) for k in schedule.kernels)
