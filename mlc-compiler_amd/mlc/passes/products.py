"""Products that absorb the pointwise kernels after them
(``Config.gemm_epilogue``).

A library GEMM writes its result and the kernels after it read it back: fc1's
bias and GELU, the bias and re-layout of merged q/k/v. Where such kernels
follow an ``mm`` directly, are its result's only readers and each read it at a
map that a tile of the result can invert, the runtime runs the group as one
launch (``codegen/hip_gemm``): the result is rounded to its storage type in
registers, as the library stores it, and each kernel's body is evaluated on it
there. The schedule keeps its kernels (per-kernel profiling times them one by
one); ``Schedule.merged`` names the groups. The planner keeps every buffer of a
group alive through all of it and leaves the product out, which is never
stored. What that saves it spends on not writing where the launch before has
just read (``memory_planning._pack_groups``): a GPT-2 block takes 201 MB at b32
s512 fp16, its kernels one by one 226.
"""

from __future__ import annotations

import math
from dataclasses import dataclass
from fractions import Fraction

import torch

from ..ir.graph import Value
from ..kernels import ExternKernel, KernelArg, PointwiseKernel, Schedule

FLOATS = (torch.float16, torch.bfloat16, torch.float32)


@dataclass(frozen=True)
class Read:
    """An operand at ``base + row * m + col * (n - lo)`` (``col`` 0 or 1)."""

    base: int
    row: int
    col: int


@dataclass(frozen=True)
class Part:
    """One pointwise kernel over columns ``[lo, hi)`` of the product: its
    operands (``None`` for the product itself) and, for its contiguous output,
    the terms ``(size, step, stride)`` that give an element's index from the
    row (``m_terms``) and the column past ``lo`` (``n_terms``)."""

    kernel: PointwiseKernel
    lo: int
    hi: int
    reads: tuple
    m_terms: tuple
    n_terms: tuple


def _terms(a: KernelArg):
    axis = a.index.axis("idx")
    return axis.terms if axis is not None else ()


def _radix(terms):
    """``terms`` sorted outermost first when their steps are the places of one
    mixed radix number down to 1, with its range; else None."""
    terms = sorted(terms, key=lambda t: -t[1])
    place = 1
    for size, step, _ in reversed(terms):
        if step != place:
            return None
        place *= size
    return tuple(terms), place


def _split_rows(terms, N: int):
    """Terms that run on from one row of ``N`` into the next, cut there."""
    out = []
    for size, step, stride in terms:
        per = N // stride if stride and N % stride == 0 else 0
        if 1 < per < size and size % per == 0:
            out += [(size // per, step * per, N), (per, step, stride)]
        else:
            out.append((size, step, stride))
    return tuple(out)


def _coefficients(terms, cuts):
    """Stride of each digit between neighbouring ``cuts`` of the iteration
    index; None when a term's own places are not among them."""
    found = [0] * (len(cuts) - 1)
    for size, step, stride in terms:
        if step not in cuts or step * size not in cuts:
            return None
        for i, place in enumerate(cuts[:-1]):
            if step <= place < step * size:
                found[i] = stride * (place // step)
    return found


def match_part(k: PointwiseKernel, y: Value) -> Part | None:
    """How ``k`` runs on tiles of the contiguous ``[M, N]`` product ``y``."""
    M, N = y.shape
    if len(k.outputs) != 1 or not k.outputs[0].index.is_identity():
        return None
    if any(a.dtype not in FLOATS for a in (*k.inputs, *k.outputs)):
        return None
    own = [a for a in k.inputs if a.buffer is y.buffer]
    if not own or any(a.index != own[0].index for a in own):
        return None
    terms, base = _split_rows(_terms(own[0]), N), own[0].index.base
    # the index and the place in y are the same digits in two orders
    whole = _radix(terms)
    if whole is None or whole[1] != k.numel or k.numel == 0:
        return None
    rows = _radix([(size, stride // N, step) for size, step, stride in terms if stride % N == 0])
    cols = _radix([(size, stride, step) for size, step, stride in terms if stride % N])
    if rows is None or cols is None or rows[1] != M or base + cols[1] > N:
        return None
    lo, width = base, cols[1]
    if lo % 4 or width % 4 or N % 4:
        return None
    reads = []
    for a in k.inputs:
        if a.buffer is y.buffer:
            reads.append(None)
            continue
        mine = _terms(a)
        cuts = sorted({p for t in (*terms, *mine) for p in (t[1], t[1] * t[0])} | {1, k.numel})
        if any(b % c for c, b in zip(cuts, cuts[1:])):
            return None
        at, of = _coefficients(terms, cuts), _coefficients(mine, cuts)
        if at is None or of is None:
            return None
        # every digit of the column moves the operand as far as the product
        # (or not at all), every digit of the row by one and the same pitch
        col = {Fraction(o, n) for o, n in zip(of, at) if n % N}
        row = {Fraction(o, n // N) for o, n in zip(of, at) if n % N == 0}
        pitch, step = next(iter(row), Fraction(0)), next(iter(col), Fraction(0))
        if len(col) > 1 or len(row) > 1 or step not in (0, 1) or pitch.denominator != 1:
            return None
        reads.append(Read(a.index.base, int(pitch), int(step)))
    return Part(k, lo, lo + width, tuple(reads), rows[0], cols[0])


def product_group(kernels, i: int, graph_outputs) -> tuple[int, list[Part]] | None:
    """(last index, parts) of the group that starts at the ``mm`` at ``i``."""
    k = kernels[i]
    if not isinstance(k, ExternKernel) or k.node.op != "aten.mm.default" or k.node.kwargs:
        return None
    y = k.outputs[0]
    if (len(y.shape) != 2 or y.buffer.name in graph_outputs or y.buffer.numel != math.prod(y.shape)
            or not y.layout.is_contiguous()):
        return None
    readers = [j for j, x in enumerate(kernels) if any(v.buffer is y.buffer for v in x.reads())]
    if not readers or readers != list(range(i + 1, i + 1 + len(readers))):
        return None
    parts = []
    for j in readers:
        part = match_part(kernels[j], y) if isinstance(kernels[j], PointwiseKernel) else None
        if part is None:
            return None
        parts.append(part)
    # one launch has no order between its parts: none may read another's output
    made = {p.kernel.outputs[0].buffer.name for p in parts}
    if any(a.buffer.name in made for p in parts for a in p.kernel.inputs):
        return None
    return readers[-1], parts


def merge_products(schedule: Schedule) -> int:
    """Record the groups the runtime runs as one launch; returns how many."""
    from ..codegen.hip_gemm import plan_group

    outputs = {v.buffer.name for v in schedule.graph.outputs}
    schedule.merged = {}
    for i, k in enumerate(schedule.kernels):
        found = product_group(schedule.kernels, i, outputs)
        if found is not None and plan_group(k, found[1]) is not None:
            schedule.merged[i] = found
    return len(schedule.merged)
