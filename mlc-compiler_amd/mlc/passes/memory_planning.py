"""The arena: every intermediate buffer at a fixed byte offset of one slab.

Shapes are static and each intermediate buffer is written by one kernel and
read by known later ones, so its lifetime is an interval of kernel indices.
Buffers whose intervals are disjoint may share bytes. On the GPU the arena is
one ``hipMalloc`` slab, and because every offset is fixed at compile time
every kernel argument is the same pointer on every call -- what lets the whole
schedule be captured once as a hipGraph and replayed.

Placement contract (kept bit-exact with the reference planner,
``mlc/passes/memory_planning.py:35-240``, so offsets match its golden
fixtures): buffers are taken largest first, ties by first-write index, then
name; each goes to the lowest offset whose bytes no time-overlapping buffer
already placed occupies; offsets and buffer sizes are multiples of 256 bytes.

Besides placement the planner reports the lower bound no placement can beat
(the most bytes live at one kernel) and checks its own result: any two
buffers live at the same time must not share a byte.
"""

from __future__ import annotations

from collections import defaultdict
from dataclasses import dataclass, field, replace
from itertools import accumulate

from ..config import Config
from ..ir.graph import Graph
from ..ir.types import Buffer
from ..kernels import Schedule
from ..runtime.native import STATIC_SLAB_BYTES

#: byte alignment of every arena offset (16-byte packs, library GEMM operands)
ALIGNMENT = 256


def _round_up(n: int) -> int:
    return -(-n // ALIGNMENT) * ALIGNMENT


@dataclass
class LiveRange:
    buffer: Buffer
    #: index of the kernel that first writes the buffer
    start: int
    #: index of the last kernel touching it (len(schedule) for a graph output)
    end: int
    #: bytes reserved (the buffer's size rounded up to ALIGNMENT)
    size: int

    def overlaps(self, other: "LiveRange") -> bool:
        return self.start <= other.end and other.start <= self.end


@dataclass
class AllocationPlan:
    #: "arena" (placed in one slab) or "eager" (allocated around each kernel)
    mode: str
    arena_bytes: int = 0
    offsets: dict[str, int] = field(default_factory=dict)
    #: eager mode: kernel index -> buffers to allocate before it runs
    alloc_at: dict[int, list[Buffer]] = field(default_factory=dict)
    #: eager mode: kernel index -> buffer names to drop after it runs
    free_at: dict[int, list[str]] = field(default_factory=dict)
    live_ranges: dict[str, LiveRange] = field(default_factory=dict)
    #: most bytes live at any one kernel: the bound no placement can beat
    peak_bytes: int = 0
    #: bytes if every buffer had memory of its own
    total_bytes: int = 0

    @property
    def efficiency(self) -> float:
        """Arena size over the lower bound (1.0 is optimal)."""
        return self.arena_bytes / self.peak_bytes if self.peak_bytes else 1.0

    def summary(self) -> str:
        kib = lambda n: f"{n / 1024:.1f} KiB"  # noqa: E731
        if self.mode == "arena":
            return (f"memory: arena {kib(self.arena_bytes)}, lower bound {kib(self.peak_bytes)} "
                    f"({self.efficiency:.2f}x), unplanned would be {kib(self.total_bytes)}")
        return f"memory: unplanned, peak {kib(self.peak_bytes)} of {kib(self.total_bytes)} total"


# --------------------------------------------------------------------------
# lifetimes
# --------------------------------------------------------------------------

def compute_live_ranges(graph: Graph, schedule: Schedule) -> list[LiveRange]:
    """Lifetimes of the plannable buffers, per *buffer* (a view keeps its
    whole buffer alive), in order of first appearance in the schedule. The
    product of a group that runs as one launch is never stored: it has none."""
    first: dict[str, int] = {}
    last: dict[str, int] = {}
    by_name: dict[str, Buffer] = {}

    def touch(buf: Buffer, i: int, writes: bool) -> None:
        by_name.setdefault(buf.name, buf)
        if writes:
            first.setdefault(buf.name, i)
        last[buf.name] = max(last.get(buf.name, i), i)

    # kernels that run as one launch touch their buffers from its first to its last
    span = {j: (i, end) for i, (end, _) in schedule.merged.items() for j in range(i, end + 1)}
    for i, k in enumerate(schedule.kernels):
        begin, end = span.get(i, (i, i))
        for v in k.writes():
            touch(v.buffer, begin, True)
        for v in (*k.writes(), *k.reads()):
            touch(v.buffer, end, False)
    for v in graph.outputs:  # results outlive the schedule
        by_name.setdefault(v.buffer.name, v.buffer)
        last[v.buffer.name] = len(schedule.kernels)

    unstored = {schedule.kernels[i].outputs[0].buffer.name for i in schedule.merged}
    return [LiveRange(buf, first[name], last[name], _round_up(buf.nbytes))
            for name, buf in by_name.items()
            if buf.plannable and name in first and name not in unstored]


def _rested(schedule: Schedule, ranges: list[LiveRange]) -> list[LiveRange]:
    """``ranges`` kept for one more launch (the ends of groups are launches'
    ends as they are)."""
    group_end = {i: end for i, (end, _) in schedule.merged.items()}
    final = len(schedule.kernels) - 1
    return [r if r.end >= final else replace(r, end=group_end.get(r.end + 1, r.end + 1))
            for r in ranges]


def peak_live_bytes(ranges: list[LiveRange], n_kernels: int) -> int:
    """Most bytes live at one kernel index (a lower bound on the arena)."""
    delta: dict[int, int] = defaultdict(int)
    for r in ranges:
        delta[r.start] += r.size
        delta[r.end + 1] -= r.size
    return max(accumulate(delta[t] for t in sorted(delta)), default=0) if ranges else 0


# --------------------------------------------------------------------------
# placement
# --------------------------------------------------------------------------

def _lowest_fit(busy: list[tuple[int, int]], size: int) -> int:
    """Lowest offset with ``size`` free bytes below the next busy extent;
    ``busy`` are ``[lo, hi)`` byte extents (overlapping allowed)."""
    at = 0
    for lo, hi in sorted(busy):
        if lo - at >= size:
            break
        at = max(at, hi)
    return at


def pack(ranges: list[LiveRange], rested: list[LiveRange] | None = None,
         limit: int = 0) -> tuple[dict[str, int], int]:
    """Offsets of every range and the arena size they need. ``rested``: the
    same ranges with longer ends, kept apart wherever ``limit`` bytes allow."""
    order = sorted(zip(ranges, rested or ranges),
                   key=lambda p: (-p[0].size, p[0].start, p[0].buffer.name))
    offsets: dict[str, int] = {}
    placed: list[tuple[LiveRange, LiveRange, int]] = []
    arena = 0

    def fit(r: LiveRange, resting: bool) -> int:
        return _lowest_fit([(off, _round_up(off + p.size)) for p, long, off in placed
                            if (long if resting else p).overlaps(r)], r.size)

    for r, long in order:
        off = fit(long, True)
        if rested is not None and off + r.size > limit:
            off = fit(r, False)
        offsets[r.buffer.name] = off
        placed.append((r, long, off))
        arena = max(arena, off + r.size)
    return offsets, arena


def _pack_groups(graph: Graph, schedule: Schedule, cfg: Config, ranges: list[LiveRange],
                 tight: tuple[dict[str, int], int]) -> tuple[dict[str, int], int]:
    """``tight``, or a placement that takes no more than the kernels one by
    one would and leaves what a launch has read alone for one more launch.

    What a launch reads is in the L2 of the XCDs that read it, and writing
    there at once costs: in ``tight``, a BERT-base b32 layer's LayerNorm
    writes where its product's input was (7.9 us; 5.3 elsewhere) and that
    product where the attention's was (9.4; 8.4). Forward, tight / so: every
    variant 1272 / 1229 us, product epilogues alone 1737 / 1607; GPT-2 b32
    s512 5.38 / 5.38 ms, b1 the same within 1%. Two or three launches more in
    as much memory as they take were slower (1274 so, 1313 and 1325)."""
    apart = pack(compute_live_ranges(graph, replace(schedule, merged={})))[1]
    limit = max(tight[1], min(apart, STATIC_SLAB_BYTES) if cfg.static_arena else apart)
    rested = pack(ranges, _rested(schedule, ranges), limit)
    return rested if rested[1] <= limit else tight


def verify(ranges: list[LiveRange], offsets: dict[str, int]) -> list[str]:
    """Every pair of buffers live at one time that share a byte, described.
    Two lifetimes overlap exactly when both are live at the later start, so
    the check runs once per distinct start time over the buffers live then."""
    found: list[str] = []
    reported: set[tuple[str, str]] = set()
    for t in sorted({r.start for r in ranges}):
        live = sorted(((offsets[r.buffer.name], r) for r in ranges if r.start <= t <= r.end),
                      key=lambda e: e[0])
        for i, (off_a, a) in enumerate(live):
            for off_b, b in live[i + 1:]:
                if off_b >= off_a + a.size:
                    break
                if off_a >= off_b + b.size:  # b is empty and sits at a's start
                    continue
                pair = tuple(sorted((a.buffer.name, b.buffer.name)))
                if pair in reported:
                    continue
                reported.add(pair)
                found.append(f"{a.buffer.name} bytes [{off_a}, {off_a + a.size}) kernels "
                             f"[{a.start}, {a.end}] share memory with {b.buffer.name} bytes "
                             f"[{off_b}, {off_b + b.size}) kernels [{b.start}, {b.end}]")
    return found


def plan_memory(graph: Graph, schedule: Schedule, cfg: Config) -> AllocationPlan:
    """Place (or, with ``memory_planning`` off, schedule the allocation of)
    every intermediate; records the plan on ``schedule`` and each buffer."""
    ranges = compute_live_ranges(graph, schedule)
    plan = AllocationPlan(mode="arena" if cfg.memory_planning else "eager",
                          live_ranges={r.buffer.name: r for r in ranges},
                          peak_bytes=peak_live_bytes(ranges, len(schedule.kernels)),
                          total_bytes=sum(r.size for r in ranges))
    if plan.mode == "eager":
        for r in ranges:
            plan.alloc_at.setdefault(r.start, []).append(r.buffer)
            if r.end < len(schedule.kernels):
                plan.free_at.setdefault(r.end, []).append(r.buffer.name)
    else:
        plan.offsets, plan.arena_bytes = pack(ranges)
        if schedule.merged and cfg.static_arena and plan.arena_bytes > STATIC_SLAB_BYTES:
            # a group's outputs beside its inputs may be more than its product
            # beside either: its kernels one by one may still fit
            schedule.merged = {}
            return plan_memory(graph, schedule, cfg)
        if schedule.merged:
            plan.offsets, plan.arena_bytes = _pack_groups(graph, schedule, cfg, ranges,
                                                          (plan.offsets, plan.arena_bytes))
        clashes = verify(ranges, plan.offsets)
        if clashes:
            raise AssertionError("arena placement overlaps live buffers:\n" + "\n".join(clashes))
    for b in graph.buffers():
        b.arena_offset = plan.offsets.get(b.name)
    schedule.arena_bytes = plan.arena_bytes
    schedule.plan = plan
    return plan
