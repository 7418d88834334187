"""Native matrix products for the library calls of a schedule.

``aten.mm``, ``aten.addmm`` and ``aten.bmm`` stay extern kernels of the
schedule; up to the sizes where it was measured to be at least the library's
speed, the runtime runs one of the two templates of ``templates/mlc_gemm.h`` in
the library call's place (``plan_product`` decides, from sizes, strides and
types alone; the lines are ``TILED_FLOPS`` and its neighbours). Both accumulate in fp32 and round once
to the storage type, as the library does; ``addmm``'s bias is added before that
rounding.

* **tiled** (``gemm_tile``): both operands at unit stride along k, in aligned
  rows of whole 128-byte pieces -- a linear layer's activations and its
  ``[N, K]`` weight. Operands go straight from memory into an LDS ring.
* **staged** (``gemm_staged``): any strides, sizes and alignments, through
  registers into LDS -- attention's products over strided heads or odd lengths.

Measured in graphs of 24-48 products over 12 weights, fp16, library / tiled:
16x2048x512 (M x N x K) 3.6 / 2.0 us, 128x768x768 4.6 / 2.3, 128x3072x768
7.8 / 3.7, 128x768x3072 7.6 / 4.8, 525x768x768 7.3 / 4.0, 2048x2304x768
16.1 / 10.5, 2048x768x3072 19.0 / 14.9, 4096x3072x768 24.4 / 20.8,
16384x2304x768 70 / 58 (990 TFLOP/s, of 1340 that a large library product
reaches here). fp32: 128x3072x768 15.3 / 7.6, 128x768x3072 12.0 / 9.7,
1024x768x768 13.8 / 12.8.
"""

from __future__ import annotations

import math
from dataclasses import dataclass

import torch

from ..ir.graph import Value
from ..ir.scalar import Call
from ..kernels import ExternKernel
from .hip_backend import (MAX_THREADS, STORAGE, LaunchSpec, Renderer, _subexprs as subexprs,
                          fp16_rounded, half_inputs, itemsize, value_types_of)

CUS, XCDS = 256, 8
LDS_BYTES = 160 * 1024

#: tiled form: rows and columns of a workgroup's tile, waves across them, and
#: the k-splits tried
TILES = ((16, 16, 1, 1, (1, 2, 4)), (16, 32, 1, 2, (2, 4)), (16, 32, 1, 1, (3,)),
         (32, 32, 2, 2, (1, 2, 4)), (32, 48, 2, 1, (2, 4)), (32, 64, 2, 2, (1, 2)),
         (64, 64, 2, 2, (1, 2)), (64, 96, 2, 2, (1, 2)), (64, 128, 2, 4, (1,)),
         (96, 96, 2, 2, (1,)), (128, 96, 2, 2, (1,)), (128, 128, 2, 4, (1,)),
         (128, 192, 2, 4, (1,)), (128, 256, 2, 4, (1,)), (256, 256, 4, 2, (1,)))
#: floating-point operations up to which the tiled form is at least the
#: library's speed, by element size: fp16 16384x2304x768 58 us against 70,
#: 16384x3072x768 76 against 70; with long sums 8192x768x3072 39.6 against
#: 40.4, 16384x768x3072 70 against 65; fp32 2048x768x768 21 against 27, but
#: 525x768x3072 30 against 27
TILED_FLOPS, LONG_K, LONG_K_FLOPS = {2: 60e9, 4: 2.2e9}, 1024, 40e9
#: past this many columns (a vocabulary head) the weights are most of the
#: traffic and padded rows cost in full: 512x50257x768 fp16 62 us against 66
#: and 16 rows 16.0 against 17.8, but 333 rows 58 against 46, 64 rows 20.3
#: against 19.6, 1024 rows 124 against 117
WIDE, WIDE_FLOPS = 16384, 40e9
#: the line with pointwise kernels in the epilogue, against the library and
#: those kernels after it: 16384x3072x768 + bias + GELU 114 us in a layer
#: against 84 + 38; with long sums 16384x768x3072 + bias + residual 90 against
#: 73 + 12, 8192 rows 41 against 40 + 8
MERGED_FLOPS, MERGED_LONG_K_FLOPS = 80e9, 60e9
TRANSCENDENTAL = {"erf", "exp", "tanh", "sigmoid", "sin", "cos", "log", "pow"}


@dataclass(frozen=True)
class Operand:
    """A ``[batch, rows, k]`` view of a buffer (strides in elements)."""

    value: Value
    batch: int
    row: int
    k: int
    base: int

    def aligned(self, elements: int, batches: int) -> bool:
        """Every row starts on a multiple of ``elements``."""
        return (self.k == 1 and self.row % elements == 0 and self.base % elements == 0
                and (batches == 1 or self.batch % elements == 0))

    def columns_aligned(self, elements: int, batches: int) -> bool:
        """Rows at unit stride, every k's run of them starting on a multiple
        of ``elements``."""
        return (self.k != 1 and self.row == 1 and self.k % elements == 0
                and self.base % elements == 0 and (batches == 1 or self.batch % elements == 0))


@dataclass(frozen=True)
class Product:
    """``out[z, m, n] = sum_k a[z, m, k] b[z, n, k] (+ bias[n])``."""

    batches: int
    M: int
    N: int
    K: int
    a: Operand
    b: Operand
    out: Operand      # rows m, k-axis n
    bias: Value | None
    form: tuple       # ("tiled", TM, TN, WM, WN, WK, stages) or ("staged", TM, TN)


def _operand(v: Value, row_axis: int, k_axis: int) -> Operand:
    lay = v.layout
    return Operand(v, lay.strides[0] if len(v.shape) == 3 else 0, lay.strides[row_axis],
                   lay.strides[k_axis], lay.offset)


def tile_cost(M: int, N: int, K: int, batches: int, size: int, tile: tuple) -> float:
    """Microseconds of the tiled form in one launch, fitted to 1300 timings
    (median error 6%): a launch and its epilogue, the first load's latency once
    per round of workgroups, and for the busiest CU's tiles the larger of its
    LDS reads and its matrix instructions, plus its loads."""
    TM, TN, WM, WN, WK, stages = tile
    tiles = batches * -(-M // TM) * -(-N // TN)
    steps = K * size // 128 // WK
    ring = min(stages, steps) * WK * (TM + TN) * 128
    waves = WM * WN * WK
    together = max(1, min(LDS_BYTES // ring, 16 // waves))
    per_xcd = -(-tiles // XCDS)
    per_cu = -(-per_xcd // (CUS // XCDS))
    rounds = -(-per_xcd // (CUS // XCDS * together))
    loads = (TM + TN) * K * size
    reads = (TM * WN + TN * WM) * K * size
    macs = TM * TN * K * (1 if size == 2 else 8)
    simds = min(4, waves * min(together, per_cu))
    return (1.1 + 0.8 * rounds + per_cu * (max(2.95e-6 * reads, 4.33e-7 * macs * 4 / simds)
                                           + 5.66e-6 * loads + 6e-6 * TM * TN))


def choose_tile(M: int, N: int, K: int, batches: int, size: int,
                math: bool = False) -> tuple | None:
    """The cheapest tile by ``tile_cost``, with the deepest ring that fits LDS.

    In 16 bits, a product of more than one tile per CU takes tiles of at least
    128 x 128 (smaller ones reload A and B too often: 4096x2304x768 took 21.8 us
    in 128 x 96, 18.3 in 128 x 192), and a ring of half of LDS: two workgroups
    at a time, one's epilogue and first loads under the other's products.

    A large tile over a long sum takes eight waves: four, one a SIMD, leave its
    LDS reads uncovered (4096x768x3072 took 36 us in a layer in 128 x 96 by four
    waves, 27 in 128 x 128 by eight).

    ``math``: an epilogue with a transcendental. With more than one tile per CU
    none then takes more than half of LDS, so that its arithmetic runs beside
    another tile's products (16384x3072x768 + GELU 104 us in 128 x 192, 111 in
    256 x 256); below that a CU has no second tile to run it beside.

    In fp32 a k-split of 4 is kept up to 128 rows, where the library sums k in
    as many parts: fewer, longer sums would be further from float64 than it
    is (5.0e-7 relative against 2.5e-7 at K = 768)."""
    pieces = K * size // 128
    best = None
    for TM, TN, WM, WN, splits in TILES:
        if TM > max(16, 2 * M) or (K > LONG_K and TM * TN >= 128 * 96 and WM * WN < 8):
            continue
        crowded = size == 2 and -(-batches * -(-M // TM) * -(-N // TN) // XCDS) > CUS // XCDS
        small = crowded and TM * TN < 128 * 128
        fewest = 1
        if size == 4:
            fewest = (4 if M <= 128 else 2) if TM * TN <= 32 * 48 else 2 if TM * TN <= 64 * 96 else 1
        for WK in sorted({min(n, pieces) for n in splits}):
            if pieces % WK or WK < min(fewest, pieces):
                continue
            steps = pieces // WK

            def deepest(lds: int):
                return next((n for n in (4, 3, 2)
                             if min(n, steps) * WK * (TM + TN) * 128 <= lds), None)

            stages = (deepest(LDS_BYTES // 2) if crowded else None) or deepest(LDS_BYTES)
            if stages is None or (math and crowded and deepest(LDS_BYTES // 2) is None):
                continue
            tile = (TM, TN, WM, WN, WK, min(stages, max(2, steps)))
            rank = (small, tile_cost(M, N, K, batches, size, tile))
            if best is None or rank < best[0]:
                best = (rank, tile)
    return best[1] if best else None


#: staged form: operations up to which it is used, and the rows and columns of
#: its tile
STAGED_FLOPS = 2e9


def _line(M: int, N: int, K: int, size: int, merged_flops: float) -> float:
    """Operations up to which a product runs on the tiled form."""
    if N > WIDE:
        full = M >= 0.9 * 128 * -(-M // 128)
        return WIDE_FLOPS if size == 2 and (M <= 32 or full) else 0.0
    line = TILED_FLOPS[size]
    if size == 2:
        line = max(min(line, LONG_K_FLOPS) if K > LONG_K else line, merged_flops)
    return line


def plan_product(k: ExternKernel, merged_flops: float = 0.0, math: bool = False) -> Product | None:
    """How a library call's product runs natively, or ``None`` to leave it to
    the library. ``merged_flops``: the line where pointwise kernels run in its
    epilogue, which pays for itself where the product alone does not."""
    node = k.node
    op = node.op
    if op not in ("aten.mm.default", "aten.addmm.default", "aten.bmm.default") or node.kwargs:
        return None
    args, bias = list(node.args), None
    if op == "aten.addmm.default":
        bias, args = args[0], args[1:]
    if len(args) != 2 or len(node.outputs) != 1 or not all(isinstance(v, Value) for v in args):
        return None
    x, w = args
    out = node.outputs[0]
    rank = 3 if op == "aten.bmm.default" else 2
    if any(len(v.shape) != rank for v in (x, w, out)) or len({v.dtype for v in (x, w, out)}) != 1:
        return None
    if x.dtype not in (torch.float16, torch.bfloat16, torch.float32):
        return None
    M, K, N = x.shape[-2], x.shape[-1], w.shape[-1]
    batches = x.shape[0] if rank == 3 else 1
    if w.shape[-2] != K or tuple(out.shape[-2:]) != (M, N) or min(M, N, K, batches) < 1:
        return None
    if bias is not None and not (isinstance(bias, Value) and tuple(bias.shape) == (N,)
                                 and bias.dtype == x.dtype and (N == 1 or bias.layout.strides[0] == 1)):
        return None
    operands = [v for v in (x, w, out, bias) if v is not None]
    if any(v.buffer.numel >= 2 ** 31 or min(v.layout.strides, default=0) < 0 for v in operands):
        return None
    a, b, c = _operand(x, -2, -1), _operand(w, -1, -2), _operand(out, -2, -1)
    if N > 1 and c.k != 1:
        return None
    size = itemsize(x.dtype)
    flops = 2.0 * batches * M * N * K
    E = 16 // size
    if (K * size % 128 == 0 and flops <= _line(M, N, K, size, merged_flops)
            and a.aligned(E, batches) and b.aligned(E, batches)):
        tile = choose_tile(M, N, K, batches, size, math)
        if tile is not None:
            return _launchable(Product(batches, M, N, K, a, b, c, bias, ("tiled", *tile)))
    if rank == 3 and flops <= STAGED_FLOPS:
        return _launchable(Product(batches, M, N, K, a, b, c, bias,
                                   ("staged", *staged_tile(M, N, batches))))
    return None


def _launchable(p: Product) -> Product | None:
    """``p`` unless its grid has more threads than HIP launches."""
    src = _Source(p)
    return p if src.grid * src.threads < MAX_THREADS else None


def staged_tile(M: int, N: int, batches: int) -> tuple[int, int]:
    """64 x 64, or 32 wide along an axis where 64 leaves half of the chip idle."""
    TM = TN = 64
    if batches * -(-M // 64) * -(-N // 64) < CUS:
        TM = 32
        if batches * -(-M // 32) * -(-N // 64) < CUS:
            TN = 32
    return TM, TN


@dataclass(frozen=True)
class _Source:
    """The pieces of a product's kernel around its epilogue."""

    p: Product

    @property
    def storage(self) -> str:
        return STORAGE[self.p.a.value.dtype]

    @property
    def tile(self) -> tuple[int, int]:
        return self.p.form[1], self.p.form[2]

    @property
    def threads(self) -> int:
        return 64 * math.prod(self.p.form[3:6]) if self.p.form[0] == "tiled" else 256

    @property
    def grid(self) -> int:
        return XCDS * -(-self.p.batches * self._tiles[0] * self._tiles[1] // XCDS)

    @property
    def _tiles(self) -> tuple[int, int]:
        return -(-self.p.M // self.tile[0]), -(-self.p.N // self.tile[1])

    def head(self, params: list[str]) -> list[str]:
        p, T = self.p, self.storage
        params = [f"const {T}* __restrict__ a", f"const {T}* __restrict__ b", *params]
        L = [f"extern \"C\" __global__ void __launch_bounds__({self.threads}) "
             f"KERNEL({', '.join(params)}) {{",
             f"  // {p.form[0]}: {p.batches} x [{p.M} x {p.K}] x [{p.K} x {p.N}], "
             f"{self.tile[0]} x {self.tile[1]} tiles",
             "  int z, mt, nt;",
             f"  if (!mlc::tile_index<{p.batches}, {self._tiles[0]}, {self._tiles[1]}>(z, mt, nt)) return;"]
        return L + [self.move("a", p.a), self.move("b", p.b)]

    def move(self, name: str, o: Operand) -> str:
        """``name`` at this batch's first element."""
        return f"  {name} += (int64_t)z * {o.batch if self.p.batches > 1 else 0} + {o.base};"

    def tail(self, transposed: str = "false", store_t: str = "store") -> list[str]:
        p, T = self.p, self.storage
        (TM, TN), E = self.tile, 16 // itemsize(p.a.value.dtype)
        if p.form[0] == "tiled":
            return [f"  mlc::gemm_tile<{T}, {p.M}, {p.N}, {p.K}, {p.a.row}, {p.b.row}, "
                    f"{', '.join(map(str, p.form[1:]))}>(a, b, mt * {TM}, nt * {TN}, store, "
                    f"{transposed}, {store_t});", "}"]
        flags = ", ".join(str(o.aligned(E, p.batches) or o.columns_aligned(E, p.batches)).lower()
                          for o in (p.a, p.b))
        return [f"  mlc::gemm_staged<{T}, {p.M}, {p.N}, {p.K}, {p.a.row}, {p.a.k}, {p.b.row}, {p.b.k}, "
                f"{TM}, {TN}, {8 * E}, {flags}>(a, b, mt * {TM}, nt * {TN}, store);", "}"]

    def spec(self, kind: str, values: list[Value]) -> LaunchSpec:
        return LaunchSpec("", self.grid, self.threads, 0,
                          {"kind": kind, "form": self.p.form,
                           "buffers": [v.buffer.name for v in values],
                           "dtypes": [v.buffer.dtype for v in values],
                           "numels": [v.buffer.numel for v in values]})


def emit_product(k: ExternKernel) -> tuple[str, LaunchSpec] | None:
    """Source (with the placeholder name ``KERNEL``) and launch spec of a
    library call's native product, or ``None``."""
    p = plan_product(k)
    if p is None:
        return None
    src = _Source(p)
    T = src.storage
    packed = p.N % 4 == 0 and p.out.aligned(4, p.batches)
    params = [f"const {T}* __restrict__ bias"] if p.bias is not None else []
    L = src.head(params + [f"{T}* __restrict__ c"])
    L += [src.move("c", p.out),
          "  auto store = [&](int m, int n, mlc::float4v s) {",
          "    float v[4] = {s[0], s[1], s[2], s[3]};"]
    if p.bias is not None:
        L += ["#pragma unroll",
              f"    for (int i = 0; i < 4; ++i) if (n + i < {p.N}) "
              f"v[i] += mlc::ld(bias + {p.bias.layout.offset} + n + i);"]
    L += [f"    mlc::store4<{T}, {p.M}, {p.N}, {p.out.row}, {str(packed).lower()}>(c, m, n, v);",
          "  };"]
    values = [p.a.value, p.b.value, *([p.bias] if p.bias is not None else []), p.out.value]
    return "\n".join(L + src.tail()), src.spec("gemm", values)


# --------------------------------------------------------------------------
# products with the pointwise kernels after them
# --------------------------------------------------------------------------

def plan_group(k: ExternKernel, parts) -> Product | None:
    """The product of a group that runs as one launch (``passes/products``),
    or ``None`` where the kernels stay apart."""
    if any(a.buffer.numel >= 2 ** 31 for part in parts
           for a in (*part.kernel.inputs, *part.kernel.outputs)):
        return None
    calls = {e.fn for part in parts for _, x in part.kernel.body for e in subexprs(x)
             if isinstance(e, Call)}
    K = k.node.args[0].shape[-1]
    return plan_product(k, MERGED_LONG_K_FLOPS if K > LONG_K else MERGED_FLOPS,
                        bool(calls & TRANSCENDENTAL))


def _place(terms, var: str) -> str:
    """Index of an output element from one coordinate (``Part.m_terms``),
    in unsigned arithmetic: most sizes are powers of two, so their divisions
    are shifts."""
    top = max((size * step for size, step, _ in terms), default=1)
    parts = []
    for size, step, stride in terms:
        t = var if step == 1 else f"{var} / {step}u"
        t = t if size * step == top else f"{t} % {size}u"
        parts.append(f"({t}) * {stride}u")
    return " + ".join(parts) or "0u"


def _transposed(part, p: Product) -> bool:
    """Whether a part's stores run along the rows of whole tiles (a per-head V
    transposed for the attention): four rows of a column go out together."""
    TM, TN, WK = p.form[1], p.form[2], p.form[5]
    inner = next((t for t in part.m_terms if t[1] == 1), (1, 1, 0))
    others = [t for t in (*part.m_terms, *part.n_terms) if t is not inner]
    return (WK == 1 and p.M % 4 == 0 and inner[2] == 1 and inner[0] % 4 == 0
            and all(t[2] % 4 == 0 for t in others) and _whole_tiles(part, TN, p.N))


def _whole_tiles(part, TN: int, N: int) -> bool:
    return part.lo % TN == 0 and (part.hi % TN == 0 or part.hi == N)


def _in_part(part, N: int, TN: int) -> str:
    """The test for a part's columns: where they are whole tiles, one scalar
    branch per workgroup."""
    if part.lo == 0 and part.hi == N:
        return "true"
    if _whole_tiles(part, TN, N):
        return f"nt >= {part.lo // TN} && nt < {-(-part.hi // TN)}"
    return f"n >= {part.lo} && n < {part.hi}"


def _part_lines(part, i: int, N: int, TN: int, along_m: bool = False) -> list[str]:
    """One pointwise kernel's work on four consecutive columns of row ``m`` from
    ``n`` (four consecutive rows of column ``n`` from ``m``): ``x`` holds the
    product, already rounded to its storage type."""
    k = part.kernel
    out = k.outputs[0]
    L = [f"    if ({_in_part(part, N, TN)}) {{", f"      const uint32_t q = n - {part.lo}, row = m;"]
    names: list[str] = []
    for slot, (a, read) in enumerate(zip(k.inputs, part.reads)):
        if read is None:
            names.append("x[j]")
            continue
        step = read.row if along_m else read.col
        at = f"p{i}_{slot} + (row * {read.row}u + {read.base}u" + (" + q)" if read.col else ")")
        if step:
            packed = step == 1 and read.row % 4 == 0 and read.base % 4 == 0
            L.append(f"      float v{slot}[4];" + (f" mlc::load_pack<4>(v{slot}, {at});" if packed else
                     f" for (int j = 0; j < 4; ++j) v{slot}[j] = mlc::ld({at} + j * {step});"))
            names.append(f"v{slot}[j]")
        else:
            L.append(f"      const float v{slot} = mlc::ld({at});")
            names.append(f"v{slot}")
    types: dict[str, str] = {}
    r = Renderer(lambda s: (names[s], "float"), lambda n: (n, types[n]), half_inputs(k), dict(k.body),
                 fp16_rounded(k), value_types_of(k))
    L += ["      float o[4];", "#pragma unroll", "      for (int j = 0; j < 4; ++j) {"]
    for name, expr in k.body:
        code, types[name] = r.bind(name, expr)
        L.append(f"        const {types[name]} {name} = {code};")
    code, _ = r.store(k.out_expr[out.value.name], out.dtype == torch.float16)
    inner = next((t for t in part.n_terms if t[1] == 1), (1, 1, 1))
    terms = (*part.m_terms, *part.n_terms)
    packed = along_m or (inner[2] == 1 and inner[0] % 4 == 0
                         and all(t is inner or t[2] % 4 == 0 for t in terms))
    L += [f"        o[j] = {code};", "      }"]
    if not along_m and inner[0] % 4:  # the four columns may run on into the next digit
        return L + ["#pragma unroll", "      for (int j = 0; j < 4; ++j)",
                    f"        mlc::st(o{i} + (({_place(part.m_terms, 'row')}) "
                    f"+ ({_place(part.n_terms, '(q + j)')})), o[j]);", "    }"]
    L.append(f"      {STORAGE[out.dtype]}* w = o{i} + (({_place(part.m_terms, 'row')}) "
             f"+ ({_place(part.n_terms, 'q')}));")
    if packed:
        L.append("      mlc::store_pack<4>(w, o);")
    else:
        L += ["#pragma unroll",
              f"      for (int j = 0; j < 4; ++j) mlc::st(w + j * {inner[2]}, o[j]);"]
    return L + ["    }"]


def emit_group(k: ExternKernel, parts) -> tuple[str, LaunchSpec]:
    """A product and the pointwise kernels after it as one kernel."""
    p = plan_group(k, parts)
    src = _Source(p)
    T = src.storage
    params, values = [], [p.a.value, p.b.value]
    for i, part in enumerate(parts):
        for slot, (a, read) in enumerate(zip(part.kernel.inputs, part.reads)):
            if read is not None:
                params.append(f"const {STORAGE[a.dtype]}* __restrict__ p{i}_{slot}")
                values.append(a.value)
        out = part.kernel.outputs[0]
        params.append(f"{STORAGE[out.dtype]}* __restrict__ o{i}")
        values.append(out.value)
    L = src.head(params)
    turned = {i for i, part in enumerate(parts) if p.form[0] == "tiled" and _transposed(part, p)}

    def epilogue(name: str, which, along_m: bool) -> list[str]:
        lines = [f"  auto {name} = [&](int m, int n, mlc::float4v s) {{"]
        if p.M % src.tile[0] or p.N % src.tile[1]:
            lines.append(f"    if (m >= {p.M} || n >= {p.N}) return;")
        lines.append("    const float x[4] = {"
                     + ", ".join(f"mlc::ld_of<{T}>(s[{j}])" for j in range(4)) + "};")
        for i, part in enumerate(parts):
            if i in which:
                lines += _part_lines(part, i, p.N, src.tile[1], along_m)
        return lines + ["  };"]

    # a workgroup whose columns belong to turned parts alone stores along m
    mixed = [i for i in range(len(parts)) if i not in turned]
    clear = all(parts[i].hi <= parts[t].lo or parts[i].lo >= parts[t].hi
                for i in mixed for t in turned)
    if not turned or not clear:
        L += epilogue("store", range(len(parts)), False)
        return "\n".join(L + src.tail()), src.spec("gemm+pointwise", values)
    L += epilogue("store", mixed, False) + epilogue("store_t", turned, True)
    test = " || ".join(f"({_in_part(parts[t], p.N, src.tile[1])})" for t in sorted(turned))
    return "\n".join(L + src.tail(test, "store_t")), src.spec("gemm+pointwise", values)
