"""Load and launch the generated HIP module through ``libmlc_hip.so``.

The counterpart of the reference's ``TritonRuntime``
(``mlc/runtime/triton_runtime.py:60-97``) behind the same seam: it is built
from a schedule, exposes ``source`` (the module text, a ``str``), ``path``
(where that text was written) and ``launch_table``, resolves a
kernel against the buffer table once (``bind``) and launches it
(``launch``/``run_bound``) on torch's current stream. On top of that it owns
the per-model native state the MI355X design adds:

* one context per compiled model (device binding, the arena slab, the graph);
* the arena as one ``hipMalloc`` slab, handed to torch through DLPack so the
  extern library calls write into the same memory (``arena``);
* the pre-resolved plan as a native launch table: consecutive generated
  kernels run as one ``mlc_plan_run`` call (``compile_runs``);
* hipGraph capture and replay of the whole schedule (``capture_begin``,
  ``capture_end``, ``replay``);
* hipEvent timing of one bound kernel in place (``time_bound``);
* the invalid-input word: the native embedding gather flags an id outside
  its table there (torch raises ``IndexError`` for one). It is coherent host
  memory, so a pass enqueues nothing for it and ``pending_error`` reads it
  without waiting for the device;
* the caller's inputs: read where they are by launches made one by one
  (``bind_inputs``, ``call``), or copied in by one launch in front of the graph
  (``graph_call``).
"""

from __future__ import annotations

import ctypes
import struct
from dataclasses import dataclass

import torch

from ..codegen.hip_backend import LaunchSpec, build_module, build_products
from ..config import Config
from ..kernels import ExternKernel, Kernel, Schedule
from . import native

_CAPSULE_NAME = b"dltensor"
_PyCapsule_New = ctypes.pythonapi.PyCapsule_New
_PyCapsule_New.restype = ctypes.py_object
_PyCapsule_New.argtypes = [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]


@dataclass
class Bound:
    """One generated kernel resolved against the buffer table."""

    name: str
    fn: int
    grid: int
    block: int
    lds: int
    args: bytes


@dataclass
class Range:
    """Entries ``[begin, end)`` of the native launch plan."""

    plan: int
    begin: int
    end: int


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _on_16_bytes(spec: LaunchSpec | None, buffers: dict[str, torch.Tensor]) -> bool:
    return spec is not None and all(buffers[n].data_ptr() % 16 == 0 for n in spec.meta["buffers"])


class HipRuntime:
    name = "hip"

    def __init__(self, schedule: Schedule, cfg: Config, device: torch.device) -> None:
        if device.type != "cuda":
            raise native.NativeError(f"HipRuntime needs a ROCm GPU device, got {device}")
        self.device = device
        self.index = device.index if device.index is not None else torch.cuda.current_device()
        self.lib = native.load_library()
        self.module = build_module(schedule, cfg)
        #: the generated HIP module text (``TritonRuntime.source``)
        self.source: str = self.module.source
        self.launch_table: dict[str, LaunchSpec] = self.module.launches
        #: library products that run natively, by kernel name; their module
        #: is loaded beside the generated one when there are any
        products, self.group_table = build_products(schedule)
        self.product_table: dict[str, LaunchSpec] = products.launches
        objects = native.compile_code_objects(
            [self.source] + ([products.source] if products.functions else []))
        self.path, self.code_object_path = objects[0]

        self._ctx = ctypes.c_void_p()
        native.check(self.lib.mlc_ctx_create(self.index, ctypes.byref(self._ctx)), "mlc_ctx_create")
        self._mods: list[ctypes.c_void_p] = []
        self.functions: dict[str, int] = {}
        for (_, path), table in zip(objects, (self.launch_table,
                                              {**self.product_table, **self.group_table})):
            self._load(path.read_bytes(), sorted({s.symbol for s in table.values()}))
        self._plans: list[ctypes.c_void_p] = []
        #: native plan -> its launches, by entry
        self._launches: dict[int, list[Bound]] = {}
        self._arena_tensor: torch.Tensor | None = None
        self._static_arena = bool(getattr(cfg, "static_arena", False))
        #: device address of the context's invalid-input word, if a kernel
        #: of this module can flag one (the native embedding gather)
        self._error_word: int | None = None
        if any(spec.meta.get("error_word") for spec in self.launch_table.values()):
            word = ctypes.c_void_p()
            native.check(self.lib.mlc_error_word(self._ctx, ctypes.byref(word)), "mlc_error_word")
            self._error_word = word.value

    def _load(self, image: bytes, symbols: list[str]) -> None:
        mod = ctypes.c_void_p()
        buf = ctypes.create_string_buffer(image, len(image))
        native.check(self.lib.mlc_module_load(self._ctx, buf, len(image), ctypes.byref(mod)),
                     "mlc_module_load")
        self._mods.append(mod)
        for symbol in symbols:
            fn = ctypes.c_void_p()
            native.check(self.lib.mlc_function(mod, symbol.encode(), ctypes.byref(fn)),
                         f"mlc_function({symbol})")
            self.functions[symbol] = fn.value

    # -- the reference seam ---------------------------------------------------

    def bind(self, k: Kernel, buffers: dict[str, torch.Tensor]) -> Bound:
        """Resolve a launch once: function handle, geometry and the packed
        kernel arguments (``in0..in{n-1}, out0..out{m-1}`` buffer base
        pointers, ``mlc/runtime/triton_runtime.py:67-83``)."""
        if isinstance(k, ExternKernel):
            raise TypeError("extern kernels do not go through the HIP runtime")
        spec = self.launch_table[k.name]
        ptrs = []
        for a in list(k.inputs) + list(k.outputs):
            t = buffers[a.value.buffer.name]
            if t.device.type != "cuda":
                raise native.NativeError(f"{k.name}: buffer {a.value.buffer.name} is on {t.device}")
            if t.dtype != a.value.buffer.dtype or t.numel() < a.value.buffer.numel:
                raise native.NativeError(
                    f"{k.name}: buffer {a.value.buffer.name} is {t.dtype}[{t.numel()}], the kernel "
                    f"was generated for {a.value.buffer.dtype}[{a.value.buffer.numel}]")
            if t.data_ptr() % 16:
                raise native.NativeError(f"{k.name}: buffer {a.value.buffer.name} is not 16-byte "
                                         "aligned; the kernel's packed accesses assume it is")
            ptrs.append(t.data_ptr())
        args = struct.pack(f"<{len(ptrs)}Q", *ptrs)
        return Bound(k.name, self.functions[spec.symbol], spec.grid, spec.block, spec.lds_bytes,
                     args)

    def bind_native_extern(self, k: ExternKernel, buffers: dict[str, torch.Tensor]) -> Bound | None:
        """An extern op this module implements natively (``aten.embedding``),
        resolved like a generated kernel; ``None`` leaves it to the library."""
        return self._bind_extern(k, self.launch_table.get(k.name), buffers)

    def bind_product(self, k: ExternKernel, buffers: dict[str, torch.Tensor]) -> Bound | None:
        """A matrix product this module runs in the library's place, resolved
        like a generated kernel; ``None`` leaves it to the library, whose
        operands may lie anywhere (a weight at an odd place in flat storage)."""
        spec = self.product_table.get(k.name)
        return self._bind_extern(k, spec, buffers) if _on_16_bytes(spec, buffers) else None

    def bind_group(self, k: ExternKernel, buffers: dict[str, torch.Tensor]) -> Bound | None:
        """The group of kernels starting at ``k`` that runs as one launch;
        ``None`` leaves its kernels apart, as ``bind_product`` does."""
        spec = self.group_table[k.name]
        return self._bind_extern(k, spec, buffers) if _on_16_bytes(spec, buffers) else None

    def _bind_extern(self, k: ExternKernel, spec: LaunchSpec | None,
                     buffers: dict[str, torch.Tensor]) -> Bound | None:
        if spec is None:
            return None
        ptrs = []
        for name, dtype, numel in zip(spec.meta["buffers"], spec.meta["dtypes"],
                                      spec.meta["numels"]):
            t = buffers[name]
            if t.device.type != "cuda" or t.dtype != dtype or t.numel() < numel:
                raise native.NativeError(f"{k.name}: buffer {name} is {t.dtype}[{t.numel()}] on "
                                         f"{t.device}, expected {dtype}[{numel}] on the GPU")
            if t.data_ptr() % 16:
                raise native.NativeError(f"{k.name}: buffer {name} is not 16-byte aligned")
            ptrs.append(t.data_ptr())
        if spec.meta.get("error_word"):
            ptrs.append(self._error_word)
        return Bound(k.name, self.functions[spec.symbol], spec.grid, spec.block, spec.lds_bytes,
                     struct.pack(f"<{len(ptrs)}Q", *ptrs))

    # -- invalid inputs ------------------------------------------------------------
    @property
    def flags_errors(self) -> bool:
        """Whether a kernel of this module can flag an invalid input."""
        return self._error_word is not None

    def fetch_errors(self, stream: int | None = None) -> None:
        """Nothing to enqueue: the word is host memory that kernels write. Kept
        for callers of the time when a run copied it back."""

    def pending_error(self) -> str | None:
        """The message for an invalid input flagged by a completed run, read
        without waiting for the device; ``None`` if no completed run flagged
        one. Runs still in flight are seen by a later call."""
        if self._error_word is None:
            return None
        value = ctypes.c_int32()
        native.check(self.lib.mlc_error_poll(self._ctx, ctypes.byref(value)), "mlc_error_poll")
        if value.value == 0:
            return None
        return ("an embedding id was outside its table (torch raises IndexError for such an "
                "id); the rows it addressed were written as zeros")

    def clear_errors(self) -> None:
        """Wait for the device, then zero the word."""
        if self._error_word is not None:
            native.check(self.lib.mlc_error_clear(self._ctx), "mlc_error_clear")

    def check_errors(self) -> None:
        """Synchronize and raise :class:`native.NativeError` if any run so far
        flagged an invalid input (clearing the flag)."""
        if self._error_word is None:
            return
        torch.cuda.synchronize(self.device)
        msg = self.pending_error()
        if msg is not None:
            self.clear_errors()
            raise native.NativeError(msg)

    def launch(self, k: Kernel, buffers: dict[str, torch.Tensor]) -> None:
        self.run_bound(self.bind(k, buffers))

    def run_bound(self, payload) -> None:
        if isinstance(payload, Bound) and payload.grid == 0:
            return  # a reduction over zero rows: nothing to launch
        if isinstance(payload, Range):
            native.check(self.lib.mlc_plan_run(payload.plan, payload.begin, payload.end, _stream()),
                         "mlc_plan_run")
            return
        native.check(self.lib.mlc_launch(payload.fn, payload.grid, payload.block, payload.lds,
                                         payload.args, len(payload.args), _stream()),
                     f"mlc_launch({payload.name})")

    # -- the pre-resolved plan ----------------------------------------------------
    def compile_runs(self, plan: list) -> list:
        """Turn ``[(kind, payload)]`` into runs where every maximal sequence of
        generated kernels is one ``Range`` of a native launch plan."""
        def native_of(kind, payload):
            if kind == "kernel":
                return payload if payload.grid else None
            if kind == "extern" and getattr(payload, "module", None) is self:
                return payload.bound  # a library op this module claimed
            return None

        kernels = [b for b in (native_of(kind, p) for kind, p in plan) if b is not None]
        handle = ctypes.c_void_p()
        native.check(self.lib.mlc_plan_create(self._ctx, len(kernels), ctypes.byref(handle)),
                     "mlc_plan_create")
        self._plans.append(handle)
        self._launches[handle.value] = kernels
        for i, b in enumerate(kernels):
            native.check(self.lib.mlc_plan_set(handle, i, b.fn, b.grid, b.block, b.lds, b.args,
                                               len(b.args)), "mlc_plan_set")
        runs: list = []
        i = 0
        for kind, payload in plan:
            if native_of(kind, payload) is not None:
                if runs and runs[-1][0] == "kernel":
                    runs[-1][1].end = i + 1
                else:
                    runs.append(("kernel", Range(handle.value, i, i + 1)))
                i += 1
            else:
                runs.append((kind, payload))
        return runs

    def bind_inputs(self, runs: list, addresses: dict[int, int]) -> None:
        """Let ``call`` replace the buffers at ``addresses`` (address of an
        input's own buffer -> the input's position) wherever a launch of
        ``runs`` reads them."""
        for kind, payload in runs:
            if kind != "kernel":
                continue
            for i in range(payload.begin, payload.end):
                args = self._launches[payload.plan][i].args
                for at, (ptr,) in enumerate(struct.iter_unpack("<Q", args)):
                    if ptr in addresses:
                        native.check(self.lib.mlc_plan_input(payload.plan, i, 8 * at,
                                                             addresses[ptr]), "mlc_plan_input")

    def call(self, runs: list, inputs, stream: int) -> None:
        """Launch ``runs`` one by one on the given input addresses."""
        n = len(inputs)
        ptrs = (ctypes.c_void_p * n)(*inputs)
        for kind, payload in runs:
            if kind == "kernel":
                native.check(self.lib.mlc_plan_call(payload.plan, payload.begin, payload.end, ptrs,
                                                    n, stream), "mlc_plan_call")
            elif kind == "extern":
                payload.run()

    # -- arena -----------------------------------------------------------------
    def arena(self, nbytes: int) -> torch.Tensor:
        """The arena: one ``hipMalloc`` slab of at least ``nbytes``, or with
        ``Config(static_arena=True)`` the library's static device array
        (``mlc_slab_static``, nothing allocated), as a uint8 tensor that
        aliases it (DLPack, no copy)."""
        if self._arena_tensor is not None and self._arena_tensor.numel() >= nbytes:
            return self._arena_tensor
        self._arena_tensor = None
        ptr = ctypes.c_void_p()
        if self._static_arena:
            native.check(self.lib.mlc_slab_static(self._ctx, nbytes, ctypes.byref(ptr)),
                         "mlc_slab_static")
        else:
            native.check(self.lib.mlc_slab_alloc(self._ctx, nbytes, ctypes.byref(ptr)),
                         "mlc_slab_alloc")
        managed = ctypes.c_void_p()
        native.check(self.lib.mlc_slab_dlpack(self._ctx, ctypes.byref(managed)), "mlc_slab_dlpack")
        capsule = _PyCapsule_New(managed, _CAPSULE_NAME, None)
        t = torch.utils.dlpack.from_dlpack(capsule)
        if t.data_ptr() != ptr.value or t.device.type != "cuda":
            raise native.NativeError("the slab's DLPack export does not alias the slab")
        self._arena_tensor = t
        return t

    # -- graph -----------------------------------------------------------------
    def capture_begin(self, stream: int) -> None:
        native.check(self.lib.mlc_graph_begin(self._ctx, stream), "mlc_graph_begin")

    def capture_end(self) -> None:
        native.check(self.lib.mlc_graph_end(self._ctx), "mlc_graph_end")

    def replay(self, stream: int) -> None:
        native.check(self.lib.mlc_graph_replay(self._ctx, stream), "mlc_graph_replay")

    #: copies ``graph_call`` takes at once
    MAX_COPIES = 8

    def graph_call(self, copies: list[tuple[int, int, int]], stream: int) -> None:
        """``(dst, src, bytes)`` device copies as one launch, then the graph."""
        n = len(copies)
        dst, src = (ctypes.c_void_p * n)(), (ctypes.c_void_p * n)()
        size = (ctypes.c_size_t * n)()
        for i, (d, s, b) in enumerate(copies):
            dst[i], src[i], size[i] = d, s, b
        native.check(self.lib.mlc_graph_call(self._ctx, n, dst, src, size, stream), "mlc_graph_call")

    def graph_nodes(self) -> int:
        n = ctypes.c_size_t()
        native.check(self.lib.mlc_graph_node_count(self._ctx, ctypes.byref(n)),
                     "mlc_graph_node_count")
        return n.value

    # -- profiling -------------------------------------------------------------
    def time_bound(self, payload: Bound, iters: int, stream: int) -> float:
        """Average ms of ``iters`` back-to-back launches of one bound kernel,
        timed with hipEvents on ``stream``."""
        if payload.grid == 0:
            return 0.0
        handle = ctypes.c_void_p()
        native.check(self.lib.mlc_plan_create(self._ctx, 1, ctypes.byref(handle)), "mlc_plan_create")
        try:
            native.check(self.lib.mlc_plan_set(handle, 0, payload.fn, payload.grid, payload.block,
                                               payload.lds, payload.args, len(payload.args)),
                         "mlc_plan_set")
            ms = ctypes.c_float()
            native.check(self.lib.mlc_time_entry(handle, 0, iters, stream, ctypes.byref(ms)),
                         "mlc_time_entry")
            return float(ms.value)
        finally:
            self.lib.mlc_plan_destroy(handle)

    def synchronize(self) -> None:
        native.check(self.lib.mlc_device_synchronize(self._ctx), "mlc_device_synchronize")

    def close(self) -> None:
        lib = self.lib
        for p in self._plans:
            lib.mlc_plan_destroy(p)
        self._plans = []
        self._arena_tensor = None
        # the context owns the graph that names the module's functions: it goes first
        if getattr(self, "_ctx", None) is not None and self._ctx.value:
            lib.mlc_ctx_destroy(self._ctx)
            self._ctx = None
        for mod in getattr(self, "_mods", []):
            lib.mlc_module_unload(mod)
        self._mods = []

    def __del__(self) -> None:
        try:
            self.close()
        except Exception:
            pass
