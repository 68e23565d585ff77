"""The launcher ``matmul`` and the BLAS-like ``matmatmul_`` / ``mul_`` (reference src/matmul.jl;
Julia's ``matmatmul!`` / ``mul!`` lose their ``!`` in Python).

Device arrays are torch CUDA tensors in COLUMN-MAJOR order like Julia's CuArrays: a logical
(rows, cols) matrix is a tensor with ``stride(0) == 1`` (see ``gemmkernels.colmajor``).  torch is
only the owner of the memory and of the stream; every flop runs in libgemmkernels_hip.so.
"""
from __future__ import annotations

import contextlib
import ctypes
import math
from typing import Optional

import numpy as np

from . import _lib
from . import cta_swizzle as CTASwizzle
from . import epilogue as Epilogue
from . import kernel as Kernel
from . import layout as Layout
from . import operator as Operator
from . import transform as Transform
from .config import _MFMA_TILE_COST, Config, _mfma_cost, default_block_shape, get_config as _get_config, larger_tile, product_block_shape, sliced_block_shape, split_k_block_shape
from .config import _product_slices
from .dtypes import BFloat16, DType, Float16, Float32, Float64, from_torch, promote_type
from .errors import ConfigError, DimensionMismatch
from ._native import Prepared, load as load_native
from .tiling import NT

_HOOKS = ("transform_global_to_shared_a", "transform_global_to_shared_b", "transform_global_to_shared_c",
          "transform_shared_to_global_d", "transform_shared_to_regs_a", "transform_shared_to_regs_b",
          "transform_shared_to_regs_c", "transform_regs_to_shared_d")


def _ptr(x) -> Optional[int]:
    if x is None:
        return None
    if isinstance(x, int):
        return x
    return int(x.data_ptr())


_NO_LD = (Layout.ZERO, Layout.DIAGONAL, Layout.GETT_KIND)
_INTERLEAVED = (Layout.INTERLEAVED_COL_MAJOR, Layout.INTERLEAVED_ROW_MAJOR)


_SPLIT = (Layout.SPLIT_COL_MAJOR, Layout.SPLIT_ROW_MAJOR)


def _leading_dim(x, layout) -> int:
    """Leading dimension, in elements, of a column-major device matrix."""
    kind = layout.kind
    if x is None or kind in _NO_LD or isinstance(x, int):
        return 0
    shape, stride = x.shape, x.stride()
    if kind in _INTERLEAVED:
        # interleaved complex data: a real tensor of logical shape (2, rows, cols), column-major,
        # or a complex tensor of shape (rows, cols); the leading dimension counts complex elements
        if x.is_complex():
            if len(shape) != 2 or (shape[0] > 1 and stride[0] != 1):
                raise ConfigError("complex operands must be column-major matrices")
            return int(stride[1]) if shape[1] > 1 else max(int(shape[0]), 1)
        if len(shape) != 3 or shape[0] != 2 or stride[0] != 1 or (shape[1] > 1 and stride[1] != 2):
            raise ConfigError("interleaved complex operands must have shape (2, rows, cols) in column-major order")
        return int(stride[2]) // 2 if shape[2] > 1 else max(int(shape[1]), 1)
    if kind in _SPLIT:
        # planar complex data: a real tensor of logical shape (rows, cols, 2), column-major, the
        # imaginary plane right behind the real one
        if len(shape) != 3 or shape[2] != 2 or (shape[0] > 1 and stride[0] != 1) or stride[2] != stride[1] * shape[1]:
            raise ConfigError("planar complex operands must have shape (rows, cols, 2) in column-major order")
        return int(stride[1])
    if len(shape) != 2:
        raise ConfigError("matrix operands must be 2-dimensional")
    if shape[0] > 1 and stride[0] != 1:
        raise ConfigError("matrix operands must be column-major (stride(0) == 1); see gemmkernels.colmajor")
    return int(stride[1]) if shape[1] > 1 else max(int(shape[0]), 1)


def _current_stream() -> int:
    """Raw handle of torch's current HIP stream."""
    import torch
    if _native is not None:
        return _native.current_stream()
    try:
        return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())
    except AttributeError:
        return torch.cuda.current_stream().cuda_stream


_native = None              # the module gk_torch, once a call has been made (None as well where it is not built)


def _gk_matmul(conf_c, a, b, c, d, trans, epi, code: int, stream: int) -> int:
    """gk_matmul on descriptors and addresses; its status."""
    if _native is not None:
        return _native.matmul(ctypes.addressof(conf_c), a, b, c, d, None if trans is None else ctypes.addressof(trans), None if epi is None else ctypes.addressof(epi), code, stream)
    return _lib.lib().gk_matmul(ctypes.byref(conf_c), a, b, c, d, ctypes.byref(trans) if trans is not None else None,
                                ctypes.byref(epi) if epi is not None else None, code, stream)


_workspaces = {}            # (device, stream) -> buffer of eager launches
_recorded = {}              # (device, stream) -> buffers of graphs captured without torch
_pool_of_capture = {}       # (device, stream, capture) -> whether torch keeps the capture's memory for the graph
_COUNTER_BYTES = 2048       # arrival counters at the head of a workspace (kSplitCounterBytes of the library)


def split_k_workspace(conf_c, stream: int):
    """Device workspace for a K-split launch of ``conf_c`` on ``stream``, as a byte tensor (None: the product runs
    unsplit).  The slices of an output tile leave their partial tiles there and the last one to arrive adds them
    up in slice order (``gk_matmul_split_k``).  One zero-initialised buffer per device and stream, grown when a
    launch needs more: launches on one stream are ordered, so they can share it, and every launch leaves the
    arrival counters at its head at zero.  The caller keeps the tensor until the launch is on its stream: another
    thread may replace the buffer by a larger one meanwhile."""
    return _workspace(_split_k_bytes(conf_c), stream)


def _split_k_bytes(conf_c) -> int:
    need = ctypes.c_size_t()
    rc = _lib.lib().gk_split_k_workspace_size(ctypes.byref(conf_c), ctypes.byref(need))
    if rc != _lib.GK_OK:
        _raise(rc)
    return need.value


def _sliced_bytes(conf_c, trans, epi) -> int:
    """Workspace of a launch that runs in slices of K (``gk_matmul_sliced``), 0 of any other."""
    shape, block = conf_c.matmul_shape, conf_c.block_shape
    if conf_c.op.kind == Operator.MFMA and (shape.K < 1280 or block.M != block.N or -(-shape.M // block.M) * -(-shape.N // block.N) > 170):
        return 0              # (what the library cuts has fewer tiles and a longer K: a first launch need not ask)
    need = ctypes.c_size_t()
    rc = _lib.lib().gk_sliced_workspace_size(ctypes.byref(conf_c), ctypes.byref(trans) if trans is not None else None,
                                             ctypes.byref(epi) if epi is not None else None, ctypes.byref(need))
    if rc != _lib.GK_OK:
        _raise(rc)
    return need.value


def _span(buf):
    """What the library is told of a workspace: its address and size."""
    return (int(buf.data_ptr()), int(buf.numel())) if buf is not None else (0, 0)


def _on(stream: int):
    """torch's current stream set to ``stream`` (a raw handle): what is allocated and cleared under it belongs to it, so the
    clear runs in front of a launch on it and whatever gets the memory next runs behind that launch."""
    import torch
    if stream == _current_stream():
        return contextlib.nullcontext()
    return torch.cuda.stream(torch.cuda.ExternalStream(stream) if stream else torch.cuda.default_stream())


def _capture_of(stream: int):
    """The id of the capture that ``stream`` is part of, or None."""
    capturing, capture = ctypes.c_int32(), ctypes.c_uint64()
    rc = _lib.lib().gk_stream_capture(stream, ctypes.byref(capturing), ctypes.byref(capture))
    if rc != _lib.GK_OK:
        _raise(rc)
    return capture.value if capturing.value else None


def _in_graph_pool(buf, stream: int, capture: int) -> bool:
    """Whether a buffer allocated during a capture lies in a memory pool of the graph (``torch.cuda.graph``), which keeps
    its memory as long as the graph lives, or in the allocator's common one, which hands it out again.  One answer for all
    of a stream's part in a capture."""
    import torch
    key = (buf.device.index, stream, capture)
    known = _pool_of_capture.get(key)
    if known is None:
        p = buf.data_ptr()
        pools = [tuple(s["segment_pool_id"]) for s in torch.cuda.memory_snapshot()
                 if s["device"] == buf.device.index and s["address"] <= p < s["address"] + s["total_size"]]
        known = bool(pools) and pools[0] != (0, 0)
        if len(_pool_of_capture) >= 64:
            _pool_of_capture.clear()
        _pool_of_capture[key] = known
    return known


def _workspace(need: int, stream: int):
    if need == 0:
        return None
    import torch
    stream = int(stream)
    key = (torch.cuda.current_device(), stream)
    capture = _capture_of(stream)
    if capture is not None:
        # a buffer of the graph's own, cleared by every replay: one that eager launches or other graphs use as well could be
        # in use, replaced by a larger one or not yet cleared when this graph runs
        with _on(stream):
            buf = torch.empty(need, dtype=torch.uint8, device="cuda")
            if not _in_graph_pool(buf, stream, capture):
                # a capture that torch does not know of: nobody else keeps the memory for the graph, so it is never given
                # back.  The graphs captured so on one stream share a buffer (as launches on one stream do: their replays
                # must not overlap), and a larger one is at least twice as large, which bounds all of them together
                kept = _recorded.setdefault(key, [])
                if not kept or kept[-1].numel() < need:
                    kept.append(buf if not kept else torch.empty(max(need, 2 * kept[-1].numel()), dtype=torch.uint8, device="cuda"))
                buf = kept[-1]
            buf[:_COUNTER_BYTES].zero_()
        return buf
    buf = _workspaces.get(key)
    if buf is None or buf.numel() < need:
        with _on(stream):
            buf = _workspaces[key] = torch.zeros(max(need, 1 << 20), dtype=torch.uint8, device="cuda")
        if _native is not None:
            _native.use_workspace(key[0], stream, buf.data_ptr(), buf.numel(), buf)
    return buf


_RETRY_AFTER = 256          # calls, after an allocation that failed: each one gives the allocator's cache back and waits for the device
_calls_without = {}         # (device, stream) -> calls that go without before memory is asked for again


def _workspace_if_any(need: int, stream: int):
    """``_workspace`` for a launch that is in slices of K without having been asked to: None where there is no memory for it (the library then
    launches it unsplit)."""
    import torch
    key = (torch.cuda.current_device(), int(stream))
    waiting = _calls_without.get(key, 0)
    if waiting > 0:
        buf = _workspaces.get(key)
        if buf is None or buf.numel() < need:
            _calls_without[key] = waiting - 1
            return None
    try:
        return _workspace(need, stream)
    except torch.OutOfMemoryError:
        _calls_without[key] = _RETRY_AFTER - 1
        return None


def _launch_sliced(conf_c, a, b, c, d, trans, epi, code: int, need: int, stream: int) -> int:
    """gk_matmul_sliced on descriptors and addresses, with the workspace of the stream; its status."""
    native = _load_native()
    if native is not None:
        rc = native.sliced_at(ctypes.addressof(conf_c), a, b, c, d, None if trans is None else ctypes.addressof(trans),
                              None if epi is None else ctypes.addressof(epi), code, need, stream)
        if rc == _lib.GK_OK:
            return rc
    workspace = _workspace_if_any(need, stream)
    if native is not None and workspace is not None:
        import torch
        key = (torch.cuda.current_device(), stream)
        if _workspaces.get(key) is workspace:
            native.use_workspace(*key, *_span(workspace), workspace)
    return _lib.lib().gk_matmul_sliced(ctypes.byref(conf_c), a, b, c, d, ctypes.byref(trans) if trans is not None else None,
                                       ctypes.byref(epi) if epi is not None else None, code, *_span(workspace), stream)


_IDENTITY = Transform.Elementwise()
_DEFAULT_EPILOGUE = Epilogue.Default()
_lowered = {}


def lower_transforms(transforms: dict) -> Optional[_lib.gk_transforms]:
    if all(t.is_identity for t in transforms.values()):
        return None
    if any(t.expr is not None for t in transforms.values()):
        raise ConfigError("expression transforms need a specialised kernel (gemmkernels.specialize)")
    return _lower(transforms)


def _lower(transforms: dict) -> Optional[_lib.gk_transforms]:
    """``lower_transforms`` of transforms without expressions.  (What it gives is kept for good: matmul() knows it by its identity.)"""
    key = tuple([transforms[name].ops for name in _HOOKS])
    hit = _lowered.get(key)
    if hit is not None:
        return hit
    if not any(key):
        return None
    out = _lowered[key] = _lib.gk_transforms()
    for i, name in enumerate(_HOOKS):
        ops = transforms[name].ops
        out.hook[i].n_ops = len(ops)
        for j, (kind, p0, p1) in enumerate(ops):
            out.hook[i].ops[j].kind, out.hook[i].ops[j].p0, out.hook[i].ops[j].p1 = kind, p0, p1
    return out


def _raise(rc: int):
    msg = _lib.last_error()
    if rc == _lib.GK_ERR_DIMENSION_MISMATCH:
        raise DimensionMismatch(msg)
    raise ConfigError(msg, rc)


class SpecializedKernel:
    """A kernel compiled at run time (hipRTC) for one configuration with its transform hooks inlined:
    arbitrary C expressions in x, and block shapes outside the table compiled into the library.  The
    counterpart of the reference's one-JIT-compiled-kernel-per-Config with inlined functors
    (src/matmul.jl:38, src/transform.jl:26-30).  The first construction for a given configuration and
    set of expressions compiles (seconds); later ones are served from the library's cache."""

    def __init__(self, conf: Config, transforms: dict):
        self.conf = conf
        exprs = (ctypes.c_char_p * 8)()
        self.expressions = []
        for i, name in enumerate(_HOOKS):
            t = transforms.get(name) or _IDENTITY
            e = t.c_expression()
            self.expressions.append(e)
            exprs[i] = e.encode() if e is not None else None
        handle = ctypes.c_void_p()
        cconf = conf.to_c()
        rc = _lib.lib().gk_rtc_compile(ctypes.byref(cconf), exprs, Kernel.matmul_pipelined.code, ctypes.byref(handle))
        if rc != _lib.GK_OK:
            _raise(rc)
        self._handle = handle
        buf = ctypes.create_string_buffer(200)
        _lib.lib().gk_rtc_kernel_name(handle, buf, len(buf))
        self.name = buf.value.decode()

    def plan(self, a, b, c, d, epilogue=None) -> "Plan":
        return Plan(self.conf, a, b, c, d, {}, _DEFAULT_EPILOGUE if epilogue is None else epilogue, Kernel.matmul_pipelined,
                    specialized=self)

    def __call__(self, a, b, c, d, epilogue=None, stream=None):
        return self.plan(a, b, c, d, epilogue)(stream)


def specialize(conf: Config, *,
               transform_global_to_shared_a=None, transform_global_to_shared_b=None,
               transform_global_to_shared_c=None, transform_shared_to_global_d=None,
               transform_shared_to_regs_a=None, transform_shared_to_regs_b=None,
               transform_shared_to_regs_c=None, transform_regs_to_shared_d=None) -> SpecializedKernel:
    """Compile (or fetch from the cache) the kernel of ``conf`` with these hooks inlined.  A hook is a
    ``Transform.Elementwise`` (op list or ``expr="..."``) or directly a C expression string in x."""
    given = dict(transform_global_to_shared_a=transform_global_to_shared_a, transform_global_to_shared_b=transform_global_to_shared_b,
                 transform_global_to_shared_c=transform_global_to_shared_c, transform_shared_to_global_d=transform_shared_to_global_d,
                 transform_shared_to_regs_a=transform_shared_to_regs_a, transform_shared_to_regs_b=transform_shared_to_regs_b,
                 transform_shared_to_regs_c=transform_shared_to_regs_c, transform_regs_to_shared_d=transform_regs_to_shared_d)
    return SpecializedKernel(conf, {k: (Transform.Elementwise(expr=v) if isinstance(v, str) else v) for k, v in given.items()})


def _launched_as(conf: Config, operands, lds, cconf, trans, transforms, hooks: bool, slices: bool) -> Optional[Config]:
    """``larger_tile`` of ``conf`` where the operands, but for their addresses, are what the aligned layouts of ``conf`` ask for (the library refuses others, and is
    left to) and no op list keeps the launch on its tile, or None."""
    larger = larger_tile(conf, hooks, slices)
    if larger is None or trans is not None and _lists_in_the_k_loop(conf, cconf, trans, transforms):
        return None
    for x, layout, ld in zip(operands, (conf.global_a_layout, conf.global_b_layout, conf.global_c_layout, conf.global_d_layout), lds):
        if layout.kind != Layout.ZERO and not _takes_larger_tile(x, layout, ld):
            return None
    return larger


def _takes_larger_tile(x, layout, ld: int) -> bool:
    # (the offsets in a tile are kept in 32 bits: 256 columns of 2^22 elements are left to a tile with fewer)
    return x is not None and ld * layout.T.size % 16 == 0 and ld < 1 << 21


_AB_HOOKS = ("transform_global_to_shared_a", "transform_shared_to_regs_a", "transform_global_to_shared_b", "transform_shared_to_regs_b")
_lists = {}


def _lists_in_the_k_loop(conf: Config, cconf, trans, transforms: dict) -> bool:
    """Whether the hooks of A and B stay in the K loop as op lists (one factor per operand is folded or multiplied in, see the library's fused levels).  Such a launch
    keeps its tile: its time is that of the lists, of which the estimates know nothing.  Of 67 drawn plans that a larger tile took 20 were slower on it, up to twice
    (3648 x 3456 x 4032 'T','N' with a list on B 783 -> 1629 us), and those on the tile that stands for slices, of which there are none with lists, all were (1088 x 1088 x 5248 'N','T' with one on A 240 -> 437).
    With hooks on C and D, a bias or factors all of 53 were faster."""
    if conf.operator.kind != Operator.MFMA or all(transforms[h].is_identity for h in _AB_HOOKS):
        return False
    key = (conf.global_a_layout.kind, conf.global_a_layout.T.name, *(transforms[h].ops for h in _AB_HOOKS))
    known = _lists.get(key)
    if known is None:
        if len(_lists) >= 256:
            _lists.clear()
        name = ctypes.create_string_buffer(256)
        if _lib.lib().gk_kernel_name(ctypes.byref(cconf), ctypes.byref(trans), None, Kernel.matmul_pipelined.code, name, len(name)) != _lib.GK_OK:
            return True                   # (refused: the launch says why)
        known = _lists[key] = name.value.endswith(b"_fused_ab")
    return known


def _routes_of(conf: Config, lds, cconf, trans, transforms, epi, operands):
    """What a launch of ``conf`` on operands of these leading dimensions tries, in this order: descriptor, workspace (0: not in slices of K), and whether
    it takes operands at 16-byte boundaries only."""
    mfma = conf.operator.kind == Operator.MFMA
    larger = _launched_as(conf, operands, lds, cconf, trans, transforms, trans is not None or epi is not None, mfma) if mfma else None
    of = [cconf] if larger is None else [larger.to_c(*lds), cconf]
    return [(c, _sliced_bytes(c, trans, epi) if mfma else 0, c is not cconf) for c in of]


class Plan:
    """One launch with everything but the stream lowered ahead of time: the descriptors of the
    configuration, the transforms and the epilogue, and the operand addresses.  Calling the plan is
    one call into the library, which runs every launch-time check of reference
    src/matmul.jl:28-41 on the first call and, where the launch needs no workspace, keeps what they found from the second on (``prepare``).  The plan keeps its operands alive; they must not be resized or freed by
    other means while it is in use.  For loops that launch the same GEMM many times, where the
    microseconds a general ``matmul`` call spends on lowering would rival the kernel itself."""

    __slots__ = ("_fn", "_conf", "_trans", "_epi", "_args", "_keep", "_split_k", "_sliced", "_slices", "_as_given", "_direct", "_calls", "d", "kernel_names")

    def __init__(self, conf: Config, a, b, c, d, transforms: dict, epilogue, kernel, specialized=None, slices=False):
        if specialized is None and any(t.expr is not None for t in transforms.values()):
            specialized = SpecializedKernel(conf, transforms)       # expression hooks: a run-time compiled kernel
        lds = (_leading_dim(a, conf.global_a_layout), _leading_dim(b, conf.global_b_layout),
               _leading_dim(c, conf.global_c_layout), _leading_dim(d, conf.global_d_layout))
        self._conf = _lib.gk_config.from_buffer_copy(conf.to_c(*lds))        # to_c hands out a cached, shared descriptor
        self._trans = None if specialized is not None else lower_transforms(transforms)
        self._as_given = None                                      # (what is launched where the library refuses the larger tile)
        hooks = self._trans is not None or epilogue.kind != Epilogue.DEFAULT
        larger = None
        if specialized is None and kernel is not Kernel.matmul_split_k:
            larger = _launched_as(conf, (a, b, c, d), lds, self._conf, self._trans, transforms, hooks, slices)
            if larger is not None and any(x is not None and _ptr(x) % 16 != 0 for x in (a, b, c, d)):
                larger = None
        if larger is not None:
            self._as_given, self._conf = self._conf, _lib.gk_config.from_buffer_copy(larger.to_c(*lds))
        self._epi = None
        self._split_k, self._sliced, self._slices = False, 0, slices
        if epilogue.kind != Epilogue.DEFAULT:
            self._epi = _lib.gk_epilogue()
            self._epi.kind = epilogue.kind
            self._epi.bias = _ptr(epilogue.bias)
        epi_ref = ctypes.byref(self._epi) if self._epi is not None else None
        if specialized is not None:
            self._fn = _lib.lib().gk_rtc_matmul
            self._args = (specialized._handle, ctypes.byref(self._conf), _ptr(a), _ptr(b), _ptr(c), _ptr(d), epi_ref)
        elif kernel is Kernel.matmul_split_k:
            self._fn = _lib.lib().gk_matmul_split_k
            self._args = (ctypes.byref(self._conf), _ptr(a), _ptr(b), _ptr(c), _ptr(d),
                          ctypes.byref(self._trans) if self._trans is not None else None, epi_ref)
            self._split_k = True
        else:
            self._sliced = _sliced_bytes(self._conf, self._trans, self._epi) if slices else 0
            self._fn = _lib.lib().gk_matmul_sliced if self._sliced else _lib.lib().gk_matmul
            self._args = (ctypes.byref(self._conf), _ptr(a), _ptr(b), _ptr(c), _ptr(d),
                          ctypes.byref(self._trans) if self._trans is not None else None, epi_ref, kernel.code)
        self._keep = (a, b, c, d, epilogue, specialized)
        self._direct = None           # (from the second call on, see prepare)
        self._calls = 0 if specialized is None and not self._split_k and not self._sliced else 2
        self.d = d
        self.kernel_names = ()      # filled in by the BLAS-level front end

    def prepare(self):
        """Has the library check the launch once for all calls to come (gk_prepare): a few microseconds, which a plan that is called once does not pay."""
        self._calls = 2
        if _load_native() is not None:
            prepared = Prepared(self._conf, self._trans, self._epi, self._args[-1])
            if prepared.handle is not None:
                self._direct = prepared, (prepared.handle, *self._args[1:5])         # (one object: a thread that uses it holds it)

    def __call__(self, stream=None):
        if self._calls < 2:
            self._calls += 1
            if self._calls == 2:
                self.prepare()
        stream = _current_stream() if stream is None else int(stream)
        if self._split_k:
            workspace = split_k_workspace(self._conf, stream)
            rc = self._fn(*self._args, *_span(workspace), stream)
            if rc != _lib.GK_OK:
                _raise(rc)
            return self.d
        if self._sliced:
            rc = _launch_sliced(self._conf, *self._args[1:5], self._trans, self._epi, self._args[-1], self._sliced, stream)
        else:
            direct = self._direct
            if direct is not None and _native.run_at(*direct[1], stream) == _lib.GK_OK:
                return self.d
            rc = self._fn(*self._args, stream)
        if rc != _lib.GK_OK and self._as_given is not None:
            need = _sliced_bytes(self._as_given, self._trans, self._epi) if self._slices else 0
            if need:
                rc = _launch_sliced(self._as_given, *self._args[1:5], self._trans, self._epi, self._args[-1], need, stream)
            else:
                rc = _lib.lib().gk_matmul(ctypes.byref(self._as_given), *self._args[1:], stream)
        if rc != _lib.GK_OK:
            _raise(rc)
        return self.d


def _collect(given: dict) -> dict:
    return {k: (_IDENTITY if v is None else v) for k, v in given.items()}


def plan(conf: Config, a, b, c, d, *,
         transform_global_to_shared_a=None, transform_global_to_shared_b=None,
         transform_global_to_shared_c=None, transform_shared_to_global_d=None,
         transform_shared_to_regs_a=None, transform_shared_to_regs_b=None,
         transform_shared_to_regs_c=None, transform_regs_to_shared_d=None,
         epilogue=None, kernel=Kernel.matmul_singlestage) -> Plan:
    """Same arguments as ``matmul``; returns a ``Plan`` whose call launches on the current stream."""
    from . import complex_planar
    if complex_planar.is_planar(conf) and not complex_planar.planes_adjacent(a, b, c, d):
        return complex_planar.PlanarComplexPlan(conf, a, b, c, d)
    transforms = _collect(dict(transform_global_to_shared_a=transform_global_to_shared_a,
                               transform_global_to_shared_b=transform_global_to_shared_b,
                               transform_global_to_shared_c=transform_global_to_shared_c,
                               transform_shared_to_global_d=transform_shared_to_global_d,
                               transform_shared_to_regs_a=transform_shared_to_regs_a,
                               transform_shared_to_regs_b=transform_shared_to_regs_b,
                               transform_shared_to_regs_c=transform_shared_to_regs_c,
                               transform_regs_to_shared_d=transform_regs_to_shared_d))
    # (FPUOp: a configured launch is one fma chain per output, whatever its sizes)
    return Plan(conf, a, b, c, d, transforms, _DEFAULT_EPILOGUE if epilogue is None else epilogue, kernel, slices=conf.operator.kind == Operator.MFMA)


_PREPARED_MAX = 64


class _Sliced:
    """What gk_torch launches in slices of K where ``Prepared`` holds a launch checked once: the descriptor, the kind of kernel and the workspace."""

    __slots__ = ("handle", "args", "_conf")

    def __init__(self, conf_c, code: int, need: int):
        self._conf = _lib.gk_config.from_buffer_copy(conf_c)
        self.handle, self.args = None, (ctypes.addressof(self._conf), code, need)


def _prepare(conf: Config, cconf, lds, kernel, need: int = 0) -> None:
    """Keeps the launch that ``matmul`` made for operands of these leading dimensions (no address) with its configuration."""
    kept = conf.__dict__.get("_prepared")
    if _load_native() is None or kept is not None and (lds, kernel) in kept:
        return
    if conf.__dict__.get("_launched") != (lds, kernel):             # (a configuration that is launched once does not pay for it)
        conf.__dict__["_launched"] = (lds, kernel)
        return
    made = _Sliced(cconf, kernel.code, need) if need else Prepared(cconf, None, None, kernel.code)
    if not need and made.handle is None:
        return
    if kept is None or len(kept) > _PREPARED_MAX:
        forms = {**dict.fromkeys(_NO_LD, 0), **dict.fromkeys(_INTERLEAVED, 2), **dict.fromkeys(_SPLIT, 3)}
        kept = {"forms": tuple(forms.get(l.kind, 1) for l in (conf.global_a_layout, conf.global_b_layout, conf.global_c_layout, conf.global_d_layout))}
    kept[(lds, kernel)] = made
    conf.__dict__["_prepared"] = kept


def matmul(conf: Config, a, b, c, d, *,
           transform_global_to_shared_a=None, transform_global_to_shared_b=None,
           transform_global_to_shared_c=None, transform_shared_to_global_d=None,
           transform_shared_to_regs_a=None, transform_shared_to_regs_b=None,
           transform_shared_to_regs_c=None, transform_regs_to_shared_d=None,
           epilogue=None, kernel=Kernel.matmul_singlestage, stream=None):
    """reference src/matmul.jl:7-44: launch geometry, checks (ConfigError) and the asynchronous
    launch on the current stream.  Same positional and keyword arguments as the reference."""
    hooked = not (transform_global_to_shared_a is None and transform_global_to_shared_b is None and
                  transform_global_to_shared_c is None and transform_shared_to_global_d is None and transform_shared_to_regs_a is None and
                  transform_shared_to_regs_b is None and transform_shared_to_regs_c is None and transform_regs_to_shared_d is None)
    plain = epilogue is None and not hooked
    prepared = conf.__dict__.get("_prepared") if plain else None
    if prepared is not None and stream is None:
        # (a launch of these leading dimensions was made before: a Config is immutable once built)
        lds = _native.leading_dims(prepared["forms"], a, b, c, d)
        again = prepared.get((lds, kernel)) if lds is not None else None
        if again is not None and (_native.run(again.handle, a, b, c, d) if again.handle is not None else _native.run_sliced(*again.args, a, b, c, d)):
            return d
    from . import complex_planar
    if complex_planar.is_planar(conf) and not complex_planar.planes_adjacent(a, b, c, d):
        return complex_planar.PlanarComplexPlan(conf, a, b, c, d)(stream)
    ctrans = None
    if hooked:
        collected = _collect(dict(
            transform_global_to_shared_a=transform_global_to_shared_a, transform_global_to_shared_b=transform_global_to_shared_b,
            transform_global_to_shared_c=transform_global_to_shared_c, transform_shared_to_global_d=transform_shared_to_global_d,
            transform_shared_to_regs_a=transform_shared_to_regs_a, transform_shared_to_regs_b=transform_shared_to_regs_b,
            transform_shared_to_regs_c=transform_shared_to_regs_c, transform_regs_to_shared_d=transform_regs_to_shared_d))
        if any(t.expr is not None for t in collected.values()):
            return Plan(conf, a, b, c, d, collected, _DEFAULT_EPILOGUE if epilogue is None else epilogue, kernel)(stream)
        ctrans = _lower(collected)

    lds = (_leading_dim(a, conf.global_a_layout), _leading_dim(b, conf.global_b_layout),
           _leading_dim(c, conf.global_c_layout), _leading_dim(d, conf.global_d_layout))
    cconf = conf.to_c(*lds)
    cepi = None
    if epilogue is not None and epilogue.kind != Epilogue.DEFAULT:
        cepi = _lib.gk_epilogue()
        cepi.kind = epilogue.kind
        cepi.bias = _ptr(epilogue.bias)
    stream = _current_stream() if stream is None else int(stream)
    if kernel is Kernel.matmul_split_k:
        workspace = split_k_workspace(cconf, stream)
        rc = _lib.lib().gk_matmul_split_k(ctypes.byref(cconf), _ptr(a), _ptr(b), _ptr(c), _ptr(d),
                                          ctypes.byref(ctrans) if ctrans is not None else None,
                                          ctypes.byref(cepi) if cepi is not None else None,
                                          *_span(workspace), stream)
    else:
        pointers = (_ptr(a), _ptr(b), _ptr(c), _ptr(d))
        routes = conf.__dict__.setdefault("_routes", {})                 # (a Config is immutable once built, and lowered transforms are kept)
        key = (lds, 0 if ctrans is None else id(ctrans), 0 if cepi is None else cepi.kind)
        route = routes.get(key)
        if route is None:
            if len(routes) >= _PREPARED_MAX:
                routes.clear()
            route = routes[key] = _routes_of(conf, lds, cconf, ctrans, collected if ctrans is not None else None, cepi, (a, b, c, d))
        rc = _lib.GK_ERR_UNSUPPORTED
        for of, need, aligned in route:                                   # (the tile asked for where the library refuses the larger one)
            if aligned and any(p is not None and p % 16 != 0 for p in pointers):
                continue
            rc = _launch_sliced(of, *pointers, ctrans, cepi, kernel.code, need, stream) if need else _gk_matmul(of, *pointers, ctrans, cepi, kernel.code, stream)
            if rc == _lib.GK_OK:
                if plain:
                    _prepare(conf, of, lds, kernel, need)
                break
    if rc != _lib.GK_OK:
        _raise(rc)
    return d


def kernel_name(conf: Config, kernel=Kernel.matmul_singlestage, transforms=None, epilogue=None) -> str:
    """Name of the compiled kernel instance a launch of ``conf`` runs (for logs and profiles)."""
    cconf = conf.to_c()
    buf = ctypes.create_string_buffer(256)
    ctrans = None
    if transforms:
        full = {k: transforms.get(k, Transform.Elementwise()) for k in _HOOKS}
        ctrans = lower_transforms(full)
    cepi = None
    if epilogue is not None and epilogue.kind != Epilogue.DEFAULT:
        cepi = _lib.gk_epilogue()
        cepi.kind = epilogue.kind
    rc = _lib.lib().gk_kernel_name(ctypes.byref(cconf), ctypes.byref(ctrans) if ctrans is not None else None,
                                   ctypes.byref(cepi) if cepi is not None else None, kernel.code, buf, len(buf))
    if rc != _lib.GK_OK:
        raise ConfigError(_lib.last_error(), rc)
    return buf.value.decode()


# ------------------------------------------------------------------------------------------------
# BLAS-like
# ------------------------------------------------------------------------------------------------

def _select_kernel(layout_a, layout_b):
    """reference src/matmul.jl:52-56: the pipelined kernel when both operands are aligned."""
    if layout_a.is_aligned and layout_b.is_aligned:
        return Kernel.matmul_pipelined
    return Kernel.matmul_singlestage


_configs = {}


def get_config(*args):
    """Memoised create_config (reference src/matmul.jl:58-65)."""
    val = _configs.get(args)
    if val is None:
        val = _configs[args] = create_config(*args)
    return val


def create_config(A: DType, sizeA, stridesA, transA: bool, B: DType, sizeB, stridesB, transB: bool,
                  C: DType, sizeC, stridesC, alpha: type, zeroAlpha: bool, beta: type, zeroBeta: bool, wmma=None,
                  aligned_pointers=(True, True, True), factor: Optional[str] = None):
    """reference src/matmul.jl:66-183, with the MI355X operator and block-shape choices.  ``aligned_pointers``
    says whether A, B and C start on 16-byte boundaries: the reference decides on the aligned layouts from the
    strides alone (a misaligned view then traps on the device, src/layout.jl:22-25); here such an operand gets
    the bounds-checked layout, which takes any address.  ``factor``: how alpha is applied to A
    in the K loop (None: not there), see ``split_k_block_shape``."""
    m = sizeA[1 if transA else 0]
    k = sizeA[0 if transA else 1]
    n = sizeB[0 if transB else 1]
    if m != sizeC[0] or n != sizeC[1] or k != sizeB[1 if transB else 0]:
        raise DimensionMismatch("Dimensions do not match")

    a_layout_base = Layout.RowMajor if transA else Layout.ColMajor
    b_layout_base = Layout.RowMajor if transB else Layout.ColMajor
    a_aligned_layout_base = Layout.UnsafeAlignedRowMajor if transA else Layout.UnsafeAlignedColMajor
    b_aligned_layout_base = Layout.UnsafeAlignedRowMajor if transB else Layout.UnsafeAlignedColMajor

    # operator: the matrix cores for 16-bit inputs with fp32 accumulation (src/matmul.jl:85-91)
    mfma_types = [(Float16, Float16, Float32), (BFloat16, BFloat16, Float32), (Float16, Float16, Float16)]
    compute_type = promote_type(A, B)
    use_mfma = ((compute_type, compute_type, C) in mfma_types) if wmma is None else bool(wmma)

    shared_a_layout = Layout.Padded[a_aligned_layout_base[compute_type if use_mfma else A], 8]
    shared_b_layout = Layout.Padded[b_aligned_layout_base[compute_type if use_mfma else B], 8]
    shared_c_layout = Layout.Zero[C] if zeroBeta else Layout.UnsafeAlignedColMajor[C]
    shared_d_layout = Layout.UnsafeAlignedColMajor[C]

    if use_mfma:
        operator = Operator.MFMAOp[32, 32, 16, compute_type, Float32 if C == Float16 else C]
    else:
        operator = Operator.FPUOp[8, 8, 1, 8, 8, 1, compute_type, C]
    a_aligned = (stridesA[1] * A.size) % 16 == 0 and aligned_pointers[0]
    b_aligned = (stridesB[1] * B.size) % 16 == 0 and aligned_pointers[1]
    c_aligned = (stridesC[1] * C.size) % 16 == 0 and aligned_pointers[2]

    def layouts_for(block_shape):
        # src/matmul.jl:121-156: vector loads and stores need 16-byte aligned columns and whole tiles
        if zeroAlpha:
            ga, gb = Layout.Zero[A], Layout.Zero[B]
        else:
            ga = (a_aligned_layout_base[A] if a_aligned and m % block_shape.M == 0 and k % block_shape.K == 0
                  else a_layout_base[A])
            gb = (b_aligned_layout_base[B] if b_aligned and k % block_shape.K == 0 and n % block_shape.N == 0
                  else b_layout_base[B])
        cd_aligned = c_aligned and m % block_shape.M == 0 and n % block_shape.N == 0
        gc = Layout.Zero[C] if zeroBeta else (Layout.UnsafeAlignedColMajor[C] if cd_aligned else Layout.ColMajor[C])
        gd = Layout.UnsafeAlignedColMajor[C] if cd_aligned else Layout.ColMajor[C]
        return ga, gb, gc, gd

    # The library runs a 16-bit product on bounds-checked layouts on the aligned kernels all the same (any address
    # and leading dimension; tiles over the edge clamp their loads and mask their stores; the last K tile is
    # repaired in LDS when a 16-byte chunk reaches over the end of an operand) as long as A and B hold one whole
    # chunk of 8 elements along their contiguous index; floating-point FPUOp takes any size and alignment on every tile.  Then the tile is chosen among all tiles, not only those
    # that divide the sizes (4096 x 4096 x 4000: the 64-deep tile with a partial last step instead of the 32-deep
    # one), and the operands it does not divide get the bounds-checked layouts, as the reference's rule says.
    edge_ok = not zeroAlpha and (((k if transA else m) >= 8 and (n if transB else k) >= 8) if use_mfma
                                 else compute_type in (Float16, Float32, Float64))
    block_shape = None
    if use_mfma and edge_ok:
        block_shape = sliced_block_shape(m, n, k, max(stridesA[1], stridesB[1]), not (a_aligned and b_aligned)) or split_k_block_shape(m, n, k, max(0 if transA else stridesA[1], stridesB[1] if transB else 0), factor)
    if block_shape is None:
        block_shape = default_block_shape(operator, NT(M=m, N=n, K=k), tile_sized=not edge_ok, a_kmajor=transA, b_kmajor=not transB)
        if use_mfma and edge_ok:
            odd = (not a_aligned and transA) + (not b_aligned and not transB), (not a_aligned and not transA) + (not b_aligned and transB)
            block_shape = product_block_shape(block_shape, m, n, k, transA, not transB, odd, C.size * (1 if zeroBeta else 2),
                                              stridesA[1], stridesB[1])
    global_a_layout, global_b_layout, global_c_layout, global_d_layout = layouts_for(block_shape)
    if not edge_ok and any(l.kind in (Layout.COL_MAJOR, Layout.ROW_MAJOR) for l in (global_a_layout, global_b_layout, global_c_layout, global_d_layout)):
        # some operand needs bounds checks (and C = beta C, the zero alpha): one tile shape
        block_shape = NT(M=64, N=64, K=32)
        global_a_layout, global_b_layout, global_c_layout, global_d_layout = layouts_for(block_shape)

    conf = _get_config(gemm_shape=NT(M=m, N=n, K=k), block_shape=block_shape, operator=operator,
                       global_a_layout=global_a_layout, global_b_layout=global_b_layout,
                       global_c_layout=global_c_layout, global_d_layout=global_d_layout,
                       shared_a_layout=shared_a_layout, shared_b_layout=shared_b_layout,
                       shared_c_layout=shared_c_layout, shared_d_layout=shared_d_layout,
                       is_a_col_major=not transA, is_b_col_major=not transB)
    return conf, compute_type, _select_kernel(global_a_layout, global_b_layout)


def _round_to(dtype: DType, x: float) -> float:
    if dtype == Float16:
        return float(np.float16(x))
    if dtype == BFloat16:
        import torch
        return float(torch.tensor(x, dtype=torch.bfloat16))
    if dtype == Float32:
        return float(np.float32(x))
    return float(x)


_FOLDED = frozenset(2.0 ** e for e in range(-4, 5))


def _single_plan(C, tA: bool, tB: bool, A, B, alpha, beta, wmma=None) -> Plan:
    """One launch for C = alpha * op(A) * op(B) + beta * C: the configuration ``create_config`` picks."""
    # (a power of two within 2^-4 .. 2^4 leaves the K loop, see the folded scales of the library)
    factor = None if abs(float(alpha)) in _FOLDED else "per fragment"
    conf, compute_type, kernel = get_config(
        from_torch(A.dtype), tuple(A.shape), tuple(A.stride()), tA,
        from_torch(B.dtype), tuple(B.shape), tuple(B.stride()), tB,
        from_torch(C.dtype), tuple(C.shape), tuple(C.stride()),
        type(alpha), alpha == 0, type(beta), beta == 0, wmma, tuple(x.data_ptr() % 16 == 0 for x in (A, B, C)), factor)
    alpha_c = _round_to(compute_type, float(alpha))          # convert(compute_type, alpha), :196
    beta_c = _round_to(from_torch(C.dtype), float(beta))     # convert(eltype(C), beta), :197
    for name, value in (("alpha", alpha_c), ("beta", beta_c)):
        if float(np.float32(value)) != value:
            # transform parameters travel as binary32; Float64 (or large integer) factors that do not
            # fit would silently change the result
            raise ConfigError(f"{name} = {value!r} is not representable in binary32, the parameter type of the transform hooks")
    # beta = 0 has already turned C into a Zero layout: nothing is loaded, nothing to scale
    ta = Transform.Elementwise(ops=[] if alpha_c == 1.0 else [(Transform.SCALE, alpha_c, 0.0)])
    tc = Transform.Elementwise(ops=[] if beta_c == 1.0 or beta == 0 else [(Transform.SCALE, beta_c, 0.0)])
    if conf.operator.kind == Operator.MFMA:
        # few output tiles and a long K loop (skinny products): the K-split kind cuts K into slices so that every CU gets
        # work (the library decides how many, and runs the product unsplit when slices would be too short or the tile
        # has no K-split instance; the bounds-checked kernel takes slices too).  Its sum is
        # ordered, so the result is the same on every run, like the reference's mul!.
        bs, ms = conf.block_shape, conf.matmul_shape
        tiles = -(-ms.M // bs.M) * -(-ms.N // bs.N)
        sliced = _product_slices((bs.M, bs.N, bs.K), ms.M, ms.N, ms.K) > 1
        if not sliced and (bs == split_k_block_shape(ms.M, ms.N, ms.K, 0, factor) or tiles <= 128 and ms.K >= 2048):
            kernel = Kernel.matmul_split_k
    else:
        sliced = conf.operator.kind == Operator.FPU
    # (floating-point FPUOp and 128 x 128: the library takes slices of K where one chain per output would leave the chip idle, gk_matmul_sliced)
    p = Plan(conf, A, B, C, C, _collect({**dict.fromkeys(_HOOKS), "transform_shared_to_regs_a": ta, "transform_shared_to_regs_c": tc}),
             _DEFAULT_EPILOGUE, kernel, slices=sliced)
    p.kernel_names = (kernel_name(conf, kernel, dict(transform_shared_to_regs_a=ta, transform_shared_to_regs_c=tc)),)
    return p


def matmatmul_plan(C, transA: str, transB: str, A, B, alpha, beta, *, wmma=None):
    """The launch ``matmatmul_`` would make, as a ``Plan`` to call any number of times: one launch of the
    configuration ``create_config`` picks (reference src/matmul.jl:185-204), whatever the sizes.  A 16-bit
    product whose sizes are not whole tiles, whose leading dimensions are odd or whose operands start off a
    16-byte boundary still runs on the aligned kernels (``create_config``); the bounds-checked kernel is left
    with operands that have fewer than 8 elements along their contiguous index."""
    return _single_plan(C, transA == 'T', transB == 'T', A, B, alpha, beta, wmma)


def matmatmul_(C, transA: str, transB: str, A, B, alpha, beta, *, wmma=None):
    """``matmatmul!`` (reference src/matmul.jl:185-204): C = alpha * op(A) * op(B) + beta * C."""
    tA, tB = transA == 'T', transB == 'T'
    a, b, c = A.data_ptr(), B.data_ptr(), C.data_ptr()
    key = None
    if type(alpha) in _PLAIN_NUMBERS and type(beta) in _PLAIN_NUMBERS:
        key = (tA, tB, A.dtype, A.shape, A.stride(), B.dtype, B.shape, B.stride(), C.dtype, C.shape, C.stride(),
               alpha, beta, wmma, a % 16 == 0, b % 16 == 0, c % 16 == 0)
        hit = _mul_launches.get(key)
        if hit is not None:
            if wmma is None:
                _remember(C, A, B, tA, tB, alpha, beta, hit)
            hit(a, b, c, _current_stream())
            return C
    p = _single_plan(C, tA, tB, A, B, alpha, beta, wmma)
    # (an alpha that is infinite in A's type would make NaN of the zeros that fill a copy up)
    packed = packed_leading_dims(p._conf, a, b) if not p._split_k and not p._sliced and math.isfinite(_round_to(from_torch(A.dtype), float(alpha))) else None
    launch = _MulLaunch(p) if packed is None else _MulLaunchOnCopies(p, packed)
    if key is not None:
        if len(_mul_launches) >= _MUL_LAUNCHES_MAX:
            _mul_launches.clear()
        _mul_launches[key] = launch
    launch(a, b, c, _current_stream())
    if key is not None and wmma is None:
        _remember(C, A, B, tA, tB, alpha, beta, launch)
    return C


def _load_native():
    global _native, _native_mul
    if _native is None:
        _native = load_native()
        if _native is not None:
            _native_mul = _native.mul
    return _native


def _native_mul(C, A, B, tA, tB, alpha, beta) -> bool:
    """gk_torch's ``mul`` once it is loaded: True when the call is on its way."""
    return False


def _remember(C, A, B, tA, tB, alpha, beta, launch) -> None:
    """Leaves the launch of this kind of operands with gk_torch, which makes the next ones (``mul_``), and the workspace of the stream."""
    native = _load_native()
    if native is None or type(launch) is not _MulLaunch or type(alpha) is not float or type(beta) is not float:
        return
    import torch
    form, need = (2, launch._workspace) if launch._workspace is not None else (1, launch._sliced) if launch._sliced else (0, 0)
    what, owner, trans = ctypes.addressof(launch._conf), None, 0 if launch._trans is None else ctypes.addressof(launch._trans)
    if form == 0 and all(x.data_ptr() % 16 == 0 for x in (A, B, C)):           # (part of the kind)
        owner = launch._prepared
        if owner is None:
            owner = launch._prepared = Prepared(launch._conf, launch._trans, None, launch._code)
        if owner.handle is not None:
            form, what = 3, owner.handle
    if native.remember(C, A, B, tA, tB, alpha, beta, form, what, trans, launch._code or 0, need, (launch, owner)) and need:
        key = (torch.cuda.current_device(), _current_stream())
        buf = _workspaces.get(key)
        if buf is not None:
            native.use_workspace(*key, buf.data_ptr(), buf.numel(), buf)


_PLAIN_NUMBERS = (float, int, bool)


def _stored(which: int, kind: int, extent: int, k: int):
    """Rows (contiguous) and columns of operand A (0) or B (1) as it lies in memory."""
    row_major = kind in (Layout.ROW_MAJOR, Layout.ALIGNED_ROW_MAJOR)
    return (k, extent) if row_major == (which == 0) else (extent, k)


_PACK_MIN_WORK, _PACK_MIN_WORK_ONE = 24 * 10 ** 9, 80 * 10 ** 9      # M N K with both operands, with one of them
_PACK_MAX_BYTES = 512 << 20
_PACK_SHARE, _PACK_SHARE_ONE = (0.29, 0.325, 0.36), 0.13             # of the product's time; both operands: by how many are contiguous along k


def packed_leading_dims(conf_c, a: int, b: int):
    """Leading dimensions of copies of A and of B (None: the operand stays as it is) on which a product runs faster, the
    copying included, or None.

    An operand whose columns start off 16-byte boundaries costs a launch more requests to the L2 than its bytes need: a 128-byte row of a
    tile lies on two lines where k is contiguous, one of 512 bytes on five (4001 x 4003 x 4005 'T','N': 18.0 million requests, 10.1 on copies and 1.6 for
    copying; memory sees the same traffic either way).  Copies with columns on 128-byte lines are read and written at 5.3 TB/s while
    they and the operands fit the memory-side cache (4 TB/s beyond), and they pay where that is a small enough share of the product
    (_mfma_cost); copies of both operands end in whole K tiles as well (_MulLaunchOnCopies).  BF16, us without and with copies, each on the same inputs over
    and over / on inputs that rotate through 600 MB / alone on new ones, by that share:
      0.08 8001 x 8003 x 2005 'N','T' 366 307 / 441 309 / 450 328, 'T','N' 396 292 / 468 292 / 483 311;
      0.18 3001 x 3003 x 3005 'N','T' 82 83 / 105 86 / 100 104, 'T','N' 83 76 / 113 80 / 101 99; 2501 x 8003 x 4005 'N','N' 202 190 / 268 197 / 288 225;
      0.24 4001 x 4003 x 4005 'N','N' 133 126 / 171 143 / 153 151, 'N','T' 129 129 / 168 144 / 145 147, 'T','N' 137 126 / 178 143 / 155 149;
      0.28 801 x 5003 x 6005 'N','N' 117 99 / 134 102 / 131 117; 0.30 2001 x 2003 x 6005 'N','T' 71 78 / 88 81 / 89 101, 'N','N' 78 73 / 105 78 / 97 94;
      0.27 2501 x 8003 x 8005 'N','T' 4 % slower / 22 % faster / 12 % faster; 0.34 1001 x 8003 x 4005 'N','N' 90 91 / 122 93 / 148 124, 'N','T' 86 91 / 108 94 / 120 131,
      'T','N' 94 88 / 125 91 / 148 122; 0.39 4001 x 4003 x 8100 6 to 9 % slower / 13 to 20 % faster / between;
      0.48 1501 x 8003 x 8005 'N','N' 193 233 / 249 233 / 270 287.
    Below 2.4e10 products the copies take what they save (2001 x 2003 x 4005, 3001 x 3003 x 1505).  One odd operand, contiguous along k:
      4000 x 4000 x 4001 'N','N' 111 114 / 139 125 / 125 128 (6.4e10, not copied), 5000 x 5000 x 5001 258 239 / 337 281 / 342 296, 6000 x 6000 x 6001 'N','N' 387 389 / 440 417 /
      466 443 and 'T','T' 408 439 / 509 441 / 526 466, 8000 x 8000 x 8001 915 796 / 929 795 / 944 794; a share of 0.3 2000 x 8000 x 8001 210 242 / 255 243 / 253 264;
      along m or n: not worth a copy (4001 x 4000 x 4000 'N','N' 123 125 / 160 155)."""
    shape, layouts = conf_c.matmul_shape, (conf_c.global_a_layout, conf_c.global_b_layout)
    work = shape.M * shape.N * shape.K
    tile = (conf_c.block_shape.M, conf_c.block_shape.N, conf_c.block_shape.K)
    if conf_c.op.kind != Operator.MFMA or work < _PACK_MIN_WORK or min(shape.M, shape.N) < 512 or shape.K < 1000 or tile not in _MFMA_TILE_COST:
        return None
    if any(layout.kind == Layout.ZERO for layout in layouts):        # (alpha = 0)
        return None
    odd = tuple(layout.ld % 8 != 0 or address % 16 != 0 for layout, address in zip(layouts, (a, b)))
    k_major = tuple(layouts[which].kind in ((Layout.ROW_MAJOR, Layout.ALIGNED_ROW_MAJOR) if which == 0 else (Layout.COL_MAJOR, Layout.ALIGNED_COL_MAJOR))
                    for which in (0, 1))
    if not all(odd) and (work < _PACK_MIN_WORK_ONE or not any(o and k for o, k in zip(odd, k_major))):
        return None
    k = -(-shape.K // 64) * 64 if all(odd) else shape.K
    stored = tuple(_stored(which, layouts[which].kind, (shape.M, shape.N)[which], k) for which in (0, 1))
    packed = tuple(-(-rows // 64) * 64 if o else None for o, (rows, _) in zip(odd, stored))
    total = sum(2 * ld * cols for ld, (_, cols) in zip(packed, stored) if ld is not None)
    if total > _PACK_MAX_BYTES or max(rows for rows, _ in stored) > _PACK_MAX_ROWS:
        return None
    copying = 2 * total / (5.3e6 if total < 100e6 else 4.0e6)
    share = _PACK_SHARE[sum(k_major)] if all(odd) else _PACK_SHARE_ONE
    return packed if copying <= share * _mfma_cost(tile, shape.M, shape.N, shape.K) else None


_PACK_MAX_ROWS = 255 * 512          # of one launch of gk_pack_columns


class _MulLaunch:
    """What ``matmatmul_`` hands to the library for operands of one kind (element types, sizes, strides, alignment) and one
    pair of factors: descriptors only, no address and no tensor, so any operands of that kind can use it, on any
    stream and from any thread.  (What is written after it is made is the launch checked once for gk_torch: threads that meet there make one too
    many.)  Lowering the same call again takes 22 us of
    interpreter time, the whole of a small product: mul! at 256^3 in Float32 takes 5 us on the device."""

    __slots__ = ("_fn", "_conf", "_trans", "_conf_ref", "_trans_ref", "_code", "_workspace", "_sliced", "_prepared")

    def __init__(self, p: Plan):
        self._conf, self._trans = p._conf, p._trans         # (own the memory that the references point to)
        self._conf_ref = ctypes.byref(self._conf)
        self._trans_ref = ctypes.byref(self._trans) if self._trans is not None else None
        self._fn = p._fn
        self._workspace = _split_k_bytes(self._conf) if p._split_k else None
        self._code = None if p._split_k else p._args[-1]
        self._sliced = p._sliced
        self._prepared = None

    def __call__(self, a: int, b: int, c: int, stream: int) -> None:
        if self._sliced:
            workspace = _workspace_if_any(self._sliced, stream)
            rc = self._fn(self._conf_ref, a, b, c, c, self._trans_ref, None, self._code, *_span(workspace), stream)
        elif self._workspace is None:
            rc = self._fn(self._conf_ref, a, b, c, c, self._trans_ref, None, self._code, stream)
        else:
            workspace = _workspace(self._workspace, stream)
            rc = self._fn(self._conf_ref, a, b, c, c, self._trans_ref, None, *_span(workspace), stream)
        if rc != _lib.GK_OK:
            _raise(rc)


class _MulLaunchOnCopies(_MulLaunch):
    """The same on copies of the operands whose columns start off a 16-byte boundary (``packed_leading_dims``).  Copies of both operands
    are filled up with zeros to whole K tiles of 64: the partial one, which the kernels run outside their pipeline, takes some 10 us per
    round of tiles (the product on copies 4001 x 4003 x 4005 110 -> 100 us, from memory 136 -> 127), and sums of zeros change no bit.

    A call that finds no memory for the copies costs milliseconds (the allocator gives its cache back and waits for the device before it
    says so), so the calls behind it run on the operands as they lie and only every 256th tries again.  (The count is the one thing written
    after the launch is made: threads that meet on it try once more or less.)"""

    __slots__ = ("_packed", "_packed_ref", "_copies", "_copy_bytes", "_calls_without")

    def __init__(self, p: Plan, packed):
        super().__init__(p)
        self._packed = _lib.gk_config.from_buffer_copy(self._conf)
        self._packed_ref = ctypes.byref(self._packed)
        shape, self._copies, at = self._conf.matmul_shape, [], 0
        k = shape.K if None in packed else -(-shape.K // 64) * 64
        self._packed.matmul_shape.K = k
        for which, (layout, mine, ld, extent) in enumerate(((self._packed.global_a_layout, self._conf.global_a_layout, packed[0], shape.M),
                                                            (self._packed.global_b_layout, self._conf.global_b_layout, packed[1], shape.N))):
            if ld is None:
                continue
            (rows, cols), (rows_copy, cols_copy) = _stored(which, mine.kind, extent, shape.K), _stored(which, mine.kind, extent, k)
            self._copies.append((which, at, (rows, cols, mine.ld), (ld, rows_copy, cols_copy)))
            layout.ld = ld
            at += 2 * ld * cols_copy
        self._copy_bytes, self._calls_without = at, 0

    def _on_copies(self, a: int, b: int, c: int, stream: int) -> bool:
        """The product on copies of the operands whose columns start off a 16-byte boundary (the same launch, the same bits).
        False: not here -- no memory for the copies, or a capture, whose graph would have to keep them."""
        import torch
        # (`stream` is torch's current one: what torch says of captures and allocates is that stream's)
        if torch.cuda.is_current_stream_capturing():
            return False
        if self._calls_without > 0:
            self._calls_without -= 1
            return False
        # memory of this call alone, in the order of the stream: what gets it next on this stream runs behind the product
        try:
            copies = torch.empty(self._copy_bytes, dtype=torch.uint8, device="cuda")
        except torch.OutOfMemoryError:
            self._calls_without = _RETRY_AFTER - 1
            return False
        base, operands, jobs = copies.data_ptr(), [a, b], []
        for which, at, source, copy in self._copies:
            jobs += (operands[which], *source, base + at, *copy)
            operands[which] = base + at
        rc = _lib.lib().gk_pack_columns_padded(*jobs, *((None, 0, 0, 0, None, 0, 0, 0) if len(jobs) == 8 else ()), stream)
        if rc == _lib.GK_OK:
            rc = self._fn(self._packed_ref, *operands, c, c, self._trans_ref, None, self._code, stream)
        if rc != _lib.GK_OK:
            _raise(rc)
        return True

    def __call__(self, a: int, b: int, c: int, stream: int) -> None:
        if not self._on_copies(a, b, c, stream):
            super().__call__(a, b, c, stream)


# launches by kind of operands and factors; a program has few kinds, one that has more pays for lowering again
_mul_launches = {}
_MUL_LAUNCHES_MAX = 1024


class Transpose:
    """Lazy transpose wrapper, Julia's ``transpose(A)`` / ``A'`` (no conjugation, src/matmul.jl:211-213)."""

    def __init__(self, parent):
        self.parent = parent


Adjoint = Transpose


def mul_(C, A, B, alpha=True, beta=False):
    """``mul!`` (reference src/matmul.jl:207-215): unwraps Transpose/Adjoint and forwards."""
    tA, tB = isinstance(A, Transpose), isinstance(B, Transpose)
    if tA:
        A = A.parent
    if tB:
        B = B.parent
    alpha, beta = float(alpha), float(beta)
    if _native_mul(C, A, B, tA, tB, alpha, beta):
        return C
    return matmatmul_(C, 'T' if tA else 'N', 'T' if tB else 'N', A, B, alpha, beta)
