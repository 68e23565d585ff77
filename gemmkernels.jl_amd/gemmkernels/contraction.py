"""Planner for tensor contractions written the TCCG way, e.g. ``"abc-bda-dc"`` for
``D[a,b,c] = sum_d A[b,d,a] * B[d,c]`` (the contraction of the reference's benchmark script,
benchmarks/tensor-contractions/run.jl:10-21, where the index arithmetic is hand-written into four
Layout types, :22-85).  Here the arithmetic is derived from the mode strings:

1. modes are classified (M: in A and D, N: in B and D, K: in A and B);
2. neighbouring modes that are neighbours, in the same order, in both tensors that hold them are
   fused into one longer mode (longer first modes are what the kernel's 16-byte vectors and 32-wide
   accumulator blocks need);
3. both assignments of the two inputs to the kernel's A and B operands are tried (swapping them
   swaps the roles of M and N; the sum is the same);
4. a tile with tensor-contraction addressing is chosen whose BLOCK_K divides the first K mode;
5. the library validates the result; if no candidate passes, the reasons are reported.

Tensors are dense and column-major (first index fastest), as Julia arrays are.  Nothing is copied
or permuted: a contraction either maps onto one launch of the GEMM kernel or is refused.
"""
from __future__ import annotations

import ctypes
from dataclasses import dataclass
from typing import Dict, List, Optional, Sequence, Tuple

from . import _lib
from . import kernel as Kernel
from . import layout as Layout
from . import operator as Operator
from ._native import Prepared, load as native
from .config import _GETT_TILES, _mfma_cost, get_config
from .dtypes import BFloat16, DType, Float16, Float32
from .errors import ConfigError
from .tiling import NT


def parse(spec: str) -> Tuple[str, str, str]:
    """``"D-A-B"`` -> (d_modes, a_modes, b_modes); one letter per mode."""
    parts = spec.replace(" ", "").split("-")
    if len(parts) != 3 or not all(parts):
        raise ValueError(f"a contraction is written 'D-A-B' with one letter per mode, got {spec!r}")
    d, a, b = parts
    for name, modes in (("D", d), ("A", a), ("B", b)):
        if len(set(modes)) != len(modes):
            raise ValueError(f"mode repeated in {name}: {modes!r}")
    return d, a, b


def classify(d: str, a: str, b: str) -> Tuple[List[str], List[str], List[str]]:
    """M, N and K modes; batch modes (in all three tensors) and modes summed over a single tensor are
    not GEMM-shaped and are refused."""
    m = [ch for ch in a if ch in d and ch not in b]
    n = [ch for ch in b if ch in d and ch not in a]
    k = [ch for ch in a if ch in b and ch not in d]
    odd = [ch for ch in set(a + b + d) if ch not in m + n + k]
    if odd:
        raise ValueError("modes " + ", ".join(sorted(odd)) + " appear in all three tensors or in only one: not a GEMM-shaped contraction")
    if not m or not n or not k:
        raise ValueError("a contraction needs at least one M mode (A and D), one N mode (B and D) and one K mode (A and B)")
    return m, n, k


def fuse(d: str, a: str, b: str, extents: Dict[str, int]) -> Tuple[str, str, str, Dict[str, int], Dict[str, str]]:
    """Fuses modes x, y that directly follow each other (x before y) in every tensor that holds them.
    Returns the new mode strings and extents, and for every surviving letter the letters it stands for."""
    groups = {ch: ch for ch in set(d + a + b)}
    ext = dict(extents)
    tensors = [d, a, b]
    changed = True
    while changed:
        changed = False
        for t in tensors:
            for i in range(len(t) - 1):
                x, y = t[i], t[i + 1]
                holders = [u for u in tensors if x in u or y in u]
                if all((x in u) and (y in u) and u.index(y) == u.index(x) + 1 for u in holders):
                    ext[x] = ext[x] * ext[y]
                    groups[x] = groups[x] + groups[y]
                    del ext[y], groups[y]
                    tensors = [u.replace(y, "") for u in tensors]
                    changed = True
                    break
            if changed:
                break
    d2, a2, b2 = tensors
    return d2, a2, b2, ext, groups


@dataclass
class ContractionPlan:
    """What the planner decided, and the launch (``plan(...)`` returns it ready to call)."""
    spec: str
    swapped: bool                 # the second input runs as the kernel's A operand
    fused: Dict[str, str]         # surviving mode -> original modes it stands for
    conf: object
    gemm_shape: Tuple[int, int, int]
    kernel_name: str
    _launch: object = None

    def __call__(self, stream=None):
        return self._launch(stream)


def _shape_extents(modes: str, x, extents: Dict[str, int], name: str) -> None:
    shape = tuple(int(s) for s in x.shape)
    if len(shape) != len(modes):
        raise ConfigError(f"{name} has {len(shape)} dimensions, its mode string {modes!r} has {len(modes)}")
    stride = 1
    for ch, e, s in zip(modes, shape, x.stride()):
        if extents.setdefault(ch, e) != e:
            raise ConfigError(f"mode {ch!r} has extent {extents[ch]} in one tensor and {e} in {name}")
        if e > 1 and int(s) != stride:
            raise ConfigError(f"{name} must be dense and column-major (first index fastest); see gemmkernels.colmajor")
        stride *= e


def candidates(spec: str, extents: Dict[str, int], ab_type: DType = Float16, cd_type: DType = Float32, zero_c: bool = True):
    """Yields (swapped, fused groups, configuration or None, reason) for both operand assignments and
    every tile with contraction addressing, best first.  Needs no GPU."""
    from .matmul import kernel_name
    d, a, b = parse(spec)
    classify(d, a, b)
    d2, a2, b2, ext, groups = fuse(d, a, b, extents)
    for swapped in (False, True):
        am, bm = (b2, a2) if swapped else (a2, b2)
        gmap = Layout.gett_map(am, bm, d2, ext)
        M, N, K = gmap.extent("m"), gmap.extent("n"), gmap.extent("k")
        tiles = [t for t in _GETT_TILES if M % t[0] == 0 and N % t[1] == 0 and K % t[2] == 0]
        if not tiles:
            yield swapped, groups, None, (f"no tile divides M = {M}, N = {N} and K = {K} "
                                          f"(tiles {_GETT_TILES})")
            continue
        # the tile with the shortest estimated launch first; the library says which of them tile the K modes
        for t in sorted(tiles, key=lambda t: _mfma_cost(t, M, N, K, False)):
            try:
                conf = get_config(gemm_shape=NT(M=M, N=N, K=K), operator=Operator.MFMAOp[32, 32, 16, ab_type, Float32],
                                  global_a_layout=Layout.GETT[ab_type, gmap], global_b_layout=Layout.GETT[ab_type, gmap],
                                  global_c_layout=Layout.Zero[cd_type] if zero_c else Layout.GETT[cd_type, gmap],
                                  global_d_layout=Layout.GETT[cd_type, gmap],
                                  shared_a_layout=Layout.UnsafeAlignedColMajor[ab_type], shared_b_layout=Layout.UnsafeAlignedColMajor[ab_type],
                                  shared_c_layout=Layout.Zero[cd_type] if zero_c else Layout.UnsafeAlignedColMajor[cd_type],
                                  shared_d_layout=Layout.UnsafeAlignedColMajor[cd_type],
                                  block_shape=NT(M=t[0], N=t[1], K=t[2]), kernel=Kernel.matmul_pipelined)
                yield swapped, groups, conf, kernel_name(conf, Kernel.matmul_pipelined)
            except ConfigError as e:
                yield swapped, groups, None, f"tile {t}: {e.message}"


def plan(spec: str, a, b, d, c=None, ab_type: Optional[DType] = None, cd_type: Optional[DType] = None) -> ContractionPlan:
    """Plans ``D = sum A * B (+ C)`` for device tensors (dense, column-major) and returns the launch.
    ``c`` has the modes and the element type of ``d``; ``d`` may be ``c``."""
    from .dtypes import from_torch
    from .matmul import Plan, _DEFAULT_EPILOGUE, _IDENTITY, _HOOKS
    dm, am, bm = parse(spec)
    extents: Dict[str, int] = {}
    _shape_extents(am, a, extents, "A")
    _shape_extents(bm, b, extents, "B")
    _shape_extents(dm, d, extents, "D")
    if c is not None:
        _shape_extents(dm, c, extents, "C")
        if c.dtype != d.dtype:         # (the kernel reads C as it writes D: elements of another size lie elsewhere, also behind the end of C)
            raise ConfigError(f"C must have the element type of D: {c.dtype} and {d.dtype}")
    ab_type = ab_type or from_torch(a.dtype)
    cd_type = cd_type or from_torch(d.dtype)
    if ab_type not in (Float16, BFloat16) or from_torch(b.dtype) != ab_type:
        raise ConfigError("contractions run on the matrix cores: A and B must both be Float16 or both BFloat16")
    reasons = []
    for swapped, groups, conf, info in candidates(spec, extents, ab_type, cd_type, zero_c=c is None):
        if conf is None:
            reasons.append(("B as the A operand: " if swapped else "") + info)
            continue
        x, y = (b, a) if swapped else (a, b)
        launch = Plan(conf, x, y, c, d, {k: _IDENTITY for k in _HOOKS}, _DEFAULT_EPILOGUE, Kernel.matmul_pipelined, slices=True)
        ms = conf.matmul_shape
        return ContractionPlan(spec, swapped, groups, conf, (ms.M, ms.N, ms.K), info, launch)
    raise ConfigError("contraction " + spec + " does not map onto the GEMM kernel: " + "; ".join(reasons))


def contract(spec: str, a, b, d, c=None, stream=None):
    """``D[...] = sum A[...] * B[...] (+ C[...])`` in one launch on the current stream; returns ``d``."""
    from .matmul import _current_stream
    key = (spec, a.dtype, a.shape, a.stride(), b.dtype, b.shape, b.stride(), d.dtype, d.shape, d.stride(),
           None if c is None else (c.dtype, c.shape, c.stride()))
    launch = _launches.get(key)
    if launch is None:
        launch = _Launch(plan(spec, a, b, d, c))
        if len(_launches) >= _LAUNCHES_MAX:
            _launches.clear()
        _launches[key] = launch
    ready = launch.ready if stream is None else None             # (held while it is used)
    if ready is None or not ready[0](ready[1].handle, *((b, a) if launch._swapped else (a, b)), c, d):
        launch(a.data_ptr(), b.data_ptr(), None if c is None else c.data_ptr(), d.data_ptr(), _current_stream() if stream is None else int(stream))
    return d


class _Launch:
    """What ``contract`` hands to the library for operands of one kind (mode string, element types, extents, strides): the descriptor
    the planner arrived at, no address and no tensor; the library checks the addresses at every launch.  (What is written after it is made is how often it was
    called and, from the second call on, the launch checked once: threads that meet there make one too many.)  Planning again took 70 us of interpreter time a call, several times the kernel of a small contraction."""

    __slots__ = ("_conf", "_conf_ref", "_swapped", "_fn", "_code", "_sliced", "ready", "_calls")

    def __init__(self, p: ContractionPlan):
        self._conf = p._launch._conf                      # (owns the memory that the reference points to)
        self._conf_ref = ctypes.byref(self._conf)
        self._swapped = p.swapped
        self._fn, self._code, self._sliced = p._launch._fn, p._launch._args[-1], p._launch._sliced
        # (the launch checked once and gk_torch's way to it, for operands on 16-byte boundaries)
        self.ready = None
        self._calls = 0

    def __call__(self, a: int, b: int, c: Optional[int], d: int, stream: int) -> None:
        self._calls += 1
        if self._calls == 2 and not self._sliced and native() is not None:
            prepared = Prepared(self._conf, None, None, self._code)
            if prepared.handle is not None:
                self.ready = native().run, prepared
        x, y = (b, a) if self._swapped else (a, b)
        if self._sliced:
            from .matmul import _launch_sliced
            rc = _launch_sliced(self._conf, x, y, c, d, None, None, self._code, self._sliced, stream)
        else:
            from .matmul import _gk_matmul
            rc = _gk_matmul(self._conf, x, y, c, d, None, None, self._code, stream)
        if rc != _lib.GK_OK:
            from .matmul import _raise
            _raise(rc)


# launches by kind of operands; a program has few kinds, one that has more pays for planning again
_launches: Dict[tuple, _Launch] = {}
_LAUNCHES_MAX = 256
