"""Config and get_config (reference src/config.jl), with defaults re-derived for the MI355X:
64-lane wavefronts, 160 KiB of LDS per workgroup, MFMA 32x32x16 blocks."""
from __future__ import annotations

import ctypes
import math
import struct
from dataclasses import dataclass, fields
from typing import Optional

from . import _lib
from . import layout as Layout
from . import operator as Operator
from . import cta_swizzle as CTASwizzle
from .errors import ConfigError
from .tiling import NT

WARP_SIZE = 64   # lanes per wavefront; the reference's 32 (src/matmul.jl:24) becomes 64 here


@dataclass
class Config:
    """reference src/config.jl:3-41, field for field."""
    matmul_shape: NT
    block_shape: NT
    warps_per_block: int
    mem_a_warp: NT
    mem_a_thread: NT
    mem_b_warp: NT
    mem_b_thread: NT
    mem_cd_warp: NT
    mem_cd_thread: NT
    compute_warp: NT
    compute_op_shape: NT
    global_a_layout: Layout.LayoutType
    global_b_layout: Layout.LayoutType
    global_c_layout: Layout.LayoutType
    global_d_layout: Layout.LayoutType
    shared_a_layout: Layout.LayoutType
    shared_b_layout: Layout.LayoutType
    shared_c_layout: Layout.LayoutType
    shared_d_layout: Layout.LayoutType
    operator: Operator.OperatorType
    is_a_col_major: bool
    is_b_col_major: bool
    cta_swizzle: CTASwizzle.SwizzleType

    def __str__(self):
        # reference src/config.jl:43-76
        width = max(len(f.name) for f in fields(self)) + 2
        return "\n".join(f"{(f.name + ':').ljust(width)}{getattr(self, f.name)}" for f in fields(self)) + "\n"

    def __getstate__(self):
        # (copies and pickles: the fields and whether the tile was left open; descriptors and launches that were kept are made again)
        mine = {f.name: getattr(self, f.name) for f in fields(self)}
        if "_tile_left_open" in self.__dict__:
            mine["_tile_left_open"] = self.__dict__["_tile_left_open"]
        return mine

    def to_c(self, lda: int = 0, ldb: int = 0, ldc: int = 0, ldd: int = 0) -> _lib.gk_config:
        """Lower to the POD of the C ABI; leading dimensions come from the arrays of the call.
        The result is cached per set of leading dimensions (a Config is immutable once built)."""
        cache = self.__dict__.setdefault("_c_cache", {})
        key = (lda, ldb, ldc, ldd)
        hit = cache.get(key)
        if hit is not None:
            return hit
        c = _lib.gk_config()
        # (whole structs at their offsets: member by member this was half of a first launch's time on the host)
        mine = self.__dict__
        for name, at in _SHAPES_AT:
            src = mine[name].get
            try:
                _SHAPE.pack_into(c, at, int(src("M", 0)), int(src("N", 0)), int(src("K", 0)))
            except struct.error:
                raise ConfigError(f"{name} must be below 2^31, got {tuple(mine[name].values())}") from None
        c.warps_per_block = int(self.warps_per_block)
        for (name, at), ld in zip(_LAYOUTS_AT, (lda, ldb, ldc, ldd, 0, 0, 0, 0)):
            src = mine[name]
            _LAYOUT.pack_into(c, at, src.kind, src.T.code, src.pad, 0, int(ld))
        op = self.operator
        c.op.kind, c.op.M, c.op.N, c.op.K = op.kind, op.M, op.N, op.K
        c.op.mb, c.op.nb, c.op.kb = op.mb, op.nb, op.kb
        c.op.compute_type, c.op.accum_type = op.CT.code, op.AT.code
        c.is_a_col_major, c.is_b_col_major = int(self.is_a_col_major), int(self.is_b_col_major)
        c.cta_swizzle.kind, c.cta_swizzle.param = self.cta_swizzle.kind, self.cta_swizzle.param
        gmap = None
        for l in (self.global_a_layout, self.global_b_layout, self.global_c_layout, self.global_d_layout):
            if l.kind == Layout.GETT_KIND and l.gett is not None:
                gmap = l.gett
        if gmap is not None:
            for dst, src in ((c.gett.m, gmap.m), (c.gett.n, gmap.n), (c.gett.k, gmap.k)):
                if len(src) > _lib.GK_MAX_MODES:
                    raise ConfigError(f"at most {_lib.GK_MAX_MODES} tensor modes per GEMM dimension")
                dst.nmodes = len(src)
                for i, (e, s0, s1) in enumerate(src):
                    dst.extent[i], dst.stride0[i], dst.stride1[i] = int(e), int(s0), int(s1)
        cache[key] = c                      # (whole: other threads may look for it meanwhile)
        return c


_SHAPE, _LAYOUT = struct.Struct("=3i"), struct.Struct("=4iq")
_SHAPES_AT = tuple((name, getattr(_lib.gk_config, name).offset) for name in (
    "matmul_shape", "block_shape", "mem_a_warp", "mem_a_thread", "mem_b_warp", "mem_b_thread", "mem_cd_warp", "mem_cd_thread", "compute_warp", "compute_op_shape"))
_LAYOUTS_AT = tuple((name, getattr(_lib.gk_config, name).offset) for name in (
    "global_a_layout", "global_b_layout", "global_c_layout", "global_d_layout", "shared_a_layout", "shared_b_layout", "shared_c_layout", "shared_d_layout"))
assert _SHAPE.size == ctypes.sizeof(_lib.gk_shape) and _LAYOUT.size == ctypes.sizeof(_lib.gk_layout)


def heuristic_block_shape(shared_a_layout, shared_b_layout, shared_c_layout, shared_d_layout) -> NT:
    """The reference's block-shape heuristic, unchanged (src/config.jl:84-120): grow M and N while
    a C/D tile fits 64 KiB, then K while the A and B tiles fit 64 KiB together."""
    def nbytes(layout, a, b):
        size = Layout.physical_size(layout, (a, b))
        n = 1
        for s in size:
            n *= s
        return n * layout.T.size

    def num_bytes_cd(M, N, K):
        return max(nbytes(shared_c_layout, M, N), nbytes(shared_d_layout, M, N))

    def num_bytes_ab(M, N, K):
        return nbytes(shared_a_layout, M, K) + nbytes(shared_b_layout, K, N)

    def next_mn(M, N, K):
        return (2 * M, N, K) if M == N else (M, 2 * N, K)

    cur = (1, 1, 1)
    nxt = next_mn(*cur)
    while num_bytes_cd(*nxt) <= 64 * 1024:
        cur, nxt = nxt, next_mn(*nxt)
    nxt = (cur[0], cur[1], 2 * cur[2])
    while num_bytes_ab(*nxt) <= 64 * 1024:
        cur, nxt = nxt, (nxt[0], nxt[1], 2 * nxt[2])
    return NT(M=cur[0], N=cur[1], K=cur[2])


def adjacent_elements(num: int, parent_size: NT, is_col_major: bool) -> NT:
    """reference src/config.jl:124-134."""
    p = tuple(parent_size.values())
    if is_col_major:
        t = (min(num, p[0]), num // min(num, p[0]))
    else:
        t = (num // min(num, p[1]), min(num, p[1]))
    return NT(zip(parent_size.keys(), t))


# MFMA tile table of the library: block shape -> waves (M x N).  The wave tile (compute_warp) is
# block / waves; every entry is made of 32x32 MFMA blocks.
_MFMA_TILES = [
    ((256, 256, 64), (2, 4)),
    ((256, 256, 32), (2, 4)),     # for K that is a multiple of 32 only (6 % behind 256x256x64; 4 x 2 waves: 10 %)
    ((256, 128, 64), (2, 2)),
    ((128, 256, 64), (2, 2)),
    ((128, 128, 32), (2, 2)),     # four stages: measured ahead of 128x128x64 with two stages on 2048-sized problems
    ((128, 128, 64), (2, 2)),
    ((64, 64, 64), (2, 2)),
    ((64, 64, 32), (2, 2)),       # four stages; the one-wave instance (the tensor-contraction kernels have only that) is 1.5 - 2.7 times slower
]
# Tiles with a side of 192: they fill the chip where 256 x 256 leaves CUs idle (3072^2: 192 tiles instead of 144,
# 56 us instead of 68).  Compiled per transpose: 256 x 192 for 'N','N', 'T','N' and 'N','T'; 192 x 256 for
# 'T','N' and 'T','T' (the third entry says whether a transpose (a_kmajor, b_kmajor) has the tile).
_MFMA_TILES_192 = [((256, 192, 64), (4, 2), lambda a_kmajor, b_kmajor: b_kmajor or not a_kmajor),
                   ((192, 256, 64), (2, 4), lambda a_kmajor, b_kmajor: a_kmajor)]
NUM_CUS = 256

# measured winners by problem (filled by gemmkernels.tuning.install / load, or from the JSON file
# named by the environment variable GEMMKERNELS_TUNING_TABLE)
TUNED = {}


# tiles compiled with tensor-contraction addressing
_GETT_TILES = [(256, 256, 64), (128, 128, 64), (64, 64, 64), (64, 64, 32)]


def _tiles_k_modes(extents, block_k) -> bool:
    """Whether a K tile of a contraction is a whole number of leading K modes times a divisor of the next one."""
    whole = 1
    for extent in extents:
        if block_k % whole != 0:
            return False
        need = block_k // whole
        if need <= extent:
            return extent % need == 0
        whole *= extent
    return False


def _mfma_tiles(a_kmajor: bool, b_kmajor: bool):
    return [t for t, _ in _MFMA_TILES] + [t for t, _, has in _MFMA_TILES_192 if has(a_kmajor, b_kmajor)]


def default_block_shape(operator, gemm_shape, tile_sized: bool = True, gett: bool = False, planar: bool = False,
                        a_kmajor: bool = False, b_kmajor: bool = True, k_modes=None) -> NT:
    """MI355X block shape: of the tiles of the table that divide the problem, the one with the shortest
    estimated launch (tiles per CU times the cost of a tile).  ``a_kmajor``: A is stored K x M ('T');
    ``b_kmajor``: B is stored K x N ('N'); they admit the tiles with a side of 192.  ``k_modes``: extents of the K modes of a
    contraction, which a K tile has to divide evenly as well."""
    M, N, K = gemm_shape["M"], gemm_shape["N"], gemm_shape["K"]
    if operator.kind in (Operator.FPU, Operator.FPU_TROPICAL):
        costs = _FPU_TILE_COST.get((operator.CT.name, operator.AT.name), {}) if operator.kind == Operator.FPU else {}
        fitting = [t for t in costs if not tile_sized or (M % t[0] == 0 and N % t[1] == 0 and K % t[2] == 0)]
        if not fitting:
            return NT(M=64, N=64, K=32)

        def fpu_cost(t):
            rounds = -(-(-(-M // t[0]) * -(-N // t[1])) // NUM_CUS)
            return costs[t][0] if rounds == 1 else costs[t][1] * rounds
        best = min(fitting, key=fpu_cost)
        return NT(M=best[0], N=best[1], K=best[2])
    if operator.kind in (Operator.MFMA_COMPLEX, Operator.MFMA_DUAL):
        # complex tiles, in complex elements
        table = _complex_tiles(operator, planar, a_kmajor, b_kmajor)
        fitting = [t for t, _ in table if M % t[0] == 0 and N % t[1] == 0 and K % t[2] == 0]
        if not fitting:
            return NT(M=64, N=64, K=32)
        # (one real product of twice the rows and columns; 32 x 32 x 64 has four LDS stages, of which a CU holds two tiles)
        fitting = [t for t in fitting if t != (32, 32, 64) or (M // 32) * (N // 32) <= 2 * NUM_CUS] or fitting
        best = min(fitting, key=lambda t: (_mfma_cost((2 * t[0], 2 * t[1], t[2]), 2 * M, 2 * N, K, False), fitting.index(t)))
        return NT(M=best[0], N=best[1], K=best[2])
    # sizes need not be whole tiles when the layouts are the bounds-checked ones (the aligned kernels mask the
    # last tile row / column and zero the end of the last K tile)
    table = _mfma_tiles(a_kmajor, b_kmajor)
    fitting = [t for t in table if not tile_sized or (M % t[0] == 0 and N % t[1] == 0 and K % t[2] == 0)]
    if gett:
        fitting = [t for t in fitting if t in _GETT_TILES and (k_modes is None or _tiles_k_modes(k_modes, t[2]))]
    if not fitting:
        return NT(M=64, N=64, K=32)
    # the shortest estimated launch (_MFMA_TILE_COST); ties go to the tile listed first
    best = min(fitting, key=lambda t: (_mfma_cost(t, M, N, K, not gett), fitting.index(t)))
    return NT(M=best[0], N=best[1], K=best[2])


def split_k_block_shape(M, N, K, widest_ld=0, factor=None) -> Optional[NT]:
    """The tile of a 16-bit product with few output tiles and a long K, which is cut into slices of K (``Kernel.matmul_split_k``), or None (the
    default tile, and one chain over K).  us, slices and unsplit on four LDS stages, inputs that rotate through 400 MB, 'N','N':
        64 tiles (4096 x 64)        K = 1280 9.6 and 10.7, 2048 10.4 and 14.3, 4096 14.0 and 25.6
        128 tiles (8192 x 64)       K = 1280 10.6 and 11.1, 2048 13.7 and 14.8
        165 tiles, three slices     K = 3072 15.5 and 17.0, 4096 17.9 and 21.3

    171 to 256 tiles leave two slices, which are there for the error as well: half the chain has 2.9e-7 of the norm where the whole has 4.1e-7
    (K = 4096, FP16 uniform in [-1, 1); 1.5e-7 and 3e-7 on values of one sign; 4.1 and 5.7e-7, 2.2 and 4.3e-7 at K = 8192).  Their time, two
    slices and unsplit, 'N','N' / 'T','N':
        K = 3072     256 tiles 21.0 and 19.3 / 19.2 and 17.2
        K = 4096     180 tiles 19.4 and 21.7 / 18.4 and 20.6, 256 tiles 25.3 and 24.3 / 22.6 and 20.6
        K = 8192     180 tiles 32.1 and 39.3 / 30.7 and 35.8, 210 tiles 32.4 and 38.7 / 31.5 and 36.3, 256 tiles 43.4 and 44.9 / 36.9 and 36.5
        K = 16384    256 tiles 79.9 and 86.4 / 68.4 and 70.7
        K = 3328     1001 x 704 24.8 and 23.4 / 19.3 and 18.0;    K = 4004     1024 x 768 26.2 and 30.7 / 32.6 and 32.1
    Not where K and the output are both ragged (1001 x 700 x 3333, 1000 x 1000 x 4000).

    ``factor``: alpha stays in the K loop (None: it does not), which makes it longer, and two slices are taken whatever the extents.  FP16
    111 x 2629 x 1477 (84 tiles) 12.9 and 16.4.  BF16, two slices and unsplit: 768 x 1024 x 4096 23.6 and 26.5, 960 x 896 x 8192 41.0 and 49.0,
    1024 x 1024 x 4096 26.6 and 26.9, 1001 x 1001 x 5001 42.2 and 41.6, 1000 x 900 x 3001 26.4 and 26.1; and with an extent that fills no tile or
    one, where the slices are behind, 70 x 7000 x 3500 28.9 and 26.1, 12000 x 64 x 4096 32.3 and 27.8.

    ``widest_ld``: the larger leading dimension of the operands whose rows are the k of a tile; the kernel keeps the offsets in a tile in 32
    bits, so 64 rows of 2^24 elements are left to a tile with fewer."""
    if 64 * widest_ld * 2 >= 1 << 31:
        return None
    tiles = -(-M // 64) * -(-N // 64)
    if tiles <= 128:
        worth = K >= 1280
    else:
        two = factor is not None or K % 64 == 0 or M % 64 == 0 and N % 64 == 0
        worth = K >= 3000 and (tiles <= 170 or tiles <= 256 and two)
    return NT(M=64, N=64, K=64) if worth else None


def sliced_block_shape(M, N, K, widest_ld=0, odd=False) -> Optional[NT]:
    """128 x 128 x 64 for a 16-bit product whose tiles of that size leave CUs idle and whose K is long enough for slices of them to be ahead of
    tiles of 64 x 64, cut or not (``gk_matmul_sliced``), or None.  A 64 x 64 tile brings twice the bytes per product into a CU, and more than 256 of
    them are not cut (a few more than 256 take as long as 512).  us, 64 x 64 -> 128 x 128 in slices, inputs that rotate:
        1472 x 768 x 5888 'N','T' 34.2 -> 24.0, 1088 x 1088 x 5248 'N','T' 31.5 -> 24.3, 704 x 1664 x 4544 'T','T' 26.6 -> 22.3,
        2944 x 384 x 3712 24.0 -> 19.2; below the line 384 x 4160 x 2496 18.0 and 21.5, 1088 x 1728 x 3136 21.6 and 26.7.
    ``odd``: an operand whose columns start off 16-byte boundaries, whose rows of a small tile lie on relatively more lines:
        326 x 3462 x 3056 'T','T' 26.6 -> 19.5, 2048 x 560 x 2542 'T','N' 22.3 -> 18.5, 2624 x 517 x 3296 32.1 -> 24.1,
        539 x 2592 x 7990 with a factor 79.9 -> 50.7.
    Error against 64 bits: never larger than that of the one chain it replaces (two slices or three).
    ``widest_ld``: the largest leading dimension; the kernel keeps the offsets in a tile in 32 bits."""
    tiles, small = -(-M // 128) * -(-N // 128), -(-M // 64) * -(-N // 64)
    if small <= 256 or tiles > 128 or K < (2500 if odd else 3500) or 128 * widest_ld * 2 >= 1 << 31:
        return None
    return NT(M=128, N=128, K=64)


# Estimated launch time of a tile, in microseconds: what a launch costs whatever its size, per 1000 k and round, per further tile of
# a CU, for a partial last K tile (times the square root of the rounds), for tiles over the edges.  Fitted, weighted towards the tiles near the
# best, to timings of every tile at 61 sizes from 1000 x 1000 x 64 to 4416 x 4416 x 1024 ('N','N' and 'T','N'; whole tiles, multiples of 64 and odd ones; inputs
# that rotate through 200 MB and more): the tile the estimate picks is 1.5 % behind the best one on average, 11 % at most.  E.g. 1024^3 7.6 us on 64 x 64 x 64,
# 12.6 on 128 x 128 x 64, 25.8 on 256 x 256 x 64; 2048^3 26.6, 23.5 and 41.1; 4096 x 2048 x 4096 92, 64.5 and 71.9; 3072^3 51.8 on
# 256 x 192 x 64, 58.8 on 256 x 256 x 64; 5913 x 6229 x 20 39.0 on 64 x 64 x 32, 53.4 on 64 x 64 x 64, 66.6 on 256 x 256 x 64.
_MFMA_TILE_COST = {(256, 256, 64): (12.0, 16.4, 39.0, 21.0, 1.2), (256, 256, 32): (12.2, 29.2, 20.7, 5.7, 6.8),
                   (256, 128, 64): (8.8, 13.5, 7.8, 15.5, 7.9), (128, 256, 64): (8.9, 12.9, 7.4, 17.4, 7.4),
                   (128, 128, 32): (6.7, 7.5, 1.9, 4.9, 3.6), (128, 128, 64): (6.7, 7.5, 1.9, 8.5, 3.6),
                   (64, 64, 64): (3.5, 3.5, 0.4, 3.7, 1.6), (64, 64, 32): (3.3, 4.6, 0.4, 2.0, 1.6),
                   (256, 192, 64): (5.4, 17.1, 19.3, 9.1, 7.9), (192, 256, 64): (5.0, 17.1, 15.3, 10.4, 7.9)}


# The same for plain products on any leading dimension, closer: the five above, per operand whose columns start off 16-byte boundaries (contiguous
# along k, along m or n) what the K loop takes longer, per MB of C and D, and of the smaller tiles how many tile times one to two (a + b (tiles per
# CU - 1)) and more of them in a CU take.  Fitted to 1500 products drawn like those that `mul_` is timed on, extents 16 to 8192, every tile of each,
# and the sliced launches of 128 x 128 x 64 (us, per 1000 k, per slice, per workgroup of a CU, for a partial last K tile).  _MFMA_TILE_COST stays the
# estimate of what this one knows nothing of: contractions, complex and configured products, copies, and the default that it has to be ahead of.
_PRODUCT_COST = {(256, 256, 64): (1.89, 20.31, 8.62, 2.54, 3.74, 0.22, 0.08, 0.16), (256, 256, 32): (0, 23.88, 4.11, 1.26, 5.98, 0.17, 0.01, 0.19),
                 (256, 128, 64): (4.72, 12.53, 5.58, 2.69, 1.4, 0.18, 0.08, 0.13), (128, 256, 64): (4.74, 13, 5.41, 3, 1.35, 0.18, 0.1, 0.13),
                 (128, 128, 32): (3.71, 7.92, 1.13, 0.9, 0.82, 0.34, 0.08, 0.12), (128, 128, 64): (3.65, 7.93, 0.99, 1.52, 0.78, 0.22, 0.11, 0.12),
                 (64, 64, 64): (2.88, 3.35, 0, 0.76, 0.52, 0.22, 0.22, 0.11), (64, 64, 32): (3.05, 3.56, 0.03, 0.44, 0.39, 0.23, 0.19, 0.11),
                 (256, 192, 64): (0.06, 18.16, 2.52, 1.82, 4.96, 0.2, 0.08, 0.19), (192, 256, 64): (3.72, 19.02, 2.44, 2.94, 0.35, 0.15, 0.14, 0.19)}
_PRODUCT_ROUNDS = {(128, 128, 32): (0.75, 0.09, 1.59), (128, 128, 64): (0.49, 0.23, 1.66), (64, 64, 64): (0.75, 0.33, 1.08), (64, 64, 32): (0.62, 0.41, 1.12)}
_PRODUCT_IN_SLICES = (2.88, 8.35, 1.06, 3.36, 0.04)
_PRODUCT_FITTED_TO = 8192


def _product_slices(t, M, N, K) -> int:
    """How many slices of K the library cuts a plain product on this tile into (``gk_matmul_sliced``; 128 x 128 x 64 only)."""
    tiles = -(-M // t[0]) * -(-N // t[1])
    return min(NUM_CUS // tiles, K // (768 if tiles <= 85 else 1024)) if t == (128, 128, 64) and tiles <= 128 and K >= 2048 else 1


def _product_cost(t, M, N, K, odd, cd_bytes):
    """Estimated microseconds of a plain product; ``odd``: operands whose columns start off 16-byte boundaries, contiguous along k and not;
    ``cd_bytes``: of C and D per output."""
    fixed, per_k, further, tail, edges, odd_k, odd_mn, per_mb = _PRODUCT_COST[t]
    tiles = -(-M // t[0]) * -(-N // t[1])
    per_k *= 1.0 + odd_k * odd[0] + odd_mn * odd[1]
    always = per_mb * 1e-6 * M * N * cd_bytes + (edges if M % t[0] or N % t[1] else 0.0)
    slices = _product_slices(t, M, N, K)
    if slices > 1:
        own = _PRODUCT_IN_SLICES
        chain = own[1] * per_k / _PRODUCT_COST[t][1] * -(-K // (64 * slices)) * 0.064
        return always + own[0] + chain + own[2] * slices + own[3] * slices * tiles / NUM_CUS + (own[4] if K % 64 else 0.0)
    per_cu = tiles / NUM_CUS
    if t not in _PRODUCT_ROUNDS:
        rounds = -(-tiles // NUM_CUS)
    elif per_cu <= 1:
        rounds = 1.0
    else:
        second, more, full = _PRODUCT_ROUNDS[t]
        rounds = 1.0 + second + more * (per_cu - 1.0) if per_cu <= 2 else full * (-(-tiles // (2 * NUM_CUS)) if t[0] == 128 else per_cu)
    return always + fixed + rounds * per_k * K * 1e-3 + further * max(per_cu - 1.0, 0.0) + (tail * rounds ** 0.5 if K % t[2] else 0.0)


def product_block_shape(block, M, N, K, a_kmajor, b_kmajor, odd, cd_bytes, lda=0, ldb=0) -> NT:
    """The tile of a plain 16-bit product whose default is ``block``: another one where the closer estimate has it 8 % ahead, which it was at every
    one of 344 products that the fit had not seen (at 5 % one in a hundred was slower, by up to 7 %).  Not for products small enough to end within
    the launch and its ends, nor for odd operands of a product that may run on copies of them.  us on the default and on this one, inputs that
    rotate: 1110 x 6976 x 1284 'T','N' 43.7 and 34.1, 646 x 5207 x 960 'N','T' 23.2 and 18.7, 2336 x 266 x 7288 'N','T' 34.5 and 24.7 (in slices),
    6236 x 96 x 6584 35.3 and 27.6 (in slices), 2632 x 2392 x 259 with C 20.5 and 18.1; the other 51 of 60 drawn ones within 2 %.

    The fit knows extents up to 8192.  Beyond (to 262144), of 70 drawn products that it moved 17 were slower, none of them in slices
    (1387 x 169454 x 71 253.6 and 424.4, 14832 x 552 x 64584 1391 and 1559), so only the slices are taken there: of 50 others all faster, on
    average 1.7 times (1792 x 464 x 65960 309 and 195, 568 x 1424 x 37808 227 and 111).

    ``lda``, ``ldb``: a tile whose rows lie too far apart for the kernels' offsets in 32 bits is refused by the library, so it is none of the
    candidates."""
    work = M * N * K
    if work < 5e8 or sum(odd) and work >= 2.4e10:
        return block
    own = (block.M, block.N, block.K)
    tiles = _mfma_tiles(a_kmajor, b_kmajor)
    if max(M, N, K) > _PRODUCT_FITTED_TO:
        tiles = [t for t in tiles if t == own or _product_slices(t, M, N, K) > 1]
    tiles = [t for t in tiles if t == own or max((t[0] if a_kmajor else t[2]) * lda, (t[1] if b_kmajor else t[2]) * ldb) * 2 < 1 << 31]
    cost = {t: _product_cost(t, M, N, K, odd, cd_bytes) for t in tiles}
    best = min(cost, key=cost.get)
    return NT(M=best[0], N=best[1], K=best[2]) if own in cost and cost[best] < 0.92 * cost[own] else block


def _rounds(t, tiles):
    """How many tile times a launch of ``tiles`` tiles of shape ``t`` takes.  A CU holds one workgroup of the tiles with
    144 or 128 KiB of LDS at a time: whole rounds.  The 128 x 128 tiles run one per CU on four LDS stages where every tile has a CU,
    and two per CU on two stages beyond that (tiles per CU and tile times: 1.1 1.55, 1.27 1.6, 1.56 1.77, 2.0 1.9; 2.25 3.7, 3.5 3.9, 4.8 6.7).  The 64 x 64
    tiles: two of four stages side by side take 1.8 times one (2048 x 1024 x 4096 29.5 us, 1024 x 1024 x 4096 18.7), more of two stages share a CU
    at one tile time each."""
    per_cu = tiles / NUM_CUS
    if t[0] * t[1] >= 128 * 256:
        return -(-tiles // NUM_CUS)
    if per_cu <= 1:
        return 1.0
    if t[0] * t[1] >= 128 * 128:
        rounds = 1.3 + 0.28 * per_cu if per_cu <= 2 else 1.85 * -(-tiles // (2 * NUM_CUS))
        return rounds if t[2] >= 64 else 1.15 * rounds
    return 1.0 + 0.82 * (per_cu - 1.0) if per_cu <= 2 else 0.95 * per_cu


def _mfma_cost(t, M, N, K, pairs=True):
    """Estimated microseconds of a product in real tiles of shape ``t`` (``pairs``: a plain one)."""
    tiles = -(-M // t[0]) * -(-N // t[1])
    if pairs and t == (64, 64, 32) and tiles <= 2 * NUM_CUS and (K % 64 == 0 or K >= 1536):
        # the library runs these on 64 x 64 x 64 with four stages; a lone workgroup on a long K is named 64 x 64 x 32 (any leading dimension)
        return _mfma_cost((64, 64, 64), M, N, K) - (0.01 if tiles <= NUM_CUS and K >= 2048 else 0.0)
    fixed, per_k, further, tail, edges = _MFMA_TILE_COST[t]
    rounds = _rounds(t, tiles)
    return (fixed + rounds * per_k * K * 1e-3 + further * max(tiles / NUM_CUS - 1.0, 0.0) + (tail * rounds ** 0.5 if K % t[2] else 0.0)
            + (edges if M % t[0] or N % t[1] else 0.0))


# FPUOp on the FP32 / FP64 matrix instructions: time of a tile per 1000 k, in microseconds, when every CU has one tile at most
# and per tile when a CU has several (they are bound by the matrix cores, so the tiles of a CU add up, and a launch
# takes as long as the CU with the most).  Measured, e.g. Float32: 2048^3 134 us on 128 x 128 (256 tiles), 142 on 64 x 64 (1024);
# 2560^3 324 against 302 (400 and 1600 tiles: 2 and 7 rounds); 1024^3 68, 24.5 and 26 us on 128 x 128, 64 x 64 (256 tiles) and
# 32 x 32 (1024); 768^3 53, 19 and 17 (576 tiles of 32 x 32).  Float64: 1000^3 41.3 us on 64 x 64, 41.1 on 32 x 32; 2048^3 270, 305.
_FPU_TILE_COST = {("Float32", "Float32"): {(128, 128, 32): (65.0, 63.0), (64, 64, 32): (21.0, 17.8), (32, 32, 32): (9.0, 6.1)},
                  ("Float64", "Float64"): {(64, 64, 32): (38.0, 33.0), (32, 32, 32): (14.0, 9.8)}}

# complex / dual tiles (complex elements) -> waves: one real product of the real views of A and B, whose real tile
# has twice the rows and columns; the same table for every transpose
_COMPLEX_PAIR_TILES = [((128, 128, 64), (2, 4)), ((64, 64, 64), (2, 2)), ((64, 64, 32), (2, 2)), ((32, 32, 64), (2, 2)), ((32, 32, 32), (2, 2))]

# complex tiles (complex elements) of the kernel for planar global matrices -> waves; the real tile has twice
# the rows and columns (both planes of A, B and D)
_PLANAR_TILES = [((128, 128, 64), (2, 4)), ((64, 64, 64), (2, 2)), ((64, 64, 32), (2, 2)), ((32, 32, 64), (2, 2)), ((32, 32, 32), (2, 2))]

# tiles of FPUOp and of the bounds-checked MFMA kernel
_FPU_TILES = [((64, 64, 32), (2, 2)), ((128, 128, 16), (2, 2)), ((128, 128, 32), (2, 2)), ((32, 32, 32), (2, 2)), ((32, 32, 32), (1, 1))]
_CHECKED_TILES = [((64, 64, 32), (2, 2))]


def _complex_tiles(operator, planar, a_kmajor, b_kmajor):
    """(tile, waves) of the complex / dual instances for these layouts, in order of preference."""
    return _PLANAR_TILES if planar else _COMPLEX_PAIR_TILES


# One wave per SIMD: 256 x 256 x 64 on four waves with 128 x 128 wave tiles (a third fewer LDS reads per MFMA than
# 2 x 4 waves, and a K loop written out slot by slot: 105 against 116 us at 4096^3).  Compiled for plain products
# without hooks (whole tiles, or any extents with an FP32 C / D) and with hooks of D in closed form; the library runs
# the 2 x 4 arrangement of the same block shape, with the same bits, for any other launch of such a configuration.
_SOLO_TILE, _SOLO_WAVES = (256, 256, 64), (2, 2)
_SOLO_COMPLEX_TILE = (128, 128, 64)        # in complex elements


def _default_waves(operator, block_shape, checked=False, planar=False, gett=False, a_kmajor=False, b_kmajor=True, whole_tiles=False):
    key = (block_shape["M"], block_shape["N"], block_shape["K"])
    if gett and key == (64, 64, 32):
        return (1, 1)
    if operator.kind == Operator.MFMA and key == _SOLO_TILE and whole_tiles:
        return _SOLO_WAVES
    # ... and the tiles with a side of 192 (wave tiles of 128 x 96 / 96 x 128; 3072^3: 56 us against 62 on eight waves,
    # 'N','T' 57 against 65); the library runs the eight waves for what these instances do not cover (hooks, a bias,
    # tiles over the edges, a C / D that does not take 16-byte accesses)
    if operator.kind == Operator.MFMA and not gett and whole_tiles and any(key == t for t, _, _ in _MFMA_TILES_192):
        return _SOLO_WAVES
    # ... and the complex / dual product on interleaved matrices of an 'N','N' launch, whose real tile is that tile
    # (planar matrices: every transpose)
    if (operator.kind in (Operator.MFMA_COMPLEX, Operator.MFMA_DUAL) and key == _SOLO_COMPLEX_TILE and whole_tiles
            and (planar or (not a_kmajor and b_kmajor))):
        return _SOLO_WAVES
    if operator.kind in (Operator.FPU, Operator.FPU_TROPICAL):
        table = _FPU_TILES
    elif operator.kind == Operator.MFMA and checked and any(t == key for t, _ in _CHECKED_TILES):
        table = _CHECKED_TILES
    elif operator.kind in (Operator.MFMA_COMPLEX, Operator.MFMA_DUAL):
        table = _complex_tiles(operator, planar, a_kmajor, b_kmajor)
    else:
        table = _MFMA_TILES + [(t, w) for t, w, _ in _MFMA_TILES_192]
    for t, w in table:
        if t == key:
            return w
    return None


def require_tile_sized_global(layout) -> bool:
    """reference src/config.jl:175-178."""
    return layout.kind not in (Layout.ZERO, Layout.COL_MAJOR, Layout.ROW_MAJOR)


def get_config(*, gemm_shape, operator, global_a_layout, global_c_layout, **params) -> Config:
    """reference src/config.jl:180-316.  Same keywords; defaults for the parameters the caller
    leaves out are chosen for the MI355X.  All checks of the reference are run (by the library,
    through gk_validate) and raise ConfigError."""
    gemm_shape = NT(gemm_shape)
    global_b_layout = params.get("global_b_layout", global_a_layout)
    global_d_layout = params.get("global_d_layout", global_c_layout)

    def padded(l):
        return Layout.Padded[l, 16 // l.T.size] if l.kind not in (Layout.ZERO, Layout.DIAGONAL, Layout.GETT_KIND) else l

    shared_a_layout = params.get("shared_a_layout", padded(global_a_layout))
    shared_b_layout = params.get("shared_b_layout", padded(global_b_layout))
    shared_c_layout = params.get("shared_c_layout", global_c_layout)
    shared_d_layout = params.get("shared_d_layout", global_d_layout)

    tile_sized = any(require_tile_sized_global(l) for l in (global_a_layout, global_b_layout, global_c_layout, global_d_layout))
    block_shape = params.get("block_shape")
    if block_shape is None and operator.kind == Operator.MFMA and TUNED:
        # a measured winner for exactly this problem (gemmkernels.tuning), unless the caller chose otherwise
        key = (f"mfma/{global_a_layout.T.name}/{'N' if params.get('is_a_col_major', True) else 'T'}"
               f"{'N' if params.get('is_b_col_major', True) else 'T'}/{gemm_shape.M}x{gemm_shape.N}x{gemm_shape.K}")
        hit = TUNED.get(key)
        aligned = all(l.kind in (Layout.ALIGNED_COL_MAJOR, Layout.ALIGNED_ROW_MAJOR, Layout.ZERO)
                      for l in (global_a_layout, global_b_layout, global_c_layout, global_d_layout))
        if hit is not None and aligned:
            bm, bn, bk = hit["block"]
            wm, wn = hit["waves"]
            block_shape = NT(M=bm, N=bn, K=bk)
            params.setdefault("warps_per_block", wm * wn)
            params.setdefault("compute_warp", NT(M=bm // wm, N=bn // wn, K=16))
            params.setdefault("cta_swizzle", CTASwizzle.XCDAware[int(hit.get("panel", 4))])
    if block_shape is None and global_a_layout.kind == Layout.DIAGONAL and gemm_shape.M % 64 == 0 and gemm_shape.N % 64 == 0:
        # a diagonal A makes the product a streaming pass over B and D: many small workgroups keep more
        # memory requests in flight than a few large ones (measured against HBM with rotating buffers)
        block_shape = NT(M=64, N=64, K=32 if gemm_shape.K % 32 == 0 else gemm_shape.K)
        params.setdefault("warps_per_block", 4)
        params.setdefault("compute_warp", NT(M=32, N=32, K=16))
        # consecutive workgroups on consecutive pieces of memory: the XCD-aware walk (made for tiles that
        # share operands) costs a streaming kernel 8 % here
        params.setdefault("cta_swizzle", CTASwizzle.Identity)
    is_gett = any(l.kind == Layout.GETT_KIND for l in (global_a_layout, global_b_layout, global_c_layout, global_d_layout))
    planar = global_a_layout.kind in (Layout.SPLIT_COL_MAJOR, Layout.SPLIT_ROW_MAJOR)
    a_kmajor = global_a_layout.kind in (Layout.ROW_MAJOR, Layout.ALIGNED_ROW_MAJOR, Layout.INTERLEAVED_ROW_MAJOR, Layout.SPLIT_ROW_MAJOR)
    b_kmajor = global_b_layout.kind in (Layout.COL_MAJOR, Layout.ALIGNED_COL_MAJOR, Layout.INTERLEAVED_COL_MAJOR, Layout.SPLIT_COL_MAJOR)
    if block_shape is None:
        k_modes = [mode[0] for mode in global_a_layout.gett.k] if global_a_layout.kind == Layout.GETT_KIND else None
        block_shape = default_block_shape(operator, gemm_shape, tile_sized, is_gett, planar, a_kmajor=a_kmajor, b_kmajor=b_kmajor, k_modes=k_modes)
    block_shape = NT(block_shape)
    op_shape = Operator.shape(operator)

    checked = any(l.kind in (Layout.COL_MAJOR, Layout.ROW_MAJOR) for l in (global_a_layout, global_b_layout, global_c_layout, global_d_layout))
    whole_tiles = gemm_shape.M % block_shape.M == 0 and gemm_shape.N % block_shape.N == 0 and gemm_shape.K % block_shape.K == 0
    if operator.kind == Operator.MFMA and not is_gett:
        # (the plain product also where tiles stick out over the edges; the library runs the eight-wave arrangement
        # where C / D are not FP32)
        whole_tiles = whole_tiles or (gemm_shape.M >= 8 and gemm_shape.K >= 64)
    waves = _default_waves(operator, block_shape, checked, planar, is_gett, a_kmajor, b_kmajor, whole_tiles)
    if waves is not None:
        warps_default = waves[0] * waves[1]
        compute_warp_default = NT(M=block_shape.M // waves[0], N=block_shape.N // waves[1], K=op_shape.K)
    else:
        # reference src/config.jl:216-229: 8 warps as 4 x 2 unless the block is too small for that
        warps_default = 8
        compute_warp_default = NT(M=block_shape.M // 4, N=block_shape.N // 2, K=op_shape.K)
        if op_shape.M > 0 and op_shape.N > 0 and ((block_shape.M // op_shape.M) < 4 or (block_shape.N // op_shape.N) < 2):
            compute_warp_default = NT(M=max(op_shape.M, block_shape.M // 4), N=max(op_shape.N, block_shape.N // 2), K=op_shape.K)
            warps_default = min(block_shape.M // op_shape.M, 4) * min(block_shape.N // op_shape.N, 2)
    warps_per_block = params.get("warps_per_block", warps_default)
    compute_warp = NT(params.get("compute_warp", compute_warp_default))
    if "warps_per_block" in params and "compute_warp" not in params and waves is not None and warps_per_block != warps_default:
        # keep the reference's 4 x 2 style split for a caller-chosen wave count
        wm = 4 if warps_per_block % 4 == 0 and warps_per_block >= 8 else (2 if warps_per_block % 2 == 0 else 1)
        compute_warp = NT(M=block_shape.M // wm, N=block_shape.N // max(1, warps_per_block // wm), K=op_shape.K)

    is_a_col_major = params.get("is_a_col_major", True)
    is_b_col_major = params.get("is_b_col_major", True)
    is_cd_col_major = params.get("is_cd_col_major", True)

    # reference src/config.jl:240-260 with 64 lanes: 16 bytes per lane, as few lanes per row as possible
    lanes = WARP_SIZE * max(1, warps_per_block)
    n_a = max(1, min(16 // global_a_layout.T.size, (block_shape.M * block_shape.K) // lanes))
    n_b = max(1, min(16 // global_b_layout.T.size, (block_shape.K * block_shape.N) // lanes))
    n_c = max(1, min(16 // global_c_layout.T.size, (block_shape.M * block_shape.N) // lanes))
    mk, kn, mn = NT(M=block_shape.M, K=block_shape.K), NT(K=block_shape.K, N=block_shape.N), NT(M=block_shape.M, N=block_shape.N)
    mem_a_warp = NT(params.get("mem_a_warp", adjacent_elements(WARP_SIZE * n_a, mk, is_a_col_major)))
    mem_b_warp = NT(params.get("mem_b_warp", adjacent_elements(WARP_SIZE * n_b, kn, is_b_col_major)))
    mem_cd_warp = NT(params.get("mem_cd_warp", adjacent_elements(WARP_SIZE * n_c, mn, is_cd_col_major)))
    mem_a_thread = NT(params.get("mem_a_thread", adjacent_elements(n_a, mk, is_a_col_major)))
    mem_b_thread = NT(params.get("mem_b_thread", adjacent_elements(n_b, kn, is_b_col_major)))
    mem_cd_thread = NT(params.get("mem_cd_thread", adjacent_elements(n_c, mn, is_cd_col_major)))

    # src/config.jl:277-279 defaults to Identity; on the MI355X the XCD-aware walk is the default
    # (panels 4 tiles high; 8 once every CU has a tile: 4096^3 is 0.2 - 1.0 us faster with it in every transpose, 8192^3
    # 10 %; 16 from four thousand tiles on: 16384 x 16384 x 4096 1771 us against 1789 and 1871 us with 8 and 4)
    n_tiles = -(-gemm_shape.M // block_shape.M) * -(-gemm_shape.N // block_shape.N)
    cta_swizzle = params.get("cta_swizzle", CTASwizzle.XCDAware[16 if n_tiles >= 4096 else (8 if n_tiles >= NUM_CUS else 4)])

    conf = Config(gemm_shape, block_shape, warps_per_block, mem_a_warp, mem_a_thread, mem_b_warp, mem_b_thread,
                  mem_cd_warp, mem_cd_thread, compute_warp, op_shape,
                  global_a_layout, global_b_layout, global_c_layout, global_d_layout,
                  shared_a_layout, shared_b_layout, shared_c_layout, shared_d_layout,
                  operator, is_a_col_major, is_b_col_major, cta_swizzle)
    if not params.get("specialize", False):
        # ``specialize=True``: the block shape need not be in the library's table because the kernel
        # will be compiled at run time (gemmkernels.specialize); that compilation and every launch run
        # the same checks, minus the table lookup
        check_config(conf, params.get("kernel"))
        conf.__dict__["_tile_left_open"] = not any(k in params for k in _TILE_CHOICES)
    return conf


_TILE_CHOICES = ("block_shape", "warps_per_block", "compute_warp", "mem_a_warp", "mem_b_warp", "mem_cd_warp", "mem_a_thread", "mem_b_thread",
                 "mem_cd_thread", "cta_swizzle")
_ANY_SIZE = {Layout.ALIGNED_COL_MAJOR: Layout.ColMajor, Layout.ALIGNED_ROW_MAJOR: Layout.RowMajor}


def larger_tile(conf: Config, hooks: bool, slices: bool = False) -> Optional[Config]:
    """The configuration that a launch of ``conf`` runs on where the tile was left to the default and one that does not divide the sizes is faster,
    or None.

    Aligned layouts ask for sizes in whole tiles (reference src/config.jl:268-275), so most multiples of 64 leave only the 64 x 64 tiles, which
    bring every operand into the CUs four times as often as 256 x 256 ones do.  The kernels take tiles over the edges on any layout, so the launch
    is that of the bounds-checked layouts on the tile with the shortest estimate, once the operands have passed for what the aligned ones ask
    (``matmul``): every output is summed in the same order, except in slices.  us on the tile that divides and on the larger one, and the ratio of
    the estimates, inputs that rotate:
        2240 x 5568 x 2304 'N','N' with C 100.0 and 69.9 (0.52), 4544 x 2048 x 2368 'T','N' 70.8 and 47.9 (0.68), 1344 x 2880 x 5696 'T','T' 64.7 and
        58.3 (0.71), 1600 x 4480 x 2048 'N','T' with C 54.9 and 47.5 (0.75), 5632 x 2240 x 384 24.2 and 20.7 (0.84), 5120 x 4224 x 5888 with C 285.8
        and 269.4 (0.84); beyond the line 1920 x 1856 x 2368 27.9 and 29.2 (0.90), 2368 x 3072 x 896 with C 28.4 and 30.0 (0.90).
    Extents up to 131072, with and without hooks: 81 drawn ones all faster, 1.01 to 2.5 times.
    ``hooks``: transforms or a bias, which tiles of 256 x 256 over the edges run on eight waves (5376 x 2176 x 768 with C 47.5 and 53.0,
    3520 x 2432 x 2048 72.4 and 76.1, so not those) and which the estimates leave out: 5696 x 5760 x 4160 with C 440 and 320 on 128 x 128 (0.57),
    4992 x 1344 x 4416 99.6 and 73.7 (0.70), 4608 x 832 x 6080 75.5 and 61.6 (0.71); beyond the line 5056 x 768 x 2176 29.1 and 31.0 (0.85).  (Not for
    op lists on A or B, see ``matmul``.)
    ``slices``: the launch may run in slices of K (``sliced_block_shape``)."""
    if not conf.__dict__.get("_tile_left_open") or conf.operator.kind != Operator.MFMA or conf.global_a_layout.kind not in _ANY_SIZE:
        return None
    name = ("_larger_tile_with_hooks" if hooks else "_larger_tile") + ("_in_slices" if slices else "")
    if name not in conf.__dict__:
        op, layouts = conf.operator, (conf.global_a_layout, conf.global_b_layout, conf.global_c_layout, conf.global_d_layout)
        shared = (conf.shared_a_layout, conf.shared_b_layout, conf.shared_c_layout, conf.shared_d_layout)
        # (kept by value: a program that makes a configuration for every product finds the answer of the ones before)
        key = (*conf.matmul_shape.values(), *conf.block_shape.values(), hooks, slices, op.kind, op.M, op.N, op.K, op.CT.name, op.AT.name, conf.is_a_col_major, conf.is_b_col_major,
               *((l.kind, l.T.name, l.pad) for l in layouts + shared))
        found = _larger_tiles.get(key, False)
        if found is False:
            found = _find_larger_tile(tuple(conf.matmul_shape.values()), tuple(conf.block_shape.values()), op, layouts, shared,
                                      conf.is_a_col_major, conf.is_b_col_major, hooks, slices)
            if len(_larger_tiles) >= 256:
                _larger_tiles.clear()
            _larger_tiles[key] = found
        conf.__dict__[name] = found
    return conf.__dict__[name]


_larger_tiles = {}


def _find_larger_tile(shape, own, operator, layouts, shared, is_a_col_major, is_b_col_major, hooks, slices) -> Optional[Config]:
    if operator.kind != Operator.MFMA or any(l.kind not in _ANY_SIZE and not (i == 2 and l.kind == Layout.ZERO) for i, l in enumerate(layouts)):
        return None
    M, N, K = shape
    if own not in _MFMA_TILE_COST:
        return None
    a_kmajor, b_kmajor = layouts[0].kind == Layout.ALIGNED_ROW_MAJOR, layouts[1].kind == Layout.ALIGNED_COL_MAJOR
    sliced = sliced_block_shape(M, N, K) if slices and own[:2] == (64, 64) else None
    if sliced is not None:
        best = tuple(sliced.values())
    else:
        best = min(_mfma_tiles(a_kmajor, b_kmajor), key=lambda t: math.inf if hooks and t[:2] == (256, 256) else _mfma_cost(t, M, N, K))
        if best == own or _mfma_cost(best, M, N, K) > (0.8 if hooks else 0.86) * _mfma_cost(own, M, N, K):
            return None
    a, b, c, d = (_ANY_SIZE[l.kind][l.T] if l.kind in _ANY_SIZE else l for l in layouts)
    try:
        return get_config(gemm_shape=NT(M=M, N=N, K=K), operator=operator, block_shape=NT(M=best[0], N=best[1], K=best[2]),
                          global_a_layout=a, global_b_layout=b, global_c_layout=c, global_d_layout=d,
                          shared_a_layout=shared[0], shared_b_layout=shared[1], shared_c_layout=shared[2], shared_d_layout=shared[3],
                          is_a_col_major=is_a_col_major, is_b_col_major=is_b_col_major)
    except ConfigError:
        return None


def check_config(conf: Config, kernel=None) -> None:
    """Every ConfigError of the reference (src/config.jl:203-275, src/matmul.jl:28-41), decided by
    the library on the host."""
    c = conf.to_c()
    code = 0 if kernel is None else kernel.code
    rc = _lib.lib().gk_validate(ctypes.byref(c), code)
    if rc != _lib.GK_OK:
        raise ConfigError(_lib.last_error(), rc)


def _load_tuning_table_from_environment() -> None:
    import json
    import os
    path = os.environ.get("GEMMKERNELS_TUNING_TABLE")
    if path and os.path.exists(path):
        with open(path) as f:
            TUNED.update(json.load(f))


_load_tuning_table_from_environment()
