"""FPUOp on the FP32 / FP64 matrix instructions (reference src/operator.jl:35-153): bit-identical to the sequential fma
chain of the oracle at the sizes where a tile, a vector or a K tile ends."""
import numpy as np
import pytest
import torch

import gemmkernels as gk
from gemmkernels import Epilogue, Float16, Float32, Float64, Kernel, Layout, NT, Operator, Transform
import helpers
from test_fpu_types_gpu import TORCH, operand

pytestmark = pytest.mark.gpu

TYPES = {"f32": (Float32, Float32, np.float32, np.float32), "f64": (Float64, Float64, np.float64, np.float64),
         "f16_f32": (Float16, Float32, np.float16, np.float32), "f32_f64": (Float32, Float64, np.float32, np.float64)}
TILES = {"f32": [((128, 128, 32), (2, 2)), ((128, 128, 16), (2, 2)), ((64, 64, 32), (2, 2)), ((32, 32, 32), (2, 2)), ((32, 32, 32), (1, 1))],
         "f64": [((64, 64, 32), (2, 2)), ((32, 32, 32), (2, 2))], "f16_f32": [((64, 64, 32), (2, 2))], "f32_f64": [((64, 64, 32), (2, 2))]}
# (M, N, K) around a tile (BM, BN, BK): fewer rows or k than a vector, one beyond a vector, a tile less and more one, K tiles 0 .. 4
SIZES = [lambda m, n, k: (1, 1, 1), lambda m, n, k: (3, 2, 3), lambda m, n, k: (5, n + 1, k - 1), lambda m, n, k: (m, n, k),
         lambda m, n, k: (m - 1, n - 3, 2 * k + 2), lambda m, n, k: (m + 2, 2 * n + 1, 3 * k + 5), lambda m, n, k: (2 * m, n, 4 * k)]


def config(M, N, K, ta, tb, types, tile, zero_c):
    AB, CD = TYPES[types][:2]
    (bm, bn, bk), (wm, wn) = tile
    return gk.get_config(gemm_shape=NT(M=M, N=N, K=K), block_shape=NT(M=bm, N=bn, K=bk), warps_per_block=wm * wn,
                         compute_warp=NT(M=bm // wm, N=bn // wn, K=1), operator=Operator.FPUOp[8, 8, 1, 8, 8, 1, AB, CD],
                         global_a_layout=(Layout.RowMajor if ta else Layout.ColMajor)[AB], global_b_layout=(Layout.RowMajor if tb else Layout.ColMajor)[AB],
                         global_c_layout=Layout.Zero[CD] if zero_c else Layout.ColMajor[CD], global_d_layout=Layout.ColMajor[CD],
                         is_a_col_major=not ta, is_b_col_major=not tb)


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("types", list(TYPES))
def test_every_tile_at_its_edges(gpu, types, ta, tb):
    _, _, np_in, np_out = TYPES[types]
    for tile in TILES[types]:
        for n, size in enumerate(SIZES):
            M, N, K = size(*tile[0])
            a, b = operand((K, M) if ta else (M, K), np_in, 10 + n), operand((N, K) if tb else (K, N), np_in, 20 + n)
            c = None if n % 2 else operand((M, N), np_out, 30 + n)
            conf = config(M, N, K, ta, tb, types, tile, c is None)
            hooks = {}
            if n % 3 == 1:          # a scale of A in the K loop, C scaled
                hooks = dict(transform_shared_to_regs_a=Transform.Elementwise(lambda x: x * 1.5), transform_shared_to_regs_c=Transform.Elementwise(lambda x: x * 0.5))
            if n == 6:              # lists of four on C alone, a scale of B, lists in both hooks of D
                steps = Transform.Elementwise(lambda x: (x * 0.5 + 1) * 3 - 2)
                hooks = dict(transform_global_to_shared_c=steps, transform_shared_to_regs_c=steps, transform_global_to_shared_b=Transform.Elementwise(lambda x: x * -0.75),
                             transform_regs_to_shared_d=steps, transform_shared_to_global_d=steps)
            if n % 3 == 2:          # lists in both hooks of A and one of B (x + 1 leaves no zero behind K), and of D
                hooks = dict(transform_global_to_shared_a=Transform.Elementwise(lambda x: x + 1), transform_shared_to_regs_a=Transform.Elementwise(lambda x: x * 0.75),
                             transform_global_to_shared_b=Transform.Elementwise(lambda x: (x + 1) * 3), transform_shared_to_global_d=Transform.Elementwise(Transform.relu))
            print("case", types, tile, (M, N, K), ta, tb, gk.kernel_name(conf, Kernel.matmul_singlestage), flush=True)
            d = helpers.run_gpu(conf, a, b, c, (M, N), d_dtype=TORCH[np_out], transforms=hooks)
            assert np.array_equal(d, helpers.run_oracle(conf, a, b, c, (M, N), d_dtype=np_out, transforms=hooks)), (tile, (M, N, K))


@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_zeros_infinities_and_subnormals_go_through_as_in_an_fma_chain(gpu, ta, tb):
    """Signed zeros, infinities (and the NaN they make) and values whose products and sums are subnormal."""
    for types in ("f32", "f64"):
        _, _, np_in, np_out = TYPES[types]
        M, N, K = 70, 66, 44          # (whole steps of four k: the zeros behind K would make +0 of a sum that underflowed to -0)
        r = np.random.RandomState(3)
        pick = np.array([0.0, -0.0, 1.0, -2.5, np.finfo(np_in).tiny, -np.finfo(np_in).tiny / 4, np.finfo(np_in).tiny * 0.5, 0.375], np_in)
        a, b = np.asfortranarray(r.choice(pick, (K, M) if ta else (M, K))), np.asfortranarray(r.choice(pick, (N, K) if tb else (K, N)))
        (a.T if ta else a)[5, 7], (b if not tb else b.T)[9, 11] = np.inf, -np.inf
        conf = config(M, N, K, ta, tb, types, TILES[types][0], True)
        d = helpers.run_gpu(conf, a, b, None, (M, N), d_dtype=TORCH[np_out])
        ref = helpers.run_oracle(conf, a, b, None, (M, N), d_dtype=np_out)
        assert np.array_equal(np.isnan(d), np.isnan(ref)) and np.array_equal(d[~np.isnan(ref)], ref[~np.isnan(ref)])
        assert np.array_equal(np.signbit(d[ref == 0]), np.signbit(ref[ref == 0]))


@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_nothing_behind_k_meets_an_infinite_factor(gpu, ta, tb):
    """A scale by infinity makes NaN of a zero: the values behind a partial K tile are none of the product's."""
    times_inf = Transform.Elementwise(lambda x: x * float("inf"))
    for types in TYPES:
        _, _, np_in, np_out = TYPES[types]
        for K in (1, 5, 34, 45, 67):
            M, N = 66, 70
            a, b = abs(operand((K, M) if ta else (M, K), np_in, 61)) + np_in(1), abs(operand((N, K) if tb else (K, N), np_in, 62)) + np_in(1)
            for hooks in (dict(transform_shared_to_regs_a=times_inf), dict(transform_global_to_shared_b=times_inf)):
                conf = config(M, N, K, ta, tb, types, TILES[types][-1], True)
                d = helpers.run_gpu(conf, a, b, None, (M, N), d_dtype=TORCH[np_out], transforms=hooks)
                ref = helpers.run_oracle(conf, a, b, None, (M, N), d_dtype=np_out, transforms=hooks)
                assert np.all(np.isposinf(ref)) and np.array_equal(d, ref), (types, K, list(hooks))


def test_operands_at_the_end_of_an_allocation_and_off_16_byte_boundaries(gpu):
    """Leading dimensions and first elements at any multiple of the element size; bias per column and per row."""
    for types in ("f32", "f64"):
        _, _, np_in, np_out = TYPES[types]
        M, N, K = 67, 129, 101
        for ta, tb in ((False, False), (True, True)):
            a, b = operand((K, M) if ta else (M, K), np_in, 41), operand((N, K) if tb else (K, N), np_in, 42)

            def at_end(x):          # the last element of the matrix is the last of the allocation
                flat = torch.full((3 + (x.shape[0] + 5) * x.shape[1] - 5,), float("nan"), dtype=TORCH[np_in], device="cuda")
                view = flat[3:].as_strided(x.shape, (1, x.shape[0] + 5))
                view.copy_(torch.from_numpy(np.ascontiguousarray(x)).cuda())
                return view
            for epilogue in ((None, Epilogue.Bias, Epilogue.BiasRow) if hasattr(Epilogue, "BiasRow") and types == "f32" else (None,)):
                conf = config(M, N, K, ta, tb, types, TILES[types][-1], True)
                d = gk.colmajor_empty((M, N), TORCH[np_out])
                bias = operand((max(M, N), 1), np.float32, 43)[:, 0]
                epi = None if epilogue is None else epilogue(torch.from_numpy(bias).cuda())
                gk.matmul(conf, at_end(a), at_end(b), None, d, epilogue=epi)
                torch.cuda.synchronize()
                ref = helpers.run_oracle(conf, a, b, None, (M, N), d_dtype=np_out, epilogue=None if epilogue is None else epilogue(0), bias=bias)
                assert np.array_equal(gk.to_numpy(d), ref), (types, ta, tb, epilogue)


def test_zero_alpha_reads_neither_a_nor_b(gpu):
    for types in ("f32", "f64"):
        _, _, np_in, np_out = TYPES[types]
        a, b, c = operand((100, 40), np_in, 51), operand((40, 70), np_in, 52), operand((100, 70), np_out, 53)
        A, B, C = (gk.colmajor(x) for x in (np.full_like(a, np.nan), b, c))
        gk.matmatmul_(C, "N", "N", A, B, 0.0, 2.0)
        torch.cuda.synchronize()
        assert np.array_equal(gk.to_numpy(C), 2 * c)


def test_leading_dimensions_beyond_32_bits_of_tile_offsets(gpu):
    """128 rows of 2^23 Float32 lie 4 GiB apart: the offsets in a tile are 64 bits wide, so the 128 x 128 tile takes every
    leading dimension that the 64 x 64 tile takes."""
    M, N, K, ld = 128, 70, 37, (1 << 23) + 3
    a, b = operand((K, M), np.float32, 71), operand((K, N), np.float32, 72)
    A = torch.empty(ld * (M - 1) + K, device="cuda").as_strided((K, M), (1, ld))
    A.copy_(torch.from_numpy(np.ascontiguousarray(a)))
    for tile in TILES["f32"][:3]:
        conf = config(M, N, K, True, False, "f32", tile, True)
        D = gk.colmajor_empty((M, N), torch.float32)
        gk.matmul(conf, A, gk.colmajor(b), None, D)
        torch.cuda.synchronize()
        assert np.array_equal(gk.to_numpy(D), helpers.run_oracle(conf, a, b, None, (M, N), d_dtype=np.float32)), tile


@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
@pytest.mark.parametrize("types", ["f32", "f64"])
def test_instances_for_one_workgroup_per_cu_and_for_more(gpu, types, ta, tb):
    """At most 256 tiles run on instances of their own (32 x 32 x 32 in pairs of K tiles from K = 512 on), more on the others: the same fma
    chains either way, with factors on A and C, at tile counts on both sides and K around a pair."""
    _, _, np_in, np_out = TYPES[types]
    half = dict(transform_shared_to_regs_a=Transform.Elementwise(lambda x: x * 1.5), transform_shared_to_regs_c=Transform.Elementwise(lambda x: x * 0.5))
    for tile, (M, N), Ks in ((((32, 32, 32), (2, 2)), (37, 61), (511, 512, 543, 577, 640)), (((32, 32, 32), (2, 2)), (512, 512), (512,)), (((32, 32, 32), (2, 2)), (545, 512), (66, 520)),
                             (((64, 64, 32), (2, 2)), (65, 130), (31, 64, 101)), (((64, 64, 32), (2, 2)), (1030, 1021), (70,))):
        for K in Ks:
            a, b = operand((K, M) if ta else (M, K), np_in, K), operand((N, K) if tb else (K, N), np_in, K + 1)
            for hooks in ({}, half):
                c = operand((M, N), np_out, K + 2) if hooks else None
                conf = config(M, N, K, ta, tb, types, tile, c is None)
                name = gk.kernel_name(conf, Kernel.matmul_singlestage, hooks)
                few = -(-M // tile[0][0]) * -(-N // tile[0][1]) <= 256
                assert ("_s3_" in name or "_pairs_" in name) == (few and (tile[0][0] == 64 or K >= 512)), name
                print("case", types, tile, (M, N, K), ta, tb, name, flush=True)
                d = helpers.run_gpu(conf, a, b, c, (M, N), d_dtype=TORCH[np_out], transforms=hooks)
                assert np.array_equal(d, helpers.run_oracle(conf, a, b, c, (M, N), d_dtype=np_out, transforms=hooks)), (tile, (M, N, K))
