"""Products of 257 to 512 tiles of 64 x 64 and a long K in slices of K on 128 x 128 x 64 (``sliced_block_shape``): exact on small whole numbers against 64 bits at the
edges of the rule, whatever the ends of K and of the tiles, from ``mul_``, plans and ``matmul``, the same bits on every run and from a graph; no larger error than one chain."""
import pytest

import gemmkernels as gk
from gemmkernels import Epilogue, Kernel, NT, Transform, configs
from gemmkernels.config import larger_tile, sliced_block_shape

pytestmark = pytest.mark.gpu
TILE = NT(M=128, N=128, K=64)


def whole(gen, rows, cols, dtype, span=2):
    import torch
    return torch.randint(-span, span + 1, (cols, rows), generator=gen, device="cuda").to(dtype).t()


def mul_plan(c, a, b, ta, tb, alpha, beta):
    import sys
    return sys.modules["gemmkernels.matmul"].matmatmul_plan(c, "NT"[ta], "NT"[tb], a, b, alpha, beta)


# whole tiles, K ending 1, 8 and 63 into a tile, extents one over and one under a tile, odd leading dimensions, 65 and 128 tiles, two and three slices
@pytest.mark.parametrize("M,N,K", [(1024, 2048, 3520), (2048, 1024, 8192), (1025, 1025, 2561), (1000, 1111, 4104), (513, 2175, 2623), (127, 8255, 2500), (16384, 128, 3584)])
@pytest.mark.parametrize("dtype,out,alpha,beta", [("float16", "float32", 1.0, 0.0), ("bfloat16", "float32", 1.5, 0.5), ("float16", "float16", 1.0, 0.0)])
def test_mul(gpu, M, N, K, dtype, out, alpha, beta):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    for ta in (False, True):
        for tb in (False, True):
            # (FP16 results: sums of magnitude below 2048 stay whole)
            a = whole(gen, *((K, M) if ta else (M, K)), getattr(torch, dtype), 1 if out == "float16" else 2)
            b = whole(gen, *((N, K) if tb else (K, N)), getattr(torch, dtype), 1 if out == "float16" else 2)
            c0 = whole(gen, M, N, getattr(torch, out))
            p = mul_plan(c0, a, b, ta, tb, alpha, beta)
            assert p._sliced > 0 and p._conf.block_shape.M == 128, (M, N, K)
            want = alpha * ((a.double().t() if ta else a.double()) @ (b.double().t() if tb else b.double())) + beta * c0.double()
            for _ in range(3):
                c = c0.clone()
                gk.mul_(c, gk.Transpose(a) if ta else a, gk.Transpose(b) if tb else b, alpha, beta)
                assert torch.equal(c.double(), want.to(c.dtype).double()), (M, N, K, ta, tb)


def test_configured(gpu):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(5)
    for M, N, K, hooks in ((1088, 1024, 3520, False), (2048, 1024, 4096, True), (704, 1984, 5056, False), (192, 5696, 3712, True)):
        a, b, c, bias = whole(gen, K, M, torch.float16), whole(gen, K, N, torch.float16), whole(gen, M, N, torch.float32), torch.randint(-3, 4, (N,), generator=gen, device="cuda").float()
        conf = configs.mfma_config(M, N, K, True, False)
        assert larger_tile(conf, hooks, True).block_shape == TILE
        options = dict(transform_shared_to_global_d=Transform.Elementwise(Transform.relu), epilogue=Epilogue.Bias(bias)) if hooks else {}
        d = gk.colmajor_empty((M, N), torch.float32)
        launch = gk.plan(conf, a, b, c, d, kernel=Kernel.matmul_pipelined, **options)
        assert launch._sliced > 0 and launch._conf.block_shape.M == 128, (M, N, K)
        want = a.double().t() @ b.double() + c.double()
        if hooks:
            want = torch.relu(want + bias.double())
        for run in (launch, lambda: gk.matmul(conf, a, b, c, d, kernel=Kernel.matmul_pipelined, **options)):
            for _ in range(3):
                d.fill_(float("nan"))
                run()
                assert torch.equal(d.double(), want), (M, N, K)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            launch()
        for _ in range(3):
            d.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(d.double(), want), (M, N, K)
            launch()
            torch.cuda.synchronize()
            assert torch.equal(d.double(), want), (M, N, K)


def test_error_of_a_shorter_chain(gpu):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(7)
    M, N, K = 1024, 1088, 4096
    a, b = (torch.rand(s, generator=gen, device="cuda").mul_(2).sub_(1).half().t() for s in ((K, M), (N, K)))
    c, one = gk.colmajor_empty((M, N), torch.float32), gk.colmajor_empty((M, N), torch.float32)
    gk.mul_(c, a, b, 1.0, 0.0)
    chain = configs.mfma_config(M, N, K, block_shape=(64, 64, 64), zero_c=True)
    gk.matmul(chain, a, b, None, one, kernel=Kernel.matmul_pipelined)
    want = a.double() @ b.double()
    error = lambda x: ((x.double() - want).norm() / want.norm()).item()
    assert error(c) <= error(one), (error(c), error(one))


def test_refused_and_other_tiles(gpu):
    """Nothing above 128 tiles, below the line of K, or with a tile that was asked for."""
    import torch
    assert sliced_block_shape(2049, 1024, 4096) is None and sliced_block_shape(1024, 1088, 3496) is None and sliced_block_shape(1024, 1088, 2496, odd=True) is None and sliced_block_shape(1024, 1088, 2504, odd=True) == TILE and sliced_block_shape(1024, 1024, 8192) is None
    conf = configs.mfma_config(1024, 2048, 4096, block_shape=(64, 64, 64), zero_c=True)
    half = lambda m, n: torch.empty(n, m, device="cuda", dtype=torch.float16).t()
    launch = gk.plan(conf, half(1024, 4096), half(4096, 2048), None, gk.colmajor_empty((1024, 2048), torch.float32), kernel=Kernel.matmul_pipelined)
    assert launch._sliced == 0 and launch._conf.block_shape.M == 64


def test_k_split_launches_of_the_tile_within_a_limit_of_lds(gpu):
    """Their slices have four LDS stages (128 KiB); where less is allowed the launch runs unsplit on two, and is not refused."""
    import torch
    from gemmkernels import _lib
    gen = torch.Generator(device="cuda").manual_seed(11)
    M, N, K = 512, 384, 4096
    a, b = whole(gen, M, K, torch.float16), whole(gen, K, N, torch.float16)
    conf = configs.mfma_config(M, N, K, block_shape=(128, 128, 64), zero_c=True)
    want = a.double() @ b.double()
    try:
        for limit in (0, 65536):
            _lib.lib().gk_set_device_limits(limit, 0)
            d = gk.colmajor_empty((M, N), torch.float32)
            gk.matmul(conf, a, b, None, d, kernel=Kernel.matmul_split_k)
            assert torch.equal(d.double(), want), limit
    finally:
        _lib.lib().gk_set_device_limits(0, 0)
