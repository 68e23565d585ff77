"""Plain products on the tile that the closer estimate takes instead of the default (``product_block_shape``): exact on small whole numbers against 64 bits, and where the line lies."""
import pytest

import gemmkernels as gk
from gemmkernels import NT
from gemmkernels.config import product_block_shape


def test_the_line():
    small, large = NT(M=64, N=64, K=32), NT(M=256, N=256, K=64)
    assert product_block_shape(small, 2326, 1029, 855, False, False, (0, 2), 4) == NT(M=128, N=128, K=32)
    assert product_block_shape(small, 300, 300, 300, False, True, (1, 1), 4) == small                 # ends within the launch and its ends
    assert product_block_shape(small, 4001, 4003, 4005, True, True, (2, 0), 4) == small                # may run on copies of its operands
    assert product_block_shape(large, 4096, 4096, 4096, False, True, (0, 0), 4) == large
    assert product_block_shape(NT(M=32, N=32, K=64), 2326, 1029, 855, False, False, (0, 2), 4) == NT(M=32, N=32, K=64)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,ta,tb,tile", [(2326, 1029, 855, False, True, (128, 128, 32)), (991, 3293, 565, True, False, (128, 128, 64)), (3596, 2319, 285, False, True, (256, 192, 64)),
                                              (826, 3725, 462, True, True, (128, 128, 32)), (2336, 266, 7288, False, True, (128, 128, 64))])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (1.5, 0.5)])
def test_mul(gpu, M, N, K, ta, tb, tile, alpha, beta):
    import sys

    import torch
    gen = torch.Generator(device="cuda").manual_seed(K)
    whole = lambda rows, cols, t: torch.randint(-2, 3, (cols, rows), generator=gen, device="cuda").to(t).t()
    a, b = whole(*((K, M) if ta else (M, K)), torch.float16), whole(*((N, K) if tb else (K, N)), torch.float16)
    c = whole(M, N, torch.float32)
    p = sys.modules["gemmkernels.matmul"].matmatmul_plan(c, "NT"[ta], "NT"[tb], a, b, alpha, beta)
    if beta == 0.0:
        assert (p._conf.block_shape.M, p._conf.block_shape.N, p._conf.block_shape.K) == tile
    want = alpha * ((a.double().t() if ta else a.double()) @ (b.double().t() if tb else b.double())) + beta * c.double()
    gk.mul_(c, gk.Transpose(a) if ta else a, gk.Transpose(b) if tb else b, alpha, beta)
    assert torch.equal(c.double(), want)
