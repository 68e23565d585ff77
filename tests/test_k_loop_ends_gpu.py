"""The ends of the K loop of the products on the matrix cores: no tile, fewer tiles than LDS stages, as many, one more, each with and without a last tile
outside the pipeline, over tiles at the edge of D or not, with and without C.  Operands are small whole numbers, so every sum is exact in whatever order it
is made and the results are compared with == ."""
import pytest

import gemmkernels as gk

pytestmark = pytest.mark.gpu

KS = [8, 9, 31, 32, 33, 63, 64, 65, 96, 100, 127, 128, 129, 160, 191, 192, 193, 200, 255, 256, 257, 319, 320, 321]


def integers(gen, rows, cols, dtype):
    import torch
    return torch.randint(-3, 4, (cols, rows), generator=gen, device="cuda").to(dtype).t()


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("types", ["f16_f32", "bf16_f32", "f16_f16"])
def test_every_end(gpu, ta, tb, types):
    import torch
    ab, cd = {"f16_f32": (torch.float16, torch.float32), "bf16_f32": (torch.bfloat16, torch.float32), "f16_f16": (torch.float16, torch.float16)}[types]
    gen = torch.Generator(device="cuda").manual_seed(11)
    for M, N in ((64, 128), (67, 130), (130, 9), (700, 1500), (2048, 1100)):
        for K in KS:
            a, b = integers(gen, *((K, M) if ta else (M, K)), ab), integers(gen, *((N, K) if tb else (K, N)), ab)
            exact = (a.double().t() if ta else a.double()) @ (b.double().t() if tb else b.double())
            for alpha, beta in ((1.0, 0.0), (1.0, 1.0), (1.5, 1.0)):          # (whole and half numbers below 2^13, exact; in an FP16 C below 2^10)
                if cd is torch.float16 and 9 * 1.5 * K + 3 >= 1024:
                    continue
                c = integers(gen, M, N, cd)
                want = alpha * exact + beta * c.double()
                got = gk.mul_(c, gk.Transpose(a) if ta else a, gk.Transpose(b) if tb else b, alpha, beta)
                assert torch.equal(got.double(), want), (M, N, K, alpha, beta)


def test_operands_that_end_where_their_memory_ends(gpu):
    """The tile outside the pipeline reads nothing behind an operand: NaN in front of it and behind it change no result."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(12)

    def fenced(x):
        flat = torch.full((x.numel() + 64,), float("nan"), dtype=x.dtype, device="cuda")
        inside = flat[32:32 + x.numel()].view(x.shape[1], x.shape[0])
        inside.copy_(x.t())
        return inside.t()
    for M, N, K in ((67, 130, 33), (130, 67, 97), (33, 515, 200), (65, 65, 8), (1001, 301, 129)):
        for ta in (False, True):
            for tb in (False, True):
                a, b = integers(gen, *((K, M) if ta else (M, K)), torch.float16), integers(gen, *((N, K) if tb else (K, N)), torch.float16)
                want = (a.double().t() if ta else a.double()) @ (b.double().t() if tb else b.double())
                fa, fb = fenced(a), fenced(b)
                c = fenced(torch.zeros(N, M, device="cuda").t())
                gk.mul_(c, gk.Transpose(fa) if ta else fa, gk.Transpose(fb) if tb else fb, 1.0, 1.0)
                assert torch.equal(c.double(), want), (M, N, K, ta, tb)
