"""Contractions and configured products on 64 x 64 x 64 tiles in slices of K: exact on small whole numbers against 64 bits, with and without C, whatever K modes a
slice starts in, the same bits on every run; and which launches are cut."""
import pytest

import gemmkernels as gk
from gemmkernels import Epilogue, Kernel, Transform, configs
from gemmkernels import contraction

pytestmark = pytest.mark.gpu

# (mode string, extents): K modes e, f with K = 2048 .. 4160; slices start inside f, inside e, with three K modes and with one
CASES = [("abcd-aebf-dfce", dict(a=32, b=12, c=6, d=64, e=64, f=64)), ("abcd-aebf-dfce", dict(a=64, b=2, c=4, d=32, e=32, f=192)),
         ("abcd-aebf-dfce", dict(a=32, b=8, c=20, d=32, e=64, f=64)), ("abc-adbe-edc", dict(a=64, b=3, c=64, d=48, e=64)),
         ("ab-aefg-ebfg", dict(a=192, b=128, e=32, f=8, g=16)), ("ab-ae-eb", dict(a=128, b=64, e=4096))]


def tensor(gen, modes, ext, dtype):
    import torch
    shape = [ext[m] for m in modes]
    return torch.randint(-2, 3, tuple(reversed(shape)), generator=gen, device="cuda").to(dtype).permute(*reversed(range(len(shape))))


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("with_c", [False, True])
def test_contractions(gpu, case, with_c):
    import torch
    spec, ext = CASES[case]
    dm, am, bm = spec.split("-")
    gen = torch.Generator(device="cuda").manual_seed(case)
    a, b = tensor(gen, am, ext, torch.float16), tensor(gen, bm, ext, torch.float16)
    c = tensor(gen, dm, ext, torch.float32) if with_c else None
    d = gk.colmajor_empty(tuple(ext[m] for m in dm), torch.float32)
    p = contraction.plan(spec, a, b, d, c)
    assert p._launch._sliced > 0, p.kernel_name
    want = torch.einsum(f"{am},{bm}->{dm}", a.cpu().double(), b.cpu().double())
    if with_c:
        want = want + c.cpu().double()
    for _ in range(5):
        d.fill_(float("nan"))
        gk.contract(spec, a, b, d, c)
        assert torch.equal(d.cpu().double(), want)
        d.fill_(float("nan"))
        p()
        assert torch.equal(d.cpu().double(), want)


def test_configured_products(gpu):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(3)
    for M, N, K, hooks in ((512, 576, 4480, False), (384, 256, 3776, True), (640, 704, 5312, False), (64, 64, 1280, True), (128, 192, 1344, False)):
        for ta in (False, True):
            for tb in (False, True):
                a, b = tensor(gen, "km" if ta else "mk", dict(m=M, k=K), torch.float16), tensor(gen, "nk" if tb else "kn", dict(n=N, k=K), torch.float16)
                c, bias = tensor(gen, "mn", dict(m=M, n=N), torch.float32), torch.randint(-3, 4, (N,), generator=gen, device="cuda").float()
                conf = configs.mfma_config(M, N, K, ta, tb)
                options = dict(transform_shared_to_global_d=Transform.Elementwise(Transform.relu), epilogue=Epilogue.Bias(bias)) if hooks else {}
                d = gk.colmajor_empty((M, N), torch.float32)
                launch = gk.plan(conf, a, b, c, d, kernel=Kernel.matmul_pipelined, **options)
                assert launch._sliced > 0, (M, N, K)
                want = (a.double().t() if ta else a.double()) @ (b.double().t() if tb else b.double()) + c.double()
                if hooks:
                    want = torch.relu(want + bias.double())
                launch()
                assert torch.equal(d.double(), want), (M, N, K, ta, tb)
                d.fill_(float("nan"))
                gk.matmul(conf, a, b, c, d, kernel=Kernel.matmul_pipelined, **options)
                assert torch.equal(d.double(), want), (M, N, K, ta, tb)


def test_which_are_cut(gpu):
    import torch
    half = lambda m, n: torch.empty(n, m, device="cuda", dtype=torch.float16).t()
    for M, N, K in ((1024, 1024, 4096), (512, 512, 1024), (4096, 4096, 4096), (2048, 1088, 8192)):
        launch = gk.plan(configs.mfma_config(M, N, K, zero_c=True), half(M, K), half(K, N), None, gk.colmajor_empty((M, N), torch.float32), kernel=Kernel.matmul_pipelined)
        assert launch._sliced == 0, (M, N, K)
