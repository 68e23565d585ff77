"""Float32 and Float64 products in slices of K (``gk_matmul_sliced``): which launches take them, their results at the edges of tiles and of slices, their error
beside the error of one chain, the same bits on every run, and replays of a graph."""
import ctypes

import pytest

import gemmkernels as gk
from gemmkernels import Kernel, _lib, configs

TYPES = ["float32", "float64"]


def sliced_bytes(M, N, K, dtype, transforms=None):
    import torch
    from gemmkernels.dtypes import from_torch
    T = from_torch(getattr(torch, dtype))
    conf = configs_fpu(M, N, K, T).to_c()
    need = ctypes.c_size_t()
    assert _lib.lib().gk_sliced_workspace_size(ctypes.byref(conf), transforms, None, ctypes.byref(need)) == _lib.GK_OK
    return need.value


def configs_fpu(M, N, K, T):
    import importlib
    return importlib.import_module("gemmkernels.matmul").create_config(T, (M, K), (1, M), False, T, (K, N), (1, K), False, T, (M, N), (1, M), float, False, float, True)[0]


def test_which_launches_are_cut():
    # (no GPU) few tiles and a long K; not few K, not tiles enough for the chip, not another operator
    assert sliced_bytes(64, 64, 8000, "float32") > 0 and sliced_bytes(64, 64, 8000, "float64") > 0
    assert sliced_bytes(448, 31, 7872, "float64") > 0 and sliced_bytes(1000, 1000, 4000, "float32") > 0
    for dtype in TYPES:
        assert sliced_bytes(96, 96, 100, dtype) == 0 and sliced_bytes(256, 256, 64, dtype) == 0
        assert sliced_bytes(2048, 2048, 2048, dtype) == 0 and sliced_bytes(1000, 1000, 1000, dtype) == 0
    conf = configs.mfma_config(4096, 4096, 4096).to_c()
    need = ctypes.c_size_t(1)
    assert _lib.lib().gk_sliced_workspace_size(ctypes.byref(conf), None, None, ctypes.byref(need)) == _lib.GK_OK and need.value == 0
    assert _lib.lib().gk_sliced_workspace_size(None, None, None, ctypes.byref(need)) == _lib.GK_ERR_INVALID_ARGUMENT
    assert _lib.lib().gk_matmul_sliced(None, None, None, None, None, None, None, 0, None, 0, None) == _lib.GK_ERR_INVALID_ARGUMENT
    # a caller's limit of LDS that the slices do not fit
    conf = configs_fpu(64, 64, 8000, gk.Float32).to_c()
    try:
        _lib.lib().gk_set_device_limits(16 * 1024, 0)
        assert _lib.lib().gk_sliced_workspace_size(ctypes.byref(conf), None, None, ctypes.byref(need)) == _lib.GK_OK and need.value == 0
    finally:
        _lib.lib().gk_set_device_limits(0, 0)


SIZES = [(16, 56, 746), (33, 31, 1001), (64, 64, 8000), (320, 24, 1914), (1, 100, 3000), (5, 3, 2049), (448, 31, 4099), (100, 200, 515), (153, 180, 7164), (900, 900, 2003), (32, 32, 1024)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_exact_on_whole_numbers(gpu, dtype, ta, tb):
    import torch
    T = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(5)
    integers = lambda m, n: torch.randint(-4, 5, (n, m), generator=gen, device="cuda").to(T).t()
    for M, N, K in SIZES:
        a, b = integers(*((K, M) if ta else (M, K))), integers(*((N, K) if tb else (K, N)))
        exact = (a.double().t() if ta else a.double()) @ (b.double().t() if tb else b.double())
        for alpha, beta in ((1.0, 0.0), (1.0, 1.0), (1.5, 0.5)):
            c = integers(M, N)
            want = alpha * exact + beta * c.double()
            got = gk.mul_(c, gk.Transpose(a) if ta else a, gk.Transpose(b) if tb else b, alpha, beta)
            assert torch.equal(got.double(), want), (M, N, K, alpha, beta)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", TYPES)
def test_error_and_reproducibility(gpu, dtype):
    """Against 64 bits (Float64: against a sum in twice its digits, on the CPU), no further off than the chain gk_matmul makes of the same launch; the same bits on every run."""
    import numpy as np
    import torch
    T = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(6)
    for M, N, K in ((64, 64, 8000), (320, 24, 1914), (100, 200, 515), (448, 31, 4099)):
        assert sliced_bytes(M, N, K, dtype) > 0
        for lo in (0.0, -1.0):
            a = (torch.rand(K, M, generator=gen, device="cuda", dtype=T) * (1 - lo) + lo).t()
            b = (torch.rand(N, K, generator=gen, device="cuda", dtype=T) * (1 - lo) + lo).t()
            c = torch.zeros(N, M, device="cuda", dtype=T).t()
            first = gk.mul_(c, a, b).clone()
            for _ in range(20):
                assert torch.equal(gk.mul_(c, a, b), first)
            conf = configs_fpu(M, N, K, gk.Float32 if dtype == "float32" else gk.Float64)
            chain = torch.zeros(N, M, device="cuda", dtype=T).t()
            gk.matmul(conf, a, b, None, chain, kernel=Kernel.matmul_singlestage)
            wide = np.float64 if dtype == "float32" else np.longdouble
            exact = a.cpu().numpy().astype(wide) @ b.cpu().numpy().astype(wide)
            off = lambda x: float(np.linalg.norm((x.cpu().numpy().astype(wide) - exact).astype(np.float64)) / np.linalg.norm(exact.astype(np.float64)))
            assert off(first) <= off(chain) * 1.05, (M, N, K, lo, off(first), off(chain))


@pytest.mark.gpu
def test_infinite_factors_and_values(gpu):
    """beta scales C in the first slice alone (0 times infinity in the others would be NaN); infinities come through."""
    import torch
    a, b = torch.ones(2000, 40, device="cuda").t(), torch.ones(50, 2000, device="cuda").t()
    c = torch.ones(50, 40, device="cuda").t()
    assert bool(torch.isinf(gk.mul_(c, a, b, 1.0, float("inf"))).all())
    a[3, 1999] = float("inf")
    c.fill_(0)
    gk.mul_(c, a, b)
    assert bool(torch.isinf(c[3]).all()) and bool((c[4] == 2000).all())


@pytest.mark.gpu
def test_graph_replays(gpu):
    import torch
    for dtype in TYPES:
        T = getattr(torch, dtype)
        a, b, c = torch.rand(3000, 70, device="cuda", dtype=T).t(), torch.rand(90, 3000, device="cuda", dtype=T).t(), torch.zeros(90, 70, device="cuda", dtype=T).t()
        gk.mul_(c, a, b)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            gk.mul_(c, a, b)
        for i in range(4):
            a.copy_(torch.rand(3000, 70, device="cuda", dtype=T).t())
            c.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            replayed = c.clone()
            gk.mul_(c, a, b)              # (eager launches between the replays)
            assert torch.equal(replayed, c)
