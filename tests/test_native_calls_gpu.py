"""Calls that go from torch tensors to the library through the module gk_torch: the module is there and takes them, what is out of the ordinary goes the way through Python
with the same results and the same refusals, streams and threads have their own workspaces, and limits set after a launch was prepared hold."""
import threading

import pytest

import gemmkernels as gk
from gemmkernels import ConfigError, Kernel, _lib, _native, configs

pytestmark = pytest.mark.gpu


def integers(rows, cols, dtype, seed=0):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-3, 4, (cols, rows), generator=gen, device="cuda").to(dtype).t()


def test_the_module_takes_the_second_call(gpu):
    import torch
    native = _native.load()
    assert native is not None, "gk_torch.so is not built"
    for M, N, K, dtype in ((33, 20, 17, torch.float32), (64, 64, 4000, torch.float64), (100, 60, 40, torch.float16), (512, 64, 4096, torch.bfloat16)):
        a, b, c = integers(M, K, dtype, 1), integers(K, N, dtype, 2), integers(M, N, torch.float64 if dtype is torch.float64 else torch.float32, 3)
        want = a.double() @ b.double()
        gk.mul_(c, a, b)
        assert torch.equal(c.double(), want)
        c.fill_(float("nan"))
        assert native.mul(c, a, b, False, False, 1.0, 0.0) is True
        assert torch.equal(c.double(), want)
        # another kind: not seen before
        assert native.mul(c, a, b, False, False, 2.0, 0.0) is False and native.mul(c, a, b, True, False, 1.0, 0.0) is False


def test_out_of_the_ordinary(gpu):
    import torch

    class Sub(torch.Tensor):
        pass
    native = _native.load()
    a, b, c = integers(40, 24, torch.float32, 1), integers(24, 16, torch.float32, 2), integers(40, 16, torch.float32, 3)
    want = a.double() @ b.double()
    gk.mul_(c, a, b)
    sub = a.as_subclass(Sub)
    assert native.mul(c, sub, b, False, False, 1.0, 0.0) is False and native.mul(c, a.cpu(), b, False, False, 1.0, 0.0) is False and native.mul(c, 3, b, False, False, 1.0, 0.0) is False
    c.zero_()
    gk.mul_(c, sub, b)
    assert torch.equal(c.double(), want)
    for bad in (lambda: gk.mul_(c, b, b), lambda: gk.mul_(c.t(), a, b)):
        for _ in range(2):
            with pytest.raises((ConfigError, gk.DimensionMismatch) if hasattr(gk, "DimensionMismatch") else Exception):
                bad()
    # more kinds than are kept
    for i in range(1100):
        gk.mul_(c, a, b, 1.0, float(i % 7) + i / 2048.0)
    c.zero_()
    gk.mul_(c, a, b)
    assert torch.equal(c.double(), want)


def test_limits_set_after_a_launch_was_prepared(gpu):
    import torch
    conf = configs.mfma_config(512, 512, 512, zero_c=True, block_shape=(256, 256, 64))
    a, b, d = integers(512, 512, torch.float16, 1), integers(512, 512, torch.float16, 2), gk.colmajor_empty((512, 512), torch.float32)
    plan = gk.plan(conf, a, b, None, d, kernel=Kernel.matmul_pipelined)
    launches = (plan, lambda: gk.matmul(conf, a, b, None, d, kernel=Kernel.matmul_pipelined))
    for launch in launches:
        launch()
        launch()
    try:
        _lib.lib().gk_set_device_limits(64 * 1024, 0)
        for launch in launches:
            with pytest.raises(ConfigError, match="shared memory"):
                launch()
    finally:
        _lib.lib().gk_set_device_limits(0, 0)
    for launch in launches:
        d.fill_(float("nan"))
        launch()
        assert torch.equal(d.double(), a.double() @ b.double())


def test_configured_launches_look_at_their_operands(gpu):
    """After a launch was kept: operands off 16-byte boundaries, of other leading dimensions and of shapes that a layout does not take."""
    import torch
    conf = configs.diagonal_config(256, 320, zero_c=True)
    a, b, d = torch.randn(256, device="cuda").half(), integers(256, 320, torch.float16), gk.colmajor_empty((256, 320), torch.float32)
    for _ in range(2):
        gk.matmul(conf, a, b, None, d, kernel=Kernel.matmul_singlestage)
    off = torch.empty(256 * 320 + 1, device="cuda", dtype=torch.float16)[1:].view(320, 256).t()
    with pytest.raises(ConfigError, match="aligned"):
        gk.matmul(conf, a, off, None, d, kernel=Kernel.matmul_singlestage)
    with pytest.raises(ConfigError, match="column-major"):
        gk.matmul(conf, a, b.t().contiguous(), None, d, kernel=Kernel.matmul_singlestage)
    wide = torch.empty(320, 512, device="cuda", dtype=torch.float16).t()[:256]
    wide.copy_(b)
    want = a.double()[:, None] * b.double()
    for x in (wide, b, wide):
        d.fill_(float("nan"))
        gk.matmul(conf, a, x, None, d, kernel=Kernel.matmul_singlestage)
        assert torch.equal(d.double(), want)
    for planar in (False, True):
        make = configs.complex_planar_config if planar else configs.complex_config
        shape = (lambda m, n: (m, n, 2)) if planar else (lambda m, n: (2, m, n))
        t = lambda s, dtype: torch.randint(-3, 4, tuple(reversed(s)), device="cuda").to(dtype).permute(2, 1, 0)
        conf = make(128, 64, 192, False, False, zero_c=True)
        x, y, z = t(shape(128, 192), torch.float16), t(shape(192, 64), torch.float16), t(shape(128, 64), torch.float32)
        parts = lambda v: torch.complex(v[..., 0].double(), v[..., 1].double()) if planar else torch.complex(v[0].double(), v[1].double())
        for _ in range(3):
            z.fill_(float("nan"))
            gk.matmul(conf, x, y, None, z, kernel=Kernel.matmul_pipelined)
            assert torch.equal(parts(z), parts(x) @ parts(y))


def test_threads_and_streams(gpu):
    """Products in slices from four threads on four streams, each against its own result: a workspace per stream."""
    import torch
    shapes = [(64, 64, 4000), (300, 24, 1900), (512, 64, 4096), (128, 192, 3000)]
    wrong = []

    def work(i):
        torch.cuda.set_device(0)
        M, N, K = shapes[i]
        dtype = torch.float32 if i < 2 else torch.float16
        with torch.cuda.stream(torch.cuda.Stream()):
            a, b, c = integers(M, K, dtype, i), integers(K, N, dtype, i + 9), integers(M, N, torch.float32, i)
            want = a.double() @ b.double()
            for _ in range(60):
                c.fill_(float("nan"))
                gk.mul_(c, a, b)
                if not torch.equal(c.double(), want):
                    wrong.append(i)
                    return
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
