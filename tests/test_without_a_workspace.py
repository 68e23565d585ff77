"""Launches that run in slices of K without having been asked to run unsplit where there is no memory for their workspace, as they did before there were slices."""
import contextlib
import sys

import pytest

import gemmkernels as gk
from gemmkernels import Kernel, configs

torch = pytest.importorskip("torch")
mm = sys.modules["gemmkernels.matmul"]


def test_a_plan_without_memory_seldom_asks_again(monkeypatch):
    """No GPU: the launches are recorded, the allocation fails."""
    conf = configs.mfma_config(384, 256, 3776, zero_c=True)
    half = lambda m, n: torch.empty((n, m), dtype=torch.float16).t()
    launch = gk.plan(conf, half(384, 3776), half(3776, 256), None, torch.empty((256, 384)).t(), kernel=Kernel.matmul_pipelined)
    assert launch._sliced > 0
    ran, asked = [], []

    class Library:
        gk_matmul_sliced = staticmethod(lambda *args: ran.append(args[-3:]) or 0)

    def none(*args, **kwargs):
        asked.append(len(ran))
        raise torch.OutOfMemoryError("no memory")
    monkeypatch.setattr(torch, "zeros", none)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(mm, "_load_native", lambda: None)
    monkeypatch.setattr(mm._lib, "lib", lambda: Library)
    monkeypatch.setattr(mm, "_capture_of", lambda stream: None)
    monkeypatch.setattr(mm, "_on", lambda stream: contextlib.nullcontext())
    monkeypatch.setattr(mm, "_workspaces", {})
    monkeypatch.setattr(mm, "_calls_without", {})
    for _ in range(600):
        launch(stream=7)
    assert ran == [(0, 0, 7)] * 600 and asked == [0, 256, 512]


@pytest.mark.gpu
def test_every_entry(gpu, monkeypatch):
    gen = torch.Generator(device="cuda").manual_seed(3)
    whole = lambda m, n, t: torch.randint(-3, 4, (n, m), generator=gen, device="cuda").to(t).t()
    M, N, K = 384, 256, 3776
    a, b, conf = whole(M, K, torch.float16), whole(K, N, torch.float16), configs.mfma_config(M, N, K, zero_c=True)
    d = gk.colmajor_empty((M, N), torch.float32)
    want = a.double() @ b.double()
    single, other = whole(64, 4000, torch.float32), whole(4000, 48, torch.float32)
    e = gk.colmajor_empty((64, 48), torch.float32)
    big = whole(1088, 5248, torch.float16), whole(5248, 1088, torch.float16)
    f = gk.colmajor_empty((1088, 1088), torch.float32)
    x, y, g = whole(128, 4096, torch.float16), whole(4096, 64, torch.float16), gk.colmajor_empty((128, 64), torch.float32)
    entries = [(lambda: gk.matmul(conf, a, b, None, d, kernel=Kernel.matmul_pipelined), d, want),
               (lambda: gk.plan(conf, a, b, None, d, kernel=Kernel.matmul_pipelined)(), d, want),
               (lambda: gk.mul_(e, single, other), e, single.double() @ other.double()),
               (lambda: gk.mul_(f, *big), f, big[0].double() @ big[1].double()),
               (lambda: gk.contract("ab-ae-eb", x, y, g), g, x.double() @ y.double())]
    stream = torch.cuda.Stream()

    def none(*args, **kwargs):
        raise torch.OutOfMemoryError("no memory")
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for out_of_memory in (True, False):
            if out_of_memory:
                monkeypatch.setattr(torch, "zeros", none)
            else:
                monkeypatch.undo()
                mm._calls_without.clear()
            for run, result, right in entries:
                for _ in range(3):
                    result.fill_(float("nan"))
                    run()
                    assert torch.equal(result.double(), right), out_of_memory
    stream.synchronize()
    assert mm._workspaces[(torch.cuda.current_device(), stream.cuda_stream)].numel() > 0
