"""matmul() launches what a plan with the same arguments launches: the same bits, on values whose sum in slices of K is not that of one chain."""
import pytest

import gemmkernels as gk
from gemmkernels import BFloat16, Float32, Kernel, Layout, Operator, Transform, configs

pytestmark = pytest.mark.gpu

LIST = Transform.Elementwise(lambda x: x * 0.5 + 0.25)
HOOKS = [dict(), dict(transform_shared_to_global_d=Transform.Elementwise(Transform.relu)), dict(transform_shared_to_regs_a=Transform.Elementwise(lambda x: x * 1.5)),
         dict(transform_global_to_shared_a=LIST, transform_shared_to_global_d=LIST)]


@pytest.mark.parametrize("hooks", range(len(HOOKS)))
@pytest.mark.parametrize("M,N,K,slices", [(384, 256, 3776, True), (1088, 1088, 5248, True), (2240, 1344, 2304, False)])
@pytest.mark.parametrize("bf16,bias", [(False, False), (False, True), (True, False)])
def test_the_same_bits(gpu, M, N, K, slices, hooks, bf16, bias):
    import torch
    from gemmkernels import Epilogue
    gen = torch.Generator(device="cuda").manual_seed(K + hooks)
    rand = lambda m, n, t: torch.rand((n, m), generator=gen, device="cuda").mul_(2).sub_(1).to(t).t()
    dtype = torch.bfloat16 if bf16 else torch.float16
    a, b, c = rand(M, K, dtype), rand(K, N, dtype), rand(M, N, torch.float32)
    types = {} if not bf16 else dict(operator=Operator.MFMAOp[32, 32, 16, BFloat16, Float32], global_a_layout=Layout.UnsafeAlignedColMajor[BFloat16],
                                     global_b_layout=Layout.UnsafeAlignedColMajor[BFloat16])
    conf = configs.mfma_config(M, N, K, **types)
    options = dict(HOOKS[hooks])
    if bias:
        options["epilogue"] = Epilogue.Bias(torch.randn(N, generator=gen, device="cuda"))
    one, other = gk.colmajor_empty((M, N), torch.float32), gk.colmajor_empty((M, N), torch.float32)
    launch = gk.plan(conf, a, b, c, one, kernel=Kernel.matmul_pipelined, **options)
    lists = hooks == 3
    assert (launch._sliced > 0) == (slices and (not lists or bf16 and M == 384))
    for _ in range(3):
        one.fill_(float("nan"))
        other.fill_(float("nan"))
        launch()
        gk.matmul(conf, a, b, c, other, kernel=Kernel.matmul_pipelined, **options)
        assert torch.equal(one, other)


def test_repeated_launches_in_slices(gpu):
    """From the third on they go from the tensors to the library in C++: on other operands, other streams and in several threads, under capture, and refused
    where the first one would be."""
    import threading
    import torch
    from gemmkernels import ConfigError
    gen = torch.Generator(device="cuda").manual_seed(9)
    whole = lambda m, n: torch.randint(-3, 4, (n, m), generator=gen, device="cuda").to(torch.float16).t()
    M, N, K = 1088, 1088, 5248
    conf = configs.mfma_config(M, N, K, zero_c=True)
    sets = []
    for _ in range(3):
        a, b = whole(M, K), whole(K, N)
        sets.append((a, b, gk.colmajor_empty((M, N), torch.float32), a.double() @ b.double()))
    run = lambda s: gk.matmul(conf, s[0], s[1], None, s[2], kernel=Kernel.matmul_pipelined)
    for _ in range(3):
        for s in sets:
            s[2].fill_(float("nan"))
            run(s)
            assert torch.equal(s[2].double(), s[3])
    assert any(getattr(x, "args", None) for x in conf.__dict__["_prepared"].values())
    off = torch.empty(M * K + 8, dtype=torch.float16, device="cuda")[1:1 + M * K].view(K, M).t()               # starts off a 16-byte boundary
    with pytest.raises(ConfigError, match="aligned"):
        gk.matmul(conf, off, sets[0][1], None, sets[0][2], kernel=Kernel.matmul_pipelined)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(sets[1])
    for _ in range(3):
        sets[1][2].fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(sets[1][2].double(), sets[1][3])
        run(sets[0])
        torch.cuda.synchronize()
    failed = []

    def work(s):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                s[2].fill_(float("nan"))
                run(s)
                if not torch.equal(s[2].double(), s[3]):
                    failed.append(s)
    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(s,)) for s in sets]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
