"""Configurations whose tile is left to the default and whose sizes only small tiles divide: the launch runs on a larger tile over the edges
(``config.larger_tile``), with the bits of the tile that divides and with everything refused that was refused."""
import pytest

import gemmkernels as gk
from gemmkernels import ConfigError, Epilogue, Kernel, Transform, configs
from gemmkernels.config import larger_tile
from gemmkernels.errors import DimensionMismatch


def shape(conf):
    return None if conf is None else tuple(conf.block_shape[x] for x in "MNK")


def test_the_rule():
    # (no GPU: where the line lies, and what a caller's own choices do to it)
    open_ = configs.mfma_config(2240, 5568, 2304)
    assert shape(open_) == (64, 64, 64)
    assert shape(larger_tile(open_, False)) == (256, 256, 64) and shape(larger_tile(open_, True)) == (128, 128, 64)
    assert larger_tile(configs.mfma_config(1920, 1856, 2368), False) is None          # too little to win
    assert larger_tile(configs.mfma_config(4096, 4096, 4096), False) is None          # the best tile divides
    assert larger_tile(configs.mfma_config(2240, 5568, 2304, block_shape=(64, 64, 64)), False) is None
    assert larger_tile(configs.mfma_config(2240, 5568, 2304, warps_per_block=4), False) is None
    assert larger_tile(configs.complex_config(1088, 1600, 2112), False) is None
    for conf in (open_, larger_tile(open_, False)):
        assert gk.kernel_name(conf, Kernel.matmul_pipelined)


LIST = Transform.Elementwise(lambda x: x * 0.5 + 0.25)


@pytest.mark.parametrize("M,N,K,larger", [(1088, 1088, 5248, (128, 128, 64)), (2240, 5568, 2304, (128, 128, 64)), (3648, 3456, 4032, (128, 256, 64))])
@pytest.mark.parametrize("hooks,moves", [(dict(transform_shared_to_regs_a=Transform.Elementwise(lambda x: x * 1.5)), True), (dict(transform_global_to_shared_b=Transform.Elementwise(lambda x: -x)), True),
                                         (dict(transform_shared_to_global_d=LIST), True), (dict(transform_global_to_shared_a=LIST), False),
                                         (dict(transform_shared_to_regs_b=Transform.Elementwise(Transform.relu)), False),
                                         (dict(transform_global_to_shared_a=Transform.Elementwise(lambda x: x * 1.5), transform_shared_to_regs_a=Transform.Elementwise(lambda x: x * 3)), False)])
def test_op_lists_in_the_k_loop_keep_their_tile(M, N, K, larger, hooks, moves):
    # (no GPU: a plan is lowered, not launched)
    torch = pytest.importorskip("torch")
    conf = configs.mfma_config(M, N, K, zero_c=True)
    half = lambda m, n: torch.empty((n, m), dtype=torch.float16).t()
    launch = gk.plan(conf, half(M, K), half(K, N), None, torch.empty((N, M)).t(), kernel=Kernel.matmul_pipelined, **hooks)
    block = launch._conf.block_shape
    assert (block.M, block.N, block.K) == (larger if moves else shape(conf))
    assert (launch._sliced > 0) == (moves and M == 1088)


CASES = [(2240, 5568, 2304, False), (4544, 2048, 2368, False), (2368, 5376, 384, False), (2752, 3712, 1984, True), (1152, 5184, 4800, True), (2240, 2496, 5696, True)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_same_bits_as_the_tile_that_divides(gpu, case):
    import torch
    M, N, K, hooks = CASES[case]
    ta, tb, with_c = case % 2 == 1, case // 2 % 2 == 1, case % 3 != 2
    gen = torch.Generator(device="cuda").manual_seed(case)
    rand = lambda m, n, dtype: torch.rand((n, m), generator=gen, device="cuda").mul_(2).sub_(1).to(dtype).t()
    a, b = rand(*((K, M) if ta else (M, K)), torch.float16), rand(*((N, K) if tb else (K, N)), torch.float16)
    c = rand(M, N, torch.float32) if with_c else None
    options = dict(transform_shared_to_global_d=Transform.Elementwise(Transform.relu), epilogue=Epilogue.Bias(torch.randn(N, generator=gen, device="cuda"))) if hooks else {}
    conf = configs.mfma_config(M, N, K, ta, tb, zero_c=not with_c)
    assert larger_tile(conf, hooks) is not None, shape(conf)
    own = configs.mfma_config(M, N, K, ta, tb, zero_c=not with_c, block_shape=shape(conf))
    print("case", (M, N, K), ta, tb, with_c, hooks, shape(conf), shape(larger_tile(conf, hooks)), flush=True)
    results = []
    for through_plan in (False, True):
        for which in (own, conf):
            d = gk.colmajor_empty((M, N), torch.float32)
            d.fill_(float("nan"))
            if through_plan:
                launch = gk.plan(which, a, b, c, d, kernel=Kernel.matmul_pipelined, **options)
                assert (launch._conf.block_shape.M > 64) == (which is conf)
                launch()
            else:
                gk.matmul(which, a, b, c, d, kernel=Kernel.matmul_pipelined, **options)
            results.append(d)
    assert all(torch.equal(results[0], r) for r in results[1:])


@pytest.mark.gpu
def test_what_was_refused_stays_refused(gpu):
    import torch
    M, N, K = 2240, 5568, 2304
    conf = configs.mfma_config(M, N, K, zero_c=True)
    a, b, d = gk.colmajor_empty((M, K), torch.float16), gk.colmajor_empty((K, N), torch.float16), gk.colmajor_empty((M, N), torch.float32)
    off = torch.empty(M * K + 1, dtype=torch.float16, device="cuda")[1:].view(K, M).t()               # starts off a 16-byte boundary
    odd = torch.empty((K, M + 1), dtype=torch.float16, device="cuda")[:, :M].t()                       # odd leading dimension
    for bad in (off, odd):
        for launch in (lambda: gk.matmul(conf, bad, b, None, d, kernel=Kernel.matmul_pipelined), gk.plan(conf, bad, b, None, d, kernel=Kernel.matmul_pipelined)):
            with pytest.raises(ConfigError, match="aligned|multiple of 16 bytes"):
                launch()
    small = gk.colmajor_empty((M - 64, K), torch.float16)                                               # (an operand that the configuration does not fit)
    with pytest.raises(DimensionMismatch):
        gk.matmul(conf, small, b, None, d, kernel=Kernel.matmul_pipelined)
