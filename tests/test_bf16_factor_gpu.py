"""One factor on A of a BF16 product: applied per fragment (widened, multiplied in fp32, rounded once), so the result is that of the
product with A scaled and rounded beforehand, bit for bit -- for every tile, transpose and factor, infinities, NaN and subnormals included."""
import numpy as np
import pytest
import torch

import gemmkernels as gk
from gemmkernels import BFloat16, Float32, Kernel, Layout, Operator, Transform, configs, tuning
from gemmkernels.config import get_config
from gemmkernels.errors import ConfigError
from gemmkernels.tiling import NT

CANDIDATES = tuning.MFMA_CANDIDATES
FACTORS = (1.5, -0.3, 3.0e38, 1.0e-39, float("inf"), 0.0)


def conf_for(M, N, K, ta, tb, block, waves, kernel):
    whole = M % block[0] == 0 and N % block[1] == 0 and K % block[2] == 0
    col, row = (Layout.UnsafeAlignedColMajor, Layout.UnsafeAlignedRowMajor) if whole else (Layout.ColMajor, Layout.RowMajor)
    shared = Layout.Padded[Layout.UnsafeAlignedColMajor[BFloat16], 8]
    return get_config(gemm_shape=NT(M=M, N=N, K=K), operator=Operator.MFMAOp[32, 32, 16, BFloat16, Float32], block_shape=NT(M=block[0], N=block[1], K=block[2]),
                      warps_per_block=waves[0] * waves[1], compute_warp=NT(M=block[0] // waves[0], N=block[1] // waves[1], K=16),
                      global_a_layout=(row if ta else col)[BFloat16], global_b_layout=(row if tb else col)[BFloat16], shared_a_layout=shared, shared_b_layout=shared,
                      global_c_layout=Layout.Zero[Float32], global_d_layout=col[Float32], shared_c_layout=Layout.Zero[Float32],
                      shared_d_layout=Layout.UnsafeAlignedColMajor[Float32], is_a_col_major=not ta, is_b_col_major=not tb, kernel=kernel)


def operands(M, N, K, ta, tb, special):
    g = torch.Generator(device="cuda")
    g.manual_seed(M + 3 * N + 7 * K)
    flat = lambda shape: (torch.rand(tuple(reversed(shape)), generator=g, device="cuda") * 2 - 1).to(torch.bfloat16)
    a, b = flat((K, M) if ta else (M, K)), flat((N, K) if tb else (K, N))
    if special:
        values = torch.tensor([float("inf"), -float("inf"), float("nan"), 3.3e38, 1e-40, -0.0], dtype=torch.bfloat16, device="cuda")
        a.view(-1)[:: a.numel() // 5] = values[: len(a.view(-1)[:: a.numel() // 5])]
    return a.permute(1, 0), b.permute(1, 0)


def test_level_of_the_kernel():
    """No GPU: one scale on A runs on level 1, a scale on B and op lists on level 2."""
    conf = conf_for(512, 512, 512, False, False, (128, 128, 64), (2, 2), Kernel.matmul_pipelined)
    scale = Transform.Elementwise(lambda x: x * 1.5)
    name = lambda **t: gk.kernel_name(conf, Kernel.matmul_pipelined, t)
    assert name(transform_shared_to_regs_a=scale).endswith("_bf16_fused") and name(transform_global_to_shared_a=scale).endswith("_bf16_fused")
    assert name(transform_shared_to_regs_b=scale).endswith("_fused_ab") and name(transform_shared_to_regs_a=Transform.Elementwise(lambda x: x + 1.5)).endswith("_fused_ab")


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("block,waves", CANDIDATES, ids=[f"{b[0]}x{b[1]}x{b[2]}w{w[0]}x{w[1]}" for b, w in CANDIDATES])
def test_factor_on_a_equals_a_scaled_beforehand(gpu, block, waves, ta, tb):
    for M, N, K, factors, special in ((2 * block[0], block[1], 3 * block[2], FACTORS, False), (block[0] + 9, block[1] - 5, 2 * block[2] + 11, (1.5,), True),
                                      (block[0], block[1], block[2], (-0.3, 2.0e38), True)):
        try:
            conf = conf_for(M, N, K, ta, tb, block, waves, Kernel.matmul_pipelined)
        except ConfigError:
            pytest.skip("not compiled for this transpose")
        a, b = operands(M, N, K, ta, tb, special)
        for f in factors:
            hook = Transform.Elementwise(ops=[(Transform.SCALE, f, 0.0)])
            scaled = (a.float() * f).to(torch.bfloat16)
            d, want = (gk.colmajor_empty((M, N), torch.float32) for _ in range(2))
            print("case", block, waves, (M, N, K), ta, tb, f, flush=True)
            gk.matmul(conf, a, b, None, d, transform_shared_to_regs_a=hook, kernel=Kernel.matmul_pipelined)
            gk.matmul(conf, scaled, b, None, want, kernel=Kernel.matmul_pipelined)
            assert torch.equal(d.isnan(), want.isnan()) and torch.equal(d.nan_to_num(nan=0.0), want.nan_to_num(nan=0.0)), (M, N, K, f)


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_slices_of_k_and_the_default_launch(gpu, ta, tb):
    """Integers and an exact factor: every sum is exact, whatever tile and slices mul! picks."""
    for M, N, K in ((70, 61, 2049), (256, 192, 4096), (1030, 1026, 321), (300, 1001, 64)):
        g = torch.Generator(device="cuda")
        g.manual_seed(K)
        ints = lambda shape: torch.randint(-3, 4, tuple(reversed(shape)), generator=g, device="cuda")
        a, b, c = (ints(s).to(t).permute(1, 0) for s, t in (((K, M) if ta else (M, K), torch.bfloat16), ((N, K) if tb else (K, N), torch.bfloat16), ((M, N), torch.float32)))
        want = 1.5 * ((a.T if ta else a).double() @ (b.T if tb else b).double()) + 0.5 * c.double()
        gk.matmatmul_(c, "NT"[ta], "NT"[tb], a, b, 1.5, 0.5)
        assert torch.equal(c.double(), want), (M, N, K)
