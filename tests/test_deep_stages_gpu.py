"""The small tiles with four LDS stages that launches with few workgroups run on, at the sizes where they can go wrong: fewer K tiles than
stages, partial last K tiles, BLOCK_K = 32 fetched in pairs, tile counts on either side of the rule; integers, so that every sum is
exact and the result equals the float64 product bit for bit."""
import numpy as np
import pytest
import torch

import gemmkernels as gk
from gemmkernels import BFloat16, Float16, Float32, Kernel, Layout, Operator, _lib, configs, contraction
from gemmkernels.config import get_config
from gemmkernels.tiling import NT

DEEP = "_w2x2_s4"


def conf_for(M, N, K, ta, tb, block, T=Float16, zero_c=True):
    """Aligned layouts where the tile divides the sizes, the bounds-checked ones elsewhere."""
    whole = M % block[0] == 0 and N % block[1] == 0 and K % block[2] == 0
    col, row = (Layout.UnsafeAlignedColMajor, Layout.UnsafeAlignedRowMajor) if whole else (Layout.ColMajor, Layout.RowMajor)
    shared = Layout.Padded[Layout.UnsafeAlignedColMajor[T], 8]
    return get_config(gemm_shape=NT(M=M, N=N, K=K), operator=Operator.MFMAOp[32, 32, 16, T, Float32], block_shape=NT(M=block[0], N=block[1], K=block[2]),
                      global_a_layout=(row if ta else col)[T], global_b_layout=(row if tb else col)[T], shared_a_layout=shared, shared_b_layout=shared,
                      global_c_layout=Layout.Zero[Float32] if zero_c else col[Float32], global_d_layout=col[Float32],
                      shared_c_layout=Layout.Zero[Float32] if zero_c else Layout.UnsafeAlignedColMajor[Float32],
                      shared_d_layout=Layout.UnsafeAlignedColMajor[Float32], is_a_col_major=not ta, is_b_col_major=not tb)


def integers(shape, dtype, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    flat = torch.randint(-3, 4, tuple(reversed(shape)), generator=g, device="cuda").to(dtype)
    return flat.permute(*reversed(range(len(shape))))


def test_which_launches_are_deep():
    """No GPU: the rule as gk_kernel_name reports it, and the shallow instance under a limit of 64 KiB of LDS."""
    name = lambda *size, **kw: gk.kernel_name(conf_for(*size, False, False, **kw), Kernel.matmul_pipelined)
    assert DEEP in name(2048, 2048, 512, block=(128, 128, 64)) and DEEP + "_pairs" in name(2048, 2048, 512, block=(128, 128, 32))
    assert "_s2" in name(2048, 2176, 512, block=(128, 128, 64)) and "_pairs" not in name(2048, 2176, 512, block=(128, 128, 32))
    assert "_pairs" not in name(512, 512, 96, block=(128, 128, 32)) and "_pairs" not in name(512, 512, 96, block=(64, 64, 32))
    assert DEEP in name(2048, 1024, 512, block=(64, 64, 64)) and "_s2" in name(2048, 1088, 512, block=(64, 64, 64))
    assert DEEP + "_pairs" in name(512, 512, 512, block=(64, 64, 32)) and DEEP + "_pairs" in name(501, 333, 1601, block=(64, 64, 32))
    assert "_pairs" not in name(501, 333, 1001, block=(64, 64, 32)) and "_pairs" not in name(512, 512, 1632, block=(64, 64, 32))
    limit = _lib.lib().gk_set_device_limits
    try:
        limit(64 * 1024, 0)
        assert "_s2" in name(512, 512, 512, block=(128, 128, 64)) and "_pairs" not in name(512, 512, 512, block=(128, 128, 32))
        assert "_w2x2" in gk.kernel_name(configs.complex_config(128, 128, 128, block_shape=NT(M=64, N=64, K=64)), Kernel.matmul_pipelined)
    finally:
        limit(0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("block", [(64, 64, 64), (64, 64, 32), (128, 128, 64), (128, 128, 32)])
@pytest.mark.parametrize("T", [Float16, BFloat16])
def test_plain_products(gpu, T, block, ta, tb):
    dtype = torch.float16 if T is Float16 else torch.bfloat16
    for M, N, K in ((128, 256, 64), (128, 128, 128), (256, 128, 192), (128, 128, 320), (128, 256, 576), (200, 136, 72), (137, 67, 333), (131, 201, 1601)):
        a, b = integers((K, M) if ta else (M, K), dtype, 1), integers((N, K) if tb else (K, N), dtype, 2)
        c = integers((M, N), torch.float32, 3)
        want = (a.T if ta else a).double() @ (b.T if tb else b).double()
        for zero_c in (True, False):
            conf = conf_for(M, N, K, ta, tb, block, T, zero_c)
            print("case", gk.kernel_name(conf, Kernel.matmul_pipelined), (M, N, K), flush=True)
            d = gk.colmajor_empty((M, N), torch.float32)
            d.fill_(float("nan"))
            gk.matmul(conf, a, b, None if zero_c else c, d, kernel=Kernel.matmul_pipelined)
            assert torch.equal(d.double(), want if zero_c else want + c.double()), (M, N, K, zero_c)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,block", [((1024, 2048, 128), (64, 64, 64)), ((1024, 2112, 128), (64, 64, 64)), ((2048, 2048, 192), (128, 128, 32)), ((2048, 2176, 192), (128, 128, 32))])
def test_tile_counts_on_either_side_of_the_rule(gpu, dims, block):
    M, N, K = dims
    a, b = integers((M, K), torch.float16, 1), integers((N, K), torch.float16, 2)
    d = gk.colmajor_empty((M, N), torch.float32)
    gk.matmul(conf_for(M, N, K, False, True, block), a, b, None, d, kernel=Kernel.matmul_pipelined)
    assert torch.equal(d.double(), a.double() @ b.T.double())


@pytest.mark.gpu
@pytest.mark.parametrize("ext", [dict(a=32, b=2, c=2, d=32, e=32, f=2), dict(a=32, b=4, c=2, d=64, e=64, f=6), dict(a=64, b=2, c=6, d=32, e=32, f=32), dict(a=64, b=34, c=18, d=64, e=32, f=4)])
def test_contractions_on_the_small_tiles(gpu, ext):
    """One K tile and many, K modes that share a K tile, tile counts below and above the rule."""
    a, b = integers([ext[m] for m in "aebf"], torch.float16, 1), integers([ext[m] for m in "dfce"], torch.float16, 2)
    d = gk.colmajor_empty([ext[m] for m in "abcd"], torch.float32)
    d.fill_(float("nan"))
    p = contraction.plan("abcd-aebf-dfce", a, b, d)
    print("case", p.kernel_name, ext, flush=True)
    gk.contract("abcd-aebf-dfce", a, b, d)
    want = np.einsum("aebf,dfce->abcd", a.double().cpu().numpy(), b.double().cpu().numpy(), optimize=True)
    assert np.array_equal(d.cpu().numpy(), want)
    # other operands of the same kind through the launch that is kept for it, and their views of another alignment refused
    a2 = integers([ext[m] for m in "aebf"], torch.float16, 5)
    gk.contract("abcd-aebf-dfce", a2, b, d, c=d)
    want2 = want + np.einsum("aebf,dfce->abcd", a2.double().cpu().numpy(), b.double().cpu().numpy(), optimize=True)
    assert np.array_equal(d.cpu().numpy(), want2)
    flat = torch.empty(a.numel() + 1, dtype=torch.float16, device="cuda")
    off = flat[1:].view(tuple(reversed(a.shape))).permute(*reversed(range(a.dim())))
    with pytest.raises(gk.ConfigError):
        gk.contract("abcd-aebf-dfce", off, b, d)


@pytest.mark.gpu
@pytest.mark.parametrize("planar", [False, True])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_complex_products(gpu, planar, ta, tb):
    for block, dims in (((32, 32, 64), (64, 32, 64)), ((32, 32, 64), (96, 64, 320)), ((64, 64, 64), (128, 64, 128)), ((64, 64, 64), (64, 192, 384)), ((64, 64, 64), (1088, 1088, 64))):
        M, N, K = dims
        shape = (lambda s: s + (2,)) if planar else (lambda s: (2,) + s)
        make = configs.complex_planar_config if planar else configs.complex_config
        conf = make(M, N, K, ta, tb, block_shape=NT(M=block[0], N=block[1], K=block[2]), zero_c=False)
        a, b = integers(shape((K, M) if ta else (M, K)), torch.float16, 1), integers(shape((N, K) if tb else (K, N)), torch.float16, 2)
        c = integers(shape((M, N)), torch.float32, 3)
        d = gk.colmajor_empty(shape((M, N)), torch.float32)
        gk.matmul(conf, a, b, c, d, kernel=Kernel.matmul_pipelined)
        part = (lambda x, i: x[..., i].double()) if planar else (lambda x, i: x[i].double())
        ar, ai, br, bi = (part(x, i).T if t else part(x, i) for x, t in ((a, ta), (b, tb)) for i in (0, 1))
        print("case", gk.kernel_name(conf, Kernel.matmul_pipelined), dims, flush=True)
        assert torch.equal(part(d, 0), ar @ br - ai @ bi + part(c, 0)), (block, dims)
        assert torch.equal(part(d, 1), ar @ bi + ai @ br + part(c, 1)), (block, dims)
