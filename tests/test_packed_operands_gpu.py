"""Large 16-bit products whose columns start off 16-byte boundaries: ``mul_`` copies such operands to columns on 128-byte lines
first.  The launch is the same one, so the result is that of the product on the operands as they lie, bit for bit."""
import itertools

import pytest
import torch

import gemmkernels as gk
from gemmkernels import _lib
from gemmkernels.matmul import matmatmul_plan, packed_leading_dims


class _Layouts:
    """The fields of a lowered configuration that the rule looks at, of op(A) op(B) on matrices with the leading dimensions given."""

    def __new__(cls, M, N, K, ta, tb, lda, ldb):
        conf = _lib.gk_config()
        conf.op.kind = gk.Operator.MFMA
        conf.matmul_shape.M, conf.matmul_shape.N, conf.matmul_shape.K = M, N, K
        conf.global_a_layout.kind, conf.global_b_layout.kind = 1 + ta, 1 + tb        # ColMajor, RowMajor
        conf.global_a_layout.ld, conf.global_b_layout.ld = lda, ldb
        tile = gk.default_block_shape(gk.Operator.MFMAOp[32, 32, 16, gk.BFloat16, gk.Float32], gk.NT(M=M, N=N, K=K), tile_sized=False, a_kmajor=ta, b_kmajor=not tb)
        conf.block_shape.M, conf.block_shape.N, conf.block_shape.K = tile.M, tile.N, tile.K
        return conf


def test_the_rule():
    """No GPU: which products are worth the copies."""
    dims = lambda M, N, K, ta, tb, a=0, b=0: packed_leading_dims(_Layouts(M, N, K, ta, tb, K if ta else M, N if tb else K), a, b)
    assert dims(4001, 4003, 4005, True, False) == (4032, 4032)
    assert dims(4001, 4003, 4005, False, True) == (4032, 4032)
    assert dims(6001, 5003, 7100, False, False) == (6016, 7104)
    assert dims(4001, 4003, 8100, False, False) is None                           # (copies and operands outgrow the memory-side cache)
    assert dims(4000, 4000, 4000, True, False) is None and dims(4096, 4096, 4096, False, False) is None
    assert dims(4096, 4096, 4096, False, False, 2, 6) == (4096, 4096)             # misaligned addresses
    assert dims(5000, 5000, 5001, False, False) == (None, 5056)                   # one operand, contiguous along k
    assert dims(4000, 4000, 4001, False, False) is None                           # (less work: level or slower but for rotating inputs)
    assert dims(2000, 8000, 8001, False, False) is None                           # (a copy of most of what is read)
    # both operands: by the share of the product's time that copying them takes, more where they are contiguous along k
    assert all(dims(1501, 8003, 8005, ta, tb) is None for ta, tb in itertools.product((False, True), repeat=2))
    assert [dims(1001, 8003, 4005, ta, tb) is not None for ta, tb in ((False, False), (False, True), (True, False), (True, True))] == [False, False, True, False]
    assert [dims(2001, 2003, 6005, ta, tb) is not None for ta, tb in ((False, False), (False, True), (True, False), (True, True))] == [True, False, True, True]
    assert all(dims(3001, 3003, 3005, ta, tb) is not None for ta, tb in itertools.product((False, True), repeat=2))
    assert dims(4001, 4000, 4000, False, False) is None                           # one operand, contiguous along m
    assert dims(2001, 2003, 4005, True, False) is None                            # too little work
    assert dims(131, 8191, 31111, True, False) is None                            # too few rows
    assert dims(16001, 16001, 16001, True, False) is None                         # copies of more than 512 MiB


def test_a_launch_without_memory_for_copies_seldom_asks_again(monkeypatch):
    """No GPU: the launches are recorded, the allocation fails."""
    import sys
    matmul = sys.modules["gemmkernels.matmul"]
    host = lambda rows, cols, dtype: torch.empty((cols, rows), dtype=dtype).t()
    p = matmatmul_plan(host(3001, 2999, torch.float32), 'N', 'N', host(3001, 3003, torch.float16), host(3003, 2999, torch.float16), 1.0, 0.0)
    launch = matmul._MulLaunchOnCopies(p, packed_leading_dims(p._conf, 0, 0))
    plain, asked = [], []
    launch._fn = lambda conf, a, b, c, d, *rest: plain.append((a, b, c)) or _lib.GK_OK

    def none(*args, **kwargs):
        asked.append(len(plain))
        raise torch.OutOfMemoryError("no memory")
    monkeypatch.setattr(torch, "empty", none)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    for _ in range(600):
        launch(2, 4, 6, 0)
    assert plain == [(2, 4, 6)] * 600 and asked == [0, 256, 512]


def _odd(rows, cols, ld, dtype, gen, offset=0):
    buffer = (torch.rand(ld * (cols - 1) + rows + offset, generator=gen, device="cuda") * 2 - 1).to(dtype)      # ends with the last column
    return torch.as_strided(buffer, (rows, cols), (1, ld), offset)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,ld,offset", [(1, 1, 1, 0), (7, 17, 9, 1), (8, 16, 8, 0), (511, 33, 513, 3), (512, 5, 515, 1), (515, 20, 515, 0), (1029, 3, 2001, 7)])
def test_pack_columns(rows, cols, ld, offset):
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x, y = _odd(rows, cols, ld, torch.float16, gen, offset), _odd(rows + 1, cols + 2, ld + 1, torch.float16, gen)
    dims = [(-(-r // 8) * 8) for r in (rows, rows + 1)]
    copies = [torch.full((c, d), -2.0, dtype=torch.float16, device="cuda") for c, d in zip((cols, cols + 2), dims)]
    job = lambda m, copy, d: (m.data_ptr(), m.shape[0], m.shape[1], m.stride(1) if m.shape[1] > 1 else m.shape[0], copy.data_ptr(), d)
    stream = torch.cuda.current_stream().cuda_stream
    assert _lib.lib().gk_pack_columns(*job(x, copies[0], dims[0]), *job(y, copies[1], dims[1]), stream) == _lib.GK_OK, _lib.last_error()
    for m, copy in zip((x, y), copies):
        assert torch.equal(copy[:, :m.shape[0]].t(), m) and bool((copy[:, m.shape[0]:] == -2.0).all())
    copies[0].fill_(-2.0)
    assert _lib.lib().gk_pack_columns(*job(x, copies[0], dims[0]), None, 0, 0, 0, None, 0, stream) == _lib.GK_OK, _lib.last_error()
    assert torch.equal(copies[0][:, :rows].t(), x) and bool((copies[0][:, rows:] == -2.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,ld,offset", [(1, 1, 1, 0), (7, 17, 9, 1), (8, 16, 8, 0), (9, 4, 9, 2), (511, 33, 513, 3), (512, 5, 515, 1), (519, 20, 519, 0), (1029, 3, 2001, 7)])
@pytest.mark.parametrize("more_rows,more_cols", [(0, 0), (1, 0), (9, 3), (63, 16), (520, 1)])
def test_pack_columns_padded(rows, cols, ld, offset, more_rows, more_cols):
    """Zeros behind the rows and the columns of the matrix, what lies behind the rows of the copy left alone; NaN in the source behind its columns."""
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x = _odd(rows, cols, ld, torch.float16, gen, offset)
    if cols > 1:
        torch.as_strided(x, (ld - rows, cols - 1), (1, ld), offset + rows).fill_(float("nan"))
    rows_copy, cols_copy = rows + more_rows, cols + more_cols
    ld_copy = -(-rows_copy // 8) * 8 + 8
    copies = [torch.full((cols_copy + 1, ld_copy), -2.0, dtype=torch.float16, device="cuda") for _ in range(2)]
    job = lambda copy: (x.data_ptr(), rows, cols, ld, copy.data_ptr(), ld_copy, rows_copy, cols_copy)
    stream = torch.cuda.current_stream().cuda_stream
    assert _lib.lib().gk_pack_columns_padded(*job(copies[0]), *job(copies[1]), stream) == _lib.GK_OK, _lib.last_error()
    want = torch.full((cols_copy + 1, ld_copy), -2.0, dtype=torch.float16, device="cuda")
    want[:cols_copy, :rows_copy] = 0
    want[:cols, :rows] = x.t()
    assert torch.equal(copies[0].view(torch.int16), want.view(torch.int16)) and torch.equal(copies[1].view(torch.int16), want.view(torch.int16))


def test_pack_columns_refuses():
    """No GPU: nothing is launched."""
    pack = _lib.lib().gk_pack_columns
    none = (None, 0, 0, 0, None, 0, None)
    assert pack(None, 8, 8, 8, 256, 8, *none) == _lib.GK_ERR_INVALID_ARGUMENT
    assert pack(256, 8, 8, 7, 256, 8, *none) == _lib.GK_ERR_INVALID_ARGUMENT
    assert pack(256, 9, 8, 9, 256, 9, *none) == _lib.GK_ERR_INVALID_ARGUMENT
    assert pack(257, 8, 8, 8, 256, 8, *none) == _lib.GK_ERR_ALIGNMENT
    assert pack(256, 8, 8, 8, 264, 8, *none) == _lib.GK_ERR_ALIGNMENT
    assert pack(256, 8, 8, 8, 256, 8, 256, 8, -1, 8, 256, 8, None) == _lib.GK_ERR_INVALID_ARGUMENT
    assert pack(256, 1 << 20, 8, 1 << 20, 256, 1 << 20, *none) == _lib.GK_ERR_INVALID_ARGUMENT
    padded = _lib.lib().gk_pack_columns_padded
    none = (None, 0, 0, 0, None, 0, 0, 0, None)
    assert padded(256, 8, 8, 8, 256, 16, 7, 8, *none) == _lib.GK_ERR_INVALID_ARGUMENT
    assert padded(256, 8, 8, 8, 256, 16, 8, 7, *none) == _lib.GK_ERR_INVALID_ARGUMENT
    assert padded(256, 8, 8, 8, 256, 16, 17, 8, *none) == _lib.GK_ERR_INVALID_ARGUMENT


class _Poisoned:
    """Buffers of bytes that ``torch.empty`` makes are full of NaN (0xFF), whatever the allocator had left there; counts them."""

    def __init__(self, monkeypatch):
        self.made, empty = 0, torch.empty

        def poisoned(*args, **kwargs):
            out = empty(*args, **kwargs)
            if kwargs.get("dtype") is torch.uint8:
                self.made += 1
                out.fill_(255)
            return out
        monkeypatch.setattr(torch, "empty", poisoned)


@pytest.mark.gpu
@pytest.mark.parametrize("ab,cd", [(torch.bfloat16, torch.float32), (torch.float16, torch.float32), (torch.float16, torch.float16)])
@pytest.mark.parametrize("ta,tb", list(itertools.product((False, True), repeat=2)))
def test_product_on_copies(ta, tb, ab, cd, monkeypatch):
    """Against the plan of the same product, which launches on the operands as they lie; a call under capture does so too.  What
    the copies do not fill is NaN."""
    M, N, K = 3001, 2999, 3003
    poisoned = _Poisoned(monkeypatch)
    gen = torch.Generator(device="cuda").manual_seed(5)
    a = _odd(K, M, K, ab, gen, 1) if ta else _odd(M, K, M + 2, ab, gen)
    b = _odd(N, K, N, ab, gen) if tb else _odd(K, N, K, ab, gen, 3)
    c = (torch.rand(N, M, generator=gen, device="cuda") * 2 - 1).to(cd).t()
    for alpha, beta in ((1.0, 0.0), (1.5, 0.5)):
        ref, out, captured = (c.clone(memory_format=torch.preserve_format) for _ in range(3))
        matmatmul_plan(ref, 'T' if ta else 'N', 'T' if tb else 'N', a, b, alpha, beta)()
        call = lambda d: gk.mul_(d, gk.Transpose(a) if ta else a, gk.Transpose(b) if tb else b, alpha, beta)
        before = poisoned.made
        call(out)
        assert poisoned.made == before + 1
        assert torch.equal(out, ref)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call(captured)
        assert poisoned.made == before + 1
        for _ in range(2):
            captured.copy_(c)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(captured, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_one_operand_on_a_copy(ta, tb, monkeypatch):
    """The operand that is contiguous along an odd K is copied, the other stays: the partial K tile runs as it does on the operands
    as they lie, next to NaN behind the rows of the copy."""
    M, N, K = 4800, 4992, 3501
    poisoned = _Poisoned(monkeypatch)
    gen = torch.Generator(device="cuda").manual_seed(8)
    a = _odd(K, M, K, torch.float16, gen) if ta else _odd(M, K, M, torch.float16, gen)
    b = _odd(N, K, N, torch.float16, gen) if tb else _odd(K, N, K, torch.float16, gen)
    ref, out = (gk.colmajor_empty((M, N), torch.float32) for _ in range(2))
    p = matmatmul_plan(ref, 'T' if ta else 'N', 'T' if tb else 'N', a, b, 1.0, 0.0)
    assert packed_leading_dims(p._conf, a.data_ptr(), b.data_ptr()) == ((3520, None) if ta else (None, 3520))
    p()
    gk.mul_(out, gk.Transpose(a) if ta else a, gk.Transpose(b) if tb else b)
    assert poisoned.made == 1 and torch.equal(out, ref)


@pytest.mark.gpu
def test_streams_and_no_memory(monkeypatch):
    """On a stream of its own, beside the default one, and where the copies find no memory: the same bits."""
    M = N = K = 3001
    gen = torch.Generator(device="cuda").manual_seed(6)
    a, b = _odd(M, K, M, torch.bfloat16, gen), _odd(K, N, K, torch.bfloat16, gen)
    ref, out, other = (gk.colmajor_empty((M, N), torch.float32) for _ in range(3))
    p = matmatmul_plan(ref, 'N', 'N', a, b, 1.0, 0.0)
    assert packed_leading_dims(p._conf, a.data_ptr(), b.data_ptr()) is not None
    p()
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    for _ in range(3):
        gk.mul_(out, a, b)
        with torch.cuda.stream(stream):
            gk.mul_(other, a, b)
    torch.cuda.synchronize()
    assert torch.equal(out, ref) and torch.equal(other, ref)
    out.zero_()

    asked = []

    def none(*args, **kwargs):
        asked.append(args)
        raise torch.OutOfMemoryError("no memory")
    monkeypatch.setattr(torch, "empty", none)
    gk.mul_(out, a, b)
    monkeypatch.undo()
    assert len(asked) == 1 and torch.equal(out, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("ab", [torch.float16, torch.bfloat16])
def test_an_infinite_factor_and_infinite_values(ab):
    """K = 6048 is whole tiles of 32, on which the product runs, and 94.5 of 64: zeros behind it must not meet an infinite alpha (values of one
    sign: every output is infinite), nor change what infinities and NaN in A and B give."""
    M, N, K = 2001, 2003, 6048
    gen = torch.Generator(device="cuda").manual_seed(7)
    a, b = _odd(K, M, K + 3, ab, gen).abs_(), _odd(K, N, K + 1, ab, gen).abs_()
    for spoil in (False, True):
        if spoil:
            a[K - 1, 5], a[0, M - 1], b[K - 1, 7] = float("inf"), float("nan"), float("-inf")
        for alpha in (float("inf"), 1e6, 1.5, 1.0):                 # (1e6 is infinite in FP16)
            ref, out = (gk.colmajor_empty((M, N), torch.float32) for _ in range(2))
            p = matmatmul_plan(ref, 'T', 'N', a, b, alpha, 0.0)
            assert packed_leading_dims(p._conf, a.data_ptr(), b.data_ptr()) is not None and p._conf.block_shape.K == 32
            p()
            gk.mul_(out, gk.Transpose(a), b, alpha, 0.0)
            assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.nan_to_num(), ref.nan_to_num())
            assert spoil or bool((out == float("inf")).all() if alpha == float("inf") or alpha == 1e6 and ab is torch.float16 else out.isfinite().all())
