"""Products whose operand holds 2^31 elements or more and whose last K tile runs outside the pipeline: every chunk of that tile comes from inside the operand
(``tail_chunk``, whose arithmetic test_tail_chunks.py walks on the host).  Whole numbers, so every sum is exact and the results are compared with == ."""
import pytest

import gemmkernels as gk

pytestmark = pytest.mark.gpu

# M, N, K, A transposed, leading dimension of the wide operand (0: dense).  Tiles of 128 x 256, 256 x 256 (four
# waves), 256 x 128, 64 x 64 in slices of K, and 64 x 64 because the rows of larger tiles lie too far apart
CASES = [(80, 131072, 16400, False, 0), (4096, 131072, 16400, False, 0), (65536, 72, 50264, True, 0), (10000, 64, 4100, True, 215000),
         (991, 3293, 565, True, 1 << 23)]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_more_than_2_31_elements(gpu, case):
    import torch
    M, N, K, ta, ld = CASES[case]
    print("case", CASES[case], flush=True)
    gen = torch.Generator(device="cuda").manual_seed(case)
    wide = torch.empty((M if ta else N, ld or K), dtype=torch.float16, device="cuda")
    assert wide.numel() >= 2 ** 31
    wide = wide[:, :K].random_(-3, 4, generator=gen).t()       # contiguous along k
    other = torch.randint(-3, 4, (N, K) if ta else (K, M), generator=gen, device="cuda").to(torch.float16).t()        # K x N, or M x K
    c = gk.colmajor_empty((M, N), torch.float32)
    c.fill_(float("nan"))
    gk.mul_(c, gk.Transpose(wide) if ta else other, other if ta else wide, 1.0, 0.0)
    # (exact in FP32: at most 9 K < 2^24)
    rows, step = wide.shape[1], 8192
    for at in range(0, rows, step):
        part = wide[:, at:at + step].float()
        want = part.t() @ other.float() if ta else other.float() @ part
        got = c[at:at + step] if ta else c[:, at:at + step]
        assert torch.equal(got, want), at
    del wide, other, c
    torch.cuda.empty_cache()
