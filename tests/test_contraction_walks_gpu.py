"""Contractions whose K, M or N index is three or four modes: the carries of the walk over K, from every mode that a K tile can
end in, and the digits of the rows and columns of a tile.  Small integers, so the sums are exact in any order."""
import numpy as np
import pytest

import gemmkernels as gk
from gemmkernels import contraction


def check(spec, ext):
    import torch
    dm, am, bm = contraction.parse(spec)
    rs = np.random.RandomState(3)
    A = np.asfortranarray(rs.randint(-2, 3, size=[ext[ch] for ch in am]).astype(np.float16))
    B = np.asfortranarray(rs.randint(-2, 3, size=[ext[ch] for ch in bm]).astype(np.float16))
    d = gk.colmajor_empty(tuple(ext[ch] for ch in dm), torch.float32)
    d.fill_(float("nan"))
    gk.contract(spec, gk.colmajor(A), gk.colmajor(B), d)
    torch.cuda.synchronize()
    want = np.einsum(f"{am},{bm}->{dm}", A.astype(np.float64), B.astype(np.float64), optimize=True)
    assert np.array_equal(gk.to_numpy(d).astype(np.float64), want)


# a K tile is one step or several inside the first K mode, whole first modes and a step along the next one, or ends with a mode
@pytest.mark.gpu
@pytest.mark.parametrize("spec,efgh", [("ad-aefgh-dhgfe", e) for e in ((64, 2, 3, 2), (128, 3, 2, 2), (64, 1, 3, 2))] +
                         [("ad-aehgf-dfghe", e) for e in ((64, 2, 3, 2), (192, 2, 2, 3), (8, 16, 3, 2), (16, 4, 5, 3), (4, 2, 32, 3))],
                         ids=lambda e: e if isinstance(e, str) else "x".join(map(str, e)))
def test_walk_over_k(gpu, spec, efgh):
    check(spec, dict(zip("efgh", efgh), a=128, d=64))


@pytest.mark.gpu
@pytest.mark.parametrize("abc", [(64, 3, 2), (32, 2, 3), (16, 4, 2), (64, 1, 4)], ids=lambda e: "x".join(map(str, e)))
@pytest.mark.parametrize("spec", ["adbec-abcf-dfe", "aebdc-acbf-dfe"])
def test_walk_over_rows_and_columns(gpu, spec, abc):
    check(spec, dict(zip("abc", abc), d=32, e=4, f=192))
