"""GPU parity of the FP64 Gram kernel (qumasun_amd/csrc/qg_dense64.hip) against extended precision at
the edges of its tiles, blocks and point ranges.

Tolerance: a sum of K products rounds by at most K eps |a||b|; the products of random columns are held
to 1e-13 of the columns' norms (K <= 20,000: the worst case is 4e-12, the expected sqrt(K) eps 3e-14).
"""
import ctypes

import numpy as np
import pytest

import qumasun_amd as Q
from qumasun_amd import _native as N

pytestmark = pytest.mark.gpu

# points, columns of A and of B: one tile, tile remainders, small / middle / large blocks, several
# blocks, ranges with a partial last step, an odd number of points (the library's path)
CASES = [(2, 1, 1), (514, 16, 16), (1000, 17, 33), (4098, 31, 64), (3330, 90, 100), (2062, 97, 129), (20000, 144, 144),
         (1030, 160, 193), (700, 161, 385), (999, 20, 20)]


@pytest.mark.parametrize("K,M,Nc", CASES)
def test_gram64(gpu, K, M, Nc):
    import torch
    print(f"gram64 {K} {M} {Nc}", flush=True)
    rng = np.random.default_rng(K + M)
    A = rng.standard_normal((M, K)) * 10.0 ** rng.uniform(-3, 3, (M, 1))
    B = rng.standard_normal((Nc, K))
    a, b = torch.from_numpy(A).to(gpu), torch.from_numpy(B).to(gpu)
    ldc = M + 3
    c = torch.full((Nc, ldc), float("nan"), dtype=torch.float64, device=gpu)
    p = [ctypes.c_void_p(t.data_ptr()) for t in (a, b, c)]
    N.check(Q.lib().qg_gram(N.QG_F64, p[0], p[1], K, M, Nc, K, K, p[2], ldc, None))
    torch.cuda.synchronize()
    got = c.cpu().numpy()
    assert np.isnan(got[:, M:]).all()       # nothing written between the columns
    ref = (A.astype(np.longdouble) @ B.T.astype(np.longdouble)).T if K <= 5000 else (A @ B.T).T
    scale = np.linalg.norm(B, axis=1)[:, None] * np.linalg.norm(A, axis=1)[None, :]
    assert float(np.max(np.abs(got[:, :M] - ref) / scale)) <= 1e-13


def test_gram64_special_values(gpu):
    """Values of unused points and bands do not reach the result; infinities and NaN stay in their entries."""
    import torch
    print("gram64 special values", flush=True)
    K, M = 1034, 20
    rng = np.random.default_rng(3)
    buf = torch.full((2, M + 1, K + 6), float("nan"), dtype=torch.float64, device=gpu)
    A = rng.standard_normal((M, K))
    A[4, 7] = np.inf
    A[9, K - 1] = np.nan
    buf[0, :M, :K] = torch.from_numpy(A).to(gpu)
    B = rng.standard_normal((M, K))
    buf[1, :M, :K] = torch.from_numpy(B).to(gpu)
    c = torch.empty((M, M), dtype=torch.float64, device=gpu)
    N.check(Q.lib().qg_gram(N.QG_F64, ctypes.c_void_p(buf[0].data_ptr()), ctypes.c_void_p(buf[1].data_ptr()), K, M, M,
                            K + 6, K + 6, ctypes.c_void_p(c.data_ptr()), M, None))
    torch.cuda.synchronize()
    got = c.cpu().numpy()
    keep = [i for i in range(M) if i not in (4, 9)]
    ref = (A[keep] @ B.T).T
    scale = np.linalg.norm(B, axis=1)[:, None] * np.linalg.norm(A[keep], axis=1)[None, :]
    assert float(np.max(np.abs(got[:, keep] - ref) / scale)) <= 1e-13
    assert np.isnan(got[:, 9]).all() and np.isinf(got[:, 4]).all()
