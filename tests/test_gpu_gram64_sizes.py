"""GPU parity of every size of the FP64 Gram kernel (qumasun_amd/csrc/qg_dense64.hip: half of the block's tile
rows x quarter of its tile columns), one block and several, where the rule chooses it; and the library's
product where that is chosen.  The kernel that ran is told by its name.

Tolerance 1e-13 of the columns' norms (K = 4098 and 13,826: the worst case of K rounded products is
K eps = 9e-13 and 3e-12, the expected sqrt(K) eps 1.4e-14 and 2.6e-14)."""
import ctypes

import numpy as np
import pytest

import qumasun_amd as Q
from qumasun_amd import _native as N
from test_gpu_kernel_families import _kernels

pytestmark = pytest.mark.gpu

SIZES = {(1, 1): (16, 20), (1, 2): (1, 193), (1, 3): (17, 385), (2, 1): (33, 1), (2, 2): (49, 65), (2, 3): (50, 260),
         (3, 1): (177, 10), (3, 2): (161, 210), (3, 3): (90, 129), (4, 1): (97, 30), (4, 2): (200, 193), (4, 3): (200, 260),
         (5, 1): (300, 1), (5, 2): (129, 65), (5, 3): (144, 129)}
SEVERAL = {(5, 3): (300, 260)}


def _gram(gpu, K, M, Nc):
    import torch
    rng = np.random.default_rng(M * 1000 + Nc)
    A, B = rng.standard_normal((M, K)), rng.standard_normal((Nc, K))
    a, b = torch.from_numpy(A).to(gpu), torch.from_numpy(B).to(gpu)
    c = torch.full((Nc, M), float("nan"), dtype=torch.float64, device=gpu)
    names = _kernels(lambda: N.check(Q.lib().qg_gram(N.QG_F64, *[ctypes.c_void_p(t.data_ptr()) for t in (a, b)], K, M, Nc, K, K,
                                                     ctypes.c_void_p(c.data_ptr()), M, None)))
    scale = np.linalg.norm(B, axis=1)[:, None] * np.linalg.norm(A, axis=1)[None, :]
    assert float(np.max(np.abs(c.cpu().numpy() - (A @ B.T).T) / scale)) <= 1e-13
    return names


@pytest.mark.parametrize("size", sorted(SIZES))
def test_every_size(gpu, size):
    print(f"gram64 size {size}", flush=True)
    names = _gram(gpu, 4098, *SIZES[size])
    assert any("gram64_kernel<%d, %d>" % size in n for n in names), names


def test_several_blocks_of_the_largest(gpu):
    print("gram64 several blocks", flush=True)
    assert any("gram64_kernel<5, 3>" in n for n in _gram(gpu, 13826, *SEVERAL[5, 3]))


@pytest.mark.parametrize("K,M,Nc", [(64000, 256, 256), (1030, 160, 193)])
def test_library_where_it_is_faster(gpu, K, M, Nc):
    print(f"gram library {K} {M} {Nc}", flush=True)
    assert not any("gram64_kernel" in n for n in _gram(gpu, K, M, Nc))
