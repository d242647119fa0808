"""Which kernels the nonlocal forces run (told by their names): FP64 states the one pass over psi, FP32
states the chain of gradient blocks and row or table projections, whose order of rounding their forces keep.
Forces against the oracle: relative 2-norm FP64 <= 1e-10, FP32 <= 2e-5, as for every force form."""
import numpy as np
import pytest

import qumasun_amd as Q
from test_gpu_kernel_families import Cell, _any, _dtype, _kernels
from test_gpu_sphere import GAUSS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(32, 21, 19), (33, 21, 19)])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_force_kernels(gpu, oracle, prec, n):
    import torch
    print(f"force kernels {prec} {n}", flush=True)
    c = Cell(oracle, n, GAUSS, 6)
    x = torch.from_numpy(c.X).to(gpu).to(_dtype(prec))
    occ = np.array([2.0, 2.0, 0.0, 1.5, 1.0, 0.0])
    res = []
    names = _kernels(lambda: res.append(c.integ.EnergyForceNonlocal(x, occ)))
    if prec == "f64":
        assert _any(names, "sphere_force_kernel") and not _any(names, "gradient8_kernel"), names
    else:
        assert _any(names, "gradient8_kernel") and not _any(names, "sphere"), names
    onl = oracle.OracleNL(c.n, c.h, c.pos, np.zeros(len(c.pos), np.int32), c.projs)
    e_ref, f_ref = oracle.nonlocal_energy_force(c.n, c.h, onl, c.X, occ, np.zeros(len(c.pos), np.int32), c.projs)
    e, f = res[0]
    tol = 1e-10 if prec == "f64" else 2e-5
    assert abs(e - e_ref) <= tol * abs(e_ref) and np.linalg.norm(f - f_ref) <= tol * np.linalg.norm(f_ref)
