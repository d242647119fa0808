"""GPU parity of the sphere force pass (qumasun_amd/csrc/qg_sphere.hip) against the FP64 oracle on
grids whose last point group overlaps its neighbour, with crowded images, several halo vectors per
thread, separate band runs, and one and two bands per workgroup.

Tolerances (relative 2-norm), as for every force form: FP64 <= 1e-10, FP32 <= 2e-5."""
import numpy as np
import pytest

import qumasun_amd as Q
from test_gpu_sphere import GAUSS, TABLE

pytestmark = pytest.mark.gpu

CASES = {
    "ragged": ((13, 9, 11), 0.42, 5, GAUSS, 4),
    "crowded": ((24, 20, 16), 0.3, 40, GAUSS, 3),
    "tables_ragged": ((21, 25, 10), 0.33, 6, TABLE, 5),
    "wide_rows": ((134, 10, 9), 0.3, 6, GAUSS, 3),
    "two_bands": ((40, 44, 9), 0.3, 8, GAUSS, 131),
}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_forces_against_oracle(gpu, oracle, name, prec):
    import torch
    n, h0, nat, projs, nb = CASES[name]
    print(f"sphere forces {name} {prec}", flush=True)
    h = (h0, 1.05 * h0, 0.95 * h0)
    rng = np.random.default_rng(9)
    pos = rng.uniform(0, 1, (nat, 3)) * np.array([n[d] * h[d] for d in range(3)])
    species = (np.arange(nat) % len(projs)).astype(np.int32)
    ng = n[0] * n[1] * n[2]
    psi = rng.standard_normal((nb, ng)) * 0.05
    occ = rng.uniform(0.1, 2.0, nb)
    occ[1] = 0.0
    onl = oracle.OracleNL(n, h, pos, species, projs)
    e_ref, f_ref = oracle.nonlocal_energy_force(n, h, onl, psi, occ, species, projs)
    integ = Q.PseudoPotIntegrator(Q.Grid(*n, *h), projs)
    integ.UpdatePosition(pos, species)
    x = torch.from_numpy(psi).to(gpu).to(torch.float64 if prec == "f64" else torch.float32)
    e, f = integ.EnergyForceNonlocal(x, occ)
    tol = 1e-10 if prec == "f64" else 2e-5
    assert abs(e - e_ref) <= tol * abs(e_ref), (e, e_ref)
    assert np.linalg.norm(f - f_ref) <= tol * np.linalg.norm(f_ref)
    e2, f2 = integ.EnergyForceNonlocal(x, occ)
    assert e2 == e and np.array_equal(f, f2)     # the same sums in the same order
