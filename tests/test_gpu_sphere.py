"""GPU parity of the sphere apply pass (qumasun_amd/csrc/qg_sphere.hip) against the FP64 oracle at
the sizes where its tiles, lists and layouts have edges.

Tolerances (relative 2-norm over the block), as for every H psi form: FP64 <= 1e-12, FP32 <= 2e-6.
"""
import numpy as np
import pytest

import qumasun_amd as Q

pytestmark = pytest.mark.gpu

GAUSS = [[Q.gaussian_projector(0, 1.0, 0.6, 2.4), Q.gaussian_projector(1, -0.5, 0.5, 2.4)]]


def _table(l, e, width, cutoff):
    xi = np.linspace(np.log(1e-4), np.log(12.0), 240)
    r = np.exp(xi)
    return Q.table_projector(l, e, cutoff, xi[0], (xi[-1] - xi[0]) / 239, r ** l * np.exp(-r * r / (2 * width ** 2)))


# p before s, two cutoffs, 2 + 2 channels; a second species with one s channel only
TABLE = [[_table(1, -0.5, 0.5, 2.2), _table(0, 1.0, 0.55, 1.7), _table(1, 0.4, 0.7, 2.2), _table(0, -0.3, 0.8, 1.7)],
         [Q.gaussian_projector(0, 0.7, 0.5, 1.5)]]

# grid, spacing, atoms, projectors, bands
CASES = {
    "ragged_rows": ((13, 9, 11), 0.42, 5, GAUSS, 3),          # Nx odd, sphere wider than the cell
    "smallest_rows": ((8, 8, 8), 0.5, 2, GAUSS, 2),           # the smallest axes the pass takes
    "crowded": ((24, 20, 16), 0.3, 40, GAUSS, 3),             # far more images per point than stay in registers
    "tables_two_species": ((22, 17, 19), 0.31, 6, TABLE, 5),
    "tables_ragged": ((21, 25, 10), 0.33, 6, TABLE, 4),
    "wide_rows": ((134, 10, 9), 0.3, 6, GAUSS, 2),            # FP64: several halo vectors per thread
    "widest_rows": ((1022, 9, 8), 0.3, 8, GAUSS, 1),          # one row per tile in FP64
    "tile_remainder": ((40, 29, 13), 0.3, 8, GAUSS, 65),      # partial last tile, slab and band pair
}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_hpsi_against_oracle(gpu, oracle, name, prec):
    import torch
    n, h0, nat, projs, nb = CASES[name]
    print(f"sphere hpsi {name} {prec}", flush=True)
    h = (h0, 1.05 * h0, 0.95 * h0)
    rng = np.random.default_rng(7)
    pos = rng.uniform(0, 1, (nat, 3)) * np.array([n[d] * h[d] for d in range(3)])
    pos[0] = [3 * h[0], 2 * h[1], 5 * h[2]]     # a nucleus on a grid point
    species = (np.arange(nat) % len(projs)).astype(np.int32)
    ng = n[0] * n[1] * n[2]
    V = rng.uniform(-2, 1, ng)
    X = rng.standard_normal((nb, ng))
    onl = oracle.OracleNL(n, h, pos, species, projs)
    ref = oracle.hamiltonian_block(n, h, V, onl, X)
    g = Q.Grid(*n, *h)
    integ = Q.PseudoPotIntegrator(g, projs)
    integ.UpdatePosition(pos, species)
    H = Q.Hamiltonian(g, V, integ)
    x = torch.from_numpy(X).to(gpu).to(torch.float64 if prec == "f64" else torch.float32)
    out = torch.full_like(x, float("nan"))
    H.apply(x, out)
    torch.cuda.synchronize()
    err = float(np.linalg.norm(out.double().cpu().numpy() - ref) / np.linalg.norm(ref))
    assert err <= (1e-12 if prec == "f64" else 2e-6), err


def test_moved_nuclei_and_plans(gpu, oracle):
    """The lists follow qg_nonlocal_update, and every tile height and band count gives one result."""
    import torch
    n, h = (40, 22, 12), (0.3, 0.3, 0.3)
    rng = np.random.default_rng(8)
    ng = n[0] * n[1] * n[2]
    g = Q.Grid(*n, *h)
    integ = Q.PseudoPotIntegrator(g, GAUSS)
    box = np.array([n[d] * h[d] for d in range(3)])
    integ.UpdatePosition(rng.uniform(0, 1, (4, 3)) * box)
    V = rng.uniform(-2, 1, ng)
    H = Q.Hamiltonian(g, V, integ)
    X = rng.standard_normal((5, ng))
    x = torch.from_numpy(X).to(gpu)
    out = torch.empty_like(x)
    H.apply(x, out)
    pos = rng.uniform(0, 1, (7, 3)) * box
    integ.UpdatePosition(pos)
    ref = oracle.hamiltonian_block(n, h, V, oracle.OracleNL(n, h, pos, np.zeros(7, np.int32), GAUSS), X)
    for ty, nb, tz in ((0, 0, 0), (1, 1, 3), (5, 2, 12), (9, 4, 1), (22, 2, 7)):
        H.set_plan(rows_ty=ty, rows_bands=nb, rows_tz=tz)
        out.fill_(float("nan"))
        H.apply(x, out)
        torch.cuda.synchronize()
        err = float(np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref))
        assert err <= 1e-12, (ty, nb, tz, err)
