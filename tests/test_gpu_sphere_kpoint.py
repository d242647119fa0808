"""GPU parity of the sphere passes of the k-point Hamiltonian (qumasun_amd/csrc/qg_sphere.hip) against
the FP64 oracle where their tiles, lists and layouts have edges.

Tolerances (relative 2-norm over the block), as for every k-point apply: complex128 <= 1e-12,
complex64 <= 2e-6.
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
    "ragged_rows": ((13, 9, 11), 0.42, 5, GAUSS, 3),      # Nx odd, sphere wider than the cell
    "smallest_rows": ((8, 8, 8), 0.5, 2, GAUSS, 2),
    "crowded": ((24, 20, 16), 0.3, 40, GAUSS, 2),
    "tables_two_species": ((22, 17, 19), 0.31, 6, TABLE, 3),
    "tables_ragged": ((21, 25, 10), 0.33, 6, TABLE, 2),
    "wide_rows": ((134, 10, 9), 0.3, 6, GAUSS, 1),        # complex128: two halo vectors per thread
    "half_tile": ((76, 29, 13), 0.3, 8, GAUSS, 5),        # complex128: the low tile, last one partial
}


@pytest.mark.parametrize("prec", ["z128", "c64"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_kpoint_against_oracle(gpu, oracle, name, prec):
    import torch
    n, h0, nat, projs, nb = CASES[name]
    print(f"sphere kpoint {name} {prec}", flush=True)
    h, k = (h0, 1.05 * h0, 0.95 * h0), (0.4, -0.25, 0.3)
    rng = np.random.default_rng(9)
    box = np.array([n[d] * h[d] for d in range(3)])
    species = (np.arange(nat) % len(projs)).astype(np.int32)
    ng = n[0] * n[1] * n[2]
    V = rng.uniform(-2, 1, ng)
    U = rng.standard_normal((nb, ng)) + 1j * rng.standard_normal((nb, ng))
    g = Q.Grid(*n, *h)
    integ = Q.PseudoPotIntegrator(g, projs)
    integ.UpdatePosition(rng.uniform(0, 1, (nat, 3)) * box, species)
    H = Q.Hamiltonian(g, V, integ)
    Hk = Q.KpointHamiltonian(H, k)
    u = torch.from_numpy(U).to(gpu).to(torch.complex128 if prec == "z128" else torch.complex64)
    out = torch.empty_like(u)
    for _ in range(2):      # the second pass with the nuclei moved under the same handle
        pos = rng.uniform(0, 1, (nat, 3)) * box
        integ.UpdatePosition(pos, species)
        out.fill_(float("nan"))
        Hk.apply(u, out)
        torch.cuda.synchronize()
        ref = oracle.kpoint_hamiltonian(n, h, V, oracle.OracleNL(n, h, pos, species, projs), k, U)
        err = float(np.linalg.norm(out.cpu().numpy() - ref) / np.linalg.norm(ref))
        assert err <= (1e-12 if prec == "z128" else 2e-6), err
