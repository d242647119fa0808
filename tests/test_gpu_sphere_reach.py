"""Spheres that reach more than a thousand grid points (a fine spacing along one axis, a cell shorter than
the sphere, so that the points of an image lie far from its centre): beyond what a list entry can address,
the other kernels serve.  Projections and the projector term of H psi against the oracle.

Tolerances: projections FP64 1e-12, FP32 2e-6; the projector term (H psi minus its local part, which is
1e6 times as large) 1e-6 in FP64."""
import numpy as np
import pytest

import qumasun_amd as Q

pytestmark = pytest.mark.gpu

PROJ = [[Q.gaussian_projector(0, 1.0, 1.1, 2.7), Q.gaussian_projector(1, -0.5, 1.0, 2.7)]]


@pytest.mark.parametrize("axis", [0, 1])
def test_far_points(gpu, oracle, axis):
    import torch
    n, h = [10, 10, 10], [0.5, 0.55, 0.5]
    n[axis], h[axis] = (120, 800)[axis], 0.0025
    print(f"far points {n}", flush=True)
    rng = np.random.default_rng(6)
    g = Q.Grid(*n, *h)
    pos = rng.uniform(0, 1, (1, 3)) * np.array(n) * np.array(h)
    integ = Q.PseudoPotIntegrator(g, PROJ)
    integ.UpdatePosition(pos)
    V = rng.uniform(-1, 1, g.size)
    H = Q.Hamiltonian(g, V, integ)
    onl = oracle.OracleNL(tuple(n), tuple(h), pos, np.zeros(1, np.int32), PROJ)
    X = rng.standard_normal((3, g.size)) + 2.0
    cref = np.stack([onl.project(x.copy()) for x in X])
    for dt, tol in ((torch.float64, 1e-12), (torch.float32, 2e-6)):
        c = integ.InnerNonlocalPsi(torch.from_numpy(X).to(gpu).to(dt)).cpu().numpy()
        assert np.linalg.norm(c - cref) <= tol * np.linalg.norm(cref), (dt, c, cref)
    x = torch.from_numpy(X).to(gpu)
    out = torch.empty_like(x)
    H.apply(x, out)
    loc = oracle.hamiltonian_block(tuple(n), tuple(h), V, None, X)
    ref = oracle.hamiltonian_block(tuple(n), tuple(h), V, onl, X) - loc
    got = out.cpu().numpy() - loc
    assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)
