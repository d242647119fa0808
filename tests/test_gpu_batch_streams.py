"""GPU parity of a batch whose cells run on two streams (qumasun_amd/csrc/qg_hpsi.hip): one handle and
one set of projectors used several times in a batch, odd grids, and one cell alone.

Tolerances (relative 2-norm over the block), as for every H psi form: FP64 <= 1e-12, FP32 <= 2e-6.
"""
import numpy as np
import pytest

import qumasun_amd as Q

pytestmark = pytest.mark.gpu

GAUSS = [[Q.gaussian_projector(0, 1.0, 0.6, 2.0), Q.gaussian_projector(1, -0.5, 0.5, 2.0)]]
GRIDS = [(24, 20, 16), (13, 9, 11), (16, 16, 16)]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("order", [(0,), (0, 0, 0), (1, 2, 0, 3, 0, 2, 1, 3)])
def test_batch_shares(gpu, oracle, order, prec):
    import torch
    print(f"batch shares {order} {prec}", flush=True)
    rng = np.random.default_rng(12)
    h = (0.32, 0.3, 0.34)
    cells = []
    for n in GRIDS:
        pos = rng.uniform(0, 1, (5, 3)) * np.array([n[d] * h[d] for d in range(3)])
        g = Q.Grid(*n, *h)
        integ = Q.PseudoPotIntegrator(g, GAUSS)
        integ.UpdatePosition(pos)
        V = rng.uniform(-2, 1, g.size)
        cells.append((n, V, oracle.OracleNL(n, h, pos, np.zeros(5, np.int32), GAUSS), integ, Q.Hamiltonian(g, V, integ)))
    n, V, onl, integ, H = cells[0]      # a second potential over the first cell's projectors
    V = rng.uniform(-2, 1, V.size)
    cells.append((n, V, onl, integ, Q.Hamiltonian(Q.Grid(*n, *h), V, integ)))
    dt = torch.float64 if prec == "f64" else torch.float32
    X = [rng.standard_normal((3 + i, cells[c][1].size)) for i, c in enumerate(order)]
    xs = [torch.from_numpy(x).to(gpu).to(dt) for x in X]
    outs = [torch.full_like(x, float("nan")) for x in xs]
    for _ in range(3):
        Q.batch_apply([cells[c][4] for c in order], xs, outs)
    torch.cuda.synchronize()
    for c, x, o in zip(order, X, outs):
        n, V, onl = cells[c][:3]
        ref = oracle.hamiltonian_block(n, h, V, onl, x)
        err = float(np.linalg.norm(o.double().cpu().numpy() - ref) / np.linalg.norm(ref))
        assert err <= (1e-12 if prec == "f64" else 2e-6), (c, err)
