"""Grid points closer to a nucleus than the first point of its radial table, which r_min leaves to the
table (r_min below exp(xi_min), or zero with a nucleus on a grid point): the first value holds there, so the
projections and H psi are those of r_min = exp(xi_min), to the bit."""
import numpy as np
import pytest

import qumasun_amd as Q

pytestmark = pytest.mark.gpu


def _projectors(r_min):
    xi = np.log(0.3) + 0.2 * np.arange(14)
    r = np.exp(xi)
    return [[Q.table_projector(l, e, 2.0, xi[0], 0.2, np.exp(-r * r), r_min=r_min) for l, e in ((0, 1.0), (1, -0.5))]]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("r_min", [0.0, 0.05])
def test_points_below_the_table(gpu, prec, r_min):
    import torch
    print(f"below the radial table {prec} {r_min}", flush=True)
    n, h = (21, 20, 18), 0.4
    rng = np.random.default_rng(4)
    # 0.1 and 0.2 from a grid point, on one (only r_min = 0 looks beyond r_min there)
    pos = np.array([[4.1, 3.0, 2.0], [6.0, 5.0, 4.2], [2.0, 6.0, 5.2]]) * 1.0
    pos = np.rint(pos / h) * h + np.array([[0.1, 0, 0], [0, 0.2, 0], [0, 0, 0]])
    g = Q.Grid(*n, h, h, h)
    V = rng.uniform(-1, 1, g.size)
    x = torch.from_numpy(rng.standard_normal((4, g.size))).to(gpu).to(torch.float64 if prec == "f64" else torch.float32)
    res = []
    for rm in (r_min, float(np.exp(np.log(0.3)))):
        integ = Q.PseudoPotIntegrator(g, _projectors(rm))
        integ.UpdatePosition(pos)
        out = torch.empty_like(x)
        Q.Hamiltonian(g, V, integ).apply(x, out)
        res.append((integ.InnerNonlocalPsi(x).cpu().numpy(), out.cpu().numpy()))
    assert np.isfinite(res[0][0]).all() and np.abs(res[0][0]).min() > 0
    for a, b in zip(*res):
        assert np.array_equal(a, b)
