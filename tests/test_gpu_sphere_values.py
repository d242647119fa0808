"""Infinities and NaN at grid points outside every projector sphere do not reach the projections, the
forces or H psi at the spheres' points (qumasun_amd/csrc/qg_sphere.hip works on groups of points and
lists of planes, in which the points outside a sphere have projector value zero).

Results equal those of the same states without the bad values: relative 2-norm FP64 <= 1e-12,
FP32 <= 2e-6 (forces 1e-10; those of FP32 states 2e-5), as against the oracle elsewhere; the other bands
of the block are as clean as before."""
import numpy as np
import pytest

import qumasun_amd as Q
from test_gpu_sphere import GAUSS, TABLE

pytestmark = pytest.mark.gpu

# grid, spacing, atoms, projectors: whole and ragged rows, tables with two cutoffs, slabs and tiles cut short
CASES = {"whole": ((32, 20, 24), 0.42, 2, GAUSS), "ragged": ((33, 21, 29), 0.42, 2, TABLE),
         "narrow": ((40, 9, 16), 0.6, 2, GAUSS)}
BAD = {"inf": np.inf, "nan": np.nan}


def _cell(name):
    n, h0, nat, projs = CASES[name]
    h = (h0, 1.05 * h0, 0.95 * h0)
    rng = np.random.default_rng(15)
    pos = rng.uniform(0, 1, (nat, 3)) * np.array([n[d] * h[d] for d in range(3)])
    species = (np.arange(nat) % len(projs)).astype(np.int32)
    inside = np.zeros((n[2], n[1], n[0]), bool)
    ax = [np.arange(n[d]) * h[d] for d in range(3)]
    for R, s in zip(pos, species):
        cut = max(p["cutoff"] for p in projs[s])
        d = [((ax[k] - R[k] + n[k] * h[k] / 2) % (n[k] * h[k]) - n[k] * h[k] / 2) ** 2 for k in range(3)]
        inside |= d[0][None, None, :] + d[1][None, :, None] + d[2][:, None, None] <= cut * cut
    reach = inside.copy()       # the points that a stencil at the spheres' points reads
    for axis in range(3):
        for m in range(-4, 5):
            reach |= np.roll(inside, m, axis)
    assert (~reach).any()
    g = Q.Grid(*n, *h)
    integ = Q.PseudoPotIntegrator(g, projs)
    integ.UpdatePosition(pos, species)
    return g, integ, rng.uniform(-2, 1, g.size), inside.reshape(-1), reach.reshape(-1), rng


def _close(a, b, tol):
    assert np.isfinite(a).all()
    assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)


@pytest.mark.parametrize("bad", sorted(BAD))
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_real_bands(gpu, name, prec, bad):
    import torch
    print(f"values outside spheres {name} {prec} {bad}", flush=True)
    g, integ, V, inside, reach, rng = _cell(name)
    H = Q.Hamiltonian(g, V, integ)
    dt = torch.float64 if prec == "f64" else torch.float32
    tol = 1e-12 if prec == "f64" else 2e-6
    x = torch.from_numpy(rng.standard_normal((6, g.size)) * 0.1).to(gpu).to(dt)
    clean = x.clone()
    out, ref = torch.empty_like(x), torch.empty_like(x)
    H.apply(clean, ref)
    cref = integ.InnerNonlocalPsi(clean).cpu().numpy()
    eref, fref = integ.EnergyForceNonlocal(clean, np.full(6, 2.0))
    x[4, torch.from_numpy(~inside).to(gpu)] = BAD[bad]
    c = integ.InnerNonlocalPsi(x).cpu().numpy()
    _close(c[4], cref[4], tol)
    _close(c, cref, tol)
    x.copy_(clean)
    x[4, torch.from_numpy(~reach).to(gpu)] = BAD[bad]
    H.apply(x, out)
    torch.cuda.synchronize()
    o, r = out.double().cpu().numpy(), ref.double().cpu().numpy()
    _close(o[4, inside], r[4, inside], tol)
    _close(np.delete(o, 4, 0), np.delete(r, 4, 0), tol)
    e, f = integ.EnergyForceNonlocal(x, np.full(6, 2.0))
    _close(np.array([e]), np.array([eref]), 1e-10 if prec == "f64" else 2e-5)
    _close(f, fref, 1e-10 if prec == "f64" else 2e-5)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_complex_bands(gpu, name, prec):
    import torch
    print(f"values outside spheres, k point {name} {prec}", flush=True)
    g, integ, V, inside, reach, rng = _cell(name)
    Hk = Q.KpointHamiltonian(Q.Hamiltonian(g, V, integ), (0.4, -0.25, 0.3))
    x = rng.standard_normal((3, g.size)) + 1j * rng.standard_normal((3, g.size))
    x = torch.from_numpy(x).to(gpu).to(torch.complex128 if prec == "f64" else torch.complex64)
    out, ref = torch.empty_like(x), torch.empty_like(x)
    Hk.apply(x, ref)
    x[1, torch.from_numpy(~reach).to(gpu)] = complex(np.nan, np.inf)
    Hk.apply(x, out)
    torch.cuda.synchronize()
    o, r = out.cpu().numpy(), ref.cpu().numpy()
    tol = 1e-12 if prec == "f64" else 2e-6
    _close(o[1, inside], r[1, inside], tol)
    _close(np.delete(o, 1, 0), np.delete(r, 1, 0), tol)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_infinity_inside(gpu, prec):
    """An infinity at a sphere's point gives infinite (signed) coefficients of that atom alone."""
    import torch
    g, integ, V, inside, reach, rng = _cell("whole")
    x = torch.from_numpy(rng.standard_normal((2, g.size))).to(gpu).to(torch.float64 if prec == "f64" else torch.float32)
    cref = integ.InnerNonlocalPsi(x).cpu().numpy()
    unit = torch.zeros_like(x)
    at = int(np.flatnonzero(inside)[57])
    unit[0, at] = 1.0
    beta = integ.InnerNonlocalPsi(unit).cpu().numpy()[0]    # dV beta_j at the point
    x[0, at] = np.inf
    c = integ.InnerNonlocalPsi(x).cpu().numpy()
    assert (beta != 0).any() and (beta == 0).any()
    assert np.array_equal(c[0][beta != 0], np.copysign(np.inf, beta[beta != 0]))
    tol = 1e-12 if prec == "f64" else 2e-6
    _close(c[0][beta == 0], cref[0][beta == 0], tol)
    _close(c[1], cref[1], tol)
