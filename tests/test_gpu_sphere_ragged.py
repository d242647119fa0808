"""Rows that are no whole number of point groups (qumasun_amd/csrc/qg_sphere.hip): the last group of a row
overlaps its neighbour and both store the shared points, so both must store the same bits.

A cell and its states moved by whole groups along x give H psi moved by as much, bit for bit, at every
point of the sphere: spacing 1/2 makes the move exact, and one non-zero value per band, at the first point
of a group in both places, makes the projections the same sum.  After the move the sphere lies over the
end of the rows; 17 points put some of the pairs of groups into different wavefronts.  (In 64 bits the
displacements of such a cell are exact in any form; 32 bits round them.)"""
import numpy as np
import pytest

import qumasun_amd as Q

pytestmark = pytest.mark.gpu

PROJ = [[Q.gaussian_projector(0, 1.0, 0.6, 1.75), Q.gaussian_projector(1, -0.7, 0.5, 1.75)]]
N, H0, MOVE = (17, 24, 9), 0.5, 8


def _pair(rng, complex_bands):
    """(V, nucleus, states) of the two places; the sphere does not wrap in x."""
    ng = N[0] * N[1] * N[2]
    # of 40 binary places, so that the move rounds nothing
    centre = np.rint(np.array([5 + rng.uniform(0.2, 0.4), rng.uniform(0, N[1]), rng.uniform(0, N[2])]) * 2.0 ** 40) / 2.0 ** 40
    V = rng.uniform(-1, 1, N[::-1])
    nb = 12
    X = np.zeros((nb, *N[::-1]), complex if complex_bands else float)
    for b in range(nb):
        j = int(np.rint(centre[1])) + b % 5 - 2
        k = int(np.rint(centre[2])) + b // 5 - 1
        X[b, k % N[2], j % N[1], 4] = rng.uniform(0.5, 1.0) * (np.exp(2j * b) if complex_bands else 1.0)
    out = []
    for m in (0, MOVE):
        pos = (centre + [m, 0, 0]) * H0
        out.append((np.roll(V, m, 2).reshape(-1), pos[None], np.roll(X, m, 3).reshape(nb, ng)))
    return out


@pytest.mark.parametrize("kind", ["f64", "f32", "c128", "c64"])
def test_moved_by_whole_groups(gpu, kind):
    import torch
    print(f"ragged rows {kind}", flush=True)
    dt = dict(f64=torch.float64, f32=torch.float32, c128=torch.complex128, c64=torch.complex64)[kind]
    rng = np.random.default_rng(77)
    for trial in range(8):
        res = []
        for V, pos, X in _pair(rng, kind[0] == "c"):
            g = Q.Grid(*N, H0, H0, H0)
            integ = Q.PseudoPotIntegrator(g, PROJ)
            integ.UpdatePosition(pos)
            H = Q.Hamiltonian(g, V, integ)
            if kind[0] == "c":
                H = Q.KpointHamiltonian(H, (0.0, 0.25, 0.3))
            x = torch.from_numpy(X).to(gpu).to(dt)
            out = torch.empty_like(x)
            H.apply(x, out)
            torch.cuda.synchronize()
            res.append(out.cpu().numpy().reshape(len(X), *N[::-1]))
        a, b = res[0][..., 2:9], res[1][..., 2 + MOVE:9 + MOVE]
        off = int((a != b).sum())
        assert off == 0, (trial, off)
        assert float(np.abs(a).max()) > 0
