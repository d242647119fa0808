"""The FP64 block update of the solver (qumasun_amd/csrc/qg_dense64.hip) at the edges of its tiles and
blocks, through two preconditioned iterations: every block that leaves them has been updated several
times, so the returned states are orthonormal and their Rayleigh quotients are the returned values only
if every point and band was.

Tolerance 1e-9 (states of norm 1, energies of order 1-100 Ha), as for the solver's trajectories.
"""
import numpy as np
import pytest

import qumasun_amd as Q
from qumasun_amd import _native as N

pytestmark = pytest.mark.gpu

# grid (points a multiple of the 128-point tile, or not; an odd number: the library's product), bands (the
# smallest and largest of each range the kernel takes, tile remainders, and the sizes beside them)
CASES = [((16, 16, 16), 16), ((10, 9, 7), 17), ((16, 16, 16), 32), ((24, 20, 10), 33), ((10, 9, 7), 50),
         ((10, 9, 7), 76), ((10, 9, 7), 77), ((24, 20, 10), 129), ((24, 20, 10), 144), ((24, 20, 10), 153),
         ((24, 20, 10), 154), ((9, 11, 13), 20)]


@pytest.mark.parametrize("n,nb", CASES)
def test_states_after_updates(gpu, n, nb):
    import torch
    print(f"update64 {n} {nb}", flush=True)
    h = (0.5, 0.45, 0.55)
    rng = np.random.default_rng(nb)
    g = Q.Grid(*n, *h)
    H = Q.Hamiltonian(g, rng.uniform(-1, 1, g.size))
    X = torch.from_numpy(Q.random_states(g.size, nb, g.dvol)).to(gpu)
    P = torch.zeros_like(X)
    e, _ = Q.Eigen_d_multi(H, X, P, 0, precision=N.QG_PREC_F64, max_iter=2, precond=N.QG_PRECOND_KINETIC,
                           precond_shift=1.0)
    HX = torch.empty_like(X)
    H.apply(X, HX)
    torch.cuda.synchronize()
    x, hx = X.cpu().numpy(), HX.cpu().numpy()
    assert np.abs(x @ x.T * g.dvol - np.eye(nb)).max() <= 1e-9
    e = np.asarray(e)
    assert np.abs((x * hx).sum(axis=1) * g.dvol - e).max() <= 1e-9 * max(1.0, np.abs(e).max())
