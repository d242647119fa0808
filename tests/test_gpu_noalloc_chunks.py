"""GPU test of the allocation-free H psi where its band chunks are uneven: 216 atoms, 120^3, FP32, band
counts of which a shorter chunk takes more slabs than a longer one, so that its partials need more of the
fixed scratch.  Every band equals qg_hamiltonian_apply's (relative 2-norm <= 2e-6, as for every FP32 form)."""
import ctypes

import pytest

import qumasun_amd as Q
from qumasun_amd import _native as N

pytestmark = pytest.mark.gpu


def test_uneven_chunks(gpu):
    import torch
    s = Q.diamond_system(3, 40)
    g = Q.Grid(*[s["n"]] * 3, *[s["h"]] * 3)
    integ = Q.PseudoPotIntegrator(g, s["projectors"])
    integ.UpdatePosition(s["positions"])
    H = Q.Hamiltonian(g, s["V"], integ)
    lib = Q.lib()
    x = torch.randn((729, g.size), device=gpu, dtype=torch.float32)
    ref, got = torch.empty_like(x), torch.empty_like(x)
    H.apply(x, ref)
    for nb in (313, 627, 729):
        print(f"noalloc {nb} bands", flush=True)
        got.fill_(float("nan"))
        N.check(lib.qg_hamiltonian_apply_noalloc(H._h, N.QG_F32, nb, ctypes.c_void_p(x.data_ptr()), g.size,
                                                 ctypes.c_void_p(got.data_ptr()), g.size, None))
        torch.cuda.synchronize()
        err = (got[:nb] - ref[:nb]).norm(dim=1) / ref[:nb].norm(dim=1)
        assert float(err.max()) <= 2e-6, (nb, err.max())
        assert bool(got[nb:].isnan().all())
