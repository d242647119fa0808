"""GPU test of H psi, forces and k points where the entry lists of the sphere passes may not be built
(QG_SPHERE_KB, the bytes one projector set's lists may take): what does not fit is served by the row and
table kernels, with the oracle's results.

Tolerances (relative 2-norm over the block), as for every form: FP64 <= 1e-12, FP32 <= 2e-6; forces 1e-10."""
import ctypes

import numpy as np
import pytest

import qumasun_amd as Q
from qumasun_amd import _native as N
from test_gpu_kernel_families import Cell, TOL, _dtype, _kernels
from test_gpu_sphere import GAUSS, TABLE

pytestmark = pytest.mark.gpu


def _family(names):
    apply = next(f for f in ("sphere_hpsi", "rows_hpsi", "fused_hpsi") if any(f in n for n in names))
    project = next(f for f in ("sphere_project", "rows_project", "::project_kernel") if any(f in n for n in names))
    return project, apply


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("grid", ["rows", "tables"])
def test_hpsi_within_the_budget(gpu, oracle, monkeypatch, grid, prec):
    import torch
    print(f"list budget {grid} {prec}", flush=True)
    seen = set()
    for kb in [0, *(int(100 * 1.5 ** i) for i in range(20)), 1 << 20]:
        monkeypatch.setenv("QG_SPHERE_KB", str(kb))
        c = Cell(oracle, (32, 21, 19), GAUSS, 5) if grid == "rows" else Cell(oracle, (33, 21, 19), TABLE[:1], 5)
        x = torch.from_numpy(c.X).to(gpu).to(_dtype(prec))
        out = torch.full_like(x, float("nan"))
        seen.add(_family(_kernels(lambda: c.H.apply(x, out))))
        c.check(out, prec)
        if grid == "rows":      # prepared by the update of the nuclei, whichever kernels serve
            out.fill_(float("nan"))
            N.check(Q.lib().qg_hamiltonian_apply_noalloc(c.H._h, N.QG_F64 if prec == "f64" else N.QG_F32, len(c.X),
                                                         ctypes.c_void_p(x.data_ptr()), c.g.size,
                                                         ctypes.c_void_p(out.data_ptr()), c.g.size, None))
            torch.cuda.synchronize()
            c.check(out, prec)
    plain = ("rows_project", "rows_hpsi") if grid == "rows" else ("::project_kernel", "fused_hpsi")
    # nothing fits, the apply's lists alone, all
    assert seen == {plain, (plain[0], "sphere_hpsi"), ("sphere_project", "sphere_hpsi")}


@pytest.mark.parametrize("kb", [0, 1 << 20])
def test_kpoint_and_forces_within_the_budget(gpu, oracle, monkeypatch, kb):
    import torch
    print(f"list budget, k point and forces {kb}", flush=True)
    monkeypatch.setenv("QG_SPHERE_KB", str(kb))
    c = Cell(oracle, (33, 21, 19), GAUSS, 4)
    onl = oracle.OracleNL(c.n, c.h, c.pos, np.zeros(len(c.pos), np.int32), c.projs)
    k = (0.4, -0.25, 0.3)
    U = c.X + 1j * c.rng.standard_normal(c.X.shape)
    Hk = Q.KpointHamiltonian(c.H, k)
    u = torch.from_numpy(U).to(gpu)
    out = torch.empty_like(u)
    names = _kernels(lambda: Hk.apply(u, out))
    assert any("sphere_kpoint_kernel" in n for n in names) == (kb > 0), names
    ref = oracle.kpoint_hamiltonian(c.n, c.h, c.V, onl, k, U)
    assert np.linalg.norm(out.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)
    occ = np.full(len(c.X), 2.0)
    e_ref, f_ref = oracle.nonlocal_energy_force(c.n, c.h, onl, c.X, occ, np.zeros(len(c.pos), np.int32), c.projs)
    e, f = c.integ.EnergyForceNonlocal(torch.from_numpy(c.X).to(gpu), occ)
    assert abs(e - e_ref) <= 1e-10 * abs(e_ref) and np.linalg.norm(f - f_ref) <= 1e-10 * np.linalg.norm(f_ref)
