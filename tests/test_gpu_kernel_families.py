"""Which kernels an H psi runs: a plan that asks for the row or table kernels gets them, on grids that the
sphere passes serve too, and each family gives the oracle's H psi.  Families are told apart by the names of
the kernels launched.

Tolerances (relative 2-norm over the block), as for every H psi form: FP64 <= 1e-12, FP32 <= 2e-6."""
import ctypes

import numpy as np
import pytest

import qumasun_amd as Q
from qumasun_amd import _native as N
from test_gpu_sphere import GAUSS

pytestmark = pytest.mark.gpu

# p before s with two cutoffs; three s channels (more than the sphere passes hold); the channels of one l
# share their cutoff, as in the reference
MIXED = [[Q.gaussian_projector(1, 0.8, 0.5, 2.0), Q.gaussian_projector(0, -0.3, 0.7, 1.6)]]
THREE = [[Q.gaussian_projector(0, 1.0, 0.6, 2.0), Q.gaussian_projector(0, 0.4, 0.5, 2.0),
          Q.gaussian_projector(0, -0.3, 0.7, 2.0), Q.gaussian_projector(1, -0.5, 0.6, 1.6)]]
TOL = {"f64": 1e-12, "f32": 2e-6}


def _kernels(f):
    """Names of the engine's kernels that f launches."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        f()
        torch.cuda.synchronize()
    return {e.name for e in p.events() if "qg::" in e.name}


def _any(names, part):
    return any(part in n for n in names)


class Cell:
    def __init__(self, oracle, n, projs, nb, seed=5, nat=7):
        self.nat, self.n, self.h, self.projs, self.oracle = nat, n, (0.3, 0.32, 0.28), projs, oracle
        self.rng = np.random.default_rng(seed)
        self.g = Q.Grid(*n, *self.h)
        self.integ = Q.PseudoPotIntegrator(self.g, projs)
        self.V = self.rng.uniform(-2, 1, self.g.size)
        self.X = self.rng.standard_normal((nb, self.g.size))
        self.move()
        self.H = Q.Hamiltonian(self.g, self.V, self.integ)

    def move(self):
        self.pos = self.rng.uniform(0, 1, (self.nat, 3)) * np.array([self.n[d] * self.h[d] for d in range(3)])
        self.integ.UpdatePosition(self.pos)

    def check(self, out, prec):
        onl = self.oracle.OracleNL(self.n, self.h, self.pos, np.zeros(len(self.pos), np.int32), self.projs)
        ref = self.oracle.hamiltonian_block(self.n, self.h, self.V, onl, self.X)
        err = np.linalg.norm(out.double().cpu().numpy() - ref) / np.linalg.norm(ref)
        assert err <= TOL[prec], err


def _dtype(prec):
    import torch
    return torch.float64 if prec == "f64" else torch.float32


ROWS = [dict(), dict(rows_ty=5, rows_tz=3), dict(rows_bands=1, rows_tzp=5, rows_nbp=4), dict(rows_bands=2), dict(rows_bands=4)]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("projs", ["one_s_one_p", "mixed"])
def test_row_plan_runs_row_kernels(gpu, oracle, prec, projs):
    import torch
    print(f"row plan {prec} {projs}", flush=True)
    c = Cell(oracle, (32, 21, 19), GAUSS if projs == "one_s_one_p" else MIXED, 13)
    x = torch.from_numpy(c.X).to(gpu).to(_dtype(prec))
    out = torch.empty_like(x)
    assert _any(_kernels(lambda: c.H.apply(x, out)), "sphere_hpsi_kernel")
    for shape in ROWS:
        c.H.set_plan(kernels=N.QG_KERNELS_ROWS, **shape)
        out.fill_(float("nan"))
        names = _kernels(lambda: c.H.apply(x, out))
        assert _any(names, "rows_hpsi_kernel") and _any(names, "rows_project_kernel") and not _any(names, "sphere"), names
        c.check(out, prec)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_row_plan_without_allocation(gpu, oracle, prec):
    """The plan's geometry is there without an application before, and again after the nuclei moved."""
    import torch
    print(f"row plan, no allocation {prec}", flush=True)
    c = Cell(oracle, (32, 21, 19), GAUSS, 5)
    c.H.set_plan(kernels=N.QG_KERNELS_ROWS)
    x = torch.from_numpy(c.X).to(gpu).to(_dtype(prec))
    for _ in range(2):
        out = torch.full_like(x, float("nan"))
        free = torch.cuda.mem_get_info()[0]
        names = _kernels(lambda: N.check(Q.lib().qg_hamiltonian_apply_noalloc(
            c.H._h, N.QG_F64 if prec == "f64" else N.QG_F32, len(c.X), ctypes.c_void_p(x.data_ptr()), c.g.size,
            ctypes.c_void_p(out.data_ptr()), c.g.size, None)))
        assert _any(names, "rows_hpsi_kernel") and not _any(names, "sphere"), names
        assert torch.cuda.mem_get_info()[0] == free
        c.check(out, prec)
        c.move()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("case", ["few_planes", "three_s"])
def test_row_kernels_where_the_lists_do_not_serve(gpu, oracle, prec, case):
    import torch
    print(f"row kernels by themselves {case} {prec}", flush=True)
    c = Cell(oracle, (32, 21, 7), MIXED, 6, nat=2) if case == "few_planes" else Cell(oracle, (32, 21, 19), THREE, 6)
    x = torch.from_numpy(c.X).to(gpu).to(_dtype(prec))
    out = torch.full_like(x, float("nan"))
    names = _kernels(lambda: c.H.apply(x, out))
    assert _any(names, "rows_hpsi_kernel") and not _any(names, "sphere"), names
    c.check(out, prec)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_batch_of_table_plans(gpu, oracle, prec):
    """One cell with a table plan puts the whole batch on the persistent table kernels."""
    import torch
    print(f"batch of table plans {prec}", flush=True)
    cells = [Cell(oracle, n, GAUSS, nb, seed=nb) for n, nb in (((24, 20, 16), 5), ((13, 9, 11), 9), ((40, 16, 12), 3))]
    cells[1].H.set_plan(kernels=N.QG_KERNELS_TABLES)
    xs = [torch.from_numpy(c.X).to(gpu).to(_dtype(prec)) for c in cells]
    outs = [torch.full_like(x, float("nan")) for x in xs]
    names = _kernels(lambda: Q.batch_apply([c.H for c in cells], xs, outs))
    assert _any(names, "fused_batch_kernel") and _any(names, "project_batch_kernel") and not _any(names, "sphere"), names
    for c, o in zip(cells, outs):
        c.check(o, prec)
