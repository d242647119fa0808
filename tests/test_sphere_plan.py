"""Host check of the sphere passes' size rules (qumasun_amd/csrc/qg_sphere_plan.hpp).

Chunks of the allocation-free application: for every band count, each chunk (the shorter last one too)
fits the fixed scratch, the chunks cover the bands, and the slabs of a chunk cover the grid.  Cells:
(tile columns, most images of one, channels, coefficients, bands per workgroup, planes) of 216 atoms on
120^3 in FP32 and FP64, 512 atoms on 128^3, 1000 atoms on 120^3 in FP64, and one band that fills the
scratch by itself."""
import os
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++") or shutil.which("c++")
CAPACITY = 8 << 20


@pytest.fixture(scope="module")
def plan():
    if not CXX:
        pytest.skip("no host compiler")
    d = tempfile.mkdtemp()
    exe = os.path.join(d, "sphere_plan")
    r = subprocess.run([CXX, "-O1", "-std=c++17", os.path.join(ROOT, "tests", "harness", "sphere_plan.cpp"), "-o", exe],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
    yield lambda *a: subprocess.run([exe, *map(str, a)], stdout=subprocess.PIPE, text=True, timeout=60,
                                    check=True).stdout.split("\n")[:-1]
    shutil.rmtree(d, ignore_errors=True)


CELLS = [(15, 113, 4, 864, 4, 120), (15, 113, 4, 864, 2, 120), (16, 250, 4, 2048, 4, 128), (15, 520, 4, 4000, 2, 120),
         (40, 1000, 8, 8000, 1, 64), (2, 20, 4, 32, 4, 24)]


@pytest.mark.parametrize("cell", CELLS)
def test_every_chunk_fits(plan, cell):
    nz = cell[-1]
    for nbands in [*range(1, 330, 7), 121, 137, 241, 313, 512, 625, 626, 627, 729, 1089]:
        lines = plan("chunks", nbands, *cell, CAPACITY)
        rows = [list(map(int, s.split())) for s in lines[1:]]
        assert sum(r[0] for r in rows) == nbands
        for bands, slabs, planes, doubles in rows:
            assert 1 <= bands <= int(lines[0]) and doubles <= CAPACITY
            assert slabs * planes >= nz > (slabs - 1) * planes and planes % 8 == 0


def test_band_that_does_not_fit(plan):
    assert plan("chunks", 3, 1000, 1000, 8, 8, 4, 64, CAPACITY) == ["1"] + ["1 1 64 8000008"] * 3
    assert plan("chunks", 3, 1100, 1000, 8, 8, 4, 64, CAPACITY) == ["0"]
