"""Host check of the sphere passes' size rules (qumasun_amd/csrc/qg_sphere_plan.hpp).

Chunks of the allocation-free application: for every band count, each chunk (the shorter last one too)
fits the fixed scratch, the chunks cover the bands, and the slabs of a chunk cover the grid.  Cells:
(tile columns, most images of one, channels, coefficients, bands per workgroup, planes) of 216 atoms on
120^3 in FP32 and FP64, 512 atoms on 128^3, 1000 atoms on 120^3 in FP64, and one band that fills the
scratch by itself.

Entry lists: their parts do not overlap, every load that the kernels issue ahead lies inside the
allocation (also where an offset past a list's last entry is not checked), and what is built fits."""
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


@pytest.mark.parametrize("nv", [2, 4])
@pytest.mark.parametrize("trips,slots", [(1, 0), (1, 1), (1, 2), (7, 3), (5000, 900), (1 << 20, 0)])
def test_list_layout(plan, nv, trips, slots):
    vals, slot_vals, words, slot_words, size, _ = map(int, plan("lists", nv, trips, slots, 0)[0].split())
    ahead = 4                       # entries a wavefront loads before it looks at their number
    assert vals == 0 and slot_vals >= vals + 1024 * nv * trips
    assert words >= slot_vals + 1024 * nv * 8 * slots and slot_words >= words + 256 * trips
    assert size >= slot_words + 256 * slots
    # from the end of the last plane's entries; a slot without points is addressed from the lists' start
    assert vals + 1024 * nv * (trips + ahead) <= size and words + 256 * (trips + ahead) <= size
    assert slot_vals + 1024 * nv * 8 * slots + 1024 * nv <= size and slot_words + 256 * (slots + ahead) <= size


def test_lists_within_their_room(plan):
    def fit(room):
        return int(plan("lists", 2, 1000, 400, room)[0].split()[5])

    both, trips = (int(plan("lists", 2, 1000, n, 0)[0].split()[4]) for n in (400, 0))
    assert trips < both
    assert [fit(r) for r in (0, trips - 1, trips, both - 1, both, 2 ** 63)] == [0, 0, 1, 1, 2, 2]
