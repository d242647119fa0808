"""The tabulated radial functions read nothing outside their table (qumasun_amd/csrc/qg_radial.hpp, compiled
for the host and the device alike): below the first point, where r_min leaves room for one, the first
value; beyond the last, zero; in between the interpolation, which is exact for a straight line."""
import os
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++")


@pytest.fixture(scope="module")
def radial():
    if not CXX:
        pytest.skip("no host compiler")
    d = tempfile.mkdtemp()
    exe = os.path.join(d, "radial_range")
    r = subprocess.run([CXX, "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                        os.path.join(ROOT, "tests", "harness", "radial_range.cpp"), "-o", exe],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    if r.returncode != 0 and "asan" in r.stdout:
        pytest.skip("no sanitizer runtime")
    assert r.returncode == 0, r.stdout[-2000:]
    env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}

    def run(n, rels):
        r = subprocess.run([exe, str(n), *map(repr, rels)], stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True,
                           timeout=60, env=env)
        assert r.returncode == 0, r.stderr[-1500:]
        return [float(s) for s in r.stdout.split()]

    yield run
    shutil.rmtree(d, ignore_errors=True)


@pytest.mark.parametrize("n", [5, 6, 7, 9])
def test_values_and_range(radial, n):
    inf = float("inf")
    below = [-inf, -1e300, -1e10, -2.5, -1.0, -0.4, -1e-17]
    assert radial(n, below) == [1.0] * len(below)
    beyond = [n - 1, n - 0.5, n + 3, 1e9, 1e300, inf]
    assert radial(n, beyond) == [0.0] * len(beyond)
    inside = [k * (n - 1) / 40 for k in range(40)]
    for rel, got in zip(inside, radial(n, inside)):
        assert abs(got - (1.0 + rel)) <= 1e-13 * (1.0 + rel)
