"""Host check of what the kinetic preconditioner keeps between calls (qumasun_amd/csrc/qg_plan_store.hpp):
a step that throws (no memory for the symbol, a plan that cannot be made) leaves nothing that a later call
takes for made, and nothing unreleased."""
import os
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++") or shutil.which("c++")


def test_plan_store():
    if not CXX:
        pytest.skip("no host compiler")
    d = tempfile.mkdtemp()
    try:
        exe = os.path.join(d, "plan_store")
        r = subprocess.run([CXX, "-O1", "-std=c++17", os.path.join(ROOT, "tests", "harness", "plan_store.cpp"), "-o", exe],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
        assert r.returncode == 0, r.stdout[-2000:]
        r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=60)
        assert r.returncode == 0, r.stdout
    finally:
        shutil.rmtree(d, ignore_errors=True)
