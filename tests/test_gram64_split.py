"""Host check of the FP64 Gram kernel's split and of the rule that chooses between it and the library's
product (qumasun_amd/csrc/qg_gram64_split.hpp), at products that were timed both ways (us, kernel : library)
and of which one side is at least a tenth faster."""
import os
import shutil
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++") or shutil.which("c++")

# points, M, N, kernel us, library us
TIMED = [(13824, 8, 8, 25, 138), (13824, 128, 128, 100, 139), (13824, 240, 240, 103, 142), (13824, 512, 512, 189, 151),
         (64000, 16, 48, 32, 89), (64000, 144, 432, 204, 277), (64000, 192, 192, 127, 150), (64000, 256, 512, 388, 282),
         (64000, 352, 704, 727, 529), (64000, 528, 1584, 2844, 2085), (512000, 8, 24, 78, 273), (512000, 64, 64, 163, 336),
         (512000, 96, 192, 438, 551), (512000, 128, 256, 670, 595), (512000, 144, 144, 490, 757), (512000, 136, 408, 1316, 1484),
         (512000, 192, 576, 2560, 1966), (512000, 168, 504, 2393, 1582), (512000, 256, 512, 3038, 2195),
         (512000, 512, 512, 5691, 4333), (512000, 528, 1584, 21624, 15309), (1728000, 32, 96, 407, 4396),
         (1728000, 144, 432, 4547, 9012), (1728000, 192, 192, 2658, 4447), (1728000, 288, 576, 10572, 14545),
         (1728000, 240, 720, 12407, 9683), (1728000, 432, 864, 24838, 22317), (1728000, 512, 512, 18457, 14966),
         (1728000, 528, 1056, 42234, 36039), (1728000, 528, 1584, 72395, 54790)]


@pytest.fixture(scope="module")
def split():
    if not CXX:
        pytest.skip("no host compiler")
    d = tempfile.mkdtemp()
    exe = os.path.join(d, "gram64_split")
    r = subprocess.run([CXX, "-O1", "-std=c++17", os.path.join(ROOT, "tests", "harness", "gram64_split.cpp"), "-o", exe],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]

    def run(sizes):
        lines = "".join(f"{k} {m} {n} {max(1, min(64, k // 2048))}\n" for k, m, n in sizes)
        out = subprocess.run([exe], input=lines, stdout=subprocess.PIPE, text=True, timeout=60, check=True).stdout
        return [tuple(map(int, s.split())) for s in out.splitlines()]

    yield run
    shutil.rmtree(d, ignore_errors=True)


def test_the_faster_side_is_chosen(split):
    for (k, m, n, own, lib), r in zip(TIMED, split([t[:3] for t in TIMED])):
        assert max(own, lib) >= 1.1 * min(own, lib)
        assert r[0] == int(own < lib), (k, m, n, own, lib)


def test_split_covers_the_product(split):
    sizes = [(k, m, n) for k in (2, 510, 4098, 64000, 1728000) for m in (1, 16, 160, 161, 528) for n in (1, 192, 193, 1584, 9000)]
    for (k, m, n), (_, nch, per, mb, nb, bm, bn) in zip(sizes, split(sizes)):
        assert nch * per >= k > (nch - 1) * per and per % 16 == 0
        assert mb * bm * 16 >= m and nb * bn * 16 >= n and bm <= 10 and bn <= 12
        blocks = mb * nb
        # whole rounds of one workgroup per CU are not exceeded
        assert nch == 1 or nch * blocks <= (256 if blocks <= 32 else 1024)
