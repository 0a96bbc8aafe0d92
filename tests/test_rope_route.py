"""CPU: the rule that sends a RoPE call to the vector kernel (sulimo_amd/csrc/rope_route.h,
compiled here), against the sizes its 32-bit thread numbers and its loads allow."""
import os
import shutil
import subprocess

import pytest

from sulimo_amd import hip

CSRC = os.path.join(os.path.dirname(hip.__file__), "csrc")
INT_MAX = 2**31 - 1


@pytest.fixture(scope="module")
def grids(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    d = tmp_path_factory.mktemp("rope")
    (d / "r.cpp").write_text('''#include "rope_route.h"
#include <stdio.h>
int main() {
  int h, hd, rd, n;
  while (scanf("%d %d %d %d", &h, &hd, &rd, &n) == 4) {
    const sulimo::RopeVecGrid g = sulimo::rope_vec_grid(h, hd, rd, n);
    printf("%u %u\\n", g.x, g.y);
  }
}
''')
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "r.cpp"), "-o", str(d / "r")], check=True)

    def run(shapes):
        text = "".join("%d %d %d %d\n" % s for s in shapes)
        out = subprocess.run([str(d / "r")], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, ln.split())) for ln in out.splitlines()]

    return run


def test_vector_kernel_takes_only_what_its_thread_numbers_hold(grids):
    # one head of 128 reaches 2^31 threads at 2^27 tokens: a 34 GB buffer
    edge = [(h, hd, rd, n) for hd, rd in ((128, 128), (64, 40), (8, 8), (256, 64)) for h in (1, 5)
            for n in {(INT_MAX // (rd // 8) + d) for d in range(-600, 3)} | {2**27, 2**31 - 300} if n <= INT_MAX]
    edge += [(h, 8, 8, 3) for h in (262139, 262140, 262141, 300000)]
    for (h, hd, rd, n), (x, y) in zip(edge, grids(edge)):
        last = -(-n * (rd // 8) // 256) * 256 - 1  # the last workgroup's last thread number
        fits = last < INT_MAX and -(-h // 4) <= 65535
        assert (x > 0) == fits, (h, hd, rd, n)
        if x:
            assert x * 256 - 1 == last and y * 4 >= h > (y - 1) * 4


def test_vector_kernel_loads_are_aligned_and_whole(grids):
    shapes = [(h, hd, rd, n) for h in (1, 3, 4, 9) for hd in range(2, 140, 2) for rd in range(0, hd + 1, 2) for n in (1, 70)]
    for (h, hd, rd, n), (x, y) in zip(shapes, grids(shapes)):
        assert (x > 0) == (rd > 0 and rd % 8 == 0 and hd % 8 == 0), (h, hd, rd, n)
        if x:
            assert x * 256 >= n * (rd // 8) > (x - 1) * 256
            for i in range(0, rd // 2, 4):  # elements 2i and 2i+4 (Norm), i and i + rd/2 (NeoX) of a head
                assert all((2 * o) % 8 == 0 and o + 4 <= rd for o in (2 * i, 2 * i + 4, i, i + rd // 2))
