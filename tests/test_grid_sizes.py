"""Launch sizes of the kernels that take several lanes per item, over all item counts that the engine accepts: the header that
the kernels' launches use, compiled for the host."""
import os
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include "grid.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
  const gsj::ItemGrid g = gsj::item_grid(strtoull(argv[1], nullptr, 10), (uint32_t)atoi(argv[2]));
  printf("%u %u\n", g.x, g.y);
}
"""


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    (d / "grid.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "postgis-cuda_amd", "csrc"), "-o", d / "grid", d / "grid.cpp"], check=True)
    return lambda n, lanes: [int(v) for v in subprocess.run([d / "grid", str(n), str(lanes)], check=True, capture_output=True, text=True).stdout.split()]


# 2^28 and 2^29: where one row of 16 or 8 lanes per item reaches the launch limit; candidates and rings end below 2^32
@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 256, 257, 2**26, 2**26 + 1, 2**28 - 1, 2**28, 2**29, 2**32 - 1])
@pytest.mark.parametrize("lanes", [8, 16])
def test_blocks_cover_the_items_within_a_launch(blocks, n, lanes):
    (x, y), per = blocks(n, lanes), 256 // lanes
    assert 0 < x * 256 < 2**32 and 0 < y < 2**16
    assert n <= x * y * per and n > x * (y - 1) * per
    if n <= 2**26:   # one row of as many blocks as the items fill
        assert y == 1 and (x - 1) * per < n
