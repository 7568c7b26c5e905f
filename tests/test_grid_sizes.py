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
  for (int k = 1; k + 1 < argc; k += 2) printf("%u\n", gsj::stride_blocks(strtoull(argv[k], nullptr, 10), (uint32_t)atoi(argv[k + 1])));
}
"""


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    (d / "grid.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "postgis-cuda_amd", "csrc"), "-o", d / "grid", d / "grid.cpp"], check=True)
    return lambda n, lanes: int(subprocess.run([d / "grid", str(n), str(lanes)], check=True, capture_output=True, text=True).stdout)


# 2^28 and 2^29: where a round of 16 or 8 lanes per item reaches the launch limit; candidates and rings end below 2^32
@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 256, 257, 2**26, 2**26 + 1, 2**28 - 1, 2**28, 2**29, 2**32 - 1])
@pytest.mark.parametrize("lanes", [8, 16])
def test_blocks_cover_the_items_within_a_launch(blocks, n, lanes):
    b, per = blocks(n, lanes), 256 // lanes
    assert 0 < b * 256 < 2**32
    if n <= 2**26:   # a single round of as many blocks as the items fill
        assert (b - 1) * per < n <= b * per
