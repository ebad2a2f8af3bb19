"""Grids of the kernels that pass once over all cells of a stored pvar
(cell_blocks): enough workgroups for the mesh, independent of the height of
the RHS kernel's strips, and no more partials than the buffers hold."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fosite_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
SIZES = [(4, 4), (4, 5000), (64, 64), (65, 9), (251, 333), (512, 1024), (1024, 2048), (3000, 2001), (65, 100003)]
PROGRAM = """
#include <cstdio>
#include "fv_device.h"
int main() {
  int i, j;
  while (std::scanf("%d %d", &i, &j) == 2)
    std::printf("%d %d %d %d\\n", fv::cell_blocks(i, j), fv::tile_blocks(i, j),
                fv::strip_cols(i) * fv::strip_blocks(j, 1) + 1, fv::SCRATCH_MAX_BLOCKS);
}
"""


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch_sizes")
    src, exe = str(d / "sizes.cpp"), str(d / "sizes")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", ROCM + "/include", "-I", CSRC,
                           "-o", exe, src])
    text = "\n".join("%d %d" % s for s in SIZES)
    out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
    return dict(zip(SIZES, (tuple(map(int, line.split())) for line in out.splitlines())))


@pytest.mark.parametrize("size", SIZES)
def test_cell_blocks_cover_the_mesh_and_fit_the_partials(blocks, size):
    n, tiles, partials, scratch = blocks[size]
    cells = (size[0] + 4) * (size[1] + 4)
    # two cells of the interior a thread; a mesh narrower than a strip has fewer, never idle workgroups
    assert n == min(-(-size[0] // 64) * -(-size[1] // 8), -(-cells // 256))
    assert 1 <= n <= partials
    assert tiles > scratch or n <= scratch  # (the allocation-free step refuses more tiles)
