"""k_rhs at the edges of its strips (64 columns x 1..8 rows per wave, four
strips per workgroup): meshes of fewer columns than a strip's halo, one column
more or less than a strip, a last strip of one and two columns (whose halo
reaches into the neighbour's x ghost cells), fewer rows than a workgroup, and
a tall mesh with eight rows per strip and a short last one; against the oracle
as in test_gpu_parity (bit-exact without absorbing boundaries, relative L1
<= 1e-12 with them)."""
import numpy as np
import pytest

from fosite_amd import setups
from tests.parity import rel_l1, run_pair

PROBLEMS = {
    "euler_nograd": lambda ni, nj: dict(setups.riemann2d_config(n=8), inum=ni, jnum=nj),
    "euler_periodic_prim": lambda ni, nj: dict(setups.shear_box_config(8, recvars=setups.PRIMITIVE), inum=ni, jnum=nj),
    "disk_fargo": lambda ni, nj: setups.kepler_disk_config(ni=ni, nj=nj),
    "euler_disk_dp5": lambda ni, nj: setups.euler_disk_config(ni=ni, nj=nj),
}
SIZES = [(4, 4), (5, 9), (63, 13), (64, 4), (65, 7), (66, 10), (127, 5), (129, 36)]


def compare(cfg, nsteps):
    exact = setups.ABSORBING not in cfg["bc"]
    I = (slice(None), slice(2, -2), slice(2, -2))
    for n, cv, sc, rc, rs in run_pair(cfg, nsteps):
        assert sc["n_adj"] == rs["n_adj"] and sc["brk"] == rs["brk"], (n, sc, rs)
        if exact:
            assert sc["time"] == rs["time"] and sc["dt"] == rs["dt"], (n, sc, rs)
            assert np.array_equal(cv[I], rc[I]), (n, np.abs(cv[I] - rc[I]).max())
        else:
            assert (rel_l1(cv, rc) <= 1e-12).all(), (n, rel_l1(cv, rc))


@pytest.mark.gpu
@pytest.mark.parametrize("ni,nj", SIZES)
@pytest.mark.parametrize("problem", list(PROBLEMS))
def test_gpu_strip_edges(problem, ni, nj):
    print("strips", problem, ni, nj, flush=True)
    compare(PROBLEMS[problem](ni, nj), 4)


@pytest.mark.gpu
@pytest.mark.parametrize("nj", [3701, 5001])
@pytest.mark.parametrize("problem", ["euler_nograd", "disk_fargo"])
def test_gpu_tall_strips(problem, nj):
    """Two strips of columns; 3701 rows: eight rows per strip, five in the last;
    5001: ten rows (the edge columns in two passes), one in the last."""
    print("tall strips", problem, nj, flush=True)
    compare(PROBLEMS[problem](65, nj), 2)
