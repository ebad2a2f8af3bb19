"""k_visc at the edges of its strips (up to 60 columns of the ghost-inclusive
mesh x 4 .. 16 rows per wave): meshes narrower than a strip, strips that end
with the first, at and behind the east ghost cells (widths of 60, 59 and 58
columns), fewer rows than a strip and a short last one, corner cells of every
pair of boundary rules; against the oracle (bit for bit without absorbing
boundaries, relative L1 <= 1e-12 with them)."""
import numpy as np
import pytest

from fosite_amd import setups as S
from tests.parity import rel_l1, run_pair

PROBLEMS = {
    "euler_nograd": lambda ni, nj: dict(S.riemann2d_config(n=8), inum=ni, jnum=nj, ymax=float(nj) / ni, vismodel=1,
                                       dynconst=1e-4),
    "euler_periodic": lambda ni, nj: S.shear_box_config(n=ni, jnum=nj, fargo=0, vismodel=1, dynconst=1e-3),
    "disk_alpha_absorbing": lambda ni, nj: dict(S.kepler_disk_config(ni=ni, nj=nj), fargo=0, vismodel=2,
                                                dynconst=0.01),
    "disk_alpha_fargo_nograd": lambda ni, nj: dict(S.kepler_disk_config(ni=ni, nj=nj), fargo=1, vismodel=2,
                                                   dynconst=0.01, omega=0.3, rotframe=1,
                                                   bc=[S.NO_GRADIENTS] * 2 + [S.PERIODIC] * 2),
}
SIZES = [(4, 4), (56, 9), (57, 12), (58, 13), (59, 28), (117, 10), (118, 29), (3537, 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("problem,ni,nj", [(p, ni, nj) for p in PROBLEMS for ni, nj in SIZES
                                           if (p, ni) != ("euler_nograd", 3537)])  # (breaks after 270 substeps)
def test_gpu_visc_strip_edges(problem, ni, nj):
    print("viscous strips", problem, ni, nj, flush=True)
    cfg = PROBLEMS[problem](ni, nj)
    exact = S.ABSORBING not in cfg["bc"]
    I = (slice(None), slice(2, -2), slice(2, -2))
    for n, cv, sc, rc, rs in run_pair(cfg, 3):
        assert sc["n_adj"] == rs["n_adj"] and sc["brk"] == rs["brk"], (n, sc, rs)
        if exact:
            assert sc["time"] == rs["time"] and sc["dt"] == rs["dt"], (n, sc, rs)
            assert np.array_equal(cv[I], rc[I], equal_nan=True), (n, np.abs(cv[I] - rc[I]).max())
        else:
            assert (rel_l1(cv, rc) <= 1e-12).all(), (n, rel_l1(cv, rc))


@pytest.mark.gpu
def test_gpu_visc_tall_strips_molecular():
    """16 rows per strip (the most), the last strip one row."""
    print("viscous tall strips", flush=True)
    cfg = PROBLEMS["euler_periodic"](8, 32989)
    for n, cv, sc, rc, rs in run_pair(cfg, 1):
        assert sc["time"] == rs["time"] and sc["dt"] == rs["dt"], (n, sc, rs)
        assert np.array_equal(cv[:, 2:-2, 2:-2], rc[:, 2:-2, 2:-2], equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("vismodel", [2, 3])
def test_gpu_visc_tall_strips_rotation(vismodel):
    """The same with a viscosity from the local rotation (ALPHA, BETA): e_phi/r
    at 32989 angles."""
    print("viscous tall strips", vismodel, flush=True)
    cfg = dict(PROBLEMS["disk_alpha_fargo_nograd"](8, 32989), vismodel=vismodel)
    for n, cv, sc, rc, rs in run_pair(cfg, 1):
        assert sc["time"] == rs["time"] and sc["dt"] == rs["dt"], (n, sc, rs)
        assert np.array_equal(cv[:, 2:-2, 2:-2], rc[:, 2:-2, 2:-2], equal_nan=True)
