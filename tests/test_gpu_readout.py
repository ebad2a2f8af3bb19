"""Host arrays to and from the device state (k_load, k_readout): conversions
and padding on odd meshes, every cell, ghosts included, bit for bit against
numpy in FP64; the FP32 form stores the FP64 values rounded once."""
import numpy as np
import pytest

from fosite_amd import setups


def cons(p, g):
    u = [p[0], p[0] * p[1], p[0] * p[2]]
    if len(p) == 4:
        u.append(p[3] / (g - 1.0) + 0.5 * p[0] * (p[1] * p[1] + p[2] * p[2]))
    return np.stack(u)


def prim(u, g):
    inv = 1.0 / u[0]
    p = [u[0], u[1] * inv, u[2] * inv]
    if len(u) == 4:
        p.append((g - 1.0) * (u[3] - 0.5 * inv * (u[1] * u[1] + u[2] * u[2])))
    return np.stack(p)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
@pytest.mark.parametrize("euler", [False, True])
@pytest.mark.parametrize("ni,nj", [(4, 4), (13, 70), (129, 6), (257, 130)])
def test_gpu_state_in_and_out(ni, nj, euler, dtype):
    import fosite_amd
    cfg = (dict(setups.riemann2d_config(n=8), inum=ni, jnum=nj) if euler else setups.kepler_disk_config(ni=ni, nj=nj))
    cfg["dtype"] = dtype
    rng = np.random.default_rng(ni * nj)
    V, shape = (4 if euler else 3), (nj + 4, ni + 4)
    p = np.stack([rng.uniform(0.1, 2, shape), rng.normal(size=shape), rng.normal(size=shape),
                  rng.uniform(0.1, 2, shape)][:V])
    stored = lambda u: u.astype(np.float32).astype(np.float64) if dtype == "fp32" else u  # noqa: E731
    print("readout", ni, nj, euler, dtype, flush=True)
    sim = fosite_amd.Fosite(cfg)
    init = setups.initial(cfg)
    sim.set_initial(p, init.get("bccsound"), init.get("fcsound"), init.get("w"))
    for u in (cons(p, 1.4), cons(p, 1.4) * 0.75):
        cv, pv = sim.state()
        assert np.array_equal(cv, stored(u))
        assert np.array_equal(pv, prim(stored(u), cfg["gamma"]))
        sim.set_conservative(cons(p, 1.4) * 0.75)
    sim.close()
