"""The FARGO remap formed while the end-of-step evaluation marches along y, at
the rows where a ring wraps: rings of 4 to 19 rows, background velocities of
both signs from a fraction of a cell to more than a ring per step (and zero),
in the strips' columns and their edge columns; with a y boundary that is not
periodic the separate remap kernel runs.  Bit for bit against the oracle (no
absorbing boundaries), host steps and device rounds."""
import numpy as np
import pytest

import fosite_amd
import oracle
from fosite_amd import setups as S

I = (slice(None), slice(2, -2), slice(2, -2))


def build(physics, ni, nj, amp, bcy):
    cfg = S.shear_box_config(n=ni, jnum=nj, physics=physics)
    cfg["bc"] = cfg["bc"][:2] + [bcy, bcy]
    init = S.initial(cfg)
    i = np.arange(ni + 4)
    w = amp * np.sin(2 * np.pi * (i - 2) / ni)
    w[i == 2] = 0.0
    init["pvar"][2] += w[None, :] - init["w"][None, :]
    init["w"] = w
    return cfg, init


def start(sim, init):
    sim.set_initial(init["pvar"], init.get("bccsound"), init.get("fcsound"), init["w"])
    sim.first_step()


@pytest.mark.gpu
@pytest.mark.parametrize("bcy", [S.PERIODIC, S.NO_GRADIENTS])
@pytest.mark.parametrize("amp", [0.3, 20.0, 3000.0])
@pytest.mark.parametrize("ni,nj", [(20, 4), (65, 5), (66, 19)])
@pytest.mark.parametrize("physics", [S.EULER, S.EULER_ISOTHERM])
def test_gpu_fargo_rings_that_wrap(physics, ni, nj, amp, bcy):
    print("fargo march", physics, ni, nj, amp, bcy, flush=True)
    cfg, init = build(physics, ni, nj, amp, bcy)
    sim, rounds, ref = fosite_amd.Fosite(cfg), fosite_amd.Fosite(cfg), oracle.Oracle(cfg)
    for s in (sim, rounds, ref):
        start(s, init)
    for _ in range(6):
        assert sim.step() == ref.step()
    rounds.run(6)
    want, _, rs = ref.state()
    for s in (sim, rounds):
        cv, _ = s.state()
        sc = s.scalars()
        for k in ("iter", "n_adj", "brk", "time", "dt"):
            assert sc[k] == rs[k], (k, sc, rs)
        assert np.array_equal(cv[I], want[I], equal_nan=True)
        s.close()
