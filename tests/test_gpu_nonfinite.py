"""Values that leave the FP64 range: quotients that overflow, divisors that are
exactly zero.  The reference's IEEE divisions give Inf there, which its sound
speed, wave speeds, time step and data checks act on (a run then ends with
dt = 0 or a break); the device has to take the same decisions in the same step
and leave the same values (NaN for NaN).  Against the oracle, host steps and
device rounds, bit for bit (no transcendental functions are involved).  Not with
the limiters that compare signs: the sign of a NaN is the hardware's choice."""
import numpy as np
import pytest

import fosite_amd
import oracle
from fosite_amd import setups as S

I = (slice(None), slice(2, -2), slice(2, -2))


def gas(cfg, rho=1.0, pressure=1.0):
    pv = np.zeros((4, cfg["jnum"] + 4, cfg["inum"] + 4))
    pv[0], pv[3] = rho, pressure
    return pv


def overflowing_sound_speed(limiter, recvars):
    """gamma*P/rho overflows in one cell: cs = Inf, 1/dt = Inf."""
    cfg = dict(S.riemann2d_config(n=16), limiter=limiter, recvars=recvars)
    pv = gas(cfg)
    pv[0, 9, 7], pv[3, 9, 7] = 1e-300, 1e10
    return cfg, pv


def overflowing_inverse_step(limiter, recvars):
    """A finite velocity over a cell's length overflows: 1/dt = Inf."""
    cfg = dict(S.shear_box_config(n=32, physics=S.EULER_ISOTHERM, fargo=0, recvars=recvars), limiter=limiter)
    pv = S.initial(cfg)["pvar"]
    pv[0, 9, 7], pv[1, 9, 7] = 1e-300, -1e308
    return cfg, pv


def zero_face(along):
    """The linear slope through 1, 1, 5 without a limiter makes the lower face of
    the middle cell exactly zero, which no check of the cells sees."""
    def build(limiter, recvars):
        cfg = dict(S.riemann2d_config(n=16), limiter=limiter, recvars=recvars)
        pv = gas(cfg)
        pv[(0, 9, 8) if along == "x" else (0, 8, 9)] = 5.0
        return cfg, pv
    return build


def overflowing_slopes(limiter, recvars):
    """Van Leer's numerator overflows (differences of 1e160), the fields do not."""
    cfg = dict(S.riemann2d_config(n=16), limiter=limiter, recvars=recvars)
    pv = gas(cfg)
    pv[3, :, 8:] = 1e160
    pv[3, :, 9:] = 3e160
    return cfg, pv


PROBLEMS = {
    "overflowing_sound_speed": (overflowing_sound_speed, [S.VANLEER, S.OSPRE]),
    "overflowing_inverse_step": (overflowing_inverse_step, [S.VANLEER, S.OSPRE]),
    "zero_face_x": (zero_face("x"), [S.NOLIMIT]),
    "zero_face_y": (zero_face("y"), [S.NOLIMIT]),
    "overflowing_slopes": (overflowing_slopes, [S.VANLEER, S.OSPRE]),
}


@pytest.mark.gpu
@pytest.mark.parametrize("recvars", [S.PRIMITIVE, S.CONSERVATIVE])
@pytest.mark.parametrize("problem,limiter", [(p, l) for p in PROBLEMS for l in PROBLEMS[p][1]])
def test_gpu_nonfinite(problem, limiter, recvars):
    print("nonfinite", problem, limiter, recvars, flush=True)
    cfg, pv = PROBLEMS[problem][0](limiter, recvars)
    init = S.initial(cfg)
    sims = fosite_amd.Fosite(cfg), fosite_amd.Fosite(cfg)
    ref = oracle.Oracle(cfg)
    for s in sims + (ref,):
        s.set_initial(pv, init.get("bccsound"), init.get("fcsound"), init.get("w"))
        s.first_step()

    def compare(s):
        want, _, rs = ref.state()
        cv, _ = s.state()
        sc = s.scalars()
        for k in ("iter", "n_adj", "brk", "time", "dt"):
            assert np.array_equal(sc[k], rs[k], equal_nan=True), (k, sc, rs)
        assert np.array_equal(cv[I], want[I], equal_nan=True)

    for s in sims:
        compare(s)
    steps = 0
    while steps < 3:
        ended = ref.step()
        assert sims[0].step() == ended
        compare(sims[0])
        steps += 1
        if ended:
            break
    sims[1].run(steps)
    compare(sims[1])
    for s in sims:
        s.close()
