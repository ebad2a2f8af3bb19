"""Batches whose members take different ways through the FARGO remap: in the
end-of-step evaluation (periodic in y), as the separate remap launch before it
(NO_GRADIENTS in y) and none (no FARGO), mixed and alone, in rounds of an odd
and an even number of steps; bit for bit the members run alone, and those
against the oracle."""
import numpy as np
import pytest

import oracle
from fosite_amd import setups as S
from tests.test_gpu_batch import check_same, run_batch

I = (slice(None), slice(2, -2), slice(2, -2))


def member(physics, ni, nj, fargo, bcy, **kw):
    cfg = S.shear_box_config(n=ni, jnum=nj, physics=physics, fargo=fargo, **kw)
    cfg["bc"] = cfg["bc"][:2] + [bcy, bcy]
    return cfg


def mixed(physics, dtype):
    ways = [(66, 19, 2, S.NO_GRADIENTS), (40, 33, 2, S.PERIODIC), (65, 24, 0, S.PERIODIC), (20, 9, 0, S.NO_GRADIENTS),
            (130, 12, 2, S.NO_GRADIENTS)]
    return [dict(member(physics, *w), dtype=dtype) for w in ways]


@pytest.mark.gpu
@pytest.mark.parametrize("tiling", [0, 3])
@pytest.mark.parametrize("chunks", [[7, 5], [6, 8]])
@pytest.mark.parametrize("which", ["mixed", "separate"])
@pytest.mark.parametrize("physics,dtype", [(S.EULER, "fp64"), (S.EULER_ISOTHERM, "fp64"), (S.EULER_ISOTHERM, "fp32")])
def test_gpu_batch_remap_ways(physics, dtype, which, chunks, tiling):
    print("batch remap", physics, dtype, which, chunks, tiling, flush=True)
    cfgs = mixed(physics, dtype)
    if which == "separate":
        cfgs = [cfgs[0], cfgs[4]]
    res, info = run_batch(cfgs, chunks, autotune=False, tiling=tiling)
    assert info["device_steps"] > 0
    check_same(cfgs, res, chunks)
    if dtype == "fp32":
        return
    for cfg, (taken, cv, sc, _) in zip(cfgs, res):
        init = S.initial(cfg)
        ref = oracle.Oracle(cfg)
        ref.set_initial(init["pvar"], init.get("bccsound"), init.get("fcsound"), init.get("w"))
        ref.first_step()
        for _ in range(taken):
            ref.step()
        want, _, rs = ref.state()
        assert sc["iter"] == rs["iter"] and sc["n_adj"] == rs["n_adj"] and sc["time"] == rs["time"], (sc, rs)
        assert np.array_equal(cv[I], want[I])
