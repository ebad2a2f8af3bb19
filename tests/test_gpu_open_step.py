"""Device rounds whose first stages take the step control of the step before
along, against the same steps controlled by the host, bit for bit: rounds of
1, 2, 3, 8 and 17 steps (the two step-control headers alternate, graphs and
single launches end on either), one after the other, and meshes of 512 and
513 workgroups (up to 512 the first stages take the control along, beyond
each step has its own launch)."""
import numpy as np
import pytest

import fosite_amd
from fosite_amd import setups as S

CASES = {
    "disk": (S.kepler_disk_config(ni=72, nj=100), (1, 2, 3, 8, 17)),
    "disk_fp32": (dict(S.kepler_disk_config(ni=72, nj=100), dtype="fp32"), (1, 2, 3, 8, 17)),
    "riemann": (S.riemann2d_config(n=65), (3, 8, 1, 17)),
    # rejected steps: rounds that halt in between
    "disk_cfl": (dict(S.kepler_disk_config(ni=48, nj=64), cfl=0.9), (5, 9, 17)),
    "blocks_512": (S.kepler_disk_config(ni=64, nj=512 * 64), (2, 3)),
    "blocks_513": (S.kepler_disk_config(ni=64, nj=512 * 64 + 1), (2, 3)),
}


def make(cfg):
    init = S.initial(cfg)
    sim = fosite_amd.Fosite(cfg)
    sim.set_initial(init["pvar"], init.get("bccsound"), init.get("fcsound"), init.get("w"))
    sim.first_step()
    return sim


@pytest.mark.gpu
@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_gpu_rounds_equal_host_steps(name, single):
    cfg, rounds = CASES[name]
    print("open step", name, single, flush=True)
    sim, ref = make(cfg), make(cfg)
    if single:
        sim.profile(True)  # launches one by one
    for n in rounds:
        assert sim.run(n) == n
        for _ in range(n):
            assert not ref.step()
        a, b = sim.scalars(), ref.scalars()
        for k in ("iter", "n_adj", "brk", "time", "dt"):
            assert a[k] == b[k], (n, k, a, b)
        assert np.array_equal(sim.state()[0], ref.state()[0]), n
    sim.close()
    ref.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rounds", [(1, 2, 3, 8, 17), (4, 7)])
def test_gpu_batch_rounds_equal_host_steps(rounds):
    cfgs = [S.kepler_disk_config(ni=72, nj=100), S.kepler_disk_config(ni=40, nj=64)]
    print("open step batch", rounds, flush=True)
    sims, refs = [make(c) for c in cfgs], [make(c) for c in cfgs]
    with_batch = fosite_amd.Batch(sims)
    for n in rounds:
        assert list(with_batch.run(n)) == [n, n]
        for s, r in zip(sims, refs):
            for _ in range(n):
                r.step()
            assert s.scalars()["time"] == r.scalars()["time"]
            assert np.array_equal(s.state()[0], r.state()[0]), n
    with_batch.close()
    for s in sims + refs:
        s.close()
