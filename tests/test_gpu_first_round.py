"""The first rounds of a new state, in which the long graph of steps is built
while the device works on the pairs ahead of it: round lengths about one and
two long graphs (8 steps), odd and even, each as a first round and as the
second one behind it; bit for bit the same steps controlled by the host."""
import numpy as np
import pytest

from fosite_amd import setups as S
from tests.test_gpu_open_step import make

CONFIGS = {
    "disk": S.kepler_disk_config(ni=40, nj=64),                     # step control inside the first stages
    "disk_fargo1": dict(S.kepler_disk_config(ni=40, nj=64), fargo=1),  # a launch of its own
}


@pytest.mark.gpu
@pytest.mark.parametrize("n", [7, 8, 9, 15, 16, 17, 24, 25])
@pytest.mark.parametrize("name", list(CONFIGS))
def test_gpu_first_rounds_equal_host_steps(name, n):
    print("first round", name, n, flush=True)
    sim, ref = make(CONFIGS[name]), make(CONFIGS[name])
    for _ in range(2):
        assert sim.run(n) == n
        for _ in range(n):
            assert not ref.step()
        a, b = sim.scalars(), ref.scalars()
        for k in ("iter", "n_adj", "brk", "time", "dt"):
            assert a[k] == b[k], (k, a, b)
        assert np.array_equal(sim.state()[0], ref.state()[0])
    sim.close()
    ref.close()
