"""Drawn dipoles against the oracle, bit for bit: the disc test is exact, the
root and its two products round once each, on the host as on the device."""
import numpy as np
import pytest

from tests.helpers import print_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [1, 0xFFFFFFFFFFFFFFFF])
def test_random_lattice_is_the_oracles(sn, oracle, seed):
    rp = sn.ReplicaParams(32, 32, 30, seed=seed)
    print_case("draws", N=rp.N, seed=seed)
    with sn.StarryNight(rp) as ctx:
        ctx.init_lattice_random(0)
        got = ctx.get_lattice()[:, :3]
    want = np.array([oracle.counter_draw(seed, 0, 0xFFFFFFFF, i)[0] for i in range(rp.N)])
    assert np.array_equal(got, want)
