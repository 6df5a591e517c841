"""Energy differences of proposed moves at the edges of the lane groups.

1 to 16 lanes share a move and take the offset table in rounds: tables shorter than
a round, of whole rounds and with a rest, one move, a group's worth and one
more, and more moves than groups in flight.  The bar is that of the other
site-energy tests: FP64 on both sides, only the summation order differs.
"""
import numpy as np
import pytest

from tests.helpers import oracle_model, print_case, rand_lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,rc", [((25, 25, 1), 1), ((6, 7, 1), 5), ((8, 9, 1), 2), ((9, 5, 3), 1), ((4, 6, 3), 2),
                                     ((7, 9, 11), 4), ((20, 20, 20), 5)])
def test_moves_of_any_count(sn, oracle, dims, rc):
    rp = sn.ReplicaParams(*dims, DipoleCutOff=rc, CageStrain=0.7, Efield=(0.01, -0.02, 0.03), K=0.2)
    print_case("moves", dims=dims, rc=rc)
    rng = np.random.default_rng(sum(dims) + rc)
    lat = rand_lattice(rp.N, rng, mixed=True)
    o = oracle_model(oracle, rp)
    with sn.StarryNight(rp) as ctx:
        ctx.set_lattice(lat)
        for n in (1, 16, 17, 16384, 16385, 33000):
            sites = rng.integers(0, rp.N, n).astype(np.int32)
            props = rand_lattice(n, rng, mixed=False)[:, :3].copy()
            got = ctx.site_energy_batch(sites, props)
            check = slice(None) if n < 100 else slice(n - 200, n)
            want, _ = o.site_energy_batch(lat, sites[check], props[check])
            assert np.allclose(got[check], want, rtol=0, atol=1e-10 * max(1.0, np.abs(want).max()))
            # a move's answer does not depend on its place in the list
            assert np.array_equal(got[:200], ctx.site_energy_batch(sites[:200], props[:200]))
