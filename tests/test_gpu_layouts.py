"""Sweep parity at the edges of the staging and round layouts.

The GPU lattice and its counts equal the oracle's, site for site, after sweeps
in the GPU's own visit order (the bars of test_gpu_sweep):
  * tile staging: planes of more rows than threads (18 x 18 rows of 256
    threads), of exactly as many and of a few; tiles of more than two proposal
    chunks (1000 sites: four), at 256 and 512 threads; ragged tiles;
  * whole lattices: two sites per lane group and round with an odd site left
    over, one site, several runs of proposals, LDS blocks just full and just
    begun (256 and 257 sites), replicas of different sizes in one launch.
"""
import numpy as np
import pytest

from tests.helpers import print_case, rand_lattice
from tests.test_gpu_sweep import run_pair

pytestmark = pytest.mark.gpu

TILES = {
    "wide_rows": (dict(X=24, Y=24, Z=24), dict(kernel=2, tile=(4, 12, 12))),
    "rows_equal_threads": (dict(X=20, Y=20, Z=20), dict(kernel=2, tile=(4, 10, 10))),
    "few_rows": (dict(X=26, Y=12, Z=12, DipoleCutOff=2), dict(kernel=2, tile=(8, 3, 3))),
    "four_chunks": (dict(X=20, Y=20, Z=20, DipoleCutOff=2), dict(kernel=2, tile=(10, 10, 10))),
    "four_chunks_512": (dict(X=20, Y=20, Z=20, DipoleCutOff=4), dict(kernel=2, tile=(10, 10, 10), block_threads=512)),
    "ragged": (dict(X=19, Y=22, Z=25), dict(kernel=2)),
    "flat_ragged": (dict(X=41, Y=67, Z=1), dict(kernel=2)),
}


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("name", TILES)
def test_tile_layouts(sn, oracle, name, mixed):
    box, tuning = TILES[name]
    rp = sn.ReplicaParams(**box, T=300, Efield=(0.0, 0.03, -0.02), seed=77)
    print_case("tile_layout", name=name, mixed=mixed)
    lat = rand_lattice(rp.N, np.random.default_rng(len(name) + mixed), mixed=mixed)
    run_pair(sn, oracle, [rp], [lat], tuning, nsweeps=2)


WHOLE = {
    "two_sites_odd": [(12, 12, 12)],             # 54 sites a colour on 16 groups
    "one_block": [(16, 16, 1)],                  # 256 sites
    "block_and_one": [(257, 5, 1)],              # 1285 = 5 blocks and 5 sites
    "several_runs": [(16, 16, 16)],
    "uneven": [(12, 12, 12), (16, 12, 12), (12, 12, 16)],
}


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("name", WHOLE)
def test_whole_lattice_layouts(sn, oracle, name, mixed):
    rc = 1 if name == "block_and_one" else 3
    reps = [sn.ReplicaParams(*b, DipoleCutOff=rc, T=250 + 50 * k, K=0.1 * k, seed=90 + k) for k, b in enumerate(WHOLE[name])]
    print_case("whole_layout", name=name, mixed=mixed)
    rng = np.random.default_rng(len(name) + mixed)
    run_pair(sn, oracle, reps, [rand_lattice(r.N, rng, mixed=mixed) for r in reps], dict(kernel=3), nsweeps=3)
