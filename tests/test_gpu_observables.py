"""Observable kernels at the edges of their tiles, against the oracle.

Bars as in test_gpu_energy: FP64 on both sides, only the summation order
differs; counts exact.
"""
import numpy as np
import pytest

from tests.helpers import oracle_model, print_case, rand_lattice

pytestmark = pytest.mark.gpu

# workgroups of 4 rows x up to 16 z walk along x over a ring of ten planes:
# rows left over, z split unevenly, one plane, more planes than the ring has,
# every axis shorter than the reach of 8 sites
RADIAL = [(2, 2, 1), (2, 3, 2), (2, 5, 17), (9, 4, 16), (23, 6, 33), (64, 2, 3), (31, 7, 1)]


@pytest.mark.parametrize("dims", RADIAL)
def test_radial_order_tiles(sn, oracle, dims):
    rp = sn.ReplicaParams(*dims, DipoleCutOff=1)
    print_case("radial_tiles", dims=dims)
    lat = rand_lattice(rp.N, np.random.default_rng(sum(dims)), mixed=True)
    with sn.StarryNight(rp) as ctx:
        ctx.set_lattice(lat)
        fe, afe, cnt = ctx.radial_order()
    few, afew, cntw = oracle_model(oracle, rp).radial_order(lat)
    assert np.array_equal(cnt, cntw)
    assert np.abs(fe - few).max() <= 1e-12 and np.abs(afe - afew).max() <= 1e-12


# rows held whole by the lanes (several to a wave below 33 sites) and cut at
# Z > 64; rows of a workgroup left over; an odd X; axes shorter than the reach
STENCIL = [(2, 3, 2), (5, 70, 1), (3, 9, 31), (4, 17, 64), (3, 5, 65), (7, 4, 130)]


@pytest.mark.parametrize("dims", STENCIL)
def test_stencil_tiles(sn, oracle, dims):
    rp = sn.ReplicaParams(*dims, DipoleCutOff=1)
    print_case("stencil_tiles", dims=dims)
    lat = rand_lattice(rp.N, np.random.default_rng(sum(dims)), mixed=True)
    o = oracle_model(oracle, rp)
    with sn.StarryNight(rp) as ctx:
        ctx.set_lattice(lat)
        assert np.abs(ctx.dipole_potential() - o.dipole_potential(lat)).max() <= 1e-12
        for cutoff in range(1, 10):
            assert np.abs(ctx.dipole_efield(cutoff) - o.dipole_efield(lat, cutoff)).max() <= 1e-12


# rows held whole or cut (Z = 180: halo inside the lattice), rows and x left
# over by the workgroups, workgroups of several steps along x, one and two x a
# step, plane (2D) lattices of more rows than lanes, an axis of two sites,
# lattices without a tiling
ENERGY = [((8, 7, 6), 3), ((7, 30, 5), 2), ((9, 12, 180), 4), ((10, 9, 70), 1), ((33, 20, 16), 5), ((16, 600, 1), 3),
          ((300, 10, 1), 5), ((64, 64, 64), 3),
          ((2, 40, 5), 1), ((6, 7, 8), 5), ((6, 9, 1), 5)]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("dims,rc", ENERGY)
def test_energy_workgroups(sn, oracle, dims, rc, mixed):
    rp = sn.ReplicaParams(*dims, DipoleCutOff=rc, CageStrain=0.7, Efield=(0.01, -0.02, 0.03), K=0.2)
    print_case("energy_workgroups", dims=dims, rc=rc, mixed=mixed)
    lat = rand_lattice(rp.N, np.random.default_rng(sum(dims) + rc), mixed=mixed)
    with sn.StarryNight(rp) as ctx:
        ctx.set_lattice(lat)
        e, parts = ctx.energy()
        g, dp, e2 = ctx.gradient()
    o = oracle_model(oracle, rp)
    ew, pw = o.energy(lat)
    gw, dpw = o.gradient(lat)
    scale = np.abs(pw).sum() + 1.0
    assert abs(e - ew) <= 1e-12 * scale and e2 == e
    assert np.abs(parts - pw).max() <= 1e-12 * scale
    assert np.abs(g - gw).max() <= 1e-11 * (np.abs(gw).max() + 1.0)
    assert np.abs(dp - dpw).max() <= 1e-11 * (np.abs(dpw).max() + 1.0)
