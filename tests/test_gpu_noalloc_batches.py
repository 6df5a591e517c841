"""sn_gradient_all_device_noalloc where the batch's partial sums do not fit the
fixed scratch at once: a launch per replica, in stream order, over the same
rows.  13,200 untiled replicas take a workgroup each (131,072 doubles hold
13,107 rows of ten)."""
import ctypes as C

import numpy as np
import pytest

from tests.helpers import print_case, rand_lattice

pytestmark = pytest.mark.gpu

ROWS = 131072 // 10


@pytest.mark.parametrize("mixed", [False, True])
def test_noalloc_adjoint_a_replica_at_a_time(sn, mixed):
    import torch
    R, X = ROWS + 93, 4
    print_case("noalloc_batches", replicas=R, X=X, mixed=mixed)
    rng = np.random.default_rng(7)
    reps = [sn.ReplicaParams(X, X, X, T=300, K=0.1 * (k % 2), Efield=(0, 0, 0.01 * (k % 3)), seed=k + 1)
            for k in range(R)]
    with sn.StarryNight(reps, sn.TuningParams(kernel=2)) as ctx:
        for r, rp in enumerate(reps):
            ctx.set_lattice(rand_lattice(rp.N, rng, mixed=mixed and r % 2 == 0), r)
        g_one, g_each = (torch.full((R * X ** 3, 3), float("nan"), dtype=torch.float64, device="cuda:0")
                         for _ in range(2))
        torch.cuda.synchronize()
        dp_one, e_one = ctx.gradient_all_device(g_one)
        dp_each, e_each = np.empty((R, 6)), np.empty(R)
        pd = C.POINTER(C.c_double)
        st = sn.lib().sn_gradient_all_device_noalloc(ctx._h, C.c_void_p(g_each.data_ptr()), dp_each.ctypes.data_as(pd),
                                                     e_each.ctypes.data_as(pd))
        assert st == 0, sn.lib().sn_last_error(ctx._h)
        torch.cuda.synchronize()
    # the same sums per site; per replica 64 terms of at most ~150 in another
    # order, and lengths applied before or after the sum over neighbours: some
    # 200 roundings of 2^-53
    tol = 200 * 2.0 ** -53
    assert float((g_one - g_each).abs().max()) <= tol * float(g_one.abs().max())
    assert np.abs(dp_one - dp_each).max() <= 64 * tol * np.abs(dp_one).max()
    assert np.abs(e_one - e_each).max() <= 64 * tol * np.abs(e_one).max()
