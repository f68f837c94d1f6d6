"""The listener ACA around the edges of its batches of eight crosses and of its 64-row blocks: rank limits below, at and
above a batch, listener counts around a wavefront. A limited factorisation is the beginning of the unlimited one, bit
for bit, and the unlimited one reproduces the matrix."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("LL", [2, 9, 63, 64, 65, 129])
def test_limits_and_batches(ctx, capi, oracle, small_relief, LL):
    P, E, _ = small_relief
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=32, factor=1.5)
    oc = oracle.Ctx(P, g.E, g.dense, g.lowrank)
    k = 2 * np.pi * 2000.0 / 343.0
    d = np.random.default_rng(LL).standard_normal((LL, 3))
    L = 5.0 * d / np.linalg.norm(d, axis=1, keepdims=True)
    L[:, 1] = np.abs(L[:, 1]) + 0.5
    tol = 1e-7
    q = g.listener_aca(k, L, tol)
    U, V = q.factors()
    r = U.shape[1]
    assert 0 < r <= LL - 1
    if r < min(LL, g.N) - 1:  # stopped by the rule
        assert rel(U @ V, oc.listener_matrix(k, L)) < 1e3 * tol
    for lim in (1, 7, 8, 9, 16, 17):
        if lim >= LL:
            continue
        Ul, Vl = g.listener_aca(k, L, tol, max_rank=lim).factors()
        n = min(lim, r)
        assert Ul.shape == (LL, n) and Vl.shape == (n, g.N)
        assert np.array_equal(Ul, U[:, :n]) and np.array_equal(Vl, V[:n])
