"""Receiver products at the edges of their tiles: listener and element counts around 4 and 16, right-hand sides around
a tile of 8 and a pass of 40, forward and transposed, against the oracle's listener matrix. Both sums are FP64 over
at most 741 elements: rounding of 1e-16 per term, entries accurate to 1e-13, hence 1e-12."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,LL", [(1, 1), (1, 181), (3, 4), (8, 5), (9, 15), (37, 16), (40, 17), (41, 19), (83, 33)])
def test_receivers_vs_oracle(ctx, capi, oracle, small_relief, nr, LL):
    P, E, _ = small_relief
    E = E[:len(E) - 3]  # N not a multiple of 4
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=16, factor=1.5)
    assert g.N % 4 and g.N % 16
    rng = np.random.default_rng(nr)
    L = rng.standard_normal((LL, 3)) + [0.0, 5.0, 0.0]
    k = 2 * np.pi * 2000.0 / 343.0
    Q = oracle.Ctx(P, g.E, g.dense, g.lowrank).listener_matrix(k, L)
    X = rng.standard_normal((nr, g.N)) + 1j * rng.standard_normal((nr, g.N))
    V = rng.standard_normal((nr, LL)) + 1j * rng.standard_normal((nr, LL))
    print("receivers nr=%d LL=%d" % (nr, LL), flush=True)
    y = g.receivers(k, L, ctx.to_device(X), nr).numpy()
    b = g.receivers(k, L, ctx.to_device(V), nr, transpose=True).numpy()
    assert rel(y, X @ Q.T) < 1e-12 and rel(b, V @ Q) < 1e-12
    # a right-hand side alone gets the bits it gets in the batch
    j = nr - 1
    assert np.array_equal(g.receivers(k, L, ctx.to_device(X[j:]), 1).numpy()[0], y[j])
    assert np.array_equal(g.receivers(k, L, ctx.to_device(V[j:]), 1, transpose=True).numpy()[0], b[j])
