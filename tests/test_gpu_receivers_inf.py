"""Infinite inputs of the receiver products where the sum does not fill the last group of four: an infinity in the last
element (or, transposed, the last receiver) gives infinities of its entries' signs, and nothing else changes. (The
surplus entries of that group are zeros, and zero times infinity is not.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("drop", [0, 1, 2, 3])
def test_infinity_in_the_last_place(ctx, capi, oracle, small_relief, drop):
    P, E, _ = small_relief
    E = E[:len(E) - drop]
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=16, factor=1.5)
    rng = np.random.default_rng(drop)
    LL, k = 20 - drop, 2 * np.pi * 2000.0 / 343.0
    L = rng.standard_normal((LL, 3)) + [0.0, 5.0, 0.0]
    Q = oracle.Ctx(P, g.E, g.dense, g.lowrank).listener_matrix(k, L)
    print("infinity: N %% 4 = %d, LL %% 4 = %d" % (g.N % 4, LL % 4), flush=True)
    for transpose in (False, True):
        n = LL if transpose else g.N
        x = rng.standard_normal((2, n)) + 1j * rng.standard_normal((2, n))
        plain = g.receivers(k, L, ctx.to_device(x), 2, transpose).numpy()
        x[0, n - 1] = complex(np.inf, 0.0)
        y = g.receivers(k, L, ctx.to_device(x), 2, transpose).numpy()
        q = Q[n - 1] if transpose else Q[:, n - 1]
        assert np.all(q.real != 0) and np.all(q.imag != 0)
        assert np.array_equal(y[0].real, np.sign(q.real) * np.inf) and np.array_equal(y[0].imag, np.sign(q.imag) * np.inf)
        assert np.array_equal(y[1], plain[1])
