"""Pair tiles of the shape gradient at their edges: rows (touched elements) and columns (elements, listeners) that
do not fill 16 x 16 tiles, fewer columns than one tile per wavefront, right-hand-side counts around the GEMM's step
of two, against the oracle. Both sides evaluate the same sums in FP64: up to 700 terms of rounding 1e-16 each, amplified
by the cancellation of near-element derivatives (1e-12 at worst), give the bound 1e-11."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup(ctx, capi, oracle, small_relief):
    P, E, top = small_relief
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=16, factor=1.5)
    return g, oracle.Ctx(P, g.E, g.dense, g.lowrank), top


# (right-hand sides, listeners, differentiable vertices): one row, 17 rows, all; 1, 15, 16, 17, 65 and 181 columns
@pytest.mark.parametrize("nr,LL,ndiff", [(1, 1, 1), (2, 15, 3), (3, 16, 20), (4, 17, 256), (5, 65, 77), (37, 181, 256),
                                         (41, 19, 5)])
def test_pair_tiles_vs_oracle(setup, ctx, capi, nr, LL, ndiff):
    g, oc, top = setup
    rng = np.random.default_rng(nr)
    L = rng.standard_normal((LL, 3)) * 3.0 + [0.0, 20.0, 0.0]
    k = 2 * np.pi * 1500.0 / 343.0
    X, Lm = (rng.standard_normal((nr, g.N)) + 1j * rng.standard_normal((nr, g.N)) for _ in range(2))
    VF = rng.standard_normal((nr, LL)) + 1j * rng.standard_normal((nr, LL))
    src = rng.standard_normal((nr, 3))
    src /= np.linalg.norm(src, axis=1)[:, None]
    diff = rng.permutation(top)[:ndiff]
    print("pairs nr=%d LL=%d ndiff=%d" % (nr, LL, ndiff), flush=True)
    got = g.shape_grad(k, L, diff, nr, ctx.to_device(X), ctx.to_device(Lm), ctx.to_device(VF), capi.ARH_RHS_PLANE, src)
    want = [np.zeros(len(diff)) for _ in range(3)]
    for j in range(nr):
        for w, o in zip(want, oc.shape_grad(k, L, diff, X[j], Lm[j], VF[j], capi.ARH_RHS_PLANE, src[j])):
            w += o
    for a, b in zip(got, want):
        assert rel(a, b) < 1e-11
