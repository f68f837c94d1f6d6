"""Products with few right-hand sides, whose packed rows hold exactly that many values (1 to 4), against those with more
(rows of whole tiles): the columns of a product are independent, so every right-hand side gets the same bits, in both
precisions, both directions and every leaf class (2, 4 and 8 row tiles)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaf", [16, 64, 128])
@pytest.mark.parametrize("transpose", [False, True])
def test_narrow_products_equal_wide(ctx, capi, small_relief, leaf, transpose):
    P, E, _ = small_relief
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=leaf, factor=1.5)
    H = g.assemble(2 * np.pi * 1500.0 / 343.0, 1e-5, storage=capi.ARH_MIXED)
    rng = np.random.default_rng(leaf)
    x = rng.standard_normal((11, g.N)) + 1j * rng.standard_normal((11, g.N))
    for precision in (capi.ARH_FP64, capi.ARH_MIXED):
        want = H.matvec_np(x, transpose=transpose, precision=precision)
        for r in (1, 2, 3, 4, 5, 8, 9):
            print("narrow leaf=%d precision=%d nr=%d" % (leaf, precision, r), flush=True)
            got = H.matvec_np(x[:r], transpose=transpose, precision=precision)
            assert np.array_equal(got, want[:r])
