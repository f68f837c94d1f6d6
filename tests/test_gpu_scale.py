"""arh_scale: every element of a complex array times a real factor, over and around the grid's first stride; -1 is exact
(the right-hand sides of the solves)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1024 * 256, 1024 * 256 + 3])
def test_scale(ctx, n):
    rng = np.random.default_rng(n)
    a = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    d = ctx.to_device(a)
    ctx.scale(d, -1.0)
    assert np.array_equal(d.numpy(), -a)
    ctx.scale(d, 3.0)
    assert np.array_equal(d.numpy(), -3.0 * a)
