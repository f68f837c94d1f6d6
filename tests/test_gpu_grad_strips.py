"""Shape gradient with more touched elements than one strip of partial sums holds. A vertex's gradient depends on its own
elements alone, so calls for a few vertices at a time, whose pairs are taken one way, give the same numbers: sums of the
same terms in another order and by another formula. A term is good to about 1e-14 of its largest factor (tests/
test_gpu_grad_pairs.py has 1e-11 for sums over 700 elements, dominated by the neighbours' near-cancelling terms, and the
rounding of a sum grows like the root of its length): 1e-10 of the gradient's norm for 22,000. The partial sums stay within
their strip: less than 96 MB in the device memory cache after a call that starts from an empty one."""
import gc

import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,grid", [(1, 88), (3, 96)])
def test_strips_against_subsets(ctx, capi, nr, grid):
    from acoustic_reliefs_amd import meshes
    P, E, top = meshes.relief_config(0.9, grid, 0.15)[:3]
    top = np.asarray(top)
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=64, factor=1.5)
    T = int(np.isin(g.E, top).any(axis=1).sum())
    print("strips: nr=%d, %d touched of %d, %d blocks" % (nr, T, g.N, (T + 63) // 64), flush=True)
    assert 48 * T * ((T + 63) // 64 // 2 + 1) > 64 << 20
    rng = np.random.default_rng(nr)
    LL = 19
    L = rng.standard_normal((LL, 3)) * 3.0 + [0.0, 20.0, 0.0]
    k = 2 * np.pi * 1000.0 / 343.0
    X, Lm, VF = (ctx.to_device(rng.standard_normal((nr, n)) + 1j * rng.standard_normal((nr, n))) for n in (g.N, g.N, LL))
    src = rng.standard_normal((nr, 3))
    src /= np.linalg.norm(src, axis=1)[:, None]

    def grad(diff):
        return np.stack(g.shape_grad(k, L, diff, nr, X, Lm, VF, capi.ARH_RHS_PLANE, src))

    gc.collect()  # what earlier tests left
    ctx.synchronize()
    capi.device_trim(0)
    full = grad(top)
    left = capi.device_cached(0)
    print("cached after the call: %.1f MB" % (left / 1e6), flush=True)
    assert left < 96e6
    # the first, the last and some in between, a few hundred touched elements each
    for i0 in (0, len(top) // 3, len(top) // 2, len(top) - 100):
        part = grad(top[i0:i0 + 100])
        for a, b in zip(full[:, i0:i0 + 100], part):
            assert rel(a, b) < 1e-10
    assert np.array_equal(full, grad(top))
