"""The solver's fused vector updates at the edges of their tiles: right-hand sides around multiples of the four columns of a workgroup
and the 40 of a product pass, sizes that do not fill the last rows, both precisions, columns that stop at
different iterations. A batch gives every right-hand side the bits it gets alone (the updates of one right-hand side
see nothing of the others), and the true residual meets the tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def geom(ctx, capi):
    from acoustic_reliefs_amd import meshes
    P, E, _ = meshes.relief_config(0.3, 14, 0.05, seed=2)
    return capi.Geometry.from_mesh(ctx, P, E, leaf=16, factor=1.5)


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("nr", [1, 15, 16, 17, 32, 39, 40, 41])
def test_batch_equals_alone(geom, ctx, capi, storage, nr):
    k = 2 * np.pi * 2000.0 / 343.0
    H = geom.assemble(k, 1e-6, storage=storage)
    rng = np.random.default_rng(nr)
    b = rng.standard_normal((nr, geom.N)) + 1j * rng.standard_normal((nr, geom.N))
    b[::3] = -geom.rhs(k, capi.ARH_RHS_PLANE, np.tile([0.6, -0.8, 0.0], (len(b[::3]), 1))).numpy()  # fewer iterations
    print("solver updates storage=%d nr=%d" % (storage, nr), flush=True)
    x, st = H.solve_np(b, tol=1e-8, true_residual=True)
    assert np.all(st["true_res"] <= 1e-8)
    for j in sorted({0, 1 % nr, nr - 1}):
        xj, sj = H.solve_np(b[j:j + 1], tol=1e-8, true_residual=True)
        assert np.array_equal(xj[0], x[j])
        assert sj["iters_per_rhs"][0] == st["iters_per_rhs"][j]
