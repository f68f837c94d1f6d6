"""The solver's start on the device: zero right-hand sides, right-hand sides that meet the tolerance with x = 0, and
ones that iterate, alone and in one batch. Those that do not iterate return x = 0 after no iteration; the others get
the bits they get alone; no products are counted where nothing iterates."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hmat(ctx, capi):
    from acoustic_reliefs_amd import meshes
    P, E, _ = meshes.relief_config(0.3, 14, 0.05, seed=2)
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=16, factor=1.5)
    return {s: g.assemble(2 * np.pi * 1000.0 / 343.0, 1e-6, storage=s) for s in (0, 1)}


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("zero", [(), (0,), (2,), (0, 1, 2, 3, 4)])
@pytest.mark.parametrize("tol", [1e-7, 2.0])
def test_start(hmat, storage, zero, tol):
    H = hmat[storage]
    rng = np.random.default_rng(7)
    b = rng.standard_normal((5, H.geom.N)) + 1j * rng.standard_normal((5, H.geom.N))
    b[list(zero)] = 0.0
    x, st = H.solve_np(b, tol=tol, hist_cap=4)
    runs = [j for j in range(5) if j not in zero and (tol < 1.0 or storage == 1)]  # mixed: inner tolerance 0.5
    for j in range(5):
        assert (st["iters_per_rhs"][j] > 0) == (j in runs)
        if j not in runs:
            assert np.all(x[j] == 0.0) and st["true_res"][j] == (0.0 if j in zero else 1.0)
    if not runs:
        assert st["matvecs"] == 1  # the true residual
    for j in runs[:2]:
        xj, sj = H.solve_np(b[j:j + 1], tol=tol, hist_cap=4)
        assert np.array_equal(xj[0], x[j])
        assert np.array_equal(sj["hist"][0], st["hist"][j]) and st["hist"][j][0] == 1.0
