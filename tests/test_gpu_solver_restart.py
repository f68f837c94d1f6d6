"""BiCGSTAB's breakdown restarts, which a right-hand side waits for between two products of a batch of iterations, and whole
solves on the generic products (leaves above 128).

The mesh makes a right-hand side break down exactly. One element lies in the plane z = 0 with its centroid at the origin; the
others lie in the planes x = 0 and y = 0. The origin is in all three planes, so every entry of the first element's row is an
exact zero but the -1/2 of its own: with b = c e_1 the first step gives r = s - w t with (r)_1 = 0 exactly, r0^H r = 0 while
|r| is not small. The restart takes r0 = r, whose first component stays 0, and the solve converges on the
rest. The same holds for the complex-FP32 operator."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K = 2 * np.pi * 4000.0 / 343.0


def corner_mesh(n):
    P = [[1 / 32, 0, 0], [-1 / 64, 1 / 64, 0], [-1 / 64, -1 / 64, 0]]
    E = [[0, 1, 2]]
    t = np.linspace(0.05, 0.65, n + 1)
    for plane in (0, 1):
        o = len(P)
        P += [([0.0, u, z] if plane == 0 else [u, 0.0, z]) for z in t for u in t]
        for i in range(n):
            for j in range(n):
                a = o + i * (n + 1) + j
                E += [[a, a + 1, a + n + 2], [a, a + n + 2, a + n + 1]]
    return np.array(P, dtype=np.float64), np.array(E, dtype=np.int32)


@pytest.fixture(scope="module")
def mesh():
    return corner_mesh(24)


@pytest.fixture(scope="module", params=[24, 128, 256])
def geom(request, mesh, ctx, capi):
    g = capi.Geometry.from_mesh(ctx, *mesh, leaf=request.param, factor=1.5)
    c = np.asarray(g.P)[np.asarray(g.E)].mean(axis=1)
    g.first = int(np.argmin(np.abs(c).sum(axis=1)))
    return g


def batch(g, nr):
    rng = np.random.default_rng(nr)
    b = rng.standard_normal((nr, g.N)) + 1j * rng.standard_normal((nr, g.N))
    paused = list(range(1, nr, 3)) if nr > 1 else [0]
    for j in paused:
        b[j] = 0.0
        b[j, g.first] = 1.0 + j
    return b, paused


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("nr", [1, 2, 7, 43])
def test_restarts(geom, storage, nr):
    H = geom.assemble(K, 1e-8, storage=storage)
    b, paused = batch(geom, nr)
    print("restarts: storage=%d nr=%d N=%d, %d low-rank blocks" % (storage, nr, geom.N, len(geom.lowrank)), flush=True)
    row = np.zeros((1, geom.N), complex)
    row[0, geom.first] = 1.0
    for prec in ([0] if storage == 0 else [0, 1]):
        y = H.matvec_np(row, precision=prec)[0]
        assert y[geom.first] == -0.5 and np.count_nonzero(y) > geom.N // 2
    x, st = H.solve_np(b, tol=1e-7, true_residual=True)
    assert st["restarts"] == len(paused)
    assert np.all(st["true_res"] <= 1e-7)
    for j in sorted({0, nr - 1, *paused[:2]}):
        xj, sj = H.solve_np(b[j:j + 1], tol=1e-7, true_residual=True)
        assert np.array_equal(xj[0], x[j])
        assert sj["iters_per_rhs"][0] == st["iters_per_rhs"][j] and sj["restarts"] == (j in paused)


def test_iterations_of_the_oracle(geom, oracle):
    """On the library's own operator as a matrix (the ACA's stopping rule leaves out much of the blocks that hold exact
    zeros). Eigen's counter starts again at the restart; the library's counts all iterations, one more here."""
    H = geom.assemble(K, 1e-10)
    A = H.matvec_np(np.eye(geom.N)).T
    b, _ = batch(geom, 2)
    x, st = H.solve_np(b, tol=1e-6)
    for j in (0, 1):
        xo, it, err, hist = oracle.bicgstab_dense(A, b[j], 1e-6)
        print("column %d: %d iterations, oracle %d" % (j, st["iters_per_rhs"][j], it), flush=True)
        assert abs(st["iters_per_rhs"][j] - (it + j)) <= 1
        assert np.linalg.norm(A @ x[j] - b[j]) <= 2e-6 * np.linalg.norm(b[j])
