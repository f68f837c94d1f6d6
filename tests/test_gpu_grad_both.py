"""Shape gradient with enough touched elements that their pairs are taken both ways at once: odd and even numbers of
64-element blocks, blocks that are not full, with and without elements that no differentiable vertex touches, against
the oracle. The sums are those of tests/test_gpu_grad_pairs.py over up to 2,618 elements instead of 700: its bound of
1e-11 times four."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup(ctx, capi, oracle):
    from acoustic_reliefs_amd import meshes
    P, E, top = meshes.relief_config(0.6, 32)[:3]
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=32, factor=1.5)
    return g, oracle.Ctx(P, g.E, g.dense, g.lowrank), np.asarray(top)


# differentiable vertices, of the first rows of the top grid (blocks of touched elements); None: every vertex
@pytest.mark.parametrize("nr,rows", [(1, 19), (3, 20), (2, 21), (5, 32), (37, 32), (1, None)])
def test_blocks_vs_oracle(setup, ctx, capi, nr, rows):
    g, oc, top = setup
    rng = np.random.default_rng(nr)
    diff = np.arange(g.V) if rows is None else top[:32 * rows]
    T = int(np.isin(g.E, diff).any(axis=1).sum())
    print("both ways: nr=%d, %d touched of %d, %d blocks" % (nr, T, g.N, (T + 63) // 64), flush=True)
    LL = 33
    L = rng.standard_normal((LL, 3)) * 3.0 + [0.0, 20.0, 0.0]
    k = 2 * np.pi * 1500.0 / 343.0
    X, Lm = (rng.standard_normal((nr, g.N)) + 1j * rng.standard_normal((nr, g.N)) for _ in range(2))
    VF = rng.standard_normal((nr, LL)) + 1j * rng.standard_normal((nr, LL))
    src = rng.standard_normal((nr, 3))
    src /= np.linalg.norm(src, axis=1)[:, None]
    got = g.shape_grad(k, L, diff, nr, ctx.to_device(X), ctx.to_device(Lm), ctx.to_device(VF), capi.ARH_RHS_PLANE, src)
    want = [np.zeros(len(diff)) for _ in range(3)]
    for j in range(nr):
        for w, o in zip(want, oc.shape_grad(k, L, diff, X[j], Lm[j], VF[j], capi.ARH_RHS_PLANE, src[j])):
            w += o
    for a, b in zip(got, want):
        assert rel(a, b) < 4e-11
