"""Block ACA over the size classes of its kernel: up to 64 x 64 (one wavefront, entries shared by 3, 2 or 1 lanes:
edges at 21, 32 and 64), one wavefront looping, a workgroup, ranks over one batch of eight stored crosses, single
rows. The stopping rule bounds the last cross by tol times the block's norm estimate, so each block is within 30 tol
of the exact one (the bound of the oracle's own check); ranks follow the oracle's to +-2 (pivots at near-ties)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def far_patches(m, n):
    """Two patches of m and n small triangles, a few sizes apart: one admissible block each way."""
    rng = np.random.default_rng(m * 1000 + n)
    P, E = [], []
    for count, x0 in ((m, 0.0), (n, 1.0)):
        c = rng.uniform(0.0, 0.25, (count, 3)) + [x0, 0.0, 0.0]
        for p in c:
            t = p + rng.uniform(-0.01, 0.01, (3, 3))
            E.append([len(P), len(P) + 1, len(P) + 2])
            P += list(t)
    return np.array(P), np.array(E, dtype=np.int32)


@pytest.mark.parametrize("m,n", [(1, 7), (2, 2), (20, 21), (21, 22), (31, 33), (32, 32), (64, 64), (63, 65), (65, 21),
                                 (130, 64), (200, 255), (256, 256), (300, 400)])
@pytest.mark.parametrize("tol", [1e-3, 1e-8])
def test_blocks_of_every_class(ctx, capi, oracle, m, n, tol):
    P, E = far_patches(m, n)
    N = m + n
    k = 40.0
    print("aca m=%d n=%d tol=%g" % (m, n, tol), flush=True)
    dense = np.array([[0, m, 0, m], [m, N, m, N]], np.int32)
    low = np.array([[0, m, m, N], [m, N, 0, m]], np.int32)
    g = capi.Geometry(ctx, P, E, dense, low)
    H = g.assemble(k, tol)
    oc = oracle.Ctx(P, E, dense, low)
    A = oc.dense_matrix(k)
    oc.assemble(k, tol)
    for a, (rs, re, cs, ce) in enumerate(low):
        U, V = H.factors(a)
        B = A[rs:re, cs:ce]
        lim = min(100, re - rs - 1, ce - cs - 1)
        rank = H.ranks()[a]
        assert U.shape[1] <= rank <= max(lim, 0)
        assert abs(int(rank) - int(oc.ranks()[a])) <= 2
        if 0 < rank < lim:  # stopped by the rule
            assert np.linalg.norm(B - U @ V) <= 30 * tol * np.linalg.norm(B)
