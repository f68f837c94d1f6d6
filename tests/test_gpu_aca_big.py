"""Big ACA blocks beside small ones: a few big blocks take more wavefronts each than many do, on a stream beside the
small blocks' one. A block's crosses depend on its own entries alone, so the factors of a pair of patches are the same
bits in a small and in a large crowd, run after run, and they approximate the block as the stopping rule promises."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def patches(sizes):
    P, E = [], []
    for a, count in enumerate(sizes):
        rng = np.random.default_rng(a)
        for p in rng.uniform(0.0, 0.25, (count, 3)) + [float(a), 0.0, 0.0]:
            E.append([len(P), len(P) + 1, len(P) + 2])
            P += list(p + rng.uniform(-0.01, 0.01, (3, 3)))
    o = np.concatenate([[0], np.cumsum(sizes)])
    pairs = [(i, j) for i in range(len(sizes)) for j in range(len(sizes)) if i != j]
    dense = np.array([[o[i], o[i + 1], o[i], o[i + 1]] for i in range(len(sizes))], np.int32)
    low = np.array([[o[i], o[i + 1], o[j], o[j + 1]] for i, j in pairs], np.int32)
    return np.array(P), np.array(E, dtype=np.int32), dense, low, pairs


def test_few_and_many(ctx, capi, oracle):
    tol, k = 1e-6, 20.0
    got = {}
    for big in (3, 17):  # 6 and 272 blocks of 261 + 257 rows and columns and more
        sizes = [261, 257, 300] + [260] * (big - 3) + [40, 9, 70]
        P, E, dense, low, pairs = patches(sizes)
        print("big ACA blocks: %d of %d" % (big * (big - 1), len(low)), flush=True)
        g = capi.Geometry(ctx, P, E, dense, low)
        for _ in range(3):
            H = g.assemble(k, tol)
            f = {p: H.factors(a) for a, p in enumerate(pairs) if max(p) < 3}
            for p, (U, V) in f.items():
                u, v = got.setdefault(p, (U, V))
                assert np.array_equal(U, u) and np.array_equal(V, v)
        if big == 3:
            A = oracle.Ctx(P, E, dense, low).dense_matrix(k)
            for a, (rs, re, cs, ce) in enumerate(low):
                U, V = H.factors(a)
                B = A[rs:re, cs:ce]
                if 0 < H.ranks()[a] < min(100, re - rs - 1, ce - cs - 1):  # stopped by the rule
                    assert np.linalg.norm(B - U @ V) <= 30 * tol * np.linalg.norm(B)
