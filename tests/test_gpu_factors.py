"""The factors of low-rank blocks by block: the same whichever block is read first and in whatever order, and for a copy
of the operator read from two threads at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_any_order(ctx, capi):
    from acoustic_reliefs_amd import meshes
    P, E, _ = meshes.relief_config(0.3, 14, 0.05, seed=2)
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=16, factor=1.5)
    n = len(g.lowrank)
    H = [g.assemble(2 * np.pi * 1000.0 / 343.0, 1e-5) for _ in range(3)]
    want = [H[0].factors(a) for a in range(n)]

    def same(a, f):
        return all(np.array_equal(x, y) for x, y in zip(want[a], f))

    assert all(same(a, H[1].factors(a)) for a in reversed(range(n)))
    got = [None] * n

    def read(first):
        for a in range(first, n, 2):
            got[a] = H[2].factors(a)

    threads = [threading.Thread(target=read, args=(first,)) for first in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(same(a, f) for a, f in enumerate(got))
