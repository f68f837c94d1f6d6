"""The room a mixed assembly takes: the ACA scratch is free again when the FP32 layout is built. With ranks of at most 6 the
layout's panels (24 MB) fit a freed scratch block (28 MB; the device memory cache hands out blocks of up to a quarter more
than the request), so an assembly that starts from an empty cache leaves less there than the scratch was; with scratch
and layout side by side it leaves all of it."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRANULE = 2 << 20  # of the cache's blocks above 1 MiB


def granules(n):
    return (n + GRANULE - 1) // GRANULE * GRANULE


def test_layout_takes_the_scratch(ctx, capi):
    from acoustic_reliefs_amd import meshes
    P, E = meshes.icosphere(4, 0.5)
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=32, factor=1.5)
    k, max_rank = 2 * np.pi * 500.0 / 343.0, 6
    low = np.asarray(g.lowrank, dtype=np.int64)
    m, n = low[:, 1] - low[:, 0], low[:, 3] - low[:, 2]
    lim = np.minimum(max_rank, np.minimum(m, n) - 1)
    us, vs = (granules(16 * int((lim * x).sum())) for x in (m, n))
    H = g.assemble(k, 1e-13, max_rank, capi.ARH_MIXED)
    assert np.array_equal(H.ranks(), lim)
    del H
    gc.collect()  # what earlier tests left
    ctx.synchronize()
    capi.device_trim(0)
    assert capi.device_cached(0) == 0
    H = g.assemble(k, 1e-13, max_rank, capi.ARH_MIXED)
    left = capi.device_cached(0)
    print("FP32 layout %.1f MB, scratch %.1f + %.1f MB, cached after the assembly %.1f MB"
          % (H.info()["bytes_fp32"] / 1e6, us / 1e6, vs / 1e6, left / 1e6), flush=True)
    assert left < us + vs
