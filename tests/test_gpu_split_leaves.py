"""Narrow products of leaves that are split over many tasks (one, a few, more than the eight tiles of a summing batch):
the task that happens to finish last sums the tiles in task order, so repeated products give the same bits, and those
of the wide product, whose tiles a kernel of its own sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,leaf,all_dense", [(8, 16, False), (32, 32, False), (32, 128, True), (32, 40, True)])
def test_split_leaves(ctx, capi, grid, leaf, all_dense):
    from acoustic_reliefs_amd import meshes
    P, E = meshes.relief_config(0.6, grid)[:2]
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=leaf, factor=1.5, all_dense=all_dense)
    H = g.assemble(2 * np.pi * 1000.0 / 343.0, 1e-5, storage=capi.ARH_MIXED)
    rng = np.random.default_rng(grid)
    x = rng.standard_normal((5, g.N)) + 1j * rng.standard_normal((5, g.N))
    print("split leaves grid=%d leaf=%d" % (grid, leaf), flush=True)
    for precision in (capi.ARH_FP64, capi.ARH_MIXED):
        for tr in (False, True):
            want = H.matvec_np(x, transpose=tr, precision=precision)
            for r in (1, 2, 3, 4, 1, 4, 2) * 3:
                assert np.array_equal(H.matvec_np(x[:r], transpose=tr, precision=precision), want[:r])
