"""What the device makes of the ACA's ranks: factor offsets over more and fewer than the 1024 blocks of a workgroup, ranks
of zero, stacks and panel columns. The products equal those of the stored blocks, in both directions (FP64: rounding,
1e-12; the complex-FP32 copy: 2e-6), and the totals are the sums over the blocks. A NaN in a dense block is still an
error, and the geometry's next operator is right."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _product(h, x, transpose):
    y = -0.5 * x
    blocks = [(r, h.dense_block(b), None) for b, r in enumerate(h.geom.dense)]
    blocks += [(r,) + h.factors(a) for a, r in enumerate(h.geom.lowrank)]
    for (rs, re, cs, ce), A, B in blocks:
        i, o = (slice(rs, re), slice(cs, ce)) if transpose else (slice(cs, ce), slice(rs, re))
        f = [A] if B is None else [A, B]
        v = x[i]
        for m in ([m.T for m in f] if transpose else f[::-1]):
            v = m @ v
        y[o] += v
    return y


@pytest.fixture(scope="module")
def geoms(ctx, capi):
    from acoustic_reliefs_amd import meshes
    P, E, _ = meshes.relief_config(0.3, 14, 0.05, seed=2)
    return {leaf: capi.Geometry.from_mesh(ctx, P, E, leaf=leaf, factor=1.5) for leaf in (4, 16, 40)}


@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("max_rank", [0, 1, 2, 100])
@pytest.mark.parametrize("leaf", [4, 16, 40])
def test_lists(geoms, leaf, max_rank, storage):
    g = geoms[leaf]
    H = g.assemble(2 * np.pi * 2000.0 / 343.0, 1e-5, max_rank=max_rank, storage=storage)
    rng = np.random.default_rng(leaf + max_rank)
    x = rng.standard_normal(g.N) + 1j * rng.standard_normal(g.N)
    print("block lists leaf=%d max_rank=%d storage=%d: %d blocks" % (leaf, max_rank, storage, len(g.lowrank)), flush=True)
    info = H.info()
    assert info["sum_rank"] == sum(H.factors(a)[0].shape[1] for a in range(len(g.lowrank)))
    assert info["max_rank"] == H.ranks().max() <= max_rank
    for tr in (False, True):
        ref = _product(H, x, tr)
        for prec in ([0] if storage == 0 else [0, 1]):
            y = H.matvec_np(x, transpose=tr, precision=prec)
            assert np.linalg.norm(y - ref) <= (1e-12 if prec == 0 else 2e-6) * np.linalg.norm(ref)


def test_block_counts(geoms):
    n = sorted(len(g.lowrank) for g in geoms.values())
    assert 0 < n[0] < 1024 and n[-1] > 2048


def test_nan_in_a_dense_block(ctx, capi, geoms):
    g0 = geoms[16]
    E = np.array(g0.E)
    E[1] = E[1, 0]  # an element of no extent: its collocation point is its quadrature points, r = 0
    g = capi.Geometry(ctx, g0.P, E, g0.dense, g0.lowrank)
    for storage in (0, 1):
        with pytest.raises(Exception, match="NaN in a dense"):
            g.assemble(20.0, 1e-4, storage=storage)
    x = np.ones(g0.N, complex)
    a, b = (g0.assemble(20.0, 1e-4).matvec_np(x) for _ in range(2))
    assert np.array_equal(a, b)
