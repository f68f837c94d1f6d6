"""The listener term of the shape gradient against 80-bit arithmetic. Far from the surface the error is that of the phase
k r: the roundings of the coordinates' differences, of r and of the product, each of 2^-53, times k r (up to 2,900 here).
Plain double precision with a correctly rounded root makes the same roundings, so its own error on the same inputs is the
measure: the kernel's may not be larger than that by more than a tenth (both are sums over 61 listeners x 6 points of errors
that are independent, so their norms over 256 vertices scatter by a few percent)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RULE = [(w, a, b) for w, p, q in ((0.223381589678011, 0.445948490915965, 0.108103018168070),
                                  (0.109951743655322, 0.091576213509771, 0.816847572980459))
        for a, b in ((p, q), (p, p), (q, p))]


def listener_term(real, P, E, diff, k, L, X, VF):
    """A by its definition (Q = 1/2 sum w F s, F = e^{-ikr} (-1 - ikr) / (4 pi r^3), s = -(d . n)) in the given precision."""
    one = np.ones(1, real)[0]
    pi = one * 4 * np.arctan(one)
    P, L, k = P.astype(real), L.astype(real), one * k
    a, b, c = (P[E[:, j]][:, None] for j in range(3))
    u, v = b - a, c - a
    n = np.cross(u, v)
    up = np.array([0, 1, 0], real)
    dn = [np.cross(up, b - c), np.cross(up, v), np.cross(u, up)]
    dQ = [0, 0, 0]
    for w, xi, eta in RULE:
        w, xi, eta = one * w, one * xi, one * eta
        d = L[None] - (a + xi * u + eta * v)
        r = np.sqrt((d * d).sum(axis=-1))
        e = np.cos(k * r) - 1j * np.sin(k * r)
        F = e * (-1 - 1j * k * r) / (4 * pi * r ** 3)
        H = e * (-k * k / r ** 2 + 3 * (1 + 1j * k * r) / r ** 4) / (4 * pi)
        s = -(d * n).sum(axis=-1)
        for j, beta in enumerate((1 - xi - eta, xi, eta)):
            dQ[j] = dQ[j] + w / 2 * (-H * beta * d[..., 1] * s / r + F * (beta * n[..., 1] - (d * dn[j]).sum(axis=-1)))
    slot = np.full(len(P), -1)
    slot[diff] = np.arange(len(diff))
    A = np.zeros(len(diff), real)
    for j in range(3):
        t = sum((x * (dQ[j] @ f)).real for x, f in zip(X, VF))
        on = slot[E[:, j]] >= 0
        np.add.at(A, slot[E[:, j]][on], t[on])
    return A


@pytest.mark.parametrize("f,radius,nr", [(1000.0, 50.0, 1), (3150.0, 50.0, 1), (4000.0, 5.0, 3)])
def test_listener_term(ctx, capi, f, radius, nr):
    from acoustic_reliefs_amd import meshes
    P, E, top = meshes.relief_config(0.6, 16)
    g = capi.Geometry.from_mesh(ctx, P, E, leaf=32, factor=1.5)
    P, E, top, k = np.asarray(g.P), np.asarray(g.E), np.asarray(top), 2 * np.pi * f / 343.0
    L = meshes.semicircle_receivers(radius, 61)
    rng = np.random.default_rng(int(f) + nr)
    X, Lm = (rng.standard_normal((nr, g.N)) + 1j * rng.standard_normal((nr, g.N)) for _ in range(2))
    VF = rng.standard_normal((nr, 61)) + 1j * rng.standard_normal((nr, 61))
    src = np.tile([0.0, -1.0, 0.0], (nr, 1))
    A = g.shape_grad(k, L, top, nr, ctx.to_device(X), ctx.to_device(Lm), ctx.to_device(VF), capi.ARH_RHS_PLANE, src)[0]
    exact = listener_term(np.longdouble, P, E, top, k, L, X, VF)
    plain = listener_term(np.float64, P, E, top, k, L, X, VF)
    err, own = (float(np.linalg.norm((v - exact).astype(float)) / np.linalg.norm(exact.astype(float))) for v in (A, plain))
    print("listener term f=%g radius=%g: error %.3e, plain double %.3e" % (f, radius, err, own), flush=True)
    assert err <= 1.1 * own
