"""What one GCR cycle (max_outer = 1) leaves of the residual."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

EPS = 0.3


def _source(L, point):
    return O.point_source(L, (1, 0, 1, 1), 1, 2) if point else O.spinor_gaussian(L, 62)


def _one_cycle(Q, L, b, kappa, mu, op, eo, prec, n, seed=61):
    lat = Q.Lattice(L)
    g = Q.Gauge(lat).upload(O.gauge_generate(L, EPS, seed))
    fb, fx = Q.Spinor(lat).upload(b), Q.Spinor(lat)
    S = Q.Solver(lat, g, n_restart=n, tol=1e-15, inner_prec=prec, op=op, eo=eo, max_outer=1)
    r = S.solve(fx, fb, kappa, mu, check=False)
    S.close()
    assert r["rc"] in (0, 6) and r["outer"] == 1
    return r["relres"]


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
@pytest.mark.parametrize("op", ["Q", "D"])
@pytest.mark.parametrize("L", [(6, 3, 5, 3), (8, 6, 4, 6), (16, 8, 8, 8)])
@pytest.mark.parametrize("kappa,mu", [(0.12, 0.0), (0.12, 0.04), (0.139, 0.0)])
def test_longer_cycles_reach_no_less(gpu, prec, op, L, kappa, mu):
    """A block of steps that is too long is left out, the last one of a cycle
    too: |res| stays within twice the smallest of any shorter cycle."""
    Q = gpu
    b = _source(L, True)
    least = 1.0
    for n in (8, 16, 24, 28, 32, 36, 40, 44, 48, 56, 64):
        r = _one_cycle(Q, L, b, kappa, mu, op, 0, prec, n)
        assert r <= 2.0 * least
        least = min(least, r)


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
@pytest.mark.parametrize("links,kappa", [(1.0, 1e-5), (1e-8, 0.12), (0.0, 0.12)])
@pytest.mark.parametrize("point", [0, 1])
def test_residual_of_zero_ends_the_cycle(gpu, prec, links, kappa, point):
    """Local operators, but for little: a few steps, or none for an even point
    source, leave a residual that is stored as exactly 0."""
    Q = gpu
    L = (8, 6, 4, 6)
    lat, u = Q.Lattice(L), links * O.gauge_generate(L, EPS, 61)
    b = O.point_source(L, (0, 0, 0, 0), 1, 2) if point else _source(L, 0)
    for eo in (0, 1):
        for n in (4, 12, 32):
            fb, fx = Q.Spinor(lat).upload(b), Q.Spinor(lat)
            S = Q.Solver(lat, Q.Gauge(lat).upload(u), n_restart=n, tol=1e-10, inner_prec=prec, op="D", eo=eo, max_outer=20)
            S.solve(fx, fb, kappa)
            assert O.b_minus_Dx(O.Geometry(L), fx.download(), b, u, kappa) <= 1e-10


@pytest.mark.parametrize("prec", ["f32", "f16"])
@pytest.mark.parametrize("op,eo,kappa,mu,links,n", [("Q", 0, 1e-12, 0.0, 1.0, 4), ("D", 0, 0.12, 1e10, 1.0, 4),
                                                    ("D", 1, 0.12, 1e10, 1.0, 4), ("Q", 0, 0.12, 0.0, 1e6, 32)])
@pytest.mark.parametrize("graph", [0, 1])
def test_operators_of_large_norm(gpu, prec, op, eo, kappa, mu, links, n, graph):
    """Powers of the operator leave the range of FP32: solved in single steps.
    The solver then does an ordinary solve as a new one does."""
    Q = gpu
    if prec == "f16" and links > 6e4:
        pytest.skip("FP16 links end at 65504")
    L = (8, 6, 4, 6)
    lat, u, b = Q.Lattice(L), O.gauge_generate(L, EPS, 61), _source(L, 0)
    fb, fx, fy = Q.Spinor(lat).upload(b), Q.Spinor(lat), Q.Spinor(lat)
    kw = dict(n_restart=n, tol=1e-10, inner_prec=prec, op=op, eo=eo, max_outer=100, graph=graph)
    g, big = Q.Gauge(lat).upload(u), Q.Gauge(lat).upload(links * u)
    S = Q.Solver(lat, big, **kw)
    for _ in range(2):
        S.solve(fx, fb, kappa, mu)
        assert O.b_minus_Dx(O.Geometry(L), fx.download(), b, links * u, kappa, mu) <= 1e-10
    S.set_gauge(g)
    r = S.solve(fx, fb, 0.05, 0.03)
    assert r == {**Q.Solver(lat, g, **kw).solve(fy, fb, 0.05, 0.03), "seconds": r["seconds"]}
    assert np.array_equal(fx.download(), fy.download())
