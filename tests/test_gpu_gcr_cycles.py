"""What one GCR cycle (max_outer = 1) leaves of the residual, also against the
smallest residual of its Krylov space, which Arnoldi's process finds on the CPU,
one step after another, with the oracle's operator."""
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


@pytest.mark.parametrize("op,eo,kappa,mu,links,n,prec", [
    ("Q", 0, 1e-12, 0.0, 1.0, 4, "f32"), ("Q", 0, 1e-12, 0.0, 1.0, 4, "f16"),
    ("D", 0, 0.12, 1e10, 1.0, 4, "f32"), ("D", 0, 0.12, 1e10, 1.0, 4, "f16"),
    ("D", 1, 0.12, 1e10, 1.0, 4, "f32"), ("D", 1, 0.12, 1e10, 1.0, 4, "f16"),
    ("Q", 0, 0.12, 0.0, 1e6, 32, "f32")])   # (FP16 links end at 65504)
@pytest.mark.parametrize("graph", [0, 1])
def test_operators_of_large_norm(gpu, prec, op, eo, kappa, mu, links, n, graph):
    """Powers of the operator leave the range of FP32: solved in single steps.
    The solver then does an ordinary solve as a new one does."""
    Q = gpu
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


def _schur(geo, u, m, mu, b):
    """D^ v = D_oo v - D_oe D_ee^-1 D_eo v and its source, on full vectors whose even sites are 0."""
    t, x, y, z = np.unravel_index(np.arange(geo.V), geo.L, order="F")
    odd = ((t + x + y + z) % 2 == 1)[:, None, None]
    diag = (m + 4.0) + 1j * mu * np.array([1.0, 1.0, -1.0, -1.0])[None, :, None]

    def D(v):
        return O.dslash(geo, np.ascontiguousarray(v), u, m, mu)

    assert np.abs(np.where(odd, D(np.where(odd, b, 0)) - diag * b, 0)).max() <= 1e-12 * np.abs(b).max()
    even = lambda v: np.where(odd, 0, v / diag)
    return (lambda v: np.where(odd, D(v) - D(even(D(v))), 0)), np.where(odd, b - D(even(b)), 0)


_reference = {}


def _least_residuals(L, op, eo, kappa, mu, point, n):
    """|b - D x| / |b| after 0 .. n steps of minimal residual."""
    key = (L, op, eo, kappa, mu, point)
    if key not in _reference:
        geo, u, b, m = O.Geometry(L), O.gauge_generate(L, EPS, 61), _source(L, point), 1 / (2 * kappa) - 4
        if eo:
            A, r = _schur(geo, u, m, mu, b)
        elif op == "Q":
            A, r = (lambda v: O.qtm(geo, v, u, m, mu)), b * np.array([1j, 1j, -1j, -1j])[None, :, None]
        else:
            A, r = (lambda v: O.dslash(geo, v, u, m, mu)), b
        V, H, e = [r / np.linalg.norm(r)], np.zeros((n + 1, n), complex), np.eye(n + 1)[0]
        res = [1.0]
        for j in range(n):
            w = A(V[j])
            for _ in range(2):
                for i in range(j + 1):
                    h = np.vdot(V[i], w)
                    H[i, j] += h
                    w = w - h * V[i]
            H[j + 1, j] = np.linalg.norm(w)
            V.append(w / H[j + 1, j])
            Hj = H[:j + 2, :j + 1]
            res.append(np.linalg.norm(e[:j + 2] - Hj @ np.linalg.lstsq(Hj, e[:j + 2], rcond=None)[0]))
        _reference[key] = np.array(res) * np.linalg.norm(r) / np.linalg.norm(b)
    return _reference[key]


@pytest.mark.parametrize("prec,eps", [("f64", 2.0**-53), ("f32", 2.0**-24), ("f16", 2.0**-11)])
@pytest.mark.parametrize("op,eo,kappa,mu", [("D", 0, 0.12, 0.0), ("D", 0, 0.12, 0.04), ("D", 1, 0.12, 0.0),
                                            ("D", 1, 0.139, 0.04), ("Q", 0, 0.12, 0.0), ("Q", 0, 0.12, 0.04),
                                            ("Q", 0, 0.139, 0.0)])
@pytest.mark.parametrize("point", [0, 1])
def test_a_cycle_reaches_the_least_residual(gpu, prec, eps, op, eo, kappa, mu, point):
    """No direction is lost, in blocks of 8, 4, 2 and 1 and from one to the next:
    2% are less than what one step takes off.  The stored w_k, off by eps of
    themselves, leave eps |res_k| each, four times that through the basis of a
    block.  (FP16 cycles of Q beyond 27 steps, and FP32 ones beyond 40, lose their
    orthogonality.)"""
    Q = gpu
    L = (8, 6, 4, 6)
    b = _source(L, point)
    for n in (1, 2, 3, 5, 8, 13, 16, 27, 40, 64):
        if (prec == "f16" and op == "Q" and n > 27) or (prec == "f32" and op == "Q" and n > 40):
            continue
        ref = _least_residuals(L, op, eo, kappa, mu, point, 64)
        r = _one_cycle(Q, L, b, kappa, mu, op, eo, prec, n)
        assert r <= 1.02 * ref[n] + 4 * eps * np.sqrt((ref[:n]**2).sum()) + 1e-15
        assert r >= 0.98 * ref[n] - 2 * eps - 1e-15   # (1e-15: the reference's own rounding)


# 12 288 sites, the longest short vectors of FP32 and FP64, and longer ones whose
# last tile has 60, 58, 4 and (half lattice) 56 of 64 sites
@pytest.mark.parametrize("L,op,eo", [((16, 16, 6, 8), "D", 0), ((14, 21, 6, 7), "D", 0), ((15, 13, 9, 14), "Q", 0),
                                     ((30, 21, 18, 11), "D", 0), ((10, 6, 14, 30), "D", 1)])
@pytest.mark.parametrize("prec,eps", [("f64", 2.0**-53), ("f32", 2.0**-24), ("f16", 2.0**-11)])
def test_long_vectors_with_partial_tiles(gpu, L, op, eo, prec, eps):
    """Blocks of 8 (FP16: 4), 4, 2 and 1: the least residual, and the same bits
    alone and in a batch."""
    Q = gpu
    kappa, mu, n = 0.12, 0.04, 15
    lat, g = Q.Lattice(L), Q.Gauge(Q.Lattice(L)).upload(O.gauge_generate(L, EPS, 61))
    b = [_source(L, 0), O.spinor_gaussian(L, 63)]
    fb, sols = Q.Spinor(lat, nrhs=2), []
    for r in range(2):
        fb.upload(b[r], rhs=r)
    # (a tuned FP16 batch may take the matrix cores, which round differently)
    Q.dslash_set_config(Q.Spinor(lat, Q.PREC[prec]), Q.Gauge(lat, Q.PREC[prec]), 2 | (4 << 8), 0)
    for batch in (1, 2):
        fx = Q.Spinor(lat, nrhs=2)
        S = Q.Solver(lat, g, n_restart=n, tol=1e-15, inner_prec=prec, op=op, eo=eo, max_outer=1, batch=batch)
        S.solve(fx, fb, kappa, mu, check=False)
        S.close()
        sols.append([fx.download(r) for r in range(2)])
    for r in range(2):
        assert np.array_equal(sols[0][r], sols[1][r])
    ref = _least_residuals(L, op, eo, kappa, mu, 0, n)
    res = O.b_minus_Dx(O.Geometry(L), sols[0][0], b[0], O.gauge_generate(L, EPS, 61), kappa, mu)
    assert res <= 1.02 * ref[n] + 4 * eps * np.sqrt((ref[:n]**2).sum()) + 1e-15
    assert res >= 0.98 * ref[n] - 2 * eps
