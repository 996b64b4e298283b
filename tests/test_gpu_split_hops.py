"""One wavefront per hop (launches of few sites) against the one-site kernels:
the same bits, on partial tiles, extents of 2, batches and every precision."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

THETA = (np.pi, 0.3, -0.5, 0.7)
PRECS = ["f64", "f32", "f16"]


@pytest.mark.parametrize("L", [(2, 2, 2, 2), (6, 3, 5, 3), (8, 4, 4, 4), (10, 2, 7, 11)])
@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("nrhs", [1, 3])
def test_dslash_matches_forced_traversal(gpu, L, prec, nrhs):
    Q = gpu
    lat = Q.Lattice(L, THETA)
    u = Q.gauge_generate(L, 0.4, 71)
    psi = [Q.spinor_gaussian(L, 72 + r) for r in range(nrhs)]
    p = Q.PREC[prec]
    g = Q.Gauge(lat, p)
    Q.convert(g, Q.Gauge(lat).upload(u))
    x, y = Q.Spinor(lat, p, nrhs), Q.Spinor(lat, p, nrhs)
    for r in range(nrhs):
        x.upload(psi[r], rhs=r)
    for op in (Q.OP_D, Q.OP_Q):
        Q.dslash_tune(y, x, g)   # launches of this size take one wavefront per hop
        Q.dslash(y, x, g, 0.1, 0.07, op)
        got = [y.download(r) for r in range(nrhs)]
        Q.dslash_set_config(x, g, 2 | (1 << 8), 0)   # one site per lane
        Q.dslash(y, x, g, 0.1, 0.07, op)
        for r in range(nrhs):
            assert np.array_equal(got[r], y.download(r))
            if prec == "f64":
                ref = (O.qtm if op == Q.OP_Q else O.dslash)(O.Geometry(L, THETA), psi[r], u, 0.1, 0.07)
                assert np.linalg.norm(got[r] - ref) <= 1e-13 * np.linalg.norm(ref)


@pytest.mark.parametrize("L", [(4, 2, 2, 2), (8, 4, 6, 4), (12, 6, 6, 6)])
@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("nrhs", [1, 2, 5])
def test_schur_matches_one_site_kernels(gpu, L, prec, nrhs):
    Q = gpu
    lat, half = Q.Lattice(L, THETA), Q.Lattice((L[0] // 2,) + L[1:])
    p = Q.PREC[prec]
    g = Q.Gauge(lat, p)
    Q.convert(g, Q.Gauge(lat).upload(Q.gauge_generate(L, 0.4, 73)))
    x, y = Q.Spinor(half, p, nrhs), Q.Spinor(half, p, nrhs)
    for r in range(nrhs):
        x.upload(Q.spinor_gaussian(half.L, 74 + r), rhs=r)
    out = []
    try:
        for zlen in (0, 1):
            Q.eo_set_zlen(zlen)
            Q.dslash_schur(y, x, g, 0.1, 0.07)
            out.append([y.download(r) for r in range(nrhs)])
    finally:
        Q.eo_set_zlen(0)
    for a, b in zip(*out):
        assert np.array_equal(a, b)
