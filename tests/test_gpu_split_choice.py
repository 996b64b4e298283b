"""One wavefront per hop, forced (traversal 7), against the one-site kernels, and
which launches take it."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

THETA = (np.pi, 0.3, -0.5, 0.7)
SPLIT, ONE_SITE = 7, 2 | (1 << 8)


# less than a tile, 2 sites of the last one, a few, whole tiles
@pytest.mark.parametrize("L", [(2, 2, 2, 2), (2, 3, 3, 25), (6, 3, 5, 3), (10, 2, 7, 11), (8, 4, 4, 4)])
@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
@pytest.mark.parametrize("nrhs", [1, 4, 6])   # row groups of 4, with and without a rest
def test_forced_split_matches_one_site_kernels(gpu, L, prec, nrhs):
    Q = gpu
    lat, p = Q.Lattice(L, THETA), Q.PREC[prec]
    u = Q.gauge_generate(L, 0.4, 71)
    psi = [Q.spinor_gaussian(L, 72 + r) for r in range(nrhs)]
    g = Q.Gauge(lat, p)
    Q.convert(g, Q.Gauge(lat).upload(u))
    x, y = Q.Spinor(lat, p, nrhs), Q.Spinor(lat, p, nrhs)
    for r in range(nrhs):
        x.upload(psi[r], rhs=r)
    for op in (Q.OP_D, Q.OP_Q):
        out = []
        for cfg in (SPLIT, ONE_SITE):
            Q.dslash_set_config(x, g, cfg, 0)
            assert Q.dslash_chosen(x, g, nrhs) == cfg
            Q.dslash(y, x, g, 0.1, 0.07, op)
            out.append([y.download(r) for r in range(nrhs)])
        for r in range(nrhs):
            assert np.array_equal(out[0][r], out[1][r])
        if prec == "f64":
            ref = (O.qtm if op == Q.OP_Q else O.dslash)(O.Geometry(L, THETA), psi[-1], u, 0.1, 0.07)
            assert np.linalg.norm(out[0][-1] - ref) <= 1e-13 * np.linalg.norm(ref)


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
def test_batches_of_a_lattice_tuned_on_one_rhs(gpu, prec):
    """Up to 4 rhs, as for batches that were timed: more were slower."""
    Q = gpu
    L = (8, 4, 6, 4)
    lat, p = Q.Lattice(L), Q.PREC[prec]
    g = Q.Gauge(lat, p)
    x, y = Q.Spinor(lat, p), Q.Spinor(lat, p)
    Q.dslash_tune(y, x, g)
    one = Q.dslash_chosen(x, g)
    for count in (2, 4):
        assert (Q.dslash_chosen(x, g, count) == SPLIT) == (one == SPLIT)
    for count in (5, 12, 80):   # 61 440 (site, rhs) pairs
        assert Q.dslash_chosen(x, g, count) != SPLIT


def test_forced_split_where_it_does_not_apply(gpu):
    """FP16 links under FP32 spinors: the z-march instead."""
    Q = gpu
    L = (6, 4, 5, 4)
    lat = Q.Lattice(L)
    u, psi = Q.gauge_generate(L, 0.4, 71), Q.spinor_gaussian(L, 72)
    g = Q.Gauge(lat, Q.F16)
    Q.convert(g, Q.Gauge(lat).upload(u))
    x, y = Q.Spinor(lat, Q.F32).upload(psi), Q.Spinor(lat, Q.F32)
    out = []
    for cfg in (SPLIT, 2 | (6 << 8)):
        Q.dslash_set_config(x, g, cfg, 0)
        assert Q.dslash_chosen(x, g) == 2 | (6 << 8)
        Q.dslash(y, x, g, 0.1, 0.07)
        out.append(y.download())
    assert np.array_equal(*out)
    with pytest.raises(Q.QcdError):
        Q.dslash_set_config(x, g, 8, 0)
