"""GCR cycles where their kernels change shape: restart lengths at both ends
and around the vectors-in-flight groups, lattices of partial tiles, and vector
lengths on both sides of the short / long split and of the separate
coefficient kernel.  Every solution is accepted by the oracle's b - D x."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

KAPPA = 0.12


def _fields(Q, L, nrhs, eps=0.2):
    u = Q.gauge_generate(L, eps, 61)
    lat = Q.Lattice(L)
    b = [Q.spinor_gaussian(L, 62 + r) for r in range(nrhs)]
    fb = Q.Spinor(lat, nrhs=nrhs)
    for r in range(nrhs):
        fb.upload(b[r], rhs=r)
    return u, lat, Q.Gauge(lat).upload(u), b, fb


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
@pytest.mark.parametrize("n", [1, 2, 3, 8, 9, 16, 17, 33, 64])
def test_restart_lengths_on_partial_tiles(gpu, prec, n):
    Q = gpu
    L = (6, 3, 5, 3)   # 270 sites: four tiles and 14 sites
    u, lat, g, b, fb = _fields(Q, L, 2)
    fx = Q.Spinor(lat, nrhs=2)
    S = Q.Solver(lat, g, n_restart=n, tol=1e-10, inner_prec=prec, batch=2, op="D", max_outer=500)   # (Q is indefinite: GCR(1) stalls on it)
    S.solve(fx, fb, KAPPA, 0.03)
    for r in range(2):
        assert O.b_minus_Dx(O.Geometry(L), fx.download(r), b[r], u, KAPPA, 0.03) <= 1e-10


# inner vectors of 4096 and 4608 (FP16 split), 8192 and 8448 (FP32, FP64), and
# 33 024 sites (more workgroups than the update adds up by itself)
@pytest.mark.parametrize("L,eo", [((16, 8, 8, 8), 1), ((16, 8, 8, 9), 0), ((8, 8, 18, 8), 1), ((16, 8, 8, 8), 0),
                                  ((22, 8, 8, 6), 0), ((16, 16, 16, 16), 1), ((43, 8, 8, 24), 0)])
@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
def test_short_and_long_vectors(gpu, prec, L, eo):
    """A rhs gets the same bits alone and in a batch of 3, and converges."""
    Q = gpu
    u, lat, g, b, fb = _fields(Q, L, 3)
    sols = []
    for batch in (1, 3):
        fx = Q.Spinor(lat, nrhs=3)
        Q.Solver(lat, g, n_restart=11, tol=1e-10, inner_prec=prec, batch=batch, eo=eo, max_outer=500).solve(fx, fb, KAPPA)
        sols.append([fx.download(r) for r in range(3)])
    for r in range(3):
        assert np.array_equal(sols[0][r], sols[1][r])
    assert O.b_minus_Dx(O.Geometry(L), sols[1][2], b[2], u, KAPPA) <= 1e-10


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
@pytest.mark.parametrize("eo", [0, 1])
def test_exhausted_krylov_space(gpu, prec, eo):
    """U = 1 and a point source: the Krylov space ends long before the cycle does."""
    Q = gpu
    L = (4, 4, 4, 4)
    u = np.zeros((256, 4, 3, 3), dtype=np.complex128)
    u[:, :, [0, 1, 2], [0, 1, 2]] = 1.0
    lat = Q.Lattice(L)
    fb, fx = Q.Spinor(lat).upload(Q.point_source(L, (1, 2, 3, 0), 2, 1)), Q.Spinor(lat)
    S = Q.Solver(lat, Q.Gauge(lat).upload(u), n_restart=64, tol=1e-10, inner_prec=prec, eo=eo, max_outer=100)
    S.solve(fx, fb, 0.11)
    assert O.b_minus_Dx(O.Geometry(L), fx.download(), Q.point_source(L, (1, 2, 3, 0), 2, 1), u, 0.11) <= 1e-10
