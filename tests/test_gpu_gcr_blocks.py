"""GCR steps in blocks: every remainder of a cycle by blocks of 4, 2 and 1, on
the operators that take them differently (D and the even-odd Schur complement
with their local term left out of the directions, with and without a twisted
mass; Q, whose steps are nearly empty every other time), with random and point
sources, on vector lengths whose partial sums are added in one and in two
stages.  Each cycle has to reach the smallest residual that its Krylov space
holds: the number of cycles is the FP64 one (a cycle's reduction is that of
GMRES(n), so it does not depend on how the steps are taken), and the solution
passes the oracle's b - D x."""
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

KAPPA, TOL = 0.12, 1e-10


def _solve(Q, L, src, prec, n, op, eo, mu):
    lat = Q.Lattice(L)
    u = Q.gauge_generate(L, 0.2, 71)
    fb, fx = Q.Spinor(lat).upload(src), Q.Spinor(lat)
    S = Q.Solver(lat, Q.Gauge(lat).upload(u), n_restart=n, tol=TOL, inner_prec=prec, op=op, eo=eo, max_outer=2000)
    r = S.solve(fx, fb, KAPPA, mu)
    assert O.b_minus_Dx(O.Geometry(L), fx.download(), src, u, KAPPA, mu) <= TOL
    return r["outer"]


@pytest.mark.parametrize("op,eo,mu", [("D", 0, 0.0), ("D", 1, 0.04), ("Q", 0, 0.0), ("Q", 0, 0.04)])
@pytest.mark.parametrize("n", [4, 5, 6, 7, 12, 18])
@pytest.mark.parametrize("point", [0, 1])
def test_cycles_of_every_remainder(gpu, op, eo, mu, n, point):
    Q = gpu
    L = (8, 6, 4, 6)
    src = Q.point_source(L, (1, 2, 3, 0), 2, 1) if point else Q.spinor_gaussian(L, 72)
    ref = _solve(Q, L, src, "f64", n, op, eo, mu)
    for prec in ("f32", "f16"):
        # FP16 storage (2^-11) adds at most its own share to a residual that a
        # cycle of at most 18 steps reduces by more than that
        got = _solve(Q, L, src, prec, n, op, eo, mu)
        assert abs(got - ref) <= max(1, ref // 8)


# 256 and 257 to 1024 workgroups of the dots: the sums in one and in two stages
@pytest.mark.parametrize("L,prec", [((32, 16, 16, 8), "f16"), ((32, 16, 16, 9), "f16"), ((16, 16, 16, 12), "f32"),
                                    ((32, 16, 16, 16), "f32"), ((32, 16, 16, 16), "f64"), ((12, 8, 16, 8), "f64")])
def test_sums_in_two_stages(gpu, L, prec):
    Q = gpu
    _solve(Q, L, Q.spinor_gaussian(L, 73), prec, 11, "D", 0, 0.0)


@pytest.mark.parametrize("op,eo,mu", [("D", 0, 0.04), ("D", 1, 0.0), ("Q", 0, 0.0), ("Q", 0, 0.04)])
@pytest.mark.parametrize("n", [8, 9, 15, 16, 27, 31, 64])
@pytest.mark.parametrize("point", [0, 1])
def test_blocks_of_eight(gpu, op, eo, mu, n, point):
    """Cycles with blocks of eight and every shorter one behind them: the FP32
    and FP64 cycle counts agree (a cycle that FP32 storage, 6e-8, ends early
    leaves the next one as much to do)."""
    Q = gpu
    L = (8, 6, 4, 6)
    src = Q.point_source(L, (1, 2, 3, 0), 2, 1) if point else Q.spinor_gaussian(L, 74)
    ref = _solve(Q, L, src, "f64", n, op, eo, mu)
    assert abs(_solve(Q, L, src, "f32", n, op, eo, mu) - ref) <= max(1, ref // 8)


@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
@pytest.mark.parametrize("op,eo,mu", [("D", 0, 0.0), ("D", 1, 0.0), ("Q", 0, 0.0), ("D", 1, 5.0)])
@pytest.mark.parametrize("n", [12, 24])
def test_heavy_masses(gpu, prec, op, eo, mu, n):
    """kappa 0.005: a few steps reach the rounding of the stored vectors, the
    rest of the cycle works in their noise and has to leave the solution alone."""
    Q = gpu
    L = (8, 6, 4, 6)
    src, u, lat = Q.spinor_gaussian(L, 75), Q.gauge_generate(L, 0.2, 71), Q.Lattice(L)
    fb, fx = Q.Spinor(lat).upload(src), Q.Spinor(lat)
    S = Q.Solver(lat, Q.Gauge(lat).upload(u), n_restart=n, tol=TOL, inner_prec=prec, op=op, eo=eo, max_outer=30)
    S.solve(fx, fb, 0.005, mu)
    assert O.b_minus_Dx(O.Geometry(L), fx.download(), src, u, 0.005, mu) <= TOL
