"""Link smearing where its kernels change course: y slabs that do not divide
the extent, the two forms of the stout exponential, and projections of badly
conditioned or badly scaled matrices."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(4, 3, 2, 3), (4, 3, 9, 5), (10, 4, 17, 3), (2, 2, 8, 2)])
def test_smearing_on_ragged_slabs(gpu, L):
    Q = gpu
    u = Q.gauge_generate(L, 0.3, 31)
    geo, lat = O.Geometry(L), Q.Lattice(L)
    g, out = Q.Gauge(lat).upload(u), Q.Gauge(lat)
    a = u
    for n in range(1, 4):   # one to three steps: both ping-pong fields and their temporal links
        a = O.ape3d(geo, a, 0.5)
        Q.ape_smear(out, g, 0.5, n)
        assert np.abs(out.download() - a).max() <= 1e-13
    for ndim in (3, 4):
        s = u
        for n in range(1, 4):
            s = O.stout(geo, s, 0.1, ndim)
            Q.stout_smear(out, g, 0.1, ndim, n)
            assert np.abs(out.download() - s).max() <= 1e-13


@pytest.mark.parametrize("rho", [1e-9, 0.1, 0.35, 0.6, 2.0])
def test_stout_exponential_both_forms(gpu, rho):
    """Series (eigenvalues of Q up to 1), closed form, and both in one wavefront."""
    Q = gpu
    L = (8, 4, 4, 4)
    u = Q.gauge_generate(L, 0.5, 32)
    lat = Q.Lattice(L)
    out = Q.Gauge(lat)
    Q.stout_smear(out, Q.Gauge(lat).upload(u), rho, 4, 1)
    # the closed form divides by 9 u^2 - w^2: a few 1e-14 from the oracle's own
    assert np.abs(out.download() - O.stout(O.Geometry(L), u, rho, 4)).max() <= (1e-13 if rho <= 0.6 else 1e-12)


@pytest.mark.parametrize("scale", [1.0, 1e-40, 1e40])
def test_projection_of_ill_conditioned_links(gpu, scale):
    Q = gpu
    L = (4, 4, 4, 4)
    rng = np.random.default_rng(33)
    m = rng.normal(size=(256, 4, 3, 3)) + 1j * rng.normal(size=(256, 4, 3, 3))
    v, s, w = np.linalg.svd(m)
    s[..., 2] = s[..., 0] * 10.0 ** rng.uniform(-6, 0, size=s.shape[:-1])
    s = np.sort(s, axis=-1)[..., ::-1]
    m = (v * s[..., None, :]) @ w
    # the polar factor of an FP64 matrix is defined to eps times its condition number
    tol = 1e-14 * (10 + s[..., 0] / s[..., 2])
    lat = Q.Lattice(L)
    out = Q.Gauge(lat)
    Q.ape_smear(out, Q.Gauge(lat).upload(scale * m), 0.0, 1)
    got = out.download()[:, 1:]
    assert (np.abs(got - O.project_su3(m[:, 1:])).max(axis=(-1, -2)) <= tol[:, 1:]).all()
    uu = got @ got.conj().swapaxes(-1, -2)
    assert np.abs(uu - np.eye(3)).max() <= 1e-14 and np.abs(np.linalg.det(got) - 1).max() <= 1e-14


def test_gauss_march_lengths_agree(gpu):
    """A launch long enough to march (6 rhs: 2 planes a lane, 12 rhs: 3, the last
    z chunk shorter) against one rhs, one plane a lane: the same bits."""
    Q = gpu
    L = (2, 32, 32, 34)
    u = Q.gauge_generate(L, 0.3, 34)
    lat = Q.Lattice(L)
    g = Q.Gauge(lat).upload(u)
    src = [Q.spinor_gaussian(L, 35 + r) for r in range(2)]
    ref = []
    for s in src:
        f = Q.Spinor(lat).upload(s)
        Q.gauss_smear(f, g, 4.0, -1, 3)
        ref.append(f.download())
    for n in (6, 12):
        f = Q.Spinor(lat, nrhs=n)
        for r in range(n):
            f.upload(src[r % 2], rhs=r)
        Q.gauss_smear(f, g, 4.0, -1, 3)
        for r in (0, n // 2, n - 1):
            assert np.array_equal(f.download(r), ref[r % 2])
    v, geo = src[0], O.Geometry(L)
    for _ in range(3):
        v = O.gauss3d_all(geo, v, u, 4.0)
    assert np.linalg.norm(ref[0] - v) <= 1e-13 * np.linalg.norm(v)


# 128 columns per workgroup: partial last one, rows longer than it, planes
# shorter than it; chunks of 1 to 8 planes with a shorter last one
@pytest.mark.parametrize("L,slice_,nrhs", [((4, 34, 29, 31), 1, 12), ((2, 150, 9, 40), 0, 3), ((4, 6, 5, 350), 3, 12),
                                           ((8, 18, 14, 22), -1, 7), ((2, 48, 40, 50), 0, 12)])
@pytest.mark.parametrize("prec", ["f64", "f32", "f16"])
def test_gauss_tiles_match_columns(gpu, prec, L, slice_, nrhs):
    """Large launches take another kernel than one rhs alone: same bits."""
    Q = gpu
    lat = Q.Lattice(L)
    g64, g = Q.Gauge(lat), Q.Gauge(lat, Q.PREC[prec])
    Q.gauge_generate_device(g64, 0.3, 41)
    Q.convert(g, g64)
    v = Q.Spinor(lat, Q.PREC[prec], nrhs)
    src = [Q.spinor_gaussian(L, 42 + r) for r in (0, 1)]
    for r in range(nrhs):
        v.upload(src[r % 2], rhs=r)
    Q.gauss_smear(v, g, 0.6, slice_, 3)
    for r in (0, nrhs - 1):
        one = Q.Spinor(lat, Q.PREC[prec]).upload(src[r % 2])
        Q.gauss_smear(one, g, 0.6, slice_, 3)
        assert np.array_equal(one.download(), v.download(r))
