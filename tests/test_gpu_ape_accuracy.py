"""Rounding of an APE step against the same step in extended precision."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

LD = np.clongdouble


def _dag(m):
    return np.conj(np.swapaxes(m, -1, -2))


def _project(m):
    """SU(3) projection by Newton's iteration; the inverse refined in extended precision."""
    x, one = m, np.eye(3, dtype=LD)
    for _ in range(60):
        inv = np.linalg.inv(x.astype(np.complex128)).astype(LD)
        for _ in range(3):
            inv = inv @ (2 * one - x @ inv)
        n = (x + _dag(inv)) / 2
        done = np.abs(n - x).max() < 1e-18
        x = n
        if done:
            break
    d = (np.cross(m[..., 1, :], m[..., 2, :]) * m[..., 0, :]).sum(-1)
    ph = np.arctan2(d.imag, d.real) / 3
    return x * (np.cos(ph) - 1j * np.sin(ph)).astype(LD)[..., None, None]


def _ape(L, u, alpha):
    def at(f, mu, step):   # f at x + step mu
        return np.roll(f.reshape(L[::-1] + f.shape[1:]), -step, axis=3 - mu).reshape(f.shape)

    out = u.copy()
    for mu in (1, 2, 3):
        s = np.zeros_like(u[:, 0])
        for nu in (1, 2, 3):
            if nu != mu:
                m, n, b = u[:, mu], u[:, nu], at(u, nu, -1)
                s = s + n @ at(m, nu, 1) @ _dag(at(n, mu, 1)) + _dag(b[:, nu]) @ b[:, mu] @ at(b[:, nu], mu, 1)
        out[:, mu] = _project(u[:, mu] + alpha * s)
    return out


@pytest.mark.parametrize("eps", [0.1, 0.2, 0.3])
def test_ape_step_rounding(gpu, eps):
    """Half an ulp of the elements (3^-1/2 in the mean) covers the rounding of the
    stored link and of the products before it, added in the mean square."""
    Q = gpu
    L = (4, 6, 4, 6)
    u = O.gauge_generate(L, eps, 90)
    ref = _ape(L, u.astype(LD), np.longdouble(0.5))
    lat = Q.Lattice(L)
    out = Q.Gauge(lat)
    Q.ape_smear(out, Q.Gauge(lat).upload(u), 0.5, 1)
    err = (out.download() - ref)[:, 1:]
    assert np.sqrt((np.abs(err)**2).mean()) <= 2.0**-53 / np.sqrt(3.0)
