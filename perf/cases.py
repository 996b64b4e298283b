"""The work a user of this library has it do, as measurable cases.

Every case goes through the Python front end (or, for the host-struct API,
through the C entry point a C program calls) with inputs in hand: fields in
HBM, the solver workspace created once, host structs for the drop-in calls.
Gauge fields are U = exp(i eps H), H traceless Hermitian from N(0,1) draws.

Outputs are device fields.  `run` returns them as lists that fetch the values
only when they are read (DeviceOutput): a program that keeps its fields in HBM
does not copy them to the host in every pass.  Values come back in the type of
the field they were stored in (FP16 spinors as float16).
"""
import ctypes

import numpy as np
import torch

import qcd_amd as Q

THETA = (np.pi, 0.0, 0.0, 0.0)   # antiperiodic in time
TWISTED = (np.pi, 0.3, -0.5, 0.7)
SPINOR_BYTES = {"f64": 192, "f32": 96, "f16": 52}
LINK_BYTES = {"f64": 576, "f32": 288, "f16": 144}


def listed():
    return [
        # One operator application on the smallest configuration: launch latency.
        {"name": "dslash_f64_8c16", "kind": "dslash", "T": 16, "X": 8, "Y": 8, "Z": 8, "prec": "f64", "nrhs": 1,
         "op": "D", "mu": 0.0, "kappa": 0.125, "eps": 0.2},
        # The benchmark's headline: one FP64 application on 24^3x48.
        {"name": "dslash_f64_24c48", "kind": "dslash", "T": 48, "X": 24, "Y": 24, "Z": 24, "prec": "f64", "nrhs": 1,
         "op": "D", "mu": 0.0, "kappa": 0.132, "eps": 0.3},
        # Q with a twisted mass and phases in all directions over a few FP32
        # vectors on extents that fill neither tiles nor wavefronts evenly.
        {"name": "dslash_q_f32_ragged", "kind": "dslash", "T": 30, "X": 21, "Y": 18, "Z": 22, "prec": "f32", "nrhs": 3,
         "op": "Q", "mu": 0.05, "kappa": 0.130, "eps": 0.3},
        # The operator over a batch of FP16 vectors, as the mixed solver's users apply it.
        {"name": "dslash_f16_16rhs_24c48", "kind": "dslash", "T": 48, "X": 24, "Y": 24, "Z": 24, "prec": "f16",
         "nrhs": 16, "op": "D", "mu": 0.0, "kappa": 0.132, "eps": 0.3},
        # A propagator (12 point sources) on the smallest lattice of the serving mix.
        {"name": "solve_f16_12rhs_8c16", "kind": "solve", "T": 16, "X": 8, "Y": 8, "Z": 8, "prec": "f16", "nrhs": 12,
         "n_restart": 32, "eo": True, "mu": 0.0, "kappa": 0.125, "eps": 0.2},
        # The propagator of the solves benchmark, with its shorter restart length.
        {"name": "solve_f16_12rhs_16c32", "kind": "solve", "T": 32, "X": 16, "Y": 16, "Z": 16, "prec": "f16",
         "nrhs": 12, "n_restart": 12, "eo": True, "mu": 0.0, "kappa": 0.130, "eps": 0.3},
        # invert.c's own solve: one vector, FP64, GCR(32) on Q, no preconditioning.
        {"name": "solve_f64_1rhs_16c32", "kind": "solve", "T": 32, "X": 16, "Y": 16, "Z": 16, "prec": "f64", "nrhs": 1,
         "n_restart": 32, "eo": False, "mu": 0.0, "kappa": 0.130, "eps": 0.3},
        # A propagator on 24^3x48 in one mixed-precision even-odd batch.
        {"name": "solve_f16_12rhs_24c48", "kind": "solve", "T": 48, "X": 24, "Y": 24, "Z": 24, "prec": "f16",
         "nrhs": 12, "n_restart": 12, "eo": True, "mu": 0.0, "kappa": 0.132, "eps": 0.3},
        # Source smearing of a propagator: 50 Gauss iterations of 12 vectors on one time slice.
        {"name": "gauss_f64_12rhs_32c64", "kind": "gauss", "T": 64, "X": 32, "Y": 32, "Z": 32, "prec": "f64",
         "nrhs": 12, "niter": 50, "slice": 5, "eps": 0.3},
        # Link smearing of one configuration before its sources are smeared.
        {"name": "ape_10steps_24c48", "kind": "ape", "T": 48, "X": 24, "Y": 24, "Z": 24, "steps": 10, "eps": 0.3},
        {"name": "stout4d_4steps_24c48", "kind": "stout", "T": 48, "X": 24, "Y": 24, "Z": 24, "steps": 4, "ndim": 4,
         "eps": 0.3},
        # The host-struct call of a program written against the reference's
        # header: host arrays in, host arrays out.
        {"name": "dropin_apply_16c32", "kind": "dropin", "T": 32, "X": 16, "Y": 16, "Z": 16, "mu": 0.0,
         "kappa": 0.130, "eps": 0.3},
    ]


def _extent(rng, lo, hi, even=False):
    """An extent spread over the logarithm of [lo, hi]; odd ones among them unless even."""
    n = int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))
    return n + (n & 1) if even else n


def _lattice(rng, lo, hi, most_sites, even=False):
    while True:
        L = {"T": _extent(rng, 2 * lo, 2 * hi, even)}
        L.update({d: _extent(rng, lo, hi, even) for d in "XYZ"})
        V = L["T"] * L["X"] * L["Y"] * L["Z"]
        if V % 2 == 0 and V <= most_sites:
            return L


def draw(rng):
    kind = rng.choice(["dslash", "dslash", "dslash", "solve", "solve", "gauss", "ape", "stout", "dropin"])
    eps = round(rng.uniform(0.1, 0.3), 3)
    if kind == "dslash":
        prec = rng.choice(["f64", "f32", "f16"])
        nrhs = rng.choice([1, 1, 2, 3, 5, 8, 12, 16, 17])
        L = _lattice(rng, 6, 30, 40_000_000 // max(nrhs, 40))
        return {"kind": kind, **L, "prec": prec, "nrhs": nrhs, "op": rng.choice("DQ"),
                "mu": rng.choice([0.0, round(rng.uniform(0.01, 0.1), 3)]), "kappa": round(rng.uniform(0.12, 0.135), 4),
                "eps": eps}
    if kind == "solve":
        prec = rng.choice(["f16", "f16", "f32", "f64"])
        eo = rng.random() < 0.7
        nrhs = rng.choice([1, 3, 12]) if eo else 1
        L = _lattice(rng, 6, 22, 400_000 if prec == "f16" else 150_000, even=eo)
        return {"kind": kind, **L, "prec": prec, "nrhs": nrhs, "n_restart": rng.choice([8, 12, 16, 32]), "eo": eo,
                "mu": rng.choice([0.0, round(rng.uniform(0.01, 0.1), 3)]), "kappa": round(rng.uniform(0.115, 0.125), 4),
                "eps": eps}
    if kind == "gauss":
        nrhs = rng.choice([1, 5, 12])
        L = _lattice(rng, 6, 32, 2_100_000)
        return {"kind": kind, **L, "prec": rng.choice(["f64", "f64", "f32", "f16"]), "nrhs": nrhs,
                "niter": rng.choice([3, 20, 50, 51]), "slice": rng.choice([-1, 0, L["T"] - 1]) if L["T"] <= 16 else
                rng.randrange(L["T"]), "eps": eps}
    if kind == "ape":
        return {"kind": kind, **_lattice(rng, 6, 24, 700_000), "steps": rng.randint(1, 10), "eps": eps}
    if kind == "stout":
        return {"kind": kind, **_lattice(rng, 6, 24, 700_000), "steps": rng.randint(1, 4), "ndim": rng.choice([3, 4]),
                "eps": eps}
    return {"kind": kind, **_lattice(rng, 6, 16, 140_000), "mu": rng.choice([0.0, 0.05]),
            "kappa": round(rng.uniform(0.12, 0.135), 4), "eps": eps}


# ---------------------------------------------------------------- inputs
def _extents(case):
    return tuple(int(case[d]) for d in "TXYZ")


def _theta(case):
    return TWISTED if case.get("mu", 0.0) else THETA


def _mass(case):
    return 1.0 / (2.0 * case["kappa"]) - 4.0


def _mul(a, b):
    """3x3 products of [..., 3, 3] arrays, written out over the inner index."""
    return sum(a[..., :, k, None] * b[..., None, k, :] for k in range(3))


def _dag(a):
    return a.conj().transpose(-1, -2)


def _trace(a):
    return a[..., 0, 0] + a[..., 1, 1] + a[..., 2, 2]


def _eye(like):
    return torch.eye(3, dtype=like.dtype, device=like.device)


def _exp(x):
    """Matrix exponential of small 3x3 matrices (norm up to about 2), by its series."""
    p, one = _eye(x).expand_as(x), _eye(x)
    for n in range(28, 0, -1):
        p = one + _mul(x, p) / n
    return p


def _normal(gen, *shape):
    return torch.view_as_complex(torch.randn(*shape, 2, generator=gen, dtype=torch.float64, device=gen.device))


def _links(case, seed):
    """Links [V, 4, 3, 3] on the GPU."""
    L = _extents(case)
    gen = torch.Generator(device="cuda").manual_seed(2 * int(seed) + 1)
    a = _normal(gen, int(np.prod(L)), 4, 3, 3)
    h = (a + _dag(a)) / 2
    h = h - (_trace(h) / 3)[..., None, None] * _eye(h)
    return _exp(1j * case["eps"] * h)


def _vectors(case, seed):
    """Spinors [V, 4, 3], one after another: N(0,1) entries."""
    V = int(np.prod(_extents(case)))
    gen = torch.Generator(device="cuda").manual_seed(2 * int(seed))
    for _ in range(case.get("nrhs", 1)):
        yield _normal(gen, V, 4, 3)


def _source_site(case, seed):
    """Where the point sources of a propagator sit, (t, x, y, z)."""
    L = _extents(case)
    rng = np.random.default_rng(int(seed))
    t = case["slice"] if case.get("slice", -1) >= 0 else int(rng.integers(0, L[0]))
    return (t,) + tuple(int(rng.integers(0, L[d])) for d in (1, 2, 3))


def _host(t):
    return t.cpu().numpy()


class DeviceOutput(list):
    """Output fields on the device (or host memory of the state), fetched in full when iterated over."""

    def __init__(self, n, fetch):
        super().__init__([None] * n)
        self.fetch = fetch

    def __iter__(self):
        return (self.fetch(r) for r in range(len(self)))

    def __getitem__(self, r):
        return self.fetch(r)


def _stored(a, prec):
    """Host values of a field in the type it holds on the device."""
    if prec == "f64":
        return a
    return a.astype(np.complex64) if prec == "f32" else a.view(np.float64).astype(np.float16)


class DropInCall:
    """Host structs of one program: geometry, vectors, links."""

    def __init__(self, case, seed):
        self.d = Q.DropIn(_extents(case), _theta(case))
        self.v = self.d.vector(_host(next(_vectors(case, seed))))
        self.u = self.d.gauge(_host(_links(case, seed)))
        self.out = self.d.vector()

    def fetch(self, r):
        return self.d.view(self.out, 12).copy()

    def __del__(self):
        self.d.close()


def prepare(case, seed):
    kind, L = case["kind"], _extents(case)
    if kind == "dropin":
        return {"case": case, "call": DropInCall(case, seed)}
    lat = Q.Lattice(L, _theta(case))
    g64 = Q.Gauge(lat).upload(_host(_links(case, seed)))
    s = {"case": case, "lat": lat, "g64": g64}
    if kind in ("ape", "stout"):
        s["out"] = Q.Gauge(lat)
        return s
    p = Q.PREC[case["prec"]]
    nrhs = case["nrhs"]
    if kind == "solve":   # a propagator: point sources, one per (spin, colour)
        s["b"], s["x"] = Q.Spinor(lat, Q.F64, nrhs), Q.Spinor(lat, Q.F64, nrhs)
        for r in range(nrhs):
            Q.point_source_device(s["b"], r, _source_site(case, seed), r // 3, r % 3)
        s["solver"] = Q.Solver(lat, g64, n_restart=case["n_restart"], tol=1e-12, max_outer=2000,
                               inner_prec=case["prec"], batch=nrhs, eo=int(case["eo"]),
                               op=Q.OP_D if case["eo"] else Q.OP_Q)
        return s
    g = g64
    if p != Q.F64:
        g = Q.Gauge(lat, p)
        Q.convert(g, g64)
    s["g"] = g
    if kind == "dslash":
        s["x"], s["y"] = Q.Spinor(lat, p, nrhs), Q.Spinor(lat, p, nrhs)
        for r, v in enumerate(_vectors(case, seed)):
            s["x"].upload(_host(v), rhs=r)
        return s
    s["site"] = _source_site(case, seed)
    s["src"] = s["v"] = Q.Spinor(lat, Q.F64, nrhs)
    if p != Q.F64:
        s["v"] = Q.Spinor(lat, p, nrhs)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "dslash":
        Q.dslash(s["y"], s["x"], s["g"], _mass(case), case["mu"], Q.OP_Q if case["op"] == "Q" else Q.OP_D)
        y, prec = s["y"], case["prec"]
        return DeviceOutput(y.nrhs, lambda r: _stored(y.download(r), prec))
    if kind == "solve":
        s["solver"].solve(s["x"], s["b"], case["kappa"], case["mu"])
        x = s["x"]
        return DeviceOutput(x.nrhs, lambda r: x.download(r))
    if kind == "gauss":
        # smearing works in place: a pass makes the propagator's sources and smears them
        v, prec = s["v"], case["prec"]
        for r in range(v.nrhs):
            Q.point_source_device(s["src"], r, s["site"], r // 3, r % 3)
        if v is not s["src"]:
            Q.convert(v, s["src"])
        Q.gauss_smear(v, s["g"], 4.0, case["slice"], case["niter"])
        return DeviceOutput(v.nrhs, lambda r: _stored(v.download(r), prec))
    if kind == "ape":
        Q.ape_smear(s["out"], s["g64"], 0.5, case["steps"])
    elif kind == "stout":
        Q.stout_smear(s["out"], s["g64"], 0.1, case["ndim"], case["steps"])
    else:
        c = s["call"]
        rc = Q.lib().qcd_applyWilsonTMOp(ctypes.byref(c.out), ctypes.byref(c.v), ctypes.byref(c.u), _mass(case),
                                         case["mu"])
        assert rc == 0
        return DeviceOutput(1, c.fetch)
    out = s["out"]
    return DeviceOutput(1, lambda r: out.download())


# ---------------------------------------------------------------- work
def work(case):
    """Compulsory bytes (inputs read once, outputs written once) and operations of one pass."""
    L = _extents(case)
    V, kind = int(np.prod(L)), case["kind"]
    if kind == "dslash":
        n = case["nrhs"]
        return {"bytes": V * (2 * n * SPINOR_BYTES[case["prec"]] + LINK_BYTES[case["prec"]]), "flops": V * n * 1392}
    if kind == "dropin":
        return {"bytes": V * 960, "flops": V * 1392}
    if kind == "solve":   # the iteration count depends on the data: one operator application at least
        n = case["nrhs"]
        return {"bytes": V * (2 * n * 192 + 576), "flops": V * n * 1392}
    if kind == "gauss":
        sites, n = V if case["slice"] < 0 else V // L[0], case["nrhs"]
        f64 = case["prec"] == "f64"
        return {"bytes": V * n * (192 if f64 else 192 + SPINOR_BYTES[case["prec"]])
                + sites * (2 * n * SPINOR_BYTES[case["prec"]] + 3 * LINK_BYTES[case["prec"]] // 4),
                "flops": sites * n * case["niter"] * (6 * 4 * 72 + 48)}
    # per link and step: 2 (ndim - 1) staples of two 3x3 products each, then
    # the projection (about six Newton steps) or the exponential
    nd = 3 if kind == "ape" else case["ndim"]
    per_link = 2 * (nd - 1) * 2 * 216 + (6 * 350 if kind == "ape" else 1100)
    return {"bytes": V * 2 * 576, "flops": V * nd * case["steps"] * per_link}


# ---------------------------------------------------------------- exact
# The chiral gamma basis of the reference (lib/src/qcd_gamma.c:46-88): gamma_mu
# in units of i^p at (row, column).
_GAMMA = {0: ((0, 2, 2), (1, 3, 2), (2, 0, 2), (3, 1, 2)), 1: ((0, 3, 3), (1, 2, 3), (2, 1, 1), (3, 0, 1)),
          2: ((0, 3, 2), (1, 2, 0), (2, 1, 0), (3, 0, 2)), 3: ((0, 2, 3), (1, 3, 1), (2, 0, 1), (3, 1, 3))}
_AXIS = {0: 3, 1: 2, 2: 1, 3: 0}   # direction (t, x, y, z) -> axis of [Z, Y, X, T, ...]


def _gamma(mu, like):
    g = torch.zeros(4, 4, dtype=torch.complex128, device=like.device)
    for r, c, p in _GAMMA[mu]:
        g[r, c] = 1j ** p
    return g


def _grid(a, L):
    return a.reshape((L[3], L[2], L[1], L[0]) + tuple(a.shape[1:]))


def _at(a, mu, step):
    """The value at x + step mu, at x."""
    return torch.roll(a, -step, _AXIS[mu])


def _spin(m, psi):
    return sum(m[:, s, None] * psi[..., s, None, :] for s in range(4))


def _colour(u, psi):
    """u psi on the colour index of [..., 4, 3]."""
    return sum(u[..., None, :, c] * psi[..., :, c, None] for c in range(3))


def _apply_d(psi, u, L, theta, m, mu, op="D"):
    """D psi, or i gamma5 D psi, of a grid [Z, Y, X, T, 4, 3]."""
    g5 = torch.tensor([1.0, 1.0, -1.0, -1.0], dtype=torch.complex128, device=psi.device)[:, None]
    one = torch.eye(4, dtype=torch.complex128, device=psi.device)
    out = (m + 4.0) * psi + 1j * mu * g5 * psi
    for d in range(4):
        ph, g = complex(np.exp(1j * theta[d] / L[d])), _gamma(d, psi)
        ud = u[..., d, :, :]
        out = out - 0.5 * ph * _colour(ud, _spin(one - g, _at(psi, d, 1)))
        out = out - 0.5 * ph.conjugate() * _at(_colour(_dag(ud), _spin(one + g, psi)), d, -1)
    return 1j * g5 * out if op == "Q" else out


def _as_output(grid, V):
    return grid.reshape((V,) + tuple(grid.shape[4:])).cpu().numpy()


def _solve(b, u, case, L):
    """x with D x = b by conjugate gradients on D^+ D (g5 D(mu)^+ g5 = D(-mu))."""
    th, m, mu = _theta(case), _mass(case), case["mu"]
    g5 = torch.tensor([1.0, 1.0, -1.0, -1.0], dtype=torch.complex128, device=b.device)[:, None]

    def dag(v):
        return g5 * _apply_d(g5 * v, u, L, th, m, -mu)

    x = torch.zeros_like(b)
    for _ in range(3):   # restarts from the true residual
        r = dag(b - _apply_d(x, u, L, th, m, mu))
        p, rr = r.clone(), r.abs().square().sum()
        for _ in range(400):
            w = _apply_d(p, u, L, th, m, mu)
            a = rr / w.abs().square().sum()
            x = x + a * p
            r = r - a * dag(w)
            new = r.abs().square().sum()
            p, rr = r + (new / rr) * p, new
            if float(rr) < 1e-30:
                break
    return x


def _gauss(v, u, case):
    n = 1.0 / (1.0 + 6.0 * 4.0)
    for _ in range(case["niter"]):
        s = torch.zeros_like(v)
        for d in (1, 2, 3):
            ud = u[..., d, :, :]
            s = s + _colour(ud, _at(v, d, 1)) + _at(_colour(_dag(ud), v), d, -1)
        v = n * (v + 4.0 * s)
    return v


def _staples(u, mu, dims):
    s = 0
    for nu in dims:
        if nu != mu:
            a, b = u[..., nu, :, :], u[..., mu, :, :]
            s = s + _mul(_mul(a, _at(b, nu, 1)), _dag(_at(a, mu, 1)))
            s = s + _at(_mul(_dag(a), _mul(b, _at(a, mu, 1))), nu, -1)
    return s


def _inverse(a):
    r0, r1, r2 = a[..., 0, :], a[..., 1, :], a[..., 2, :]

    def cross(x, y):
        return torch.stack([x[..., 1] * y[..., 2] - x[..., 2] * y[..., 1], x[..., 2] * y[..., 0] - x[..., 0] * y[..., 2],
                            x[..., 0] * y[..., 1] - x[..., 1] * y[..., 0]], -1)

    c = torch.stack([cross(r1, r2), cross(r2, r0), cross(r0, r1)], -1)
    det = (r0 * c[..., :, 0]).sum(-1)
    return c / det[..., None, None], det


def _project(a):
    """The unitary polar factor times exp(-i arg(det) / 3), by Newton's iteration."""
    det = _inverse(a)[1]
    x = a
    for _ in range(12):
        x = 0.5 * (x + _dag(_inverse(x)[0]))
    return x * torch.exp(-1j * torch.angle(det) / 3)[..., None, None]


def _ape(u, case):
    new = u.clone()
    for mu in (1, 2, 3):
        new[..., mu, :, :] = _project(u[..., mu, :, :] + 0.5 * _staples(u, mu, (1, 2, 3)))
    return new


def _stout(u, case):
    dims = tuple(range(4 - case["ndim"], 4))
    new = u.clone()
    for mu in dims:
        w = _mul(_staples(u, mu, dims), _dag(u[..., mu, :, :]))
        a = w - _dag(w)
        a = a - (_trace(a) / 3)[..., None, None] * _eye(a)
        new[..., mu, :, :] = _mul(_exp(0.05 * a), u[..., mu, :, :])   # i Q = rho/2 A
    return new


def exact(case, seed):
    kind, L = case["kind"], _extents(case)
    V = int(np.prod(L))
    if kind == "solve" and V * case["nrhs"] > 2_000_000:
        return None
    u = _grid(_links(case, seed), L)
    if kind in ("dslash", "dropin"):
        return [_as_output(_apply_d(_grid(v, L), u, L, _theta(case), _mass(case), case["mu"], case.get("op", "D")), V)
                for v in _vectors(case, seed)]
    if kind in ("ape", "stout"):
        for _ in range(case["steps"]):
            u = (_ape if kind == "ape" else _stout)(u, case)
        return [_as_output(u, V)]
    t, x, y, z = _source_site(case, seed)
    out = []
    for r in range(case["nrhs"]):
        b = torch.zeros(V, 4, 3, dtype=torch.complex128, device=u.device)
        b[t + L[0] * (x + L[1] * (y + L[2] * z)), r // 3, r % 3] = 1.0
        b = _grid(b, L)
        if kind == "solve":
            b = _solve(b, u, case, L)
        elif case["slice"] < 0:
            b = _gauss(b, u, case)
        else:
            k = case["slice"]
            b[:, :, :, k:k + 1] = _gauss(b[:, :, :, k:k + 1], u[:, :, :, k:k + 1], case)
        out.append(_as_output(b, V))
    return out
