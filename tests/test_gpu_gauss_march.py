"""The z march of the one-column Gauss kernel over several planes per lane, which
launches take with QCD_HIP_GAUSS_ZLEN set, or unasked on large whole FP16 fields:
the bits of one plane per lane and of the tiled kernel."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# slice, whole field, and a slice large enough for the tiled kernel where no length is set
CASES = [((6, 9, 7, 11), 2, 3), ((4, 5, 6, 10), -1, 2), ((2, 48, 40, 50), 0, 2)]
RUN = """
import sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import qcd_amd as Q
out = {}
for i, (L, t, nrhs) in enumerate(eval(sys.argv[2])):
    lat = Q.Lattice(L)
    for prec in ("f64", "f32", "f16"):
        g64, g, v = Q.Gauge(lat), Q.Gauge(lat, Q.PREC[prec]), Q.Spinor(lat, Q.PREC[prec], nrhs)
        Q.gauge_generate_device(g64, 0.3, 41)
        Q.convert(g, g64)
        for r in range(nrhs):
            v.upload(Q.spinor_gaussian(L, 42 + r), rhs=r)
        Q.gauss_smear(v, g, 0.6, t, 3)
        for r in range(nrhs):
            out[f"{i}{prec}{r}"] = v.download(r)
np.savez(sys.argv[3], **out)
"""


def test_set_lengths(gpu, tmp_path):
    """3 (no divisor of 11 and 10, one lane's last chunk shorter), 4 and 64 (all planes) against none set."""
    files = []
    for zlen in ("", "1", "3", "4", "64"):
        env = {k: v for k, v in os.environ.items() if k != "QCD_HIP_GAUSS_ZLEN"}
        if zlen:
            env["QCD_HIP_GAUSS_ZLEN"] = zlen
        files.append(str(tmp_path / f"z{zlen}.npz"))
        subprocess.run([sys.executable, "-c", RUN, ROOT, repr(CASES), files[-1]], check=True, env=env, timeout=100)
    ref = np.load(files[0])
    for f in files[1:]:
        got = np.load(f)
        assert sorted(got.files) == sorted(ref.files)
        for k in ref.files:
            assert np.array_equal(got[k], ref[k])


def test_whole_fp16_field(gpu):
    """6 x 32 x 32 x 34 sites, 3 rhs: two planes per lane; 5 rhs: four, the last chunk two."""
    Q = gpu
    L = (6, 32, 32, 34)
    lat = Q.Lattice(L)
    g64, g = Q.Gauge(lat), Q.Gauge(lat, Q.F16)
    Q.gauge_generate_device(g64, 0.3, 41)
    Q.convert(g, g64)
    src = [Q.spinor_gaussian(L, 42 + r) for r in range(2)]
    ref = []
    for s in src:
        one = Q.Spinor(lat, Q.F16).upload(s)
        Q.gauss_smear(one, g, 0.6, -1, 2)
        ref.append(one.download())
    for n in (3, 5):
        v = Q.Spinor(lat, Q.F16, n)
        for r in range(n):
            v.upload(src[r % 2], rhs=r)
        Q.gauss_smear(v, g, 0.6, -1, 2)
        for r in (0, n - 1):
            assert np.array_equal(v.download(r), ref[r % 2])
