"""The Chebyshev degree that a caller gives holds on the finest and on the intermediate levels."""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import PKG, ROOT

pytestmark = pytest.mark.gpu

# in a process of its own: the switches are read once
CODE = """
import sys
import numpy as np
sys.path[:0] = [%r, %r]
import dtc_amd as dtc
from dtc_amd import synth
d = dtc.Domain(synth.trabecular(%d, seed=5, sigma=2.0, bvtv=0.35), delta=(0.01,) * 3, micro_nen=%d)
r = dtc.solve_domain(d, precision=1, precond=1, rel_tol=1e-10, rotation=False)
assert r["status"] == 0
np.savez(sys.argv[1], ff=r["ff"], iterations=r["iterations"])
"""


@pytest.mark.parametrize("n,nen", [(40, 8), (20, 20)])
def test_given_degree_is_the_levels_degree(tmp_path, n, nen):
    """Degree 2 given, against the default (degree 2 on the finest level) with the degree and the
    interval of the intermediate levels switched to those of degree 2: the same iteration
    to the last bit, and another one than the default with its degree 4 below."""
    import dtc_amd as dtc
    from dtc_amd import synth
    d = dtc.Domain(synth.trabecular(n, seed=5, sigma=2.0, bvtv=0.35), delta=(0.01,) * 3, micro_nen=nen)
    kw = dict(precision=1, precond=1, rel_tol=1e-10, rotation=False)
    two, plain = dtc.solve_domain(d, mg_degree=2, **kw), dtc.solve_domain(d, **kw)
    assert two["status"] == plain["status"] == 0
    env = dict(os.environ, DTC_MG_LDEG="2", DTC_MG_LRATIO="12")
    out = str(tmp_path / "r.npz")
    subprocess.run([sys.executable, "-c", CODE % (ROOT, PKG, n, nen), out], env=env, check=True, timeout=100)
    ref = np.load(out)
    assert two["iterations"] == int(ref["iterations"])
    assert np.array_equal(two["ff"], ref["ff"])
    assert not np.array_equal(two["ff"], plain["ff"])


@pytest.mark.parametrize("degree", [1, 2, 3, 4, 6])
def test_every_degree_converges(degree):
    import dtc_amd as dtc
    from dtc_amd import synth
    d = dtc.Domain(synth.trabecular(36, seed=8, sigma=2.0, bvtv=0.35), delta=(0.01,) * 3)
    r = dtc.solve_domain(d, precision=1, precond=1, rel_tol=1e-10, rotation=False, mg_degree=degree)
    p = dtc.solve_domain(d, precision=1, precond=1, rel_tol=1e-10, rotation=False)
    assert r["status"] == 0 and r["precision_used"] == dtc.DTC_FP32_REFINE
    # two solutions of relative residual 1e-10, condition below the square of the edge: 2e-10 * 1.3e3 < 1e-6
    assert np.abs(r["ff"] - p["ff"]).max() <= 1e-6 * np.abs(p["ff"]).max()
