"""HEX20 batches of very unlike domains: one large among many single voxels, and the other way
round, so that the element pass's work list has groups of one and of many workgroups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,precond", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("at", [0, 37, 60])
def test_one_large_domain_among_single_voxels(monkeypatch, at, prec, precond):
    """Against solves alone, to rel-res 1e-11.  A single voxel has Dirichlet nodes only: its
    forces carry rounding alone.  The large one: an error of the residual grows by at most the
    condition of the Jacobi-scaled quadratic operator, ten times the square of the edge
    (< 1e3): 2e-11 * 1e3 < 1e-7."""
    import dtc_amd as dtc
    monkeypatch.setenv("DTC_CONCURRENT", "1")
    one = lambda E: dtc.Domain(np.ones((1, 1, 1), np.int8), delta=(0.01,) * 3, micro_nen=20, E=E)
    doms = [one(1000.0 * (i + 1)) for i in range(60)]
    big = dtc.Domain(np.ones((9, 8, 7), np.int8), delta=(0.01,) * 3, micro_nen=20)
    doms.insert(at, big)
    kw = dict(precision=prec, precond=precond, rel_tol=1e-11, rotation=False)
    res = dtc.solve_batch(doms, **kw)
    assert [r["status"] for r in res] == [0] * 61
    alone = dtc.solve_domain(big, **kw)
    assert np.abs(res[at]["ff"] - alone["ff"]).max() <= 1e-7 * np.abs(alone["ff"]).max()
    unit = dtc.solve_domain(one(1000.0), **kw)["ff"]
    for i, r in enumerate(r for k, r in enumerate(res) if k != at):
        assert np.abs(r["ff"] - (i + 1) * unit).max() <= 1e-12 * (i + 1) * np.abs(unit).max(), i
