"""Solid voxels of modulus 0: their nodes stay in the mesh, their elements carry nothing, so
the matvec meets clusters of nodes without a single element, at the front, inside and at
the end of its tables, and in tables without any element at all."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NX, NY, NZ = 17, 9, 9
# (z, y, x) ranges of modulus 0
ZERO = {"first corner": np.s_[0:4, 0:4, 0:8], "first half": np.s_[:, :, 0:9], "last corner": np.s_[4:, 4:, 8:],
        "inside": np.s_[1:8, 1:8, 1:16]}
MODES = [(0, 0), (1, 0), (1, 1)]     # precision, preconditioner


def _domain(dtc, zero, nen=8, **kw):
    mod = np.random.default_rng(5).uniform(2000.0, 8000.0, (NZ, NY, NX))
    if zero:
        mod[ZERO[zero]] = 0.0
    return dtc.Domain(np.ones(mod.shape, np.int8), delta=(0.01,) * 3, xa_n=(2, 2, 2), modulus=mod, micro_nen=nen, **kw)


def _oracle(d):
    from oracle import oracle as O
    nodes, elems = O.mesh(d.phi, 1, d.micro_nen, d.delta, d.xa_n)
    ijk = np.rint(nodes[elems[:, 0] - 1] / 0.01 - 1).astype(int)
    emod = d.modulus[ijk[:, 2], ijk[:, 1], ijk[:, 0]]
    mn, mx, dim = d.box()
    o = O.solve_domain(nodes, elems, 1.0, d.nu, d.a(), mn, mx, dim, tol=1e-13, emod=emod, want_u=True, want_r=True)
    held = np.zeros(len(nodes), bool)
    held[elems[emod > 0.0] - 1] = True          # nodes that some stiffness holds
    return o, np.repeat(held, 3)


@pytest.mark.parametrize("prec,precond", MODES)
@pytest.mark.parametrize("zero", ZERO)
def test_fields_match_the_oracle(zero, prec, precond):
    """Relative residual 1e-11.  An error of the residual grows by at most the condition of
    the Jacobi-scaled operator, about the square of the longest edge (< 3e2), times the
    moduli's spread (4) and 4 for the surfaces without a prescribed displacement:
    1e-11 * 5e3 < 1e-7.  The displacement of a node that nothing holds is free."""
    import dtc_amd as dtc
    d = _domain(dtc, zero)
    r = dtc.solve_domain(d, want_u=True, want_r=True, precision=prec, precond=precond, rel_tol=1e-11, rotation=False)
    assert r["status"] == 0
    o, held = _oracle(d)
    assert 0 < held.sum() < held.size
    for k in ("r", "ff"):
        assert np.abs(r[k] - o[k]).max() <= 1e-7 * np.abs(o[k]).max(), k
    assert np.abs(r["u"] - o["u"])[:, held].max() <= 1e-7 * np.abs(o["u"]).max()
    assert np.isfinite(r["u"]).all()


@pytest.mark.parametrize("prec,precond", MODES)
def test_in_one_batch(monkeypatch, prec, precond):
    """Such a domain first, inside and last in one sub-batch, and one that carries nothing."""
    import dtc_amd as dtc
    monkeypatch.setenv("DTC_CONCURRENT", "1")
    names = ["first half", None, "inside", None, "last corner"]
    doms = [_domain(dtc, z) for z in names]
    doms[3].modulus = np.zeros((NZ, NY, NX))
    res = dtc.solve_batch(doms, precision=prec, precond=precond, rel_tol=1e-11, rotation=False)
    assert [r["status"] for r in res] == [0] * 5
    for i, (d, r) in enumerate(zip(doms, res)):
        if i == 3:
            assert not r["ff"].any() and r["iterations"] == 0
        else:
            o, _ = _oracle(d)
            assert np.abs(r["ff"] - o["ff"]).max() <= 1e-7 * np.abs(o["ff"]).max(), i


@pytest.mark.parametrize("prec,precond", MODES)
@pytest.mark.parametrize("nen", [8, 20])
def test_nothing_carries(nen, prec, precond):
    """A domain alone whose every modulus is 0: no force, no iteration."""
    import dtc_amd as dtc
    d = _domain(dtc, None, nen)
    d.modulus = np.zeros((NZ, NY, NX))
    r = dtc.solve_domain(d, want_r=True, precision=prec, precond=precond, rel_tol=1e-11, rotation=False)
    assert r["status"] == 0 and r["iterations"] == 0
    assert not r["ff"].any() and not r["r"].any()


@pytest.mark.parametrize("prec,precond", [(0, 0), (1, 1)])
def test_quadratic_elements(prec, precond):
    """HEX20 over the same voxels (its coarse space is the HEX08 matvec)."""
    import dtc_amd as dtc
    d = _domain(dtc, "first half", 20)
    d.phi, d.modulus = d.phi[:5, :5, :13], d.modulus[:5, :5, :13]
    r = dtc.solve_domain(d, precision=prec, precond=precond, rel_tol=1e-11, rotation=False)
    assert r["status"] == 0
    o, _ = _oracle(d)
    assert np.abs(r["ff"] - o["ff"]).max() <= 1e-7 * np.abs(o["ff"]).max()
