"""The two-pass HEX20 operator at the sizes where it can go wrong (element counts around
its 4 and 8 elements per workgroup, node counts around its 32-node bricks, domains of
unlike size in one launch), and the node tables of the multigrid transfers on even, odd
and unlike edge lengths."""
import numpy as np
import pytest

from helpers import random_mask

pytestmark = pytest.mark.gpu

# (nx, ny, nz, solid share)
SHAPES = [(1, 1, 1, 1.0), (3, 1, 1, 1.0), (4, 1, 1, 1.0), (5, 1, 1, 1.0), (2, 2, 2, 1.0), (3, 3, 1, 1.0), (4, 3, 2, 0.6),
          (6, 5, 4, 0.7)]


def _domain(dtc, nx, ny, nz, p):
    rng = np.random.default_rng(nx * 100 + ny * 10 + nz)
    phi = np.ones((nz, ny, nx), np.int8) if p == 1.0 else random_mask((nz, ny, nx), p, nx + ny + nz)
    phi[0] = 1
    return dtc.Domain(phi, delta=(0.01,) * 3, xa_n=(2, 2, 2), micro_nen=20, modulus=rng.uniform(2000.0, 8000.0, phi.shape))


@pytest.mark.parametrize("prec,precond", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("nx,ny,nz,p", SHAPES)
def test_fields_match_the_oracle(nx, ny, nz, p, prec, precond):
    """Displacements and reactions to rel-res 1e-11.  An error of the residual grows by at
    most the condition of the Jacobi-scaled quadratic operator, ten times the square of
    the longest edge (< 400) times the moduli's spread (4): 1e-11 * 2e3 < 1e-7."""
    import dtc_amd as dtc
    from oracle import oracle as O
    d = _domain(dtc, nx, ny, nz, p)
    r = dtc.solve_domain(d, want_u=True, want_r=True, precision=prec, precond=precond, rel_tol=1e-11, rotation=False)
    assert r["status"] == 0
    nodes, elems = O.mesh(d.phi, 1, 20, d.delta, d.xa_n)
    ijk = np.rint(nodes[elems[:, 0] - 1] / 0.01 - 1).astype(int)
    mn, mx, dim = d.box()
    o = O.solve_domain(nodes, elems, 1.0, d.nu, d.a(), mn, mx, dim, tol=1e-13,
                       emod=d.modulus[ijk[:, 2], ijk[:, 1], ijk[:, 0]], want_u=True, want_r=True)
    for k in ("u", "r", "ff"):
        assert np.abs(r[k] - o[k]).max() <= 1e-7 * np.abs(o[k]).max(), k


@pytest.mark.parametrize("prec,precond", [(0, 0), (1, 1)])
def test_domains_of_unlike_size_in_one_launch(prec, precond):
    """One batch against solves alone to rel-res 1e-11: the bound above, on both sides."""
    import dtc_amd as dtc
    doms = [_domain(dtc, *s) for s in SHAPES]
    kw = dict(rel_tol=1e-11, rotation=False, precision=prec, precond=precond)
    for d, m in zip(doms, dtc.solve_batch(doms, **kw)):
        one = dtc.solve_domain(d, **kw)
        assert one["status"] == m["status"] == 0
        assert np.abs(one["ff"] - m["ff"]).max() <= 2e-7 * np.abs(one["ff"]).max()


@pytest.mark.parametrize("nx,ny,nz,nen", [(40, 17, 9, 8), (33, 32, 31, 8), (24, 8, 47, 8), (16, 9, 12, 20), (13, 14, 8, 20)])
def test_multigrid_transfers_keep_the_cycle_mesh_independent(nx, ny, nz, nen):
    """On a solid block the V-cycle leaves a condition number of at most 4: conjugate
    gradients gain a factor (sqrt(4) + 1) / (sqrt(4) - 1) = 3 per iteration, so 1e-8 takes
    log(2e8) / log(3) < 18.  A wrong or missing interpolation leaves some of the smooth
    modes to the smoother, whose condition grows with the square of the edge."""
    import dtc_amd as dtc
    d = dtc.Domain(np.ones((nz, ny, nx), np.int8), delta=(0.01,) * 3, micro_nen=nen)
    r = dtc.solve_domain(d, precision=1, precond=1, rel_tol=1e-8, rotation=False)
    assert r["status"] == 0 and r["iterations"] <= 18, r["iterations"]
