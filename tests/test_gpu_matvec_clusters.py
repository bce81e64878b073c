"""The element-by-element matvec over clusters of nodes at the sizes where it can go
wrong: clusters of a single element, of one brick, of several bricks, pieces of one
brick (more nodes than a cluster holds), edges that are no multiple of the 8x4x4
bricks, per-voxel moduli, and grids narrow and wide enough for both lane splits."""
import numpy as np
import pytest

from helpers import random_mask

pytestmark = pytest.mark.gpu

# (nx, ny, nz, solid share); full blocks exceed a cluster within one brick
SHAPES = [(1, 1, 1, 1.0), (2, 1, 3, 1.0), (7, 3, 3, 1.0), (8, 4, 4, 1.0), (9, 5, 5, 1.0), (16, 8, 8, 1.0), (17, 9, 7, 1.0),
          (13, 11, 10, 0.6), (19, 6, 12, 0.5), (25, 5, 9, 0.7)]


@pytest.mark.parametrize("prec,precond", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("nx,ny,nz,p", SHAPES)
def test_fields_match_the_oracle(nx, ny, nz, p, prec, precond):
    """Displacements and reactions of every load case to rel-res 1e-11 (FP64 and mixed,
    Jacobi and multigrid).  An error of the residual grows by at most the condition of
    the Jacobi-scaled operator, about the square of the longest edge (< 1e3) times the
    moduli's spread (4): 1e-11 * 4e3 < 1e-7."""
    import dtc_amd as dtc
    from oracle import oracle as O
    rng = np.random.default_rng(nx * 100 + ny * 10 + nz)
    phi = np.ones((nz, ny, nx), np.int8) if p == 1.0 else random_mask((nz, ny, nx), p, nx + ny + nz)
    phi[0] = 1
    mod = rng.uniform(2000.0, 8000.0, phi.shape)
    d = dtc.Domain(phi, delta=(0.01,) * 3, xa_n=(2, 2, 2), modulus=mod)
    r = dtc.solve_domain(d, want_u=True, want_r=True, precision=prec, precond=precond, rel_tol=1e-11, rotation=False)
    assert r["status"] == 0
    nodes, elems = O.mesh(phi, 1, 8, d.delta, d.xa_n)
    ijk = np.rint(nodes[elems[:, 0] - 1] / 0.01 - 1).astype(int)
    mn, mx, dim = d.box()
    o = O.solve_domain(nodes, elems, 1.0, d.nu, d.a(), mn, mx, dim, tol=1e-13,
                       emod=mod[ijk[:, 2], ijk[:, 1], ijk[:, 0]], want_u=True, want_r=True)
    for k in ("u", "r", "ff"):
        assert np.abs(r[k] - o[k]).max() <= 1e-7 * np.abs(o[k]).max(), k


def test_sums_do_not_depend_on_the_batch(monkeypatch):
    """30 FP64 Jacobi-PCG iterations on a domain alone (fewer clusters than the wide lane
    split starts at) and inside a batch (more): the same bits."""
    import dtc_amd as dtc
    from dtc_amd import synth
    monkeypatch.setenv("DTC_CONCURRENT", "1")
    doms = [dtc.Domain(synth.trabecular(40, seed=60 + i, sigma=2.0, bvtv=0.3), delta=(0.01,) * 3) for i in range(6)]
    kw = dict(precision=0, rel_tol=1e-12, max_iter=30, rotation=False)
    many = dtc.solve_batch(doms, **kw)
    alone = dtc.solve_domain(doms[2], **kw)
    assert alone["iterations"] == many[2]["iterations"] == 30
    for k in ("ff", "K_macro", "C", "relres"):
        assert np.array_equal(alone[k], many[2][k]), k
