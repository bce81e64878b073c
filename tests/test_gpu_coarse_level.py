"""The one-launch Chebyshev pass of the coarsest multigrid level, at the lattice sizes where its
workgroup changes (256, 384, 512 and 729 nodes) and on domains that are their own coarsest
level; the phases of the block iteration on a domain whose FP32 recursion loses its way."""
import numpy as np
import pytest

from helpers import random_mask

pytestmark = pytest.mark.gpu

# (nx, ny, nz): 2 x 2 x 2, 252, 256, 288, 384, 392, 512, 567 and 729 lattice nodes, and larger ones above it
SHAPES = [(1, 1, 1), (8, 6, 3), (7, 7, 3), (8, 7, 3), (7, 7, 5), (6, 6, 7), (7, 7, 7), (8, 8, 6), (8, 8, 8), (9, 8, 8),
          (16, 15, 14), (17, 5, 9)]


@pytest.mark.parametrize("nx,ny,nz", SHAPES)
def test_pass_preconditions_like_its_polynomial(nx, ny, nz):
    """Solid blocks of at most 8 voxels an edge: degree 6 on [l/50, l] leaves the spectrum
    within 1 +- 1 / T_6(51/49) = 1 +- 0.35, condition 2.1, so conjugate gradients gain 5.5 per
    iteration: 1e-6 takes ln(2e6) / ln(5.5) < 9 iterations, the rest to 1e-8 four, and one
    each for the residual replacements: at most 16.  Larger blocks see the pass below a
    V-cycle of condition 4 at most: 18."""
    import dtc_amd as dtc
    d = dtc.Domain(np.ones((nz, ny, nx), np.int8), delta=(0.01,) * 3)
    r = dtc.solve_domain(d, precision=1, precond=1, rel_tol=1e-8, rotation=False)
    assert r["status"] == 0 and r["iterations"] <= (16 if max(nx, ny, nz) <= 8 else 18), r["iterations"]


@pytest.mark.parametrize("nx,ny,nz", SHAPES)
def test_porous_domains_match_fp64(nx, ny, nz):
    """Per-voxel moduli, missing voxels and nodes, several domains of unlike size in one
    batch: within 2 x 1e-11 times the condition (square of the edge times the moduli's
    spread, below 4e3) of the plain FP64 solve."""
    import dtc_amd as dtc
    rng = np.random.default_rng(nx * 100 + ny * 10 + nz)
    doms = []
    for k in range(3):
        phi = random_mask((nz, ny, nx), 0.7, nx + ny + nz + k)
        phi[0] = 1
        doms.append(dtc.Domain(phi, delta=(0.01,) * 3, modulus=rng.uniform(2000.0, 8000.0, phi.shape)))
    doms.append(dtc.Domain(np.ones((4, 5, 3), np.int8), delta=(0.01,) * 3))
    kw = dict(rel_tol=1e-11, rotation=False)
    for m, p in zip(dtc.solve_batch(doms, precision=1, precond=1, **kw), dtc.solve_batch(doms, precision=0, **kw)):
        assert m["status"] == p["status"] == 0
        assert np.abs(m["ff"] - p["ff"]).max() <= 1e-7 * np.abs(p["ff"]).max()


def test_a_stuck_phase_is_cut_short():
    """A trabecular 64^3 domain whose second FP32 phase got stuck and ran to the cap of 400
    twice: with phases bound to one and a half times the first one's length (and 16) it
    takes at most the first phase, three such phases and the last steps."""
    import dtc_amd as dtc
    from dtc_amd import synth
    d = dtc.Domain(synth.trabecular(64, seed=107), llimit=1, delta=(0.01,) * 3, xa_n=(2, 2, 2))
    one = dtc.solve_domain(d, precision=1, precond=1, rel_tol=1e-5, rotation=False)
    r = dtc.solve_domain(d, precision=1, precond=1, rel_tol=1e-11, rotation=False)
    assert r["status"] == 0 and r["relres"] <= 1e-11
    n1 = one["iterations"]
    assert r["iterations"] <= n1 + 3 * (n1 + n1 // 2 + 16) + 64, (n1, r["iterations"])
