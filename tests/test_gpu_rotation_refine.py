"""The chain of refinements of the rotation search at its ends: one refinement, all sixteen,
first grids of a few points, several tensors in one search."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tensor(seed):
    from dtc_amd import synth
    from oracle import oracle as O
    rng = np.random.default_rng(seed)
    n = rng.standard_normal(3)
    return O.rotate66(synth.orthotropic_C(rng), n / np.linalg.norm(n), rng.uniform(0.2, 1.2))


@pytest.mark.parametrize("criterion", [1, 2])
@pytest.mark.parametrize("step,num_zero", [(90.0, 1e-9), (30.0, 1e-9), (7.0, 1e-9), (5.0, 1e30), (5.0, 1e-300)])
def test_refinements_match_the_oracle(criterion, step, num_zero):
    """num_zero 1e30 stops after the first refinement (jj = 1), 1e-300 runs on until two
    minima agree to the bit, at most 16.  The criterion is a sum of squares of entries, each
    formed from about 40 products: 1e-9 of sum T^2 leaves 1e5 ulps for the two orders."""
    import dtc_amd as dtc
    from oracle import oracle as O
    T = _tensor(int(step))
    g, o = dtc.rotation_search(T, criterion, step, num_zero), O.rotation_search(T, criterion, step, num_zero)
    if num_zero > 1.0:
        assert g["jj"] == o["jj"] == 1
    assert 1 <= g["jj"] <= 16
    assert abs(g["crit"] - o["crit"]) <= 1e-9 * np.sum(T ** 2)


def test_searches_of_a_batch_equal_single_searches():
    import dtc_amd as dtc
    from dtc_amd import synth
    doms = [dtc.Domain(synth.trabecular(9, seed=40 + i, sigma=1.4, bvtv=0.5), delta=(0.01,) * 3) for i in range(5)]
    for r in dtc.solve_batch(doms, precision=0, rel_tol=1e-8, rotation=True):
        for c in (1, 2):
            one = dtc.rotation_search(r["EE"], c)
            assert all(np.array_equal(one[k], r["rot"][c - 1][k]) for k in ("jj", "alpha", "n", "aa", "EE_opt", "crit"))
