"""Device memory that one-shot calls leave to the next: calls of unlike sizes from several
threads return the bits of the same calls made one by one, and what is kept is bounded."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _calls():
    import dtc_amd as dtc
    from dtc_amd import synth
    grey, modulus = synth.greyscale(11, seed=3, bvtv=0.4)
    doms = [dtc.Domain(synth.trabecular(n, seed=n, sigma=1.5, bvtv=0.4), delta=(0.01,) * 3, micro_nen=nen)
            for n, nen in ((9, 8), (17, 8), (26, 8), (6, 20), (10, 20))]
    doms.append(dtc.Domain(grey, llimit=1, delta=(0.01,) * 3, modulus=modulus, E=1e4))
    calls = []
    for d in doms:
        for kw in (dict(precision=0), dict(precision=1, precond=1)):
            calls.append(lambda d=d, kw=kw: dtc.solve_domain(d, rel_tol=1e-8, rotation=True, want_u=True, **kw))
        calls.append(lambda d=d: dict(zip(("nodes", "elems"), dtc.mesh(d.phi, d.llimit, d.micro_nen, d.delta, d.xa_n))))
    return calls


def _same(a, b):
    keys = [k for k, v in a.items() if isinstance(v, np.ndarray)]
    assert keys
    return all(np.array_equal(a[k], b[k], equal_nan=True) for k in keys)


def test_calls_from_threads_return_the_bits_of_single_calls():
    calls = _calls()
    alone = [c() for c in calls]
    wrong, errors = [], []

    def work(k):
        try:
            for i in np.random.default_rng(k).permutation(len(calls)):
                if not _same(alone[i], calls[i]()):
                    wrong.append((k, int(i)))
        except Exception as e:   # reported by the main thread
            errors.append(e)

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors, errors
    assert not wrong, wrong


def test_kept_memory_is_bounded():
    """At most 4 GiB stay with the library whatever sizes were asked for."""
    import ctypes as C
    import dtc_amd as dtc
    from dtc_amd._lib import load

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert load().hipMemGetInfo(C.byref(free), C.byref(total)) == 0   # the library's own runtime
        return free.value

    free0 = free_bytes()
    for n in range(40, 200, 16):
        phi = np.zeros((n, n, n), np.int32)
        phi[:2] = 1
        dtc.mesh(phi, 1, 20, (0.01,) * 3, (2, 2, 2))
    assert free0 - free_bytes() <= (4 << 30) + (256 << 20)
