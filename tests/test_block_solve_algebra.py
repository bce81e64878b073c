"""The 24 x 24 solves of the block PCG (csrc/bsolve.hpp), compiled for the CPU with one
context per lane of the wave, against their definition in numpy: a factor with dropped
pivots, right-hand sides of the kept directions, and what a direction that is not finite
may touch."""
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG

R = 24
MAIN = r"""
#include <ucontext.h>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>
#define __global__ static
#define __launch_bounds__(n)
constexpr int R = 24, RR = R * R, WAVE = 64;
struct Index { int x; };
static Index blockIdx, threadIdx;
static ucontext_t lanes[WAVE], caller;
static double slot[2][WAVE];
static int calls[WAVE], finished;
static void switch_to(int t) {           // lanes run in turn, one exchange at a time
    const int me = threadIdx.x;
    threadIdx.x = t;
    swapcontext(&lanes[me], &lanes[t]);
}
static double lane_f64(double v, int lane) {
    const int t = threadIdx.x, p = calls[t]++ & 1;
    slot[p][t] = v;
    switch_to((t + 1) % WAVE);
    return slot[p][lane];
}
#include "bsolve.hpp"
static int mode, n;
static std::vector<int> done;
static std::vector<double> g, l;
static std::vector<float> c;
static void body() {
    if (mode == 0) k_bsolve<0>(done.data(), g.data(), l.data(), c.data());
    if (mode == 1) k_bsolve<1>(done.data(), g.data(), l.data(), c.data());
    if (mode == 2) k_bsolve<2>(done.data(), g.data(), l.data(), c.data());
    if (++finished == WAVE) setcontext(&caller);
    switch_to((threadIdx.x + 1) % WAVE);
}
int main(int, char** argv) {
    mode = atoi(argv[1]);
    n = atoi(argv[2]);                    // domains one after another
    g.resize((size_t)n * 2 * RR);
    l.resize((size_t)n * RR);
    c.resize((size_t)n * RR);
    done.resize(n);
    FILE* f = fopen(argv[3], "rb");
    if (fread(g.data(), 8, g.size(), f) != g.size() || fread(l.data(), 8, l.size(), f) != l.size()) return 1;
    fclose(f);
    std::vector<char> stacks((size_t)WAVE << 16);
    for (int d = 0; d < n; ++d) {
        blockIdx.x = d;
        finished = 0;
        for (int t = 0; t < WAVE; ++t) {
            calls[t] = 0;
            getcontext(&lanes[t]);
            lanes[t].uc_stack.ss_sp = &stacks[(size_t)t << 16];
            lanes[t].uc_stack.ss_size = 1 << 16;
            makecontext(&lanes[t], body, 0);
        }
        threadIdx.x = 0;
        swapcontext(&caller, &lanes[0]);
    }
    f = fopen(argv[4], "wb");
    fwrite(l.data(), 8, l.size(), f);
    fwrite(c.data(), 4, c.size(), f);
    fclose(f);
}
"""


@pytest.fixture(scope="module")
def solve(tmp_path_factory):
    d = tmp_path_factory.mktemp("bsolve")
    (d / "m.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-I", os.path.join(PKG, "csrc"), str(d / "m.cpp"), "-o",
                    str(d / "m")], check=True)

    def run(mode, g0, g1=None, lfac=None):
        """g0, g1, lfac: (n, 24, 24); returns the factors and the coefficients."""
        n = len(g0)
        g = np.stack([g0, np.zeros_like(g0) if g1 is None else g1], 1)
        with open(d / "in", "wb") as f:
            f.write(g.tobytes() + (np.zeros_like(g0) if lfac is None else lfac).tobytes())
        subprocess.run([str(d / "m"), str(mode), str(n), str(d / "in"), str(d / "out")], check=True, timeout=60)
        raw = (d / "out").read_bytes()
        return (np.frombuffer(raw, np.float64, n * R * R).reshape(n, R, R),
                np.frombuffer(raw, np.float32, n * R * R, offset=n * R * R * 8).reshape(n, R, R))
    return run


def _factor(W, drop):
    """L with zero columns for the pivots at or below drop of their diagonal entry."""
    W = 0.5 * (W + W.T)
    A, L = W.copy(), np.zeros_like(W)
    for k in range(R):
        if A[k, k] > drop * W[k, k] and A[k, k] < np.inf:
            L[k:, k] = A[k:, k] / np.sqrt(A[k, k])
            A -= np.outer(L[:, k], L[:, k])
    return L


def _apply(L, B, forward=True):
    """Y of L L^T Y = B (forward) or L^T Y = B over the kept directions, zero rows elsewhere."""
    keep = np.flatnonzero(np.diag(L) > 0.0)
    Lk, Y = L[np.ix_(keep, keep)], np.zeros_like(B)
    Z = np.linalg.solve(Lk, B[keep]) if forward else B[keep]
    Y[keep] = np.linalg.solve(Lk.T, Z)
    return Y


def _grams(n):
    """Grams of blocks of 24 random columns, of condition below 1e3; in half of them some
    columns are zero or a sum of earlier ones."""
    rng = np.random.default_rng(3)
    P = rng.standard_normal((n, 200, R))
    for i in range(1, n, 2):
        P[i][:, 5] = 0.0
        P[i][:, 9] = P[i][:, 2] - P[i][:, 7]
        P[i][:, 23] = P[i][:, 0] + P[i][:, 22]
    return np.einsum("nri,nrj->nij", P, P), rng.standard_normal((n, R, R))


def test_modes_match_their_definition(solve):
    """FP64 with a condition below 1e3, results rounded to FP32: 2^-24 of the largest
    entry, and 24 x 1e3 x 2^-52 for the solves; together below 1e-6."""
    W, B = _grams(4)
    L, c0 = solve(0, W, B)
    _, c1 = solve(1, B, lfac=L)
    _, c2 = solve(2, W)
    for i in range(len(W)):
        ref = _factor(W[i], 1e-9)
        assert np.abs(L[i] - ref).max() <= 1e-9 * np.abs(ref).max()
        assert (np.diag(ref) > 0).sum() == (21 if i % 2 else 24)
        for got, want in ((c0[i], _apply(ref, B[i])), (c1[i], -_apply(ref, B[i])),
                          (c2[i], _apply(_factor(W[i], 1e-10), np.eye(R), False))):
            assert np.abs(got - want).max() <= 1e-6 * np.abs(want).max()


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("col", [0, 11, 23])
def test_a_direction_that_is_not_finite_is_dropped(solve, col, bad):
    """Its row and column of the Gram are not finite: its column of L is zero, and the
    others get the factor and the coefficients of a block without it."""
    W, B = _grams(2)
    without = W.copy()
    for M, v in ((W, bad), (without, 0.0)):
        M[:, col, :] = v
        M[:, :, col] = v
    B[:, col] = bad
    L, c0 = solve(0, W, B)
    _, c1 = solve(1, B, lfac=L)
    _, c2 = solve(2, W)
    B[:, col] = 0.0
    for i in range(len(W)):
        ref = _factor(without[i], 1e-9)
        assert not L[i][:, col].any()
        rest = [r for r in range(R) if r != col]
        assert np.abs(L[i] - ref)[rest].max() <= 1e-9 * np.abs(ref).max()
        for got, want in ((c0[i], _apply(ref, B[i])), (c1[i], -_apply(ref, B[i])),
                          (c2[i], _apply(_factor(without[i], 1e-10), np.eye(R), False))):
            assert not got[col].any()
            assert np.abs(got - want).max() <= 1e-6 * np.abs(want).max()
