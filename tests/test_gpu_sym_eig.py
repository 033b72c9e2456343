"""The symmetric eigen-decompositions of the matrix-ODE steps at the edges of their sizes
(8, 16 and 32 pairs in one workgroup, the shifted one-sided form above k = 64): a step whose
S sub-step and column flows run in them, with variable coefficients, against the CPU oracle
at the tolerance of the other one-step tests (1e-10 on Y)."""
import numpy as np
import pytest

from oracle.data import random_factors
from oracle.metrics import rel_err
from tests.test_gpu_de import operator_pair, oracle_one, run_one, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [1, 2, 3, 15, 16, 17, 31, 32, 33, 63, 64])
def test_bug_ranks(lri, r):
    n, m, N = 150, 120, 4
    dev, host = operator_pair(lri, n, m, 1, False, True, seed=r)
    u = random_factors(np.random.default_rng(r), n, m, r)
    got, ref = run_one(lri, "bug", dev, u, 0.01, N), oracle_one("bug", host, u, 0.01, N)
    e = rel_err(*got, *ref)
    say(f"case: r={r} rel err {e:.2e}")
    assert e <= 1e-10


@pytest.mark.parametrize("r", [1, 8, 9, 16, 17, 32, 33])  # decompositions of size 2 r
def test_augmented_sizes(lri, r):
    n, m, N = 150, 120, 4
    dev, host = operator_pair(lri, n, m, 1, False, True, seed=r)
    u = random_factors(np.random.default_rng(r), n, m, r)
    got, ref = run_one(lri, "ra", dev, u, 0.01, N, tol=1e-9), oracle_one("ra", host, u, 0.01, N, tol=1e-9)
    assert got[1].shape == ref[1].shape
    e = rel_err(*got, *ref)
    say(f"case: 2r={2 * r} rel err {e:.2e}")
    assert e <= 1e-10
