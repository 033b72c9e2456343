"""The S sub-step of the quadratic operator (k_quad_sstep) at the edges of its 16-wide
blocks: k = 1, 15, 16 (one block), 17, 31, 32 (two), both signs and a transposed start,
with and without forcing.  Against the CPU oracle; FP64, <= 1e-10 on Y."""
import numpy as np
import pytest

from oracle.data import random_factors
from oracle.metrics import rel_err
from tests.test_gpu_burgers import oracle_one, random_quadratic, run_one, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [1, 2, 15, 16, 17, 31, 32])
@pytest.mark.parametrize("name,q", [("bug", 0), ("primal", 2), ("dual", 1)])
def test_blocks(lri, name, q, r):
    n, m, N = 60, 45, 3
    say(f"case: {name} r={r} q={q}")
    dev, host = random_quadratic(lri, n, m, q, True, seed=r)
    u = random_factors(np.random.default_rng(r + 1), n, m, r)
    dt = 1e-3
    got, ref = run_one(lri, name, dev, u, dt, N), oracle_one(name, host, u, dt, N)
    e = rel_err(*got, *ref)
    say(f"  rel err {e:.2e}")
    assert e <= 1e-10


@pytest.mark.parametrize("r", [8, 13])  # the augmented core: 2 r = 16, 26
def test_augmented(lri, r):
    dev, host = random_quadratic(lri, 60, 45, 1, False, seed=r)
    u = random_factors(np.random.default_rng(r), 60, 45, r)
    got = run_one(lri, "ra", dev, u, 1e-3, 2, tol=1e-6)
    ref = oracle_one("ra", host, u, 1e-3, 2, tol=1e-6)
    assert got[1].shape == ref[1].shape
    assert rel_err(*got, *ref) <= 1e-10
