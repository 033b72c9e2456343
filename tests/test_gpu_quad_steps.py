"""The fused RK4 steps of the quadratic sub-problems (k_quad_steps) at the edges of their
tiles: 16 and 48 own rows per workgroup, fewer rows than one tile with its halo,
column blocks of 4 and 16, odd and even numbers of RK4 steps, the tensor in LDS and in
global memory.  Against the CPU oracle; FP64, <= 1e-10 on Y as the other one-step tests."""
import numpy as np
import pytest

from oracle.data import random_factors
from oracle.metrics import rel_err
from tests.test_gpu_burgers import oracle_one, random_quadratic, run_one, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,r,N,periodic", [
    (3, 3, 1, 1, True), (5, 16, 4, 2, True), (5, 16, 4, 3, False), (16, 17, 5, 16, True), (31, 33, 16, 5, False),
    (64, 48, 17, 6, True), (100, 49, 24, 7, True), (90, 70, 32, 4, False), (8200, 97, 15, 5, True),
    (8191, 200, 24, 4, False)])
@pytest.mark.parametrize("name", ["bug", "primal"])
def test_tile_edges(lri, name, n, m, r, N, periodic):
    say(f"case: {name} n={n} m={m} r={r} N={N} periodic={periodic}")
    dev, host = random_quadratic(lri, n, m, 1, periodic, seed=n + r)
    u = random_factors(np.random.default_rng(n + 1), n, m, r)
    dt = 2e-4 * N  # small steps: well conditioned whatever the size
    got, ref = run_one(lri, name, dev, u, dt, N), oracle_one(name, host, u, dt, N)
    e = rel_err(*got, *ref)
    say(f"  rel err {e:.2e}")
    assert e <= 1e-10
