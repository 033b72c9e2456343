"""The Jacobi SVD (k_jacobi_svd) at the edges of its sizes (8 R rows for R = 2, 4, 6, 8, 10,
12, 16) and at odd ones: k = r in the two-factor Greedy step, k = 2 r and the truncation
rank in the rank-adaptive one, with the tolerances of their other one-step tests."""
import numpy as np
import pytest

from oracle import dlra
from oracle.data import random_factors
from oracle.metrics import rel_err
from tests.test_gpu_greedy import run_greedy
from tests.test_gpu_parity import one_step_case, run_native_step, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r", [1, 2, 3, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64])
def test_polar(lri, r):
    n, m = 150, 140
    say(f"case: two-factor Greedy step n={n} m={m} r={r}")
    rng = np.random.default_rng(r)
    u = random_factors(rng, n, m, r)
    X = u.to_matrix() + 1e-2 * rng.standard_normal((n, m)) / np.sqrt(m)
    Z0 = u.V @ u.S.T
    U, _, Z = run_greedy(lri, u.U, np.eye(r), Z0, [X], twofactor=True)
    Uo, Zo = dlra.greedy_step_twofactor(u.U, Z0, X)
    e = np.linalg.norm(U @ Z.T - Uo @ Zo.T) / np.linalg.norm(Uo @ Zo.T)
    say(f"  rel err {e:.2e}")
    assert e <= 1e-10
    assert np.linalg.norm(U.T @ U - np.eye(r)) <= 1e-12


@pytest.mark.parametrize("tol", [1e-14, 1e-2])
@pytest.mark.parametrize("r", [1, 8, 9, 16, 17, 24, 25, 32, 33, 40, 41, 48, 49, 64])
def test_rank_adaptive(lri, r, tol):
    n, m = 200, 170
    say(f"case: RA step n={n} m={m} r={r} tol={tol}")
    u, A0, A1 = one_step_case(100 + r, n, m, r, inc=1e-2)
    Uo, So, Vo, r1 = dlra.rank_adaptive_bug_step(u.U, u.S, u.V, A1 - A0, tol, 64)
    U, S, V = run_native_step(lri, "ra", u, [A0, A1], tol=tol, rmax=64)
    say(f"  rank {S.shape[0]} (oracle {r1}), rel err {rel_err(U, S, V, Uo, So, Vo):.2e}")
    assert S.shape[0] == r1
    assert rel_err(U, S, V, Uo, So, Vo) <= 1e-9
    assert np.allclose(np.diag(S), np.diag(So), rtol=1e-10, atol=1e-14)
