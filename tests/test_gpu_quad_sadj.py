"""The reverse S sub-step of the quadratic operator (k_quad_sadj16 for k <= 16, the general
kernel above) at the edges of its 16-wide block, one reverse BUG step against the CPU
oracle with the tolerance of the other one-step adjoint tests (1e-9)."""
import numpy as np
import pytest

from oracle import adjoint_de as ad
from tests.test_gpu_adjoint_de import context, random_operator, random_state, rel, say, tangential

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r,q,N", [(1, 0, 1), (2, 1, 2), (15, 2, 3), (16, 0, 2), (17, 1, 2)])
def test_reverse_s_step_blocks(lri, r, q, N):
    n, m, dt = 70, 50, 0.002
    say(f"case: reverse BUG step r={r} q={q} N={N}")
    dev, host = random_operator(lri, n, m, q, True, seed=r)
    rng = np.random.default_rng(r + 40)
    U, S, V = random_state(rng, n, m, r)
    cot = [rng.standard_normal(x.shape) for x in (U, S, V)]
    with context(lri, dev, U, S, V) as ctx:
        Ub, Sb, Vb, (a, b) = ctx.step_de_bug_adjoint(dt, N, *cot)
    ref = ad.bug_de_step_vjp(host, U, S, V, dt, N, *cot)
    errs = [rel(tangential(U, Ub), tangential(U, ref[0])), rel(Sb, ref[1]),
            rel(tangential(V, Vb), tangential(V, ref[2])), abs(a - ref[3]) / abs(ref[3]), abs(b - ref[4]) / abs(ref[4])]
    say(f"  errors {errs}")
    assert max(errs) <= 1e-9
