"""The one-launch CholeskyQR (k_qr) at the edges of its shapes: one workgroup alone (up to
512 rows at r <= 16, 256 above), the first row of a second one, 20 and 21 workgroups
(whose sums are shared out), 64 with growing tiles, the largest it takes and one row more
(the separate kernels).  Against the CPU oracle in FP64 (<= 1e-10 on Y, as the other
one-step tests), on tall problems with a short other side."""
import numpy as np
import pytest

from oracle import dlra
from oracle.metrics import rel_err
from tests.test_gpu_parity import one_step_case, run_native_step, say

pytestmark = pytest.mark.gpu

STEP = {"primal": dlra.ksl_primal_step, "dual": dlra.ksl_dual_step, "bug": dlra.bug_step}


@pytest.mark.parametrize("kind", ["primal", "dual", "bug"])
@pytest.mark.parametrize("n,r", [(16, 1), (33, 16), (256, 17), (257, 32), (512, 16), (513, 5), (2560, 32),
                                 (2561, 32), (3000, 26), (3969, 32), (5121, 16), (6144, 32), (6145, 17),
                                 (16385, 16), (49152, 9), (49153, 16)])
def test_shapes(lri, kind, n, r):
    m = 48
    say(f"case: {kind} n={n} m={m} r={r}")
    u, A0, A1 = one_step_case(n + r, n, m, min(r, 16) if n == 16 else r)
    got = run_native_step(lri, kind, u, [A0, A1])
    got = got[:3]
    ref = STEP[kind](u.U, u.S, u.V, A1 - A0)
    e = rel_err(*got, *ref)
    say(f"  rel err {e:.2e}")
    assert e <= 1e-10


@pytest.mark.parametrize("n,r", [(200, 32), (8192, 32), (8193, 17), (16384, 32), (16385, 20)])
def test_three_passes(lri, n, r):
    """The shifted form, in the Greedy step (U1 = orth(X V0), V1 = orth(X' U0), S1 = U1' X V1)."""
    u, X, _ = one_step_case(n + r, n, 48, r)
    with lri.native.Context(n, 48, r) as ctx:
        ctx.set_state(u.U, u.S, u.V)
        ctx.reserve(1, lri.native.F64)
        ctx.upload(0, lri.api._encode(X, "f64"))
        ctx.step_greedy(0)
        got = ctx.get_state()
    e = rel_err(*got, *dlra.greedy_step(u.U, u.S, u.V, X))
    say(f"case: greedy n={n} r={r} rel err {e:.2e}")
    assert e <= 1e-10


@pytest.mark.parametrize("n,r", [(6000, 32), (16384, 16), (700, 13), (4099, 24)])
def test_repeats_bit_for_bit(lri, n, r):
    """The sums over workgroups are in workgroup order whatever their timing."""
    u, A0, A1 = one_step_case(5, n, 64, r)
    runs = [run_native_step(lri, "primal", u, [A0, A1])[:3] for _ in range(3)]
    for g in runs[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(g, runs[0]))
