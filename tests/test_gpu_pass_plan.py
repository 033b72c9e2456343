"""The split plan of the product passes at the edges of its rule: a reduction of one,
exactly one and just more than one quantum of 256, workgroups below and above 512 and (FP64)
1536, tall, wide and ragged.  dA V and dA' U against NumPy in FP64.

Tolerance, entry by entry against |dA| |B|: a sum of K rounded products errs by at
most (K + 2) u, u = 2^-53 in FP64 and 2^-24 in FP32; in the mixed precision the operand B
is rounded to FP32 (u) or to two BF16 parts (2^-16), dA to FP32 or two BF16 parts as well."""
import numpy as np
import pytest

from oracle.data import bf16_round, random_factors
from tests.test_zz_no_alloc import _Hip, context_product, noalloc_product, say

pytestmark = pytest.mark.gpu


def data(n, m, r, dtype, seed):
    rng = np.random.default_rng(seed)
    u = random_factors(rng, n, m, r)
    A0, A1 = rng.standard_normal((n, m)).astype(np.float32), rng.standard_normal((n, m)).astype(np.float32)
    if dtype == "bf16":
        A0, A1 = bf16_round(A0), bf16_round(A1)
    return u, A0.astype(np.float64), A1.astype(np.float64)


def check(got, u, A0, A1, which, dtype, precision):
    d = A1 - A0
    d, B = (d, u.V) if which == 0 else (d.T, u.U)
    K = d.shape[1]
    tol = (K + 2) * 2.0 ** -53
    if precision:
        tol = (K + 4) * 2.0 ** -24 + (2.0 ** -14 if dtype == "bf16" else 0.0)
    bound = tol * (np.abs(d) @ np.abs(B))
    err = np.abs(got - d @ B) - (K + 2) * 2.0 ** -53 * (np.abs(d) @ np.abs(B))  # NumPy's own
    assert np.all(err <= bound), (which, float((err / bound).max()))


@pytest.mark.parametrize("dtype,precision", [("f64", 0), ("f32", 1), ("bf16", 1), ("bf16", 0)])
@pytest.mark.parametrize("n,m,r", [(255, 256, 8), (257, 513, 17), (2000, 1500, 21), (1025, 1537, 48), (33, 9001, 5),
                                   (9001, 40, 33), (4099, 1023, 64)])
def test_products(lri, n, m, r, dtype, precision):
    say(f"case: passes n={n} m={m} r={r} {dtype} precision={precision}")
    u, A0, A1 = data(n, m, r, dtype, n + m)
    for which in (0, 1):
        check(context_product(lri, which, u, A0, A1, dtype, precision), u, A0, A1, which, dtype, precision)


@pytest.mark.parametrize("n,m", [(22000, 1025), (20000, 1024)])
def test_noalloc_at_its_limit(lri, n, m):
    """22000 x 1025 at r = 64: three splits' partial results exceed the static scratch, the
    coarse plan's one fits; 20000 x 1024: two splits fit."""
    say(f"case: noalloc product n={n} m={m} r=64")
    lri.native.lib()
    hip = _Hip()
    u, A0, A1 = data(n, m, 64, "f32", 3)
    check(noalloc_product(lri, hip, 0, u, A0, A1, "f32", 0), u, A0, A1, 0, "f32", 0)
    hip.free()
