"""The measured work of this framework: what its users have it do, through its public entry
points, from the smallest solve to the largest snapshots.

A case is a dict with a ``kind``:

* ``solve``     ``solve(MatrixDataProblem, alg)``, the whole call: context, steps, every state.
* ``data``      steps over snapshots that are resident on the GPU, on a context that the
                program keeps (initial factors in and final factors out as device arrays).
* ``adjoint``   reverse steps over such snapshots, the cotangents on the device.
* ``de``        matrix-ODE steps dX/dt = A X + X B' + a b' on a context that the program keeps.
* ``burgers``   ``solve(MatrixDEProblem, alg, dt)`` of the viscous Burgers problem, the whole call.
* ``gradient``  ``solve_gradient`` of a loss of the final state of such a solve, the whole call.
* ``batch``     rank-adaptive steps of many independent heat equations of uneven sizes.
"""
import ctypes
import math

import numpy as np
import torch

import __graft_entry__

DEV = "cuda:0"
BYTES = {"f64": 8, "f32": 4, "bf16": 2}
TORCH = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}


def package():
    torch.cuda.init()  # torch's device before the library's first call
    return __graft_entry__.load_package()


def listed():
    return [
        # the basic use and the smallest: a 100-step solve of a 256 x 256 problem at rank 8, the
        # snapshots made on the GPU; launches and latency
        dict(name="solve_ksl_f64_256", kind="solve", alg="ksl", n=256, m=256, r=8, steps=100),
        # an ordinary FP64 tracking run, uneven sides and an odd rank
        dict(name="ksl_f64_2000x1500", kind="data", alg="ksl", n=2000, m=1500, r=21, dtype="f64", steps=20),
        # the headline: BF16 snapshots of 16384 x 16384 at rank 32
        dict(name="ksl_bf16_16384", kind="data", alg="ksl", n=16384, m=16384, r=32, dtype="bf16", steps=8),
        # FP32 snapshots, ragged sides that no tile divides
        dict(name="bug_f32_10007x4099", kind="data", alg="bug", n=10007, m=4099, r=24, dtype="f32", steps=8),
        # FP64 throughout at a rank above 32; both sweep directions in one step
        dict(name="strang_f64_6144x8192", kind="data", alg="strang", n=6144, m=8192, r=48, dtype="f64", steps=2),
        # rank adaptation on data: augmented bases, the small SVD, the read-back of the rank
        dict(name="ra_bug_bf16_8192x3000", kind="data", alg="bug_ra", n=8192, m=3000, r=20, dtype="bf16", steps=6),
        # the snapshot itself instead of increments
        dict(name="greedy_bf16_16384", kind="data", alg="greedy", n=16384, m=16384, r=32, dtype="bf16", steps=6),
        # the reverse direction over data
        dict(name="adjoint_bug_bf16_12288", kind="adjoint", alg="bug", n=12288, m=12288, r=32, dtype="bf16", steps=4),
        # the heat equation with a source at 4096 x 4096, rank 32, stiff (5369 RK4 sub-steps)
        dict(name="de_bug_4096", kind="de", alg="bug", n=4096, r=32, steps=10, variable=False, dt=1e-4),
        # Burgers with one parameter sample per column, the notebook's size and rank
        dict(name="burgers_bug_1000x400", kind="burgers", alg="bug", n=1000, m=400, r=15, steps=20, substeps=16),
        # the gradient of a loss through a Burgers solve, checkpointed
        dict(name="gradient_burgers_2048x1024", kind="gradient", alg="bug", n=2048, m=1024, r=16, steps=8, substeps=7,
             checkpoint=4),
        # many small heat equations of uneven size and rank at once
        dict(name="batch_ra_64", kind="batch", count=64, nmin=256, nmax=2048, rmin=4, rmax=28, steps=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "data", "data", "data", "data", "adjoint", "de", "burgers", "gradient", "batch"])
    if kind == "solve":
        n, m, r = _log(rng, 100, 1500), _log(rng, 100, 1500), rng.randint(4, 24)
        return dict(kind=kind, alg=rng.choice(["ksl", "bug"]), n=n, m=m, r=r, steps=rng.randint(20, 100))
    if kind in ("data", "adjoint"):
        dtype = rng.choice(["bf16", "bf16", "f32", "f64"])
        alg = rng.choice(["ksl", "dual", "strang", "bug", "bug_ra", "greedy"] if kind == "data" else
                         ["bug", "ksl", "ksl_dual"])
        top = {"bf16": 16384, "f32": 12000, "f64": 8192}[dtype]
        n, m = _log(rng, 500, top), _log(rng, 500, top)
        return dict(kind=kind, alg=alg, n=n, m=m, r=rng.randint(4, 28 if alg == "bug_ra" else 64), dtype=dtype,
                    steps=rng.randint(2, 8 if kind == "data" else 4))
    if kind == "de":
        variable = rng.random() < 0.4
        n = _log(rng, 300, 1500 if variable else 4096)
        alg = rng.choice(["bug", "bug", "bug_ra"])
        return dict(kind=kind, alg=alg, n=n, r=rng.randint(6, 32 if alg == "bug" else 20), steps=rng.randint(3, 10),
                    variable=variable, dt=1e-4 if alg == "bug" else BATCH["dt"])
    if kind == "burgers":
        n = _log(rng, 300, 2000)
        return dict(kind=kind, alg=rng.choice(["bug", "ksl"]), n=n, m=_log(rng, 100, 1000), r=rng.randint(6, 24),
                    steps=rng.randint(4, 20), substeps=_burgers_substeps(n))
    if kind == "gradient":
        n = _log(rng, 400, 2048)
        return dict(kind=kind, alg=rng.choice(["bug", "ksl"]), n=n, m=_log(rng, 200, 1024), r=rng.randint(6, 20),
                    steps=rng.randint(3, 8), substeps=max(2, math.ceil(7 * (n / 2048) ** 2) + 1),
                    checkpoint=rng.randint(2, 5))
    return dict(kind=kind, count=rng.randint(8, 64), nmin=256, nmax=_log(rng, 500, 2048), rmin=4,
                rmax=rng.randint(8, 28), steps=rng.randint(2, 8))


# ------------------------------------------------------------------------------------------ inputs


def _gen(seed, what=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1009 + what)
    return g


def _orth(rows, cols, g, dtype=torch.float64):
    """Orthonormal columns, from a Gaussian, by two Cholesky QRs (torch's QR is slow for tall matrices)."""
    X = torch.randn(rows, cols, generator=g, device=DEV, dtype=torch.float64)
    for _ in range(2):
        L = torch.linalg.cholesky(X.t() @ X)
        X = torch.linalg.solve_triangular(L, X.t(), upper=False).t()
    return X.contiguous()


def _pitch(n, dtype):
    """Column pitch in elements: the padding that the library recommends for BF16 columns of a multiple of 4 KB."""
    return n + 64 if dtype == "bf16" and (2 * n) % 4096 == 0 else n


def _snapshots(case, seed, count):
    """A(t_k) = Q1(t_k) D(t_k) Q2(t_k)' + noise with slowly turning orthonormal Q1, Q2 and singular
    values that grow with e^t; t_k = k / 199 as in a 200-snapshot run. Stored column-major: X[k] is
    the m x n row-major transpose, in a buffer of the column pitch. With them the exact rank-r
    factors at t = 0."""
    n, m, r, dtype = case["n"], case["m"], case["r"], case["dtype"]
    g = _gen(seed)
    q = min(r + 8, min(n, m) // 2)
    Q1, Q2 = _orth(n, 2 * q, g), _orth(m, 2 * q, g)
    # rank adaptation: singular values with clear gaps around the tolerance, and little noise
    ra = case["alg"] == "bug_ra"
    sig = 10.0 ** (-torch.arange(q, device=DEV, dtype=torch.float64) / 8) if ra else \
        10.0 ** (-1.5 * torch.arange(q, device=DEV, dtype=torch.float64) / max(1, r - 1))
    work = torch.float64 if dtype == "f64" else torch.float32
    scale = (1e-7 if ra else 1e-3) / math.sqrt(max(n, m))
    C1 = torch.randn(m, n, generator=g, device=DEV, dtype=work) * scale
    C2 = torch.randn(m, n, generator=g, device=DEV, dtype=work) * scale
    ld = _pitch(n, dtype)
    X = []
    for k in range(count):
        t = k / 199.0 * (8.0 if ra else 1.0)
        a, b = math.cos(t), math.sin(t)
        left = (Q1[:, :q] * a + Q1[:, q:] * b).to(work)
        right = ((Q2[:, :q] * a - Q2[:, q:] * b) * (sig * math.exp(t))).to(work)
        A = right @ left.t()
        A.add_(C1, alpha=a).add_(C2, alpha=b)
        buf = torch.empty(m, ld, device=DEV, dtype=TORCH[dtype])
        buf[:, :n].copy_(A)
        X.append(buf[:, :n])
        del A
    return X, Q1[:, :r].contiguous(), torch.diag(sig[:r]), Q2[:, :r].contiguous()


def _ptr(t):
    return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))


class _Factors:
    """Factors on the device, column-major (a tensor (r, n) row-major is n x r column-major)."""

    def __init__(self, n, m, r):
        self.n, self.m, self.r = n, m, r
        self.U = torch.zeros(r, n, device=DEV, dtype=torch.float64)
        self.S = torch.zeros(r, r, device=DEV, dtype=torch.float64)
        self.V = torch.zeros(r, m, device=DEV, dtype=torch.float64)

    def set(self, U, S, V):
        self.U.copy_(U.t())
        self.S.copy_(S.t())
        self.V.copy_(V.t())
        return self


def _host(U, s, V):
    """U, diag(s), V as host arrays, column-major."""
    return tuple(np.asfortranarray(x.cpu().numpy()) for x in (U, torch.diag(s), V))


def _set_state(lri, ctx, f):
    """The context's factors from device arrays. They are copied on the default stream; the library's own
    stream is another one, so that the steps come after a wait."""
    lri.native.check(lri.native.lib().lri_set_state(ctx.h, f.r, _ptr(f.U), f.n, _ptr(f.S), f.r, _ptr(f.V), f.m), ctx.h)
    torch.cuda.current_stream().synchronize()


def _get_state(lri, ctx, f):
    """The context's factors into f; returns their rank."""
    k = ctypes.c_int64()
    lri.native.check(lri.native.lib().lri_get_state(ctx.h, ctypes.byref(k), _ptr(f.U), f.n, _ptr(f.S), f.r, _ptr(f.V),
                                                    f.m), ctx.h)
    return int(k.value)


def _rank_cap(case):
    return min(64, case["n"], case["m"]) if case["alg"] == "bug_ra" else case["r"]


def _ra_tol(case):
    """Between two of the cumulative tails of the singular values 10^(-j/8): keeps about r + 3 of r + 8."""
    return 0.8 * 10.0 ** (-(case["r"] + 3) / 8)


def _count(case):
    """Snapshots that a data pass walks over, in a ring."""
    return 5 if case["alg"] == "strang" else 4


def _pairs(case):
    """(previous, [middle,] next) of every step; the walk goes up the ring and back down."""
    c = _count(case)
    walk = list(range(c)) + list(range(c - 2, 0, -1))
    hop = 2 if case["alg"] == "strang" else 1
    at = [walk[i % len(walk)] for i in range(hop * case["steps"] + 1)]
    return [tuple(at[i * hop:i * hop + hop + 1]) for i in range(case["steps"])]


# ------------------------------------------------------------------------------------------ prepare


def prepare(case, seed):
    lri = package()
    return {"solve": _prepare_solve, "data": _prepare_data, "adjoint": _prepare_data, "de": _prepare_de,
            "burgers": _prepare_burgers, "gradient": _prepare_burgers, "batch": _prepare_batch}[case["kind"]](
                lri, case, seed)


def _algorithm(lri, name):
    return lri.ProjectorSplitting(lri.PrimalLieTrotter()) if name == "ksl" else lri.UnconventionalAlgorithm()


def _prepare_solve(lri, case, seed):
    X, U, S, V = _snapshots(dict(case, dtype="f64"), seed, case["steps"] + 1)
    u0 = lri.SVDLikeRepresentation(*_host(U, torch.diagonal(S), V))
    prob = lri.MatrixDataProblem([x.t() for x in X], u0)
    return dict(case=case, lri=lri, prob=prob, alg=_algorithm(lri, case["alg"]))


def _prepare_data(lri, case, seed):
    n, m, r = case["n"], case["m"], case["r"]
    X, U, S, V = _snapshots(case, seed, _count(case))
    cap = _rank_cap(case)
    ctx = lri.native.Context(n, m, cap)
    ctx.bind([x.data_ptr() for x in X], lri.native.DTYPES[case["dtype"]], X[0].stride(0), owners=X)
    ctx.set_precision(lri.native.PREC_F64 if case["dtype"] == "f64" else lri.native.PREC_MIXED)
    st = dict(case=case, lri=lri, ctx=ctx, X=X, start=_Factors(n, m, r).set(U, S, V), out=_Factors(n, m, cap))
    if case["kind"] == "adjoint":
        g = _gen(seed, 1)
        rand = [torch.randn(*s, generator=g, device=DEV, dtype=torch.float64) for s in ((n, r), (r, r), (m, r))]
        st["bar"] = _Factors(n, m, r).set(*rand)
        torch.cuda.synchronize()
        _set_state(lri, ctx, st["start"])
    if case["alg"] == "bug_ra":
        st["probe"] = torch.randn(n, generator=_gen(seed, 2), device=DEV, dtype=torch.float64)
    return st


def _smooth(n, r, g):
    """n x r orthonormal columns that mix the 2 r smoothest sines: heat-equation data that lives longer than a step."""
    return _sines(n, min(n, 2 * r)) @ _orth(min(n, 2 * r), r, g)


def _sines(n, k):
    """The first k eigenvectors of tridiag(1, -2, 1); whole periods leave the argument first, so that the
    sines are exact to rounding."""
    i, j = (torch.arange(1, x + 1, device=DEV, dtype=torch.float64) for x in (n, k))
    angle = torch.remainder(i[:, None] * j[None, :], 2 * (n + 1)) * (math.pi / (n + 1))
    return torch.sin(angle) * math.sqrt(2.0 / (n + 1))


def _heat(case, seed):
    """Smooth orthonormal factors, singular values 10^(-i/8), a source a b'; for variable coefficients the
    diffusion a(x) = 1 + 0.5 sin(2 pi x + phase) on the cell faces."""
    n, r = case["n"], case["r"]
    g = _gen(seed)
    U, V = _smooth(n, r, g), _smooth(n, r, g)
    s = 10.0 ** (-torch.arange(r, device=DEV, dtype=torch.float64) / 8)
    a, b = (torch.randn(n, generator=g, device=DEV, dtype=torch.float64) for _ in range(2))
    phase = float(torch.rand(1, generator=g, device=DEV))
    face = (1.0 + 0.5 * np.sin(2 * np.pi * (np.arange(n + 1) / n + phase))) if case["variable"] else np.ones(n + 1)
    d, e = -(face[:-1] + face[1:]) * float(n * n), face[1:-1] * float(n * n)
    return U, s, V, a, b, d, e


def _heat_substeps(d, e, dt):
    up = np.zeros_like(d)
    up[:-1] += np.abs(e)
    up[1:] += np.abs(e)
    return max(1, math.ceil(dt * 2 * float(np.max(np.abs(d) + up)) / 2.5))


def _prepare_de(lri, case, seed):
    n, r = case["n"], case["r"]
    U, s, V, a, b, d, e = _heat(case, seed)
    cap = min(64, n) if case["alg"] == "bug_ra" else r
    ctx = lri.native.Context(n, n, cap)
    ctx.set_operator_lyapunov(d, e, False, d, e, False, a.cpu().numpy(), b.cpu().numpy())
    if not case["variable"]:
        ctx.set_resident_eigenbasis(True)  # as init() does for constant coefficients
    return dict(case=case, lri=lri, ctx=ctx, start=_host(U, s, V),
                out=_Factors(n, n, cap), substeps=_heat_substeps(d, e, case["dt"]),
                probe=torch.randn(n, generator=_gen(seed, 2), device=DEV, dtype=torch.float64))


def _burgers_substeps(n):
    """RK4 sub-steps of the Burgers steps (dt 1e-2, viscosity 0.005, period pi) with some headroom."""
    return max(2, math.ceil(1e-2 * (4 * 0.005 * (n / math.pi) ** 2 + 4 * n / math.pi) / 2.2))


def _burgers(case, seed):
    """burgers: the initial profile of the reference's Burgers test (data_agnostic_approximation.jl:35-44)
    plus a Fourier sine series with random coefficients, one sample per column, period pi; gradient: a sine
    series with random coefficients on [0, 1). As rank-r factors (host), with viscosity, cell and step."""
    n, m, r = case["n"], case["m"], case["r"]
    rng = np.random.default_rng(seed)
    if case["kind"] == "burgers":
        nu, dx, dt = 0.005, math.pi / n, 1e-2
        x = dx / 2 + dx * np.arange(n)
        modes = np.stack([np.sin(2 * k * x) for k in range(1, r + 4)], axis=1)
        amp = 0.5 / np.arange(1, r + 4) ** 1.5
        xi = rng.uniform(-1.0, 1.0, (r + 3, m))
        profile = 0.5 * (np.exp(np.cos(2 * x)) - 1.5) * np.sin(2 * x + 0.74 * math.pi)
        left = np.concatenate([profile[:, None], modes * amp], axis=1)
        right = np.concatenate([np.ones((1, m)), xi], axis=0)
    else:
        nu, dx, dt = 1e-2, 1.0 / n, 1e-4
        x = dx * np.arange(n)
        left = np.stack([np.sin(2 * math.pi * k * x) / k for k in range(1, r + 1)], axis=1)
        right = rng.standard_normal((r, m))
    Ql, Rl = np.linalg.qr(left)
    Qr, Rr = np.linalg.qr(right.T)
    A, s, Bt = np.linalg.svd(Rl @ Rr.T)
    return np.asfortranarray(Ql @ A[:, :r]), np.diag(s[:r]), np.asfortranarray(Qr @ Bt[:r].T), nu, dx, dt


def _prepare_burgers(lri, case, seed):
    n, m = case["n"], case["m"]
    U, S, V, nu, dx, dt = _burgers(case, seed)
    A = lri.SymTridiagonal(-2.0 * nu / dx ** 2 * np.ones(n), nu / dx ** 2 * np.ones(n), periodic=True)
    B = lri.SymTridiagonal(np.zeros(m), np.zeros(m - 1))
    D = lri.Tridiagonal(-0.5 / dx * np.ones(n), np.zeros(n), 0.5 / dx * np.ones(n), periodic=True)
    prob = lri.MatrixDEProblem(lri.QuadraticOperator(A, B, D), lri.SVDLikeRepresentation(U, S, V),
                               (0.0, case["steps"] * dt))
    return dict(case=case, lri=lri, prob=prob, alg=_algorithm(lri, case["alg"]), dt=dt)


def _members(case, seed):
    """Sizes log-uniform, ranks uniform; smooth orthonormal factors, singular values 10^(-i/8)."""
    rng = np.random.default_rng(seed)
    ns = np.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"]), case["count"])).astype(int)
    rs = rng.integers(case["rmin"], case["rmax"] + 1, case["count"])
    g = _gen(seed)
    ns, rs = ns.tolist(), rs.tolist()
    return [(n, r, _smooth(n, r, g), 10.0 ** (-torch.arange(r, device=DEV, dtype=torch.float64) / 8), _smooth(n, r, g))
            for n, r in zip(ns, rs)]


BATCH = dict(dt=2e-5, tol=1e-7, cap=64)


def _prepare_batch(lri, case, seed):
    mem, cap = _members(case, seed), BATCH["cap"]
    b = lri.native.Batch([x[0] for x in mem], [x[0] for x in mem], [cap] * len(mem))
    sub, start = [], []
    for (n, r, U, s, V), c in zip(mem, b.members):
        L = lri.laplacian_1d(n)
        c.set_operator_lyapunov(L.d, L.e, False, L.d, L.e, False)
        c.set_resident_eigenbasis(True)
        sub.append(_heat_substeps(L.d, L.e, BATCH["dt"]))
        start.append(_host(U, s, V))
    top = case["nmax"]
    U, V = (torch.zeros(len(mem), cap, top, device=DEV, dtype=torch.float64) for _ in range(2))
    S = torch.zeros(len(mem), cap, cap, device=DEV, dtype=torch.float64)
    return dict(case=case, lri=lri, batch=b, sub=np.array(sub, dtype=np.int64), start=start, U=U, S=S, V=V, top=top,
                probe=torch.randn(top, generator=_gen(seed, 2), device=DEV, dtype=torch.float64))


# ---------------------------------------------------------------------------------------------- run


def run(state):
    return {"solve": _run_solve, "data": _run_data, "adjoint": _run_adjoint, "de": _run_de, "burgers": _run_burgers,
            "gradient": _run_gradient, "batch": _run_batch}[state["case"]["kind"]](state)


def _run_solve(st):
    sol = st["lri"].solve(st["prob"], st["alg"])
    return [np.stack([y.U for y in sol.Y]), np.stack([y.S for y in sol.Y]), np.stack([y.V for y in sol.Y])]


def _finish(st):
    """The final factors on the device. After rank adaptation S is diagonal: K = U S and L = V S', with the sign
    of each singular pair that makes probe' U positive."""
    f, k = st["out"], _get_state(st["lri"], st["ctx"], st["out"])
    if st["case"]["alg"] != "bug_ra":
        return [f.U, f.S, f.V, k]
    s = (torch.sign(f.U @ st["probe"]) * torch.diagonal(f.S))[:, None]
    return [f.U * s, f.S, f.V * s, k]


def _run_data(st):
    case, lri, ctx = st["case"], st["lri"], st["ctx"]
    alg = case["alg"]
    _set_state(lri, ctx, st["start"])
    for at in _pairs(case):
        if alg == "ksl":
            ctx.step_ksl(lri.native.PRIMAL, *at)
        elif alg == "dual":
            ctx.step_ksl(lri.native.DUAL, *at)
        elif alg == "strang":
            ctx.step_ksl_strang(*at)
        elif alg == "bug":
            ctx.step_bug(*at)
        elif alg == "greedy":
            ctx.step_greedy(at[1])
        else:
            ctx.step_bug_ra(*at, _ra_tol(case), 64)
    return _finish(st)


def _run_adjoint(st):
    """Reverse steps at the context's state over the increments, last first, the cotangents updated in place."""
    case, ctx, f, b = st["case"], st["ctx"], st["out"], st["bar"]
    f.U.copy_(b.U)
    f.S.copy_(b.S)
    f.V.copy_(b.V)
    torch.cuda.current_stream().synchronize()  # the library reads them on its own stream
    for at in reversed(_pairs(case)):
        ctx.step_adjoint_ptr(case["alg"], *at, f.U.data_ptr(), f.n, f.S.data_ptr(), f.r, f.V.data_ptr(), f.m)
    return [f.U, f.S, f.V]


def _run_de(st):
    case, ctx = st["case"], st["ctx"]
    ctx.set_state(*st["start"])
    for _ in range(case["steps"]):
        if case["alg"] == "bug":
            ctx.step_de_bug(case["dt"], st["substeps"])
        else:
            ctx.step_de_bug_ra(case["dt"], st["substeps"], BATCH["tol"], 64)
    return _finish(st)


def _run_burgers(st):
    sol = st["lri"].solve(st["prob"], st["alg"], st["dt"], substeps=st["case"]["substeps"])
    return [np.stack([y.U for y in sol.Y[1:]]), np.stack([y.S for y in sol.Y[1:]]), np.stack([y.V for y in sol.Y[1:]])]


def _loss(U, S, V):
    """|| mean over the columns of U S V' ||^2 and its gradient."""
    w = S @ V.mean(axis=0)
    z = U @ w
    back = 2.0 * (U.T @ z)
    return float(z @ z), 2.0 * np.outer(z, w), np.outer(back, V.mean(axis=0)), \
        np.outer(np.full(V.shape[0], 1.0 / V.shape[0]), S.T @ back)


def _run_gradient(st):
    case = st["case"]
    value, bars, scales = st["lri"].solve_gradient(st["prob"], st["alg"], _loss, st["dt"],
                                                   checkpoint=case["checkpoint"], substeps=case["substeps"])
    return [value, *bars, scales[0]]  # scales[1] is the derivative along B = 0


def _run_batch(st):
    lri, b = st["lri"], st["batch"]
    for f, c in zip(st["start"], b.members):
        c.set_state(*f)
    for _ in range(st["case"]["steps"]):
        ranks = b.step_de_bug_ra(BATCH["dt"], st["sub"], BATCH["tol"], BATCH["cap"])
    b.synchronize()
    L, top, cap = lri.native.lib(), st["top"], BATCH["cap"]
    k = ctypes.c_int64()
    for i, c in enumerate(b.members):
        lri.native.check(L.lri_get_state(c.h, ctypes.byref(k), _ptr(st["U"][i]), top, _ptr(st["S"][i]), cap,
                                         _ptr(st["V"][i]), top), c.h)
    s = (torch.sign(st["U"] @ st["probe"]) * torch.diagonal(st["S"], dim1=1, dim2=2))[:, :, None]  # as _finish
    return [st["U"] * s, st["S"], st["V"] * s, ranks]


# --------------------------------------------------------------------------------- work, tolerance


def work(case):
    """Bytes: each snapshot that a product needs is read once per product that depends on the one before
    it (dA V0 and dA' U0 share one read), and the factors are read and written once per step. Flops: the
    products, 2 n m r each, or the row and core work of a step."""
    k, steps = case["kind"], case.get("steps", 1)
    if k in ("solve", "data", "adjoint"):
        n, m, r = case["n"], case["m"], case["r"]
        alg = case["alg"]
        e = BYTES[case.get("dtype", "f64")]
        reads, prods = {"ksl": (2, 2), "dual": (2, 2), "strang": (4, 4), "bug": (2, 3), "bug_ra": (2, 4),
                        "greedy": (2, 3), "ksl_dual": (4, 4)}[alg]
        if k == "adjoint":  # with the forward step recomputed
            reads, prods = (3, 6) if alg == "bug" else (4, 4)
        snaps = 1 if alg == "greedy" else 2
        return {"bytes": steps * (reads * snaps * n * m * e + 16.0 * (n + m + r) * r),
                "flops": steps * (2.0 * prods * n * m * r + 8.0 * (n + m) * r * r)}
    if k == "de":
        n, r = case["n"], case["r"]
        return {"bytes": steps * 32.0 * n * r, "flops": steps * (16.0 * n * r * r)}
    if k in ("burgers", "gradient"):
        n, m, r = case["n"], case["m"], case["r"]
        stages = 4 * case["substeps"]
        per = stages * 2.0 * ((n + m) * r ** 3 + 3 * r ** 4)  # the quadratic terms through their tensors
        times = 1 if k == "burgers" else 4  # forward, recomputed twice over, and reversed
        return {"bytes": steps * 16.0 * (n + m + r) * r * times, "flops": steps * per * times}
    n = math.sqrt(case["nmin"] * case["nmax"])
    r = (case["rmin"] + case["rmax"]) / 3
    return {"bytes": case["count"] * (steps * 32.0 * n * r + 16.0 * n * n),
            "flops": case["count"] * steps * 32.0 * n * r * r}


def tolerance(case):
    """About four times the largest error against exact() over some 60 drawn cases."""
    k = case["kind"]
    if k in ("data", "adjoint") and case["dtype"] != "f64":
        return {"rel": 2e-6}  # three BF16 products per FP32 one, or FP32, with FP32 sums
    if k == "batch" or k == "de":
        return {"rel": 1e-6}  # FP64, times the conditioning of the graded bases that stiff flows leave
    if k in ("gradient", "adjoint"):
        return {"rel": 1e-7}  # FP64, times the conditioning of R in the reverse QR
    return {"rel": 1e-11}


# -------------------------------------------------------------------------------------------- exact


def _qr(A):
    """QR with a positive diagonal of R, of a tensor on the device, on the host (differentiable)."""
    Q, R = torch.linalg.qr(A.cpu())
    s = torch.where(torch.diagonal(R) < 0, -1.0, 1.0)
    return (Q * s).to(A.device), (R * s[:, None]).to(A.device)


def _tail_rank(s, tol, cap):
    tail = np.sqrt(np.append(np.cumsum(s[::-1] ** 2)[::-1], 0.0))
    return min(cap, next(k for k in range(1, len(s) + 1) if tail[k] <= tol))


def _truncate(Uh, Sh, Vh, tol, probe):
    a, s, bt = torch.linalg.svd(Sh.cpu())
    k = _tail_rank(s.numpy(), tol, 64)
    U, V, s = Uh @ a[:, :k].to(DEV), Vh @ bt[:k].t().to(DEV), s[:k].to(DEV)
    return U, torch.diag(s), V, torch.sign(probe @ U) * s  # the last as _finish scales U and V


def _step(alg, U, S, V, D):
    """One step over the increment (or, for greedy, the snapshot) D, given by D(X) = D X and D(X, True) = D' X."""
    if alg == "ksl":
        P = D(V)
        U1, R = _qr(U @ S + P)
        V1, R = _qr(V @ (R - U1.t() @ P).t() + D(U1, True))
        return U1, R.t(), V1
    if alg in ("dual", "ksl_dual"):
        Q = D(U, True)
        V1, R = _qr(V @ S.t() + Q)
        U1, R = _qr(U @ (R.t() - Q.t() @ V1) + D(V1))
        return U1, R, V1
    if alg == "bug":
        U1, _ = _qr(U @ S + D(V))
        V1, _ = _qr(V @ S.t() + D(U, True))
        return U1, (U1.t() @ U) @ S @ (V.t() @ V1) + U1.t() @ D(V1), V1
    U1, _ = _qr(D(V))
    V1, _ = _qr(D(U, True))
    return U1, U1.t() @ D(V1), V1


def exact(case, seed):
    if case["kind"] in ("solve", "data", "adjoint"):
        return _exact_data(case, seed)
    if case["kind"] == "de":
        return _exact_de(case, seed)
    if case["kind"] == "batch":
        return _exact_batch(case, seed)
    return _exact_burgers(case, seed)


def _exact_data(case, seed):
    alg = case["alg"]
    whole = case["kind"] == "solve"
    at = dict(case, dtype=case.get("dtype", "f64"))
    X, U, S, V = _snapshots(at, seed, case["steps"] + 1 if whole else _count(case))

    def increment(p, q):
        W = X[q].double() if p is None else X[q].double() - X[p].double()  # m x n, the transpose
        return lambda Z, t=False: W @ Z if t else W.t() @ Z

    if whole:
        Y = [(U, S, V)]
        for k in range(case["steps"]):
            Y.append(_step(alg, *Y[-1], increment(k, k + 1)))
        return [torch.stack([y[i] for y in Y]) for i in range(3)]
    if case["kind"] == "adjoint":
        n, m, r = case["n"], case["m"], case["r"]
        g = _gen(seed, 1)
        bars = [torch.randn(*s, generator=g, device=DEV, dtype=torch.float64) for s in ((n, r), (r, r), (m, r))]
        for p, q in reversed(_pairs(case)):
            ins = [x.clone().requires_grad_(True) for x in (U, S, V)]
            bars = list(torch.autograd.grad(_step(alg, *ins, increment(p, q)), ins, bars))
        return [x.t().contiguous() for x in bars]
    sign = None
    if alg == "bug_ra":
        probe = torch.randn(case["n"], generator=_gen(seed, 2), device=DEV, dtype=torch.float64)
    for pq in _pairs(case):
        if alg == "strang":
            U, S, V = _step("ksl", U, S, V, increment(pq[0], pq[1]))
            U, S, V = _step("dual", U, S, V, increment(pq[1], pq[2]))
        elif alg == "bug_ra":
            D = increment(*pq)
            Uh, _ = _qr(torch.cat([U, U @ S + D(V)], 1))
            Vh, _ = _qr(torch.cat([V, V @ S.t() + D(U, True)], 1))
            Sh = (Uh.t() @ U) @ S @ (V.t() @ Vh) + Uh.t() @ D(Vh)
            U, S, V, sign = _truncate(Uh, Sh, Vh, _ra_tol(case), probe)
        elif alg == "greedy":
            U, S, V = _step(alg, U, S, V, increment(None, pq[1]))
        else:
            U, S, V = _step(alg, U, S, V, increment(*pq))
    return _laid_out(U, S, V, sign, _rank_cap(case))


def _laid_out(U, S, V, sign, cap):
    """As _finish returns it: column-major, zero columns up to the capacity."""
    k = U.shape[1]
    f = _Factors(U.shape[0], V.shape[0], cap)
    f.U[:k], f.S[:k, :k], f.V[:k] = (U if sign is None else U * sign).t(), S.t(), (V if sign is None else V * sign).t()
    return [f.U, f.S, f.V, k]


def _flow(z, N):
    """N RK4 steps of y' = a y + b as y -> g y + (g - 1) b / a, for z = h a; returns g."""
    return (1 + z * (1 + z / 2 * (1 + z / 3 * (1 + z / 4)))) ** N


def _sub(Y, lam, mu, F, dt, N):
    """N RK4 steps of Y_ij' = (lam_i + mu_j) Y_ij + F_ij."""
    a = lam[:, None] + mu[None, :]
    g = _flow(a * (dt / N), N)
    return g * Y + (g - 1) * F / a


def _eigen(d, e, constant):
    n = len(d)
    if constant:  # e tridiag(1, -2, 1); 2 cos(x) - 2 = -4 sin(x / 2)^2 without its cancellation
        k = torch.arange(1, n + 1, device=DEV, dtype=torch.float64)
        return -4.0 * float(e[0]) * torch.sin(k * (math.pi / (2 * (n + 1)))) ** 2, _sines(n, n)
    w, Q = np.linalg.eigh(np.diag(d) + np.diag(e, 1) + np.diag(e, -1))
    return torch.from_numpy(w).to(DEV), torch.from_numpy(Q).to(DEV)


def _de_step(ra, U, S, V, lam, f, h, dt, N, probe, tol):
    """A (rank-adaptive) BUG step of X' = diag(lam) X + X diag(lam) + f h' in the eigenbasis."""
    def side(U, S, V, f, h):  # K' = A K + K (V'BV) + f (h'V)
        mu, W = torch.linalg.eigh(((V.t() * lam) @ V).cpu())
        mu, W = mu.to(DEV), W.to(DEV)
        return _sub(U @ S @ W, lam, mu, torch.outer(f, h @ V @ W), dt, N) @ W.t()

    K, L = side(U, S, V, f, h), side(V, S.t(), U, h, f)
    U1, _ = _qr(torch.cat([U, K], 1) if ra else K)
    V1, _ = _qr(torch.cat([V, L], 1) if ra else L)
    al, Wa = (x.to(DEV) for x in torch.linalg.eigh(((U1.t() * lam) @ U1).cpu()))
    be, Wb = (x.to(DEV) for x in torch.linalg.eigh(((V1.t() * lam) @ V1).cpu()))
    S0 = Wa.t() @ (U1.t() @ U) @ S @ (V.t() @ V1) @ Wb
    S1 = Wa @ _sub(S0, al, be, torch.outer(Wa.t() @ (U1.t() @ f), Wb.t() @ (V1.t() @ h)), dt, N) @ Wb.t()
    return _truncate(U1, S1, V1, tol, probe) if ra else (U1, S1, V1, None)


def _exact_de(case, seed):
    U, s, V, a, b, d, e = _heat(case, seed)
    lam, Q = _eigen(d, e, not case["variable"])
    probe = torch.randn(case["n"], generator=_gen(seed, 2), device=DEV, dtype=torch.float64)
    N = _heat_substeps(d, e, case["dt"])
    U, S, V, f, h, p = Q.t() @ U, torch.diag(s), Q.t() @ V, Q.t() @ a, Q.t() @ b, Q.t() @ probe
    for _ in range(case["steps"]):
        U, S, V, sign = _de_step(case["alg"] == "bug_ra", U, S, V, lam, f, h, case["dt"], N, p, BATCH["tol"])
    return _laid_out(Q @ U, S, Q @ V, sign, min(64, case["n"]) if case["alg"] == "bug_ra" else case["r"])


def _exact_batch(case, seed):
    mem, cap, top = _members(case, seed), BATCH["cap"], case["nmax"]
    probe = torch.randn(top, generator=_gen(seed, 2), device=DEV, dtype=torch.float64)
    Us, Vs = (torch.zeros(len(mem), cap, top, device=DEV, dtype=torch.float64) for _ in range(2))
    Ss, ranks = torch.zeros(len(mem), cap, cap, device=DEV, dtype=torch.float64), []
    for i, (n, r, U, s, V) in enumerate(mem):
        d, e = -2.0 * float(n * n) * np.ones(n), float(n * n) * np.ones(n - 1)
        lam, Q = _eigen(d, e, True)
        N, z = _heat_substeps(d, e, BATCH["dt"]), torch.zeros(n, device=DEV, dtype=torch.float64)
        U, S, V, p = Q.t() @ U, torch.diag(s), Q.t() @ V, Q.t() @ probe[:n]
        for _ in range(case["steps"]):
            U, S, V, sign = _de_step(True, U, S, V, lam, z, z, BATCH["dt"], N, p, BATCH["tol"])
        k = U.shape[1]
        ranks.append(k)
        Us[i, :k, :n], Vs[i, :k, :n], Ss[i, :k, :k] = (Q @ (U * sign)).t(), (Q @ (V * sign)).t(), S
    return [Us, Ss, Vs, np.array(ranks, dtype=np.int64)]


def _exact_burgers(case, seed):
    U, S, V, nu, dx, dt = _burgers(case, seed)
    U, S, V = (torch.from_numpy(np.ascontiguousarray(x)).to(DEV) for x in (U, S, V))
    N, alg = case["substeps"], case["alg"]
    h = dt / N

    def F(Y, c):  # c nu u_xx - u u_x, periodic, central differences
        up, dn = torch.roll(Y, -1, 0), torch.roll(Y, 1, 0)
        return (c * nu / dx ** 2) * (up - 2 * Y + dn) - (up - dn) * (0.5 / dx) * Y

    def rk4(f, y):
        for _ in range(N):
            a = f(y)
            b = f(y + h / 2 * a)
            c = f(y + h / 2 * b)
            d = f(y + h * c)
            y = y + h / 6 * (a + 2 * b + 2 * c + d)
        return y

    def step(U, S, V, c):
        K = rk4(lambda K: F(K @ V.t(), c) @ V, U @ S)
        U1, R = _qr(K)
        if alg == "ksl":
            S1 = rk4(lambda Z: -(U1.t() @ F(U1 @ Z @ V.t(), c) @ V), R)
            V1, R = _qr(rk4(lambda L: F(U1 @ L.t(), c).t() @ U1, V @ S1.t()))
            return U1, R.t(), V1
        V1, _ = _qr(rk4(lambda L: F(U @ L.t(), c).t() @ U, V @ S.t()))
        S0 = (U1.t() @ U) @ S @ (V.t() @ V1)
        return U1, rk4(lambda Z: U1.t() @ F(U1 @ Z @ V1.t(), c) @ V1, S0), V1

    one = torch.ones((), device=DEV, dtype=torch.float64)
    Y = [(U, S, V)]
    for _ in range(case["steps"]):
        Y.append(step(*Y[-1], one))
    if case["kind"] == "burgers":
        return [torch.stack([y[i] for y in Y[1:]]) for i in range(3)]
    ins = [x.clone().requires_grad_(True) for x in Y[-1]]
    value = (ins[0] @ (ins[1] @ ins[2].mean(0))).square().sum()
    bars, scale = list(torch.autograd.grad(value, ins)), torch.zeros_like(one)
    for y in reversed(Y[:-1]):
        ins = [x.clone().requires_grad_(True) for x in (*y, one)]
        *bars, c = torch.autograd.grad(step(*ins), ins, bars)
        scale = scale + c
    return [float(value.detach()), *bars, float(scale)]
