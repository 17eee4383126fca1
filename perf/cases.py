"""The work that programs have this library do, as cases that can be timed.

A case is a dict of plain values.  listed() names the fixed ones, draw() gives
further ones of the same ranges, prepare() makes what a program holds before the
call (seeded inputs on the device, and the plan where it keeps one), run() is one
pass through the public entry points, exact() the same results in 64 bits from
plain torch, work() the bytes and operations a pass cannot do without.

Inputs are LQR Schur complements with random stable dynamics (A = I + dt G), the
systems that trajectory optimisation solves at every step; the initial guess is
zero unless the case re-solves a shifted horizon.  FP32 solves stop at a relative
residual of 1e-5, FP64 ones at 1e-10.  Ranges: stateSize 2 to 32 (FP64: to 24,
and 28), horizons 3 to 512, batches of 4 to 512 systems.

Kinds:
  solve   synchronous solve on device tensors, Pinv given (a control loop that
          needs lambda and the record before it goes on)
  form    the same with no Pinv: the library forms it (the reference's default)
  async   stream-ordered solve, the result left on the device
  host    the host-pointer call on numpy arrays (the reference's call shape)
  train   differentiable solve: forward, then backward to gamma and S
  step    one step of a controller on the device: Schur complement, symmetric
          stair preconditioner, solve
  batch   a plan over many systems, run once
"""
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "gbd-pcg_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "gbd-pcg_amd"))

import gbdpcg  # noqa: E402
from gbdpcg.autograd import pcg_solve  # noqa: E402

MAX_ITER = 173
_RECUR = {"fused": gbdpcg.RECUR_FUSED, "reference": gbdpcg.RECUR_REFERENCE}
_DTYPE = {"f32": torch.float32, "f64": torch.float64}


def listed():
    return [
        # the smallest call: the size of the compile example, block-Jacobi, waited for
        dict(name="solve_n2_N3", kind="solve", dtype="f32", n=2, N=3, recurrence="reference", precond="jacobi"),
        # a quadrotor with a quaternion attitude, an odd horizon, everything left at the defaults
        dict(name="form_n13_N50", kind="form", dtype="f32", n=13, N=50, recurrence="reference", precond="ss"),
        # the benchmark's system: a seven-joint arm, 128 knots
        dict(name="async_n14_N128", kind="async", dtype="f32", n=14, N=128, recurrence="fused", precond="ss"),
        # a long horizon in double precision
        dict(name="async_n14_N256_f64", kind="async", dtype="f64", n=14, N=256, recurrence="fused", precond="ss"),
        # a floating-base model in double precision, the reference's iteration
        dict(name="async_n18_N75_f64", kind="async", dtype="f64", n=18, N=75, recurrence="reference", precond="ss"),
        # the reference's own call: host arrays in, host lambda out
        dict(name="host_n12_N64", kind="host", dtype="f32", n=12, N=64, recurrence="reference", precond="ss"),
        # a differentiable layer
        dict(name="train_n14_N64", kind="train", dtype="f32", n=14, N=64, recurrence="fused", precond="ss"),
        # a quadrotor's controller step from its linearisation
        dict(name="step_n12_N100", kind="step", dtype="f32", n=12, N=100, recurrence="fused", precond="ss"),
        # a training batch: 64 horizons, both directions
        dict(name="batch64_n14_N128", kind="batch", dtype="f32", sizes="14", N_lo=128, N_hi=128, count=64,
             adjoint=True, recurrence="fused", warm=False),
        # many uneven problems of the sizes of common robots
        dict(name="batch512_uneven", kind="batch", dtype="f32", sizes="6,12,14,28", N_lo=16, N_hi=256, count=512,
             adjoint=False, recurrence="fused", warm=False),
        # arbitrary sizes with the plan's default recurrence
        dict(name="batch96_any", kind="batch", dtype="f32", sizes="3,4,7,9,10,13,17,20,24,31", N_lo=5, N_hi=120,
             count=96, adjoint=False, recurrence="reference", warm=False),
        # receding-horizon re-solve of large systems in double precision, both directions
        dict(name="resolve32_n28_N512_f64", kind="batch", dtype="f64", sizes="28", N_lo=512, N_hi=512, count=32,
             adjoint=True, recurrence="fused", warm=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["solve", "form", "async", "async", "host", "train", "step", "batch", "batch", "batch"])
    dtype = "f64" if rng.random() < 0.3 else "f32"
    top = 24 if dtype == "f64" else 32
    case = dict(kind=kind, dtype=dtype, recurrence=rng.choice(["fused", "reference"]))
    if kind == "batch":
        count = _log_int(rng, 4, 256)
        case["sizes"] = ",".join(str(s) for s in sorted(rng.sample(range(2, top + 1), rng.choice([1, 2, 4]))))
        case["N_lo"] = _log_int(rng, 3, 64)
        case["N_hi"] = case["N_lo"] + rng.randrange(0, 129)
        case.update(count=count, adjoint=rng.random() < 0.4, warm=rng.random() < 0.3)
        return case
    case.update(n=rng.randrange(2, top + 1), N=_log_int(rng, 3, 512),
                precond="ss" if kind in ("train", "step") else rng.choice(["ss", "ss", "jacobi"]))
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _tol(case):
    return 1e-10 if case["dtype"] == "f64" else 1e-5


def _shapes(case):
    """(n, N) of every system of a case: stateSizes in turn, horizons spread over
    the range by a fixed stride."""
    if case["kind"] != "batch":
        return [(case["n"], case["N"])]
    sizes = [int(s) for s in case["sizes"].split(",")]
    span = case["N_hi"] - case["N_lo"] + 1
    return [(sizes[i % len(sizes)], case["N_lo"] + (i * 37) % span) for i in range(case["count"])]


def _invert(M):
    """Inverses of a batch of positive definite matrices (Gauss-Jordan, in place)."""
    for c in range(M.shape[-1]):
        piv = M[:, c, c].clone()
        row = M[:, c, :] / piv[:, None]
        col = M[:, :, c].clone()
        M -= col[:, :, None] * row[:, None, :]
        M[:, c, :] = row
        M[:, :, c] = -col / piv[:, None]
        M[:, c, c] = 1 / piv
    return M


def _linearisation(n, m, knots, gen, dev):
    """A, B, Q, R of `knots` stages (Q and R diagonal), in 64 bits."""
    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=dev, dtype=torch.float64)

    def uniform(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=gen, device=dev, dtype=torch.float64)
    A = torch.eye(n, device=dev, dtype=torch.float64) + 0.1 * 0.1 * normal(knots, n, n)
    return A, 0.1 * normal(knots, n, m), uniform(0.1, 10.0, knots, n), uniform(0.01, 1.0, knots, m)


def _schur(A, B, Q, R, first):
    """theta (k, k) and phi (k, k-1) of a chain of stages; `first` marks the first
    knot of each system, which has no predecessor."""
    keep = (~first).to(A.dtype)[:, None, None]
    Ap, Bp, Qp, Rp = A.roll(1, 0), B.roll(1, 0), Q.roll(1, 0), R.roll(1, 0)
    AQ = Ap / Qp[:, None, :]
    theta = keep * (AQ @ Ap.mT + (Bp / Rp[:, None, :]) @ Bp.mT) + torch.diag_embed(1 / Q)
    return (theta + theta.mT) / 2, -AQ * keep


def _cbtd(diag, low, first):
    """Block rows (k, k-1), (k, k), (k, k+1), each column-major, with the upper
    blocks the transposes of the lower ones."""
    up = (low.mT * (~first).to(low.dtype)[:, None, None]).roll(-1, 0)
    return torch.stack([low.mT, diag.mT, up.mT], 1)


def _stair(theta, phi, first, kind):
    inv = _invert(theta.clone())
    low = torch.zeros_like(phi) if kind == "jacobi" else -inv @ phi @ inv.roll(1, 0)
    return _cbtd(inv, low, first)


def _first(Ns, dev):
    first = torch.zeros(sum(Ns), dtype=torch.bool, device=dev)
    at = 0
    for N in Ns:
        first[at] = True
        at += N
    return first


def _inputs(case, seed):
    """The systems of a case, as tensors on the device: every system's S, Pinv,
    gamma, g_lambda (and the guess), in the case's precision."""
    dev, dt = torch.device("cuda"), _DTYPE[case["dtype"]]
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    shapes = _shapes(case)
    out = [None] * len(shapes)
    for n in sorted({s[0] for s in shapes}):
        which = [i for i, s in enumerate(shapes) if s[0] == n]
        Ns = [shapes[i][1] for i in which]
        first, knots = _first(Ns, dev), sum(Ns)
        A, B, Q, R = (x.to(dt).double() for x in _linearisation(n, max(n // 2, 1), knots, gen, dev))
        vec = torch.randn(3, knots, n, generator=gen, device=dev, dtype=torch.float64).to(dt)
        lqr = [x.to(dt) for x in (A, B, Q, R)]
        if case["kind"] == "step":
            S = P = None
        else:
            theta, phi = _schur(A, B, Q, R, first)
            S = _cbtd(theta, phi, first).to(dt)
            P = _stair(theta, phi, first, case.get("precond", "ss")).to(dt)
        at = 0
        for i, N in zip(which, Ns):
            s = slice(at, at + N)
            out[i] = dict(n=n, N=N, gamma=vec[0, s].reshape(-1).clone(), glam=vec[1, s].reshape(-1).clone(),
                          guess=vec[2, s].reshape(-1).clone())
            if S is not None:
                out[i].update(S=S[s].reshape(-1).clone(), Pinv=P[s].reshape(-1).clone())
            if case["kind"] == "step":
                out[i].update(lqr=[x[s].contiguous() for x in lqr])
            at += N
    return out


def _pool(lengths, dt, dev):
    """One buffer holding a tensor of each length, each on a 256-byte boundary."""
    step = 256 // torch.empty(0, dtype=dt).element_size()
    at, views = 0, []
    for c in lengths:
        views.append((at, c))
        at += -(-c // step) * step
    buf = torch.zeros(at, dtype=dt, device=dev)
    return buf, [buf[a:a + c] for a, c in views]


def _pooled(parts):
    buf, views = _pool([p.numel() for p in parts], parts[0].dtype, parts[0].device)
    for v, p in zip(views, parts):
        v.copy_(p)
    return buf, views


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def prepare(case, seed):
    systems = _inputs(case, seed)
    kw = dict(tol=_tol(case), max_iter=MAX_ITER, exit_mode=gbdpcg.EXIT_REL_RESID,
              recurrence=_RECUR[case["recurrence"]])
    one = systems[0]
    st = dict(kind=case["kind"], kw=kw, n=one["n"], N=one["N"], dtype=_DTYPE[case["dtype"]])
    if case["kind"] != "batch":
        st.update(gamma=one["gamma"], lam=torch.zeros_like(one["gamma"]), glam=one["glam"])
        if "S" in one:
            st.update(S=one["S"], Pinv=one["Pinv"])
        if case["kind"] == "form":
            st["precond"] = gbdpcg.PRECOND_SS if case["precond"] == "ss" else gbdpcg.PRECOND_JACOBI
        if case["kind"] == "host":
            st.update({k: st[k].cpu().numpy() for k in ("S", "Pinv", "gamma", "lam")})
        if case["kind"] == "train":
            st["S"].requires_grad_(True)
            st["gamma"].requires_grad_(True)
        if case["kind"] == "step":
            st.update(lqr=one["lqr"], m=max(one["n"] // 2, 1), S=torch.empty(one["N"] * 3 * one["n"] ** 2,
                      dtype=st["dtype"], device="cuda"))
            st["Pinv"] = torch.empty_like(st["S"])
        return st
    guess, _ = _pooled([s["guess"] for s in systems])
    st["guess"] = guess if case["warm"] else torch.zeros_like(guess)
    st["gamma0"], _ = _pooled([s["gamma"] for s in systems])
    st["gamma"], gammas = _pooled([s["gamma"] for s in systems])
    st["lam"], lams = _pool([s["gamma"].numel() for s in systems], st["dtype"], guess.device)
    st["warm"], st["adjoint"], st["seed"] = case["warm"], case["adjoint"], seed
    plan = [dict(S=s["S"], Pinv=s["Pinv"], gamma=g, lam=l, n=s["n"], N=s["N"]) for s, g, l in
            zip(systems, gammas, lams)]
    if case["adjoint"]:
        st["ggamma"], ggs = _pool([s["gamma"].numel() for s in systems], st["dtype"], guess.device)
        st["gS"], gSs = _pool([s["S"].numel() for s in systems], st["dtype"], guess.device)
        for d, s, gg, gS in zip(plan, systems, ggs, gSs):
            d.update(adjoint=True, glam=s["glam"], ggamma=gg, gS=gS)
    st["plan"] = gbdpcg.Batch(plan, tol=kw["tol"], max_iter=MAX_ITER, exit_mode=kw["exit_mode"],
                              recurrence=kw["recurrence"])
    return st


def run(st):
    kind, n, N, kw = st["kind"], st["n"], st["N"], st["kw"]
    if kind == "solve":
        st["lam"].zero_()
        gbdpcg.solve(st["S"], st["gamma"], st["lam"], n, N, st["Pinv"], **kw)
        return st["lam"]
    if kind == "form":
        st["lam"].zero_()
        gbdpcg.solve(st["S"], st["gamma"], st["lam"], n, N, precond=st["precond"], **kw)
        return st["lam"]
    if kind == "async":
        st["lam"].zero_()
        gbdpcg.solve_async(st["S"], st["gamma"], st["lam"], n, N, st["Pinv"], **kw)
        return st["lam"]
    if kind == "host":
        st["lam"].fill(0)
        gbdpcg.solve_host(st["S"], st["gamma"], st["lam"], n, N, st["Pinv"], **kw)
        return st["lam"]
    if kind == "train":
        st["S"].grad = st["gamma"].grad = None
        lam = pcg_solve(st["S"], st["gamma"], st["Pinv"], n, N, **kw)
        lam.backward(st["glam"])
        return {"lam": lam.detach(), "ggamma": st["gamma"].grad, "gS": st["S"].grad}
    if kind == "step":
        gbdpcg.lqr_schur_device(*st["lqr"], st["S"], n, st["m"], N)
        gbdpcg.precond_device(st["S"], st["Pinv"], n, N)
        st["lam"].zero_()
        gbdpcg.solve_async(st["S"], st["gamma"], st["lam"], n, N, st["Pinv"], **kw)
        return {"S": st["S"], "Pinv": st["Pinv"], "lam": st["lam"]}
    st["lam"].copy_(st["guess"])
    if st["warm"]:
        # the next step of a receding horizon: the last solution moved one knot,
        # the right-hand side changed a little
        st["gamma"].copy_(st["gamma0"])
        st["plan"].warm_start(st["seed"], 1e-2)
    st["plan"].run()
    out = {"lam": st["lam"]}
    if st["warm"]:
        out["gamma"] = st["gamma"]
    if st["adjoint"]:
        out.update(ggamma=st["ggamma"], gS=st["gS"])
    return out


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _direct(S, rhs):
    """x of S x = b for systems of one stateSize: S (B, N, 3, n, n) in cbtd order,
    rhs (B, N, n, c), by block elimination on the CPU in 64 bits."""
    S = S.mT
    N = S.shape[1]
    D, b = [S[:, 0, 1]], [rhs[:, 0]]
    for k in range(1, N):
        both = torch.linalg.solve(D[-1], torch.cat([S[:, k - 1, 2], b[-1]], -1))
        n = S.shape[-1]
        D.append(S[:, k, 1] - S[:, k, 0] @ both[..., :n])
        b.append(rhs[:, k] - S[:, k, 0] @ both[..., n:])
    x = [torch.linalg.solve(D[-1], b[-1])]
    for k in range(N - 2, -1, -1):
        x.append(torch.linalg.solve(D[k], b[k] - S[:, k, 2] @ x[-1]))
    return torch.stack(x[::-1], 1)


def _gradient(lam, gg):
    """-1/2 (gg lam^T + lam gg^T) on the block-tridiagonal pattern, cbtd order."""
    N, n = lam.shape
    out = torch.zeros(N, 3, n, n, dtype=torch.float64)
    for j, s in ((0, 1), (1, 0), (2, -1)):
        L, G = lam.roll(s, 0), gg.roll(s, 0)
        out[:, j] = -0.5 * (L[:, :, None] * gg[:, None, :] + G[:, :, None] * lam[:, None, :])
    out[0, 0] = 0
    out[N - 1, 2] = 0
    return out


def _solutions(systems, adjoint):
    """lambda (and g_gamma) of every system, systems of one stateSize together
    (short horizons continued with identity blocks)."""
    for n in sorted({s["n"] for s in systems}):
        group = [s for s in systems if s["n"] == n]
        top = max(s["N"] for s in group)
        S = torch.zeros(len(group), top, 3, n, n, dtype=torch.float64)
        S[:, :, 1] = torch.eye(n, dtype=torch.float64)
        b = torch.zeros(len(group), top, n, 2, dtype=torch.float64)
        for i, s in enumerate(group):
            S[i, :s["N"]] = s["S"].double().cpu().reshape(s["N"], 3, n, n)
            b[i, :s["N"], :, 0] = s["gamma"].double().cpu().reshape(s["N"], n)
            b[i, :s["N"], :, 1] = s["glam"].double().cpu().reshape(s["N"], n)
        x = _direct(S, b if adjoint else b[..., :1])
        for i, s in enumerate(group):
            s["x"] = x[i, :s["N"], :, 0]
            if adjoint:
                s["gx"] = x[i, :s["N"], :, 1]


def exact(case, seed):
    systems = _inputs(case, seed)
    adjoint = case["kind"] == "train" or case.get("adjoint", False)
    if case["kind"] == "step":
        one = systems[0]
        first = _first([one["N"]], "cpu")
        theta, phi = _schur(*[x.double().cpu() for x in one["lqr"]], first)
        one["S"] = _cbtd(theta, phi, first)
        P = _stair(theta, phi, first, "ss")
        _solutions(systems, False)
        return {"S": one["S"].reshape(-1), "Pinv": P.reshape(-1), "lam": one["x"].reshape(-1)}
    if case.get("warm"):
        # the noise that the warm start adds is the library's own sequence, known on the host too
        for i, s in enumerate(systems):
            z = gbdpcg.counter_randn(s["n"] * s["N"], seed, i, 1e-2, dtype="float64")
            s["gamma"] = s["gamma"].double() + torch.from_numpy(z).to(s["gamma"].device)
    _solutions(systems, adjoint)
    if case["kind"] != "batch":
        lam = systems[0]["x"].reshape(-1)
        if case["kind"] != "train":
            return lam
        return {"lam": lam, "ggamma": systems[0]["gx"].reshape(-1),
                "gS": _gradient(systems[0]["x"], systems[0]["gx"]).reshape(-1)}
    place = _DTYPE[case["dtype"]]
    out = {"lam": _spread([s["x"] for s in systems], place)}
    if case["warm"]:
        out["gamma"] = _spread([s["gamma"].cpu() for s in systems], place)
    if adjoint:
        out["ggamma"] = _spread([s["gx"] for s in systems], place)
        out["gS"] = _spread([_gradient(s["x"], s["gx"]) for s in systems], place)
    return out


def _spread(parts, dt):
    """64-bit values at the offsets of a pool of type dt."""
    pool, views = _pool([p.numel() for p in parts], dt, "cpu")
    buf = torch.zeros(pool.numel(), dtype=torch.float64)
    for v, p in zip(views, parts):
        buf[v.storage_offset():v.storage_offset() + p.numel()] = p.reshape(-1)
    return buf


def work(case):
    """Each matrix and vector read once, each output written once; the operations
    of a typical iteration count at the case's tolerance."""
    size, iters = (8, 70) if case["dtype"] == "f64" else (4, 36)
    adjoint = case["kind"] == "train" or case.get("adjoint", False)
    made = case["kind"] in ("form", "step")
    values = flops = 0
    for n, N in _shapes(case):
        mat, vec = 3 * n * n * N, n * N
        values += (1 if made else 2) * mat + 3 * vec
        flops += iters * (4 * n * n * (3 * N - 2) + 10 * vec) * (2 if adjoint else 1)
        if adjoint:
            values += mat + 2 * vec
        if case["kind"] == "step":
            m = max(n // 2, 1)
            values += mat + N * (n * n + n * m + n + m)
        if made:
            flops += N * (2 * n ** 3 + 8 * n ** 3)
    return {"bytes": values * size, "flops": flops}
