"""Systems of one workgroup: adjoints of the two-rows-per-lane item (FP32, n <= 16, more
than 512 rows), exceptional values in every lone item, and outputs that are handed over
uninitialised.

Bars: those of the adjoint tests over every stateSize (tests/test_gpu_adjoint.py): counts
within one of the same-precision oracle's, lambda and g_gamma within 1e-4 of the FP64
iterate of the same count, g_S by the formula from the returned vectors."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_adjoint import _t, rel, system
from test_gpu_batched import check, make_batch
from test_gpu_parity import gpu_solve

pytestmark = pytest.mark.gpu


def two_row_horizons(n):
    """The smallest and largest N of the two-row item, and for n = 13..15 both sides of
    the 64 knots up to which a knot's rows get lanes of their own (8 of them)."""
    top = 512 // ((n + 1) // 2)
    return sorted({512 // n + 1, top} | ({64, 65} if 12 < n < 16 and top > 64 else set()))


def adjoint(S, P, g, glam, n, N, dtype, forward, lam_in, **kw):
    import gbdpcg
    a = [_t(x.astype(dtype), dtype) for x in (S, P, g, glam)]
    lam = _t(lam_in.astype(dtype), dtype)
    gg, gS = _t(np.full(n * N, np.nan, dtype), dtype), _t(np.full(3 * n * n * N, np.nan, dtype), dtype)
    res = gbdpcg.adjoint(a[0], a[2], lam, a[3], gg, gS, n, N, a[1], forward=forward, **kw)
    return *(x.cpu().numpy().astype(np.float64) for x in (lam, gg, gS)), res


@pytest.mark.parametrize("recurrence", [0, 1])
@pytest.mark.parametrize("forward", [True, False])
@pytest.mark.parametrize("n", [2, 3, 5, 8, 13, 14, 15, 16])
def test_adjoints_on_two_rows_per_lane(gpu, n, forward, recurrence):
    dtype, tol, bar = np.float32, 3e-5, 1e-4
    kw = dict(tol=tol, max_iter=600, exit_mode=1, recurrence=recurrence)
    for N in two_row_horizons(n):
        S, P, g, glam = system(n, N, 6600 + 37 * n + N, dtype)
        lam_in = np.zeros(n * N) if forward else O.pcg(S, P, g, np.zeros(n * N), n, N, 1e-8, 2000, 1)[0]
        lam, gg, gS, res = adjoint(S, P, g, glam, n, N, dtype, forward, lam_in, **kw)
        assert res.adj_status == 0 and (not forward or res.status == 0), (n, N)
        sides = [(glam, res.adj_iters, gg)] + ([(g, res.iters, lam)] if forward else [])
        for rhs, its, x in sides:
            for f in ((True, False) if recurrence == 1 else (False,)):
                _, it, *_ = O.pcg(S.astype(dtype), P.astype(dtype), rhs.astype(dtype), np.zeros(n * N, dtype), n, N,
                                  tol, 600, 1, dtype, fused=f)
                assert abs(its - it) <= 1, (n, N, its, it, f)
            ref, *_ = O.pcg(S, P, rhs, np.zeros(n * N), n, N, 0.0, its, 1, np.float64, fused=recurrence == 1)
            assert rel(x, ref) <= bar, (n, N, rel(x, ref))
        if not forward:
            assert np.array_equal(lam, lam_in.astype(dtype).astype(np.float64))
        expect = O.dense_to_cbtd(-0.5 * (np.outer(gg, lam) + np.outer(lam, gg)), n, N) * O.pattern_mask(n, N)
        assert np.allclose(gS, expect, rtol=1e-5, atol=1e-6 * np.abs(expect).max()), (n, N)


# (n, N, dtype): two rows per lane, one and two lanes per row on 512 threads, one lane per
# row on 256, the row broadcast, and 512 threads of one row per lane in FP64
LONE = [(14, 64, np.float32), (13, 73, np.float32), (5, 170, np.float32), (14, 30, np.float32), (30, 16, np.float32),
        (12, 20, np.float32), (12, 20, np.float64), (14, 12, np.float64), (6, 80, np.float64), (20, 12, np.float64)]


@pytest.mark.parametrize("n,N,dtype", LONE)
@pytest.mark.parametrize("recurrence", [0, 1])
def test_breakdown_of_lone_workgroups(gpu, n, N, dtype, recurrence):
    """p'Sp = 0 on the first direction, and r'z = 0 with r != 0, as on one wave
    (tests/test_gpu_parity.py): BREAKDOWN at iteration 0, lambda untouched."""
    import gbdpcg
    sign = np.where(np.arange(n) % 2 == 0, 1.0, -1.0)
    g = np.zeros(n * N)
    g[n * (N - 1)] = g[n * (N - 1) + 1] = 1.0
    lam0 = np.zeros(n * N, dtype)
    for s, p in ((sign, np.ones(n)), (np.full(n, 2.0), sign)):
        S, P = np.zeros((N, 3, n, n)), np.zeros((N, 3, n, n))
        S[:, 1], P[:, 1] = np.diag(s), np.diag(p)
        S, P = S.reshape(-1).astype(dtype), P.reshape(-1).astype(dtype)
        lam, res = gpu_solve(S, P, g.astype(dtype), lam0, n, N, dtype, tol=1e-6, max_iter=25, exit_mode=1,
                             recurrence=recurrence)
        _, it, st, *_ = O.pcg(S, P, g.astype(dtype), lam0, n, N, 1e-6, 25, 1, dtype, fused=recurrence == 1)
        assert st == O.BREAKDOWN and res.status == gbdpcg.BREAKDOWN and res.iters == it == 0 and not lam.any()


@pytest.mark.parametrize("n,N,dtype", LONE)
@pytest.mark.parametrize("recurrence", [0, 1])
@pytest.mark.parametrize("mode", [0, 1])
def test_exceptional_values_in_lone_workgroups(gpu, n, N, dtype, recurrence, mode):
    """NaN and infinity in the last row (the one without a partner where n is odd), an
    initial guess that solves the system, no iterations allowed, one iteration: status
    and count as the LDS-resident kernel gives them, which the oracle's tests hold."""
    import gbdpcg
    S, P, g, _ = system(n, N, 77, dtype)
    S, P, g = (a.astype(dtype) for a in (S, P, g))
    z = np.zeros(n * N, dtype)
    kw = dict(tol=1e-5, max_iter=40, exit_mode=mode, recurrence=recurrence)

    def put(a, i, v):
        b = a.copy()
        b[i] = v
        return b
    corner = (N - 1) * 3 * n * n + 2 * n * n - 1  # last element of the last diagonal block
    cases = [(S, P, put(g, -1, np.nan), z, kw), (S, P, put(g, -1, np.inf), z, kw),
             (put(S, corner, np.nan), P, g, z, kw), (S, put(P, corner, np.nan), g, z, kw),
             (S, P, z, z, kw), (S, P, g, g, dict(kw, max_iter=0)), (S, P, g, z, dict(kw, max_iter=1)),
             (S, P, g, z, dict(kw, tol=1e30))]
    want = [gbdpcg.NONFINITE] * 4 + [gbdpcg.CONVERGED, gbdpcg.MAX_ITER, gbdpcg.MAX_ITER, gbdpcg.CONVERGED]
    for i, ((a, b, c, l, k), status) in enumerate(zip(cases, want)):
        lam, res = gpu_solve(a, b, c, l, n, N, dtype, **k)
        _, ref = gpu_solve(a, b, c, l, n, N, dtype, kernel=gbdpcg.KERNEL_LDS, **k)
        assert (res.status, res.iters) == (ref.status, ref.iters) and res.status == status, (i, res.status, ref.status)
        if k["max_iter"] == 0:
            assert np.array_equal(lam, l)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("recurrence", [0, 1])
@pytest.mark.parametrize("sizes,repeat", [((14,), 1), ((6, 12, 14), 1), ((5, 13, 30), 1), ((4, 9, 15), 40)])
def test_batched_gradients_are_written_whole(gpu, dtype, recurrence, sizes, repeat):
    """g_gamma and g_S handed over full of NaN: every element is written, the padding
    blocks (zero) among them; alone and on several ranks, in one round and in several."""
    import gbdpcg
    tol = 3e-5 if dtype == np.float32 else 1e-9
    specs = [(n, N, tol) for n in sizes for N in ((4, 256 // n, 600 // n) if repeat == 1 else (256 // n + 1,))]
    systems, host = make_batch(specs, dtype, adjoint=True, seed0=16000)
    for s in systems:
        s["ggamma"].fill_(float("nan"))
        s["gS"].fill_(float("nan"))
    extra = [dict(s, lam=s["lam"].clone(), ggamma=s["ggamma"].clone(), gS=s["gS"].clone())
             for _ in range(repeat - 1) for s in systems]
    b = gbdpcg.Batch(systems + extra, exit_mode=gbdpcg.EXIT_REL_RESID, recurrence=recurrence)
    b.run()
    results = b.results()
    check(systems, host, results, dtype, recurrence, adjoint=True)
    for s, first in zip(extra, systems * (repeat - 1)):
        assert bool((s["gS"] == first["gS"]).all()) and bool((s["ggamma"] == first["ggamma"]).all())
