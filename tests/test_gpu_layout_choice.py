"""What the planners choose, by the times of whole calls: a choice that another
request of the same call beats by a margin is a fault of the planner.

Every call runs a fixed number of iterations (tolerance 0) and is the fastest of
several timed runs; the margins (10 % where both sides are the same kind of call)
are several times the spread of such minima and well below the faults they guard
against (1.2 to 1.7 times)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fastest_us(call, reps=10, tries=7):
    import torch
    for _ in range(3):
        call()
    best = float("inf")
    for _ in range(tries):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(reps):
            call()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) / reps * 1e3)
    return best


def _system(n, N, dtype):
    """Block-tridiagonal, diagonally dominant S and its block-Jacobi preconditioner."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(100 * n + N)
    S = torch.randn(N, 3, n, n, generator=gen, device="cuda", dtype=torch.float64) / (4 * n)
    S[:, 1] = (S[:, 1] + S[:, 1].mT) / 2 + torch.eye(n, device="cuda", dtype=torch.float64)
    S[1:, 0] = S[:-1, 2].mT
    P = torch.zeros_like(S)
    P[:, 1] = torch.eye(n, device="cuda", dtype=torch.float64)
    g = torch.randn(N * n, generator=gen, device="cuda", dtype=torch.float64)
    T = torch.float64 if dtype == np.float64 else torch.float32
    return S.reshape(-1).to(T), P.reshape(-1).to(T), g.to(T)


def _solve_us(n, N, dtype, recurrence, **kw):
    import torch
    import gbdpcg
    S, P, g = _system(n, N, dtype)
    lam = torch.zeros_like(g)

    def call():
        lam.zero_()
        gbdpcg.solve_async(S, g, lam, n, N, P, tol=0.0, max_iter=20, exit_mode=gbdpcg.EXIT_REL_RESID,
                           recurrence=recurrence, **kw)
    return _fastest_us(call)


@pytest.mark.parametrize("n,N,longer,recurrence", [(28, 160, 220, 1), (28, 192, 220, 1), (12, 850, 1500, 0),
                                                   (12, 1000, 1500, 1), (14, 550, 900, 1)])
def test_longer_horizons_are_no_faster(gpu, n, N, longer, recurrence):
    """FP32: an iteration on `longer` knots does all that one on N knots does.  (Four
    workgroups of one solve sharing each CU of an XCD made the shorter one slower.)"""
    short, full = (_solve_us(n, k, np.float32, recurrence) for k in (N, longer))
    assert short <= 1.1 * full, (short, full)


@pytest.mark.parametrize("dtype,n,N", [(np.float32, 15, 3000), (np.float32, 16, 3000), (np.float32, 24, 1200),
                                       (np.float32, 20, 2000), (np.float32, 31, 700), (np.float64, 10, 3000),
                                       (np.float64, 13, 3000), (np.float64, 15, 2000)])
def test_long_horizons_of_any_size_keep_up_with_lds(gpu, dtype, n, N):
    """Sizes without instances of their own, more workgroups than one XCD holds,
    reference recurrence (two exchanges per iteration over all ranks): not slower
    than the LDS-resident kernel, which has fewer ranks."""
    import gbdpcg
    auto, lds = _solve_us(n, N, dtype, 0), _solve_us(n, N, dtype, 0, kernel=gbdpcg.KERNEL_LDS)
    assert auto <= lds, (auto, lds)


@pytest.mark.parametrize("N,recurrence", [(850, 0), (890, 1)])
def test_row_broadcast_does_not_crowd_one_xcd(gpu, N, recurrence):
    """FP64 n = 12 in the row broadcast, about 62 workgroups: as above."""
    short, full = (_solve_us(12, k, np.float64, recurrence) for k in (N, 1000))
    assert short <= 1.1 * full, (short, full)


def _batch_us(n, N, count, dtype, recurrence, **kw):
    import torch
    import gbdpcg
    S, P, g = _system(n, N, dtype)
    lam = torch.zeros(count, n * N, device="cuda", dtype=g.dtype)
    b = gbdpcg.Batch([dict(S=S, Pinv=P, gamma=g, lam=lam[i], n=n, N=N) for i in range(count)], tol=0.0, max_iter=30,
                     exit_mode=gbdpcg.EXIT_REL_RESID, recurrence=recurrence, **kw)

    def call():
        lam.zero_()
        b.run()
    return _fastest_us(call)


def test_batches_spread_over_idle_cus(gpu):
    """100 one-workgroup systems on 256 CUs take no longer than 12 of them (they shared
    CUs two by two while others were idle)."""
    few, many = (_batch_us(2, 33, count, np.float64, 1) for count in (12, 100))
    assert many <= 1.1 * few, (many, few)


@pytest.mark.parametrize("n,N,cap", [(2, 16, 4), (6, 40, 12)])
def test_capped_batches_keep_up_with_lds(gpu, n, N, cap):
    """FP64, reference recurrence, a cap on the knots of a workgroup: the automatic
    choice is not slower than the LDS-resident kernel under the same cap."""
    import gbdpcg
    kw = dict(knots_per_wg=cap)
    auto, lds = _batch_us(n, N, 150, np.float64, 0, **kw), _batch_us(n, N, 150, np.float64, 0,
                                                                    kernel=gbdpcg.KERNEL_LDS, **kw)
    assert auto <= 1.1 * lds, (auto, lds)


@pytest.mark.parametrize("dtype,n,N,count,recurrence", [(np.float32, 2, 254, 1000, 1), (np.float64, 2, 180, 600, 1),
                                                        (np.float32, 16, 30, 400, 0), (np.float32, 14, 35, 600, 0)])
def test_batches_of_several_rounds_keep_up_with_512_threads(gpu, dtype, n, N, count, recurrence):
    """Systems that one workgroup of 512 threads holds and one of 256 does not: the
    automatic choice is not slower than the larger workgroups."""
    auto, wide = (_batch_us(n, N, count, dtype, recurrence, threads=t) for t in (0, 512))
    assert auto <= 1.1 * wide, (auto, wide)


@pytest.mark.parametrize("n,N", [(29, 25), (27, 9)])
def test_tuning_a_fused_request_without_a_fused_layout_costs_nothing(gpu, n, N):
    """FP64 at odd N from n = 25 on runs the reference iteration: after tuning the fused
    request, it and a plain reference solve take the untuned layout, bit for bit, unless
    a faster one was found, and neither is slower than before."""
    import torch
    import gbdpcg
    S, P, g = _system(n, N, np.float64)
    kw = dict(tol=0.0, max_iter=20, exit_mode=gbdpcg.EXIT_REL_RESID)

    def solution(recurrence):
        lam = torch.zeros_like(g)
        gbdpcg.solve(S, g, lam, n, N, P, recurrence=recurrence, **kw)
        return lam
    before = [(solution(r), _solve_us(n, N, np.float64, r)) for r in (0, 1)]
    rep = gbdpcg.tune_single(S, g, n, N, P, recurrence=gbdpcg.RECUR_FUSED, **kw)
    after = [(solution(r), _solve_us(n, N, np.float64, r)) for r in (0, 1)]
    for (lam0, us0), (lam1, us1) in zip(before, after):
        assert us1 <= 1.1 * us0, (us1, us0)
        assert rep["best_us"] < rep["default_us"] or torch.equal(lam0, lam1)


@pytest.mark.parametrize("n,N,dtype,fits", [
    (14, 3300, np.float32, True), (14, 3800, np.float32, True), (14, 4000, np.float32, False),
    (14, 4096, np.float32, False), (28, 900, np.float64, True), (28, 960, np.float64, False),
    (12, 2000, np.float64, True), (20, 3000, np.float32, True), (24, 480, np.float64, False),
    (14, 5166, np.float32, True), (12, 7306, np.float32, True), (28, 1292, np.float32, True)])
def test_what_the_scratch_takes(gpu, n, N, dtype, fits):
    """The no-allocation solve takes the horizons that its documentation names (n = 14 FP32
    up to about 3800, n = 28 FP64 up to about 900) and refuses those beyond, whatever
    layout the planner runs; horizons of which two workgroups to a CU do not hold eight
    knots each are the LDS-resident kernel's, whose records fit again.  What it takes has
    the bits of the ordinary call, or of that kernel's where only its records fit."""
    import torch
    import gbdpcg
    S, P, g = _system(n, N, dtype)
    kw = dict(tol=0.0, max_iter=5, exit_mode=gbdpcg.EXIT_REL_RESID, recurrence=gbdpcg.RECUR_FUSED)
    lam, ref = torch.zeros_like(g), torch.zeros_like(g)
    if not fits:
        with pytest.raises(gbdpcg.GbdpcgError, match="scratch"):
            gbdpcg.solve_noalloc(S, g, lam, n, N, P, **kw)
        return
    gbdpcg.solve_noalloc(S, g, lam, n, N, P, **kw)
    kernel = gbdpcg.KERNEL_LDS if (n, N) in ((14, 5166), (12, 7306)) else gbdpcg.KERNEL_AUTO
    gbdpcg.solve(S, g, ref, n, N, P, kernel=kernel, **kw)
    assert torch.equal(lam, ref)
