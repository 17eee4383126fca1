"""The register kernels for any stateSize up to 32: sizes at the edges of their
classes (n rounded up to 4), horizons at the edges of what one workgroup of 64,
256 or 512 threads holds, and one beyond, against the FP64 oracle and against the
LDS-resident kernel.

Bars: those of the sweeps over every stateSize (lambda within 1e-4 of the FP64
oracle run for the same iterations in FP32, 1e-9 in FP64; iteration counts within
one of the same-precision oracle's and of the LDS kernel's)."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_batched import check, make_batch
from test_gpu_parity import gpu_solve, lqr_system, rel

pytestmark = pytest.mark.gpu
SIZES = [1, 2, 3, 4, 5, 8, 9, 12, 13, 14, 16, 17, 20, 21, 24, 25, 28, 29, 32]


def horizons(n):
    """What one workgroup of 64, 256 or 512 lanes holds of a system without
    neighbours, one or two lanes per row or two rows per lane, and one knot more;
    where rows get 16 lanes per knot (n = 13..15 from N = 13 to 32)."""
    edges = [64 // n, 128 // n, 256 // n, 512 // n, 512 // ((n + 1) // 2)] + ([12, 32, 64] if 12 < n < 16 else [])
    return sorted({N for e in edges for N in (e, e + 1) if 2 <= N <= 300})


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("recurrence", [0, 1])
def test_edges_of_one_workgroup(gpu, dtype, recurrence):
    import gbdpcg
    tol, bar = (1e-5, 1e-4) if dtype == np.float32 else (1e-9, 1e-9)
    for n in SIZES:
        for N in horizons(n):
            S, P, g = lqr_system(n, N, 4100 + 40 * n + N, dtype)
            z = np.zeros(n * N, dtype)
            kw = dict(tol=tol, max_iter=400, exit_mode=1, recurrence=recurrence)
            lam, res = gpu_solve(S, P, g, z, n, N, dtype, **kw)
            _, res_lds = gpu_solve(S, P, g, z, n, N, dtype, kernel=gbdpcg.KERNEL_LDS, **kw)
            _, it, *_ = O.pcg(S, P, g, z, n, N, tol, 400, 1, dtype, fused=recurrence == 1)
            assert res.status == gbdpcg.CONVERGED and abs(res.iters - it) <= 1, (n, N, res.iters, it)
            assert res_lds.status == gbdpcg.CONVERGED and abs(res.iters - res_lds.iters) <= 1, (n, N)
            ref, *_ = O.pcg(S.astype(np.float64), P.astype(np.float64), g.astype(np.float64), z.astype(np.float64),
                            n, N, 0.0, res.iters)
            assert rel(lam, ref) <= bar, (n, N, rel(lam, ref))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("recurrence", [0, 1])
@pytest.mark.parametrize("top", [16, 32])
def test_batches_of_any_size(gpu, dtype, recurrence, top):
    """One plan over every class up to `top`, forward and adjoint, with horizons on
    both sides of one workgroup, the reference's |r'z| rule excluded (check() holds
    the relative residual)."""
    tol = 1e-5 if dtype == np.float32 else 1e-9
    specs = [(n, N, tol) for n in SIZES if n <= top for N in (2, 256 // n, 256 // n + 1, 512 // n + 1) if N <= 150]
    systems, host = make_batch(specs, dtype, adjoint=True, seed0=14000)
    import gbdpcg
    b = gbdpcg.Batch(systems, exit_mode=gbdpcg.EXIT_REL_RESID, recurrence=recurrence)
    b.run()
    check(systems, host, b.results(), dtype, recurrence, adjoint=True)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("recurrence", [0, 1])
def test_batches_of_several_rounds(gpu, dtype, recurrence):
    """More systems than CUs: plans on small workgroups of one lane
    per row, horizons on both sides of what one of those holds (256 // n knots)."""
    import gbdpcg
    tol = 1e-5 if dtype == np.float32 else 1e-9
    sizes = [n for n in SIZES if n <= 16 and n > 3]
    specs = [(n, 256 // n + d, tol) for _ in range(8) for n in sizes for d in (-2, -1, 0, 1, 2)]
    systems, host = make_batch(specs, dtype, seed0=15000)
    b = gbdpcg.Batch(systems, exit_mode=gbdpcg.EXIT_REL_RESID, recurrence=recurrence)
    assert b.info()["wgs_per_cu"] == (3 if dtype == np.float32 else 2)
    b.run()
    check(systems, host, b.results(), dtype, recurrence)
