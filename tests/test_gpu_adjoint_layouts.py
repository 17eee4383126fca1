"""Which layouts adjoint solves run on: alone, against the paired solve and the plain
solve of the same system, and of shapes that the autotuner has chosen a layout for."""
import os
import subprocess
import sys

import numpy as np
import pytest

from test_gpu_adjoint import run_adjoint, system

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))

TUNE = """
import sys; sys.path[:0] = [{here!r}]
import conftest, torch, numpy as np, gbdpcg
from test_gpu_adjoint import _t, system
S, P, g, glam = system({n}, {N}, 5, np.{dtype})
gbdpcg.tune_single(*(_t(a.astype(np.{dtype}), np.{dtype}) for a in (S, g)), {n}, {N},
                   _t(P.astype(np.{dtype}), np.{dtype}), tol=1e-5, max_iter=200, exit_mode=1, recurrence=1)
"""
SOLVE = """
import sys; sys.path[:0] = [{here!r}]
import conftest, torch, numpy as np, gbdpcg
from test_gpu_adjoint import run_adjoint, system
S, P, g, glam = system({n}, {N}, 5, np.{dtype})
kw = dict(tol=1e-5, max_iter=200, exit_mode=1, recurrence=1)
lam, gg, gS, res = run_adjoint(S, P, g, glam, {n}, {N}, np.{dtype}, **kw)
if not {forward}:
    lam, gg, gS, res = run_adjoint(S, P, g, glam, {n}, {N}, np.{dtype}, forward=False, lam_in=lam, **kw)
np.savez({out!r}, lam=lam, gg=gg, gS=gS)
"""


def _run(code, cache):
    r = subprocess.run([sys.executable, "-c", code], timeout=100, capture_output=True, text=True,
                       env=dict(os.environ, GBDPCG_TUNE_CACHE=str(cache)))
    assert r.returncode == 0, r.stderr[-2000:]


@pytest.mark.parametrize("n,N,dtype,kind,threads,forward", [
    (12, 21, np.float32, 4, 256, True), (6, 40, np.float32, 4, 256, True),
    (14, 20, np.float64, 6, 512, False), (12, 13, np.float64, 4, 256, False)])
def test_a_tuned_shape_keeps_its_paired_solve(gpu, tmp_path, n, N, dtype, kind, threads, forward):
    """A choice of one workgroup on an any-size instance, which runs forward and adjoint
    one after the other: forward + adjoint in one call still iterates them together
    (FP32, n = 6 and 12), and the FP64 adjoint by itself still has the bits of that solve
    where both run the row broadcast (n = 12 and 14), as untuned."""
    cache, out = tmp_path / "tune.txt", str(tmp_path / "out.npz")
    fields = dict(here=HERE, n=n, N=N, dtype=dtype.__name__, out=out, forward=forward)
    _run(TUNE.format(**fields), cache)
    key = cache.read_text().split()[0]
    cache.write_text(f"{key} {kind} {threads} 1 8\n")
    _run(SOLVE.format(**fields), cache)
    S, P, g, glam = system(n, N, 5, dtype)
    lam, gg, gS, _ = run_adjoint(S, P, g, glam, n, N, dtype, tol=1e-5, max_iter=200, exit_mode=1, recurrence=1)
    tuned = np.load(out)
    for name, untuned in (("lam", lam), ("gg", gg), ("gS", gS)):
        assert np.array_equal(tuned[name], untuned), name


@pytest.mark.parametrize("n,horizons", [(12, (4, 13, 14, 20, 42, 43, 100, 128)), (14, (4, 14, 17, 32, 36, 37, 100))])
def test_adjoint_alone_has_the_bits_of_the_paired_solve(gpu, n, horizons):
    """FP64 fused, the sizes of the row broadcast: g_gamma and g_S of forward + adjoint in
    one call and of the adjoint by itself are the same numbers."""
    kw = dict(tol=1e-10, max_iter=300, exit_mode=1, recurrence=1)
    for N in horizons:
        S, P, g, glam = system(n, N, 900 + N, np.float64)
        lam, gg, gS, _ = run_adjoint(S, P, g, glam, n, N, np.float64, **kw)
        _, gg2, gS2, _ = run_adjoint(S, P, g, glam, n, N, np.float64, forward=False, lam_in=lam, **kw)
        assert np.array_equal(gg2, gg) and np.array_equal(gS2, gS), (n, N)


@pytest.mark.parametrize("n,horizons", [(2, (4, 32, 60, 128)), (6, (8, 20, 36, 40)), (12, (15, 19)), (14, (15, 16))])
def test_adjoint_alone_runs_as_the_plain_solve(gpu, n, horizons):
    """FP64 fused, elsewhere: the paired solve adds up in another order anyhow (two rows to
    a quad of lanes), and the adjoint by itself takes the layout of a plain solve, one
    workgroup where that holds the system: g_gamma is that solve's lambda for g_lambda."""
    from test_gpu_parity import gpu_solve
    kw = dict(tol=1e-10, max_iter=300, exit_mode=1, recurrence=1)
    for N in horizons:
        S, P, g, glam = system(n, N, 900 + N, np.float64)
        z = np.zeros(n * N)
        _, gg, _, _ = run_adjoint(S, P, g, glam, n, N, np.float64, forward=False, lam_in=g, **kw)
        lam, _ = gpu_solve(S, P, glam, z, n, N, np.float64, **kw)
        assert np.array_equal(gg, lam), (n, N)
