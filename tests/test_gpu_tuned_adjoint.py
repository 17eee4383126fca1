"""Adjoint solves of shapes that the autotuner has chosen a layout for."""
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
lam, gg, gS, res = run_adjoint(S, P, g, glam, {n}, {N}, np.{dtype}, tol=1e-5, max_iter=200, exit_mode=1, recurrence=1)
np.savez({out!r}, lam=lam, gg=gg, gS=gS)
"""


def _run(code, cache):
    r = subprocess.run([sys.executable, "-c", code], timeout=100, capture_output=True, text=True,
                       env=dict(os.environ, GBDPCG_TUNE_CACHE=str(cache)))
    assert r.returncode == 0, r.stderr[-2000:]


@pytest.mark.parametrize("n,N", [(12, 21), (6, 40)])
def test_a_tuned_shape_keeps_its_paired_solve(gpu, tmp_path, n, N):
    """FP32, a choice of one workgroup on an any-size instance (kind 4: 256 threads, one
    lane per row), which runs forward and adjoint one after the other: forward +
    adjoint in one call still iterates them together, bit for bit as untuned."""
    cache, out = tmp_path / "tune.txt", str(tmp_path / "out.npz")
    fields = dict(here=HERE, n=n, N=N, dtype="float32", out=out)
    _run(TUNE.format(**fields), cache)
    key = cache.read_text().split()[0]
    cache.write_text(f"{key} 4 256 1 8\n")
    _run(SOLVE.format(**fields), cache)
    S, P, g, glam = system(n, N, 5, np.float32)
    lam, gg, gS, _ = run_adjoint(S, P, g, glam, n, N, np.float32, tol=1e-5, max_iter=200, exit_mode=1, recurrence=1)
    tuned = np.load(out)
    for name, untuned in (("lam", lam), ("gg", gg), ("gS", gS)):
        assert np.array_equal(tuned[name], untuned), name
