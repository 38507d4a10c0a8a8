"""BiCGSTAB in one launch whose waits run out (needs a GPU): with a bound of 0 ms
every block gives up at the first sum that is not there yet and exits, and the
launches repeat the solve: iterations, residuals and solutions equal to the
last bit, the first guess kept.  After it 16 solves are launches, then one
launch is tried again; with the ordinary bound it succeeds.
"""
import numpy as np
import pytest

import wavetrisk_hydrostatic_amd as W
from wavetrisk_hydrostatic_amd import cases
from test_gpu_bicgstab_launch import context

pytestmark = pytest.mark.gpu


def _solve(ctx, u0, f, tol=1e-9, maxit=60):
    ctx.fs_upload(W.FS_ETA, u0)
    ctx.fs_upload(W.FS_RHS, f)
    return ctx.elliptic_solve(W.SOLVE_BICGSTAB, tol, maxit) + (ctx.fs_download(W.FS_ETA),)


def _equal(a, b):
    return all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a, b))


@pytest.mark.parametrize("level", [4, 6, 7, 8])
def test_given_up_solve_is_repeated(level):
    print(f"one-launch BiCGSTAB given up, J{level}", flush=True)
    g, ctx, (eo, u0, f) = context(level, 10 * level)
    ctx.fs_set_graph(True)
    want = _solve(ctx, u0, f)
    ctx.fs_set_graph(False)
    assert ctx.fs_one_launch() == (0, 0)
    ctx.fs_set_wait(0.0)
    assert _equal(_solve(ctx, u0, f), want)
    assert ctx.fs_one_launch() == (1, 1)
    short = _solve(ctx, u0, f, 1e-14, 2)
    for _ in range(15):  # the rest of the 16 that the launches take
        assert _equal(_solve(ctx, u0, f, 1e-14, 2), short)
    assert ctx.fs_one_launch() == (1, 1)
    assert _equal(_solve(ctx, u0, f), want)  # tried again
    assert ctx.fs_one_launch() == (2, 2)
    assert _equal(_solve(ctx, u0, f), want)
    assert ctx.fs_one_launch() == (2, 2)  # 32 launches now
    ctx.fs_set_wait(20.0)
    assert _equal(_solve(ctx, u0, f), want)
    assert _equal(_solve(ctx, u0, f, 1e-14, 2), short)
    assert ctx.fs_one_launch() == (4, 2)
    ctx.close()


def test_coarse_solves_of_an_ensemble():
    print("one-launch coarse solves of an ensemble's V-cycles given up", flush=True)
    lev = [context(level, 7 * level) for level in (4, 5)]
    out = []
    for wait in (20.0, 0.0):
        ctxs = []
        for g, one, (eo, u0, f) in lev:
            c = W.Context(g, nlayers=1, members=3)
            topo = cases.ocean(g, 1, seed=3)[0]
            c.set_topography(np.stack([topo + 20.0 * m for m in range(3)]))
            c.fs_set_params(3000.0)
            c.fs_upload(W.FS_ETA_OLD, np.stack([eo * (m + 1) for m in range(3)]))
            c.fs_upload(W.FS_ETA, np.stack([u0] * 3))
            c.fs_upload(W.FS_RHS, np.stack([f * 10.0 ** (-4 * m) for m in range(3)]))  # members end apart
            c.fs_set_wait(wait)
            ctxs.append(c)
        h = W.Hierarchy(ctxs)
        it, res = h.solve(W.SOLVE_VCYCLE)
        out.append((np.copy(it), np.copy(res), ctxs[-1].fs_download(W.FS_ETA)))
        n, failed = ctxs[0].fs_one_launch()
        assert n > 0 and failed == (n if wait == 0.0 else 0)
        h.close()
        for c in ctxs:
            c.close()
    for _, c, _ in lev:
        c.close()
    assert _equal(*out)


def test_wait_refusals():
    print("waits out of range", flush=True)
    g, ctx, _ = context(4, 1)
    for ms in (-1.0, 1001.0, float("nan")):
        with pytest.raises(W.WtgError):
            ctx.fs_set_wait(ms)
    ctx.close()
