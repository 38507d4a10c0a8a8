"""Several Jacobi sweeps and the residual in one launch, as V-cycles run them,
against the same V-cycle put together from single sweeps and transforms (needs
a GPU): J4 (one tile a lozenge, whose rings cross several seams), J5 and J6;
no sweep, fewer, as many and more than one launch carries, with a residual or
not.  The same operations in the same order: equal to the last bit.
"""
import numpy as np
import pytest

import wavetrisk_hydrostatic_amd as W
from wavetrisk_hydrostatic_amd import cases

pytestmark = pytest.mark.gpu


def level(l):
    g = W.Grid(level=l, min_level=4, domain_level=2)
    c = W.Context(g, nlayers=1)
    c.set_topography(cases.ocean(g, 1, seed=l)[0])
    c.fs_set_params(3000.0, 0.7, 0.9)
    src = g.array("node_src")
    rng = np.random.default_rng(l)
    fields = [np.where(src >= 0, (a * rng.standard_normal(g.layout.ncells))[src], 0.0) for a in (0.5, 0.5, 1e-9)]
    c.fs_upload(W.FS_ETA_OLD, fields[0])
    return c, fields[1], fields[2]


def sweeps(c, u, f, n):
    c.fs_upload(W.FS_ETA, u)
    c.fs_upload(W.FS_RHS, f)
    c.jacobi(W.FS_ETA, W.FS_RHS, 1.0, n)
    return c.fs_download(W.FS_ETA)


def residual(c, u, f):
    c.fs_upload(W.FS_DIVF, u)
    c.elliptic_apply(W.FS_DIVF, W.FS_DIVF_OLD)
    return f - c.fs_download(W.FS_DIVF_OLD)


def cycle(h, ctxs, u, f, p):
    """one V-cycle (lin_solve.f90:102-139)"""
    res, corr = residual(ctxs[-1], u, f), [None] * len(ctxs)
    rhs = [None] * len(ctxs)
    for l in range(len(ctxs) - 1, 0, -1):
        corr[l] = sweeps(ctxs[l], 0 * res, res, p.down_iter)
        rhs[l] = residual(ctxs[l], corr[l], res)
        ctxs[l].fs_upload(W.FS_DIVF, rhs[l])
        h.forward(l, W.FS_DIVF, W.FS_DIVF_OLD, W.FS_DIVF)
        res = ctxs[l - 1].fs_download(W.FS_DIVF)
    ctxs[0].fs_upload(W.FS_ETA, 0 * res)
    ctxs[0].fs_upload(W.FS_RHS, res)
    ctxs[0].elliptic_solve(W.SOLVE_BICGSTAB, p.coarse_tol, p.coarse_iter)
    e = ctxs[0].fs_download(W.FS_ETA)
    for l in range(1, len(ctxs)):
        ctxs[l - 1].fs_upload(W.FS_DIVF, e)
        ctxs[l].fs_upload(W.FS_DIVF_OLD, 0 * rhs[l])
        h.inverse(l, W.FS_DIVF, W.FS_DIVF_OLD, W.FS_DIVF)
        e = sweeps(ctxs[l], corr[l] + ctxs[l].fs_download(W.FS_DIVF), rhs[l], p.up_iter)
    return sweeps(ctxs[-1], u + e, f, p.post_iter)


@pytest.mark.parametrize("levels", [(4, 5), (4, 5, 6)])
@pytest.mark.parametrize("down,up,post", [(2, 2, 4), (0, 0, 0), (1, 3, 5), (6, 5, 12), (7, 1, 1)])
def test_cycle_equals_single_sweeps(levels, down, up, post):
    print(f"V-cycle over levels {levels}: {down}, {up}, {post} sweeps", flush=True)
    lev = [level(l) for l in levels]
    ctxs = [c for c, _, _ in lev]
    h = W.Hierarchy(ctxs)
    p = W.MgParams.defaults(max_vcycle=1, fine_tol=1e-30, down_iter=down, up_iter=up, post_iter=post)
    _, u, f = lev[-1]
    want = cycle(h, ctxs, u, f, p)
    for c, u0, f0 in lev:
        c.fs_upload(W.FS_ETA, u0)
        c.fs_upload(W.FS_RHS, f0)
    _, res = h.solve(W.SOLVE_VCYCLE, p)
    got = ctxs[-1].fs_download(W.FS_ETA)
    own = ctxs[-1].grid.layout.owned_cells()
    src = ctxs[-1].grid.array("node_src")
    norm = [np.sqrt(ctxs[-1].fs_dot(W.FS_DIVF, W.FS_DIVF))
            for x in (residual(ctxs[-1], got, f), f) if ctxs[-1].fs_upload(W.FS_DIVF, x) is None]
    h.close()
    for c in ctxs:
        c.close()
    assert np.array_equal(got[own], want[own])
    assert np.array_equal(got[src >= 0], got[src[src >= 0]])  # halo copies
    assert res[-1] == norm[0] / norm[1]
