"""BiCGSTAB as one launch against its separate launches, which contexts take
that replay graphs (needs a GPU): J4 to J6, a cell a thread with the last block
partly filled; J7 and J8, several cells a thread; solves that converge, that stop at once, at max_iter and never
(a right-hand side of zeros or with a NaN); as the coarse solve of V-cycles;
and ensembles, whose members converge apart.  The same operations in the same
order: equal to the last bit.
"""
import numpy as np
import pytest

import wavetrisk_hydrostatic_amd as W
from wavetrisk_hydrostatic_amd import cases

pytestmark = pytest.mark.gpu


def context(level, seed):
    g = W.Grid(level=level, min_level=4, domain_level=2)
    ctx = W.Context(g, nlayers=1)
    ctx.set_topography(cases.ocean(g, 1, seed=seed)[0])
    ctx.fs_set_params(3000.0)
    rng = np.random.default_rng(seed)
    src = g.array("node_src")
    fields = []
    for amp in (0.5, 0.5, 1e-9):  # old free surface, first guess, right-hand side
        q = amp * rng.standard_normal(g.layout.ncells)
        fields.append(np.where(src >= 0, q[src], 0.0))
    ctx.fs_upload(W.FS_ETA_OLD, fields[0])
    return g, ctx, fields


@pytest.mark.parametrize("level", [4, 5, 6, 7, 8])
def test_one_launch_equals_launches(level):
    print(f"BiCGSTAB in one launch, J{level}", flush=True)
    g, ctx, (eo, u0, f) = context(level, 10 * level)
    nan = f.copy()
    nan[g.layout.owned_cells()[0]] = np.nan
    for rhs, tol, maxit in ((f, 1e-9, 400), (f, 1e-3, 400), (f, 1e30, 5), (f, 1e-14, 1), (f, 1e-14, 7),
                            (0 * f, 1e-9, 3), (nan, 1e-9, 3)):
        out = []
        for graph in (True, False):
            ctx.fs_set_graph(graph)
            ctx.fs_upload(W.FS_ETA, u0)
            ctx.fs_upload(W.FS_RHS, rhs)
            out.append(ctx.elliptic_solve(W.SOLVE_BICGSTAB, tol, maxit) + (ctx.fs_download(W.FS_ETA),))
        (i1, r1, s1), (i2, r2, s2) = out
        assert i1 == i2 and np.array_equal(r1, r2, equal_nan=True), (tol, maxit, i1, i2, r1, r2)
        assert np.array_equal(s1, s2, equal_nan=True), (tol, maxit)
    ctx.close()


def test_coarse_solves_of_cycles():
    print("V-cycles over one-launch coarse solves", flush=True)
    lev = [context(level, 7 * level) for level in (5, 6)]
    ctxs = [c for _, c, _ in lev]
    h = W.Hierarchy(ctxs)
    out = []
    for graph in (True, False):
        for _, c, (eo, u0, f) in lev:
            c.fs_set_graph(graph)
            c.fs_upload(W.FS_ETA, u0)
            c.fs_upload(W.FS_RHS, f)
        it, res = h.solve(W.SOLVE_VCYCLE)
        out.append((it.copy(), res.copy(), ctxs[-1].fs_download(W.FS_ETA)))
    h.close()
    for c in ctxs:
        c.close()
    assert all(np.array_equal(a, b, equal_nan=True) for a, b in zip(*out))


@pytest.mark.parametrize("level,members", [(4, 2), (4, 5), (5, 3)])
def test_ensemble_steps_equal_launches_of_single_runs(level, members):
    print(f"split steps over one-launch solves, J{level} x {members}", flush=True)
    g = W.Grid(level=level, min_level=4, domain_level=2)
    draws = [cases.ocean(g, 2, seed=50 + m) for m in range(members)]
    etas = np.stack([d[1].sum(0) / 1028.0 + d[0] for d in draws])

    def step(which, graph):
        one = len(which) == 1
        ctx = W.Context(g, nlayers=2, members=len(which))
        topos = np.stack([draws[m][0] for m in which])
        ctx.set_topography(topos[0] if one else topos)
        ctx.upload_state(0, *(np.concatenate([draws[m][k] for m in which]) for k in (1, 2, 3)))
        ctx.fs_set_params(1800.0, 0.6, 0.8)
        ctx.fs_upload(W.FS_ETA, etas[which[0]] if one else etas[which])
        ctx.fs_set_graph(graph)
        it = ctx.rk4_split(0, 2, 1e-11, 400)
        eta = ctx.fs_download(W.FS_ETA).reshape(len(which), -1)
        ctx.close()
        return it, eta

    it, eta = step(list(range(members)), False)
    single = [step([m], True) for m in range(members)]
    own = g.layout.owned_cells()
    assert it == max(i for i, _ in single)
    for m, (_, e) in enumerate(single):
        assert np.array_equal(eta[m][own], e[0][own])
