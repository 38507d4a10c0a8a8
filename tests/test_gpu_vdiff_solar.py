"""Vertical diffusion with a penetrative solar flux (needs a GPU): the buoyancy
rows with their irradiance in the register kernels at every unrolled size and
above, against the oracle within 1e-14 (device and host exp may differ in the
last bit); columns with a layer of negative mass, which the register kernels
leave; members; eta from the free surface.  The flux costs two exponentials an
interface, not another order of time: at most three times the call without.
"""
import time

import numpy as np
import pytest

import wavetrisk_hydrostatic_amd as W
from wavetrisk_hydrostatic_amd import cases
from conftest import maxrel
from helpers import oracle_of

pytestmark = pytest.mark.gpu

PARAMS = dict(Q_sr=80.0, c_p=3991.87, bottom_friction=4e-4)


def _case(g, L, members, seed):
    rng = np.random.default_rng(seed)
    NC = g.layout.ncells
    draws = []
    for k in range(members):
        topo, m, t, u = cases.ocean(g, L, seed=80 + k)
        f = 1.0 + 0.3 * rng.uniform(-1, 1, (L, 1)) * g.array("x")[2] / g.radius
        draws.append((topo, m * f, t * f * (1.0 + 0.05 * rng.uniform(-1, 1, (L, 1))), u * rng.uniform(-1, 1, (L, 1, 1))))
    forcing = [dict(bot=rng.uniform(-3e-7, 3e-7, NC), top=rng.uniform(-1e-6, 1e-6, NC), tau=rng.uniform(0.02, 0.2, NC),
                    wind=rng.uniform(-2e-4, 2e-4, (3, NC))) for _ in range(members)]
    coef = [(rng.uniform(1e-5, 1e-3, (L + 1, NC)), rng.uniform(1e-4, 1e-3, (L + 1, NC)), rng.uniform(1e-6, 3e-5, (L, NC)))
            for _ in range(members)]
    return draws, forcing, coef


def _context(g, L, draws, forcing, coef, **params):
    M = len(draws)
    ctx = W.Context(g, nlayers=L, members=M)
    ctx.set_topography(np.stack([d[0] for d in draws]) if M > 1 else draws[0][0])
    ctx.upload_state(0, *(np.concatenate([d[v] for d in draws]) for v in (1, 2, 3)))
    ctx.set_vdiff(**params)
    ctx.vdiff_set_coefficients(*(np.concatenate([c[v] for c in coef]) for v in range(3)))
    ctx.vdiff_set_forcing(*(np.concatenate([f[v] for f in forcing]) for v in ("bot", "top", "tau")),
                          np.concatenate([f["wind"] for f in forcing]))
    return ctx


@pytest.mark.parametrize("layers,members,tke,split", [
    (2, 1, 0, False), (3, 1, 1, False), (16, 2, 1, False), (17, 1, 0, True), (24, 1, 1, True), (25, 1, 1, False),
    (32, 1, 1, False), (33, 1, 1, False)])
def test_solar_rows_equal_oracle(layers, members, tke, split):
    print(f"vertical diffusion with a solar flux, J5 L{layers} x {members} tke {tke} split {split}", flush=True)
    g = W.Grid(level=5, min_level=5, domain_level=2)
    L, NC = layers, g.layout.ncells
    draws, forcing, coef = _case(g, L, members, layers)
    oc, oe = g.layout.owned_cells(), g.layout.owned_edge_cells()
    for d in draws:  # left to the private arrays
        d[1][L // 2, oe[::97]] *= -0.01
    ctx = _context(g, L, draws, forcing, coef, tke_closure=tke, mode_split=int(split), **PARAMS)
    eta = 0.4 * np.sin(np.arange(NC) * 0.37) if split else None
    if split:
        ctx.fs_upload(W.FS_ETA, eta)
    ctx.vertical_diffusion(0, 1800.0, 2)
    got = ctx.download_state(0) + ctx.vdiff_coefficients()
    ctx.close()
    n = (L, L, L, L + 1, L + 1, L)
    for k, (topo, m, t, u) in enumerate(draws):
        o = oracle_of(g, topo)
        st = (m.copy(), t.copy(), u.copy())
        o.ghost_fill(*st)
        res = o.vertical_diffusion(*st, 1800.0, 2, forcing[k], *coef[k], eta=eta, tke_closure=tke, **PARAMS)
        for i in range(6):
            w = oe if i == 2 else oc
            assert maxrel(got[i][k * n[i]:(k + 1) * n[i]][..., w], res[i][..., w]) <= 1e-14, i


def test_solar_flux_time():
    print("vertical diffusion's time with and without a solar flux, J6 L20", flush=True)
    g = W.Grid(level=6, min_level=6, domain_level=2)
    draws, forcing, coef = _case(g, 20, 1, 1)
    best = []
    for q in (0.0, 80.0):
        ctx = _context(g, 20, draws, forcing, coef, tke_closure=1, **{**PARAMS, "Q_sr": q})
        times = []
        for _ in range(8):
            t0 = time.perf_counter()
            ctx.vertical_diffusion(0, 900.0, 2)
            times.append(time.perf_counter() - t0)
        ctx.close()
        best.append(min(times[1:]))
    print(f"{best[0] * 1e6:.0f} us without, {best[1] * 1e6:.0f} us with", flush=True)
    assert best[1] <= 3.0 * best[0]
