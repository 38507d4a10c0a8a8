"""The vertical diffusion's register kernels where their shapes change (needs a
GPU): the fewest layers, both sides of every unrolled size, above the largest
(private arrays); several members; a negative time step, whose systems dgtsv
pivots and the register kernels leave.  TKE closure: every field equal to the
oracle bit for bit (no exponentials on this path).
"""
import numpy as np
import pytest

import wavetrisk_hydrostatic_amd as W
from wavetrisk_hydrostatic_amd import cases
from helpers import oracle_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers,members,dt,switches", [
    (3, 1, 900.0, {}), (16, 2, 900.0, {}), (17, 1, 900.0, {"patankar": 1}), (24, 1, 900.0, {"enhance_diff": 1}),
    (25, 1, 900.0, {}), (32, 1, 1800.0, {}), (33, 1, 900.0, {}), (7, 1, -3e7, {}), (20, 1, -2e8, {}), (30, 1, -4e8, {})])
def test_two_calls_equal_oracle(layers, members, dt, switches):
    print(f"vertical diffusion L{layers} x {members} dt {dt} {switches}", flush=True)
    g = W.Grid(level=5, min_level=5, domain_level=2)
    L, NC = layers, g.layout.ncells
    rng = np.random.default_rng(layers)
    draws = []
    for k in range(members):
        topo, m, t, u = cases.ocean(g, L, seed=80 + k)
        f = 1.0 + 0.3 * rng.uniform(-1, 1, (L, 1)) * g.array("x")[2] / g.radius
        draws.append((topo, m * f, t * f * (1.0 + 0.05 * rng.uniform(-1, 1, (L, 1))), u * rng.uniform(-1, 1, (L, 1, 1))))
    forcing = [dict(bot=rng.uniform(-3e-7, 3e-7, NC), top=rng.uniform(-1e-6, 1e-6, NC), tau=rng.uniform(0.02, 0.2, NC),
                    wind=rng.uniform(-2e-4, 2e-4, (3, NC))) for _ in range(members)]
    coef = [(rng.uniform(1e-5, 1e-3, (L + 1, NC)), rng.uniform(1e-4, 1e-3, (L + 1, NC)), rng.uniform(1e-6, 3e-5, (L, NC)))
            for _ in range(members)]
    ctx = W.Context(g, nlayers=L, members=members)
    ctx.set_topography(np.stack([d[0] for d in draws]) if members > 1 else draws[0][0])
    ctx.upload_state(0, *(np.concatenate([d[v] for d in draws]) for v in (1, 2, 3)))
    ctx.set_vdiff(tke_closure=1, bottom_friction=4e-4, **switches)
    ctx.vdiff_set_coefficients(*(np.concatenate([c[v] for c in coef]) for v in range(3)))
    ctx.vdiff_set_forcing(*(np.concatenate([f[v] for f in forcing]) for v in ("bot", "top", "tau")),
                          np.concatenate([f["wind"] for f in forcing]))
    for _ in range(2):
        ctx.vertical_diffusion(0, dt, 2)
    got = ctx.download_state(0) + ctx.vdiff_coefficients()
    ctx.close()
    oc, oe = g.layout.owned_cells(), g.layout.owned_edge_cells()
    for k, (topo, m, t, u) in enumerate(draws):
        o = oracle_of(g, topo)
        st, cf = (m.copy(), t.copy(), u.copy()), coef[k]
        o.ghost_fill(*st)
        for _ in range(2):
            res = o.vertical_diffusion(*st, dt, 2, forcing[k], *cf, tke_closure=1, bottom_friction=4e-4, **switches)
            st, cf = res[:3], res[3:]
        n = (L, L, L, L + 1, L + 1, L)
        for i in range(6):
            a, b = got[i][k * n[i]:(k + 1) * n[i]], res[i]
            w = oe if i == 2 else oc
            assert np.array_equal(a[..., w], b[..., w], equal_nan=True), i
