"""The vertical diffusion's register kernels on columns with infinities, NaNs
and massless layers (needs a GPU): a division through a reciprocal gives NaN
where the quotient is an infinity, so such columns take the private arrays and
every field equals the oracle bit for bit (TKE closure, no exponentials).
"""
import numpy as np
import pytest

import wavetrisk_hydrostatic_amd as W
from wavetrisk_hydrostatic_amd import cases
from helpers import oracle_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [3, 16, 20, 30])
def test_nonfinite_columns_equal_oracle(layers):
    print(f"vertical diffusion of infinities, NaNs and massless layers, J4 L{layers}", flush=True)
    g = W.Grid(level=4, min_level=4, domain_level=2)
    L, NC = layers, g.layout.ncells
    oc, oe = g.layout.owned_cells(), g.layout.owned_edge_cells()
    rng = np.random.default_rng(layers)
    topo, m, t, u = cases.ocean(g, L, seed=5)
    f = 1.0 + 0.02 * rng.uniform(-1, 1, (L, 1)) * g.array("x")[2] / g.radius
    m, t, u = m * f, t * f, u * rng.uniform(0.5, 1.5, (L, 1, 1))
    cells = rng.choice(oe, 42, replace=False).reshape(7, 6)
    for k in range(6):
        lay = (0, 1, L // 2, L - 2, L - 1, L - 1)[k]
        u[lay, k % 3, cells[0, k]], u[lay, k % 3, cells[1, k]] = np.inf, -np.inf
        t[lay, cells[2, k]], t[lay, cells[3, k]] = np.inf, np.nan
        m[lay, cells[4, k]] = 0.0  # with a temperature: t / m is an infinity
        m[lay, cells[5, k]], t[lay, cells[5, k]] = 0.0, 0.0
        m[lay, cells[6, k]] = np.inf
    forcing = dict(bot=rng.uniform(-3e-7, 3e-7, NC), top=rng.uniform(-1e-6, 1e-6, NC), tau=rng.uniform(0.02, 0.2, NC),
                   wind=rng.uniform(-2e-4, 2e-4, (3, NC)))
    coef = (rng.uniform(1e-5, 1e-3, (L + 1, NC)), rng.uniform(1e-4, 1e-3, (L + 1, NC)), rng.uniform(1e-6, 3e-5, (L, NC)))
    ctx = W.Context(g, nlayers=L)
    ctx.set_topography(topo)
    ctx.upload_state(0, m, t, u)
    ctx.set_vdiff(tke_closure=1, bottom_friction=4e-4)
    ctx.vdiff_set_coefficients(*coef)
    ctx.vdiff_set_forcing(forcing["bot"], forcing["top"], forcing["tau"], forcing["wind"])
    ctx.vertical_diffusion(0, 900.0, 2)
    got = ctx.download_state(0) + ctx.vdiff_coefficients()
    ctx.close()
    o = oracle_of(g, topo)
    st = (m.copy(), t.copy(), u.copy())
    o.ghost_fill(*st)
    with np.errstate(all="ignore"):
        res = o.vertical_diffusion(*st, 900.0, 2, forcing, *coef, tke_closure=1, bottom_friction=4e-4)
    for i in range(6):
        w = oe if i == 2 else oc
        assert np.array_equal(got[i][..., w], res[i][..., w], equal_nan=True), i
