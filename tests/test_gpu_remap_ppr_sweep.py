"""remapPPR as one sweep of the column (needs a GPU), against the oracle bit for
bit: the fewest layers it takes and the most, drifted layers onto coordinates
that refine towards the surface, several members, a uniform column, coordinates
whose ends leave the old column, and interfaces that fall or coincide, whose
columns keep the general path.
"""
import numpy as np
import pytest

import wavetrisk_hydrostatic_amd as W
from wavetrisk_hydrostatic_amd import cases
from helpers import oracle_of

pytestmark = pytest.mark.gpu


def _target(L, kind):
    s = np.arange(L + 1) / L
    b = 1.0 - s ** 0.7
    a = 1.0 - b
    if kind == "outside":  # the lowest and the highest interface beyond the old ones
        a, b = a.copy(), b.copy()
        b[0], a[-1], b[-1] = 1.02, 1.0, -0.01
    if kind == "inside":
        b = 0.02 + 0.95 * b
    if kind == "falling":
        a, b = a.copy(), b.copy()
        a[[1, 2]], b[[1, 2]] = a[[2, 1]], b[[2, 1]]
    if kind == "equal":
        a, b = a.copy(), b.copy()
        a[2], b[2] = a[1], b[1]
    return a, b


@pytest.mark.parametrize("layers,members,drift,kind", [
    (4, 1, True, "surface"), (5, 2, True, "surface"), (13, 1, False, "surface"), (64, 1, True, "surface"),
    (9, 1, True, "outside"), (9, 1, True, "inside"), (6, 1, True, "falling"), (6, 1, True, "equal"),
    (3, 1, True, "surface")])
def test_sweep_equals_oracle(layers, members, drift, kind):
    print(f"PPR sweep L{layers} x {members} drift {drift} {kind}", flush=True)
    g = W.Grid(level=5, min_level=5, domain_level=2)
    draws, x = [], g.array("x") / g.radius
    for k in range(members):
        topo, m, t, u = cases.ocean(g, layers, seed=60 + k)
        if drift:
            rng = np.random.default_rng(k)
            f = 1.0 + 0.3 * rng.uniform(-1, 1, (layers, 1)) * np.cos(9 * x[0] + x[2])
            m, t = m * f, t * f * (1.0 + 0.1 * rng.uniform(-1, 1, (layers, 1)) * x[1])
            u = u * rng.uniform(-1, 1, (layers, 1, 1))
        draws.append((topo, m, t, u))
    a, b = _target(layers, kind)
    ctx = W.Context(g, nlayers=layers, members=members)
    ctx.set_topography(np.stack([d[0] for d in draws]) if members > 1 else draws[0][0])
    ctx.upload_state(0, *(np.concatenate([d[v] for d in draws]) for v in (1, 2, 3)))
    ctx.remap(0, W.REMAP_PPR, a, b)
    got = ctx.download_state(0)
    ctx.close()
    own, own_e = g.layout.owned_cells(), g.layout.owned_edge_cells()
    for k, (topo, m, t, u) in enumerate(draws):
        o = oracle_of(g, topo)
        st = (m.copy(), t.copy(), u.copy())
        o.ghost_fill(*st)
        want = o.remap(*st, W.REMAP_PPR, a, b)
        s = slice(k * layers, (k + 1) * layers)
        assert np.array_equal(got[0][s][:, own], want[0][:, own], equal_nan=True)
        assert np.array_equal(got[1][s][:, own], want[1][:, own], equal_nan=True)
        assert np.array_equal(got[2][s][:, :, own_e], want[2][:, :, own_e], equal_nan=True)
