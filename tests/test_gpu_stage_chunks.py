"""The FP64 stage kernel where its blocks differ (needs a GPU): tiles whose
layers are split into chunks (small grids), a last chunk shorter than the
others, one layer per block, tiles with all four pentagon corners (J4), and
whole columns per block with the column sums carried from stage to stage
(J7, or an ensemble).  Same operations in the same order as the oracle: every
field equal to the last bit after two steps, of every member.
"""
import numpy as np
import pytest

import wavetrisk_hydrostatic_amd as W
from wavetrisk_hydrostatic_amd import cases
from helpers import oracle_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,layers,members", [(4, 1, 1), (4, 11, 1), (4, 64, 1), (5, 13, 1), (6, 7, 1), (6, 2, 3),
                                                  (6, 4, 4), (7, 3, 1)])
def test_two_steps_equal_oracle(level, layers, members):
    print(f"stage chunks J{level} L{layers} x {members}", flush=True)
    g = W.Grid(level=level, min_level=level, domain_level=min(2, level - 3))
    draws = [cases.ocean(g, layers, seed=31 + k) for k in range(members)]
    ctx = W.Context(g, nlayers=layers, members=members)
    ctx.set_topography(np.stack([d[0] for d in draws]) if members > 1 else draws[0][0])
    ctx.upload_state(0, *(np.concatenate([d[v] for d in draws]) for v in (1, 2, 3)))
    ctx.rk4(0, 100.0, 2)
    got = ctx.download_state(0)
    ctx.close()
    own, own_e = g.layout.owned_cells(), g.layout.owned_edge_cells()
    for k, (topo, m, t, u) in enumerate(draws):
        o = oracle_of(g, topo)
        m, t, u = m.copy(), t.copy(), u.copy()
        o.ghost_fill(m, t, u)
        want = o.rk4(m, t, u, 100.0, 2)
        s = slice(k * layers, (k + 1) * layers)
        assert np.array_equal(got[0][s][:, own], want[0][:, own])
        assert np.array_equal(got[1][s][:, own], want[1][:, own])
        assert np.array_equal(got[2][s][:, :, own_e], want[2][:, :, own_e])
