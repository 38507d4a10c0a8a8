"""The network's weight gradients where their contraction over the batch is
split into chunks (needs a GPU): one chunk, the fewest rows that give two, a
last chunk shorter than the others, and the most chunks; against the oracle
with the same bf16 roundings, the bar of the unsplit gradients (2e-2 normwise
per parameter block: an activation's bf16 rounding can fall the other way;
the FP32 sums themselves differ by less than 1e-5).
"""
import numpy as np
import pytest

import wavetrisk_hydrostatic_amd as W
from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 192, 256, 449, 5000])
def test_gradients_match_oracle(batch):
    print(f"mlp gradients, {batch} rows", flush=True)
    net = W.MLP(max_batch=batch, seed=8)
    p = net.params.astype(np.float64)
    rng = np.random.default_rng(batch)
    x = rng.standard_normal((batch, M.NI)).astype(np.float32)
    t = (0.5 * rng.standard_normal((batch, M.NO))).astype(np.float32)
    loss, g = net.gradients(x, t)
    again = net.gradients(x, t)
    net.close()
    assert loss == again[0] and np.array_equal(g, again[1])  # a fixed order of sums
    lo, go = M.loss_and_grad(p, x, t, emulate=True)
    assert abs(loss - lo) <= 1e-4 * lo
    o = 0
    for name, shape in M.SHAPES:
        n = int(np.prod(shape))
        err = np.linalg.norm(g[o:o + n] - go[o:o + n]) / np.linalg.norm(go[o:o + n])
        assert err <= 2e-2, (name, err)
        o += n
