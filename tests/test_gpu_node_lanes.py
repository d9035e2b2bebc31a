"""The tiled deposit's node sums with 8, 4, 2 and 1 lanes to a node
(csrc/deposit.hip, node_lanes): meshes at both sides of the lines between them,
with few and many particles, against the oracle."""
import numpy as np
import pytest

import openspacecharge_amd as osc
from oracle.oracle import Oracle, gaussian_bunch

pytestmark = pytest.mark.gpu
LO = (1, 1, 1)


@pytest.mark.parametrize("shape", [(32, 32, 32), (51, 50, 51), (64, 64, 64), (65, 64, 64), (64, 64, 128), (66, 63, 130)])
@pytest.mark.parametrize("n", [1500, 30001, 400009])
@pytest.mark.parametrize("width", [1.0, 0.2])
def test_rho(shape, n, width):
    O = Oracle()
    x, y, z = gaussian_bunch(n, (1e-3 * width,) * 3, seed=n)
    m = osc.Mesh3D(nhi=shape)
    m.min, m.max = np.full(3, -3.1e-3), np.full(3, 3.3e-3)
    m.delta = (m.max - m.min) / (np.array(shape) - 1)
    d = O.deposit_particles(x, y, z, LO, shape, total_charge=1e-9, resize=False, mn=m.min, mx=m.max,
                            delta=m.delta)
    ctx = osc.Context(0)
    dropped = osc.deposit_particles(x, y, z, m, total_charge=1e-9, resize_mesh=False, ctx=ctx)
    ctx.close()
    assert dropped == d["dropped"]
    # the oracle adds a node's terms one after another, at most n of them
    assert np.all(np.abs(m.rho - d["rho"]) <= n * 2.0 ** -53 * np.abs(d["rho"]) + 1e-30)
    # FP32: the terms rounded to 2^-50 n max|q|, weights and their products of
    # three (each below 1) to 2^-24
    c32 = osc.Context(0, precision=osc.OSC_PREC_FP32)
    osc.space_charge_step(x, y, z, m, total_charge=1e-9, resize_mesh=False, ctx=c32)
    c32.close()
    q = 1e-9 / n
    cells = np.zeros(np.array(shape) + 1)
    idx = [np.floor((a - lo) / h).astype(int) for a, lo, h in zip((x, y, z), m.min, m.delta)]
    ok = np.all([(i >= 0) & (i < s - 1) for i, s in zip(idx, shape)], axis=0)
    np.add.at(cells, tuple(i[ok] + 1 for i in idx), 1)
    near = sum(cells[a:a + shape[0], b:b + shape[1], c:c + shape[2]] for a in (0, 1) for b in (0, 1) for c in (0, 1))
    # a weight's rounding: 2^-24 of 1, its own and its product's
    assert np.all(np.abs(m.rho - d["rho"]) <= near * q * 8 * 2.0 ** -24)
