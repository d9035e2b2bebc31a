"""The cell sort where the number of nodes is a power of two, so that dropped
particles sort by the last node's key (csrc/deposit.hip, SortPlan), and one
node more or less: the deposit's drops and sums, the fused step's gather in
cell order, and the gather of points sorted for themselves."""
import os

import numpy as np
import pytest

import openspacecharge_amd as osc
from oracle.oracle import Oracle, gaussian_bunch

pytestmark = pytest.mark.gpu
LO = (1, 1, 1)


@pytest.fixture
def ctx():
    old = os.environ.get("OSC_TILED_DEPOSIT")
    os.environ["OSC_TILED_DEPOSIT"] = "0"
    try:
        c = osc.Context(0)
    finally:
        if old is None:
            del os.environ["OSC_TILED_DEPOSIT"]
        else:
            os.environ["OSC_TILED_DEPOSIT"] = old
    yield c
    c.close()


@pytest.mark.parametrize("shape", [(2, 2, 2), (4, 8, 8), (32, 32, 64), (27, 49, 50), (16, 16, 24)])
@pytest.mark.parametrize("n", [700, 70001])
def test_drops_sort_last(shape, n, ctx):
    O = Oracle()
    x, y, z = gaussian_bunch(n, (1e-3, 1e-3, 2e-3), seed=n)
    m = osc.Mesh3D(nhi=shape, gamma=3.0)
    # dropped particles, and some in the cell of the last nodes
    m.min, m.max = np.array([-4e-3, -4e-3, -8e-3]), np.array([1e-3, 1.2e-3, 1.5e-3])
    m.delta = (m.max - m.min) / (np.array(shape) - 1)
    d = O.deposit_particles(x, y, z, LO, shape, total_charge=1e-9, resize=False, mn=m.min, mx=m.max,
                            delta=m.delta)
    dropped = osc.deposit_particles(x, y, z, m, total_charge=1e-9, resize_mesh=False, ctx=ctx)
    assert dropped == d["dropped"] > 0
    # at most n terms a node, in another order
    assert np.all(np.abs(m.rho - d["rho"]) <= n * 2.0 ** -53 * np.abs(d["rho"]) + 1e-30)
    if min(shape) < 4:
        return
    E, B = osc.space_charge_step(x, y, z, m, total_charge=1e-9, resize_mesh=False, calc_bfield=True, ctx=ctx)
    e, b, _ = O.interpolate_field(LO, shape, m.min, m.delta, m.efield, m.bfield, x, y, z)
    assert np.array_equal(E, e.T) and np.array_equal(B, b.T)
    px, py, pz = 0.9 * y, 0.8 * x, 1.1 * z
    E, B = osc.interpolate_field(px, py, pz, m, E=True, B=True, ctx=ctx)
    e, b, _ = O.interpolate_field(LO, shape, m.min, m.delta, m.efield, m.bfield, px, py, pz)
    assert np.array_equal(E, e.T) and np.array_equal(B, b.T)
