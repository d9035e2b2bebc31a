"""One context that serves both precisions on a fixed mesh keeps an FP32 and an
FP64 spectrum under one cache entry, the FP32 one stored as a half along the
mirrored z axis, the FP64 one whole: each solve must give what a context of its
own precision gives, whatever the other left there."""
import os

import numpy as np
import pytest

import openspacecharge_amd as osc

pytestmark = pytest.mark.gpu

F32, F64 = osc.OSC_PREC_FP32, osc.OSC_PREC_FP64
# (8, 18, 24): z lengths with a plan, whose z pass is left to the multiply
SHAPES = [(24, 20, 32), (16, 12, 18), (9, 7, 8)]


def _ctx(prec, graphs=False):
    old = os.environ.get("OSC_FAR_GREEN")
    os.environ["OSC_FAR_GREEN"] = "0"  # far cells would keep the precisions' keys apart
    try:
        c = osc.Context(0, precision=prec)
    finally:
        if old is None:
            del os.environ["OSC_FAR_GREEN"]
        else:
            os.environ["OSC_FAR_GREEN"] = old
    c.set_graphs(graphs)
    return c


def _solve(ctx, shape, cathode):
    m = osc.Mesh3D(nhi=shape, gamma=4.0)
    m.min = np.array([-1e-3, -0.8e-3, 0.2e-3])
    m.delta = np.array([2e-3, 1.6e-3, 1.2e-3]) / (np.array(shape) - 1)
    m.max = m.min + m.delta * (np.array(shape) - 1)
    m.allocate()
    m.rho[...] = np.random.default_rng(sum(shape)).random(shape) * 1e-12
    osc.space_charge_3d(m, at_cathode=cathode, calc_bfield=True, ctx=ctx)
    return np.concatenate([m.efield, m.bfield], axis=-1)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("order", [(F32, F32, F64, F32, F64), (F64, F64, F32, F64, F32)])
@pytest.mark.parametrize("cathode", [False, True])
def test_precisions_share_a_context(shape, graphs, order, cathode):
    want = {}
    for prec in (F32, F64):
        c = _ctx(prec, graphs)
        want[prec] = _solve(c, shape, cathode)
        c.close()
    assert not np.array_equal(want[F32], want[F64])
    c = _ctx(order[0], graphs)
    for k, prec in enumerate(order):
        c.set_precision(prec)
        assert np.array_equal(_solve(c, shape, cathode), want[prec]), k
    c.close()
