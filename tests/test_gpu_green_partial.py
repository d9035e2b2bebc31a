"""A solve that finds one or two of its three Green spectra in the cache builds
the others together (csrc/green.hip, green_spectra): the same fields as with
none cached, on grids whose components go side by side, and on larger ones."""
import os

import numpy as np
import pytest

import openspacecharge_amd as osc

pytestmark = pytest.mark.gpu


def _solve(ctx, solver, shape, gamma):
    m = osc.Mesh3D(nhi=shape, gamma=gamma)
    m.min = np.array([-1e-3, -0.7e-3, 0.3e-3])
    m.delta = np.array([2e-3, 1.4e-3, 1.1e-3]) / (np.array(shape) - 1)
    m.max = m.min + m.delta * (np.array(shape) - 1)
    m.allocate()
    m.rho[...] = np.random.default_rng(sum(shape)).random(shape) * 1e-12
    (osc.space_charge_3d if solver == "free" else osc.space_charge_freespace)(m, ctx=ctx)
    return np.concatenate([m.efield, m.bfield], axis=-1) if solver != "free" else m.efield


@pytest.mark.parametrize("cached", [1, 2])
@pytest.mark.parametrize("shape", [(24, 20, 32), (15, 14, 25), (128, 64, 96)])
@pytest.mark.parametrize("solver", ["free", "legacy"])
@pytest.mark.parametrize("prec", [osc.OSC_PREC_FP64, osc.OSC_PREC_FP32])
def test_some_components_cached(cached, shape, solver, prec):
    old = os.environ.get("OSC_GREEN_ADMIT")
    os.environ["OSC_GREEN_ADMIT"] = "0"  # a spectrum is kept from its first build on
    try:
        c, ref = (osc.Context(0, precision=prec) for _ in range(2))
    finally:
        if old is None:
            del os.environ["OSC_GREEN_ADMIT"]
        else:
            os.environ["OSC_GREEN_ADMIT"] = old
    ref.set_green_cache(False)
    want = _solve(ref, solver, shape, 3.0)
    # room for the second geometry's spectra and `cached` of the first's
    L = [2 * n for n in shape]
    spec = (16 if prec == osc.OSC_PREC_FP64 else 8) * ((L[0] // 2 + 1 + 15) // 16 * 16) * L[1] * L[2]
    c.set_green_cache(True, spec * (3 + cached))
    for gamma in (3.0, 4.0, 3.0, 3.0):
        got = _solve(c, solver, shape, gamma)
        if gamma == 3.0:
            assert np.array_equal(got, want)
    ref.close()
    c.close()
