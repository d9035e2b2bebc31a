"""Sums of a direct and an image term per z column (k_zconv's two phases and
the x pass over pairs of parts): with B (parts kept apart) and without (added),
and axes whose length has no plan (x: the sums over full spectra, z: the
runtime-length passes)."""
import numpy as np
import pytest

import openspacecharge_amd as osc
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

SHAPES = [(8, 8, 8), (50, 8, 9), (8, 50, 9), (9, 8, 50), (16, 12, 64), (9, 16, 81), (64, 64, 24), (72, 96, 12)]


def _mesh(shape, prec):
    rng = np.random.default_rng(sum(shape))
    ctx = osc.Context(0, precision=prec)
    m = osc.Mesh3D(nhi=shape, gamma=3.0)
    m.min = np.array([-1e-3, -0.7e-3, 0.3e-3])
    m.delta = np.array([2e-3, 1.4e-3, 1.1e-3]) / (np.array(shape) - 1)
    m.max = m.min + m.delta * (np.array(shape) - 1)
    m.allocate()
    m.rho[...] = rng.random(shape) * 1e-12
    return ctx, m


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("prec", [osc.OSC_PREC_FP64, osc.OSC_PREC_FP32])
@pytest.mark.parametrize("with_b", [True, False])
def test_cathode(shape, prec, with_b):
    ctx, m = _mesh(shape, prec)
    osc.space_charge_3d(m, at_cathode=True, calc_bfield=with_b, ctx=ctx)
    ctx.close()
    O = Oracle()
    O.set_zero_unused_planes(True)
    try:
        ref, floor = O.floor(lambda: np.concatenate(O.space_charge_3d(
            m.rho, m.nlo, m.nhi, m.min, m.max, m.delta, m.gamma, at_cathode=True), axis=-1))
    finally:
        O.set_zero_unused_planes(False)
    # the floor (one ulp of the Green primitives) as in every parity test; in
    # FP32 the convolution's rounding, 1e-5 of the largest value
    tol = 1e-5 if prec == osc.OSC_PREC_FP32 else 4 * floor + 2e-14
    got = np.concatenate([m.efield, m.bfield], axis=-1) if with_b else m.efield
    for k in range(6 if with_b else 3):
        if k == 5:
            assert not np.any(got[..., 5])
            continue
        scale = np.max(np.abs(ref[..., k]))
        assert np.max(np.abs(got[..., k] - ref[..., k])) <= tol * scale, k


@pytest.mark.parametrize("shape", SHAPES[:5])
@pytest.mark.parametrize("direct", [True, False])
@pytest.mark.parametrize("method", [1, 2])
def test_legacy(shape, direct, method):
    ctx, m = _mesh(shape, osc.OSC_PREC_FP64)
    rho0 = m.rho.copy(order="F")
    osc.space_charge_cathodeimages(m, direct, True, method, ctx=ctx)
    ctx.close()
    O = Oracle()

    def run():
        _, _, e, b, _ = O.space_charge_cathodeimages(rho0, m.nlo, m.nhi, m.npad, m.min, m.delta, m.gamma,
                                                     direct, True, method)
        return np.concatenate([e, b], axis=-1)
    ref, floor = O.floor(run)
    got = np.concatenate([m.efield, m.bfield], axis=-1)
    # the potential's differences amplify its rounding by up to the node count
    tol = 4 * floor + (2e-14 if direct else 2e-14 * max(shape))
    for k in range(5):
        scale = np.max(np.abs(ref[..., k]))
        assert np.max(np.abs(got[..., k] - ref[..., k])) <= tol * scale, k
