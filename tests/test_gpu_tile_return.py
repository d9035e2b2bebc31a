"""The tiled gather's values in bin order and their return to particle order
(csrc/gather.hip: k_tile_gather, k_tile_return), and the tiled deposit's block
sizes and split node sums, at the particle counts where the work split changes
and with particles off the mesh: bit for bit against the oracle's
interpolate_field, and rho against the oracle's deposit."""
import numpy as np
import pytest

import openspacecharge_amd as osc
from oracle.oracle import Oracle, gaussian_bunch

pytestmark = pytest.mark.gpu
O = Oracle()
LO = (1, 1, 1)


def fields(shape, seed):
    rng = np.random.default_rng(seed)
    return [np.asfortranarray(rng.standard_normal(shape + (3,))) for _ in range(2)]


# 65536: the fewest points that take a deposit's kept order; the others cross
# the block and item sizes (512 * 512, 1024 * 512, ...), and meshes with tiles
# of 8^3 cells, larger ones, and fewer cells than a tile
@pytest.mark.parametrize("n", [65536, 262145, 524289, 1100003])
@pytest.mark.parametrize("shape", [(7, 9, 20), (40, 33, 17), (96, 96, 128)])
@pytest.mark.parametrize("want", ["E", "B", "EB"])
def test_return_to_particle_order(n, shape, want):
    x, y, z = gaussian_bunch(n, (1e-3, 1e-3, 2e-3), seed=n)
    m = osc.Mesh3D(nhi=shape)
    # a mesh that a few particles leave
    m.min, m.max = np.array([-3e-3, -3.5e-3, -6e-3]), np.array([3.2e-3, 3e-3, 7e-3])
    m.delta = (m.max - m.min) / (np.array(shape) - 1)
    ctx = osc.Context(0)
    d = O.deposit_particles(x, y, z, LO, shape, total_charge=1e-9, resize=False, mn=m.min, mx=m.max,
                            delta=m.delta)
    dropped = osc.deposit_particles(x, y, z, m, total_charge=1e-9, resize_mesh=False, ctx=ctx)
    assert dropped == d["dropped"] > 0
    # the oracle adds a node's terms one after another, at most n of them
    assert np.all(np.abs(m.rho - d["rho"]) <= n * 2.0 ** -53 * np.abs(d["rho"]) + 1e-30)
    m.efield, m.bfield = fields(shape, n)
    got, fl = osc.interpolate_field(x, y, z, m, E="E" in want, B="B" in want, return_clamped=True,
                                    ctx=ctx)
    ctx.close()
    e, b, c = O.interpolate_field(LO, shape, m.min, m.delta, m.efield, m.bfield, x, y, z)
    got = got if want == "EB" else (got,)
    for g, ref in zip(got, [dict(E=e, B=b)[k] for k in want]):
        assert np.array_equal(g, ref.T)
    assert np.array_equal(fl, c) and fl.any()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 63, 513, 20011, 300007])
def test_step_off_mesh(n, prec):
    """Fused steps on a fixed mesh that particles leave: every particle's field
    is the oracle's interpolation of the step's own mesh fields (FP64 exactly;
    FP32: weights, node values and eight-term sums rounded to FP32)."""
    shape = (24, 20, 33)
    x, y, z = gaussian_bunch(n, (1e-3, 1e-3, 2e-3), seed=n + 7)
    x[0] = 0.0
    y[0] = z[0] = 1e-4
    m = osc.Mesh3D(nhi=shape, gamma=3.0)
    m.min, m.max = np.array([-2e-3, -2.5e-3, -4e-3]), np.array([2.2e-3, 2e-3, 5e-3])
    m.delta = (m.max - m.min) / (np.array(shape) - 1)
    ctx = osc.Context(0, precision=osc.OSC_PREC_FP32 if prec == "fp32" else osc.OSC_PREC_FP64)
    E, B = osc.space_charge_step(x, y, z, m, total_charge=1e-9, resize_mesh=False, calc_bfield=True,
                                 ctx=ctx)
    ctx.close()
    e, b, _ = O.interpolate_field(LO, shape, m.min, m.delta, m.efield, m.bfield, x, y, z)
    for g, ref, f in ((E, e.T, m.efield), (B, b.T, m.bfield)):
        if prec == "fp64":
            assert np.array_equal(g, ref)
        else:
            for c in range(3):
                # weights (<= 1) of 2 products, 8 terms: under 16 roundings; a
                # clamped point's weights reach the number of cells it is off
                w = 16 * 2.0 ** -24 * np.max(np.abs(f[..., c]))
                far = 1 + np.abs(np.stack([x / m.delta[0], y / m.delta[1], z / m.delta[2]])).max(0) ** 3
                assert np.all(np.abs(g[:, c] - ref[:, c]) <= w * far)


@pytest.mark.parametrize("shape", [(24, 20, 33), (96, 96, 128)])
@pytest.mark.parametrize("n", [4001, 600011])
@pytest.mark.parametrize("cathode", [False, True])
def test_step_known_b(n, shape, cathode):
    """The fused step's gather, which knows how its B was formed (no z part;
    from E without a cathode), against interpolate_field of the same fields,
    which does not: bit for bit, with particles off the mesh and one that has
    no place."""
    x, y, z = gaussian_bunch(n, (1e-3, 1e-3, 2e-3), seed=n + 3)
    z += 8e-3
    x[n // 2] = np.nan
    m = osc.Mesh3D(nhi=shape, gamma=3.0)
    m.min, m.max = np.array([-2e-3, -2.5e-3, 1e-3]), np.array([2.2e-3, 2e-3, 14e-3])
    m.delta = (m.max - m.min) / (np.array(shape) - 1)
    ctx = osc.Context(0)
    E, B = osc.space_charge_step(x, y, z, m, total_charge=1e-9, resize_mesh=False, at_cathode=cathode,
                                 calc_bfield=True, ctx=ctx)
    E2, B2 = osc.interpolate_field(x, y, z, m, E=True, B=True, ctx=ctx)
    ctx.close()
    assert np.isnan(B[n // 2]).all() and np.count_nonzero(B[:, 2]) == 1
    assert np.array_equal(E, E2, equal_nan=True) and np.array_equal(B, B2, equal_nan=True)
