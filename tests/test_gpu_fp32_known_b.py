"""The FP32 step's gather, which knows how its B was formed (no z part; from E
without a cathode), bit for bit against numpy in FP32 from the step's own mesh
fields: weights formed in FP64 and rounded, node values rounded, the eight terms
in upstream's order (open_spacecharge_mod.f90:369-376)."""
import numpy as np
import pytest

import openspacecharge_amd as osc
from oracle.oracle import gaussian_bunch

pytestmark = pytest.mark.gpu

f32 = np.float32


def gather(field, p, mn, delta):
    """(n, 3) FP32 values of the mesh field at the points."""
    idx, w = [], []
    for a in range(3):
        h = 1.0 / delta[a]
        i = np.clip(np.floor((p[a] - mn[a]) * h + 1.0), 1, field.shape[a] - 1)
        idx.append(i.astype(int) - 1)
        w.append((((mn[a] - p[a]) + i * delta[a]) * h).astype(f32))
    (i, j, k), (ab, de, gh) = idx, w
    one = f32(1)
    out = np.empty((len(i), 3))
    for c in range(3):
        F = field[..., c].astype(f32)
        s = F[i, j, k] * ab * de * gh
        s = s + F[i, j + 1, k] * ab * (one - de) * gh
        s = s + F[i, j + 1, k + 1] * ab * (one - de) * (one - gh)
        s = s + F[i, j, k + 1] * ab * de * (one - gh)
        s = s + F[i + 1, j, k + 1] * (one - ab) * de * (one - gh)
        s = s + F[i + 1, j + 1, k + 1] * (one - ab) * (one - de) * (one - gh)
        s = s + F[i + 1, j + 1, k] * (one - ab) * (one - de) * gh
        s = s + F[i + 1, j, k] * (one - ab) * de * gh
        assert s.dtype == f32
        out[:, c] = s
    return out


@pytest.mark.parametrize("shape", [(24, 20, 33), (96, 96, 128)])
@pytest.mark.parametrize("n", [777, 400009])
@pytest.mark.parametrize("cathode", [False, True])
def test_bits(shape, n, cathode):
    x, y, z = gaussian_bunch(n, (1e-3, 1e-3, 2e-3), seed=n + 5)
    z += 8e-3
    m = osc.Mesh3D(nhi=shape, gamma=3.0)
    # a mesh that a few particles leave
    m.min, m.max = np.array([-2e-3, -2.5e-3, 1e-3]), np.array([2.2e-3, 2e-3, 14e-3])
    m.delta = (m.max - m.min) / (np.array(shape) - 1)
    ctx = osc.Context(0, precision=osc.OSC_PREC_FP32)
    E, B = osc.space_charge_step(x, y, z, m, total_charge=1e-9, resize_mesh=False, at_cathode=cathode,
                                 calc_bfield=True, ctx=ctx)
    ctx.close()
    p = (x, y, z)
    assert np.array_equal(E, gather(m.efield, p, m.min, m.delta))
    assert np.array_equal(B, gather(m.bfield, p, m.min, m.delta))
    assert not B[:, 2].any()
