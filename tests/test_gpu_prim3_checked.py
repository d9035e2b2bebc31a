"""k_prim3's checked and plain instantiations (csrc/green.hip) on the GPU, bit
for bit: a grid long enough in z that two transverse axes count as close to zero
takes the checked kernel, its middle planes as a grid of their own the plain one,
at the same coordinates (spacings in z are whole numbers times a power of two,
so that the planes' coordinates are exact)."""
import numpy as np
import pytest

import openspacecharge_amd as osc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [2.0 ** -166, 1.0, 2.0 ** 166])
@pytest.mark.parametrize("dx,dy,dz", [(1 / 3, 0.29, 1024.0), (0.41, 0.7 / 3, 768.0)])
@pytest.mark.parametrize("icomp", [1, 2, 3])
def test_same_bits(dx, dy, dz, scale, icomp):
    ctx = osc.Context(0)
    got = []
    for nz in (16, 64):
        g = np.zeros((64, 60, nz), dtype=np.complex128, order="F")
        osc.osc_get_cgrn_freespace(g, (dx * scale, dy * scale, dz * scale), 1.0, icomp, None, ctx=ctx)
        got.append(g)
    ctx.close()
    short, long = got
    a, b = short[:-1, :-1, :15], long[:-1, :-1, 24:39]
    assert np.isfinite(a).all() and np.abs(a).max() > 0
    assert np.array_equal(a, b)
