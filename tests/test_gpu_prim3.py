"""The FP64 offset-grid primitives of k_prim3 (csrc/green.hip), with and
without its range checks, against the oracle: grids that leave part of a block
or of its planes empty, needles and pancakes whose terms cancel, a coordinate
that an offset makes zero, and magnitudes the plain sequences do not cover."""
import numpy as np
import pytest

import openspacecharge_amd as osc
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

CASES = {
    "one-block": ((2, 2, 2), (1e-4, 1e-4, 1e-4), 1.0, None),
    "ragged": ((66, 7, 9), (1e-4, 2e-4, 3e-4), 9.78, None),
    "needle": ((8, 8, 130), (1e-5, 1e-5, 3e-3), 5.0, None),
    "pancake": ((40, 36, 6), (1e-3, 1e-3, 1e-8), 1.0, None),
    # w = 0 at one plane (the corner values of the cells there)
    "zero-plane": ((12, 10, 16), (1e-4, 1e-4, 1e-4), 1.0, (0.0, 0.0, 0.5e-4)),
    # two axes close to zero: the checked kernel
    "zero-line": ((12, 10, 16), (1e-4, 1e-4, 1e-4), 1.0, (0.0, 0.499999e-4, 0.499999e-4)),
    "huge": ((10, 8, 6), (1e62, 2e62, 1e62), 1.0, None),
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("icomp", [1, 2, 3])
def test_primitive(name, icomp):
    shape, delta, gam, off = CASES[name]
    O = Oracle()
    # the differenced cells (the last plane of each axis keeps raw primitives)
    cells = (slice(0, -1),) * 3
    ref, floor = O.floor(lambda: O.get_cgrn_freespace(shape, delta, gam, icomp, off)[cells])
    g = np.zeros(shape, dtype=np.complex128, order="F")
    ctx = osc.Context(0)
    osc.osc_get_cgrn_freespace(g, delta, gam, icomp, off, ctx=ctx)
    ctx.close()
    # each of a primitive's logarithms and arc tangents within 1.5 ulp of the
    # oracle's 0.5, on top of the floor's one ulp of the whole
    g = g[cells]
    assert np.max(np.abs(g - ref)) <= (4 * floor + 2e-14) * np.max(np.abs(ref))
