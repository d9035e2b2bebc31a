"""The integrated legacy Green functions of k_green_legacy (csrc/green.hip),
with and without its range checks, against the oracle: grids that leave part
of a block or of a thread's planes empty, needles and pancakes whose terms
cancel, corners on the plane z = 0, a shifted order of the planes, and
magnitudes the plain sequences do not cover."""
import numpy as np
import pytest

import openspacecharge_amd as osc
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

# mesh nodes, spacing, gamma
CASES = {
    "one-block": ((2, 2, 2), (1e-4, 1e-4, 1e-4), 1.0),
    "ragged": ((33, 3, 5), (1e-4, 2e-4, 3e-4), 9.78),
    "planes": ((5, 4, 33), (1.1e-4, 0.7e-4, 1.3e-4), 2.0),
    "needle": ((8, 8, 64), (1e-5, 1e-5, 3e-3), 5.0),
    "pancake": ((40, 36, 6), (1e-3, 1e-3, 1e-8), 1.0),
    "huge": ((6, 5, 4), (1e62, 2e62, 1e62), 1.0),
}


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("icomp", [0, 1, 2, 3])
def test_green(name, icomp):
    n, dl, gam = CASES[name]
    O = Oracle()
    nlo, npad = (1, 1, 1), (1, 1, 1)
    ctx = osc.Context(0)
    um = (0.0, 0.0, 2.5 * dl[2])
    calls = [lambda L, **k: L(nlo, n, npad, dl, gam, icomp, 1, **k),
             # the corners of one plane at z = 0
             lambda L, **k: L(nlo, n, npad, dl, gam, 0.5 * dl[2], icomp, 1, **k),
             lambda L, **k: L(nlo, n, npad, um, dl, gam, icomp, 1, **k)]
    fns = [(osc.osc_getgrnfree, O.getgrnfree), (osc.osc_getgrnimageshift, O.getgrnimageshift),
           (osc.osc_getgrnimageconvcorr, O.getgrnimageconvcorr)]
    for call, (dev, ora) in zip(calls, fns):
        g = call(dev, ctx=ctx)
        ref, floor = O.floor(lambda: call(ora))
        # a corner's logarithms and arc tangents are within 1.5 ulp of the
        # exact ones where the floor moves the whole value by one ulp
        assert np.max(np.abs(g - ref)) <= (4 * floor + 2e-14) * np.max(np.abs(ref))
    ctx.close()
