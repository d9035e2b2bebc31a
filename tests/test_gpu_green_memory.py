"""Device memory of Green builds on grids too large to build the three
components side by side (csrc/green.hip, build_spectra): the real arrays take
one component's place beside the spectra, and the fields are those of the other
precision to its rounding."""
import numpy as np
import pytest

import openspacecharge_amd as osc

pytestmark = pytest.mark.gpu

F32, F64 = osc.OSC_PREC_FP32, osc.OSC_PREC_FP64


def bucket(nbytes):
    """What the buffer pool allocates for a request (below 1 GiB)."""
    return 1 << max(8, (int(nbytes) - 1).bit_length())


def solve(ctx, solver, shape):
    import torch
    m = osc.Mesh3D(nhi=shape, gamma=3.0, device="cuda")
    m.min = np.array([-1e-3, -0.7e-3, 0.3e-3])
    m.delta = np.array([2e-3, 1.4e-3, 1.1e-3]) / (np.array(shape) - 1)
    m.max = m.min + m.delta * (np.array(shape) - 1)
    m.allocate()
    rho = np.random.default_rng(sum(shape)).random(shape) * 1e-12
    m.rho.copy_(torch.from_numpy(np.asfortranarray(rho)))
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    c = ctx()
    if solver in ("free", "cathode"):
        osc.space_charge_3d(m, at_cathode=solver == "cathode", calc_bfield=True, ctx=c)
    elif solver == "legacy":
        osc.space_charge_freespace(m, ctx=c)
    else:
        osc.space_charge_cathodeimages(m, ctx=c)
    c.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    out = np.concatenate([m.efield.cpu().numpy(), m.bfield.cpu().numpy()], axis=-1)
    c.close()
    return out, used


@pytest.mark.parametrize("shape", [(128, 64, 96), (90, 81, 100)])
@pytest.mark.parametrize("solver", ["free", "cathode", "legacy", "legacy-cathode"])
def test_one_real_array(solver, shape):
    # a first context: what the process keeps (code, tables) is not counted
    solve(lambda: osc.Context(0), solver, (8, 8, 8))
    L = [2 * n for n in shape]
    kxp = (L[0] // 2 + 1 + 15) // 16 * 16
    terms = 6 if "cathode" in solver else 3
    got = {}
    for prec, size in ((F64, 16), (F32, 8)):
        got[prec], used = solve(lambda: osc.Context(0, precision=prec), solver, shape)
        spec, real = bucket(size * kxp * L[1] * L[2]), bucket(8 * L[0] * L[1] * L[2])
        # the Green spectra, rho's, and for each z spectrum of an image solve in
        # FP32 or without plans; the real array; the inverse's arrays (E and B,
        # or their parts)
        full = 6 if "cathode" in solver and (prec == F32 or shape[0] == 90) else 0
        inverse = bucket(size * kxp * L[1] * shape[2] * (6 if "cathode" in solver else 3))
        most = (terms + 1 + full) * spec + real + inverse + (24 << 20)
        print(solver, shape, "fp64" if size == 16 else "fp32", used >> 20, "MB of", most >> 20, flush=True)
        assert used <= most
    scale = np.abs(got[F64]).max(axis=(0, 1, 2))
    err = np.abs(got[F32] - got[F64]).max(axis=(0, 1, 2))
    assert np.all(err[:5] <= 1e-5 * scale[:5])
    assert not got[F64][..., 5].any() and not got[F32][..., 5].any()
