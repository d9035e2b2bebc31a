"""Admission of the request loop: requests on grids whose Green components are
built through one real array are counted with one, so that a budget for two of
them runs two at a time."""
import pytest

import openspacecharge_amd as osc
from oracle.oracle import gaussian_bunch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [osc.OSC_PREC_FP32, osc.OSC_PREC_FP64])
def test_budget_for_two_runs_two(precision):
    import torch
    nhi, n = (96, 96, 128), 2_000_000
    nodes = nhi[0] * nhi[1] * nhi[2]
    # mesh arrays, ten half spectra of the doubled grid, its real array, node
    # records, particles, and a constant
    one = 3 * 64 * nodes + 10 * (nhi[0] + 1) * 4 * nhi[1] * nhi[2] * 16 + 96 * n + (64 << 20)
    t = [torch.from_numpy(a).cuda() for a in gaussian_bunch(n, (1e-3, 1e-3, 1e-3), seed=5)]
    out = [torch.empty((n, 3), dtype=torch.float64, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    srv = osc.Server(nworkers=2, max_bytes=2 * one + (1 << 20))
    tickets = [srv.submit(*t, E, nhi=nhi, gamma=9.8, total_charge=1e-9, precision=precision) for E in out]
    for k in tickets:
        srv.wait(k)
    st = srv.stats()
    srv.close()
    assert st["max_running"] == 2
    assert torch.equal(out[0], out[1])
