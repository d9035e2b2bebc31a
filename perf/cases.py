"""Performance cases of the space-charge path: what a tracking code has this
library do, through the public entry points, over the range it is used in.

A case is one pass of ``deposit -> solve -> gather``:

* ``call`` "step": the fused ``space_charge_step``; "calls": the same as three
  drop-in calls; "stream": a handful of requests on a running ``Server``.
* ``solver``: "free" and "cathode" (``space_charge_3d``), "pipe"
  (``space_charge_rectpipe``), "legacy" and "legacy-cathode"
  (``space_charge_freespace``, ``space_charge_cathodeimages``).
* ``mesh`` "bunch": the mesh follows the bunch, so that every step has a Green
  function of its own (the spectrum cache is off, as it could only hit because
  a measurement repeats its inputs); "fixed": the mesh stays, and the spectra
  cached by earlier steps are used, as in a run on one mesh.
* ``charges``: a charge per particle instead of one total charge.
* ``points`` > 0: the fields are wanted at that many other points.
* ``host``: the arrays are numpy arrays, as a Fortran caller's are.
"""
import math
import random

import numpy as np
import torch

GAMMA = 5.0e6 / 0.510998910e6
QTOT = 1e-9
PIPE_A, PIPE_B = 10e-3, 6e-3


def _case(name, call, solver, precision, nx, ny, nz, n, ratio, mesh="bunch", charges=False, points=0,
          host=False, bfield=True):
    c = dict(call=call, solver=solver, precision=precision, nx=nx, ny=ny, nz=nz, n=n, ratio=ratio,
             mesh=mesh, charges=charges, points=points, host=host, bfield=bfield)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest bunches of a parameter scan: latency and launches
        _case("step-32", "step", "free", "fp64", 32, 32, 32, 100_000, 2.0),
        # a small bunch of a batch, in the FP32 mode, a pancake (sigma_z << sigma_x)
        _case("step-48-fp32", "step", "free", "fp32", 48, 48, 48, 300_000, 0.2),
        # edges that are no product of 2s and 3s, an ordinary number of particles
        _case("step-100x75x60", "step", "free", "fp64", 100, 75, 60, 1_000_000, 0.5),
        # the headline size, in both precisions
        _case("step-128", "step", "free", "fp64", 128, 128, 128, 10_000_000, 4.0),
        _case("step-128-fp32", "step", "free", "fp32", 128, 128, 128, 10_000_000, 4.0),
        # the largest request of the served mix
        _case("step-256-fp32", "step", "free", "fp32", 256, 256, 256, 20_000_000, 1.0, bfield=False),
        # a gun: cathode images on a long mesh
        _case("cathode-128x128x256", "step", "cathode", "fp64", 128, 128, 256, 5_000_000, 0.5),
        # a beam in a rectangular pipe, its Green functions built once
        _case("pipe-64x64x128", "calls", "pipe", "fp64", 64, 64, 128, 2_000_000, 3.0, mesh="fixed"),
        # a run on one mesh with weighted macroparticles and test particles
        _case("fixed-96x96x128", "calls", "free", "fp64", 96, 96, 128, 2_000_000, 1.0, mesh="fixed",
              charges=True, points=300_000),
        # the legacy image solver on the mesh of the cathode comparison
        _case("legacy-cathode-64", "calls", "legacy-cathode", "fp64", 64, 64, 64, 2_000_000, 1.0),
        # the drop-in calls on host arrays (the free-space benchmark mesh)
        _case("host-64x64x128", "calls", "free", "fp64", 64, 64, 128, 1_000_000, 0.1, host=True),
        # a served stream: independent requests of mixed sizes in flight together
        dict(name="stream-8-fp32", call="stream", precision="fp32", requests=8, mix=7, workers=4),
    ]


def _smooth(e, primes):
    for p in primes:
        while e % p == 0:
            e //= p
    return e == 1


def _edge(rng, lo, hi):
    """A mesh edge, over its logarithm: half of them products of 2s and 3s
    (the usual choice), the others of any primes the transforms take."""
    primes = (2, 3) if rng.random() < 0.5 else (2, 3, 5, 7, 11, 13, 17, 19, 23)
    while True:
        e = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        if _smooth(e, primes):
            return e


def draw(rng):
    u = rng.random()
    if u < 0.12:
        return dict(call="stream", precision=rng.choice(["fp64", "fp32"]), requests=rng.randint(4, 8),
                    mix=rng.randrange(1 << 20), workers=rng.choice([2, 4]))
    while True:
        nx, ny, nz = (_edge(rng, 16, 200) for _ in range(3))
        if rng.random() < 0.3:
            ny = nx
        most = 128 ** 3 if all(_smooth(e, (2, 3)) for e in (nx, ny, nz)) else 56 ** 3
        if nx * ny * nz <= most:
            break
    n = int(math.exp(rng.uniform(math.log(1e4), math.log(5e6))))
    ratio = math.exp(rng.uniform(math.log(0.05), math.log(20.0)))
    if u < 0.62:
        return _case(None, "step", rng.choice(["free", "free", "cathode"]), rng.choice(["fp64", "fp32"]),
                     nx, ny, nz, n, ratio, charges=rng.random() < 0.2, bfield=rng.random() < 0.8)
    solver = rng.choice(["free", "cathode", "pipe", "legacy", "legacy-cathode"])
    fixed = solver == "pipe" or (solver == "free" and rng.random() < 0.6)
    host = rng.random() < 0.15
    return _case(None, "calls", solver, "fp64", nx, ny, nz, min(n, 1_000_000) if host else n,
                 min(ratio, 3.0) if solver == "pipe" else ratio, mesh="fixed" if fixed else "bunch",
                 charges=rng.random() < 0.3, points=rng.choice([0, 0, max(1000, n // 7)]), host=host)


def _requests(case):
    """The sizes of a stream's requests (the batch of mixed grids)."""
    rng = random.Random(case["mix"])
    out = []
    for _ in range(case["requests"]):
        nx, ny, nz = rng.choice([(32,) * 3, (48,) * 3, (64,) * 3, (96, 96, 128), (128,) * 3])
        out.append(_case(None, "step", rng.choice(["free", "free", "cathode"]), case["precision"], nx, ny, nz,
                         int(math.exp(rng.uniform(math.log(1e5), math.log(4e6)))),
                         math.exp(rng.uniform(math.log(0.05), math.log(20.0))), bfield=False))
    return out


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _sigma(case):
    if case["solver"] == "pipe":
        return 1e-3, 0.6e-3, 1e-3 * case["ratio"]
    return 1e-3, 1e-3, 1e-3 * case["ratio"]


def _gauss(gen, n, sigma, center, zpos):
    """A seeded Gaussian bunch cut at 4 sigma."""
    got, have = [], 0
    while have < n:
        r = torch.randn((int((n - have) * 1.2) + 64, 3), generator=gen, device=_DEV, dtype=torch.float64)
        r = r[(r * r).sum(1) <= 16.0]
        r = r * torch.tensor(sigma, dtype=torch.float64, device=_DEV)
        r = r + torch.tensor(center, dtype=torch.float64, device=_DEV)
        if zpos:
            r = r[r[:, 2] > 0]
        got.append(r)
        have += r.shape[0]
    r = torch.cat(got)[:n]
    return tuple(r[:, a].contiguous() for a in range(3))


def _bounds(case):
    """Corners of a fixed mesh."""
    s = _sigma(case)
    if case["solver"] == "pipe":
        return (-PIPE_A / 2, -PIPE_B / 2, -6 * s[2]), (PIPE_A / 2, PIPE_B / 2, 6 * s[2])
    return tuple(-4.1 * v for v in s), tuple(4.1 * v for v in s)


def _inputs(case, seed):
    gen = torch.Generator(device=_DEV)
    gen.manual_seed(1_000_003 * int(seed) + 17)
    s = _sigma(case)
    cathode = case["solver"] in ("cathode", "legacy-cathode")
    center = (0.0, 0.0, 1.5 * s[2] + 0.5e-3 if cathode else 0.0)
    xyz = _gauss(gen, case["n"], s, center, cathode)
    q = None
    if case["charges"]:
        q = (0.5 + torch.rand(case["n"], generator=gen, device=_DEV, dtype=torch.float64)) * (QTOT / case["n"])
    # test particles: a smaller bunch inside the first, on whose mesh they stay
    pts = xyz
    if case["points"]:
        pts = _gauss(gen, case["points"], tuple(0.5 * v for v in s), center, cathode)
    return xyz, q, pts


_STREAM = []


def _stream():
    """The one stream of the program: its tensors and the library's work are
    on it, so that a buffer torch hands out again is never still written to."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    torch.cuda.set_stream(_STREAM[0])
    return _STREAM[0].cuda_stream


def prepare(case, seed):
    import openspacecharge_amd as osc
    stream = _stream()
    prec = osc.OSC_PREC_FP32 if case["precision"] == "fp32" else osc.OSC_PREC_FP64
    if case["call"] == "stream":
        reqs = _requests(case)
        parts = [_inputs(r, 131 * int(seed) + k)[0] for k, r in enumerate(reqs)]
        E = [torch.empty((r["n"], 3), dtype=torch.float64, device="cuda") for r in reqs]
        torch.cuda.synchronize()
        return dict(case=case, reqs=reqs, parts=parts, E=E, prec=prec,
                    server=osc.Server(nworkers=case["workers"], green_cache=False))
    xyz, q, pts = _inputs(case, seed)
    torch.cuda.synchronize()
    ctx = osc.Context(0, precision=prec)
    if case["mesh"] == "bunch":
        ctx.set_green_cache(False)
    if case["host"]:
        xyz = tuple(a.cpu().numpy() for a in xyz)
        pts = xyz if not case["points"] else tuple(a.cpu().numpy() for a in pts)
        q = None if q is None else q.cpu().numpy()
    else:
        ctx.set_stream(stream)
        ctx.set_async(True)
    mesh = osc.Mesh3D(nhi=(case["nx"], case["ny"], case["nz"]), gamma=GAMMA,
                      device="host" if case["host"] else "cuda")
    if case["mesh"] == "fixed":
        lo, hi = _bounds(case)
        mesh.min, mesh.max = np.array(lo), np.array(hi)
        mesh.delta = (mesh.max - mesh.min) / (np.array(mesh.shape) - 1)
    if case["solver"] == "pipe":
        osc.osc_alloc_rectpipe_arrays(mesh.nlo, mesh.nhi, mesh.npad, ctx=ctx)
        osc.osc_getgrnpipe(GAMMA, PIPE_A, PIPE_B, mesh.delta, mesh.min, mesh.npad, ctx=ctx)
    return dict(case=case, xyz=xyz, q=q, pts=pts, ctx=ctx, mesh=mesh)


def run(state):
    import openspacecharge_amd as osc
    case = state["case"]
    if case["call"] == "stream":
        srv, tickets = state["server"], []
        for r, (x, y, z), E in zip(state["reqs"], state["parts"], state["E"]):
            tickets.append(srv.submit(x, y, z, E, nhi=(r["nx"], r["ny"], r["nz"]), gamma=GAMMA, total_charge=QTOT,
                                      solver=r["solver"], precision=state["prec"]))
        for t in tickets:
            srv.wait(t)
        return {"E": list(state["E"])}
    (x, y, z), mesh, ctx = state["xyz"], state["mesh"], state["ctx"]
    charge = dict(qa=state["q"]) if case["charges"] else dict(total_charge=QTOT)
    resize = case["mesh"] == "bunch"
    want_b = case["bfield"]
    if case["call"] == "step":
        got = osc.space_charge_step(x, y, z, mesh, resize_mesh=resize, at_cathode=case["solver"] == "cathode",
                                    calc_bfield=want_b, ctx=ctx, **charge)
    else:
        osc.deposit_particles(x, y, z, mesh, resize_mesh=resize, count_dropped=False, ctx=ctx, **charge)
        if case["solver"] in ("free", "cathode"):
            osc.space_charge_3d(mesh, at_cathode=case["solver"] == "cathode", calc_bfield=want_b, ctx=ctx)
        elif case["solver"] == "pipe":
            osc.space_charge_rectpipe(mesh, PIPE_A, PIPE_B, direct_field_calc=False, ctx=ctx)
        elif case["solver"] == "legacy":
            osc.space_charge_freespace(mesh, ctx=ctx)
        else:
            osc.space_charge_cathodeimages(mesh, ctx=ctx)
        px, py, pz = state["pts"]
        got = osc.interpolate_field(px, py, pz, mesh, E=True, B=want_b, ctx=ctx)
    E, B = got if want_b else (got, None)
    out = {"E": E, "rho": mesh.rho, "efield": mesh.efield}
    if want_b:
        out.update(B=B, bfield=mesh.bfield)
    if case["solver"] == "pipe":
        out["phi"] = mesh.phi
    return out


# ---------------------------------------------------------------------------
# compulsory work
# ---------------------------------------------------------------------------
def work(case):
    if case["call"] == "stream":
        each = [work(r) for r in _requests(case)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    P, M, n = case["n"], case["points"] or case["n"], case["nx"] * case["ny"] * case["nz"]
    per = 48 if case["bfield"] else 24
    nbytes = (32 if case["charges"] else 24) * P + per * M + (24 * M if case["points"] else 0) + (8 + per) * n
    N = 8 * n
    fft = 2.5 * N * math.log2(N)
    greens = {"free": 3, "cathode": 6, "legacy": 3, "legacy-cathode": 6, "pipe": 0}[case["solver"]]
    if case["mesh"] == "fixed":
        greens = 0
    fields = 1 if case["solver"] == "pipe" else 3
    terms = {"free": 3, "cathode": 6, "legacy": 3, "legacy-cathode": 6, "pipe": 4}[case["solver"]]
    if case["solver"] == "pipe":
        nbytes += 8 * n
    # transforms, spectral products, Green cells (three logarithms and arc
    # tangents' worth each), deposit and gather
    flops = fft * (1 + greens + fields) + 4 * N * terms + 60.0 * N * greens + 40.0 * P + 8.0 * per * M / 8 * 4
    return {"bytes": float(nbytes), "flops": float(flops)}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
_C = {"free": 299792448.0, "cathode": 299792448.0}
_FPEI = {"free": 8987551502.2918644, "cathode": 8987551502.2918644, "pipe": 8987551744.0}


def _cells(p, mn, delta, n):
    """Lower node index and weight of it, per axis."""
    out = []
    for a in range(3):
        f = (p[a] - mn[a]) / delta[a]
        i = torch.floor(f).clamp_(0, n[a] - 2)
        out.append((i.long(), 1.0 - (f - i)))
    return out


def _corners(p, mn, delta, n):
    (i, a), (j, b), (k, c) = _cells(p, mn, delta, n)
    for di in (0, 1):
        for dj in (0, 1):
            for dk in (0, 1):
                w = (1 - a if di else a) * (1 - b if dj else b) * (1 - c if dk else c)
                yield (i + di) + n[0] * ((j + dj) + n[1] * (k + dk)), w


def _deposit(p, q, mn, delta, n):
    rho = torch.zeros(n[0] * n[1] * n[2], dtype=torch.float64, device=p[0].device)
    for s in range(0, p[0].numel(), 4_000_000):
        sl = slice(s, s + 4_000_000)
        for at, w in _corners([c[sl] for c in p], mn, delta, n):
            rho.index_add_(0, at, w * (q[sl] if torch.is_tensor(q) else q))
    return rho.view(n[2], n[1], n[0])


def _gather(fields, p, mn, delta, n):
    """(3, nz, ny, nx) at the points -> (points, 3)."""
    flat = fields.reshape(3, -1)
    out = torch.zeros((p[0].numel(), 3), dtype=torch.float64, device=p[0].device)
    for s in range(0, p[0].numel(), 4_000_000):
        sl = slice(s, s + 4_000_000)
        for at, w in _corners([c[sl] for c in p], mn, delta, n):
            for a in range(3):
                out[sl, a] += flat[a][at] * w
    return out


def _primitive(x, y, z):
    """An antiderivative of x / r^3 in all three variables."""
    r = torch.sqrt(x * x + y * y + z * z)

    def logp(v, rest):  # log(r + v), without the cancellation at v near -r
        return torch.where(v >= 0, torch.log(r + v), torch.log(rest / (r - v)))
    return x * torch.atan((y * z) / (r * x)) - z * logp(y, x * x + z * z) - y * logp(z, x * x + y * y)


def _field(rho, n, delta, zoff, fpei, hole=False):
    """E (3, nz, ny, nx) of the node charges rho (nz, ny, nx): the convolution
    with the cell-averaged 1/r^2 kernel, its cells shifted by zoff in z; with
    hole, the kernel is zero in a cell around the origin, as the legacy
    solvers have it."""
    d = [delta[0], delta[1], delta[2] * GAMMA]
    L = [2 * m for m in n]
    dev = rho.device
    ax = [(torch.arange(L[a], dtype=torch.float64, device=dev) + (0.5 - n[a])) * d[a] for a in range(3)]
    ax[2] = ax[2] + zoff * GAMMA
    u, v, w = ax[0].view(1, 1, -1), ax[1].view(1, -1, 1), ax[2].view(-1, 1, 1)
    rhat = torch.fft.rfftn(rho, s=(L[2], L[1], L[0]))
    out = torch.empty((3,) + tuple(rho.shape), dtype=torch.float64, device=dev)
    for a, args in enumerate(((u, v, w), (v, w, u), (w, u, v))):
        g = _primitive(*args)
        for dim in range(3):
            g = torch.diff(g, dim=dim)
        g = torch.nn.functional.pad(g, (0, 1, 0, 1, 0, 1))
        k = round(n[2] - 1 - zoff / delta[2])
        if hole and 0 <= k < L[2] and abs((k + 1 - n[2]) * delta[2] + zoff) < 0.5 * delta[2]:
            g[k, n[1] - 1, n[0] - 1] = 0.0
        c = torch.fft.irfftn(torch.fft.rfftn(g) * rhat, s=(L[2], L[1], L[0]))
        scale = fpei * (GAMMA if a < 2 else 1.0) / (d[0] * d[1] * d[2])
        out[a] = scale * c[n[2] - 1:2 * n[2] - 1, n[1] - 1:2 * n[1] - 1, n[0] - 1:2 * n[0] - 1]
    return out


def _pipe_phi(rho, n, mn, delta):
    """The potential in the pipe: 5 x 5 modes, by their separable sums."""
    dev = rho.device
    idx = [torch.arange(m, dtype=torch.float64, device=dev) for m in n]

    def mode(a, m, size):
        f = m * math.pi / size
        dif = (idx[a].view(-1, 1) - idx[a].view(1, -1)) * delta[a]
        tot = 2.0 * mn[a] + (idx[a].view(-1, 1) + idx[a].view(1, -1)) * delta[a]
        return torch.cos(f * dif) - (-1.0) ** m * torch.cos(f * tot)
    w = (idx[2].view(-1, 1) - idx[2].view(1, -1)) * delta[2] * GAMMA
    hz = delta[2]
    phi = torch.zeros_like(rho)
    for m in range(1, 6):
        rx = rho @ mode(0, m, PIPE_A).T
        for k in range(1, 6):
            kap = math.hypot(m * math.pi / PIPE_A, k * math.pi / PIPE_B)
            ry = mode(1, k, PIPE_B) @ rx
            zf = (torch.exp(-kap * (w - hz).abs()) - 2.0 * torch.exp(-kap * w.abs())
                  + torch.exp(-kap * (w + hz).abs())) / (hz * hz * kap * kap)
            zf = zf + torch.eye(n[2], dtype=torch.float64, device=dev) * (2.0 / (hz * kap))
            phi += ((zf / kap) @ ry.reshape(n[2], -1)).reshape(phi.shape)
    return phi * (2.0 * math.pi / (PIPE_A * PIPE_B)) * _FPEI["pipe"]


def _gradient(phi, delta):
    """-grad phi as the finite-difference rule of the potential solvers."""
    out = torch.empty((3,) + tuple(phi.shape), dtype=torch.float64, device=phi.device)
    for a, dim in enumerate((2, 1, 0)):
        g = torch.gradient(phi, spacing=delta[a], dim=dim, edge_order=1)[0]
        out[a] = -g * (GAMMA if a < 2 else 1.0 / GAMMA)
    return out


def exact(case, seed):
    if case["call"] == "stream":
        return {"E": [exact(r, 131 * int(seed) + k)["E"] for k, r in enumerate(_requests(case))]}
    xyz, q, pts = _inputs(case, seed)
    n = (case["nx"], case["ny"], case["nz"])
    if case["mesh"] == "fixed":
        mn, mx = _bounds(case)
        delta = [(mx[a] - mn[a]) / (n[a] - 1) for a in range(3)]
    else:  # the bunch's extent and a millionth of a cell
        lo, hi = [float(c.min()) for c in xyz], [float(c.max()) for c in xyz]
        d = [(hi[a] - lo[a]) / (n[a] - 1) for a in range(3)]
        mn, mx = [lo[a] - 1e-6 * d[a] for a in range(3)], [hi[a] + 1e-6 * d[a] for a in range(3)]
        delta = [(mx[a] - mn[a]) / (n[a] - 1) for a in range(3)]
    rho = _deposit(xyz, q if case["charges"] else QTOT / case["n"], mn, delta, n)
    solver, phi = case["solver"], None
    cl, fpei = _C.get(solver, 299792458.0), _FPEI.get(solver, 299792458.0 ** 2 * 1e-7)
    bc = math.sqrt(1.0 - 1.0 / GAMMA ** 2) / cl
    if solver == "pipe":
        phi = _pipe_phi(rho, n, mn, delta)
        E = _gradient(phi, delta)
        Bt = E
    else:
        E = _field(rho, n, delta, 0.0, fpei)
        Bt = E
        if solver.endswith("cathode"):  # the image charges move the other way
            img = _field(-rho.flip(0), n, delta, 2 * mn[2] + (mx[2] - mn[2]), fpei, solver != "cathode")
            Bt = E - img
            E = E + img
    out = {"E": _gather(E, pts, mn, delta, n), "rho": rho.permute(2, 1, 0), "efield": E.permute(3, 2, 1, 0)}
    if case["bfield"]:
        B = torch.stack([-bc * Bt[1], bc * Bt[0], torch.zeros_like(E[0])])
        out.update(B=_gather(B, pts, mn, delta, n), bfield=B.permute(3, 2, 1, 0))
    if phi is not None:
        out["phi"] = phi.permute(2, 1, 0)
    return out
