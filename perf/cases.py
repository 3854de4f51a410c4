"""Cases of the collision operator's use: what is timed, on which inputs, and what its outputs should be.

A user of this package evaluates the collision operator for one cell or a batch of cells, advances 0D ensembles and 1D
meshes by whole steps, calls the reference's own host-buffer interface, and builds a weight table before a run. The
cases cover those entry points from one cell on a small grid to the 512-problem ensemble at N = 32, in the sizes of the
package's configurations, fixtures and tests. The precision form with FP32 products is used where its results are: in
an ensemble's time steps. Everything else runs in FP64, which is the only form that is accurate on near-equilibrium
cells.

Kinds of case:
  q       Operator.compute_q_dev on device arrays, with the projection (op "maxpreserve" or "computeq": Q(f, f);
          "pair": Q(f, g) of two different cells, as species pairs need it)
  abi     ComputeQ_maxPreserve and conserveAllMoments on host arrays, one cell: what the reference's driver calls
  run0d   Run.ensemble: Heun or Euler steps of independent problems, replayed as a HIP graph
  run1d   Run.mesh (or mesh_species): transport, collision and walls of a 1D mesh, replayed as a HIP graph
  table   generation of an anisotropic or isotropic weight table, and its copy to the host for the Weights/ file
"""
import ctypes
import math

import numpy as np
import torch

import spectralbte_amd as spb

HEAD = 64  # problems of an ensemble that exact() follows (they do not depend on each other)


def listed():
    return [
        # one evaluation through the reference's interface: the smallest call its driver makes
        {"name": "abi16", "kind": "abi", "N": 16, "Lv": 5.0, "lam": 0.0},
        # one device-resident evaluation of one small cell: launches and latency
        {"name": "cell16", "kind": "q", "N": 16, "Lv": 5.0, "lam": 0.0, "ncell": 1, "op": "maxpreserve"},
        # the BKW relaxation, 100 Heun steps of one cell: the reference's first test, at N = 16
        {"name": "bkw16", "kind": "run0d", "N": 16, "Lv": 5.0, "lam": 0.0, "ncell": 1, "order": 2, "dt": 0.01,
         "form": "fp64", "steps": 100},
        # the reference's heat-transfer test: 250 cells on its smallest grid, Euler steps between diffuse walls
        {"name": "heat8", "kind": "run1d", "N": 8, "Lv": 9.0, "lam": 1.0, "ncell": 250, "length": 1.0, "order": 1,
         "dt": 1e-4, "Kn": 3.2, "walls": "diffuse", "species": 1, "steps": 10},
        # one cell of the production grid: the reference's method, one pass over the weight table per evaluation
        {"name": "cell32", "kind": "q", "N": 32, "Lv": 6.0, "lam": 1.0, "ncell": 1, "op": "maxpreserve"},
        # a mesh's cells in one batch, at a count that fills no tile
        {"name": "mesh24", "kind": "q", "N": 24, "Lv": 8.0, "lam": 1.0, "ncell": 37, "op": "computeq"},
        # a grid that is no power of two or three
        {"name": "grid10", "kind": "q", "N": 10, "Lv": 6.0, "lam": 1.0, "ncell": 75, "op": "maxpreserve"},
        # a mixture: four pairs of species per cell, two of them with different arguments
        {"name": "mixture16", "kind": "run1d", "N": 16, "Lv": 7.0, "lam": 1.0, "ncell": 48, "length": 1.0, "order": 1,
         "dt": 1e-3, "Kn": 0.5, "walls": "diffuse", "species": 2, "steps": 2},
        # a weight table of the anisotropic generator, once per new grid or exponent
        {"name": "landau16", "kind": "table", "table": "landau", "N": 16, "Lv": 7.0, "lam": 1.0},
        # the smaller half of the ensemble configuration: a Heun step of 512 problems
        {"name": "ensemble24", "kind": "run0d", "N": 24, "Lv": 6.0, "lam": 1.0, "ncell": 512, "order": 2, "dt": 0.005,
         "form": "fp32a", "steps": 1},
        # the Mach-1.2 shock: a whole second-order step of 256 cells
        {"name": "shock32", "kind": "run1d", "N": 32, "Lv": 8.0, "lam": 1.0, "ncell": 256, "length": 10.0, "order": 2,
         "dt": 0.002, "Kn": 0.1, "walls": "copy", "species": 1, "steps": 1},
        # the headline batch as its users run it: a Heun step of 512 problems at N = 32
        {"name": "ensemble32", "kind": "run0d", "N": 32, "Lv": 6.0, "lam": 1.0, "ncell": 512, "order": 2, "dt": 0.005,
         "form": "fp32a", "steps": 1},
    ]


def _logint(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    """A case of the same ranges: any kind, grids of 6 to 32 nodes (odd ones too), one cell to as many as cost less than
    the largest listed case (at N = 32 a quarter of it, so that many can be drawn)."""
    kind = rng.choice(["q", "q", "q", "run0d", "run0d", "run1d", "run1d", "abi", "table"])
    lam = rng.choice([0.0, 1.0])
    Lv = round(rng.uniform(5.0, 8.5), 2)
    if kind == "abi":
        return {"kind": kind, "N": rng.choice([8, 9, 10, 12, 16, 18]), "Lv": Lv, "lam": lam}
    if kind == "table":
        return {"kind": kind, "table": rng.choice(["landau", "landau", "glance", "iso"]), "N": rng.choice([6, 8, 9, 10, 12, 15, 16]),
                "Lv": Lv, "lam": rng.choice([0.0, 0.5, 1.0])}
    N = rng.choice([6, 8, 9, 10, 12, 16, 16, 18, 20, 24, 24, 32, 32])
    most = {32: 128, 24: 300, 20: 120, 18: 160}.get(N, 600)  # grids without tiles of their own cost more per cell
    n = _logint(rng, 1, most)
    if kind == "q":
        return {"kind": kind, "N": N, "Lv": Lv, "lam": lam, "ncell": n, "op": rng.choice(["maxpreserve", "computeq", "pair"])}
    if kind == "run0d":
        form = rng.choice(["fp64", "fp32", "fp32a"]) if N in (16, 24, 32) else "fp64"
        return {"kind": kind, "N": N, "Lv": Lv, "lam": lam, "ncell": n, "order": rng.choice([1, 2, 2]), "dt": 0.005, "form": form,
                "steps": rng.randint(1, 3)}
    species = rng.choice([1, 1, 1, 2])
    return {"kind": kind, "N": N, "Lv": Lv, "lam": lam, "ncell": max(3, n // (species * species)), "length": 10.0,
            "order": rng.choice([1, 2]), "dt": 0.002, "Kn": rng.choice([0.1, 0.5, 1.0]), "walls": rng.choice(["copy", "diffuse"]),
            "species": species, "steps": 1}


# ------------------------------------------------------------------ grids and inputs
def _masses(case):
    return [1.0, 2.0][:case.get("species", 1)]


def _grid(case, Lv=None):
    """The 0D grid of the reference, or its 1D grid for mesh runs (the two agree for even N)."""
    N, Lv = case["N"], Lv or case["Lv"]
    dv = 2 * Lv / (N - 1)
    v = -Lv + np.arange(N) * dv
    if case["kind"] == "run1d":
        return v, -0.5 * (N - 1) * np.pi / Lv + np.arange(N) * (np.pi * (N - 1) / (N * Lv))
    deta = 2 * np.pi / N / dv
    return v, -(0.5 * N * deta if N % 2 == 0 else 0.5 * (N - 1) * deta) + np.arange(N) * deta


def _maxwellian(v, rho, u, T):
    """(n, N, N, N) of rho, T (n,) and u (n, 3)."""
    g = [torch.exp(-(v[None, :] - u[:, d, None]) ** 2 / (2 * T[:, None])) for d in range(3)]
    rho = rho * (2 * math.pi * T) ** -1.5
    return rho[:, None, None, None] * g[0][:, :, None, None] * g[1][:, None, :, None] * g[2][:, None, None, :]


def _weights3(N, v):
    w = torch.ones(N, dtype=torch.float64, device=v.device)
    w[0] = w[-1] = 0.5
    return w[:, None, None] * w[None, :, None] * w[None, None, :] * (v[1] - v[0]) ** 3


def _bimodal(case, v, n, gen):
    """Sums of two Maxwellians (weights U(0.2, 0.8), means U(-1.5, 1.5)^3, temperatures U(0.5, 2)) at unit density: the
    ensemble configuration's problems."""
    def u(*shape, a, b):
        return (a + (b - a) * torch.rand(shape, dtype=torch.float64, generator=gen)).to(v.device)
    f = sum(_maxwellian(v, u(n, a=0.2, b=0.8), u(n, 3, a=-1.5, b=1.5), u(n, a=0.5, b=2.0)) for _ in range(2))
    return f / (f * _weights3(case["N"], v)).sum((1, 2, 3), keepdim=True)


def _layer(case, v, n, gen, across=False):
    """Cells of a Mach-1.2 shock layer: blends of the states on its two sides (over the mesh, or anywhere in the layer)."""
    s = torch.rand(n, dtype=torch.float64, generator=gen).to(v.device) * 0.9 + 0.05
    if across:
        x = torch.arange(n, dtype=torch.float64, device=v.device) + 0.5 - n / 2
        shift = (torch.rand(1, dtype=torch.float64, generator=gen).to(v.device) - 0.5) * 0.2 * n
        s = 0.5 * (1 + torch.tanh((x - shift) / (20 / (2 * math.atanh(0.98)) * n / 256)))
    m2 = 1.2 ** 2
    u1, r2 = 1.2 * math.sqrt(5 / 3), 4 * m2 / (m2 + 3)
    T2 = (5 * m2 - 1) * (m2 + 3) / (16 * m2)
    one = torch.ones(1, dtype=torch.float64, device=v.device)

    def side(rho, ux, T):
        return _maxwellian(v, rho * one, torch.tensor([[ux, 0.0, 0.0]], dtype=torch.float64, device=v.device), T * one)
    s = s[:, None, None, None]
    return (1 - s) * side(1.0, u1, 1.0) + s * side(r2, u1 / r2, T2)


def _inputs(case, seed):
    """The distributions a pass starts from, as tensors on the GPU: (n, N, N, N), or (species, n, N, N, N)."""
    gen = torch.Generator().manual_seed(int(seed))
    N, n = case["N"], case.get("ncell", 1)
    v = torch.from_numpy(_grid(case)[0]).cuda()
    if case["kind"] == "q":
        make = _layer if case["op"] == "computeq" else _bimodal
        return [make(case, v, n, gen) for _ in range(2 if case["op"] == "pair" else 1)]
    if case["kind"] == "abi":
        return [_bimodal(case, v, 1, gen)]
    if case["kind"] == "run0d":
        if n > 1:
            return [_bimodal(case, v, n, gen)]
        K = 0.62 + 0.2 * float(torch.rand(1, generator=gen))  # the BKW solution at a time of the seed's
        V2 = v[:, None, None] ** 2 + v[None, :, None] ** 2 + v[None, None, :] ** 2
        return [((2 * math.pi * K) ** -1.5 * torch.exp(-V2 / (2 * K)) * ((5 * K - 3) / (2 * K) + (1 - K) / (2 * K * K) * V2))[None]]
    if case["walls"] == "copy":
        f = _layer(case, v, n, gen, across=True)
    else:  # a gas at rest between the walls, with 10% of density noise and a second, drifting part
        r = 1 + 0.1 * (torch.rand(n, dtype=torch.float64, generator=gen).to(v.device) - 0.5)
        one, u = torch.ones_like(r), torch.zeros(n, 3, dtype=torch.float64, device=v.device)
        f = _maxwellian(v, r, u, 1.2 * one) + _maxwellian(v, 0.3 * one, u + 0.8, 0.7 * one)
    return [torch.stack([f * (1 + 0.2 * l) for l in range(case["species"])])]


# ------------------------------------------------------------------ handles
_ops = {}


def _operator(case, table=True):
    """One operator per grid and exponent, as a program with one velocity grid keeps it."""
    key = (case["N"], case["Lv"], case["lam"], case["kind"] == "run1d", case.get("species", 1))
    if key not in _ops:
        v, eta = _grid(case)
        op = spb.Operator(case["N"], case["Lv"], v, eta)
        m = _masses(case)
        if len(m) > 1:
            op.set_species(m)
        for a in range(len(m)):
            for b in range(len(m)):
                op.select_table(b * len(m) + a)
                op.generate_weights_iso(case["lam"], 2.0, 2.0, m[a], m[b])
        op.select_table(0)
        _ops[key] = op
    return _ops[key]


class _View:
    """A device buffer of a run, for torch.as_tensor: the tensor keeps this object, and so the run that owns the buffer."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f8", "version": 3, "strides": None}


def _tensor(owner, ptr, shape):
    return torch.as_tensor(_View(owner, ptr, shape), device="cuda")


def _mesh(case):
    n, g = case["ncell"], case["order"]
    h = case["length"] / n
    return (np.arange(n + 2 * g) - g + 0.5) * h, np.full(n + 2 * g, h)


_abi = {}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "table":
        # the velocity domain is the seed's: a table depends on nothing else that could vary
        Lv = case["Lv"] * (1 + 0.05 * float(torch.rand(1, generator=torch.Generator().manual_seed(int(seed)))))
        v, eta = _grid(case, Lv)
        return {"case": case, "op": spb.Operator(case["N"], Lv, v, eta)}
    f = _inputs(case, seed)
    n3 = case["N"] ** 3
    if kind == "abi":
        key = (case["N"], case["Lv"], case["lam"])
        if _abi.get("key") != key:
            if _abi:
                spb.dealloc_coll()
                spb.dealloc_conservation()
            v, eta = _grid(case)
            spb.initialize_coll(case["N"], case["Lv"], v, eta)
            spb.initialize_conservation(case["N"], v[1] - v[0], v)
            _abi.update(key=key, rows=spb.WeightRows(_operator(case).get_weights()))
        return {"case": case, "f": f[0].reshape(n3).cpu().numpy(), "rows": _abi["rows"]}
    op = _operator(case)
    if kind == "q":
        f = [x.reshape(-1, n3).contiguous() for x in f]
        flags = spb.CONSERVE | (spb.MAXPRESERVE if case["op"] == "maxpreserve" else 0) | (spb.SELF if len(f) == 1 else 0)
        return {"case": case, "op": op, "f": f, "Q": torch.zeros_like(f[0]), "flags": flags}
    f = f[0].reshape(-1, case["ncell"], n3).cpu().numpy()
    if kind == "run0d":
        r = spb.Run.ensemble(op, f[0], order=case["order"], dt=case["dt"], Kn=1.0, form=case["form"])
    else:
        x, dx = _mesh(case)
        kw = dict(order=case["order"], dt=case["dt"], Kn=case["Kn"], T0=1.0, T1=2.0,
                  bc=spb.BC_DIFFUSE if case["walls"] == "diffuse" else spb.BC_COPY)
        r = spb.Run.mesh(op, f[0], x, dx, **kw) if len(f) == 1 else spb.Run.mesh_species(op, f, x, dx, **kw)
    r.use_graph(True)
    ptrs = []
    for l in range(len(f)):
        p = ctypes.c_void_p()
        spb._check(spb.lib().spbte_run_species_state(r.h, l, ctypes.byref(p)))
        ptrs.append(p.value)
    state = [_tensor(r, p, (case["ncell"], n3)) for p in ptrs]
    return {"case": case, "op": op, "run": r, "state": state}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "q":
        f = state["f"]
        state["op"].compute_q_dev(f[0].data_ptr(), f[1].data_ptr() if len(f) > 1 else None, state["Q"].data_ptr(), case["ncell"],
                                  "fp64", state["flags"])
        return state["Q"]
    if kind == "abi":
        return spb.conserveAllMoments([spb.ComputeQ_maxPreserve(state["f"], state["f"], state["rows"])])[0]
    if kind == "table":
        op = state["op"]
        if case["table"] == "landau":
            op.generate_weights_landau(case["lam"])
        elif case["table"] == "glance":
            op.generate_weights_glance(case["lam"], 0.1)
        else:
            op.generate_weights_iso(case["lam"])
        return op.get_weights()
    state["run"].step(case["steps"], sync=False)
    s = state["state"]
    if kind == "run0d" and case["ncell"] > HEAD:
        return {"first": s[0][:HEAD], "rest": s[0][HEAD:]}
    return s


def work(case):
    """The distributions are real, so half of the output modes fix the result, and Q(f, f) takes the modes c and r - c of
    a pair alike, so half of the summed modes do: P/4 table entries and products for Q(f, f), P/2 for Q(f, g), with
    P = N^6; 10 flops per product pair of ComputeQ and 18 of the maxPreserve split."""
    N, n = case["N"], case.get("ncell", 1)
    n3, P = N ** 3, N ** 6
    kind = case["kind"]
    if kind == "table":
        nodes = {"landau": 2048 * 40, "glance": 1500 * 60, "iso": 60}[case["table"]]
        return {"bytes": 8 * P, "flops": nodes * P / 48}  # an entry serves its images under the cube's 48 symmetries
    if kind in ("q", "abi"):
        op = case.get("op", "maxpreserve")
        share = 0.5 if op == "pair" else 0.25
        return {"bytes": share * P * 8 + (3 if op == "pair" else 2) * n * n3 * 8, "flops": share * P * n * (18 if op == "maxpreserve" else 10)}
    s = case.get("species", 1)
    stages = case["order"] * case["steps"]
    shares = 0.25 * s + 0.5 * (s * s - s)  # pairs of a species with itself and with another
    width = 4 if case.get("form") in ("fp32", "fp32a") else 8
    return {"bytes": shares * P * width * stages + 2 * s * n * n3 * 8 * case["steps"],
            "flops": shares * P * n * stages * (18 if kind == "run0d" else 10)}


# ------------------------------------------------------------------ the same in 64 bits, with plain torch
def _table(case, mi=1.0, mj=1.0):
    """The isotropic table for lambda 0 and 1 (closed forms of the radial integral), N^3 x N^3."""
    N, Lv, lam = case["N"], case["Lv"], case["lam"]
    v, eta = _grid(case)
    e = torch.from_numpy(eta).cuda()
    E = torch.stack(torch.meshgrid(e, e, e, indexing="ij")).reshape(3, -1)
    w = torch.ones(N, dtype=torch.float64, device="cuda")
    w[0] = w[-1] = 0.5
    wc = (w[:, None, None] * w[None, :, None] * w[None, None, :]).reshape(-1)
    pre = 16 * math.pi ** 2 * (eta[1] - eta[0]) ** 3 / (2 * math.pi) ** 1.5 / (4 * math.pi)
    mu = mj / (mi + mj)
    tiny = 1e-12

    def sinc(x):
        return torch.where(x == 0, torch.ones_like(x), torch.sin(x) / torch.where(x == 0, torch.ones_like(x), x))

    def fcos(x):
        return torch.where(x.abs() > 1e-12, (torch.cos(x) - 1) / torch.where(x.abs() > 1e-12, x * x, torch.ones_like(x)), x * x / 24 - 0.5)

    def single(c):  # the integral of r^(lam + 2) sinc(c r)
        s = torch.where(c > tiny, c, torch.ones_like(c))
        x = s * Lv
        if lam == 0:
            return torch.where(c > tiny, (torch.sin(x) - x * torch.cos(x)) / s ** 3, torch.full_like(c, Lv ** 3 / 3))
        return torch.where(c > tiny, (torch.cos(x) * (2 - x * x) + 2 * x * torch.sin(x) - 2) / s ** 4, torch.full_like(c, Lv ** 4 / 4))

    W = torch.empty(N ** 3, N ** 3, dtype=torch.float64, device="cuda")
    a1 = E.square().sum(0).sqrt()
    loss = single(a1)
    for r in range(0, N ** 3, N):
        z = mu * E[:, r:r + N]
        a0 = z.square().sum(0).sqrt()[:, None].expand(N, N ** 3)
        a2 = (E[:, None, :] - z[:, :, None]).square().sum(0).sqrt()
        both = (a0 > tiny) & (a2 > tiny)
        p, q = torch.where(both, a0, torch.ones_like(a0)), torch.where(both, a2, torch.ones_like(a2))
        d, s = (p - q) * Lv, (p + q) * Lv
        if lam == 0:
            g = Lv / (2 * p * q) * (sinc(d) - sinc(s))
        else:
            d = torch.where((p - q).abs() < 1e-10, torch.zeros_like(d), d)
            g = Lv * Lv * 0.5 / (p * q) * (sinc(d) - sinc(s) + fcos(d) - fcos(s))
        W[r:r + N] = wc * pre * (torch.where(both, g, single(torch.maximum(a0, a2))) - loss)
    return W


def _axis(case, invert):
    N = case["N"]
    v, eta = (np.asarray(x, dtype=np.longdouble) for x in _grid(case))
    pi = np.longdouble("3.141592653589793238462643383279502884")
    a, s, d, L0, L1 = (v, -1, eta[1] - eta[0], -v[0], -eta[0]) if invert else (eta, 1, v[1] - v[0], -eta[0], -v[0])
    j = np.arange(N)
    ph = s * L1 * a[:, None] - s * 2 * pi * ((j[:, None] * j) % N) / N + s * j[None, :] * L0 * d
    w = np.ones(N)
    w[0] = w[-1] = 0.5
    M = (np.cos(ph) * w).astype(np.float64) + 1j * (np.sin(ph) * w).astype(np.float64)
    return torch.from_numpy(M).cuda() * float(d) / math.sqrt(2 * math.pi)


def _transform(case, x, invert=False):
    """(N, N, N, B) complex, along the three axes."""
    M, N = _axis(case, invert), case["N"]
    for _ in range(3):  # one axis at a time, which then goes to the end of the three
        B = x.shape[3]
        x = (M @ x.reshape(N, -1)).reshape(N, N, N, B).permute(1, 2, 0, 3).contiguous()
    return x


def _sum(case, W, pairs):
    """sum over c of W[r][c] G[c] F[r - c] for each (G, F) of (N, N, N, B), added."""
    N, h = case["N"], case["N"] // 2
    B = pairs[0][0].shape[3]
    k = torch.arange(N, device="cuda")
    iz = (k[:, None] + h - k[None, :]) % N
    Gz = [G.permute(2, 0, 1, 3).contiguous() for G, _ in pairs]  # (cz, cx, cy, B)
    out = torch.empty(N, N, N, B, dtype=torch.complex128, device="cuda")
    Wv = W.view(N, N, N, N, N, N)
    step = max(1, min(B, (1 << 28) // N ** 4))
    for rx in range(N):
        Fx = [F[(rx + h - k) % N] for _, F in pairs]
        for ry in range(N):
            w = Wv[rx, ry].permute(0, 3, 1, 2).reshape(N, 1, N ** 3)
            Fy = [F[:, (ry + h - k) % N].permute(2, 0, 1, 3) for F in Fx]  # (z, cx, cy, B)
            for b in range(0, B, step):
                P = sum(G[None, ..., b:b + step] * F[iz][..., b:b + step] for G, F in zip(Gz, Fy))
                P = torch.view_as_real(P.reshape(N, N ** 3, -1)).reshape(N, N ** 3, -1)
                out[rx, ry, :, b:b + step] = torch.view_as_complex(torch.bmm(w, P).reshape(N, -1, 2))
    return out


def _split(case, f):
    """The Maxwellian of each cell's moments."""
    v = torch.from_numpy(_grid(case)[0]).cuda()
    w = _weights3(case["N"], v)
    rho = (f * w).sum((1, 2, 3))
    V = [v[:, None, None], v[None, :, None], v[None, None, :]]
    u = torch.stack([(f * w * V[d]).sum((1, 2, 3)) / rho for d in range(3)], 1)
    T = sum((f * w * (V[d] - u[:, d, None, None, None]) ** 2).sum((1, 2, 3)) for d in range(3)) / (3 * rho)
    return _maxwellian(v, rho, u, T)


def _q(case, W, f, g=None, split=False):
    """Q of (B, N, N, N) cells, not projected."""
    def hat(x):
        return _transform(case, x.permute(1, 2, 3, 0).to(torch.complex128).contiguous())
    if split:
        M = _split(case, f)
        A, M = hat(f - M), hat(M)
        pairs = [(A, A + M), (M, A)]
    else:
        F = hat(f)
        pairs = [(F if g is None else hat(g), F)]
    return _transform(case, _sum(case, W, pairs), True).real.permute(3, 0, 1, 2).contiguous()


def _project(case, Q):
    """Q[m][l] of the pair (l, m), (B, N, N, N) each, made conservative over all pairs of a cell together."""
    m = _masses(case) if len(Q) > 1 else [1.0]
    S = len(m)
    v = torch.from_numpy(_grid(case)[0]).cuda()
    w = _weights3(case["N"], v).expand(case["N"], case["N"], case["N"])
    V = [v[:, None, None], v[None, :, None], v[None, None, :]]
    C = []
    for l in range(S):
        rows = [w * m[l] if a == l else torch.zeros_like(w) for a in range(S)]
        rows += [w * m[l] * x for x in V] + [w * m[l] * 0.5 * (V[0] ** 2 + V[1] ** 2 + V[2] ** 2)]
        C.append(torch.stack(rows).reshape(S + 4, -1))
    A = sum(c @ c.T for c in C)
    mom = sum(Q[b][a].reshape(-1, C[0].shape[1]) @ C[a].T for a in range(S) for b in range(S))
    scale = torch.diagonal(A).rsqrt()
    x = torch.linalg.solve(A * scale[:, None] * scale[None, :], (mom * scale).T).T * scale
    return [[Q[b][a] - (x @ C[a]).reshape(Q[b][a].shape) / S for a in range(S)] for b in range(S)]


def _minmod(a, b, c):
    s = torch.sign(a)
    same = (s == torch.sign(b)) & (s == torch.sign(c))
    return torch.where(same, s * torch.minimum(torch.minimum(a.abs(), b.abs()), c.abs()), torch.zeros_like(a))


def _wall(case, v, f, TW, right, mass):
    """The reflected half of a diffuse wall at TW for the outgoing half of f."""
    N = case["N"]
    half = torch.arange(N, device="cuda") >= N // 2
    out = (half if right else ~half)[:, None, None]
    kb = 1.0 if _masses(case)[0] == 1.0 else 1.380658e-23
    flux = torch.where(out, f * _weights3(N, v) * v[:, None, None], torch.zeros_like(f)).sum()
    sig = (1 if right else -1) * math.sqrt(2 * math.pi * mass / (kb * TW)) * flux
    V2 = v[:, None, None] ** 2 + v[None, :, None] ** 2 + v[None, None, :] ** 2
    M = sig * (0.5 * mass / (math.pi * kb * TW)) ** 1.5 * torch.exp(-0.5 * mass / (kb * TW) * V2)
    return M, out


def _advect(case, f, mass):
    """One transport stage of (n, N, N, N) cells: first-order upwind, or the two minmod half steps and their mean."""
    x, dx = (torch.from_numpy(a).cuda() for a in _mesh(case))
    v = torch.from_numpy(_grid(case)[0]).cuda()
    up = (torch.arange(case["N"], device="cuda") >= case["N"] // 2)[:, None, None]  # from the left
    vx = v[:, None, None]
    n, dt, diffuse = case["ncell"], case["dt"], case["walls"] == "diffuse"
    if case["order"] == 1:
        lo, hi = f[:1], f[-1:]
        if diffuse:
            (a, _), (b, _) = _wall(case, v, f[0], 1.0, False, mass), _wall(case, v, f[-1], 2.0, True, mass)
            lo, hi = a[None], b[None]
        g = torch.cat([lo, f, hi])
        cfl = dt * vx / dx[1:-1, None, None, None]
        return torch.where(up, (1 - cfl) * f + cfl * g[:-2], (1 + cfl) * f - cfl * g[2:])

    def stage(f):
        g = torch.cat([2 * f[:1] - f[1:2], f, 2 * f[-1:] - f[-2:-1]])
        X, D = x[1:-1, None, None, None], dx[2:-2, None, None, None]
        s = _minmod((g[1:-1] - g[:-2]) / (X[1:-1] - X[:-2]), (g[2:] - g[1:-1]) / (X[2:] - X[1:-1]), (g[2:] - g[:-2]) / (X[2:] - X[:-2]))
        right, left = f + 0.5 * D * s, f - 0.5 * D * s  # a cell's states at its two faces
        # no-flux walls: the outgoing half leaves the cell, the incoming half has the other face's value
        fl, fr = torch.where(up, right[0], left[0]), torch.where(up, right[-1], left[-1])
        if diffuse:
            (a, out), (b, out2) = _wall(case, v, fl, 1.0, False, mass), _wall(case, v, fr, 2.0, True, mass)
            fl, fr = torch.where(out, fl, a), torch.where(out2, fr, b)
        cfl = 0.5 * dt * vx / D
        from_left = torch.cat([fl[None], right[:-1]])
        from_right = torch.cat([left[1:], fr[None]])
        return torch.where(up, f - cfl * (right - from_left), f - cfl * (from_right - left))
    return 0.5 * (f + stage(stage(f)))


class _BesselJ0:
    """J0 on [0, top] by Taylor series about the multiples of 1/16, whose derivatives are Bessel's integral by the
    trapezoid rule (torch's own is 4e-7 off near 5)."""

    def __init__(self, top):
        x = torch.arange(int(16 * top) + 2, dtype=torch.float64, device="cuda")[:, None] / 16
        t = (torch.arange(512, dtype=torch.float64, device="cuda") + 0.5) * (2 * math.pi / 512)
        s = torch.sin(t)[None]
        self.d = [(s ** m * torch.cos(x * s + 0.5 * math.pi * m)).mean(1) / math.factorial(m) for m in range(9)]

    def __call__(self, x):
        i = (16 * x).round()
        h, i = x - i / 16, i.long()
        y = self.d[8][i]
        for m in range(7, -1, -1):
            y = y * h + self.d[m][i]
        return y


def _landau(case, seed):
    Lv = case["Lv"] * (1 + 0.05 * float(torch.rand(1, generator=torch.Generator().manual_seed(int(seed)))))
    e = torch.from_numpy(_grid(case, Lv)[1]).cuda()
    E = torch.stack(torch.meshgrid(e, e, e, indexing="ij")).reshape(3, -1)
    x, w = (torch.from_numpy(a).cuda() for a in np.polynomial.legendre.leggauss(64))
    th, tw = 0.5 * math.pi * (1 + x), 0.5 * math.pi * w
    r, rw = 0.5 * Lv * (1 + x), 0.5 * Lv * w * (0.5 * Lv * (1 + x)) ** (case["lam"] + 2)
    th, tw = th[32:], 2 * tw[32:]  # even about pi/2
    n3 = E.shape[1]
    W = torch.zeros(n3, n3, dtype=torch.float64, device="cuda")
    z2 = E.square().sum(0)
    j0 = _BesselJ0(Lv * math.sqrt(3) * float(e.abs().max()) + 1)
    step = max(1, (1 << 24) // n3)
    for a in range(0, n3, step):
        zz = z2[a:a + step, None]
        dot = E[:, a:a + step].T @ E
        safe = torch.where(zz == 0, torch.ones_like(zz), zz)
        perp = torch.where(zz == 0, torch.zeros_like(dot), (z2[None] - dot * dot / safe).clamp(min=0)).sqrt()
        par, zl = torch.where(zz == 0, torch.zeros_like(dot), dot / safe.sqrt()), zz.sqrt()
        acc = torch.zeros_like(dot)
        for i in range(64):
            inner = torch.zeros_like(dot)
            for t in range(32):
                s, c = math.sin(float(th[t])), math.cos(float(th[t]))
                ph = r[i] * par * c
                inner += tw[t] * s * j0(r[i] * s * perp) * (-r[i] ** 2 * zz * s * s * torch.cos(ph) + 4 * r[i] * zl * c * torch.sin(ph))
            acc += rw[i] * inner
        W[a:a + step] = 2 * math.pi * acc
    return W


def exact(case, seed):
    kind, N = case["kind"], case["N"]
    if kind == "table":
        return _landau(case, seed).cpu().numpy() if case["table"] == "landau" else None
    f = _inputs(case, seed)
    n = case.get("ncell", 1)
    if kind in ("q", "abi"):
        W = _table(case)
        mp = case.get("op", "maxpreserve") == "maxpreserve"
        q = _project(case, [[_q(case, W, f[0], f[1] if len(f) > 1 else None, split=mp)]])[0][0]
        return q.reshape(n, -1) if kind == "q" else q.reshape(-1).cpu().numpy()
    m, f = _masses(case), f[0]
    S, h, Kn = len(m), case["dt"], case.get("Kn", 1.0)
    if kind == "run0d":
        f = f[None, :HEAD]
    W = [[_table(case, m[a], m[b]) for a in range(S)] for b in range(S)]

    def rate(y):
        Q = _project(case, [[_q(case, W[b][a], y[a], None if a == b else y[b], split=kind == "run0d") for a in range(S)] for b in range(S)])
        return torch.stack([sum(Q[b][a] for b in range(S)) for a in range(S)]) / Kn

    def advect(y):
        return torch.stack([_advect(case, y[l], m[l]) for l in range(S)]) if kind == "run1d" else y
    for _ in range(case["steps"]):
        y = advect(f)
        k = rate(y)
        if case["order"] == 1:
            f = y + h * k
            continue
        y1 = y + h * k
        f = advect(0.5 * (y + y1) + 0.5 * h * rate(y1))
    out = [f[l].reshape(f.shape[1], -1) for l in range(S)]
    return {"first": out[0], "rest": None} if kind == "run0d" and n > HEAD else out
