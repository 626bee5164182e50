"""Performance cases: the calls that programs built on this framework spend their time in.

Every case goes through the public Python mirror (``stratiflow_amd``).  Inputs are smooth in z, decay over the
horizontal modes and have a finite amplitude (0.05 of the background velocity), the state of a developed run.  A pass
starts from the same stored state each time, as FixedEvolve and the Newton and Arnoldi operators do (CopyToSolver,
start-up, steps, CopyFromSolver), so it can be repeated.

Outputs are the device buffers of the fields, looked at in place: a field in host memory goes through the reference's
full layout in double, which a program does once per snapshot and not once per call.  The pressure of FP32 steps is left
out: it is the running sum of projection residues over dt and carries their rounding (1e-3 of its norm in FP32); the
drivers' inner products leave it out as well.  FP64 cases return it.

``exact`` restates the discretisation in plain torch FP64: torch.fft for the horizontal transforms, a Thomas sweep for
the vertical systems.
"""
import ctypes
import math

import numpy as np
import torch

import stratiflow_amd as sf

LX = 2 * math.pi / 0.44
L3 = 10.0
RI, PR = 0.12, 1.0
AMPLITUDE = 0.05
SIZES_X = (24, 32, 48, 64, 96, 128, 192, 256, 384, 512)
SIZES_Y = (12, 16, 24, 32, 48, 64, 96, 128, 192)
BETA, ZETA = (1.0, 25.0 / 8.0, 9.0 / 4.0), (0.0, -17.0 / 8.0, -5.0 / 4.0)


# ---- the cases --------------------------------------------------------------
def listed():
    return [
        # one step of the smallest grid of the demos and Newton tests: launches and latency
        dict(name="evolve-2d-64-f32", kind="evolve", N1=64, N2=1, N3=64, prec=4, steps=1),
        # the Newton-Krylov configuration (256 x 256, FP64 stepping): part of one operator application
        dict(name="evolve-2d-256-f64", kind="evolve", N1=256, N2=1, N3=256, prec=8, steps=20),
        # a small 3D run with a column that does not fill whole wavefronts
        dict(name="evolve-3d-96x48x100-f32", kind="evolve", N1=96, N2=48, N3=100, prec=4, steps=4),
        # a 3D reference run in double precision
        dict(name="evolve-3d-192x96x192-f64", kind="evolve", N1=192, N2=96, N3=192, prec=8, steps=2),
        # the throughput workload of bench.py
        dict(name="evolve-3d-384x192x384-f32", kind="evolve", N1=384, N2=192, N3=384, prec=4, steps=4),
        # Arnoldi in 2D: linearised steps about a state
        dict(name="linear-2d-256-f64", kind="linear", N1=256, N2=1, N3=256, prec=8, steps=20),
        # stability of a 3D state (Stability3D): linearised 3D steps
        dict(name="linear-3d-192x96x192-f32", kind="linear", N1=192, N2=96, N3=192, prec=4, steps=2),
        # the backward pass of an adjoint loop over stored states
        dict(name="adjoint-3d-96x48x128-f32", kind="adjoint", N1=96, N2=48, N3=128, prec=4, steps=1),
        # an ensemble of uneven 2D runs advanced together
        dict(name="ensemble-16-f32", kind="ensemble", runs=16, pick=1, prec=4, steps=10),
        # nodal <-> modal transforms of one field: .fields files, plots, diagnostics
        dict(name="transform-384x192x384-f32", kind="transform", N1=384, N2=192, N3=384, prec=4),
        # a preconditioned GMRES step without its operator: preconditioner, Gram column, Gram-Schmidt
        dict(name="gmres-256-f64", kind="gmres", N1=256, N2=1, N3=256, prec=8, vectors=30),
        # the learned preconditioner applied to one Krylov vector
        dict(name="net-256-f64", kind="net", N1=256, N2=1, N3=256, prec=8, layers=4),
    ]


def draw(rng):
    most = 0.6 * max(work(c)["bytes"] for c in listed())
    while True:
        kind = rng.choice(("evolve", "evolve", "evolve", "linear", "linear", "adjoint", "ensemble", "transform",
                           "gmres", "net"))
        prec = rng.choice((4, 8))
        if kind == "ensemble":
            return dict(kind=kind, runs=rng.randint(3, 20), pick=rng.randrange(1, 1 << 20), prec=prec,
                        steps=rng.randint(4, 12))
        three = kind not in ("gmres", "net") and rng.random() < 0.6
        c = dict(kind=kind, N1=rng.choice(SIZES_X), N2=rng.choice(SIZES_Y) if three else 1,
                 N3=4 * int(round(math.exp(rng.uniform(math.log(8), math.log(128))))), prec=prec)
        if c["N1"] > 384 and prec == 8:
            continue
        if kind in ("evolve", "linear", "adjoint"):
            c["steps"] = rng.randint(1, 3 if three or kind == "adjoint" else 20)
        if kind == "gmres":
            c["vectors"] = rng.randint(4, 40)
            c["N3"] = min(c["N3"], 256)  # the advected preconditioner's largest FP64 column
        if kind == "net":
            c["layers"] = rng.randint(3, 5)
        if work(c)["bytes"] <= most:
            return c


# ---- geometry and inputs ----------------------------------------------------
def _three(c):
    return c["N2"] > 1


def _active(c):
    """Active x and y modes of the 2/3 rule."""
    return c["N1"] // 3, (2 * (c["N2"] // 3) - 1 if _three(c) else 1)


def _rows(c):
    """Spanwise index of every active y mode."""
    h = c["N2"] // 3
    return list(range(h)) + list(range(c["N2"] - h + 1, c["N2"])) if _three(c) else [0]


def _names(c):
    return ("u1", "u2", "u3", "b") if _three(c) else ("u1", "u3", "b")


def _dt(c):
    return 0.005 if _three(c) else 0.01


def _points(N):
    """The stretched grid: z, zf and their spacings."""
    x = np.linspace(-1.0, 1.0, N - 1)
    z = np.zeros(N)
    z[1:] = L3 * (2.0 * x**7 + x) / 3.0
    z *= -L3 / (0.5 * (z[1] + z[2]))
    z[0] = 2.0 * z[1] - z[2]
    zf = np.zeros(N)
    zf[1:-1] = 0.5 * (z[1:-1] + z[2:])
    zf[0], zf[-1] = 2.0 * zf[1] - zf[2], 2.0 * zf[-2] - zf[-3]
    dy, dyf = np.zeros(N), np.zeros(N)
    dy[1:] = zf[1:] - zf[:-1]
    dy[0] = dy[1]
    dyf[1:-1] = z[2:] - z[1:-1]
    dyf[-1], dyf[0] = dyf[-2], dyf[1]
    return z, zf, dy, dyf


def _background(zf):
    """tanh(z) with the ghost points of a Neumann profile."""
    u = np.tanh(zf)
    u[1] = u[2]
    u[0] = u[1]
    u[-2] = u[-3]
    u[-1] = u[-2]
    return u


def _field(c, rng, dirichlet=False):
    """A real field's active modes [y mode][z][x mode] in FP64 on the GPU, largest nodal value AMPLITUDE."""
    a1, a2 = _active(c)
    z, zf, _, _ = _points(c["N3"])
    x = (z if dirichlet else zf) / 2.0
    prof = np.stack([np.exp(-x * x) * h for h in (np.ones_like(x), 2 * x, 4 * x * x - 2, 8 * x**3 - 12 * x)])
    k1 = np.arange(a1) / max(a1, 1)
    k2 = np.abs(np.array([j if j < c["N2"] // 2 + 1 else j - c["N2"] for j in _rows(c)])) / max(c["N2"] / 3.0, 1.0)
    fall = np.exp(-4.0 * np.hypot(k1[None, :], k2[:, None]))
    co = (rng.uniform(-1, 1, (a2, a1, 4)) + 1j * rng.uniform(-1, 1, (a2, a1, 4))) * fall[:, :, None]
    dev = torch.device("cuda")
    f = torch.einsum("ajh,hz->azj", torch.tensor(co, device=dev), torch.tensor(prof, device=dev).to(torch.complex128))
    for a in range(1, (a2 + 1) // 2):
        f[a2 - a, :, 0] = f[a, :, 0].conj()
    f[0, :, 0] = f[0, :, 0].real.to(f.dtype)
    return f * (AMPLITUDE / _Reference(c).nodal(f).abs().max())


def _inputs(c, seed, sets=1):
    rng = np.random.default_rng(seed)
    return [{n: _field(c, rng, n == "u3") for n in _names(c)} for _ in range(sets)]


def _reynolds(seed):
    return float(np.random.default_rng([seed, 7]).uniform(1000.0, 3000.0))


def _ensemble(c):
    """Grids and steps of an uneven ensemble."""
    rng = np.random.default_rng(c["pick"])
    return [dict(kind="evolve", N1=int(rng.choice((64, 96, 128, 192, 256))), N2=1,
                 N3=int(rng.choice((96, 128, 192, 256, 384))), prec=c["prec"], steps=c["steps"])
            for _ in range(c["runs"])]


# ---- the framework's side ---------------------------------------------------
class _SfField(ctypes.Structure):  # struct sf_field
    _fields_ = [("ctx", ctypes.c_void_p), ("kind", ctypes.c_int), ("bc", ctypes.c_int), ("n", ctypes.c_size_t),
                ("d", ctypes.c_void_p), ("owned", ctypes.c_bool)]


class _Buffer:
    """Device memory of a field, which it keeps alive (and the field its solver) for as long as a tensor looks at it."""

    def __init__(self, field, ptr, shape, typestr):
        self.field = field
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _view(c, field):
    """A field's device values as a tensor: modal [y mode][z][x mode][re, im], nodal [y][x][z]."""
    raw = _SfField.from_address(field.h.value if hasattr(field.h, "value") else field.h)
    a1, a2 = _active(c)
    shape = (a2, c["N3"], a1, 2) if field.kind == sf.MODAL else (c["N2"], c["N1"], c["N3"])
    if raw.n != math.prod(shape) or raw.kind != field.kind or raw.bc != field.bc:
        raise RuntimeError("the layout of sf_field has changed")
    view = torch.as_tensor(_Buffer(field, raw.d, shape, "<f%d" % c["prec"]), device="cuda")
    if view.data_ptr() != raw.d:
        raise RuntimeError("the view of a field is a copy")
    return view


def _solver(c, seed):
    s = sf.IMEXRK(c["N1"], c["N2"], c["N3"], sf.THREE_D if _three(c) else sf.TWO_D, LX, LX / 2 if _three(c) else 1.0,
                  L3, _reynolds(seed), RI, PR, precision=c["prec"])
    s.SetBackground(_background(s.vertical_points()[1]))
    s.deltaT = _dt(c)
    return s


def _new(s, name):
    return s.field(sf.MODAL, sf.DIRICHLET if name == "u3" else sf.NEUMANN)


def _upload(c, s, values):
    """A StateVector's fields; p starts at zero."""
    a1, _ = _active(c)
    out = {}
    for name, f in values.items():
        full = torch.zeros((c["N2"], c["N1"] // 2 + 1, c["N3"]), dtype=torch.complex128, device="cuda")
        full[_rows(c), :a1] = f.permute(0, 2, 1)
        out[name] = _new(s, name)
        out[name].upload(full.cpu().numpy())
    return out


def _state(s, c):
    """Empty fields for a result, and what of them a pass returns."""
    out = {n: _new(s, n) for n in _names(c) + ("p",)}
    return out, {n: _view(c, f) for n, f in out.items() if n != "p" or c["prec"] == 8}


def _copy_in(s, x):
    s.CopyToSolver(x["u1"], x.get("u2"), x["u3"], x["b"], x["p"])


def _copy_out(s, x):
    s.CopyFromSolver(x["u1"], x.get("u2"), x["u3"], x["b"], x["p"])


def prepare(case, seed):
    c = case
    if c["kind"] == "ensemble":
        parts = _ensemble(c)
        runs = [_solver(p, seed + i) for i, p in enumerate(parts)]
        start, out, views = [], [], []
        for i, (p, s) in enumerate(zip(parts, runs)):
            x = _upload(p, s, _inputs(p, seed + i)[0])
            x["p"] = _new(s, "p")
            start.append(x)
            o, v = _state(s, p)
            out.append(o)
            views.append({n: t for n, t in v.items() if n != "p"})
        return dict(case=c, runs=runs, start=start, out=out, views=views, batch=sf.Batch(runs))
    s = _solver(c, seed)
    st = dict(case=c, solver=s)
    if c["kind"] == "transform":
        st["modal"] = _upload(c, s, {"u1": _inputs(c, seed)[0]["u1"]})["u1"]
        st["nodal"], st["back"] = s.field(sf.NODAL, sf.NEUMANN), _new(s, "u1")
        st["views"] = {"nodal": _view(c, st["nodal"]), "back": _view(c, st["back"])}
        return st
    if c["kind"] == "gmres":
        st["basis"] = [_upload(c, s, x) for x in _inputs(c, seed, c["vectors"])]
        for x in st["basis"]:
            norm = math.sqrt(_dot(s, x, x))
            for n in x:
                x[n] *= 1.0 / norm
        st["w"] = _upload(c, s, _inputs(c, seed + 1)[0])
        st["z"], st["q"] = {n: _new(s, n) for n in _names(c)}, {n: _new(s, n) for n in _names(c)}
        st["views"] = {k: {n: _view(c, f) for n, f in st[k].items()} for k in ("z", "q")}
        return st
    st["x"] = _upload(c, s, _inputs(c, seed)[0])
    if c["kind"] == "net":
        st["net"] = sf.Net(s, 64, c["layers"], seed=3)
        st["net"].set_dilations([1 << min(k, 3) for k in range(c["layers"])])
        st["net"].set_params(_params(st["net"].channels, seed))
        st["out"] = {n: _new(s, n) for n in _names(c)}
        st["views"] = {n: _view(c, f) for n, f in st["out"].items()}
        return st
    st["x"]["p"] = _new(s, "p")
    st["out"], st["views"] = _state(s, c)
    if c["kind"] == "linear":
        st["about"] = _upload(c, s, _inputs(c, seed + 1)[0])
    if c["kind"] == "adjoint":
        st["direct"] = [_upload(c, s, x) for x in _inputs(c, seed + 1, c["steps"] + 1)]
    return st


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "ensemble":
        for s, x in zip(state["runs"], state["start"]):
            _copy_in(s, x)
        state["batch"].step(c["steps"])
        for s, o in zip(state["runs"], state["out"]):
            _copy_out(s, o)
        return state["views"]
    s = state["solver"]
    if kind == "transform":
        state["modal"].ToNodal(state["nodal"])
        state["nodal"].ToModal(state["back"])
        return state["views"]
    if kind == "gmres":
        return _gmres_step(state)
    if kind == "net":
        order = ("u1", "u2", "u3", "b")
        state["net"].apply([state["x"].get(n) for n in order], [state["out"].get(n) for n in order])
        return state["views"]
    # FixedEvolve, LinearEvolve and AdjointEvolve at a fixed dt
    _copy_in(s, state["x"])
    if kind == "linear":
        a = state["about"]
        s.SetLinearBackground(a["u1"], a.get("u2"), a["u3"], a["b"])
    if kind == "adjoint":
        s.PrepareRunAdjoint()
        d = [[x["u1"], x.get("u2"), x["u3"], x["b"]] for x in state["direct"]]
        for k in range(c["steps"]):
            s.TimeStepAdjoint(d[c["steps"] - 1 - k], d[c["steps"] - k])
    else:
        s.FilterAll()
        s.PopulateNodalVariables()
        s.RemoveDivergence(0.0)
        if kind == "linear":
            s.TimeStepLinear(c["steps"])
        else:
            s.TimeStep(c["steps"])
    _copy_out(s, state["out"])
    return state["views"]


def _dot(s, a, b):
    """StateVector::Dot: <u, u> + Ri <b, b>."""
    return sum((RI if n == "b" else 1.0) * s.InnerProd(a[n], b[n]) for n in a)


def _gmres_step(state):
    """Flexible GMRES without its operator: z = M^-1 q, its Gram column, and the Gram-Schmidt of w."""
    s, basis, z, q = state["solver"], state["basis"], state["z"], state["q"]
    nu, T = 1.0 / s.flow["Re"], 2.0
    for n, f in basis[0].items():
        f.diffusion_precondition(z[n], T * nu / (PR if n == "b" else 1.0), 0.3, 1e9, T)
        z[n].EnforceBCs()
    gram = [_dot(s, x, z) for x in basis]
    for n, f in state["w"].items():
        q[n].assign(f)
    h = []
    for x in basis:
        h.append(_dot(s, x, q))
        for n in q:
            q[n].MulAdd(-h[-1], x[n])
    h.append(math.sqrt(_dot(s, q, q)))
    for n in q:
        q[n] *= 1.0 / h[-1]
        q[n].EnforceBCs()
    return dict(state["views"], gram=np.array(gram), h=np.array(h))


def _params(channels, seed):
    """Parameters of a trained size: W[5][out][in] and bias[out] per layer, on the padded channels."""
    rng = np.random.default_rng([seed, 11])
    p = []
    for l, (ci, co) in enumerate(zip(channels[:-1], channels[1:])):
        rin = 8 if l == 0 else ci
        rout = 6 if l == len(channels) - 2 else co
        w = np.zeros((5, co, ci))
        w[:, :rout, :rin] = rng.normal(0.0, math.sqrt(2.0 / (5 * rin)), (5, rout, rin))
        b = np.zeros(co)
        b[:rout] = rng.normal(0.0, 0.05, rout)
        p += [w.ravel(), b]
    return np.concatenate(p).astype(np.float32)


# ---- what a pass cannot do without ------------------------------------------
def work(case):
    """Bytes: every stage of a step reads and writes the state once (the vertical solves need all z of a mode, the
    products all modes of a z) and the explicit terms pass from stage to stage.  Flops: the FFTs, products and solves
    of the scheme."""
    c = case
    if c["kind"] == "ensemble":
        parts = [work(p) for p in _ensemble(c)]
        return {"bytes": sum(p["bytes"] for p in parts), "flops": sum(p["flops"] for p in parts)}
    a1, a2 = _active(c)
    modal = a1 * a2 * c["N3"]
    nodal = c["N1"] * c["N2"] * c["N3"]
    ba = modal * 2 * c["prec"]
    nf = len(_names(c))
    fft = 2.5 * nodal * math.log2(c["N1"] * c["N2"])
    if c["kind"] == "transform":
        return {"bytes": 2 * ba + 2 * nodal * c["prec"], "flops": 2 * fft}
    if c["kind"] == "gmres":
        k = c["vectors"]
        return {"bytes": (2 + 3 * k) * nf * ba, "flops": nf * modal * (60.0 + 12.0 * k)}
    if c["kind"] == "net":
        ch = [32] + [64] * (c["layers"] - 1) + [32]
        return {"bytes": 2 * nf * ba, "flops": 10.0 * modal * sum(a * b for a, b in zip(ch[:-1], ch[1:]))}
    stages = 3 * c["steps"]
    products = {"evolve": 11 if _three(c) else 6, "linear": 11 if _three(c) else 6, "adjoint": 12 if _three(c) else 6}
    forward = products[c["kind"]]
    inverse = {"evolve": nf, "linear": 2 * nf, "adjoint": nf * (4 if _three(c) else 3)}[c["kind"]]
    extra = {"evolve": 0, "linear": nf, "adjoint": 2 * nf}[c["kind"]]
    per = (2 * (nf + 1) + extra + 4.0 / 3.0 * nf) * ba
    return {"bytes": stages * per, "flops": stages * ((inverse + forward) * fft + 60.0 * nodal + nf * 250.0 * modal)}


# ---- plain FP64 -------------------------------------------------------------
def _prev(f):
    return torch.cat((torch.zeros_like(f[:, :1]), f[:, :-1]), 1)


def _next(f):
    return torch.cat((f[:, 1:], torch.zeros_like(f[:, :1])), 1)


class _Reference:
    """The scheme in FP64 on [row][z][x mode or x point] tensors."""

    def __init__(self, c, Re=1.0):
        self.c, self.Re, self.three = c, Re, _three(c)
        self.N1, self.N2, self.N3 = c["N1"], c["N2"], c["N3"]
        self.A1, self.A2 = _active(c)
        dev = torch.device("cuda")

        def col(a):
            return torch.tensor(np.asarray(a), device=dev, dtype=torch.float64).view(1, -1, 1)

        z, zf, dy, dyf = _points(self.N3)
        N = self.N3
        j = np.arange(N)
        pad = np.append(dy[1:], 1.0)
        back = np.append(1.0, dyf[:-1])
        inn, ind = (j >= 1) & (j <= N - 2), (j >= 2) & (j <= N - 2)
        self.nlo, self.nup = col(np.where(inn, 1 / dy / dyf, 0)), col(np.where(inn, 1 / pad / dyf, 0))
        self.dlo, self.dup = col(np.where(ind, 1 / back / dy, 0)), col(np.where(ind, 1 / dyf / dy, 0))
        self.dznd, self.dzdn = col(np.where(j >= 2, 1 / dy, 0)), col(np.where(j >= 1, 1 / dyf, 0))
        on = j >= 1
        self.iflo, self.ifdi = col(np.where(on, dyf / (2 * dy), 0)), col(np.where(on, back / (2 * dy), 0))
        self.itlo, self.itdi = self.ifdi, self.iflo
        self.wn = col(np.where(inn, np.append(z[1:], 0) - z, 0))
        self.wd = col(np.where(ind, zf - np.append(0, zf[:-1]), 0))
        self.ubar = col(_background(zf))
        self.half = col(np.where(on, 0.5, 0.0))
        rows = np.array(_rows(c))
        k2 = np.where(rows < self.N2 / 2, rows, rows - self.N2)
        L2 = LX / 2 if self.three else 1.0
        self.kx = torch.tensor(2 * math.pi * np.arange(self.A1) / LX, device=dev).view(1, 1, -1)
        self.ky = torch.tensor(2 * math.pi * k2 / L2, device=dev, dtype=torch.float64).view(-1, 1, 1)
        self.k2 = self.kx**2 + self.ky**2
        self.rows = torch.tensor(rows, device=dev)
        self.j = torch.arange(N, device=dev).view(1, -1, 1)

    def nodal(self, f):
        full = torch.zeros((self.N2, self.N3, self.N1 // 2 + 1), dtype=torch.complex128, device=f.device)
        full[self.rows, :, :self.A1] = f
        return torch.fft.irfft(torch.fft.ifft(full, dim=0) * self.N2, n=self.N1, dim=2) * self.N1

    def modal(self, g):
        return (torch.fft.fft(torch.fft.rfft(g, dim=2), dim=0) / (self.N1 * self.N2))[self.rows, :, :self.A1]

    def matrix(self, kind, coef):
        """Rows of kind n(eumann), d(irichlet) or p(oisson): I - coef (Dzz - k^2), or Dzz - k^2."""
        N, j = self.N3, self.j
        lo, up = (self.dlo, self.dup) if kind == "d" else (self.nlo, self.nup)
        one = torch.ones_like(self.k2 + lo)
        di = -lo - up - self.k2
        a, b, c = (lo * one, di, up * one) if kind == "p" else (-coef * lo * one, 1 - coef * di, -coef * up * one)
        ident = (j <= 2) | (j >= N - 2) if kind == "d" else (j == 0) | (j == N - 1)
        a, b, c = (torch.where(ident, v * one, m) for v, m in ((0.0, a), (1.0, b), (0.0, c)))
        if kind != "d":
            a, b, c = (torch.where(j == 1, v * one, m) for v, m in ((0.0, a), (1.0, b), (-1.0, c)))
            a, b, c = (torch.where(j == N - 2, v * one, m) for v, m in ((1.0, a), (-1.0, b), (0.0, c)))
        if kind == "p":  # the mean pressure is pinned
            b[0, 1, 0], c[0, 1, 0] = 1.0, 0.0
        return a, b, c

    def solve(self, m, d):
        a, b, c = m
        N = self.N3
        cc, x = [None] * N, [None] * N
        cc[0], x[0] = c[:, 0] / b[:, 0], d[:, 0] / b[:, 0]
        for k in range(1, N):
            r = 1.0 / (b[:, k] - a[:, k] * cc[k - 1])
            cc[k], x[k] = c[:, k] * r, (d[:, k] - a[:, k] * x[k - 1]) * r
        for k in range(N - 2, -1, -1):
            x[k] = x[k] - cc[k] * x[k + 1]
        return torch.stack(x, 1)

    def ends(self, f, dirichlet):
        j = self.j
        cut = (j <= 1) | (j >= self.N3 - 2) | ((j == 2) if dirichlet else (j < 0))
        return torch.where(cut, torch.zeros_like(f), f)

    def enforce(self, x):
        out = {}
        for n, f in x.items():
            if n == "u3":
                f = self.ends(f, True)
            elif n != "p":
                f = torch.cat((f[:, 1:2], f[:, 1:-1], f[:, -2:-1]), 1)
            out[n] = f
        return out

    def advection(self, x, about=None):
        """BuildRHS's products of x, or their derivative about a state in the direction x."""
        U = {n: self.nodal(f) for n, f in x.items()}
        W = {n: self.nodal(f) for n, f in about.items()} if about is not None else U
        if about is None:
            U = W = dict(U, u1=U["u1"] + self.ubar)
        else:
            W = dict(W, u1=W["u1"] + self.ubar)

        def both(f):  # bilinear f: f(U, U), or its derivative
            return f(U, U) if about is None else f(U, W) + f(W, U)

        def flux(n):  # ddz(Ibar(n) u3)
            def g(A, B):
                v = (self.half * _prev(A[n]) + self.half * A[n]) * B["u3"]
                hi = (0.5 * A[n] + 0.5 * _next(A[n])) * _next(B["u3"])
                return (hi - v) * self.dzdn
            return both(g)

        def q4(A, B):
            i, k = 0.5 * A["u3"] + 0.5 * _next(A["u3"]), 0.5 * B["u3"] + 0.5 * _next(B["u3"])
            return (i * k - _prev(i) * _prev(k)) * self.dznd

        def tilde(n):
            return both(lambda A, B: (self.itlo * _prev(A[n]) + self.itdi * A[n]) * B["u3"])

        def prod(n, m):
            if about is not None and n == m:
                return 2 * U[n] * W[n]
            return U[n] * W[m] if about is None else U[n] * W[m] + W[n] * U[m]

        F, ix, iy = self.modal, 1j * self.kx, 1j * self.ky
        r = {"u1": -(ix * F(prod("u1", "u1")) + F(flux("u1"))), "u3": -(ix * F(tilde("u1")) + F(both(q4))),
             "b": -(ix * F(prod("u1", "b")) + F(flux("b")))}
        if self.three:
            p = F(prod("u1", "u2"))
            r["u2"] = -(F(flux("u2")) + ix * p + iy * F(prod("u2", "u2")))
            r["u1"] -= iy * p
            r["u3"] -= iy * F(tilde("u2"))
            r["b"] -= iy * F(prod("u2", "b"))
        return r

    def buoyancy(self, x, r):
        v = RI * (self.iflo * _prev(x["b"]) + self.ifdi * x["b"])
        v[0, :, 0] = 0
        return dict(r, u3=r["u3"] + v, b=r["b"] - (0.5 * x["u3"] + 0.5 * _next(x["u3"])))

    def project(self, x, mult):
        div = 1j * self.kx * x["u1"] + self.dzdn * (_next(x["u3"]) - x["u3"])
        if self.three:
            div = div + 1j * self.ky * x["u2"]
        q = self.solve(self.matrix("p", 0.0), self.ends(div, False))
        y = dict(x, u1=x["u1"] - 1j * self.kx * q, u3=x["u3"] - self.dznd * (q - _prev(q)), p=x["p"] + mult * q)
        if self.three:
            y["u2"] = x["u2"] - 1j * self.ky * q
        return y

    def stage(self, k, x, r, old, dt):
        h = dt * (8.0, 2.0, 5.0)[k] / 15.0
        p = x["p"]
        grad = {"u1": 1j * self.kx * p, "u2": 1j * self.ky * p, "u3": self.dznd * (p - _prev(p))}
        y = dict(x)
        for n in r:
            d = n == "u3"
            c = 0.5 * h / self.Re / (PR if n == "b" else 1.0)
            lo, up = (self.dlo, self.dup) if d else (self.nlo, self.nup)
            u = x[n]
            lap = lo * _prev(u) - (lo + up) * u + up * _next(u) - self.k2 * u
            R = u + h * BETA[k] * r[n] + c * lap
            if old is not None:
                R = R + h * ZETA[k] * old[n]
            if n in grad:
                R = R - h * grad[n]
            y[n] = self.solve(self.matrix("d" if d else "n", c), self.ends(R, d))
        return self.project(y, 1.0 / h)

    def evolve(self, x, steps, dt, about=None, start_up=True):
        x = dict(x, p=torch.zeros_like(x["b"]))
        seen = {n: x[n] for n in _names(self.c)}  # the nodal fields precede the first projection
        if start_up:
            x = self.project(x, 0.0)
        for _ in range(steps):
            old = None
            for k in range(3):
                r = self.buoyancy(x, self.advection(seen, about))
                x = self.stage(k, x, r, old, dt)
                old, seen = r, {n: x[n] for n in _names(self.c)}
        return self.enforce(x)

    def adjoint_terms(self, x, t):
        U = {n: self.nodal(x[n]) for n in _names(self.c)}
        T = {n: self.nodal(f) for n, f in t.items()}
        DX = {n: self.nodal(1j * self.kx * f) for n, f in t.items()}
        DY = {n: self.nodal(1j * self.ky * f) for n, f in t.items()}

        def ibar(f):
            return self.half * _prev(f) + self.half * f

        def idir(f):
            return 0.5 * f + 0.5 * _next(f)

        def ifull(f):
            return self.iflo * _prev(f) + self.ifdi * f

        def itil(f):
            return self.itlo * _prev(f) + self.itdi * f

        def nd(f):
            return self.dznd * (f - _prev(f))

        def dn(f):
            return self.dzdn * (_next(f) - f)

        def mean(f):
            return f[0, :, 0].real.view(1, -1, 1)

        def forced(D):
            v = D["u1"] * U["u1"] + idir(D["u3"] * U["u3"]) + D["b"] * U["b"]
            return -(v + D["u2"] * U["u2"]) if self.three else -v

        w = nd(T["u1"]) * ifull(U["u1"])
        if self.three:
            w = w + nd(T["u2"]) * ifull(U["u2"])
        f3 = 0.5 * (T["b"] - mean(t["b"])) - w - ifull(dn(T["u3"])) * U["u3"] - nd(T["b"]) * ifull(U["b"])
        fb = 0.5 * (T["u3"] - mean(t["u3"])) + RI * idir(U["u3"])
        F, ix, iy = self.modal, 1j * self.kx, 1j * self.ky
        r = {"u1": ix * F(U["u1"] * T["u1"]) + F(dn(ibar(U["u1"]) * T["u3"]) + forced(DX)),
             "u3": ix * F(itil(T["u1"]) * U["u3"]) + F(nd(idir(U["u3"]) * idir(T["u3"])) + f3),
             "b": ix * F(U["b"] * T["u1"]) + F(dn(ibar(U["b"]) * T["u3"]) + fb)}
        if self.three:
            r["u1"] += iy * F(U["u1"] * T["u2"])
            r["u2"] = (iy * F(U["u2"] * T["u2"]) + ix * F(U["u2"] * T["u1"])
                       + F(dn(ibar(U["u2"]) * T["u3"]) + forced(DY)))
            r["u3"] += iy * F(itil(T["u2"]) * U["u3"])
            r["b"] += iy * F(U["b"] * T["u2"])
        return r

    def adjoint(self, x, direct, dt):
        x = self.project(dict(x, p=torch.zeros_like(x["b"])), 0.0)
        x["p"] = torch.zeros_like(x["p"])
        steps = len(direct) - 1
        for s in range(steps):
            below, above = direct[steps - 1 - s], direct[steps - s]
            old, frac = None, 0.0
            for k in range(3):
                t = {n: (1 - frac) * above[n] + frac * below[n] for n in above}
                t["u1"][0, :, 0] += self.ubar.view(-1)
                r = self.adjoint_terms(x, t)
                x = self.stage(k, x, r, old, dt)
                old = r
                frac += (8.0, 2.0, 5.0)[k] / 15.0
        return self.enforce(x)

    def dot(self, a, b):
        total = 0.0
        for n in a:
            v = (a[n].real * b[n].real + a[n].imag * b[n].imag) * (self.wd if n == "u3" else self.wn)
            total += (RI if n == "b" else 1.0) * float(2 * v.sum() - v[0, :, 0].sum())
        return total

    def precondition(self, n, f, T, delta):
        """(T L - delta)^-1 f - f/2 with L = nu (Dzz - k^2) - i kx U."""
        d = n == "u3"
        a, b, c = self.matrix("d" if d else "n", T / self.Re / (PR if n == "b" else 1.0) / delta)
        j = self.j
        plain = (j <= 2) | (j >= self.N3 - 2) if d else (j <= 1) | (j >= self.N3 - 2)
        b = torch.where(plain, b.to(f.dtype), b + 1j * T * self.kx * self.ubar / delta)
        return self.solve((a, b, c), self.ends(f, d) * (-1.0 / delta)) - 0.5 * f


def _pairs(x, c):
    return {n: torch.view_as_real(f.contiguous()) for n, f in x.items() if n != "p" or c["prec"] == 8}


def exact(case, seed):
    c = case
    if c["kind"] == "ensemble":
        out = []
        for i, p in enumerate(_ensemble(c)):
            x = _Reference(p, _reynolds(seed + i)).evolve(_inputs(p, seed + i)[0], p["steps"], _dt(p), start_up=False)
            out.append({n: f for n, f in _pairs(x, p).items() if n != "p"})
        return out
    ref = _Reference(c, _reynolds(seed))
    if c["kind"] == "transform":
        f = _inputs(c, seed)[0]["u1"]
        return {"nodal": ref.nodal(f).permute(0, 2, 1).contiguous(), "back": torch.view_as_real(f)}
    if c["kind"] == "gmres":
        basis = _inputs(c, seed, c["vectors"])
        basis = [{n: f / math.sqrt(ref.dot(x, x)) for n, f in x.items()} for x in basis]
        z = ref.enforce({n: ref.precondition(n, f, 2.0, 0.3) for n, f in basis[0].items()})
        q, h = dict(_inputs(c, seed + 1)[0]), []
        for x in basis:
            h.append(ref.dot(x, q))
            q = {n: q[n] - h[-1] * x[n] for n in q}
        h.append(math.sqrt(ref.dot(q, q)))
        q = ref.enforce({n: f / h[-1] for n, f in q.items()})
        return dict(z=_pairs(z, c), q=_pairs(q, c), gram=np.array([ref.dot(x, z) for x in basis]), h=np.array(h))
    x = _inputs(c, seed)[0]
    if c["kind"] == "net":
        return _net(c, ref, x, seed)
    dt = _dt(c)
    if c["kind"] == "linear":
        x = ref.evolve(x, c["steps"], dt, about=_inputs(c, seed + 1)[0])
    elif c["kind"] == "adjoint":
        x = ref.adjoint(x, _inputs(c, seed + 1, c["steps"] + 1), dt)
    else:
        x = ref.evolve(x, c["steps"], dt)
    return _pairs(x, c)


def _net(c, ref, x, seed):
    """in + s net(in / s) with dilated convolutions over z, one profile per mode."""
    a1, a2 = _active(c)
    f = torch.stack([v for n in _names(c) for v in (x[n].real, x[n].imag)], 1)  # [y mode][channel][z][x mode]
    s = float((f * f).sum() / (f.numel() / 2)) ** 0.5
    kx = (ref.kx / ref.kx.max()).expand(a2, c["N3"], a1).unsqueeze(1)
    y = torch.cat((f / s, kx, torch.zeros_like(kx)), 1).permute(0, 3, 1, 2).reshape(a1 * a2, -1, c["N3"])
    ch = [32] + [64] * (c["layers"] - 1) + [32]
    y = torch.nn.functional.pad(y, (0, 0, 0, ch[0] - y.shape[1]))
    p = torch.tensor(_params(ch, seed).astype(np.float64), device="cuda")
    for l, (ci, co) in enumerate(zip(ch[:-1], ch[1:])):
        w, b, p = p[:5 * co * ci].view(5, co, ci).permute(1, 2, 0), p[5 * co * ci:][:co], p[5 * co * ci + co:]
        dil = 1 << min(l, 3)
        wide = torch.nn.functional.pad(y, (2 * dil, 2 * dil))
        y = sum(torch.matmul(w[:, :, t].contiguous(), wide[:, :, t * dil:t * dil + c["N3"]].contiguous())
                for t in range(5)) + b.view(1, -1, 1)
        if l < len(ch) - 2:
            y = y.relu()
    y = y[:, :f.shape[1]].reshape(a2, a1, f.shape[1], c["N3"]).permute(0, 2, 3, 1)
    v = f + s * y
    return {n: torch.stack((v[:, 2 * i], v[:, 2 * i + 1]), -1) for i, n in enumerate(_names(c))}
