"""The work that users of this package have it do, as cases of plain values.

Every kind goes through the public Python entry points: pressure Poisson solves (`mg.Multigrid`),
whole time steps (`ts.Hydro`), the field operators and the viscous Jacobi solve on caller arrays
(`field.FieldGrid`), a solve of a sequence with the online least-squares predictor
(`guess.GuessNet` with `mg.Multigrid`) and one training step of the guess network.

Grids have 2^k + 1 nodes per direction.  Domain lengths are in proportion to the node counts, as
in the 257 x 257 x 129 convection run on (2, 2, 1), so that spacings are alike in every direction.
"""
import ctypes
import math

import torch

from saras_amd import _lib, field, guess, mg, ts, workloads

DEV = "cuda"
F64 = torch.float64


def listed():
    return [
        # the small validation solves: a user's first problem, many launches of next to no work
        dict(name="poisson_fp64_33", kind="poisson", xi=5, yi=5, zi=5, domain="PPN", mesh="UUD", precision="fp64",
             pads=0, direct=0),
        # a box with walls and stretching all round, another length in every direction
        dict(name="poisson_mixed_129x65x33", kind="poisson", xi=7, yi=6, zi=5, domain="NNN", mesh="DDD",
             precision="mixed", pads=1, direct=1),
        # an ordinary grid with the accelerated mixed precision solver
        dict(name="poisson_gcr_65", kind="poisson", xi=6, yi=6, zi=6, domain="PPN", mesh="UUD", precision="gcr",
             pads=1, direct=1),
        # the stretched-grid 257^3 Poisson problem of the benchmark in plain double precision
        dict(name="poisson_fp64_257", kind="poisson", xi=8, yi=8, zi=8, domain="PPN", mesh="UUD", precision="fp64",
             pads=0, direct=0),
        # the same problem with the fastest solver: FP32 cycles inside GCR(1), mirror pads, exact coarsest level
        dict(name="poisson_gcr_257", kind="poisson", xi=8, yi=8, zi=8, domain="PPN", mesh="UUD", precision="gcr",
             pads=1, direct=1),
        # the Taylor-Green step at 129^3, the reference's own solver parameters
        dict(name="step_tgv_129", kind="hydro", xi=7, yi=7, zi=7, domain="PPP", mesh="UUU"),
        # the Rayleigh-Benard convection step on 257 x 257 x 129 nodes
        dict(name="step_convection_257x257x129", kind="convection", xi=8, yi=8, zi=7, domain="PPN", mesh="UUD",
             precision="gcr", pads=1, direct=1),
        # one solve in a sequence: guess from the eight solves before it, solve, record
        dict(name="sequence_257x257x129", kind="sequence", xi=8, yi=8, zi=7),
        # the operators of a user's own time step on its own arrays, small with ragged sides
        dict(name="fields_33x17x65", kind="fields", xi=5, yi=4, zi=6, domain="NPN", mesh="DUD"),
        # the same on the benchmark's grid
        dict(name="fields_257", kind="fields", xi=8, yi=8, zi=8, domain="PPN", mesh="UUD"),
        # the implicit viscous solve of one velocity component on a user's arrays
        dict(name="viscous_129", kind="viscous", xi=7, yi=7, zi=7, domain="PPN", mesh="UUD", loc=1),
        # one online training step of the guess network beside a 257^3 solver
        dict(name="train_guess_257", kind="train", xi=8, yi=8, zi=8),
    ]


def draw(rng):
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        c = _draw(rng)
        if c not in known:
            return c


def _draw(rng):
    kind = rng.choice(["poisson", "poisson", "poisson", "poisson", "fields", "fields", "hydro", "convection",
                       "viscous", "sequence", "train"])
    domain, mesh = rng.choice([("PPN", "UUD"), ("PPN", "UUD"), ("NNN", "DDD"), ("NPN", "DUD"), ("PNN", "UDD")])
    c = dict(kind=kind, domain=domain, mesh=mesh)
    if kind == "hydro" and rng.random() < 0.5:
        k = rng.randint(4, 7)
        c.update(xi=k, yi=k, zi=k, domain="PPP", mesh="UUU")
        return c
    top = 7 if kind in ("hydro", "viscous") else 8
    low = 4 if kind in ("poisson", "fields") else 5
    while True:
        c["xi"], c["yi"], c["zi"] = (rng.randint(low, top) for _ in range(3))
        # the coarsest level of a solver has to fit one workgroup: sides at most a factor 8 apart
        if kind in ("fields", "viscous") or max(_ind(c)) - min(_ind(c)) <= 3:
            break
    if kind in ("poisson", "convection"):
        c["precision"] = rng.choice(["fp64", "mixed", "gcr"])
        c["pads"] = rng.randint(0, 1)
        # the exact coarsest level holds at most 1024 nodes
        m = min(c["xi"], c["yi"], c["zi"]) - 1
        nc = math.prod((1 << (c[a] - m)) + 1 for a in ("xi", "yi", "zi"))
        c["direct"] = rng.randint(0, 1) if nc <= 200 else 0
    if kind == "viscous":
        c["loc"] = rng.randint(0, 3)
    if kind in ("sequence", "train"):
        del c["domain"], c["mesh"]   # periodic in x and y, walls and stretching in z
    return c


# ---- geometry and inputs -------------------------------------------------------------------------
def _ind(c):
    return c["xi"], c["yi"], c["zi"]


def _lengths(c):
    m = min(_ind(c))
    return tuple(float(1 << (k - m)) for k in _ind(c))


def _nodes(c):
    return tuple((1 << k) + 1 for k in _ind(c))


def _axis(n, length, stretched, face):
    """Coordinates and metrics xi_x, xi_xx, xi_x^2 of one direction on the core nodes (or faces)."""
    m = n - 1 if face else n
    a = (torch.arange(m, dtype=F64) + (0.5 if face else 0.0)) / (n - 1)
    if not stretched:
        one = torch.ones(m, dtype=F64)
        return length * a, one / length, 0.0 * one, one / length ** 2
    tb = math.tanh(1.0)
    x = length * (1.0 - torch.tanh(1.0 - 2.0 * a) / tb) / 2.0
    s = 1.0 - 2.0 * x / length
    d1 = tb / (length * (1.0 - (s * tb) ** 2))
    d2 = -4.0 * tb ** 3 * s / (length ** 2 * (1.0 - (s * tb) ** 2) ** 2)
    return x, d1, d2, d1 ** 2


def _axes(c, faces=(False, False, False)):
    return [_axis(n, L, s == "D", f) for n, L, s, f in zip(_nodes(c), _lengths(c), c["mesh"], faces)]


def _pad(core):
    return torch.nn.functional.pad(core, (1, 1, 1, 1, 1, 1)).contiguous()


def _modes(c, seed, weights=None):
    """Smooth core node field: eight seeded Fourier modes that fit the domain (the right-hand sides of
    workloads.stretched_poisson, with cosines along walls)."""
    out = torch.zeros(_nodes(c), dtype=F64, device=DEV)
    kmax = max(2, min(16, min(_nodes(c)) // 4))
    xs = [a[0].to(DEV) for a in _axes(c)]
    for m, (a, kx, ky, kz, phx, phy) in enumerate(workloads.fourier_modes(seed, 8, kmax)):
        w = a if weights is None else weights[m]
        f = []
        for x, k, ph, per, L in zip(xs, (kx, ky, kz), (phx, phy, 0.0), c["domain"], _lengths(c)):
            f.append(torch.cos(2 * math.pi * k * x / L + ph) if per == "P" else torch.cos(math.pi * k * x / L))
        out += w * f[0][:, None, None] * f[1][None, :, None] * f[2][None, None, :]
    return out


def _random_field(shape, seed):
    """Padded field as a flow has it: large smooth motion with a little noise, ghosts included."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    out = 0.05 * torch.randn(shape, dtype=F64, device=DEV, generator=g)
    r = torch.rand((4, 7), dtype=F64, device=DEV, generator=g).cpu().tolist()
    xs = [torch.arange(n, dtype=F64, device=DEV) / (n - 3) for n in shape]
    for q in r:
        f = [torch.cos(2 * math.pi * ((1 + int(4 * q[d])) * xs[d] + q[3 + d])) for d in range(3)]
        out += (q[6] - 0.5) * f[0][:, None, None] * f[1][None, :, None] * f[2][None, None, :]
    return out


class _Array:
    """A torch tensor as the field operators take their arrays."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.ptr = self.t.data_ptr()


class _Memory:
    """A field of a running simulation, seen in place (and its owner kept alive)."""

    def __init__(self, ptr, shape, owner):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": "<f8", "version": 2}
        self.owner = owner


def _walls(domain):
    return field.bc([k for p in domain for k in ([field.PERIODIC] * 2 if p == "P" else [field.DIRICHLET] * 2)])


def _solver(c):
    p = mg.Parser.from_strings(mesh=c["mesh"], domain=c["domain"], vcCount=100, preSmooth=2, postSmooth=2, resType=2,
                               semantics=_lib.SR_SEM_PROJECTED, relTolerance=1e-10)
    p.xInd, p.yInd, p.zInd = _ind(c)
    p.Lx, p.Ly, p.Lz = _lengths(c)
    p.vcDepth = min(_ind(c)) - 1
    p.precision = {"fp64": _lib.SR_PREC_FP64, "mixed": _lib.SR_PREC_MIXED,
                   "gcr": _lib.SR_PREC_MIXED_GCR}[c["precision"]]
    p.padMode, p.coarseDirect = c["pads"], c["direct"]
    m = mg.Multigrid(mg.Grid(p), p)
    m.vCycle()   # the HIP runtime that torch brings reads a solve's timing events only after one eager cycle
    return m


def _stepper(desc):
    h, m = ts.Hydro(desc), ctypes.c_void_p()
    _lib.check(_lib.load().sr_ts_pressure_solver(h.h, ctypes.byref(m)))
    _lib.check(_lib.load().sr_mg_op_vcycle(m))   # as in _solver
    return h


def _centred(p):
    # periodic and Neumann boundaries fix a pressure up to a constant only: its level means nothing
    return p - p.mean()


# ---- prepare -------------------------------------------------------------------------------------
def prepare(case, seed):
    return _PREPARE[case["kind"]](dict(case), seed)


def _prepare_poisson(c, seed):
    s = {"kind": "poisson", "mg": _solver(c), "f": _pad(_modes(c, seed))}
    s["p"] = torch.zeros_like(s["f"])
    torch.cuda.synchronize()
    return s


def _snapshot(h, which):
    views = {}

    def view(w):
        ptr = h.device_ptr(w)
        if (w, ptr) not in views:
            views[w, ptr] = torch.as_tensor(_Memory(ptr, h.shape(w), h), device=DEV)
        return views[w, ptr]

    return {"h": h, "view": view, "saved": {w: view(w).clone() for w in which}}


def _prepare_hydro(c, seed):
    ind = _ind(c)
    periodic = c["domain"] == "PPP"
    L = (2 * math.pi,) * 3 if periodic else _lengths(c)
    h = _stepper(ts.ts_desc(ind=ind, L=L, domain=c["domain"], mesh=c["mesh"], depth=min(ind) - 1,
                            prob_type=2 if periodic else 1))
    h.initTGV()
    g = torch.Generator().manual_seed(seed)
    ph = (2 * math.pi * torch.rand(3, dtype=F64, generator=g)).tolist()
    amp = 0.5 + float(torch.rand(1, dtype=F64, generator=g))
    wave = [2 * math.pi / k for k in L]
    for comp, (w, sgn) in enumerate(((ts.VX, 1.0), (ts.VY, -1.0), (ts.VZ, 0.0))):
        v = torch.zeros(h.shape(w), dtype=F64)
        xs = [_axis(n, k, m == "D", d == comp)[0] for d, (n, k, m) in enumerate(zip(_nodes(c), L, c["mesh"]))]
        t = [torch.sin(wv * x + p) if d == comp else torch.cos(wv * x + p)
             for d, (x, wv, p) in enumerate(zip(xs, wave, ph))]
        v[1:-1, 1:-1, 1:-1] = sgn * amp * t[0][:, None, None] * t[1][None, :, None] * t[2][None, None, :]
        h.upload(w, v.numpy())
        h.imposeVBC(comp)
    s = _snapshot(h, (ts.VX, ts.VY, ts.VZ, ts.P, ts.PP))
    s["kind"] = "hydro"
    torch.cuda.synchronize()
    return s


def _prepare_convection(c, seed):
    prec = {"fp64": _lib.SR_PREC_FP64, "mixed": _lib.SR_PREC_MIXED, "gcr": _lib.SR_PREC_MIXED_GCR}[c["precision"]]
    h = _stepper(ts.ts_desc(ind=_ind(c), L=_lengths(c), domain=c["domain"], mesh=c["mesh"], scalar=True, rbc_type=2,
                            Ra=1e7, Pr=1.0, dt=0.01, prob_type=5, Re=1.0, semantics=_lib.SR_SEM_PROJECTED,
                            rel_tol=1e-10, vc_count=100, pre=2, post=2, res_type=2, depth=min(_ind(c)) - 1,
                            precision=prec, pad_mode=c["pads"], coarse_direct=c["direct"]))
    h.initRBC(seed=seed, amp=1e-3)
    for _ in range(3):
        h.timeAdvance()
    s = _snapshot(h, (ts.VX, ts.VY, ts.VZ, ts.T, ts.P, ts.PP))
    s["kind"] = "convection"
    torch.cuda.synchronize()
    return s


def _evolving(c, seed, n, dt=0.05):
    """Right-hand side n of a sequence that changes smoothly in time (workloads.EvolvingPoisson)."""
    modes, g = workloads.fourier_modes(seed, 8, 16), workloads.SplitMix64(seed + 7919)
    w = [0.5 + 1.5 * g.uniform() for _ in modes]
    psi = [2.0 * math.pi * g.uniform() for _ in modes]
    return _pad(_modes(c, seed, [m[0] * math.cos(a * n * dt + b) for m, a, b in zip(modes, w, psi)]))


def _prepare_sequence(c, seed):
    c.update(domain="PPN", mesh="UUD", precision="gcr", pads=1, direct=1)
    if math.prod((1 << (k - min(_ind(c)) + 1)) + 1 for k in _ind(c)) > 1000:
        c["direct"] = 0
    n = _nodes(c)
    s = {"kind": "sequence", "mg": _solver(c), "rhs": [_evolving(c, seed, k) for k in range(12)], "n": 0,
         "net": guess.GuessNet(tuple((k + 1) // 2 for k in n), fine=n, seed=0, history=8)}
    s["net"].set_policy(3)   # the predictor alone
    s["ring"] = [torch.zeros_like(s["rhs"][0]) for _ in range(3)]
    torch.cuda.synchronize()
    for _ in range(9):
        run(s)
    return s


def _prepare_fields(c, seed):
    fg = field.FieldGrid(field.fgrid_desc(ind=_ind(c), L=_lengths(c), mesh=c["mesh"], domain=c["domain"]))
    shape = [fg.shape(loc) for loc in range(4)]
    zero = lambda loc: _Array(torch.zeros(shape[loc], dtype=F64, device=DEV))  # noqa: E731
    s = {"kind": "fields", "fg": fg, "P": _Array(_random_field(shape[0], 4 * seed)),
         "V": [_Array(_random_field(shape[k], 4 * seed + k)) for k in (1, 2, 3)],
         "H": [zero(k) for k in (1, 2, 3)], "Hp": zero(0), "G": [zero(k) for k in (1, 2, 3)], "div": zero(0),
         "d1": zero(0), "d2": zero(0), "stream": torch.cuda.ExternalStream(fg.stream())}
    torch.cuda.synchronize()
    return s


def _prepare_viscous(c, seed):
    fg = field.FieldGrid(field.fgrid_desc(ind=_ind(c), L=_lengths(c), mesh=c["mesh"], domain=c["domain"]))
    shape = fg.shape(c["loc"])
    s = {"kind": "viscous", "fg": fg, "loc": c["loc"], "bc": _walls(c["domain"]),
         "F0": _random_field(shape, 2 * seed), "F": _Array(torch.zeros(shape, dtype=F64, device=DEV)),
         "G": _Array(torch.zeros(shape, dtype=F64, device=DEV)), "stream": torch.cuda.ExternalStream(fg.stream())}
    s["R"] = _Array(s["F0"] + 0.02 * _random_field(shape, 2 * seed + 1))
    torch.cuda.synchronize()
    return s


def _prepare_train(c, seed):
    c.update(domain="PPN", mesh="UUD", precision="gcr", pads=1, direct=0)
    n = _nodes(c)
    s = {"kind": "train", "mg": _solver(c), "net": guess.GuessNet(tuple((k + 1) // 2 for k in n), fine=n, seed=1)}
    fs = [_evolving(c, seed, k) for k in range(3)]
    s["p2"], s["p1"], s["p"] = (_direct(c, f[1:-1, 1:-1, 1:-1]) for f in fs)
    s["f"], s["out"] = fs[2], torch.zeros_like(fs[2])
    torch.cuda.synchronize()
    for _ in range(2):
        run(s)
    return s


_PREPARE = {"poisson": _prepare_poisson, "hydro": _prepare_hydro, "convection": _prepare_convection,
            "sequence": _prepare_sequence, "fields": _prepare_fields, "viscous": _prepare_viscous,
            "train": _prepare_train}


# ---- run -----------------------------------------------------------------------------------------
def run(state):
    return _RUN[state["kind"]](state)


def _run_poisson(s):
    s["p"].zero_()
    torch.cuda.current_stream().synchronize()   # the solver works on its own stream
    s["mg"].mgSolve_device(s["p"].data_ptr(), s["f"].data_ptr())
    return _centred(s["p"])


def _run_step(s):
    for w, a in s["saved"].items():
        s["view"](w).copy_(a)
    torch.cuda.current_stream().synchronize()
    s["h"].timeAdvance()
    out = {w: s["view"](w) for w in s["saved"] if w not in (ts.P, ts.PP)}
    return {**out, "P": _centred(s["view"](ts.P))}


def _run_sequence(s):
    n = s["n"]
    s["n"] = n + 1
    p, p1, p2 = (s["ring"][(n - k) % 3] for k in range(3))
    k = n % (2 * len(s["rhs"]) - 2)   # forth and back in time, without a jump
    f = s["rhs"][min(k, 2 * len(s["rhs"]) - 2 - k)].data_ptr()
    s["net"].predict(s["mg"], p1.data_ptr(), p2.data_ptr(), f, p.data_ptr())
    s["mg"].mgSolve_device(p.data_ptr(), f)
    s["net"].observe(s["mg"], f, p.data_ptr())
    return _centred(p)


def _run_fields(s):
    fg = s["fg"]
    with torch.cuda.stream(s["stream"]):
        for h in s["H"] + [s["Hp"]]:
            h.t.zero_()
    fg.vfComputeDiff(s["V"], s["H"])
    fg.vfComputeNLin(s["V"], s["V"], s["H"])
    fg.sfComputeDiff(s["P"], s["Hp"])
    fg.sfComputeNLin(s["V"], s["P"], s["Hp"])
    fg.gradient(s["P"], s["G"])
    fg.divergence(s["V"], s["div"])
    fg.calcDerivative1(field.NODE, 2, s["P"], s["d1"])
    fg.calcDerivative2(field.NODE, 0, s["P"], s["d2"])
    return {"H": [a.t for a in s["H"]], "Hp": s["Hp"].t, "G": [a.t for a in s["G"]], "div": s["div"].t,
            "d1": s["d1"].t, "d2": s["d2"].t}


def _run_viscous(s):
    with torch.cuda.stream(s["stream"]):
        s["F"].t.copy_(s["F0"])
    sweeps = s["fg"].jacobi(s["loc"], 1, 0.01, s["bc"], s["R"], s["F"], s["G"], coef=math.sqrt(1e-7), cn_tol=1e-6)
    return s["F"].t, sweeps


def _run_train(s):
    net = s["net"]
    net.predict(s["mg"], s["p1"].data_ptr(), s["p2"].data_ptr(), s["f"].data_ptr(), s["out"].data_ptr())
    net.train(s["p"].data_ptr())
    return {"guess": _centred(s["out"]), "weights": [net.get_layer(k) for k in range(_lib.SR_GUESS_LAYERS)]}


_RUN = {"poisson": _run_poisson, "hydro": _run_step, "convection": _run_step, "sequence": _run_sequence,
        "fields": _run_fields, "viscous": _run_viscous, "train": _run_train}


# ---- work ----------------------------------------------------------------------------------------
def work(case):
    """Bytes that must be read or written once, and, where the amount is fixed, the arithmetic.  The
    iterations of a solve are the method's, not the problem's: a solve counts its right-hand side and
    its solution."""
    n = math.prod(k + 2 for k in _nodes(case))
    kind = case["kind"]
    if kind == "poisson":
        return {"bytes": 16 * n, "flops": 13 * n}
    if kind == "hydro":      # V and P read and written, the pressure correction read and written
        return {"bytes": 8 * n * 10, "flops": 250 * n}
    if kind == "convection":
        return {"bytes": 8 * n * 12, "flops": 330 * n}
    if kind == "sequence":   # eight pairs read, one written, right-hand side read, solution written
        return {"bytes": 8 * n * 20, "flops": 40 * n}
    if kind == "fields":     # V and P read; H, Hp, G, div, d1, d2 written
        return {"bytes": 8 * n * 14, "flops": 190 * n}
    if kind == "viscous":    # the guess and the right-hand side read, the result written
        return {"bytes": 24 * n, "flops": 20 * n}
    net = math.prod((k + 1) // 2 for k in _nodes(case))
    flops = sum(2 * 27 * ci * co * net / 8 ** lv for ci, co, lv in map(guess.layer_info, range(_lib.SR_GUESS_LAYERS)))
    return {"bytes": 8 * n * 5, "flops": 3 * flops}


# ---- the same in plain torch, 64 bits --------------------------------------------------------------
def _eigen(n, length, stretched, periodic):
    """V, 1/V and the eigenvalues of one direction's second derivative on its independent nodes."""
    h = 1.0 / (n - 1)
    _, _, d2, dd = _axis(n, length, stretched, False)
    up, dn = dd / h ** 2 + d2 / (2 * h), dd / h ** 2 - d2 / (2 * h)
    m = n - 1 if periodic else n
    a = torch.zeros((m, m), dtype=F64)
    for i in range(m):
        a[i, i] -= 2 * dd[i] / h ** 2
        for j, w in ((i + 1, up[i]), (i - 1, dn[i])):
            j = j % m if periodic else 1 if j < 0 else n - 2 if j > n - 1 else j
            a[i, j] += w
    scale = torch.ones(m, dtype=F64)
    if not periodic:
        for i in range(m - 1):
            scale[i + 1] = scale[i] * torch.sqrt(a[i, i + 1] / a[i + 1, i])
    lam, q = torch.linalg.eigh((scale[:, None] * a / scale[None, :] + (scale[:, None] * a / scale[None, :]).T) / 2)
    return q / scale[:, None], q.T * scale[None, :], lam


def _direct(c, f):
    """Padded, centred solution of L p = f (core nodes) by diagonalising each direction."""
    per = [p == "P" for p in c["domain"]]
    n, L, m = _nodes(c), _lengths(c), c["mesh"]
    e = [[a.to(f.device) for a in _eigen(n[d], L[d], m[d] == "D", per[d])] for d in range(3)]
    u = f[tuple(slice(0, n[d] - 1 if per[d] else n[d]) for d in range(3))]
    for d in range(3):
        u = torch.tensordot(e[d][1], u, dims=([1], [d])).movedim(0, d)
    lam = e[0][2][:, None, None] + e[1][2][None, :, None] + e[2][2][None, None, :]
    null = lam.abs() < 1e-9 * lam.abs().max()
    u = torch.where(null, torch.zeros_like(u), u / torch.where(null, torch.ones_like(lam), lam))
    for d in range(3):
        u = torch.tensordot(e[d][0], u, dims=([1], [d])).movedim(0, d)
    for d in range(3):
        r = list(range(n[d]))
        at = [n[d] - 2, *r[:-1], 0, 1] if per[d] else [1, *r, n[d] - 2]
        u = u.index_select(d, torch.tensor(at, device=f.device))
    return _centred(u.contiguous())


def _shift(a, core, off):
    return a[tuple(slice(1 + o, 1 + o + n) for o, n in zip(off, core))]


def _exact_fields(c, seed):
    s = _prepare_fields(c, seed)
    n = _nodes(c)
    h = [1.0 / (k - 1) for k in n]
    node, face = _axes(c), _axes(c, (True, True, True))
    unit = [[int(d == e) for e in range(3)] for d in range(3)]
    core = lambda loc: [k - (d == loc - 1) for d, k in enumerate(n)]                       # noqa: E731

    def along(v, d):
        return v.to(DEV).reshape([-1 if e == d else 1 for e in range(3)])

    def step(F, loc, d, o):
        return _shift(F, core(loc), [o * q for q in unit[d]])

    def metric(loc, d, q):
        return along((face if d == loc - 1 else node)[d][q], d)

    def first(F, loc, d):
        return metric(loc, d, 1) * (step(F, loc, d, 1) - step(F, loc, d, -1)) / (2 * h[d])

    def second(F, loc, d):   # the Crank-Nicolson half of the second derivative
        return (metric(loc, d, 2) * (step(F, loc, d, 1) - step(F, loc, d, -1)) / (2 * h[d]) +
                0.5 * metric(loc, d, 3) * (step(F, loc, d, 1) - 2 * step(F, loc, d, 0) + step(F, loc, d, -1)) / h[d] ** 2)

    V, P = [v.t for v in s["V"]], s["P"].t

    def rhs(F, loc):
        out = 0.0
        for d in range(3):
            offs = [[0, 0, 0]]
            if d != loc - 1:
                offs.append([-q for q in unit[d]])
                if loc > 0:
                    offs += [[a + b for a, b in zip(o, unit[loc - 1])] for o in offs]
            adv = sum(_shift(V[d], core(loc), o) for o in offs) / len(offs)
            out = out + second(F, loc, d) - adv * first(F, loc, d)
        return _pad(out)

    def whole(fn, d):
        """A derivative of P along d on the padded node array: pads along d are zero, the others not."""
        big = list(n)
        out = torch.zeros_like(P)
        sl = [slice(None)] * 3
        sl[d] = slice(1, 1 + big[d])
        lo, hi, mid = list(sl), list(sl), sl
        lo[d], hi[d] = slice(0, big[d]), slice(2, 2 + big[d])
        out[tuple(mid)] = fn(P[tuple(hi)], P[tuple(mid)], P[tuple(lo)])
        return out

    q1, q2, q3 = (along(node[2][q], 2) for q in (1, 2, 3))
    r2, r3 = (along(node[0][q], 0) for q in (2, 3))
    div = sum(along(node[d][1], d) * (_shift(V[d], n, [0, 0, 0]) - _shift(V[d], n, [-q for q in unit[d]])) / h[d]
              for d in range(3))
    return {"H": [rhs(V[k], k + 1) for k in range(3)], "Hp": rhs(P, 0),
            "G": [_pad(along(face[k][1], k) * (step(P, k + 1, k, 1) - step(P, k + 1, k, 0)) / h[k]) for k in range(3)],
            "div": _pad(div), "d1": whole(lambda a, b, e: q1 * (a - e) / (2 * h[2]), 2),
            "d2": whole(lambda a, b, e: r2 * (a - e) / (2 * h[0]) + 0.5 * r3 * (a - 2 * b + e) / h[0] ** 2, 0)}


def exact(case, seed):
    c = dict(case)
    if c["kind"] == "poisson":
        return _direct(c, _modes(c, seed))
    if c["kind"] == "fields":
        return _exact_fields(c, seed)
    return None   # time steps, Jacobi to a tolerance, learned guesses: no closed value
