"""The kernels that march along x (saras_amd/csrc/columns.h) where chunks hold one plane, several and
uneven numbers of them and where a plane's last workgroup is nearly empty, against the oracle; and the
outputs that share memory, which the components then write in order, one launch each."""
import numpy as np
import pytest

from oracle import pyoracle as po
from helpers import rel_close

pytestmark = pytest.mark.gpu

RTOL = 1e-12

GRIDS = {
    # several planes per chunk, unevenly, and one; z periodic, with walls and walls all round
    "65x129x129": dict(ind=(6, 7, 7), L=(1.0, 2.0, 2.0), domain="PPN", mesh="UUD", beta=(1.0, 1.0, 1.2)),
    "129x129x129": dict(ind=(7, 7, 7), L=(1.0, 1.0, 1.0), domain="NNN", mesh="DDD", beta=(1.1, 0.7, 1.3)),
    "33x5x17": dict(ind=(5, 2, 4), L=(1.0, 2.0, 1.5), domain="NPP", mesh="DUU", beta=(1.1, 1.0, 1.0)),
    "65x33x65": dict(ind=(6, 5, 6), L=(2.0, 1.0, 2.0), domain="PPP", mesh="UUU"),
    "257x17x129": dict(ind=(8, 4, 7), L=(1.0, 1.0, 1.0), domain="PNP", mesh="UDU", beta=(1.0, 0.7, 1.0)),
}


def _pair(grid):
    from saras_amd import field
    g = GRIDS[grid]
    o = po.OracleTS(po.ts_params(**g))
    return o, field.FieldGrid(field.fgrid_desc(ind=g["ind"], L=g["L"], mesh=g["mesh"],
                                               beta=g.get("beta", (1.0,) * 3), domain=g["domain"]))


def _close(a, b, what):
    ok, err, s = rel_close(a, b, RTOL)
    assert a.shape == b.shape and ok, (what, err, s)


@pytest.mark.parametrize("grid", list(GRIDS))
def test_field_operators(grid):
    o, fg = _pair(grid)
    rng = np.random.default_rng(1)
    new = lambda loc: rng.standard_normal(o.loc_shape(loc))  # noqa: E731
    U, V, H, G = ([new(c) for c in (1, 2, 3)] for _ in range(4))
    F, HF = new(0), new(0)
    dU, dV, dH, dG = ([fg.array(c + 1, a[c]) for c in range(3)] for a in (U, V, H, G))
    dF, dHF, ddiv = fg.array(0, F), fg.array(0, HF), fg.array(0, new(0))
    fg.vfComputeDiff(dU, dH)
    fg.vfComputeNLin(dU, dV, dH)
    fg.vfComputeNLin(dU, dU, dH)
    fg.sfComputeDiff(dF, dHF)
    fg.sfComputeNLin(dV, dF, dHF)
    fg.gradient(dF, dG)
    fg.divergence(dV, ddiv)
    fg.sync()
    for c in range(3):
        o.fd_diff(c + 1, U[c], H[c])
        o.fd_nlin(c + 1, U[c], V, H[c])
        o.fd_nlin(c + 1, U[c], U, H[c])
        _close(dH[c].download(), H[c], f"H{c}")
    o.fd_diff(0, F, HF)
    o.fd_nlin(0, F, V, HF)
    _close(dHF.download(), HF, "node H")
    o.fd_gradient(F, G)
    for c in range(3):
        _close(dG[c].download(), G[c], f"gradient {c}")
    _close(ddiv.download(), o.fd_divergence(V), "divergence")
    for loc, a, d in ((0, F, dF), (1, U[0], dU[0]), (3, U[2], dU[2])):
        out = fg.array(loc, new(loc))
        for order in (1, 2):
            for dim in range(3):
                (fg.calcDerivative1 if order == 1 else fg.calcDerivative2)(loc, dim, d, out)
                fg.sync()
                _close(out.download(), o.fd_deriv(loc, order, dim, a), (loc, order, dim))
    fg.close()
    o.close()


@pytest.mark.parametrize("grid", list(GRIDS))
def test_right_hand_sides(grid):
    """Velocity with buoyancy and temperature, and (closed by the same pads) the velocity alone."""
    from saras_amd import ts
    for scalar in (True, False):
        kw = dict(GRIDS[grid], dt=1e-3, Re=50.0)
        if scalar:
            kw.update(scalar=True, rbc_type=1, Ra=1e4, Pr=0.7, prob_type=6)
        o, g = po.OracleTS(po.ts_params(**kw)), ts.Hydro(ts.ts_desc(**kw))
        rng = np.random.default_rng(2)
        for wo, wg in [(0, 0), (1, 1), (2, 2), (po.PRES, ts.P)] + ([(po.TEMP, ts.T)] if scalar else []):
            a = o.array(wo)
            a[...] = rng.standard_normal(a.shape)
            g.upload(wg, a)
        o.build_rhs()
        g.buildRHS()
        for wg, wo in ((ts.HX, po.HX), (ts.HY, po.HY), (ts.HZ, po.HZ)):
            _close(g.download(wg), o.array(wo), wg)
        if scalar:
            o.build_trhs()
            g.buildTRHS()
            _close(g.download(ts.TRHS), o.array(po.TRHS), "tmpRHS")
        g.close()
        o.close()


def test_outputs_that_share_memory():
    """All three outputs in one buffer: what the components leave there one after the other."""
    o, fg = _pair("33x5x17")
    rng = np.random.default_rng(3)
    shape = [o.loc_shape(c) for c in (1, 2, 3)]
    V = [rng.standard_normal(s) for s in shape]
    F, start = rng.standard_normal(o.loc_shape(0)), rng.standard_normal(o.loc_shape(0))
    dV, dF, buf = [fg.array(c + 1, V[c]) for c in range(3)], fg.array(0, F), fg.array(0, start)

    def expect(step):
        flat = start.copy().ravel()
        for c in range(3):
            n = int(np.prod(shape[c]))
            part = flat[:n].reshape(shape[c]).copy()
            step(c, part)
            flat[:n] = part.ravel()
        return flat.reshape(start.shape)

    def grad(c, part):
        G = [np.zeros(s) for s in shape]
        o.fd_gradient(F, G)
        part[1:-1, 1:-1, 1:-1] = G[c][1:-1, 1:-1, 1:-1]

    for call, step in ((lambda: fg.vfComputeDiff(dV, [buf] * 3), lambda c, a: o.fd_diff(c + 1, V[c], a)),
                       (lambda: fg.vfComputeNLin(dV, dV, [buf] * 3), lambda c, a: o.fd_nlin(c + 1, V[c], V, a)),
                       (lambda: fg.gradient(dF, [buf] * 3), grad)):
        buf.upload(start)
        call()
        fg.sync()
        _close(buf.download(), expect(step), "shared outputs")
    fg.close()
    o.close()


# an output (component) that lies over part of an input: (output, input list, its component, planes between
# the start of the first of the two and of the second).  Over another component's U anywhere; over Vx only
# its plane before the first core one, which component x does not read.
OVERLAPS = [("x", "U", "y", 3), ("z", "U", "x", 2), ("y", "U", "z", -4), ("x", "V", "x", None)]


@pytest.mark.parametrize("case", OVERLAPS, ids=str)
def test_nlin_output_over_part_of_an_input(case):
    """The components are done in order, each reading what the ones before it left in memory."""
    from saras_amd import _lib
    out, which, comp, planes = "xyz".index(case[0]), case[1], "xyz".index(case[2]), case[3]
    o, fg = _pair("33x5x17")
    rng = np.random.default_rng(5)
    shape = [o.loc_shape(c) for c in (1, 2, 3)]
    A = {n: [rng.standard_normal(s) for s in shape] for n in "UVH"}
    D = {n: [fg.array(c + 1, A[n][c]) for c in range(3)] for n in "UVH"}
    if planes is None:
        planes = shape[out][0] - 2   # the output's last core plane on the input's first plane
    step = abs(planes) * int(np.prod(shape[out][1:]))
    first = [("H", out), (which, comp)] if planes > 0 else [(which, comp), ("H", out)]
    sizes = [int(np.prod(shape[c])) for _, c in first]
    flat = rng.standard_normal(max(sizes[0], step + sizes[1]))
    buf = _lib.DeviceArray(flat.shape)
    buf.upload(flat)

    class Part:
        pass

    for (name, c), at, n in zip(first, (0, step), sizes):
        A[name][c] = flat[at:at + n].reshape(shape[c])
        D[name][c] = Part()
        D[name][c].ptr = buf.ptr + 8 * at
    fg.vfComputeNLin(D["U"], D["V"], D["H"])
    fg.sync()
    for c in range(3):
        o.fd_nlin(c + 1, A["U"][c], A["V"], A["H"][c])
    _close(buf.download(), flat, case)
    for c in range(3):
        if c != out:
            _close(D["H"][c].download(), A["H"][c], (case, c))
    fg.close()
    o.close()


@pytest.mark.parametrize("grid", list(GRIDS))
def test_jacobi_solves(grid):
    """Same sweeps and fields as the oracle where a chunk of a sweep holds several planes, with the pads and
    the z walls filled in one launch (no x and y walls) and in several."""
    from saras_amd import ts
    kw = dict(GRIDS[grid], dt=1e-3, Re=200.0)
    o, g = po.OracleTS(po.ts_params(**kw)), ts.Hydro(ts.ts_desc(**kw))
    rng = np.random.default_rng(4)
    for c in range(3):
        a = o.array(c)
        a[...] = 0.1 * rng.standard_normal(a.shape)
        g.upload(c, a)
        o.impose_vbc(c)
        g.imposeVBC(c)
        assert np.array_equal(g.download(c), a), c
    P = o.array(po.PRES)
    P[...] = 0.0
    g.upload(ts.P, P)
    o.build_rhs()
    g.buildRHS()
    for c in range(3):
        assert o.solve_v(c) == g.solveV(c), c
        _close(g.download(c), o.array(c), f"V{c}")
    g.close()
    o.close()
