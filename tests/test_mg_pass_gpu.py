"""The one-launch red-black sweep (saras_amd/csrc/mg_pass.hip) at the edges of its tiles and ranges.

V-cycles from random data (not periodic itself, so the duplicated end nodes of a periodic direction
differ) against the oracle's red-black cycle: one and several row tiles, chunks of one plane and of
several, rows of 4 entries up to 258, every image rule (periodic, mirror, antisymmetric), odd and even
sweep counts (odd ones after a prolongation mix with the half sweeps)."""
import numpy as np
import pytest

from helpers import Problem, r2_walls
from oracle import pyoracle as po
from test_mg_gpu import RTOL

pytestmark = pytest.mark.gpu

CASES = [
    # ind, domain, mesh, pre, post, Dirichlet walls (antisymmetric images below level 0)
    ((2, 2, 2), "PPN", "UUD", 2, 2, False),
    ((3, 2, 4), "NNN", "DDD", 3, 4, False),
    ((4, 6, 2), "PNP", "UDU", 1, 2, False),
    ((6, 4, 5), "PPP", "UUU", 4, 4, False),
    ((5, 4, 3), "NPP", "DUU", 2, 3, False),
    ((6, 6, 6), "NNN", "UUU", 2, 2, True),
    ((6, 6, 6), "PNN", "UDU", 2, 4, True),
    ((8, 3, 3), "PPN", "UUD", 2, 2, False),
    ((3, 8, 3), "NPN", "DUD", 2, 2, False),
    ((3, 3, 8), "PPN", "UUD", 2, 2, False),
    ((3, 3, 9), "PPP", "UUU", 2, 2, False),
    ((7, 5, 5), "PPN", "UUD", 2, 2, False),
]

# the one-workgroup coarse end (saras_amd/csrc/mg_coarse.hip): its first level with one and three entries
# per thread and with more items than threads, no pre- or post-smoothing, coarsest levels of one wave, of
# the workgroup and (17 x 17 x 5 nodes) of more nodes than the workgroup has threads, which are solved
# outside it
COARSE = [
    ((4, 4, 4), "PPN", "UUD", 2, 2, False, None),
    ((5, 5, 5), "NNN", "DDD", 2, 1, False, None),
    ((5, 5, 5), "PPP", "UUU", 0, 2, False, None),
    ((5, 5, 5), "NPN", "DUD", 1, 0, False, None),
    ((5, 5, 5), "PNP", "UDU", 0, 0, False, None),
    ((6, 6, 5), "PPN", "UUD", 2, 2, False, 3),
    ((6, 5, 4), "NNN", "UUU", 3, 2, True, None),
    ((5, 6, 5), "NNP", "UUU", 2, 2, True, None),
    ((5, 5, 5), "NNN", "UUU", 0, 2, True, None),
    ((6, 6, 4), "PPN", "UUD", 2, 2, False, 2),
]


def _problem(ind, domain, mesh, pre, post, walls, depth=None, **kw):
    n = [(1 << k) + 1 for k in ind]
    m = min(ind)
    return Problem(ind=ind, domain=domain, mesh=mesh, L=tuple(float(1 << (k - m)) for k in ind), pre=pre, post=post,
                   depth=depth, test_poisson=walls, walls=r2_walls(n) if walls else None, **kw)


@pytest.mark.parametrize("case", CASES + COARSE, ids=str)
def test_vcycle_matches_oracle(case):
    """Three iterates within the per-operator bar.  Without Dirichlet walls the operator is singular and
    the coarsest iteration runs to its limit (up to 2000 times here), each step moving the level of the
    iterate by its rounding: as for the pressures of a time step, the level is taken out."""
    pb = _problem(*case)
    o, g = pb.oracle(), pb.gpu()
    P0, F0 = np.random.default_rng(7).standard_normal(pb.shape), pb.random_rhs(8)
    o.level = 0
    o.array(po.P, 0)[...] = P0
    o.array(po.R, 0)[...] = F0
    g.upload(po.P, 0, P0)
    g.upload(po.R, 0, F0)
    for it in range(3):
        o.vcycle()
        g.vCycle()
        o.set_zero_bc(0)
        g.set_zeroBC(0)
        o.impose_bc()
        g.imposeBC()
        exp, d = o.array(po.P, 0), g.download(po.P, 0) - o.array(po.P, 0)
        if not case[5]:
            d = d - d[1:-1, 1:-1, 1:-1].mean()
        assert np.max(np.abs(d)) <= RTOL * np.max(np.abs(exp)), (it, np.max(np.abs(d)), np.max(np.abs(exp)))
    g.close()


# z directions too long for the sweeps' workgroups on the two finest levels: half sweeps, the first of which
# the restriction does on level 1, above one-launch sweeps
LONG = [((5, 5, 11), "PPN", "UUD", 2, 2, False), ((5, 5, 11), "NNN", "UUU", 3, 2, True)]


def _coarsest(pb):
    return int(np.prod([(k - 1 >> pb.depth) + 1 for k in pb.n]))


@pytest.mark.parametrize("case", LONG, ids=str)
def test_vcycle_matches_oracle_on_long_rows(case):
    test_vcycle_matches_oracle(case)


@pytest.mark.parametrize("case", CASES + COARSE + LONG, ids=str)
def test_fp32_cycle_node_by_node(case):
    """One FP32 cycle on the right-hand side against one FP64 cycle from zero, the level taken out where
    the operator is singular.  An update rounds a node to 6e-8 of its size and a cycle makes some 4 (pre +
    post) of them on every level, a coarsest iteration one more: (256 + iterations) units of the largest
    value are ten times what accumulates."""
    pb = _problem(*case, vc_count=1, rel_tol=1e-30)
    f = pb.random_rhs(5)
    for direct in (0, 1) if _coarsest(pb) <= 1024 else (0,):
        p, its = [], 0
        for precision in (0, 1):
            g = pb.gpu(precision=precision, coarse_direct=direct)
            x = np.zeros(pb.shape)
            assert g.mgSolve(x, f).cycles == 1
            its = max(its, g.info(5))
            p.append(x[1:-1, 1:-1, 1:-1])
            g.close()
        d = p[1] - p[0]
        if not case[5]:
            d = d - d.mean()
        assert np.max(np.abs(p[0])) > 0
        tol = (256 + its) * 2.0 ** -24 * max(np.max(np.abs(x)) for x in p)
        assert np.max(np.abs(d)) <= tol, (direct, its, np.max(np.abs(d)), tol)


@pytest.mark.parametrize("case", [c for c in CASES if not c[5]], ids=str)
def test_fp32_cycles_follow_fp64(case):
    """The refinement's residual history is that of the FP64 cycles up to what L makes of the rounding of
    the correction: 16 units of 6e-8 of the largest |p| times |L|, relative to the right-hand side."""
    pb = _problem(*case, vc_count=2, rel_tol=1e-30)
    f = pb.random_rhs(5)
    hist, top = [], 0.0
    for precision in (0, 1):
        g = pb.gpu(precision=precision, coarse_direct=1 if np.prod([k >> (pb.depth) for k in pb.n]) < 100 else 0)
        p = np.zeros(pb.shape)
        g.mgSolve(p, f)
        hist.append(g.history())
        c = p[1:-1, 1:-1, 1:-1]
        top = max(top, np.max(np.abs(c - c.mean())))
        g.close()
    tol = 16 * 2.0 ** -24 * _operator_norm(pb) * top * np.sqrt(np.prod(pb.n)) / np.linalg.norm(f)
    assert tol < 0.6 * hist[0][1], (tol, hist)   # below what is compared
    assert len(hist[0]) == 2 and np.max(np.abs(hist[0] - hist[1])) <= tol, (hist, tol)


def _operator_norm(pb):
    size = 0.0
    for d in range(3):
        ax, h = po.grid_axis(pb.n[d], pb.L[d], pb.gtype[d], pb.beta[d]), 1.0 / (pb.n[d] - 1)
        size += 4 * np.max(np.abs(ax["xix2"])) / h**2 + np.max(np.abs(ax["xixx"])) / h
    return size


# marching outer step (saras_amd/csrc/mg_outer.hip): also no post-smoothing, whose L e is formed on both colours
OUTER = [c for c in CASES if not c[5]] + [((5, 5, 4), "NPN", "DUD", 2, 0, False), ((4, 5, 3), "PNP", "UDU", 2, 0, False)]


@pytest.mark.parametrize("precision", [0, 1, 2], ids=["fp64", "refinement", "gcr"])
@pytest.mark.parametrize("case", OUTER, ids=str)
def test_residual_norms_match_oracle(case, precision):
    """The norm of the guess, the norm of every cycle and what the cycle left, against the oracle's
    computeError of the same iterate.  Both round r = f - L x to some 10 units of |L| |x| per node, which
    bounds the difference of the relative norms.  A GCR step is the best one along its directions, so
    that its first is no worse than the refinement step up to the rounding of L e in FP32."""
    from saras_amd import _lib
    lens = []
    for count in (1, 2, 3):
        pb = _problem(*case, vc_count=count, rel_tol=1e-30)
        f, x = pb.random_rhs(5), 1e-3 * pb.random_rhs(6)
        o = pb.oracle()
        o.level = 0
        fp = o.project_rhs(f.copy())
        size = _operator_norm(pb)

        def check(got, p):
            o.array(po.P, 0)[...] = p
            o.impose_bc()
            o.array(po.R, 0)[...] = fp
            want = o.compute_error(2)
            tol = 16 * 2.2e-16 * size * np.max(np.abs(p)) * np.sqrt(np.prod(pb.n)) / np.linalg.norm(fp[1:-1, 1:-1, 1:-1])
            assert abs(got - want) <= tol + 1e-12 * want, (count, got, want, tol)

        g = pb.gpu(precision=precision, coarse_direct=1 if np.prod([k >> (pb.depth) for k in pb.n]) < 100 else 0)
        bufs = [_lib.DeviceArray(pb.shape) for _ in range(2)]
        bufs[0].upload(x)
        bufs[1].upload(f)
        check(g.residual_device(bufs[0].ptr, bufs[1].ptr), x)
        p = x.copy()
        st = g.mgSolve(p, f)
        if precision:
            check(st.residual0, x)
        hist = g.history()
        assert len(hist) == count
        check(hist[-1], p)
        lens.append(hist)
        g.close()
    assert lens[0][0] == lens[1][0] == lens[2][0] and lens[1][1] == lens[2][1]   # the same steps each time
    if precision == 2:
        g = pb.gpu(precision=1, coarse_direct=1 if np.prod([k >> (pb.depth) for k in pb.n]) < 100 else 0)
        g.mgSolve(x.copy(), f)
        hist = lens[2]
        assert hist[0] <= g.history()[0] * (1 + 1e-5)
        assert np.all(hist[1:] <= hist[:-1] * (1 + 1e-5)), hist
        g.close()


@pytest.mark.parametrize("case", [CASES[1], CASES[3], CASES[5]], ids=str)
def test_residual_leaves_the_guess_with_its_ghosts(case):
    """sr_mg_residual without the residual field leaves level 0 as with it: the operators go on from there."""
    from saras_amd import _lib
    pb = _problem(*case)
    g = pb.gpu()
    p, f, r = (_lib.DeviceArray(pb.shape) for _ in range(3))
    p.upload(pb.random_rhs(6))
    f.upload(pb.random_rhs(5))
    state = []
    for out in (r.ptr, None):
        g.residual_device(p.ptr, f.ptr, out)
        guess = g.download(po.P, 0)
        g.computeResidual()
        state.append((guess, g.download(po.T, 0)))
    for a, b in zip(*state):
        assert np.array_equal(a, b)
    assert np.array_equal(state[0][1][1:-1, 1:-1, 1:-1], r.download()[1:-1, 1:-1, 1:-1])
    g.close()
