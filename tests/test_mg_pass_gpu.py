"""The one-launch red-black sweep (saras_amd/csrc/mg_pass.hip) at the edges of its tiles and ranges.

V-cycles from random data (not periodic itself, so the duplicated end nodes of a periodic direction
differ) against the oracle's red-black cycle: one and several row tiles, chunks of one plane and of
several, rows of 4 entries up to 258, every image rule (periodic, mirror, antisymmetric), odd and even
sweep counts (odd ones after a prolongation mix with the half sweeps)."""
import numpy as np
import pytest

from helpers import Problem, r2_walls
from test_mg_gpu import _vcycle_iterates

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


def _problem(ind, domain, mesh, pre, post, walls, **kw):
    n = [(1 << k) + 1 for k in ind]
    m = min(ind)
    return Problem(ind=ind, domain=domain, mesh=mesh, L=tuple(float(1 << (k - m)) for k in ind), pre=pre, post=post,
                   test_poisson=walls, walls=r2_walls(n) if walls else None, **kw)


@pytest.mark.parametrize("case", CASES, ids=str)
def test_vcycle_matches_oracle(case):
    pb = _problem(*case)
    o, g = pb.oracle(), pb.gpu()
    _vcycle_iterates(pb, o, g)
    g.close()


@pytest.mark.parametrize("case", [c for c in CASES if not c[5]], ids=str)
def test_fp32_cycles_follow_fp64(case):
    """The refinement's residual history is that of the FP64 cycles up to the rounding of L e in FP32:
    about 4 n^2 units of 6e-8 relative to the right-hand side for n nodes along the longest side."""
    pb = _problem(*case, vc_count=2, rel_tol=1e-30)
    f = pb.random_rhs(5)
    hist = []
    for precision in (0, 1):
        g = pb.gpu(precision=precision, coarse_direct=1 if np.prod([k >> (pb.depth) for k in pb.n]) < 100 else 0)
        g.mgSolve(np.zeros(pb.shape), f)
        hist.append(g.history())
        g.close()
    tol = 4 * max(pb.n) ** 2 * 6e-8
    assert len(hist[0]) == 2 and np.max(np.abs(hist[0] - hist[1])) <= tol * max(1.0, hist[0][0]), (hist, tol)
