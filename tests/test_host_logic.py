"""The library's host code over a HIP runtime whose kernels do nothing (fake_hip.cc).  CPU only."""
import concurrent.futures as cf
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

from saras_amd import _lib, build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host"))
    obj = [os.path.join(out, s + ".o") for s in build.HIP_SOURCES]

    def compile_one(s, o):
        subprocess.run([build.HIPCC, f"--offload-arch={build.ARCH}", "--offload-host-only", "-O1", "-std=c++17", "-fPIC",
                        "-w", "-c", os.path.join(build.CSRC, s), "-o", o], check=True, capture_output=True)

    with cf.ThreadPoolExecutor(max_workers=8) as ex:
        list(ex.map(compile_one, build.HIP_SOURCES, obj))
    # the device code, which there is none of
    names = subprocess.run(["nm", "-u", *obj], check=True, capture_output=True, text=True).stdout
    none = [f"-Wl,--defsym={s}=0" for s in sorted(set(re.findall(r"__hip_fatbin\w*", names)))]
    so = os.path.join(out, "libhost.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-o", so, *obj,
                    *[os.path.join(build.CSRC, s) for s in build.CPP_SOURCES], os.path.join(HERE, "fake_hip.cc"), *none],
                   check=True, capture_output=True)
    return so


@pytest.fixture
def fake(library, monkeypatch):
    """The package on that library, and the fake runtime's own calls."""
    monkeypatch.setattr(_lib, "LIB_PATH", library)
    monkeypatch.setattr(_lib, "_lib", None)
    L = _lib.load()
    L.fake_launched.restype = C.c_char_p
    L.fake_clear()
    L.fake_refuse_lds(0)
    yield L
    L.fake_refuse_lds(0)


def _launched(L):
    return L.fake_launched().decode().split("\n")[:-1]


def _problem(**kw):
    from helpers import Problem
    return Problem(**{**dict(ind=(4, 4, 4), domain="PPN", mesh="UUD", vc_count=3), **kw})


@pytest.mark.parametrize("precision", [0, 1, 2], ids=["fp64", "refinement", "gcr"])
def test_a_solve_whose_residuals_never_arrive_does_not_converge(fake, precision):
    """The host's mirror of the residual holds zeros here, which would pass any stop rule."""
    pb = _problem()
    g = pb.gpu(precision=precision)
    st = g.mgSolve(np.zeros(pb.shape), pb.random_rhs(0))
    assert not st.converged and st.cycles == pb.vc_count and not st.residual == st.residual
    if precision:
        assert not st.residual0 == st.residual0
    g.close()


def test_a_viscous_solve_whose_residuals_never_arrive_fails(fake):
    from saras_amd import field
    fg = field.FieldGrid(field.fgrid_desc(ind=(3, 3, 3), domain="PPN"))
    F, G, R = (fg.array(1) for _ in range(3))
    P, D = field.PERIODIC, field.DIRICHLET
    with pytest.raises(_lib.SarasError):
        fg.jacobi(1, 0, 1e-3, field.bc([P, P, P, P, D, D]), R, F, G, Re=100.0)
    for a in (F, G, R):
        a.free()
    fg.close()


@pytest.mark.parametrize("precision", [0, 1, 2], ids=["fp64", "refinement", "gcr"])
def test_without_large_lds_a_solver_runs_the_per_node_kernels(fake, precision):
    big = ("k_rb_pass", "k_march", "k_coarse_cycle")
    pb = _problem()
    for refused in (0, 1):
        fake.fake_refuse_lds(refused)
        g = pb.gpu(precision=precision)
        fake.fake_clear()
        g.vCycle()
        g.mgSolve(np.zeros(pb.shape), pb.random_rhs(0))
        ran = {b for b in big for name in _launched(fake) if b in name}
        assert ran == (set() if refused else set(big)), (refused, ran)
        g.close()


@pytest.mark.parametrize("ind", [(2, 2, 2), (2, 8, 8), (8, 2, 8), (8, 8, 2), (6, 6, 6), (7, 7, 7), (8, 8, 8), (9, 3, 9),
                                 (9, 6, 8), (10, 5, 7), (12, 2, 2), (2, 2, 12), (3, 9, 9)], ids=str)
def test_split_of_the_column_marches(fake, ind):
    """Every plane in one chunk, no chunk longer than the metrics' LDS rows; chunks of one plane (half of a
    pair of loads) only on a grid that they hardly fill the device with; a contiguous eighth of the
    workgroups, an XCD's, holds at least 16 rows of every plane or an eighth of many planes."""
    from saras_amd import field
    fg = field.FieldGrid(field.fgrid_desc(ind=ind))
    V, H, F, out = [fg.array(c) for c in (1, 2, 3)], [fg.array(c) for c in (1, 2, 3)], fg.array(0), fg.array(0)
    fake.fake_clear()
    fg.vfComputeDiff(V, H)
    fg.vfComputeNLin(V, V, H)
    fg.sfComputeNLin(V, F, out)
    fg.divergence(V, out)
    fg.calcDerivative2(0, 1, F, out)
    rows, row = (1 << ind[1]) + 3, (1 << ind[2]) + 3
    lines = _launched(fake)
    assert len(lines) == 5
    for line in lines:
        grid, threads, nb, nch, cq, cr, by_chunk = (int(x) for x in line.split()[1:])
        planes = nch * cq + cr
        assert planes == (1 << ind[0]) + (3 if "diverg" in line or "deriv" in line else 1)
        assert grid == nb * nch and nb * threads >= rows * row > (nb - 1) * threads
        assert cr < nch and 1 <= cq + (cr > 0) <= 64
        assert cq > 1 or cr >= nch - 1 or grid <= 1024, line
        assert grid <= max(2304, nb * -(-planes // 64)), line
        assert by_chunk == (rows < 16 * 8 + 2 and planes > rows), line
    for a in V + H + [F, out]:
        a.free()
    fg.close()
