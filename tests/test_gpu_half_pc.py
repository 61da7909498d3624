"""FP64 BiCGStab with three Jacobi sweeps, whose half-iterations are fused on rows of any
length, against the oracle: the first iterations, to the rounding of the dot products."""
import importlib

import numpy as np
import pytest

from helpers import interior_mask, rand_field, rel_l2, small_mesh

hip = importlib.import_module("3dalm_amd.hip")
po = importlib.import_module("pyoracle")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ok():
    return po.Kernels("oracle")


# rows of a quad and a cell; rows of whole quads; a last j tile and a last chunk of fewer
# cells; rows of three and two cells over; rows near the longest a block takes; on grids that
# the one-launch solver would take, that is told to give up (a limit of one poll)
@pytest.mark.parametrize("shape", [(7, 6, 5), (40, 20, 24), (65, 33, 31), (33, 47, 62), (20, 12, 303), (70, 97, 85)])
def test_first_iterations(ok, shape, monkeypatch):
    monkeypatch.setenv("DALM_RESIDENT_SPIN", "1")
    print(f"[half pc {shape}]", flush=True)
    mesh = small_mesh(*shape, 1.2)
    g = po.make_grid(mesh)
    A = np.zeros((mesh.L, 7))
    ok.build_A(g, A)
    m = interior_mask(mesh)
    p = rand_field(mesh, 71, 1, 0.1)
    b = rand_field(mesh, 72, 1, 1.0) * m
    c = hip.Context(mesh)
    c.upload("b", b)
    work = np.zeros(9 * mesh.L)
    it, err = po.C.c_int64(), po.C.c_double()
    # a dot product's rounding is 1e-16 of it, an iteration lets a difference grow by up to 10
    for n, bound in ((1, 1e-13), (2, 1e-13), (5, 1e-10)):
        x = p.copy()
        c.upload("p", p)
        po.lib("oracle")[0].or_run_bicgstab(po.C.byref(g), po.ptr(A), po.ptr(x), po.ptr(b), po.ptr(work), hip.PC_JACOBI,
                                            1.0, 3, po.C.byref(it), n, po.C.byref(err), 0.0)
        git, gerr, st = c.run_bicgstab(hip.PC_JACOBI, 1.0, 3, n, 0.0)
        d = rel_l2(c.download("p")[m], x[m])
        print(f"  {n} iterations: pressure {d:.2e}", flush=True)
        assert git == it.value == n and st == hip.NONCONVERGED and d <= bound
        assert np.array_equal(c.download("p")[~m], p[~m])
    c.close()
