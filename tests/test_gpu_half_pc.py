"""FP64 BiCGStab with three Jacobi sweeps, whose half-iterations are fused on rows of any
length, against the oracle: the first iterations, to the rounding of the dot products;
and against the separate kernels, bit for bit."""
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


# rows of a quad and a cell, of one quad; rows of whole quads; a last j tile and a last chunk
# of fewer cells; rows of three and two cells over; rows near the longest a block takes
# (small grids take another way unless told to)
@pytest.mark.parametrize("shape", [(7, 6, 5), (9, 30, 3), (40, 20, 24), (65, 33, 31), (33, 47, 62), (20, 12, 303),
                                   (20, 13, 383), (70, 97, 85)])
def test_first_iterations(ok, shape):
    print(f"[half pc {shape}]", flush=True)
    mesh = small_mesh(*shape, 1.2)
    g = po.make_grid(mesh)
    A = np.zeros((mesh.L, 7))
    ok.build_A(g, A)
    m = interior_mask(mesh)
    p = rand_field(mesh, 71, 1, 0.1)
    b = rand_field(mesh, 72, 1, 1.0) * m
    c, sep = hip.Context(mesh), hip.Context(mesh)
    c.set_paths(("one_launch",), ("halves",))
    sep.set_paths(("one_launch", "halves"))
    c.upload("b", b)
    sep.upload("b", b)
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
        sep.upload("p", p)
        assert sep.run_bicgstab(hip.PC_JACOBI, 1.0, 3, n, 0.0) == (git, gerr, st)
        assert np.array_equal(c.download("p"), sep.download("p"))
    assert c.paths_taken()["halves"] == sep.paths_taken()["launches"] == 3
    c.close()
    sep.close()


# a block's steps cost more than the launches saved where the blocks are few and wide
@pytest.mark.parametrize("shape, way", [((20, 12, 383), "launches"), ((30, 24, 349), "launches"), ((6, 14, 141), "launches"),
                                        ((4, 106, 53), "launches"), ((100, 98, 16), "halves"), ((39, 98, 78), "halves"),
                                        ((290, 28, 33), "halves"), ((96, 64, 64), "halves")])
def test_way_of_small_grids(shape, way):
    mesh = small_mesh(*shape, 1.2)
    c = hip.Context(mesh)
    c.upload("b", rand_field(mesh, 72, 1, 1.0) * interior_mask(mesh))
    c.run_bicgstab(hip.PC_JACOBI, 1.0, 3, 2, 0.0)
    assert c.paths_taken()[way] == 1, c.paths_taken()
    c.close()
