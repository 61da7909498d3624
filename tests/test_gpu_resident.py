"""The one-launch solvers of small grids (csrc/resident.hip) against the oracle: SOR
iterates bit for bit, BiCGStab's first iterations to the rounding of its dot products
and its converged solution, over splits into one and several slabs, odd row lengths,
a last slab of fewer planes, and a stop by the tolerance in mid-solve.  Every test
states how the grid is split and asserts which way its solves went."""
import importlib
import threading

import numpy as np
import pytest

from helpers import interior_mask, rand_field, rel_l2, small_mesh

hip = importlib.import_module("3dalm_amd.hip")
po = importlib.import_module("pyoracle")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ok():
    return po.Kernels("oracle")


def _problem(ok, shape):
    mesh = small_mesh(*shape, 1.2)
    g = po.make_grid(mesh)
    A = np.zeros((mesh.L, 7))
    ok.build_A(g, A)
    p = rand_field(mesh, 71, 1, 0.1)
    b = rand_field(mesh, 72, 1, 1.0) * interior_mask(mesh)
    c = hip.Context(mesh)
    c.upload("p", p)
    c.upload("b", b)
    return mesh, g, A, p, b, c


# shape, blocks, planes of a block, positions per thread: one slab and several, a last one
# of fewer planes, 64 of one plane, odd rows, rows longer than two wavefronts; no block:
# grids that do not fit, solved with a launch per sweep
SOR_SHAPES = [((7, 6, 5), 1, 7, 1), ((3, 12, 33), 1, 3, 1), ((5, 3, 194), 1, 5, 3), ((14, 55, 3), 1, 14, 4),
              ((64, 10, 9), 64, 1, 1), ((65, 33, 31), 33, 2, 2), ((4, 15, 203), 4, 1, 3), ((20, 64, 64), 20, 1, 4),
              ((67, 3, 263), 34, 2, 1), ((3, 11, 269), 3, 1, 4), ((130, 20, 150), 0, 0, 0)]
BI_SHAPES = [((7, 6, 5), 1, 7, 1), ((3, 12, 33), 1, 3, 2), ((3, 13, 39), 1, 3, 3), ((19, 27, 3), 1, 19, 4),
             ((64, 10, 9), 64, 1, 1), ((105, 4, 5), 53, 2, 1), ((65, 19, 27), 33, 2, 2), ((4, 39, 39), 4, 1, 3),
             ((65, 8, 97), 33, 2, 4), ((71, 4, 131), 36, 2, 2), ((65, 33, 31), 0, 0, 0), ((20, 64, 64), 0, 0, 0),
             ((130, 20, 150), 0, 0, 0)]


def _split_is(shape, what, blocks, planes, per_thread):
    s = hip.solver_split(shape, what) or dict(blocks=0, planes=0, per_thread=0)
    assert (s["blocks"], s["planes"], s["per_thread"]) == (blocks, planes, per_thread), s
    return "one_launch" if blocks else "launches"


def _ran(c, **counts):
    """The solves went these ways and no other."""
    got = c.paths_taken()
    assert {k: v for k, v in got.items() if v and not k.startswith("copy")} == counts, got


@pytest.mark.parametrize("shape, blocks, planes, per_thread", SOR_SHAPES)
def test_sor_bits(ok, shape, blocks, planes, per_thread):
    print(f"[resident sor {shape}]", flush=True)
    way = _split_is(shape, hip.SPLIT_SOR, blocks, planes, per_thread)
    mesh, g, A, p, b, c = _problem(ok, shape)
    x, r = p.copy(), np.zeros(mesh.L)
    it, err = po.C.c_int64(), po.C.c_double()
    run = lambda n, tol: po.lib("oracle")[0].or_run_sor(po.C.byref(g), po.ptr(A), po.ptr(x), po.ptr(b), po.ptr(r), 1.3,
                                                        po.C.byref(it), n, po.C.byref(err), tol)
    run(9, 0.0)
    got = c.run_sor(1.3, 9, 0.0)
    assert got[0] == it.value == 9 and got[2] == hip.NONCONVERGED
    assert np.array_equal(c.download("p"), x)
    # the sum of N squares in another order: N u / 2 relative, and far less in the mean
    assert abs(got[1] - err.value) <= 1e-13 * err.value
    # stopped by the tolerance a few iterations on: the iterate of exactly that iteration
    tol = 0.9 * err.value
    run(500, tol)
    got = c.run_sor(1.3, 500, tol)
    assert got[0] == it.value < 500 and got[2] == hip.OK
    assert np.array_equal(c.download("p"), x)
    _ran(c, **{way: 2})
    c.close()


@pytest.mark.parametrize("pc", [hip.PC_JACOBI, hip.PC_SOR])
@pytest.mark.parametrize("shape, blocks, planes, per_thread", BI_SHAPES)
def test_bicgstab(ok, shape, blocks, planes, per_thread, pc):
    print(f"[resident bicgstab {shape} pc {pc}]", flush=True)
    way = _split_is(shape, hip.SPLIT_BICGSTAB, blocks, planes, per_thread)
    mesh, g, A, p, b, c = _problem(ok, shape)
    m = interior_mask(mesh)
    lib = po.lib("oracle")[0]
    work = np.zeros(9 * mesh.L)
    it, err = po.C.c_int64(), po.C.c_double()
    for n, tol in ((2, 0.0), (5000, 1e-13)):
        x = p.copy()
        c.upload("p", p)
        lib.or_run_bicgstab(po.C.byref(g), po.ptr(A), po.ptr(x), po.ptr(b), po.ptr(work), pc, 1.1, 2, po.C.byref(it), n,
                            po.C.byref(err), tol)
        git, gerr, st = c.run_bicgstab(pc, 1.1, 2, n, tol)
        d = rel_l2(c.download("p")[m], x[m])
        print(f"  {git} against {it.value} iterations, pressure {d:.2e}", flush=True)
        if n == 2:  # the rounding of the dot products, not yet amplified by the iteration
            assert git == 2 and st == hip.NONCONVERGED and d <= 1e-13
            assert abs(gerr - err.value) <= 1e-12 * err.value
        else:  # both within 1e-13 of the same solution
            assert st == hip.OK and gerr <= 1e-13 and d <= 1e-10
        assert np.array_equal(c.download("p")[~m], p[~m])
    _ran(c, **{way: 2})
    c.close()


def test_two_contexts_at_once(ok):
    """Solves of two contexts in one launch each, from two threads, over and over: the
    oracle's iterates in both."""
    bad = []

    def work(shape):
        try:
            mesh, g, A, p, b, c = _problem(ok, shape)
            x, r = p.copy(), np.zeros(mesh.L)
            it, err = po.C.c_int64(), po.C.c_double()
            po.lib("oracle")[0].or_run_sor(po.C.byref(g), po.ptr(A), po.ptr(x), po.ptr(b), po.ptr(r), 1.3,
                                           po.C.byref(it), 60, po.C.byref(err), 0.0)
            for _ in range(20):
                c.upload("p", p)
                c.run_sor(1.3, 60, 0.0)
                assert np.array_equal(c.download("p"), x)
            _ran(c, one_launch=20)
            c.close()
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            bad.append(e)

    ts = [threading.Thread(target=work, args=(s,)) for s in ((65, 33, 31), (20, 64, 64))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_breakdown_and_nonfinite():
    """A zero residual is a breakdown before the first iteration; a NaN in b ends the
    solve after one (as the kernels of larger grids do)."""
    mesh = small_mesh(12, 9, 10, 1.2)
    c = hip.Context(mesh)
    it, err, st = c.run_bicgstab(hip.PC_JACOBI, 1.0, 3, 50, 1e-8)
    assert (it, err, st) == (0, 0.0, hip.BREAKDOWN)
    b = np.zeros(mesh.L)
    b[np.flatnonzero(interior_mask(mesh))[5]] = np.nan
    c.upload("b", b)
    it, err, st = c.run_sor(1.2, 50, 1e-8)
    assert it == 1 and st == hip.NONFINITE
    c.upload("p", np.zeros(mesh.L))
    it, err, st = c.run_bicgstab(hip.PC_JACOBI, 1.0, 3, 50, 1e-8)
    assert it == 1 and st == hip.NONFINITE
    _ran(c, one_launch=3)
    c.close()


def test_falls_back_when_a_wait_ends(ok, monkeypatch):
    """A block that gives up waiting (a limit of one poll, set by the environment) ends
    the launch, and the solve runs with one launch per sweep from the same start: the
    same iterates, then and for the context's later solves."""
    monkeypatch.setenv("DALM_RESIDENT_SPIN", "1")
    mesh, g, A, p, b, c = _problem(ok, (40, 20, 24))
    x, r = p.copy(), np.zeros(mesh.L)
    it, err = po.C.c_int64(), po.C.c_double()
    for n in (4, 3):
        po.lib("oracle")[0].or_run_sor(po.C.byref(g), po.ptr(A), po.ptr(x), po.ptr(b), po.ptr(r), 1.3, po.C.byref(it), n,
                                       po.C.byref(err), 0.0)
        got = c.run_sor(1.3, n, 0.0)
        assert got[0] == n and np.array_equal(c.download("p"), x)
    _ran(c, given_up=1, launches=2)
    c.close()


@pytest.mark.parametrize("way", ["one_launch", "launches"])
@pytest.mark.parametrize("shape", [(7, 6, 5), (64, 10, 9), (65, 33, 31), (4, 15, 203), (20, 64, 64), (67, 3, 263)])
def test_sor_mixed(shape, way):
    """The precision form's SOR of one step, in one launch and with a launch per sweep
    (as on larger grids), against the FP64 oracle's: after the same
    number of iterations (a multiple of 8) the pressure and the residual differ by the
    FP32 rounding of the corrections, 2^-24 of each (allowed: ten of them), and by that of
    the FP32 predictor in b."""
    cases, solver = importlib.import_module("3dalm_amd.cases"), importlib.import_module("3dalm_amd.solver")
    print(f"[sor mixed {shape} {way}]", flush=True)
    off = ("one_launch",) if way == "launches" else ()
    case = cases.case_c1(*shape, steps=1)
    case.max_it, case.tol = 24, 0.0
    o, s = po.OracleSolver(case), solver.Solver(case, hip.MIXED)
    s.ctx.set_paths(off)
    try:
        so, sm = o.step(), s.step()
        assert sm["it"] == so["it"] == 24
        m = interior_mask(case.mesh)
        d = rel_l2(s.field("p")[m], o.field("p")[m])
        print(f"  pressure {d:.2e}, err {sm['err']:.6e} against {so['err']:.6e}", flush=True)
        assert d <= 10 * 2.0 ** -24 * 10 and abs(sm["err"] - so["err"]) <= 1e-5 * so["err"]
        _ran(s.ctx, **{way: 1})
        case.max_it, case.tol = 2000, 0.5 * so["err"]
        s2 = solver.Solver(case, hip.MIXED)
        s2.ctx.set_paths(off)
        st = s2.step()
        assert st["it"] % 8 == 0 and st["it"] < 2000 and st["err"] <= case.tol
        _ran(s2.ctx, **{way: 1})
        s2.close()
    finally:
        s.close()


@pytest.mark.parametrize("off", [(), ("one_launch",)])
@pytest.mark.parametrize("shape", [(7, 6, 5), (64, 10, 9), (65, 33, 31), (12, 8, 8)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_sor_mixed_ghost_pressure(shape, value, off):
    """A pressure that is not finite in a ghost cell next to the interior ends the
    precision form's SOR as non-finite (its zero coefficient times it is no number), in
    one launch as with a launch per sweep; in an edge of the box no cell reads it."""
    cases, solver = importlib.import_module("3dalm_amd.cases"), importlib.import_module("3dalm_amd.solver")
    print(f"[resident sor mixed ghost {shape} {value}]", flush=True)
    case = cases.case_c1(*shape, steps=1)
    case.max_it, case.tol = 16, 0.0
    g = case.mesh.gc
    n = [q + 2 * g for q in shape]
    mid = [g + q // 2 for q in shape]
    ghosts = [(i, *mid[1:]) for i in (g - 1, n[0] - g)] + [(mid[0], j, mid[2]) for j in (g - 1, n[1] - g)] + \
        [(*mid[:2], k) for k in (g - 1, n[2] - g)]
    for ghost, want in [(q, hip.NONFINITE) for q in ghosts] + [((g - 1, g - 1, mid[2]), hip.NONCONVERGED)]:
        s = solver.Solver(case, hip.MIXED)
        s.ctx.set_paths(off)
        p = np.zeros(n)
        p[ghost] = value
        s.ctx.upload("p", p.reshape(-1))
        try:
            status = s.step()["status"]
        finally:
            s.close()
        assert status == want, (ghost, status)


@pytest.mark.parametrize("method", ["SOR mixed", "SOR", "BiCG"])
def test_pressure_like_an_empty_slot(method):
    """A pressure whose bits are the mark of an empty exchange slot: the solve is
    non-finite, and no block waits for the value."""
    cases, solver = importlib.import_module("3dalm_amd.cases"), importlib.import_module("3dalm_amd.solver")
    print(f"[resident empty mark {method}]", flush=True)
    case = cases.case_c1(64, 10, 9, steps=1)
    case.method, case.pc, case.max_it, case.tol = method.split()[0], "Jacobi", 16, 0.0
    g = case.mesh.gc
    p = np.zeros([n + 2 * g for n in (64, 10, 9)])
    p.view(np.uint64)[g + 20, g + 3, g + 4] = 0x7FF4DEADBEEF0001
    s = solver.Solver(case, hip.MIXED if method.endswith("mixed") else hip.FP64)
    try:
        s.ctx.upload("p", p.reshape(-1))
        assert s.step()["status"] == hip.NONFINITE
        _ran(s.ctx, one_launch=1)
    finally:
        s.close()


@pytest.mark.parametrize("solve, way", [
    (lambda c: c.run_sor(1.3, 20000, 1.0), "one_launch"), (lambda c: c.run_sor(1.3, 300000, 1.0), "launches"),
    (lambda c: c.run_bicgstab(hip.PC_SOR, 1.1, 5, 20000, 1.0), "one_launch"),
    (lambda c: c.run_bicgstab(hip.PC_JACOBI, 1.0, 3, 20001, 1.0), "one_launch"),
    (lambda c: c.run_bicgstab(hip.PC_SOR, 1.1, 60, 20000, 1.0), "launches"),
    (lambda c: c.run_bicgstab(hip.PC_JACOBI, 1.0, 3, 2**62, 1.0), "launches")])
def test_way_of_long_solves(ok, solve, way):
    """The work that a solve may take at most decides, not its cap of iterations alone."""
    mesh, g, A, p, b, c = _problem(ok, (12, 9, 10))
    solve(c)
    _ran(c, **{way: 1})
    c.close()
