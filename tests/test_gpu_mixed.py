"""The precision form (FP32 cell stencils, FP32 BiCGStab vectors and preconditioner
sweeps; FP64 face fluxes, pressure, dot products, norms and the residual
replacements that end every solve on the true FP64 residual) against the FP64
oracle.

Stated tolerances, against FP64:
  * every step ends with the FP64 residual test met: err <= tol, and therefore
    avg div <= 1e-6 (it is dt * max_diag * err by the projection identity);
  * turbine power within 0.1 % of the FP64 oracle;
  * velocity within 1e-4 relative L2 of the FP64 oracle over the first steps
    (FP32 storage of U rounds at 6e-8 per step);
  * pressure: the residual test err <= 1e-8 leaves a smooth pressure error that it
    hardly sees (the FP64 oracle at 1e-8 is 1.2e-3 from its own 1e-13 solution at
    64x32x32), so both are measured from the oracle's 1e-13 solution and the
    precision form may be at most ten times as far from it as the FP64 oracle at
    the same tolerance (plus 1e-5).
"""
import importlib

import numpy as np
import pytest

from helpers import interior_mask, rel_l2

hip = importlib.import_module("3dalm_amd.hip")
cases = importlib.import_module("3dalm_amd.cases")
solver = importlib.import_module("3dalm_amd.solver")
po = importlib.import_module("pyoracle")

pytestmark = pytest.mark.gpu


def _rows256():
    """A rotor case with rows of 256 interior cells (32x16x256 on a 4x2x8 box)."""
    m = cases.make_mesh(32, 16, 256, ((0.0, 4.0), (-1.0, 1.0), (0.0, 8.0)), 1.2, 1.2)
    return cases.Case("rows256", m, method="BiCG", pc="Jacobi", pc_it=3, tol=1e-8, max_it=1000, steps=4,
                      turbine=cases.default_turbine(R=0.5, tower=4.0), sites=[cases.TurbineSite((1.0, 0.0, 0.0), 12.0)],
                      ap_per_blade=4, width=0.25)


def _rows384():
    """Rows of 384 interior cells (16x8x384 on a 4x2x12 box): the four-cell kernels
    with a half-empty second tile of lanes per row, unfused."""
    m = cases.make_mesh(16, 8, 384, ((0.0, 4.0), (-1.0, 1.0), (0.0, 12.0)), 1.2, 1.2)
    return cases.Case("rows384", m, method="BiCG", pc="Jacobi", pc_it=3, tol=1e-8, max_it=1000, steps=4,
                      turbine=cases.default_turbine(R=0.5, tower=4.0), sites=[cases.TurbineSite((1.0, 0.0, 0.0), 12.0)],
                      ap_per_blade=4, width=0.25)


@pytest.mark.parametrize("builder,steps", [
    (lambda: cases.case_c2(32, 16, 16, steps=6, ap_per_blade=8), 6),
    (lambda: cases.case_c2(64, 32, 32, steps=4, ap_per_blade=16), 4),
    # rows of 256 cells: the fused half-iterations
    (lambda: _rows256(), 4),
    # rows of 384 cells: the four-cell kernels with a partial tile
    (lambda: _rows384(), 4),
])
def test_mixed_against_fp64_oracle(builder, steps):
    case = builder()
    print(f"[mixed {case.mesh.interior} steps={steps}]", flush=True)
    o = po.OracleSolver(case)
    s = solver.Solver(case, hip.MIXED)
    try:
        for n in range(steps):
            so, sm = o.step(), s.step()
            assert sm["status"] == hip.OK, sm
            assert sm["err"] <= case.tol
            assert sm["avg_div"] <= 1e-6
            assert abs(sm["power"][0] - case.sites[0].rot_speed * so["torque"][0]) <= \
                1e-3 * abs(case.sites[0].rot_speed * so["torque"][0])
        m = interior_mask(case.mesh)
        eu = rel_l2(s.field("U")[m], o.field("U")[m])
        t = builder()
        t.tol, t.max_it = 1e-13, 20000
        ot = po.OracleSolver(t)
        for _ in range(steps):
            ot.step()
        truth = ot.field("p")[m]
        ep = rel_l2(s.field("p")[m], truth)
        ep64 = rel_l2(o.field("p")[m], truth)
        print(f"mixed vs fp64: U {eu:.2e}; p from the 1e-13 solution: mixed {ep:.2e}, fp64 {ep64:.2e}",
              flush=True)
        assert eu <= 1e-4
        assert ep <= 10 * ep64 + 1e-5
    finally:
        s.close()


def test_mixed_sor_pc_and_c1():
    c = cases.case_c1(20, 12, 12, steps=3)
    c.method, c.pc, c.pc_it, c.pc_omega, c.tol = "BiCG", "SOR", 2, 1.2, 1e-9
    o = po.OracleSolver(c)
    s = solver.Solver(c, hip.MIXED)
    try:
        for _ in range(3):
            so, sm = o.step(), s.step()
            assert sm["err"] <= c.tol and sm["avg_div"] <= 1e-6
        m = interior_mask(c.mesh)
        assert rel_l2(s.field("U")[m], o.field("U")[m]) <= 1e-4
    finally:
        s.close()


@pytest.mark.parametrize("interior,tol", [((20, 12, 12), 1e-6), ((48, 24, 24), 1e-8)])
def test_mixed_sor_method(interior, tol):
    """Method SOR in the precision form: FP32 red-black sweeps on the correction,
    refined on the FP64 residual every 8 iterations.  Every solve meets the
    reference's test on the true FP64 residual, needs at most one refinement
    (8 iterations) more than the FP64 oracle's SOR, and U stays within 1e-4 of it."""
    c = cases.case_c1(*interior, steps=3)
    c.tol = tol
    print(f"[mixed SOR {interior} tol={tol}]", flush=True)
    o = po.OracleSolver(c)
    s = solver.Solver(c, hip.MIXED)
    try:
        for _ in range(3):
            so, sm = o.step(), s.step()
            assert sm["it"] % 8 == 0 and sm["it"] <= so["it"] + 8, (sm["it"], so["it"])
            if so["it"] >= c.max_it:  # the FP64 solve stopped at the cap: so must this one, as close
                assert sm["it"] == c.max_it and sm["err"] <= 1.001 * so["err"], (sm, so)
            else:
                assert sm["status"] == hip.OK, sm
                assert sm["err"] <= tol and sm["avg_div"] <= 1e-6
        m = interior_mask(c.mesh)
        assert rel_l2(s.field("U")[m], o.field("U")[m]) <= 1e-4
    finally:
        s.close()


@pytest.mark.parametrize("on", [(), ("halves",)])
@pytest.mark.parametrize("builder,cap", [(build, cap) for cap in (40, 41, 42, 43) for build in (
    lambda: cases.case_c2(48, 24, 24, steps=3, ap_per_blade=8), lambda: _rows256())])
def test_mixed_passes_and_fp64_hand_over(builder, cap, on):
    """The precision form's recovery paths: with every FP32 pass cut short after
    40 to 43 iterations (dalm_set_fp32_pass_cap), a pass that ends far
    above the tolerance is restarted from the true residual and one that ends
    within 30x of it is handed over to FP64; every solve must still end on the
    true residual with the step matching the FP64 oracle.  After an odd number of
    iterations p and q are in the other buffers of their pairs, in the FP32 halves
    and (switched on for this size) in the FP64 ones that go on from them.  Also with rows of 256
    cells (the fused half-iterations, whose pressure updates are applied eight
    iterations' at a time: caps of 40 to 43 iterations end passes with different
    numbers of them outstanding)."""
    case = builder()
    case.steps = 3
    case.tol, case.max_it = 1e-10, 4000
    print(f"[mixed recovery paths {case.mesh.interior} cap {cap}]", flush=True)
    o = po.OracleSolver(case)
    s = solver.Solver(case, hip.MIXED)
    s.ctx.set_fp32_pass_cap(cap)
    s.ctx.set_paths((), on)
    try:
        in_fp64 = 0
        for _ in range(3):
            so, sm = o.step(), s.step()
            print(f"step {sm['step']}: it {sm['it']} err {sm['err']:.3e} {s.ctx.last_solve_info()}", flush=True)
            assert sm["status"] == hip.OK, sm
            assert sm["err"] <= case.tol
            assert sm["it"] > cap  # the cut-short pass was followed by more work
            in_fp64 += s.ctx.last_solve_info()[1]
            assert abs(sm["power"][0] - case.sites[0].rot_speed * so["torque"][0]) <= \
                1e-3 * abs(case.sites[0].rot_speed * so["torque"][0])
        assert in_fp64 > 0
        m = interior_mask(case.mesh)
        assert rel_l2(s.field("U")[m], o.field("U")[m]) <= 1e-4
    finally:
        s.close()


# grids whose dot products are summed by whole units, with their k tiles
UNIT_SUMS = {(131, 130, 125): 1, (129, 127, 132): 1, (81, 154, 184): 3, (71, 67, 442): 7}


@pytest.mark.parametrize("interior, iters", [(s, n) for s in ((9, 10, 13), (33, 30, 87), (40, 24, 64), (70, 13, 30),
                                                              (82, 20, 643), (12, 10, 256)) for n in (1, 2, 9)] +
                         [((131, 130, 125), 2), ((129, 127, 132), 2), ((50, 150, 283), 2),
                          ((500, 512, 3), 2), ((81, 154, 184), 2), ((71, 67, 442), 2)])
def test_fused_half_iterations(interior, iters):
    """The fused half-iterations on rows of any length (quads that reach beyond the row,
    rows cut into k tiles, a last j tile and a last plane chunk of fewer cells, rows of 256
    cells; from two million cells on chunks and tiles of whole units, with one and several
    k tiles; rows of one quad in
    blocks of as many rows as their LDS takes): the pressure after the first iterations of a step against the FP64
    oracle's.  An iteration rounds each vector about 16 times to FP32 (2^-24), and
    BiCGStab lets that grow by up to a factor 3 per iteration; a cell, row or update left
    out is off by more than 1e-3.  After 9 iterations one group of eight pressure updates
    has been applied and one is outstanding."""
    if interior in UNIT_SUMS:
        split = hip.solver_split(interior, hip.SPLIT_HALVES_MIXED)
        assert split["unit_sums"] and split["tk"] == UNIT_SUMS[interior], split
    case = cases.case_c1(*interior, steps=1)
    case.method, case.pc, case.pc_it, case.max_it, case.tol = "BiCG", "Jacobi", 3, iters, 0.0
    print(f"[fused halves {interior} {iters} iterations]", flush=True)
    o, s = po.OracleSolver(case), solver.Solver(case, hip.MIXED)
    try:
        so, sm = o.step(), s.step()
        assert sm["it"] == so["it"] == iters
        m = interior_mask(case.mesh)
        d = rel_l2(s.field("p")[m], o.field("p")[m])
        print(f"  pressure {d:.2e}", flush=True)
        assert d <= 16 * 2.0 ** -24 * 3.0 ** (iters - 1) * 4
        outside = s.field("p")[~m]
        assert np.all(np.isfinite(outside))
        assert s.ctx.paths_taken()["halves"] == 1
    finally:
        s.close()


@pytest.mark.parametrize("interior", [(9, 10, 13), (33, 30, 87), (70, 13, 30), (12, 10, 256), (8, 3, 40)])
@pytest.mark.parametrize("sweeps, iters", [(3, 1), (3, 2), (3, 9), (1, 2), (2, 2), (4, 5)])
def test_separate_kernels(interior, sweeps, iters):
    """The update, sweeps and product as kernels of their own (any number of sweeps but
    three, rows of fewer than four cells along j, three sweeps switched off), as
    test_fused_half_iterations: the same roundings, a few more with a fourth sweep."""
    case = cases.case_c1(*interior, steps=1)
    case.method, case.pc, case.pc_it, case.max_it, case.tol = "BiCG", "Jacobi", sweeps, iters, 0.0
    print(f"[separate kernels {interior} {sweeps} sweeps {iters} iterations]", flush=True)
    o, s = po.OracleSolver(case), solver.Solver(case, hip.MIXED)
    s.ctx.set_paths(("halves",))
    try:
        so, sm = o.step(), s.step()
        assert sm["it"] == so["it"] == iters and s.ctx.paths_taken()["launches"] == 1
        m = interior_mask(case.mesh)
        d = rel_l2(s.field("p")[m], o.field("p")[m])
        print(f"  pressure {d:.2e}", flush=True)
        assert d <= 16 * 2.0 ** -24 * 3.0 ** (iters - 1) * 4
    finally:
        s.close()
