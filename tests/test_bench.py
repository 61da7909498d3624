"""The byte counts behind bench.py's rooflines, by the way the kernels run."""
import importlib

import pytest

bench = importlib.import_module("bench")


@pytest.mark.parametrize("rows256, update, p, s", [(True, 32, 36, 24), (False, 64, 28, 20)])
def test_probe_bytes(rows256, update, p, s):
    """Rows of 256 cells leave x (and the precision form r) to other kernels: the FP64
    update then moves s, t, r0, r; otherwise also x twice and both z."""
    assert [bench.probe_bytes(k, rows256) for k in ("update", "half_p_mixed", "half_s_mixed")] == [update, p, s]


@pytest.mark.parametrize("rows256, halves, fp64, mixed", [(True, True, 170, 70), (False, True, 184, 88),
                                                          (False, False, 280, 148), (True, False, 280, 148)])
def test_step_bytes(rows256, halves, fp64, mixed):
    """Bytes of an iteration: the sums over its kernels."""
    b = bench.step_bytes(rows256, halves)
    assert (b["fp64"]["per_it"], b["mixed"]["per_it"]) == (fp64, mixed)
    if halves and not rows256:
        k = {n: bench.probe_bytes(n, False) for n in bench.PROBE_BYTES_OTHER}
        assert fp64 == k["half_p"] + 2 * k["spmv"] + k["half_s"] + k["update"]
        assert mixed == k["half_p_mixed"] + k["half_s_mixed"] + k["update_mixed"]
