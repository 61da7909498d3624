"""Fields copied out of the device: every byte, at sizes around the ways they take."""
import importlib
import threading

import numpy as np
import pytest

cases = importlib.import_module("3dalm_amd.cases")
hip = importlib.import_module("3dalm_amd.hip")

pytestmark = pytest.mark.gpu


def _round_trip(interior, precision, seed, off=(), way=None):
    mesh = cases.case_c1(*interior, steps=1).mesh
    ctx = hip.Context(mesh, precision)
    ctx.set_paths(off)
    try:
        rng = np.random.default_rng(seed)
        for _ in range(2):  # the second pass finds the slots there
            for name, nc in (("p", 1), ("U", 3), ("nut", 1)):
                a = rng.standard_normal((mesh.L, nc) if nc > 1 else mesh.L)
                ctx.upload(name, a)
                want = a.astype(np.float32).astype(np.float64) if precision == hip.MIXED and name != "p" else a
                assert np.array_equal(ctx.download(name), want), name
        assert ctx.L.dalm_last_error(ctx.h) == b""
        assert way is None or ctx.paths_taken()[way] == 6, ctx.paths_taken()
    finally:
        ctx.close()


# one and three components below and above the plain copies' 2^18 values, one slot, slots of
# a quarter, full slots with a remainder
@pytest.mark.parametrize("interior, way", [((20, 12, 12), "copy_plain"), ((70, 33, 31), None),
                                           ((97, 49, 46), "copy_slots"), ((150, 90, 77), "copy_slots")])
@pytest.mark.parametrize("precision", [hip.FP64, hip.MIXED])
def test_copy_out(interior, way, precision):
    print(f"[copy out {interior} {precision}]", flush=True)
    _round_trip(interior, precision, 7, way=way)


@pytest.mark.parametrize("precision", [hip.FP64, hip.MIXED])
def test_copy_out_without_pinned_memory(precision):
    """Where the host grants no pinned memory the plain copies bring the same bytes."""
    _round_trip((97, 49, 46), precision, 7, off=("copy_slots",), way="copy_plain")


def test_copy_out_from_two_threads():
    """Two contexts copied out at once, each by its own thread."""
    bad = []

    def work(seed):
        try:
            _round_trip((97, 49, 46), hip.FP64, seed)
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            bad.append(e)

    ts = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
