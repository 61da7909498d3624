"""How the kernels that keep a part of the grid on chip split a grid (host arithmetic, no
GPU): on every size each launch fits a compute unit and its tiles cover the grid."""
import importlib
import random

import pytest

hip = importlib.import_module("3dalm_amd.hip")

LDS = 160 * 1024       # of a compute unit
HALF_STATIC = 640      # the precision halves' block sums beside the dynamic LDS
RES_STATIC = 1024      # the one-launch solvers' exchange


def _sizes():
    """Few cells along k with many rows (a block then takes hundreds of rows), and sizes
    spread over the logarithm of each extent."""
    out = [(500, 512, 3), (1000, 700, 4), (512, 531, 3), (1024, 568, 3), (16, 1500, 8), (3, 3, 3), (3, 4000, 3)]
    out += [(nx, ny, nz) for nz in (3, 4, 5, 7, 8, 9) for ny in (300, 520, 760, 1100) for nx in (40, 600)]
    out += [(20, 12, nz) for nz in (255, 256, 257, 303, 304, 305, 382, 383, 384, 385, 700)]
    rng = random.Random(5)
    out += [tuple(round(3 * (700 / 3) ** rng.random()) for _ in range(3)) for _ in range(300)]
    return [s for s in out if s[0] * s[1] * s[2] < 1 << 28]


@pytest.mark.parametrize("what", [hip.SPLIT_HALVES, hip.SPLIT_HALVES_MIXED])
@pytest.mark.parametrize("ncu", [256, 32])
def test_half_splits(what, ncu):
    mixed = what == hip.SPLIT_HALVES_MIXED
    lag, static = (3, HALF_STATIC) if mixed else (2, 0)
    taken = 0
    for nx, ny, nz in _sizes():
        s = hip.solver_split((nx, ny, nz), what, ncu)
        if s is None:
            continue
        taken += 1
        own = s["rows"] - 2 * lag
        quads = s["quads"] if s["tk"] == 1 else s["quads"] - 2
        chunks = -(-nx // s["planes"])
        assert s["lds"] + static <= LDS, (nx, ny, nz, s)
        assert s["rows"] * s["quads"] <= s["threads"] <= (1024 if mixed and nz == 256 else 768), (nx, ny, nz, s)
        assert s["threads"] % 64 == 0 and own >= 4, (nx, ny, nz, s)
        assert own * s["tj"] >= ny and 4 * quads * s["tk"] >= nz, (nx, ny, nz, s)
        assert s["blocks"] == s["tj"] * s["tk"] * chunks, (nx, ny, nz, s)
    assert taken > 100


@pytest.mark.parametrize("what", [hip.SPLIT_SOR, hip.SPLIT_BICGSTAB])
@pytest.mark.parametrize("ncu", [256, 32])
def test_one_launch_splits(what, ncu):
    most = {1: 1024, 2: 768, 3: 512, 4: 512}
    taken = 0
    for nx, ny, nz in _sizes():
        s = hip.solver_split((nx, ny, nz), what, ncu)
        if s is None:
            continue
        taken += 1
        assert s["lds"] + RES_STATIC <= LDS and s["threads"] <= most[s["per_thread"]], (nx, ny, nz, s)
        assert s["blocks"] <= max(1, min(64, ncu // 4)) and s["blocks"] * s["planes"] >= nx, (nx, ny, nz, s)
        assert (s["blocks"] - 1) * s["planes"] < nx, (nx, ny, nz, s)
        assert s["positions"] == ((nz + 1) // 2 if what == hip.SPLIT_SOR else nz)
        assert s["rows"] * s["per_thread"] >= s["planes"] * ny, (nx, ny, nz, s)
        assert s["rows"] * s["positions"] <= s["threads"], (nx, ny, nz, s)
    assert taken > 20
