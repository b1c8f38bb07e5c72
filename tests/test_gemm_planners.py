"""The GEMM planners' choices against measured launches of every kernel.

profiles/gemm_sweep_*.csv hold the time of each configuration and K slice count
of a GEMM over its range of shapes, with weights that come from HBM and with
repeated ones.  The planners estimate times from a few fitted constants; here the
kernel they pick for each shape is looked up in the table and compared with the
fastest of that shape.  The bounds are about twice what the fit left over on
average, and its worst shape plus the 3 % that two sweeps of one kernel differ
by: a constant or a limit that is off costs more than that."""
import csv
import ctypes
from pathlib import Path

import pytest

PROFILES = Path(__file__).resolve().parents[1] / "profiles"
A_I8, A_BF16 = 0, 1
OUT_F32, OUT_BF16, OUT_F32_X4 = 0, 1, 4
SMALL, TILED_I8, TILED_B16 = 0, 1, 2


def _rows(name):
    with open(PROFILES / f"gemm_sweep_{name}.csv") as f:
        return list(csv.DictReader(line for line in f if not line.startswith("#")))


def _costs(lib, name, amode, out, planes=1):
    """{weights: [(time of the choice over the best, shape, choice)]}"""
    costs = {}
    for row in _rows(name):
        M, N, K = int(row["M"]), int(row["N"]), int(row["K"])
        us = {k: float(v) for k, v in row.items() if k not in ("weights", "M", "N", "K") and v}
        cfg, split = ctypes.c_int(), ctypes.c_int()
        kernel = lib.tlk_gemm_planned(amode, out, planes * M, N, K, ctypes.byref(cfg), ctypes.byref(split))
        choice = "small" if kernel == SMALL else f"{cfg.value}/{split.value}"
        assert kernel in (SMALL, TILED_I8, TILED_B16)
        assert choice in us, (row["weights"], M, N, K, choice)
        costs.setdefault(row["weights"], []).append((us[choice] / min(us.values()), (M, N, K), choice))
    return costs


def _check(costs, bounds):
    for weights, (mean, worst) in bounds.items():
        c = costs[weights]
        assert len(c) >= 100
        got = sum(x[0] for x in c) / len(c)
        assert got <= mean, (weights, got, sorted(c)[-5:])
        assert max(c)[0] <= worst, (weights, sorted(c)[-5:])


@pytest.fixture(scope="module")
def lib(pkg):
    return ctypes.CDLL(str(pkg.LIB_PATH))


def test_w8a16_planner(lib):
    _check(_costs(lib, "w8a16", A_BF16, OUT_BF16), {"hbm": (1.007, 1.11), "repeated": (1.013, 1.17)})


def test_w8a8_planner(lib):
    _check(_costs(lib, "w8a8", A_I8, OUT_F32), {"hbm": (1.0135, 1.26), "repeated": (1.019, 1.38)})


def test_w8a32_planner(lib):
    _check(_costs(lib, "w8a32", A_I8, OUT_F32_X4, planes=4), {"hbm": (1.011, 1.17), "repeated": (1.0115, 1.21)})
