"""ILU(0) sweep plans at the bound on their merged rows' entries: a pattern past it
is planned level by level, not refused."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

import sysu_cfd_parallel_amd as s

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    so = tmp_path_factory.mktemp("ilu") / "probe.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-pthread", "-o", str(so),
                    str(ROOT / "tests/golden/ilu_plan_limit_probe.cpp"),
                    str(ROOT / "sysu_cfd_parallel_amd/csrc/device/ilu_plan.cpp")], check=True)
    lib = C.CDLL(str(so))
    lib.probe_plan.argtypes = [C.c_int] + [C.c_void_p] * 3 + [C.c_int, C.c_int, C.c_long, C.c_void_p]

    def run(mesh, upper, levels, most):
        h = s.HostMesh(mesh)
        ptr, col, diag = h.ints("CSR_ROWPTR"), h.ints("CSR_COL"), h.ints("CSR_DIAG")
        out = np.zeros(4, dtype=np.int64)
        ip = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
        assert lib.probe_plan(len(ptr) - 1, ip(ptr), ip(col), ip(diag), upper, levels, most, ip(out)) == 0
        return out.tolist()

    return run


@pytest.mark.parametrize("upper", [0, 1])
@pytest.mark.parametrize("mesh", [lambda: s.channel(40, 4, 4, jitter=0.1), lambda: s.cavity(6, tets=True, jitter=0.1)])
def test_past_the_bound_nothing_is_merged(plan, mesh, upper):
    case = mesh()
    n = s.HostMesh(case).sizes.n_cell
    by_level, merged = plan(case, upper, 1, 1 << 30), plan(case, upper, 8, 1 << 30)
    assert by_level[2] == 0 and merged[2] > 0 and merged[0] < by_level[0]
    # the entries of the merged rows lie between these
    assert plan(case, upper, 8, n) == by_level
    assert plan(case, upper, 8, 200 * n) == merged
    lo, hi = n, 200 * n
    while hi - lo > 1:  # one bound divides the two plans
        mid = (lo + hi) // 2
        got = plan(case, upper, 8, mid)
        assert got in (by_level, merged)
        lo, hi = (mid, hi) if got == by_level else (lo, mid)
    assert plan(case, upper, 8, lo) == by_level and plan(case, upper, 8, hi) == merged
