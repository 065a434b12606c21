"""Device allocations under guard: no solve writes behind a vector of its own
(row counts that are no multiple of the basis' padding).  Each test runs in a
process of its own, in which the probe's hipMalloc is the library's."""
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]

HEAD = """
import ctypes as C, sys
probe = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
probe.probe_fail_from.argtypes = [C.c_size_t]
for f in ("probe_count", "probe_live", "probe_damaged", "probe_bytes"):
    getattr(probe, f).restype = C.c_long
probe.probe_fail.argtypes = [C.c_long]
sys.path[:0] = [sys.argv[2], sys.argv[2] + "/tests"]
import numpy as np
import sysu_cfd_parallel_amd as s
from helpers import params, push, random_state
"""


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    so = tmp_path_factory.mktemp("alloc") / "probe.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", str(so),
                    str(ROOT / "tests/golden/device_alloc_probe.cpp"), "-ldl"], check=True)

    def run(body):
        r = subprocess.run([sys.executable, "-c", HEAD + body, str(so), str(ROOT)], capture_output=True, text=True,
                           timeout=100)
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
        return r.stdout

    return run


def test_solves_stay_inside_their_vectors(probe):
    out = probe("""
CASES = [s.channel(9, 1, 1), s.channel(5, 2, 1), s.cavity(3), s.channel(3, 2, 2), s.cavity(5, jitter=0.1),
         s.cavity(5, tets=True, jitter=0.1), s.cavity(7), s.channel(11, 7, 3, jitter=0.1, split=0.3, seed=2)]
rest = set()
for case in CASES:
    for precision, order in ((s.FP64, 0), (s.MIXED, 0), (s.MIXED, 2)):
        for pc in (s.PC_JACOBI, s.PC_ILU0):
            for graphs in (0, 1):
                p = params(restart=7, pc=pc)
                p.precision, p.graphs, p.inner_order = precision, graphs, order
                d = s.Solver(case, p)
                n = d.sizes.n_cell
                rest.add(n % 8)
                push(d, {k: v for k, v in random_state(n, d.sizes.n_bnd, d.sizes.n_face, 5).items()
                         if k in ("U", "V", "W", "P", "R", "APR", "DPDX", "RUFACE", "VISLAM")})
                d.call("build_velocity_matrix")
                d.solve_velocity(1e-8, 500)
                for k in ("bc_velocity", "cal_ru_face", "build_pressure_matrix"):
                    d.call(k)
                try:
                    d.solve_pressure(1e-6, 20)
                except s.NotConverged:
                    pass
                try:
                    d.update_energy()
                except s.NotConverged:
                    pass
                bad = probe.probe_damaged()
                assert bad == 0, (n, precision, order, pc, graphs, bad)
                d.close()
assert rest == set(range(1, 8)), rest
print("guards whole", probe.probe_count(), sorted(rest))
""")
    assert "guards whole" in out and int(out.split()[2]) > 1000


MOMENTUM = """
case = s.cavity(12, jitter=0.1, seed=3)

def context(precision, pc):
    p = params(restart=30, pc=pc)
    p.precision = precision
    d = s.Solver(case, p)
    global st
    st = random_state(d.sizes.n_cell, d.sizes.n_bnd, d.sizes.n_face, 5)
    push(d, {k: st[k] for k in ("U", "V", "W", "P", "R", "RUFACE")})
    d.call("build_velocity_matrix")
    return d

def solve(d):
    push(d, {k: st[k] for k in "UVW"})
    its = [i["iters"] for i in d.solve_velocity(1e-8, 500)]
    return its, [d.get(k) for k in "UVW"]

def same(a, b):
    return a[0] == b[0] and all(np.array_equal(x, y) for x, y in zip(a[1], b[1]))

FORMS = [(s.FP64, s.PC_JACOBI), (s.FP64, s.PC_ILU0), (s.MIXED, s.PC_JACOBI), (s.MIXED, s.PC_ILU0)]
"""


def test_an_allocation_that_fails_in_the_momentum_solve(probe):
    """Each allocation of the first solve in turn: the solve answers as ever or
    reports the error, and the next one answers as ever."""
    out = probe(MOMENTUM + """
tried = 0
for form in FORMS:
    d = context(*form)
    c0 = probe.probe_count()
    want = solve(d)
    count = probe.probe_count() - c0
    d.close()
    refused = 0
    for k in range(count):
        d = context(*form)
        probe.probe_fail(k)
        try:
            assert same(solve(d), want), (form, k)
        except s.S355Error as e:
            assert not isinstance(e, s.NotConverged) and "memory" in str(e), (form, k, e)
            refused += 1
        probe.probe_fail(-1)
        assert same(solve(d), want), (form, k)
        assert probe.probe_damaged() == 0
        d.close()
        tried += 1
    # the tables that every solve needs are missed, the common solve's are not
    assert refused <= count - 12, (form, refused, count)
print("allocations tried", tried)
""")
    assert "allocations tried" in out


def test_no_room_for_the_common_basis(probe):
    out = probe(MOMENTUM + """
rows = 12 ** 3
for precision, pc in FORMS:
    d = context(precision, pc)
    want = solve(d)
    d.close()
    d = context(precision, pc)
    live = probe.probe_live()
    # the basis of three components has 31 vectors of three times the rows
    probe.probe_fail_from(31 * 3 * rows * (8 if precision == s.FP64 else 4))
    assert same(solve(d), want)
    probe.probe_fail_from(0)
    assert same(solve(d), want)
    assert probe.probe_damaged() == 0
    d.close()
# an allocation that finds no room while the common solve holds some: given back
for precision in (s.FP64, s.MIXED):
    want = {}
    for pc in (s.PC_JACOBI, s.PC_ILU0):
        d = context(precision, pc)
        want[pc] = solve(d)
        d.close()
    d = context(precision, s.PC_JACOBI)
    assert same(solve(d), want[s.PC_JACOBI])
    live = probe.probe_live()
    p = params(restart=30, pc=s.PC_ILU0)
    p.precision = precision
    d.set_params(p)
    probe.probe_fail(0)
    assert same(solve(d), want[s.PC_ILU0])
    probe.probe_fail(-1)
    for pc in (s.PC_JACOBI, s.PC_ILU0):
        p = params(restart=30, pc=pc)
        p.precision = precision
        d.set_params(p)
        assert same(solve(d), want[pc])
    assert probe.probe_damaged() == 0
    d.close()
print("one after the other")
""")
    assert "one after the other" in out


def test_an_allocation_that_fails_in_a_run(probe):
    """... in the first iteration of a run that builds what the unsteady terms,
    the limiter and the inner order need: refused with the error, and the next
    run answers as ever."""
    out = probe("""
case = s.cavity(8, jitter=0.1, seed=3)

def made(order):
    p = params(restart=20, maxit=500)
    p.precision, p.inner_order = s.MIXED, order
    return s.Solver(case, p), p

def run(d, p):
    q = type(p).from_buffer_copy(p)
    q.steady, q.time_scheme, q.dt, q.total_time, q.max_outer_step, q.limiter = 0, 2, 0.05, 1e6, 2, 1
    d.set_params(q)
    d.call("init_flow_field")
    d.iterate(1)
    return [d.get(k) for k in "UVWP"]

for order in (1, 2):
    d, p = made(order)
    c0 = probe.probe_count()
    want = run(d, p)
    count = probe.probe_count() - c0
    d.close()
    for k in range(count):
        d, p = made(order)
        probe.probe_fail(k)
        try:
            got = run(d, p)
            assert all(np.array_equal(a, b) for a, b in zip(got, want)), (order, k)
        except s.S355Error as e:
            assert "memory" in str(e), (order, k, e)
        probe.probe_fail(-1)
        got = run(d, p)
        # (a second run starts its time step count where the first stopped)
        assert all(np.isfinite(a).all() for a in got), (order, k)
        if k % 4 == 0:
            assert probe.probe_damaged() == 0
        d.close()
print("allocations of a run", count)
""")
    assert "allocations of a run" in out


def test_mixed_ilu_holds_its_own_precision_only(probe):
    """What ILU(0) adds to a mixed context is less than what it adds to an FP64
    one: the tables and FP32 coefficients, no FP64 ones."""
    out = probe(MOMENTUM + """
added = {}
for precision in (s.FP64, s.MIXED):
    held = {}
    for pc in (s.PC_JACOBI, s.PC_ILU0):
        b0 = probe.probe_bytes()
        d = context(precision, pc)
        solve(d)
        held[pc] = probe.probe_bytes() - b0
        d.close()
    added[precision] = held[s.PC_ILU0] - held[s.PC_JACOBI]
assert 0 < added[s.MIXED] < added[s.FP64], added
print("added", added)
""")
    assert "added" in out
