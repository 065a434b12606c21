"""ILU(0) sweeps by groups of levels: the host plan against a plain triangular
solve (CPU), and the device's first preconditioned step against the oracle's
(GPU), at the edges of groups, classes of term counts and launch sizes."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

import sysu_cfd_parallel_amd as s
from helpers import params, push, random_state, rel_err

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    so = tmp_path_factory.mktemp("ilu") / "probe.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-pthread", "-o", str(so),
                    str(ROOT / "tests/golden/ilu_plan_probe.cpp"),
                    str(ROOT / "sysu_cfd_parallel_amd/csrc/device/ilu_plan.cpp")], check=True)
    return C.CDLL(str(so))


def random_pattern(rng, sizes, links):
    """Symmetric patterns of several cases (rows of each consecutive), sorted columns."""
    sets, a = [], 0
    for n in sizes:
        rows = [{i} for i in range(n)]
        for i in range(n):
            for j in rng.integers(max(0, i - 40), i + 1, size=rng.integers(0, links + 1)):
                rows[i].add(int(j))
                rows[int(j)].add(i)
        sets += [sorted(a + j for j in r) for r in rows]
        a += n
    ptr = np.concatenate([[0], np.cumsum([len(r) for r in sets])]).astype(np.int32)
    return ptr, np.concatenate([np.asarray(r) for r in sets]).astype(np.int32)


def mesh_pattern(case):
    h = s.HostMesh(case)
    return h.ints("CSR_ROWPTR"), h.ints("CSR_COL")


PATTERNS = {
    "single": lambda rng: (random_pattern(rng, [1], 0), [1]),
    "diagonal": lambda rng: (random_pattern(rng, [70], 0), [70]),
    "chain": lambda rng: (chain_pattern(60), [60]),
    "random": lambda rng: (random_pattern(rng, [400], 3), [400]),
    "dense_rows": lambda rng: (random_pattern(rng, [200], 9), [200]),
    "batch": lambda rng: (random_pattern(rng, [37, 1, 150, 64], 3), [37, 1, 150, 64]),
    "hexes": lambda rng: (mesh_pattern(s.cavity(9)), None),
    "tets": lambda rng: (mesh_pattern(s.cavity(5, tets=True, jitter=0.1)), None),
    "split": lambda rng: (mesh_pattern(s.channel(12, 6, 9, jitter=0.1, split=0.2)), None),
}


def chain_pattern(n):
    rows = [[j for j in (i - 1, i, i + 1) if 0 <= j < n] for i in range(n)]
    return (np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32),
            np.concatenate([np.asarray(r) for r in rows]).astype(np.int32))


def ip(a):
    return a.ctypes.data_as(C.c_void_p)


@pytest.mark.parametrize("name", sorted(PATTERNS))
@pytest.mark.parametrize("levels,rows", [(1, 65536), (2, 65536), (6, 65536), (8, 65536), (6, 40), (4, 1)])
@pytest.mark.parametrize("upper", [0, 1])
def test_sweep_plan_equals_the_triangular_solve(probe, name, levels, rows, upper):
    rng = np.random.default_rng(3)
    (ptr, col), sizes = PATTERNS[name](rng)
    n = len(ptr) - 1
    cases = np.concatenate([[0], np.cumsum(sizes or [n])]).astype(np.int32)
    row = np.repeat(np.arange(n), np.diff(ptr))
    diag = np.flatnonzero(col == row).astype(np.int32)
    # off-diagonals of a row sum to at most 0.9 of its pivot: the solve's
    # condition number is below 20 and its rounding below 1e-13
    lu = rng.uniform(-1.0, 1.0, len(col)) * 0.9 / np.maximum(np.diff(ptr)[row] - 1, 1)
    lu[diag] = rng.uniform(1.0, 1.5, n)
    r = rng.standard_normal(n)
    order = np.arange(n, dtype=np.int32) if not upper else rng.permutation(n).astype(np.int32)
    z, out = np.zeros(n), np.zeros(6, dtype=np.int64)
    assert probe.probe_sweep(n, ip(ptr), ip(col), ip(diag), upper, len(cases) - 1, ip(cases), levels, rows, ip(order),
                             ip(lu), ip(r), ip(z), ip(out)) == 0
    ref = np.zeros(n)
    for i in (range(n - 1, -1, -1) if upper else range(n)):
        lo, hi = (diag[i] + 1, ptr[i + 1]) if upper else (ptr[i], diag[i])
        ref[i] = r[i] - lu[lo:hi] @ ref[col[lo:hi]]
        if upper:
            ref[i] /= lu[diag[i]]
    assert out[5] == 0
    assert np.max(np.abs(z - ref)) <= 1e-13 * np.max(np.abs(ref))
    if levels == 1:
        assert out[4] == 0  # nothing merged
    if name == "chain" and levels == 6 and rows == 65536:
        assert out[0] == 10  # 60 levels, 6 to a launch
    # a case of a batch sums what it sums alone
    if name == "batch":
        for k in range(len(cases) - 1):
            a, e = cases[k], cases[k + 1]
            sub = slice(ptr[a], ptr[e])
            p1 = np.ascontiguousarray(ptr[a:e + 1] - ptr[a])
            c1 = np.ascontiguousarray(col[sub] - a)
            d1 = np.ascontiguousarray(diag[a:e] - ptr[a])
            o1 = np.ascontiguousarray(order[(order >= a) & (order < e)] - a)
            l1, r1 = np.ascontiguousarray(lu[sub]), np.ascontiguousarray(r[a:e])
            z1, two = np.zeros(e - a), np.array([0, e - a], dtype=np.int32)
            probe.probe_sweep(int(e - a), ip(p1), ip(c1), ip(d1), upper, 1, ip(two), levels, rows, ip(o1), ip(l1),
                              ip(r1), ip(z1), ip(out))
            assert np.array_equal(z1, z[a:e])


def shuffled(case, seed):
    """The same mesh, its cells numbered at random: few levels of many rows."""
    perm = np.arange(len(case.etype))
    vol = np.flatnonzero(case.etype >= 4)
    perm[vol] = np.random.default_rng(seed).permutation(vol)
    verts = [case.vidx[case.vptr[e]:case.vptr[e + 1]] for e in perm]
    ptr = np.concatenate([[0], np.cumsum([len(v) for v in verts])]).astype(np.int32)
    return s.CaseData(case.xyz, case.etype[perm].copy(), case.tag[perm].copy(), ptr,
                      np.concatenate(verts).astype(np.int32), case.regions, dict(case.meta))


def widest_level(ptr, col, diag):
    lev = [0] * len(diag)
    ptr, col, diag = ptr.tolist(), col.tolist(), diag.tolist()
    for i in range(len(lev)):
        lev[i] = max((lev[j] + 1 for j in col[ptr[i]:diag[i]]), default=0)
    return int(np.bincount(lev).max())


GPU_CASES = {
    "one_cell": lambda: s.cavity(1),
    "cavity3": lambda: s.cavity(3),
    "cavity17": lambda: s.cavity(17, jitter=0.1, seed=2),
    "tets": lambda: s.cavity(6, tets=True, jitter=0.1, seed=3),
    "split": lambda: s.channel(20, 9, 11, jitter=0.12, split=0.25, seed=6, re=400.0),
    "large": lambda: s.channel(120, 60, 60, jitter=0.1),
    # levels of more rows than a launch merges (and workgroups of 256 threads)
    "wide": lambda: shuffled(s.cavity(40, tets=True, jitter=0.1, seed=5), 1),
}


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [s.FP64, s.MIXED])
@pytest.mark.parametrize("name", sorted(GPU_CASES))
def test_first_preconditioned_step_matches_the_oracle(name, precision):
    """One GMRES iteration from a zero guess: x is a multiple of (LU)^-1 b, for
    each of the three momentum components."""
    from oracle.pyoracle import pc_apply

    case = GPU_CASES[name]()
    p = params(restart=30, pc=s.PC_ILU0)
    p.precision = precision
    p.graphs = 1
    d = s.Solver(case, p)
    st = random_state(d.sizes.n_cell, d.sizes.n_bnd, d.sizes.n_face, 7)
    push(d, {k: st[k] for k in ("U", "V", "W", "P", "R", "APR", "DPDX", "RUFACE")})
    d.call("build_velocity_matrix")  # momentum: no null space, three right-hand sides
    push(d, {k: np.zeros(d.sizes.n_cell) for k in ("U", "V", "W")})
    # a preconditioned step takes more than a hundredth off the residual
    info = d.solve_velocity(0.99, 1)
    assert [i["iters"] for i in info] == [1, 1, 1]
    pattern = d.ints("CSR_ROWPTR"), d.ints("CSR_COL"), d.ints("CSR_DIAG")
    if name == "wide":
        assert widest_level(*pattern) > 65536
    for k in "UVW":
        z = pc_apply(pattern[0], pattern[1], d.get("AU"), s.PC_ILU0, d.get("B%s_RHS" % k))
        x = d.get(k)
        scale = (x @ z) / (z @ z)
        # FP32 factors and sweeps: a few roundings per row, condition below 1e2
        assert rel_err(x, scale * z) <= (1e-11 if precision == s.FP64 else 3e-5), k
    d.close()
