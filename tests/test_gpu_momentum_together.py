"""The three momentum components solved together (one case) against one after
the other (a batch solves them so): the same bits, and the reference's order
of failures -- a component that fails leaves the later ones as they were."""
import numpy as np
import pytest

import sysu_cfd_parallel_amd as s
from helpers import params, push, random_state

pytestmark = pytest.mark.gpu

CASES = {
    "one": lambda: s.cavity(1),
    "odd": lambda: s.channel(11, 7, 5, jitter=0.1, split=0.35, seed=3, re=600.0),  # 1040 rows, the last tile short
    "unaligned": lambda: s.channel(9, 7, 5, jitter=0.1, re=400.0),  # 315 rows: V and W start off 16 bytes
    "hex": lambda: s.channel(11, 7, 5, jitter=0.1, re=400.0),
    "tets": lambda: s.step(2, downstream=6.0, tets=True, turbulent=False, re=400.0),
}
FORMS = [(s.FP64, s.PC_JACOBI, 0, 0), (s.FP64, s.PC_ILU0, 0, 1), (s.FP64, s.PC_NONE, 0, 1), (s.MIXED, s.PC_JACOBI, 2, 1),
         (s.MIXED, s.PC_JACOBI, 0, 0), (s.MIXED, s.PC_ILU0, 0, 0)]


def prepared(make, p):
    d = s.Solver(make(), p)
    st = random_state(d.sizes.n_cell, d.sizes.n_bnd, d.sizes.n_face, 5)
    push(d, {k: st[k] for k in ("U", "V", "W", "P", "R", "RUFACE")})
    d.call("build_velocity_matrix")
    return d, st


def form(precision, pc, order, graphs, restart=12):
    p = params(restart=restart, pc=pc)
    p.precision, p.inner_order, p.graphs = precision, order, graphs
    return p


@pytest.mark.parametrize("precision,pc,order,graphs", FORMS)
@pytest.mark.parametrize("name", sorted(CASES))
def test_together_equals_one_after_the_other(name, precision, pc, order, graphs):
    case = CASES[name]()
    p = form(precision, pc, order, graphs)
    alone, st = prepared(CASES[name], p)
    two = s.BatchSolver([case, s.cavity(2)], p)
    # the first case of a batch gets the same fields and system; its second is at rest
    for k in ("U", "V", "W", "AU", "BU_RHS", "BV_RHS", "BW_RHS"):
        f = two.get(k)
        if k == "AU":
            two.call("build_velocity_matrix")
            f = two.get(k)
        part = alone.get(k)
        f[:len(part)] = part
        two.set(k, f)
    ia = alone.solve_velocity(1e-8, 500)
    two.solve_velocity(1e-8, 500)
    ib = two.case_solve_info()
    for j, k in enumerate("UVW"):
        assert ia[j]["iters"] == ib[k][0]["iters"] and ia[j]["reason"] == ib[k][0]["reason"]
        assert np.array_equal(alone.get(k), two.case_field(0, k)), k
    alone.close()
    two.close()


@pytest.mark.parametrize("precision,pc", [(s.FP64, s.PC_JACOBI), (s.MIXED, s.PC_JACOBI), (s.FP64, s.PC_ILU0)])
def test_a_failed_component_leaves_the_later_ones(precision, pc):
    p = form(precision, pc, 0, 0, restart=30)
    d, st = prepared(CASES["odd"], p)
    full = [i["iters"] for i in d.solve_velocity(1e-8, 500)]
    done = {k: d.get(k) for k in "UVW"}
    assert min(full) > 1
    for cap in sorted({1, min(full), max(full) - 1}):
        first = next((j for j in range(3) if full[j] > cap), None)
        if first is None:
            continue
        push(d, {k: st[k] for k in "UVW"})
        with pytest.raises(s.NotConverged) as e:
            d.solve_velocity(1e-8, cap)
        for j, k in enumerate("UVW"):
            info = e.value.info[j]
            if j < first:
                assert info["reason"] > 0 and np.array_equal(d.get(k), done[k])
            elif j == first:
                assert info["reason"] < 0 and info["iters"] == cap
            else:
                assert info["iters"] == 0 and info["reason"] == 0
                assert np.array_equal(d.get(k), st[k])
    d.close()


@pytest.mark.parametrize("precision,order", [(s.FP64, 0), (s.MIXED, 0), (s.MIXED, 2)])
def test_momentum_products_are_timed(precision, order):
    """The in-solve SpMV timing sees the momentum solves, the results unchanged."""
    p = form(precision, s.PC_JACOBI, order, 0, restart=30)
    fields = []
    for on in (False, True):
        d, st = prepared(CASES["odd"], p)
        k = 1 if precision == s.MIXED else 0
        if on:
            d.spmv_profile(k, 1)
        its = [i["iters"] for i in d.solve_velocity(1e-8, 500)]
        if on:
            ms, n = d.spmv_profile(k, -1)
            assert 0 < n <= sum(its) + 3 * 8 and 0 < ms < 1
        fields.append((its, [d.get(x) for x in "UVW"]))
        d.close()
    assert fields[0][0] == fields[1][0]
    for a, b in zip(fields[0][1], fields[1][1]):
        assert np.array_equal(a, b)
