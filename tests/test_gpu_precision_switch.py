"""One context switched between the precision modes: every solve has the bits
of a context that never left its mode, whichever cycles were captured before
the switch."""
import numpy as np
import pytest

import sysu_cfd_parallel_amd as s
from helpers import params, push, random_state

pytestmark = pytest.mark.gpu


def mode(precision, pc, order):
    p = params(restart=30, pc=pc, rtol=1e-8, maxit=500)
    p.precision, p.inner_order, p.graphs = precision, order, 1
    return p


@pytest.mark.parametrize("pc,order", [(s.PC_JACOBI, 0), (s.PC_JACOBI, 2), (s.PC_NONE, 0), (s.PC_ILU0, 0)])
@pytest.mark.parametrize("first,second", [(s.MIXED, s.FP64), (s.FP64, s.MIXED)])
def test_switching_precision_there_and_back(first, second, pc, order):
    case = s.cavity(16, jitter=0.1, seed=4)

    def solve(d, rtol):
        push(d, {k: st[k] for k in "UVW"})
        its = [i["iters"] for i in d.solve_velocity(rtol, 500)]
        return its, [d.get(k) for k in "UVW"]

    def context(precision):
        d = s.Solver(case, mode(precision, pc, order))
        push(d, {k: st[k] for k in ("U", "V", "W", "P", "R", "RUFACE")})
        d.call("build_velocity_matrix")
        return d

    fresh = s.Solver(case, mode(first, pc, order))
    st = random_state(fresh.sizes.n_cell, fresh.sizes.n_bnd, fresh.sizes.n_face, 5)
    fresh.close()
    refs = {}
    for precision in (first, second):
        d = context(precision)
        refs[precision] = solve(d, 1e-8)
        d.close()
    d = context(first)
    short = solve(d, 0.1)[0]  # ends within the first captured steps
    for precision in (second, first, second, first):
        d.set_params(mode(precision, pc, order))
        its, fields = solve(d, 1e-8)
        assert its == refs[precision][0] and max(its) > max(short)
        for a, b in zip(fields, refs[precision][1]):
            assert np.array_equal(a, b)
    d.close()
