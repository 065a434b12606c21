"""Arnoldi steps of small systems in two launches (the SELL-64 product with its
dots; the sums, the update and the previous step's finalisation) against the
four launches of the one-lane CSR shape: the same sums in the same order, so the
same bits.  Sizes at the edges of tiles (256 rows), of 64-tile pieces and of
the range (256 tiles), cycles up to the longest."""
import numpy as np
import pytest

import sysu_cfd_parallel_amd as s
from helpers import params, push, random_state

pytestmark = pytest.mark.gpu

CASES = {
    "one": (lambda: s.cavity(1), 5),
    "tile": (lambda: s.channel(8, 8, 4, jitter=0.1), 30),
    "tile_and_a_bit": (lambda: s.channel(8, 8, 5, jitter=0.1, split=0.2), 8),
    "64_tiles": (lambda: s.channel(32, 32, 16), 9),
    "65_tiles": (lambda: s.channel(33, 32, 16, jitter=0.1), 64),
    "256_tiles": (lambda: s.channel(64, 32, 32, jitter=0.05), 50),
    "257_tiles": (lambda: s.channel(65, 32, 32, jitter=0.05), 16),  # past the range: four launches either way
}


@pytest.mark.parametrize("graphs", [0, 1])
@pytest.mark.parametrize("precision,order", [(s.FP64, 0), (s.MIXED, 0), (s.MIXED, 2)])
@pytest.mark.parametrize("name", sorted(CASES))
def test_two_launch_steps_equal_four(name, precision, order, graphs):
    make, restart = CASES[name]
    case = make()
    out = []
    for lanes in (1, 0):
        p = params(restart=restart, rtol=1e-8, maxit=150)
        p.precision, p.inner_order, p.graphs = precision, order, graphs
        d = s.Solver(case, p)
        d.set_kernel_shapes(1 if precision == s.MIXED else 0, lanes, rows=1, sigma=64 if lanes == 0 else 0)
        st = random_state(d.sizes.n_cell, d.sizes.n_bnd, d.sizes.n_face, 3)
        push(d, {k: st[k] for k in ("U", "V", "W", "P", "R", "APR", "DPDX", "RUFACE")})
        for k in ("bc_velocity", "cal_ru_face", "build_pressure_matrix"):
            d.call(k)
        runs = []
        for _ in range(3):  # graphs: replays with a change of the program between them
            try:
                info = d.solve_pressure(1e-8, 150)
            except s.NotConverged as e:
                info = e.info
            runs.append((info["iters"], info["reason"], info["rnorm"], d.get("DELTAP")))
            d.call("bc_deltap")
        assert all(r[:3] == runs[0][:3] and np.array_equal(r[3], runs[0][3]) for r in runs)
        out.append(runs[0])
        d.close()
    assert out[0][:3] == out[1][:3]
    assert np.array_equal(out[0][3], out[1][3])
